// Router GEMV and activation casts of the frontend, shared by the frontend kernel
// (dgm_megamoe.hip) and the fused kernel's in-kernel frontend (dgm_fused.hip). AGENT selects
// write-through agent-scope stores, for data that other workgroups of the same launch read.
#pragma once
#include "dgm_common.hpp"
#include "../../include/dgm_megamoe.h"

namespace dgm {

template <bool AGENT>
DGM_DEV void put8(uint8_t* p, uint32_t v) {
  if (AGENT) __hip_atomic_store(p, (uint8_t)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = (uint8_t)v;
}
template <bool AGENT>
DGM_DEV void put16(uint16_t* p, uint32_t v) {
  if (AGENT) __hip_atomic_store(p, (uint16_t)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = (uint16_t)v;
}
template <bool AGENT>
DGM_DEV void put32(uint32_t* p, uint32_t v) {
  if (AGENT) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}
template <bool AGENT>
DGM_DEV void put64(uint64_t* p, uint64_t v) {
  if (AGENT) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}

// Router: one wave computes the logits of expert e for tokens t0 .. t0 + 3 (rows past M are
// clamped and not written). Lane l accumulates K = 512 j + 8 l + i (j, then i ascending) with
// fp32 FMAs of exact bf16 products, then an xor butterfly (32..1) reduces the 64 lane sums: a
// fixed order, so the fp32 logits are reproducible bit for bit. Writes the fp32 logit and the
// top-k key (topk_key: orderable bf16 << 16 | 0xFFFF - e); with zero_unrouted, the keys of an
// all-zero hidden row are 0 (the token is unrouted).
// The logits of expert e (its router row wv, lane l holding K = 512 j + 8 l .. +7) for the four
// token rows xv (laid out the same way), in the order stated above; rows t0 + tt >= M are not
// written.
template <int J, bool AGENT>
DGM_DEV void router_dot4(const uint4 (&wv)[J], const uint4 (&xv)[4][J], int M, int E, int e, int t0, int lane,
                         float* __restrict__ logits, uint32_t* __restrict__ keys, bool zero_unrouted) {
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) {
    float acc = 0.f;
    uint32_t any = 0;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const uint32_t xa[4] = {xv[tt][j].x, xv[tt][j].y, xv[tt][j].z, xv[tt][j].w};
      const uint32_t wa[4] = {wv[j].x, wv[j].y, wv[j].z, wv[j].w};
#pragma unroll
      for (int qq = 0; qq < 4; ++qq) {
        acc = fmaf(__uint_as_float(xa[qq] << 16), __uint_as_float(wa[qq] << 16), acc);
        acc = fmaf(__uint_as_float(xa[qq] & 0xffff0000u), __uint_as_float(wa[qq] & 0xffff0000u), acc);
        any |= xa[qq] & 0x7fff7fffu;
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc = acc + __shfl_xor(acc, off);
    const bool unrouted = zero_unrouted && !__any(any != 0u);
    if (lane == 0 && t0 + tt < M && e < E) {
      const size_t o = (size_t)(t0 + tt) * E + e;
      put32<AGENT>(reinterpret_cast<uint32_t*>(logits) + o, __float_as_uint(acc));
      put32<AGENT>(keys + o, unrouted ? 0u : topk_key(acc, e));
    }
  }
}

template <int J, bool AGENT>
DGM_DEV void router_wave(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int M, int E, int e,
                         int t0, int lane, float* __restrict__ logits, uint32_t* __restrict__ keys,
                         bool zero_unrouted) {
  constexpr int H = J * 512;
  uint4 wv[J];
  const int ee = e < E ? e : E - 1;
#pragma unroll
  for (int j = 0; j < J; ++j) wv[j] = *reinterpret_cast<const uint4*>(w + (size_t)ee * H + 512 * j + 8 * lane);
  uint4 xv[4][J];
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) {
    const int t = t0 + tt < M ? t0 + tt : M - 1;
#pragma unroll
    for (int j = 0; j < J; ++j) xv[tt][j] = *reinterpret_cast<const uint4*>(x + (size_t)t * H + 512 * j + 8 * lane);
  }
  router_dot4<J, AGENT>(wv, xv, M, E, e, t0, lane, logits, keys, zero_unrouted);
}

// Router tile of a 256-thread workgroup for larger batches: the hidden rows of tokens
// t0 .. t0 + RT - 1 (clamped to M - 1) are staged in LDS once (xs: RT * J * 64 uint4) and wave w
// computes expert e0 + w for all of them from its router row in registers, four tokens at a
// time: each router row is read once per RT tokens and each hidden row once per four experts
// (the one-wave path reads the hidden rows once per expert). Same order of operations as
// router_wave, so the same bits.
template <int J, int RT, bool AGENT>
DGM_DEV void router_tile(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int M, int E, int e0,
                         int t0, float* __restrict__ logits, uint32_t* __restrict__ keys, bool zero_unrouted,
                         uint4* __restrict__ xs) {
  constexpr int H = J * 512, RV = RT * J * 64;       // uint4 per tile
  static_assert(RT % 4 == 0 && RV % 256 == 0, "tile of 4-token groups, whole rounds of 256 threads");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int e = e0 + wave, ee = e < E ? e : E - 1;
  uint4 wv[J];
#pragma unroll
  for (int j = 0; j < J; ++j) wv[j] = *reinterpret_cast<const uint4*>(w + (size_t)ee * H + 512 * j + 8 * lane);
  uint4 st[RV / 256];
#pragma unroll
  for (int i = 0; i < RV / 256; ++i) {
    const int v = 256 * i + tid, tt = v / (J * 64), c = v % (J * 64);
    const int t = t0 + tt < M ? t0 + tt : M - 1;
    st[i] = *reinterpret_cast<const uint4*>(x + (size_t)t * H + 8 * c);
  }
#pragma unroll
  for (int i = 0; i < RV / 256; ++i) xs[256 * i + tid] = st[i];
  __syncthreads();
#pragma unroll
  for (int g = 0; g < RT / 4; ++g) {
    uint4 xv[4][J];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
#pragma unroll
      for (int j = 0; j < J; ++j) xv[tt][j] = xs[(4 * g + tt) * (J * 64) + 64 * j + lane];
    }
    router_dot4<J, AGENT>(wv, xv, M, E, e, t0 + 4 * g, lane, logits, keys, zero_unrouted);
  }
}

// Router tile on the matrix cores: a 512-thread workgroup computes the logits of the 16 tokens
// t0 .. and 16 experts e0 .. (clamped to M - 1 and E - 1; rows and columns past them not
// written), bit for bit as router_wave does. The op V_MFMA_F32_16X16X1_4B_F32 has one K per
// instruction, so each of its results is one fp32 fma of an exact bf16 product, and its four
// blocks are four independent 16 x 16 accumulators: block b of wave w accumulates router_wave's
// lane sums of lanes l = 8 w + 4 h + b, h = 0, 1 (K = 512 j + 8 l + i, j then i ascending), for
// every (token, expert). The 64 lane sums then meet in the butterfly's order: l bits 5, 4 and 3 are
// the wave (through LDS), bit 2 is h, bits 1 and 0 the block.
// Bound by the matrix cores' fp32 rate, with the operand unpacking beside it: about 4 us per tile
// and CU at 6 x 512 K (54 clocks per op where the op alone takes 32), after 7 us for the first.
// E384 H3072, frontend + selection launch: 128 tokens 20.0 -> 12.6 us, 256 33.5 -> 17.8, 512
// 61.4 -> 26.4. Measured beside this: 16 waves of one lane group each 12.5 / 19.2 / 29.2, four waves
// of four groups (three workgroups per CU) 13.7 / 19.0 / 27.0.
struct RouterMmSmem {
  float red[8][2][16][64];      // [wave][h][accumulator register][lane]
  float blk[16][64];            // [4 block + row][lane]
  uint32_t any[8][16];          // [wave][token]: bits of the token's hidden values this wave read
};
template <int J>
DGM_DEV void router_tile_mm(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int M, int E, int e0, int t0,
                            float* __restrict__ logits, uint32_t* __restrict__ keys, bool zero_unrouted,
                            RouterMmSmem& sm) {
  typedef float v16f __attribute__((ext_vector_type(16)));
  constexpr int H = J * 512;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int b = lane >> 4, i = lane & 15;
  const uint16_t* xr = x + (size_t)(t0 + i < M ? t0 + i : M - 1) * H + 8 * (8 * wv + b);
  const uint16_t* wr = w + (size_t)(e0 + i < E ? e0 + i : E - 1) * H + 8 * (8 * wv + b);
  // (the two halves of each 128-byte line back to back)
  uint4 xv[J][2], rv[J][2];
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      xv[j][h] = *reinterpret_cast<const uint4*>(xr + 512 * j + 32 * h);
      rv[j][h] = *reinterpret_cast<const uint4*>(wr + 512 * j + 32 * h);
    }
  v16f acc[2] = {};
  uint32_t any = 0;
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int hl = 0; hl < 2; ++hl)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint32_t xa[4] = {xv[j][h].x, xv[j][h].y, xv[j][h].z, xv[j][h].w};
          const uint32_t wa[4] = {rv[j][h].x, rv[j][h].y, rv[j][h].z, rv[j][h].w};
          const uint32_t xb = hl ? xa[q] & 0xffff0000u : xa[q] << 16, wb = hl ? wa[q] & 0xffff0000u : wa[q] << 16;
          acc[h] = __builtin_amdgcn_mfma_f32_16x16x1f32(__uint_as_float(xb), __uint_as_float(wb), acc[h], 0, 0, 0);
          if (hl == 0) any |= xa[q] & 0x7fff7fffu;
        }
  // register 4 b + r of lane l: block b, token 4 (l / 16) + r, expert l % 16
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 16; ++r) sm.red[wv][h][r][lane] = acc[h][r];
  any |= (uint32_t)__shfl_xor((int)any, 16);
  any |= (uint32_t)__shfl_xor((int)any, 32);
  if (lane < 16) sm.any[wv][lane] = any;
  __syncthreads();
  // wave v sums registers 2 v and 2 v + 1: waves w and w + 4, + 2, + 1, then h
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    float s[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float a[8];
#pragma unroll
      for (int v = 0; v < 8; ++v) a[v] = sm.red[v][h][2 * wv + k][lane];
      s[h] = ((a[0] + a[4]) + (a[2] + a[6])) + ((a[1] + a[5]) + (a[3] + a[7]));
    }
    sm.blk[2 * wv + k][lane] = s[0] + s[1];
  }
  __syncthreads();
  if (wv < 4) {                 // blocks b and b + 2, then b and b + 1
    const float v = (sm.blk[wv][lane] + sm.blk[8 + wv][lane]) + (sm.blk[4 + wv][lane] + sm.blk[12 + wv][lane]);
    const int tt = 4 * b + wv, t = t0 + tt, e = e0 + i;
    if (t < M && e < E) {
      uint32_t nz = 0;
#pragma unroll
      for (int u = 0; u < 8; ++u) nz |= sm.any[u][tt];
      const size_t o = (size_t)t * E + e;
      logits[o] = v;
      keys[o] = zero_unrouted && nz == 0u ? 0u : topk_key(v, e);
    }
  }
}

// Cast lanes. MXFP4 / MXFP8: lane i of 8 per 32-element group g = i / 8 (4 elements each;
// MXFP4 rows with amax floor 1e-30, MXFP8 rows with amax floor 1e-4: the rules of
// dgm_cast_fp4_rows / dgm_cast_fp8_rows). NVFP4: 4 lanes per 16-element group (the W4A4 row
// cast: E4M3 (round to nearest even) of max(amax, 1e-30) / 6, ties-down E2M1 of x / sf). The
// lanes of a group must be adjacent and all active.
template <bool AGENT>
DGM_DEV void cast_lane_mx(const uint16_t* __restrict__ x, int act, int64_t i, uint8_t* __restrict__ q,
                          uint8_t* __restrict__ sf) {
  const int64_t g = i >> 3;
  const int part = (int)(i & 7);            // elements 4 part .. +3 of the group
  const uint2 raw = *reinterpret_cast<const uint2*>(x + g * 32 + 4 * part);
  const float v[4] = {__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u),
                      __uint_as_float(raw.y << 16), __uint_as_float(raw.y & 0xffff0000u)};
  float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
  amax = fmaxf(amax, __shfl_xor(amax, 1));
  amax = fmaxf(amax, __shfl_xor(amax, 2));
  amax = fmaxf(amax, __shfl_xor(amax, 4));
  if (act == DGM_ACT_MXFP4) {
    const uint32_t code = ceil_ue8m0_code(fmaxf(amax, 1e-30f) / 6.0f);
    const float sc = e8m0_value(code);
    uint32_t o = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) o |= e2m1_ties_down(v[k] / sc) << (4 * k);
    put16<AGENT>(reinterpret_cast<uint16_t*>(q) + g * 8 + part, o);
    if (part == 0) put8<AGENT>(sf + g, code);
  } else {
    const uint32_t code = ceil_ue8m0_code(fmaxf(amax, 1e-4f) / 448.0f);
    const float inv = 1.0f / e8m0_value(code);
    uint32_t o = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) o |= e4m3_encode(v[k] * inv) << (8 * k);
    put32<AGENT>(reinterpret_cast<uint32_t*>(q) + g * 8 + part, o);
    if (part == 0) put8<AGENT>(sf + g, code);
  }
}

template <bool AGENT>
DGM_DEV void cast_lane_nvfp4(const uint16_t* __restrict__ x, int64_t i, uint8_t* __restrict__ q,
                             uint8_t* __restrict__ sf) {
  const int64_t g = i >> 2;
  const int part = (int)(i & 3);
  const uint2 raw = *reinterpret_cast<const uint2*>(x + g * 16 + 4 * part);
  const float v[4] = {__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u),
                      __uint_as_float(raw.y << 16), __uint_as_float(raw.y & 0xffff0000u)};
  float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
  amax = fmaxf(amax, __shfl_xor(amax, 1));
  amax = fmaxf(amax, __shfl_xor(amax, 2));
  const uint32_t code = e4m3_encode(fmaxf(amax, 1e-30f) / 6.0f);
  const float sc = __builtin_amdgcn_cvt_f32_fp8((int)code, 0);
  uint32_t o = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) o |= e2m1_ties_down(v[k] / sc) << (4 * k);
  put16<AGENT>(reinterpret_cast<uint16_t*>(q) + g * 4 + part, o);
  if (part == 0) put8<AGENT>(sf + g, code);
}

// FP8 rows with one fp32 scale per 128 (per_token_cast_to_fp8(use_ue8m0=False, gran_k=128),
// deep_gemm/utils/math.py:26-38): 32 adjacent lanes per 128-element group, 4 elements each;
// sf = max(amax, 1e-4) / 448, E4M3 (round to nearest even) of x * (1 / sf) (IEEE division).
template <bool AGENT>
DGM_DEV void cast_lane_fp8f128(const uint16_t* __restrict__ x, int64_t i, uint8_t* __restrict__ q,
                               uint8_t* __restrict__ sf) {
  const int64_t g = i >> 5;
  const int part = (int)(i & 31);
  const uint2 raw = *reinterpret_cast<const uint2*>(x + g * 128 + 4 * part);
  const float v[4] = {__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u),
                      __uint_as_float(raw.y << 16), __uint_as_float(raw.y & 0xffff0000u)};
  float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
#pragma unroll
  for (int off = 1; off < 32; off <<= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
  const float s = fmaxf(amax, 1e-4f) / 448.0f;
  const float inv = 1.0f / s;
  uint32_t o = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) o |= e4m3_encode(v[k] * inv) << (8 * k);
  put32<AGENT>(reinterpret_cast<uint32_t*>(q) + g * 32 + part, o);
  if (part == 0) put32<AGENT>(reinterpret_cast<uint32_t*>(sf) + g, __float_as_uint(s));
}

// QoQ per-token int8 cast (per_token_cast_to_int8) of token t by one wave: lane l holds
// elements 512 j + 8 l .. +7; sf = max(amax, 1e-30) / 127 (fp32), q = clamp(rne(x / sf),
// +-127); the scale is repeated over the row's H / 128 slots.
template <int J, bool AGENT>
DGM_DEV void cast_qoq_token(const uint16_t* __restrict__ x, int t, int lane, uint8_t* __restrict__ q,
                            uint8_t* __restrict__ sf) {
  constexpr int H = J * 512;
  uint4 xv[J];
  float amax = 0.f;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    xv[j] = *reinterpret_cast<const uint4*>(x + (size_t)t * H + 512 * j + 8 * lane);
    const uint32_t d[4] = {xv[j].x, xv[j].y, xv[j].z, xv[j].w};
#pragma unroll
    for (int k = 0; k < 4; ++k)
      amax = fmaxf(amax, fmaxf(fabsf(__uint_as_float(d[k] << 16)), fabsf(__uint_as_float(d[k] & 0xffff0000u))));
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
  const float scale = fmaxf(amax, 1e-30f) / 127.0f;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const uint32_t d[4] = {xv[j].x, xv[j].y, xv[j].z, xv[j].w};
    uint32_t o[2] = {0u, 0u};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t bits = (k & 1) ? (d[k >> 1] & 0xffff0000u) : (d[k >> 1] << 16);
      const float v = fminf(fmaxf(rintf(__uint_as_float(bits) / scale), -127.f), 127.f);
      o[k >> 2] |= ((uint32_t)(int)v & 0xffu) << (8 * (k & 3));
    }
    put64<AGENT>(reinterpret_cast<uint64_t*>(q + (size_t)t * H + 512 * j + 8 * lane), (uint64_t)o[0] | ((uint64_t)o[1] << 32));
  }
  if (lane < H / 128) put32<AGENT>(reinterpret_cast<uint32_t*>(sf) + (size_t)t * (H / 128) + lane, __float_as_uint(scale));
}

}  // namespace dgm
