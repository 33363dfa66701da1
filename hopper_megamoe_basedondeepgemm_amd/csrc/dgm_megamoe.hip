// MegaMoE layer on MI355X (gfx950): the frontend kernels (router, top-k, activation casts), the
// combine of the calls that run the layer as several launches, and the C ABI. The experts run on
// the persistent kernel (dgm_fused.hip).
//
// Data layout in HBM (one GPU's share of the EP layer):
//  * weights: matrix-core fragment order written by dgm_transform_fp4_weights. A 16-row x
//    128-K tile is 1 KB and lane l of a wave loads bytes [16 l, 16 l + 16) of it with one
//    16-byte load: the whole wave reads the tile as one contiguous 1 KB run. Per-32 E8M0
//    scales of 4 consecutive K-tiles sit in one dword per lane.
//  * activations x: [tokens, H/2] E2M1 (low nibble = even K) or [tokens, H] E4M3, scales
//    [tokens, H/32]. Routed rows are read in place through the pool table (on one GPU the
//    per-expert pool is the list of routes; no row copies).
//  * intermediate (L1 -> L2): [pool row, I/2 | I] codes + [pool row, I/32] scales, pool rows
//    in (expert asc, token asc, slot asc) order.
//  * route outputs: bf16 [topk][tokens][H]; the combine sums valid slots in slot order.
#include "dgm_common.hpp"
#include "dgm_abi_internal.hpp"
#include "dgm_fused.hpp"
#include "dgm_frontend.hpp"

using namespace dgm;

namespace {

// ------------------------------------------------------------------ frontend
// Router rows of the grid (by < ceil(M / RTOK)): workgroup (bx, by) computes the logits and
// top-k keys of experts 4 bx .. +3 for tokens RTOK by .. +RTOK - 1 (fixed accumulation order,
// bit-reproducible fp32 logits; zero keys for an all-zero row when zero_unrouted): RT = 0, one
// wave per expert over 4 tokens (router_wave, RTOK = 4); RT > 0, the RT tokens' hidden rows
// staged in LDS and shared by the four waves (router_tile, RTOK = RT; the same bits). Cast rows
// (the rest of the grid, running beside the router rows rather than after them): MXFP4 / MXFP8
// 8 lanes per 32-element group, NVFP4 4 lanes per 16-element group, QoQ one wave per token
// (dgm_frontend.hpp).
// Tiled router rows from 64 tokens on (MI355X, E384 H3072, kernel + launch by events: 64 tokens
// 13.7 us against 15.2, 128 tokens 24.0 against 26.8; at 16 and 32 tokens the LDS staging and
// its barrier cost 1.1-1.7 us more than the hidden-row reads they save).
constexpr int FE_ROUTER_TILE = 8;         // tokens per router workgroup in the tiled form
constexpr int FE_TILE_MIN_TOKENS = 64;
// Matrix-core router tiles (router_tile_mm) beyond 64 tokens, for hidden sizes beyond 1024 only with more
// than 64 tiles of 16 tokens x 16 experts: a tile alone takes as long as a whole round of them (its
// K loop), which fewer tiles do not shorten, while the rows of eight tokens get shorter. Frontend +
// selection launch, us, rows against tiles:
//   H 3072, E 384: 80 tokens 16.8 / 12.7, 100 17.9 / 12.9, 128 20.3 / 12.8, 512 61.7 / 26.6
//           E 128: 128 tokens (64 tiles) 11.4 / 12.4, 160 (80) 12.9 / 12.8, 256 16.7 / 13.0
//           E 48: 128 tokens (24 tiles) 10.6 / 12.3, 384 (72) 13.0 / 12.9, 512 15.1 / 13.2
//   H 4096, E 128: 112 tokens (56 tiles) 12.7 / 14.7, 160 (80) 17.7 / 14.7; H 2048: 10.1 / 10.5, 11.0 / 10.6
//   H 1024, E 8: 80 tokens 8.3 / 7.5, E 48: 8.7 / 8.3; H 512, E 8: 8.1 / 6.4, E 384: 8.9 / 7.4
// Up to 64 tokens the rows stay (E 384 H 3072, 64 tokens 13.1 / 12.7, 32 tokens 10.2 / 12.3).
constexpr int FE_MM_MIN_TOKENS = 65, FE_MM_MIN_TILES = 65, FE_MM_ANY_TILES_HIDDEN = 1024;
// Phase stamps (the reference's DG_FE_STAMPS, deep_gemm/mega/__init__.py:743-756): with stamps
// non-null, workgroup b = blockIdx.y * gridDim.x + blockIdx.x < stamp_rows writes row b of 8
// int64: [0] entry, [3] (router rows) keys and logits stored by all four waves, [5] (cast rows)
// cast stored, [6] the hardware position (HW_ID | XCC_ID << 32), [7] exit; wall clock at 100 MHz.
DGM_DEV long long fe_clock() { return (long long)__builtin_amdgcn_s_memrealtime(); }
DGM_DEV long long fe_hw_position() {
  uint32_t hw, xcc;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_HW_ID)" : "=s"(hw));
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
  return (long long)hw | ((long long)(xcc & 0xffffu) << 32);
}

template <int J, int RT>
__global__ void __launch_bounds__(256) k_frontend(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                  int M, int E, int act_format, float* __restrict__ logits,
                                                  uint32_t* __restrict__ keys, int zero_unrouted,
                                                  uint8_t* __restrict__ q, uint8_t* __restrict__ sf, int router,
                                                  long long* __restrict__ stamps, int stamp_rows) {
  constexpr int H = J * 512, RTOK = RT > 0 ? RT : 4;
  __shared__ uint4 xs[RT > 0 ? RT * J * 64 : 1];
  // every argument (and the grid size) requested at entry behind one wait: left to the compiler,
  // the loads came in four dependent rounds, two of them misses on the two argument lines
  // (0.16-0.36 us of this kernel at 2-8 tokens)
  asm volatile("" ::"s"(x), "s"(w), "s"(M), "s"(E), "s"(act_format), "s"(logits), "s"(keys), "s"(zero_unrouted),
               "s"(q), "s"(sf), "s"(router), "s"(stamps), "s"(stamp_rows), "s"(gridDim.x), "s"(gridDim.y));
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ry = router ? (M + RTOK - 1) / RTOK : 0;
  const int brow = (int)(blockIdx.y * gridDim.x + blockIdx.x);
  long long* st = stamps != nullptr && brow < stamp_rows ? stamps + (size_t)brow * 8 : nullptr;
  const long long t_entry = st ? fe_clock() : 0;
  if ((int)blockIdx.y < ry) {
    if constexpr (RT > 0)
      router_tile<J, RT, false>(x, w, M, E, blockIdx.x * 4, blockIdx.y * RT, logits, keys, zero_unrouted != 0, xs);
    else
      router_wave<J, false>(x, w, M, E, blockIdx.x * 4 + wave, blockIdx.y * 4, lane, logits, keys, zero_unrouted != 0);
    if (st) {
      __syncthreads();
      if (tid == 0) {
        const long long t = fe_clock();
        st[0] = t_entry; st[1] = 0; st[2] = 0; st[3] = t; st[4] = 0; st[5] = 0;
        st[6] = fe_hw_position(); st[7] = fe_clock();
      }
    }
    return;
  }
  const int cy = (int)gridDim.y - ry, by = (int)blockIdx.y - ry;
  const int64_t lane0 = ((int64_t)by * gridDim.x + blockIdx.x) * 256 + tid;
  const int64_t nl = (int64_t)gridDim.x * cy * 256;
  if (act_format == DGM_ACT_QOQ) {
    const int nwaves = gridDim.x * cy * 4;
    for (int t = (by * (int)gridDim.x + (int)blockIdx.x) * 4 + wave; t < M; t += nwaves)
      cast_qoq_token<J, false>(x, t, lane, q, sf);
  } else if (act_format == DGM_ACT_NVFP4) {
    for (int64_t i = lane0; i < (int64_t)M * (H / 16) * 4; i += nl) cast_lane_nvfp4<false>(x, i, q, sf);
  } else if (act_format == DGM_ACT_FP8F128) {
    for (int64_t i = lane0; i < (int64_t)M * (H / 128) * 32; i += nl) cast_lane_fp8f128<false>(x, i, q, sf);
  } else {
    for (int64_t i = lane0; i < (int64_t)M * (H / 32) * 8; i += nl) cast_lane_mx<false>(x, act_format, i, q, sf);
  }
  if (st) {
    __syncthreads();
    if (tid == 0) {
      const long long t = fe_clock();
      st[0] = t_entry; st[1] = 0; st[2] = 0; st[3] = 0; st[4] = 0; st[5] = t;
      st[6] = fe_hw_position(); st[7] = fe_clock();
    }
  }
}

// The frontend by router tiles (fe_mm): workgroups [0, nr) are router tiles of 16 tokens x
// 16 experts on the matrix cores (router_tile_mm, experts fastest: with E % 128 == 0 an XCD then
// keeps one share of the router weights in its L2), the rest cast.
template <int J>
__global__ void __launch_bounds__(512, 4) k_frontend_mm(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                      int M, int E, int act_format, float* __restrict__ logits,
                                                      uint32_t* __restrict__ keys, int zero_unrouted,
                                                      uint8_t* __restrict__ q, uint8_t* __restrict__ sf, int nr,
                                                      long long* __restrict__ stamps, int stamp_rows) {
  constexpr int H = J * 512;
  __shared__ RouterMmSmem sm;
  const int tid = threadIdx.x, bid = (int)blockIdx.x;
  long long* st = stamps != nullptr && bid < stamp_rows ? stamps + (size_t)bid * 8 : nullptr;
  const long long t_entry = st ? fe_clock() : 0;
  if (bid < nr) {
    const int ne = (E + 15) / 16;
    router_tile_mm<J>(x, w, M, E, (bid % ne) * 16, (bid / ne) * 16, logits, keys, zero_unrouted != 0, sm);
  } else {
    const int64_t lane0 = (int64_t)(bid - nr) * 512 + tid, nl = (int64_t)((int)gridDim.x - nr) * 512;
    if (act_format == DGM_ACT_QOQ) {
      for (int t = (int)(lane0 >> 6); t < M; t += (int)(nl >> 6)) cast_qoq_token<J, false>(x, t, tid & 63, q, sf);
    } else if (act_format == DGM_ACT_NVFP4) {
      for (int64_t i = lane0; i < (int64_t)M * (H / 16) * 4; i += nl) cast_lane_nvfp4<false>(x, i, q, sf);
    } else if (act_format == DGM_ACT_FP8F128) {
      for (int64_t i = lane0; i < (int64_t)M * (H / 128) * 32; i += nl) cast_lane_fp8f128<false>(x, i, q, sf);
    } else {
      for (int64_t i = lane0; i < (int64_t)M * (H / 32) * 8; i += nl) cast_lane_mx<false>(x, act_format, i, q, sf);
    }
  }
  if (st) {
    __syncthreads();
    if (tid == 0) {
      const long long t = fe_clock();
      st[0] = t_entry; st[1] = 0; st[2] = 0; st[3] = bid < nr ? t : 0; st[4] = 0; st[5] = bid < nr ? 0 : t;
      st[6] = fe_hw_position(); st[7] = fe_clock();
    }
  }
}

// ------------------------------------------------------------------ top-k + softmax
// One wave per token over its key row (orderable(bf16(logit)) << 16 | (0xFFFF - e), -0 -> +0):
// k rounds of a wave-wide max select; softmax w_k = exp(v_k - v_0) / sum (sequential sum).
// Unrouted tokens (a zero first key) get idx -1 / weight 0; forced-balanced routing
// (DGM_FE_FORCE_BALANCED) gives slot s -> s G + (g + 7 s) % G with weight 1 / topk.
constexpr int SELECT_TPB = 4;           // tokens (waves) per workgroup
__global__ void __launch_bounds__(256) k_select(const uint32_t* __restrict__ keys, int M, int E, int topk, int flags,
                                                int token_offset, int64_t* __restrict__ topk_idx,
                                                float* __restrict__ topk_w) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * SELECT_TPB + (threadIdx.x >> 6);
  if (t >= M) return;
  int idx = -1;
  float wt = 0.f;
  const uint32_t* row = keys + (size_t)t * E;
  select_topk_wave([row](int e) { return row[e]; }, E, topk, (flags & DGM_FE_FORCE_BALANCED) != 0,
                   token_offset + t, lane, idx, wt);
  // (DGM_FE_RAW_WEIGHTS: the selected logit itself, no softmax)
  if ((flags & DGM_FE_RAW_WEIGHTS) && !(flags & DGM_FE_FORCE_BALANCED) && lane < topk && idx >= 0) wt = key_value(row[idx]);
  if (lane < topk) {
    topk_idx[(size_t)t * topk + lane] = idx;
    topk_w[(size_t)t * topk + lane] = wt;
  }
}

// Top-k keys of bf16 router logits [M, E] (the frontend's key of each logit, topk_key).
__global__ void __launch_bounds__(256) k_keys_bf16(const uint16_t* __restrict__ logits, int64_t n, int E,
                                                   uint32_t* __restrict__ keys) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  keys[i] = topk_key(bf16_to_f32(logits[i]), (int)(i % E));
}

// ------------------------------------------------------------------ combine
// y[t, n] = bf16(sum over valid local slots s ascending of float(partials[s, t, n])) (bf16 route
// outputs, fp32 sum).
__global__ void k_combine(const uint16_t* __restrict__ partials, int part_rows, const int64_t* __restrict__ topk_idx,
                          int M, int H, int topk, int expert_begin, int E_local, uint16_t* __restrict__ y) {
  const int t = blockIdx.y;
  const int n = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (t >= M || n >= H) return;
  // every local route's values are loaded first (one round trip), then summed in slot order
  // (fp32; a route of another rank adds nothing)
  constexpr int MAXK = 16;                         // (topk <= 16, checked on the host)
  uint2 v[MAXK];
  uint32_t use = 0;
#pragma unroll
  for (int s = 0; s < MAXK; ++s) {
    v[s] = make_uint2(0u, 0u);
    if (s < topk) {
      const int64_t g = topk_idx[(size_t)t * topk + s];
      const int64_t l = g - expert_begin;
      if (g >= 0 && l >= 0 && l < E_local) {
        use |= 1u << s;
        v[s] = *reinterpret_cast<const uint2*>(partials + ((size_t)s * part_rows + t) * H + n);
      }
    }
  }
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
#pragma unroll
  for (int s = 0; s < MAXK; ++s)
    if ((use >> s) & 1u) {
      s0 += __uint_as_float(v[s].x << 16);
      s1 += __uint_as_float(v[s].x & 0xffff0000u);
      s2 += __uint_as_float(v[s].y << 16);
      s3 += __uint_as_float(v[s].y & 0xffff0000u);
    }
  uint32_t lo = (uint32_t)f32_to_bf16(s0) | ((uint32_t)f32_to_bf16(s1) << 16);
  uint32_t hi = (uint32_t)f32_to_bf16(s2) | ((uint32_t)f32_to_bf16(s3) << 16);
  *reinterpret_cast<uint2*>(y + (size_t)t * H + n) = make_uint2(lo, hi);
}

// The counters as an L1 launch needs them, whatever the buffer held: the set that it will use (the
// parity word's; the launch itself clears the other one for the L2 launch) with no unit claimed and no
// workgroup counted. Without it a claim counter left over would pass units over, and a launch that waits
// for no arrival reports nothing.
__global__ void __launch_bounds__(64) k_open_counters(int* __restrict__ counters) {
  int* set = counters + CNT_SET0 + (counters[CNT_PARITY] & 1) * CNT_SET;
  if (threadIdx.x == 0) {
    set[CNT_STARTED] = 0;
    set[CNT_CLAIM] = 0;
  }
}

int g_cu_count = 0;

int cu_count() {
  if (g_cu_count == 0) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, dev) == hipSuccess) g_cu_count = prop.multiProcessorCount;
    if (g_cu_count <= 0) g_cu_count = 256;
  }
  return g_cu_count;
}

int launch_combine(const DgmMoeArgs* A, uint8_t* buf, const DgmBufferLayout* L, hipStream_t stream) {
  dim3 cg((A->hidden / 4 + 255) / 256, A->num_tokens);
  hipLaunchKernelGGL(k_combine, cg, dim3(256), 0, stream, (const uint16_t*)(buf + L->partials), L->max_tokens,
                     (const int64_t*)(buf + L->topk_idx), A->num_tokens, A->hidden, A->topk, A->expert_begin,
                     A->num_local_experts, (uint16_t*)A->y);
  return dgm_last_launch_status();
}

}  // namespace

// ==================================================================== C ABI
static thread_local char g_err[512];
void dgm_set_error(const char* msg) {
  strncpy(g_err, msg, sizeof(g_err) - 1);
  g_err[sizeof(g_err) - 1] = 0;
}

static bool fused_fits(const DgmMoeArgs* A);
static int fused_launch_phases(const DgmMoeArgs* A, int phases, hipStream_t stream);

extern "C" {

int dgm_version(void) { return 1; }
const char* dgm_last_error(void) { return g_err; }

int dgm_device_cu_count(void) { return cu_count(); }

int dgm_abi_struct_sizes(size_t* moe_args, size_t* buffer_layout) {
  DGM_CHECK_ARG(moe_args && buffer_layout, "null pointer");
  *moe_args = sizeof(DgmMoeArgs);
  *buffer_layout = sizeof(DgmBufferLayout);
  return 0;
}

int dgm_host_device_pointer(const void* host, void** device) {
  DGM_CHECK_ARG(host && device, "null pointer");
  hipError_t e = hipHostGetDevicePointer(device, const_cast<void*>(host), 0);
  if (e != hipSuccess) {
    dgm_set_error("hipHostGetDevicePointer failed: not pinned host memory");
    return (int)e;
  }
  return 0;
}

int dgm_fused_workgroups(int hidden, int intermediate, int act_format) {
  return dgm_fused_grid_blocks(hidden, intermediate, act_format);
}

int dgm_fused_last_form(int hidden, int intermediate, int act_format) {
  return dgm_fused_form(hidden, intermediate, act_format);
}

int dgm_fused_buffer_layout(int max_tokens, int num_experts, int num_local_experts, int topk,
                            int hidden, int intermediate, int act_format, DgmBufferLayout* out) {
  DGM_CHECK_ARG(out != nullptr, "null layout");
  DGM_CHECK_ARG(max_tokens > 0 && topk > 0 && topk <= 16, "max_tokens > 0, 0 < topk <= 16");
  DGM_CHECK_ARG(num_experts > 0 && num_experts <= 1024, "num_experts in (0, 1024]");
  DGM_CHECK_ARG(num_local_experts > 0 && num_local_experts <= num_experts, "num_local_experts");
  DGM_CHECK_ARG(hidden % 512 == 0 && intermediate % 128 == 0, "hidden % 512, intermediate % 128");
  DGM_CHECK_ARG(act_format >= DGM_ACT_MXFP4 && act_format <= DGM_ACT_FP8F128, "act_format");
  DGM_CHECK_ARG((int64_t)max_tokens * topk <= FUSED_BIG_ROUTES, "max_tokens * topk <= 4096");
  // scales: E8M0 bytes per 32 (MXFP); QoQ: fp32 per token repeated over H / 128 slots (the
  // same H / 32 bytes) and fp32 per 64 intermediate features (I / 16 bytes); NVFP4: E4M3
  // bytes per 16; FP8F128: fp32 per 128 K (H / 32 bytes) and E8M0 bytes per 32 intermediate
  // features, sized as QoQ's (so one buffer serves both layers of the split recipe)
  const DgmRowBytes rb = dgm_row_bytes(act_format, hidden, intermediate);
  const size_t xb = rb.x, mb = rb.mid, xsfb = rb.x_sf, msfb = rb.mid_sf;
  const int R = max_tokens * topk;
  size_t off = 0;
  memset(out, 0, sizeof(*out));
  out->x = off; off += dgm_align256((size_t)max_tokens * xb);
  out->x_sf = off; off += dgm_align256((size_t)max_tokens * xsfb);
  out->topk_idx = off; off += dgm_align256((size_t)R * 8);
  out->topk_weights = off; off += dgm_align256((size_t)R * 4);
  out->logits = off; off += dgm_align256((size_t)max_tokens * num_experts * 4);
  out->fe_keys = off; off += dgm_align256((size_t)max_tokens * num_experts * 4);
  out->pool = off; off += dgm_align256(dgm_pool_bytes(num_local_experts, R));
  out->mid = off; off += dgm_align256((size_t)R * mb);
  out->mid_sf = off; off += dgm_align256((size_t)R * msfb);
  out->partials = off; off += dgm_align256((size_t)R * hidden * 2);     // bf16 [topk][max_tokens][H]
  out->counters = off; off += dgm_align256((size_t)CNT_ALL * 4);
  out->total_bytes = off;
  out->x_row_bytes = (int32_t)xb;
  out->mid_row_bytes = (int32_t)mb;
  out->max_routes = R;
  out->max_tokens = max_tokens;
  out->topk = topk;
  out->num_experts = num_experts;
  out->num_local_experts = num_local_experts;
  out->hidden = hidden;
  out->intermediate = intermediate;
  out->act_format = act_format;
  out->x_sf_row_bytes = (int32_t)xsfb;
  out->mid_sf_row_bytes = (int32_t)msfb;
  return 0;
}

}  // extern "C"

int dgm_check_layout_call(const DgmBufferLayout* L, int num_tokens, int topk, int num_experts, int num_local_experts,
                          int hidden, int intermediate, int act_format) {
  DGM_CHECK_ARG(L != nullptr, "null layout");
  DGM_CHECK_ARG(L->max_routes == L->max_tokens * L->topk && L->topk > 0,
                "the layout was not made by dgm_fused_buffer_layout");
  DGM_CHECK_ARG(num_tokens >= 0 && num_tokens <= L->max_tokens, "num_tokens exceeds the buffer's max_tokens");
  DGM_CHECK_ARG(topk > 0 && topk <= L->topk, "topk exceeds the buffer's topk (route outputs are [topk][max_tokens][H])");
  DGM_CHECK_ARG(num_experts > 0 && num_experts <= L->num_experts, "num_experts exceeds the buffer's");
  DGM_CHECK_ARG(num_local_experts < 0 || num_local_experts <= L->num_local_experts,
                "num_local_experts exceeds the buffer's (dispatch table)");
  DGM_CHECK_ARG(hidden == L->hidden, "hidden differs from the buffer's");
  DGM_CHECK_ARG(intermediate < 0 || intermediate == L->intermediate, "intermediate differs from the buffer's");
  const DgmRowBytes rb = dgm_row_bytes(act_format, hidden, intermediate < 0 ? L->intermediate : intermediate);
  DGM_CHECK_ARG(rb.x <= (size_t)L->x_row_bytes && rb.x_sf <= (size_t)L->x_sf_row_bytes,
                "the activation format needs wider x / x_sf rows than the buffer's");
  DGM_CHECK_ARG(intermediate < 0 || (rb.mid <= (size_t)L->mid_row_bytes && rb.mid_sf <= (size_t)L->mid_sf_row_bytes),
                "the activation format needs wider intermediate rows than the buffer's");
  return 0;
}

static int fe_tiles(int num_tokens, int num_experts) { return ((num_experts + 15) / 16) * ((num_tokens + 15) / 16); }
// Whether the router runs as matrix-core tiles
static bool fe_mm(int num_tokens, int hidden, int num_experts, bool router) {
  return router && num_tokens >= FE_MM_MIN_TOKENS &&
         (hidden <= FE_MM_ANY_TILES_HIDDEN || fe_tiles(num_tokens, num_experts) >= FE_MM_MIN_TILES);
}

// The frontend launch's grid: router tiles (fe_mm) or rows (4 experts x 4 tokens per workgroup, 8
// tokens from FE_TILE_MIN_TOKENS on) and, beside them, cast rows of one cast lane per thread (QoQ: one wave
// per token).
static dim3 fe_grid(int num_tokens, int hidden, int num_experts, int act_format, int flags, bool router) {
  const int rx = (num_experts + 3) / 4;
  const int64_t cast_threads = act_format == DGM_ACT_QOQ       ? (int64_t)num_tokens * 64
                               : act_format == DGM_ACT_NVFP4   ? (int64_t)num_tokens * (hidden / 16) * 4
                               : act_format == DGM_ACT_FP8F128 ? (int64_t)num_tokens * (hidden / 128) * 32
                                                               : (int64_t)num_tokens * (hidden / 32) * 8;
  const int64_t cast_rows = (flags & DGM_FE_NO_CAST) ? 0 : (cast_threads + (int64_t)rx * 256 - 1) / ((int64_t)rx * 256);
  if (fe_mm(num_tokens, hidden, num_experts, router))
    return dim3(fe_tiles(num_tokens, num_experts) + ((flags & DGM_FE_NO_CAST) ? 0 : (int)((cast_threads + 511) / 512)));
  const int rtok = num_tokens >= FE_TILE_MIN_TOKENS ? FE_ROUTER_TILE : 4;
  return dim3(rx, (router ? (num_tokens + rtok - 1) / rtok : 0) + (int)cast_rows);
}

extern "C" {

int dgm_frontend_workgroups(int num_tokens, int hidden, int num_experts, int act_format, int flags, int router) {
  if (num_tokens <= 0 || hidden <= 0 || num_experts <= 0) return 0;
  const dim3 g = fe_grid(num_tokens, hidden, num_experts, act_format, flags, router != 0);
  return (int)(g.x * g.y);
}

int dgm_router_topk_launch(const void* hidden_bf16, const void* router_weight_bf16, int num_tokens,
                           int hidden, int num_experts, int topk, int act_format, int flags,
                           int token_offset, void* buffer, const DgmBufferLayout* L, hipStream_t stream) {
  return dgm_router_topk_launch_stamped(hidden_bf16, router_weight_bf16, num_tokens, hidden, num_experts, topk,
                                        act_format, flags, token_offset, buffer, L, nullptr, 0, stream);
}

int dgm_router_topk_launch_stamped(const void* hidden_bf16, const void* router_weight_bf16, int num_tokens,
                                   int hidden, int num_experts, int topk, int act_format, int flags,
                                   int token_offset, void* buffer, const DgmBufferLayout* L, int64_t* stamps,
                                   int stamp_rows, hipStream_t stream) {
  DGM_CHECK_ARG(buffer && L && (hidden_bf16 || num_tokens == 0), "null pointer");   // (no tokens: no rows)
  DGM_CHECK_ARG(topk > 0 && topk <= 16 && topk <= num_experts, "topk");
  DGM_CHECK_ARG(act_format >= DGM_ACT_MXFP4 && act_format <= DGM_ACT_FP8F128, "act_format");
  {
    const int chk = dgm_check_layout_call(L, num_tokens, topk, num_experts, -1, hidden, -1, act_format);
    if (chk) return chk;
  }
  DGM_CHECK_ARG(num_experts <= 1024, "num_experts <= 1024");
  DGM_CHECK_ARG(hidden % 512 == 0, "hidden % 512 == 0");
  DGM_CHECK_ARG(!(flags & DGM_FE_FORCE_BALANCED) || num_experts % topk == 0, "forced-balanced needs E % topk == 0");
  DGM_CHECK_ARG(act_format >= DGM_ACT_MXFP4 && act_format <= DGM_ACT_FP8F128, "act_format");
  DGM_CHECK_ARG(((uintptr_t)hidden_bf16 & 15) == 0 && ((uintptr_t)router_weight_bf16 & 15) == 0, "16-byte alignment");
  DGM_CHECK_ARG(router_weight_bf16 || !(flags & (DGM_FE_FORCE_BALANCED | DGM_FE_ZERO_ROW_UNROUTED | DGM_FE_SELECT_IN_MEGA)),
                "cast only (router_weight NULL): no routing flags");
  DGM_CHECK_ARG(router_weight_bf16 || !(flags & DGM_FE_NO_CAST), "DGM_FE_NO_CAST needs the router weight");
  if (num_tokens == 0) return 0;
  DGM_CHECK_ARG(stamp_rows >= 0 && (stamps != nullptr || stamp_rows == 0), "stamps / stamp_rows");
  uint8_t* buf = (uint8_t*)buffer;
  const int J = hidden / 512;
  const int router = router_weight_bf16 ? 1 : 0;
  const bool tiled = num_tokens >= FE_TILE_MIN_TOKENS, mm = fe_mm(num_tokens, hidden, num_experts, router != 0);
  const dim3 rg = fe_grid(num_tokens, hidden, num_experts, act_format, flags, router != 0);
  long long* stamp_ptr = (long long*)stamps;
  const uint16_t* x = (const uint16_t*)hidden_bf16;
  const uint16_t* w = (const uint16_t*)router_weight_bf16;
  float* logits = (float*)(buf + L->logits);
  uint32_t* keys = (uint32_t*)(buf + L->fe_keys);
  const int zero_unrouted = (flags & DGM_FE_ZERO_ROW_UNROUTED) ? 1 : 0;
#define DGM_FE(JJ)                                                                                           \
  if (mm)                                                                                                    \
    hipLaunchKernelGGL((k_frontend_mm<JJ>), rg, dim3(512), 0, stream, x, w, num_tokens, num_experts, act_format, \
                       logits, keys, zero_unrouted, buf + L->x, buf + L->x_sf,                               \
                       fe_tiles(num_tokens, num_experts), stamp_ptr, stamp_rows);                            \
  else if (tiled)                                                                                            \
    hipLaunchKernelGGL((k_frontend<JJ, FE_ROUTER_TILE>), rg, dim3(256), 0, stream, x, w, num_tokens, num_experts, \
                       act_format, logits, keys, zero_unrouted, buf + L->x, buf + L->x_sf, router, stamp_ptr, \
                       stamp_rows);                                                                          \
  else                                                                                                       \
    hipLaunchKernelGGL((k_frontend<JJ, 0>), rg, dim3(256), 0, stream, x, w, num_tokens, num_experts,            \
                       act_format, logits, keys, zero_unrouted, buf + L->x, buf + L->x_sf, router, stamp_ptr,   \
                       stamp_rows)
  switch (J) {
    case 1: DGM_FE(1); break;
    case 2: DGM_FE(2); break;
    case 4: DGM_FE(4); break;
    case 6: DGM_FE(6); break;
    case 8: DGM_FE(8); break;
    default: DGM_CHECK_ARG(false, "hidden must be 512, 1024, 2048, 3072 or 4096");
  }
#undef DGM_FE
  int st = dgm_last_launch_status();
  if (st || (flags & DGM_FE_SELECT_IN_MEGA) || !router) return st;
  hipLaunchKernelGGL(k_select, dim3((num_tokens + SELECT_TPB - 1) / SELECT_TPB), dim3(256), 0, stream, keys, num_tokens,
                     num_experts, topk, flags, token_offset, (int64_t*)(buf + L->topk_idx),
                     (float*)(buf + L->topk_weights));
  return dgm_last_launch_status();
}

int dgm_router_logits_topk_launch(const void* logits_bf16, int num_tokens, int num_experts, int topk, int flags,
                                  int token_offset, void* buffer, const DgmBufferLayout* L, hipStream_t stream) {
  DGM_CHECK_ARG(buffer && L && (logits_bf16 || num_tokens == 0), "null pointer");
  DGM_CHECK_ARG(topk > 0 && topk <= 16 && topk <= num_experts, "topk");
  {
    // (no activation rows are written: the buffer's own format and hidden size)
    const int chk = dgm_check_layout_call(L, num_tokens, topk, num_experts, -1, L->hidden, -1, L->act_format);
    if (chk) return chk;
  }
  DGM_CHECK_ARG(num_experts > 0 && num_experts <= 1024, "num_experts <= 1024");
  DGM_CHECK_ARG(!(flags & DGM_FE_FORCE_BALANCED) || num_experts % topk == 0, "forced-balanced needs E % topk == 0");
  DGM_CHECK_ARG(!(flags & DGM_FE_ZERO_ROW_UNROUTED), "zero-row unrouting needs the hidden rows (dgm_router_topk_launch)");
  if (num_tokens == 0) return 0;
  uint8_t* buf = (uint8_t*)buffer;
  uint32_t* keys = (uint32_t*)(buf + L->fe_keys);
  const int64_t n = (int64_t)num_tokens * num_experts;
  hipLaunchKernelGGL(k_keys_bf16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, (const uint16_t*)logits_bf16, n,
                     num_experts, keys);
  int st = dgm_last_launch_status();
  if (st || (flags & DGM_FE_SELECT_IN_MEGA)) return st;
  hipLaunchKernelGGL(k_select, dim3((num_tokens + SELECT_TPB - 1) / SELECT_TPB), dim3(256), 0, stream, keys, num_tokens,
                     num_experts, topk, flags, token_offset, (int64_t*)(buf + L->topk_idx),
                     (float*)(buf + L->topk_weights));
  return dgm_last_launch_status();
}

// The key array the top-k is selected from under select_in_mega: the caller's, else the buffer's
// (written by a DGM_FE_SELECT_IN_MEGA frontend call).
static const uint32_t* select_keys(const DgmMoeArgs* A, uint8_t* buf, const DgmBufferLayout* L) {
  return A->fe_keys ? (const uint32_t*)A->fe_keys : (const uint32_t*)(buf + L->fe_keys);
}

// Writes topk_idx / topk_weights from the select keys for the paths that read them.
static int materialize_topk(const DgmMoeArgs* A, uint8_t* buf, const DgmBufferLayout* L, hipStream_t stream) {
  hipLaunchKernelGGL(k_select, dim3((A->num_tokens + SELECT_TPB - 1) / SELECT_TPB), dim3(256), 0, stream,
                     select_keys(A, buf, L), A->num_tokens, A->num_experts, A->topk, A->fe_flags,
                     A->token_offset, (int64_t*)(buf + L->topk_idx), (float*)(buf + L->topk_weights));
  return dgm_last_launch_status();
}

// Every workgroup of the fused kernel reads all tokens' logits when it selects the top-k; that
// costs ~1 us of SIMD time per token and workgroup (the selection rounds are sequential), so
// above SELECT_IN_MEGA_FAST_TOKENS a separate selection launch (one wave per token over the
// whole GPU) comes first and the fused kernel reads the result. Forced-balanced routing scans
// no keys, so it is selected in the kernel up to SELECT_IN_MEGA_FAST_BALANCED tokens (at 16
// tokens 0.5-1.4 us less than the extra launch; at 32 and 64 no gain). The in-kernel frontend
// (fe_in_mega) selects in the kernel up to SELECT_IN_MEGA_MAX_TOKENS.
constexpr int SELECT_IN_MEGA_MAX_TOKENS = 64;
constexpr int SELECT_IN_MEGA_FAST_TOKENS = 8;     // (one token per wave)
constexpr int SELECT_IN_MEGA_FAST_BALANCED = 16;

int dgm_megamoe_fused_launch(const DgmMoeArgs* A, hipStream_t stream) {
  const int chk = dgm_check_fused_args(A);
  if (chk) return chk;
  if (A->num_tokens == 0) return 0;
  if (fused_fits(A)) return fused_launch_phases(A, 3, stream);
  DGM_CHECK_ARG(A->act_format != DGM_ACT_QOQ && A->act_format != DGM_ACT_NVFP4,
                "QoQ / NVFP4 layer: at most 1024 routes (tokens x topk), 256 tokens and 512 local experts per call");
  DGM_CHECK_ARG(!A->fe_in_mega, "fe_in_mega: the fused kernel's limits (tokens, routes, local experts) are exceeded");
  return dgm_megamoe_split_launch(A, stream);
}

}  // extern "C"

int dgm_check_fused_args(const DgmMoeArgs* A) {
  DGM_CHECK_ARG(A && A->buffer && A->layout && (A->y || A->num_tokens == 0), "null pointer");
  DGM_CHECK_ARG(A->w1_values && A->w1_scales && A->w2_values && A->w2_scales, "null weights");
  const DgmBufferLayout* L = A->layout;
  DGM_CHECK_ARG(A->topk > 0 && A->topk <= 16, "topk");
  DGM_CHECK_ARG(A->act_format >= DGM_ACT_MXFP4 && A->act_format <= DGM_ACT_FP8F128, "act_format");
  {
    const int chk = dgm_check_layout_call(L, A->num_tokens, A->topk, A->num_experts, A->num_local_experts, A->hidden,
                                          A->intermediate, A->act_format);
    if (chk) return chk;
  }
  DGM_CHECK_ARG(A->num_local_experts > 0 && A->num_local_experts <= FUSED_BIG_LOCAL, "num_local_experts");
  DGM_CHECK_ARG(A->expert_begin >= 0 && A->expert_begin + A->num_local_experts <= A->num_experts, "expert range");
  DGM_CHECK_ARG(A->act_format >= DGM_ACT_MXFP4 && A->act_format <= DGM_ACT_FP8F128, "act_format");
  DGM_CHECK_ARG(A->act_format != DGM_ACT_QOQ || (A->w1_row_scales && A->w2_row_scales),
                "QoQ needs the row scales s1 of both matrices");
  DGM_CHECK_ARG(A->topk > 0 && A->topk <= 16, "topk");
  DGM_CHECK_ARG(A->hidden % 128 == 0 && A->intermediate % 32 == 0, "shape");
  DGM_CHECK_ARG(A->intermediate % 128 == 0, "intermediate % 128 == 0");
  if (A->fe_in_mega) {
    DGM_CHECK_ARG(A->hidden_states && A->router_weight, "fe_in_mega: null hidden_states / router_weight");
    DGM_CHECK_ARG(((uintptr_t)A->hidden_states & 15) == 0 && ((uintptr_t)A->router_weight & 15) == 0, "16-byte alignment");
    DGM_CHECK_ARG(A->num_tokens <= SELECT_IN_MEGA_MAX_TOKENS, "fe_in_mega: num_tokens <= 64");
    DGM_CHECK_ARG(A->hidden % 512 == 0, "fe_in_mega: hidden % 512 == 0");
    DGM_CHECK_ARG(A->topk <= A->num_experts && A->num_experts <= 1024, "fe_in_mega: topk, num_experts");
    DGM_CHECK_ARG(!(A->fe_flags & DGM_FE_FORCE_BALANCED) || A->num_experts % A->topk == 0,
                  "forced-balanced needs E % topk == 0");
  }
  return 0;
}

// The plain persistent form's limits (route, token, expert and combine-block counts of its LDS
// tables): within them the whole layer is one launch. Beyond them MXFP4, MXFP8 and FP8F128
// activations run the large-batch form, one launch per phase, whose tables hold every call that a
// buffer layout admits.
static bool fused_fits(const DgmMoeArgs* A) {
  return !fused_needs_big(A->num_tokens, A->topk, A->num_local_experts) && A->hidden / 64 <= FUSED_MAX_NB64;
}
// One launch of the persistent kernel running `phases` (FusedParams::phases) of the layer, with
// the buffer's own workspace views.
static int fused_launch_phases(const DgmMoeArgs* A, int phases, hipStream_t stream) {
  const DgmBufferLayout* L = A->layout;
  uint8_t* buf = (uint8_t*)A->buffer;
  DgmWorkspace w;
  w.pool = buf + L->pool;
  w.mid = buf + L->mid;
  w.mid_sf = buf + L->mid_sf;
  w.partials = (uint16_t*)(buf + L->partials);
  w.part_rows = L->max_tokens;
  w.counters = (int*)(buf + L->counters);
  return dgm_fused_launch_ws(A, phases, w, stream);
}

int dgm_fused_launch_ws(const DgmMoeArgs* A, int phases, const DgmWorkspace& w, hipStream_t stream) {
  const DgmBufferLayout* L = A->layout;
  uint8_t* buf = (uint8_t*)A->buffer;
  {
    const int fast = (A->fe_flags & DGM_FE_FORCE_BALANCED) ? SELECT_IN_MEGA_FAST_BALANCED : SELECT_IN_MEGA_FAST_TOKENS;
    // (the large-batch form reads the top-k; the kernel's selection has no raw weights)
    const bool raw = (A->fe_flags & DGM_FE_RAW_WEIGHTS) && !(A->fe_flags & DGM_FE_FORCE_BALANCED);
    const bool sel = (A->fe_in_mega || (A->select_in_mega && A->num_tokens <= fast && !raw)) && (phases & 1) && fused_fits(A);
    if (A->select_in_mega && !sel && (phases & 1)) {
      int st = materialize_topk(A, buf, L, stream);
      if (st) return st;
    }
    FusedParams p;
    p.w1v = (const uint8_t*)A->w1_values;
    p.w1s = (const uint32_t*)A->w1_scales;
    p.w2v = (const uint8_t*)A->w2_values;
    p.w2s = (const uint32_t*)A->w2_scales;
    p.w1r = A->act_format == DGM_ACT_QOQ ? (const float*)A->w1_row_scales : nullptr;
    p.w2r = A->act_format == DGM_ACT_QOQ ? (const float*)A->w2_row_scales : nullptr;
    p.gs1 = A->act_format == DGM_ACT_NVFP4 ? A->l1_global_scales : nullptr;
    p.gs2 = A->act_format == DGM_ACT_NVFP4 ? A->l2_global_scales : nullptr;
    p.x = buf + L->x;
    p.xsf = buf + L->x_sf;
    p.topk_idx = (int64_t*)(buf + L->topk_idx);
    p.topk_w = (float*)(buf + L->topk_weights);
    // (the in-kernel frontend writes the buffer's own keys and logits)
    p.keys = A->fe_in_mega ? (const uint32_t*)(buf + L->fe_keys) : select_keys(A, buf, L);
    p.logits = (float*)(buf + L->logits);
    p.select = sel ? 1 : 0;
    p.fe_in = A->fe_in_mega ? 1 : 0;
    p.hidden = (const uint16_t*)A->hidden_states;
    p.router_w = (const uint16_t*)A->router_weight;
    p.fe_flags = A->fe_flags;
    p.token_offset = A->token_offset;
    p.E = A->num_experts;
    p.mid = w.mid;
    p.mid_sf = w.mid_sf;
    p.partials = w.partials;
    p.part_rows = w.part_rows;
    p.y = (uint16_t*)A->y;
    p.pool_out = w.pool;
    p.recv_stats = A->recv_stats;
    p.counters = w.counters;
    p.host_err = A->host_error;
    p.M = A->num_tokens;
    p.topk = A->topk;
    p.expert_begin = A->expert_begin;
    p.E_local = A->num_local_experts;
    p.clamp = A->activation_clamp;
    p.fast_math = A->fast_math;
    p.spin_limit = 1 << 22;
    p.stamps = (long long*)A->phase_stamps;
    // (debug bit 1: phase_stamps receives the QoQ L1 accumulators instead of stamps)
    p.stamp_rows = A->phase_stamps && !(A->debug_flags & 2) ? A->phase_stamp_rows : 0;
    p.phases = phases;
    p.debug = (int16_t)(A->debug_flags & 31);
    // (a cooperative launch costs 14-19 us of its own: only where there is something to wait for. Both
    // launches of a split call made cooperatively: E384, 2 tokens A-MXFP8 70 us, plainly 34)
    return launch_fused(p, A->hidden, A->intermediate, A->act_format, stream,
                        (A->launch_flags & DGM_LAUNCH_COOPERATIVE) && fused_launch_waits(phases, A->fe_in_mega != 0));
  }
}

extern "C" {

int dgm_megamoe_split_launch(const DgmMoeArgs* A, hipStream_t stream) {
  DGM_CHECK_ARG(A && A->buffer && A->layout && (A->y || A->num_tokens == 0), "null pointer");
  DGM_CHECK_ARG(A->act_format >= DGM_ACT_MXFP4 && A->act_format <= DGM_ACT_FP8F128, "act_format");
  DGM_CHECK_ARG(!A->fe_in_mega, "split path: fe_in_mega is a fused-launch option");
  DGM_CHECK_ARG(A->topk > 0 && A->topk <= 16, "topk");
  {
    const int chk = dgm_check_layout_call(A->layout, A->num_tokens, A->topk, A->num_experts, A->num_local_experts,
                                          A->hidden, A->intermediate, A->act_format);
    if (chk) return chk;
  }
  if (A->act_format == DGM_ACT_QOQ || A->act_format == DGM_ACT_NVFP4) {
    // two launches of the persistent kernel: dispatch + L1, then L2 + combine
    DGM_CHECK_ARG(A->w1_values && A->w1_scales && A->w2_values && A->w2_scales, "null weights");
    DGM_CHECK_ARG(A->act_format != DGM_ACT_QOQ || (A->w1_row_scales && A->w2_row_scales),
                  "QoQ needs the row scales s1 of both matrices");
    DGM_CHECK_ARG(A->num_tokens >= 0 && (int64_t)A->num_tokens * A->topk <= A->layout->max_routes,
                  "num_tokens exceeds the buffer");
    DGM_CHECK_ARG(A->topk > 0 && A->topk <= 16, "topk");
    DGM_CHECK_ARG(A->num_local_experts > 0 && A->expert_begin >= 0 &&
                  A->expert_begin + A->num_local_experts <= A->num_experts, "expert range");
    DGM_CHECK_ARG(A->hidden % 128 == 0 && A->intermediate % 128 == 0, "shape");
    if (A->num_tokens == 0) return 0;
    DGM_CHECK_ARG(fused_fits(A), "QoQ / NVFP4 layer: at most 1024 routes (tokens x topk), 256 tokens and 512 local experts per call");
    int st = fused_launch_phases(A, 1, stream);
    if (st) return st;
    return fused_launch_phases(A, 2, stream);
  }
  const DgmBufferLayout* L = A->layout;
  DGM_CHECK_ARG(A->num_tokens >= 0 && (int64_t)A->num_tokens * A->topk <= L->max_routes, "num_tokens exceeds the buffer");
  DGM_CHECK_ARG(A->num_local_experts > 0 && A->num_local_experts <= FUSED_BIG_LOCAL, "num_local_experts");
  if (A->num_tokens == 0) return 0;
  // the persistent kernel twice (dispatch + L1, then L2), then the combine: no launch has a wait
  // on another workgroup, so none needs its grid resident at once (E384, 257 tokens, FP8F128:
  // 389 us; with the launches this replaced, see FORM_BIG, 989 us). These calls keep nothing in the
  // buffer from one to the next, the counters included
  hipLaunchKernelGGL(k_open_counters, dim3(1), dim3(64), 0, stream, (int*)((uint8_t*)A->buffer + L->counters));
  int st = dgm_last_launch_status();
  if (!st) st = fused_launch_phases(A, 1, stream);
  if (!st) st = fused_launch_phases(A, 2 | 4, stream);
  return st ? st : launch_combine(A, (uint8_t*)A->buffer, L, stream);
}

}  // extern "C"
