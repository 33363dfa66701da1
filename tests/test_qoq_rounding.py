"""The QoQ packer's rounding without divisions, over every operand it can meet: the products with a
rounded reciprocal, added to a constant that ends their precision above the reciprocal's error, give
the integers that the fp32 quotients give. (fmas in float64: those sums are exact there.)"""
import numpy as np
import pytest

F, D = np.float32, np.float64


@pytest.mark.parametrize("bits", [8, 11])      # significant bits of a bf16 / fp16 source
@pytest.mark.parametrize("scale", [-60, 0, 60])
def test_row_quotients(bits, scale):
    v = np.arange(2 ** (bits - 1), 2 ** bits, dtype=D)[:, None]
    s1 = (np.arange(128, 256, dtype=D)[None] * 2.0 ** (scale - 8)).astype(F)
    r1 = (F(1) / s1).astype(F)
    for gap in range(-9, 9):
        for sign in (1, -1):
            x = (sign * v * 2.0 ** (scale + gap - bits)).astype(F)
            q = (x / s1).astype(F)
            got = (x.astype(D) * r1 + 384).astype(F) - F(384)
            seen = np.abs(q) <= 121
            np.testing.assert_array_equal(np.rint(got)[seen], np.rint(q)[seen])


def test_codes():
    q, s2, z = np.meshgrid(np.arange(-112, 113), np.arange(1, 16), np.arange(16), indexing="ij")
    q, s2, z = q.astype(F), s2.astype(F), z.astype(F)
    want = np.clip(np.rint((q / s2).astype(F) + z), 0, 15).astype(np.uint32)
    r2 = (F(1) / s2).astype(F)
    got = (q.astype(D) * r2 + (z + 2048)).astype(F) + F(2 ** 23 - 2048)
    got = np.clip(got, F(2 ** 23), F(2 ** 23 + 15)).view(np.uint32)
    np.testing.assert_array_equal(got - np.uint32(0x4B000000), want)
    # eight of them as one dword, shifted together with their exponent bits
    n = got.reshape(-1, 8).astype(np.uint64)
    word = n[:, 3]
    for i in (7, 2, 6, 1, 5, 0, 4):
        word = ((word << 4) + n[:, i]) & 0xFFFFFFFF
    word = (word - 0xFB000000) & 0xFFFFFFFF
    c = want.reshape(-1, 8).astype(np.uint64)
    ref = sum(((c[:, b] << 4) | c[:, b + 4]) << (8 * b) for b in range(4))
    np.testing.assert_array_equal(word, ref)
