"""The wide forms of the rotary embedding's kernels (floneum_amd/csrc/rope.hip) at the sizes between which they choose their
blocks, over views and odd head and row counts, bit for bit against the CPU restatements; and, on the host, the division by
multiplication that numbers their rows.
"""
import numpy as np
import pytest

import floneum_amd as fa
import oracle


def rounded(a, dtype):
    if dtype == fa.F32:
        return np.asarray(a, np.float32)
    if dtype == fa.F16:
        return np.asarray(a, np.float32).astype(np.float16).astype(np.float32)
    return fa.bf16_bits_to_f32(fa.f32_to_bf16_bits(a))


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore:overflow")
@pytest.mark.parametrize("dtype", [fa.F32, fa.F16, fa.BF16])
@pytest.mark.parametrize("D, heads, rows", [
    (64, 32, 2049), (128, 32, 1025), (256, 16, 1027),  # the larger blocks, the last one partial
    (64, 1, 7), (64, 3, 5), (128, 7, 1), (128, 5, 13), (256, 1, 3),  # the smaller ones, down to less than one
])
def test_blocks_of_rows(device, dtype, D, heads, rows):
    """Rows of zeros of either sign, of values whose squares overflow and underflow, and ordinary ones, from a [rows, heads, D]
    view, normalised and rotated, and rotated alone."""
    rng = np.random.default_rng(D * rows)
    x = rng.normal(0, 1, (1, rows, heads, D)).astype(np.float32)
    flat = x.reshape(-1, D)
    for i, s in enumerate([0.0, -0.0, 1e25 if dtype == fa.F32 else 100.0, 1e-30, 3e-6]):
        if i < len(flat):
            flat[(len(flat) // 2 + i) % len(flat)] *= np.float32(s)
    rc = fa.RopeCache(D, rows + 3, 10000.0, device)
    w = rng.normal(1, 0.2, D).astype(np.float32)
    norm = fa.RmsNorm(w, None, 1e-6, dtype, device)
    t = fa.Tensor.from_numpy(device, x, dtype).transpose(1, 2)
    xr = rounded(x, dtype).transpose(0, 2, 1, 3)
    n = rounded(oracle.rms_norm(xr, rounded(w, dtype), None, 1e-6), dtype)
    for got, want in [(rc.apply(t, 3, norm=norm), oracle.rope(n, rc.cos_host, rc.sin_host, 3)),
                      (rc.apply(t, 3), oracle.rope(np.ascontiguousarray(xr), rc.cos_host, rc.sin_host, 3))]:
        got, want = rounded(got.to_numpy(), dtype), rounded(want, dtype)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_division_by_multiplication():
    """The multiplier and shift of fill_row_job, for every divisor to 5000 and others to 2^31, at the quotients' edges."""
    rng = np.random.default_rng(1)
    ds = np.concatenate([np.arange(2, 5001), rng.integers(5001, 2 ** 31, 4000), 2 ** np.arange(1, 31), 2 ** np.arange(2, 31) + 1,
                         2 ** np.arange(2, 31) - 1]).astype(object)
    for d in ds:
        d = int(d)
        log = (d - 1).bit_length()
        mul, shift = (1 << (31 + log)) // d + 1, log - 1
        assert mul < 2 ** 32
        top = (2 ** 31 - 1) // d
        for q in {0, 1, top // 2, top}:
            for t in (q * d - 1, q * d, q * d + d - 1):
                if 0 <= t < 2 ** 31:
                    assert ((t * mul) >> 32) >> shift == t // d, (t, d)
