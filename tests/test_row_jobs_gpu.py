"""The wide forms of the rotary embedding's kernels (floneum_amd/csrc/rope.hip) at the sizes between which they choose their
blocks, over views and odd head and row counts, bit for bit against the CPU restatements; and, on the host, the division by
multiplication that numbers their rows.
"""
import ctypes

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


class RopeRows(ctypes.Structure):
    """fhip::RopeRows (floneum_amd/csrc/common.h)."""
    _fields_ = [("src", ctypes.c_void_p), ("dst", ctypes.c_void_p), ("ss", ctypes.c_int64 * 4), ("ds", ctypes.c_int64 * 4),
                ("shape", ctypes.c_uint32 * 4), ("src_dtype", ctypes.c_int32), ("dst_dtype", ctypes.c_int32),
                ("cos", ctypes.c_void_p), ("sin", ctypes.c_void_p), ("pos0", ctypes.c_int64), ("mode", ctypes.c_int32),
                ("norm_w", ctypes.c_void_p), ("norm_b", ctypes.c_void_p), ("norm_dtype", ctypes.c_int32), ("eps", ctypes.c_float),
                ("vec", ctypes.c_int32), ("few", ctypes.c_int32), ("small", ctypes.c_int32), ("mul", ctypes.c_uint32 * 3),
                ("shift", ctypes.c_uint32 * 3)]


class RowNorm(ctypes.Structure):
    _fields_ = [("weight", ctypes.c_void_p), ("bias", ctypes.c_void_p), ("dtype", ctypes.c_int32), ("eps", ctypes.c_float)]


FILL = "_ZN4fhip12fill_row_jobEPNS_8RopeRowsEPKvPKl10fhip_dtypePvS5_S6_PKjPKfSB_liPKNS_7RowNormE"


def filled(shape, mode=0, norm=False):
    """What the library's launcher passes to its kernels for contiguous rows of this shape (nothing is launched)."""
    out, at, strides = RopeRows(), ctypes.c_void_p(0x10000), (ctypes.c_int64 * 4)(*fa._contig_strides(shape))
    row_norm = RowNorm(0x10000, None, fa.F32, 1e-6)
    getattr(fa.lib(), FILL)(ctypes.byref(out), at, strides, fa.F32, at, strides, fa.F32, (ctypes.c_uint32 * 4)(*shape), at, at,
                            ctypes.c_int64(7), mode, ctypes.byref(row_norm) if norm else None)
    assert (tuple(out.shape), out.pos0, out.mode, bool(out.norm_w)) == (shape, 7, mode, norm)
    return out


def quotient(t, mul, shift):  # as the kernels divide: the upper half of a product of 32 bits, shifted
    return ((t * mul) >> 32) >> shift if mul else t


def test_division_by_multiplication():
    """The multipliers and shifts that rows and heads are numbered with, for every divisor to 5000 and others to 2^31, at the
    quotients' edges."""
    rng = np.random.default_rng(1)
    ds = np.concatenate([np.arange(1, 5001), rng.integers(5001, 2 ** 31, 4000), 2 ** np.arange(1, 31), 2 ** np.arange(2, 31) + 1,
                         2 ** np.arange(2, 31) - 1]).astype(object)
    for d in map(int, ds):
        job = filled((1, d, 1, 64))
        assert (job.mul[0], job.shift[0]) == (0, 0)
        assert tuple(filled((1, 1, d, 64)).mul)[:2] == (job.mul[1], 0)
        top = (2 ** 31 - 1) // d
        for q in {0, 1, top // 2, top}:
            for t in (q * d - 1, q * d, q * d + d - 1):
                if 0 <= t < 2 ** 31:
                    assert quotient(t, job.mul[1], job.shift[1]) == t // d, (t, d)


QUARTER_BLOCKS = 3584  # blocks of a quarter of 32 / 16 / 8 rows from which on a launch takes halves


@pytest.mark.parametrize("D, quarter", [(64, 8), (128, 4), (256, 2)])
def test_rows_of_a_block(D, quarter):
    """4: a quarter of 32 / 16 / 8 rows, 2: half of them (the heads of a position together where those are neighbours)."""
    most = (QUARTER_BLOCKS - 1) * quarter
    assert [filled((1, 1, rows, D), 0, True).few & 7 for rows in (1, most, most + 1, 10 * most)] == [4, 4, 2, 2]


@pytest.mark.parametrize("mode, norm", [(0, False), (1, False), (2, False), (0, True), (1, True), (2, True)])
def test_steps_of_a_row(mode, norm):
    """Steps per row: four pairs each, or four elements where nothing is rotated; and which inputs are numbered in 32 bits."""
    for D in (8, 64, 96, 128, 200, 256):
        job, per_row = filled((2, 3, 5, D), mode, norm), D // 4 if mode == 2 else D // 8
        assert job.small
        for t in (0, per_row - 1, per_row, 7 * per_row + per_row - 1, 30 * per_row - 1):
            assert quotient(t, job.mul[2], job.shift[2]) == t // per_row
        rows = (2 ** 31 - 1) // (1 if norm else per_row)
        assert filled((1, 1, rows, D), mode, norm).small and not filled((1, 1, rows + 1, D), mode, norm).small
        assert not filled((2 ** 20, 2 ** 20, 2 ** 25, D), mode, norm).small  # 2^65 rows


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [fa.F32, fa.F16, fa.BF16])
@pytest.mark.parametrize("D, heads, kv_heads, rows, turned", [
    (64, 5, 1, 4779, True), (64, 5, 1, 4777, True), (64, 5, 1, 4779, False),  # 3584 blocks of eight rows and a few less
    (128, 7, 2, 801, True), (256, 4, 2, 601, True), (256, 4, 2, 601, False), (128, 3, 1, 2, True),
])
def test_jobs_of_a_layer(device, dtype, D, heads, kv_heads, rows, turned):
    """q, k and v of two sequences in one launch, each with blocks of its own, against the same jobs one by one; views of
    [rows, heads, D] and of [heads, rows, D], around the sizes between which blocks change their rows and their order."""
    rng = np.random.default_rng(D + rows)

    def rows_of(h):
        x = rng.normal(0, 1, (2, rows, h, D) if turned else (2, h, rows, D)).astype(np.float32)
        t = fa.Tensor.from_numpy(device, x, dtype)
        return t.transpose(1, 2) if turned else t

    q, k, v = rows_of(heads), rows_of(kv_heads), rows_of(kv_heads)
    rope = fa.RopeCache(D, rows + 5, 10000.0, device)
    q_norm, k_norm = (fa.RmsNorm(rng.normal(1, 0.2, D).astype(np.float32), b, 1e-6, dtype, device)
                      for b in (None, rng.normal(0, 0.2, D).astype(np.float32)))
    cache = fa.KvCache(2, rows, dtype, device)
    got = cache.qkv_rope_append(rope, q, k, v, 5, False, q_norm, k_norm)
    want = [rope.apply(q, 5, norm=q_norm), rope.apply(k, 5, norm=k_norm), v]
    for g, w in zip(got, want):
        assert np.array_equal(g.to_numpy().view(np.uint32 if dtype != fa.F16 else np.uint16),
                              np.ascontiguousarray(w.to_numpy()).view(np.uint32 if dtype != fa.F16 else np.uint16))
    # the rows of one launch against the restatement: the first, the last and one between
    host = q.to_numpy()
    for r in {0, rows // 2, rows - 1}:
        x = rounded(host, dtype)[:, :, r:r + 1]
        n = rounded(oracle.rms_norm(np.ascontiguousarray(x), rounded(q_norm.weight.to_numpy()[0], dtype), None, 1e-6), dtype)
        y = rounded(oracle.rope(n, rope.cos_host, rope.sin_host, 5 + r), dtype)
        assert np.array_equal(rounded(got[0].to_numpy(), dtype)[:, :, r:r + 1].view(np.uint32), y.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [fa.F32, fa.F16, fa.BF16])
@pytest.mark.parametrize("D, heads, kv_heads, rows, turned, quarters", [
    (64, 5, 1, 2388, True, True), (64, 5, 1, 2389, True, False), (64, 5, 1, 2389, False, False), (128, 7, 2, 796, True, True),
    (128, 7, 2, 797, True, False), (256, 4, 2, 597, True, True), (256, 4, 2, 597, False, True), (256, 4, 2, 598, True, False),
])
def test_jobs_of_a_layer_on_both_sides(device, dtype, D, heads, kv_heads, rows, turned, quarters):
    """The same of two sequences whose q and k are just below and just above QUARTER_BLOCKS blocks."""
    blocks = sum(-(-2 * h * rows // {64: 8, 128: 4, 256: 2}[D]) for h in (heads, kv_heads))
    assert quarters == (blocks < QUARTER_BLOCKS) and abs(blocks - QUARTER_BLOCKS) < 8
    test_jobs_of_a_layer(device, dtype, D, heads, kv_heads, rows, turned)
