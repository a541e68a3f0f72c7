"""The merge inside the split-KV decode kernels at every number of splits it takes: two or three count their arrivals in one word, four
to eight have a mark each.  Bit for bit the two-launch form (which a call with per-sequence lengths takes), into outputs whose rows
can and cannot be stored in pieces, twice and more often in a row on one workspace, and from a recorded graph."""
import numpy as np
import pytest

import floneum_amd as fa

pytestmark = pytest.mark.gpu


def tensors(device, dtype, B, H, Hkv, Sq, Skv, D):
    rng = np.random.default_rng(Skv * 7 + D)
    return (fa.Tensor.from_numpy(device, rng.normal(0, 0.7, shp).astype(np.float32), dtype)
            for shp in [(B, H, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)])


def view(device, shape, dtype, how):
    B, H, Sq, D = shape
    if how == "contiguous":
        return fa.Tensor.from_numpy(device, np.full(shape, 7.0, np.float32), dtype)
    o = fa.Tensor.from_numpy(device, np.full((B, H, Sq, 2 * D + 1), 7.0, np.float32), dtype)
    if how == "odd rows":
        return fa.Tensor(o.buffer, dtype, shape, o.strides, 1)
    return fa.Tensor(o.buffer, dtype, shape, o.strides[:3] + (2,), 0)


@pytest.mark.parametrize("dtype, B, H, Hkv, Sq, Skv, D, splits", [
    (fa.F16, 1, 8, 4, 1, 257, 64, 3), (fa.BF16, 6, 32, 32, 1, 485, 64, 2), (fa.F16, 1, 32, 32, 1, 459, 64, 4), (fa.F16, 1, 8, 8, 1, 643, 96, 6),
    (fa.BF16, 1, 4, 4, 1, 984, 128, 8), (fa.F16, 3, 6, 3, 1, 900, 32, 8), (fa.F32, 1, 8, 8, 1, 500, 128, 8), (fa.F32, 3, 12, 3, 2, 333, 64, 6),
    (fa.F16, 1, 16, 1, 2, 600, 128, 5), (fa.BF16, 2, 32, 8, 4, 724, 128, 6), (fa.F16, 1, 8, 2, 1, 775, 256, 7), (fa.F32, 1, 16, 2, 1, 449, 256, 8),
])
@pytest.mark.parametrize("how", ["contiguous", "odd rows", "every second", "f32"])
def test_every_number_of_splits(device, dtype, B, H, Hkv, Sq, Skv, D, splits, how):
    q, k, v = tensors(device, dtype, B, H, Hkv, Sq, Skv, D)
    analytic = (True, Skv - Sq, 0) if Sq > 1 else None
    plan = q.decode_plan(k, v, D ** -0.5, analytic=analytic)
    assert (plan["nsplit"], plan["kernels"]) == (splits, 1), plan
    lens = fa.IntTensor(device, np.full(B, Skv, np.int32))
    out_dtype = fa.F32 if how == "f32" else dtype
    want = q.flash_attention(k, v, D ** -0.5, analytic=analytic, kv_lens=lens, out_dtype=out_dtype)
    assert q.decode_plan(k, v, D ** -0.5, analytic=analytic, kv_lens=lens)["kernels"] == 2
    want = want.to_numpy()
    assert np.isfinite(want).all()
    for _ in range(3):
        out = view(device, (B, H, Sq, D), out_dtype, "contiguous" if how == "f32" else how)
        q.flash_attention(k, v, D ** -0.5, analytic=analytic, out_dtype=out_dtype, out=out)
        assert np.array_equal(out.to_numpy().view(np.uint8), want.view(np.uint8))


@pytest.mark.parametrize("B, Hkv, Skv, splits", [(2, 3, 257, 3), (1, 8, 1000, 8), (7, 4, 714, 6)])
def test_replays(device, B, Hkv, Skv, splits):
    """Replays carry the tag they were recorded with: nothing of an earlier one may count, with other calls in between or not."""
    device = device.with_new_stream()
    q, k, v = tensors(device, fa.F16, B, 4 * Hkv, Hkv, 1, Skv, 64)
    assert q.decode_plan(k, v, 0.125)["nsplit"] == splits
    u = list(tensors(device, fa.F16, 3, 8, 2, 1, 900, 64))
    assert u[0].decode_plan(u[1], u[2], 0.125)["kernels"] == 1
    want = q.flash_attention(k, v, 0.125).to_numpy()
    out = fa.Tensor.empty(device, q.shape, fa.F16)
    u[0].flash_attention(u[1], u[2], 0.125)  # (the workspace has its size before the capture)
    with device.capture() as cap:
        for _ in range(3):
            q.flash_attention(k, v, 0.125, out=out)
    zero = np.zeros(q.shape, np.float16)
    for rep in range(4):
        out = fa.Tensor(out.buffer, fa.F16, q.shape)
        fa.check(fa.lib().fhip_memcpy_h2d(device.stream, fa.ctypes.c_void_p(out.buffer.ptr), zero.ctypes.data_as(fa.ctypes.c_void_p), zero.nbytes))
        cap.graph.launch()
        assert np.array_equal(out.to_numpy().view(np.uint8), want.view(np.uint8)), rep
        if rep % 2:
            u[0].flash_attention(u[1], u[2], 0.125).to_numpy()
