"""Host-only checks of how the Python mirror fills the C ABI's descriptors: packed in one go, they are byte for byte what
assigning the fields one by one gives, in every form of call and for values beyond their fields."""
import ctypes

import numpy as np
import pytest

import floneum_amd as fa


class _Device:
    stream, compute_units = None, 256


class _Memory:
    def __init__(self, ptr, device):
        self.ptr, self.device = ptr, device


def by_fields(q, k, v, out, scale, mask, analytic, lens, odt, force):
    def c4(t):
        c = fa.CTensor4()
        c.ptr, c.offset = t.buffer.ptr, t.offset
        c.shape[:], c.stride[:] = t.shape, t.strides
        return c

    a = fa.CAttnArgs()
    a.q, a.k, a.v, a.out = c4(q), c4(k), c4(v), c4(out)
    a.dtype, a.out_dtype, a.scale, a.force_kernel = q.dtype, odt, float(np.float32(scale)), force
    if mask is not None:
        a.mask, a.mask_kind = mask[0]._c2(), int(mask[1])
        if len(mask) > 2:
            a.mask_intervals = mask[2].buffer.ptr
    if isinstance(analytic, fa.CAnalyticMask):
        a.analytic = analytic
    elif analytic is not None:
        a.analytic = fa.CAnalyticMask(1, 1 if analytic[0] else 0, analytic[1], analytic[2] or 0)
    if lens is not None:
        a.kv_lens = lens.buffer.ptr + lens.offset * 4
    return a


@pytest.mark.parametrize("analytic", [None, (True, 5, 0), (False, 2 ** 40, 7), fa.CAnalyticMask(1, 1, -3, 9)])
@pytest.mark.parametrize("with_mask", [None, "mask", "mask and table"])
@pytest.mark.parametrize("rows, ptr, scale", [(3, 0x7f1234567000, 0.1), (2 ** 33 + 3, 0x1000, 0.25), (3, None, np.float32(1e-3))])
def test_packed_arguments_are_the_fields(analytic, with_mask, rows, ptr, scale):
    dev = _Device()

    def tensor(p, shape, strides=None, offset=0, dtype=fa.F16):
        return fa.Tensor(_Memory(p, dev), dtype, shape, strides, offset)

    q = tensor(ptr, (2, 8, rows, 64)).transpose(1, 2).transpose(1, 2)
    k, v = (tensor(0x2000 * i, (2, 4, 9, 64), (4 * 16 * 64, 16 * 64, 64, 1), 128 * i) for i in (1, 2))
    out = tensor(0x9000, (2, rows, 8, 64), dtype=fa.F32).transpose(1, 2)
    mask = None
    if with_mask:
        table = fa.MaskIntervals.__new__(fa.MaskIntervals)
        table.buffer = _Memory(0x5550, dev)
        mask = (tensor(0x4440, (3, 9)), fa.MaskKind.QKMask) + ((table,) if "table" in with_mask else ())
    lens = None
    if analytic is None:
        lens = fa.IntTensor.__new__(fa.IntTensor)
        lens.buffer, lens.shape, lens.offset = _Memory(0x7770, dev), (2,), 3
    got = q._attn_args(k, v, scale, mask, analytic, lens, fa.F32, fa.KERNEL_PREFILL_F32, out)
    want = by_fields(q, k, v, out, scale, mask, analytic, lens, fa.F32, fa.KERNEL_PREFILL_F32)
    assert bytes(got) == bytes(want)
    view = fa._cache_view(type("C", (), dict(device=dev, dtype=fa.F16)), v._c4())
    assert (view.buffer.ptr, view.offset, view.shape, view.strides) == (v.buffer.ptr, v.offset, v.shape, v.strides)


@pytest.mark.parametrize("which, shape, strides, other, other_strides", [
    ("k", (1, 2, 9, 64), (1, 2, 3), "v", (1, 2, 3, 4, 5)),  # strides that make up for each other's number
    ("q", (1, 2, 3, 64), (1, 2, 3, 4, 5), "out", (1, 2, 3)),
    ("out", (1, 2, 3), (6, 3, 1), "v", (1, 2, 3, 4, 5, 6)),
    ("out", (1, 2, 3), (1, 2, 3, 4, 5), None, None),
    ("out", (1, 2, 3, 4, 5), (1, 2, 3), None, None),
])
def test_ranks_and_strides_of_other_lengths_are_refused(which, shape, strides, other, other_strides):
    dev = _Device()
    t = {n: fa.Tensor(_Memory(0x1000, dev), fa.F16, (1, 2, 9 if n in "kv" else 3, 64)) for n in ("q", "k", "v", "out")}
    t[which].shape, t[which].strides = shape, strides
    if other:
        t[other].strides = other_strides
    with pytest.raises((AssertionError, ValueError, IndexError)):
        t["q"]._attn_args(t["k"], t["v"], 0.1, None, None, None, None, fa.KERNEL_AUTO, t["out"])


@pytest.mark.parametrize("shape, strides", [((3, 9), (9, 1, 1)), ((3, 9), (9,))])
def test_masks_of_other_ranks_are_refused(shape, strides):
    dev = _Device()
    q, k = (fa.Tensor(_Memory(0x1000, dev), fa.F16, (1, 2, n, 64)) for n in (3, 9))
    mask = fa.Tensor(_Memory(0x2000, dev), fa.F16, shape, strides)
    k.strides = (k.strides + (1, 1))[:8 - len(shape) - len(strides)]  # as many values in all as well-formed tensors have
    with pytest.raises((AssertionError, ValueError, IndexError)):
        q._attn_args(k, q, 0.1, (mask, fa.MaskKind.QKMask), None, None, None, fa.KERNEL_AUTO, q)


def test_a_shape_has_a_length():
    with pytest.raises(TypeError):
        fa.Tensor.empty(_Device(), (n for n in (2, 3)), fa.F16)
