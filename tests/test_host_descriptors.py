"""Host-only checks of how the Python mirror fills the C ABI's descriptors: packed in one go, they are byte for byte what
assigning the fields one by one gives, in every form of call and for values beyond their fields."""
import ctypes
import os
import subprocess
import sys
import sysconfig

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


def native(dev):
    """The native half, and tensors, a rotary cache and norms on made-up memory for it."""
    fa.lib()

    def tensor(p, shape, strides=None, offset=0, dtype=fa.F16):
        return fa.Tensor(_Memory(p, dev), dtype, shape, strides, offset)

    def norm(bias):
        n = fa.RmsNorm.__new__(fa.RmsNorm)
        n.device, n.dtype, n.eps = dev, fa.BF16, 1e-6
        n.weight, n.bias = tensor(0x3330, (1, 64)), tensor(0x3440, (1, 64)) if bias else None
        return n

    rope = fa.RopeCache.__new__(fa.RopeCache)
    rope.cos, rope.sin, rope.rows = tensor(0x6660, (9, 32)), tensor(0x6670, (9, 32)), 9
    return fa._native, tensor, norm, rope


@pytest.mark.parametrize("analytic", [None, (True, 5, 0), (False, -3, 2 ** 40)])
@pytest.mark.parametrize("with_mask", [None, "mask", "mask and table"])
@pytest.mark.parametrize("lens, out_dtype, scale", [(False, None, 0.1), (True, fa.F32, -1e-3), (True, None, float(np.float32(0.3)))])
def test_native_arguments_are_the_packed_ones(analytic, with_mask, lens, out_dtype, scale):
    dev = _Device()
    host, tensor, _, _ = native(dev)
    q = tensor(0x7f1234567000, (2, 3, 8, 64), offset=7).transpose(1, 2)
    k, v = (tensor(0x2000 * i, (2, 4, 9, 64), (-4 * 16 * 64, 16 * 64, 64, 0), 2 ** 63 + i) for i in (1, 2))
    out = tensor(0x9000, (2, 3, 8, 64), dtype=fa.F32).transpose(1, 2)
    mask = None
    if with_mask:
        table = fa.MaskIntervals.__new__(fa.MaskIntervals)
        table.buffer = _Memory(0x5550, dev)
        mask = (tensor(0x4440, (3, 9)), fa.MaskKind.QKMask) + ((table,) if "table" in with_mask else ())
    counts = None
    if lens:
        counts = fa.IntTensor.__new__(fa.IntTensor)
        counts.buffer, counts.shape, counts.offset = _Memory(0x7770, dev), (2,), 3
    a = (k, v, scale, mask, analytic, counts, out_dtype, fa.KERNEL_PREFILL_F32, out)
    assert host.attention_descriptor(q, *a) == bytes(q._attn_args(*a))


def test_calls_that_are_not_plain_are_left_to_the_general_way():
    """Each of these the mirror still accepts or refuses by itself: the native half answers None and leaves no exception."""
    dev, other = _Device(), _Device()
    host, tensor, _, _ = native(dev)
    plain = dict(q=tensor(0x1000, (1, 2, 3, 64)), k=tensor(0x2000, (1, 2, 9, 64)), v=tensor(0x3000, (1, 2, 9, 64)), scale=0.1, mask=None,
                 analytic=None, lens=None, odt=None, force=0, out=tensor(0x4000, (1, 2, 3, 64)))
    assert host.attention_descriptor(*plain.values()) is not None

    class Odd(fa.Tensor):
        pass

    lens = fa.IntTensor.__new__(fa.IntTensor)
    lens.buffer, lens.shape, lens.offset = _Memory(0x7770, dev), (2,), 0
    m = tensor(0x4440, (3, 9))
    foreign = fa.Tensor(_Memory(0x2000, other), fa.F16, (1, 2, 9, 64))
    for change in [dict(k=foreign), dict(v=foreign), dict(q=tensor(0x1000, (2, 3, 64))), dict(k=tensor(0x2000, (1, 2, 9, 64), (1, 2, 3))),
                   dict(k=tensor(0x2000, (1, 2, 9, 64), dtype=fa.F32)), dict(q=tensor(None, (1, 2, 3, 64))), dict(scale=1), dict(scale=1e39),
                   dict(scale=float("nan")), dict(scale=np.float32(0.1)), dict(q=tensor(0x1000, (1, 2, 2 ** 33, 64))), dict(out=None),
                   dict(k=tensor(0x2000, (1, 2, 9, 64), offset=-1)), dict(k=tensor(0x2000, (1, 2, 9, 64), (1, 2, 2 ** 70, 1))),
                   dict(q=Odd(_Memory(0x1000, dev), fa.F16, (1, 2, 3, 64))), dict(lens=lens), dict(lens=[1]), dict(odt="f32"), dict(force=2 ** 40),
                   dict(mask=m), dict(mask=(m,)), dict(mask=[m, fa.MaskKind.QKMask]), dict(mask=(m, None)), dict(mask=(m, 1, None)),
                   dict(mask=(tensor(0x4440, (3, 9), dtype=fa.F32), 1)), dict(mask=(tensor(0x4440, (1, 3, 9)), 1)),
                   dict(analytic=(1, 5, 0)), dict(analytic=(True, 5, None)), dict(analytic=[True, 5, 0]), dict(analytic=(True, 2 ** 70, 0)),
                   dict(analytic=fa.CAnalyticMask(1, 1, 0, 0)), dict(analytic=(True, 5))]:
        assert host.attention_descriptor(*dict(plain, **change).values()) is None, change


@pytest.mark.parametrize("q_bias, k_bias, interleaved", [(None, None, False), (False, True, True), (True, None, False)])
def test_native_append_describes_what_ctypes_does(q_bias, k_bias, interleaved):
    dev = _Device()
    host, tensor, norm, rope = native(dev)
    cache = fa.KvCache.__new__(fa.KvCache)
    cache.device, cache.dtype, cache.handle = dev, fa.F16, None
    q, k, v = (tensor(0x1000 * i, (1, 2, h, 64), offset=i).transpose(1, 2) for i, h in ((1, 8), (2, 4), (3, 4)))
    q_out = tensor(0x8000, q.shape, dtype=fa.F32)
    norms = [norm(b) if b is not None else None for b in (q_bias, k_bias)]
    got = host.append_descriptors(cache, rope, q, q_out, k, v, 5, interleaved, *norms)
    want = b"".join(bytes(t._c4()) for t in (q, q_out, k, v)) + np.array([fa.F16, fa.F32, fa.F16, fa.F16], np.int32).tobytes()
    want += bytes(rope._tables(5, interleaved)) + b"".join(bytes(n._c() if n else fa.CRmsNorm()) for n in norms)
    assert got == want
    for a in [(cache, rope, q, q_out, k, tensor(0x3000, k.shape, dtype=fa.F32), 5, False, None, None), (cache, rope, q, None, k, v, 5, False, None, None),
              (cache, rope, q, q_out, k, v, -1, False, None, None), (cache, rope, q, q_out, k, v, 5, 0, None, None),
              (cache, rope, q, q_out, k, v, 5, False, object(), None), (object(), rope, q, q_out, k, v, 5, False, None, None)]:
        assert host.append_descriptors(*a) is None
    cache.handle = None


def test_native_tensors_are_the_mirror_s():
    dev = _Device()
    host, tensor, _, _ = native(dev)
    blocks = []

    def memory(device, nbytes):
        blocks.append((device, nbytes))
        return _Memory(0x1000, device)

    for shape in [(2, 3, 4, 64), (5,), (), (2, 0, 3), (1, 1, 1, 1)]:
        t, want = host.contiguous(memory, dev, 2, fa.F16, shape), tensor(0x1000, shape)
        assert type(t) is fa.Tensor and (t.shape, t.strides, t.offset, t.dtype) == (want.shape, want.strides, want.offset, want.dtype)
        assert blocks[-1] == (dev, 2 * int(np.prod(shape))) and t.device is dev
    for shape in [[2, 3], (2, -1), (2.0, 3), (np.int64(2), 3), (2 ** 33, 1), (2 ** 31, 2 ** 31)]:
        assert host.contiguous(memory, dev, 2, fa.F16, shape) is None
    with pytest.raises(ZeroDivisionError):
        host.contiguous(lambda *_: 1 // 0, dev, 2, fa.F16, (1,))


def test_the_native_half_is_for_one_interpreter():
    """Its name says for which, so no other one loads it."""
    fa.lib()
    at = fa._native.__file__
    assert os.path.basename(at) == "_host" + sysconfig.get_config_var("EXT_SUFFIX")
    assert not os.path.exists(os.path.join(os.path.dirname(at), "_host.so"))


def test_the_mirror_without_its_native_half():
    """As under an interpreter that it was not built for: the library loads, and calls are described through ctypes."""
    program = """
import sys
sys.modules["floneum_amd._host"] = None
import floneum_amd as fa
fa.lib()
assert fa._native is None
class Device: pass
class Memory:
    def __init__(self, device, ptr): self.device, self.ptr = device, ptr
fa.Buffer = lambda device, nbytes: Memory(device, nbytes)
one, other = Device(), Device()
t = fa.Tensor.empty(one, (1, 2, 9, 64), fa.F16)
assert t.buffer.ptr == 2 * 2 * 9 * 64 and t.strides == (2 * 9 * 64, 9 * 64, 64, 1)
try:
    t.flash_attention(fa.Tensor.empty(other, (1, 2, 9, 64), fa.F16), t, 0.125)
except AssertionError as e:
    assert "different devices" in str(e)
else:
    sys.exit("accepted")
"""
    done = subprocess.run([sys.executable, "-c", program], cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))), capture_output=True, text=True)
    assert done.returncode == 0, done.stderr


@pytest.mark.parametrize("with_native", [True, False])
def test_no_result_is_allocated_for_a_call_that_is_refused(monkeypatch, with_native):
    dev, other = _Device(), _Device()
    dev.stream = other.stream = ctypes.c_void_p(0x10)  # (no call gets as far as using it)
    _, tensor, _, _ = native(dev)
    if not with_native:
        monkeypatch.setattr(fa, "_native", None)

    def allocated(*_):
        raise MemoryError("a result was allocated")

    monkeypatch.setattr(fa, "Buffer", allocated)
    q, k, v = tensor(0x1000, (1, 2, 3, 64)), tensor(0x2000, (1, 2, 9, 64)), tensor(0x3000, (1, 2, 9, 64))
    with pytest.raises(AssertionError, match="different devices"):
        q.flash_attention(fa.Tensor(_Memory(0x2000, other), fa.F16, (1, 2, 9, 64)), v, 0.125)
    with pytest.raises(fa.InvalidArgument, match="one element type"):
        q.flash_attention(k, tensor(0x3000, (1, 2, 9, 64), dtype=fa.F32), 0.125)
    with pytest.raises(fa.InvalidArgument, match="rank-4"):
        q.flash_attention(tensor(0x2000, (2, 9, 64)), v, 0.125)
    with pytest.raises(MemoryError):
        q.flash_attention(k, v, 0.125)
