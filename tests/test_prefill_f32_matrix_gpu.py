"""GPU tests of the f32 prefill kernel on the f32 matrix instruction (floneum_amd/csrc/attn_prefill_f32.hip) at head dims to 128,
which it serves for views that the kernel for these head dims cannot address: rows of K that overlap.  Against the same
formula in 64 bits, over every way a mask is applied, storage type and tile width, with the keys split over workgroups
and not.

Tolerance: a dot product of D terms and a sum over keys, each a chain of f32 roundings: a relative error of (D + Skv) 2^-25 in the
worst case and its square root, some 1e-6, in the mean; 2e-6 relative L2.
Reference semantics: fusor-ml/fusor/src/composite/flash_attention.rs:141-199.
"""
import numpy as np
import pytest

import floneum_amd as fa
from test_prefill_f32_terms_gpu import in_64_bits, tensors

pytestmark = pytest.mark.gpu
NEG_INF = float("-inf")


def overlapping(device, seed, B, Hkv, Skv, D, dtype):
    """K rows that begin half a row apart: [B, Hkv, Skv, D] over Skv / 2 rows' memory, and the same as an array."""
    step = D // 8 * 4
    length = (Skv - 1) * step + D
    flat = fa.Tensor.from_numpy(device, np.random.default_rng(seed).normal(0, 1, (B, Hkv, length)).astype(np.float32), dtype)
    view = fa.Tensor(flat.buffer, dtype, (B, Hkv, Skv, D), (Hkv * length, length, step, 1))
    host = np.asarray(flat.to_numpy(), np.float64)
    return view, np.stack([host[:, :, j * step:j * step + D] for j in range(Skv)], axis=2)


@pytest.mark.parametrize("dtype", [fa.F32, fa.F16, fa.BF16])
@pytest.mark.parametrize("D", [64, 128, 20, 96])
@pytest.mark.parametrize("Sq,Skv", [(45, 131), (21, 2111)])  # the second: keys split over workgroups
@pytest.mark.parametrize("mask", ["none", "intervals", "values", "lowest"])
def test_masks_and_types(device, mask, Sq, Skv, D, dtype):
    B, H, Hkv = 2, 4, 2
    q, _, v = tensors(20, B, H, Hkv, Sq, Skv, D)
    tk, k = overlapping(device, 21, B, Hkv, Skv, D, dtype)
    tq, tv = (fa.Tensor.from_numpy(device, a, dtype) for a in (q, v))
    m = np.zeros((B, Skv), np.float32)
    if mask == "intervals":
        m[0, Skv // 3:], m[1, :5] = NEG_INF, NEG_INF
    elif mask == "values":
        m[:] = np.random.default_rng(22).normal(0, 1, m.shape)
    elif mask == "lowest":  # one sequence of nothing else, one with visible keys
        low = {fa.F32: -3.4028235e38, fa.F16: -65504.0, fa.BF16: -3.3895314e38}[dtype]
        m[0], m[1, Skv // 2:] = low, low
    tm = None if mask == "none" else (fa.Tensor.from_numpy(device, m, dtype), fa.MaskKind.BatchKeyMask)
    out = np.asarray(tq.flash_attention(tk, tv, D ** -0.5, tm, out_dtype=fa.F32, force_kernel=fa.KERNEL_PREFILL_F32).to_numpy(), np.float64)
    bias = None if tm is None else np.asarray(tm[0].to_numpy(), np.float64)[:, None, None, :]
    q, v = (np.asarray(t.to_numpy(), np.float64) for t in (tq, tv))
    if mask == "lowest" and dtype == fa.F16:
        bias = np.asarray(bias[1:])  # -65504 does not hide the scores: sums with it round at 2^-7, which is the f32 formula's own error
        out, q, k, v = out[1:], q[1:], k[1:], v[1:]
    ref = in_64_bits(q, k, v, D ** -0.5, bias)
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    assert err <= 2e-6, f"{mask} D{D}: relative L2 {err:.2e}"
