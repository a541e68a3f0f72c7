"""GPU tests of infinite elements, and of finite ones beyond bf16's largest, in the f32 prefill kernel that splits values into
bf16 terms (floneum_amd/csrc/attn_prefill_f32_terms.hip): such an element has no sum of finite terms, so the rows that meet it
are formed again from the elements themselves.  Against the same formula in 64 bits over the keys a row sees.

Tolerance: a dot product of 128 f32 terms in a chain has a relative error of 128 * 2^-25 = 4e-6 in the worst case and some
2e-7 in the mean, the result's sum over keys the same; 2e-6 relative L2 over all rows.
Reference semantics: fusor-ml/fusor/src/composite/flash_attention.rs:141-199.
"""
import time

import numpy as np
import pytest

import floneum_amd as fa
from test_prefill_f32_terms_gpu import FORMS, causal_mask, tensors

pytestmark = pytest.mark.gpu


def expect(q, k, v, scale, mask):
    """mask: [B, Sq, Skv] to add; keys at -inf are not seen."""
    B, H, Sq, D = q.shape
    G = H // k.shape[1]
    out = np.zeros((B, H, Sq, D))
    q, k, v = (np.asarray(a, np.float64) for a in (q, k, v))
    with np.errstate(invalid="ignore", over="ignore"):
        for b in range(B):
            for h in range(H):
                s = np.where(mask[b] > -np.inf, (q[b, h] @ k[b, h // G].T) * scale + mask[b], -np.inf)
                p = np.exp(s - s.max(-1, keepdims=True))
                p /= p.sum(-1, keepdims=True)
                finite = np.where(np.isfinite(v[b, h // G]), v[b, h // G], 0.0)
                out[b, h] = p @ finite
                for j, d in np.argwhere(np.isinf(v[b, h // G])):
                    out[b, h, p[:, j] > 0, d] = v[b, h // G, j, d]
    return out


def check(out, ref):
    out = np.asarray(out, np.float64)
    assert not np.isnan(ref).any() and np.isinf(ref).any()
    np.testing.assert_array_equal(np.isinf(out), np.isinf(ref))
    assert (out[np.isinf(ref)] == ref[np.isinf(ref)]).all()
    for dims in (slice(4, 5), np.r_[0:4, 5:ref.shape[-1]]):  # dim 4 may hold far larger values than the others
        a, r = out[..., dims], ref[..., dims]
        a, r = a[np.isfinite(r)], r[np.isfinite(r)]
        err = np.linalg.norm(a - r) / np.linalg.norm(r)
        assert err <= 2e-6, f"relative L2 {err:.2e}"


def plant(q, k, v, huge):
    q[..., 0], q[..., 1] = np.abs(q[..., 0]) + 0.1, 0.0
    if k.shape[2] > 30:
        k[:, :, 7, 0] = -np.inf      # a score of -inf: the key has no weight
        if huge:
            k[:, :, 11, 1] = 3.4e38  # times zero
            v[:, :, 9, 4] = 3.4e38   # finite: its share of the result is
    j = k.shape[2] // 2
    v[:, 0, j, 3], v[:, -1, j // 2, 2] = np.inf, -np.inf


@pytest.mark.parametrize("D", [64, 128, 20])
@pytest.mark.parametrize("form", [f for f in FORMS if f != "one_key"])
def test_elements_without_finite_terms(device, form, D):
    B, H, Hkv, Sq, Skv, causal = FORMS[form]
    q, k, v = tensors(11, B, H, Hkv, Sq, Skv, D)
    plant(q, k, v, huge=True)
    tq, tk, tv = (fa.Tensor.from_numpy(device, a, fa.F32) for a in (q, k, v))
    out = tq.flash_attention(tk, tv, D ** -0.5, analytic=(True, Skv - Sq, 0) if causal else None,
                             force_kernel=fa.KERNEL_PREFILL_F32).to_numpy()
    mask = causal_mask(Sq, Skv, Skv - Sq) if causal else np.zeros((Sq, Skv))
    check(out, expect(q, k, v, D ** -0.5, np.broadcast_to(mask, (B, Sq, Skv))))


@pytest.mark.parametrize("dtype", [fa.F32, fa.F16, fa.BF16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("kind", ["rows", "keys"])
def test_with_added_masks(device, dtype, D, kind):
    B, H, Hkv, Sq, Skv = 2, 4, 2, 45, 131
    q, k, v = tensors(12, B, H, Hkv, Sq, Skv, D)
    plant(q, k, v, huge=dtype == fa.F32)
    m = np.random.default_rng(13).normal(0, 1, (Sq if kind == "rows" else B, Skv)).astype(np.float32)
    tq, tk, tv, tm = (fa.Tensor.from_numpy(device, a, dtype) for a in (q, k, v, m))
    out = tq.flash_attention(tk, tv, D ** -0.5, (tm, fa.MaskKind.QKMask if kind == "rows" else fa.MaskKind.BatchKeyMask),
                             out_dtype=fa.F32, force_kernel=fa.KERNEL_PREFILL_F32).to_numpy()
    q, k, v, m = (t.to_numpy() for t in (tq, tk, tv, tm))
    m = np.asarray(m, np.float64)
    check(out, expect(q, k, v, D ** -0.5, np.broadcast_to(m[None] if kind == "rows" else m[:, None, :], (B, Sq, Skv))))


@pytest.mark.parametrize("Sq,Skv,D,what", [(2048, 2048, 128, "V"), (512, 512, 64, "V"), (129, 8003, 128, "V"), (2048, 2048, 128, "K")])
def test_one_infinite_element_does_not_multiply_the_time(device, Sq, Skv, D, what):
    """An infinity in the first key's row reaches every row of its group; all of them in f32 arithmetic take some 3 times (V) to 4
    times (512 rows) the time of a call without it.  One row at a time they took more than 100 times as long; 10 is allowed."""
    q, k, v = tensors(14, 1, 32, 8, Sq, Skv, D)
    q[..., 0] = np.abs(q[..., 0]) + 0.1

    def best_of_three():
        tq, tk, tv = (fa.Tensor.from_numpy(device, a, fa.F32) for a in (q, k, v))
        times = []
        for _ in range(4):
            device.synchronize()
            start = time.perf_counter()
            for _ in range(5):
                tq.flash_attention(tk, tv, D ** -0.5, analytic=(True, Skv - Sq, 0), force_kernel=fa.KERNEL_PREFILL_F32)
            device.synchronize()
            times.append(time.perf_counter() - start)
        return min(times[1:])

    usual = best_of_three()
    (v if what == "V" else k)[:, :, 0, 0] = np.inf if what == "V" else -np.inf
    odd = best_of_three()
    assert odd <= 10 * usual, f"{odd / usual:.1f} times as long"
