"""GPU tests of the 256-row 16-bit prefill kernel (floneum_amd/csrc/attn_prefill_mfma.hip) at head dims between its tile
widths of 64, 96 and 128: every form its launcher chooses between, against the same formula in 64 bits.  Rows of Q, K and V
are views into wider rows whose remaining elements are NaN: the kernel must neither read dims behind head_dim nor write
them.

Tolerance: an output rounds once to the type and each probability once, so results differ from 64 bits by about one
rounding of the type in relative L2 (2^-12 mean in f16, 2^-9 in bf16); three times that is allowed.
Reference semantics: fusor-ml/fusor/src/composite/flash_attention.rs:141-199.
"""
import numpy as np
import pytest

import floneum_amd as fa

pytestmark = pytest.mark.gpu

FORMS = {  # B, H, Hkv, Sq, Skv, causal, window
    "blocks_of_256": (16, 16, 8, 300, 300, True, 0),
    "blocks_of_256_one_tile": (16, 16, 16, 257, 64, False, 0),
    "blocks_of_128": (1, 4, 2, 200, 333, True, 100),
    "keys_split": (1, 4, 4, 40, 1100, True, 0),
    "heads_share_a_block": (8, 32, 4, 21, 2100, True, 0),
    "one_key": (1, 2, 1, 33, 1, False, 0),
}


def padded(device, a, dtype, pad):
    """`a` as a view of rows that are `pad` elements longer, NaN behind it."""
    wide = np.full(a.shape[:3] + (a.shape[3] + pad,), np.nan, np.float32)
    wide[..., :a.shape[3]] = a
    return fa.Tensor.from_numpy(device, wide, dtype).narrow(3, 0, a.shape[3])


def in_64_bits(q, k, v, scale, causal, window):
    B, H, Sq, _ = q.shape
    G, Skv = H // k.shape[1], k.shape[2]
    i, j = np.arange(Sq)[:, None] + Skv - Sq, np.arange(Skv)[None, :]
    seen = (j <= i) & (j + window > i if window else True) if causal else np.ones((Sq, Skv), bool)
    out = np.empty(q.shape)
    for b in range(B):
        for h in range(H):
            s = np.where(seen, q[b, h] @ k[b, h // G].T * scale, -np.inf)
            p = np.exp(s - s.max(-1, keepdims=True))
            out[b, h] = p / p.sum(-1, keepdims=True) @ v[b, h // G]
    return out


@pytest.mark.parametrize("dtype", [fa.F16, fa.BF16])
@pytest.mark.parametrize("D", [40, 72, 80, 88, 104, 112, 120])
@pytest.mark.parametrize("form", list(FORMS))
def test_forms_and_edges(device, form, D, dtype):
    B, H, Hkv, Sq, Skv, causal, window = FORMS[form]
    rng = np.random.default_rng(D)
    shapes = [(B, H, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)]
    q, k, v = (rng.normal(0, 1, s).astype(np.float32) for s in shapes)
    if dtype == fa.F16:
        q, k, v = (a.astype(np.float16).astype(np.float32) for a in (q, k, v))
    else:
        q, k, v = (fa.bf16_bits_to_f32(fa.f32_to_bf16_bits(a)) for a in (q, k, v))
    tq, tk, tv = (padded(device, a, dtype, 8) for a in (q, k, v))
    analytic = (True, Skv - Sq, window) if causal else None
    assert tq.selected_kernel(tk, tv, D ** -0.5, analytic=analytic) == fa.KERNEL_PREFILL_MFMA
    ref = in_64_bits(*(a.astype(np.float64) for a in (q, k, v)), D ** -0.5, causal, window)
    tol = 3 * (2.0 ** -12 if dtype == fa.F16 else 2.0 ** -9)
    for out_dtype, tail in ((dtype, 8), (fa.F32, 4), (dtype, 3)):  # 16-byte stores of both widths, and element by element
        host = np.full((B, H, Sq, D + tail), 7.0, np.float32)
        whole = fa.Tensor.from_numpy(device, host, out_dtype)
        tq.flash_attention(tk, tv, D ** -0.5, analytic=analytic, out_dtype=out_dtype, out=whole.narrow(3, 0, D))
        got = whole.to_numpy().astype(np.float64)
        err = np.linalg.norm(got[..., :D] - ref) / np.linalg.norm(ref)
        assert err <= tol, f"{form} D{D}: relative L2 {err:.2e}"
        assert (got[..., D:] == 7.0).all(), f"{form} D{D}: written behind head_dim"


@pytest.mark.parametrize("dtype", [fa.F16, fa.BF16])
@pytest.mark.parametrize("form,D", [("blocks_of_128", 80), ("blocks_of_256", 80), ("blocks_of_256", 40), ("keys_split", 120),
                                    ("blocks_of_128", 64), ("blocks_of_256", 128)])
@pytest.mark.parametrize("q_std,k_std,scale", [(1e-4, 1e4, None), (1.0, 1e4, 1e-5), (1.0, 1e4, 1e-6), (1e-5, 1e4, 0.5)])
def test_small_scales_and_elements(device, form, D, dtype, q_std, k_std, scale):
    """The scale is applied to the f32 scores: elements of Q times a power of two of it would leave f16's normal range, and
    with it lose bits, for some of these.  (scores of a few units at most, so that every probability has weight)"""
    B, H, Hkv, Sq, Skv, causal, window = FORMS[form]
    scale = float(np.float32(D ** -0.5 if scale is None else scale))
    rng = np.random.default_rng(D + 1)
    stds, shapes = (q_std, k_std, 1.0), [(B, H, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)]
    tq, tk, tv = (fa.Tensor.from_numpy(device, rng.normal(0, sd, sh).astype(np.float32), dtype) for sd, sh in zip(stds, shapes))
    analytic = (True, Skv - Sq, window) if causal else None
    out = tq.flash_attention(tk, tv, scale, analytic=analytic, out_dtype=fa.F32, force_kernel=fa.KERNEL_PREFILL_MFMA).to_numpy()
    ref = in_64_bits(*(t.to_numpy().astype(np.float64) for t in (tq, tk, tv)), scale, causal, window)
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    assert err <= 3 * (2.0 ** -12 if dtype == fa.F16 else 2.0 ** -9), f"{form} D{D}: relative L2 {err:.2e}"


@pytest.mark.parametrize("dtype", [fa.F16, fa.BF16])
@pytest.mark.parametrize("D,kernel", [(256, fa.KERNEL_PREFILL_MFMA), (200, fa.KERNEL_PREFILL_MFMA),
                                      (128, fa.KERNEL_PREFILL_MFMA_ROWS64)])
@pytest.mark.parametrize("q_std,k_std,scale", [(1e-4, 1e4, None), (1e-5, 1e4, 0.5), (1.0, 1.0, None)])
def test_small_elements_in_the_kernels_of_32_and_64_rows_per_wavefront(device, D, kernel, dtype, q_std, k_std, scale):
    """The same for head dims above 192, and for the form of 64 rows per wavefront."""
    B, H, Hkv, Sq, Skv, causal, window = 2, 4, 2, 300, 300, True, 0
    scale = float(np.float32(D ** -0.5 if scale is None else scale))
    rng = np.random.default_rng(D + 2)
    stds, shapes = (q_std, k_std, 1.0), [(B, H, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)]
    tq, tk, tv = (fa.Tensor.from_numpy(device, rng.normal(0, sd, sh).astype(np.float32), dtype) for sd, sh in zip(stds, shapes))
    out = tq.flash_attention(tk, tv, scale, analytic=(True, 0, 0), out_dtype=fa.F32, force_kernel=kernel).to_numpy()
    ref = in_64_bits(*(t.to_numpy().astype(np.float64) for t in (tq, tk, tv)), scale, causal, window)
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    assert err <= 3 * (2.0 ** -12 if dtype == fa.F16 else 2.0 ** -9), f"D{D}: relative L2 {err:.2e}"
