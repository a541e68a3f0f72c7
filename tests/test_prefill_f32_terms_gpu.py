"""GPU tests of the prefill kernel that computes in f32 precision from bf16 terms on the bf16 matrix cores
(floneum_amd/csrc/attn_prefill_f32_terms.hip): every form its launcher chooses between, at the edges of its 32-row units,
32-key tiles and padded head dims, against the same formula in 64 bits.

Tolerance: the six products of terms that are formed differ from the f32 product by at most 2^-24 of it, a score rounds 9
times at its own size (once per 16 dims, and once when the two accumulators are added) and the result once per tile, so
a relative L2 of 16 roundings of 2^-24 = 1e-6 is above what any of these sizes can reach (they measure 1e-7 to 3e-7).
Reference semantics: fusor-ml/fusor/src/composite/flash_attention.rs:141-199.
"""
import numpy as np
import pytest

import floneum_amd as fa

pytestmark = pytest.mark.gpu
NEG_INF = float("-inf")


def in_64_bits(q, k, v, scale, mask=None):
    """mask: [Sq, Skv] or [B, 1, 1, Skv] to add, or None."""
    G = q.shape[1] // k.shape[1]
    k, v = (np.repeat(np.asarray(a, np.float64), G, axis=1) for a in (k, v))
    s = np.asarray(q, np.float64) @ k.transpose(0, 1, 3, 2) * scale
    if mask is not None:
        s = s + mask
    p = np.exp(s - s.max(-1, keepdims=True))
    return (p / p.sum(-1, keepdims=True)) @ v


def close(out, ref, what):
    out = np.asarray(out, np.float64)
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    assert err <= 1e-6, f"{what}: relative L2 {err:.2e}"


def tensors(seed, B, H, Hkv, Sq, Skv, D, stds=(1.0, 1.0, 1.0)):
    rng = np.random.default_rng(seed)
    return [rng.normal(0, s, shp).astype(np.float32)
            for s, shp in zip(stds, [(B, H, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)])]


def causal_mask(Sq, Skv, off):
    return np.where(np.arange(Skv)[None, :] > np.arange(Sq)[:, None] + off, NEG_INF, 0.0)


FORMS = {
    # the workgroups of 256 compute units decide: (B, H, Hkv, Sq, Skv, causal)
    "two_units_four_key_groups": (1, 6, 2, 33, 61, True),       # head_dim <= 64; above: two units, two key groups
    "two_units_two_key_groups": (2, 32, 8, 510, 510, True),     # 64; above: four units, two key groups
    "four_units_two_key_groups": (2, 16, 16, 515, 545, False),  # 64; above: two units, two key groups
    "four_units": (34, 16, 16, 40, 65, False),
    "few_rows_keys_split": (1, 8, 2, 21, 2111, True),
    "short_prompt_keys_split": (1, 16, 4, 545, 545, True),      # above 64: four units, two key groups, three shares
    "shorter_prompt_keys_split": (1, 8, 2, 385, 385, True),     # above 64: two units, two key groups, three shares
    "one_tile": (1, 4, 4, 32, 32, True),
    "one_key": (3, 4, 1, 40, 1, False),
}


@pytest.mark.parametrize("D", [64, 128, 20, 80, 96])
@pytest.mark.parametrize("form", list(FORMS))
def test_forms_and_edges(device, form, D):
    B, H, Hkv, Sq, Skv, causal = FORMS[form]
    q, k, v = tensors(1, B, H, Hkv, Sq, Skv, D)
    tq, tk, tv = (fa.Tensor.from_numpy(device, a, fa.F32) for a in (q, k, v))
    out = tq.flash_attention(tk, tv, D ** -0.5, analytic=(True, Skv - Sq, 0) if causal else None,
                             force_kernel=fa.KERNEL_PREFILL_F32).to_numpy()
    close(out, in_64_bits(q, k, v, D ** -0.5, causal_mask(Sq, Skv, Skv - Sq) if causal else None), f"{form} D{D}")


WIDE = {
    # above head_dim 128: (B, H, Hkv, Sq, Skv, causal)
    "one_tile": (1, 4, 1, 65, 32, False), "unsplit": (2, 16, 4, 130, 65, False), "one_key": (3, 4, 1, 70, 1, False),
    "even_shares": (1, 8, 4, 148, 1251, True), "uneven_shares": (1, 8, 4, 417, 417, True), "shares_some_rows_do_not_see": (1, 4, 4, 801, 801, True),
    "shares_behind_a_cache": (1, 8, 4, 500, 801, True), "shares_of_odd_heads": (2, 6, 3, 330, 330, True),
    "few_rows": (1, 4, 2, 33, 2500, True), "few_rows_in_f32": (1, 4, 2, 33, 1500, True),
    # (few keys, unsplit, take the f32 instruction above 192 dims unless the grid is large; half-filled workgroups of units do)
    "unsplit_of_many": (8, 16, 4, 130, 65, False), "half_filled": (2, 16, 16, 40, 700, True), "half_filled_long": (2, 4, 4, 40, 2500, True),
}


@pytest.mark.parametrize("D", [256, 192, 132, 160, 228])
@pytest.mark.parametrize("form", list(WIDE))
def test_wide_heads(device, form, D):
    B, H, Hkv, Sq, Skv, causal = WIDE[form]
    q, k, v = tensors(6, B, H, Hkv, Sq, Skv, D)
    tq, tk, tv = (fa.Tensor.from_numpy(device, a, fa.F32) for a in (q, k, v))
    out = tq.flash_attention(tk, tv, D ** -0.5, analytic=(True, Skv - Sq, 0) if causal else None,
                             force_kernel=fa.KERNEL_PREFILL_F32).to_numpy()
    close(out, in_64_bits(q, k, v, D ** -0.5, causal_mask(Sq, Skv, Skv - Sq) if causal else None), f"{form} D{D}")


@pytest.mark.parametrize("D", [256, 160])
@pytest.mark.parametrize("of", ["V", "Q"])
@pytest.mark.parametrize("form", ["unsplit", "uneven_shares"])
def test_wide_heads_beyond_bf16(device, form, of, D):
    """Rows that are formed once more in f32: magnitudes at the bottom of f32's range, and an infinity that one key's V holds."""
    B, H, Hkv, Sq, Skv, causal = WIDE[form]
    q, k, v = tensors(7, B, H, Hkv, Sq, Skv, D, {"V": (1, 1, 2.0 ** -120), "Q": (2.0 ** -120, 2.0 ** 120, 1)}[of])
    if of == "V":
        v[0, 0, 3, 7] = np.inf
    tq, tk, tv = (fa.Tensor.from_numpy(device, a, fa.F32) for a in (q, k, v))
    out = tq.flash_attention(tk, tv, D ** -0.5, analytic=(True, Skv - Sq, 0) if causal else None, force_kernel=fa.KERNEL_PREFILL_F32).to_numpy()
    ref = in_64_bits(q, k, np.where(np.isinf(v), 0.0, v), D ** -0.5, causal_mask(Sq, Skv, Skv - Sq) if causal else None)
    if of == "V":
        seen = np.arange(Sq) + (Skv - Sq) >= 3 if causal else np.full(Sq, True)
        assert np.all(out[0, :H // Hkv, :, 7][:, seen] == np.inf)
        out, ref = out.copy(), ref.copy()
        out[0, :H // Hkv, :, 7][:, seen] = ref[0, :H // Hkv, :, 7][:, seen] = 0.0
    close(out, ref, f"{form} {of}")


@pytest.mark.parametrize("D", [256, 160])
@pytest.mark.parametrize("of", ["V", "Q"])
def test_wide_heads_beyond_bf16_of_many(device, of, D):
    """The same of an unsplit grid that is large enough for the terms kernel at every head_dim."""
    test_wide_heads_beyond_bf16(device, "unsplit_of_many", of, D)


@pytest.mark.parametrize("stds", [(1.0, 1.0, 1e30), (1e-12, 1e12, 1e-30), (1e4, 1e-4, 1.0)])
def test_magnitudes(device, stds):
    """The terms keep f32's range."""
    q, k, v = tensors(2, 1, 4, 2, 70, 200, 128, stds)
    tq, tk, tv = (fa.Tensor.from_numpy(device, a, fa.F32) for a in (q, k, v))
    close(tq.flash_attention(tk, tv, 128 ** -0.5).to_numpy(), in_64_bits(q, k, v, 128 ** -0.5), f"{stds}")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("form", ["two_units_four_key_groups", "two_units_two_key_groups", "few_rows_keys_split"])
@pytest.mark.parametrize("of", ["V", "Q", "K", "a dim of V"])
def test_elements_whose_last_term_bf16_cannot_hold(device, of, form, D):
    """Magnitudes down to f32's smallest normal one: results as small as V, and products of small elements with large ones.  (A
    result of 2^-120 is rounded at 2^-144.)"""
    B, H, Hkv, Sq, Skv, causal = FORMS[form]
    small, large = 2.0 ** -120, 2.0 ** 120
    q, k, v = tensors(16, B, H, Hkv, Sq, Skv, D, {"V": (1, 1, small), "Q": (small, large, 1), "K": (large, small, 1)}.get(of, (1, 1, 1)))
    if of == "a dim of V":
        v[..., 5] *= np.float32(small)
    tq, tk, tv = (fa.Tensor.from_numpy(device, a, fa.F32) for a in (q, k, v))
    out = tq.flash_attention(tk, tv, D ** -0.5, analytic=(True, Skv - Sq, 0) if causal else None,
                             force_kernel=fa.KERNEL_PREFILL_F32).to_numpy()
    ref = in_64_bits(q, k, v, D ** -0.5, causal_mask(Sq, Skv, Skv - Sq) if causal else None)
    close(out, ref, of)
    close(out[..., 5], ref[..., 5], of)


@pytest.mark.parametrize("dtype", [fa.F32, fa.F16, fa.BF16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("rows", ["some", "many"])
def test_added_masks_in_every_storage_type(device, dtype, D, rows):
    """Finite mask values, in 16-bit storage (two terms or one) as in f32: the products stay exact, so an f32 result has
    f32's precision.  The layout of the result is [b, seq, heads * hd]."""
    B, H, Hkv, Sq, Skv = (2, 4, 2, 45, 100) if rows == "some" else (17, 16, 16, 70, 97)
    q, k, v = tensors(3, B, H, Hkv, Sq, Skv, D)
    bias = np.random.default_rng(4).normal(0, 1, (Sq, Skv)).astype(np.float32)
    tq, tk, tv, tm = (fa.Tensor.from_numpy(device, a, dtype) for a in (q, k, v, bias))
    out = fa.Tensor.empty(device, (B, Sq, H, D), fa.F32)
    tq.flash_attention(tk, tv, D ** -0.5, (tm, fa.MaskKind.QKMask), out_dtype=fa.F32, out=out.transpose(1, 2))
    q, k, v, bias = (t.to_numpy() for t in (tq, tk, tv, tm))
    close(out.to_numpy().transpose(0, 2, 1, 3), in_64_bits(q, k, v, D ** -0.5, np.asarray(bias, np.float64)), f"D{D}")


@pytest.mark.parametrize("dtype", [fa.F16, fa.BF16])
def test_16_bit_results(device, dtype):
    """Head dims that only this kernel takes in 16 bits (multiples of 4 that are not of 8): the f32 result, rounded once."""
    q, k, v = tensors(5, 2, 4, 2, 70, 133, 100)
    tq, tk, tv = (fa.Tensor.from_numpy(device, a, dtype) for a in (q, k, v))
    f32 = tq.flash_attention(tk, tv, 0.1, out_dtype=fa.F32).to_numpy()
    out = tq.flash_attention(tk, tv, 0.1).to_numpy()
    want = f32.astype(np.float16) if dtype == fa.F16 else fa.bf16_bits_to_f32(fa.f32_to_bf16_bits(f32))
    assert np.array_equal(out, want)


def test_rows_without_keys_and_views(device):
    """Sequences without a key give NaN rows; overlapping K rows (a broadcast view) run on the f32 matrix instruction."""
    q, k, v = tensors(6, 3, 4, 2, 40, 70, 64)
    tq, tk, tv = (fa.Tensor.from_numpy(device, a, fa.F32) for a in (q, k, v))
    lens = [70, 0, 33]
    out = tq.flash_attention(tk, tv, 0.125, kv_lens=fa.IntTensor(device, lens)).to_numpy()
    assert np.isnan(out[1]).all()
    for b in (0, 2):
        n = lens[b]
        close(out[b:b + 1], in_64_bits(q[b:b + 1], k[b:b + 1, :, :n], v[b:b + 1, :, :n], 0.125), f"batch {b}")
    one = tk.narrow(2, 5, 1).broadcast_to((3, 2, 70, 64))
    close(tq.flash_attention(one, tv, 0.125).to_numpy(), in_64_bits(q, np.repeat(k[:, :, 5:6], 70, axis=2), v, 0.125), "broadcast")
