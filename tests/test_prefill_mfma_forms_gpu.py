"""GPU tests of the 16-bit prefill kernel of head dims to 128 (floneum_amd/csrc/attn_prefill_mfma.hip): its two workgroup
forms at every tile width, with key counts around the ends of their rings of 64-key tiles, and grids that its launcher gives
to the one or the other, against the same formula in 64 bits.

Tolerance: probabilities and results are rounded to the type once each, half a unit in the last place apart, which is a relative
L2 of at most 2^-11 (f16) or 2^-8 (bf16) for either; twice that bounds both.
Reference semantics: fusor-ml/fusor/src/composite/flash_attention.rs:141-199.
"""
import numpy as np
import pytest

import floneum_amd as fa

pytestmark = pytest.mark.gpu


def run(device, dtype, B, H, Hkv, Sq, Skv, D, causal=False):
    rng = np.random.default_rng(Sq * 1009 + Skv)
    tq, tk, tv = (fa.Tensor.from_numpy(device, rng.normal(0, 1, shp).astype(np.float32), dtype)
                  for shp in [(B, H, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)])
    analytic = (True, Skv - Sq, 0) if causal else None
    assert tq.selected_kernel(tk, tv, D ** -0.5, analytic=analytic) == fa.KERNEL_PREFILL_MFMA
    out = tq.flash_attention(tk, tv, D ** -0.5, analytic=analytic).to_numpy()
    q, k, v = (np.asarray(t.to_numpy(), np.float64) for t in (tq, tk, tv))
    k, v = (np.repeat(a, H // Hkv, axis=1) for a in (k, v))
    s = q @ k.transpose(0, 1, 3, 2) * D ** -0.5
    if causal:
        s = np.where(np.arange(Skv)[None, :] > np.arange(Sq)[:, None] + Skv - Sq, -np.inf, s)
    p = np.exp(s - s.max(-1, keepdims=True))
    ref = (p / p.sum(-1, keepdims=True)) @ v
    err = np.linalg.norm(np.asarray(out, np.float64) - ref) / np.linalg.norm(ref)
    assert err <= (2.0 ** -10 if dtype == fa.F16 else 2.0 ** -7), f"relative L2 {err:.2e}"


@pytest.mark.parametrize("dtype", [fa.F16, fa.BF16])
@pytest.mark.parametrize("D", [64, 80, 96, 112, 128])
def test_grids_of_even_rows_keep_the_256_row_form(device, dtype, D):
    """Eight query blocks per head on more than half of the compute units, every row with the same keys."""
    run(device, dtype, 1, 18, 6, 1801, 333, D)


@pytest.mark.parametrize("D", [64, 72, 96, 128])
@pytest.mark.parametrize("Skv", [1, 63, 65, 128, 129, 192, 193, 257, 320, 321, 449])
def test_key_counts_around_the_rings_of_tiles(device, D, Skv):
    """One tile to more than either ring holds (four; five of K in the key-split form), the last one whole, short by a key or a
    single key.  130 heads give 129 rows to the 256-row form, four heads to the key-split form (from three tiles on)."""
    run(device, fa.F16, 1, 130, 130, 129, Skv, D)
    run(device, fa.BF16, 1, 4, 2, 130, Skv, D)
    if Skv >= 130:
        run(device, fa.F16, 1, 4, 2, 130, Skv, D, causal=True)
