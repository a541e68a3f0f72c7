"""GPU tests of the 16-bit prefill kernel of head dims to 128 (floneum_amd/csrc/attn_prefill_mfma.hip): its two workgroup
forms at every tile width, with key counts around the ends of their rings of 64-key tiles, and grids that its launcher gives
to the one or the other, against the same formula in 64 bits.

Tolerance: probabilities and results are rounded to the type once each, half a unit in the last place apart, which is a relative
L2 of at most 2^-11 (f16) or 2^-8 (bf16) for either; twice that bounds both.
Reference semantics: fusor-ml/fusor/src/composite/flash_attention.rs:141-199.
"""
import ctypes

import numpy as np
import pytest

import floneum_amd as fa

CUS = 256


def block_rows(B, H, Sq, Skv, later_rows_see=0, window=0, compute_units=CUS):
    """Query rows per workgroup (256, or 128 in the key-split form), from the function that the launcher asks."""
    rule = fa.lib()._ZN4fhip23prefill_mfma_block_rowsEiiiiilli
    return rule(B, H, Sq, Skv, 1, ctypes.c_int64(later_rows_see), ctypes.c_int64(window), compute_units)


@pytest.mark.parametrize("B, H, Sq, before, window, rows", [
    # rows with a whole window behind the first of them, whose keys begin with that window: 256 rows a block, but for a 128-row grid of
    # one workgroup per CU
    (1, 16, 2364, 1398, 1399, 256), (1, 12, 3132, 2620, 2512, 256), (2, 12, 1939, 300, 208, 256), (1, 12, 2668, 451, 452, 128),
    # half a window: 256 from one and a quarter workgroups per CU on; less than half: as a prompt
    (1, 24, 2048, 511, 1024, 256), (1, 24, 2048, 510, 1024, 128), (1, 20, 2048, 511, 1024, 128), (1, 24, 2048, 0, 1024, 128),
    (1, 24, 2048, 2047, 2049, 128),  # of a window longer than the rows the line of the keys per row decides
])
def test_which_form_under_a_window(B, H, Sq, before, window, rows):
    first = max(0, before - window + 1) // 128 * 128
    later = before - first + Sq
    assert block_rows(B, H, Sq, later, later, window) == rows


@pytest.mark.parametrize("B, H, Sq, Skv, later_rows_see, window, rows", [
    (1, 16, 4096, 4096, 0, 0, 256), (1, 32, 2048, 8192, 0, 0, 256), (1, 32, 2048, 2048, 2048, 0, 128),  # even rows; a prompt
    (1, 32, 2048, 4096, 4096, 0, 128), (1, 32, 2048, 5120, 5120, 0, 128), (1, 32, 2048, 5121, 5121, 0, 256),  # the line
    (1, 24, 2048, 16384, 16384, 0, 256), (1, 32, 2048, 8192, 2048, 0, 128),  # rows at the end and the beginning of a longer view
    (1, 32, 2048, 4096, 4096, 1024, 256), (1, 32, 2048, 4096, 4096, 4096, 128), (1, 32, 2048, 4095, 4095, 1024, 128),  # windows
    (1, 33, 2048, 2048, 2048, 0, 256), (1, 32, 1792, 1792, 1792, 0, 256), (1, 18, 1792, 1792, 1792, 0, 128),  # more than a workgroup
    (4, 32, 128, 300, 0, 0, 128), (4, 32, 129, 300, 0, 0, 128), (8, 32, 129, 300, 0, 0, 256), (1, 4, 200, 128, 0, 0, 256),  # per CU
])
def test_which_form(B, H, Sq, Skv, later_rows_see, window, rows):
    assert block_rows(B, H, Sq, Skv, later_rows_see, window) == rows


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


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [fa.F16, fa.BF16])
@pytest.mark.parametrize("D", [64, 80, 96, 112, 128])
def test_grids_of_even_rows_keep_the_256_row_form(device, dtype, D):
    """Eight query blocks per head on more than half of the compute units, every row with the same keys."""
    assert block_rows(1, 18, 1801, 333, 0, 0, device.compute_units) == 256
    run(device, dtype, 1, 18, 6, 1801, 333, D)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Skv, rows", [(4502, 128), (4505, 256)])
def test_causal_grids_on_both_sides_of_the_line(device, D, Skv, rows):
    assert block_rows(1, 17, 1801, Skv, Skv, 0, device.compute_units) == rows
    run(device, fa.F16, 1, 17, 17, 1801, Skv, D, causal=True)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 72, 96, 128])
@pytest.mark.parametrize("Skv", [1, 63, 65, 128, 129, 192, 193, 257, 320, 321, 449])
def test_key_counts_around_the_rings_of_tiles(device, D, Skv):
    """One tile to more than either ring holds (four; five of K in the key-split form), the last one whole, short by a key or a
    single key.  130 heads give 129 rows to the 256-row form, four heads to the key-split form (from three tiles on)."""
    assert block_rows(1, 130, 129, Skv, 0, 0, device.compute_units) == 256
    assert block_rows(1, 4, 130, Skv, 0, 0, device.compute_units) == (128 if Skv > 128 else 256)
    run(device, fa.F16, 1, 130, 130, 129, Skv, D)
    run(device, fa.BF16, 1, 4, 2, 130, Skv, D)
    if Skv >= 130:
        run(device, fa.F16, 1, 4, 2, 130, Skv, D, causal=True)
