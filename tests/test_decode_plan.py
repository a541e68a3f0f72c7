"""How a split-KV decode call's keys are divided: where chunks of the ordinary length would leave the last few workgroups a
round of their own, fewer and longer ones are taken, and the workspace stays that of the ordinary ones; and such calls against
the formula in 64 bits.

Tolerance: as tests/test_prefill_mfma_forms_gpu.py for 16-bit tensors.  In f32 a score rounds D / 4 times, once per step of the
matrix instruction, and twice more before the exponential, a result once per 16 keys of a wavefront (24) and a dozen times
in the merges, each up to 2^-24 of either sign at a size of about 1: (160 / 4 + 2)^0.5 and 36^0.5 of them, 8.9 2^-24 = 5.3e-7 in
the mean square, and twice that as the bound.
"""
import ctypes
import random

import numpy as np
import pytest

import floneum_amd as fa
from test_abi import FAKE, make_args

CUS = 256


def workspace(B, H, Hkv, rows, Skv, D, dtype, lens=False):
    a, need = make_args(B=B, H=H, Hkv=Hkv, Sq=rows, Skv=Skv, D=D, dtype=dtype), ctypes.c_size_t()
    if lens:
        a.kv_lens = FAKE
    assert fa.lib().fhip_flash_attention_workspace_bytes(ctypes.byref(a), CUS, ctypes.byref(need)) == fa.OK
    return need.value


def planned_splits(B, H, Hkv, rows, Skv, D, dtype, lens=False):
    """The library's own plan, through its planning function (the C ABI's query of it asks for a GPU's stream)."""
    plan = fa.lib()._ZN4fhip11decode_planEiiiiiibbPiS0_S0_S0_
    chunk, n, waves, reported = (ctypes.c_int() for _ in range(4))
    plan(B, Hkv, H // Hkv * rows, Skv, D, CUS, ctypes.c_bool(lens), ctypes.c_bool(dtype == fa.F32), *map(ctypes.byref, (chunk, n, waves, reported)))
    assert (n.value - 1) * chunk.value < Skv <= n.value * chunk.value and n.value <= reported.value
    return n.value


def bytes_of(B, H, Hkv, D, n):
    if n <= 1:
        return 0
    cols = padded = H // Hkv
    for gt in (16, 32):
        if cols > gt:
            padded = max(padded, (cols + gt - 1) // gt * gt)
    partials = B * Hkv * padded * n * (D + 2) * 4
    return partials if n > 8 else partials + B * Hkv * ((cols + 15) // 16) * (n * 128 + 4) + 256


def ordinary_splits(B, Hkv, cols, Skv, D, f32, lens=False):
    """Of chunks of at most 1024 keys (512 for many sequences of lengths of their own), for as many workgroups as the chip holds
    (None: the eight-wavefront form's own rule)."""
    mfma = D % 32 == 0 and 32 <= D <= 256 and not (f32 and D > 192 and cols <= 4)
    gt = (32 if cols > 16 and D <= (192 if f32 else 128) else 16) if mfma else 1 if cols <= 1 else 2 if cols <= 2 else 4 if cols <= 4 else 8
    units = B * Hkv * ((cols + gt - 1) // gt)
    if mfma and not f32 and D <= 128 and Skv > 2048 and (units >= CUS or cols > 8):
        return None
    target = CUS * (1 if mfma and D > 128 else 2 if mfma or f32 else 4)
    step = 64 if f32 else 128
    if not mfma:
        step = min(128, 16 * (64 // (4 if D <= 32 else 8 if D <= 64 else 16 if D <= 128 else 32)))
    n = max(min(-(-target // units), -(-Skv // step)), -(-Skv // (512 if lens and units >= target else 1024)), 1)
    if Skv <= 256 and mfma:
        n = 1
    chunk = -(-(-(-Skv // n)) // step) * step
    return -(-Skv // chunk)


def test_the_workspace_is_that_of_the_ordinary_splits():
    """Reported for them also where fewer are run, and what those write fits into it."""
    rng = random.Random(3)
    fewer = 0
    for _ in range(3000):
        B, (H, Hkv) = rng.randint(1, 40), rng.choice([(32, 8), (16, 4), (16, 16), (8, 4), (32, 32), (7, 7), (40, 2)])
        D, rows, dtype = rng.choice([32, 64, 80, 96, 128, 192, 256]), rng.choice([1, 1, 2, 4]), rng.choice([fa.F32, fa.F16, fa.BF16])
        Skv, lens = int(2 ** rng.uniform(7, 15)), rng.random() < 0.3
        n = ordinary_splits(B, Hkv, H // Hkv * rows, Skv, D, dtype == fa.F32, lens)
        if n is None or B * H * Skv * D > 2 ** 33:
            continue
        call = (B, H, Hkv, rows, Skv, D, dtype, lens)
        need, run = workspace(*call), planned_splits(*call)
        assert need == bytes_of(B, H * rows, Hkv, D, n), call
        assert bytes_of(B, H * rows, Hkv, D, run) <= need, call
        assert run == n or not lens, call
        fewer += run < n
    assert fewer > 50


@pytest.mark.parametrize("B, H, Hkv, Skv, D, dtype", [(20, 16, 4, 4001, 256, fa.BF16), (20, 32, 8, 4500, 128, fa.F32)])
def test_calls_share_a_workspace(B, H, Hkv, Skv, D, dtype):
    """With and without per-sequence lengths, and at the lengths that a growing cache has been through."""
    need = workspace(B, H, Hkv, 1, Skv, D, dtype)
    assert workspace(B, H, Hkv, 1, Skv, D, dtype, lens=True) == need
    assert all(workspace(B, H, Hkv, 1, n, D, dtype) <= need for n in range(1, Skv))


@pytest.mark.parametrize("B, H, Hkv, Skv, D, dtype, splits", [
    (16, 32, 8, 4096, 128, fa.F16, 4), (16, 32, 8, 4104, 128, fa.F16, 4), (16, 32, 8, 8192, 128, fa.F16, 8),
    (20, 16, 4, 4001, 256, fa.BF16, 3), (20, 32, 8, 4500, 128, fa.F32, 3), (9, 32, 8, 4096, 128, fa.F32, 8), (12, 32, 8, 3000, 128, fa.F16, 6),
])
def test_splits(B, H, Hkv, Skv, D, dtype, splits):
    assert planned_splits(B, H, Hkv, 1, Skv, D, dtype) == splits


@pytest.mark.parametrize("B, H, Hkv, rows, Skv, D, dtype", [
    (26, 16, 16, 1, 9663, 64, fa.F32), (16, 32, 8, 1, 8200, 128, fa.F16),  # more than four workgroups per CU
    (21, 8, 4, 1, 4701, 256, fa.BF16), (21, 8, 4, 1, 1512, 160, fa.F32),   # eleven units of three splits on an XCD of 32 CUs
    (8, 32, 8, 1, 8946, 32, fa.F16), (17, 16, 4, 1, 9008, 128, fa.F16),    # from nine splits to seven
    (13, 32, 8, 4, 6032, 48, fa.F16), (11, 32, 8, 1, 15870, 80, fa.BF16),  # the vector variant
])
def test_calls_that_keep_their_ordinary_splits(B, H, Hkv, rows, Skv, D, dtype):
    assert planned_splits(B, H, Hkv, rows, Skv, D, dtype) == ordinary_splits(B, Hkv, H // Hkv * rows, Skv, D, dtype == fa.F32)


@pytest.mark.parametrize("B, H, Hkv, rows, Skv, D, dtype, splits", [
    (3, 32, 8, 1, 13774, 96, fa.BF16, 18), (10, 8, 4, 2, 10826, 96, fa.F16, 11), (9, 16, 4, 1, 9000, 128, fa.F16, 12), (3, 32, 8, 1, 13774, 96, fa.F32, 20),
])
def test_splits_counted_down_to_one_round(B, H, Hkv, rows, Skv, D, dtype, splits):
    """A few workgroups beyond what the chip holds are taken back above 8 splits; calls with per-sequence lengths keep them, and both
    report the same workspace."""
    call = (B, H, Hkv, rows, Skv, D, dtype)
    ordinary = ordinary_splits(B, Hkv, H // Hkv * rows, Skv, D, dtype == fa.F32)
    assert planned_splits(*call) == splits < ordinary and B * Hkv * splits <= 2 * CUS < B * Hkv * ordinary
    assert planned_splits(*call, lens=True) == ordinary
    assert workspace(*call) == workspace(*call, lens=True) == bytes_of(B, H * rows, Hkv, D, ordinary)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [fa.F32, fa.F16, fa.BF16])
@pytest.mark.parametrize("B, H, Hkv, rows, Skv, D", [(16, 8, 8, 1, 4104, 32), (17, 16, 8, 2, 4500, 32), (20, 8, 4, 1, 3000, 160)])
def test_long_chunks(device, dtype, B, H, Hkv, rows, Skv, D):
    rng = np.random.default_rng(Skv)
    tq, tk, tv = (fa.Tensor.from_numpy(device, rng.normal(0, 1, shp).astype(np.float32), dtype)
                  for shp in [(B, H, rows, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)])
    analytic = (True, Skv - rows, 0) if rows > 1 else None
    assert tq.selected_kernel(tk, tv, D ** -0.5, analytic=analytic) == fa.KERNEL_DECODE_SPLITKV
    assert tq.decode_plan(tk, tv, D ** -0.5, analytic=analytic)["nsplit"] > 1
    out = np.asarray(tq.flash_attention(tk, tv, D ** -0.5, analytic=analytic).to_numpy(), np.float64)
    q, k, v = (np.asarray(t.to_numpy(), np.float64) for t in (tq, tk, tv))
    k, v = (np.repeat(a, H // Hkv, axis=1) for a in (k, v))
    s = q @ k.transpose(0, 1, 3, 2) * D ** -0.5
    if analytic:
        s = np.where(np.arange(Skv)[None, :] > np.arange(rows)[:, None] + Skv - rows, -np.inf, s)
    p = np.exp(s - s.max(-1, keepdims=True))
    ref = (p / p.sum(-1, keepdims=True)) @ v
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    assert err <= {fa.F32: 1.1e-6, fa.F16: 2.0 ** -10, fa.BF16: 2.0 ** -7}[dtype], f"relative L2 {err:.2e}"
