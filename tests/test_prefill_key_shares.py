"""Calls whose rows all see about the same keys (chunks of a prompt, follow-up messages, images): into how many shares their keys go,
by the workspace the library asks for, and such calls against the formula in 64 bits, into outputs of any stride and type.

Tolerance: 16-bit results as in tests/test_prefill_mfma_forms_gpu.py.  In f32 a score sums D products in terms of which each is
exact, 2^-24 and less of its size apart from a rounding per slice of 16, the probabilities and the shares' sums round a dozen times each:
40 roundings of 2^-24 and either sign bound the relative L2 by 40^0.5 2^-24 = 3.8e-7; twice that.
"""
import ctypes

import numpy as np
import pytest

import floneum_amd as fa
from test_abi import make_args

CUS = 256


def shares(B, H, Hkv, Sq, Skv, D, dtype, causal=True, window=0):
    a, need = make_args(B=B, H=H, Hkv=Hkv, Sq=Sq, Skv=Skv, D=D, dtype=dtype), ctypes.c_size_t()
    if causal:
        a.analytic.enabled, a.analytic.causal, a.analytic.q_pos_offset, a.analytic.window = 1, 1, Skv - Sq, window
    assert fa.lib().fhip_flash_attention_workspace_bytes(ctypes.byref(a), CUS, ctypes.byref(need)) == fa.OK
    per = B * H * Sq * (D + (2 if dtype == fa.F32 else 4)) * 4
    assert need.value % per == 0
    return need.value // per


@pytest.mark.parametrize("call, want", [
    # 16-bit: short views of more than 64 rows, full rounds of workgroups, no split where one round is there already
    ((1, 8, 4, 189, 1993, 80, fa.F16), 8), ((4, 32, 8, 207, 4303, 96, fa.F16), 0), ((1, 32, 32, 49, 3032, 128, fa.BF16), 8),
    ((1, 32, 8, 231, 14900, 64, fa.F16), 8), ((1, 16, 16, 4096, 4096, 80, fa.F16, False), 0),
    # f32: even rows in the shares of least time; up to 128 rows, squares and up to 768 keys by the former rule
    ((2, 32, 8, 275, 2911, 64, fa.F32), 3), ((1, 16, 16, 1156, 1156, 128, fa.F32, False), 3), ((1, 16, 16, 1156, 1156, 128, fa.F32), 0),
    ((1, 16, 16, 768, 768, 128, fa.F32, False), 2), ((1, 32, 8, 128, 8192, 128, fa.F32), 4), ((1, 32, 8, 129, 8003, 128, fa.F32), 6),
    # above 128 dims in f32: one round of workgroups, of a square those whose rows see a key; up to 64 rows the former rule
    ((1, 16, 4, 148, 3510, 256, fa.F32), 11), ((1, 16, 4, 300, 700, 256, fa.F32), 6), ((1, 8, 4, 1024, 1024, 256, fa.F32), 6),
    ((1, 16, 4, 2048, 2048, 256, fa.F32), 0), ((1, 16, 4, 1024, 1024, 256, fa.F32, False), 2), ((1, 16, 4, 64, 4096, 256, fa.F32), 16),
    # above 128 dims: up to four shares of 512 keys
    ((1, 16, 4, 141, 2659, 256, fa.BF16), 4), ((1, 16, 4, 141, 1000, 256, fa.BF16), 0),
    # but not of many rows, whose partials' bytes cost more than the rounds of tiles gain
    ((3, 12, 12, 413, 1858, 256, fa.BF16), 0), ((2, 12, 12, 893, 2927, 256, fa.BF16, True, 1734), 0), ((3, 6, 3, 1209, 2620, 192, fa.F16), 0),
])
def test_shares(call, want):
    assert shares(*call) == want


@pytest.mark.parametrize("call, want", [((8, 16, 4, 1278, 21043, 128), 0), ((4, 16, 16, 2363, 21840, 128), 0), ((2, 16, 16, 2826, 9136, 128), 0),
                                        ((2, 16, 16, 2320, 14643, 80), 2), ((8, 12, 12, 458, 30160, 96), 0)])
def test_the_partials_of_a_call_are_limited(call, want):
    """16-bit calls: 64 MiB where the time asks for more shares than the rules (the first of these asked for 165, the next for 152)."""
    B, H, _, rows, _, D = call
    assert shares(*call, fa.BF16) == want and want * B * H * rows * (D + 4) * 4 <= 64 << 20


@pytest.mark.parametrize("call, known, unknown", [
    ((2, 6, 3, 84, 1416, 80, fa.F16), 8, 0), ((4, 16, 4, 75, 1187, 128, fa.F16), 3, 0), ((3, 12, 12, 271, 1201, 256, fa.F16), 2, 0),
    ((1, 32, 8, 360, 1844, 128, fa.F32), 5, 2), ((1, 16, 4, 765, 1999, 96, fa.F32), 5, 2), ((3, 16, 4, 321, 1323, 128, fa.F32), 3, 0),
])
def test_rows_that_may_see_fewer_keys_than_the_call_has(call, known, unknown):
    """Sequences with lengths of their own take more shares than by rule only for 30 % of the time; masks over (query, key) are planned as
    causal ones, whose bits they have."""
    B, H, Hkv, rows, keys, D, dtype = call
    a, need = make_args(B=B, H=H, Hkv=Hkv, Sq=rows, Skv=keys, D=D, dtype=dtype), ctypes.c_size_t()
    per = B * H * rows * (D + (2 if dtype == fa.F32 else 4)) * 4

    def asked():
        assert fa.lib().fhip_flash_attention_workspace_bytes(ctypes.byref(a), CUS, ctypes.byref(need)) == fa.OK
        return need.value / per

    assert shares(*call, causal=False) == known and asked() == known
    a.kv_lens = 0x1000
    assert asked() == unknown
    a.kv_lens = None
    a.mask_kind, a.mask.ptr, a.mask_intervals = fa.MaskKind.QKMask, 0x10000, 0x20000
    a.mask.shape[:], a.mask.stride[:] = (rows, keys), (keys, 1)
    assert asked() == known == shares(*call)


@pytest.mark.parametrize("dtype, D", [(fa.F32, 64), (fa.F32, 100), (fa.F32, 128), (fa.F32, 256), (fa.F16, 64), (fa.BF16, 128), (fa.F16, 192), (fa.F16, 256)])
def test_a_mask_tensor_shares_the_plan_of_the_causal_mask(dtype, D):
    """The tensor of a causal mask gives the bits of the analytic call, so chunks of a prompt are shared out alike."""
    rng = np.random.default_rng(D)
    for _ in range(300):
        rows, Hkv = int(rng.integers(65, 1500)), int(rng.choice([1, 2, 4, 8]))
        keys, B, H = 2 * rows + int(rng.integers(0, 6000)), int(rng.integers(1, 5)), Hkv * int(rng.choice([1, 2, 4]))
        asked = []
        for masked in (False, True):
            a, need = make_args(B=B, H=H, Hkv=Hkv, Sq=rows, Skv=keys, D=D, dtype=dtype), ctypes.c_size_t()
            if masked:
                a.mask_kind, a.mask.ptr, a.mask_intervals = fa.MaskKind.QKMask, 0x10000, 0x20000
                a.mask.shape[:], a.mask.stride[:] = (rows, keys), (keys, 1)
            else:
                a.analytic.enabled, a.analytic.causal, a.analytic.q_pos_offset = 1, 1, keys - rows
            assert fa.lib().fhip_flash_attention_workspace_bytes(ctypes.byref(a), CUS, ctypes.byref(need)) == fa.OK
            asked.append(need.value)
        assert asked[0] == asked[1], (B, H, Hkv, rows, keys)


@pytest.mark.parametrize("call", [(1, 32, 32, 2859, 7370, 80), (8, 16, 16, 689, 6007, 80), (8, 4, 1, 2154, 6748, 96)])
def test_full_grids_are_split_for_a_tenth_of_their_time(call):
    """16-bit grids of more than half the chip, which two shares slow down (us 209 -> 238, 210 -> 245, 190 -> 211)."""
    assert shares(*call, fa.F16) == 0


@pytest.mark.parametrize("D, dtype", [(64, fa.F32), (96, fa.F32), (256, fa.F32), (64, fa.F16), (128, fa.BF16), (256, fa.F16)])
@pytest.mark.parametrize("before", [0, 1, 127, 128, 4000, 20000])
def test_a_window_is_planned_on_its_keys(D, dtype, before):
    """A view with more keys in front of the window asks for what the window's own keys ask for, to the next 128."""
    rows, window = 300, 2048
    seen = rows + window - 1
    got = shares(2, 16, 4, rows, before + seen, D, dtype, window=window)
    assert got in {shares(2, 16, 4, rows, n, D, dtype) for n in range(seen, seen + 128)}


@pytest.mark.parametrize("D", [256, 192, 160])
@pytest.mark.parametrize("H, Hkv, rows", [(4, 1, 3000), (8, 4, 2000), (16, 8, 1000), (12, 12, 1693)])
def test_a_windowed_prompt_is_not_shared_out_as_a_whole_one(H, Hkv, rows, D):
    """Above 128 dims a row block under a narrow window would meet one or two of the shares that the whole prompt has."""
    whole = shares(1, H, Hkv, rows, rows, D, fa.F32)
    assert whole >= 3
    assert all(shares(1, H, Hkv, rows, rows, D, fa.F32, window=w) == 0 for w in (1, 32, 128))
    assert all(shares(1, H, Hkv, rows, rows, D, fa.F32, window=w) == whole for w in (rows - 1, rows, 2 * rows, 2 ** 40, 2 ** 63 - 1))


@pytest.mark.parametrize("call, want", [((1, 4, 4, 1768, 1768, 160), 3), ((1, 4, 4, 1985, 1985, 192), 3), ((1, 6, 3, 1603, 2289, 160), 3),
                                        ((3, 12, 12, 413, 700, 256), 0), ((2, 16, 4, 1205, 1205, 160), 0), ((1, 6, 3, 1256, 1256, 256), 2)])
def test_squares_with_a_mask_tensor_are_split_to_one_round(call, want):
    """16-bit calls above head_dim 128 whose rows may see from one to all of the keys."""
    B, H, Hkv, rows, keys, D = call
    a, need = make_args(B=B, H=H, Hkv=Hkv, Sq=rows, Skv=keys, D=D, dtype=fa.F16), ctypes.c_size_t()
    a.mask_kind, a.mask.ptr, a.mask_intervals = fa.MaskKind.QKMask, 0x10000, 0x20000
    a.mask.shape[:], a.mask.stride[:] = (rows, keys), (keys, 1)
    assert fa.lib().fhip_flash_attention_workspace_bytes(ctypes.byref(a), CUS, ctypes.byref(need)) == fa.OK
    assert need.value == want * B * H * rows * (D + 4) * 4


class TermsCall(ctypes.Structure):  # floneum_amd/csrc/common.h
    _fields_ = [(n, ctypes.c_int) for n in ("B", "Hkv", "G", "Sq", "Skv", "D", "cus")] + [
        ("uneven", ctypes.c_bool), ("window", ctypes.c_int64), ("f32", ctypes.c_bool), ("causal", ctypes.c_bool)]


@pytest.mark.parametrize("call, want", [
    # workgroups of half the units, or of two key groups, see fewer keys beside a window's (us in those of four units and now: 21.7 and
    # 13.9, 19.2 and 13.4, 14.2 and 10.4, 18.3 and 13.6, 16.4 and 13.4, 27.1 and 24.0)
    ((3, 16, 1, 156, 314, 96, 32), (2, 2)), ((1, 16, 1, 228, 319, 80, 24), (2, 2)), ((1, 8, 2, 224, 249, 80, 25), (2, 2)),
    ((1, 16, 1, 1558, 1580, 64, 27), (2, 2)), ((1, 4, 2, 155, 309, 96, 29), (2, 2)), ((4, 16, 1, 273, 444, 96, 82), (4, 2)),
])
def test_forms_under_a_narrow_window(call, want):
    """The form of an unsplit f32 chunk (batch, KV heads, heads each, rows, keys seen, head_dim, window), from what the launcher asks."""
    rule = fa.lib()._ZN4fhip22prefill_f32_terms_formERKNS_9TermsCallEi
    rule.restype, rule.argtypes = ctypes.c_uint64, [ctypes.POINTER(TermsCall), ctypes.c_int]
    form = rule(ctypes.byref(TermsCall(*call[:6], CUS, False, call[6], True, True)), 1)
    assert (form & 0xffffffff, form >> 32) == want


@pytest.mark.parametrize("call, want", [((1, 8, 4, 162, 390, 64), 4), ((1, 16, 4, 154, 445, 64), 4), ((8, 8, 2, 516, 2456, 64), 2), ((8, 32, 8, 180, 2905, 64), 2)])
def test_f32_tensors_are_shared_out_by_the_quickest_form(call, want):
    """(us, in these shares and in those of the least time of the form that runs: 12.8 and 14.6, 13.3 and 14.9, 143 and 162, 199 and 238)"""
    assert shares(*call, fa.F32) == want


@pytest.mark.parametrize("call", [(4, 8, 4, 1071, 2216, 128), (1, 32, 8, 1494, 2990, 96), (3, 8, 2, 1832, 3665, 96), (1, 16, 4, 2436, 5021, 80)])
def test_long_chunks_are_not_split_for_rows_that_see_few_keys(call):
    """Chunks of more than a round of workgroups, whose later rounds see the fewest keys under a causal mask (us unsplit and in the two shares
    that calls without one take: 203 and 257, 245 and 284, 287 and 339, 348 and 433)."""
    assert shares(*call, fa.F32) == 0 and shares(*call, fa.F32, causal=False) >= 2


@pytest.mark.parametrize("H, Hkv, rows, keys, D, causal, want", [
    (16, 4, 1500, 1500, 100, False, 2), (32, 8, 200, 3000, 100, True, 7), (32, 8, 200, 3000, 36, True, 7), (16, 8, 400, 2500, 60, True, 8),
])
def test_16_bit_tensors_on_the_f32_kernel_are_planned_for_their_one_form(H, Hkv, rows, keys, D, causal, want):
    """Head dims that are no multiple of 8.  (f32 tensors have other forms, and other shares, to choose from.)"""
    a, need = make_args(B=1, H=H, Hkv=Hkv, Sq=rows, Skv=keys, D=D, dtype=fa.F16), ctypes.c_size_t()
    if causal:
        a.analytic.enabled, a.analytic.causal, a.analytic.q_pos_offset = 1, 1, keys - rows
    assert fa.lib().fhip_flash_attention_workspace_bytes(ctypes.byref(a), CUS, ctypes.byref(need)) == fa.OK
    assert need.value == want * H * rows * (D + 2) * 4
    assert shares(1, H, Hkv, rows, keys, D, fa.F32, causal=causal) < want


def test_narrow_windows_are_not_shared_out():
    """Above 192 dims a short walk is quicker unsplit on the f32 instruction than in shares of the terms kernel."""
    assert [shares(1, 32, 32, 396, 396, 256, fa.F32, window=w) for w in (130, 156, 200, 300)] == [0, 0, 0, 3]
    assert [shares(1, 32, 32, 175, 175, 256, fa.F32, window=w) for w in (50, 0)] == [0, 2]


@pytest.mark.parametrize("H, Hkv, rows, keys, D, window, want", [
    # of three shares two would hold no key of a row block
    (32, 8, 173, 1420, 80, 334, 0), (32, 8, 173, 1420, 80, 0, 3), (32, 8, 173, 1420, 80, 1400, 3),
])
def test_a_windowed_chunk_is_not_shared_out_as_a_whole_one(H, Hkv, rows, keys, D, window, want):
    assert shares(3, H, Hkv, rows, keys, D, fa.F32, window=window) == want


def test_a_wide_window_is_planned_as_none():
    assert [shares(1, 32, 8, 1100, 4357, 128, fa.F32, window=w) for w in (1000, 2885, 4357)] == [0, 2, 2]
    assert shares(2, 32, 32, 728, 3304, 64, fa.F32, window=2549) == 2


def test_rows_behind_a_window_see_alike():
    """A chunk of more rows than its window is planned as an even call from the keys on at which the first row sees half a window."""
    assert [shares(1, 8, 4, 1200, keys, 128, fa.F32, window=600) for keys in (1200, 1498, 1499, 1799, 4000)] == [3, 3, 0, 0, 0]
    assert shares(1, 4, 1, 1804, 6014, 256, fa.F32, window=1515) >= 3  # (above 128 dims uneven shares know their window)


@pytest.mark.parametrize("at", [2 ** 20, 2 ** 62 - 2, 2 ** 62, 2 ** 63 - 1 - 1156])
def test_rows_far_behind_the_keys_see_alike(at):
    """Rows and a window at the end of the 64 bits: every row sees every key, as without a mask."""
    a, need = make_args(B=1, H=16, Hkv=16, Sq=1156, Skv=1156, D=128, dtype=fa.F32), ctypes.c_size_t()
    a.analytic.enabled, a.analytic.causal, a.analytic.q_pos_offset, a.analytic.window = 1, 1, at, at + 1156
    assert fa.lib().fhip_flash_attention_workspace_bytes(ctypes.byref(a), CUS, ctypes.byref(need)) == fa.OK
    assert need.value == shares(1, 16, 16, 1156, 1156, 128, fa.F32, causal=False) * 16 * 1156 * 130 * 4 > 0


@pytest.mark.gpu
@pytest.mark.parametrize("D", [256, 160])
@pytest.mark.parametrize("H, Hkv, rows, keys, window, how, want", [
    (4, 1, 800, 800, 500, "window", 9), (4, 2, 513, 513, 300, "window", 6), (4, 1, 700, 700, 33, "window", 0), (4, 4, 640, 800, 450, "window", 9),
    (4, 1, 650, 650, 0, "table", 7), (4, 2, 417, 417, 200, "table", 5), (4, 1, 300, 640, 0, "lens", 10), (2, 2, 129, 333, 0, "lens", 4),
])
def test_wide_heads_in_shares(device, H, Hkv, rows, keys, window, how, want, D):
    """Uneven shares and their levels above 128 dims under a window, a mask tensor's interval table and lengths of two sequences (one of
    them in the first share alone)."""
    B = 2 if how == "lens" else 1
    rng = np.random.default_rng(rows * 7 + D)
    q, k, v = tensor(device, rng, fa.F32, (B, H, rows, D)), tensor(device, rng, fa.F32, (B, Hkv, keys, D)), tensor(device, rng, fa.F32, (B, Hkv, keys, D))
    i, j = np.arange(rows)[:, None] + keys - rows, np.arange(keys)[None, :]
    hidden = np.broadcast_to((j > i) | ((j + window <= i) if window else False), (B, rows, keys))
    analytic = mask = lens = None
    if how == "window":
        analytic = (True, keys - rows, window)
    elif how == "table":
        m = fa.Tensor.from_numpy(device, np.where(hidden[0], -np.inf, 0.0).astype(np.float32), fa.F32)
        mask = (m, fa.MaskKind.QKMask)
    else:
        counts = np.array([keys, 20], np.int32)
        lens, hidden = fa.IntTensor(device, counts), np.broadcast_to(np.arange(keys)[None, None, :] >= counts[:, None, None], (B, rows, keys))
    assert shares(B, H, Hkv, rows, keys, D, fa.F32, causal=how != "lens", window=window if how == "window" else 0) == want
    out = q.flash_attention(k, v, D ** -0.5, mask, analytic=analytic, kv_lens=lens).to_numpy().astype(np.float64)
    a, b, c = (t.to_numpy().astype(np.float64) for t in (q, k, v))
    b, c = (np.repeat(t, H // Hkv, axis=1) for t in (b, c))
    s = np.where(hidden[:, None], -np.inf, a @ b.transpose(0, 1, 3, 2) * D ** -0.5)
    p = np.exp(s - s.max(-1, keepdims=True))
    ref = (p / p.sum(-1, keepdims=True)) @ c
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    assert err <= 7.6e-7, f"relative L2 {err:.2e}"


def tensor(device, rng, dtype, shape):
    return fa.Tensor.from_numpy(device, rng.normal(0, 1, shape).astype(np.float32), dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype, B, H, Hkv, Sq, Skv, D, causal, window", [
    (fa.F16, 1, 8, 4, 189, 1993, 80, True, 0), (fa.BF16, 1, 4, 4, 65, 1291, 128, True, 0), (fa.F16, 1, 4, 2, 201, 3333, 64, True, 700),
    (fa.F16, 2, 4, 1, 33, 1409, 96, True, 0), (fa.BF16, 1, 4, 4, 300, 1000, 72, False, 0), (fa.F16, 1, 4, 2, 140, 1999, 256, True, 0),
    (fa.F32, 1, 4, 2, 275, 2911, 64, True, 0), (fa.F32, 1, 4, 4, 1156, 1156, 128, False, 0), (fa.F32, 1, 8, 2, 131, 3000, 80, True, 900),
    (fa.F32, 1, 2, 2, 129, 1025, 36, False, 0), (fa.F32, 2, 4, 2, 150, 900, 256, True, 0),
])
@pytest.mark.parametrize("out", ["contiguous", "turned", "odd rows", "every second"])
def test_shared_keys(device, dtype, B, H, Hkv, Sq, Skv, D, causal, window, out):
    """Every form of the merge's stores: rows of four, rows that are not aligned, elements apart; f32 results of 16-bit calls."""
    rng = np.random.default_rng(Sq * 31 + Skv)
    q, k, v = tensor(device, rng, dtype, (B, H, Sq, D)), tensor(device, rng, dtype, (B, Hkv, Skv, D)), tensor(device, rng, dtype, (B, Hkv, Skv, D))
    analytic = (True, Skv - Sq, window) if causal else None
    out_dtype = fa.F32 if out in ("turned", "every second") else dtype
    if out == "odd rows":
        o = fa.Tensor.from_numpy(device, np.full((B, H, Sq, D + 1), 7.0, np.float32), out_dtype)
        view = fa.Tensor(o.buffer, out_dtype, (B, H, Sq, D), o.strides, 1)
    elif out == "every second":
        o = fa.Tensor.from_numpy(device, np.full((B, H, Sq, 2 * D), 7.0, np.float32), out_dtype)
        view = fa.Tensor(o.buffer, out_dtype, (B, H, Sq, D), o.strides[:3] + (2,), 0)
    else:
        o = fa.Tensor.from_numpy(device, np.full((B, Sq, H, D) if out == "turned" else (B, H, Sq, D), 7.0, np.float32), out_dtype)
        view = o.transpose(1, 2) if out == "turned" else o
    q.flash_attention(k, v, D ** -0.5, analytic=analytic, out_dtype=out_dtype, out=view)
    whole = np.asarray(o.to_numpy(), np.float64)
    got = whole[..., 1:] if out == "odd rows" else whole[..., ::2] if out == "every second" else whole.transpose(0, 2, 1, 3) if out == "turned" else whole
    if out == "odd rows":
        assert np.all(whole[..., 0] == 7.0)
    if out == "every second":
        assert np.all(whole[..., 1::2] == 7.0)
    a, b, c = (np.asarray(t.to_numpy(), np.float64) for t in (q, k, v))
    b, c = (np.repeat(t, H // Hkv, axis=1) for t in (b, c))
    s = a @ b.transpose(0, 1, 3, 2) * D ** -0.5
    if causal:
        i, j = np.arange(Sq)[:, None] + Skv - Sq, np.arange(Skv)[None, :]
        s = np.where((j > i) | ((j + window <= i) if window else False), -np.inf, s)
    p = np.exp(s - s.max(-1, keepdims=True))
    ref = (p / p.sum(-1, keepdims=True)) @ c
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= {fa.F32: 7.6e-7, fa.F16: 2.0 ** -10, fa.BF16: 2.0 ** -7}[dtype], f"relative L2 {err:.2e}"


@pytest.mark.gpu
@pytest.mark.parametrize("keys, lengths", [(800, (800,)), (900, (613, )), (769, (1, )), (801, (801, 260))])
@pytest.mark.parametrize("hidden", [-10000.0, -np.inf, float(np.finfo(np.float32).min)])
@pytest.mark.parametrize("D", [64, 128])
def test_padded_sequences_in_shares(device, keys, lengths, hidden, D):
    """Squares of more than 768 keys with a key mask: the mask-adding form and the interval form in even shares, some of which a
    sequence's keys do not reach."""
    B, H = len(lengths), 12
    rng = np.random.default_rng(keys + D)
    q, k, v = (tensor(device, rng, fa.F32, (B, H, keys, D)) for _ in range(3))
    bias = np.where(np.arange(keys)[None, :] >= np.array(lengths)[:, None], hidden, 0.0).astype(np.float32)
    assert shares(B, H, H, keys, keys, D, fa.F32, causal=False) >= 2
    out = q.flash_attention(k, v, D ** -0.5, (fa.Tensor.from_numpy(device, bias, fa.F32), fa.MaskKind.BatchKeyMask)).to_numpy().astype(np.float64)
    a, b, c = (t.to_numpy().astype(np.float64) for t in (q, k, v))
    s = a @ b.transpose(0, 1, 3, 2) * D ** -0.5 + bias.astype(np.float64)[:, None, None, :]
    p = np.exp(s - s.max(-1, keepdims=True))
    ref = (p / p.sum(-1, keepdims=True)) @ c
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    assert err <= 7.6e-7, f"relative L2 {err:.2e}"
