"""GPU tests of how the term-splitting f32 prefill kernel (floneum_amd/csrc/attn_prefill_f32_terms.hip) reads a mask it adds:
whole tiles four keys at a time, the last one and strided masks element by element, and a padding mask's row looked at by
the kernel itself.  Against the same formula in 64 bits.

Tolerance: 1e-6 relative L2 as for the kernel's other forms (a score and its mask value are added with one rounding, 2^-24
of a score of up to some 10 for the values used here, which moves a probability by at most 6e-7 and their mean by far less).
Reference semantics: fusor-ml/fusor/src/composite/flash_attention.rs:161-177.
"""
import numpy as np
import pytest

import floneum_amd as fa
from test_prefill_f32_terms_gpu import close, in_64_bits, tensors

pytestmark = pytest.mark.gpu
NEG_INF = float("-inf")


def padding_rows(Skv):
    """One row of every kind: an interval at the start, one inside, finite values, two runs, and no visible key."""
    m = np.zeros((5, Skv), np.float32)
    m[0, (Skv + 1) // 2:] = NEG_INF
    m[1, :Skv // 3] = NEG_INF
    m[1, Skv - Skv // 4:] = NEG_INF
    m[2] = np.random.default_rng(Skv).normal(0, 1, Skv)
    m[2, (Skv + 1) // 2:] = -10000.0
    m[3, Skv // 2:(Skv + 1) // 2 + Skv // 5] = NEG_INF
    m[4] = NEG_INF
    return m


@pytest.mark.parametrize("Skv", [1, 5, 31, 32, 33, 255, 257, 1000, 1023, 1024, 1025])
@pytest.mark.parametrize("D", [64, 40])
@pytest.mark.parametrize("layout", ["rows", "columns"])
def test_padding_masks(device, Skv, D, layout):
    """1024 keys and fewer in rows: no scan launch; more keys, or a mask whose keys are not neighbours: one."""
    q, k, v = tensors(7, 5, 4, 2, 37, Skv, D)
    m = padding_rows(Skv)
    tq, tk, tv = (fa.Tensor.from_numpy(device, a, fa.F32) for a in (q, k, v))
    tm = (fa.Tensor.from_numpy(device, m, fa.F32) if layout == "rows"
          else fa.Tensor.from_numpy(device, np.ascontiguousarray(m.T), fa.F32).transpose(0, 1))
    out = tq.flash_attention(tk, tv, D ** -0.5, (tm, fa.MaskKind.BatchKeyMask), force_kernel=fa.KERNEL_PREFILL_F32).to_numpy()
    seen = [b for b in range(5) if (m[b] > NEG_INF).any()]
    assert np.isnan(out[[b for b in range(5) if b not in seen]]).all()
    ref = in_64_bits(q[seen], k[seen], v[seen], D ** -0.5, np.asarray(m[seen], np.float64)[:, None, None, :])
    close(out[seen], ref, f"Skv {Skv}")


@pytest.mark.parametrize("dtype", [fa.F32, fa.F16, fa.BF16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("first", [0, 1, 4])
@pytest.mark.parametrize("Skv", [63, 64, 129])
def test_views_of_a_score_mask(device, dtype, D, first, Skv):
    """A mask inside a wider one: aligned to a four-key piece, to an element only, and rows of an odd length."""
    Sq, wide = 45, 140 if Skv == 64 else 139
    q, k, v = tensors(8, 2, 4, 2, Sq, Skv, D)
    m = np.random.default_rng(9).normal(0, 1, (Sq, wide)).astype(np.float32)
    tq, tk, tv, tm = (fa.Tensor.from_numpy(device, a, dtype) for a in (q, k, v, m))
    view = tm.narrow(1, first, Skv)
    out = tq.flash_attention(tk, tv, D ** -0.5, (view, fa.MaskKind.QKMask), out_dtype=fa.F32,
                             force_kernel=fa.KERNEL_PREFILL_F32).to_numpy()
    q, k, v, m = (t.to_numpy() for t in (tq, tk, tv, tm))
    close(out, in_64_bits(q, k, v, D ** -0.5, np.asarray(m, np.float64)[:, first:first + Skv]), f"D{D}")


@pytest.mark.parametrize("dtype", [fa.F32, fa.BF16])
@pytest.mark.parametrize("D", [64, 128, 40])
@pytest.mark.parametrize("kind", ["rows", "keys"])
@pytest.mark.parametrize("Sq,Skv", [(45, 131), (21, 2111)])  # the second: keys split over workgroups
def test_lowest_finite_values(device, dtype, D, kind, Sq, Skv):
    """Padding with the type's lowest finite value, which is no -inf: beside a zero it has no weight, but a row of nothing else
    takes the mean of its keys (every score vanishes beside it), and of two such values the higher one takes all."""
    low = np.float32(-3.4028235e38 if dtype == fa.F32 else -3.3895314e38)
    B = 3 if kind == "keys" else 2
    q, k, v = tensors(10, B, 4, 2, Sq, Skv, D)
    m = np.zeros((B if kind == "keys" else Sq, Skv), np.float32)
    m[0] = low
    m[1, : Skv // 3] = low
    m[2, ::3] = low
    m[2, m[2] == 0] = low * np.float32(0.8125)
    tq, tk, tv, tm = (fa.Tensor.from_numpy(device, a, dtype) for a in (q, k, v, m))
    out = tq.flash_attention(tk, tv, D ** -0.5, (tm, fa.MaskKind.QKMask if kind == "rows" else fa.MaskKind.BatchKeyMask),
                             out_dtype=fa.F32, force_kernel=fa.KERNEL_PREFILL_F32).to_numpy()
    q, k, v, m = (np.asarray(t.to_numpy(), np.float64) for t in (tq, tk, tv, tm))
    close(out, in_64_bits(q, k, v, D ** -0.5, m if kind == "rows" else m[:, None, None, :]), f"D{D} {kind}")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Sq,Skv", [(300, 300), (21, 2111)])
def test_one_rounding_at_the_size_of_the_mask(device, D, Sq, Skv):
    """Scores with mask values about -1000 added lie between -1024 and -512, where neighbours are 2^-14 apart.  The sum rounds
    once there, as the reference's does: an error uniform over 2^-14, deviation 2^-14 / sqrt(12) = 1.76e-5, which is the
    relative error of each probability and, the keys' errors being independent, of the result.  A second rounding, of
    the score times log2(e), would bring it to 3.0e-5; 2.2e-5 is allowed."""
    q, k, v = tensors(14, 2, 4, 2, Sq, Skv, D)
    m = (-1000 + np.random.default_rng(15).normal(0, 1, (2, Skv))).astype(np.float32)
    tq, tk, tv, tm = (fa.Tensor.from_numpy(device, a, fa.F32) for a in (q, k, v, m))
    out = np.asarray(tq.flash_attention(tk, tv, D ** -0.5, (tm, fa.MaskKind.BatchKeyMask),
                                        force_kernel=fa.KERNEL_PREFILL_F32).to_numpy(), np.float64)
    ref = in_64_bits(q, k, v, D ** -0.5, np.asarray(m, np.float64)[:, None, None, :])
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    assert err <= 2.2e-5, f"relative L2 {err:.2e}"
