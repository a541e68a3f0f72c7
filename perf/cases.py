"""The attention work that users of this framework have it do, as cases that can be timed and compared.

Five kinds of calls, each through the package's public entry points:

  step     one attention layer of one chat stream generating one token: rotary embedding of q and k, the new key and
           value into the (full, sliding) cache, attention over the cache
  layer    the same layer on a whole prompt: q / k norms, rotary embedding, cache, attention with the causal mask tensor
  decode   attention of one to four new tokens per sequence over a batch's cache, even or ragged lengths
  prefill  attention of many new rows: a prompt, a prompt fed in chunks under a sliding window, a follow-up message on a
           long cache, an image's patches without a mask
  encoder  bidirectional attention with an additive padding mask of finite values

Tensors are N(0, std^2), with std 1 where rows are normalised projections and 0.5 for long caches, like the rest of the
repository's measurements.
"""
import math
import random

import numpy as np
import torch

import floneum_amd as fa

TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
FHIP = {"f32": fa.F32, "f16": fa.F16, "bf16": fa.BF16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}


def _case(kind, dtype, batch, heads, kv_heads, head_dim, rows, keys, causal=False, window=0, ragged=False, std=1.0, name=None):
    c = dict(kind=kind, dtype=dtype, batch=batch, heads=heads, kv_heads=kv_heads, head_dim=head_dim, rows=rows, keys=keys,
             causal=causal, window=window, ragged=ragged, std=std)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # one chat stream generating a token on a context of 4096 positions, in the f32 that the reference keeps its cache in
        _case("step", "f32", 1, 32, 8, 128, 1, 4096, name="chat_step_f32"),
        # a serving batch generating one token per sequence, 16-bit cache
        _case("decode", "f16", 16, 32, 8, 128, 1, 4096, std=0.5, name="decode_batch_f16"),
        # the same for a model with a key length of 256, with odd lengths
        _case("decode", "bf16", 16, 16, 4, 256, 1, 4001, std=0.5, name="decode_batch_d256_bf16"),
        # a ragged serving batch without grouped heads: 128 to 32768 cached keys per sequence
        _case("decode", "f16", 32, 32, 32, 96, 1, 32768, ragged=True, name="decode_ragged_f16"),
        # the first layer work of a 512-token prompt, as the reference calls it: f32, norms, rotary embedding, mask tensor
        _case("layer", "f32", 1, 32, 8, 64, 512, 512, causal=True, name="prompt_layer_f32"),
        # a 4096-token prompt in f32
        _case("prefill", "f32", 1, 32, 8, 128, 4096, 4096, causal=True, name="prompt_f32"),
        # an 8192-token prompt in f16
        _case("prefill", "f16", 1, 32, 8, 128, 8192, 8192, causal=True, name="prompt_f16"),
        # a 4096-token prompt at key length 256
        _case("prefill", "bf16", 1, 16, 4, 256, 4096, 4096, causal=True, name="prompt_d256_bf16"),
        # the next 512 tokens of four prompts fed in chunks under a 4096-key window, after 16384 cached ones that were cut to it
        _case("prefill", "bf16", 4, 32, 8, 128, 512, 4096, causal=True, window=4096, name="window_chunk_bf16"),
        # a follow-up message on a long conversation: odd sizes, few rows on many keys
        _case("prefill", "f32", 1, 32, 8, 128, 129, 8003, causal=True, name="chat_turn_f32"),
        # an image's patches in a vision block of head_dim 80: no mask
        _case("prefill", "f16", 1, 16, 16, 80, 4096, 4096, name="vision_f16"),
        # a batch of padded sentences in an encoder: -10000 on the padding
        _case("encoder", "f32", 8, 12, 12, 64, 512, 512, name="encoder_padding_f32"),
    ]


def _between(rng, lo, hi):
    """A whole number in [lo, hi], even over the logarithm: odd ones as often as even ones."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "layer", "decode", "decode", "prefill", "prefill", "prefill", "encoder"])
    dtype = rng.choice(["f32", "f16", "bf16"])
    heads, kv_heads = rng.choice([(32, 8), (16, 4), (16, 16), (8, 4), (32, 32)])
    if kind == "step":
        return _case("step", dtype, 1, heads, kv_heads, rng.choice([64, 128]), 1, _between(rng, 300, 16000))
    if kind == "layer":
        return _case("layer", dtype, 1, heads, kv_heads, rng.choice([64, 128]), *[_between(rng, 30, 2000)] * 2, causal=True)
    if kind == "encoder":
        rows = _between(rng, 60, 1000)
        return _case("encoder", "f32", _between(rng, 1, 16), 12, 12, 64, rows, rows)
    if kind == "decode":
        head_dim, rows, ragged = rng.choice([64, 96, 128, 256]), rng.choice([1, 1, 1, 2, 4]), rng.random() < 0.3
        keys = _between(rng, 300, 16000)
        most = int(4e9 / (2 * BYTES[dtype] * kv_heads * keys * head_dim))  # 4 GB of cache at most
        batch = _between(rng, 1, max(1, min(32, most)))
        return _case("decode", dtype, batch, heads, kv_heads, head_dim, rows, keys, causal=rows > 1 and not ragged,
                     ragged=ragged, std=0.5)
    # prefill
    head_dim = rng.choice([64, 80, 96, 128, 128, 256])
    shape = rng.choice(["prompt", "chunk", "turn", "image"])
    batch, window = 1, 0
    if head_dim == 256 and heads == 32:
        heads, kv_heads = 16, 4
    if shape == "prompt":
        rows = keys = _between(rng, 100, 4000)
    elif shape == "image":
        rows = keys = _between(rng, 200, 4000)
        head_dim, heads, kv_heads = rng.choice([64, 80, 128]), 16, 16
    elif shape == "chunk":
        rows, window, batch = _between(rng, 100, 1000), 4096, rng.choice([1, 2] if dtype == "f32" else [1, 2, 4])
        keys = rows + _between(rng, 1000, 7000)
    else:
        rows = _between(rng, 9, 300)
        keys = rows + _between(rng, 1000, 16000)
    return _case("prefill", dtype, batch, heads, kv_heads, head_dim, rows, keys, causal=shape != "image", window=window)


def _lengths(c):
    """Key counts of a ragged batch, or tokens of padded sentences: spread evenly over what such a batch holds."""
    r = random.Random(c["batch"] * 100003 + c["keys"])
    low = 128 if c["kind"] == "decode" else max(1, c["keys"] // 4)
    low = min(low, c["keys"])
    return [r.randint(low, c["keys"]) for _ in range(c["batch"])]


class _TorchBuffer:
    """Memory of a torch tensor as the buffer of a floneum_amd.Tensor."""

    def __init__(self, device, tensor):
        self.device, self.tensor, self.ptr = device, tensor, tensor.data_ptr()


class _Alias:
    """Device memory of a cache view as torch sees it."""

    def __init__(self, view, shape):
        n = BYTES[{v: k for k, v in FHIP.items()}[view.dtype]]
        self.view = view
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<f4" if n == 4 else "<i2", version=2,
                                             data=(view.buffer.ptr + view.offset * n, False),
                                             strides=tuple(s * n for s in view.strides))


def _wrap(device, tensor, dtype):
    return fa.Tensor(_TorchBuffer(device, tensor), FHIP[dtype], tuple(tensor.shape))


def _unwrap(view, dtype, shape=None):
    t = torch.as_tensor(_Alias(view, shape or view.shape), device="cuda")
    return t if dtype == "f32" else t.view(TORCH[dtype])


def prepare(case, seed):
    c, dev = case, fa.Device.default()
    gen = torch.Generator(device="cuda").manual_seed(seed)
    B, H, Hkv, D, rows, keys, dtype = (c[k] for k in ("batch", "heads", "kv_heads", "head_dim", "rows", "keys", "dtype"))

    def normal(*shape):
        return torch.empty(shape, dtype=TORCH[dtype], device="cuda").normal_(0.0, c["std"], generator=gen)

    s = dict(case=c, scale=D ** -0.5, out=torch.empty((B, rows, H, D), dtype=TORCH[dtype], device="cuda"))
    # the output as the projection behind attention reads it: [batch, rows, heads * head_dim]
    s["fa_out"] = _wrap(dev, s["out"], dtype).transpose(1, 2)
    if c["kind"] in ("step", "layer"):
        # projections as a model holds them, [batch, rows, heads, head_dim]
        q, k, v = normal(B, rows, H, D), normal(B, rows, Hkv, D), normal(B, rows, Hkv, D)
        s["q"], s["k"], s["v"] = (_wrap(dev, t, dtype).transpose(1, 2) for t in (q, k, v))
        s["cache"] = fa.KvCache(2, keys, FHIP[dtype], dev)
        s["start"] = keys if c["kind"] == "step" else 0
        s["rope"] = fa.RopeCache(D, s["start"] + rows, 10000.0, dev)
    if c["kind"] == "step":
        torch.cuda.synchronize()
        for _ in range(2):  # a cache at its limit, which slides from here on: every row of its memory has been written
            k0, v0 = normal(B, Hkv, keys, D), normal(B, Hkv, keys, D)
            torch.cuda.synchronize()
            views = s["cache"].append(dev, _wrap(dev, k0, dtype), _wrap(dev, v0, dtype))
            dev.synchronize()
        views = s["cache"].append(dev, s["k"], s["v"])
        whole = [fa.Tensor(x.buffer, x.dtype, (B, Hkv, x.strides[1] // D, D)) for x in views]
        s["cached"] = [_unwrap(x, dtype) for x in whole]
    elif c["kind"] == "layer":
        w = [torch.empty(D, device="cuda").normal_(1.0, 0.2, generator=gen).cpu().numpy() for _ in range(2)]
        s["q_norm"], s["k_norm"] = (fa.RmsNorm(x, None, 1e-6, FHIP[dtype], dev) for x in w)
        mask = fa.MaskCache(FHIP[dtype]).get_mask_on_device(rows, 0, None, dev)
        s["mask"] = (mask.mask(), fa.MaskKind.QKMask, mask.intervals())
        s["attention_mask"] = mask
        s["cached"], s["at"] = None, None
    else:
        q, k, v = normal(B, H, rows, D), normal(B, Hkv, keys, D), normal(B, Hkv, keys, D)
        s["q"], s["k"], s["v"] = (_wrap(dev, t, dtype) for t in (q, k, v))
        s["analytic"] = (True, keys - rows, c["window"]) if c["causal"] else None
        s["lens"] = s["mask"] = None
        if c["ragged"] or c["kind"] == "encoder":
            lens = _lengths(c)
            random.Random(seed).shuffle(lens)
            if c["ragged"]:
                s["lens"] = fa.IntTensor(dev, np.asarray(lens, np.int32))
            else:
                bias = (torch.arange(keys, device="cuda")[None, :] >= torch.tensor(lens, device="cuda")[:, None]) * -10000.0
                s["mask"] = (_wrap(dev, bias.to(TORCH[dtype]), dtype), fa.MaskKind.BatchKeyMask)
    torch.cuda.synchronize()
    return s


def run(s):
    kind = s["case"]["kind"]
    if kind == "step":
        q, k, v = s["cache"].qkv_rope_append(s["rope"], s["q"], s["k"], s["v"], s["start"])
        q.flash_attention(k, v, s["scale"], out=s["fa_out"])
        return [s["out"]] + s["cached"]
    if kind == "layer":
        s["cache"].reset()
        q, k, v = s["cache"].qkv_rope_append(s["rope"], s["q"], s["k"], s["v"], 0, False, s["q_norm"], s["k_norm"])
        q.flash_attention(k, v, s["scale"], s["mask"], out=s["fa_out"])
        if s["at"] != (k.buffer.ptr, v.buffer.ptr):
            s["at"], s["cached"] = (k.buffer.ptr, v.buffer.ptr), [_unwrap(k, s["case"]["dtype"]), _unwrap(v, s["case"]["dtype"])]
        return [s["out"]] + s["cached"]
    s["q"].flash_attention(s["k"], s["v"], s["scale"], s["mask"], analytic=s["analytic"], kv_lens=s["lens"], out=s["fa_out"])
    return s["out"]


def _pairs(c):
    """(query row, key) pairs that count, summed over the batch."""
    rows, keys, B = c["rows"], c["keys"], c["batch"]
    if c["ragged"]:
        return rows * sum(_lengths(c))
    if not c["causal"]:
        return B * rows * keys
    pos = np.arange(keys - rows, keys, dtype=np.int64)
    low = np.maximum(pos - c["window"] + 1, 0) if c["window"] else 0
    return B * int(np.sum(pos + 1 - low))


def work(case):
    c, e = case, BYTES[case["dtype"]]
    B, H, Hkv, D, rows, keys = (c[k] for k in ("batch", "heads", "kv_heads", "head_dim", "rows", "keys"))
    kv_rows = sum(_lengths(c)) if c["ragged"] else B * keys
    if c["causal"] and c["window"]:  # keys before the first row's window are not read
        kv_rows = B * min(keys, rows + c["window"] - 1)
    b = e * (2 * B * H * rows * D + 2 * kv_rows * Hkv * D)  # q and out, keys and values
    f = 4 * D * H * _pairs(c)
    if c["kind"] == "step":    # new k and v in, rows of the cache out, tables
        b += e * 4 * B * Hkv * D + 4 * D
    elif c["kind"] == "layer":  # the cache's rows are written here and read by nobody else: k and v in and out
        b += e * 2 * B * Hkv * rows * D + 4 * rows * D + e * 2 * D + e * rows * keys
        f += 6 * B * (H + Hkv) * rows * D
    elif c["kind"] == "encoder":
        b += e * B * keys
    return {"bytes": b, "flops": f}


def tolerance(case):
    # About four times the largest difference from the same call in 64 bits, over the listed cases and a dozen drawn ones:
    # 5.7e-7 in f32, 2.9e-4 in f16, 2.4e-3 in bf16 (results and, in the matrix kernels, probabilities rounded to the type).
    if case["dtype"] == "f32":
        return {"rel": 2.5e-6}
    return {"rel": 1e-3} if case["dtype"] == "f16" else {"rel": 1e-2}
