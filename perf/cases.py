"""The work whose speed this framework is held to, through its public entry points (``amdgpu_rustdsl_amd.ops``).

Three kinds of call:

* ``attend``: ``fmha_fwd_mxfp8`` on tensors that are already MXFP8 (a serving engine's Q and its KV cache);
* ``attend_bf16``: ``fmha_fwd_bf16_via_mxfp8``, bf16 in and bf16 out, the quantisers included;
* ``quantize``: ``quantize_mxfp8`` of K and ``quantize_v`` / ``quantize_v_seq32`` of V, what filling a KV cache costs.

The listed cases are the repository's own configurations (one block, the headline, the long sequence, the causal
prefill, the short query over a long KV range) and the calls around them that a serving program makes: ragged
prompts, grouped-query heads, a decode step, a whole bf16 layer, the cache's quantisation. ``draw`` gives others of
the same ranges.
"""
import math

import torch

from amdgpu_rustdsl_amd import ops

D = 128
LOG2E = 1.4426950408889634


def _attend(name, B, H, HK, S, SK, **kw):
    c = dict(kind="attend", B=B, H=H, HK=HK, S=S, SK=SK, causal=False, lse=False, splits=0, seq32=False, scaled=False,
             partials="fp16")
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest: one head of one short prompt; launch and host latency
        _attend("tiny_B1H1S256", 1, 1, 1, 256, 256),
        # an ordinary ragged cross-length prompt (queries and keys of different, odd lengths)
        _attend("ragged_B1H8S1000_SK1337", 1, 8, 8, 1000, 1337),
        # the headline configuration, with the LSE that a caller merging or differentiating keeps
        _attend("prefill_B4H8S2048_lse", 4, 8, 8, 2048, 2048, lse=True),
        # one medium prompt: too few query tiles for the chip, so the KV range is split
        _attend("prefill_B1H8S2048", 1, 8, 8, 2048, 2048),
        # a long prompt
        _attend("long_B1H8S8192", 1, 8, 8, 8192, 8192),
        # a ragged batch: a last wave of blocks that does not fill the chip
        _attend("ragged_B3H8S3001", 3, 8, 8, 3001, 3001),
        # causal prefill, as a decoder model runs it
        _attend("causal_B2H8S2048_lse", 2, 8, 8, 2048, 2048, causal=True, lse=True),
        # the largest: a long causal prefill with grouped-query heads, the softmax scale applied in the kernel
        _attend("causal_B1H32HK8S6144", 1, 32, 8, 6144, 6144, causal=True, scaled=True),
        # a short query chunk over a long KV cache, on the KV split (a ragged tail)
        _attend("chunk_B1H8S128_SK16000", 1, 8, 8, 128, 16000, splits=8),
        # a decode step: one query token per sequence of a batch, grouped-query heads, a long KV cache
        _attend("decode_B8H32HK8S1_SK8192", 8, 32, 8, 1, 8192),
        # a whole bf16 attention layer through the MXFP8 path: three quantisers, then the attention
        dict(name="layer_bf16_B2H8S2048", kind="attend_bf16", B=2, H=8, HK=8, S=2048, SK=2048, causal=False, lse=False,
             seq32=False, scaled=False),
        # filling a KV cache: K rows, and V with one scale per 32 keys and column
        dict(name="cache_B4HK8_SK2048_seq32", kind="quantize", B=4, HK=8, SK=2048, seq32=True),
    ]


def _logsize(rng, lo, hi):
    """Spread over the logarithm of [lo, hi]; a third of them multiples of 128, the rest as they fall."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.33:
        n = (n + 127) // 128 * 128
    return max(lo, min(hi, n))


def draw(rng):
    """One more case of the ranges above. What a case may cost is bounded by the largest listed one: by its padded
    (query, key) pairs on whole 256-row query tiles, and by the bytes of its K and V."""
    kind = rng.choice(["prefill", "prefill", "causal", "chunk", "decode", "decode", "attend_bf16", "quantize"])
    while True:
        # the bf16 entry point allocates its scales for as many K heads as Q heads
        group = 1 if kind == "attend_bf16" else rng.choice([1, 1, 2, 4, 8])
        HK = rng.choice([1, 2, 3, 4, 8])
        H = HK * group
        B = rng.choice([1, 1, 2, 3, 4, 6, 8])
        if kind == "quantize":
            SK = _logsize(rng, 64, 16384)
            if B * SK * HK > 8 * 8192 * 8:
                continue
            return dict(kind="quantize", B=B, HK=HK, SK=SK, seq32=rng.random() < 0.5)
        if kind == "decode":
            S, SK = rng.choice([1, 1, 1, 2, 4, 7, 16]), _logsize(rng, 512, 16384)
        elif kind == "chunk":
            S, SK = _logsize(rng, 17, 512), _logsize(rng, 1024, 16384)
        else:
            S = _logsize(rng, 64, 8192)
            SK = S if rng.random() < 0.6 else min(16384, S + _logsize(rng, 16, 4096))
        causal = kind == "causal" or (kind == "attend_bf16" and rng.random() < 0.5)
        pairs = B * H * ((S + 255) // 256 * 256) * SK
        if pairs > 32 * 6144 * 6144 * (1.0 if causal else 0.5) or B * SK * HK > 8 * 8192 * 8:
            continue
        opts = dict(causal=causal, seq32=rng.random() < 0.2, scaled=rng.random() < 0.3, lse=False)
        if kind in ("prefill", "causal", "attend_bf16"):
            # the LSE is an output of the full-sequence kernels, not of the KV split
            opts["lse"] = rng.random() < 0.4 and (causal or ops.select_path(B, H, S, SK)[0] != "kvsplit")
        if kind == "attend_bf16":
            return dict(kind="attend_bf16", B=B, H=H, HK=HK, S=S, SK=SK, **opts)
        if kind in ("chunk", "decode") and SK >= 4096 and rng.random() < 0.3:
            opts["splits"] = rng.choice([4, 8])
            opts["partials"] = rng.choice(["fp16", "fp32"])
        return _attend(None, B, H, HK, S, SK, **opts)


def _generator(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFFFFFFFFFF)
    return g


def _normal(shape, seed, salt):
    return torch.randn(shape, generator=_generator(seed, salt), device="cuda", dtype=torch.float32)


def _source(case, seed):
    """The float tensors behind a case. Q, K and V are N(0, 1) as the repository's generator draws them, K with the
    uneven channels that a trained key projection has (gains of about 0.6 to 1.7)."""
    B, HK, SK = case["B"], case["HK"], case["SK"]
    gain = torch.exp(0.3 * _normal((1, 1, HK, D), seed, 1))
    k = (_normal((B, SK, HK, D), seed, 2) * gain).to(torch.bfloat16)
    v = _normal((B, SK, HK, D), seed, 3).to(torch.bfloat16)
    q = None
    if case["kind"] != "quantize":
        q = _normal((B, case["S"], case["H"], D), seed, 4).to(torch.bfloat16)
    return q, k, v


def _block_scale(amax):
    """E8M0 byte of block maxima: clamp(floor(log2 amax) - 8 + 127, 0, 254)."""
    e = torch.frexp(amax)[1].to(torch.int32) - 1
    return torch.where(amax > 0, (e - 8 + 127).clamp(0, 254), torch.zeros_like(e))


def _e4m3(x):
    return (x + 0.0).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).view(torch.uint8)


def _rows_to_mxfp8(x, mul):
    """Rows [..., 128] -> (e4m3 bytes, E8M0 [..., 4]): one scale per 32 elements of x * mul."""
    xs = (x.to(torch.float32) * mul).unflatten(-1, (4, 32))
    e = _block_scale(xs.abs().amax(-1))
    q = _e4m3(xs * torch.exp2((127 - e).to(torch.float32)).unsqueeze(-1))
    return q.flatten(-2), e.to(torch.uint8)


def _tensor_to_e4m3(x):
    """(e4m3 bytes, descale): one float32 descale amax / 448 per tensor."""
    xf = x.to(torch.float32)
    d = xf.abs().max() / 448.0
    return _e4m3(xf / d), d.reshape(1)


def _seq32_to_mxfp8(x):
    """[B, SK, HK, 128] -> (e4m3 bytes, E8M0 [B, ceil(SK / 32), HK, 128]): one scale per 32 keys and column."""
    B, SK, HK, _ = x.shape
    nb = (SK + 31) // 32
    xf = torch.zeros(B, nb * 32, HK, D, device=x.device)
    xf[:, :SK] = x.to(torch.float32)
    xb = xf.view(B, nb, 32, HK, D)
    e = _block_scale(xb.abs().amax(2))
    q = _e4m3(xb * torch.exp2((127 - e).to(torch.float32)).unsqueeze(2))
    return q.view(B, nb * 32, HK, D)[:, :SK].contiguous(), e.to(torch.uint8)


def _mxfp8_inputs(case, seed):
    """(q, k, v, q scales, k scales, V scale) as plain tensors, without the kernels' padding."""
    q, k, v = _source(case, seed)
    q8, qs = _rows_to_mxfp8(q, 1.0 if case["scaled"] else LOG2E / math.sqrt(D))
    k8, ks = _rows_to_mxfp8(k, 1.0)
    v8, vs = _seq32_to_mxfp8(v) if case["seq32"] else _tensor_to_e4m3(v)
    return q8, k8, v8, qs, ks, vs


def _with_slack(scales, slack):
    """The scales at the front of an allocation with the zeroed slack behind them that the entry point asks for."""
    base = torch.zeros(scales.numel() + slack, dtype=torch.uint8, device=scales.device)
    base[:scales.numel()] = scales.flatten()
    return base[:scales.numel()].view(scales.shape)


def prepare(case, seed):
    B, HK, SK = case["B"], case["HK"], case["SK"]
    if case["kind"] == "quantize":
        _, k, v = _source(case, seed)
        return dict(case=case, k=k, v=v, ks=ops.alloc_scales(B, SK, HK, "cuda"))
    S, H = case["S"], case["H"]
    lse = torch.empty(B, H, S, dtype=torch.float32, device="cuda") if case["lse"] else None
    out = torch.empty(B, S, H, D, dtype=torch.bfloat16, device="cuda")
    if case["kind"] == "attend_bf16":
        q, k, v = _source(case, seed)
        return dict(case=case, q=q, k=k, v=v, out=out, lse=lse)
    q8, k8, v8, qs, ks, vs = _mxfp8_inputs(case, seed)
    qsp, ksp = _with_slack(qs, 2048 * H), _with_slack(ks, 2560 * H)
    if not case["seq32"]:
        d = vs   # at the front of the 4 KiB buffer that the entry point asks for
        vs = torch.zeros(1024, dtype=torch.float32, device="cuda")
        vs[:1] = d
    return dict(case=case, q=q8, k=k8, v=v8, qs=qsp, ks=ksp, vs=vs, out=out, lse=lse)


def run(state):
    c = state["case"]
    if c["kind"] == "quantize":
        k8 = ops.quantize_mxfp8(state["k"], state["ks"])
        if c["seq32"]:
            v8, vs = ops.quantize_v_seq32(state["v"])
        else:
            v8, vs = ops.quantize_v(state["v"])
            vs = vs[:1]   # the descale; the rest of the buffer is padding that the attention requires
        return k8, state["ks"], v8, vs
    if c["kind"] == "attend_bf16":
        ops.fmha_fwd_bf16_via_mxfp8(state["q"], state["k"], state["v"], state["out"], causal=c["causal"], lse=state["lse"],
                                    v_scales="seq32" if c["seq32"] else "tensor", scale_in_kernel=c["scaled"])
        return (state["out"], state["lse"]) if c["lse"] else state["out"]
    ops.fmha_fwd_mxfp8(state["q"], state["k"], state["v"], state["qs"], state["ks"], state["vs"], state["out"],
                       path="kvsplit" if c["splits"] else "auto", splits=c["splits"] or None, lse=state["lse"],
                       causal=c["causal"], partials=c["partials"],
                       softmax_scale=1.0 / math.sqrt(D) if c["scaled"] else None)
    return (state["out"], state["lse"]) if c["lse"] else state["out"]


def work(case):
    B, HK, SK = case["B"], case["HK"], case["SK"]
    nkv = B * SK * HK
    vscale = B * ((SK + 31) // 32) * HK * D if case["seq32"] else 4
    if case["kind"] == "quantize":
        # bf16 K and V in; bytes and scales out
        return {"bytes": 2 * nkv * D * 2 + 2 * nkv * D + nkv * 4 + vscale, "flops": 0}
    S, H = case["S"], case["H"]
    pairs = S * SK
    if case["causal"]:
        # row i sees keys 0 .. i + SK - S; SK >= S in every causal case here
        pairs = S * (SK - S) + S * (S + 1) // 2
    flops = 4 * B * H * pairs * D
    nq = B * S * H
    if case["kind"] == "attend_bf16":
        return {"bytes": (2 * nkv + nq) * D * 2 + nq * D * 2, "flops": flops}
    lse = nq * 4 if case["lse"] else 0
    return {"bytes": nq * (D + 4) + nkv * (2 * D + 4) + vscale + nq * D * 2 + lse, "flops": flops}


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"
    # The path computes the softmax weights in e4m3 (3 mantissa bits, about 2.5 % of each weight) after a
    # piecewise-linear exp2: against float64 the outputs are about 3 % off, and orders that quantise the weights against
    # another running maximum differ by up to 4 % from each other (measured at 2048 keys). The largest difference of one
    # element, over the outputs' root mean square, belongs to a row that few keys decide: 0.43 between two such orders,
    # and 0.62 against float64 under the causal mask, whose first rows see one to a few keys.
    return {"rel": 0.03, "max": 0.9 if case["causal"] else 0.5}


def _attention64(q, k, v, causal, scale, lse):
    """softmax(scale q k^T) v in float64, one head and one block of rows at a time: [B, S, H, D] and [B, H, S]."""
    B, S, H, _ = q.shape
    SK, HK = k.shape[1], k.shape[2]
    out = torch.empty(B, S, H, D, dtype=torch.float64, device=q.device)
    ls = torch.empty(B, H, S, dtype=torch.float64, device=q.device) if lse else None
    keys = torch.arange(SK, device=q.device)
    step = max(1, min(S, (1 << 25) // SK))
    for b in range(B):
        for h in range(H):
            kh, vh = k[b, :, h // (H // HK)].double(), v[b, :, h // (H // HK)].double()
            for r in range(0, S, step):
                s = (q[b, r:r + step, h].double() @ kh.T.contiguous()) * scale
                if causal:
                    rows = torch.arange(r, r + s.shape[0], device=q.device)
                    s.masked_fill_(keys[None] > rows[:, None] + (SK - S), -math.inf)
                m = s.amax(1, keepdim=True)
                p = torch.exp(s - m)
                l = p.sum(1, keepdim=True)
                out[b, r:r + step, h] = (p @ vh) / l
                if lse:
                    ls[b, h, r:r + step] = (m + torch.log(l))[:, 0]
    return (out, ls) if lse else out


def exact(case, seed):
    if case["kind"] == "quantize":
        _, k, v = _source(case, seed)
        k8, ks = _rows_to_mxfp8(k, 1.0)
        v8, vs = _seq32_to_mxfp8(v) if case["seq32"] else _tensor_to_e4m3(v)
        return k8, ks, v8, vs
    if case["kind"] == "attend_bf16":
        q, k, v = _source(case, seed)
        return _attention64(q, k, v, case["causal"], 1.0 / math.sqrt(D), case["lse"])
    q8, k8, v8, qs, ks, vs = _mxfp8_inputs(case, seed)

    def rows(x, e):
        s = torch.exp2(e.to(torch.float64) - 127.0)
        return (x.view(torch.float8_e4m3fn).to(torch.float64).unflatten(-1, (4, 32)) * s.unsqueeze(-1)).flatten(-2)

    v = v8.view(torch.float8_e4m3fn).to(torch.float64)
    if case["seq32"]:
        v = v * torch.exp2(vs.to(torch.float64) - 127.0).repeat_interleave(32, 1)[:, :case["SK"]]
    else:
        v = v * vs.to(torch.float64)
    # the scale folded into Q carries log2(e): softmax2(q k) = softmax(ln 2 q k)
    scale = 1.0 / math.sqrt(D) if case["scaled"] else math.log(2.0)
    return _attention64(rows(q8, qs), rows(k8, ks), v, case["causal"], scale, case["lse"])
