"""Performance cases of the MLA decode library: what a serving program has it do.

A case is one call (or one serving step) through the public entry points of
``mlc_decode_amd`` and ``mla_decode``, described by plain values:

  kind      "paged"     ``flash_mla_with_kvcache`` with the schedule in hand (a layer of a step)
            "auto"      ``mla_decode_with_kvcache``: schedules and decodes
            "sparse"    ``flash_mla_with_kvcache(indices=...)``: top-k tokens per sequence
            "absorbed"  ``mla_decode_absorbed``: decode and the per-head value projection
            "legacy"    a contiguous-cache kernel object called as kernel(q, q_pe, kv, k_pe, out)
            "step"      ``kv_append``, ``get_mla_metadata``, ``flash_mla_with_kvcache``
            "append"    ``kv_append`` of a block of new tokens per sequence
            "quantize"  ``quantize_kv_cache`` of a whole cache
  batch, heads, s_q     sequences, query heads, query tokens per sequence
  lo, hi                cached tokens per sequence, uniform in [lo, hi] (or three groups: "skew")
  cache     "native" (the query dtype) or "fp8" (e4m3 codes with power-of-two scales)
  dtype     "bf16" or "f16"
  splits    0 = the balanced schedule, n = every sequence cut into n page ranges
  topk, n_new           keys per sequence (sparse); new tokens per sequence (step, append)

The lengths of a case are fixed by its values, so that its work is known; page order, queries,
cache contents, index lists and weights come from the seed.  Values are N(0, sigma^2), as in
the repository's benchmark protocol.
"""
from __future__ import annotations

import random

import torch

import mla_decode
import mlc_decode_amd as M

PAGE, D_QK, D_V, D_ROPE, D_OUT = 64, 576, 512, 64, 128
_DT = {"bf16": torch.bfloat16, "f16": torch.float16}
_BASE = dict(kind="paged", batch=1, heads=16, s_q=1, lo=1024, hi=1024, skew=False, cache="native", dtype="bf16",
             sigma=1.0, splits=0, topk=0, n_new=0)


def _case(name, **kw):
    return dict(_BASE, name=name, **kw)


def listed():
    return [
        # the smallest call: one short conversation on one tensor-parallel rank; launches and latency count
        _case("auto_b1_h16_l1024", kind="auto"),
        # the headline: all 128 heads of a token on one GPU, 64 sequences of 4096 tokens
        _case("paged_b64_h128_l4096", batch=64, heads=128, lo=4096, hi=4096),
        # one of eight tensor-parallel ranks, a ragged batch: bound by the cache's bytes
        _case("paged_b128_h16_ragged", batch=128, heads=16, lo=256, hi=8192),
        # long contexts, two query tokens (multi-token prediction), all heads: the largest case
        _case("paged_b32_s2_h128_l16384", batch=32, s_q=2, heads=128, lo=16384, hi=16384, splits=8),
        # a skewed batch in fp16: one long, some medium and many tiny sequences
        _case("paged_b132_h64_f16_skew", batch=132, heads=64, dtype="f16", sigma=0.5, skew=True, lo=1, hi=16384),
        # two query tokens on a tensor-parallel rank, ragged: 32 query rows
        _case("paged_b64_s2_h16_ragged", batch=64, s_q=2, heads=16, lo=256, hi=8192),
        # the headline's shape over the fp8 cache
        _case("fp8_b64_h128_l4096", batch=64, heads=128, lo=4096, hi=4096, cache="fp8"),
        # sparse attention: the top 2048 tokens of 8192-token contexts, all heads
        _case("sparse_b64_h128_top2048", kind="sparse", batch=64, heads=128, lo=8192, hi=8192, topk=2048),
        # an attention layer's decode with the value projection, ragged, all heads
        _case("absorbed_b32_h128_ragged", kind="absorbed", batch=32, heads=128, lo=512, hi=8192),
        # the contiguous-cache kernel call at batch 1 and a long context, fp16
        _case("legacy_b1_h16_f16_l32768", kind="legacy", heads=16, dtype="f16", sigma=0.1, lo=32768, hi=32768),
        # a whole serving step on a tensor-parallel rank: append a token, schedule, decode (fp8 cache)
        _case("step_fp8_b128_h16_ragged", kind="step", batch=128, heads=16, lo=256, hi=8192, cache="fp8", n_new=1),
        # a prompt's tokens written to the fp8 cache, 64 per sequence and call
        _case("append_fp8_b32_n64", kind="append", batch=32, lo=1, hi=4096, cache="fp8", n_new=64),
    ]


def _log_int(rng, lo, hi):
    """An integer in [lo, hi], uniform over its logarithm."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    """One more case of the ranges above: sizes log-uniform, odd and ragged ones among them."""
    top = listed()[3]
    most = work(top)
    while True:
        kind = rng.choice(("paged", "paged", "paged", "paged", "auto", "sparse", "absorbed", "legacy", "step", "append", "quantize"))
        c = dict(_BASE, kind=kind, batch=_log_int(rng, 1, 256))
        c["heads"] = rng.choice((8, 16, 16, 24, 32, 40, 64, 96, 128, 128))
        c["cache"] = rng.choice(("native", "native", "fp8")) if kind != "legacy" else "native"
        c["dtype"] = rng.choice(("bf16", "bf16", "f16")) if c["cache"] == "native" else "bf16"
        c["sigma"] = rng.choice((1.0, 0.5))
        hi = _log_int(rng, 64, 32768)
        c["lo"], c["hi"] = (hi, hi) if rng.random() < 0.3 else (max(1, hi // rng.choice((2, 8, 32))), hi)
        if kind in ("paged", "auto", "absorbed", "step"):
            c["s_q"] = rng.choice((1, 1, 1, 2, 2, 3, 4))
        if kind in ("paged", "auto"):
            c["splits"] = rng.choice((0, 0, 0, 0, _log_int(rng, 1, 12)))
        if kind == "sparse":
            c["topk"] = _log_int(rng, 64, 2048)
            c["lo"] = c["hi"] = max(c["hi"], c["topk"])
        if kind == "legacy":
            c["batch"], c["lo"], c["sigma"] = _log_int(rng, 1, 16), c["hi"], 0.1
        if kind == "step":
            c["n_new"] = c["s_q"]
        if kind == "append":
            c["n_new"] = _log_int(rng, 1, 64)
        if kind == "quantize":
            c.update(heads=0, batch=1, dtype="bf16", cache="fp8", lo=c["hi"] * 64, hi=c["hi"] * 64)  # up to 2 M tokens
        w, tokens = work(c), sum(_cached(c))
        if w["bytes"] <= most["bytes"] and w["flops"] <= most["flops"] and tokens <= 1 << 20 and c["batch"] * c["s_q"] * c["heads"] <= 1 << 14:
            return c


# ---------------------------------------------------------------------------------------
# sizes
# ---------------------------------------------------------------------------------------
def _cached(c):
    """Cached tokens of each sequence before the call."""
    r = random.Random("%d %d %d" % (c["batch"], c["lo"], c["hi"]))
    if c["skew"]:
        return [16384] + [r.randint(2048, 8192) for _ in range(31)] + [r.randint(1, 128) for _ in range(c["batch"] - 32)]
    return [r.randint(c["lo"], c["hi"]) for _ in range(c["batch"])]


def work(c):
    """Each input read once, each output written once; QK and PV of every visible (row, key) pair."""
    B, rows, e = c["batch"], c["batch"] * c["s_q"] * c["heads"], 2
    tok = 656 if c["cache"] == "fp8" else D_QK * e
    if c["kind"] == "quantize":
        return {"bytes": c["hi"] * (D_QK * e + 656), "flops": 0}
    if c["kind"] == "append":
        return {"bytes": B * c["n_new"] * (D_QK * e + tok), "flops": 0}
    lens = [c["topk"]] * B if c["kind"] == "sparse" else [n + c["n_new"] for n in _cached(c)]
    causal = c["s_q"] > 1
    seen = sum(max(0, n - (i if causal else 0)) for n in lens for i in range(c["s_q"])) * c["heads"]
    b = sum(lens) * tok + rows * D_QK * e + rows * (D_OUT if c["kind"] == "absorbed" else D_V) * e + rows * 4
    f = 2 * seen * (D_QK + D_V)
    if c["kind"] == "sparse":
        b += 4 * sum(lens)
    if c["kind"] == "absorbed":
        b, f = b + c["heads"] * D_V * D_OUT * e, f + 2 * rows * D_V * D_OUT
    if c["kind"] == "step":
        b += B * c["n_new"] * (D_QK * e + tok)
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------
def _pages(tokens):
    return (tokens + PAGE - 1) // PAGE


def _fp8(kv):
    """bf16 rows [..., 576] -> (codes [..., 512] uint8, scales [..., 4] fp32, rope [..., 64]): the
    scale of a 128-dim block is the smallest power of two s with amax <= 448 s (1 for zeros)."""
    x = kv[..., :D_V].unflatten(-1, (4, 128)).float()
    a = x.abs().amax(-1)
    e = torch.ceil(torch.log2(a.double() / 448)).clamp(-126, 127)
    e = torch.where(a.double() > 448 * torch.exp2(e), e + 1, e)
    e = torch.where(a.double() <= 448 * torch.exp2(e - 1), e - 1, e).clamp(-126, 127)
    s = torch.where(a == 0, torch.ones_like(a), torch.exp2(e).float())
    codes = (x / s[..., None]).to(torch.float8_e4m3fn).view(torch.uint8).flatten(-2)
    return codes, s, kv[..., D_V:].contiguous()


def _fp8_pool(kv):
    """The fp8 cache (latent, scale, rope) of bf16 pages [n, 64, 576], some pages at a time."""
    parts = [_fp8(p) for p in kv.split(1024)]
    latent, scale, rope = (torch.cat([p[i] for p in parts]) for i in range(3))
    return latent, scale.transpose(1, 2).contiguous(), rope


def _inputs(c, seed):
    """Everything on the GPU, from the seed alone (plain tensors, nothing of the library)."""
    g = torch.Generator("cuda").manual_seed(seed)
    dt, B, H, S = _DT[c["dtype"]], c["batch"], c["heads"], c["s_q"]
    randn = lambda *shape: torch.randn(*shape, generator=g, dtype=torch.bfloat16 if dt == torch.bfloat16 else dt, device="cuda") * c["sigma"]  # noqa: E731
    x = {}
    if c["kind"] == "quantize":
        x["kv"] = randn(_pages(c["hi"]), PAGE, 1, D_QK)
        return x
    lens = _cached(c)
    x["lens"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
    if c["kind"] == "legacy":
        x["q"], x["q_pe"] = randn(B, H, D_V), randn(B, H, D_ROPE)
        x["kv"], x["k_pe"] = randn(B, c["hi"], 1, D_V), randn(B, c["hi"], 1, D_ROPE)
        return x
    pages = [_pages(n + c["n_new"]) for n in lens]
    ids = torch.randperm(sum(pages), generator=g, device="cuda").to(torch.int32)
    x["table"] = torch.zeros(B, max(pages), dtype=torch.int32, device="cuda")
    row, col = [], []
    for b, n in enumerate(pages):
        row += [b] * n
        col += range(n)
    x["table"][torch.tensor(row, device="cuda"), torch.tensor(col, device="cuda")] = ids
    x["kv"] = randn(sum(pages), PAGE, 1, D_QK)
    if c["kind"] != "append":
        x["q"] = randn(B, S, H, D_QK)
    if c["n_new"]:
        x["kv_new"] = randn(B, c["n_new"], D_QK)
    if c["cache"] == "fp8":
        x["latent"], x["scale"], x["rope"] = _fp8_pool(x.pop("kv").squeeze(2))
    if c["kind"] == "sparse":
        # a random subset of each sequence's tokens, in no order, as pool token ids
        pos = torch.rand(B, c["hi"], generator=g, device="cuda").topk(c["topk"], dim=1).indices
        page = torch.gather(x["table"].long(), 1, pos // PAGE)
        x["indices"] = (page * PAGE + pos % PAGE).to(torch.int32).unsqueeze(1)
    if c["kind"] == "absorbed":
        x["w_uv"] = (torch.randn(H, D_V, D_OUT, generator=g, device="cuda") * D_V ** -0.5).to(dt)
    return x


def prepare(c, seed):
    """The inputs, and what a program has ready before the call: the cache, the step's schedule (shared
    by all layers), the weight in the library's layout, the kernel object of a shape."""
    x = _inputs(c, seed)
    st = {"case": c, "x": x, "scale": D_QK ** -0.5}
    if c["kind"] == "quantize":
        return st
    if c["kind"] == "legacy":
        st["kernel"] = mla_decode.build_kernel_from_config(c["batch"], c["heads"], 1, c["hi"], D_V, D_ROPE, {"num_split": None})
        st["out"] = torch.empty_like(x["q"])
        return st
    st["cache"] = M.Fp8KVCache(x["latent"], x["scale"], x["rope"]) if c["cache"] == "fp8" else x["kv"]
    rows = c["s_q"] * c["heads"]
    if c["kind"] in ("paged", "absorbed"):
        st["sched"] = M.get_mla_metadata(x["lens"], rows, 1, forced_splits=c["splits"])
    elif c["kind"] == "sparse":
        st["sched"] = M.get_mla_metadata(x["lens"], rows, 1, topk=c["topk"])
    if c["kind"] == "absorbed":
        st["w"] = M.prepare_w_uv(x["w_uv"])
    return st


def run(st):
    c, x, scale = st["case"], st["x"], st["scale"]
    kind, causal = c["kind"], c["s_q"] > 1
    if kind == "quantize":
        return tuple(M.quantize_kv_cache(x["kv"]))
    if kind == "legacy":
        st["kernel"](x["q"], x["q_pe"], x["kv"], x["k_pe"], st["out"])
        return st["out"]
    cache = st["cache"]
    if kind == "paged":
        return M.flash_mla_with_kvcache(x["q"], cache, x["table"], x["lens"], D_V, *st["sched"], softmax_scale=scale, causal=causal)
    if kind == "auto":
        return M.mla_decode_with_kvcache(x["q"], cache, x["table"], x["lens"], num_splits=c["splits"] or None, sm_scale=scale, causal=causal)
    if kind == "sparse":
        return M.flash_mla_with_kvcache(x["q"], cache, None, None, D_V, *st["sched"], softmax_scale=scale, indices=x["indices"])
    if kind == "absorbed":
        return M.mla_decode_absorbed(x["q"], cache, x["table"], x["lens"], *st["sched"], st["w"], softmax_scale=scale, causal=causal)
    # the accepted lengths of the last step: append advances them in place
    lens = x["lens"].clone()
    M.kv_append(x["kv_new"], cache, x["table"], lens)
    written = tuple(cache) if c["cache"] == "fp8" else (cache,)
    if kind == "append":
        return written + (lens,)
    sched, splits = M.get_mla_metadata(lens, c["s_q"] * c["heads"], 1)
    out, lse = M.flash_mla_with_kvcache(x["q"], cache, x["table"], lens, D_V, sched, splits, softmax_scale=scale, causal=causal)
    return out, lse, lens, written


# ---------------------------------------------------------------------------------------
# comparison
# ---------------------------------------------------------------------------------------
def tolerance(c):
    """Appends and conversions are bytes.  A decode's output is rounded to 16 bits and so are its
    softmax weights before the second product."""
    if c["kind"] in ("append", "quantize"):
        return "exact"
    return {"rel": 1e-2, "max": 0.1} if c["dtype"] == "bf16" else {"rel": 1.5e-3, "max": 0.015}


def _attend(q, k, visible, scale):
    """q [S, H, 576], k [L, 576] in 64 bits, visible [S] keys per query -> out [S, H, 512], lse [H, S]."""
    S, H, _ = q.shape
    s = (q.reshape(S * H, D_QK) @ k.T).mul_(scale).reshape(S, H, -1)
    at = torch.arange(k.shape[0], device=k.device)
    for i, n in enumerate(visible):
        s[i].masked_fill_(at >= n, float("-inf"))
    lse = torch.logsumexp(s, -1)
    p = torch.exp(s - lse[..., None])
    p = torch.nan_to_num(p, nan=0.0)  # rows without a visible key
    o = (p.reshape(S * H, -1) @ k[:, :D_V]).reshape(S, H, D_V)
    return o, lse.T


def exact(c, seed):
    """What run() returns, in 64 bits and plain torch (bytes that are only moved: None)."""
    x = _inputs(c, seed)
    scale, kind = D_QK ** -0.5, c["kind"]
    if kind == "quantize":
        _, s, rope = _fp8_pool(x["kv"].squeeze(2))
        return None, s.double(), rope.double()
    if kind == "legacy":
        rows = [_attend(torch.cat([x["q"][b], x["q_pe"][b]], -1).double()[None],
                        torch.cat([x["kv"][b, :, 0], x["k_pe"][b, :, 0]], -1).double(), [c["hi"]], scale)[0][0] for b in range(c["batch"])]
        return torch.stack(rows)
    lens, written = _cached(c), None
    if c["n_new"]:
        pos = x["lens"].long()[:, None] + torch.arange(c["n_new"], device="cuda")
        page, row = torch.gather(x["table"].long(), 1, pos // PAGE), pos % PAGE
        if c["cache"] == "fp8":
            codes, s, rope = _fp8(x["kv_new"])
            x["latent"][page, row], x["rope"][page, row] = codes, rope
            x["scale"].transpose(1, 2)[page, row] = s
            written = (None, x["scale"].double(), x["rope"].double())
        else:
            x["kv"][page, row, 0] = x["kv_new"]
            written = (None,)
        lens = [n + c["n_new"] for n in lens]
        if kind == "append":
            return written + (None,)

    def keys(page, row):  # pool rows in 64 bits
        if c["cache"] == "fp8":
            v = x["latent"][page, row].view(torch.float8_e4m3fn).double().unflatten(-1, (4, 128))
            v = v * x["scale"].transpose(1, 2)[page, row].double()[..., None]
            return torch.cat([v.flatten(-2), x["rope"][page, row].double()], -1)
        return x["kv"][page, row, 0].double()

    outs, lses = [], []
    for b in range(c["batch"]):
        if kind == "sparse":
            i = x["indices"][b, 0].long()
            k, n = keys(i // PAGE, i % PAGE), c["topk"]
        else:
            t = torch.arange(lens[b], device="cuda")
            k, n = keys(x["table"][b].long()[t // PAGE], t % PAGE), lens[b]
        visible = [n - (c["s_q"] - 1 - i if c["s_q"] > 1 else 0) for i in range(c["s_q"])]
        o, lse = _attend(x["q"][b].double(), k, visible, scale)
        if kind == "absorbed":
            o = torch.stack([o[:, h] @ x["w_uv"][h].double() for h in range(c["heads"])], 1)
        outs.append(o)
        lses.append(lse)
    out, lse = torch.stack(outs), torch.stack(lses)
    return (out, lse, None, (None,) * len(written)) if kind == "step" else (out, lse)
