"""The work a server has this package do, as cases that can be timed and checked.

Every case is one call (or one layer's calls) through the public functions of
``tinyserver_amd.kernels``, as the serving loop makes them: the fused decode
step of a small batch, paged decode attention of large batches, the prefill's
norm/RoPE/store and varlen attention, and the batched sampler. Shapes are the
Qwen3 attention shapes (head_dim 128, 8 kv heads, 2, 4 or 8 query heads per kv
head, a vocabulary of 151,936), page sizes the server's default (256), the
benchmark's (16) and the one the model-level validation uses (4, in float32).

``listed`` gives the cases, ``draw`` more of the same ranges; ``prepare``
makes what a program holds before the call, ``run`` makes the call, ``exact``
computes the same outputs in 64 bits with plain torch.
"""

import math
import random

import torch

from tinyserver_amd.kernels import (
    flash_attn_varlen_func,
    paged_attention_forward,
    paged_decode_step,
    qk_norm_rope_store,
    sample_tokens,
)

D = 128
HKV = 8
VOCAB = 151936
EPS = 1e-6
THETA = 1.0e6
DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}

# The costliest listed work, which drawn cases stay under.
MAX_KV_TOKENS = 32 * 32768  # tokens in the paged cache of one decode batch
MAX_PREFILL_PAIRS = 64 * 16384 * 16385 // 2  # (q-head, query, key) pairs of one prefill
MAX_F32_PAIRS = 16 * 8 * 512 * 513 // 2  # the same in float32


def listed():
    return [
        # A few short chats on the smallest model: one layer's decode step
        # (norm, RoPE, K/V store and attention of the new tokens). Launch
        # latency and host work are most of it.
        dict(name="decode_step_0.6b_bs4", kind="decode_step", batch=4, heads=16, lo=16, hi=512, page=16, dtype="bf16",
             lens=1),
        # The server's default settings (at most 8 sequences, 256-token
        # pages) with contexts of a few thousand tokens.
        dict(name="decode_step_1.7b_bs8_p256", kind="decode_step", batch=8, heads=16, lo=128, hi=4096, page=256,
             dtype="bf16", lens=2),
        # The headline: paged decode attention of a busy Qwen3-8B server.
        dict(name="decode_8b_bs64", kind="decode", batch=64, heads=32, lo=512, hi=4096, page=16, dtype="bf16", lens=3),
        # Long-context decode, the largest K/V read.
        dict(name="decode_32b_bs32_32k", kind="decode", batch=32, heads=64, lo=32768, hi=32768, page=16, dtype="bf16",
             lens=4),
        # A checkpoint served in float32 on 4-token pages (what the
        # model-level validation and comparison runs use).
        dict(name="decode_0.6b_f32_p4", kind="decode", batch=8, heads=16, lo=16, hi=1024, page=4, dtype="f32", lens=5),
        # The prefill's norm/RoPE/store of 16 packed prompts.
        dict(name="norm_store_8b_16seq", kind="norm_store", seqs=16, heads=32, lo=128, hi=2048, page=16, dtype="bf16",
             lens=6),
        # The same prompts' varlen causal attention.
        dict(name="prefill_8b_16seq", kind="prefill", seqs=16, heads=32, lo=128, hi=2048, dtype="bf16", lens=6),
        # A full prefill step of a default server: 8 prompts, about 4096
        # tokens, two query heads per kv head.
        dict(name="prefill_1.7b_8seq", kind="prefill", seqs=8, heads=16, lo=64, hi=960, dtype="bf16", lens=8),
        # One long document on the largest model.
        dict(name="prefill_32b_16k", kind="prefill", seqs=1, heads=64, lo=16384, hi=16384, dtype="bf16", lens=9),
        # Prompts in float32 (validation and comparison runs).
        dict(name="prefill_0.6b_f32", kind="prefill", seqs=8, heads=16, lo=32, hi=512, dtype="f32", lens=10),
        # Sampling for 64 sequences with the server's default request
        # (temperature 1, top_p 0.95, no top_k).
        dict(name="sample_bs64_default", kind="sample", batch=64, mix="default", dtype="bf16"),
        # Sampling for 8 sequences whose requests differ: greedy, the
        # default, top-k with top-p, top-p alone.
        dict(name="sample_bs8_mixed", kind="sample", batch=8, mix="mixed", dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode_step", "decode", "decode", "norm_store", "prefill", "prefill", "sample"])
    heads = rng.choice([16, 32, 64])
    lens = rng.randrange(1, 1 << 20)
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16"])
    if kind == "decode_step":
        # Small steps: the glue takes the fused step up to 16384 tiles of 16
        # tokens in the block tables of all 8 kv heads, 32768 tokens.
        batch = _log_int(rng, 1, 16)
        hi = min(_log_int(rng, 64, 8192), 32768 // batch // 256 * 256)
        return dict(kind=kind, batch=batch, heads=heads, lo=max(1, hi // rng.choice([2, 8, 32])), hi=hi,
                    page=rng.choice([16, 256]), dtype=dtype, lens=lens)
    if kind == "decode":
        if rng.random() < 0.3:
            hi = _log_int(rng, 32, 1024)
            return dict(kind=kind, batch=_log_int(rng, 1, 8), heads=16, lo=max(1, hi // 8), hi=hi,
                        page=rng.choice([4, 16]), dtype="f32", lens=lens)
        batch = _log_int(rng, 1, 128)
        hi = min(_log_int(rng, 256, 32768), MAX_KV_TOKENS // batch)
        return dict(kind=kind, batch=batch, heads=heads, lo=max(1, hi // rng.choice([1, 4, 16])), hi=hi,
                    page=rng.choice([16, 256]), dtype=dtype, lens=lens)
    if kind == "norm_store":
        hi = _log_int(rng, 16, 2048)
        return dict(kind=kind, seqs=_log_int(rng, 1, 16), heads=heads, lo=max(1, hi // 8), hi=hi,
                    page=rng.choice([16, 256]), dtype=dtype, lens=lens)
    if kind == "prefill":
        if rng.random() < 0.3:
            seqs = _log_int(rng, 1, 8)
            hi = min(_log_int(rng, 32, 1024), int(math.sqrt(2 * MAX_F32_PAIRS / 16 / seqs)) - 1)
            return dict(kind=kind, seqs=seqs, heads=16, lo=max(1, hi // 8), hi=hi, dtype="f32", lens=lens)
        seqs = _log_int(rng, 1, 32)
        hi = min(_log_int(rng, 32, 16384), int(math.sqrt(2 * MAX_PREFILL_PAIRS / heads / seqs)) - 1)
        return dict(kind=kind, seqs=seqs, heads=heads, lo=max(1, hi // rng.choice([1, 4, 16])), hi=hi, dtype=dtype,
                    lens=lens)
    return dict(kind="sample", batch=_log_int(rng, 1, 64), mix=rng.choice(["default", "mixed", "topk", "greedy"]),
                dtype=dtype, lens=lens)


# ------------------------------------------------------------------ inputs --
def _lengths(case):
    """The case's sequence lengths: fixed by the case, the same for every seed."""
    n = case["batch"] if "batch" in case else case["seqs"]
    r = random.Random(1000003 * case["lens"] + 17 * case["hi"] + n)
    return [r.randint(case["lo"], case["hi"]) for _ in range(n)]


def _randn(gen, *shape, dtype):
    return torch.randn(*shape, generator=gen, device=DEVICE, dtype=torch.float32).to(dtype)


def _pool(gen, pages, page, dtype):
    out = torch.empty(pages, HKV, page, D, device=DEVICE, dtype=dtype)
    step = max(1, (1 << 27) // (HKV * page * D))
    for i in range(0, pages, step):
        n = min(step, pages - i)
        out[i : i + n] = _randn(gen, n, HKV, page, D, dtype=dtype)
    return out


def _tables(gen, lens, page):
    """Shuffled pages of a pool with a tenth of it free, and the zero-padded block tables."""
    need = [-(-n // page) for n in lens]
    pages = math.ceil(sum(need) * 1.1)
    perm = torch.randperm(pages, generator=gen, device=DEVICE).to(torch.int32)
    width = max(need)
    starts = torch.tensor([sum(need[:i]) for i in range(len(need))], device=DEVICE)
    col = torch.arange(width, device=DEVICE)
    used = col[None, :] < torch.tensor(need, device=DEVICE)[:, None]
    idx = (starts[:, None] + col[None, :]).clamp(max=pages - 1)
    return torch.where(used, perm[idx], 0).to(torch.int32).contiguous(), pages


def _cos_sin(positions, dtype):
    inv = 1.0 / (THETA ** (torch.arange(0, D, 2, dtype=torch.float32, device=DEVICE) / D))
    ang = positions.to(DEVICE, torch.float32)[:, None] * inv[None, :]
    emb = torch.cat((ang, ang), dim=-1)
    return emb.cos().to(dtype), emb.sin().to(dtype)


def _norm_weight(gen, dtype):
    return (1.0 + 0.1 * torch.randn(D, generator=gen, device=DEVICE)).to(dtype)


def _cu(lens):
    cu = torch.zeros(len(lens) + 1, dtype=torch.int32)
    cu[1:] = torch.cumsum(torch.tensor(lens), 0).to(torch.int32)
    return cu.to(DEVICE)


def _sampling_rows(mix, batch):
    """(temperature, top_k, top_p) of each row's request."""
    kinds = {"default": [(1.0, 0, 0.95)], "topk": [(0.8, 50, 0.9)], "greedy": [(0.0, 0, 1.0)],
             "mixed": [(0.0, 0, 1.0), (1.0, 0, 0.95), (0.8, 50, 0.9), (0.8, 0, 0.9)]}[mix]
    return [kinds[i % len(kinds)] for i in range(batch)]


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind, dt = case["kind"], DTYPES[case["dtype"]]
    s = {"kind": kind}
    if kind == "sample":
        b = case["batch"]
        x = torch.randn(b, VOCAB, generator=gen, device=DEVICE) * 2.5
        hot = torch.randint(0, VOCAB, (b, 8), generator=gen, device=DEVICE)
        x.scatter_add_(1, hot, torch.rand(b, 8, generator=gen, device=DEVICE) * 12)
        rows = _sampling_rows(case["mix"], b)
        s["logits"] = x.to(dt)
        s["temperature"] = torch.tensor([r[0] for r in rows], device=DEVICE)
        s["top_k"] = torch.tensor([r[1] for r in rows], dtype=torch.int64, device=DEVICE)
        s["top_p"] = torch.tensor([r[2] for r in rows], device=DEVICE)
        s["uniforms"] = torch.rand(b, generator=gen, device=DEVICE)
        return s
    lens, hq = _lengths(case), case["heads"]
    if kind in ("decode", "decode_step"):
        b = len(lens)
        s["tables"], pages = _tables(gen, lens, case["page"])
        s["k_cache"] = _pool(gen, pages, case["page"], dt)
        s["v_cache"] = _pool(gen, pages, case["page"], dt)
        s["page"] = case["page"]
        s["q"] = _randn(gen, b, hq, D, dtype=dt)
        s["seq_lens"] = torch.tensor(lens, dtype=torch.int32, device=DEVICE)
        if kind == "decode_step":
            s["k"] = _randn(gen, b, HKV, D, dtype=dt)
            s["v"] = _randn(gen, b, HKV, D, dtype=dt)
            s["qw"], s["kw"] = _norm_weight(gen, dt), _norm_weight(gen, dt)
            s["cos"], s["sin"] = _cos_sin(s["seq_lens"] - 1, dt)
        return s
    t = sum(lens)
    s["cu"], s["max_len"] = _cu(lens), max(lens)
    s["q"] = _randn(gen, t, hq, D, dtype=dt)
    s["k"] = _randn(gen, t, HKV, D, dtype=dt)
    s["v"] = _randn(gen, t, HKV, D, dtype=dt)
    if kind == "norm_store":
        s["tables"], pages = _tables(gen, lens, case["page"])
        s["k_cache"] = torch.zeros(pages, HKV, case["page"], D, device=DEVICE, dtype=dt)
        s["v_cache"] = torch.zeros_like(s["k_cache"])
        s["qw"], s["kw"] = _norm_weight(gen, dt), _norm_weight(gen, dt)
        s["cos"], s["sin"] = _cos_sin(torch.cat([torch.arange(n) for n in lens]), dt)
    return s


# --------------------------------------------------------------- the calls --
def run(s):
    kind = s["kind"]
    if kind == "decode_step":
        out = paged_decode_step(s["q"], s["k"], s["v"], s["qw"], s["kw"], s["cos"], s["sin"], EPS, s["k_cache"],
                                s["v_cache"], s["tables"], s["seq_lens"])
        return {"out": out, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    if kind == "decode":
        return paged_attention_forward(s["q"], s["k_cache"], s["v_cache"], s["tables"], s["page"], s["seq_lens"])
    if kind == "norm_store":
        q, k = qk_norm_rope_store(s["q"], s["k"], s["v"], s["qw"], s["kw"], s["cos"], s["sin"], EPS, s["k_cache"],
                                  s["v_cache"], s["tables"], s["cu"])
        return {"q": q, "k": k, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    if kind == "prefill":
        return flash_attn_varlen_func(s["q"], s["k"], s["v"], s["cu"], s["cu"], s["max_len"], s["max_len"], True)
    return sample_tokens(s["logits"], s["temperature"], s["top_k"], s["top_p"], s["uniforms"])


def work(case):
    kind = case["kind"]
    eb = 4 if case["dtype"] == "f32" else 2
    if kind == "sample":
        # Logits in, tokens and the requests' settings; one exponential a logit.
        b = case["batch"]
        return {"bytes": b * VOCAB * eb + b * 28, "flops": 2 * b * VOCAB}
    lens, hq = _lengths(case), case["heads"]
    t = sum(lens)
    if kind in ("decode", "decode_step"):
        b = len(lens)
        kv = 2 * t * HKV * D * eb
        tables = 4 * sum(-(-n // case["page"]) for n in lens) + 4 * b
        extra = 0
        if kind == "decode_step":  # new K/V in and into the cache, cos/sin, weights
            extra = (4 * b * HKV * D + 2 * b * D + 2 * D) * eb
            kv -= 2 * b * HKV * D * eb  # the new tokens' cache rows are written, not read
        return {"bytes": kv + 2 * b * hq * D * eb + tables + extra, "flops": 4 * t * hq * D}
    if kind == "norm_store":
        # q, k, v, cos, sin in; rotated q and k and both cache rows out.
        return {"bytes": eb * (t * D * (2 * hq + 5 * HKV) + 2 * t * D + 2 * D) + 4 * sum(-(-n // case["page"])
                                                                                       for n in lens),
                "flops": 10 * t * (hq + HKV) * D}
    pairs = sum(n * (n + 1) // 2 for n in lens)
    return {"bytes": eb * t * D * (2 * hq + 2 * HKV), "flops": 4 * D * hq * pairs}


def tolerance(case):
    """About four times what the calls differ by from 64-bit arithmetic on the same inputs."""
    kind, f16 = case["kind"], case["dtype"] == "f16"
    if kind == "sample":
        return "exact"
    if case["dtype"] == "f32":  # 3e-7 to 6e-7 measured
        return {"rel": 2.5e-6, "max": 1e-4}
    if kind == "norm_store":  # the model's four roundings a value: 3.1e-3 in bf16
        return {"rel": 1.6e-3 if f16 else 1.2e-2, "max": 5e-2}
    if kind == "decode_step":  # those and the output's own: 3.7e-3 in bf16
        return {"rel": 2e-3 if f16 else 1.5e-2, "max": 5e-2}
    return {"rel": 1.2e-3 if f16 else 8e-3, "max": 5e-2}  # 1.7e-3 (decode), 2.0e-3 (prefill) in bf16


# ------------------------------------------------------- the same in 64 bits --
def _norm_rope64(x, w, cos, sin):
    x = x.double()
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()
    rot = torch.cat((-y[..., D // 2 :], y[..., : D // 2]), dim=-1)
    return y * cos.double()[:, None, :] + rot * sin.double()[:, None, :]


def _rows(cache, table, n, page):
    """One sequence's (HKV, n, D) rows of a paged cache, in 64 bits."""
    used = table[: -(-n // page)].long()
    return cache[used].double().transpose(0, 1).reshape(HKV, -1, D)[:, :n].contiguous()


def _decode64(q, k_cache, v_cache, tables, page, lens):
    out = torch.empty(q.shape, dtype=torch.float64, device=DEVICE)
    for i, n in enumerate(lens):
        k, v = _rows(k_cache, tables[i], n, page), _rows(v_cache, tables[i], n, page)
        qi = q[i].double().reshape(HKV, -1, D).transpose(1, 2).contiguous()
        p = torch.softmax(torch.bmm(k, qi) / math.sqrt(D), dim=1).transpose(1, 2).contiguous()
        out[i] = torch.bmm(p, v).reshape(-1, D)
    return out


def _prefill64(q, k, v, lens):
    out = torch.empty(q.shape, dtype=torch.float64, device=DEVICE)
    group, start = q.shape[1] // HKV, 0
    for n in lens:
        for h in range(HKV):
            kt = k[start : start + n, h].double().t().contiguous()
            vh = v[start : start + n, h].double().contiguous()
            for r in range(0, n, 1024):
                m = min(1024, n - r)
                rows = slice(start + r, start + r + m)
                qs = q[rows, h * group : (h + 1) * group].double().transpose(0, 1).reshape(group * m, D).contiguous()
                sc = torch.mm(qs, kt[:, : r + m].contiguous()).reshape(group, m, r + m) / math.sqrt(D)
                late = torch.arange(r + m, device=DEVICE)[None, :] > torch.arange(r, r + m, device=DEVICE)[:, None]
                p = torch.softmax(sc.masked_fill_(late, float("-inf")), dim=-1).reshape(group * m, r + m)
                o = torch.mm(p, vh[: r + m]).reshape(group, m, D)
                out[rows, h * group : (h + 1) * group] = o.transpose(0, 1)
        start += n
    return out


def _sample64(s):
    x = s["logits"].double() / s["temperature"].double().clamp(min=1e-5)[:, None]
    xs, order = torch.sort(x, dim=-1, descending=True, stable=True)
    ranks = torch.arange(VOCAB, device=DEVICE)[None, :]
    keep = torch.where(s["top_k"] > 0, s["top_k"], VOCAB)[:, None]
    probs = torch.softmax(xs.masked_fill(ranks >= keep, float("-inf")), dim=-1)
    cut = (torch.cumsum(probs, -1) - probs) > s["top_p"].double()[:, None]
    cut[:, 0] = False
    cdf = torch.cumsum(probs.masked_fill(cut, 0.0), -1)
    pick = torch.searchsorted(cdf, s["uniforms"].double()[:, None] * cdf[:, -1:]).clamp(max=VOCAB - 1)
    pick = torch.where(s["temperature"][:, None] <= 0, 0, pick)
    return order.gather(-1, pick).squeeze(-1)


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "sample":
        return _sample64(s)
    lens = _lengths(case)
    if kind == "decode":
        return _decode64(s["q"], s["k_cache"], s["v_cache"], s["tables"], case["page"], lens)
    if kind == "prefill":
        return _prefill64(s["q"], s["k"], s["v"], lens)
    q = _norm_rope64(s["q"], s["qw"], s["cos"], s["sin"])
    k = _norm_rope64(s["k"], s["kw"], s["cos"], s["sin"])
    k_cache, v_cache = s["k_cache"].double(), s["v_cache"].double()
    if kind == "decode_step":
        seq = torch.arange(len(lens), device=DEVICE)
        pos = s["seq_lens"].long() - 1
    else:
        seq = torch.cat([torch.full((n,), i) for i, n in enumerate(lens)]).to(DEVICE)
        pos = torch.cat([torch.arange(n) for n in lens]).to(DEVICE)
    block, slot = s["tables"][seq, pos // case["page"]].long(), pos % case["page"]
    k_cache[block, :, slot] = k
    v_cache[block, :, slot] = s["v"].double()
    if kind == "norm_store":
        return {"q": q, "k": k, "k_cache": k_cache, "v_cache": v_cache}
    out = _decode64(q, k_cache, v_cache, s["tables"], case["page"], lens)
    return {"out": out, "k_cache": k_cache, "v_cache": v_cache}
