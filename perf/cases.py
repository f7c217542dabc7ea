"""Performance cases of sparse_attn_sharedkv: what a serving or training
program has the operator do, through its public entry points.

A case is a dict of plain values. ``op`` is the call:

``attn``   one attention forward (``sparse_attn_sharedkv``, out and LSE);
``train``  a forward recorded for autograd and its backward
           (``sparse_attn_sharedkv_autograd``): out and every gradient;
``bwd``    the backward alone, from a forward's out and LSE
           (``sparse_attn_sharedkv_backward``);
``write``  new KV rows into a paged cache (``write_kv_cache``).

The other fields are the shape: ``B`` sequences of ``q_lo .. q_hi`` query
tokens over caches of ``kv_lo .. kv_hi`` rows (a prefill, ``whole``, queries
its whole sequence), drawn from ``lens`` so that the lengths are part of the
case; ``H`` heads, ``D`` channels, window ``win``, top-k ``K``, compressed
ratio ``ratio``, block size ``bs``, row type ``dt``.

Sequence lengths and tables are device tensors, as a serving loop keeps
them, but for the dense compressed scenario (``cfa``), whose slot count
follows the longest sequence and is read from the lengths: host tensors.
Queries, cache rows and output gradients are N(0, 1), the top-k positions of
a token distinct and uniform below its causal threshold, -1 padded, and the
physical blocks of a cache a random permutation.
"""

import math
import random

import torch

from dsv4_amd.api import (sparse_attn_sharedkv, sparse_attn_sharedkv_autograd,
                          sparse_attn_sharedkv_backward)
from dsv4_amd.cache import write_kv_cache

DV = 512
DEV = "cuda"


def _attn(name, op="attn", kind="scfa", B=1, H=64, D=576, K=512, ratio=4, win=128, bs=64, dt="bf16",
          q=(1, 1), kv=(2048, 2048), whole=False, layout="TND", lens=0):
    return {"name": name, "op": op, "kind": kind, "B": B, "H": H, "D": D, "K": K if kind == "scfa" else 0,
            "ratio": ratio, "win": win, "bs": bs, "dt": dt, "q_lo": q[0], "q_hi": q[1], "kv_lo": kv[0],
            "kv_hi": kv[1], "whole": whole, "layout": layout, "lens": lens}


def _write(name, B, per_seq, kv, dt, bs=64, lens=0):
    return {"name": name, "op": "write", "B": B, "q_lo": per_seq[0], "q_hi": per_seq[1], "kv_lo": kv[0],
            "kv_hi": kv[1], "D": 576, "bs": bs, "dt": dt, "whole": False, "lens": lens}


def listed():
    return [
        # one user's decode step with few heads: a call's latency
        _attn("decode_1", B=1, H=16, K=64, kv=(2048, 2048)),
        # a serving batch's decode step over mixed contexts
        _attn("decode_32", B=32, H=64, K=512, kv=(8192, 32768), lens=1),
        # decode with draft tokens: 1 to 4 query tokens a sequence, 128 heads
        _attn("decode_drafts", B=16, H=128, K=1024, q=(1, 4), kv=(1024, 65536), lens=2),
        # long contexts in fp8 cache rows, compressed 128 to 1
        _attn("decode_fp8_128k", B=8, H=128, K=1024, ratio=128, kv=(131072, 131072), dt="fp8"),
        # one prompt of 4096 tokens
        _attn("prefill_4k", B=1, K=512, kv=(4096, 4096), whole=True),
        # a window-only layer over a prompt of 8192 tokens
        _attn("prefill_window_8k", kind="swa", B=1, D=512, bs=128, kv=(8192, 8192), whole=True),
        # a dense compressed layer, 128 to 1, in fp16
        _attn("prefill_dense_8k", kind="cfa", B=1, D=512, ratio=128, bs=128, kv=(8192, 8192), whole=True, dt="fp16"),
        # chunks of four prompts continued over fp8 caches
        _attn("prefill_chunks_fp8", B=4, K=512, q=(200, 900), kv=(4096, 16384), dt="fp8", lens=3),
        # a training step of the layer on one sequence of 4096 tokens
        _attn("train_4k", op="train", B=1, K=512, kv=(4096, 4096), whole=True),
        # the backward of packed sequences of unequal lengths, 128 heads, fp16
        _attn("backward_packed", op="bwd", B=4, H=128, K=512, kv=(150, 1300), whole=True, dt="fp16", lens=4),
        # a prompt chunk of 32768 new rows quantised into an fp8 cache
        _write("write_fp8_32k", B=8, per_seq=(4096, 4096), kv=(4096, 16384), dt="fp8", lens=5),
        # a decode step's new rows, one a sequence
        _write("write_step", B=32, per_seq=(1, 1), kv=(1024, 8192), dt="bf16", lens=6),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    limit = max(work(c)["flops"] for c in listed())
    while True:
        c = _draw(rng)
        del c["name"]
        if work(c)["flops"] <= limit:
            return c


def _draw(rng):
    lens = rng.randrange(1 << 20)
    kind = rng.choices(["scfa", "swa", "cfa"], [6, 2, 2])[0]
    D = rng.choice([576, 576, 512])
    bs = rng.choice([64, 64, 128, 16])
    H = rng.choice([16, 32, 64, 64, 64, 128])
    K = rng.choice([64, 128, 512, 512, 1024, rng.randrange(40, 1100)])
    ratio = rng.choice([4, 4, 8, 128]) if kind == "scfa" else 128
    win = rng.choice([128, 128, 128, 64, rng.randrange(1, 257)])
    what = rng.choices(["decode", "prefill", "chunks", "train", "bwd", "write"], [4, 3, 2, 1, 2, 2])[0]
    dt = rng.choice(["bf16", "bf16", "fp16"])
    if what == "write":
        per = _log(rng, 1, 4096)
        return _write("", B=rng.randrange(1, 33 if per < 1000 else 9), per_seq=(max(1, per // 2), per),
                      kv=(per, per + _log(rng, 64, 16384)), dt=rng.choice(["fp8", "fp8", "bf16", "fp16"]), bs=bs,
                      lens=lens)
    if what in ("decode", "chunks") and rng.random() < 0.4:
        dt, D = "fp8", 576
    shape = dict(kind=kind, H=H, D=D, K=K, ratio=ratio, win=win, bs=bs, dt=dt, lens=lens)
    if what == "decode":
        hi = _log(rng, 300, 65536)
        return _attn("", B=_log(rng, 1, 64), q=(1, rng.choice([1, 1, 2, 4])), kv=(max(4, hi // rng.choice([1, 4, 30])), hi),
                     **shape)
    if what == "chunks":
        hi = _log(rng, 64, 1500)
        kv = _log(rng, 2048, 32768)
        return _attn("", B=rng.randrange(1, 6), q=(max(1, hi // 4), hi), kv=(kv // 2, kv), **shape)
    if what == "prefill":
        hi = _log(rng, 200, 8192)
        B = rng.randrange(1, max(2, min(8, 8192 // hi) + 1))
        lo = max(1, hi // rng.choice([1, 1, 3]))
        return _attn("", B=B, kv=(lo, hi), whole=True, layout="BSND" if lo == hi and rng.random() < 0.3 else "TND", **shape)
    hi = _log(rng, 128, 6000)
    B = rng.randrange(1, max(2, min(8, 6000 // hi) + 1))
    return _attn("", op=what, B=B, kv=(max(1, hi // rng.choice([1, 4])), hi), whole=True, **shape)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _lengths(c):
    r = random.Random(c["lens"])
    kv = [r.randint(c["kv_lo"], c["kv_hi"]) for _ in range(c["B"])]
    q = list(kv) if c["whole"] else [min(r.randint(c["q_lo"], c["q_hi"]), n) for n in kv]
    return q, kv


def _table(lens, bs, gen):
    """Shuffled block table of the sequences, -1 = unused, and the pool's blocks."""
    n = [max(1, -(-x // bs)) for x in lens]
    pool = sum(n) + 3
    perm = torch.randperm(pool, generator=gen, device=DEV).to(torch.int32)
    table = torch.full((len(n), max(n)), -1, dtype=torch.int32, device=DEV)
    at = 0
    for b, m in enumerate(n):
        table[b, :m] = perm[at:at + m]
        at += m
    return table, pool


def _normal(shape, dtype, gen):
    out = torch.empty(shape, dtype=dtype, device=DEV)
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 27):
        part = flat[i:i + (1 << 27)]
        part.copy_(torch.randn(part.numel(), generator=gen, device=DEV))
    return out


def _fp8_rows(blocks, bs, gen):
    """Cache rows of 656 bytes: 512 e4m3 latent values, four scales, 64 bf16
    rope channels, from N(0, 1) channels (amax / 448 a 128-channel group)."""
    rows = torch.empty((blocks * bs, 656), dtype=torch.uint8, device=DEV)
    for i in range(0, rows.shape[0], 1 << 17):
        part = rows[i:i + (1 << 17)]
        n = part.shape[0]
        x = torch.randn((n, 576), generator=gen, device=DEV).to(torch.bfloat16).float()
        lat = x[:, :512].reshape(n, 4, 128)
        scale = lat.abs().amax(-1) / 448.0
        part[:, :512] = (lat / scale[..., None]).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8).reshape(n, 512)
        part[:, 512:528] = scale.contiguous().view(torch.uint8)
        part[:, 528:] = x[:, 512:].to(torch.bfloat16).contiguous().view(torch.uint8)
    return rows.view(blocks, bs, 1, 656)


def _top_k(q_lens, kv_lens, c, gen):
    """Per token: distinct positions, uniform below the causal threshold."""
    K = c["K"]
    parts = []
    for ql, kl in zip(q_lens, kv_lens):
        thr = (torch.arange(ql, device=DEV) + (kl - ql + 1)) // c["ratio"]
        n = max(kl // c["ratio"], 1)
        idx = torch.full((ql, K), -1, dtype=torch.int32, device=DEV)
        step = max(1, (1 << 25) // n)
        for i in range(0, ql, step):
            t = thr[i:i + step, None]
            score = torch.rand((t.shape[0], n), generator=gen, device=DEV)
            score.masked_fill_(torch.arange(n, device=DEV)[None, :] >= t, -1.0)
            best, at = score.topk(min(K, n), dim=1)
            idx[i:i + step, :at.shape[1]] = torch.where(best >= 0, at, -1).to(torch.int32)
        parts.append(idx)
    return torch.cat(parts).unsqueeze(1)


_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp8": torch.bfloat16}


def _inputs(c, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    q_lens, kv_lens = _lengths(c)
    dt = _DT[c["dt"]]
    if c["op"] == "write":
        table, pool = _table(kv_lens, c["bs"], gen)
        n = sum(q_lens)
        row = 656 if c["dt"] == "fp8" else c["D"]
        seq = torch.repeat_interleave(torch.arange(c["B"], device=DEV), torch.tensor(q_lens, device=DEV)).to(torch.int32)
        pos = torch.cat([torch.arange(k - m, k, device=DEV) for m, k in zip(q_lens, kv_lens)]).to(torch.int32)
        return {"kv": _normal((n, c["D"]), dt, gen), "table": table, "seq": seq, "pos": pos,
                "cache": torch.zeros((pool, c["bs"], 1, row), dtype=torch.uint8 if c["dt"] == "fp8" else dt, device=DEV)}
    T = sum(q_lens)
    rows = (lambda n: _fp8_rows(n, c["bs"], gen)) if c["dt"] == "fp8" else (
        lambda n: _normal((n, c["bs"], 1, c["D"]), dt, gen))
    host = c["kind"] == "cfa"
    i32 = dict(dtype=torch.int32, device="cpu" if host else DEV)
    cu = [0]
    for m in q_lens:
        cu.append(cu[-1] + m)
    table, pool = _table(kv_lens, c["bs"], gen)
    kw = {"ori_kv": rows(pool), "ori_block_table": table, "seqused_kv": torch.tensor(kv_lens, **i32),
          "sinks": torch.randn(c["H"], generator=gen, device=DEV), "softmax_scale": 1.0 / math.sqrt(c["D"]),
          "ori_win_left": c["win"] - 1}
    if c["kind"] != "swa":
        kw["cmp_block_table"], pool = _table([k // c["ratio"] for k in kv_lens], c["bs"], gen)
        kw["cmp_kv"] = rows(pool)
        kw["cmp_ratio"] = c["ratio"]
    if c["kind"] == "scfa":
        kw["cmp_sparse_indices"] = _top_k(q_lens, kv_lens, c, gen)
    q = _normal((T, c["H"], c["D"]), dt, gen)
    if c["layout"] == "BSND":
        S = q_lens[0]
        q = q.view(c["B"], S, c["H"], c["D"])
        if "cmp_sparse_indices" in kw:
            kw["cmp_sparse_indices"] = kw["cmp_sparse_indices"].view(c["B"], S, 1, c["K"])
        kw["layout_q"] = "BSND"
    else:
        kw["cu_seqlens_q"] = torch.tensor(cu, **i32)
    s = {"q": q, "kw": kw}
    if c["op"] != "attn":
        s["dout"] = _normal((T, c["H"], DV), dt, gen)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s["op"] = case["op"]
    if case["op"] == "bwd":
        s["out"], s["lse"] = sparse_attn_sharedkv(s["q"], return_softmax_lse=True, **s["kw"])
    if case["op"] == "train":
        kw = dict(s["kw"])
        s["leaf"] = {k: kw.pop(k).requires_grad_(True) for k in ("ori_kv", "cmp_kv", "sinks") if k in kw}
        s["q"].requires_grad_(True)
        s["kw"] = kw
    return s


def run(s):
    op = s["op"]
    if op == "attn":
        out, lse = sparse_attn_sharedkv(s["q"], return_softmax_lse=True, **s["kw"])
        return {"out": out, "lse": lse}
    if op == "bwd":
        dq, d_ori, d_cmp, d_sinks = sparse_attn_sharedkv_backward(s["dout"], s["q"], s["out"], s["lse"], **s["kw"])
        r = {"dq": dq, "d_ori": d_ori, "d_sinks": d_sinks}
        if d_cmp is not None:
            r["d_cmp"] = d_cmp
        return r
    if op == "train":
        out = sparse_attn_sharedkv_autograd(s["q"], **s["leaf"], **s["kw"])
        names = list(s["leaf"])
        grads = torch.autograd.grad(out, [s["q"]] + [s["leaf"][n] for n in names], s["dout"])
        r = {"out": out.detach(), "dq": grads[0]}
        r.update({{"ori_kv": "d_ori", "cmp_kv": "d_cmp", "sinks": "d_sinks"}[n]: g for n, g in zip(names, grads[1:])})
        return r
    write_kv_cache(s["kv"], s["cache"], s["table"], s["seq"], s["pos"])
    return s["cache"]


# ---------------------------------------------------------------------------
# work, tolerance, 64-bit results
# ---------------------------------------------------------------------------

def _pairs(c):
    """(token, key) pairs that count, and the distinct cache rows they name
    at most, window and compressed."""
    q_lens, kv_lens = _lengths(c)
    pairs = rows = 0
    for ql, kl in zip(q_lens, kv_lens):
        sg = torch.arange(kl - ql, kl)
        w = torch.clamp(sg + 1, max=c["win"]).sum().item()
        thr = (sg + 1) // c["ratio"]
        k = 0 if c["kind"] == "swa" else (torch.clamp(thr, max=c["K"]) if c["kind"] == "scfa" else thr).sum().item()
        pairs += w + k
        rows += min(kl, ql + c["win"] - 1)
        rows += 0 if c["kind"] == "swa" else min(kl // c["ratio"], k)
    return int(pairs), int(rows)


def work(case):
    c = case
    if c["op"] == "write":
        n = sum(_lengths(c)[0])
        return {"bytes": n * (c["D"] * 2 + (656 if c["dt"] == "fp8" else c["D"] * 2) + 8), "flops": 0}
    pairs, rows = _pairs(c)
    T, H, D = sum(_lengths(c)[0]), c["H"], c["D"]
    row = 656 if c["dt"] == "fp8" else D * 2
    fwd = T * H * (D * 2 + DV * 2 + 4) + rows * row + T * c["K"] * 4
    bwd = T * H * (D * 2 + 2 * DV * 2 + 4 + D * 2) + rows * (row + D * 4) + T * c["K"] * 4
    f, b = pairs * H * 2 * (D + DV), pairs * H * 2 * (3 * D + 2 * DV)
    return {"attn": {"bytes": fwd, "flops": f}, "bwd": {"bytes": bwd, "flops": b},
            "train": {"bytes": fwd + bwd, "flops": f + b}}[c["op"]]


def tolerance(case):
    if case["op"] == "write":
        return "exact"
    # four times what the outputs and gradients measure against 64 bits: the
    # rounding of P, dS and the outputs, 2.6e-3 in bf16 and 3e-4 in fp16
    return {"rel": 1.2e-3 if case["dt"] == "fp16" else 1e-2}


def _rows64(cache, fp8, flat):
    """fp64 cache rows [..., D] at flat row indices."""
    r = cache.detach().reshape(-1, cache.shape[-1])[flat.reshape(-1)]
    if fp8:
        lat = r[:, :512].contiguous().view(torch.float8_e4m3fn).double().view(-1, 4, 128)
        scale = r[:, 512:528].contiguous().view(torch.float32).double()
        rope = r[:, 528:].contiguous().view(torch.bfloat16).double()
        r = torch.cat([(lat * scale[..., None]).view(-1, 512), rope], 1)
    return r.double().view(*flat.shape, -1)


def exact(case, seed):
    c = case
    if c["op"] == "write":
        return None
    s = _inputs(c, seed)
    kw, q = s["kw"], s["q"]
    lead = q.shape[:-2]
    T, H, D = sum(_lengths(c)[0]), c["H"], c["D"]
    fp8, bs, dev = c["dt"] == "fp8", c["bs"], DEV
    q = q.reshape(T, H, D)
    dout = s.get("dout")
    q_lens, kv_lens = _lengths(c)
    out = torch.empty((T, H, DV), dtype=torch.float64, device=dev)
    lse = torch.empty((T, H), dtype=torch.float64, device=dev)
    has_cmp = c["kind"] != "swa"
    dq = torch.zeros((T, H, D), dtype=torch.float64, device=dev) if dout is not None else None
    d_ori = torch.zeros((kw["ori_kv"].numel() // D, D), dtype=torch.float64, device=dev) if dout is not None else None
    d_cmp = torch.zeros((kw["cmp_kv"].numel() // D, D), dtype=torch.float64, device=dev) if dout is not None and has_cmp else None
    d_sinks = torch.zeros(H, dtype=torch.float64, device=dev)
    sinks, scale = kw["sinks"].double(), kw["softmax_scale"]
    t0 = 0
    for b, (ql, kl) in enumerate(zip(q_lens, kv_lens)):
        J = c["win"] + (c["K"] if c["kind"] == "scfa" else kl // c["ratio"] if has_cmp else 0)
        step = max(1, (1 << 25) // (J * D))
        for i in range(0, ql, step):
            m = min(step, ql - i)
            sg = torch.arange(i, i + m, device=dev) + (kl - ql)
            pos = sg[:, None] - torch.arange(c["win"], device=dev)[None, :]
            ok = pos >= 0
            pos = pos.clamp(min=0)
            flat = kw["ori_block_table"][b].long()[pos // bs] * bs + pos % bs
            keys, valid = [_rows64(kw["ori_kv"], fp8, flat.masked_fill(~ok, 0))], [ok]
            if has_cmp:
                n = J - c["win"]
                at = (kw["cmp_sparse_indices"].reshape(T, -1)[t0 + i:t0 + i + m].long() if c["kind"] == "scfa"
                      else torch.arange(n, device=dev)[None, :].expand(m, n))
                okc = (at >= 0) & (at < ((sg + 1) // c["ratio"])[:, None])
                at = at.masked_fill(~okc, 0)
                flat_c = (kw["cmp_block_table"][b].long()[at // bs] * bs + at % bs).masked_fill(~okc, 0)
                keys.append(_rows64(kw["cmp_kv"], fp8, flat_c))
                valid.append(okc)
            k, v = torch.cat(keys, 1), torch.cat(valid, 1)[:, None, :]
            qq = q.detach()[t0 + i:t0 + i + m].double()
            x = torch.matmul(qq, k.transpose(1, 2).contiguous()) * scale
            x = x.masked_fill(~v, -math.inf)
            l = torch.logsumexp(torch.cat([x, sinks.view(1, H, 1).expand(m, H, 1)], 2), 2)
            p = torch.exp(x - l[..., None])
            o = torch.matmul(p, k[..., :DV].contiguous())
            sl = slice(t0 + i, t0 + i + m)
            out[sl], lse[sl] = o, l
            if dout is None:
                continue
            g = dout[sl].double()
            delta = (g * o).sum(-1)
            ds = p * (torch.matmul(g, k[..., :DV].transpose(1, 2).contiguous()) - delta[..., None]) * scale
            dq[sl] = torch.matmul(ds, k)
            dk = torch.matmul(ds.transpose(1, 2).contiguous(), qq)
            dk[..., :DV] += torch.matmul(p.transpose(1, 2).contiguous(), g)
            d_sinks -= (torch.exp(sinks - l) * delta).sum(0)
            w = c["win"]
            d_ori.index_add_(0, flat[ok], dk[:, :w][ok])
            if has_cmp:
                d_cmp.index_add_(0, flat_c[okc], dk[:, w:][okc])
        t0 += ql
    if c["op"] == "attn":
        return {"out": out.view(*lead, H, DV), "lse": lse.view(*lead, H)}
    r = {"dq": dq, "d_ori": d_ori.view(kw["ori_kv"].shape), "d_sinks": d_sinks}
    if has_cmp:
        r["d_cmp"] = d_cmp.view(kw["cmp_kv"].shape)
    if c["op"] == "train":
        r["out"] = out
    return r
