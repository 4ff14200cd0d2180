"""Performance cases of the paged-attention library: what an engine asks of
libvcpp_attn.so through its binding (vllm-cpp_amd/pyvcpp.py), from one short
sequence to whole prefill batches.

A case is a dict of plain values; `kind` names the entry points it calls:

  decode        vcpp_paged_decode, one query token per sequence
  decode_step   a decode step's layers (vcpp_write_kv of the new tokens, then
                vcpp_paged_decode) captured in a HIP graph and replayed
  prefill       vcpp_paged_prefill, chunks of new tokens on paged prefixes
  prefill_split vcpp_paged_prefill_split, few chunks on long prefixes
  mixed         vcpp_paged_mixed_step, decodes and prefill chunks in one step
  token_prep    vcpp_qk_norm_rope on q and k, then vcpp_write_kv of k and v
  dense         flash_attention_cuda, contiguous keys

Sequence and chunk lengths are drawn uniformly from the case's bounds by its
`lens` seed, so that a case is the same work whatever its inputs hold.
"""
import ctypes
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "vllm-cpp_amd"))
import pyvcpp  # noqa: E402

KV = {"f32": pyvcpp.KV_F32, "f16": pyvcpp.KV_F16, "i8": pyvcpp.KV_I8, "fp8": pyvcpp.KV_FP8}
ESIZE = {"f32": 4, "f16": 2, "i8": 1, "fp8": 1}
DEV = "cuda:0"
LAYERS = 4  # layers of a captured decode step


def listed():
    return [
        # One chat with a short history on an fp32 cache, the precision of the
        # CPU engine: the smallest call, bound by launches and latency.
        dict(name="decode_f32_single", kind="decode", kv="f32", seqs=1, ctx_min=512, ctx_max=512,
             heads=64, kv_heads=8, dim=80, block=16, lens=1),
        # A serving step of a few interactive requests, replayed as a graph
        # the way a token loop does: each layer writes its new K/V, then attends.
        dict(name="decode_step_graph", kind="decode_step", kv="f16", seqs=3, ctx_min=40, ctx_max=1200,
             heads=32, kv_heads=8, dim=128, block=16, lens=2),
        # One user on a long document: a single sequence has to fill the GPU.
        dict(name="decode_f16_one_long", kind="decode", kv="f16", seqs=1, ctx_min=32768, ctx_max=32768,
             heads=64, kv_heads=8, dim=80, block=16, lens=3),
        # A loaded server's ragged decode batch (the headline benchmark's sizes).
        dict(name="decode_f16_batch", kind="decode", kv="f16", seqs=64, ctx_min=128, ctx_max=4096,
             heads=64, kv_heads=8, dim=80, block=16, lens=2024),
        # The same kind of batch on byte pages, for a model of 7 query heads
        # to a kv head with wide heads, and larger pages.
        dict(name="decode_fp8_batch", kind="decode", kv="fp8", seqs=40, ctx_min=100, ctx_max=5000,
             heads=28, kv_heads=4, dim=128, block=32, lens=5),
        # Chunked prefill at full load: long chunks on cached prefixes.
        dict(name="prefill_f16_chunks", kind="prefill", kv="f16", chunks=8, new_min=2048, new_max=2048,
             prefix_min=1024, prefix_max=1024, heads=64, kv_heads=8, dim=80, block=16, lens=6),
        # Fresh prompts of ordinary, uneven lengths admitted together.
        dict(name="prefill_f16_prompts", kind="prefill", kv="f16", chunks=6, new_min=9, new_max=700,
             prefix_min=0, prefix_max=100, heads=32, kv_heads=8, dim=128, block=16, lens=7),
        # One chunk of a very long request.
        dict(name="prefill_split_long", kind="prefill_split", kv="f16", chunks=1, new_min=512, new_max=512,
             prefix_min=32768, prefix_max=32768, heads=64, kv_heads=8, dim=80, block=16, lens=8),
        # Follow-up turns: short new messages on cached conversations.
        dict(name="prefill_split_suffix", kind="prefill_split", kv="f16", chunks=3, new_min=11, new_max=70,
             prefix_min=6000, prefix_max=9000, heads=32, kv_heads=8, dim=128, block=16, lens=9),
        # A full scheduler step on a quantised cache: many long decodes with a
        # few prefill chunks.
        dict(name="mixed_step_i8", kind="mixed", kv="i8", seqs=128, ctx_min=1024, ctx_max=8192,
             chunks=4, new_min=512, new_max=512, prefix_min=1024, prefix_max=1024,
             heads=64, kv_heads=8, dim=80, block=16, lens=10),
        # The work in front of a prefill's attention: q/k norm and rotation,
        # then the new K/V into their pages.
        dict(name="token_prep_f16", kind="token_prep", kv="f16", tokens=16384, heads=64, kv_heads=8,
             dim=80, block=16, lens=11),
        # The contiguous-cache slot, a small batch of requests.
        dict(name="dense_small_batch", kind="dense", kv="f32", batch=2, kv_len=2048, heads=32, dim=128, q_len=1),
    ]


# (query heads, kv heads): group sizes 1 to 8, 2 to 32 kv heads
HEADS = [(64, 8), (32, 8), (28, 4), (16, 8), (32, 4), (12, 2), (16, 16), (24, 8)]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges: any kind, page type, head
    shape and page size, batch sizes and lengths spread over their logarithm."""
    limit = _cost(listed()[5])
    while True:
        kind = rng.choice(["decode", "decode", "decode", "decode_step", "prefill", "prefill", "prefill_split",
                           "prefill_split", "mixed", "token_prep", "dense"])
        heads, kv_heads = rng.choice(HEADS)
        case = dict(kind=kind, heads=heads, kv_heads=kv_heads, dim=rng.choice([64, 80, 80, 128, 128]),
                    block=rng.choice([16, 16, 32]), lens=rng.randrange(1 << 20))
        if kind in ("decode", "decode_step", "token_prep"):
            case["kv"] = rng.choice(["f32", "f16", "f16", "i8", "fp8"])
        else:
            case["kv"] = rng.choice(["f16", "f16", "i8", "fp8"])
        if kind in ("decode", "decode_step", "mixed"):
            top = {"decode": 128, "decode_step": 16, "mixed": 128}[kind]
            case["seqs"] = _log_int(rng, 1, top)
            hi = _log_int(rng, 64, 32768 if case["seqs"] <= 16 else 8192)
            case["ctx_max"] = hi
            case["ctx_min"] = max(1, int(hi * rng.uniform(0.02, 1.0)))
        if kind in ("prefill", "prefill_split", "mixed"):
            case["chunks"] = rng.randint(1, 3) if kind == "prefill_split" else _log_int(rng, 1, 8)
            hi = _log_int(rng, 8, 2048 if kind == "prefill" else 512)
            case["new_max"] = hi
            case["new_min"] = max(1, int(hi * rng.uniform(0.1, 1.0)))
            hi = _log_int(rng, 2048, 32768) if kind == "prefill_split" else rng.choice([0, _log_int(rng, 16, 4096)])
            case["prefix_max"] = hi
            case["prefix_min"] = int(hi * rng.uniform(0.5, 1.0))
        if kind == "token_prep":
            case["tokens"] = _log_int(rng, 1, 16384)
        if kind == "dense":
            case = dict(kind=kind, kv="f32", batch=_log_int(rng, 1, 16), kv_len=_log_int(rng, 64, 8192), heads=heads,
                        dim=case["dim"], q_len=rng.choice([1, 1, 3]))
        if _cost(case) <= limit:
            return case


def _lens(case):
    """(context lengths, chunk lengths, prefix lengths) of a case."""
    r = random.Random(case.get("lens", 0))
    ctx = [r.randint(case["ctx_min"], case["ctx_max"]) for _ in range(case.get("seqs", 0))]
    new = [r.randint(case["new_min"], case["new_max"]) for _ in range(case.get("chunks", 0))]
    prefix = [r.randint(case["prefix_min"], case["prefix_max"]) for _ in range(case.get("chunks", 0))]
    return ctx, new, prefix


def _row_bytes(case):
    """Bytes of one token's K and V in its pages (int8: with its scales)."""
    scales = 2 * case["kv_heads"] * 2 if case["kv"] == "i8" else 0
    return 2 * case["kv_heads"] * case["dim"] * ESIZE[case["kv"]] + scales


def work(case):
    """Bytes read or written once and multiply-add flops of one pass."""
    D, H = case["dim"], case["heads"]
    if case["kind"] == "dense":
        pairs = case["batch"] * H
        return {"bytes": pairs * (case["kv_len"] * (2 * D + 1) * 4 + 2 * D * 4), "flops": pairs * case["kv_len"] * 4 * D}
    if case["kind"] == "token_prep":
        rows = case["tokens"] * (H + case["kv_heads"]) * D * 4
        v = case["tokens"] * case["kv_heads"] * D * 4
        return {"bytes": 2 * rows + v + case["tokens"] * (_row_bytes(case) + 12),
                "flops": case["tokens"] * (H + case["kv_heads"]) * D * 8}
    ctx, new, prefix = _lens(case)
    block, row = case["block"], _row_bytes(case)
    layers = LAYERS if case["kind"] == "decode_step" else 1
    table = sum(-(-n // block) for n in ctx) + sum(-(-(n + p) // block) for n, p in zip(new, prefix))
    q_bytes = len(ctx) * H * D * 8 + sum(new) * H * D * 6
    kv_bytes = (sum(ctx) + sum(new) + sum(prefix)) * row
    if case["kind"] == "decode_step":  # the new token's fp32 K and V, and its page row
        kv_bytes += len(ctx) * (2 * case["kv_heads"] * D * 4 + row)
    pairs = sum(ctx) + sum(n * p + n * (n + 1) // 2 for n, p in zip(new, prefix))
    return {"bytes": layers * (kv_bytes + q_bytes + 4 * table), "flops": layers * pairs * 4 * D * H}


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 8e12, w["flops"] / 2.5e15)


def tolerance(case):
    """Relative error another correct implementation shows: about four times
    this library's own error against 64-bit arithmetic, as measured (decode
    2e-7 to 3e-6, prefill 1e-4 to 3e-4, q/k norm and rotation 1e-7)."""
    if case["kind"] == "dense":
        return {"rel": 2e-6, "max": 1e-4}
    if case["kind"] == "token_prep":
        # the rounded pages: a value on a rounding boundary moves by one step
        return {"rel": 1e-4, "max": 0.01, "differ": 1e-4}
    if case["kind"] in ("decode", "decode_step"):
        return {"rel": 1e-5, "max": 1e-3}
    # P (and int8 V) enter the matrix product in 16 bits
    return {"rel": 1.2e-3, "max": 0.03}


# ---- inputs -----------------------------------------------------------------


class _Pool:
    """Pages of a paged KV cache with random block tables for the given
    lengths, a quarter larger than they need."""

    def __init__(self, case, lens, gen, empty=False):
        bs, hkv, D = case["block"], case["kv_heads"], case["dim"]
        used = [-(-n // bs) for n in lens]
        nb = max(1, (sum(used) * 5 + 3) // 4)
        self.kv, self.bs = case["kv"], bs
        perm = torch.randperm(nb, generator=gen, device=DEV).to(torch.int32)
        self.tables = torch.full((len(lens), max(used + [1])), -1, dtype=torch.int32, device=DEV)
        at = 0
        for i, n in enumerate(used):
            self.tables[i, :n] = perm[at:at + n]
            at += n
        self.ks = self.vs = None
        std = 0.5 if case["kind"] in ("prefill", "prefill_split") else 1.0
        self.k, self.ks = self._values((nb, bs, hkv, D), std, gen, empty)
        self.v, self.vs = self._values((nb, bs, hkv, D), std, gen, empty)
        self.pages = pyvcpp.kv_pages(KV[self.kv], self.k, self.v, bs, hkv, D, nb, bs * hkv * D, self.ks, self.vs,
                                     hkv * bs if self.kv == "i8" else 0)

    def _values(self, shape, std, gen, empty):
        if empty:
            dt = {"f32": torch.float32, "f16": torch.float16, "i8": torch.int8, "fp8": torch.uint8}[self.kv]
            scale = torch.zeros(shape[0], shape[2], shape[1], dtype=torch.float16, device=DEV)
            return torch.zeros(shape, dtype=dt, device=DEV), scale if self.kv == "i8" else None
        if self.kv == "f16":
            return torch.randn(shape, generator=gen, device=DEV, dtype=torch.float16) * std, None
        x = torch.randn(shape, generator=gen, device=DEV) * std
        if self.kv == "f32":
            return x, None
        if self.kv == "fp8":
            return x.to(torch.float8_e4m3fn).view(torch.uint8), None
        scale = (x.abs().amax(-1) / 127).to(torch.float16)
        q = torch.round(x / scale.float().unsqueeze(-1)).clamp_(-127, 127).to(torch.int8)
        return q, scale.transpose(1, 2).contiguous()

    def rows(self, i, n):
        """K and V of the first n positions of sequence i, in 64 bits: [n][kv heads][dim]."""
        ids = self.tables[i, :-(-n // self.bs)].long()
        got = []
        for x, s in ((self.k, self.ks), (self.v, self.vs)):
            x = x[ids]
            x = x.view(torch.float8_e4m3fn) if self.kv == "fp8" else x
            x = x.double()
            if self.kv == "i8":
                x = x * s[ids].double().transpose(1, 2).unsqueeze(-1)
            got.append(x.reshape(-1, *x.shape[2:])[:n])
        return got

    def buffers(self):
        out = {"k": self.k, "v": self.v}
        if self.kv == "i8":
            out.update(ks=self.ks, vs=self.vs)
        return out


def _ints(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def _randn(gen, *shape, dtype=torch.float32, std=1.0):
    return torch.randn(shape, generator=gen, device=DEV, dtype=dtype) * std


def _inv_freq(D):
    return (1.0 / 10000.0 ** (torch.arange(0, D, 2, dtype=torch.float64) / D)).float().to(DEV)


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    H, D = case["heads"], case["dim"]
    s = {"case": case, "kind": case["kind"], "H": H}
    if case["kind"] == "dense":
        B, n = case["batch"], case["kv_len"]
        s["q"] = _randn(gen, B, H, case["q_len"], D)
        s["k"], s["v"] = _randn(gen, B, H, n, D), _randn(gen, B, H, n, D)
        s["out"] = torch.zeros(B, H, D, device=DEV)
        s["weights"] = torch.zeros(B, H, n, device=DEV)
        return s
    if case["kind"] == "token_prep":
        n = case["tokens"]
        s["pool"] = _Pool(case, [n], gen, empty=True)
        s["q"], s["k"], s["v"] = (_randn(gen, n, h, D) for h in (H, case["kv_heads"], case["kv_heads"]))
        s["qw"], s["kw"] = (1.0 + 0.1 * _randn(gen, D) for _ in range(2))
        s["positions"] = torch.arange(1024, 1024 + n, dtype=torch.int32, device=DEV) % 4096
        s["inv_freq"] = _inv_freq(D)
        s["slots"] = _slots(s["pool"], 0, 0, n)
        return s
    ctx, new, prefix = _lens(case)
    if case["kind"] == "decode_step":
        s["pools"] = [_Pool(case, ctx, gen) for _ in range(LAYERS)]
        s["q"] = [_randn(gen, len(ctx), H, D) for _ in range(LAYERS)]
        s["new"] = [(_randn(gen, len(ctx), case["kv_heads"], D), _randn(gen, len(ctx), case["kv_heads"], D))
                    for _ in range(LAYERS)]
        s["out"] = [torch.zeros_like(q) for q in s["q"]]
        s["ctx"], s["max_ctx"] = _ints(ctx), max(ctx)
        s["slots"] = [torch.cat([_slots(p, i, n - 1, n) for i, n in enumerate(ctx)]) for p in s["pools"]]
        need = pyvcpp.decode_workspace_size(s["pools"][0].pages, len(ctx), H, s["max_ctx"])
        s["ws"] = torch.zeros(max(need, 16), dtype=torch.uint8, device=DEV)
        _step(s)  # once outside the capture, as a program does before it records
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            _step(s)
        return s
    lens = ctx + [n + p for n, p in zip(new, prefix)]
    s["pool"] = pool = _Pool(case, lens, gen)
    if ctx:
        s["dq"] = _randn(gen, len(ctx), H, D)
        s["dout"] = torch.zeros_like(s["dq"])
        s["ctx"], s["max_ctx"] = _ints(ctx), max(ctx)
        s["dtables"] = pool.tables[:len(ctx)].contiguous()
    if new:
        start = [0]
        for n in new:
            start.append(start[-1] + n)
        s["pq"] = _randn(gen, start[-1], H, D, dtype=torch.float16, std=0.5 if case["kind"] != "mixed" else 1.0)
        s["pout"] = torch.zeros(start[-1], H, D, device=DEV)
        s["q_start"], s["prefix"] = _ints(start), _ints(prefix)
        s["max_new"], s["max_prefix"] = max(new), max(prefix)
        s["ptables"] = pool.tables[len(ctx):].contiguous()
    need = 0
    if case["kind"] == "decode":
        need = pyvcpp.decode_workspace_size(pool.pages, len(ctx), H, s["max_ctx"])
    elif case["kind"] == "mixed":
        need = pyvcpp.mixed_workspace_size(pool.pages, len(ctx), H, s["max_ctx"], s["ptables"].shape[1])
    elif case["kind"] == "prefill_split":
        need = pyvcpp.prefill_workspace_size(pool.pages, len(new), s["max_new"], s["max_prefix"], H)
    s["ws"] = torch.zeros(max(need, 16), dtype=torch.uint8, device=DEV)
    return s


def _slots(pool, i, lo, hi):
    """Physical slots of positions lo .. hi - 1 of sequence i."""
    pos = torch.arange(lo, hi, device=DEV)
    return pool.tables[i, pos // pool.bs].long() * pool.bs + pos % pool.bs


def _step(s):
    for i, pool in enumerate(s["pools"]):
        pyvcpp.write_kv(pool.pages, s["new"][i][0], s["new"][i][1], s["slots"][i])
        pyvcpp.paged_decode(pool.pages, s["q"][i], s["out"][i], pool.tables, s["ctx"], s["max_ctx"], s["H"],
                            workspace=s["ws"])


# ---- one pass ---------------------------------------------------------------


def run(s):
    kind, H = s["kind"], s["H"]
    if kind == "decode":
        return pyvcpp.paged_decode(s["pool"].pages, s["dq"], s["dout"], s["dtables"], s["ctx"], s["max_ctx"], H,
                                   workspace=s["ws"])
    if kind == "decode_step":
        s["graph"].replay()
        return {"out": s["out"]}
    if kind == "prefill":
        return pyvcpp.paged_prefill(s["pool"].pages, s["pq"], s["pout"], s["ptables"], s["q_start"], s["prefix"],
                                    s["max_new"], H)
    if kind == "prefill_split":
        return pyvcpp.paged_prefill_split(s["pool"].pages, s["pq"], s["pout"], s["ptables"], s["q_start"],
                                          s["prefix"], s["max_new"], s["max_prefix"], H, workspace=s["ws"])
    if kind == "mixed":
        pyvcpp.paged_mixed_step(s["pool"].pages, s["dq"], s["dout"], s["dtables"], s["ctx"], s["max_ctx"], s["pq"],
                                s["pout"], s["ptables"], s["q_start"], s["prefix"], s["max_new"], H,
                                workspace=s["ws"])
        return {"decode": s["dout"], "prefill": s["pout"]}
    if kind == "token_prep":
        pyvcpp.qk_norm_rope(s["q"], s["k"], s["positions"], s["inv_freq"], s["qw"], s["kw"])
        pyvcpp.write_kv(s["pool"].pages, s["k"], s["v"], s["slots"])
        return dict(s["pool"].buffers(), q=s["q"])
    c = s["case"]
    pyvcpp.lib().flash_attention_cuda(*(ctypes.c_void_p(s[x].data_ptr()) for x in ("q", "k", "v", "out", "weights")),
                                      c["batch"], H, c["dim"], c["q_len"], c["kv_len"], None)
    return {"out": s["out"], "weights": s["weights"]}


# ---- the same in 64 bits ----------------------------------------------------


def _attend(q, k, v, first):
    """Attention of q [n][H][D] over k, v [m][kv heads][D]: row i sees
    positions 0 .. first + i."""
    n, H, D = q.shape
    m, hkv = k.shape[0], k.shape[1]
    out = torch.empty(n, H, D, dtype=torch.float64, device=q.device)
    hidden = torch.arange(m, device=q.device)[None, :] > first + torch.arange(n, device=q.device)[:, None]
    for h in range(hkv):
        qh = q[:, h * (H // hkv):(h + 1) * (H // hkv)].transpose(0, 1)
        w = torch.matmul(qh, k[:, h].t().contiguous()) / math.sqrt(D)
        w = torch.softmax(w.masked_fill_(hidden, -math.inf), -1)
        out[:, h * (H // hkv):(h + 1) * (H // hkv)] = torch.matmul(w, v[:, h].contiguous()).transpose(0, 1)
    return out


def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "dense":
        w = torch.matmul(s["q"][:, :, :1].double(), s["k"].double().transpose(2, 3).contiguous())
        w = torch.softmax(w / math.sqrt(case["dim"]), -1)
        return {"out": torch.matmul(w, s["v"].double())[:, :, 0], "weights": w[:, :, 0]}
    if case["kind"] == "token_prep":
        return _exact_prep(case, s)
    ctx, new, prefix = _lens(case)
    if case["kind"] == "decode_step":
        outs = []
        for i, pool in enumerate(s["pools"]):  # the pages hold the new tokens from prepare's first step
            outs.append(torch.cat([_attend(s["q"][i][j:j + 1].double(), *pool.rows(j, n), n - 1)
                                   for j, n in enumerate(ctx)]))
        return {"out": outs}
    pool, dout, pout = s["pool"], None, None
    if ctx:
        dout = torch.cat([_attend(s["dq"][i:i + 1].double(), *pool.rows(i, n), n - 1) for i, n in enumerate(ctx)])
    if new:
        parts, at = [], 0
        for i, (n, p) in enumerate(zip(new, prefix)):
            k, v = pool.rows(len(ctx) + i, n + p)
            for lo in range(0, n, 512):
                hi = min(n, lo + 512)
                parts.append(_attend(s["pq"][at + lo:at + hi].double(), k, v, p + lo))
            at += n
        pout = torch.cat(parts)
    if case["kind"] == "mixed":
        return {"decode": dout, "prefill": pout}
    return dout if ctx else pout


def _exact_prep(case, s):
    theta = (s["inv_freq"][None, :] * s["positions"][:, None].float()).double()  # an fp32 angle by definition
    c, sn = torch.cos(theta)[:, None], torch.sin(theta)[:, None]

    def prep(x, w):
        x = x.double()
        x = x * w.double() / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * c - b * sn, a * sn + b * c], -1).flatten(-2)

    out = {"q": prep(s["q"], s["qw"])}
    blocks, at = s["slots"] // case["block"], s["slots"] % case["block"]
    for name, x in (("k", prep(s["k"], s["kw"])), ("v", s["v"].double())):
        if case["kv"] in ("i8", "fp8"):  # codes, whole numbers
            out[name] = None
            continue
        page = torch.zeros(s["pool"].k.shape, dtype=torch.float64, device=DEV)
        page[blocks, at] = x
        out[name] = page
    return out
