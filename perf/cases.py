"""Performance cases of the paged-attention framework: the attention work of one
engine step, taken through the public entry points a serving engine calls.

A pass is one step's attention over ``layers`` decoder layers: the K/V write of
the step's new tokens and the attention over every sequence's history, layer
after layer, with that step's metadata already on the device (as the engine's
scheduler leaves it) and a context object made for the step. Shapes are the
Qwen2.5 0.5B and 7B attention shapes this framework is built and benchmarked
for (14 q / 2 kv heads of 64, 28 q / 4 kv heads of 128, block size 16).

``kind`` of a case:

- ``decode``: one new token per sequence through ``paged_attention``, with the
  metadata in one of three forms: ``tables`` (block tables and context
  lengths), ``reference`` (``gather_slots`` + additive mask, recognised on the
  device) or ``masked`` (the same with the fused path switched off, the
  reference engine's default flag);
- ``graph``: a decode step through ``HipGraphDecoder.decode`` from host lists;
- ``prefill``: packed query chunks after cached prefixes (and, with
  ``decodes``, one-token rows packed first: a mixed step), in the same three
  forms, through ``paged_attention`` or, with ``rope``, ``rope_paged_attention``
  (with ``lists``, the step's metadata is built by ``prefill_context`` in the
  pass);
- ``mixed``: decode rows and chunks as one captured graph (``MixedStep``).
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
ESIZE = {"bf16": 2, "fp16": 2, "fp32": 4}
SMALL = {"hq": 14, "hkv": 2, "d": 64}  # Qwen2.5-0.5B attention
LARGE = {"hq": 28, "hkv": 4, "d": 128}  # Qwen2.5-7B attention


def listed() -> list[dict]:
    return [
        # a handful of chats on the small model, fp32: the smallest step, where
        # launches and host work count
        _decode("decode-small-fp32", SMALL, "fp32", seqs=8, lo=1, hi=512, layers=4),
        # the same batch as a serving loop runs it: a whole 24-layer step
        # replayed as a graph, its metadata built from the scheduler's lists
        {"name": "graph-small-fp32", "kind": "graph", **SMALL, "dtype": "fp32", "bs": 16, "seqs": 8, "lo": 1,
         "hi": 512, "dist": "uniform", "layers": 24, "layout": "head_major"},
        # the headline decode: 64 chats of 512..4096 tokens on the 7B shape
        _decode("decode-7b-bf16", LARGE, "bf16", seqs=64, lo=512, hi=4096, layers=8),
        # few sequences, a long tail of contexts (documents among chats), fp16
        _decode("decode-skewed-fp16", LARGE, "fp16", seqs=16, lo=16, hi=32768, layers=8, dist="lognormal"),
        # an unchanged reference caller: gather_slots + mask, its contiguous
        # pool layout, a batch that is no power of two
        _decode("decode-reference-bf16", LARGE, "bf16", seqs=37, lo=100, hi=3000, layers=8, form="reference",
                layout="slot_major"),
        # the reference engine's default flag: no fused path, mask read as given
        _decode("decode-masked-bf16", LARGE, "bf16", seqs=24, lo=64, hi=2048, layers=4, form="masked"),
        # chunked prefill: 512-token chunks after cached prefixes of up to 8k,
        # pairs of sequences sharing prefix blocks
        _prefill("prefill-7b-bf16", LARGE, "bf16", seqs=8, lo=512, hi=512, prefix=8192, layers=3, share=True),
        # short fresh prompts of odd lengths on the small model, rotary
        # embedding and K/V write in the framework's fused call, the step's
        # metadata built from the scheduler's lists
        _prefill("prefill-short-fp16", SMALL, "fp16", seqs=12, lo=9, hi=300, prefix=0, layers=8, rope=True,
                 lists=True),
        # fp32 chunks after short prefixes (the reference's CPU-parity dtype)
        _prefill("prefill-fp32", SMALL, "fp32", seqs=6, lo=64, hi=512, prefix=1500, layers=2),
        # an unchanged reference caller's packed step: decodes and chunks in one
        # frame, one varlen mask
        _prefill("prefill-reference-bf16", LARGE, "bf16", seqs=4, lo=128, hi=400, prefix=2000, layers=4,
                 form="reference", decodes=13),
        # the same kind of frame with the reference engine's default flag
        _prefill("prefill-masked-bf16", LARGE, "bf16", seqs=3, lo=100, hi=256, prefix=1000, layers=2,
                 form="masked", decodes=5),
        # the mixed continuous-batching step of the 7B shape as one graph
        {"name": "mixed-7b-bf16", "kind": "mixed", **LARGE, "dtype": "bf16", "bs": 16, "seqs": 224, "lo": 256,
         "hi": 4096, "dist": "uniform", "chunks": 4, "chunk": 256, "prefix": 0, "layers": 6},
    ]


def _named(name, case):
    return case if name is None else {"name": name, **case}


def _decode(name, shape, dtype, *, seqs, lo, hi, layers, dist="uniform", form="tables", layout="head_major", bs=16):
    return _named(name, {"kind": "decode", **shape, "dtype": dtype, "bs": bs, "seqs": seqs, "lo": lo, "hi": hi,
                         "dist": dist, "layers": layers, "form": form, "layout": layout})


def _prefill(name, shape, dtype, *, seqs, lo, hi, prefix, layers, form="tables", decodes=0, rope=False, share=False,
             lists=False, layout="head_major", bs=16):
    return _named(name, {"kind": "prefill", **shape, "dtype": dtype, "bs": bs, "seqs": seqs, "lo": lo, "hi": hi,
                         "prefix": prefix, "layers": layers, "form": form, "decodes": decodes, "rope": rope,
                         "share": share, "lists": lists, "layout": layout})


def draw(rng: random.Random) -> dict:
    """One more case of the listed ranges (no name): sizes log-uniform."""

    def log(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["decode", "decode", "decode", "graph", "prefill", "prefill", "prefill", "mixed"])
    small = rng.random() < 0.35
    shape = SMALL if small else LARGE
    bs = rng.choice([16, 16, 16, 32])
    layout = rng.choice(["head_major", "head_major", "slot_major"])
    if kind in ("decode", "graph"):
        seqs = log(1, 96 if kind == "decode" else 16)
        hi = log(48, 4096 if kind == "decode" else 512)
        dtype = rng.choice(["fp32", "bf16", "fp16"] if small else ["bf16", "bf16", "fp16"])
        lo = max(1, hi // rng.choice([2, 8, 500]))
        if kind == "graph":
            return {"kind": "graph", **shape, "dtype": dtype, "bs": bs, "seqs": seqs, "lo": lo, "hi": hi,
                    "dist": "uniform", "layers": rng.randint(4, 24), "layout": layout}
        form = rng.choice(["tables", "tables", "reference", "masked"])
        if form == "masked":
            seqs, hi = min(seqs, 24), min(hi, 2048)
            lo = min(lo, hi)
        dist = rng.choice(["uniform", "uniform", "lognormal"]) if form == "tables" else "uniform"
        if dist == "lognormal":
            seqs, lo, hi = min(seqs, 16), 16, 32768
        return _decode(None, shape, dtype, seqs=seqs, lo=lo, hi=hi, layers=rng.randint(2, 6), dist=dist, form=form,
                       layout=layout, bs=bs)
    if kind == "mixed":
        hi = log(64, 4096)
        return {"kind": "mixed", **LARGE, "dtype": rng.choice(["bf16", "fp16"]), "bs": bs, "seqs": log(8, 224),
                "lo": max(1, hi // 16), "hi": hi, "dist": "uniform", "chunks": rng.randint(1, 4),
                "chunk": log(16, 256), "prefix": rng.choice([0, 0, log(1, 2000)]), "layers": rng.randint(1, 4)}
    form = rng.choice(["tables", "tables", "reference", "masked"])
    if form == "tables":
        dtype = rng.choice(["fp32", "bf16", "fp16"] if small else ["bf16", "bf16", "fp16"])
        if dtype == "fp32":
            seqs, hi, prefix = log(1, 8), log(4, 512), rng.choice([0, log(1, 1500)])
        else:
            seqs, hi, prefix = log(1, 16), log(4, 512), rng.choice([0, log(1, 4096)])
        decodes = rng.choice([0, 0, log(1, 32)])
        return _prefill(None, shape, dtype, seqs=seqs, lo=max(1, hi // rng.choice([1, 4, 16])), hi=hi, prefix=prefix,
                        layers=rng.randint(1, 3), decodes=decodes, rope=rng.random() < 0.3, share=rng.random() < 0.3,
                        lists=decodes > 0, layout=layout, bs=bs)
    hi = log(4, 400 if form == "reference" else 256)
    return _prefill(None, shape, rng.choice(["bf16", "fp16"]), seqs=rng.randint(1, 4 if form == "reference" else 3),
                    lo=max(1, hi // rng.choice([1, 4])), hi=hi,
                    prefix=rng.choice([0, log(1, 2000 if form == "reference" else 1000)]), layers=rng.randint(1, 2),
                    form=form, decodes=rng.choice([0, log(1, 16)]), layout=layout, bs=bs)


# ---------------------------------------------------------------- sizes (a function of the case alone)


def _sizes(case: dict) -> tuple[list[int], list[int]]:
    """(cached tokens, new tokens) of every sequence, in packing order."""
    r = np.random.default_rng([case["seqs"], case["hi"], case.get("layers", 1)])

    def contexts(n):
        if case.get("dist") == "lognormal":
            x = np.round(r.lognormal(8.0, 1.2, n))
            return [int(v) for v in np.clip(x, case["lo"], case["hi"])]
        return [int(v) for v in r.integers(case["lo"], case["hi"] + 1, n)]

    if case["kind"] in ("decode", "graph"):
        return [c - 1 for c in contexts(case["seqs"])], [1] * case["seqs"]
    if case["kind"] == "mixed":
        n = case["chunks"]
        return [c - 1 for c in contexts(case["seqs"])] + [case["prefix"]] * n, [1] * case["seqs"] + [case["chunk"]] * n
    new = [int(v) for v in r.integers(case["lo"], case["hi"] + 1, case["seqs"])]
    cached = [int(v) for v in r.integers(0, case["prefix"] + 1, case["seqs"])]
    nd = case["decodes"]
    dec = [int(v) for v in r.integers(0, max(case["prefix"], 256) + 1, nd)]
    return dec + cached, [1] * nd + new


def _shared(case: dict, cached: list[int], new: list[int]) -> list[int]:
    """Leading blocks sequence i shares with sequence i - 1 (chunk pairs with a
    common cached prefix)."""
    out = [0] * len(cached)
    if case.get("share"):
        nd = case["decodes"]
        for i in range(nd + 1, len(cached), 2):
            out[i] = min(cached[i - 1], cached[i]) // case["bs"]
    return out


def work(case: dict) -> dict:
    cached, new = _sizes(case)
    es, hq, hkv, d = ESIZE[case["dtype"]], case["hq"], case["hkv"], case["d"]
    total, bs = sum(new), case["bs"]
    shared = _shared(case, cached, new)
    keys = sum(c + n for c, n in zip(cached, new)) - bs * sum(shared)
    pairs = sum(n * c + n * (n + 1) // 2 for c, n in zip(cached, new))
    # K/V of every key once (the new ones from the step's rows), the new rows'
    # pool write, q and out, write slots
    layer = 2 * keys * hkv * d * es + 2 * total * hkv * d * es + 2 * total * hq * d * es + 8 * total
    step = 0
    if case.get("form") in ("reference", "masked"):
        if case["kind"] == "decode":
            t = max(cached) + 1
            step = len(new) * t * (8 + es)
        else:
            allk = sum(c + n for c, n in zip(cached, new))
            step = allk * 8 + total * allk * es
    else:
        step = sum(-(-(c + n) // bs) for c, n in zip(cached, new)) * 4
    if case.get("rope"):
        layer += 2 * total * d * 4
    return {"bytes": case["layers"] * layer + step, "flops": case["layers"] * 4 * hq * d * pairs}


def tolerance(case: dict) -> dict:
    # about four times the largest difference measured from 64-bit arithmetic
    # over the same inputs (bf16 3.4e-3, fp16 6.2e-4, fp32 5.6e-7): 16-bit
    # queries, probabilities and outputs, or 32-bit sums
    return {"rel": {"bf16": 1.3e-2, "fp16": 2.5e-3, "fp32": 2.5e-6}[case["dtype"]]}


# ---------------------------------------------------------------- inputs (made from the seed alone)


def _inputs(case: dict, seed: int) -> dict:
    """Block tables, pool contents and the step's activations as plain tensors."""
    cached, new = _sizes(case)
    bs, dt, L = case["bs"], DTYPES[case["dtype"]], case["layers"]
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    shared = _shared(case, cached, new)
    nblk = [-(-(c + n) // bs) for c, n in zip(cached, new)]
    own = [b - s for b, s in zip(nblk, shared)]
    num_blocks = math.ceil(1.25 * sum(own)) + 1
    perm = np.random.default_rng(seed).permutation(num_blocks).tolist()
    tables, off = [], 0
    for i, (s, o) in enumerate(zip(shared, own)):
        tables.append((tables[i - 1][:s] if s else []) + perm[off : off + o])
        off += o
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rnd(*shape, scale=1.0):
        x = torch.randn(*shape, generator=g, device="cuda", dtype=dt)
        return x if scale == 1.0 else x * scale

    total = sum(new)
    out = {
        "cached": cached, "new": new, "tables": tables, "num_blocks": num_blocks,
        "k_pool": rnd(L, num_blocks * bs, hkv, d), "v_pool": rnd(L, num_blocks * bs, hkv, d),
        "q": rnd(L, total, hq, d, scale=1.5), "k": rnd(L, total, hkv, d), "v": rnd(L, total, hkv, d),
    }
    pos = np.concatenate([np.arange(c, c + n) for c, n in zip(cached, new)])
    seq = np.repeat(np.arange(len(new)), new)
    slots = np.array([tables[s][p // bs] * bs + p % bs for s, p in zip(seq.tolist(), pos.tolist())], dtype=np.int64)
    out["write_slots"] = torch.from_numpy(slots).cuda()
    if case.get("rope"):
        inv = 1.0 / (10000.0 ** (torch.arange(0, d, 2, dtype=torch.float64) / d))
        ang = torch.from_numpy(pos).double()[:, None] * inv[None, :]
        ang = torch.cat([ang, ang], dim=1)
        out["cos"], out["sin"] = ang.cos().float().cuda(), ang.sin().float().cuda()
    return out


def _tables_tensor(tables) -> torch.Tensor:
    bt = np.zeros((len(tables), max(len(t) for t in tables)), dtype=np.int32)
    for i, t in enumerate(tables):
        bt[i, : len(t)] = t
    return torch.from_numpy(bt).cuda()


def _history_slots(table, n, bs) -> np.ndarray:
    p = np.arange(n)
    return np.asarray(table, dtype=np.int64)[p // bs] * bs + p % bs


def _reference_metadata(case: dict, x: dict) -> tuple[torch.Tensor, torch.Tensor]:
    """``gather_slots`` and the additive mask as the reference engine builds them."""
    bs, dt = case["bs"], DTYPES[case["dtype"]]
    lens = [c + n for c, n in zip(x["cached"], x["new"])]
    low = torch.finfo(dt).min
    if case["kind"] == "decode":
        gs = np.zeros((len(lens), max(lens)), dtype=np.int64)
        for i, n in enumerate(lens):
            gs[i, :n] = _history_slots(x["tables"][i], n, bs)
        cols = torch.arange(max(lens), device="cuda")
        hide = cols[None, :] >= torch.tensor(lens, device="cuda")[:, None]
        mask = torch.zeros(len(lens), 1, 1, max(lens), dtype=dt, device="cuda")
        return torch.from_numpy(gs).cuda(), mask.masked_fill_(hide[:, None, None, :], low)
    gs = np.concatenate([_history_slots(t, n, bs) for t, n in zip(x["tables"], lens)])[None]
    k_seq = torch.from_numpy(np.repeat(np.arange(len(lens)), lens)).cuda()
    k_pos = torch.from_numpy(np.concatenate([np.arange(n) for n in lens])).cuda()
    q_seq = torch.from_numpy(np.repeat(np.arange(len(lens)), x["new"])).cuda()
    q_pos = torch.from_numpy(np.concatenate([np.arange(c, c + n) for c, n in zip(x["cached"], x["new"])])).cuda()
    hide = (q_seq[:, None] != k_seq[None, :]) | (k_pos[None, :] > q_pos[:, None])
    mask = torch.zeros(1, 1, len(q_seq), len(k_seq), dtype=dt, device="cuda")
    return torch.from_numpy(gs).cuda(), mask.masked_fill_(hide[None, None], low)


def prepare(case: dict, seed: int) -> dict:
    from infrared_amd import PagedKVPool
    from infrared_amd.hip_graph import HipGraphDecoder
    from infrared_amd.mixed_step import MixedBatch, MixedInputs, MixedStep

    x = _inputs(case, seed)
    dt = DTYPES[case["dtype"]]
    pool = PagedKVPool(case["layers"], x["num_blocks"], case["bs"], case["hkv"], case["d"], dt, device="cuda",
                       layout=case.get("layout", "head_major"))
    pool.k.copy_(x.pop("k_pool"))
    pool.v.copy_(x.pop("v_pool"))
    s = {"case": case, "pool": pool, **x}
    kind, n = case["kind"], len(x["new"])
    if kind == "mixed":
        nd = case["seqs"]
        cu = [i * case["chunk"] for i in range(case["chunks"] + 1)]
        batch = MixedBatch(
            write_slots=x["write_slots"], dec_tables=_tables_tensor(x["tables"][:nd]),
            dec_ctx=torch.tensor([c + 1 for c in x["cached"][:nd]], dtype=torch.int32).cuda(),
            pre_tables=_tables_tensor(x["tables"][nd:]), cu_seqlens_q=torch.tensor(cu, dtype=torch.int32).cuda(),
            q_start=torch.full((case["chunks"],), case["prefix"], dtype=torch.int32).cuda(), max_q_len=case["chunk"])
        inputs = MixedInputs(q_dec=x["q"][:, :nd].contiguous(), q_pre=x["q"][:, nd:].contiguous(), k_new=x["k"],
                             v_new=x["v"])
        s["step"] = MixedStep(pool, batch, inputs, case["d"] ** -0.5)
        s["step"].capture()
        return s
    if kind == "graph":
        from infrared_amd import paged_attention

        scale, n_rep = case["d"] ** -0.5, case["hq"] // case["hkv"]

        def layers(buf, paged):
            rows = [i if i < n else 0 for i in range(buf.ids.shape[0])]  # pad rows repeat row 0
            if "rows" not in s:
                s["rows"] = [t[:, rows].unsqueeze(2) for t in (x["q"], x["k"], x["v"])]
            q, k, v = s["rows"]
            outs = [paged_attention(q[i], k[i], v[i], paged, buf.mask, i, scale, n_rep)
                    for i in range(case["layers"])]
            return torch.stack(outs, dim=1)

        t_max = -(-case["hi"] // case["bs"]) * case["bs"]
        s["decoder"] = HipGraphDecoder(None, pool, max_num_seqs=n, t_max=t_max, block_size=case["bs"],
                                       step_fn=layers)
        s["decoder"].decode(x["tables"], x["cached"], [0] * n)  # captured once, as at a server's start
        return s
    form = case["form"]
    if kind == "prefill":
        s["qkv"] = [t.unsqueeze(1) for t in (x["q"], x["k"], x["v"])]  # [L, 1, tokens, heads, d]
        if case["rope"]:
            s["cs"] = [x["cos"].unsqueeze(0), x["sin"].unsqueeze(0)]
    else:
        s["qkv"] = [t.unsqueeze(2) for t in (x["q"], x["k"], x["v"])]  # [L, B, 1, heads, d]
    if form in ("reference", "masked"):
        s["gather_slots"], s["mask"] = _reference_metadata(case, x)
        return s
    s["block_tables"] = _tables_tensor(x["tables"])
    s["context_lens"] = torch.tensor([c + m for c, m in zip(x["cached"], x["new"])], dtype=torch.int32).cuda()
    s["q_start"] = torch.tensor(x["cached"], dtype=torch.int32).cuda()
    s["cu"] = torch.tensor([0, *np.cumsum(x["new"]).tolist()], dtype=torch.int32).cuda()
    return s


def _returns_pool(case: dict, num_blocks: int) -> bool:
    """Small pools, which the step has updated, are outputs too (the larger
    ones' new rows show in the attention over them)."""
    rows = case["layers"] * num_blocks * case["bs"]
    return rows * case["hkv"] * case["d"] * ESIZE[case["dtype"]] <= 48 << 20


def run(s: dict):
    out = _run(s)
    out = list(out) if isinstance(out, list) else [out]
    return [*out, s["pool"].k, s["pool"].v] if _returns_pool(s["case"], s["num_blocks"]) else out


def _run(s: dict):
    from infrared_amd import PagedContext, metadata, paged_attention, rope_paged_attention

    case, pool = s["case"], s["pool"]
    kind = case["kind"]
    if kind == "mixed":
        s["step"].replay()
        return [s["step"].out_dec, s["step"].out_pre]
    if kind == "graph":
        return s["decoder"].decode(s["tables"], s["cached"], [0] * len(s["new"]))
    q, k, v = s["qkv"]
    mask = None
    if case["form"] in ("reference", "masked"):
        # a step's metadata arrives as new tensor objects, its buffers reused
        mask = s["mask"].view(s["mask"].shape)
        gather = s["gather_slots"].view(s["gather_slots"].shape)
        paged = PagedContext(pool, s["write_slots"], gather, case["form"] == "reference")
    elif kind == "prefill" and case["lists"]:
        paged, _ = metadata.prefill_context(pool, s["tables"], s["cached"], s["new"])
    elif kind == "prefill":
        paged = PagedContext(pool, s["write_slots"], None, True, s["block_tables"], None, s["cu"], s["q_start"],
                             max(s["new"]))
    else:
        paged = PagedContext(pool, s["write_slots"], None, True, s["block_tables"], s["context_lens"])
    scale, n_rep = case["d"] ** -0.5, case["hq"] // case["hkv"]
    outs = []
    for i in range(case["layers"]):
        if case.get("rope"):
            outs.append(rope_paged_attention(q[i], k[i], v[i], *s["cs"], paged, mask, i, scale, n_rep))
        else:
            outs.append(paged_attention(q[i], k[i], v[i], paged, mask, i, scale, n_rep))
    return outs


# ---------------------------------------------------------------- 64-bit reference


def exact(case: dict, seed: int):
    x = _inputs(case, seed)
    out = _exact(case, x)
    if not _returns_pool(case, x["num_blocks"]):
        return out
    pools = []
    for pool, new in (("k_pool", _rotated(case, x, x["k"].double())), ("v_pool", x["v"].double())):
        pools.append(x[pool].double())
        pools[-1][:, x["write_slots"]] = new
    return [*out, *pools]


def _rotated(case: dict, x: dict, t: torch.Tensor) -> torch.Tensor:
    """Rotary embedding of ``[.., tokens, heads, d]`` when the case has one."""
    if not case.get("rope"):
        return t
    cos, sin, half = x["cos"].double()[:, None], x["sin"].double()[:, None], case["d"] // 2
    return t * cos + torch.cat([-t[..., half:], t[..., :half]], dim=-1) * sin


def _exact(case: dict, x: dict) -> list[torch.Tensor]:
    cached, new, bs = x["cached"], x["new"], case["bs"]
    hkv, d, rep = case["hkv"], case["d"], case["hq"] // case["hkv"]
    outs = []
    for layer in range(case["layers"]):
        q, k, v = (x[n][layer].double() for n in ("q", "k", "v"))
        q, k = _rotated(case, x, q), _rotated(case, x, k)
        out = torch.empty_like(q)
        row = 0
        for table, c, n in zip(x["tables"], cached, new):
            slots = torch.from_numpy(_history_slots(table, c, bs)).cuda()
            kk = torch.cat([x["k_pool"][layer, slots].double(), k[row : row + n]])  # [T, hkv, d]
            vv = torch.cat([x["v_pool"][layer, slots].double(), v[row : row + n]])
            hide = (torch.arange(c + n, device="cuda")[None, :] > torch.arange(c, c + n, device="cuda")[:, None])
            for h in range(hkv):
                qh = q[row : row + n, h * rep : (h + 1) * rep].reshape(n * rep, d)
                sc = (qh @ kk[:, h].T.contiguous()) * d**-0.5
                sc = sc.masked_fill(hide.repeat_interleave(rep, 0), -math.inf)
                out[row : row + n, h * rep : (h + 1) * rep] = (sc.softmax(-1) @ vv[:, h].contiguous()).view(n, rep, d)
            row += n
        outs.append(out)
    if case["kind"] == "mixed":
        nd = case["seqs"]
        return [torch.stack([o[:nd] for o in outs]), torch.stack([o[nd:] for o in outs])]
    if case["kind"] == "graph":
        return [torch.stack(outs, dim=1).unsqueeze(2)]
    if case["kind"] == "decode":
        return [o.unsqueeze(1) for o in outs]
    return [o.unsqueeze(0) for o in outs]
