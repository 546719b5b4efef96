"""The work whose time is measured, through the package's public entry points.

The path is the sparse-attention inference path: the quantiser that produces the fp8 indexer's
inputs, the lightning indexer with its top-k, the top-k selector alone, and the attention kernels
over the selected rows (latent MLA, its joined-rope decode entry, the window + compressed-KV
attention with sinks, grouped 128-wide heads).  ``listed()`` holds the shapes of this
repository's benchmark and tests, ``draw(rng)`` more of the same ranges.  A state is made on the
GPU from the seed alone; ``run`` is one call.
"""
import math

import torch

from __graft_entry__ import load_package

_FP8 = torch.float8_e4m3fn
_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32, "fp8": _FP8, "int8": torch.int8}
_SIZE = {"bf16": 2, "fp16": 2, "fp32": 4, "fp8": 1, "int8": 1}


def listed():
    return [
        # The smallest call: one token of the decode entry that takes latent and rope parts apart
        # (128 heads, 128-row blocks, 2048 of 2560 visible keys, a pool of 6400 rows).
        dict(name="sfa_decode", kind="sfa", T=1, H=128, pool=6400, act=2560, topk=2048, block=128, causal=0,
             dtype="bf16"),
        # The selector example: 64 rows of 4096 scores, 2048 kept.
        dict(name="topk_example", kind="topk", rows=64, n=4096, k=2048, lens=False, values=False),
        # A decode batch of the window + selected-compressed-rows attention: 24 sequences, one
        # query each, about 8K keys.
        dict(name="v4_decode", kind="v4", mode="csa", B=24, S=1, kv=8193, H=64, K=512, win=127, block=128,
             dtype="bf16"),
        # A decode batch of the latent attention: 64 sequences of 64K tokens in a paged cache.
        dict(name="mla_decode", kind="mla", B=64, S=1, kv=65536, H=128, topk=2048, block=64, dtype="bf16"),
        # Grouped 128-wide heads at the grouped example's shape (odd query and key counts, fp16).
        dict(name="gqa_example", kind="gqa", B=2, S=273, kv=44444, H=64, G=4, topk=2048, dtype="fp16"),
        # Quantising the index queries of a 4096-token chunk: 64 heads of 128.
        dict(name="quant_queries", kind="quant", rows=262144, n=128, dtype="bf16", out="fp8", round_scale=False),
        # The indexer of a decode step: 32 sequences of 128K keys, paged fp8 keys with scales.
        dict(name="indexer_decode", kind="indexer", layout="paged", B=32, S=1, kv=131072, H=64, D=128, K=2048,
             dtype="fp8", block=64),
        # Packed ragged batches of the 16-bit indexer (24 heads), causal, uneven lengths.
        dict(name="indexer_packed", kind="indexer", layout="packed", B=3, S=1021, kv=9001, H=24, D=128, K=2048,
             dtype="bf16", block=0),
        # A prefill chunk of the window + selected-compressed-rows attention: 8192 rows.
        dict(name="v4_prefill", kind="v4", mode="csa", B=1, S=8192, kv=8192, H=64, K=512, win=127, block=128,
             dtype="bf16"),
        # The indexer of a 4096-token prefill chunk at the end of 32K keys.
        dict(name="indexer_prefill", kind="indexer", layout="dense", B=1, S=4096, kv=32768, H=64, D=128, K=2048,
             dtype="fp8", block=0),
        # The same at the end of 128K keys, where the selection is streamed out of the indexer.
        dict(name="indexer_long", kind="indexer", layout="dense", B=1, S=4096, kv=131072, H=64, D=128, K=2048,
             dtype="fp8", block=0),
        # The latent attention of a whole 16K-token prompt, causal: the largest call.
        dict(name="mla_prefill", kind="mla", B=1, S=16384, kv=16384, H=128, topk=2048, block=0, dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]: odd sizes as often as even ones."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["sfa", "topk", "v4", "v4", "mla_decode", "mla_prefill", "mla_prefill", "gqa", "quant",
                       "indexer_decode", "indexer_packed", "indexer_dense", "indexer_dense"])
    dt = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "sfa":
        pool = 128 * rng.randint(20, 375)
        return dict(kind="sfa", T=rng.randint(1, 8), H=rng.choice([16, 32, 64, 128]), pool=pool,
                    act=rng.randint(1100, pool), topk=rng.choice([512, 1024, 2048]), block=128,
                    causal=rng.randint(0, 1), dtype=dt)
    if kind == "topk":
        n = _log_int(rng, 1000, 131072)
        return dict(kind="topk", rows=_log_int(rng, 1, max(2, min(4096, (1 << 28) // n))), n=n,
                    k=min(n, rng.choice([64, 128, 512, 1000, 2048])), lens=rng.random() < 0.3,
                    values=rng.random() < 0.5)
    if kind == "v4":
        mode = rng.choice(["swa", "hca", "csa"])
        B, S = (_log_int(rng, 1, 64), 1) if rng.random() < 0.5 else (rng.randint(1, 3), _log_int(rng, 64, 2700))
        return dict(kind="v4", mode=mode, B=B, S=S, kv=S + _log_int(rng, 200, 12000), H=64, K=512, win=127, block=128,
                    dtype=dt)
    if kind == "mla_decode":
        return dict(kind="mla", B=_log_int(rng, 1, 64), S=rng.choice([1, 1, 1, 2]), kv=_log_int(rng, 4096, 65536),
                    H=rng.choice([16, 64, 128, 128]), topk=rng.choice([512, 1024, 2048, 2048]), block=64, dtype=dt)
    if kind == "mla_prefill":
        S = _log_int(rng, 64, 12000)
        return dict(kind="mla", B=1 if S > 4000 else rng.randint(1, 2), S=S, kv=S + rng.choice([0, 0, 3968, 30001]),
                    H=rng.choice([16, 32, 64, 128, 128]), topk=rng.choice([512, 1024, 2048, 2048]), block=0,
                    dtype=dt)
    if kind == "gqa":
        return dict(kind="gqa", B=rng.randint(1, 2), S=_log_int(rng, 16, 400), kv=_log_int(rng, 8192, 50000),
                    H=rng.choice([32, 64]), G=rng.choice([2, 4]), topk=rng.choice([512, 1024, 2048]), dtype=dt)
    if kind == "quant":
        n = rng.choice([128, 128, 128, 64, 512, 576, 7168])
        return dict(kind="quant", rows=_log_int(rng, 64, 33554432 // n), n=n, dtype=rng.choice(["bf16", "bf16", "fp16",
                    "fp32"]), out=rng.choice(["fp8", "fp8", "int8"]), round_scale=rng.random() < 0.3)
    if kind == "indexer_decode":
        return dict(kind="indexer", layout="paged", B=_log_int(rng, 1, 32), S=rng.choice([1, 1, 1, 2]),
                    kv=_log_int(rng, 4096, 131072), H=rng.choice([32, 64, 64]), D=128, K=2048,
                    dtype=rng.choice(["fp8", "fp8", "bf16"]), block=64)
    if kind == "indexer_packed":
        return dict(kind="indexer", layout="packed", B=rng.randint(1, 4), S=_log_int(rng, 32, 1500),
                    kv=_log_int(rng, 2500, 20000), H=rng.choice([8, 16, 24, 32, 64]), D=rng.choice([64, 128, 128]),
                    K=rng.choice([512, 2048]), dtype=rng.choice(["fp8", dt]), block=0)
    S = _log_int(rng, 64, 4096)
    return dict(kind="indexer", layout="dense", B=1, S=S, kv=max(S, _log_int(rng, 4096, 131072)),
                H=rng.choice([32, 64, 64]), D=128, K=rng.choice([1024, 2048, 2048]), dtype="fp8", block=0)


# ------------------------------------------------------------------------------- inputs


def _gen(seed):
    dev = torch.device("cuda")
    return dev, torch.Generator(device=dev).manual_seed(seed)


def _normal(g, dev, shape, dtype, scale=1.0):
    return torch.randn(shape, generator=g, device=dev).mul_(scale).to(dtype)


def _choose(g, dev, limits, width, k):
    """Per row r: min(k, limits[r]) distinct positions of [0, limits[r]) in random order, then -1."""
    rows = limits.numel()
    out = torch.full((rows, k), -1, dtype=torch.int32, device=dev)
    cols = torch.arange(width, device=dev).view(1, -1)
    step = max(1, (1 << 27) // width)
    kk = min(k, width)
    for r in range(0, rows, step):
        u = torch.rand((min(step, rows - r), width), generator=g, device=dev)
        u.masked_fill_(cols >= limits[r:r + step].view(-1, 1), -1.0)
        v, i = torch.topk(u, kk, dim=1)
        out[r:r + step, :kk] = torch.where(v >= 0, i, -1).to(torch.int32)
    return out


def _fp8_rows(x):
    """fp8 rows with an fp32 scale of absmax / 448 each."""
    s = x.abs().amax(dim=-1).div(448.0)
    return (x / s.unsqueeze(-1)).clamp_(-448, 448).to(_FP8), s


def _uneven(total, B, least):
    """B lengths that sum to about ``total``, uneven and mostly odd."""
    part = [max(least, (total * (2 * b + 1)) // (B * B) - b) for b in range(B)]
    return part


def _limits(S, kv, dev):
    """Keys a causal query row sees: the last row sees all kv."""
    return torch.arange(kv - S + 1, kv + 1, device=dev)


def prepare(case, seed):
    pkg = load_package()
    pkg.load_library()
    dev, g = _gen(seed)
    c = dict(case)
    dt = _DT[c["dtype"]] if "dtype" in c else torch.float32
    st = {"pkg": pkg, "case": c}
    kind = c["kind"]
    if kind == "quant":
        st["x"] = _normal(g, dev, (c["rows"], c["n"]), dt, 3.0)
    elif kind == "topk":
        st["x"] = torch.randn((c["rows"], c["n"]), generator=g, device=dev)
        st["len"] = (torch.randint(c["n"] // 2, c["n"] + 1, (c["rows"],), generator=g, device=dev).to(torch.int32)
                     if c["lens"] else None)
    elif kind == "sfa":
        T, nb = c["T"], c["pool"] // c["block"]
        st["q"] = _normal(g, dev, (T, c["H"], 512), dt, 0.5)
        st["key"] = _normal(g, dev, (nb, c["block"], 1, 512), dt, 0.5)
        st["qr"] = _normal(g, dev, (T, c["H"], 64), dt, 0.5)
        st["kr"] = _normal(g, dev, (nb, c["block"], 1, 64), dt, 0.5)
        lim = _limits(T, c["act"], dev) if c["causal"] else torch.full((T,), c["act"], device=dev)
        st["idx"] = _choose(g, dev, lim, c["act"], c["topk"]).view(T, 1, -1)
        st["table"] = torch.randperm(nb, generator=g, device=dev).to(torch.int32).view(1, nb)
        st["qlen"] = torch.full((1,), T, dtype=torch.int32, device=dev)
        st["klen"] = torch.full((1,), c["act"], dtype=torch.int32, device=dev)
    elif kind == "mla":
        B, S, kv = c["B"], c["S"], c["kv"]
        st["q"] = _normal(g, dev, (B, S, c["H"], 576), dt, 0.5)
        st["table"] = st["qlen"] = st["klen"] = None
        if c["block"]:
            nb = -(-kv // c["block"])
            st["kv"] = _normal(g, dev, (B * nb, c["block"], 1, 576), dt, 0.5)
            st["table"] = torch.randperm(B * nb, generator=g, device=dev).to(torch.int32).view(B, nb)
            st["klen"] = torch.full((B,), kv, dtype=torch.int32, device=dev)
        else:
            st["kv"] = _normal(g, dev, (B, kv, 1, 576), dt, 0.5)
        # Row t sits at position kv - S + t; rows with fewer keys than the top-k end in empty slots.
        st["idx"] = _choose(g, dev, _limits(S, kv, dev).repeat(B), kv, c["topk"]).view(B, S, 1, c["topk"])
    elif kind == "gqa":
        B, S, G = c["B"], c["S"], c["G"]
        st["q"] = _normal(g, dev, (B, S, c["H"], 128), dt)
        st["kv"] = _normal(g, dev, (B, c["kv"], G, 128), dt)
        st["qlen"] = torch.full((B,), S, dtype=torch.int32, device=dev)
        st["klen"] = torch.full((B,), c["kv"], dtype=torch.int32, device=dev)
        lim = _limits(S, c["kv"], dev).view(1, S, 1).expand(B, S, G).reshape(-1)
        st["idx"] = _choose(g, dev, lim, c["kv"], c["topk"]).view(B, S, G, c["topk"])
    elif kind == "v4":
        B, S, bs = c["B"], c["S"], c["block"]
        ratio = 128 if c["mode"] == "hca" else 4
        # Ragged batches: a sequence's context is up to a tenth shorter than the longest one.
        lens = [c["kv"] - (c["kv"] - S) * b // (10 * B) for b in range(B)]
        nb = -(-c["kv"] // bs)
        st["q"] = _normal(g, dev, (B * S, c["H"], 512), dt, 0.5)
        st["ori"] = _normal(g, dev, (B * nb, bs, 1, 512), dt, 0.5)
        st["obt"] = torch.randperm(B * nb, generator=g, device=dev).to(torch.int32).view(B, nb)
        st["cu"] = torch.arange(B + 1, dtype=torch.int32, device=dev) * S
        st["lens"] = torch.tensor(lens, dtype=torch.int32, device=dev)
        st["sinks"] = torch.randn(c["H"], generator=g, device=dev)
        st["ratio"] = ratio
        st["cmp"] = st["cbt"] = st["idx"] = None
        if c["mode"] != "swa":
            cnb = max(1, -(-(c["kv"] // ratio) // bs))
            st["cmp"] = _normal(g, dev, (B * cnb, bs, 1, 512), dt, 0.5)
            st["cbt"] = torch.randperm(B * cnb, generator=g, device=dev).to(torch.int32).view(B, cnb)
        if c["mode"] == "csa":
            thr = torch.cat([_limits(S, n, dev) // ratio for n in lens])
            st["idx"] = _choose(g, dev, thr, max(1, c["kv"] // ratio), c["K"]).view(B * S, 1, c["K"])
    elif kind == "indexer":
        B, S, kv, H, D = c["B"], c["S"], c["kv"], c["H"], c["D"]
        st["table"] = st["ks"] = st["qlen"] = st["klen"] = None
        if c["layout"] == "packed":
            ql, kl = _uneven(B * S, B, 1), _uneven(B * kv, B, B * S)
            st["qlen"] = torch.tensor(ql, device=dev).cumsum(0).to(torch.int32)
            st["klen"] = torch.tensor(kl, device=dev).cumsum(0).to(torch.int32)
            q, k, w = (sum(ql), H, D), (sum(kl), 1, D), (sum(ql), H)
        elif c["layout"] == "paged":
            nb = -(-kv // c["block"])
            st["table"] = torch.randperm(B * nb, generator=g, device=dev).to(torch.int32).view(B, nb)
            st["klen"] = torch.full((B,), kv, dtype=torch.int32, device=dev)
            st["qlen"] = torch.full((B,), S, dtype=torch.int32, device=dev)
            q, k, w = (B, S, H, D), (B * nb, c["block"], 1, D), (B, S, H)
        else:
            q, k, w = (B, S, H, D), (B, kv, 1, D), (B, S, H)
        st["q"] = _normal(g, dev, q, dt)
        kf = torch.randn(k, generator=g, device=dev)
        if dt == _FP8:
            st["k"], ks = _fp8_rows(kf)
            st["ks"] = ks.reshape(ks.shape[:-1]).contiguous()
        else:
            st["k"] = kf.to(dt)
        st["w"] = torch.randn(w, generator=g, device=dev) / 8
    else:
        raise ValueError(kind)
    return st


# ------------------------------------------------------------------------------- one call


def run(st):
    pkg, c = st["pkg"], st["case"]
    kind = c["kind"]
    if kind == "quant":
        return pkg.act_quant(st["x"], round_scale=c["round_scale"], dtype=_DT[c["out"]])
    if kind == "topk":
        return pkg.topk_selector(st["x"], c["k"], row_len=st["len"], return_values=c["values"])
    if kind == "sfa":
        return pkg.sparse_attn_tilelang(st["q"], st["key"], st["key"], st["idx"], 576 ** -0.5, 1, st["qlen"],
                                        st["klen"],
                                        query_rope=st["qr"], key_rope=st["kr"], layout_query="TND",
                                        layout_kv="PA_BSND", sparse_mode=3 if c["causal"] else 0,
                                        block_table=st["table"])
    if kind == "mla":
        return pkg.sparse_mla_fwd(st["q"], st["kv"], st["idx"], 576 ** -0.5, block_table=st["table"],
                                  actual_seq_lengths_query=st["qlen"], actual_seq_lengths_kv=st["klen"])
    if kind == "gqa":
        return pkg.sparse_gqa_fwd(st["q"], st["kv"], st["idx"], actual_seq_lengths_query=st["qlen"],
                                  actual_seq_lengths_kv=st["klen"])
    if kind == "v4":
        return pkg.sparse_flash_mla(st["q"], ori_kv=st["ori"], cmp_kv=st["cmp"], cmp_sparse_indices=st["idx"],
                                    ori_block_table=st["obt"], cmp_block_table=st["cbt"], cu_seqlens_q=st["cu"],
                                    seqused_kv=st["lens"], sinks=st["sinks"], softmax_scale=512 ** -0.5,
                                    cmp_ratio=st["ratio"], ori_win_left=c["win"], return_softmax_lse=True)
    if c["layout"] == "packed":
        return pkg.lightning_indexer(st["q"], st["k"], st["w"], actual_seq_lengths_query=st["qlen"],
                                     actual_seq_lengths_key=st["klen"], layout_query="TND", layout_key="TND",
                                     sparse_count=c["K"], return_value=True, key_scale=st["ks"])
    if c["layout"] == "paged":  # the paged form returns positions only
        return pkg.lightning_indexer(st["q"], st["k"], st["w"], actual_seq_lengths_query=st["qlen"],
                                     actual_seq_lengths_key=st["klen"], block_table=st["table"],
                                     layout_key="PA_BSND", sparse_count=c["K"], key_scale=st["ks"])[0]
    return pkg.lightning_indexer(st["q"], st["k"], st["w"], sparse_count=c["K"], return_value=True,
                                 key_scale=st["ks"])


# ------------------------------------------------------------------------------- what a call cannot do without


def _seen(S, kv, cap):
    """Sum over the S causal rows ending at kv keys of min(keys seen, cap)."""
    return sum(min(kv - S + 1 + t, cap) for t in range(S))


def _pairs(case):
    """(query, key) pairs of an indexer call."""
    c = case
    if c["layout"] == "packed":
        lens = zip(_uneven(c["B"] * c["S"], c["B"], 1), _uneven(c["B"] * c["kv"], c["B"], c["B"] * c["S"]))
        return sum(_seen(s, n, n) for s, n in lens)
    return c["B"] * _seen(c["S"], c["kv"], c["kv"])


def work(case):
    c = case
    kind = c["kind"]
    sz = _SIZE[c.get("dtype", "fp32")]
    if kind == "quant":
        return {"bytes": c["rows"] * (c["n"] * (sz + 1) + 4), "flops": 0}
    if kind == "topk":
        return {"bytes": c["rows"] * (4 * c["n"] + c["k"] * (8 if c["values"] else 4)), "flops": 0}
    if kind == "sfa":
        slots = _seen(c["T"], c["act"], c["topk"]) if c["causal"] else c["T"] * min(c["topk"], c["act"])
        rows = min(slots, c["act"])
        return {"bytes": c["T"] * c["H"] * (576 + 512) * 2 + rows * 1152 + 4 * c["T"] * c["topk"],
                "flops": 2 * c["H"] * 1088 * slots}
    if kind == "mla":
        slots = c["B"] * _seen(c["S"], c["kv"], c["topk"])
        rows = min(slots, c["B"] * c["kv"])
        qo = c["B"] * c["S"] * c["H"]
        return {"bytes": qo * (1088 * 2 + 4) + rows * 1152 + 4 * c["B"] * c["S"] * c["topk"],
                "flops": 2 * c["H"] * 1088 * slots}
    if kind == "gqa":
        slots = c["B"] * c["G"] * _seen(c["S"], c["kv"], c["topk"])
        rows = min(slots, c["B"] * c["G"] * c["kv"])
        qo = c["B"] * c["S"] * c["H"]
        return {"bytes": qo * (256 * 2 + 4) + rows * 256 + 4 * c["B"] * c["G"] * c["S"] * c["topk"],
                "flops": 4 * c["H"] // c["G"] * 128 * slots}
    if kind == "v4":
        ratio = 128 if c["mode"] == "hca" else 4
        lens = [c["kv"] - (c["kv"] - c["S"]) * b // (10 * c["B"]) for b in range(c["B"])]
        keys = rows = 0
        for n in lens:
            own = comp = 0
            for p in range(n - c["S"], n):
                own += min(p, c["win"]) + 1
                if c["mode"] == "hca":
                    comp += (p + 1) // ratio
                elif c["mode"] == "csa":
                    comp += min((p + 1) // ratio, c["K"])
            keys += own + comp
            rows += min(own, c["S"] + c["win"], n) + min(comp, n // ratio)
        qo = c["B"] * c["S"] * c["H"]
        return {"bytes": qo * (1024 * 2 + 4) + rows * 1024 + (4 * c["B"] * c["S"] * c["K"] if c["mode"] == "csa"
                                                             else 0), "flops": 4 * c["H"] * 512 * keys}
    if c["layout"] == "packed":
        T, keys = sum(_uneven(c["B"] * c["S"], c["B"], 1)), sum(_uneven(c["B"] * c["kv"], c["B"], c["B"] * c["S"]))
    else:
        T, keys = c["B"] * c["S"], c["B"] * c["kv"]
    out = T * c["K"] * (4 if c["layout"] == "paged" else 4 + max(2, 4 if c["dtype"] == "fp8" else 2))
    return {"bytes": T * c["H"] * (c["D"] * sz + 4) + keys * (c["D"] * sz + (4 if c["dtype"] == "fp8" else 0)) + out,
            "flops": 2 * c["H"] * c["D"] * _pairs(c)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("quant", "topk"):  # codes, scales and an ordered selection: one right answer
        return "exact"
    if kind == "indexer":
        # Scores a few fp32 roundings apart change places when the heads are summed in another order
        # (heads permuted: up to 4.5e-4 of the positions).  The values stay within the f16 products
        # of the fp8 path (1.6e-4 off the 64-bit scores) or one rounding to 16 bits.
        return {"rel": {"fp8": 6e-4, "bf16": 4e-3, "fp16": 6e-4}[case["dtype"]], "max": 0.03, "differ": 0.002}
    # 16-bit probabilities and outputs, rounded once each: with the index lists reversed the outputs
    # move by up to 3.8e-3 (bf16; the largest by 6e-2) and 2.1e-4 (fp16).
    return {"rel": 1.5e-2, "max": 0.25} if case["dtype"] == "bf16" else {"rel": 1.5e-3, "max": 0.03}


# ------------------------------------------------------------------------------- 64-bit results


def _attend(q, k, v, valid, scale, sink=None):
    """softmax(scale q k^T) v over the valid keys in 64 bits: q [n, H, d], k / v [n, L, *], valid [n, L]."""
    s = torch.bmm(q, k.transpose(1, 2).contiguous()).mul_(scale)
    s.masked_fill_(~valid.unsqueeze(1), -math.inf)
    lse = torch.logsumexp(s, dim=-1)
    if sink is not None:
        lse = torch.logaddexp(lse, sink.view(1, -1))
    ref = torch.where(torch.isinf(lse), torch.zeros_like(lse), lse)
    return torch.bmm(s.sub_(ref.unsqueeze(-1)).exp_(), v.contiguous()), lse


def _gathered(q, pool, rows, valid, scale, dv, sink=None):
    """_attend over pool[rows] in slabs of query rows: q [N, H, d], pool [R, d], rows / valid [N, L]."""
    N, H, _ = q.shape
    out = torch.empty((N, H, dv), dtype=torch.float64, device=q.device)
    lse = torch.empty((N, H), dtype=torch.float64, device=q.device)
    step = max(1, (1 << 27) // (rows.shape[1] * max(pool.shape[1], H)))
    for r in range(0, N, step):
        k = pool[rows[r:r + step].clamp(min=0).long()].double()
        out[r:r + step], lse[r:r + step] = _attend(q[r:r + step].double(), k, k[..., :dv], valid[r:r + step], scale,
                                                   sink)
    return out, lse


def _paged_rows(idx, table, block):
    """Physical rows of positions idx [B, L] behind table [B, blocks]."""
    p = idx.clamp(min=0).long()
    return table.long().gather(1, p // block) * block + p % block


def _exact_mla(st):
    c = st["case"]
    B, S, H, _ = st["q"].shape
    idx = st["idx"].view(B, S * c["topk"])
    if st["table"] is not None:
        rows = _paged_rows(idx, st["table"], c["block"])
    else:
        rows = idx.clamp(min=0).long() + torch.arange(B, device=idx.device).view(B, 1) * c["kv"]
    out, lse = _gathered(st["q"].view(B * S, H, 576), st["kv"].view(-1, 576), rows.view(B * S, -1),
                         idx.view(B * S, -1) >= 0, 576 ** -0.5, 512)
    return out.view(B, S, H, 512), lse.view(B, S, H)


def _exact_sfa(st):
    c = st["case"]
    q = torch.cat((st["q"], st["qr"]), dim=-1)
    pool = torch.cat((st["key"], st["kr"]), dim=-1).view(-1, 576)
    idx = st["idx"].view(1, -1)
    rows = _paged_rows(idx, st["table"], c["block"]).view(c["T"], -1)
    return _gathered(q, pool, rows, idx.view(c["T"], -1) >= 0, 576 ** -0.5, 512)[0]


def _exact_gqa(st):
    c = st["case"]
    B, S, H, G = c["B"], c["S"], c["H"], c["G"]
    outs, lses = [], []
    for b in range(B):
        for h in range(G):
            idx = st["idx"][b, :, h]
            o, l = _gathered(st["q"][b].view(S, G, H // G, 128)[:, h], st["kv"][b, :, h].contiguous(), idx, idx >= 0,
                             128 ** -0.5, 128)
            outs.append(o)
            lses.append(l)
    out = torch.stack(outs).view(B, G, S, H // G, 128).permute(0, 2, 1, 3, 4).reshape(B, S, H, 128)
    return out, torch.stack(lses).view(B, G, S, H // G).permute(0, 2, 1, 3).reshape(B, S, H)


def _exact_v4(st):
    c = st["case"]
    bs, S, win, ratio = c["block"], c["S"], c["win"], st["ratio"]
    ori = st["ori"].view(-1, 512)
    pool = ori if st["cmp"] is None else torch.cat((ori, st["cmp"].view(-1, 512)))
    outs, lses = [], []
    for b, n in enumerate(st["lens"].tolist()):
        pos = torch.arange(n - S, n, device=ori.device).view(-1, 1)
        own = pos - win + torch.arange(win + 1, device=ori.device)
        rows, valid = [_paged_rows(own.view(1, -1), st["obt"][b:b + 1], bs).view(S, -1)], [own >= 0]
        if c["mode"] != "swa":
            if c["mode"] == "hca":
                pick = torch.arange(max(1, n // ratio), device=ori.device).view(1, -1).expand(S, -1)
                ok = pick < (pos + 1) // ratio
            else:
                pick = st["idx"][b * S:(b + 1) * S, 0]
                ok = pick >= 0
            at = _paged_rows(pick.reshape(1, -1), st["cbt"][b:b + 1], bs).view(S, -1)
            rows.append(at + ori.shape[0])
            valid.append(ok)
        o, l = _gathered(st["q"][b * S:(b + 1) * S], pool, torch.cat(rows, 1), torch.cat(valid, 1), 512 ** -0.5, 512,
                         st["sinks"].double())
        outs.append(o)
        lses.append(l)
    return torch.cat(outs), torch.cat(lses)


def _top_scores(q, k, w, ks, K):
    """The K largest 64-bit scores of each causal row: q [S, H, D], k [n, D], w [S, H], ks [n] or None."""
    S, n = q.shape[0], k.shape[0]
    kt = k.double().t().contiguous()
    out = torch.full((S, K), -math.inf, dtype=torch.float64, device=q.device)
    cols = torch.arange(n, device=q.device).view(1, -1)
    step = max(1, (1 << 28) // (n * q.shape[1]))
    for r in range(0, S, step):
        m = min(step, S - r)
        s = (q[r:r + m].double().reshape(-1, q.shape[2]) @ kt).clamp_(min=0).view(m, -1, n)
        s = torch.bmm(w[r:r + m].double().unsqueeze(1), s).squeeze(1)
        if ks is not None:
            s.mul_(ks.double().view(1, -1))
        s.masked_fill_(cols > torch.arange(n - S + r, n - S + r + m, device=q.device).view(-1, 1), -math.inf)
        out[r:r + m, :min(K, n)] = torch.topk(s, min(K, n), dim=1).values
    return out


def _exact_indexer(st):
    c = st["case"]
    if c["layout"] == "packed":
        vals, q0, k0 = [], 0, 0
        for q1, k1 in zip(st["qlen"].tolist(), st["klen"].tolist()):
            ks = None if st["ks"] is None else st["ks"].reshape(-1)[k0:k1]
            vals.append(_top_scores(st["q"][q0:q1], st["k"][k0:k1, 0], st["w"][q0:q1], ks, c["K"]))
            q0, k0 = q1, k1
        return None, torch.cat(vals).unsqueeze(1)
    vals = [_top_scores(st["q"][b], st["k"][b, :, 0], st["w"][b], None if st["ks"] is None else
                        st["ks"].reshape(c["B"], -1)[b], c["K"]) for b in range(c["B"])]
    return None, torch.stack(vals).unsqueeze(2)


def _exact_quant(st):
    c = st["case"]
    x = st["x"].double()
    top = 127.0 if c["out"] == "int8" else 448.0
    s = x.abs().amax(dim=1, keepdim=True).clamp_(min=1e-4) / top
    if c["round_scale"]:
        s = torch.exp2(torch.ceil(torch.log2(s)))
    return (x / s if c["out"] == "fp8" else None), s


def exact(case, seed):
    if case["kind"] == "topk" or case.get("layout") == "paged":  # positions alone
        return None
    st = prepare(case, seed)
    return {"quant": _exact_quant, "sfa": _exact_sfa, "mla": _exact_mla, "gqa": _exact_gqa, "v4": _exact_v4,
            "indexer": _exact_indexer}[case["kind"]](st)
