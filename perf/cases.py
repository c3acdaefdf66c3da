"""What the paged-KV attention is timed on: the calls a serving engine makes of this library, over the range of sizes it
makes them in.

A case is one engine step on the attention side of one or several layers:
  attend    decode rows or verify trees whose Q, K and V rows are ready: the attention of one layer.
  fused     a decode step from the fp32 projection: norm, rotary, append and attention as one call per layer.
  prefill   prompt chunks from the fp32 projection: prep with the append folded in, then the attention, for every layer
            (sliding layers keep rings and save their rows after the attention); decode rows may ride in the same pass.
  slot      a slot checkpoint: every layer's blocks exported to the file's layout, and another slot's imported.

The sequences of a case: `seqs` trees with `rows` rows each (`rows_lo` .. `rows` where prompts differ in length) behind
`lo` .. `hi` cached keys, drawn from `lens`; `riders` more trees of one row. Layers: `full` ones that keep every key in
listed blocks, `sliding` ones with a ring of `window` positions.
"""
import math
import random

import numpy as np
import torch

from espetero_amd import abi, device, host, synth

F16, BF16 = "fp16", "bf16"
_DT = {F16: (abi.ESP_F16, torch.float16), BF16: (abi.ESP_BF16, torch.bfloat16)}
_GATE_WIDTH = 2560      # model width of the head-wise output gate's dots


def _case(kind, heads, dtype, bt, **kw):
    H, Hkv, hd = heads
    c = dict(kind=kind, H=H, Hkv=Hkv, hd=hd, dtype=dtype, bt=bt, full=1, sliding=0, window=0, seqs=1, lo=0, hi=0, rows_lo=0, rows=1,
             riders=0, lens=1, prep="", gate=False)
    c.update(kw)
    return c


def listed():
    named = lambda name, *a, **kw: dict(_case(*a, **kw), name=name)  # noqa: E731
    return [
        # One user, a short conversation: the smallest call, launches and latency.
        named("decode_one", "attend", (32, 4, 128), F16, 16, lo=1024, hi=1024),
        # Sixteen users of one model, contexts from a prompt to a long conversation: the everyday decode batch.
        named("decode_batch", "attend", (32, 4, 128), F16, 16, seqs=16, lo=512, hi=8192, lens=2),
        # A busy server: many short conversations, five query heads per KV head, 64-token blocks, from the projection on.
        named("decode_many", "fused", (40, 8, 128), BF16, 64, seqs=48, lo=60, hi=3000, lens=3, prep="omni"),
        # One period of a sliding / full layer mix (5 : 1) decoding eight long documents.
        named("decode_layers", "fused", (16, 8, 256), F16, 16, seqs=8, lo=12000, hi=16384, lens=4, sliding=5, window=1024, prep="gemma"),
        # Speculative decoding at long context: four draft rows per sequence.
        named("verify_drafts", "attend", (32, 4, 128), F16, 16, seqs=8, lo=32768, hi=32768, rows=4),
        # The 512-dim heads of full-attention layers, few sequences of very different length.
        named("decode_wide_head", "attend", (16, 2, 512), BF16, 16, seqs=5, lo=900, hi=16384, lens=5),
        # A handful of fresh user prompts batched into one pass, ragged lengths, head-wise output gate.
        named("prefill_prompts", "prefill", (32, 4, 128), F16, 16, seqs=6, rows_lo=40, rows=900, lens=6, prep="omni", gate=True),
        # The last 2048-token chunk of an 8192-token document.
        named("prefill_chunk", "prefill", (40, 8, 128), BF16, 16, lo=6144, hi=6144, rows=2048, prep="omni"),
        # One period of the sliding / full mix on prompt chunks of 1024 rows of long documents: the largest step.
        named("prefill_layers", "prefill", (16, 8, 256), F16, 16, seqs=8, lo=15360, hi=15360, rows=1024, sliding=5, window=1024, prep="gemma"),
        # Prompt chunks on the 512-dim heads.
        named("prefill_wide_head", "prefill", (16, 2, 512), F16, 64, seqs=2, lo=3000, hi=7000, rows_lo=700, rows=1024, lens=7, prep="gemma"),
        # Continuous batching: one prompt's chunk and a dozen decoding users in the same pass.
        named("pass_mixed", "prefill", (32, 4, 128), F16, 16, lo=2048, hi=2048, rows=512, riders=12, lens=8, prep="omni"),
        # A conversation is put away and another one taken up again: six layers' blocks, 6000 tokens.
        named("slot_checkpoint", "slot", (16, 8, 256), F16, 64, lo=6000, hi=6000, full=6),
    ]


_HEADS = {128: [(32, 4, 128), (40, 8, 128), (16, 8, 128), (8, 2, 128)], 256: [(16, 8, 256), (8, 2, 256), (24, 4, 256)], 512: [(16, 2, 512)]}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _drawn(rng):
    what = rng.choice(["decode", "decode", "verify", "fused", "fused", "prompts", "chunk", "layers", "mixed", "slot"])
    dtype, bt, lens = rng.choice([F16, BF16]), rng.choice([16, 16, 64]), rng.randrange(1 << 20)
    heads = lambda *hds: rng.choice(_HEADS[rng.choice(hds)])  # noqa: E731
    if what == "decode":
        hi = _log(rng, 200, 32768)
        return _case("attend", heads(128, 128, 256, 512), dtype, bt, seqs=_log(rng, 1, 64), lo=max(1, hi // rng.choice([1, 4, 16])), hi=hi, lens=lens)
    if what == "verify":
        h = heads(128, 128, 256, 512)
        most = {128: 32, 256: 16, 512: 32}[h[2]] * h[1] // h[0]
        hi = _log(rng, 400, 32768)
        return _case("attend", h, dtype, bt, seqs=_log(rng, 1, 16), lo=max(1, hi // rng.choice([1, 8])), hi=hi, rows=rng.randint(2, min(8, most)), lens=lens)
    if what == "fused":
        h = heads(128, 256)
        hi = _log(rng, 200, 16384)
        sliding = rng.choice([0, 5]) if h[2] == 256 else 0
        return _case("fused", h, dtype, bt, seqs=_log(rng, 1, 48), lo=max(1, hi // rng.choice([1, 4, 16])), hi=hi, lens=lens, sliding=sliding,
                     window=1024 if sliding else 0, prep="omni" if h[2] == 128 else rng.choice(["gemma", "qwen35"]) if not sliding else "gemma")
    if what == "prompts":
        h = heads(128, 256, 512)
        hi = _log(rng, 24, 2048)
        return _case("prefill", h, dtype, bt, seqs=_log(rng, 1, 8), rows_lo=max(1, hi // rng.choice([1, 4, 16])), rows=hi, lens=lens,
                     prep="omni" if h[2] == 128 else "gemma", gate=rng.random() < 0.5)
    if what == "chunk":
        h = heads(128, 128, 256, 512)
        rows = _log(rng, 64, 2048)
        P = rng.choice([16 * _log(rng, 1, 1000), _log(rng, 10, 16000)])
        return _case("prefill", h, dtype, bt, lo=P, hi=P, rows=rows, lens=lens,
                     prep="omni" if h[2] == 128 else "gemma" if h[2] == 512 else rng.choice(["gemma", "qwen35"]))
    if what == "layers":
        h = heads(256)
        hi, rows = _log(rng, 500, 16000), _log(rng, 64, 1024)
        return _case("prefill", h, dtype, bt, seqs=rng.randint(1, 8), lo=max(1, hi // rng.choice([1, 4])), hi=hi, rows_lo=max(1, rows // rng.choice([1, 2])),
                     rows=rows, sliding=5, window=1024, lens=lens, prep="gemma")
    if what == "mixed":
        h = heads(128, 256)
        P = _log(rng, 16, 8000)
        return _case("prefill", h, dtype, bt, seqs=rng.randint(1, 2), lo=P, hi=P, rows_lo=64, rows=_log(rng, 64, 1024), riders=_log(rng, 1, 32), lens=lens,
                     prep="omni" if h[2] == 128 else "gemma")
    n = _log(rng, 100, 12000)
    return _case("slot", heads(128, 256), dtype, bt, lo=n, hi=n, full=rng.randint(1, 8), lens=lens)


def draw(rng):
    """One more case of these ranges, no larger than the largest listed one (a drawn full-attention or 512-dim prefill is held to a
    part of it: those run at a lower rate)."""
    most = max(_cost(c) for c in listed())
    while True:
        c = _drawn(rng)
        if _cost(c) <= 0.5 * most:
            return c


def _cost(case):
    w = work(case)
    return w["flops"] / {128: 9e14, 256: 7e14, 512: 5e14}[case["hd"]] + w["bytes"] / 4e12


def _sequences(case):
    """[(cached keys, rows)] of the pass's trees."""
    rng = random.Random(case["lens"])
    out = [(rng.randint(case["lo"], case["hi"]), rng.randint(case["rows_lo"] or case["rows"], case["rows"])) for _ in range(case["seqs"])]
    return out + [(_log(rng, 200, 6000), 1) for _ in range(case["riders"])]


def _pairs(seqs, window):
    """(visible query-key pairs, cached keys some row sees) of one layer. Plain causal rows; verify chains the same."""
    pairs = keys = 0
    for P, M in seqs:
        q = P + np.arange(M, dtype=np.int64)
        n = np.minimum(q + 1, window) if window else q + 1
        pairs += int(n.sum())
        keys += min(P, window - 1) if window else P
    return pairs, keys


def work(case):
    seqs, e = _sequences(case), 2
    H, Hkv, hd = case["H"], case["Hkv"], case["hd"]
    rows = sum(M for _, M in seqs)
    kv = 2 * Hkv * hd * e                                   # bytes of one key and value
    if case["kind"] == "slot":
        blocks = sum(-(-P // case["bt"]) for P, _ in seqs)
        return {"bytes": 2 * 2 * blocks * case["bt"] * kv * case["full"], "flops": 0}
    io = 2 * rows * H * hd * e if case["kind"] == "attend" else rows * (H * (2 if case["prep"] == "qwen35" else 1) + 2 * Hkv) * hd * 4 + rows * H * hd * e
    total = {"bytes": 0, "flops": 0}
    for window, count in ((0, case["full"]), (case["window"], case["sliding"])):
        pairs, keys = _pairs(seqs, window)
        b = io + (keys + rows) * kv                         # cached keys and this pass's own rows, read or written once
        f = 4 * hd * H * pairs
        if case["gate"]:
            b += (rows + H) * _GATE_WIDTH * e
            f += 2 * rows * H * _GATE_WIDTH
        total["bytes"] += count * b
        total["flops"] += count * f
    return total


def tolerance(case):
    """Outputs are stored in 16 bits and every probability is rounded to them before P.V: against float64 on the path's own
    inputs the listed cases read 2.5e-4 to 2.9e-4 (fp16) and 2.1e-3 to 2.4e-3 (bf16), single values up to 2.5e-3 and 1.1e-2;
    four times that."""
    if case["kind"] == "slot":
        return "exact"
    return {"rel": 1.2e-3, "max": 1e-2} if case["dtype"] == F16 else {"rel": 9.5e-3, "max": 4.4e-2}


class _Layer:
    """One layer's share of a step: its pool region, records and buffers, as an engine keeps them."""

    def __init__(self, case, seqs, window, gen):
        H, Hkv, hd, bt = case["H"], case["Hkv"], case["hd"], case["bt"]
        dt, tdt = _DT[case["dtype"]]
        kind = case["kind"]
        n_rows = sum(M for _, M in seqs)
        self.n_rows = n_rows
        ring = -(-window // bt) if window else 0
        per = [ring or -(-(P + M) // bt) for P, M in seqs]
        n_blocks = sum(per)
        scale = 1.0 if case["prep"] == "omni" else hd ** -0.5
        p = synth.make_params(H, Hkv, hd, dt, bt, window=window, ring=ring, scale=scale, rows_per_tile=case["rows"])
        if kind == "prefill":
            p.rows_per_tile = 128
            p.rows_per_tile = device.plan_hint3(p)[2]
        self.p = p
        # Pool: keys as they leave the norm, values half as large; pages in a seeded order.
        self.pool = torch.empty(n_blocks * 2 * bt * Hkv * hd, dtype=tdt, device="cuda").normal_(generator=gen)
        self.pool.view(n_blocks * Hkv, 2, bt * hd)[:, 1] *= 0.5
        order = torch.randperm(n_blocks, generator=gen, device="cuda").cpu().numpy().astype(np.int32)
        trees, pos = np.zeros(len(seqs), abi.TREE_DT), np.zeros((n_rows, 4), np.int32)
        where = np.zeros((n_rows, 2), np.int32)             # (block, position) each row is kept at
        base = used = 0
        for i, ((P, M), nb) in enumerate(zip(seqs, per)):
            trees[i] = (base, P, used, M)
            q = P + np.arange(M)
            pos[base:base + M, :3] = q[:, None]
            where[base:base + M, 0] = used + (q // bt) % ring if ring else order[used + q // bt]
            where[base:base + M, 1] = q % bt
            base += M
            used += nb
        desc = None
        if kind == "attend" and case["rows"] > 1:
            desc = np.concatenate([synth.verify_desc(M, 1) for _, M in seqs])
        resident, groups = device.plan_hint(p)
        tiles, jobs, n_parts = host.plan_tiles(trees, groups, window, pos if window else None, host.options_mi355x(p.rows_per_tile, resident))
        # A full layer's rows can be read from the pool, where the prep has put them, if its 16-row groups are groups there too.
        self.in_pool = kind == "prefill" and not ring and all((P - int(t["base"])) % 16 == 0 for (P, _), t in zip(seqs, trees))
        self.dp = device.DevicePass(p, trees, tiles, jobs, n_parts, n_rows, order, desc, pos, pool_blocks=n_blocks, fused=kind == "fused",
                                    rows_in_pool=self.in_pool)
        make = lambda cols: torch.empty(n_rows, cols, dtype=tdt, device="cuda")  # noqa: E731
        self.O = torch.zeros(n_rows, H * hd, dtype=tdt, device="cuda")
        if kind == "attend":
            self.Q, self.Kb, self.Vb = make(H * hd).normal_(generator=gen), make(Hkv * hd).normal_(generator=gen), make(Hkv * hd).normal_(generator=gen)
            self.Vb *= 0.5
            return
        pp, a = synth.make_prep(case["prep"], H, Hkv, hd, dt, 1, seed=1, bt=bt)
        self.pp = pp
        dev = lambda x: None if x is None else torch.from_numpy(x).cuda()  # noqa: E731
        f32 = dict(dtype=torch.float32, device="cuda")
        self.X = torch.empty(n_rows, pp.x_ld, **f32).normal_(0.0, 1.5, generator=gen)
        self.qn, self.kn = (torch.empty(hd, **f32).normal_(1.0, 0.25, generator=gen) for _ in range(2))
        self.pos, self.inv_freq, self.sel = self.dp.pos, dev(a["inv_freq"]), dev(a["rope_sel"])
        table = np.full((n_rows, 4), -1, np.int32)
        table[:, :2] = where
        self.table = dev(table)
        if case["prep"] == "qwen35":                        # the projection holds a gate beside each query head
            p.gate, p.gate_ld, p.gate_hs, p.gate_off, p.gate_headwise = self.X.data_ptr(), pp.x_ld, 2 * hd, hd, 0
        if kind == "fused":
            return
        self.Q = make(H * hd)
        self.Kb, self.Vb = (None, None) if self.in_pool else (make(Hkv * hd), make(Hkv * hd))
        self.saves = None
        if ring:                                            # the rows the next token can still see join the ring after the attention
            keep = np.concatenate([np.arange(max(0, M - window), M) + int(t["base"]) for (_, M), t in zip(seqs, trees)])
            e = np.zeros(len(keep), abi.KVSAVE_DT)
            e["src_row"], e["block"], e["pos"] = keep, where[keep, 0], where[keep, 1]
            self.saves, self.n_saves, self.table = device.to_dev(e), len(e), None
        self.dots = None
        if case["gate"]:
            g = self.gp = abi.GateParams()
            g.H, g.head_dim, g.D, g.dtype, g.q_ld, g.x_ld = H, hd, _GATE_WIDTH, dt, H * hd, _GATE_WIDTH
            self.xn = make(_GATE_WIDTH).normal_(generator=gen)
            self.Wg = torch.empty(H, _GATE_WIDTH, dtype=tdt, device="cuda").normal_(0.0, 2.0 * _GATE_WIDTH ** -0.5, generator=gen)
            self.dots = torch.empty(n_rows, H, **f32)
            p.gate, p.gate_ld, p.gate_hs, p.gate_off, p.gate_headwise = self.dots.data_ptr(), H, 1, 0, 1

    def fused(self):
        device.decode_fused(self.pp, self.p, self.X, self.qn, self.kn, self.pos, self.inv_freq, self.sel, self.table, self.pool, self.dp, self.O)

    def prefill(self):
        device.attn_prep(self.pp, self.X, self.qn, self.kn, self.pos, self.inv_freq, self.sel, self.Q, self.Kb, self.Vb, self.table,
                         self.pool if self.table is not None else None, self.n_rows)
        if self.dots is not None:
            device.head_gate(self.gp, None, self.xn, self.Wg, self.dots, self.n_rows)
        self.dp.run(self.Q, self.Kb, self.Vb, self.pool, self.O)
        if self.saves is not None:
            device.kv_save(self.p, self.Kb, self.Vb, self.pool, self.saves, self.n_saves)


def _slot_state(case, gen):
    H, Hkv, hd, bt = case["H"], case["Hkv"], case["hd"], case["bt"]
    dt, tdt = _DT[case["dtype"]]
    n = sum(-(-P // bt) for P, _ in _sequences(case))
    block, layers = 2 * bt * Hkv * hd, case["full"]
    order = torch.randperm(2 * n, generator=gen, device="cuda").to(torch.int32)
    params = []
    for layer in range(layers):
        p = synth.make_params(H, Hkv, hd, dt, bt)
        p.kv_base = layer * 2 * n * block
        params.append(p)
    pool = torch.empty(layers * 2 * n * block, dtype=tdt, device="cuda").normal_(generator=gen)
    return dict(kind="slot", n=n, params=params, pool=pool, away=order[:n].contiguous(), back=order[n:].contiguous(),
                file_out=torch.empty(layers, n * block, dtype=tdt, device="cuda"),
                file_in=torch.empty(layers, n * block, dtype=tdt, device="cuda").normal_(generator=gen))


def prepare(case, seed):
    device.init(0)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    if case["kind"] == "slot":
        return _slot_state(case, gen)
    seqs = _sequences(case)
    layers = [_Layer(case, seqs, case["window"], gen) for _ in range(case["sliding"])] + [_Layer(case, seqs, 0, gen) for _ in range(case["full"])]
    return dict(kind=case["kind"], layers=layers)


def run(state):
    if state["kind"] == "slot":
        for p, out, back in zip(state["params"], state["file_out"], state["file_in"]):
            device.kv_export_blocks(p, state["pool"], state["away"], state["n"], out)
            device.kv_import_blocks(p, back, state["back"], state["n"], state["pool"])
        return [state["file_out"], state["pool"]]
    layers = state["layers"]
    if state["kind"] == "attend":
        for lay in layers:
            lay.dp.run(lay.Q, lay.Kb, lay.Vb, lay.pool, lay.O)
        return [lay.O for lay in layers]
    for lay in layers:
        lay.fused() if state["kind"] == "fused" else lay.prefill()
    return [lay.O for lay in layers] + [lay.pool for lay in layers]
