"""The workloads this framework's speed is measured on: one dict per case, made, run and checked
by the functions below.

Kinds of case and what each stands for in a serving process:
  layer    the GPU half of one MoE layer (kt_gguf_hot.moe_layer) on routed tokens: decode windows,
           short prompts and prefill chunks, for every weight type; weights as a slot tensor or
           as a table of slot addresses
  decode   one decode step's hot-expert layers as a server replays them: several layers with
           their own weights in one captured HIP graph
  stream   one layer of streamed prefill (KTStreamPrefillGGUF.run_tensors): the experts' blocks
           come over the host link from pinned banks while groups compute
  gemv     the stand-alone GGUF expert GEMV of a decode window (moe_a8_vec_multi)
  dequant  a group of experts' blocks expanded to bf16 rows (dequant_experts)
  route    the hot registry's lookup and counts for one layer (kt_hot_cache.route_native)

Shapes are those of the package's own workloads (synth.WORKLOADS) and smaller generic ones.
Inputs follow the same recipe: activations ~ N(0, 1), Zipf expert popularity, top-k of
Gumbel-perturbed logits, weights whose codes are distributed as quantised normals.
"""
from __future__ import annotations

import importlib.util
import math
import sys
from pathlib import Path

import torch

_ROOT = Path(__file__).resolve().parent.parent


def _package():
    name = "kt_prefill_lend_amd"
    if name not in sys.modules:
        root = _ROOT / "kt-prefill-lend_amd"
        spec = importlib.util.spec_from_file_location(name, root / "__init__.py", submodule_search_locations=[str(root)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    import kt_prefill_lend_amd.kt_gguf_dequant as DQ
    import kt_prefill_lend_amd.kt_gguf_hot as H
    import kt_prefill_lend_amd.kt_gguf_moe_multi as M
    import kt_prefill_lend_amd.kt_hot_cache as C
    import kt_prefill_lend_amd.kt_stream_prefill as SP

    return H, M, DQ, C, SP


Q8_0, Q4_K, Q6_K, IQ3_S = 8, 12, 14, 21
BLOCK = {Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210), IQ3_S: (256, 110)}  # values, bytes


def _row_bytes(cols, t):
    return cols // BLOCK[t][0] * BLOCK[t][1]


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # a single user's decode step: one token through eight hot-expert layers of a small-expert
        # model, replayed as a graph; launch latency is what counts
        dict(name="decode-1-graph", kind="decode", t13=Q4_K, t2=Q4_K, hidden=2048, inter=512, experts=256, hot=32,
             top_k=8, zipf=1.1, tokens=1, layers=8),
        # a small batch's decode window of a large-expert model, eager
        dict(name="decode-5-large", kind="layer", t13=Q4_K, t2=Q6_K, hidden=7168, inter=2048, experts=256, hot=24,
             top_k=8, zipf=1.1, tokens=5, table=False),
        # a batch's decode window with 3-bit weights, top-10 of 512 experts
        dict(name="decode-13-iq3_s", kind="layer", t13=IQ3_S, t2=IQ3_S, hidden=2048, inter=512, experts=512, hot=48,
             top_k=10, zipf=1.2, tokens=13, table=False),
        # a larger decode batch (or a multi-token verify window) with 8-bit weights, read
        # through the table of slot addresses
        dict(name="window-24-q8_0", kind="layer", t13=Q8_0, t2=Q8_0, hidden=2048, inter=768, experts=128, hot=16,
             top_k=8, zipf=1.1, tokens=24, table=True),
        # a short prompt, or a decode batch of some eighty users
        dict(name="chunk-77", kind="layer", t13=Q4_K, t2=Q6_K, hidden=2048, inter=512, experts=256, hot=40,
             top_k=8, zipf=1.1, tokens=77, table=False),
        # a prompt of ordinary length with 8-bit weights
        dict(name="chunk-512-q8_0", kind="layer", t13=Q8_0, t2=Q8_0, hidden=2048, inter=768, experts=128, hot=16,
             top_k=8, zipf=1.1, tokens=512, table=False),
        # a long prompt's ragged last chunk with 3-bit weights
        dict(name="chunk-2047-iq3_s", kind="layer", t13=IQ3_S, t2=IQ3_S, hidden=2048, inter=512, experts=512, hot=48,
             top_k=10, zipf=1.2, tokens=2047, table=False),
        # a full prefill chunk, the bench's headline shape
        dict(name="prefill-16384", kind="layer", t13=Q4_K, t2=Q6_K, hidden=2048, inter=512, experts=256, hot=40,
             top_k=8, zipf=1.1, tokens=16384, table=False),
        # one streamed layer of a large-expert model: 24 experts over the host link
        dict(name="stream-6144", kind="stream", t13=Q4_K, t2=Q6_K, hidden=7168, inter=2048, experts=24, top_k=8,
             zipf=1.1, tokens=6144),
        # the gate/up GEMV of a decode window as a caller of the bare kernel runs it
        dict(name="gemv-4", kind="gemv", t=Q4_K, rows=1024, cols=2048, experts=32, top_k=8, cold=0.4, tokens=4,
             dtype="bf16"),
        # a streamed group of eight large experts' down weights expanded to bf16
        dict(name="dequant-8-q6_k", kind="dequant", t=Q6_K, rows=7168, cols=2048, n=8),
        # a prefill chunk's lookup in the hot registry
        dict(name="route-16384", kind="route", experts=256, hot=40, top_k=8, zipf=1.1, tokens=16384),
    ]


_TYPES = [(Q8_0, Q8_0), (Q4_K, Q4_K), (Q4_K, Q6_K), (IQ3_S, IQ3_S)]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "layer", "layer", "decode", "stream", "gemv", "dequant", "route"])
    if kind == "stream":
        t13, t2 = rng.choice(_TYPES)
        small = rng.random() < 0.5
        return dict(kind="stream", t13=t13, t2=t2, hidden=2048 if small else 7168, inter=512 if small else 2048,
                    experts=rng.randint(9, 24) if t13 != Q8_0 else rng.randint(5, 12), top_k=rng.choice([4, 8]),
                    zipf=1.1, tokens=_log_int(rng, 512, 6144))
    if kind == "gemv":
        t = rng.choice([Q8_0, Q4_K, Q6_K, IQ3_S])
        rows, cols = rng.choice([(1024, 2048), (2048, 512), (1536, 2048), (2048, 768), (4096, 7168), (7168, 2048)])
        if t != Q8_0 and cols % 256:
            cols = 512
        return dict(kind="gemv", t=t, rows=rows, cols=cols, experts=rng.choice([16, 32, 48]), top_k=rng.choice([4, 8, 10]),
                    cold=round(rng.uniform(0.0, 0.6), 2), tokens=_log_int(rng, 1, 32),
                    dtype=rng.choice(["bf16", "bf16", "f16", "f32"]))
    if kind == "dequant":
        t = rng.choice([Q8_0, Q4_K, Q6_K, IQ3_S])
        rows, cols = rng.choice([(1024, 2048), (2048, 512), (768, 2048), (4096, 7168), (7168, 2048), (2047, 1024)])
        return dict(kind="dequant", t=t, rows=rows, cols=cols, n=rng.randint(1, 8))
    if kind == "route":
        return dict(kind="route", experts=rng.choice([128, 256, 512]), hot=rng.choice([16, 40, 64]),
                    top_k=rng.choice([4, 8, 10]), zipf=1.1, tokens=_log_int(rng, 1, 32768))
    t13, t2 = rng.choice(_TYPES)
    if kind == "decode":
        return dict(kind="decode", t13=t13, t2=t2, hidden=2048, inter=rng.choice([512, 768]), experts=256,
                    hot=rng.choice([24, 32, 40]), top_k=8, zipf=1.1, tokens=rng.randint(1, 32), layers=rng.randint(4, 8))
    size = rng.random()
    hidden, inter = rng.choice([(2048, 512), (2048, 768), (4096, 1024), (7168, 2048)])
    if inter == 2048:
        tokens = _log_int(rng, 1, 6144)
    else:
        tokens = _log_int(rng, 1, 32) if size < 0.35 else _log_int(rng, 33, 600) if size < 0.7 else _log_int(rng, 601, 16384)
    return dict(kind="layer", t13=t13, t2=t2, hidden=hidden, inter=inter, experts=rng.choice([128, 256]),
                hot=rng.randint(12, 48) if inter < 2048 else rng.randint(8, 24), top_k=rng.choice([4, 8, 8, 10]),
                zipf=rng.choice([0.8, 1.1]), tokens=tokens, table=rng.random() < 0.25)


# ---------------------------------------------------------------- inputs

def _gen(seed, *salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + sum((i + 1) * 7919 * int(s) for i, s in enumerate(salt))) % (1 << 62))
    return g


def _codes(g, shape, mid, std, lo, hi):
    """Integer codes of a quantised normal, uint8/int in [lo, hi]."""
    v = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return v.mul_(std).add_(mid).round_().clamp_(lo, hi).to(torch.int16)


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(*v.shape, 2)


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo


def _blocks(g, t, rows, cols):
    """GGUF rows uint8 [rows, row bytes] of values distributed about as N(0, 0.02)."""
    bv, bb = BLOCK[t]
    n = rows * (cols // bv)
    out = torch.empty((n, bb), dtype=torch.uint8, device="cuda")
    if t == Q8_0:
        out[:, :2] = _f16_bytes(_uniform(g, (n,), 3e-4, 6e-4))
        out[:, 2:] = _codes(g, (n, 32), 0.0, 45.0, -127, 127).to(torch.int8).view(torch.uint8)
    elif t == Q4_K:
        sc = torch.randint(24, 64, (n, 8), generator=g, device="cuda", dtype=torch.int16)
        m = (sc + torch.randint(-4, 5, (n, 8), generator=g, device="cuda", dtype=torch.int16)).clamp_(0, 63)
        d = _uniform(g, (n,), 1.2e-4, 1.8e-4)
        out[:, :2] = _f16_bytes(d)
        out[:, 2:4] = _f16_bytes(7.5 * d)
        s = torch.empty((n, 12), dtype=torch.int16, device="cuda")
        s[:, 0:4] = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
        s[:, 4:8] = m[:, :4] | ((m[:, 4:] >> 4) << 6)
        s[:, 8:12] = (sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)
        out[:, 4:16] = s.to(torch.uint8)
        q = _codes(g, (n, 4, 2, 32), 7.5, 3.0, 0, 15)
        out[:, 16:] = (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(n, 128).to(torch.uint8)
    elif t == Q6_K:
        q = _codes(g, (n, 2, 4, 32), 32.0, 11.0, 0, 63)  # [half, run of 32]
        lo = torch.stack([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
        out[:, :128] = lo.reshape(n, 128).to(torch.uint8)
        hi = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
        out[:, 128:192] = hi.reshape(n, 64).to(torch.uint8)
        sc = torch.randint(40, 128, (n, 16), generator=g, device="cuda", dtype=torch.int16)
        neg = torch.rand((n, 16), generator=g, device="cuda") < 0.5
        out[:, 192:208] = torch.where(neg, -sc, sc).to(torch.int8).view(torch.uint8)
        out[:, 208:] = _f16_bytes(_uniform(g, (n,), 1.5e-5, 2.8e-5))
    else:
        out[:] = torch.randint(0, 256, (n, bb), generator=g, device="cuda", dtype=torch.uint8)
        out[:, :2] = _f16_bytes(_uniform(g, (n,), 1.5e-4, 3.0e-4))
    return out.reshape(rows, -1)


def _experts(seed, salt, t, n, rows, cols):
    out = torch.empty((n, rows, _row_bytes(cols, t)), dtype=torch.uint8, device="cuda")
    for e in range(n):
        out[e] = _blocks(_gen(seed, salt, e, t), t, rows, cols)
    return out


def _routing(seed, salt, tokens, experts, top_k, zipf):
    """(ids [T, k] int32 with expert 0 the most popular, weights [T, k] fp32)."""
    g = _gen(seed, salt, 11)
    logp = -zipf * torch.log(torch.arange(1, experts + 1, device="cuda", dtype=torch.float32))
    u = torch.rand((tokens, experts), generator=g, device="cuda").clamp_(1e-9, 1 - 1e-7)
    sel, ids = torch.topk(logp - torch.log(-torch.log(u)), top_k, dim=1)
    return ids.to(torch.int32), torch.softmax(sel, dim=1).to(torch.float32)


def _slots(seed, ids, experts, hot):
    """The slot of each id: the `hot` most popular experts, in a shuffled slot order; else -1."""
    g = _gen(seed, 12)
    table = torch.full((experts,), -1, dtype=torch.int32, device="cuda")
    table[:hot] = torch.randperm(hot, generator=g, device="cuda").to(torch.int32)
    return table[ids.long()]


def _x(seed, salt, tokens, hidden, dtype=torch.bfloat16):
    return torch.randn((tokens, hidden), generator=_gen(seed, salt, 13), device="cuda").to(dtype)


def _layer_inputs(case, seed, li=0):
    S, K, N = case["hot"], case["hidden"], case["inter"]
    ids, w = _routing(seed, 100 * li, case["tokens"], case["experts"], case["top_k"], case["zipf"])
    return dict(x=_x(seed, 100 * li, case["tokens"], K), w=w, slots=_slots(seed + li, ids, case["experts"], S),
                w13=_experts(seed, 100 * li + 1, case["t13"], S, 2 * N, K),
                w2=_experts(seed, 100 * li + 2, case["t2"], S, K, N))


_DTYPE = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _gemv_inputs(case, seed):
    g = _gen(seed, 21)
    T, k, E = case["tokens"], case["top_k"], case["experts"]
    ids = torch.rand((T, E), generator=g, device="cuda").topk(k, dim=1).indices.to(torch.int32)
    ids[torch.rand((T, k), generator=g, device="cuda") < case["cold"]] = -1
    return _x(seed, 22, T, case["cols"], _DTYPE[case["dtype"]]), ids.reshape(-1).contiguous(), _experts(
        seed, 23, case["t"], E, case["rows"], case["cols"])


def _route_inputs(case, seed):
    E = case["experts"]
    perm = torch.randperm(E, generator=_gen(seed, 32), device="cuda")
    ids, _ = _routing(seed, 31, case["tokens"], E, case["top_k"], case["zipf"])
    slot = torch.full((E,), -1, dtype=torch.int32, device="cuda")
    slot[perm[: case["hot"]]] = torch.arange(case["hot"], dtype=torch.int32, device="cuda")
    cpu = torch.where(slot >= 0, -1, torch.arange(E, dtype=torch.int32, device="cuda")).to(torch.int32)
    return perm[ids.long()].to(torch.int32), slot, cpu


# ---------------------------------------------------------------- prepare and run

def _table(t):
    """The slots' addresses as the pointer-table form of the weights takes them."""
    stride = t.stride(0) * t.element_size()
    return torch.tensor([t.data_ptr() + s * stride for s in range(t.shape[0])], dtype=torch.int64, device="cuda")


def _desc(H, case, a, table):
    w13, w2 = (_table(a["w13"]), _table(a["w2"])) if table else (a["w13"], a["w2"])
    return H.layer_desc(w13, w2, case["hidden"], case["inter"], case["t13"], case["t2"], table), (w13, w2)


def prepare(case, seed):
    H, M, DQ, C, SP = _package()
    kind = case["kind"]
    if kind == "layer":
        a = _layer_inputs(case, seed)
        desc, keep = _desc(H, case, a, case["table"])
        return dict(kind=kind, H=H, desc=desc, keep=(keep, a), x=a["x"], w=a["w"], slots=a["slots"])
    if kind == "decode":
        layers = []
        for li in range(case["layers"]):
            a = _layer_inputs(case, seed, li)
            layers.append((_desc(H, case, a, False)[0], a))

        def step():
            return [H.moe_layer(d, a["x"], a["w"], a["slots"]) for d, a in layers]

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outs = step()
        return dict(kind=kind, graph=graph, outs=outs, keep=layers)
    if kind == "stream":
        E, K, N = case["experts"], case["hidden"], case["inter"]
        types = (case["t13"], case["t13"], case["t2"])
        st = SP.KTStreamPrefillGGUF.standalone(N, K, case["top_k"], types, device=torch.device("cuda", 0))
        bank = SP.Bank.pinned(E, SP.part_bytes(types, N, K), types)
        for e in range(E):
            w13 = _blocks(_gen(seed, 1, e, case["t13"]), case["t13"], 2 * N, K)
            bank.gate[e].copy_(w13[:N].reshape(-1))
            bank.up[e].copy_(w13[N:].reshape(-1))
            bank.down[e].copy_(_blocks(_gen(seed, 2, e, case["t2"]), case["t2"], K, N).reshape(-1))
        st.set_bank(0, bank)
        ids, w = _routing(seed, 0, case["tokens"], E, case["top_k"], case["zipf"])
        return dict(kind=kind, st=st, x=_x(seed, 0, case["tokens"], K), w=w, ids=ids)
    if kind == "gemv":
        x, ids, w = _gemv_inputs(case, seed)
        return dict(kind=kind, M=M, x=x, ids=ids, w=w, case=case)
    if kind == "dequant":
        raw = _experts(seed, 41, case["t"], case["n"], case["rows"], case["cols"]).reshape(case["n"], -1)
        pad = -raw.shape[1] % 16  # the entry point's expert stride
        raw = torch.nn.functional.pad(raw, (0, pad)).contiguous()
        out = torch.empty((case["n"], case["rows"], case["cols"]), dtype=torch.bfloat16, device="cuda")
        return dict(kind=kind, DQ=DQ, raw=raw, out=out, case=case)
    ids, slot, cpu = _route_inputs(case, seed)
    counts = torch.zeros((case["experts"],), dtype=torch.float32, device="cuda")
    return dict(kind=kind, C=C, ids=ids, slot=slot, cpu=cpu, counts=counts)


def run(state):
    kind = state["kind"]
    if kind == "layer":
        return state["H"].moe_layer(state["desc"], state["x"], state["w"], state["slots"])
    if kind == "decode":
        state["graph"].replay()
        return state["outs"]
    if kind == "stream":
        return state["st"].run_tensors(0, state["x"], state["w"], state["ids"])
    if kind == "gemv":
        c = state["case"]
        return state["M"].moe_a8_vec_multi(state["x"], state["w"], state["ids"], c["top_k"], c["t"], c["rows"], c["tokens"])
    if kind == "dequant":
        c, raw = state["case"], state["raw"]
        state["DQ"].dequant_experts(raw, raw.stride(0), c["t"], c["n"], c["rows"], c["cols"], state["out"])
        return state["out"]
    state["counts"].zero_()  # the counts of this call alone, so that every pass returns the same
    slot_ids, cpu_ids = state["C"].route_native(state["ids"], state["slot"], state["cpu"], state["counts"])
    return slot_ids, cpu_ids, state["counts"]


# ---------------------------------------------------------------- work and tolerance

def _expected_routes(case, hot):
    """(expected routes to the hot experts, expected distinct hot experts) of one call: each
    token takes top_k of the experts, the r-th most popular with a chance that grows as r^-zipf
    (capped at 1: the top-k of a token are distinct)."""
    E, k, T = case["experts"], case["top_k"], case["tokens"]
    p = [r ** -case["zipf"] for r in range(1, E + 1)]
    lo, hi = 0.0, 1e6  # inclusion of expert r: 1 - exp(-lam p_r), lam so that they sum to k
    for _ in range(60):
        mid = (lo + hi) / 2
        lo, hi = (mid, hi) if sum(1 - math.exp(-mid * v) for v in p) < k else (lo, mid)
    inc = [1 - math.exp(-lo * v) for v in p]
    return T * sum(inc[:hot]), sum(1 - (1 - v) ** T for v in inc[:hot])


def work(case):
    kind, T = case["kind"], case.get("tokens", 0)
    if kind in ("layer", "decode"):
        K, N = case["hidden"], case["inter"]
        routes, used = _expected_routes(case, case["hot"])
        per = 2 * N * _row_bytes(K, case["t13"]) + K * _row_bytes(N, case["t2"])
        n = case.get("layers", 1)
        return {"bytes": n * (used * per + 4 * T * K + 8 * T * case["top_k"]), "flops": n * 6.0 * K * N * routes}
    if kind == "stream":  # the experts' bytes out of host memory once, x in and y out
        K, N = case["hidden"], case["inter"]
        per = 2 * N * _row_bytes(K, case["t13"]) + K * _row_bytes(N, case["t2"])
        return {"bytes": case["experts"] * per + 4 * T * K, "flops": 6.0 * K * N * T * case["top_k"]}
    if kind == "gemv":
        hot = T * case["top_k"] * (1 - case["cold"])
        used = case["experts"] * (1 - (1 - 1 / case["experts"]) ** hot)
        size = 4 if case["dtype"] == "f32" else 2
        return {"bytes": used * case["rows"] * _row_bytes(case["cols"], case["t"])
                + size * T * (case["cols"] + case["top_k"] * case["rows"]), "flops": 2.0 * hot * case["rows"] * case["cols"]}
    if kind == "dequant":
        return {"bytes": case["n"] * case["rows"] * (_row_bytes(case["cols"], case["t"]) + 2 * case["cols"]), "flops": 0}
    return {"bytes": 12 * T * case["top_k"] + 12 * case["experts"], "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind in ("dequant", "route"):
        return "exact"  # single roundings of exact products; whole numbers
    if kind == "gemv":  # fp32 sums of the same int8 products, one rounding to the output type
        return {"rel": {"bf16": 7e-3, "f16": 1e-3, "f32": 4e-6}[case["dtype"]], "max": {"bf16": 3e-2, "f16": 4e-3, "f32": 1e-3}[case["dtype"]]}
    # against 64 bits a decode window is off by 1.3e-2 where its activations are quantised to 8
    # bits (the GGUF GEMV's numerics) and by 4.7e-3 with bf16 operands, as every longer chunk
    window = kind != "stream" and case["tokens"] * case["top_k"] <= 256
    return {"rel": 2.5e-2 if window else 1.8e-2, "max": 0.5 if window else 0.25}


# ---------------------------------------------------------------- the same in 64 bits

def _iq3s_grid():
    """The 512 codebook entries of the IQ3_S format, four magnitudes each."""
    text = (_ROOT / "kt-prefill-lend_amd" / "csrc" / "iq3s_grid.inc").read_text()
    v = [int(w, 16) for w in text.replace(",", " ").replace("u", " ").split() if w.startswith("0x")]
    assert len(v) == 512
    g = torch.tensor(v, dtype=torch.int64, device="cuda")
    return torch.stack([(g >> (8 * i)) & 255 for i in range(4)], 1).to(torch.float64)


def _values(t, rows, cols):
    """The dequantised values of GGUF rows uint8 [n, row bytes], fp64 [n, cols]."""
    bv, bb = BLOCK[t]
    b = rows.reshape(-1, bb)
    n = b.shape[0]

    def f16(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).to(torch.float64)  # [n, 1]

    if t == Q8_0:
        v = f16(0) * b[:, 2:].contiguous().view(torch.int8).to(torch.float64)
    elif t == Q4_K:
        s = b[:, 4:16].to(torch.int32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).to(torch.float64)
        m = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).to(torch.float64)
        q = b[:, 16:].reshape(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32).to(torch.float64)
        v = (f16(0) * sc)[:, :, None] * q - (f16(2) * m)[:, :, None]
    elif t == Q6_K:
        ql, qh = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)
        hi = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (lo | (hi << 4)).to(torch.float64) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).to(torch.float64)
        v = (f16(208) * sc)[:, :, None] * q.reshape(n, 16, 16)
    else:
        qh = b[:, 66:74].to(torch.int64)
        idx = b[:, 2:66].reshape(n, 8, 8).to(torch.int64) | torch.stack([((qh >> k) & 1) << 8 for k in range(8)], 2)
        sg = b[:, 74:106].reshape(n, 8, 4, 1).to(torch.int64) >> torch.arange(8, device="cuda")
        sign = 1.0 - 2.0 * (sg & 1).reshape(n, 8, 32).to(torch.float64)
        s = b[:, 106:110].reshape(n, 4, 1).to(torch.int64)
        nib = torch.cat([s & 15, s >> 4], 2).reshape(n, 8).to(torch.float64)
        v = (f16(0) * (1 + 2 * nib))[:, :, None] * _iq3s_grid()[idx].reshape(n, 8, 32) * sign
    return v.reshape(rows.shape[0], cols)


def _ffn(x, w, slots, n, weights):
    """sum over k of w[t, k] * FFN of expert slots[t, k], fp64; weights(e) -> (w13, w2)."""
    y = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
    xd = x.to(torch.float64)
    for e in range(n):
        tok, k = (slots == e).nonzero(as_tuple=True)
        if not tok.numel():
            continue
        w13, w2 = weights(e)
        N = w2.shape[1]
        h = xd[tok] @ w13.t().contiguous()
        h = torch.nn.functional.silu(h[:, :N]) * h[:, N:]
        y.index_add_(0, tok, (h @ w2.t().contiguous()) * w[tok, k].to(torch.float64)[:, None])
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind in ("layer", "decode"):
        K, N = case["hidden"], case["inter"]
        outs = []
        for li in range(case.get("layers", 1)):
            a = _layer_inputs(case, seed, li)
            outs.append(_ffn(a["x"], a["w"], a["slots"], case["hot"],
                             lambda e, a=a: (_values(case["t13"], a["w13"][e], K), _values(case["t2"], a["w2"][e], N))))
        return outs if kind == "decode" else outs[0]
    if kind == "stream":
        K, N = case["hidden"], case["inter"]
        ids, w = _routing(seed, 0, case["tokens"], case["experts"], case["top_k"], case["zipf"])
        return _ffn(_x(seed, 0, case["tokens"], K), w, ids, case["experts"], lambda e: (
            _values(case["t13"], _blocks(_gen(seed, 1, e, case["t13"]), case["t13"], 2 * N, K), K),
            _values(case["t2"], _blocks(_gen(seed, 2, e, case["t2"]), case["t2"], K, N), N)))
    if kind == "gemv":
        # the operation is defined on q8_1 activations: per 32 values d = max|x| / 127 in fp32
        # (kept as fp16), q = x / d rounded half away from zero
        x, ids, w = _gemv_inputs(case, seed)
        xb = x.to(torch.float32).reshape(x.shape[0], -1, 32)
        d = xb.abs().amax(2, keepdim=True) / 127.0
        r = torch.where(d > 0, xb / d, torch.zeros_like(xb))
        q = torch.sign(r) * torch.floor(r.abs() + 0.5)
        xq = (q.to(torch.float64) * d.to(torch.float16).to(torch.float64)).reshape(x.shape)
        y = torch.zeros((ids.numel(), case["rows"]), dtype=torch.float64, device="cuda")
        for e in torch.unique(ids[ids >= 0]).tolist():
            p = (ids == e).nonzero().squeeze(1)
            y[p] = xq[p // case["top_k"]] @ _values(case["t"], w[e], case["cols"]).t().contiguous()
        return y
    if kind == "dequant":
        raw = _experts(seed, 41, case["t"], case["n"], case["rows"], case["cols"])
        return torch.stack([_values(case["t"], raw[e], case["cols"]) for e in range(case["n"])])
    ids, slot, cpu = _route_inputs(case, seed)
    counts = torch.bincount(ids.reshape(-1).long(), minlength=case["experts"]).to(torch.float64)
    return slot[ids.long()], cpu[ids.long()], counts
