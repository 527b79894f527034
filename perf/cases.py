"""Performance cases of the INT4 weight-only matmul path on one MI355X.

The listed cases are the workloads that the path exists for, through the
public entry points of `cascadia_amd`, at the sizes of this repository's own
benchmark and tests: the decode GEMV and FFN chain, prefill GEMMs, the shell
projections and experts of the group-32 model shapes, sparse-MoE layers from
one token to a 1024-token prefill, and the load-time quantisation.  `draw`
spreads further cases over the same ranges (rows, matrix shapes, group sizes,
scale and activation types, weight layouts, routing).

Every input is made from the seed alone.  Weights are uniform nibbles with
scales |N(0, 0.02)| + 1e-3, activations N(0, 1); MoE routing logits are N(0, 1)
("even") or N(0, 1) with a Zipf(1.1) skew over the experts ("zipf").  Weights
are uploaded once and, except where a case says "crate", converted once to the
MFMA-tiled device layout, as a serving process does at load.
"""
from __future__ import annotations

import math

import torch

import cascadia_amd as cl

DEV = "cuda"
ZIPF = 1.1


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # the smallest call: one 4096 x 4096 GEMV of one f32 token (decode, latency)
        _gemm("gemv_4096_one_token", rows=1, n=4096, k=4096, group=128, scale="f16", x="f32"),
        # prefill of a Llama-3-8B-shaped projection, bf16 in and out: a short
        # prompt over a square matrix, and a long one over the FFN's width
        _gemm("prefill_512_4096", rows=512, n=4096, k=4096, group=128, scale="f16", x="bf16",
              y="bf16"),
        _gemm("prefill_2048_14336", rows=2048, n=14336, k=4096, group=128, scale="f16", x="bf16",
              y="bf16"),
        # a shell projection (o_proj) of the group-32 model over a ragged
        # prompt, f32 activations as that runner holds them
        _gemm("o_proj_f32_333", rows=333, n=7168, k=8192, group=32, scale="bf16", x="f32"),
        # decode FFN of eight layers, one token and a batch of 16, captured
        # once in a graph and replayed per step, as a decode loop runs it
        _ffn("decode_ffn_one_token", tokens=1, hidden=4096, inter=14336, group=128, scale="f16",
             layers=8),
        _ffn("decode_ffn_batch_16", tokens=16, hidden=4096, inter=14336, group=128, scale="f16",
             layers=8),
        # one group-32 expert over the tokens of a mid-sized prompt chunk
        _ffn("expert_g32_200", tokens=200, hidden=7168, inter=2048, group=32, scale="bf16"),
        # a MoE layer of 256 experts, softmax over the top 8, a decode batch of 32
        _moe("moe_256_batch_32", tokens=32, hidden=3072, inter=1536, experts=256, group=128,
             route="softmax", skew="even", shared=0),
        # a MoE layer of 384 experts and a shared one, group 32, skewed
        # routing: one token, a large decode batch, a prefill chunk
        _moe("moe_384_one_token", tokens=1, hidden=7168, inter=2048, experts=384, group=32,
             route="sigmoid", skew="zipf", shared=2048),
        _moe("moe_384_batch_64", tokens=64, hidden=7168, inter=2048, experts=384, group=32,
             route="sigmoid", skew="zipf", shared=2048),
        _moe("moe_384_prefill_1024", tokens=1024, hidden=7168, inter=2048, experts=384, group=32,
             route="sigmoid", skew="zipf", shared=2048),
        # loading: a bf16 matrix of the model shell quantised and tiled
        {"name": "load_quantize_7168", "kind": "load", "n": 7168, "k": 8192, "group": 32},
    ]


def _gemm(name, rows, n, k, group, scale, x, y="f32", layout="tiled"):
    return {"name": name, "kind": "gemm", "rows": rows, "n": n, "k": k, "group": group,
            "scale": scale, "x": x, "y": y, "layout": layout}


def _ffn(name, tokens, hidden, inter, group, scale, layers=1, x="bf16"):
    return {"name": name, "kind": "ffn", "tokens": tokens, "hidden": hidden, "inter": inter,
            "group": group, "scale": scale, "layers": layers, "x": x}


def _moe(name, tokens, hidden, inter, experts, group, route, skew, shared):
    return {"name": name, "kind": "moe", "tokens": tokens, "hidden": hidden, "inter": inter,
            "experts": experts, "group": group, "top_k": 8, "route": route, "skew": skew,
            "shared": shared}


def _log(rng, lo, hi):
    """An integer of [lo, hi], its logarithm uniform."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "ffn", "ffn", "moe", "moe", "load"])
    group = rng.choice([32, 32, 64, 128, 128])
    if kind == "gemm":
        layout = rng.choice(["tiled", "tiled", "tiled", "crate"])
        # (crate-layout weights serve decode and short prompts)
        rows = _log(rng, 1, 2048 if layout == "tiled" else 128)
        x = rng.choice(["f32", "bf16"])
        c = _gemm("", rows, _log(rng, 384, 14336), group * _log(rng, 1024 // group, 14336 // group),
                  group, rng.choice(["bf16", "f16"]), x,
                  rng.choice(["f32", "bf16"]) if x == "bf16" else "f32", layout)
        while c["rows"] * c["n"] * c["k"] > 2048 * 14336 * 4096 // (8 if x == "f32" else 1):
            c["rows"] = (c["rows"] + 1) // 2
    elif kind == "ffn":
        tokens = _log(rng, 1, 1024)
        c = _ffn("", tokens, 128 * _log(rng, 16, 56), 128 * _log(rng, 8, 112), group,
                 rng.choice(["bf16", "f16"]), 4 if tokens <= 16 else 1, rng.choice(["bf16", "f32"]))
        while c["tokens"] * c["hidden"] * c["inter"] > 1024 * 7168 * 3072:
            c["tokens"] = (c["tokens"] + 1) // 2
    elif kind == "moe":
        hidden, inter = 128 * _log(rng, 16, 56), 128 * _log(rng, 6, 16)
        c = _moe("", _log(rng, 1, 1024), hidden, inter, rng.choice([60, 128, 256, 384]), group,
                 rng.choice(["softmax", "sigmoid"]), rng.choice(["even", "zipf"]),
                 rng.choice([0, inter]))
        # no more expert bytes than the largest listed layer reads
        while c["experts"] * 3 * hidden * inter > 130 * 3 * 7168 * 2048:
            c["experts"] //= 2
        c["experts"] = max(16, c["experts"])
    else:
        c = {"name": "", "kind": "load", "n": _log(rng, 384, 7168), "group": group,
             "k": group * _log(rng, 1024 // group, 8192 // group)}
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 13)
    return g


def _bytes(g, n):
    w = torch.randint(-2**31, 2**31 - 1, ((n + 3) // 4,), generator=g, device=DEV,
                      dtype=torch.int32)
    return w.view(torch.uint8)[:n]


def _scales(g, n, kind):
    s = torch.randn(n, generator=g, device=DEV).abs_().mul_(0.02).add_(1e-3)
    return s.to(torch.float16 if kind == "f16" else torch.bfloat16)


def _matrix(g, n, k, group, kind):
    """(packed, scales) of one crate-layout matrix."""
    return _bytes(g, n * k // 2), _scales(g, n * (k // group), kind)


def _sdt(case):
    return cl.SCALE_F16 if case.get("scale", "f16") == "f16" else cl.SCALE_BF16


def _act(g, shape, kind):
    x = torch.randn(shape, generator=g, device=DEV)
    return x if kind == "f32" else x.to(torch.bfloat16)


def _gemm_inputs(case, seed):
    g = _gen(seed)
    w = _matrix(g, case["n"], case["k"], case["group"], case["scale"])
    return w, _act(g, (case["rows"], case["k"]), case["x"])


def _ffn_inputs(case, seed):
    g = _gen(seed)
    h, i, grp = case["hidden"], case["inter"], case["group"]
    w = [[_matrix(g, n, k, grp, case["scale"]) for n, k in ((i, h), (i, h), (h, i))]
         for _ in range(case["layers"])]
    return w, [_act(g, (case["tokens"], h), case["x"]) for _ in range(case["layers"])]


def _flat(mats):
    """One expert's flat blob: gate, up, down, each codes then scales."""
    return torch.cat([t.view(torch.uint8) for m in mats for t in m])


def _moe_inputs(case, seed):
    g = _gen(seed)
    h, i, grp, e = case["hidden"], case["inter"], case["group"], case["experts"]
    per = cl.expert_bytes(h, i, grp)
    stride = (per + 255) // 256 * 256
    blobs = _bytes(g, stride * e)
    mat, sc = i * h // 2, i * (h // grp)
    for at in (mat, 2 * mat + 2 * sc, 3 * mat + 4 * sc):  # gate, up and down scales
        blobs.view(e, stride)[:, at:at + 2 * sc] = _scales(g, e * sc, "f16").view(torch.uint8).view(
            e, 2 * sc)
    shared = None
    if case["shared"]:
        s = case["shared"]
        shared = [_matrix(g, n, k, grp, "f16") for n, k in ((s, h), (s, h), (h, s))]
    x = _act(g, (case["tokens"], h), "bf16").float()  # bf16 activations, held in f32
    residual = _act(g, (case["tokens"], h), "f32")
    logits = _logits(case, g, DEV)
    bias = torch.randn(e, generator=g, device=DEV).mul_(0.01) if case["route"] == "sigmoid" else None
    return blobs, stride, shared, x, residual, logits, bias


def _logits(case, g, device):
    t, e = case["tokens"], case["experts"]
    v = torch.randn((t, e), generator=g, device=device)
    if case["skew"] == "zipf":
        v -= ZIPF * torch.log1p(torch.randperm(e, generator=g, device=device).float())[None, :]
    return v


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------

def prepare(case, seed):
    return {"gemm": _prepare_gemm, "ffn": _prepare_ffn, "moe": _prepare_moe,
            "load": _prepare_load}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_gemm(case, seed):
    (p, s), x = _gemm_inputs(case, seed)
    n, k, grp = case["n"], case["k"], case["group"]
    tiling = cl.TILING_CRATE
    if case["layout"] == "tiled":
        p, s = cl.tile_weights(p, s, n, k, grp)
        tiling = cl.TILING_MFMA
    y = torch.empty((case["rows"], n), device=DEV,
                    dtype=torch.float32 if case["y"] == "f32" else torch.bfloat16)
    return {"run": _run_gemm, "p": p, "s": s, "x": x, "y": y, "n": n, "k": k,
            "rows": case["rows"], "opts": {"group_size": grp, "scale_dtype": _sdt(case),
                                           "tiling": tiling}}


def _run_gemm(st):
    if st["y"].dtype == torch.bfloat16:
        return cl.gemm_int4_bf16(st["p"], st["s"], st["x"], st["n"], st["k"], st["rows"], st["y"],
                                 **st["opts"])
    if st["rows"] == 1 and st["x"].dtype == torch.float32:
        return cl.dequant_gemv_int4(st["p"], st["s"], st["x"], st["n"], st["k"], st["y"],
                                    **st["opts"])
    return cl.dequant_gemm_int4_multi_auto(st["p"], st["s"], st["x"], st["n"], st["k"], st["rows"],
                                           st["y"], **st["opts"])


def _prepare_ffn(case, seed):
    w, xs = _ffn_inputs(case, seed)
    h, i, grp, sdt = case["hidden"], case["inter"], case["group"], _sdt(case)
    layers = [cl.ExpertWeights(_flat(m), h, i, grp, sdt).tiled() for m in w]
    outs = [torch.empty_like(x) for x in xs]
    ws = torch.empty(max(256, cl.ffn_workspace_bytes(h, i, case["tokens"], grp)),
                     dtype=torch.uint8, device=DEV)
    st = {"run": _run_ffn, "layers": layers, "x": xs, "out": outs, "ws": ws,
          "f32": case["x"] == "f32"}
    if case["layers"] == 1:
        return st
    # a decode loop's step: every layer's FFN in one captured graph
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _run_ffn(st)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _run_ffn(st)
    st["run"], st["graph"] = _run_graph, graph
    return st


def _run_ffn(st):
    for w, x, out in zip(st["layers"], st["x"], st["out"]):
        opts = {"group_size": w.group_size, "scale_dtype": w.scale_dtype, "workspace": st["ws"],
                "tiling": w.tiling}
        if st["f32"]:
            cl.ffn_forward_sparse_f32(x, w.hidden, w.inter, *w.slices(), out, 0.0, **opts)
        else:
            cl.expert_forward(x, *w.slices(), out, **opts)
    return st["out"]


def _run_graph(st):
    st["graph"].replay()
    return st["out"]


def _prepare_moe(case, seed):
    blobs, stride, shared, x, residual, logits, bias = _moe_inputs(case, seed)
    h, i, grp, e = case["hidden"], case["inter"], case["group"], case["experts"]
    sh = None
    if shared is not None:
        sh = cl.ExpertWeights(_flat(shared), h, case["shared"], grp, cl.SCALE_F16)
    ex = cl.MoEExperts.from_crate(blobs, e, h, i, grp, cl.SCALE_F16, stride, sh)
    t, k = case["tokens"], case["top_k"]
    ws = torch.empty(cl.moe_workspace_bytes(ex, k, t), dtype=torch.uint8, device=DEV)
    return {"run": _run_moe, "experts": ex, "x": x, "out": torch.empty_like(x),
            "residual": residual, "logits": logits, "bias": bias, "ws": ws, "k": k,
            "mode": cl.ROUTE_SIGMOID_BIAS if case["route"] == "sigmoid" else cl.ROUTE_SOFTMAX_TOPK,
            "scale": _route_scale(case),
            "ids": torch.empty((t, k), dtype=torch.int32, device=DEV),
            "weights": torch.empty((t, k), dtype=torch.float32, device=DEV)}


def _route_scale(case):
    return 2.5 if case["route"] == "sigmoid" else 1.0


def _run_moe(st):
    cl.moe_forward(st["experts"], st["x"], st["out"], top_k=st["k"], logits=st["logits"],
                   bias=st["bias"], mode=st["mode"], scale=st["scale"], residual=st["residual"],
                   ids_out=st["ids"], weights_out=st["weights"], workspace=st["ws"])
    return {"out": st["out"], "ids": st["ids"], "weights": st["weights"]}


def _load_inputs(case, seed):
    g = _gen(seed)
    return torch.randn((case["n"], case["k"]), generator=g, device=DEV).mul_(0.02).to(torch.bfloat16)


def _prepare_load(case, seed):
    return {"run": _run_load, "w": _load_inputs(case, seed), "n": case["n"], "k": case["k"],
            "group": case["group"]}


def _run_load(st):
    p, s = cl.quantize_int4_group(st["w"], st["n"], st["k"], st["group"])
    pt, stl = cl.tile_weights(p, s, st["n"], st["k"], st["group"])
    return {"packed": p, "scales": s, "packed_tiled": pt, "scales_tiled": stl}


# ---------------------------------------------------------------------------
# what one pass cannot do without
# ---------------------------------------------------------------------------

def _mat_bytes(n, k, group):
    return n * k // 2 + n * (k // group) * 2


def _unique_experts(case):
    """Experts that a batch of these routing logits selects, averaged over a few draws."""
    t, e, k, total, reps = case["tokens"], case["experts"], case["top_k"], 0, 4
    for s in range(reps):
        g = torch.Generator()
        g.manual_seed(s)
        total += torch.topk(_logits(case, g, "cpu"), k, dim=1).indices.unique().numel()
    return total / reps


def work(case):
    grp = case["group"]
    if case["kind"] == "gemm":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": _mat_bytes(n, k, grp) + m * k * (4 if case["x"] == "f32" else 2)
                + m * n * (4 if case["y"] == "f32" else 2), "flops": 2 * m * n * k}
    if case["kind"] == "ffn":
        t, h, i = case["tokens"], case["hidden"], case["inter"]
        b = 2 * _mat_bytes(i, h, grp) + _mat_bytes(h, i, grp) + 2 * t * h * (
            4 if case["x"] == "f32" else 2)
        return {"bytes": case["layers"] * b, "flops": case["layers"] * 6 * t * h * i}
    if case["kind"] == "moe":
        t, h, i, k, s = case["tokens"], case["hidden"], case["inter"], case["top_k"], case["shared"]
        per = 2 * _mat_bytes(i, h, grp) + _mat_bytes(h, i, grp)
        b = _unique_experts(case) * per + 3 * t * h * 4 + t * case["experts"] * 4 + t * k * 8
        if s:
            b += 2 * _mat_bytes(s, h, grp) + _mat_bytes(h, s, grp)
        return {"bytes": b, "flops": 6 * t * h * (k * i + s)}
    n, k = case["n"], case["k"]
    return {"bytes": n * k * 2 + 2 * _mat_bytes(n, k, grp), "flops": n * k}


# ---------------------------------------------------------------------------
# what a pass returns, in 64 bits
# ---------------------------------------------------------------------------

def _dequant(p, s, n, k, group):
    """float64 [n, k] of a crate-layout matrix: (nibble - 8) * scale."""
    b = p.view(n, k // 2)
    q = torch.stack((b & 15, b >> 4), dim=2).view(n, k).to(torch.float64).sub_(8.0)
    return q.view(n, k // group, group).mul_(s.view(n, k // group, 1).double()).view(n, k)


def _swiglu64(x, mats, h, i, group):
    """x (float64 [m, h]) through one expert, in 64 bits."""
    g = x @ _dequant(*mats[0], i, h, group).T
    u = x @ _dequant(*mats[1], i, h, group).T
    return (g * torch.sigmoid(g) * u) @ _dequant(*mats[2], h, i, group).T


def exact(case, seed):
    if case["kind"] == "gemm":
        (p, s), x = _gemm_inputs(case, seed)
        return x.double() @ _dequant(p, s, case["n"], case["k"], case["group"]).T
    if case["kind"] == "ffn":
        w, xs = _ffn_inputs(case, seed)
        return [_swiglu64(x.double(), m, case["hidden"], case["inter"], case["group"])
                for m, x in zip(w, xs)]
    if case["kind"] == "load":
        return None  # integers and rounded scales: compared exactly
    return _exact_moe(case, seed)


def _exact_moe(case, seed):
    blobs, stride, shared, x, residual, logits, bias = _moe_inputs(case, seed)
    h, i, grp, k = case["hidden"], case["inter"], case["group"], case["top_k"]
    v = logits.double()
    if case["route"] == "sigmoid":
        sc = torch.sigmoid(v)
        ids = torch.topk(sc + bias.double(), k, dim=1).indices
        w = sc.gather(1, ids)
        w = w / (w.sum(1, keepdim=True) + 1e-20) * _route_scale(case)
    else:
        top = torch.topk(v, k, dim=1)
        ids, w = top.indices, torch.softmax(top.values, dim=1) * _route_scale(case)
    out = residual.double()
    xd = x.double()
    if shared is not None:
        out = out + _swiglu64(xd, shared, h, case["shared"], grp)
    mat, sc2 = i * h // 2, i * (h // grp) * 2
    for e in ids.unique().tolist():
        tok, slot = (ids == e).nonzero(as_tuple=True)
        b = blobs[e * stride:(e + 1) * stride]
        mats = []
        for j in range(3):
            at = j * (mat + sc2)
            mats.append((b[at:at + mat], b[at + mat:at + mat + sc2].view(torch.float16)))
        y = _swiglu64(xd[tok], mats, h, i, grp)
        out.index_add_(0, tok, y * w[tok, slot].unsqueeze(1))
    return {"out": out, "ids": ids.to(torch.int32), "weights": w}


def tolerance(case):
    # 32-bit outputs: f32 sums over activations held as two bf16 planes (about
    # 17 bits); bf16 outputs: their own rounding.  A MoE layer rounds each
    # expert's output to bf16 before the weighted sum; near-ties of the
    # router's scores may select in another order.
    if case["kind"] == "load":
        return "exact"
    if case["kind"] == "moe":
        return {"rel": 6e-3, "differ": 2e-3}
    if case["kind"] == "gemm":
        return {"rel": 2e-5 if case["x"] == "f32" else 5e-6} if case["y"] == "f32" else {
            "rel": 7e-3}
    return {"rel": 4e-5 if case["x"] == "f32" else 7e-3}
