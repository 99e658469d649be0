"""Workloads of the verify path, from its smallest calls to its largest, each through the public
entry points of ds41_gfx950 as a serving program makes them.

Families (`case["path"]`):
  experts  the component kernel API over a list of expert jobs, in the order an engine calls it:
           MXFP8 of the gathered rows, gate, up, SwiGLU times the route weight, MXFP8, down. At most 8
           rows a job through the decode projections, up to 256 through the chunked (prefill) ones.
  shared   the checkpoint's FP8 W8A8 shared expert through the dense calls.
  layer    one verify MoE layer (router, plan, routed experts, shared expert) of 1..8 rows.
  stack    a verify step through several layers with the caller's route ids.
  drafter  the MTP drafter's routed-expert service.
  prefill  one MoE layer over a chunk of tokens.
  accept   draft sampling and rejection sampling from logits.
  measures rejection sampling from fp32 measures.

Weights are uniform e2m1 codes with e8m0 scales of 2^-8..2^-4, activations bf16 N(0, 1), logits
N(0, 2.5^2) with drafts at N(0, 0.5^2) around them, routes of a chunk Zipf(1.1) over the experts.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.abspath("deepseek-v4.1-flash-pro6000_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import ds41_gfx950 as G  # noqa: E402

DEV = "cuda"
LIMIT = 10.0   # SwiGLU clamp of the model
SCALE = 1.5    # route scale of the model
NAMES = ("gate", "gate_scale", "up", "up_scale", "down", "down_scale")


def listed():
    return [
        # one small expert, one token: six launches, nothing but latency
        dict(name="expert_1row", path="experts", hidden=1024, inter=512, jobs=1, rows=1, chunked=False),
        # the routed experts of a T=4 verify step, called job by job as an engine without the fused layer does
        dict(name="experts_decode", path="experts", hidden=4096, inter=2880, jobs=23, rows=2, chunked=False),
        # a batch of a prefill sweep: few experts, many and uneven rows each
        dict(name="experts_chunked", path="experts", hidden=4096, inter=2880, jobs=8, rows=256, chunked=True),
        # the shared expert of a checkpoint at the verify width
        dict(name="shared_fp8", path="shared", hidden=4096, inter=2880, rows=4),
        # plain decode (no drafts) with the checkpoint's FP8 shared expert
        dict(name="layer_1row_fp8", path="layer", hidden=4096, inter=2880, experts=384, topk=6, rows=1, tiled=True, shared="fp8"),
        # the verify width the model serves with: 1 committed + 3 drafts
        dict(name="layer_4rows", path="layer", hidden=4096, inter=2880, experts=384, topk=6, rows=4, tiled=True, shared="mxfp4"),
        # the widest verify step, weights as the checkpoint has them
        dict(name="layer_8rows_rowmajor", path="layer", hidden=4096, inter=2880, experts=384, topk=6, rows=8, tiled=False, shared="mxfp4"),
        # a verify step whose routes the engine has already: layer after layer in one call (two, as the
        # 8-bit activation codes between layers turn single roundings into whole code steps, more each layer)
        dict(name="stack_4rows", path="stack", hidden=4096, inter=2880, experts=384, topk=6, rows=4, layers=2),
        # one stage of the MTP drafter
        dict(name="drafter_5rows", path="drafter", hidden=5120, inter=2304, rows=5),
        # one layer of a prefill chunk
        dict(name="prefill_512", path="prefill", hidden=4096, inter=2880, experts=384, topk=6, tokens=512),
        # a sampling step: 3 drafts drawn, then verified, nucleus 0.95
        dict(name="accept_top_p", path="accept", vocab=129280, drafts=3, temperature=1.0, top_p=0.95),
        # the same decisions from fp32 measures
        dict(name="measures", path="measures", vocab=129280, drafts=3, greedy=False),
    ]


#: hidden and intermediate sizes: the target's, the drafter's, and smaller and ragged ones
SIZES = ((4096, 2880), (5120, 2304), (2048, 1408), (2560, 1056), (1024, 512), (512, 256))
VOCABS = (129280, 32000, 50257, 151936, 100003)


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(("experts", "experts", "experts", "shared", "layer", "layer", "stack", "drafter", "prefill", "prefill", "accept", "accept",
                       "measures"))
    hidden, inter = rng.choice(SIZES)
    if path == "experts":
        chunked = rng.random() < 0.5
        return dict(path=path, hidden=hidden, inter=inter, jobs=_log(rng, 1, 32), rows=_log(rng, 9, 256) if chunked else rng.randint(1, 8),
                    chunked=chunked)
    if path == "shared":
        return dict(path=path, hidden=hidden, inter=inter, rows=rng.randint(1, 8))
    if path == "layer":
        return dict(path=path, hidden=hidden, inter=inter, experts=rng.choice((96, 128, 256, 384)), topk=rng.choice((4, 6, 8)),
                    rows=rng.randint(1, 8), tiled=rng.random() < 0.6, shared=rng.choice(("mxfp4", "mxfp4", "fp8")))
    if path == "stack":
        return dict(path=path, hidden=hidden, inter=inter, experts=rng.choice((128, 256)), topk=6, rows=rng.randint(1, 8), layers=2)
    if path == "drafter":
        hidden, inter = rng.choice(((5120, 2304), (2048, 1408), (1024, 512)))
        return dict(path=path, hidden=hidden, inter=inter, rows=rng.randint(1, 8))
    if path == "prefill":
        return dict(path=path, hidden=hidden, inter=inter, experts=rng.choice((96, 128, 256, 384)), topk=rng.choice((4, 6)),
                    tokens=_log(rng, 12, 512))
    vocab, drafts = rng.choice(VOCABS + (rng.randint(20000, 160000),)), rng.randint(1, 5)
    if path == "accept":
        greedy = rng.random() < 0.2
        return dict(path=path, vocab=vocab, drafts=drafts, temperature=0.0 if greedy else rng.choice((0.6, 1.0)),
                    top_p=1.0 if greedy else rng.choice((1.0, 0.95, 0.9)))
    return dict(path=path, vocab=vocab, drafts=drafts, greedy=rng.random() < 0.2)


# ---- inputs, from the seed alone -----------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _bytes(g, *shape):
    """Uniform bytes (two uniform e2m1 codes each)."""
    n = math.prod(shape)
    t = torch.empty((n + 3) // 4, dtype=torch.int32, device=DEV)
    t.random_(-2**31, 2**31, generator=g)
    return t.view(torch.uint8)[:n].view(*shape)


def _scales(g, *shape):
    return torch.empty(shape, dtype=torch.uint8, device=DEV).random_(119, 124, generator=g)


def _experts(g, count, H, I, down=0):
    """MXFP4 experts as [count] stacks of their six tensors; down scales times 2^-down."""
    return dict(gate=_bytes(g, count, I, H // 2), gate_scale=_scales(g, count, I, H // 32),
                up=_bytes(g, count, I, H // 2), up_scale=_scales(g, count, I, H // 32),
                down=_bytes(g, count, H, I // 2), down_scale=_scales(g, count, H, I // 32) - down)


def _fp8_expert(g, H, I):
    """An FP8 W8A8 expert: finite E4M3 codes of |v| < 2, one E8M0 scale per 32 x 32 block."""
    def w(n, k):
        c = _bytes(g, n, k)
        return (c & 0x80) | ((c & 0x7F) % 0x40)
    def s(n, k):
        return torch.empty((n // 32, k // 32), dtype=torch.uint8, device=DEV).random_(119, 124, generator=g)
    return dict(gate=w(I, H), gate_scale=s(I, H), up=w(I, H), up_scale=s(I, H), down=w(H, I), down_scale=s(H, I))


def _rows(g, n, H):
    return torch.randn((n, H), generator=g, device=DEV).to(torch.bfloat16)


def _job_rows(case):
    """Rows of each job: the most for the first, falling off with the rank (at least 1)."""
    return [max(1, round(case["rows"] / (1 + j / 2))) for j in range(case["jobs"])]


def _zipf(rng, tokens, experts, topk):
    """topk distinct experts per token from Zipf(1.1) over a permutation of the experts."""
    perm = rng.permutation(experts)
    keys = -1.1 * np.log(np.arange(1, experts + 1)) + rng.gumbel(size=(tokens, experts))
    return perm[np.argsort(-keys, axis=1)[:, :topk]].astype(np.int32)


def _route_weights(g, n, k):
    w = torch.rand((n, k), generator=g, device=DEV) + 0.1
    return w / w.sum(1, keepdim=True) * SCALE


def _router(g, E, H):
    return torch.randn((E, H), generator=g, device=DEV) * 0.02, torch.zeros(E, device=DEV)


def _logits(case, seed):
    g = _gen(seed)
    k, V = case["drafts"], case["vocab"]
    target = torch.randn((k + 1, V), generator=g, device=DEV) * 2.5
    return target, target[:k] + torch.randn((k, V), generator=g, device=DEV) * 0.5


def _inputs(case, seed):
    g, H, I = _gen(seed), case["hidden"], case["inter"]
    path = case["path"]
    if path == "experts":
        rows = _job_rows(case)
        return dict(P=_experts(g, case["jobs"], H, I), x=_rows(g, sum(rows), H), w=torch.rand(sum(rows), generator=g, device=DEV) * 0.5 + 0.05)
    if path == "shared":
        return dict(S=_fp8_expert(g, H, I), x=_rows(g, case["rows"], H))
    if path == "layer":
        E = case["experts"]
        wg, bias = _router(g, E, H)
        fp8 = case["shared"] == "fp8"
        return dict(P=_experts(g, E + (not fp8), H, I), S=_fp8_expert(g, H, I) if fp8 else None, wg=wg, bias=bias, x=_rows(g, case["rows"], H))
    if path == "stack":
        E, L = case["experts"], case["layers"]
        rng = np.random.default_rng(seed)
        # smaller down scales: a layer's output, the next one's input, keeps its own input's magnitude
        layers = [(_experts(g, E + 1, H, I, 7), *_router(g, E, H)) for _ in range(L)]
        ids = np.stack([_zipf(rng, case["rows"], E, case["topk"]) for _ in range(L)])
        return dict(layers=layers, ids=torch.from_numpy(ids).to(DEV), x=_rows(g, case["rows"], H))
    if path == "drafter":
        scores = torch.rand((case["rows"], 128), generator=g, device=DEV)
        return dict(P=_experts(g, 128, H, I), ids=scores.topk(3, dim=1).indices.to(torch.int32).contiguous(),
                    w=torch.rand((case["rows"], 3), generator=g, device=DEV) + 0.1, x=_rows(g, case["rows"], H))
    assert path == "prefill"
    E, T, K = case["experts"], case["tokens"], case["topk"]
    ids = _zipf(np.random.default_rng(seed), T, E, K)
    return dict(P=_experts(g, E + 1, H, I), ids=torch.from_numpy(ids).to(DEV), w=_route_weights(g, T, K), x=_rows(g, T, H))


def _table(P):
    n = P["gate"].shape[0]
    return G.device_table([{k: P[k][e] for k in NAMES} for e in range(n)], DEV)[0]


# ---- one pass ------------------------------------------------------------------------------
def prepare(case, seed):
    path = case["path"]
    if path == "accept":
        k, V = case["drafts"], case["vocab"]
        target, draft = _logits(case, seed)
        return dict(case=case, target=target, draft=draft, proposals=torch.empty(k, dtype=torch.int32, device=DEV), seed=seed,
                    result=torch.zeros(40, dtype=torch.uint8, device=DEV), ws=G.accept_workspace(k, V), sws=G.sample_workspace(k, V))
    if path == "measures":
        k, V = case["drafts"], case["vocab"]
        target, draft = _logits(case, seed)
        p, q = torch.softmax(target, 1), torch.softmax(draft, 1)
        d = p[:k].argmax(1) if case["greedy"] else torch.multinomial(q, 1, generator=_gen(seed + 1))[:, 0]
        return dict(case=case, p=p.contiguous(), q=q.contiguous(), drafts=d.to(torch.int32), seed=seed,
                    result=torch.zeros(40, dtype=torch.uint8, device=DEV))
    s, H, I = _inputs(case, seed), case["hidden"], case["inter"]
    s["case"] = case
    def empty(*shape, dtype=torch.bfloat16):
        return torch.empty(shape, dtype=dtype, device=DEV)
    if path == "experts":
        R, ng = s["x"].shape[0], H // 32
        s.update(table=_table(s["P"]), xq=empty(R, H, dtype=torch.uint8), xs=empty(R, ng, dtype=torch.uint8), gate=empty(R, I), up=empty(R, I),
                 h=empty(R, I), hq=empty(R, I, dtype=torch.uint8), hs=empty(R, I // 32, dtype=torch.uint8), y=empty(R, H))
        jobs, at = dict(gate=[], up=[], down=[]), 0
        for j, n in enumerate(_job_rows(case)):
            r = slice(at, at + n)
            jobs["gate"].append((j, n, s["xq"][r], s["xs"][r], s["gate"][r]))
            jobs["up"].append((j, n, s["xq"][r], s["xs"][r], s["up"][r]))
            jobs["down"].append((j, n, s["hq"][r], s["hs"][r], s["y"][r]))
            at += n
        s["jobs"] = {k: G.device_jobs(v, DEV) for k, v in jobs.items()}
    elif path == "layer":
        T, E, K, fp8 = case["rows"], case["experts"], case["topk"], case["shared"] == "fp8"
        s.update(table=_table(s["P"]), y=empty(T, H), ids=empty(T, K, dtype=torch.int32), w=empty(T, K, dtype=torch.float32),
                 ws=torch.zeros(G.layer_workspace_bytes(T, H, I, E, K), dtype=torch.uint8, device=DEV))
        s["args"] = G.make_layer_args(s["x"], s["wg"], s["bias"], s["table"], 0, -1 if fp8 else E, T, H, I, E, K, s["y"], s["ws"],
                                      ids_out=s["ids"], weights_out=s["w"])
        s["args"].weight_layout = 1 if case["tiled"] else 0
        if fp8:
            s["fp8"] = G.fp8_expert(s["S"])
            s["args"].shared_fp8 = ctypes.addressof(s["fp8"])
    elif path == "stack":
        T, E, L, K = case["rows"], case["experts"], case["layers"], case["topk"]
        s["tables"] = [_table(P) for P, _, _ in s["layers"]]
        s["stack"] = G.VerifyStack([dict(router_w=wg, router_bias=b, table=t, shared_index=E) for (_, wg, b), t in zip(s["layers"], s["tables"])],
                                   8, H, I, E, K, weight_layout=1)
        s.update(y=empty(T, H), out=empty(L - 1, T, H), w=empty(L, T, K, dtype=torch.float32), ids_out=empty(L, T, K, dtype=torch.int32))
    elif path == "drafter":
        s.update(table=_table(s["P"]), y=empty(case["rows"], 3, H))
        s["service"] = G.TargetExperts(s["table"], 0, H, I, weight_layout=1)
    elif path == "prefill":
        T, E, K = case["tokens"], case["experts"], case["topk"]
        s.update(table=_table(s["P"]), y=empty(T, H), ws=torch.zeros(G.prefill_workspace_bytes(T, H, I, E, K), dtype=torch.uint8, device=DEV))
        s["args"] = G.make_prefill_args(s["x"], s["ids"], s["w"], s["table"], 0, E, T, H, I, E, K, s["y"], s["ws"])
    return s


def _quantize(x, q, s, stream):
    G.check(G.lib().ds41_quantize_mxfp8(G._p(x), G._p(q), G._p(s), x.shape[0], x.shape[1], stream), "quantize_mxfp8")


def run(s):
    case = s["case"]
    path = case["path"]
    if path == "accept":
        k, t, top = case["drafts"], case["temperature"], case["top_p"]
        G.sample_logits(s["draft"], t, top, s["seed"], 7, 0, 1, s["proposals"], s["sws"])
        G.verify_logits(s["target"], s["draft"] if t else None, s["proposals"], t, top, s["seed"], 7, s["result"], s["ws"])
        return dict(proposals=s["proposals"], result=s["result"].view(torch.int32))
    if path == "measures":
        G.verify_gpu_v2(s["drafts"], None if case["greedy"] else s["q"], s["p"], int(case["greedy"]), s["seed"], 7, s["result"])
        return dict(result=s["result"].view(torch.int32))
    H, I = case["hidden"], case["inter"]
    if path == "experts":
        stream, n = G._stream(), case["jobs"]
        def project(which, proj, rows, cols):
            if case["chunked"]:
                G.grouped_prefill(s["table"], s["jobs"][which], n, proj, rows, cols, case["rows"])
            else:
                G.grouped(s["table"], s["jobs"][which], n, proj, rows, cols)
        _quantize(s["x"], s["xq"], s["xs"], stream)
        project("gate", G.PROJ_GATE, I, H)
        project("up", G.PROJ_UP, I, H)
        G.check(G.lib().ds41_swiglu(G._p(s["gate"]), G._p(s["up"]), G._p(s["w"]), G._p(s["h"]), s["h"].shape[0], I, ctypes.c_float(LIMIT), stream),
                "swiglu")
        _quantize(s["h"], s["hq"], s["hs"], stream)
        project("down", G.PROJ_DOWN, H, I)
        return dict(gate=s["gate"], up=s["up"], h=s["h"], y=s["y"])
    if path == "shared":
        S = s["S"]
        a, sa = G.dense_quant(s["x"])
        g = G.dense_fp8(a, sa, S["gate"], S["gate_scale"], I)
        u = G.dense_fp8(a, sa, S["up"], S["up_scale"], I)
        z, b, sb = G.dense_shared_act(g, u)
        return dict(gate=g, up=u, h=z, y=G.dense_fp8(b, sb, S["down"], S["down_scale"], H))
    if path == "layer":
        G.moe_layer(s["args"])
        return dict(y=s["y"], ids=s["ids"], w=s["w"])
    if path == "stack":
        s["stack"].step(s["x"], s["y"], route_ids=s["ids"], layer_out=s["out"], ids_out=s["ids_out"], weights_out=s["w"])
        return dict(y=s["y"], out=s["out"], ids=s["ids_out"], w=s["w"])
    if path == "drafter":
        return dict(y=s["service"](0, s["x"], s["ids"], s["w"], s["y"]))
    G.moe_prefill(s["args"])
    return dict(y=s["y"])


# ---- what a pass cannot do without -----------------------------------------------------------
def _mx(n, k):
    return n * k // 2 + n * k // 32


def work(case):
    path = case["path"]
    if path in ("accept", "measures"):
        V, k = case["vocab"], case["drafts"]
        greedy = case["greedy"] if path == "measures" else case["temperature"] == 0
        rows = k + 1 if greedy and path == "measures" else 2 * k + 1
        # measures: a reject ends the call early; about half of the rows are looked at
        return dict(bytes=rows * V * 4, flops=rows * V * 4)
    H, I = case["hidden"], case["inter"]
    expert = 2 * _mx(I, H) + _mx(H, I)
    if path == "experts":
        R = sum(_job_rows(case))
        io = R * (2 * H + 2 * H) + R * I * 6
        return dict(bytes=case["jobs"] * expert + io, flops=R * 6 * H * I)
    if path == "shared":
        T = case["rows"]
        return dict(bytes=3 * (H * I + H * I // 1024) + T * (4 * H + 6 * I), flops=T * 6 * H * I)
    if path == "drafter":
        T = case["rows"]
        return dict(bytes=128 * (1 - (1 - 3 / 128) ** T) * expert + T * 8 * H, flops=T * 18 * H * I)
    E, K = case["experts"], case["topk"]
    if path == "layer":
        T = case["rows"]
        used = E * (1 - (1 - K / E) ** T)
        shared = 3 * (H * I + H * I // 1024) if case["shared"] == "fp8" else expert
        return dict(bytes=used * expert + shared + E * H * 4 + T * 4 * H, flops=T * ((K + 1) * 6 * H * I + 2 * E * H))
    if path == "stack":
        T, L = case["rows"], case["layers"]
        used = np.mean([len(np.unique(_zipf(np.random.default_rng(i), T, E, K))) for i in range(16)])
        return dict(bytes=L * (float(used + 1) * expert + float(used) * H * 4 + T * 4 * H), flops=L * T * (K + 1) * 6 * H * I)
    T = case["tokens"]
    used = np.mean([len(np.unique(_zipf(np.random.default_rng(i), T, E, K))) for i in range(4)])
    return dict(bytes=float(used + 1) * expert + T * 4 * H, flops=T * (K + 1) * 6 * H * I)


def tolerance(case):
    """Accept decisions and tokens are whole numbers and fixed by the sampler's definition. bf16
    outputs behind sums of thousands of products differ by single roundings, and where a changed
    rounding moves an 8-bit activation code, by 1/8 of one value; in a stack such code
    steps are the second layer's input."""
    if case["path"] in ("accept", "measures"):
        return "exact"
    return {"rel": {"stack": 3e-2, "layer": 6e-3, "drafter": 6e-3, "prefill": 6e-3, "experts": 6e-3, "shared": 6e-3}[case["path"]]}


# ---- the same in 64 bits ----------------------------------------------------------------------
_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _mx_weight(w, s, tiled):
    """[N][K] float64 of an MXFP4 matrix, row-major or in 16-row tiles of 16-byte pieces."""
    n, k = s.shape[0], s.shape[1] * 32
    if tiled:
        w = w.reshape(n // 16, k // 32, 16, 16).permute(0, 2, 1, 3).reshape(n, k // 2)
    lut = torch.tensor(_E2M1, dtype=torch.float64, device=DEV)
    v = torch.stack((lut[(w & 15).int()], lut[(w >> 4).int()]), -1).view(n, k // 32, 32)
    return (v * torch.exp2(s.double() - 127)[..., None]).view(n, k)


def _e4m3(t):
    return t.view(torch.float8_e4m3fn).float().double()


def _mx_rows(x):
    """bf16 rows through the MXFP8 format (E4M3 codes, one power-of-two scale per 32 values)."""
    v = x.float().view(x.shape[0], -1, 32)
    b = (v.abs().amax(-1).clamp_min(1e-4) * np.float32(1 / 448)).view(torch.int32)
    scale = torch.exp2(((b >> 23) + ((b & 0x7FFFFF) != 0)).double() - 127)[..., None]
    codes = (v.double() / scale).clamp(-448, 448).float().to(torch.float8_e4m3fn)
    return (codes.double() * scale).view(x.shape)


def _bf16(v):
    return v.float().to(torch.bfloat16)


def _ffn(xr, gate, up, down, w):
    """One expert over MXFP8 rows in 64-bit sums; between its projections the path's own formats."""
    g, u = xr @ gate.T, xr @ up.T
    gb, ub = _bf16(g).double().clamp(max=LIMIT), _bf16(u).double().clamp(-LIMIT, LIMIT)
    h = gb / (1 + torch.exp(-gb)) * ub
    h = h if w is None else w.double()[:, None] * h
    return g, u, h, _mx_rows(_bf16(h)) @ down.T


def _mx_ffn(P, e, xr, w, tiled):
    return _ffn(xr, *(_mx_weight(P[n][e], P[n + "_scale"][e], tiled) for n in ("gate", "up", "down")), w)


def _fp8_ffn(S, xr):
    def m(n):
        return _e4m3(S[n]) * torch.exp2(S[n + "_scale"].double() - 127).repeat_interleave(32, 0).repeat_interleave(32, 1)
    return _ffn(xr, m("gate"), m("up"), m("down"), None)


def _moe(x, ids, w, P, tiled, shared):
    xr = _mx_rows(x)
    y = torch.zeros(x.shape, dtype=torch.float64, device=DEV)
    for e in torch.unique(ids).tolist():
        t, k = torch.nonzero(ids == e, as_tuple=True)
        y.index_add_(0, t, _bf16(_mx_ffn(P, e, xr[t], w[t, k], tiled)[3]).double())
    return y + _bf16(shared(xr)).double()


def _weights_of(x, wg, ids=None, topk=0):
    z = x.double() @ wg.double().T
    u = torch.sqrt(torch.nn.functional.softplus(z, threshold=50))
    ids = u.topk(topk, dim=1).indices if ids is None else ids
    u = u.gather(1, ids.long())
    return ids, u / u.sum(1, keepdim=True) * SCALE


def exact(case, seed):
    path = case["path"]
    if path in ("accept", "measures"):
        return None
    s = _inputs(case, seed)
    x = s["x"]
    if path == "experts":
        outs, at, xr = [], 0, _mx_rows(x)
        for j, n in enumerate(_job_rows(case)):
            outs.append(_mx_ffn(s["P"], j, xr[at:at + n], s["w"][at:at + n], False))
            at += n
        return dict(zip(("gate", "up", "h", "y"), (torch.cat(v) for v in zip(*outs))))
    if path == "shared":
        return dict(zip(("gate", "up", "h", "y"), _fp8_ffn(s["S"], _mx_rows(x))))
    if path == "layer":
        ids, w = _weights_of(x, s["wg"], topk=case["topk"])
        shared = (lambda xr: _fp8_ffn(s["S"], xr)[3]) if s["S"] else (lambda xr: _mx_ffn(s["P"], case["experts"], xr, None, case["tiled"])[3])
        return dict(y=_moe(x, ids, w.float(), s["P"], case["tiled"], shared), ids=None, w=w)
    if path == "stack":
        out, ws = [], []
        for l, (P, wg, _) in enumerate(s["layers"]):
            _, w = _weights_of(x, wg, s["ids"][l])
            out.append(_moe(x, s["ids"][l], w.float(), P, True, lambda xr: _mx_ffn(P, case["experts"], xr, None, True)[3]))
            ws.append(w)
            x = _bf16(out[-1])
        return dict(y=out[-1], out=torch.stack(out[:-1]), ids=None, w=torch.stack(ws))
    if path == "drafter":
        xr, y = _mx_rows(x), torch.empty((x.shape[0], 3, x.shape[1]), dtype=torch.float64, device=DEV)
        for e in torch.unique(s["ids"]).tolist():
            t, k = torch.nonzero(s["ids"] == e, as_tuple=True)
            y[t, k] = _mx_ffn(s["P"], e, xr[t], s["w"][t, k], True)[3]
        return dict(y=y)
    return dict(y=_moe(x, s["ids"], s["w"], s["P"], False, lambda xr: _mx_ffn(s["P"], case["experts"], xr, None, False)[3]))
