"""The work that users of this library have it do, as measurable cases.

Five kinds, each through the entry points that a program calls:

  decode   moe_route + fused_deep_moe: one decode step of a MoE layer on one EP rank.  The routed ids cover all E
           experts; the rank holds the first L of them and skips the other picks.  Eager, or as a program serves
           it, captured once in a HIP graph and replayed.
  prefill  MoePrefillPlan: route + layout + count exchange + dispatch, then the combine of expert outputs.
  ops      the same through the five reference-shaped operators, with their allocations and the host read of the
           received row count.
  layer    MoeLayerPlan.forward: a whole prefill layer on one EP rank holding L of E experts.
  gmm      grouped_matmul_swiglu + grouped_matmul over ragged expert groups.

Ranges: 1 to 8192 tokens (decode to 512), 1024 to 7168 columns, 8 to 256 experts, top-1 to top-8, expert widths of
128 to 14336; bf16, int8 (W8A8) and fp8 e4m3 (1x128 / 128x128 scales).
"""
import functools
import math

import torch

import umdk_amd  # noqa: F401  (registers the operators)
from umdk_amd.plan import MoeLayerPlan, MoePrefillPlan

OPS = torch.ops.umdk_cam_op_lib
QUANT = {"bf16": 0, "int8": 2, "fp8": 3}
DEV = "cuda:0"


def listed():
    return [
        # a single user's next token on a small model: nothing but launches and host time
        dict(name="decode_one_token", kind="decode", dtype="bf16", T=1, H=1024, E=8, L=8, K=2, I=512, shared=0,
             smooth=False, graph=False),
        # the headline decode step: a 128-sequence batch, 32 of 256 experts on the rank, replayed from a graph
        dict(name="decode_fp8_graph", kind="decode", dtype="fp8", T=128, H=7168, E=256, L=32, K=8, I=2048, shared=0,
             smooth=False, graph=True),
        # the reference's own decode mode: int8 weights, smooth-quant scales and a shared expert
        dict(name="decode_int8_shared", kind="decode", dtype="int8", T=128, H=7168, E=256, L=32, K=8, I=2048,
             shared=2048, smooth=True, graph=False),
        # a large decode batch on a model whose experts all sit on the GPU, in bf16
        dict(name="decode_bf16_batch", kind="decode", dtype="bf16", T=400, H=2048, E=64, L=64, K=6, I=1408, shared=0,
             smooth=False, graph=False),
        # the headline dispatch + combine step: a 4096-token prefill chunk at the one-rank shape
        dict(name="prefill_fp8", kind="prefill", dtype="fp8", T=4096, H=7168, E=256, K=8),
        # a short ragged prompt through the operators, rows kept in bf16
        dict(name="ops_bf16_ragged", kind="ops", dtype="bf16", T=1021, H=5120, E=160, K=6),
        # the reference's prefill sample: the operators with use_quant, a full chunk
        dict(name="ops_int8", kind="ops", dtype="int8", T=4096, H=7168, E=256, K=8),
        # a prefill layer of one rank under skewed expert load: a few heavy experts, many light ones
        dict(name="layer_fp8_skewed", kind="layer", dtype="fp8", T=4096, H=7168, E=256, L=32, K=8, I=2048, skew=1.1),
        # the same layer with the reference's int8 weights
        dict(name="layer_int8_skewed", kind="layer", dtype="int8", T=4096, H=7168, E=256, L=32, K=8, I=2048, skew=1.1),
        # a dense-ish prefill layer: few wide experts, all local, bf16
        dict(name="layer_bf16_wide", kind="layer", dtype="bf16", T=8192, H=4096, E=8, L=8, K=2, I=14336, skew=0.0),
        # the expert GEMMs of a long prefill: thousands of rows per expert, compute-bound
        dict(name="gmm_fp8_large", kind="gmm", dtype="fp8", M=65536, L=32, H=7168, I=2048, kmajor=True),
        # the expert GEMMs of an ordinary chunk: about a hundred ragged rows per expert, scales as dispatched
        dict(name="gmm_fp8_ragged", kind="gmm", dtype="fp8", M=6000, L=48, H=4096, I=1408, kmajor=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _one_draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "ops", "layer", "layer", "gmm", "gmm"])
    dtype = rng.choice(["bf16", "int8", "fp8"])
    H = 256 * _log_int(rng, 4, 28)
    if kind == "decode":
        E = rng.choice([8, 16, 32, 64, 128, 160, 256])
        L = E // rng.choice([d for d in (1, 2, 4, 8) if E // d >= 8])
        return dict(kind=kind, dtype=dtype, T=_log_int(rng, 1, 512), H=H, E=E, L=L, K=rng.randint(1, 8),
                    I=128 * _log_int(rng, 1, 16), shared=128 * _log_int(rng, 1, 16) if rng.random() < 0.3 else 0,
                    smooth=dtype == "int8" and rng.random() < 0.5, graph=rng.random() < 0.5)
    if kind in ("prefill", "ops"):
        if rng.random() < 0.5:  # widths that are no power of two and no multiple of the kernels' chunks
            H = 128 * rng.randint(8, 56) if dtype == "fp8" else 16 * rng.randint(64, 448)
        E = rng.choice([8, 16, 60, 64, 128, 160, 256])
        return dict(kind=kind, dtype=dtype, T=_log_int(rng, 32, 8192), H=H, E=E, K=rng.randint(1, 8))
    if kind == "layer":
        E = rng.choice([8, 16, 32, 64, 128, 160, 256])
        L = E // rng.choice([d for d in (1, 2, 4, 8) if E // d >= 4])
        return dict(kind=kind, dtype=dtype, T=_log_int(rng, 128, 8192), H=H, E=E, L=L, K=rng.randint(1, 8),
                    I=128 * _log_int(rng, 2, 112), skew=rng.choice([0.0, 0.5, 1.1]))
    return dict(kind=kind, dtype=dtype, M=_log_int(rng, 256, 65536), L=rng.choice([4, 8, 16, 24, 32, 48, 64]), H=H,
                I=128 * _log_int(rng, 2, 112), kmajor=dtype == "fp8" and rng.random() < 0.5)


def draw(rng):
    most = [work(c) for c in listed()]
    top = {q: max(w[q] for w in most) for q in ("bytes", "flops")}
    while True:
        c = _one_draw(rng)
        w = work(c)
        if w["bytes"] <= top["bytes"] and w["flops"] <= top["flops"]:
            return c


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _tokens(T, H, g):
    """bf16 activations whose scale differs from token to token."""
    x = torch.randn(T, H, generator=g, device=DEV)
    return (x * torch.exp(0.5 * torch.randn(T, 1, generator=g, device=DEV))).bfloat16()


def _weight(L, n, k, dtype, g):
    """[L, n, k] weights ~ N(0, 0.02) and their scales: fp8 per 128 x 128 block, int8 per output channel."""
    w = torch.randn(L, n, k, generator=g, device=DEV, dtype=torch.float32).mul_(0.02)
    if dtype == "bf16":
        return w.bfloat16(), None
    if dtype == "int8":
        s = w.abs().amax(dim=2).clamp(min=1e-6) / 127.0
        return w.div_(s[:, :, None]).round_().clamp_(-127, 127).to(torch.int8), s.contiguous()
    wb = w.view(L, n // 128, 128, k // 128, 128)
    s = wb.abs().amax(dim=(2, 4)).clamp(min=1e-6) / 448.0
    q = wb.div_(s[:, :, None, :, None]).to(torch.float8_e4m3fn).view(L, n, k)
    return q, s.contiguous()


def _bias(c, g):
    """Per-expert routing bias.  skew s: popularity 1 / rank^s, the rank's experts holding every (E / L)-th rank in an
    order of the seed's, so that its load does not hang on the seed."""
    E, L, s = c["E"], c.get("L", c["E"]), c.get("skew", 0.0)
    if not s:
        return torch.randn(E, generator=g, device=DEV) * 0.5
    step = E // L
    mine = torch.arange(L, device=DEV) * step + step // 2
    other = torch.ones(E, dtype=torch.bool, device=DEV)
    other[mine] = False
    rest = other.nonzero().flatten()
    rank = torch.cat([mine[torch.randperm(L, generator=g, device=DEV)],
                      rest[torch.randperm(E - L, generator=g, device=DEV)]])
    return -s * torch.log(1.0 + rank.float())


def _groups(c, g):
    """Rows per expert, M in all: expert popularity varies by a factor of e^(0.5 N(0, 1))."""
    p = torch.softmax(0.5 * torch.randn(c["L"], generator=g, device=DEV), 0).cpu().double()
    n = torch.floor(p * c["M"]).long()
    n[: c["M"] - int(n.sum())] += 1
    return n.to(DEV)


def _quant_rows(x, dtype, kmajor):
    """bf16 rows as the dispatch hands them to the GEMMs: (rows, scales)."""
    if dtype == "bf16":
        return x, None
    f = x.float()
    if dtype == "int8":
        s = 127.0 / (f.abs().amax(dim=1) + 1e-12)
        return torch.round(f * s[:, None]).to(torch.int8), 1.0 / s
    M, H = f.shape
    a = f.view(M, H // 128, 128).abs().amax(dim=2).clamp(min=1e-4)
    q = (f.view(M, H // 128, 128) * (448.0 / a)[:, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn).view(M, H)
    s = a / 448.0
    return q, (s.t().contiguous().t() if kmajor else s)


def prepare(c, seed):
    g = _gen(seed)
    kind, dtype = c["kind"], c["dtype"]
    s = {"c": c}
    if kind == "gmm":
        s["groups"] = _groups(c, g)
        s["x"], s["xs"] = _quant_rows(_tokens(c["M"], c["H"], g), dtype, c["kmajor"])
        s["w1"], s["s1"] = _weight(c["L"], 2 * c["I"], c["H"], dtype, g)
        s["w2"], s["s2"] = _weight(c["L"], c["H"], c["I"], dtype, g)
        return s
    T, H, E, K = c["T"], c["H"], c["E"], c["K"]
    s["x"] = _tokens(T, H, g)
    s["logits"] = torch.randn(T, E, generator=g, device=DEV)
    if kind != "decode":
        s["bias"] = _bias(c, g)
    if kind in ("prefill", "ops"):
        s["y"] = torch.randn(T * K, H, generator=g, device=DEV).bfloat16()  # the experts' outputs, in dispatch order
        if kind == "prefill":
            s["plan"] = MoePrefillPlan(T, H, E, K, quant_mode=QUANT[dtype], device=DEV)
        return s
    L, I = c["L"], c["I"]
    s["w1"], s["s1"] = _weight(L, 2 * I, H, dtype, g)
    s["w2"], s["s2"] = _weight(L, H, I, dtype, g)
    if kind == "layer":
        s["plan"] = MoeLayerPlan(T, H, E, K, L, I, dtype=dtype, device=DEV)
        return s
    if c["shared"]:
        s["sw1"], s["ss1"] = (None if v is None else v[0] for v in _weight(1, 2 * c["shared"], H, dtype, g))
        s["sw2"], s["ss2"] = (None if v is None else v[0] for v in _weight(1, H, c["shared"], dtype, g))
    if c["smooth"]:
        s["smooth"] = torch.exp(0.3 * torch.randn(L, H, generator=g, device=DEV))
        s["share_smooth"] = torch.exp(0.3 * torch.randn(H, generator=g, device=DEV)) if c["shared"] else None
    if c["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _decode(s)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            s["held"] = _decode(s)
        s["graph"] = graph
    return s


# ---------------------------------------------------------------- one pass
def _decode(s):
    c = s["c"]
    idx, w = OPS.moe_route(s["logits"], None, c["K"])
    t = lambda v: None if v is None else v.transpose(-1, -2)  # noqa: E731  (logical [.., k, n] of k-contiguous storage)
    lst = lambda v: [] if v is None else [v]  # noqa: E731
    out, share, counts = OPS.fused_deep_moe(
        s["x"], idx, [t(s["w1"])], lst(s["s1"]), [t(s["w2"])], lst(s["s2"]), w, t(s.get("sw1")), s.get("ss1"),
        t(s.get("sw2")), s.get("ss2"), s.get("smooth"), s.get("share_smooth"), None, "ep", 1, 0, c["L"], 0, c["T"])
    r = {"idx": idx, "w": w, "out": out, "counts": counts}
    if c["shared"]:
        r["share"] = share
    return r


def _bytes(t):
    return t.view(torch.uint8) if t.dtype == torch.float8_e4m3fn else t


def run(s):
    c = s["c"]
    kind, dtype = c["kind"], c["dtype"]
    if kind == "decode":
        if c["graph"]:
            s["graph"].replay()
            return s["held"]
        return _decode(s)
    if kind == "prefill":
        p = s["plan"]
        p.dispatch_step(s["logits"], s["x"], s["bias"])
        out = p.combine_step(s["y"])
        return _rows({"idx": p.topk_idx, "w": p.topk_w, "out": out, "rows": _bytes(p.expand_x), "src": p.expand_idx,
                      "counts": p.recv_tokens_per_expert}, dtype, p.scales)
    if kind == "ops":
        idx, w = OPS.moe_route(s["logits"], s["bias"], c["K"])
        per_expert, rank = OPS.get_dispatch_layout(idx, c["E"], 1)
        rows, scales, src, recv, counts = OPS.moe_dispatch_prefill(
            s["x"], idx, w, per_expert, rank, "ep", 0, 1, dtype == "int8", 3 if dtype == "fp8" else -1)
        out = OPS.moe_combine_prefill(s["y"], idx, w, src, recv, "ep", 0, 1)
        return _rows({"idx": idx, "w": w, "out": out, "rows": _bytes(rows), "src": src, "counts": counts}, dtype,
                     scales)
    if kind == "layer":
        p = s["plan"]
        out = p.forward(s["x"], s["logits"], s["bias"], s["w1"], s["s1"], s["w2"], s["s2"])
        return {"idx": p.topk_idx, "w": p.topk_w, "out": out, "counts": p.recv_tokens_per_expert}
    h, hs = OPS.grouped_matmul_swiglu(s["x"], s["xs"], s["groups"], s["w1"], s["s1"], QUANT[dtype])
    y = OPS.grouped_matmul(h, hs if dtype != "bf16" else None, s["groups"], s["w2"], s["s2"])
    r = {"h": _bytes(h), "y": y}
    if dtype != "bf16":
        r["hs"] = hs
    return r


def _rows(r, dtype, scales):
    if dtype != "bf16":  # bf16 rows have no scales
        r["scales"] = scales
    return r


# ---------------------------------------------------------------- what a pass cannot do without
@functools.lru_cache(maxsize=None)
def _local_rows(T, E, L, K, skew):
    """(rows routed to the L local experts, experts of them with a row), on average over tokens; skew as in _bias."""
    if not skew:
        return T * K * L / E, L * (1 - (1 - K / E) ** T)
    g = torch.Generator().manual_seed(0)
    n = min(T, 8192)
    step = E // L
    rank = torch.arange(E)
    logits = torch.randn(n, E, generator=g) - skew * torch.log(1.0 + rank.float())
    hit = torch.zeros(E).index_add_(0, logits.topk(K, dim=1).indices.flatten(), torch.ones(n * K)) / n
    mine = hit[torch.arange(L) * step + step // 2]
    return float(mine.sum()) * T, float((1 - (1 - mine.clamp(max=1.0)) ** T).sum())


def _weight_bytes(n, k, dtype):
    if dtype == "bf16":
        return 2 * n * k
    return n * k + 4 * (n if dtype == "int8" else n * k // 16384)


def _row_bytes(n, dtype):
    return 2 * n if dtype == "bf16" else n + 4 if dtype == "int8" else n + 4 * (n // 128)


def work(c):
    kind, dtype, H = c["kind"], c["dtype"], c["H"]
    if kind == "gmm":
        M, L, I = c["M"], c["L"], c["I"]
        b = M * (_row_bytes(H, dtype) + _row_bytes(I, dtype) + 2 * H) + 8 * L
        b += L * (_weight_bytes(2 * I, H, dtype) + _weight_bytes(H, I, dtype))
        return {"bytes": b, "flops": 6 * M * H * I}
    T, E, K = c["T"], c["E"], c["K"]
    b = T * (2 * H + 4 * E + 8 * K + 2 * H)  # x, logits, the routing, the output
    if kind in ("prefill", "ops"):
        b += T * K * (_row_bytes(H, dtype) + 12 + 2 * H) + 8 * E  # dispatched rows and their sources, expert outputs
        return {"bytes": b, "flops": 2 * T * K * H}
    L, I, sh = c["L"], c["I"], c.get("shared", 0)
    rows, touched = _local_rows(T, E, L, K, c.get("skew", 0.0))
    b += touched * (_weight_bytes(2 * I, H, dtype) + _weight_bytes(H, I, dtype)) + 8 * L
    if sh:
        b += _weight_bytes(2 * sh, H, dtype) + _weight_bytes(H, sh, dtype) + 2 * T * H
    if c.get("smooth"):
        b += 4 * H * (touched + (1 if sh else 0))
    return {"bytes": int(b), "flops": int(6 * H * (rows * I + T * sh) + 2 * rows * H)}


def tolerance(c):
    """Four times what the path is seen to differ by from its 64-bit form: the output's rounding to bf16 (an rms of
    1.7e-3), and in the expert paths the values of h (and of x, where it is scaled first) that fall on the other side
    of a rounding step.  Whole values: the codes of h that do so (the dispatched rows are rounded the same way by
    every correct implementation)."""
    if c["kind"] in ("prefill", "ops"):
        return {"rel": 7e-3, "max": 0.05, "differ": 0.0}
    return {"rel": 1e-2, "max": 0.1, "differ": 1e-3 if c["kind"] == "gmm" else 0.0}


# ---------------------------------------------------------------- the same in 64 bits
def _route64(logits, bias, K):
    score = logits if bias is None else logits + bias  # the ids are defined on the 32-bit scores, ties to the lower
    idx = torch.sort(score, dim=1, descending=True, stable=True).indices[:, :K]
    return idx, torch.softmax(torch.gather(logits.double(), 1, idx), dim=1)


def _codes(x, dtype, fused, smooth=None):
    """(codes as 64-bit values, their scales, broadcast) of rows [n, H], at x's own width.  A bf16 store on the way is
    no part of what a path computes and is left out."""
    if dtype == "bf16":
        return x.double(), 1.0
    if smooth is not None:
        x = x * smooth
    if dtype == "int8":
        a = x.abs().amax(dim=1, keepdim=True)
        sc = torch.full_like(a, 127.0) / (a if fused else a + 1e-12)  # a true division: number / tensor is none
        return torch.round(x * sc).double(), torch.ones_like(a) / sc
    n, H = x.shape
    b = x.view(n, H // 128, 128)
    a = b.abs().amax(dim=2, keepdim=True).clamp(min=1e-4)
    q = (b * (torch.full_like(a, 448.0) / a)).clamp(-448, 448).float().to(torch.float8_e4m3fn).double()
    return q, a / 448.0


def _quantised(x, dtype, fused=False, smooth=None):
    """(what rows [n, H] stand for once quantised, in 64 bits; their scales)."""
    q, sc = _codes(x, dtype, fused, smooth)
    if dtype == "bf16":
        return q, None
    return (q * sc.double()).view(x.shape), sc.view(x.shape[0], -1) if dtype == "fp8" else sc.flatten()


def _weight64(w, sc, dtype):
    if dtype == "bf16":
        return w.double()
    if dtype == "int8":
        return w.double() * sc.double()[:, None]
    n, k = w.shape
    return (w.double().view(n // 128, 128, k // 128, 128) * sc.double()[:, None, :, None]).view(n, k)


def _expert64(x, w1, s1, w2, s2, dtype):
    """One expert on rows x in 64 bits: (y, h, scales of h)."""
    gu = x @ _weight64(w1, s1, dtype).t()
    I = gu.shape[1] // 2
    h, hs = _quantised(torch.nn.functional.silu(gu[:, :I]) * gu[:, I:], dtype, fused=True)
    return h @ _weight64(w2, s2, dtype).t(), h, hs


def _scale(sc, e):
    return None if sc is None else sc[e]


def exact(c, seed):
    s = prepare(dict(c, graph=False), seed)
    kind, dtype = c["kind"], c["dtype"]
    if kind == "gmm":
        x = s["x"].double()
        if dtype == "int8":
            x *= s["xs"].double()[:, None]
        elif dtype == "fp8":
            x = (x.view(c["M"], -1, 128) * s["xs"].double()[:, :, None]).view(c["M"], -1)
        ys, h, hss, at = [], [], [], 0
        for e, n in enumerate(s["groups"].tolist()):
            y, he, hs = _expert64(x[at:at + n], s["w1"][e], _scale(s["s1"], e), s["w2"][e], _scale(s["s2"], e), dtype)
            ys.append(y)
            h.append(he)
            hss.append(hs)
            at += n
        r = {"h": torch.cat(h) if dtype == "bf16" else None, "y": torch.cat(ys)}
        if dtype != "bf16":
            r["hs"] = torch.cat(hss)
        return r
    T, K = c["T"], c["K"]
    idx, w = _route64(s["logits"], s.get("bias"), K)
    order = torch.sort(idx.flatten(), stable=True).indices  # the (t, k) of each dispatched row
    # the ids and the codes of x are defined on 32-bit scores and rows (ties are common: bf16 values over a bf16
    # maximum), so they are made in 32 bits here too
    x = s["x"].float()
    if kind in ("prefill", "ops"):
        row = torch.empty_like(order)
        row[order] = torch.arange(T * K, device=DEV)
        out = torch.zeros(T, c["H"], dtype=torch.float64, device=DEV)
        for k in range(K):
            out += s["y"].double()[row.view(T, K)[:, k]] * w[:, k, None]
        _, scales = _quantised(x, dtype)
        return _rows({"idx": None, "w": w, "out": out, "rows": x[order // K] if dtype == "bf16" else None, "src": None,
                      "counts": None}, dtype, None if scales is None else scales[order // K])
    fused = kind == "decode"
    out = torch.zeros(T, c["H"], dtype=torch.float64, device=DEV)
    for e in range(c["L"]):
        t, k = (idx == e).nonzero(as_tuple=True)
        if t.numel():
            q, _ = _quantised(x[t], dtype, fused, s["smooth"][e] if c.get("smooth") else None)
            y, _, _ = _expert64(q, s["w1"][e], _scale(s["s1"], e), s["w2"][e], _scale(s["s2"], e), dtype)
            out.index_add_(0, t, y * w[t, k][:, None])
    r = {"idx": None, "w": w, "out": out, "counts": None}
    if c.get("shared"):
        x, _ = _quantised(x, dtype, fused, s["share_smooth"] if c["smooth"] else None)
        r["share"], _, _ = _expert64(x, s["sw1"], s["ss1"], s["sw2"], s["ss2"], dtype)
    return r
