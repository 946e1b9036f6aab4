"""The fused op's shared expert as one more expert of the routed GEMMs (it is as wide as they are) against launches of
its own: the same weights padded with zero columns to twice the width keep their own launches and give the same bits
(the padding's h is 0: it adds zeros to every sum and no maximum).  The own launches are compared with the oracle in
test_gpu_fused.py and test_gpu_int8.py."""
import pytest
import torch

import test_gpu_fused as F
import test_gpu_int8 as Q

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import umdk_amd  # noqa: F401
    return torch.ops.umdk_cam_op_lib


def widen(w, dim, halves):
    """w with zeros after it along dim (halves 2: after each half, the gate and the up columns)."""
    return torch.cat([v for p in w.chunk(halves, dim) for v in (p, torch.zeros_like(p))], dim)


def routed(d, int8, lists=False):
    """The routed experts' weight arguments: one stacked tensor each, or one per expert."""
    t = lambda v: None if v is None else v.transpose(-1, -2)  # noqa: E731
    one = lambda v: [] if v is None else list(v.unbind(0)) if lists else [v]  # noqa: E731
    w1, w2 = (d["w1"], d["w2"]) if int8 else (t(d["w1"]), t(d["w2"]))
    return one(w1), one(d["s1"]), one(w2), one(d["s2"])


def call(ops, d, E, mask, sw, int8, weights=None):
    return ops.fused_deep_moe(d["x"], d["ids"], *(weights or routed(d, int8)), d["scales"], sw[0], sw[1], sw[2], sw[3],
                              d.get("sm"), d.get("ssm"), mask, "ep", 1, 0, E, 0, 0)


# decode sizes with the layout in the dispatch, the same at its limit (2048 picks), past it (8-wave GEMMs, wave-per-token
# int8 rows above 3072 picks), and past the single-launch layouts (8192 picks), where the expert keeps its own launches
SIZES = [(3, 1024, 128, 8, 2), (40, 2048, 256, 16, 4), (256, 1024, 256, 8, 8), (300, 1024, 256, 16, 8),
         (600, 1024, 128, 8, 8), (1100, 1024, 128, 8, 8),
         # int8 rows by the block per destination and, one token on, by the wave per token: 3072 picks, 2048 of wide rows
         (384, 1024, 128, 16, 8), (385, 1024, 128, 16, 8), (256, 2304, 128, 8, 8), (257, 2304, 128, 8, 8)]


@pytest.mark.parametrize("kind", ["bf16", "fp8", "int8", "int8_smooth"])
@pytest.mark.parametrize("size", SIZES)
def test_shared_expert_in_the_routed_gemms(ops, kind, size):
    bs, H, I, E, K = size
    print(f"shared expert {kind} {size}", flush=True)
    int8 = kind.startswith("int8")
    if int8:
        d = Q.make_fused(bs + I, bs, H, I, E, K, ish=I, smooth=kind == "int8_smooth")
        d = {k: v.cuda() for k, v in d.items()}
        g = torch.Generator(device="cuda").manual_seed(bs)
        w1 = torch.randint(-9, 10, (H, 2 * I), dtype=torch.int8, device="cuda", generator=g)
        w2 = torch.randint(-9, 10, (I, H), dtype=torch.int8, device="cuda", generator=g)
        own = (w1, d["ss1"], w2, d["ss2"])
        wide = (widen(w1, 1, 2), widen(d["ss1"], 0, 2), widen(w2, 0, 1), d["ss2"])
    else:
        d = F.make(bs + I, bs, H, I, E, K, kind, ish=I)
        own = (d["sw1"].T, d["ss1"], d["sw2"].T, d["ss2"])
        raw = lambda w: w.view(torch.uint8) if kind == "fp8" else w  # noqa: E731  (cat of fp8 bytes)
        wide = (widen(raw(d["sw1"]), 0, 2).view(d["sw1"].dtype).T, None if kind == "bf16" else widen(d["ss1"], 0, 2),
                widen(raw(d["sw2"]), 1, 1).contiguous().view(d["sw2"].dtype).T,
                None if kind == "bf16" else widen(d["ss2"], 1, 1).contiguous())
    d["ids"][bs // 2, 0] = -1
    mask = torch.arange(bs, device="cuda") < bs - bs // 4
    a, sa, na = call(ops, d, E, mask, own, int8)
    b, sb, nb = call(ops, d, E, mask, wide, int8)
    torch.cuda.synchronize()
    assert torch.equal(na, nb)
    assert torch.equal(a.view(torch.int16), b.view(torch.int16)), "routed output"
    assert torch.equal(sa.view(torch.int16), sb.view(torch.int16)), "shared output"
    assert bool(sa.float().abs().sum(1).gt(0).all())


@pytest.mark.parametrize("kind", ["bf16", "fp8", "int8_smooth"])
def test_shared_expert_beside_weight_lists_and_in_a_graph(ops, kind):
    # the routed weights as per-expert lists (pointer tables of the L routed experts, the shared one after them) give the
    # stacked weights' bits, and a graph captured on either replays them
    bs, H, I, E, K = 40, 2048, 256, 16, 4
    print(f"shared expert beside weight lists {kind}", flush=True)
    int8 = kind.startswith("int8")
    if int8:
        d = {k: v.cuda() for k, v in Q.make_fused(bs, bs, H, I, E, K, ish=I, smooth=True).items()}
        for k in ("w1", "w2", "sw1", "sw2"):  # the kernels' own layout: no converted copies, which a capture cannot make
            d[k] = d[k].transpose(-1, -2).contiguous().transpose(-1, -2)
        own = (d["sw1"], d["ss1"], d["sw2"], d["ss2"])
    else:
        d = F.make(bs, bs, H, I, E, K, kind, ish=I)
        own = (d["sw1"].T, d["ss1"], d["sw2"].T, d["ss2"])
    same = lambda p, q: all(torch.equal(u.view(torch.int16), v.view(torch.int16)) for u, v in zip(p, q))  # noqa: E731
    both = [routed(d, int8), routed(d, int8, lists=True)]
    ref = [v.clone() for v in call(ops, d, E, None, own, int8, both[0])[:2]]
    assert same(ref, call(ops, d, E, None, own, int8, both[1])[:2])
    torch.cuda.synchronize()
    for lists, weights in enumerate(both):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = call(ops, d, E, None, own, int8, weights)
        for r in range(3):
            junk = torch.randn(1 << 20, device="cuda") * r  # eager work between replays
            for v in got[:2]:
                v.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert same(ref, got[:2]), f"replay {r}, lists {lists}"
            del junk
