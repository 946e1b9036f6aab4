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


def call(ops, d, E, mask, sw, int8):
    t = lambda v: None if v is None else v.transpose(-1, -2)  # noqa: E731
    one = lambda v: [] if v is None else [v]  # noqa: E731
    w1, w2 = (d["w1"], d["w2"]) if int8 else (t(d["w1"]), t(d["w2"]))
    return ops.fused_deep_moe(d["x"], d["ids"], [w1], one(d["s1"]), [w2], one(d["s2"]), d["scales"], sw[0], sw[1], sw[2],
                              sw[3], d.get("sm"), d.get("ssm"), mask, "ep", 1, 0, E, 0, 0)


# decode sizes with the layout in the dispatch, the same at its limit (2048 picks), past it (8-wave GEMMs, wave-per-token
# int8 rows above 4096 picks), and past the single-launch layouts (8192 picks), where the expert keeps its own launches
SIZES = [(3, 1024, 128, 8, 2), (40, 2048, 256, 16, 4), (256, 1024, 256, 8, 8), (300, 1024, 256, 16, 8),
         (600, 1024, 128, 8, 8), (1100, 1024, 128, 8, 8)]


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
