"""Which block runs which tile of a grouped GEMM: row counts at the edges of the tile classes (32 | 33, 128 | 129,
383 | 384 rows), with and without heavy experts, more and fewer tiles than blocks.  A schedule that drops, repeats or
misplaces a tile leaves wrong rows: the chained launch is compared bit for bit with the two calls (themselves compared
with the oracle in test_gpu_gmm.py), the int8 GEMM with its exact integer sums."""
import copy

import pytest
import torch
import torch.nn.functional as F

from test_gmm_plan import plan, tiles  # noqa: F401 (plan is a fixture)
from test_gpu_chain import DT_BF16, DT_FP8, Case, lib  # noqa: F401 (lib is a fixture)

pytestmark = pytest.mark.gpu

EDGES = [32, 33, 128, 129, 383, 1, 0, 64]
PREFILL = [
    (EDGES, 2048, 2048),                                # no heavy expert
    (EDGES + [384], 2048, 2048),                        # heavy tiles on some blocks, the others free at once
    ([384, 700] * 9 + EDGES, 2048, 2048),               # more heavy tiles than blocks
    ([40, 20, 130] * 12, 2048, 2048),                   # several rounds of light tiles through the queue
    (EDGES, 256, 384),                                  # reductions of 2 and 3 k-steps: no tile primes the next
    # heavy experts alone: the last round of the two calls' 256-row tiles as halves (the chained launch keeps them whole)
    ([384, 700, 641], 2048, 2048),                      # the only round
    ([2304, 2290], 2048, 2048),                         # after a full one
]


@pytest.mark.parametrize("dt", [DT_FP8, DT_BF16])
@pytest.mark.parametrize("case", range(len(PREFILL)))
def test_chained_prefill_tiles_at_class_edges(lib, dt, case):  # noqa: F811
    counts, H, I = PREFILL[case]
    print(f"chained schedule counts={counts} dt={dt}", flush=True)
    c = Case(counts, H, I, dt, 50 + case)
    assert c.cap > 48 * c.L  # the 8-wave kernel
    for _ in range(2):
        c.new_outputs()
        c.run_pair(lib)
        c.run_chain(lib)
        c.assert_same()
    assert lib.sync_status() == 0


@pytest.mark.parametrize("counts", [[1, 0, 1, 0, 0, 0, 0, 0], [0, 3], [33, 1, 32, 40], [1] * 40, [64, 65, 31] * 8 + [0] * 8,
                                    [40] * 48])
@pytest.mark.parametrize("dt", [DT_FP8, DT_BF16])
def test_chained_decode_tiles(lib, dt, counts):  # noqa: F811
    # fewer GMM2 tiles than blocks without GMM1 work (they spread over the free blocks), 32-row tiles throughout; the
    # last: 64-row tiles alone
    print(f"chained decode counts={counts} dt={dt}", flush=True)
    c = Case(counts, 1024, 512, dt, 70)
    c.run_pair(lib)
    c.run_chain(lib)
    c.assert_same()
    assert lib.sync_status() == 0


# 32- and 64-row tiles in one 4-wave launch, some experts of several 64-row tiles (GMM1's second round begins in the
# 64-row tiles, in the 32-row ones, between them)
BOTH = [([64, 65, 31, 7] * 12, 2048, 1024), ([33, 1, 130, 32, 40] * 10, 1024, 1408), ([64, 65, 31] * 8 + [0] * 8, 1024, 2048)]


def rows_to(c, cap):
    """The case's groups with a capacity of cap rows."""
    b = copy.copy(c)
    b.x = F.pad(c.x.view(torch.uint8 if c.dt == DT_FP8 else torch.int16), (0, 0, 0, cap - c.cap)).view(c.x.dtype)
    b.xs = None if c.xs is None else F.pad(c.xs, (0, cap - c.cap)).contiguous()
    b.cap = cap
    b.new_outputs()
    return b


@pytest.mark.parametrize("dt", [DT_FP8, DT_BF16])
@pytest.mark.parametrize("counts,H,I", BOTH)
def test_decode_tiles_of_both_heights(lib, plan, counts, H, I, dt):  # noqa: F811
    # against the same groups at a prefill capacity: the 8-wave kernels, every sum in the same order
    print(f"decode tiles of both heights counts={counts[:5]}.. dt={dt}", flush=True)
    c = Case(counts, H, I, dt, 90)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert c.cap <= 48 * c.L and not plan.rows32(*tiles(counts, I // 128), cus) and min(n for n in counts if n) <= 32
    b = rows_to(c, 48 * c.L + 1)
    for _ in range(2):
        c.new_outputs()
        c.run_pair(lib)
        c.run_chain(lib)
        c.assert_same()
    b.run_pair(lib)
    torch.cuda.synchronize()
    u = lambda t: t.view(torch.uint8) if t.dtype == torch.float8_e4m3fn else t.view(torch.int16)  # noqa: E731
    (h0, hs0, y0), (h1, hs1, y1) = b.out["pair"], c.out["pair"]
    assert torch.equal(u(h0)[:c.M], u(h1)[:c.M]) and torch.equal(u(y0)[:c.M], u(y1)[:c.M])
    assert hs0 is None or torch.equal(hs0[:, :c.M], hs1[:, :c.M])
    assert lib.sync_status() == 0


@pytest.mark.parametrize("counts,H,I", BOTH)
def test_int8_decode_tiles_of_both_heights(counts, H, I):
    import umdk_amd  # noqa: F401
    print(f"int8 decode tiles of both heights counts={counts[:5]}..", flush=True)
    ops, L, M = torch.ops.umdk_cam_op_lib, len(counts), sum(counts)
    g = torch.Generator(device="cuda").manual_seed(M)
    codes = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device="cuda", generator=g)  # noqa: E731
    rand = lambda *s: torch.rand(*s, device="cuda", generator=g) * 0.01  # noqa: E731
    x, xs, w1, s1, w2, s2 = codes(M, H), rand(M), codes(L, 2 * I, H), rand(L, 2 * I), codes(L, H, I), rand(L, H)
    gl = torch.tensor(counts, dtype=torch.int64, device="cuda")
    more = 48 * L + 1 - M  # a capacity for the 8-wave kernels
    h, hs = ops.grouped_matmul_swiglu(x, xs, gl, w1, s1, 2)
    h8, hs8 = ops.grouped_matmul_swiglu(F.pad(x, (0, 0, 0, more)), F.pad(xs, (0, more)), gl, w1, s1, 2)
    assert torch.equal(h, h8[:M]) and torch.equal(hs, hs8[:M])
    y, at = ops.grouped_matmul(h, hs, gl, w2, s2), 0
    for e, n in enumerate(counts):  # exact sums, as in the test below
        ref = (((h[at:at + n].double() @ w2[e].double().T).float() * s2[e]) * hs[at:at + n, None]).bfloat16()
        assert torch.equal(y[at:at + n].view(torch.int16), ref.view(torch.int16)), f"expert {e} of {n} rows"
        at += n


@pytest.mark.parametrize("counts", [EDGES, EDGES + [384, 900], [2100, 40, 2100, 150, 3, 129, 128], [384, 0, 900]])
def test_int8_tiles_at_class_edges(counts):
    # int8 x int8 sums in fp64 are exact (|sum| < 2^53), then the kernel's own fp32 sequence and bf16 rounding
    import umdk_amd  # noqa: F401
    print(f"int8 schedule counts={counts}", flush=True)
    L, M, H, I = len(counts), sum(counts), 4096, 2048
    g = torch.Generator(device="cuda").manual_seed(len(counts))
    x = torch.randint(-127, 128, (M, I), dtype=torch.int8, device="cuda", generator=g)
    w = torch.randint(-127, 128, (L, H, I), dtype=torch.int8, device="cuda", generator=g)
    xs = torch.rand(M, device="cuda", generator=g) * 0.01
    ws = torch.rand(L, H, device="cuda", generator=g) * 0.01
    gl = torch.tensor(counts, dtype=torch.int64, device="cuda")
    y = torch.ops.umdk_cam_op_lib.grouped_matmul(x, xs, gl, w, ws)
    at = 0
    for e, n in enumerate(counts):
        acc = x[at:at + n].double() @ w[e].double().T
        ref = ((acc.float() * ws[e]) * xs[at:at + n, None]).bfloat16()
        assert torch.equal(y[at:at + n].view(torch.int16), ref.view(torch.int16)), f"expert {e} of {n} rows"
        at += n
