"""The one-launch dispatch layout at the edges of its chunks (1024 entries) and of its range (32768 entries of 4096
tokens; past either the three-launch layout runs), against the oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,E", [(1, 1, 1), (1023, 1, 7), (1024, 1, 8), (1025, 1, 512), (341, 3, 160), (171, 6, 160),
                                   (1300, 7, 60), (2048, 16, 512), (4096, 8, 256), (4097, 2, 256), (4096, 9, 64)])
def test_layout_matches_oracle(T, K, E):
    import umdk_amd  # noqa: F401
    print(f"layout T={T} K={K} E={E}", flush=True)
    g = torch.Generator().manual_seed(T * K + E)
    for skew in (False, True):
        hot = max(K, E // 8) if skew else E  # skewed: few experts take every pick
        ids = torch.rand(T, hot, generator=g).argsort(1)[:, :K].contiguous() if hot >= K else torch.randint(E, (T, K))
        ids[torch.rand(T, K, generator=g) < 0.05] = -1
        nte, sti = torch.ops.umdk_cam_op_lib.get_dispatch_layout(ids.cuda(), E, 1)
        _, rnte, _, rsti = orc.dispatch_layout(ids.numpy().astype(np.int64), E, 1)
        assert np.array_equal(nte.cpu().numpy(), rnte)
        assert np.array_equal(sti.cpu().numpy(), rsti)


@pytest.mark.parametrize("T,K,E", [(1025, 1, 3), (2048, 16, 512), (4096, 8, 8)])
def test_layout_of_equal_picks_matches_oracle(T, K, E):
    # one expert takes (nearly) every pick, within a token too: whole waves agree, then a few lanes differ or are out of
    # range, among them a wave's first
    import umdk_amd  # noqa: F401
    print(f"layout of equal picks T={T} K={K} E={E}", flush=True)
    g = torch.Generator().manual_seed(T + K)
    for others in (0.0, 0.02):
        ids = torch.full((T, K), E - 1)
        odd = torch.rand(T, K, generator=g) < others
        ids[odd] = torch.randint(-1, E + 1, (int(odd.sum()),), generator=g)
        ids.view(-1)[64:65] = -1 if others else E - 1
        nte, sti = torch.ops.umdk_cam_op_lib.get_dispatch_layout(ids.cuda(), E, 1)
        _, rnte, _, rsti = orc.dispatch_layout(ids.numpy().astype(np.int64), E, 1)
        assert np.array_equal(nte.cpu().numpy(), rnte)
        assert np.array_equal(sti.cpu().numpy(), rsti)
