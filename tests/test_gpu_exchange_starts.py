"""The exchange finds where every source's rows for an expert start by a scan of its counts, 64 experts at a time: local experts on either side of that,
more sources than waves, one that sends nothing, experts without rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from iris_testing_amd import utils  # noqa: E402
from iris_testing_amd.layers import custom_a2a  # noqa: E402
from iris_testing_amd.layers.all_to_all import SimulatedWorld, simulated_world  # noqa: E402

DEV = "cuda"


@pytest.mark.parametrize("W,E_l,cap", [(1, 1, 3), (9, 2, 5), (7, 63, 4), (8, 64, 3), (7, 65, 4), (2, 200, 2), (1, 512, 3)])
def test_starts(W, E_l, cap, H=24):
    g = torch.Generator().manual_seed(W * 1000 + E_l)
    counts = torch.randint(0, cap + 1, (W, E_l), generator=g).to(torch.int32)
    counts[W - 1, E_l - 1] = cap
    world, rows, silent = SimulatedWorld(W, rank=0), [], 1 if W > 2 else -1
    for s in range(W):
        rows.append(torch.randn(3 * s + int(counts[s].sum()), H, generator=g).bfloat16().to(DEV))
        full = torch.zeros(W, E_l, dtype=torch.int32)
        full[0] = counts[s]
        if s != silent:
            world.post(s, rows[s], full.to(DEV), torch.tensor([3 * s] + [0] * (W - 1), dtype=torch.int32, device=DEV))
    bufs = utils.alloc_shmem_buffers(None, W, E_l, cap, H, torch.bfloat16)
    bufs.token_buf.fill_(9.0)
    with simulated_world(world):
        out = custom_a2a(*world.sends[0], bufs.pca, bufs.token_buf, bufs.counts_ready, bufs.token_sync, None, W * E_l, cap).cpu()
    for s in range(W):
        at, src = 3 * s, rows[s].cpu()
        for e in range(E_l):
            c = 0 if s == silent else int(counts[s, e])
            assert torch.equal(out[e, s, :c], src[at:at + c]) and not bool(out[e, s, c:].any()), (s, e)
            at += c
