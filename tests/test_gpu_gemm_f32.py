"""fp32 grouped GEMM around the ends of its slabs of 128 and 256 of K (one slab, two, odd numbers of them, a last one of few values), with and without
16-byte loads, with one and two sets of waves and both tile sizes, against the product in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from iris_testing_amd import ops  # noqa: E402

EPS = 2.0 ** -24


@pytest.mark.parametrize("rows,groups,N", [(1, 1, 4), (33, 1, 36), (95, 3, 60), (300, 2, 132), (700, 4, 509), (2100, 2, 1028)])
@pytest.mark.parametrize("K", [4, 128, 129, 132, 252, 256, 260, 384, 388, 512, 516, 640, 772])
def test_every_number_of_slabs(rows, groups, N, K):
    g = torch.Generator().manual_seed(rows * 1000 + K)
    a, w = torch.randn((rows, K), generator=g), torch.randn((groups, K, N), generator=g)
    cnt = torch.full((groups,), rows // groups, dtype=torch.int32)
    cnt[0] += rows - int(cnt.sum())
    got = ops.grouped_gemm(a.cuda(), w.cuda(), cnt.cuda()).cpu().double()
    r0 = 0
    for e, n in enumerate(cnt.tolist()):
        x, y = a[r0:r0 + n].double(), w[e].double()
        # any order of K products and sums in fp32: each rounds once, (K + 1) eps of the sum of magnitudes at most
        bound = (K + 1) * EPS * (x.abs() @ y.abs())
        assert bool(((got[r0:r0 + n] - x @ y).abs() <= bound).all()), f"group {e}"
        r0 += n
