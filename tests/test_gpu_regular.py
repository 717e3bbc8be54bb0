"""Products over a regular layout (every expert has the same rows), which need no work list: rows per expert around the
streaming limit and the tile heights, experts of many row tiles (walked in bands), both tile sizes, one expert alone, ragged
contractions.  Against the product in float64."""
import pytest
import torch

from oracle import yamoe_oracle as O
from tests.util import REL_L2_TOL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,C,K,N", [(3, 32, 64, 264), (3, 33, 72, 264), (40, 96, 64, 304), (7, 128, 128, 640), (7, 129, 200, 640),
                                     (5, 256, 64, 1032), (5, 257, 72, 1032), (130, 40, 64, 520), (1, 5000, 128, 264),
                                     (2, 4097, 64, 1288), (300, 65, 64, 264)])
def test_batch_mm_regular(gpu, E, C, K, N):
    import yamoe_amd
    print("regular", E, C, K, N, flush=True)
    g = torch.Generator().manual_seed(E + C)
    x, w = torch.randn(E, C, K, generator=g).to(torch.bfloat16), (torch.randn(E, K, N, generator=g) * 0.05).to(torch.bfloat16)
    y = torch.full((E, C, N), float("nan"), dtype=torch.bfloat16, device=gpu)
    yamoe_amd.batch_mm(x.to(gpu), w.to(gpu), torch.arange(1, E + 1, dtype=torch.int32, device=gpu) * C, y)
    torch.cuda.synchronize()
    for e in range(E):  # expert by expert: a tile at the wrong place is not lost in the mean
        assert O.rel_l2(y[e].cpu(), x[e].double() @ w[e].double()) < REL_L2_TOL[torch.bfloat16], e
