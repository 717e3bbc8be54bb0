"""Helper ops at the edges of their forms: sorted input of a bin count (a wave whose values are all one, all but one, out of
range), bin counts around a wave and a block, and scatters around the slot count that one workgroup indexes and around the
expert count whose bins fit LDS."""
import numpy as np
import pytest
import torch

from oracle import yamoe_oracle as O
from tests.util import REL_L2_TOL, report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bins", [1, 63, 64, 65, 1023, 1024, 1025, 2049])
@pytest.mark.parametrize("n", [1, 64, 65, 4096, 4097, 5000])
def test_bincount_of_sorted_values(gpu, n, bins):
    import yamoe_amd
    v = np.sort(np.random.default_rng(n + bins).integers(-1, bins + 1, size=n)).astype(np.int32)
    v[: n // 2] = v[0]
    out = torch.full((bins + 3,), 77, dtype=torch.int32, device=gpu)
    yamoe_amd.bincount_cumsum(torch.from_numpy(v).to(gpu), out, bins)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), O.bincount_cumsum(v, bins + 3, bins))


@pytest.mark.parametrize("T,K,E", [(1536, 4, 8), (1537, 4, 8), (2048, 3, 1024), (700, 2, 1025), (4000, 2, 1100),
                                   (1280, 4, 32), (1707, 3, 32), (1024, 4, 33), (4097, 1, 1024), (1024, 2, 1025), (683, 3, 1025)])
def test_scatter_index_forms(gpu, T, K, E):
    import yamoe_amd
    H, C = 8, T * K // E + 2
    print("scatter T=%d K=%d E=%d C=%d" % (T, K, E, C), flush=True)
    ids = np.random.default_rng(T + E).integers(0, E, size=T * K).astype(np.int32)
    keys, pos = O.sort_pairs(ids, 32)
    bins = O.bincount_cumsum(keys, E, E)
    g = torch.Generator().manual_seed(T)
    src, w, y0 = torch.randn(E, C, H, generator=g), torch.rand(T * K, generator=g), torch.randn(T, H, generator=g)
    y = y0.clone().to(gpu)
    yamoe_amd.scatter(src.to(gpu), torch.from_numpy(pos).to(gpu), torch.from_numpy(bins).to(gpu), w.to(gpu), y, T, E, C, K)
    torch.cuda.synchronize()
    want = O.padded_scatter(src, pos, bins, w, y0, T, E, C, K)
    assert report("scatter", y.cpu().double(), want, REL_L2_TOL[torch.float32]) < REL_L2_TOL[torch.float32]


@pytest.mark.parametrize("n,out_len", [(2**31 - 4096, 3), (2**31 - 4095, 3), (2**31 - 2000, 3), (2**31 - 1, 3), (5, 2**31 - 1)])
def test_bincount_near_the_largest_size(gpu, n, out_len):
    """Sizes whose last step of loads or stores ends beyond 2^31 - 1."""
    import yamoe_amd
    print("bincount", n, out_len, flush=True)
    v = torch.zeros(n, dtype=torch.int32, device=gpu)
    v[-1], v[n // 2] = 1, -1
    out = torch.full((out_len,), 7, dtype=torch.int32, device=gpu)
    yamoe_amd.bincount_cumsum(v, out, 3)
    torch.cuda.synchronize()
    assert out[:3].tolist() == [n - 2, n - 1, n - 1]
    assert not out[3:].any()
