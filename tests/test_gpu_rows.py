"""The row movers by slots per token: the combine of the fused op and the helper scatter take 1, 2, 4 or 8 slots in one
form each and any other number, width or alignment in a general one; few tokens are shared by several waves."""
import numpy as np
import pytest
import torch

from oracle import yamoe_oracle as O
from tests.util import REL_L2_TOL, args, oracle_forward, report, to_dev
from yamoe_amd.workloads import make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,K,capacity", [(3, 1, 3), (70, 3, 12), (33, 5, 33), (40, 8, 20), (21, 9, 21), (2100, 2, 150), (4200, 4, 900)])
def test_combine_slots(gpu, dtype, T, K, capacity):
    import yamoe_amd
    d = make_inputs(T, 64, 64, 16, K, dtype, seed=K, w_std=0.1, bias_std=0.1)
    out = yamoe_amd.experts(*args(to_dev(d, gpu)), capacity, 16, K)
    assert report("combine", out.cpu(), oracle_forward(d, capacity), REL_L2_TOL[dtype]) < REL_L2_TOL[dtype]


def test_combine_skips_dropped_rows_that_are_not_finite(gpu):
    """A dropped slot adds nothing, whatever the row that is requested in its place holds."""
    import yamoe_amd
    T, H, E, K = 40, 64, 4, 2
    d = make_inputs(T, H, 64, E, K, torch.bfloat16, seed=1)
    first = int(d["router_indices"].min())             # the expert of sorted row 0
    d["down_proj_bias"][first] = float("nan")
    capacity = 3
    out = yamoe_amd.experts(*args(to_dev(d, gpu)), capacity, E, K).cpu()
    order = np.argsort(d["router_indices"].reshape(-1).numpy(), kind="stable")
    ids = d["router_indices"].reshape(-1).numpy()[order]
    kept_first = {int(f) // K for f in order[ids == first][:capacity]}
    bad = {t for t in range(T) if not torch.isfinite(out[t].float()).all()}
    assert bad == kept_first


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float64])
@pytest.mark.parametrize("T,H,K,shift", [(9, 64, 1, 0), (50, 72, 3, 0), (31, 64, 8, 0), (17, 64, 9, 0), (40, 64, 2, 1), (8200, 16, 2, 0),
                                         (2100, 24, 8, 0)])
def test_scatter_slots(gpu, dtype, T, H, K, shift):
    """`shift`: y starts that many elements into its storage (rows that are not 16-byte aligned)."""
    import yamoe_amd
    E, C = 11, 2 * T * K // 11 // 3 + 1
    g = torch.Generator().manual_seed(T + K)
    ids, pos = O.sort_pairs(torch.randint(0, E, (T * K,), generator=g, dtype=torch.int32).numpy(), 32)
    bins = O.bincount_cumsum(ids, E, E)
    src = torch.randn(E, C, H, generator=g).to(dtype)
    w = torch.rand(T * K, generator=g).to(dtype)
    y0 = torch.randn(T, H, generator=g).to(dtype)
    y = torch.empty(T * H + shift, dtype=dtype, device=gpu)[shift:].view(T, H)
    y.copy_(y0)
    yamoe_amd.scatter(src.to(gpu), torch.from_numpy(np.asarray(pos, dtype=np.int32)).to(gpu),
                      torch.from_numpy(np.asarray(bins, dtype=np.int32)).to(gpu), w.to(gpu), y, T, E, C, K)
    want = O.padded_scatter(src, pos, bins, w, y0, T, E, C, K)
    assert report("scatter", y.cpu().double(), want, REL_L2_TOL[dtype]) < REL_L2_TOL[dtype]


@pytest.mark.parametrize("dt", [torch.int16, torch.int32, torch.int64])
@pytest.mark.parametrize("n,end_bit", [(64, 3), (1025, 8), (4096, 4), (16383, 9), (16384, 15), (16385, 4)])
def test_sort_by_one_workgroup(gpu, dt, n, end_bit):
    import yamoe_amd
    x = torch.randint(0, 1 << 14, (n,), generator=torch.Generator().manual_seed(n)).to(dt)
    k, p = torch.empty_like(x, device=gpu), torch.empty_like(x, device=gpu)
    yamoe_amd.sort(x.to(gpu), end_bit, k, p)
    want_k, want_p = O.sort_pairs(x.numpy(), end_bit)
    assert np.array_equal(k.cpu().numpy(), want_k) and np.array_equal(p.cpu().numpy(), want_p)
