"""The routing gradient writes every entry itself: output memory that held something else before, experts beyond a wave, more
slots than a wave has lanes, as many slots as experts, slots that repeat an expert or name none, tokens that name none at all,
dropped assignments."""
import pytest
import torch

from oracle import yamoe_oracle as O
from tests.util import REL_L2_TOL, args, to_dev
from yamoe_amd.workloads import make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,K,capacity", [(5, 3, 2, 5), (33, 64, 8, 33), (40, 65, 3, 2), (17, 130, 70, 17), (9, 200, 1, 1), (300, 16, 4, 50),
                                            (30, 4, 4, 9), (21, 64, 64, 21)])  # as many slots as experts: the dense layout
@pytest.mark.parametrize("per_slot", [False, True])
def test_every_entry_is_written(gpu, T, E, K, capacity, per_slot):
    import yamoe_amd
    H = I = 64
    print("routing grad", T, E, K, capacity, per_slot, flush=True)
    d = make_inputs(T, H, I, E, K, torch.float32, seed=T, w_std=0.1, bias_std=0.1)
    if K > 1:
        d["router_indices"][::3, 1] = d["router_indices"][::3, 0]  # an expert named twice
    d["router_indices"][1::4, K - 1] = E   # the token's last slot names nobody
    d["router_indices"][2::4, :] = -1      # no slot does
    if per_slot:
        d["routing_weights"] = torch.rand(T, K, generator=torch.Generator().manual_seed(3))
    gy = torch.randn(T, H, generator=torch.Generator().manual_seed(4))
    want = O.experts_backward(gy, *args(d), capacity, compute_dtype=torch.float64)[1]
    g = to_dev(d, gpu)
    for _ in range(2):  # the second call's output takes memory that held a poisoned tensor
        got = yamoe_amd.experts_backward(gy.to(gpu), *args(g), capacity, E, K)[1]
        assert got.shape == want.shape
        assert O.rel_l2(got.cpu(), want) < REL_L2_TOL[torch.float32]
        assert (got.cpu()[want == 0] == 0).all()
        got.fill_(float("nan"))
        del got
