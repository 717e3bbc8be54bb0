"""A capacity that leaves no expert more rows than the streaming kernels take: every expert is theirs, whatever the number of
assignments.  The forward then gives the bits of the stages called one by one (whose products are launches of their own), not
those of streamed experts that ride in a tile launch (other partial sums); one row more of capacity and there are tiles."""
import pytest
import torch

from oracle import yamoe_oracle as O
from tests.util import REL_L2_TOL, args, to_dev
from yamoe_amd.workloads import make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("capacity", [1, 16, 17, 32, 33])
@pytest.mark.parametrize("T,H,I,E,K", [(400, 640, 320, 8, 2), (700, 264, 520, 5, 1)])
def test_small_capacity(gpu, T, H, I, E, K, capacity, dtype):
    import yamoe_amd
    from yamoe_amd import _cabi
    print("capacity", T, H, I, E, K, capacity, dtype, flush=True)
    d = make_inputs(T, H, I, E, K, dtype, seed=T + capacity, w_std=0.05, bias_std=0.1)
    g = to_dev(d, gpu)
    out = yamoe_amd.experts(*args(g), capacity, E, K)
    torch.cuda.synchronize()
    want = O.experts_capacity(*args(d), capacity, compute_dtype=torch.float32)
    assert O.rel_l2(out.cpu(), want) < REL_L2_TOL[dtype]
    if capacity <= 32:
        _, si, counts, offsets, inv = _cabi.route(g["router_indices"], E, capacity)
        sched = _cabi.build_schedule(counts, offsets, T * K, capacity, 32)
        act = _cabi.gate_up(g["hidden"], si, g["gate_up_proj"], g["gate_up_proj_bias"], sched, K)
        y = _cabi.down(act, g["down_proj"], g["down_proj_bias"], sched)
        assert torch.equal(out, _cabi.combine(y, inv, g["router_indices"], g["routing_weights"], T, K, E))
