"""fp32 products with more output tiles than the 512 resident workgroups: every workgroup goes on from tile to tile, past
experts without rows, with one row, one slab of rows, whole tiles and remainders, and the last round is dealt out in halves."""
import pytest
import torch

from oracle import yamoe_oracle as O
from tests.util import REL_L2_TOL, args, report, to_dev
from yamoe_amd.workloads import make_inputs

pytestmark = pytest.mark.gpu

ROWS = [300, 0, 20, 129, 1, 31, 128, 640, 0, 1000, 33, 900, 777, 1024, 257, 2000]


@pytest.mark.parametrize("H,I", [(1024, 1024), (1000, 900)])
def test_gradients_over_several_rounds_of_tiles(gpu, H, I):
    import yamoe_amd
    T, E = sum(ROWS), len(ROWS)
    row_tiles = sum(-(-r // 128) for r in ROWS)
    for cols in (H, I):
        assert 512 < row_tiles * -(-cols // 128) <= 512 + 128        # input gradients: a second round, in halves
    assert E * -(-I // 128) * -(-H // 128) >= 1024                   # weight gradients: two rounds and more
    g = torch.Generator().manual_seed(H)
    d = make_inputs(T, H, I, E, 1, torch.float32, seed=H, w_std=0.05, bias_std=0.1)
    d["router_indices"] = torch.repeat_interleave(torch.arange(E), torch.tensor(ROWS))[torch.randperm(T, generator=g)].view(T, 1)
    d["routing_weights"] = torch.rand(T, E, generator=g)
    gy = torch.randn(T, H, generator=g)
    print("f32 walk", H, I, flush=True)
    dev = to_dev(d, gpu)
    out = yamoe_amd.experts(*args(dev), T, E, 1)
    grads = yamoe_amd.experts_backward(gy.to(gpu), *args(dev), T, E, 1)
    torch.cuda.synchronize()
    want = (O.experts_loop(*args(d), compute_dtype=torch.float32), *O.experts_backward_closed(gy, *args(d), T, compute_dtype=torch.float64))
    names = ("out", "d_hidden", "d_routing", "d_gate_up_proj", "d_gate_up_proj_bias", "d_down_proj", "d_down_proj_bias")
    for n, a, b in zip(names, (out, *grads), want):
        assert report(n, a.cpu(), b, REL_L2_TOL[torch.float32]) < REL_L2_TOL[torch.float32], n


@pytest.mark.parametrize("H,I", [(64, 72), (132, 260), (516, 36)])
@pytest.mark.parametrize("rows", [17, 31, 32, 33, 64, 65, 95, 96, 97, 127, 128, 129, 160, 161, 224, 225])
def test_odd_blocks_of_rows(gpu, H, I, rows):
    """Tiles of one to four blocks of 32 rows: the last of an odd number is shared by the two wave rows, k-step by k-step."""
    import yamoe_amd
    d = make_inputs(rows, H, I, 1, 1, torch.float32, seed=rows, w_std=0.05, bias_std=0.1)
    d["routing_weights"] = 0.1 + torch.rand(rows, 1, generator=torch.Generator().manual_seed(rows))
    g = args(to_dev(d, gpu))
    out = yamoe_amd.experts(*g, rows, 1, 1)
    assert O.rel_l2(out.cpu(), O.experts_capacity(*args(d), rows, compute_dtype=torch.float64)) < REL_L2_TOL[torch.float32]
    gy = torch.randn(rows, H, generator=torch.Generator().manual_seed(5))
    want = O.experts_backward(gy, *args(d), rows, compute_dtype=torch.float64)
    for a, b in zip(yamoe_amd.experts_backward(gy.to(gpu), *g, rows, 1, 1), want):
        assert O.rel_l2(a.cpu(), b) < REL_L2_TOL[torch.float32]
