"""Products on both sides of the line between 128 x 128 and 256 x 256 tiles: the same layers on few experts (the small
tiles: at most about one per CU) and on many, with contractions of whole and of partial slab pairs, shorter and longer than
the pipelined loop, row counts around the tile edges.  Forward and all six gradients against the oracle at the tolerance of
the dtype."""
import pytest
import torch

from oracle import yamoe_oracle as O
from tests.util import REL_L2_TOL, args, to_dev
from yamoe_amd.workloads import make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,I", [(56, 392), (648, 72), (776, 648), (640, 384), (128, 576)])
@pytest.mark.parametrize("T,E", [(960, 48), (257, 2), (385, 3)])
def test_both_tile_sizes(gpu, dtype, H, I, T, E):
    import yamoe_amd
    print("tiles", dtype, T, H, I, E, flush=True)
    d = make_inputs(T, H, I, E, 2, dtype, seed=H + I, w_std=0.05, bias_std=0.1)
    g = to_dev(d, gpu)
    out = yamoe_amd.experts(*args(g), T, E, 2)
    gy = torch.randn(T, H, generator=torch.Generator().manual_seed(5)).to(dtype)
    grads = yamoe_amd.experts_backward(gy.to(gpu), *args(g), T, E, 2)
    torch.cuda.synchronize()
    want = (O.experts_capacity(*args(d), T, compute_dtype=torch.float32),
            *O.experts_backward(gy, *args(d), T, compute_dtype=torch.float32))
    names = ("out", "d_hidden", "d_routing", "d_gate_up_proj", "d_gate_up_proj_bias", "d_down_proj", "d_down_proj_bias")
    for n, a, b in zip(names, (out, *grads), want):
        r = O.rel_l2(a.cpu(), b)
        assert r < REL_L2_TOL[dtype], (n, r)
