"""Contraction lengths that are not multiples of 64 on the 16-bit tile kernels: the forward contracts over H and I, the
input gradients over H and 2I.  Lengths below and above the pipelined loop's eight slabs of 32, that end in the first or in
the second slab of the last pair, by one piece of 8 or all but one; forward and all six gradients against the oracle at the
tolerance of the dtype."""
import pytest
import torch

from oracle import yamoe_oracle as O
from tests.util import REL_L2_TOL, args, to_dev
from yamoe_amd.workloads import make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,I", [(8, 24), (56, 72), (120, 136), (200, 184), (248, 264), (456, 520), (1032, 328)])
@pytest.mark.parametrize("T,E", [(300, 3), (90, 2)])
def test_contractions_that_end_inside_a_slab_pair(gpu, dtype, H, I, T, E):
    import yamoe_amd
    print("ragged", dtype, T, H, I, E, flush=True)
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
