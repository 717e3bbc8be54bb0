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


def _with_infinite_up_weights(H, I, dtype):
    """Infinite weights in the last row of two up columns of every expert: what they reach is clamped, so the result is
    finite, unless a kernel takes that row once more to fill a slab and multiplies it by zero."""
    d = make_inputs(300, H, I, 3, 2, dtype, seed=H, w_std=0.05, bias_std=0.1)
    d["gate_up_proj"][:, H - 1, [1, 2 * I - 1]] = float("inf")
    return d


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,I", [(8, 24), (56, 72), (104, 40), (152, 264), (168, 40), (264, 72), (456, 520), (1032, 328), (1064, 1032)])
def test_infinite_weights_at_the_end_of_the_contraction(gpu, dtype, H, I):
    import yamoe_amd
    print("ragged inf", dtype, H, I, flush=True)
    d = _with_infinite_up_weights(H, I, dtype)
    out = yamoe_amd.experts(*args(to_dev(d, gpu)), 300, 3, 2)
    torch.cuda.synchronize()
    want = O.experts_loop(*args(d), compute_dtype=torch.float32)
    assert torch.isfinite(want).all()
    assert O.rel_l2(out.cpu(), want) < REL_L2_TOL[dtype]


def test_infinite_gradient_in_an_experts_last_row_fp32(gpu):
    import yamoe_amd
    d = make_inputs(301, 96, 64, 3, 3, torch.float32, seed=3, w_std=0.05, bias_std=0.1)  # every expert: rows 0 .. 300
    gy = torch.randn(301, 96, generator=torch.Generator().manual_seed(5))
    gy[300, 7] = float("inf")
    got = yamoe_amd.experts_backward(gy.to(gpu), *args(to_dev(d, gpu)), 301, 3, 3)[4].cpu()
    assert not torch.isnan(got).any()
    assert torch.isinf(got[:, :, 7]).all() and torch.isfinite(got[:, :, :7]).all() and torch.isfinite(got[:, :, 8:]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,E,I", [(300, 3, 40), (960, 48, 776)])
@pytest.mark.parametrize("H", [72, 136, 200, 584])
def test_infinite_weight_where_the_last_slab_of_an_input_gradient_begins(gpu, dtype, H, T, E, I):
    """The down projection's input gradient contracts over H with its weights stored [n][k].  An infinite weight in what the
    last slab's copies read once more past the end makes the row's gradient and its routing gradient infinite, and not NaN.
    (Few and many experts: both tile sizes of the 16-bit kernels.)"""
    import yamoe_amd
    print("ragged dgrad inf", dtype, T, H, I, E, flush=True)
    d = make_inputs(T, H, I, E, 2, dtype, seed=H, w_std=0.05, bias_std=0.1)
    slab = 32 if dtype == torch.float32 else 64
    d["down_proj"][:, 3, (H - 1) // slab * slab] = float("inf")
    gy = torch.randn(T, H, generator=torch.Generator().manual_seed(5)).to(dtype)
    gy[gy == 0] = 1.0
    d_routing = yamoe_amd.experts_backward(gy.to(gpu), *args(to_dev(d, gpu)), T, E, 2)[1].cpu()
    picked = torch.zeros(T, E, dtype=torch.bool).scatter_(1, d["router_indices"], True)
    assert torch.isinf(d_routing[picked]).all() and torch.all(d_routing[~picked] == 0)
