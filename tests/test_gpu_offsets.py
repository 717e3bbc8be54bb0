"""16-bit operands that begin in the middle of a dword (contiguous views at an odd offset into their storage): the operators
give the bits that they give for operands of their own."""
import pytest
import torch

from tests.util import args, to_dev
from yamoe_amd.workloads import make_inputs

pytestmark = pytest.mark.gpu


def at_odd_offset(t):
    if t.element_size() != 2:
        return t
    s = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    v = s[1:].view(t.shape)
    assert v.is_contiguous() and v.data_ptr() % 4 == 2
    return v.copy_(t)


@pytest.mark.parametrize("T,H,I", [(300, 128, 192), (300, 72, 40), (3, 128, 192), (3, 72, 40)])
def test_experts(gpu, T, H, I):
    import yamoe_amd
    E, K = 8, 2
    d = to_dev(make_inputs(T, H, I, E, K, torch.bfloat16, seed=T, w_std=0.1, bias_std=0.1), gpu)
    gy = torch.randn(T, H, generator=torch.Generator().manual_seed(7)).to(torch.bfloat16).to(gpu)
    odd = {k: at_odd_offset(v) for k, v in d.items()}
    assert torch.equal(yamoe_amd.experts(*args(odd), T, E, K), yamoe_amd.experts(*args(d), T, E, K))
    got = yamoe_amd.experts_backward(at_odd_offset(gy), *args(odd), T, E, K)
    for a, b in zip(got, yamoe_amd.experts_backward(gy, *args(d), T, E, K)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("E", [8, 72])
def test_router(gpu, E):
    import yamoe_amd
    g = torch.Generator().manual_seed(E)
    x, w, b = (torch.randn(*s, generator=g).to(torch.float16).to(gpu) for s in ((100, 144), (E, 144), (E,)))
    idx, scores = yamoe_amd.router_topk(x, w, b, 3)
    got_idx, got_scores = yamoe_amd.router_topk(*(at_odd_offset(t) for t in (x, w, b)), 3)
    assert torch.equal(got_idx, idx) and torch.equal(got_scores, scores)
    ds = torch.randn(100, E, generator=g).to(torch.float16).to(gpu)
    got = yamoe_amd.router_topk_backward(at_odd_offset(ds), idx, *(at_odd_offset(t) for t in (scores, x, w)))
    for a, b in zip(got, yamoe_amd.router_topk_backward(ds, idx, scores, x, w)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("C,Kd", [(100, 128), (100, 40), (8, 128)])
def test_batch_mm(gpu, C, Kd):
    import yamoe_amd
    g = torch.Generator().manual_seed(C)
    x, w = (torch.randn(*s, generator=g).to(torch.bfloat16).to(gpu) for s in ((4, C, Kd), (4, Kd, 72)))
    sizes = torch.full((4,), C, dtype=torch.int32, device=gpu)
    want = yamoe_amd.batch_mm(x, w, sizes, torch.empty(4, C, 72, dtype=x.dtype, device=gpu))
    assert torch.equal(yamoe_amd.batch_mm(at_odd_offset(x), at_odd_offset(w), sizes, torch.empty_like(want)), want)
