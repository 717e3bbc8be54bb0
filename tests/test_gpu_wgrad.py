"""Weight gradients at the sizes where their kernel changes its way: expert rows around whole slabs of 32 and around the
four slabs from which it pipelines, fewer and more row tiles than a band of four, a last band that is not full.  One group
of rows per call (and one beside it without any), all six gradients against the oracle at the tolerance of the dtype."""
import pytest
import torch

from oracle import yamoe_oracle as O
from tests.util import REL_L2_TOL, args, to_dev
from yamoe_amd.workloads import make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,I", [(264, 648), (1032, 128), (1160, 512)])
@pytest.mark.parametrize("rows", [1, 64, 95, 96, 97, 127, 128, 129, 160, 161, 193])
def test_weight_gradients_by_rows(gpu, dtype, H, I, rows):
    import yamoe_amd
    print("wgrad", dtype, H, I, rows, flush=True)
    d = make_inputs(rows, H, I, 2, 1, dtype, seed=rows, w_std=0.05, bias_std=0.1)
    d["router_indices"] = torch.ones_like(d["router_indices"])
    d["routing_weights"] = (0.1 + torch.rand(rows, 2, generator=torch.Generator().manual_seed(rows))).to(dtype)
    g = to_dev(d, gpu)
    gy = torch.randn(rows, H, generator=torch.Generator().manual_seed(5)).to(dtype)
    grads = yamoe_amd.experts_backward(gy.to(gpu), *args(g), rows, 2, 1)
    torch.cuda.synchronize()
    want = O.experts_backward(gy, *args(d), rows, compute_dtype=torch.float32)
    names = ("d_hidden", "d_routing", "d_gate_up_proj", "d_gate_up_proj_bias", "d_down_proj", "d_down_proj_bias")
    for n, a, b in zip(names, grads, want):
        r = O.rel_l2(a.cpu(), b)
        assert r < REL_L2_TOL[dtype], (n, r)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,I", [(24, 72), (128, 136), (264, 500 // 8 * 8), (1024, 128)])
@pytest.mark.parametrize("rows", [1, 31, 32, 33, 64, 65, 80, 97, 111, 112, 113, 128, 129, 160, 193])
def test_weight_and_bias_gradients_of_one_expert(gpu, dtype, H, I, rows):
    """Either kernel (small tiles up to 32 rows per expert on average, and up to 112 where no routing gives an expert more than 128:
    with a single expert, up to 112), rows around whole slabs; gradients of fewer than 32 rows, of whole and of cut tiles, of
    whole and of cut cache lines; the bias gradients, which they sum beside."""
    import yamoe_amd
    print("wgrad one", dtype, H, I, rows, flush=True)
    d = make_inputs(rows, H, I, 1, 1, dtype, seed=rows, w_std=0.05, bias_std=0.1)
    d["routing_weights"] = (0.1 + torch.rand(rows, 1, generator=torch.Generator().manual_seed(rows))).to(dtype)
    g = to_dev(d, gpu)
    gy = torch.randn(rows, H, generator=torch.Generator().manual_seed(5)).to(dtype)
    grads = yamoe_amd.experts_backward(gy.to(gpu), *args(g), rows, 1, 1)
    torch.cuda.synchronize()
    want = O.experts_backward(gy, *args(d), rows, compute_dtype=torch.float32)
    names = ("d_hidden", "d_routing", "d_gate_up_proj", "d_gate_up_proj_bias", "d_down_proj", "d_down_proj_bias")
    for n, a, b in zip(names, grads, want):
        r = O.rel_l2(a.cpu(), b)
        assert r < REL_L2_TOL[dtype], (n, r)
