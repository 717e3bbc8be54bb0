"""The streaming kernels where a call has few (expert, column slab) pairs and several workgroups share one: contractions of a
few steps and of many, whole and cut slabs, one and two blocks of 16 rows, experts in chunks of 32 rows; fp32 on the same path.
The parts are added up in their order, so a call gives the same bits every time, also when it is replayed from a graph."""
import ctypes

import pytest
import torch

from oracle import yamoe_oracle as O
from tests.util import REL_L2_TOL, args, to_dev
from yamoe_amd.workloads import make_inputs

pytestmark = pytest.mark.gpu

SHAPES = [  # T, H, I, E, K, one expert for all
    (1, 64, 72, 8, 1, False), (1, 128, 256, 8, 2, False), (2, 520, 1032, 16, 2, False), (1, 2880, 360, 32, 4, False),
    (3, 1000, 40, 4, 1, False), (16, 1024, 200, 8, 2, False), (17, 264, 128, 16, 1, True), (31, 1536, 64, 8, 1, True),
    (1, 512, 64, 8, 2, False), (1, 520, 136, 32, 1, False), (4, 768, 384, 32, 2, False),  # fewer steps in a part than eight waves
    (32, 256, 264, 8, 1, True), (33, 2048, 128, 16, 1, True), (64, 512, 264, 16, 1, True), (40, 136, 520, 64, 4, False),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H,I,E,K,one", SHAPES)
def test_shared_slabs(gpu, T, H, I, E, K, one, dtype):
    import yamoe_amd
    print("stream parts", T, H, I, E, K, one, dtype, flush=True)
    d = make_inputs(T, H, I, E, K, dtype, seed=T + H, w_std=0.05, bias_std=0.1)
    if one:
        d["router_indices"] = torch.full_like(d["router_indices"], E - 2)
        d["routing_weights"] = (0.1 + torch.rand(T, E, generator=torch.Generator().manual_seed(T))).to(dtype)
    g = args(to_dev(d, gpu))
    out = yamoe_amd.experts(*g, T, E, K)
    want = O.experts_capacity(*args(d), T, compute_dtype=torch.float64 if dtype == torch.float32 else torch.float32)
    assert O.rel_l2(out.cpu(), want) < REL_L2_TOL[dtype]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        again = yamoe_amd.experts(*g, T, E, K)
    for _ in range(3):
        again.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, again)
        assert torch.equal(out, yamoe_amd.experts(*g, T, E, K))


@pytest.mark.parametrize("capacity", [0, 1, 16, 17, 32, 40])
def test_fp32_streams_up_to_a_capacity(gpu, capacity):
    """48 tokens of one expert among 16: chunks of 32 rows, cut by the capacity; gradients of a kept forward as of a recomputed one."""
    import yamoe_amd
    T, H, I, E, K = 48, 264, 520, 16, 1
    d = make_inputs(T, H, I, E, K, torch.float32, seed=capacity, w_std=0.05, bias_std=0.1)
    d["router_indices"] = torch.full_like(d["router_indices"], 3)
    d["routing_weights"] = 0.1 + torch.rand(T, E, generator=torch.Generator().manual_seed(1))
    g = args(to_dev(d, gpu))
    out, kept = yamoe_amd.experts_keep(*g, capacity, E, K)
    assert torch.equal(out, yamoe_amd.experts(*g, capacity, E, K))
    want = O.experts_capacity(*args(d), capacity, compute_dtype=torch.float64)
    assert O.rel_l2(out.cpu(), want) < REL_L2_TOL[torch.float32] or (capacity == 0 and not out.any())
    gy = torch.randn(T, H, generator=torch.Generator().manual_seed(3)).to(gpu)
    for a, b in zip(yamoe_amd.experts_backward_kept(gy, *g, kept, capacity, E, K), yamoe_amd.experts_backward(gy, *g, capacity, E, K)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("C", [1, 15, 16, 17, 32, 33])
def test_fp32_batch_mm_of_few_rows(gpu, C):
    import yamoe_amd
    E, Kd, Nd = 3, 148, 260
    gen = torch.Generator().manual_seed(C)
    x, w = torch.randn(E, C, Kd, generator=gen), torch.randn(E, Kd, Nd, generator=gen)
    y = torch.empty(E, C, Nd, device=gpu)
    yamoe_amd.batch_mm(x.to(gpu), w.to(gpu), torch.full((E,), C, dtype=torch.int32, device=gpu), y)
    assert O.rel_l2(y.cpu(), torch.bmm(x.double(), w.double())) < REL_L2_TOL[torch.float32]


@pytest.mark.parametrize("T,H,I,E,K,one", [(60, 264, 200, 8, 2, False), (128, 136, 264, 8, 1, True), (129, 136, 264, 8, 1, True),
                                           (64, 512, 1000, 16, 4, False), (65, 512, 72, 16, 4, False)])
def test_fp32_up_to_sixteen_assignments_per_expert(gpu, T, H, I, E, K, one):
    """Streamed up to there, tiles beyond; a whole batch on one expert in chunks of 32 rows."""
    import yamoe_amd
    d = make_inputs(T, H, I, E, K, torch.float32, seed=T, w_std=0.05, bias_std=0.1, zipf=1.2)
    if one:
        d["router_indices"] = torch.full_like(d["router_indices"], 5)
        d["routing_weights"] = 0.1 + torch.rand(T, E, generator=torch.Generator().manual_seed(T))
    g = args(to_dev(d, gpu))
    out = yamoe_amd.experts(*g, T, E, K)
    assert O.rel_l2(out.cpu(), O.experts_capacity(*args(d), T, compute_dtype=torch.float64)) < REL_L2_TOL[torch.float32]
    gy = torch.randn(T, H, generator=torch.Generator().manual_seed(3))
    want = O.experts_backward(gy, *args(d), T, compute_dtype=torch.float64)
    for a, b in zip(yamoe_amd.experts_backward(gy.to(gpu), *g, T, E, K), want):
        assert O.rel_l2(a.cpu(), b) < REL_L2_TOL[torch.float32]


@pytest.mark.parametrize("rows,streams", [([16] * 128, True), ([2048] + [0] * 127, False), ([600] * 3 + [8] * 25 + [0] * 100, False),
                                          ([500] + [12] * 127, True), ([33] * 30 + [8] * 98, True), ([400] * 5 + [0] * 123, False),
                                          ([129] * 8 + [8] * 120, True)])
def test_fp32_streams_everything_or_nothing_by_the_routing(gpu, rows, streams):
    """At most 16 assignments per expert on average, and more of them than streaming can take from a single expert at no loss: the
    device decides between the two kernels.  The work lists (behind the five lists of the routing) tell which; both give the
    oracle's result, and a recomputation takes the way of the forward."""
    import yamoe_amd
    from yamoe_amd import _cabi
    T, H, I, E = sum(rows), 1024, 512, 128
    print("fp32 either", rows[:8], flush=True)
    gen = torch.Generator(device=gpu).manual_seed(T)
    r = lambda *s: torch.randn(*s, generator=gen, device=gpu) * 0.05
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(rows)])
    ids = ids[torch.randperm(T, generator=torch.Generator().manual_seed(1))].view(T, 1).to(gpu)
    g = [r(T, H), ids, 0.1 + torch.rand(T, E, generator=gen, device=gpu), r(E, H, 2 * I), r(E, 2 * I), r(E, I, H), r(E, H)]
    p = _cabi.problem(*g[:4], T)
    ws = torch.zeros(_cabi.lib().yamoe_experts_workspace_bytes(ctypes.byref(p)), dtype=torch.uint8, device=gpu)
    out = _cabi.experts_forward(*g, T, workspace=ws, out=torch.full_like(g[0], float("nan")))
    up = lambda n: (n + 255) // 256 * 256
    at = 3 * up(4 * T) + up(4 * E) + up(4 * E + 4)
    tiles, listed, active, kept = ws[at:at + 16].view(torch.int32).tolist()
    assert (active, kept) == (sum(n > 0 for n in rows), T)
    assert (tiles == 0, listed > 0) == (streams, streams)
    used = [e for e, n in enumerate(rows) if n][:6]     # (the oracle on a few experts' tokens: 800 MB of weights)
    some = torch.isin(ids.view(-1).cpu(), torch.tensor(used)).nonzero().view(-1)[:200]
    x, e, w = (t.cpu()[some] for t in g[:3])
    sub = [x, torch.searchsorted(torch.tensor(used), e.view(-1)).view(-1, 1), w[:, used].contiguous()] + [t[used].cpu() for t in g[3:]]
    assert O.rel_l2(out[some.to(gpu)].cpu(), O.experts_capacity(*sub, T, compute_dtype=torch.float64)) < REL_L2_TOL[torch.float32]
    again, k = yamoe_amd.experts_keep(*g, T, E, 1)
    assert torch.equal(again, out)
    gy = r(T, H)
    for a, b in zip(yamoe_amd.experts_backward_kept(gy, *g, k, T, E, 1), yamoe_amd.experts_backward(gy, *g, T, E, 1)):
        assert torch.equal(a, b)


def test_fp32_choice_is_made_anew_at_every_replay(gpu):
    """Captured once; the routing in the captured buffer changes between replays from one that streams to one that is tiled."""
    import yamoe_amd
    T, H, I, E = 2048, 1024, 512, 128
    gen = torch.Generator(device=gpu).manual_seed(9)
    r = lambda *s: torch.randn(*s, generator=gen, device=gpu) * 0.05
    g = [r(T, H), torch.zeros(T, 1, dtype=torch.int64, device=gpu), 0.1 + torch.rand(T, E, generator=gen, device=gpu), r(E, H, 2 * I), r(E, 2 * I),
         r(E, I, H), r(E, H)]
    even, one = (torch.arange(T, device=gpu) % E).view(T, 1), torch.full((T, 1), 7, device=gpu)
    yamoe_amd.experts(*g, T, E, 1)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = yamoe_amd.experts(*g, T, E, 1)
    for ids in (even, one, even, one):
        g[1].copy_(ids)
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, yamoe_amd.experts(*g, T, E, 1))
