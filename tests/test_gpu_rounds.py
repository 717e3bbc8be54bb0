"""Launches of few rounds of tiles whose XCD shares (equal cost, not equal length) hold more tiles than the XCD's CUs take in
those rounds: the excess goes to workgroups of other XCDs.  Experts of few rows in front, of many behind, so that the
first XCDs' shares are the long ones; one round exactly filled, one tile more, and fewer; both tile sizes.  Every output row
against the oracle: a tile that nobody took, or that two workgroups took, shows."""
import pytest
import torch

from oracle import yamoe_oracle as O
from tests.util import REL_L2_TOL, args, to_dev
from yamoe_amd.workloads import make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("light,light_rows,heavy,heavy_rows,I", [(125, 40, 125, 250, 64),   # 250 tiles of 256 x 256, one round
                                                                 (128, 40, 128, 250, 64),   # 256: exactly one round
                                                                 (129, 40, 128, 250, 64),   # 257: two rounds
                                                                 (60, 40, 68, 250, 160),    # two column tiles in the gate_up product
                                                                 (95, 20, 25, 250, 128)])   # 240 pairs of 128 x 128 tiles
def test_excess_of_a_share(gpu, light, light_rows, heavy, heavy_rows, I):
    import yamoe_amd
    E, H = light + heavy, 64
    T = light * light_rows + heavy * heavy_rows
    print("rounds", E, T, I, flush=True)
    d = make_inputs(T, H, I, E, 1, torch.bfloat16, seed=E, w_std=0.05, bias_std=0.1)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor([light_rows] * light + [heavy_rows] * heavy))
    d["router_indices"] = ids[torch.randperm(T, generator=torch.Generator().manual_seed(1))].view(T, 1).to(d["router_indices"].dtype)
    d["routing_weights"] = torch.zeros(T, E).scatter_(1, d["router_indices"].long(), 1.0).to(torch.bfloat16)
    g = to_dev(d, gpu)
    out = yamoe_amd.experts(*args(g), T, E, 1)
    torch.cuda.synchronize()
    want = O.experts_capacity(*args(d), T, compute_dtype=torch.float32)
    # row by row: activations rounded once (2^-9) and the output once more, so 1e-2 for the whole holds for most rows; a row
    # of 64 values that nearly cancel may lie above it by its share of the norm, a missing row at 1
    err = (out.cpu().float() - want.float()).norm(dim=1) / want.float().norm(dim=1)
    assert err.max() < 2 * REL_L2_TOL[torch.bfloat16], float(err.max())


@pytest.mark.parametrize("rows,capacity", [([1, 15, 16, 17, 0, 2] + [140] * 6, None),   # some stream behind the tiles
                                           ([300, 1, 300, 1, 9], None),
                                           ([100] * 8, 24),                             # a capacity that leaves only streamed ones
                                           ([100] * 4, 32)])
@pytest.mark.parametrize("H,I", [(64, 64), (200, 328)])
def test_streamed_experts_in_the_tiles_launch(gpu, rows, capacity, H, I):
    """More than 32 assignments per expert on average and few tiles: one launch of 128 x 128 tiles does these and the streamed
    experts.  With the capacities everybody streams, in launches without tiles."""
    import yamoe_amd
    E, T = len(rows), sum(rows)
    capacity = T if capacity is None else capacity
    print("carried", rows, capacity, H, I, flush=True)
    d = make_inputs(T, H, I, E, 1, torch.bfloat16, seed=T, w_std=0.05, bias_std=0.1)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(rows))
    d["router_indices"] = ids[torch.randperm(T, generator=torch.Generator().manual_seed(2))].view(T, 1).to(d["router_indices"].dtype)
    d["routing_weights"] = torch.zeros(T, E).scatter_(1, d["router_indices"].long(), 1.0).to(torch.bfloat16)
    out = yamoe_amd.experts(*args(to_dev(d, gpu)), capacity, E, 1)
    torch.cuda.synchronize()
    want = O.experts_capacity(*args(d), capacity, compute_dtype=torch.float32)
    assert O.rel_l2(out.cpu(), want) < REL_L2_TOL[torch.bfloat16]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,invalid", [([1, 15, 16, 17, 0, 2, 9] + [300] * 10, 0),      # streamed beside one and two row tiles
                                          ([5, 700, 1, 500, 16, 400, 1000, 3] * 2, 10),    # more row tiles per expert
                                          ([32, 17, 31, 1, 16, 0, 25, 8] * 2, 3000)])      # invalid ids leave no tile at all
@pytest.mark.parametrize("H,I", [(1408, 704), (1416, 712)])  # contractions that are multiples of 64 and not
def test_streamed_experts_in_a_launch_of_large_tiles(gpu, rows, invalid, H, I, dtype):
    """As above with 256 x 256 tiles in both products (too many tiles of 128 x 128: at least 23 x 11), and streamed experts of 17
    to 32 rows, which only invalid ids leave there.  Expert by expert, so that a lost slab of one row shows."""
    import yamoe_amd
    E, T = len(rows), sum(rows) + invalid
    assert (T + 64 * E) // 128 * 11 > 320 and T > 32 * E
    print("carried by large tiles", rows, invalid, H, I, dtype, flush=True)
    d = make_inputs(T, H, I, E, 1, dtype, seed=T, w_std=0.05, bias_std=0.1)
    ids = torch.cat([torch.repeat_interleave(torch.arange(E), torch.tensor(rows)), torch.tensor([-1, E])[torch.arange(invalid) % 2]])
    ids = ids[torch.randperm(T, generator=torch.Generator().manual_seed(3))]
    d["router_indices"] = ids.view(T, 1).to(d["router_indices"].dtype)
    d["routing_weights"] = torch.zeros(T, E).scatter_(1, ids.clamp(0, E - 1).view(T, 1), 1.0).to(dtype)
    out = yamoe_amd.experts(*args(to_dev(d, gpu)), T, E, 1)
    torch.cuda.synchronize()
    want = O.experts_capacity(*args(d), T, compute_dtype=torch.float32)
    out = out.cpu()
    for e in range(E):
        if rows[e]:
            assert O.rel_l2(out[ids == e], want[ids == e]) < REL_L2_TOL[dtype], e
    assert not out[(ids < 0) | (ids >= E)].any()
