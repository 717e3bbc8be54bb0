"""Who works off the streaming list where a call has at most 32 assignments per expert on average: the tile launches, where the
routing makes tiles, and launches of its own, where it makes none.  Routings made for either, and for both kinds of expert in
one call; contractions of whole and of cut slab pairs, 128 x 128 tiles and (further down) 256 x 256 ones."""
import ctypes

import pytest
import torch

from oracle import yamoe_oracle as O
from tests.util import REL_L2_TOL, args, to_dev
from yamoe_amd.workloads import make_inputs

pytestmark = pytest.mark.gpu


def routed(rows):
    """Expert ids that give expert e rows[e] assignments, in a scrambled order."""
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(rows)])
    return ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(len(ids)))].view(-1, 1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,I", [(256, 192), (136, 520), (1024, 1032)])
@pytest.mark.parametrize("rows", [[16] * 8, [32, 1, 17, 0, 31, 5, 30, 16], [33, 1, 17, 0, 31, 5, 30, 16], [200, 0, 0, 3, 16, 17, 0, 1],
                                  [40] * 3 + [0] * 5, [0] * 7 + [255], [1] * 7 + [120]])
def test_streamed_beside_tiles_or_alone(gpu, dtype, H, I, rows):
    import yamoe_amd
    print("carried", dtype, H, I, rows, flush=True)
    T, E = sum(rows), len(rows)
    d = make_inputs(T, H, I, E, 1, dtype, seed=T, w_std=0.05, bias_std=0.1)
    d["router_indices"] = routed(rows)
    d["routing_weights"] = (0.1 + torch.rand(T, E, generator=torch.Generator().manual_seed(T))).to(dtype)
    g = args(to_dev(d, gpu))
    out = yamoe_amd.experts(*g, T, E, 1)
    want = O.experts_capacity(*args(d), T, compute_dtype=torch.float32)
    assert O.rel_l2(out.cpu(), want) < REL_L2_TOL[dtype]
    assert torch.equal(out, yamoe_amd.experts(*g, T, E, 1))


@pytest.mark.parametrize("E,H,I", [(32, 1032, 520), (32, 1088, 576),  # both products on 256 x 256 tiles, in up to four estimated rounds
                                   (64, 264, 4088)])                  # gate_up on such tiles, in more than four
@pytest.mark.parametrize("tiled,streamed,few", [(0, 8, 8), (0, 31, 3), (1, 8, 8), (1, 16, 1), (3, 5, 0), (8, 2, 3)])
def test_large_tiles_carry_the_list_or_leave_it(gpu, E, H, I, tiled, streamed, few):
    """`tiled` experts of 33 to 160 rows, the others of up to `streamed`; expert by expert, so that one that nobody serves shows."""
    import yamoe_amd
    print("large tiles", E, H, I, tiled, streamed, few, flush=True)
    rows = [33 + 127 * e // max(tiled - 1, 1) for e in range(tiled)] + [(streamed, few)[e % 2] for e in range(E - tiled)]
    T, cols = sum(rows), lambda n, width: (n + width - 1) // width
    rounds = (T + 128 * E) // 256 * cols(max(H, 2 * I), 256) / 256
    assert 4 * E < T <= 32 * E and E * cols(2 * I, 128) > 256          # not everything streams, gate_up on large tiles
    assert rounds <= 4 and E * cols(H, 128) > 256 if E == 32 else 4 < rounds <= 16 and T <= 24 * E
    d = make_inputs(T, H, I, E, 1, torch.bfloat16, seed=T, w_std=0.05, bias_std=0.1)
    d["router_indices"] = routed(rows)
    d["routing_weights"] = (0.1 + torch.rand(T, E, generator=torch.Generator().manual_seed(T))).to(torch.bfloat16)
    out = yamoe_amd.experts(*args(to_dev(d, gpu)), T, E, 1).cpu()
    want = O.experts_capacity(*args(d), T, compute_dtype=torch.float32)
    for e in range(E):
        mine = d["router_indices"][:, 0] == e
        assert not mine.any() or O.rel_l2(out[mine], want[mine]) < REL_L2_TOL[torch.bfloat16], e


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,I", [(64, 2304), (136, 2312)])
@pytest.mark.parametrize("rows,capacity", [([270] * 8, 0), ([257, 288, 256, 289, 512, 513, 544, 545], 0), ([288] * 7 + [20], 0),
                                           ([300] * 8, 272), ([400] * 8, 256), ([1, 16, 33, 0] + [272] * 8, 0)])
def test_last_rows_beside_whole_tiles(gpu, dtype, H, I, rows, capacity):
    """Experts of a few rows more than whole tiles, in numbers that make the gate_up product a round longer, up to
    more of them than stream."""
    import yamoe_amd
    print("remainders", dtype, H, I, rows, capacity, flush=True)
    T, E = sum(rows), len(rows)
    d = make_inputs(T, H, I, E, 1, dtype, seed=T, w_std=0.05, bias_std=0.1)
    d["router_indices"] = routed(rows)
    d["routing_weights"] = (0.1 + torch.rand(T, E, generator=torch.Generator().manual_seed(T))).to(dtype)
    g = args(to_dev(d, gpu))
    capacity = capacity or T
    out, kept = yamoe_amd.experts_keep(*g, capacity, E, 1)
    assert torch.equal(out, yamoe_amd.experts(*g, capacity, E, 1))
    want = O.experts_capacity(*args(d), capacity, compute_dtype=torch.float32)
    assert O.rel_l2(out.cpu(), want) < REL_L2_TOL[dtype]
    gy = torch.randn(T, H, generator=torch.Generator().manual_seed(3)).to(dtype).to(gpu)
    for a, b in zip(yamoe_amd.experts_backward_kept(gy, *g, kept, capacity, E, 1), yamoe_amd.experts_backward(gy, *g, capacity, E, 1)):
        assert O.rel_l2(a.cpu(), b.cpu()) < REL_L2_TOL[dtype]


@pytest.mark.parametrize("H,I", [(64, 2304), (136, 2296)])
@pytest.mark.parametrize("rows,tiles,listed", [
    ([270] * 3 + [512] * 4 + [256], 12, 3), ([257, 288, 273] + [512] * 4 + [256], 12, 3),  # a round less, few enough rows
    ([270] * 8, 8, 8), ([270] * 14, 28, 0), ([270] * 11 + [512] * 2 + [256], 27, 0),       # up to four slabs for five CUs
    ([512] * 5 + [270, 0, 0], 12, 0),                                                      # no round less
    ([768] * 13 + [522, 256, 0], 42, 1),                                                   # the fourth round
    ([38 * 256 + 10] + [256] * 4 + [0] * 11, 43, 0)])                                      # the same, most rows on one expert
def test_which_last_rows_stream(gpu, H, I, rows, tiles, listed):
    """The work lists themselves, read from the workspace, behind the five lists of the routing."""
    from yamoe_amd import _cabi
    print("last rows", H, I, rows[:8], flush=True)
    T, E = sum(rows), len(rows)
    d = make_inputs(T, H, I, E, 1, torch.bfloat16, seed=T, w_std=0.05, bias_std=0.1)
    d["router_indices"] = routed(rows)
    d["routing_weights"] = (0.1 + torch.rand(T, E, generator=torch.Generator().manual_seed(T))).to(torch.bfloat16)
    g = args(to_dev(d, gpu))
    p = _cabi.problem(*g[:4], T)
    ws = torch.zeros(_cabi.lib().yamoe_experts_workspace_bytes(ctypes.byref(p)), dtype=torch.uint8, device=gpu)
    out = _cabi.experts_forward(*g, T, workspace=ws, out=torch.full_like(g[0], float("nan")))
    up = lambda n: (n + 255) // 256 * 256
    at = 3 * up(4 * T) + up(4 * E) + up(4 * E + 4)
    assert ws[at:at + 16].view(torch.int32).tolist() == [tiles, listed, sum(n > 0 for n in rows), T]
    assert O.rel_l2(out.cpu(), O.experts_capacity(*args(d), T, compute_dtype=torch.float32)) < REL_L2_TOL[torch.bfloat16]
