"""The calls this package is measured on: what a program that uses it has it do, through the public entry points, from
the smallest call to the largest.

Five kinds of call ("path"), each with listed cases and a range that `draw` covers:

  experts   the fused expert layer in inference: one decoded token up to a 16 384-token prefill batch, 16-bit and fp32,
            whole layers and the slices of one that a tensor-parallel rank holds, even and Zipf-skewed routing
  layer     `Yamoe.forward`, the router step and the experts, in inference
  train     forward and backward of `experts_autograd`, without and with kept activations
  train_layer  forward and backward of `Yamoe.forward` with a trained router
  helpers   the helper operators composed by hand around one projection (sort, bins, gather, batch_mm, scatter)

Layer widths are the ones the package's workloads, sweep and tests use (1024, 2048, 2880), with 16, 32, 64 or 128 experts
and 2, 4 or 8 of them per token.  Weights and biases are N(0, 0.02), hidden states and output gradients N(0, 1), routing a
softmax over the top-k of random logits, as in the package's workloads; the fp32 shape of the README has unit-variance
weights and zero biases.
"""
import functools
import types

import torch

import yamoe_amd
from yamoe_amd.workloads import make_routing

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(name, path, dtype, tokens, hidden, inter, experts, top_k, zipf=0.0, capacity_factor=0.0, keep=False, w_std=0.02,
          bias_std=0.02):
    c = dict(path=path, dtype=dtype, tokens=tokens, hidden=hidden, inter=inter, experts=experts, top_k=top_k, zipf=zipf,
             capacity_factor=capacity_factor, keep=keep, w_std=w_std, bias_std=bias_std)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one user's next token on the 128-expert layer: four experts' weights, latency
        _case("decode_1", "experts", "bf16", 1, 2880, 2880, 128, 4),
        # a batch of 64 decoding users on the same layer: nearly every expert's weights for one or two rows each
        _case("decode_64", "experts", "bf16", 64, 2880, 2880, 128, 4),
        # a scheduler's step that mixes prompt chunks and decoding users: about 30 rows per expert, an odd number of tokens
        _case("chunk_1001", "experts", "bf16", 1001, 2880, 2880, 128, 4),
        # prefill of 8 x 512 tokens on the 32-expert layer
        _case("prefill_4096", "experts", "bf16", 4096, 2880, 2880, 32, 4),
        # a large prefill batch whose routing favours some experts (Zipf), 128 experts
        _case("zipf_16384", "experts", "bf16", 16384, 2880, 2880, 128, 4, zipf=1.2),
        # the README's example: 16 x 256 tokens in fp32, 8 experts
        _case("readme_fp32", "experts", "fp32", 4096, 2880, 2880, 8, 2, w_std=1.0, bias_std=0.0),
        # one rank's slice of the 32-expert layer, split four ways along the intermediate size; ragged token count
        _case("shard_2003", "experts", "bf16", 2003, 2880, 720, 32, 4),
        # the MLP block of a small model in inference, router included: one sequence of 2048 tokens
        _case("layer_2048", "layer", "fp16", 2048, 1024, 1024, 16, 2),
        # a training step of the 32-expert layer on 4096 tokens, memory as the default leaves it (recomputation)
        _case("train_4096", "train", "bf16", 4096, 2880, 2880, 32, 4),
        # a training step of the MLP block with its router, 64 experts, top-8, activations kept
        _case("train_layer_1536", "train_layer", "bf16", 1536, 2048, 2048, 64, 8, keep=True),
        # a small layer trained in fp32, assignments beyond 1.25 times an expert's fair share dropped
        _case("train_fp32", "train", "fp32", 1500, 1024, 1024, 16, 2, capacity_factor=1.25),
        # code written against the helper operators: the padded layout around one projection
        _case("helpers_2048", "helpers", "fp16", 2048, 1024, 1024, 16, 2, capacity_factor=1.5),
    ]


# ---- drawn cases -------------------------------------------------------------------------------------------------
_LAYERS = [(16, 2), (32, 4), (64, 8), (128, 4)]   # (experts, experts per token)
_FP32_COST = 16                                   # how much dearer an fp32 operation is than a 16-bit one (matrix rates)
_MOST_COST = 3.2e12                               # of zipf_16384, in 16-bit operations; readme_fp32 costs twice that


def _log_int(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def _cost(c):
    return work(c)["flops"] * (_FP32_COST if c["dtype"] == "fp32" else 1)


def draw(rng):
    path = rng.choice(["experts", "experts", "experts", "layer", "train", "train_layer", "helpers"])
    fp32 = path in ("experts", "train") and rng.random() < 0.2
    experts, top_k = rng.choice(_LAYERS[:2] if fp32 else _LAYERS if path in ("experts", "layer") else _LAYERS[:3])
    hidden = rng.choice([1024, 2048, 2880])
    inter = hidden
    if path in ("experts", "train") and rng.random() < 0.4:  # a slice of a layer, or a layer that is not square
        inter = 8 * rng.randint(hidden // 64, hidden // 8)
    low, high = {"experts": (1, 16384), "layer": (1, 8192), "train": (128, 4096), "train_layer": (128, 4096),
                 "helpers": (64, 8192)}[path]
    tokens = _log_int(rng, low, high)
    dtype = "fp32" if fp32 else rng.choice(["bf16", "bf16", "fp16"])
    zipf = rng.choice([0.0, 0.0, 1.2]) if path in ("experts", "train") else 0.0
    factor = 1.5 if path == "helpers" else rng.choice([0.0, 0.0, 0.0, 1.25]) if path == "train" else 0.0
    keep = path.startswith("train") and rng.random() < 0.5
    c = _case(None, path, dtype, tokens, hidden, inter, experts, top_k, zipf, factor, keep)
    while _cost(c) > _MOST_COST:
        c["tokens"] = c["tokens"] * 2 // 3
    return c


# ---- inputs ------------------------------------------------------------------------------------------------------
def _capacity(c):
    """Rows an expert keeps at most: all, or capacity_factor times its fair share."""
    if not c["capacity_factor"]:
        return c["tokens"]
    return max(1, int(c["capacity_factor"] * c["tokens"] * c["top_k"] / c["experts"]))


class _Block(torch.nn.Module):
    """A host model's MLP block as `Yamoe.forward` expects it."""

    def __init__(self, draw, E, H, I, K, keep):
        super().__init__()
        self.router, self.experts = torch.nn.Module(), torch.nn.Module()
        self.router.weight = torch.nn.Parameter(draw((E, H), H ** -0.5))
        self.router.bias = torch.nn.Parameter(draw((E,), 0.5))
        self.experts.gate_up_proj = torch.nn.Parameter(draw((E, H, 2 * I), 0.02))
        self.experts.gate_up_proj_bias = torch.nn.Parameter(draw((E, 2 * I), 0.02))
        self.experts.down_proj = torch.nn.Parameter(draw((E, I, H), 0.02))
        self.experts.down_proj_bias = torch.nn.Parameter(draw((E, H), 0.02))
        self.num_experts, self.top_k = E, K
        self.enable_router_grads, self.save_activations = True, keep


def prepare(case, seed):
    T, H, I, E, K = (case[k] for k in ("tokens", "hidden", "inter", "experts", "top_k"))
    dtype, dev = DTYPES[case["dtype"]], torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)

    def draw(shape, std):
        t = torch.empty(shape, dtype=dtype, device=dev)
        for part in (t if len(shape) == 3 else [t]):  # expert by expert: no fp32 copy of a whole weight tensor
            part.copy_(torch.randn(part.shape, generator=gen, device=dev) * std)
        return t

    s = types.SimpleNamespace(case=case, capacity=_capacity(case))
    s.x = draw((T, H), 1.0)
    s.gy = draw((T, H), 1.0) if case["path"].startswith("train") else None
    if "layer" in case["path"]:
        s.block = _Block(draw, E, H, I, K, case["keep"])
        s.x = s.x.view(1, T, H)
        if s.gy is not None:
            s.gy = s.gy.view(1, T, H)
            s.x.requires_grad_()
            m = s.block
            s.wrt = [s.x, m.router.weight, m.router.bias, m.experts.gate_up_proj, m.experts.gate_up_proj_bias,
                     m.experts.down_proj, m.experts.down_proj_bias]
        return s
    idx, dense = make_routing(T, E, K, torch.Generator().manual_seed(seed), renorm=case["w_std"] < 1.0, zipf=case["zipf"])
    s.idx, s.weights = idx.to(dev), dense.to(dtype).to(dev)
    if case["path"] == "helpers":
        s.w = draw((E, H, I), 0.02)
        s.slot_weights = torch.gather(s.weights, 1, s.idx).reshape(-1).contiguous()
        s.slot_experts = s.idx.reshape(-1).to(torch.int32)
        return s
    s.args = [s.x, s.idx, s.weights, draw((E, H, 2 * I), case["w_std"]), draw((E, 2 * I), case["bias_std"]),
              draw((E, I, H), case["w_std"]), draw((E, H), case["bias_std"])]
    if case["path"] == "train":
        s.wrt = [t.requires_grad_() for t in s.args if t.is_floating_point()]
    return s


# ---- one pass ----------------------------------------------------------------------------------------------------
def _helpers(s):
    c, dev = s.case, s.x.device
    T, H, I, E, K, C = c["tokens"], c["hidden"], c["inter"], c["experts"], c["top_k"], s.capacity
    ids, order = torch.empty_like(s.slot_experts), torch.empty_like(s.slot_experts)
    yamoe_amd.sort(s.slot_experts, max(1, (E - 1).bit_length()), ids, order)
    bins = torch.empty(E, dtype=torch.int32, device=dev)
    yamoe_amd.bincount_cumsum(ids, bins, E)
    x_padded = torch.empty(E, C, H, dtype=s.x.dtype, device=dev)
    yamoe_amd.gather(s.x, order, bins, x_padded, E, C, K)
    y_padded = torch.empty(E, C, I, dtype=s.x.dtype, device=dev)
    yamoe_amd.batch_mm(x_padded, s.w, bins, y_padded)
    w_sorted = yamoe_amd.index_select_out(torch.empty_like(s.slot_weights), s.slot_weights, order)
    y = torch.zeros(T, I, dtype=s.x.dtype, device=dev)
    yamoe_amd.scatter(y_padded, order, bins, w_sorted, y, T, E, C, K)
    return [y, ids, order, bins]


def run(state):
    s, c = state, state.case
    if c["path"] == "helpers":
        return _helpers(s)
    if c["path"] == "experts":
        return yamoe_amd.experts(*s.args, s.capacity, c["experts"], c["top_k"])
    if c["path"] == "layer":
        with torch.no_grad():
            return yamoe_amd.Yamoe.forward(s.block, s.x)
    if c["path"] == "train":
        out = yamoe_amd.experts_autograd(*s.args, s.capacity, c["experts"], c["top_k"], save_activations=c["keep"])
        return [out, *torch.autograd.grad(out, s.wrt, s.gy)]
    out, scores = yamoe_amd.Yamoe.forward(s.block, s.x)
    return [out, scores, *torch.autograd.grad(out, s.wrt, s.gy)]


# ---- what a pass cannot do without, and how exact it is ----------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _routed(tokens, experts, top_k, zipf, capacity):
    """(assignments kept, experts that get any) for one routing of this kind."""
    idx, _ = make_routing(tokens, experts, top_k, torch.Generator().manual_seed(0), zipf=zipf)
    counts = torch.bincount(idx.reshape(-1), minlength=experts).clamp(max=capacity)
    return int(counts.sum()), int((counts > 0).sum())


def work(case):
    T, H, I, E, K = (case[k] for k in ("tokens", "hidden", "inter", "experts", "top_k"))
    b = 4 if case["dtype"] == "fp32" else 2
    rows, active = _routed(T, E, K, case["zipf"], _capacity(case))
    if case["path"] == "helpers":
        return {"bytes": active * H * I * b + T * (H + I) * b + T * K * (4 + 8 + b) + 4 * E, "flops": 2 * H * I * rows}
    one = (3 * H * I + 2 * I + H) * b                            # an expert's weights and biases
    routing = T * K * 8 + T * E * b
    bytes_, flops = active * one + 2 * T * H * b + routing, 6 * H * I * rows
    if "layer" in case["path"]:                                  # the router's weights, product and scores
        bytes_ += (E * H + E) * b - T * K * 8
        flops += 2 * T * H * E
    if case["path"].startswith("train"):                         # each product twice more, every gradient written once
        bytes_ += E * one + 2 * T * H * b + (E * H + E if "layer" in case["path"] else T * E) * b
        flops *= 3
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    # about four times the distance of the outputs from the same pass in float64
    return {"rel": {"bf16": 1e-2, "fp16": 2e-3, "fp32": 8e-6}[case["dtype"]]}
