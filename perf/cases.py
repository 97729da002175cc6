r"""The workloads whose time counts: whole MoE layers through the package's public
entry points, as a training step or an inference call of a user's program makes them.

A case is one layer and one batch:

  gate      "naive" (NaiveGate, the default), "chosen" (a user's own gate: Zipf(1.2)
            choices clipped by `limit_by_capacity` at factor 1.25), "gshard" (GShardGate
            with its balance loss), "switch" (SwitchGate, top-1)
  dtype     "bf16", "f16" or "f32": parameters, inputs and outputs
  tokens, d_model, d_hidden, experts, top_k
  dead      experts whose gate bias keeps every token away from them
  train     True: forward, backward, gradients of the input and of every parameter;
            False: forward under no_grad
  layout    "fused": expert parameters as [E, out, in]; "list": one module per expert
  act       the activation between the two expert layers: "gelu" (the default) or "relu"

Weights are N(0, 0.02), inputs and output gradients N(0, 1), gate weights scaled so that
the logits are N(0, 1): near-uniform expert load with the raggedness of random routing.
"""
import math

import torch
import torch.nn.functional as F

from fastmoe_amd import BaseGate, FMoETransformerMLP, GShardGate, NaiveGate, SwitchGate
from fastmoe_amd.gates import limit_by_capacity

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
ZIPF_S, CAPACITY_FACTOR = 1.2, 1.25
FIELDS = ("gate", "dtype", "tokens", "d_model", "d_hidden", "experts", "top_k", "dead", "train",
          "layout", "act")


def _case(name, *values):
    return dict(zip(("name",) + FIELDS, (name,) + values))


def listed():
    return [
        # the smallest training step: the layer of a toy or unit-test model, all launches
        _case("train_small", "naive", "f32", 512, 128, 256, 4, 2, 0, True, "fused", "gelu"),
        # a balanced layer of an ordinary language model
        _case("train_balanced", "naive", "bf16", 8192, 1024, 4096, 16, 2, 0, True, "fused", "gelu"),
        # popular and unpopular experts, the popular ones cut off at their capacity
        _case("train_capacity", "chosen", "bf16", 16384, 2048, 8192, 64, 2, 0, True, "fused", "gelu"),
        # the largest layer of one GPU: few wide experts, the GEMMs are everything
        _case("train_large", "naive", "bf16", 16384, 4096, 14336, 8, 2, 0, True, "fused", "gelu"),
        # many narrow experts, eight per token, some never chosen
        _case("train_fine", "naive", "bf16", 8192, 2048, 1408, 128, 8, 13, True, "fused", "gelu"),
        # GShard in half precision on a ragged batch: capacity, balance loss, ReLU experts
        _case("train_gshard", "gshard", "f16", 3001, 768, 3072, 16, 2, 0, True, "fused", "relu"),
        # a module per expert (the layout of existing checkpoints) in full precision
        _case("train_list", "naive", "f32", 2000, 512, 2048, 8, 2, 0, True, "list", "gelu"),
        # feature sizes that no tile divides: word-vector sized embeddings
        _case("train_odd", "naive", "bf16", 1000, 300, 1200, 8, 2, 0, True, "fused", "gelu"),
        # one decode step of a batch of sequences through an ordinary layer
        _case("decode", "naive", "bf16", 32, 1024, 4096, 16, 2, 0, False, "fused", "gelu"),
        # the same through the largest layer: every expert's weights for a few rows each
        _case("decode_large", "naive", "bf16", 64, 4096, 14336, 8, 2, 0, False, "fused", "gelu"),
        # a prompt through many narrow experts
        _case("prefill_fine", "naive", "bf16", 2047, 2048, 1408, 128, 8, 13, False, "fused", "gelu"),
        # top-1 evaluation
        _case("eval_switch", "switch", "bf16", 4096, 768, 3072, 32, 1, 0, False, "fused", "relu"),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        gate = rng.choice(("naive", "naive", "naive", "chosen", "gshard", "switch"))
        dtype = rng.choice(("bf16", "bf16", "bf16", "f16", "f32"))
        train = rng.random() < 0.6
        tokens = _spread(rng, 128, 16384) if train else _spread(rng, 16, 16384)
        d_model = _spread(rng, 128, 4096)
        d_hidden = int(d_model * rng.choice((0.6875, 2, 3.5, 4)))
        kind = rng.random()
        step = 64 if kind < 0.7 else (8 if kind < 0.9 else 2)
        d_model = max(step, d_model // step * step)
        d_hidden = max(step, d_hidden // step * step)
        experts = 2 ** rng.randint(2, 7)
        top_k = {"gshard": 2, "switch": 1, "chosen": 2}.get(gate) or rng.choice((1, 2, 2, 2, 4, 8))
        layout = "list" if experts <= 8 and rng.random() < 0.25 else "fused"
        act = "relu" if gate in ("gshard", "switch") else "gelu"
        dead = experts // 10 if gate == "naive" and rng.random() < 0.25 else 0
        flops = (12.0 if train else 4.0) * tokens * top_k * d_model * d_hidden
        if top_k > experts - dead or experts * d_model * d_hidden > 2 ** 30:
            continue
        if gate in ("gshard", "switch") and tokens < experts:   # a capacity of no rows at all
            continue
        # full precision costs about 16 times as much, sizes off the 16-byte grid up to 100
        odd = d_model % 8 or d_hidden % 8
        if flops * (100 if odd else 16 if dtype == "f32" else 1) > 1.5e13:
            continue
        return dict(zip(FIELDS, (gate, dtype, tokens, d_model, d_hidden, experts, top_k, dead,
                                 train, layout, act)))


class _ChosenGate(BaseGate):
    """A user's own gate: choices made elsewhere (Zipf popularity), scored by a learned
    softmax and clipped to the experts' capacity."""

    def __init__(self, d_model, num_expert, world_size, top_k=2):
        super().__init__(num_expert, world_size)
        self.logits = torch.nn.Parameter(torch.zeros(1, top_k))

    def fill(self, case, gen):
        t, e, k = case["tokens"], case["experts"], case["top_k"]
        p = torch.arange(1, e + 1, dtype=torch.float32, device="cuda") ** -ZIPF_S
        self.idx = torch.multinomial(p.expand(t, -1), k, replacement=False, generator=gen)
        self.logits.data = torch.randn(t, k, device="cuda", generator=gen)
        self.capacity = math.ceil(CAPACITY_FACTOR * t * k / e)
        self.dtype = DTYPES[case["dtype"]]

    def forward(self, inp):
        score = F.softmax(self.logits, dim=-1).to(self.dtype)
        _, _, idx = limit_by_capacity(self.idx, self.num_expert, 1, self.capacity)
        return idx, score


class _GShard(GShardGate):
    """GShardGate without its random dropping, so that equal inputs give equal outputs."""

    def __init__(self, d_model, num_expert, world_size, topk=2, gate_bias=True):
        super().__init__(d_model, num_expert, world_size, topk, random_routing=False,
                         gate_bias=gate_bias)


class _Switch(SwitchGate):
    """SwitchGate without its jitter, for the same reason."""

    def __init__(self, d_model, num_expert, world_size, topk=1, gate_bias=True):
        super().__init__(d_model, num_expert, world_size, topk, switch_eps=0.0,
                         gate_bias=gate_bias)


GATES = {"naive": NaiveGate, "chosen": _ChosenGate, "gshard": _GShard, "switch": _Switch}


def _layer(case):
    # parameters are born on the GPU: a billion of them on the host would take seconds
    torch.set_default_tensor_type(torch.cuda.FloatTensor)
    try:
        layer = FMoETransformerMLP(
            num_expert=case["experts"], d_model=case["d_model"], d_hidden=case["d_hidden"],
            top_k=case["top_k"], gate=GATES[case["gate"]], fused=case["layout"] == "fused",
            activation=torch.nn.GELU() if case["act"] == "gelu" else torch.nn.ReLU())
    finally:
        torch.set_default_tensor_type(torch.FloatTensor)
    return layer.to(DTYPES[case["dtype"]])


def prepare(case, seed):
    dtype = DTYPES[case["dtype"]]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    layer = _layer(case)
    with torch.no_grad():
        for p in layer.experts.parameters():
            p.normal_(0.0, 0.02, generator=gen)
        if case["gate"] == "chosen":
            layer.gate.fill(case, gen)
        else:
            lin = layer.gate.gate
            lin.weight.normal_(0.0, case["d_model"] ** -0.5, generator=gen)
            lin.bias.zero_()
            for i in range(case["dead"]):
                lin.bias[i * case["experts"] // case["dead"]] = -1e4
    shape = (case["tokens"], case["d_model"])
    x = torch.randn(shape, device="cuda", dtype=dtype, generator=gen)
    if not case["train"]:
        return {"layer": layer.eval(), "x": x, "train": False}
    dy = torch.randn(shape, device="cuda", dtype=dtype, generator=gen)
    return {"layer": layer.train(), "x": x.requires_grad_(True), "dy": dy, "train": True,
            "params": list(layer.parameters()), "balance": case["gate"] in ("gshard", "switch")}


def run(state):
    layer, x = state["layer"], state["x"]
    if not state["train"]:
        with torch.no_grad():
            return layer(x)
    params = state["params"]
    x.grad = None
    for p in params:
        p.grad = None
    y = layer(x)
    if state["balance"]:
        torch.autograd.backward([y, layer.gate.get_loss()], [state["dy"], None])
    else:
        y.backward(state["dy"])
    return [y.detach(), x.grad] + [p.grad for p in params]


def _rows(case):
    """Expected number of live (token, expert) slots."""
    n, e = case["tokens"] * case["top_k"], case["experts"]
    if case["gate"] != "chosen":
        return n
    p = [(i + 1) ** -ZIPF_S for i in range(e)]
    total = sum(p)
    return sum(min(n * v / total, CAPACITY_FACTOR * n / e) for v in p)


def work(case):
    t, d, h, e = case["tokens"], case["d_model"], case["d_hidden"], case["experts"]
    size = 4 if case["dtype"] == "f32" else 2
    rows = _rows(case)
    live = min(e - case["dead"], case["tokens"] * case["top_k"])
    weights = 2 * d * h + d + h                    # of one expert
    gate = 0 if case["gate"] == "chosen" else e * d + e
    flops = 4.0 * rows * d * h + 2.0 * t * gate
    values = 2.0 * t * d + live * weights + gate   # x, y and the parameters in use
    if case["train"]:
        flops *= 3
        values += 2.0 * t * d + e * weights + gate  # dy, dx and every gradient
    return {"bytes": values * size, "flops": flops}


def tolerance(case):
    # one rounding of the storage type per intermediate, sums in 32 bits
    return {"rel": {"bf16": 1e-2, "f16": 2e-3, "f32": 1e-5}[case["dtype"]]}
