"""Performance cases of the FfnAgent FFN path: what its users run, at the sizes they run it.

Five kinds of pass, each through public entry points only:

``dense``       one Dense FFN layer: ``FfnAgent.execute`` gathers mailbox rows by slot id, applies the
                RMSNorm, runs gate_up with SiLU * up and down, and scatters to the slots of the output
                mailbox.  Decode is a handful of rows, prefill hundreds to thousands.
``request``     the same layer as one Transport mailbox transaction (submit, execute, settle), which is
                what an attached ``ffn_shim`` call does.
``stack``       one decode step of a whole model's FFN layers with residual additions, captured once into
                a graph and replayed, as serving engines run decode.
``moe``         one MoE layer: gather + RMSNorm, Router, routing finalisation, grouped Experts, combine.
``operator``    the operator layer's Dense for what the agent's templates do not take: CONCATENATED
                Gate/Up rows, GELU, projection biases.
``projection``  one prepared ``Gemm`` with a bias and any payload dtype and width.

Row capacities are powers of two, as deployments configure them, so most row counts run on a template
larger than they are.  Activations are N(0, 1), weights N(0, 0.02), norm weights 1 + N(0, 0.1).
"""

from __future__ import annotations

import math

import torch

from crosspool_amd.agent import FfnAgent
from crosspool_amd.ffn import (
    DpRowLayout,
    ForwardMode,
    GateTransform,
    GateUpOrder,
    GeluActivation,
    OutputRequirement,
    RouterAlgorithm,
    RouterProjectionPrecision,
    SiluActivation,
)
from crosspool_amd.moe import MoeFfnWeights, MoeLayerSpec, MoeRouterWeights
from crosspool_amd.operators import (
    Activation,
    Dense,
    DenseExecutionPlan,
    DenseSignature,
    Gemm,
    GemmPlan,
    ProjectionLayout,
    TensorLayout,
)
from crosspool_amd.transport import FfnRequestMetadata, TransportResident
from crosspool_amd.weights import DenseFfnWeights, ProjectionWeights

EPS = 1e-6
WEIGHT_STD = 0.02
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# (hidden, intermediate) of the Dense layers: Qwen3 0.6B, 1.7B, 4B, 8B, a hidden-1536 model and one of
# 8 tensor-parallel shards of Qwen3-32B.
DENSE_SHAPES = ((1024, 3072), (2048, 6144), (2560, 9728), (4096, 12288), (1536, 8960), (5120, 3200))
# (hidden, intermediate, experts, top-k) of the MoE layers: Qwen3-30B-A3B and a smaller generic one.
MOE_SHAPES = ((2048, 768, 128, 8), (1024, 512, 64, 6))
# The largest listed case in floating-point operations: a drawn case stays below it.
LARGEST_FLOPS = 6.0 * 8192 * 5120 * 3200


def dense(name: str, hidden: int, intermediate: int, rows: int, dtype: str = "bf16", kind: str = "dense") -> dict:
    return {"name": name, "kind": kind, "hidden": hidden, "intermediate": intermediate, "rows": rows, "dtype": dtype}


def moe(name: str, shape: tuple[int, int, int, int], rows: int, dtype: str = "bf16", scores: str = "softmax") -> dict:
    hidden, intermediate, experts, topk = shape
    return {"name": name, "kind": "moe", "hidden": hidden, "intermediate": intermediate, "experts": experts,
            "topk": topk, "rows": rows, "dtype": dtype, "scores": scores}


def listed() -> list[dict]:
    return [
        # A single-token request of the smallest model: latency, launches and the host path.
        dense("request_1024_1", 1024, 3072, 1, kind="request"),
        # A decode step of a small model's 28 FFN layers at a small batch.
        {"name": "stack_1024_7", "kind": "stack", "hidden": 1024, "intermediate": 3072, "layers": 28, "rows": 7,
         "dtype": "bf16"},
        # Decode of an 8B model with few sequences: weight streaming.
        dense("dense_4096_4", 4096, 12288, 4),
        # Decode of an 8B model with a mid-size batch: still bound by the weights.
        dense("dense_4096_45", 4096, 12288, 45),
        # A ragged prefill chunk of a 4B model in fp16.
        dense("dense_2560_517_fp16", 2560, 9728, 517, "fp16"),
        # Prefill of an 8B model at the usual chunk.
        dense("dense_4096_2048", 4096, 12288, 2048),
        # The largest prefill: one tensor-parallel shard of a 32B model.
        dense("dense_5120_8192", 5120, 3200, 8192),
        # MoE decode with few sequences.
        moe("moe_2048_3", MOE_SHAPES[0], 3),
        # MoE decode with a mid-size batch; sigmoid scores over fp32 logits with a correction bias, a shared
        # expert and a routed scaling factor.
        moe("moe_2048_51_sigmoid", MOE_SHAPES[0], 51, scores="sigmoid"),
        # MoE prefill.
        moe("moe_2048_2048", MOE_SHAPES[0], 2048),
        # A GELU-gated layer whose Gate/Up rows are CONCATENATED, with projection biases, mid-size batch.
        {"name": "operator_2048_130", "kind": "operator", "hidden": 2048, "intermediate": 6144, "rows": 130,
         "dtype": "bf16", "order": "concatenated", "activation": "gelu", "bias": True},
        # One biased fp32 projection of odd sizes.
        {"name": "projection_2053_257_fp32", "kind": "projection", "hidden": 2053, "width": 1030, "rows": 257,
         "dtype": "fp32", "gated": False},
    ]


def _log_rows(rng, low: int, high: int) -> int:
    """Row counts spread over their logarithm; most of them odd or ragged."""

    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng) -> dict:
    kind = rng.choices(("dense", "request", "stack", "moe", "operator", "projection"), (36, 8, 6, 28, 14, 8))[0]
    if kind in ("dense", "request"):
        hidden, intermediate = rng.choice(DENSE_SHAPES)
        high = min(8192, int(LARGEST_FLOPS / (6.0 * hidden * intermediate)))
        rows = _log_rows(rng, 1, high if kind == "dense" else 64)
        return {"kind": kind, "hidden": hidden, "intermediate": intermediate, "rows": rows,
                "dtype": rng.choice(("bf16", "bf16", "bf16", "fp16"))}
    if kind == "stack":
        return {"kind": kind, "hidden": 1024, "intermediate": 3072, "layers": rng.choice((16, 28)),
                "rows": _log_rows(rng, 1, 256), "dtype": rng.choice(("bf16", "fp16"))}
    if kind == "moe":
        hidden, intermediate, experts, topk = rng.choice((MOE_SHAPES[0], MOE_SHAPES[0], MOE_SHAPES[1]))
        return {"kind": kind, "hidden": hidden, "intermediate": intermediate, "experts": experts, "topk": topk,
                "rows": _log_rows(rng, 1, 4096), "dtype": rng.choice(("bf16", "bf16", "bf16", "fp16")),
                "scores": rng.choice(("softmax", "softmax", "sigmoid"))}
    if kind == "operator":
        hidden, intermediate = rng.choice(DENSE_SHAPES[:3])
        return {"kind": kind, "hidden": hidden, "intermediate": intermediate, "rows": _log_rows(rng, 1, 1024),
                "dtype": rng.choice(("bf16", "fp16")), "order": rng.choice(("concatenated", "interleaved")),
                "activation": rng.choice(("silu", "gelu")), "bias": rng.choice((True, False))}
    dtype = rng.choice(("bf16", "fp16", "fp32"))
    return {"kind": kind, "hidden": rng.randrange(64, 4097), "width": 2 * rng.randrange(32, 2049),
            "rows": _log_rows(rng, 1, 2048), "dtype": dtype, "gated": rng.choice((True, False))}


# ------------------------------------------------------------------ inputs
def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed * 7919 + 17)


def _normal(generator: torch.Generator, shape: tuple[int, ...], dtype: torch.dtype, std: float = 1.0,
            mean: float = 0.0) -> torch.Tensor:
    """N(mean, std) drawn in fp32, in pieces so that large weights need no fp32 copy of themselves."""

    out = torch.empty(shape, dtype=dtype, device="cuda")
    flat = out.view(-1)
    piece = 1 << 26
    for first in range(0, flat.numel(), piece):
        part = flat[first:first + piece]
        values = torch.empty(part.shape, dtype=torch.float32, device="cuda")
        part.copy_(values.normal_(mean, std, generator=generator))
    return out


def _mailbox(generator: torch.Generator, case: dict) -> tuple[torch.Tensor, torch.Tensor]:
    """A mailbox with twice the request's rows, and the slots the request's rows are in, in no order."""

    rows = case["rows"]
    slot_count = max(64, 2 * rows)
    pool = _normal(generator, (slot_count, case["hidden"]), DTYPES[case["dtype"]])
    slots = torch.randperm(slot_count, generator=generator, device="cuda")[:rows].to(torch.int32)
    return pool, slots


def _dense_weights(generator: torch.Generator, hidden: int, intermediate: int, dtype: torch.dtype) -> tuple:
    gate_up = _normal(generator, (2 * intermediate, hidden), dtype, WEIGHT_STD)
    down = _normal(generator, (hidden, intermediate), dtype, WEIGHT_STD)
    return gate_up, down, _normal(generator, (hidden,), dtype, 0.1, 1.0)


def _layer_inputs(case: dict, seed: int) -> dict:
    """Mailbox and layer weights of a dense, request or stack case."""

    generator = _generator(seed)
    pool, slots = _mailbox(generator, case)
    layers = [_dense_weights(generator, case["hidden"], case["intermediate"], pool.dtype)
              for _ in range(case.get("layers", 1))]
    return {"pool": pool, "slots": slots, "layers": layers}


def _moe_inputs(case: dict, seed: int) -> dict:
    generator = _generator(seed)
    pool, slots = _mailbox(generator, case)
    hidden, intermediate, dtype = case["hidden"], case["intermediate"], pool.dtype
    shared = 1 if case["scores"] == "sigmoid" else 0
    total = case["experts"] + shared
    return {
        "pool": pool,
        "slots": slots,
        "i_proj": _normal(generator, (total, 2 * intermediate, hidden), dtype, WEIGHT_STD),
        "o_proj": _normal(generator, (total, hidden, intermediate), dtype, WEIGHT_STD),
        "router": _normal(generator, (case["experts"], hidden), dtype, WEIGHT_STD),
        "correction": _normal(generator, (case["experts"],), torch.float32, 0.05) if shared else None,
        "norm": _normal(generator, (hidden,), dtype, 0.1, 1.0),
    }


def _moe_spec(case: dict) -> MoeLayerSpec:
    if case["scores"] == "sigmoid":
        return MoeLayerSpec(
            routed_expert_count=case["experts"], routed_topk=case["topk"], shared_expert_count=1,
            routed_scaling_factor=2.5, router_algorithm=RouterAlgorithm.SIGMOID,
            router_projection_precision=RouterProjectionPrecision.FP32_LOGITS,
        )
    return MoeLayerSpec(routed_expert_count=case["experts"], routed_topk=case["topk"])


def _operator_inputs(case: dict, seed: int) -> dict:
    generator = _generator(seed)
    hidden, intermediate, dtype = case["hidden"], case["intermediate"], DTYPES[case["dtype"]]
    gate_up, down, _ = _dense_weights(generator, hidden, intermediate, dtype)
    biased = case["bias"]
    return {
        "x": _normal(generator, (case["rows"], hidden), dtype),
        "gate_up": gate_up,
        "down": down,
        "gate_up_bias": _normal(generator, (2 * intermediate,), torch.float32, 0.1) if biased else None,
        "down_bias": _normal(generator, (hidden,), torch.float32, 0.1) if biased else None,
    }


def _projection_inputs(case: dict, seed: int) -> dict:
    generator = _generator(seed)
    dtype = DTYPES[case["dtype"]]
    return {
        "x": _normal(generator, (case["rows"], case["hidden"]), dtype),
        "w": _normal(generator, (case["width"], case["hidden"]), dtype, WEIGHT_STD),
        "bias": _normal(generator, (case["width"],), torch.float32, 0.1),
    }


def _capacity(rows: int) -> int:
    return 1 << (rows - 1).bit_length()


# ------------------------------------------------------------------ state and pass
class State:
    """What one user holds: tensors, and the agent or plan over them, released with the state."""

    def __init__(self, case: dict) -> None:
        self.case = case
        self.agent: FfnAgent | None = None
        self.transport: TransportResident | None = None
        self.graph: torch.cuda.CUDAGraph | None = None

    def __del__(self) -> None:
        self.graph = None
        if self.transport is not None:
            self.transport.close()
        if self.agent is not None:
            self.agent.close()


def _open_agent(state: State) -> None:
    state.agent.materialize(maximum_row_capacity=_capacity(state.case["rows"]))
    # Rows outside the request keep what the output mailbox held.
    state.out_pool = torch.zeros_like(state.pool)


def _register_dense(state: State, layers: list[tuple]) -> None:
    state.agent = FfnAgent()
    for ordinal, (gate_up, down, norm) in enumerate(layers):
        state.agent.register_layer(instance_index=0, layer_ordinal=ordinal, norm_weight=norm, eps=EPS,
                                   weights=DenseFfnWeights.from_tensors(gate_up, down))
    _open_agent(state)


def _prepare_layer(state: State, seed: int) -> None:
    case = state.case
    inputs = _layer_inputs(case, seed)
    state.pool, state.slots = inputs["pool"], inputs["slots"]
    _register_dense(state, inputs["layers"])
    if case["kind"] == "request":
        state.transport = TransportResident(state.agent.device, [(_capacity(case["rows"]), 1)])
        state.transport.open()
        state.request = FfnRequestMetadata(
            layer_ordinal=0, forward_mode=ForwardMode.DECODE, output_requirement=OutputRequirement.PER_RANK_COMPLETE,
            dp_row_layout=DpRowLayout.NONE,
        )
    elif case["kind"] == "stack":
        state.states = torch.empty_like(state.pool)
        state.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state.graph):
            state.states.copy_(state.pool)
            for ordinal in range(case["layers"]):
                state.agent.execute(instance_index=0, layer_ordinal=ordinal, pool=state.states, slots=state.slots,
                                    out_pool=state.out_pool, stream=torch.cuda.current_stream())
                state.states.add_(state.out_pool)


def _prepare_moe(state: State, seed: int) -> None:
    inputs = _moe_inputs(state.case, seed)
    state.pool, state.slots = inputs["pool"], inputs["slots"]
    state.agent = FfnAgent()
    state.agent.register_moe_layer(
        instance_index=0, layer_ordinal=0, spec=_moe_spec(state.case), norm_weight=inputs["norm"], eps=EPS,
        weights=MoeFfnWeights(inputs["i_proj"], inputs["o_proj"],
                              MoeRouterWeights(inputs["router"], inputs["correction"])),
    )
    _open_agent(state)


def _prepare_operator(state: State, seed: int) -> None:
    case = state.case
    inputs = _operator_inputs(case, seed)
    dtype, rows = DTYPES[case["dtype"]], case["rows"]
    function = GeluActivation(approximate="tanh") if case["activation"] == "gelu" else SiluActivation()
    order = GateUpOrder.CONCATENATED if case["order"] == "concatenated" else GateUpOrder.INTERLEAVED
    state.x = inputs["x"]
    state.weights = DenseFfnWeights(i_proj=ProjectionWeights(inputs["gate_up"], bias=inputs["gate_up_bias"]),
                                    o_proj=ProjectionWeights(inputs["down"], bias=inputs["down_bias"]))
    plan = DenseExecutionPlan.prepare(DenseSignature(
        payload_dtype=dtype, payload_row_capacity=_capacity(rows), hidden_size=case["hidden"],
        local_intermediate_size=case["intermediate"], activation=Activation(function=function, gate=GateTransform()),
        i_proj=ProjectionLayout.of(state.weights.i_proj, order=order), o_proj=ProjectionLayout.of(state.weights.o_proj),
    ))
    workspace = torch.empty(max(plan.workspace.nbytes, 16), dtype=torch.uint8, device="cuda")
    state.dense = Dense(plan, workspace)
    state.output = torch.empty((rows, case["hidden"]), dtype=dtype, device="cuda")


def _prepare_projection(state: State, seed: int) -> None:
    case = state.case
    inputs = _projection_inputs(case, seed)
    dtype, rows, width = DTYPES[case["dtype"]], case["rows"], case["width"]
    gated = case["gated"]
    state.x = inputs["x"]
    state.weights = ProjectionWeights(inputs["w"], bias=inputs["bias"])
    out_width = width // 2 if gated else width
    plan = GemmPlan.prepare(
        input_layout=TensorLayout((rows, case["hidden"]), dtype),
        weight_layout=ProjectionLayout.of(state.weights, order=GateUpOrder.INTERLEAVED if gated else None),
        result_layout=TensorLayout((rows, out_width), dtype),
        activation=Activation(function=SiluActivation(), gate=GateTransform()) if gated else None,
    )
    state.gemm = Gemm(plan, torch.empty(max(plan.workspace.nbytes, 16), dtype=torch.uint8, device="cuda"))
    state.output = torch.empty((rows, out_width), dtype=dtype, device="cuda")


def prepare(case: dict, seed: int) -> State:
    state = State(case)
    makers = {"dense": _prepare_layer, "request": _prepare_layer, "stack": _prepare_layer, "moe": _prepare_moe,
              "operator": _prepare_operator, "projection": _prepare_projection}
    makers[case["kind"]](state, seed)
    return state


def run(state: State) -> torch.Tensor:
    kind = state.case["kind"]
    if kind == "stack":
        state.graph.replay()
        return state.states
    if kind == "operator":
        state.dense.run_into(hidden_states=state.x, layer_weights=state.weights, output=state.output)
        return state.output
    if kind == "projection":
        state.gemm.run_into(state.x, state.weights, output=state.output)
        return state.output
    stream = torch.cuda.current_stream()
    if kind == "request":
        state.transport.submit(0, state.case["rows"], state.request, stream=stream)
    state.agent.execute(instance_index=0, layer_ordinal=0, pool=state.pool, slots=state.slots,
                        out_pool=state.out_pool, stream=stream)
    if kind == "request":
        state.transport.settle(0, state.out_pool, state.agent.lanes[0].fault_word, stream=stream)
    return state.out_pool


# ------------------------------------------------------------------ work, tolerance, 64-bit results
def work(case: dict) -> dict:
    rows, hidden, size = case["rows"], case["hidden"], DTYPES[case["dtype"]].itemsize
    if case["kind"] == "projection":
        width = case["width"]
        out = width // 2 if case["gated"] else width
        return {"bytes": size * (rows * hidden + width * hidden + rows * out) + 4 * width,
                "flops": 2.0 * rows * hidden * width}
    intermediate = case["intermediate"]
    layer = 3 * hidden * intermediate
    if case["kind"] == "moe":
        shared = 1 if case["scores"] == "sigmoid" else 0
        # The experts that evenly spread routes reach, and the shared one.
        touched = case["experts"] * (1.0 - (1.0 - case["topk"] / case["experts"]) ** rows) + shared
        routes = rows * (case["topk"] + shared)
        return {"bytes": size * (touched * layer + case["experts"] * hidden + 2 * rows * hidden + hidden) + 4 * rows,
                "flops": 2.0 * routes * layer + 2.0 * rows * hidden * case["experts"]}
    if case["kind"] == "operator":
        biases = 4 * (2 * intermediate + hidden) if case["bias"] else 0
        return {"bytes": size * (layer + 2 * rows * hidden) + biases, "flops": 2.0 * rows * layer}
    layers = case.get("layers", 1)
    return {"bytes": layers * size * (layer + hidden) + size * 2 * rows * hidden + 4 * rows,
            "flops": layers * 2.0 * rows * layer}


def tolerance(case: dict) -> dict:
    """About four times the path's own distance from its 64-bit result.

    A 16-bit layer rounds the projection, the activation and the output (bf16 4.2e-3, fp16 5.3e-4); a MoE
    layer also rounds each route's output, and a logit at a rounding boundary may pick another expert.  Over a
    stack's layers the roundings add up (bf16 6.4e-3 to 1.1e-2).
    """

    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    if case["kind"] == "moe":
        return {"rel": 2e-2 if case["dtype"] == "bf16" else 1e-2, "max": 0.99}
    if case["kind"] == "stack":
        return {"rel": 2.5e-2 if case["dtype"] == "bf16" else 4e-3}
    return {"rel": 1.6e-2 if case["dtype"] == "bf16" else 2e-3}


def _normed(rows: torch.Tensor, norm: torch.Tensor) -> torch.Tensor:
    x = rows.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * norm.double()


def _gated(projected: torch.Tensor, activation: str, order: str) -> torch.Tensor:
    if order == "interleaved":
        gate, up = projected[:, 0::2], projected[:, 1::2]
    else:
        gate, up = projected.chunk(2, dim=1)
    if activation == "gelu":
        return torch.nn.functional.gelu(gate, approximate="tanh") * up
    return gate * torch.sigmoid(gate) * up


def _exact_layer(x: torch.Tensor, gate_up: torch.Tensor, down: torch.Tensor) -> torch.Tensor:
    return _gated(x @ gate_up.double().t(), "silu", "interleaved") @ down.double().t()


def _exact_moe(case: dict, seed: int) -> torch.Tensor:
    inputs = _moe_inputs(case, seed)
    dtype, experts, topk = inputs["pool"].dtype, case["experts"], case["topk"]
    # The Router reads the normalised rows in the payload dtype; softmax layers hold its logits in it too.
    x = _normed(inputs["pool"][inputs["slots"].long()], inputs["norm"]).to(dtype).double()
    logits = x @ inputs["router"].double().t()
    rows = logits.shape[0]
    if case["scores"] == "sigmoid":
        scores = torch.sigmoid(logits)
        ids = (scores + inputs["correction"].double()).topk(topk, dim=1).indices
        scale = 2.5
    else:
        scores = torch.softmax(logits.to(dtype).double(), dim=1)
        # Equal logits go to the lower expert.
        ids = scores.sort(dim=1, descending=True, stable=True).indices[:, :topk]
        scale = 1.0
    picked = scores.gather(1, ids)
    weights = torch.zeros((rows, inputs["i_proj"].shape[0]), dtype=torch.float64, device="cuda")
    weights.scatter_(1, ids, picked / picked.sum(1, keepdim=True))
    if case["scores"] == "sigmoid":
        weights[:, experts] = 1.0 / scale
    total = torch.zeros((rows, case["hidden"]), dtype=torch.float64, device="cuda")
    for expert in range(weights.shape[1]):
        live = weights[:, expert].nonzero().view(-1)
        if live.numel():
            y = _exact_layer(x[live], inputs["i_proj"][expert], inputs["o_proj"][expert])
            total.index_add_(0, live, y * weights[live, expert, None])
    out = torch.zeros(inputs["pool"].shape, dtype=torch.float64, device="cuda")
    out[inputs["slots"].long()] = total * scale
    return out


def exact(case: dict, seed: int) -> torch.Tensor:
    if case["kind"] == "moe":
        return _exact_moe(case, seed)
    if case["kind"] == "projection":
        inputs = _projection_inputs(case, seed)
        projected = inputs["x"].double() @ inputs["w"].double().t() + inputs["bias"].double()
        return _gated(projected, "silu", "interleaved") if case["gated"] else projected
    if case["kind"] == "operator":
        inputs = _operator_inputs(case, seed)
        projected = inputs["x"].double() @ inputs["gate_up"].double().t()
        if case["bias"]:
            projected += inputs["gate_up_bias"].double()
        out = _gated(projected, case["activation"], case["order"]) @ inputs["down"].double().t()
        return out + inputs["down_bias"].double() if case["bias"] else out
    inputs = _layer_inputs(case, seed)
    slots = inputs["slots"].long()
    x = inputs["pool"][slots].double()
    if case["kind"] == "stack":
        for gate_up, down, norm in inputs["layers"]:
            x = x + _exact_layer(_normed(x, norm), gate_up, down)
        out = inputs["pool"].double()
        out[slots] = x
        return out
    gate_up, down, norm = inputs["layers"][0]
    out = torch.zeros(inputs["pool"].shape, dtype=torch.float64, device="cuda")
    out[slots] = _exact_layer(_normed(x, norm), gate_up, down)
    return out
