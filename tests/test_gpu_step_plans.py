"""Steps between a template's capacities: the plan each row count takes.

A template of more than 64 rows keeps tile choices for several row counts; replays at a
tile's edges must agree with fp64 whatever the choice (192 x 256 and 128 x 256 tiles, K splits
that are no power of two, column splits, rotated weight streams, weight tile counts that do
not divide over the XCDs), repeat bit for bit, and give the same bits through graph dispatch.
"""

from __future__ import annotations

import ctypes
import math
import os
import subprocess
import sys
import time
from pathlib import Path

import pytest
import torch

from crosspool_amd import _native
from crosspool_amd.agent import ExecutorLane, FfnAgent
from crosspool_amd.ffn import GeluActivation, ReluActivation, RouterAlgorithm, RouterProjectionPrecision, SiluActivation
from crosspool_amd.moe import MoeFfnWeights, MoeLayerSpec, MoeRouterWeights
from crosspool_amd.weights import DenseFfnWeights

pytestmark = pytest.mark.gpu


def _layer(device, hidden, intermediate, dtype):
    generator = torch.Generator(device=device).manual_seed(hidden + intermediate)
    gate_up = (torch.randn((2 * intermediate, hidden), device=device, generator=generator) * 0.02).to(dtype)
    down = (torch.randn((hidden, intermediate), device=device, generator=generator) * 0.02).to(dtype)
    norm = (1 + 0.1 * torch.randn((hidden,), device=device, generator=generator)).to(dtype)
    return gate_up, down, norm


def _expected(rows, gate_up, down, norm):
    """The step in fp64 with the path's rounding points."""

    dtype = rows.dtype
    x = rows.double()
    x = (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * norm.double()).to(dtype).double()
    projected = (x @ gate_up.double().t()).to(dtype).double()
    gate, up = projected[:, 0::2], projected[:, 1::2]
    return (gate * torch.sigmoid(gate) * up).to(dtype).double() @ down.double().t()


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize(
    "hidden,intermediate,capacity,rows_list",
    (
        (2560, 9728, 1024, (257, 517, 576, 577)),     # 192 x 256 gate_up, K splits of down
        (1536, 8960, 512, (192, 193, 320, 321)),      # 70 weight tiles of 256
        (5120, 3200, 2048, (1025, 1152, 2048)),       # 25 weight tiles, column splits
        (4096, 1032, 128, (33, 64, 65, 128)),         # rotated weight streams, ragged N
        (8192, 4096, 128, (17, 33, 64, 65, 128)),     # the same over K ranges
        (8192, 264, 64, (33, 64)),                    # the same at another multiple of 8 KB
        (1032, 1000, 300, (65, 128, 129, 300)),       # ragged K and N, a capacity between two steps
        (2048, 6144, 1024, (600, 640, 641)),          # 128 x 256 gate_up
    ),
)
def test_steps_between_capacities(device, hidden, intermediate, capacity, rows_list, dtype):
    gate_up, down, norm = _layer(device, hidden, intermediate, dtype)
    generator = torch.Generator(device=device).manual_seed(5)
    pool = torch.randn((capacity + 40, hidden), device=device, generator=generator).to(dtype)
    slots = torch.randperm(pool.shape[0], device=device, generator=generator).to(torch.int32)
    outputs = {}
    for graph_dispatch in (False, True):
        with FfnAgent(device, graph_dispatch=graph_dispatch) as agent:
            agent.register_layer(instance_index=0, layer_ordinal=0, norm_weight=norm, eps=1e-6,
                                 weights=DenseFfnWeights.from_tensors(gate_up, down))
            agent.materialize(maximum_row_capacity=capacity)
            for rows in rows_list + rows_list[:1]:
                print(f"step plan {hidden}x{intermediate} {rows}/{capacity} {dtype} graph={graph_dispatch}", flush=True)
                out = torch.zeros_like(pool)
                agent.execute(instance_index=0, layer_ordinal=0, pool=pool, slots=slots, rows=rows, out_pool=out)
                agent.check_health()
                previous = outputs.setdefault(rows, out)
                assert torch.equal(out.view(torch.int16), previous.view(torch.int16)), "replays differ"
    for rows, out in outputs.items():
        live = slots[:rows].long()
        expected = _expected(pool[live], gate_up, down, norm)
        # Sums in another order round a few values the other way: one ulp of activations and outputs.
        error = (out[live].double() - expected).norm() / expected.norm()
        ulp = 2.0**-8 if dtype is torch.bfloat16 else 2.0**-11
        assert error <= ulp, f"{rows} rows: relative error {error:.2e}"
        untouched = torch.ones(pool.shape[0], dtype=torch.bool, device=device)
        untouched[live] = False
        assert not out[untouched].any()


# 8-row weight blocks (16-row ones would fill at most half the CUs): N around the last block,
# K ranges that end inside a chunk, one and two token groups, gate_up with the gather fused.
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize("hidden,intermediate", ((1024, 3072), (1016, 1000), (264, 40), (2048, 6144)))
def test_half_block_steps(device, hidden, intermediate, dtype):
    gate_up, down, norm = _layer(device, hidden, intermediate, dtype)
    pool = torch.randn((64, hidden), device=device, generator=torch.Generator(device=device).manual_seed(9)).to(dtype)
    slots = torch.randperm(64, device=device).to(torch.int32)
    with FfnAgent(device) as agent:
        agent.register_layer(instance_index=0, layer_ordinal=0, norm_weight=norm, eps=1e-6,
                             weights=DenseFfnWeights.from_tensors(gate_up, down))
        agent.materialize(maximum_row_capacity=16)
        for rows in (1, 2, 7, 8, 9, 16):
            print(f"half blocks {hidden}x{intermediate} {rows} {dtype}", flush=True)
            out = torch.zeros_like(pool)
            agent.execute(instance_index=0, layer_ordinal=0, pool=pool, slots=slots, rows=rows, out_pool=out)
            agent.check_health()
            live = slots[:rows].long()
            expected = _expected(pool[live], gate_up, down, norm)
            error = (out[live].double() - expected).norm() / expected.norm()
            assert error <= (2.0**-8 if dtype is torch.bfloat16 else 2.0**-11), f"{rows} rows: {error:.2e}"


# The eager step keeps the capacity's own choice where a workspace has no room for the refined
# one's K ranges, takes no K ranges where it has none for either, and refuses only a workspace
# without room for the batch and the intermediate.
@pytest.mark.parametrize("rows", (257, 517))
def test_eager_step_runs_in_the_smallest_accepted_workspace(device, rows):
    hidden, intermediate = 2560, 9728
    regions = rows * (hidden + intermediate) * 2
    scratch = _native.gemm_workspace_bytes(rows, hidden, intermediate, False) + _native.gemm_workspace_bytes(
        rows, 2 * intermediate, hidden, True)
    sizes = (_native.dense_workspace_bytes(rows, hidden, intermediate), (regions + 255) // 256 * 256 + scratch, regions)
    assert sizes[0] > sizes[1] > sizes[2]
    _check_eager_steps(device, hidden, intermediate, rows, sizes, refused=regions - 16)


# A workspace for a capacity serves the row counts below it whose own K ranges would need more.
@pytest.mark.parametrize("hidden,intermediate,capacity,rows",
                         ((4096, 12288, 256, 154), (1024, 3072, 128, 72), (5120, 3200, 512, 43), (2048, 6144, 64, 22),
                          (4096, 12288, 16, 9)))
def test_eager_step_runs_in_the_workspace_of_a_capacity(device, hidden, intermediate, capacity, rows):
    _check_eager_steps(device, hidden, intermediate, rows, (_native.dense_workspace_bytes(capacity, hidden, intermediate),
                                                            rows * (hidden + intermediate) * 2))


def _check_eager_steps(device, hidden, intermediate, rows, sizes, refused=None):
    gate_up, down, norm = _layer(device, hidden, intermediate, torch.bfloat16)
    pool = torch.randn((700, hidden), device=device).bfloat16()
    slots = torch.randperm(700, device=device)[:rows].to(torch.int32)
    expected = _expected(pool[slots.long()], gate_up, down, norm)

    def pointer(tensor):
        return ctypes.c_void_p(tensor.data_ptr())

    def step(nbytes):
        print(f"eager step {hidden}x{intermediate} {rows} rows workspace {nbytes}", flush=True)
        workspace = torch.full((nbytes + 256,), 0x7f, dtype=torch.uint8, device=device)
        out = torch.zeros_like(pool)
        _native.call("xp_dense_step", pointer(pool), pointer(out), 700, pointer(slots), rows, hidden, intermediate,
                     pointer(gate_up), pointer(down), pointer(norm), 1e-6, pointer(workspace), nbytes, None,
                     ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert bool((workspace[nbytes:] == 0x7f).all()), "writes outside the workspace"
        error = (out[slots.long()].double() - expected).norm() / expected.norm()
        assert error <= 2.0**-8

    for nbytes in sizes:
        step(nbytes)
    if refused is not None:
        with pytest.raises(_native.NativeError, match="workspace is smaller"):
            step(refused)


# A Lane whose workspace has no room for the K ranges of the plans between two capacities takes the
# capacity's own choice at every row count.
@pytest.mark.parametrize("hidden,intermediate,capacity", ((8192, 4096, 512), (1536, 8960, 512), (4096, 12288, 2048)))
def test_template_runs_in_a_lane_for_the_capacitys_own_choice(device, hidden, intermediate, capacity):
    gate_up, down, norm = _layer(device, hidden, intermediate, torch.bfloat16)
    pool = torch.randn((capacity, hidden), device=device, generator=torch.Generator(device=device).manual_seed(4)).bfloat16()
    slots = torch.randperm(capacity, device=device).to(torch.int32)
    regions = capacity * (hidden + intermediate) * 2
    scratch = _native.gemm_workspace_bytes(capacity, hidden, intermediate, False) + _native.gemm_workspace_bytes(
        capacity, 2 * intermediate, hidden, True)
    nbytes = (regions + 255) // 256 * 256 + scratch if scratch else regions
    assert nbytes < _native.dense_workspace_bytes(capacity, hidden, intermediate)
    with FfnAgent(device) as agent:
        agent.register_layer(instance_index=0, layer_ordinal=0, norm_weight=norm, eps=1e-6,
                             weights=DenseFfnWeights.from_tensors(gate_up, down))
        agent.materialize(maximum_row_capacity=capacity)
        template = next(t for t in agent.templates.values() if t.signature.payload_row_capacity == capacity)
        for graph_dispatch in (False, True):
            lane = ExecutorLane(agent, nbytes, graph_dispatch=graph_dispatch)
            lane.capture(template)
            for rows in (1, capacity // 2 + 1, capacity):
                print(f"small lane {hidden}x{intermediate} {rows}/{capacity} graph={graph_dispatch}", flush=True)
                out = torch.zeros_like(pool)
                lane.replay(instance_index=0, layer_ordinal=0, pool=pool, slots=slots, rows=rows, out_pool=out)
                lane.synchronize()
                live = slots[:rows].long()
                expected = _expected(pool[live], gate_up, down, norm)
                assert (out[live].double() - expected).norm() <= 2.0**-8 * expected.norm()
            lane.close()
        lane = ExecutorLane(agent, nbytes - 256)
        with pytest.raises(_native.NativeError, match="smaller than the template needs"):
            lane.capture(template)
        lane.close()


# A MoE template keeps expert tiles for several row counts: every tile family below one capacity,
# against fp64 over the GPU's own routing, and the same bits through graph dispatch.
@pytest.mark.parametrize("capacity,rows_list", ((1024, (64, 65, 300, 449, 832, 1024)), (2304, (145, 1100, 2304))))
def test_moe_steps_between_capacities(device, capacity, rows_list):
    hidden, intermediate, experts, topk = 256, 128, 8, 2
    generator = torch.Generator(device=device).manual_seed(3)

    def normal(*shape, std=1.0):
        return (torch.randn(shape, device=device, generator=generator) * std).bfloat16()

    weights = MoeFfnWeights(normal(experts, 2 * intermediate, hidden, std=0.05), normal(experts, hidden, intermediate, std=0.05),
                            MoeRouterWeights(normal(experts, hidden, std=0.05)))
    pool = normal(capacity + 8, hidden)
    slots = torch.randperm(pool.shape[0], device=device).to(torch.int32)
    x = pool.double()
    logits = (x @ weights.router.projection.double().t()).bfloat16().double()
    picked, ids = torch.softmax(logits, 1).sort(dim=1, descending=True, stable=True)
    picked, ids = picked[:, :topk] / picked[:, :topk].sum(1, keepdim=True), ids[:, :topk]
    expected = torch.zeros_like(x)
    for expert in range(experts):
        projected = (x @ weights.i_proj[expert].double().t()).bfloat16().double()
        gate, up = projected[:, 0::2], projected[:, 1::2]
        y = (gate * torch.sigmoid(gate) * up).bfloat16().double() @ weights.o_proj[expert].double().t()
        expected += y * (picked * (ids == expert)).sum(1, keepdim=True)
    outputs = {}
    for graph_dispatch in (False, True):
        with FfnAgent(device, graph_dispatch=graph_dispatch) as agent:
            agent.register_moe_layer(instance_index=0, layer_ordinal=0, weights=weights,
                                     spec=MoeLayerSpec(routed_expert_count=experts, routed_topk=topk))
            agent.materialize(maximum_row_capacity=capacity)
            for rows in rows_list + rows_list[:1]:
                print(f"moe step plan {rows}/{capacity} graph={graph_dispatch}", flush=True)
                out = torch.zeros_like(pool)
                agent.execute(instance_index=0, layer_ordinal=0, pool=pool, slots=slots, rows=rows, out_pool=out)
                agent.check_health()
                previous = outputs.setdefault(rows, out)
                assert torch.equal(out.view(torch.int16), previous.view(torch.int16)), "replays differ"
    for rows, out in outputs.items():
        live = slots[:rows].long()
        difference = (out[live].double() - expected[live]).norm(dim=1) / expected[live].norm(dim=1)
        # Two route roundings, the combine's and flipped activations; a logit at a rounding
        # boundary may pick another expert in a few rows.
        assert difference.median() <= 2.0**-7 and (difference > 2.0**-5).float().mean() <= 0.01, f"{rows} rows"


# The same with what a MoE layer can add to the plain one: a sigmoid Router with a correction, a
# shared expert, projection biases, another activation and a scaling factor.
@pytest.mark.parametrize("activation", (SiluActivation(), ReluActivation(), GeluActivation("none")))
def test_moe_steps_of_extended_layers(device, activation):
    hidden, intermediate, routed, topk, capacity, scaling = 256, 128, 8, 2, 1024, 2.5
    experts = routed + 1
    generator = torch.Generator(device=device).manual_seed(3)

    def normal(*shape, std=1.0):
        return torch.randn(shape, device=device, generator=generator) * std

    correction = normal(routed, std=0.1)
    weights = MoeFfnWeights(
        normal(experts, 2 * intermediate, hidden, std=0.05).bfloat16(), normal(experts, hidden, intermediate, std=0.05).bfloat16(),
        MoeRouterWeights(normal(routed, hidden, std=0.05), correction),
        normal(experts, 2 * intermediate, std=0.2), normal(experts, hidden, std=0.2))
    pool = normal(capacity + 8, hidden).bfloat16()
    slots = torch.randperm(pool.shape[0], device=device).to(torch.int32)
    x = pool.double()
    scores = torch.sigmoid(x @ weights.router.projection.double().t())
    ids = (scores + correction.double()).topk(topk, dim=1).indices
    picked = scores.gather(1, ids)
    share = torch.zeros((x.shape[0], experts), dtype=torch.float64, device=device)
    share.scatter_(1, ids, picked / picked.sum(1, keepdim=True))
    share[:, routed] = 1.0 / scaling
    expected = torch.zeros_like(x)
    for expert in range(experts):
        projected = x @ weights.i_proj[expert].double().t() + weights.i_proj_bias[expert].double()
        gate, up = projected.bfloat16().double()[:, 0::2], projected.bfloat16().double()[:, 1::2]
        function = {SiluActivation: torch.nn.functional.silu, ReluActivation: torch.relu,
                    GeluActivation: torch.nn.functional.gelu}[type(activation)]
        y = (function(gate) * up).bfloat16().double() @ weights.o_proj[expert].double().t() + weights.o_proj_bias[expert].double()
        expected += scaling * y * share[:, expert: expert + 1]
    spec = MoeLayerSpec(routed_expert_count=routed, routed_topk=topk, shared_expert_count=1, routed_scaling_factor=scaling,
                        router_algorithm=RouterAlgorithm.SIGMOID, activation=activation,
                        router_projection_precision=RouterProjectionPrecision.FP32)
    with FfnAgent(device) as agent:
        agent.register_moe_layer(instance_index=0, layer_ordinal=0, weights=weights, spec=spec)
        agent.materialize(maximum_row_capacity=capacity)
        # 16-route, 64-, 128- and 256-row expert tiles, plans below and at a capacity
        for rows in (1, 8, 9, 64, 65, 140, 256, 300, 577, 1000, 1024):
            print(f"extended moe step {type(activation).__name__} {rows}/{capacity}", flush=True)
            out = torch.zeros_like(pool)
            agent.execute(instance_index=0, layer_ordinal=0, pool=pool, slots=slots, rows=rows, out_pool=out)
            agent.check_health()
            live = slots[:rows].long()
            difference = (out[live].double() - expected[live]).norm(dim=1) / expected[live].norm(dim=1)
            # Two route roundings, the combine's and flipped activations; a score within 2^-20 of
            # another may pick another expert in a few rows.
            assert difference.median() <= 2.0**-7 and (difference > 2.0**-5).double().mean() <= 0.01, f"{rows} rows"
            untouched = torch.ones(pool.shape[0], dtype=torch.bool, device=device)
            untouched[live] = False
            assert not out[untouched].any()


@pytest.mark.parametrize("precision", (RouterProjectionPrecision.FP32, RouterProjectionPrecision.FP32_LOGITS))
def test_moe_template_runs_in_a_lane_without_router_scratch(device, precision):
    hidden, intermediate, experts, topk, capacity = 2048, 64, 128, 4, 256
    generator = torch.Generator(device=device).manual_seed(3)

    def normal(*shape):
        return torch.randn(shape, device=device, generator=generator)

    router = normal(experts, hidden) * 0.1
    router = router if precision is RouterProjectionPrecision.FP32 else router.bfloat16()
    weights = MoeFfnWeights((normal(experts, 2 * intermediate, hidden) * 0.05).bfloat16(),
                            (normal(experts, hidden, intermediate) * 0.05).bfloat16(), MoeRouterWeights(router))
    pool = normal(capacity, hidden).bfloat16()
    slots = torch.randperm(capacity, device=device, generator=generator).to(torch.int32)
    with FfnAgent(device) as agent:
        agent.register_moe_layer(
            instance_index=0, layer_ordinal=0, weights=weights,
            spec=MoeLayerSpec(routed_expert_count=experts, routed_topk=topk, router_projection_precision=precision))
        agent.materialize(maximum_row_capacity=capacity)
        template = next(t for t in agent.templates.values() if t.signature.payload_row_capacity == capacity)
        layout = _native.moe_step_workspace_layout(template.signature.native_descriptor(), capacity)
        scratch = layout[2] - layout[1] - capacity * experts * 4
        assert scratch > 0
        print(f"moe lane {precision.name} {layout[7]} less {scratch} bytes", flush=True)
        lane = ExecutorLane(agent, layout[7] - scratch)
        lane.capture(template)
        for rows in (1, 100, capacity):
            out, expected = torch.zeros_like(pool), torch.zeros_like(pool)
            lane.replay(instance_index=0, layer_ordinal=0, pool=pool, slots=slots, rows=rows, out_pool=out)
            agent.execute(instance_index=0, layer_ordinal=0, pool=pool, slots=slots, rows=rows, out_pool=expected)
            torch.cuda.synchronize()
            # The Router's fp32 sums in another order: its weights move by a few 2^-24.
            assert (out.double() - expected.double()).norm() <= 2.0**-8 * expected.double().norm()
        lane.close()
        with pytest.raises(_native.NativeError, match="smaller than the template needs"):
            small = ExecutorLane(agent, layout[7] - scratch - 256)
            try:
                small.capture(template)
            finally:
                small.close()


def test_moe_replays_prepare_in_the_same_time_at_every_capacity(device):
    # What follows from the template alone (its workspace, the Router's K ranges) is settled at
    # capture: the host time of a replay does not grow with the capacity.
    hidden, intermediate, experts, capacity = 256, 64, 16, 32768
    generator = torch.Generator(device=device).manual_seed(3)

    def normal(*shape):
        return torch.randn(shape, device=device, generator=generator) * 0.05

    weights = MoeFfnWeights(normal(experts, 2 * intermediate, hidden).bfloat16(), normal(experts, hidden, intermediate).bfloat16(),
                            MoeRouterWeights(normal(experts, hidden)))
    pool = normal(capacity, hidden).bfloat16()
    slots = torch.arange(capacity, device=device, dtype=torch.int32)
    out = torch.zeros_like(pool)
    spec = MoeLayerSpec(routed_expert_count=experts, routed_topk=2, router_projection_precision=RouterProjectionPrecision.FP32)
    with FfnAgent(device) as agent:
        agent.register_moe_layer(instance_index=0, layer_ordinal=0, weights=weights, spec=spec)
        agent.materialize(maximum_row_capacity=capacity)

        def host_us(rows):
            best = math.inf
            for _ in range(30):
                torch.cuda.synchronize()
                started = time.perf_counter()
                for _ in range(4):
                    agent.execute(instance_index=0, layer_ordinal=0, pool=pool, slots=slots, rows=rows, out_pool=out)
                best = min(best, (time.perf_counter() - started) / 4)
            torch.cuda.synchronize()
            return best * 1e6

        small, large = host_us(64), host_us(capacity // 2 + 1)
        print(f"host us per replay: {small:.1f} at 64 rows, {large:.1f} at {capacity // 2 + 1}", flush=True)
        # The search over this capacity's row counts, twice a replay, took it from 45 to 96 us.
        assert large <= 1.5 * small


# A program of its own, so that the HIP runtime logs its calls.
GRAPH_PROGRAM = """
import sys
import torch
from crosspool_amd.agent import FfnAgent
from crosspool_amd.moe import MoeFfnWeights, MoeLayerSpec, MoeRouterWeights
from crosspool_amd.weights import DenseFfnWeights

device = torch.device("cuda:0")


def normal(*shape):
    return (torch.randn(shape, device=device) * 0.05).bfloat16()


pool = normal(512, 256)
slots = torch.arange(512, device=device, dtype=torch.int32)
with FfnAgent(device, graph_dispatch=sys.argv[1] == "capture") as agent:
    agent.register_layer(instance_index=0, layer_ordinal=0, weights=DenseFfnWeights.from_tensors(normal(512, 256), normal(256, 256)))
    agent.register_moe_layer(instance_index=0, layer_ordinal=1, spec=MoeLayerSpec(routed_expert_count=8, routed_topk=2),
                             weights=MoeFfnWeights(normal(8, 256, 256), normal(8, 256, 128), MoeRouterWeights(normal(8, 256))))
    agent.materialize(maximum_row_capacity=512)
    agent.lanes[0].set_graph_dispatch(True)
    print("REPLAYS", file=sys.stderr, flush=True)
    for rows in (1, 64, 65, 100, 128, 129, 193, 256, 257, 321, 400, 512):
        for ordinal in (0, 1):
            agent.execute(instance_index=0, layer_ordinal=ordinal, pool=pool, slots=slots, rows=rows)
    agent.check_health()
    print("END", file=sys.stderr, flush=True)
"""


@pytest.mark.parametrize("switched_on", ("capture", "later"))
def test_graph_dispatch_instantiates_no_graph_in_a_replay(switched_on):
    print(f"graph dispatch switched on at {switched_on}", flush=True)
    root = Path(__file__).resolve().parent.parent
    result = subprocess.run(
        [sys.executable, "-c", GRAPH_PROGRAM, switched_on], cwd=root, capture_output=True, text=True, timeout=100,
        env={**os.environ, "PYTHONPATH": str(root), "AMD_LOG_LEVEL": "3"},
    )
    assert result.returncode == 0, result.stderr[-2000:]
    before, after = result.stderr.split("REPLAYS\n")
    replays, rest = after.split("END\n")
    assert before.count("hipGraphInstantiate") > 0 and replays.count("hipGraphLaunch") > 0
    assert replays.count("hipGraphInstantiate") == 0 and replays.count("hipGraphCreate") == 0
