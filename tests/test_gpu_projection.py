"""The general projection at the edges of its tiles, slabs and K ranges.

Against fp64: an fp32 sum of K products differs from the exact one by at most
``(K + ranges) 2^-24 sum |x w|`` whatever its order; the stored value adds one rounding to the
payload dtype (at most one ulp once the sum may sit on the other side of a rounding boundary).
"""

from __future__ import annotations

import ctypes

import pytest
import torch

from crosspool_amd import _native
from crosspool_amd.ffn import RouterProjectionPrecision
from crosspool_amd.moe import MoeRouterWeights, Router

pytestmark = pytest.mark.gpu

CODES = {torch.bfloat16: _native.XP_DTYPE_BF16, torch.float16: _native.XP_DTYPE_F16, torch.float32: _native.XP_DTYPE_F32}
MANTISSA = {torch.bfloat16: 7, torch.float16: 10, torch.float32: 23}


def _pointer(tensor):
    return None if tensor is None else ctypes.c_void_p(tensor.data_ptr())


def _project(x, w, bias, out, workspace, nbytes):
    _native.call(
        "xp_projection_split", _pointer(x), x.shape[0], x.shape[1], _pointer(w), w.shape[0], _pointer(bias),
        _pointer(out), CODES[x.dtype], None, _pointer(workspace) if nbytes else None, nbytes,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream),
    )
    torch.cuda.synchronize()


def _assert_within_bound(out, x, w, bias):
    exact = x.cpu().double() @ w.cpu().double().t()
    magnitude = x.cpu().double().abs() @ w.cpu().double().abs().t()
    if bias is not None:
        exact += bias.cpu().double()
        magnitude += bias.cpu().double().abs()
    sums = (x.shape[1] + 17) * 2.0**-24 * magnitude
    rounding = exact.abs() * 2.0 ** -MANTISSA[out.dtype] if out.dtype is not torch.float32 else 0.0
    floor = 2.0**-24 if out.dtype is torch.float16 else 0.0  # half an fp16 subnormal step
    excess = (out.cpu().double() - exact).abs() - sums - rounding - floor
    assert bool((excess <= 0).all()), f"largest excess over the bound {excess.max():.3e}"


def _operands(device, rows, k, n, dtype, offset=0):
    generator = torch.Generator(device=device).manual_seed(rows * 131 + k * 17 + n)
    # `offset` leaves every operand aligned to its element only.
    x = torch.randn(rows * k + offset, device=device, generator=generator).to(dtype)[offset:].view(rows, k)
    w = torch.randn(n * k + offset, device=device, generator=generator).to(dtype)[offset:].view(n, k)
    bias = torch.randn(n, device=device, generator=generator)
    out = torch.full((rows * n + offset + 16,), 7.0, device=device, dtype=dtype)
    return x, w, bias, out


# Rows and columns around the 64- and 128-row tiles, K around a chunk (8 or 4 columns), a slab
# (64 or 32) and the K ranges.
@pytest.mark.parametrize("dtype", tuple(CODES))
@pytest.mark.parametrize(
    "rows,k,n",
    ((1, 1, 1), (1, 7, 3), (63, 9, 65), (64, 64, 64), (65, 63, 66), (3, 65, 129), (129, 31, 2), (2, 33, 63),
     (5, 1025, 67), (257, 2053, 65), (300, 129, 4097), (1030, 40, 4100)),
)
def test_projection_edges(device, dtype, rows, k, n):
    print(f"projection {dtype} {rows}x{n}x{k}", flush=True)
    x, w, bias, out = _operands(device, rows, k, n, dtype, offset=1)
    nbytes = _native.library().xp_projection_workspace_bytes(rows, n, k, CODES[dtype])
    workspace = torch.full((max(nbytes, 16),), 0xff, device=device, dtype=torch.uint8)
    _project(x, w, bias, out[1:], workspace, nbytes)
    _assert_within_bound(out[1: 1 + rows * n].view(rows, n), x, w, bias)
    assert bool((out[:1] == 7).all()) and bool((out[1 + rows * n:] == 7).all()), "stores outside the output"


# A workspace below the query splits K less, down to not at all; every split agrees with fp64.
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float32))
def test_projection_splits_k_by_its_workspace(device, dtype):
    rows, k, n = 33, 3001, 130
    x, w, bias, out = _operands(device, rows, k, n, dtype)
    full = _native.library().xp_projection_workspace_bytes(rows, n, k, CODES[dtype])
    plane = rows * n * 4
    assert full >= 4 * plane
    for nbytes in (0, plane, 2 * plane + 5, 3 * plane, full):
        print(f"projection workspace {nbytes} of {full}", flush=True)
        workspace = torch.full((full,), 0xff, device=device, dtype=torch.uint8)
        _project(x, w, bias, out, workspace, nbytes)
        _assert_within_bound(out[: rows * n].view(rows, n), x, w, bias)
        assert bool((workspace[nbytes:] == 0xff).all()), "sums outside the workspace"


def test_projection_keeps_infinities_and_nan_in_their_rows(device):
    rows, k, n = 70, 77, 66
    x, w, bias, out = _operands(device, rows, k, n, torch.bfloat16)
    x[3, 5], x[69, 76], w[65, 0] = float("inf"), float("nan"), float("inf")
    _project(x, w, bias, out, None, 0)
    got, expected = out[: rows * n].view(rows, n).float().cpu(), x.float().cpu() @ w.float().cpu().t() + bias.cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(expected))
    assert torch.equal(torch.isinf(got), torch.isinf(expected)) and torch.equal(got[torch.isinf(got)], expected[torch.isinf(expected)])


# The Router's fp32 logits: unsplit and K-split projections, capacities above the live rows,
# 16-bit and fp32 weights, widths that are no multiple of 8.
@pytest.mark.parametrize("precision", (RouterProjectionPrecision.FP32, RouterProjectionPrecision.FP32_LOGITS))
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize("rows,capacity,hidden,experts", ((1, 1, 40, 17), (9, 16, 2048, 128), (33, 66, 2048, 128), (65, 128, 1003, 130)))
def test_router_fp32_logits(device, precision, dtype, rows, capacity, hidden, experts):
    print(f"router {precision.name} {dtype} {rows}/{capacity}x{experts}x{hidden}", flush=True)
    generator = torch.Generator(device=device).manual_seed(rows + hidden)
    x = torch.randn((capacity, hidden), device=device, generator=generator).to(dtype)
    weight_dtype = torch.float32 if precision is RouterProjectionPrecision.FP32 else dtype
    w = torch.randn((experts, hidden), device=device, generator=generator).to(weight_dtype)
    router = Router(row_capacity=capacity, hidden_size=hidden, routed_expert_count=experts, routed_topk=4,
                    precision=precision, device=device, payload_dtype=dtype)
    router.run_into(hidden_states=x, router_weights=MoeRouterWeights(w), rows=rows)
    torch.cuda.synchronize()
    _assert_within_bound(router.logits[:rows], x[:rows], w, None)
    scores, order = torch.softmax(router.logits[:rows].cpu(), dim=1).sort(dim=1, descending=True, stable=True)
    assert torch.equal(router.ids[:rows].cpu().long(), order[:, :4])
    torch.testing.assert_close(router.weights[:rows].cpu(), scores[:, :4] / scores[:, :4].sum(1, keepdim=True), rtol=1e-5,
                               atol=1e-6)


# A Router splits K as far as its workspace has room for the sums: one that holds the logits
# only, and one sized for a capacity whose own choice needs less scratch than the live rows'.
@pytest.mark.parametrize("precision", tuple(RouterProjectionPrecision))
@pytest.mark.parametrize("rows,capacity,hidden,experts", ((9, 16, 2048, 128), (33, 66, 2048, 128), (639, 640, 2048, 128),
                                                          (512, 513, 4096, 256), (65, 128, 1003, 130)))
def test_router_runs_in_smaller_workspaces(device, precision, rows, capacity, hidden, experts):
    generator = torch.Generator(device=device).manual_seed(rows + hidden)
    x = torch.randn((capacity, hidden), device=device, generator=generator).bfloat16()
    weight_dtype = torch.float32 if precision is RouterProjectionPrecision.FP32 else torch.bfloat16
    w = torch.randn((experts, hidden), device=device, generator=generator).to(weight_dtype)
    router = Router(row_capacity=capacity, hidden_size=hidden, routed_expert_count=experts, routed_topk=4,
                    precision=precision, device=device)
    whole = router.workspace
    logits = rows * experts * router.logits.element_size()
    for nbytes in (whole.numel(), (logits + 255) // 256 * 256):
        print(f"router {precision.name} {rows}/{capacity}x{experts}x{hidden} workspace {nbytes}", flush=True)
        whole.fill_(0x7f)
        router.workspace = whole[:nbytes]
        router.run_into(hidden_states=x, router_weights=MoeRouterWeights(w), rows=rows)
        torch.cuda.synchronize()
        _assert_within_bound(router.logits[:rows], x[:rows], w, None)
        assert bool((whole[nbytes:] == 0x7f).all()), "sums outside the workspace"


# 16-bit projections of whole 16-byte rows, which the tuned kernels serve: every epilogue, with
# and without the workspace, around the decode sizes and the tiles.
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize("epilogue", ("none", "bias", "silu", "bias+silu", "gelu", "bias+gelu"))
def test_aligned_projections(device, dtype, epilogue):
    gated = epilogue not in ("none", "bias")
    for rows, k, n in ((1, 64, 16), (8, 1000, 528), (9, 2048, 2064), (17, 4096, 272), (33, 512, 1040), (65, 64, 32),
                       (130, 2048, 2064), (257, 1000, 4112), (300, 6144, 272), (520, 4096, 528)):
        print(f"aligned projection {dtype} {epilogue} {rows}x{n}x{k}", flush=True)
        x, w, bias, _ = _operands(device, rows, k, n, dtype)
        w.mul_(k**-0.5)
        bias = bias if "bias" in epilogue else None
        desc = None
        if gated:
            desc = _native.ActivationDesc()
            desc.function = _native.XP_ACTIVATION_GELU if "gelu" in epilogue else _native.XP_ACTIVATION_SILU
            desc.approximate_tanh, desc.alpha, desc.gated = int("gelu" in epilogue), 1.0, 1
            desc.has_limit, desc.limit, desc.up_offset = 1, 3.0, 0.5
        projected = x.double() @ w.double().t() + (0.0 if bias is None else bias.double())
        if gated:
            rounded = projected.to(dtype).double()
            gate, up = rounded[:, 0::2].clamp(max=3.0), rounded[:, 1::2].clamp(-3.0, 3.0)
            act = torch.nn.functional.gelu(gate, approximate="tanh") if "gelu" in epilogue else gate * torch.sigmoid(gate)
            expected = act * (up + 0.5)
        nbytes = _native.library().xp_projection_workspace_bytes(rows, n, k, CODES[dtype])
        workspace = torch.empty(max(nbytes, 16), device=device, dtype=torch.uint8)
        for size in sorted({0, nbytes}):
            out = torch.full((rows, n // 2 if gated else n), 7.0, device=device, dtype=dtype)
            _native.call(
                "xp_projection_split", _pointer(x), rows, k, _pointer(w), n, _pointer(bias), _pointer(out), CODES[dtype],
                None if desc is None else ctypes.byref(desc), _pointer(workspace) if size else None, size,
                ctypes.c_void_p(torch.cuda.current_stream().cuda_stream),
            )
            torch.cuda.synchronize()
            if gated:
                # One rounding of the output and the few activations whose input rounds the other way.
                error = (out.double() - expected).norm() / expected.norm()
                assert error <= 2.0 ** -(MANTISSA[dtype] + 1), f"{rows}x{n}x{k} workspace {size}: {error:.2e}"
            else:
                _assert_within_bound(out, x, w, bias)


# The other epilogues of the same routes: ReLU, GELU by erf and its tanh approximation, and Gates
# without a limit, where the tile kernels or the general one apply them and over K ranges.
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize("biased", (False, True))
@pytest.mark.parametrize("function", ("silu", "relu", "gelu", "gelu_tanh"))
@pytest.mark.parametrize("limit", (None, 1.5))
def test_aligned_projection_activations(device, dtype, biased, function, limit):
    code = {"silu": _native.XP_ACTIVATION_SILU, "relu": _native.XP_ACTIVATION_RELU}.get(function, _native.XP_ACTIVATION_GELU)
    desc = _native.ActivationDesc()
    desc.function, desc.approximate_tanh, desc.alpha, desc.gated = code, int(function == "gelu_tanh"), 1.25, 1
    desc.has_limit, desc.limit, desc.up_offset = int(limit is not None), limit or 0.0, 0.25
    for rows, k, n in ((64, 2048, 2064), (65, 2048, 8208), (130, 2048, 2064), (257, 4096, 4112), (700, 1000, 8192)):
        print(f"activation {dtype} biased={biased} {function} limit={limit} {rows}x{n}x{k}", flush=True)
        x, w, bias, _ = _operands(device, rows, k, n, dtype)
        w.mul_(k**-0.5)
        projected = x.double() @ w.double().t() + (bias.double() if biased else 0.0)
        gate, up = projected.to(dtype).double()[:, 0::2], projected.to(dtype).double()[:, 1::2]
        if limit is not None:
            gate, up = gate.clamp(max=limit), up.clamp(-limit, limit)
        if function == "silu":
            act = gate / (1.0 + torch.exp(-1.25 * gate))
        elif function == "relu":
            act = gate.clamp(min=0.0)
        else:
            act = torch.nn.functional.gelu(gate, approximate="tanh" if function == "gelu_tanh" else "none")
        expected = act * (up + 0.25)
        nbytes = _native.library().xp_projection_workspace_bytes(rows, n, k, CODES[dtype])
        workspace = torch.empty(max(nbytes, 16), device=device, dtype=torch.uint8)
        for size in sorted({0, nbytes}):
            out = torch.full((rows, n // 2), 7.0, device=device, dtype=dtype)
            _native.call(
                "xp_projection_split", _pointer(x), rows, k, _pointer(w), n, _pointer(bias) if biased else None, _pointer(out),
                CODES[dtype], ctypes.byref(desc), _pointer(workspace) if size else None, size,
                ctypes.c_void_p(torch.cuda.current_stream().cuda_stream),
            )
            torch.cuda.synchronize()
            # One rounding of the output and the few activations whose input rounds the other way.
            error = (out.double() - expected).norm() / expected.norm()
            assert error <= 2.0 ** -(MANTISSA[dtype] + 1), f"{rows}x{n}x{k} workspace {size}: {error:.2e}"


# Infinities and NaN stay in their rows and columns on every route: K ends inside a slab and rows
# and weight rows inside tiles, where a kernel's padding must not meet them.
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize("epilogue", ("none", "bias", "silu", "bias+silu", "relu", "bias+gelu"))
def test_aligned_projections_keep_infinities_and_nan_in_their_rows(device, dtype, epilogue):
    gated = epilogue not in ("none", "bias")
    desc = _native.ActivationDesc()
    desc.function = (_native.XP_ACTIVATION_GELU if "gelu" in epilogue else _native.XP_ACTIVATION_RELU if "relu" in epilogue
                     else _native.XP_ACTIVATION_SILU)
    desc.alpha, desc.gated = 1.0, 1
    for rows, k, n in ((7, 1000, 528), (13, 2056, 272), (40, 1000, 528), (70, 1000, 528), (130, 2056, 2064), (300, 3000, 1040)):
        print(f"infinities {dtype} {epilogue} {rows}x{n}x{k}", flush=True)
        x, w, bias, _ = _operands(device, rows, k, n, dtype)
        w.mul_(k**-0.5)
        # the first and last columns of rows inside and at the end of a tile
        x[2, 0], x[4, k - 1], x[rows - 1, 5], w[n - 1, 3], w[33, k - 1] = (
            float("inf"), float("nan"), float("-inf"), float("inf"), float("nan"))
        bias = bias if "bias" in epilogue else None
        projected = x.float().cpu() @ w.float().cpu().t() + (0.0 if bias is None else bias.cpu())
        expected = projected
        if gated:
            gate, up = projected.to(dtype).float()[:, 0::2], projected.to(dtype).float()[:, 1::2]
            if "relu" in epilogue:
                act = torch.where(gate.isnan() | (gate > 0), gate, torch.zeros_like(gate))
            elif "gelu" in epilogue:
                act = 0.5 * gate * (1.0 + torch.erf(gate * 0.5**0.5))
            else:
                act = gate / (1.0 + torch.exp(-gate))
            expected = act * up
        expected = expected.to(dtype).float()
        nbytes = _native.library().xp_projection_workspace_bytes(rows, n, k, CODES[dtype])
        workspace = torch.empty(max(nbytes, 16), device=device, dtype=torch.uint8)
        for size in sorted({0, nbytes}):
            out = torch.full((rows, n // 2 if gated else n), 7.0, device=device, dtype=dtype)
            _native.call(
                "xp_projection_split", _pointer(x), rows, k, _pointer(w), n, _pointer(bias), _pointer(out), CODES[dtype],
                ctypes.byref(desc) if gated else None, _pointer(workspace) if size else None, size,
                ctypes.c_void_p(torch.cuda.current_stream().cuda_stream),
            )
            torch.cuda.synchronize()
            got = out.float().cpu()
            assert torch.equal(torch.isnan(got), torch.isnan(expected)), f"{rows}x{n}x{k} workspace {size}"
            assert torch.equal(torch.isinf(got), torch.isinf(expected))
            assert torch.equal(got[torch.isinf(got)], expected[torch.isinf(expected)])


# A SiLU epilogue is evaluated with expf and an IEEE divide whichever kernel the row count, the
# bias and the workspace choose.  Every row of x is a unit vector, so the projected values are the
# weights themselves and only the activation and the store round (alpha is a power of two).  The
# activation's fp32 steps (expf within one ulp, one addition, one division, one product, half an
# ulp each) leave at most 2.5 x 2^-24 of an output, so it rounds the other way only within that of
# a tie: a share of at most 2 x 2.5 x 2^-24 of one spacing, which is at least 2^-m / 2 of the
# output.  (rcp and __expf are several times further off at these Gates, where the product with
# log2(e) has lost bits.)
@pytest.mark.parametrize("dtype,alpha,gates,ups", ((torch.bfloat16, 1.0, (-86.0, -40.0), (1.0, 2.0)),
                                                   (torch.float16, 2.0**-11, (-60000.0, -50000.0), (30000.0, 60000.0))))
@pytest.mark.parametrize("biased", (False, True))
@pytest.mark.parametrize("rows", (8, 64, 65, 256))
def test_silu_epilogues_are_evaluated_in_full_precision(device, dtype, alpha, gates, ups, biased, rows):
    print(f"silu epilogue {dtype} biased={biased} {rows} rows", flush=True)
    k, n = 1024, 16384
    generator = torch.Generator(device=device).manual_seed(rows)
    w = torch.empty((n, k), device=device, dtype=dtype)
    for offset, (low, high) in enumerate((gates, ups)):
        w[offset::2] = (low + (high - low) * torch.rand((n // 2, k), device=device, generator=generator)).to(dtype)
    x = torch.eye(k, device=device, dtype=dtype)[:rows].contiguous()
    bias = torch.zeros(n, device=device) if biased else None
    desc = _native.ActivationDesc()
    desc.function, desc.alpha, desc.gated = _native.XP_ACTIVATION_SILU, alpha, 1
    nbytes = _native.library().xp_projection_workspace_bytes(rows, n, k, CODES[dtype])
    workspace = torch.empty(max(nbytes, 16), device=device, dtype=torch.uint8)
    gate, up = w[0::2, :rows].cpu().double().t(), w[1::2, :rows].cpu().double().t()
    expected = (gate / (1.0 + torch.exp(-alpha * gate)) * up).to(dtype)
    for size in sorted({0, nbytes}):
        out = torch.empty((rows, n // 2), device=device, dtype=dtype)
        _native.call(
            "xp_projection_split", _pointer(x), rows, k, _pointer(w), n, _pointer(bias), _pointer(out), CODES[dtype],
            ctypes.byref(desc), _pointer(workspace) if size else None, size,
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream),
        )
        torch.cuda.synchronize()
        share = (out.cpu() != expected).double().mean().item()
        bound = 2 * 2.5 * 2.0**-24 / 2.0 ** -(MANTISSA[dtype] + 1)
        assert share <= bound, f"workspace {size}: share of other roundings {share:.2e} of at most {bound:.2e}"


# Grids whose weight tiles do not split over the XCDs: every tile is computed once, whatever the
# blocks of an XCD's run (runs shorter than a block, one band of 8 token tiles and several).
@pytest.mark.parametrize("n", (384, 640, 896, 1536, 2568, 3328))
def test_tile_order_covers_every_tile(device, n):
    k = 520
    generator = torch.Generator(device=device).manual_seed(n)
    w = (torch.randn((n, k), device=device, generator=generator) * k**-0.5).bfloat16()
    for rows in (65, 130, 163, 275, 358, 520, 700, 1100, 2100):
        print(f"tile order {rows}x{n}x{k} {_native.gemm_variant(rows, n, k, False)}", flush=True)
        x = torch.randn((rows, k), device=device, generator=generator).bfloat16()
        out = torch.full((rows, n), 7.0, device=device, dtype=torch.bfloat16)
        nbytes = _native.gemm_workspace_bytes(rows, n, k, False)
        workspace = torch.empty(max(nbytes, 16), device=device, dtype=torch.uint8)
        _native.call("xp_gemm_down", _pointer(x), rows, k, _pointer(w), n, _pointer(out), None, rows,
                     _pointer(workspace) if nbytes else None, nbytes,
                     ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        _assert_within_bound(out, x, w, None)
