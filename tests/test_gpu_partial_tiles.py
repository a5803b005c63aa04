"""Stacks that end inside a tile, where the other files do not reach: Gram-form stacks widened to hold two m x m
stacks, the apply with guarded memory around its parameters, and fp32 blocks whose singular values span decades."""
import ctypes as C

import pytest
import torch

from monarch_muon_amd import MonarchMuonOptimizer, _abi
from monarch_muon_amd.plan import NS_COEFFS, MuonPlanner
from oracle.truth import ns_fp64, rel_fro
from test_gpu_parity import _spectrum_stack, run_ns_only, test_ns_bf16_against_fp64_truth_and_reference as check_chain
from test_gpu_stages import panels, test_partial_tiles_against_fp64_products as check_stages

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
GUARD = 4096  # elements before and after the guarded parameters

# the sides in whole 256-wide tiles qualify for the Gram form, their finer padding alone does not: np = 2 mp
WIDENED = [(2, 200, 264), (2, 776, 456), (2, 456, 776)]


def ids(s):
    return "x".join(map(str, s))


@pytest.mark.parametrize("shape", WIDENED, ids=ids)
def test_widened_stacks_stage_by_stage(shape):
    lay = _abi.ns_layout(*shape[1:], _abi.BF16, shape[0])
    assert lay.np_ == 2 * lay.mp > -(-lay.n // 64) * 64
    print("stages", shape, flush=True)
    check_stages(shape)


@pytest.mark.parametrize("form", ["auto", "standard"])
@pytest.mark.parametrize("shape", WIDENED + [(2, 264, 96)], ids=ids)
def test_widened_stacks_in_both_forms(shape, form):
    plan = _abi.ns_plan(*shape[1:], _abi.BF16, 5, _abi.NS_STANDARD if form == "standard" else 0)
    assert any(op.kind == _abi.NSOP_SYMM for op in plan) == (form == "auto")
    print("chain", shape, form, flush=True)
    check_chain(shape, form)


def guarded(shape, dtype, seed):
    """A parameter between two guards of random values, and the whole storage."""
    gen = torch.Generator().manual_seed(seed)
    n = shape[0] * shape[1] * shape[2]
    hold = (torch.randn(n + 2 * GUARD, generator=gen) * 0.02).to(DEV, dtype)
    return hold[GUARD:GUARD + n].view(shape), hold


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("shape", WIDENED + [(2, 264, 96), (3, 64, 64), (2, 72, 200), (2, 200, 72), (3, 384, 384), (2, 520, 2056),
                                             (2, 1000, 344), (2, 30, 70)], ids=ids)
def test_apply_of_partial_tiles(shape, dtype):
    """PX + apply on its own: param + alpha s P X, X' rounded to bf16 (half a step at the largest entry, a step
    allowed), the sum rounded to the parameter's type (half a step of each); nothing beside the parameters moves."""
    print("apply", shape, dtype, flush=True)
    p, hold = guarded(shape, dtype, 5)
    before = hold.clone()
    gen = torch.Generator().manual_seed(6)
    grad = (torch.randn(shape, generator=gen) * 1e-3).to(DEV, dtype)
    (gl,) = MuonPlanner().plan([p], [grad], [torch.zeros(shape, device=DEV)], torch.bfloat16)
    lib, stream, lay, ws, nb = _abi.lib(), _abi.stream_handle(DEV), gl.ws.layout, gl.ws, gl.nblocks
    coeffs, alpha = (C.c_float * 3)(*NS_COEFFS), -0.05
    for t in (ws.x0, ws.x1, ws.a, ws.p):
        t.view(torch.bfloat16).fill_(float("nan"))

    def run(kind, in0, in1, out, scaled=0):
        op = _abi.NsOp(kind, in0, in1, out, scaled, 0)
        _abi.check(lib.mmuon_ns_run_op(C.byref(gl.struct), C.byref(op), coeffs, C.c_float(alpha), stream), "run_op")
        torch.cuda.synchronize()

    _abi.check(lib.mmuon_momentum_pack(C.byref(gl.struct), 0.0, stream), "pack")
    run(_abi.NSOP_SYRK, _abi.NSB_X0, -1, _abi.NSB_A, 1)
    run(_abi.NSOP_POLY, _abi.NSB_A, -1, _abi.NSB_P)
    assert torch.equal(hold, before)
    run(_abi.NSOP_PX_APPLY, _abi.NSB_P, _abi.NSB_X0, _abi.NSB_PARAM, 1)
    tile = torch.arange(lay.mp, device=DEV) // 256
    pm = panels(ws.p, nb, lay.mp, lay.mp)
    pm = torch.where(tile[:, None] <= tile[None, :], pm, pm.transpose(1, 2))
    u = ws.scale.double().view(nb, 1, 1) * (pm @ panels(ws.x0, nb, lay.mp, lay.np_))
    u = u[:, :lay.m, :lay.n]
    u = u.transpose(1, 2) if gl.transposed else u
    n = p.numel()
    old = before[GUARD:GUARD + n].view(shape).double()
    want = old + alpha * u
    step = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23
    bound = abs(alpha) * 2.0 ** -8 * u.abs().amax((1, 2), keepdim=True) + step * want.abs()
    assert torch.all((p.double() - want).abs() <= bound)
    assert torch.equal(hold[:GUARD], before[:GUARD]) and torch.equal(hold[GUARD + n:], before[GUARD + n:])


@pytest.mark.parametrize("ns", ["bf16", "own"])
@pytest.mark.parametrize("shape", WIDENED + [(3, 150, 200), (2, 130, 130), (2, 8, 16), (5, 33, 70), (70, 384, 384)],
                         ids=ids)
def test_a_step_writes_its_parameters_only(shape, ns):
    print("step", shape, ns, flush=True)
    dtype = torch.bfloat16 if ns == "bf16" else torch.float32
    p, hold = guarded(shape, dtype, 7)
    p = p.requires_grad_()
    before = hold.clone()
    p.grad = (torch.randn(shape, generator=torch.Generator().manual_seed(8)) * 1e-3).to(DEV, dtype)
    MonarchMuonOptimizer([p], [], ns_dtype=torch.bfloat16 if ns == "bf16" else None).step()
    torch.cuda.synchronize()
    n = p.numel()
    assert torch.isfinite(hold).all() and not torch.equal(hold[GUARD:GUARD + n], before[GUARD:GUARD + n])
    assert torch.equal(hold[:GUARD], before[:GUARD]) and torch.equal(hold[GUARD + n:], before[GUARD + n:])


@pytest.mark.parametrize("sides", [(256, 256), (512, 1376), (136, 96), (1024, 1024)], ids=ids)
def test_fp32_with_singular_values_over_four_decades(sides):
    """The fp32 path's bar, 1e-5 per block, where small singular values make the iterations amplify rounding errors
    most (one bf16 term less in the split, and the bar is missed)."""
    print("four decades", sides, flush=True)
    m, n = min(sides), max(sides)
    g = _spectrum_stack(m, n, [torch.logspace(0, -4, m, dtype=torch.float64)] * 2, 3).float()
    g = g.transpose(1, 2).contiguous() if sides[0] > sides[1] else g
    e = rel_fro(run_ns_only(g.to(DEV), None).double(), ns_fp64(g.double()))
    print("vs fp64", e.tolist())
    assert e.max() < 1e-5, e


@pytest.mark.parametrize("sides", [(256, 256), (512, 640), (1032, 520)], ids=ids)
def test_fp32_blocks_do_not_depend_on_their_number(sides):
    """One to 24 blocks: dealt to the XCDs whole (8, 16, 24) or spread over them, in 64- and in 128-wide tiles; a
    block's result is the same, bit for bit."""
    print("number of blocks", sides, flush=True)
    g = (torch.randn((24, *sides), generator=torch.Generator().manual_seed(9)) * 1e-3).to(DEV)
    want = run_ns_only(g, None)
    assert rel_fro(want[:2].double(), ns_fp64(g[:2].cpu().double())).max() < 1e-5
    for n in (1, 2, 3, 5, 8, 12, 16, 20, 23):
        assert torch.equal(run_ns_only(g[:n], None), want[:n]), n
