"""GPU parity: the HIP step (through the C ABI) against the CPU oracle and the
reference's own golden vectors.

Bars: updated weights and momentum within 1e-2 relative
Frobenius error per block with bf16 Newton-Schulz, within 1e-5 in fp32;
identical block grouping and ordering.  The momentum update is elementwise and
is checked bit for bit.  bf16 Newton-Schulz output itself is held to 1.5x the
reference's own bf16 error against the fp64 truth.
"""
import ctypes as C
import io

import numpy as np
import pytest
import torch

from golden_inputs import CASES, make_case
from monarch_muon_amd import CoatStateMonarchMuon, MonarchMuonOptimizer, QuantizationConfig, _abi
from monarch_muon_amd.plan import NS_COEFFS, MuonPlanner
from monarch_muon_amd.workloads import WORKLOADS, parameter_inventory
from oracle import codec
from oracle.step import ReferenceMonarchMuon, newton_schulz_batched
from oracle.truth import ns_fp64, rel_fro

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
GOLDEN = __import__("pathlib").Path(__file__).resolve().parent / "golden"
BF16_TOL, F32_TOL = 1e-2, 1e-5


def blocks_rel(a, b):
    """Per-block relative Frobenius error of two (nb, r, c) (or 1-D/2-D) tensors."""
    a, b = a.detach().cpu().double(), b.detach().cpu().double()
    if a.dim() < 3:
        a, b = a.reshape(1, 1, -1), b.reshape(1, 1, -1)
    return rel_fro(a, b)


# ---------------------------------------------------------------- Newton-Schulz alone
NS_SHAPES = [(4, 256, 256), (2, 512, 1368), (2, 1376, 512), (2, 1024, 1024), (1, 1024, 2752),
             (2, 96, 136), (2, 136, 96), (3, 64, 64), (2, 96, 600), (1, 600, 96)]


def run_ns_only(g: torch.Tensor, ns_dtype, flags: int = 0) -> torch.Tensor:
    """Newton-Schulz of the stack ``g`` through the library: pack with momentum 0
    (buf <- 0*buf + g = g), then the NS plan without the apply (``flags``:
    ``NS_STANDARD`` for the three-product chain on every group)."""
    p = torch.zeros_like(g, dtype=torch.bfloat16 if ns_dtype == torch.bfloat16 else torch.float32)
    buf = torch.zeros_like(g, dtype=torch.float32)
    grad = g.to(p.dtype)
    planner = MuonPlanner()
    (gl,) = planner.plan([p], [grad], [buf], ns_dtype)
    lib = _abi.lib()
    stream = _abi.stream_handle(DEV)
    _abi.check(lib.mmuon_momentum_pack(C.byref(gl.struct), 0.0, stream), "pack")
    coeffs = (C.c_float * 3)(*NS_COEFFS)
    _abi.check(lib.mmuon_newton_schulz_apply(C.byref(gl.struct), 5, coeffs, 0.0, _abi.NS_NO_APPLY | flags,
                                             stream), "ns")
    torch.cuda.synchronize()
    lay = gl.ws.layout
    out = _abi.ns_output_buffer(gl.rows, gl.cols, lay.ns_dtype, 5, flags)
    x = gl.ws.x_view(out, torch.bfloat16 if lay.ns_dtype == _abi.BF16 else torch.float32, gl.nblocks)
    x = x[:, :lay.m, :lay.n].float().cpu()
    return x.transpose(1, 2) if gl.transposed else x


@pytest.mark.parametrize("form", ["auto", "standard"])
@pytest.mark.parametrize("shape", NS_SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_ns_bf16_against_fp64_truth_and_reference(shape, form):
    """Both evaluation orders (the Gram form runs on the rectangular shapes with
    a long side at least twice the short one after padding) against fp64."""
    gen = torch.Generator().manual_seed(11)
    g = (torch.randn(shape, generator=gen) * 1e-3).to(DEV)
    ours = run_ns_only(g, torch.bfloat16, _abi.NS_STANDARD if form == "standard" else 0)
    ref_bf16 = newton_schulz_batched(g.cpu().to(torch.bfloat16)).float()
    truth = ns_fp64(g.cpu().to(torch.bfloat16).double())
    e_ours = rel_fro(ours, truth)
    e_ref = rel_fro(ref_bf16, truth)
    d_ref = rel_fro(ours, ref_bf16)
    print(f"NS {shape} {form}: ours vs fp64 {e_ours.max():.4f}, reference-bf16 vs fp64 {e_ref.max():.4f}, "
          f"ours vs reference-bf16 {d_ref.max():.4f}")
    assert torch.all(e_ours <= 1.5 * e_ref + 2e-3), (e_ours, e_ref)
    # the two bf16 evaluations differ from each other by no more than their
    # independent rounding errors explain (they add in quadrature: measured
    # d_ref / sqrt(e_ours^2 + e_ref^2) = 0.98-1.00 on these shapes; an error of
    # ours opposite to the reference's would approach e_ours + e_ref)
    assert torch.all(d_ref <= 1.15 * torch.sqrt(e_ours ** 2 + e_ref ** 2) + 1e-3), (d_ref, e_ours, e_ref)


def _spectrum_stack(m, n, spectra, seed):
    """One (m x n) block per singular-value profile: U diag(s) V^T with random
    orthonormal U, V (fp64, rounded to fp32)."""
    gen = torch.Generator().manual_seed(seed)
    out = []
    for sv in spectra:
        u, _ = torch.linalg.qr(torch.randn(m, m, generator=gen, dtype=torch.float64))
        v, _ = torch.linalg.qr(torch.randn(n, m, generator=gen, dtype=torch.float64))
        out.append(((u * sv) @ v.T).float())
    return torch.stack(out)


@pytest.mark.parametrize("shape", [(1024, 2752), (512, 1376), (2752, 1024)], ids=lambda s: "x".join(map(str, s)))
def test_ns_bf16_ill_conditioned_blocks(shape):
    """Blocks whose singular values span decades (where a Gram recursion in bf16
    without the rebuild of X drifts by up to 1.3 in relative Frobenius error):
    both evaluation orders stay within 1.5x the reference's own bf16 error."""
    r, c = shape
    m, n = min(r, c), max(r, c)
    d = torch.float64
    spectra = [torch.logspace(0, -3, m, dtype=d), torch.logspace(0, -5, m, dtype=d),
               torch.cat([torch.logspace(0, -1, 16, dtype=d), torch.full((m - 16,), 1e-3, dtype=d)]),
               torch.cat([torch.ones(1, dtype=d), torch.full((m - 1,), 1e-4, dtype=d)])]
    g = _spectrum_stack(m, n, spectra, seed=21)
    if r > c:
        g = g.transpose(1, 2).contiguous()
    ref_bf16 = newton_schulz_batched(g.to(torch.bfloat16)).float()
    truth = ns_fp64(g.to(torch.bfloat16).double())
    e_ref = rel_fro(ref_bf16, truth)
    for flags in (0, _abi.NS_STANDARD):
        ours = run_ns_only(g.to(DEV), torch.bfloat16, flags)
        e_ours = rel_fro(ours, truth)
        print(f"NS {shape} flags {flags}: ours {[round(float(e), 4) for e in e_ours]}, "
              f"reference {[round(float(e), 4) for e in e_ref]}")
        assert torch.all(e_ours <= 1.5 * e_ref + 2e-3), (flags, e_ours, e_ref)


@pytest.mark.parametrize("shape", [(4, 256, 256), (2, 256, 688), (2, 688, 256), (2, 96, 136), (2, 512, 512),
                                   (2, 1376, 512), (2, 512, 1376), (3, 200, 72)],
                         ids=lambda s: "x".join(map(str, s)))
def test_ns_fp32_against_fp64_truth(shape):
    """fp32 Newton-Schulz (the pretrain copy's, fp32 momentum) against fp64 on
    the same fp32 input: within 1e-5 relative Frobenius per block, the
    reference CPU oracle's fp32 error printed beside it."""
    gen = torch.Generator().manual_seed(12)
    g = (torch.randn(shape, generator=gen) * 1e-3).to(DEV)
    ours = run_ns_only(g, None)
    truth = ns_fp64(g.cpu().double())
    e = rel_fro(ours, truth)
    e_ref = rel_fro(newton_schulz_batched(g.cpu()).double(), truth)
    print(f"NS fp32 {shape}: ours vs fp64 {e.max():.2e}, oracle fp32 vs fp64 {e_ref.max():.2e}")
    assert e.max() < 1e-5, (e, e_ref)


# both tile sizes of the fp32 kernels (128-wide from 256 such tiles per launch), K extents that end in an odd or a
# single step, and 64-wide tiles that hold only padding
@pytest.mark.parametrize("shape", [(26, 512, 512), (256, 104, 128), (60, 200, 264), (64, 264, 136), (3, 150, 200),
                                   (2, 8, 16), (1, 16, 8), (2, 130, 130)], ids=lambda s: "x".join(map(str, s)))
def test_ns_fp32_tiles_against_fp64_truth(shape):
    """The bar of the fp32 path, 1e-5; one block of the stack set to NaN and one holding an infinity come out
    non-finite and leave the others untouched."""
    gen = torch.Generator().manual_seed(21)
    g = (torch.randn(shape, generator=gen) * 1e-3).to(DEV)
    ours = run_ns_only(g, None)
    e = rel_fro(ours, ns_fp64(g.cpu().double()))
    print(f"NS fp32 {shape}: vs fp64 {e.max():.2e}")
    assert e.max() < 1e-5, e
    if shape[0] > 2:
        bad = g.clone()
        bad[0] = float("nan")
        bad[2, 1, 3] = float("inf")
        out = run_ns_only(bad, None)
        assert not torch.isfinite(out[0]).any() and not torch.isfinite(out[2]).any()
        assert torch.equal(out[1], ours[1]) and torch.equal(out[3:], ours[3:])


@pytest.mark.parametrize("shape", [(2, 256, 256), (2, 256, 688), (2, 688, 256)], ids=lambda s: "x".join(map(str, s)))
def test_ns_zero_block_gives_zero(shape):
    """A zero block stays zero, alone and beside a non-zero block of the same
    stack (the Gram form's polynomials of a zero Gram matrix are a^k I, finite,
    applied to a zero X)."""
    g = torch.zeros(shape, device=DEV)
    assert torch.count_nonzero(run_ns_only(g, torch.bfloat16)) == 0
    g[1] = torch.randn(shape[1:], generator=torch.Generator().manual_seed(3)).to(DEV) * 1e-3
    out = run_ns_only(g, torch.bfloat16)
    assert torch.count_nonzero(out[0]) == 0 and bool(torch.isfinite(out).all())
    truth = ns_fp64(g[1:].cpu().to(torch.bfloat16).double())
    assert float(rel_fro(out[1:], truth).max()) < 0.03


# ---------------------------------------------------------------- golden vectors (reference-written)
def _run_case_gpu(case):
    muon, adamw, bufs = make_case(case, device=DEV)
    opt = MonarchMuonOptimizer(muon, adamw, lr=case["lr"], momentum=0.95,
                               ns_dtype=torch.bfloat16 if case["variant"] == "membench" else None)
    if bufs is not None:
        for p, b in zip(muon, bufs):
            opt.state[p]["momentum_buffer"] = b
    for _ in range(case["steps"]):
        opt.step()
    torch.cuda.synchronize()
    return muon, adamw, opt


@pytest.mark.parametrize("case", CASES, ids=[c["name"] for c in CASES])
def test_step_matches_reference_golden(case):
    gold = torch.load(GOLDEN / f"{case['name']}.pt", weights_only=True)
    muon, adamw, opt = _run_case_gpu(case)
    tol = BF16_TOL if case["variant"] == "membench" else F32_TOL
    for p, q in zip(muon, gold["muon_params"]):
        assert blocks_rel(p, q).max() <= tol
    for p, q in zip(muon, gold["momentum"]):
        ours = opt.state[p]["momentum_buffer"].cpu()
        if ours.dtype == torch.bfloat16:
            # torch's CPU foreach kernels (which wrote the golden) round the scalar
            # momentum to bf16 before multiplying a bf16 tensor; its GPU kernels,
            # the reference's platform, keep it in fp32 (checked bit for bit below)
            ulps = (ours.view(torch.int16).int() - q.view(torch.int16).int()).abs()
            assert ulps.max() <= 1
        else:
            assert torch.equal(ours, q), "momentum must be bit-exact"
    for p, q in zip(adamw, gold["adamw_params"]):
        assert blocks_rel(p, q).max() <= tol
    for p, q, r in zip(adamw, gold["exp_avg"], gold["exp_avg_sq"]):
        assert blocks_rel(opt.state[p]["exp_avg"], q).max() <= tol
        assert blocks_rel(opt.state[p]["exp_avg_sq"], r).max() <= tol


def test_bf16_momentum_bit_exact_against_torch_gpu_semantics():
    # the reference's op sequence executed by torch on this GPU (the oracle module
    # run on device tensors): the momentum update must agree bit for bit
    case = CASES[1]
    muon, adamw, opt = _run_case_gpu(case)
    rm, ra, _ = make_case(case, device=DEV)
    ropt = ReferenceMonarchMuon(rm, ra, lr=case["lr"], momentum=0.95, variant="membench")
    for _ in range(case["steps"]):
        ropt.step()
    torch.cuda.synchronize()
    for p, q in zip(muon, rm):
        assert torch.equal(opt.state[p]["momentum_buffer"], ropt.state[q]["momentum_buffer"])
        assert blocks_rel(p, q).max() <= BF16_TOL


@pytest.mark.parametrize("variant", ["membench", "pretrain"])
def test_adamw_bf16_bit_exact_against_torch_gpu_ops(variant):
    """The AdamW group with bf16 parameters, gradients and (optimizer-created)
    states against the reference's op sequence executed by torch on this GPU
    (membench monarch_muon.py:176-208 as foreach ops; pretrain :176-201 per
    tensor): parameters, exp_avg and exp_avg_sq bit for bit over four steps
    with new gradients before each.  Gradients span 1e-30 to 1e2 (so the second
    moments reach bf16's subnormal range and its top), with exact zeros; the
    shapes give ragged tails and 16-B misaligned tensors."""
    gen = torch.Generator().manual_seed(23)
    shapes = [(512, 300), (1000,), (77,), (33, 129), (2, 3, 5), (4096, 64)]
    w0 = [torch.randn(s, generator=gen) * 0.02 for s in shapes]
    grads = []
    for _ in range(4):
        step_g = []
        for s in shapes:
            mag = 10.0 ** torch.randint(-30, 3, s, generator=gen).double()
            g = (torch.randn(s, generator=gen).double() * mag).float()
            g[torch.rand(s, generator=gen) < 0.05] = 0.0
            step_g.append(g)
        grads.append(step_g)

    def run(cls, **kw):
        muon = [(torch.randn(2, 64, 64, generator=torch.Generator().manual_seed(3)) * 0.02)
                .bfloat16().to(DEV).requires_grad_(True)]
        adamw = [w.bfloat16().to(DEV).requires_grad_(True) for w in w0]
        opt = cls(muon, adamw, lr=0.02, momentum=0.95, **kw)
        for step_g in grads:
            muon[0].grad = torch.full_like(muon[0], 1e-3)
            for p, g in zip(adamw, step_g):
                p.grad = g.bfloat16().to(DEV)
            opt.step()
        torch.cuda.synchronize()
        return adamw, opt

    ours, gopt = run(MonarchMuonOptimizer, ns_dtype=torch.bfloat16 if variant == "membench" else None)
    ref, ropt = run(ReferenceMonarchMuon, variant=variant)
    for p, q in zip(ours, ref):
        assert p.dtype == q.dtype == torch.bfloat16
        assert torch.equal(p, q), "parameters"
        for name in ("exp_avg", "exp_avg_sq"):
            a, b = gopt.state[p][name], ropt.state[q][name]
            assert a.dtype == b.dtype == torch.bfloat16
            assert torch.equal(a, b), name


# ---------------------------------------------------------------- BASELINE configs (reduced where the CPU oracle is slow)
def _workload_params(name, layers=None, adamw_rows=None, seed=0):
    """Seeded fp32 draws in parameter order (W, g, buf per Muon param; W, g per
    AdamW param), cast to the workload dtypes."""
    w = WORKLOADS[name]
    inv = parameter_inventory(w)
    if layers is not None:
        inv = [(n, s, m) for n, s, m in inv if ".h." not in n or int(n.split(".")[2]) < layers]
    gen = torch.Generator().manual_seed(seed)
    out = []
    for n, s, muon in inv:
        if not muon and adamw_rows is not None and len(s) == 2:
            s = (adamw_rows, s[1])
        W = torch.randn(s, generator=gen) * 0.02
        G = torch.randn(s, generator=gen) * 1e-3
        B = torch.randn(s, generator=gen) * 1e-3 if (muon and w.prefill_momentum) else None
        out.append((n, muon, W, G, B))
    return w, out


def _build(w, draws, device, opt_cls, **kw):
    muon, adamw, bufs = [], [], []
    for _, is_muon, W, G, B in draws:
        p = W.to(w.param_dtype).to(device).requires_grad_(True)
        p.grad = G.to(w.param_dtype).to(device)
        (muon if is_muon else adamw).append(p)
        if is_muon:
            bufs.append(B)
    opt = opt_cls(muon, adamw, lr=0.02, momentum=0.95, **kw)
    if w.prefill_momentum and w.momentum_dtype != "fp8":
        for p, b in zip(muon, bufs):
            opt.state[p]["momentum_buffer"] = b.to(w.momentum_dtype).to(device)
    return muon, adamw, opt, bufs


@pytest.mark.parametrize("name,layers,rows,form", [("toy", None, None, "auto"), ("257m-nb2", 2, 512, "auto"),
                                                   ("1.3b-nb4", 1, 256, "auto"), ("1.3b-nb4", 1, 256, "standard"),
                                                   ("6.89b-nb4", 1, 256, "auto"), ("6.89b-nb4", 1, 256, "standard"),
                                                   ("6.89b-nb4-bf16mom", 1, 256, "auto")])
def test_workload_step_matches_oracle(name, layers, rows, form):
    w, draws = _workload_params(name, layers, rows)
    gm, ga, gopt, _ = _build(w, draws, DEV, MonarchMuonOptimizer, ns_dtype=w.ns_dtype, ns_form=form)
    variant = "membench" if w.ns_dtype == torch.bfloat16 else "pretrain"
    cm, ca, copt, _ = _build(w, draws, "cpu", ReferenceMonarchMuon, variant=variant)
    # bf16 momentum: the update as torch's GPU kernels execute the reference's
    # foreach ops (buf *= mu; buf += g; mu kept in fp32), bit for bit
    gpu_mom = None
    if w.momentum_dtype == torch.bfloat16:
        gpu_mom = [(B.to(torch.bfloat16).to(DEV), G.to(torch.bfloat16).to(DEV)) for _, m, _, G, B in draws if m]
    for _ in range(2):
        gopt.step()
        copt.step()
        if gpu_mom is not None:
            bufs = [b for b, _ in gpu_mom]
            torch._foreach_mul_(bufs, 0.95)
            torch._foreach_add_(bufs, [g for _, g in gpu_mom])
    torch.cuda.synchronize()
    tol = BF16_TOL if variant == "membench" else F32_TOL
    worst = 0.0
    for i, (p, q) in enumerate(zip(gm, cm)):
        e = blocks_rel(p, q).max().item()
        worst = max(worst, e)
        assert e <= tol
        ours, ref = gopt.state[p]["momentum_buffer"], copt.state[q]["momentum_buffer"]
        if gpu_mom is None:
            assert torch.equal(ours.cpu(), ref)
        else:
            assert torch.equal(ours, gpu_mom[i][0])
            # torch's CPU kernels round mu to bf16 first (0.9492 for 0.95), which
            # moves entries where mu*buf and g nearly cancel by many bf16 steps;
            # against the CPU oracle the bar is the north star's per-block one
            assert blocks_rel(ours, ref).max() <= BF16_TOL
    for p, q in zip(ga, ca):
        assert blocks_rel(p, q).max() <= tol
    print(f"{name}: worst per-block weight error {worst:.3e} (bar {tol})")


@pytest.mark.parametrize("form", ["auto", "standard"])
def test_ten_steps_with_fresh_gradients_against_oracle(form):
    """Ten steps of one 1.3B layer (square, tall and wide groups; the tall and
    wide ones share their launches and, by default, run the Gram form), a new
    gradient tensor for every parameter before each step, against the oracle
    fed the same gradients: momentum bit for bit after every step, weights
    within the per-block bar after every step (the per-step update errors do not
    compound past it).  The Muon group only: the CPU oracle's bf16 AdamW rounds
    its Python scalars to bf16 (torch's CPU kernels do), which ten steps of
    random gradients move past the bar, while the GPU semantics this build
    follows keep them fp32; AdamW is checked against those elsewhere."""
    w, draws = _workload_params("1.3b-nb4", layers=1)
    draws = [d for d in draws if d[1]]
    gm, ga, gopt, _ = _build(w, draws, DEV, MonarchMuonOptimizer, ns_dtype=torch.bfloat16, ns_form=form)
    cm, ca, copt, _ = _build(w, draws, "cpu", ReferenceMonarchMuon, variant="membench")
    gen = torch.Generator().manual_seed(31)
    worst = 0.0
    for step in range(10):
        for p, q in zip(gm + ga, cm + ca):
            g = (torch.randn(q.shape, generator=gen) * 1e-3).to(q.dtype)
            q.grad = g
            p.grad = g.to(DEV)              # a new tensor at a new address
        gopt.step()
        copt.step()
        torch.cuda.synchronize()
        for p, q in zip(gm, cm):
            assert torch.equal(gopt.state[p]["momentum_buffer"].cpu(), copt.state[q]["momentum_buffer"])
            e = blocks_rel(p, q).max().item()
            worst = max(worst, e)
            assert e <= BF16_TOL, (step, e)
    print(f"ten steps ({form}): worst per-block weight error {worst:.3e}")


# ---------------------------------------------------------------- FP8 codec and FP8-state step
def _narrow_groups(n_groups, spread, mag, seed):
    """Groups of 128 whose |values| lie within a factor ``spread`` of each other
    around ``mag`` (random signs): expand is large there (ratio 1.01 gives
    about 1156), so it magnifies every rounding of |x|/smm."""
    rng = np.random.default_rng(seed)
    a = mag * np.exp(rng.uniform(0, np.log(spread), size=(n_groups, 128)))
    return (a * rng.choice([-1.0, 1.0], size=a.shape)).astype(np.float32).reshape(-1)


@pytest.mark.parametrize("emin", [16, 8])
@pytest.mark.parametrize("fmt", ["E4M3", "E5M2"])
@pytest.mark.parametrize("signed", [True, False], ids=["signed", "unsigned"])
def test_fp8_codec_against_oracle(signed, fmt, emin):
    """The stand-alone codec against the oracle: 129-column values over 7
    decades (the reference test's tensor, ``test_coat_state_muon.py:27-28``,
    with a short last group), then narrow-range groups (spread 1.01 and 1.1 at
    1e-3 and 1e-7).  Expand and sqrt_minmax as the oracle's, codes at most one
    code apart on a small fraction of elements, decoding within 4e-6."""
    rng = np.random.default_rng(13)
    n = 1000 * 129
    wide = (rng.standard_normal(n) * np.logspace(-6, 1, n)).astype(np.float32)
    narrow = np.concatenate([_narrow_groups(256, sp, mag, 14 + k)
                             for k, (sp, mag) in enumerate([(1.01, 1e-3), (1.01, 1e-7), (1.1, 1e-3), (1.1, 1e-7)])])
    dt = {"E4M3": torch.float8_e4m3fn, "E5M2": torch.float8_e5m2}[fmt]
    for label, x, bar in (("wide", wide, 2e-3), ("narrow", narrow, 2e-3)):
        if not signed:
            x = x * x
        v = torch.from_numpy(x).to(DEV)
        G = (x.size + 127) // 128
        codes = torch.empty(x.size, dtype=torch.uint8, device=DEV)
        meta = [torch.empty(G, device=DEV) for _ in range(3)]
        _abi.fp8_quantize(v, codes, *meta, signed=signed, fmt=dt, expand_min=emin)
        q, sc, ex, smm = codec.quantize(x, signed, fmt, emin)
        torch.cuda.synchronize()
        ex_ours = meta[1].cpu().numpy()
        # expand = floor(16 log2(fmax^2/2) / log2(ratio)) / 16: the device log2 is
        # not correctly rounded, so where the quotient lies within an ulp of an
        # integer (a few groups of narrow ranges, where it is ~10^4) the floor
        # may take the neighbour; elsewhere it is exact
        ok = ex_ours == ex
        if label == "wide":
            assert ok.all()
        else:
            assert np.mean(ok) >= 0.99, np.mean(ok)
        np.testing.assert_allclose(meta[2].cpu().numpy(), smm, rtol=2e-7)
        np.testing.assert_allclose(meta[0].cpu().numpy()[ok], sc[ok], rtol=4e-6 if label == "wide" else 2e-4)
        okel = np.repeat(ok, 128)[:x.size]
        ours = codes.cpu().numpy()
        diff = np.abs(ours.astype(int) - q.astype(int))[okel]
        frac = float(np.mean(diff != 0))
        print(f"codec {fmt} emin {emin} {'signed' if signed else 'unsigned'} {label}: code mismatch {frac:.2e}")
        assert frac < bar and diff.max() <= 1, (label, frac, diff.max())    # pow/log2 ulps at code ties
        out = torch.empty(x.size, device=DEV)
        _abi.fp8_dequantize(torch.from_numpy(q).to(DEV), *(torch.from_numpy(t).to(DEV) for t in (sc, ex, smm)),
                            out, signed=signed, fmt=dt)
        np.testing.assert_allclose(out.cpu().numpy(), codec.dequantize(q, sc, ex, smm, signed, fmt), rtol=4e-6, atol=0)


def test_6p89b_layer_newton_schulz_output_against_fp64():
    """The update itself on the headline workload: one 6.89B layer's momentum
    after its update (44 blocks of 1024x1024, 8 of 2752x1024, 4 of 1024x2752),
    packed and orthogonalised by the library without the apply
    (MMUON_NS_NO_APPLY), against fp64 Newton-Schulz of the same bf16 input;
    bar: 1.5x the reference's own bf16 error (+2e-3), on every rectangular
    block and every fourth square block."""
    w, draws = _workload_params("6.89b-nb4", layers=1, adamw_rows=64)
    muon, _, opt, bufs = _build(w, draws, DEV, MonarchMuonOptimizer, ns_dtype=torch.bfloat16)
    params = [p for p in muon]
    grads = [p.grad for p in params]
    mbufs = [opt._get_momentum_buffer(p) for p in params]
    planner = MuonPlanner()
    launches = planner.plan(params, grads, mbufs, torch.bfloat16)
    lib = _abi.lib()
    stream = _abi.stream_handle(DEV)
    coeffs = (C.c_float * 3)(*NS_COEFFS)
    # the oracle's momentum (fp32: mu*buf, then + g, each rounded)
    ref_bufs = [(b.float() * 0.95 + G.to(torch.bfloat16).float()) for b, G in
                zip(bufs, [G for _, m, _, G, _ in draws if m])]
    worst = {}
    for gl in launches:
        _abi.check(lib.mmuon_momentum_pack(C.byref(gl.struct), 0.95, stream), "pack")
        _abi.check(lib.mmuon_newton_schulz_apply(C.byref(gl.struct), 5, coeffs, 0.0, _abi.NS_NO_APPLY, stream),
                   "ns")
        torch.cuda.synchronize()
        lay = gl.ws.layout
        out = _abi.ns_output_buffer(gl.rows, gl.cols, lay.ns_dtype, 5)
        x = gl.ws.x_view(out, torch.bfloat16, gl.nblocks)[:, :lay.m, :lay.n].float().cpu()
        ours = x.transpose(1, 2) if gl.transposed else x
        stack = torch.cat([ref_bufs[i] for i in gl.members]).to(torch.bfloat16)
        sel = list(range(0, gl.nblocks, 4)) if gl.rows == gl.cols else list(range(gl.nblocks))
        truth = ns_fp64(stack[sel].double())
        ref_bf16 = newton_schulz_batched(stack[sel]).float()
        e_ours, e_ref = rel_fro(ours[sel], truth), rel_fro(ref_bf16, truth)
        worst[(gl.rows, gl.cols)] = (float(e_ours.max()), float(e_ref.max()))
        assert torch.all(e_ours <= 1.5 * e_ref + 2e-3), (gl.rows, gl.cols, e_ours.max(), e_ref.max())
    # the momentum the pack wrote back is the oracle's, bit for bit
    for b, r in zip(mbufs, ref_bufs):
        assert torch.equal(b.cpu(), r)
    print("6.89B layer Newton-Schulz (ours, reference bf16) vs fp64:", worst)


# ---------------------------------------------------------------- edge cases and optimizer API
def test_grad_none_skipped_zero_grad_no_update_and_determinism():
    gen = torch.Generator().manual_seed(14)
    mk = lambda s: (torch.randn(s, generator=gen) * 0.02).to(torch.bfloat16).to(DEV).requires_grad_(True)
    a, b, c = mk((2, 256, 256)), mk((1, 512, 256)), mk((3, 256, 256))
    b.grad = torch.zeros_like(b)
    c.grad = (torch.randn(c.shape, generator=gen) * 1e-3).to(torch.bfloat16).to(DEV)
    a0, b0 = a.detach().clone(), b.detach().clone()
    c_init = c.detach().clone()
    opt = MonarchMuonOptimizer([a, b, c], [])
    opt.step()
    torch.cuda.synchronize()
    assert torch.equal(a, a0) and "momentum_buffer" not in opt.state[a]
    assert torch.equal(b, b0)
    c1 = c.detach().clone()
    # the same step again from the same start gives the same bits
    with torch.no_grad():
        c.copy_(c_init)
    opt2 = MonarchMuonOptimizer([c], [])
    opt2.step()
    torch.cuda.synchronize()
    assert torch.equal(c, c1)


def test_state_dict_round_trip_and_param_groups():
    case = CASES[0]
    muon, adamw, opt = _run_case_gpu(case)
    sd = opt.state_dict()
    assert [g["update_type"] for g in sd["param_groups"]] == ["muon", "adamw"]
    assert sd["param_groups"][0]["params"] == list(range(len(muon)))
    assert set(sd["state"][0]) == {"momentum_buffer"}
    assert set(sd["state"][len(muon)]) == {"step", "exp_avg", "exp_avg_sq"}
    buf = io.BytesIO()
    torch.save(sd, buf)
    buf.seek(0)
    muon2, adamw2, _ = make_case(case, device=DEV)
    opt2 = MonarchMuonOptimizer(muon2, adamw2, lr=case["lr"])
    opt2.load_state_dict(torch.load(buf, weights_only=True))
    for k, entry in opt2.state_dict()["state"].items():
        for name, v in entry.items():
            if torch.is_tensor(v):
                ref = sd["state"][k][name]
                # torch.optim casts floating state to the param dtype on load (reference behaviour)
                assert torch.equal(v, ref.to(v.dtype))


def test_fp8_state_dict_round_trip_is_exact():
    case = CASES[0]
    muon, adamw, bufs = make_case(case, device=DEV)
    opt = CoatStateMonarchMuon(muon, adamw, lr=0.02, qargs=QuantizationConfig())
    opt.step()
    opt.step()
    sd = opt.state_dict()
    buf = io.BytesIO()
    torch.save(sd, buf)
    buf.seek(0)
    m2, a2, _ = make_case(case, device=DEV)
    opt2 = CoatStateMonarchMuon(m2, a2, lr=0.02, qargs=QuantizationConfig())
    opt2.load_state_dict(torch.load(buf, weights_only=True))
    for k, entry in opt2.state_dict()["state"].items():
        for name, v in entry.items():
            if torch.is_tensor(v):
                assert v.dtype == sd["state"][k][name].dtype, name
                assert torch.equal(v.view(torch.uint8) if v.dtype == torch.float8_e4m3fn else v,
                                   sd["state"][k][name].view(torch.uint8)
                                   if v.dtype == torch.float8_e4m3fn else sd["state"][k][name])
