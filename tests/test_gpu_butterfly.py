"""HIP butterfly forward/backward (mmuon_butterfly_fwd / _bwd through the C ABI) against the
oracle (oracle/butterfly.py, pinned by tests/test_oracle_butterfly.py).

Inputs are bf16, the oracle multiplies the same bf16 values in fp32 and rounds each product to
bf16 where the reference's bmms round.  Only the summation order differs, so an output element
differs by at most a bf16 rounding step where the fp32 sums straddle one.  Bar: relative Frobenius
error <= 2e-3 per output, five times tighter than the bf16 tolerance of the optimizer path (1e-2);
the measured errors are printed and sit between 2e-5 and 2e-4.  Shapes: the Monarch factors of
the benchmark models (toy nb=2, 257M nb=2, 1.3B nb=4, 6.89B nb=4: square, tall-w2 and wide-w1
layers), token counts that are not multiples of the 256-row tile, split-K weight gradients with a
ragged last split, and the empty and single-token edge cases.
"""
import pytest
import torch

from monarch_muon_amd import butterfly_blk, butterfly_blk_bwd_op, butterfly_blk_op
from oracle import butterfly as bf
from oracle.truth import rel_fro

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
TOL = 2e-3

# (tokens, nblocks, q, p, s): w1 (nb, q, p), w2 (nb, s, q), x (tokens, nb p)
CASES = [
    (1000, 2, 256, 256, 688),     # toy gate/up (in 512 -> out 1376)
    (1000, 2, 256, 688, 256),     # toy down
    (700, 2, 512, 512, 1368),     # 257M up
    (700, 2, 512, 1368, 512),     # 257M down
    (600, 4, 512, 512, 1376),     # 1.3B up
    (512, 4, 1024, 1024, 1024),   # 6.89B q/k/v/o
    (300, 4, 1024, 1024, 2752),   # 6.89B gate/up
    (300, 4, 1024, 2752, 1024),   # 6.89B down
    (5000, 4, 256, 256, 256),     # split-K weight gradients, ragged last split
    (1, 4, 256, 256, 256),
    (300, 1, 256, 512, 384),      # one block: the riffle is the identity
    (200, 8, 256, 256, 264),      # eight blocks: 32-column planes, s not a multiple of 16
    (200, 16, 512, 256, 520),     # sixteen blocks (the most the kernels take): 16-column planes
]


def make(tokens, nb, q, p, s, seed=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(tokens, nb * p, generator=g).bfloat16()
    w1 = (torch.randn(nb, q, p, generator=g) / p ** 0.5).bfloat16()
    w2 = (torch.randn(nb, s, q, generator=g) / q ** 0.5).bfloat16()
    dout = torch.randn(tokens, nb, s, generator=g).bfloat16()
    return x, w1, w2, dout


def gpu(*ts):
    return [t.to(DEV) for t in ts]


def rel(a, b):
    return float(rel_fro(a.detach().cpu().double().reshape(1, 1, -1), b.detach().cpu().double().reshape(1, 1, -1)).max())


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_forward_and_backward_match_oracle(case):
    print("butterfly case", case, flush=True)
    x, w1, w2, dout = make(*case)
    ref_out, ref_out1 = bf.butterfly_fwd(x, w1, w2)
    ref_dx, ref_dw1, ref_dw2 = bf.butterfly_bwd(x, w1, w2, ref_out1, dout)
    xg, w1g, w2g, dg = gpu(x, w1, w2, dout)
    out, out1 = butterfly_blk_op(xg, w1g, w2g)
    # the backward from the oracle's intermediate, so each op is checked on its own inputs
    dx, dw1, dw2 = butterfly_blk_bwd_op(xg, w1g, w2g, ref_out1.to(DEV), dg)
    torch.cuda.synchronize()
    errs = {"out1": rel(out1, ref_out1), "out": rel(out, ref_out), "dx": rel(dx, ref_dx),
            "dw1": rel(dw1, ref_dw1), "dw2": rel(dw2, ref_dw2)}
    print(case, {k: f"{v:.2e}" for k, v in errs.items()})
    assert out.shape == ref_out.shape and out1.shape == ref_out1.shape
    for k, v in errs.items():
        assert v <= TOL, (k, v)


# one case for each tile size (64-, 128- and 256-wide) beside those above, an unsplit and a split weight gradient at
# each, row counts one past and one short of a tile, and rows that are no multiple of the interleaving pass's stride
LINEAR_CASES = CASES + [(1, 4, 1024, 1024, 2752), (65, 2, 64, 136, 72), (127, 2, 192, 192, 200), (4096, 4, 512, 512, 512),
                        (2049, 2, 512, 1368, 520), (8191, 4, 256, 256, 264), (3001, 4, 1024, 1024, 1024),
                        (0, 2, 256, 256, 256)]


@pytest.mark.parametrize("case", LINEAR_CASES, ids=lambda c: "x".join(map(str, c)))
def test_layer_form_equals_the_blocked_pair(case):
    """butterfly_blk (feature-order output and gradient) against the blocked op pair, bit for bit: the same products
    with the same summation order, their results stored elsewhere.  The pair against the oracle's products in fp32."""
    print("butterfly case", case, flush=True)
    tokens, nb, q, p, s = case
    x, w1, w2, dout = gpu(*make(*case, seed=3))
    out, out1 = butterfly_blk_op(x, w1, w2)
    grads = butterfly_blk_bwd_op(x, w1, w2, out1, dout)
    xg, w1g, w2g = (t.clone().requires_grad_() for t in (x, w1, w2))
    y = butterfly_blk(xg, w1g, w2g)
    dy = dout.transpose(1, 2).reshape(tokens, s * nb)
    got = torch.autograd.grad(y, (xg, w1g, w2g), dy)
    torch.cuda.synchronize()
    assert torch.equal(y, out.transpose(1, 2).reshape(tokens, s * nb))
    for u, v in zip(got, grads):
        assert torch.equal(u, v)
    if tokens:
        ref_out, ref_out1 = bf.butterfly_fwd(x, w1, w2)
        ref = (ref_out, ref_out1) + bf.butterfly_bwd(x, w1, w2, out1, dout)
        for u, v in zip((out, out1) + tuple(grads), ref):
            assert rel(u, v) <= TOL


@pytest.mark.parametrize("tokens", [1, 16, 17, 32, 33, 64, 65])
@pytest.mark.parametrize("dims", [(2, 64, 136, 72), (4, 256, 344, 1096), (1, 1024, 1024, 520), (16, 512, 264, 56)],
                         ids=lambda c: "x".join(map(str, c)))
def test_forward_for_few_tokens(tokens, dims):
    """The few-token kernel at the edges of its token tiles, with fewer and more K steps than its waves' rings hold,
    features and K that end inside a tile, and inputs that fill no tile: rows beyond the tokens must not be read into
    the result (the poison behind them is NaN).  fp32 products of bf16 inputs, rounded once: each result within half
    a bf16 step of the exact sum, a step at a rounding boundary (2^-8 of it), and fp32 summation noise."""
    print("few tokens", tokens, dims, flush=True)
    nb, q, p, s = dims
    x, w1, w2, _ = make(tokens, nb, q, p, s, seed=tokens)
    hold = torch.full((80, nb * p), float("nan"), dtype=torch.bfloat16, device=DEV)
    hold[:tokens] = x.to(DEV)
    w1g, w2g = gpu(w1, w2)
    out, out1 = butterfly_blk_op(hold[:tokens], w1g, w2g)
    y = butterfly_blk(hold[:tokens], w1g, w2g)
    torch.cuda.synchronize()
    mid = torch.einsum("bkp,kqp->bkq", x.double().view(tokens, nb, p), w1.double())  # out1[b][kk][jq]
    t = mid.reshape(tokens, q, nb).permute(2, 0, 1)                                  # the riffle: t[ll][b][i]
    got1 = out1.cpu().double()
    assert torch.all((got1.reshape(t.shape) - t).abs() <= t.abs() * 2.0 ** -8 + p * 2.0 ** -22)
    ref = torch.einsum("lbi,lsi->bls", got1.reshape(t.shape), w2.double())
    assert torch.all((out.cpu().double().reshape(ref.shape) - ref).abs() <= ref.abs() * 2.0 ** -8 + q * 2.0 ** -22)
    assert torch.equal(y, out.transpose(1, 2).reshape(tokens, s * nb))


# token counts on both sides of every switch of kernel and tile width: 16 / 32 / 64 tokens per workgroup, 64-, 128- and
# 256-wide tiles (the largest count takes the 256-wide ones); K in whole slices and ending inside one
@pytest.mark.parametrize("dims", [(4, 512, 512, 512), (2, 512, 1096, 264), (1, 1024, 2744, 520), (16, 512, 264, 56)],
                         ids=lambda c: "x".join(map(str, c)))
def test_rows_do_not_depend_on_the_token_count(dims):
    """A row of the forward and of dx is the same, bit for bit, whatever number of tokens shares its call."""
    print("rows", dims, flush=True)
    nb, q, p, s = dims
    x, w1, w2, dout = gpu(*make(16384, nb, q, p, s, seed=11))
    out, out1 = butterfly_blk_op(x, w1, w2)
    y = butterfly_blk(x, w1, w2)
    dx = butterfly_blk_bwd_op(x, w1, w2, out1, dout)[0]
    for n in (1, 8, 16, 17, 32, 33, 64, 65, 128, 300, 1000, 2000, 4096):
        print("  tokens", n, flush=True)
        o, o1 = butterfly_blk_op(x[:n], w1, w2)
        assert torch.equal(o1, out1[:, :n]) and torch.equal(o, out[:n]), n
        assert torch.equal(butterfly_blk(x[:n], w1, w2), y[:n]), n
        assert torch.equal(butterfly_blk_bwd_op(x[:n], w1, w2, o1, dout[:n])[0], dx[:n]), n


@pytest.mark.parametrize("dims", [(16, 2048, 264, 136), (16, 1024, 520, 1032), (4, 4096, 72, 4104)],
                         ids=lambda c: "x".join(map(str, c)))
def test_few_tokens_of_many_features(dims):
    """Where the few-token kernel gives way to the tiles by the number of features, one product or both, on both sides
    of each token count: the rows of a call of 300 tokens, which are within the pair's bar."""
    print("many features", dims, flush=True)
    x, w1, w2, _ = gpu(*make(300, *dims, seed=13))
    out, out1 = butterfly_blk_op(x, w1, w2)
    y = butterfly_blk(x, w1, w2)
    ref_out, ref_out1 = bf.butterfly_fwd(x, w1, w2)
    assert rel(out, ref_out) <= TOL and rel(out1, ref_out1) <= TOL
    for n in (1, 16, 17, 32, 33, 48, 49, 64, 65):
        o, o1 = butterfly_blk_op(x[:n], w1, w2)
        assert torch.equal(o1, out1[:, :n]) and torch.equal(o, out[:n]), n
        assert torch.equal(butterfly_blk(x[:n], w1, w2), y[:n]), n


@pytest.mark.parametrize("how", ["compile", "saved_hooks", "expanded_grad", "second_order"])
def test_layer_operator_under_torch(how):
    """The native operator traced by torch.compile, with saved-tensor hooks and with a gradient that is no dense
    tensor, against the plain call; a second derivative is refused."""
    x, w1, w2, _ = gpu(*make(96, 2, 64, 64, 72, seed=4))
    a, b = ([t.clone().requires_grad_() for t in (x, w1, w2)] for _ in range(2))
    y = butterfly_blk(*a)
    if how == "second_order":
        (g, *_) = torch.autograd.grad(y.float().pow(2).sum(), a, create_graph=True)
        with pytest.raises(RuntimeError, match="no autograd formula"):
            torch.autograd.grad(g.float().sum(), a)
        return
    want = torch.autograd.grad(y, a, torch.ones_like(y))
    if how == "compile":
        z = torch.compile(lambda *t: butterfly_blk(*t), backend="aot_eager", fullgraph=True)(*b)
    elif how == "saved_hooks":
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(DEV)):
            z = butterfly_blk(*b)
    else:
        z = butterfly_blk(*b)
    got = torch.autograd.grad(z.sum(), b)   # an expanded gradient
    assert torch.equal(y, z) and all(torch.equal(u, v) for u, v in zip(got, want))


@pytest.mark.parametrize("start", [1, 3, 7])
def test_gradient_that_starts_anywhere(start):
    """A gradient that is a contiguous view ``start`` elements into its storage, as torch.cat's backward hands out."""
    x, w1, w2, _ = gpu(*make(96, 2, 64, 64, 72, seed=4))
    a, b = ([t.clone().requires_grad_() for t in (x, w1, w2)] for _ in range(2))
    y = butterfly_blk(*a)
    dy = torch.randn(y.shape, generator=torch.Generator().manual_seed(1)).to(DEV, torch.bfloat16)
    want = torch.autograd.grad(y, a, dy)
    head = torch.zeros(start, dtype=torch.bfloat16, device=DEV)
    z = torch.cat([head, butterfly_blk(*b).flatten()])
    got = torch.autograd.grad(z, b, torch.cat([head, dy.flatten()]))
    assert all(torch.equal(u, v) for u, v in zip(got, want))


def test_gradient_through_the_intermediate_alone_is_zero():
    """out1 carries no gradient of its own; asking for one through it alone gives zeros."""
    x, w1, w2, _ = gpu(*make(64, 2, 64, 64, 64))
    x.requires_grad_()
    (g,) = torch.autograd.grad(butterfly_blk_op(x, w1, w2)[1].sum(), (x,))
    assert not g.any()


def test_zero_tokens():
    x, w1, w2, dout = make(0, 4, 256, 256, 256)
    xg, w1g, w2g, dg = gpu(x, w1, w2, dout)
    out, out1 = butterfly_blk_op(xg, w1g, w2g)
    dx, dw1, dw2 = butterfly_blk_bwd_op(xg, w1g, w2g, out1, dg)
    torch.cuda.synchronize()
    assert out.shape == (0, 4, 256) and out1.shape == (4, 0, 256) and dx.shape == (0, 1024)
    assert not dw1.abs().any() and not dw2.abs().any()


def test_results_are_deterministic():
    x, w1, w2, dout = gpu(*make(2600, 4, 256, 512, 256, seed=7))
    a = butterfly_blk_op(x, w1, w2)
    b = butterfly_blk_op(x, w1, w2)
    ga = butterfly_blk_bwd_op(x, w1, w2, a[1], dout)
    gb = butterfly_blk_bwd_op(x, w1, w2, b[1], dout)
    torch.cuda.synchronize()
    for u, v in zip(a + ga, b + gb):
        assert torch.equal(u, v)


def test_autograd_through_butterfly_blk_under_autocast():
    """fp32 parameters under bf16 autocast, as the reference trains: butterfly_blk casts, the
    custom op's backward runs, the gradients land in fp32 on the parameters."""
    tokens, nb, q, p, s = 384, 4, 512, 512, 1376
    x, w1, w2, _ = make(tokens, nb, q, p, s, seed=11)
    dy = torch.randn(tokens, s * nb, generator=torch.Generator().manual_seed(12)).bfloat16()
    xg = x.float().to(DEV).requires_grad_()
    w1g = w1.float().to(DEV).requires_grad_()
    w2g = w2.float().to(DEV).requires_grad_()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = butterfly_blk(xg.reshape(3, 128, nb * p), w1g, w2g)
    assert y.shape == (3, 128, s * nb) and y.dtype == torch.bfloat16
    y.backward(dy.reshape(3, 128, -1).to(DEV))
    torch.cuda.synchronize()
    ref_y = bf.butterfly_blk(x, w1, w2)
    _, ref_out1 = bf.butterfly_fwd(x, w1, w2)
    ref_dx, ref_dw1, ref_dw2 = bf.butterfly_bwd(x, w1, w2, ref_out1, bf.blocked_grad(dy, nb))
    assert w1g.grad.dtype == torch.float32
    assert rel(y.reshape(tokens, -1), ref_y) <= TOL
    assert rel(xg.grad, ref_dx) <= TOL
    assert rel(w1g.grad, ref_dw1) <= TOL
    assert rel(w2g.grad, ref_dw2) <= TOL


def test_full_size_layer_against_fp32_products():
    """6.89B gate/up layer at the benchmark's 4096 tokens: the oracle's products run on the GPU in
    fp32 (same rounding points) as the checker at this size."""
    x, w1, w2, dout = gpu(*make(4096, 4, 1024, 1024, 2752, seed=5))
    out, out1 = butterfly_blk_op(x, w1, w2)
    dx, dw1, dw2 = butterfly_blk_bwd_op(x, w1, w2, out1, dout)
    ref_out, ref_out1 = bf.butterfly_fwd(x, w1, w2)
    ref = bf.butterfly_bwd(x, w1, w2, ref_out1, dout)
    torch.cuda.synchronize()
    assert rel(out1, ref_out1) <= TOL and rel(out, ref_out) <= TOL
    for u, v in zip((dx, dw1, dw2), ref):
        assert rel(u, v) <= TOL


def test_rejects_what_the_kernels_do_not_cover():
    x, w1, w2, _ = gpu(*make(16, 4, 256, 256, 256))
    with pytest.raises(TypeError, match="bfloat16"):
        butterfly_blk_op(x.float(), w1.float(), w2.float())
    xb, w1b, w2b, _ = gpu(*make(16, 4, 64, 64, 64))   # q / nblocks = 16, not a multiple of 32
    with pytest.raises(RuntimeError, match="multiple of 32"):
        butterfly_blk_op(xb, w1b, w2b)
