"""The one-launch row kernels of a training step (projections and exponents, output projection and feed-forward)
against float64 autograd, at the row counts where their tiles change."""
import math

import pytest
import torch

from crystalformer_amd import hip_funcs, ops
from crystalformer_amd.attention import make_positive_func
from crystalformer_amd.lib import CrystalformerHipError

pytestmark = pytest.mark.gpu

# a tile of 16 rows less one, exactly, plus one; shares of 32 atoms (8 heads) and 64 of them: 2048
ROWS = [1, 15, 16, 17, 33, 1774, 2047, 2048, 2049, 4161]
# a sum of n products of float32 numbers, in any order, is within about sqrt(n) 2^-24 of its terms' 2-norm; here n is
# at most 512 a layer, two layers deep, or the row count for a weight's gradient
TOL = 2e-6


def rel(x, ref):
    x, ref = x.detach().double(), ref.detach()
    return float((x - ref).norm() / ref.norm().clamp_min(1e-30))


def leaves(dev, *shapes, scale=0.1):
    return [(torch.randn(s, device=dev) * scale).requires_grad_() for s in shapes]


def packed_of(wo, w1, w2, wq, wk, wv):
    return ops.PackedBlocks([tuple(w.detach() for w in (wo, w1, w2, wq, wk, wv))] * 2).block(1)


@pytest.mark.parametrize("n", ROWS)
def test_block_tail(dev, n):
    torch.manual_seed(n)
    att, x = leaves(dev, (n, 128), (n, 128), scale=1.0)
    wo, bo, w1, b1, w2, b2 = leaves(dev, (128, 128), (128,), (512, 128), (512,), (128, 512), (128,))
    packed = packed_of(wo, w1, w2, wo, wo, wo)
    g = torch.randn(n, 128, device=dev)
    y = hip_funcs.BlockTailHIP.apply(att, x, wo, bo, w1, b1, w2, b2, packed)
    ins = (att, x, wo, bo, w1, b1, w2, b2)
    got = torch.autograd.grad(y, ins, g)
    d = [t.detach().double().requires_grad_() for t in ins]
    s = d[1] + d[0] @ d[2].T + d[3]
    pre = s @ d[4].T + d[5]
    # (the kernel's own decision at the ReLU: a pre-activation within rounding of zero may fall on either side)
    h = ops.block_tail(att.detach(), x.detach(), packed[0], bo.detach(), b1.detach(), b2.detach())[2]
    ref = s + (pre * (h > 0)) @ d[6].T + d[7]
    assert rel(y, ref.detach()) < TOL
    for name, a, b in zip("att x wo bo w1 b1 w2 b2".split(), got, torch.autograd.grad(ref, d, g.double())):
        assert rel(a, b) < TOL, name


@pytest.mark.parametrize("n", ROWS)
@pytest.mark.parametrize("heads,func,normalize", [(8, "elu=0.1", True), (4, "abs", True), (16, "exp=0.3", False)])
def test_block_head(dev, n, heads, func, normalize):
    torch.manual_seed(n + heads)
    x, = leaves(dev, (n, 128), scale=1.0)
    wq, wk, wv, b_in, w_pos = leaves(dev, (128, 128), (128, 128), (128, 128), (384,), (128,))
    big = torch.zeros(512, 128, device=dev)
    packed = packed_of(wq, big, big.T.contiguous(), wq, wk, wv)
    name, _, beta = func.partition("=")
    beta = float(beta or 1.0)
    lb, coef, q_scale = 0.5, -0.3, 1 / math.sqrt(128 // heads)
    for stored in (False, True) if normalize else (True,):
        if not stored and n * heads < 2:
            continue
        gauss = torch.tensor([0.8, -0.1] if stored else [0.0, 0.0], device=dev)
        packed[2].zero_()
        a, qs, k, v, xc = hip_funcs.BlockHeadHIP.apply(x, wq, wk, wv, b_in, w_pos, gauss, heads, packed, normalize, True,
                                                       name, beta, lb, coef, q_scale)
        gs = [torch.randn_like(t) for t in (a, qs, k, v, xc)]
        ins = (x, wq, wk, wv, b_in, w_pos)
        got = torch.autograd.grad((a, qs, k, v, xc), ins, gs)
        d = [t.detach().double().requires_grad_() for t in ins]
        q64, k64, v64 = (d[0] @ torch.cat(d[1:4]).T + d[4]).split(128, 1)
        alpha = (q64 * d[5]).view(n, heads, -1).sum(2)
        if normalize:
            scale, shift = (0.8, -0.1) if stored else (1 / alpha.detach().std(), -alpha.detach().mean())
            alpha = (alpha + shift) * scale
            if not stored:
                assert rel(gauss, torch.stack([scale, shift])) < 1e-5
        a64 = make_positive_func(func)(alpha, lb) * coef
        outs = (a64, q64 * q_scale, k64, v64, d[0] * 1.0)
        for what, t, r in zip("a qs k v x".split(), (a, qs, k, v, xc), outs):
            # (batch statistics of n * heads values divide by their spread)
            assert rel(t, r.detach()) < (TOL if stored else 1e-5), what
        for what, t, r in zip("x wq wk wv b_in w_pos".split(), got, torch.autograd.grad(outs, d, [g.double() for g in gs])):
            assert rel(t, r) < (TOL if stored else 1e-5), what


def test_absent_gradients(dev):
    """Outputs that nobody used have no gradient; the launch takes zeros for them."""
    x, = leaves(dev, (37, 128), scale=1.0)
    wq, wk, wv, w_pos = leaves(dev, (128, 128), (128, 128), (128, 128), (128,))
    big = torch.zeros(512, 128, device=dev)
    packed = packed_of(wq, big, big.T.contiguous(), wq, wk, wv)
    out = hip_funcs.BlockHeadHIP.apply(x, wq, wk, wv, None, w_pos, torch.tensor([0.8, -0.1], device=dev), 8, packed, True,
                                       False, "elu", 0.1, 0.5, -0.3, 0.25)
    gx, gv = torch.autograd.grad(out[3].sum(), (x, wv))
    assert rel(gx, torch.ones(37, 128, device=dev).double() @ wv.double()) < TOL
    assert rel(gv, torch.ones(37, 128, device=dev).double().T @ x.double()) < TOL


@pytest.mark.parametrize("n", ROWS)
@pytest.mark.parametrize("heads,func,normalize", [(8, "elu", True), (4, "abs", True), (16, "exp", False)])
def test_same_bits_as_the_operators_one_by_one(dev, n, heads, func, normalize):
    """Outputs and gradients are those of the separate launches to the bit (a training step amplifies any
    difference: see block_rows.hip)."""
    torch.manual_seed(n + heads)
    x, = leaves(dev, (n, 128), scale=1.0)
    head = leaves(dev, (128, 128), (128, 128), (128, 128), (384,), (128,))
    tail = leaves(dev, (128, 128), (128,), (512, 128), (512,), (128, 512), (128,))
    wq, wk, wv, b_in, w_pos = head
    wo, bo, w1, b1, w2, b2 = tail
    for stored in (False, True):
        if not stored and n * heads < 2:
            continue
        start = torch.tensor([0.8, -0.1] if stored else [0.0, 0.0], device=dev)
        conf = (func, 0.1, 0.5, -0.3, 1 / math.sqrt(128 // heads))
        g_one, g_two = start.clone(), start.clone()
        q, k, v, carry = hip_funcs.FusedLinearHIP.apply(x, b_in, None, False, True, wq, wk, wv)
        a, qs = hip_funcs.GaussianExponentsHIP.apply(q.view(n, heads, -1), w_pos, g_one, normalize, True, *conf)
        att = (qs.view(n, 128) + k) * v * a.repeat_interleave(128 // heads, 1)
        s, = hip_funcs.FusedLinearHIP.apply(att, bo, carry, False, False, wo)
        y = hip_funcs.FusedFeedForwardHIP.apply(s, w1, b1, w2, b2)
        packed = packed_of(wo, w1, w2, wq, wk, wv)
        a2, qs2, k2, v2, carry2 = hip_funcs.BlockHeadHIP.apply(x, wq, wk, wv, b_in, w_pos, g_two, heads, packed, normalize,
                                                               True, *conf)
        att2 = (qs2 + k2) * v2 * a2.repeat_interleave(128 // heads, 1)
        y2 = hip_funcs.BlockTailHIP.apply(att2, carry2, wo, bo, w1, b1, w2, b2, packed)
        assert torch.equal(g_one, g_two)
        for what, one, two in zip(("a", "qs", "k", "v", "y"), (a, qs.view(n, 128), k, v, y), (a2, qs2, k2, v2, y2)):
            assert torch.equal(one, two), what
        g = torch.randn(n, 128, device=dev)
        names = "x wq wk wv b_in w_pos wo bo w1 b1 w2 b2".split()
        for what, one, two in zip(names, torch.autograd.grad(y, (x, *head, *tail), g),
                                  torch.autograd.grad(y2, (x, *head, *tail), g)):
            assert torch.equal(one, two), what


def test_operands_of_other_shapes_are_refused(dev):
    """Before any launch: the kernels read whole rows, heads and weights by these counts."""
    n = 20
    w = [torch.randn(s, device=dev) for s in ((128, 128), (512, 128), (128, 512)) + ((128, 128),) * 3]
    blocks = ops.PackedBlocks([tuple(w)] * 2)
    fwd, bwd, counter = blocks.block(0)
    x, w_pos, gauss = torch.randn(n, 128, device=dev), torch.randn(128, device=dev), torch.ones(2, device=dev)
    conf = ("elu", 0.1, 0.5, -0.3, 0.25)
    a, qs, k, v, q, alpha_n, used = ops.block_head(x, 8, fwd, counter, None, w_pos, gauss, True, False, *conf)
    y, s, h = ops.block_tail(x, x, fwd, None, None, None)
    refused = pytest.raises(CrystalformerHipError)
    for packed, count in ((blocks.forward, counter), (fwd[:-1], counter), (fwd.double(), counter), (fwd, counter.long()),
                          (fwd, counter.cpu())):
        with refused:
            ops.block_head(x, 8, packed, count, None, w_pos, gauss, True, False, *conf)
    with refused:
        ops.block_tail(x, x, blocks.forward, None, None, None)
    good = dict(ga=a, gqs=qs, gk=k, gv=v, carry=x, q=q, w_pos=w_pos, alpha_n=alpha_n, used=used, packed_bwd=bwd)
    ops.block_head_bwd(*good.values(), *conf)
    for name, wrong in (("ga", a[1:]), ("gqs", qs[1:]), ("gk", k[:, 1:]), ("gv", v[1:]), ("carry", x[:-1]), ("q", q[1:]),
                        ("q", q[:, :64]), ("w_pos", w_pos[1:]), ("alpha_n", alpha_n[1:]), ("used", used[:1]),
                        ("packed_bwd", bwd[:-1])):
        with refused:
            ops.block_head_bwd(*dict(good, **{name: wrong}).values(), *conf)
    for g, hidden, packed in ((y[1:], h, bwd), (y, h[1:], bwd), (y, h[:, 1:], bwd), (y[:, 1:], h, bwd), (y, h, bwd[:-1])):
        with refused:
            ops.block_tail_bwd(g, hidden, packed)


def test_no_atoms(dev):
    x, = leaves(dev, (0, 128))
    wq, wk, wv, b_in, w_pos = leaves(dev, (128, 128), (128, 128), (128, 128), (384,), (128,))
    big = torch.zeros(512, 128, device=dev)
    packed = packed_of(wq, big, big.T.contiguous(), wq, wk, wv)
    full = torch.full((1 << 16,), 7.0, device=dev)         # (what a freed buffer may hold)
    del full
    out = hip_funcs.BlockHeadHIP.apply(x, wq, wk, wv, b_in, w_pos, torch.tensor([0.8, -0.1], device=dev), 8, packed, True,
                                       False, "elu", 0.1, 0.5, -0.3, 0.25)
    for g in torch.autograd.grad([t.sum() for t in out], (wq, wk, wv, b_in, w_pos)):
        assert torch.equal(g, torch.zeros_like(g))
