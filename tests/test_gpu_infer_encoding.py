"""The encoding of an inference forward (``csrc/real_enc_infer.hip``: units staged once, split matrix products) against the
operators' kernels, which have the reference's sums in fp32, and against the oracle in float64: the edges of its groups
(16), chunks (64) and images (832), of its bin and row tiles, and the units its staging leaves to the blocks."""
import contextlib
import dataclasses

import pytest
import torch

from crystalformer_amd import executor, hip_funcs, lib, ops
from crystalformer_amd.graphs import GraphedForward
from crystalformer_amd.latticeformer import default_params
from crystalformer_amd.synthetic import CrystalBatch, lattice_from_parameters
from oracle import torch_model as om
from tests.helpers import RTOL, assert_close, atol_rows
from tests.test_gpu_forward import batch_of, both_ways, scaled

pytestmark = pytest.mark.gpu


def crystals(lengths, sizes, seed=1, angles=None, shift=0):
    """Crystals with cells of these lengths; ``shift`` moves atoms by up to that many whole cells."""
    g = torch.Generator().manual_seed(seed)
    L = torch.tensor(lengths, dtype=torch.float32)
    trans = lattice_from_parameters(L, torch.full_like(L, 90.0) if angles is None else torch.tensor(angles))
    s = torch.tensor(sizes)
    batch = torch.repeat_interleave(torch.arange(len(s)), s)
    frac = torch.rand(len(batch), 3, generator=g)
    if shift:
        frac = frac + torch.randint(-shift, shift + 1, frac.shape, generator=g)
    pos = (frac[:, None, :] @ trans[batch]).squeeze(1).contiguous()
    x = torch.eye(98)[torch.randint(0, 94, (len(batch),), generator=g)]
    return CrystalBatch(x, pos, batch, trans, s)


@contextlib.contextmanager
def blocks_staged():
    """Within it, how many blocks of each native forward were encoded from staged units, and of how many."""
    counts, real = [], lib.load()

    class Asked:
        def __getattr__(self, name):
            return getattr(real, name)

        def cf_forward(self, args, blocks, *rest):
            counts.append((real.cf_forward_staged(args, blocks), len(blocks)))
            return real.cf_forward(args, blocks, *rest)
    with pytest.MonkeyPatch.context() as m:
        m.setattr(executor._lib, "load", Asked)
        yield counts


def served(model, b, staged=True):
    """``both_ways``, whose native call must have taken the staged encoding in every block (or in none)."""
    with blocks_staged() as counts:
        both = both_ways(model, b)
    assert counts and all(got == (of if staged else 0) for got, of in counts), counts
    return both


def compare(dev, b, rtol=RTOL, staged=True, **options):
    model = scaled(default_params(num_layers=2, **options)).to(dev).eval()
    native, modules = served(model, b.to(dev), staged)
    assert_close(native, modules, "encoder", rtol=rtol, atol=atol_rows(modules))


# bin tiles (1, 2, 4 and 8 of 16) less than full, full and one over; head groups of eight; row tiles of 16
@pytest.mark.parametrize("adaptive", [-3.5, 0.0, 2.0])
@pytest.mark.parametrize("bins", [1, 16, 17, 33, 64, 65, 128])
def test_bin_tiles(dev, bins, adaptive):
    compare(dev, batch_of([1, 7, 20]), value_pe_dist_real=bins, adaptive_cutoff_sigma=adaptive)


@pytest.mark.parametrize("adaptive", [-3.5, 0.0])
@pytest.mark.parametrize("width, heads", [(128, 16), (128, 4), (64, 8), (96, 8), (64, 4), (32, 1)])
def test_heads_and_row_tiles(dev, width, heads, adaptive):
    compare(dev, batch_of([3, 0, 18]), model_dim=width, embedding_dim=[width], ff_dim=64, head_num=heads,
            adaptive_cutoff_sigma=adaptive)


# cells from one translation a unit to several hundred: 16, 64 and 128 staged translations lie in between; the smallest ones
# have more than an image holds, and boxes beyond fifteen cells
@pytest.mark.parametrize("options", [dict(), dict(adaptive_cutoff_sigma=0.0)])
@pytest.mark.parametrize("r0", [1.4, 3.0])
@pytest.mark.parametrize("length", [30.0, 9.0, 6.0, 4.5, 3.5, 2.4, (1.1, 9.0, 9.0), (20.0, 4.0, 3.0)])
def test_translations_a_unit(dev, length, r0, options):
    cell = list(length) if isinstance(length, tuple) else [length, 1.1 * length, 0.9 * length]
    compare(dev, crystals([cell, [8.0, 7.0, 9.0]], [6, 9]), scale_real=[r0], **options)


# boxes longest along each axis, whose translations are walked along one of the three; more than 64 staged, and counts on both
# sides of what an image holds
@pytest.mark.parametrize("length", [(20.0, 3.0, 4.0), (3.0, 20.0, 4.0), (4.0, 3.0, 20.0), (2.5, 2.5, 9.0), (9.0, 2.5, 2.5),
                                    (2.5, 9.0, 2.5), (2.7,) * 3, (2.9,) * 3, (3.1,) * 3, (3.3,) * 3])
def test_boxes_along_each_axis(dev, length):
    compare(dev, crystals([list(length)] * 3, [4, 9, 1], angles=[[80.0, 95.0, 110.0]] * 3), scale_real=[3.0])


LEAST_BYTES = 4096 * (32 + 832 * 6)                        # (of a slice in adaptive boxes; the fixed cube's entries are fewer)


@pytest.mark.parametrize("adaptive", [-3.5, 0.0])
@pytest.mark.parametrize("owner", ["STAGED_UNITS_MAX_BYTES", "STAGED_RINGS_MAX_BYTES"])
def test_less_room_than_units_need(dev, monkeypatch, adaptive, owner):
    """As many slices of pairs as the room asks for give the same bits as one; below the least slice's the operators'
    kernels serve."""
    b = crystals([[4.0, 4.0, 5.0], [9.0, 9.0, 9.0], [2.4, 2.5, 2.6], [3.0, 12.0, 7.0]], [92, 90, 91, 34]).to(dev)
    units = int((b.sizes * (b.sizes + 1)).sum()) // 2
    assert units > 3 * 4096 and units % 8
    model = scaled(default_params(num_layers=2, scale_real=[3.0], adaptive_cutoff_sigma=adaptive)).to(dev).eval()
    whole, modules = served(model, b)
    assert_close(whole, modules, "encoder", atol=atol_rows(modules))
    least = LEAST_BYTES if adaptive else 4096 * (32 + 128 * 4)
    for limit in (least, 5 * least // 2, least - 1, 0):
        monkeypatch.setattr(executor if owner == "STAGED_UNITS_MAX_BYTES" else ops, owner, limit)
        sliced, _ = served(model, b, staged=limit >= least)
        if limit >= least:
            assert torch.equal(sliced, whole)
        else:
            assert_close(sliced, modules, "encoder", atol=atol_rows(modules))


@pytest.mark.parametrize("crystals_", [5, 150])
def test_a_capacity_graph_has_the_eager_bits_whatever_its_capacity(dev, monkeypatch, crystals_):
    """Units with more entries than a large capacity's share of the room, in a graph and eagerly; crystals by themselves too."""
    monkeypatch.setattr(executor, "STAGED_UNITS_MAX_BYTES", LEAST_BYTES)
    b = crystals([[4.0, 4.0, 5.0], [3.0, 3.5, 4.0], [2.4, 2.5, 2.6], [3.0, 12.0, 7.0]], [12, 10, 7, 5]).to(dev)
    model = scaled(default_params(num_layers=2, scale_real=[3.0]))
    with torch.no_grad():
        for layer in model.encoder.layers:
            layer.self_attn.gauss_scale.copy_(torch.tensor([0.8, -0.1]))
    model = model.to(dev).eval()
    graph = GraphedForward(model, b, capacity=(crystals_, 12 * crystals_, 144 * crystals_))
    with torch.no_grad(), blocks_staged() as counts:
        eager = model(b).clone()
        assert counts == [(2, 2)]
        for _ in range(3):
            assert torch.equal(graph(b), eager)
        n = int(b.sizes[0])
        alone = model(CrystalBatch(b.x[:n], b.pos[:n], b.batch[:n], b.trans_vec[:1], b.sizes[:1]))
    assert torch.equal(alone, eager[:1])


@pytest.mark.parametrize("adaptive", [-3.5, 0.0])
def test_atoms_outside_their_cells(dev, adaptive):
    """The nearest image outside the cube: columns with references of their own.  (1e-4: differences of squared distances
    of some thousand, as in the operators' own test of this.)"""
    compare(dev, crystals([[5.0, 6.0, 7.0], [3.0, 12.0, 4.0]], [9, 8], shift=4), rtol=1e-4, adaptive_cutoff_sigma=adaptive,
            scale_real=[2.0])


@pytest.mark.parametrize("floor", [True, False])
def test_skewed_cells_with_and_without_a_floor(dev, floor, monkeypatch):
    b = crystals([[25.0, 5.0, 6.0], [4.0, 7.0, 5.0]], [30, 11], angles=[[60.0, 110.0, 70.0], [120.0, 55.0, 90.0]])
    model = scaled(default_params(num_layers=2, scale_real=[2.0])).to(dev).eval()
    if not floor:
        monkeypatch.setattr(hip_funcs.KernelManager, "MINIMUM_RANGE", 0)
    native, modules = served(model, b.to(dev))
    assert_close(native, modules, "encoder", atol=atol_rows(modules))


@pytest.mark.parametrize("bound", [0.0, 0.05, 0.099, 0.1, 0.25, 0.9])
@pytest.mark.parametrize("adaptive", [-3.5, 0.0])
def test_bounds_of_the_exponents(dev, bound, adaptive):
    # (staged in the box of the weakest exponent, which only a bound holds down)
    compare(dev, batch_of([5, 14]), staged=adaptive == 0.0 or bound >= 0.1, gauss_lb_real=bound, positive_func="abs",
            adaptive_cutoff_sigma=adaptive)


def test_blocks_that_share_units_and_blocks_that_do_not(dev):
    compare(dev, batch_of([12, 3, 25]), scale_real=[1.4, 3.0])
    model = scaled(default_params(num_layers=34, t_fixup_init=True)).to(dev).eval()    # (more blocks than are packed at once)
    native, modules = served(model, batch_of([9, 5]).to(dev))
    assert_close(native, modules, "encoder of 34 blocks", rtol=34 * RTOL)


@pytest.mark.parametrize("r0", [1.4, 3.0])
def test_no_further_from_float64_than_the_operators(dev, r0):
    """Root mean square of the distance to the oracle in float64, one block: no larger than that of the kernels whose
    products are fp32, within a tenth (an estimate from 10^4 values has a spread of one in a hundred)."""
    cfg = default_params(num_layers=1, adaptive_cutoff_sigma=0.0, scale_real=[r0])
    model = scaled(cfg)
    b = batch_of([40, 17, 25, 8])
    P = {k: v.detach().double() for k, v in model.state_dict().items()}
    b64 = dataclasses.replace(b, x=b.x.double(), pos=b.pos.double(), trans_vec=b.trans_vec.double())
    with torch.no_grad():
        x = torch.nn.functional.linear(b64.x, P["input_embeddings.weight"])
        want = om.encoder_forward(P, cfg, x, b64.pos, b64.batch, b64.trans_vec, b64.sizes)
    want = want[0] if isinstance(want, tuple) else want
    native, modules = served(model.to(dev).eval(), b.to(dev))
    err = [float((t.cpu().double() - want).square().mean().sqrt()) for t in (native, modules)]
    print("\nrms from float64: staged %.3e, operators %.3e" % tuple(err), flush=True)
    assert err[0] <= 1.1 * err[1], err


def distances_from_float64(dev, cfg, change, b):
    """Root mean squares of the distance to the oracle in float64: (native call, operators), one block after ``change``."""
    model = scaled(cfg)
    with torch.no_grad():
        change(model)
    P = {k: v.detach().double() for k, v in model.state_dict().items()}
    with torch.no_grad():
        x = torch.nn.functional.linear(b.x.double(), P["input_embeddings.weight"])
        want = om.encoder_forward(P, cfg, x, b.pos.double(), b.batch, b.trans_vec.double(), b.sizes)
    want = want[0] if isinstance(want, tuple) else want
    return [float((t.cpu().double() - want).square().mean().sqrt()) for t in served(model.to(dev).eval(), b.to(dev))]


# Bins whose weights are up to 2^24 apart: within a tenth of the fp32 products' own distance.
@pytest.mark.parametrize("bins", [16, 64])
def test_projections_of_any_magnitude(dev, bins):
    def change(model):
        g = torch.Generator().manual_seed(12)
        model.encoder.layers[0].self_attn.pe_dist_proj.mul_(torch.exp2(torch.randint(-24, 1, (bins,), generator=g).float()))
    cfg = default_params(num_layers=1, adaptive_cutoff_sigma=0.0, value_pe_dist_real=bins)
    err = distances_from_float64(dev, cfg, change, batch_of([40, 17, 25, 8]))
    assert err[0] <= 1.1 * err[1], err


def test_infinite_projection_weights(dev):
    model = scaled(default_params(num_layers=1)).to(dev).eval()
    with torch.no_grad():
        model.encoder.layers[0].self_attn.pe_dist_proj[0, 3, 5, 20] = float("inf")
        model.encoder.layers[0].self_attn.out_proj.weight[:, 3 * 16 + 5] = 0.0
        model.encoder.layers[0].self_attn.out_proj.weight[7, 3 * 16 + 5] = 1.0
    native, modules = served(model, batch_of([1, 7, 20]).to(dev))
    for same in (torch.isposinf, torch.isneginf, torch.isnan):
        assert torch.equal(same(native), same(modules))
