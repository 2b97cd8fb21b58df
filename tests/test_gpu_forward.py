"""The native inference forward (``executor``) against the same model run module by module, and
against the CPU oracle: the sizes at which its kernels can go wrong (one atom, row tiles and their
remainders, empty crystals), the options it serves and those it leaves to the modules."""
import pytest
import torch

from crystalformer_amd import executor, hip_funcs
from crystalformer_amd.graphs import GraphedForward
from crystalformer_amd.latticeformer import Latticeformer, default_params
from crystalformer_amd.synthetic import CrystalBatch, make_batch
from oracle import torch_model as om
from tests.helpers import RTOL, assert_close, atol_rows

pytestmark = pytest.mark.gpu


def batch_of(sizes, seed=3):
    """Crystals of exactly these sizes (zeros allowed)."""
    full = make_batch(len(sizes), (max(sizes), max(sizes)), False, (3.0, 11.0), (65.0, 115.0), seed=seed)
    keep = torch.cat([torch.arange(max(sizes)) < n for n in sizes])
    s = torch.tensor(sizes)
    return CrystalBatch(full.x[keep], full.pos[keep].contiguous(), torch.repeat_interleave(torch.arange(len(s)), s),
                        full.trans_vec, s)


def both_ways(model, b):
    """(native, module by module) outputs of the encoder: a forward hook sends it through the modules."""
    x = torch.nn.functional.linear(b.x, model.input_embeddings.weight)
    args = (x, b.pos, b.batch, b.trans_vec, b.sizes)
    with torch.no_grad():
        native = executor.encode(model.encoder, *args)
        assert native is not None
        handle = model.encoder.layers[0].linear1.register_forward_hook(lambda m, i, o: None)
        try:
            assert executor.encode(model.encoder, *args) is None
            return native, model.encoder(*args)
        finally:
            handle.remove()


def scaled(cfg, seed=5):
    torch.manual_seed(seed)
    model = Latticeformer(cfg)
    with torch.no_grad():
        model.input_embeddings.weight.normal_()            # (the initialisation's features are near zero)
        for layer in model.encoder.layers:
            for p in (layer.self_attn.in_proj_bias, layer.self_attn.out_proj.bias, layer.linear1.bias,
                      layer.linear2.bias):
                p.normal_(0.0, 0.3)
    return model


# sizes: one atom; a tile of rows less one, exactly, plus one; more than one tile; empty crystals
@pytest.mark.parametrize("sizes", [[1], [15], [16], [17], [1, 2, 30], [5, 0, 0, 64, 3], [200]])
@pytest.mark.parametrize("options", [dict(), dict(adaptive_cutoff_sigma=0.0), dict(value_pe_dist_real=0),
                                     dict(value_pe_dist_real=24, head_num=4, positive_func="abs"),
                                     dict(model_dim=64, embedding_dim=[64], ff_dim=96, normalize_gauss=False),
                                     dict(domain="multihead"), dict(domain="multihead-real", head_num=4),
                                     dict(domain="multihead", value_pe_dist_real=0, adaptive_cutoff_sigma=0.0)])
def test_native_forward_equals_the_modules(dev, sizes, options):
    model = scaled(default_params(num_layers=2, **options)).to(dev).eval()
    b = batch_of(sizes).to(dev)
    native, modules = both_ways(model, b)
    # every output element is a chain of sums over up to 512 products of its row
    assert_close(native, modules, "encoder", rtol=RTOL, atol=atol_rows(modules))
    with torch.no_grad():
        for layer in model.encoder.layers:                 # stored statistics instead of the batch's
            layer.self_attn.gauss_scale.copy_(torch.tensor([0.7, -0.2]))
    native, modules = both_ways(model, b)
    assert_close(native, modules, "encoder, stored statistics", rtol=RTOL, atol=atol_rows(modules))


@pytest.mark.parametrize("r0", [1.4, 3.0])               # nearly all pairs keep the cube; most leave it
def test_adaptive_boxes_either_side_of_the_staged_rings(dev, r0):
    """Below three rounds of the chip the blocks stage for themselves, above they share staged rings: both are the
    module path's results, which always uses the rings."""
    per_round = 16 * torch.cuda.get_device_properties(0).multi_processor_count
    for units in (3 * per_round - 10, 3 * per_round, 3 * per_round + 1, 3 * per_round + 127, 5 * per_round):
        crystals, rest = divmod(units, 16 * 17 // 2)
        b = batch_of([16] * crystals + [1] * rest).to(dev)
        model = scaled(default_params(num_layers=2, scale_real=[r0])).to(dev).eval()
        native, modules = both_ways(model, b)
        assert_close(native, modules, str(units), rtol=RTOL, atol=atol_rows(modules))


@pytest.mark.parametrize("options", [dict(), dict(targets=["a", "b", "c"]), dict(embedding_dim=[128, 64]),
                                     dict(pre_pooling_op="w+relu", embedding_dim=[128, 128])])
def test_native_forward_with_its_head(dev, options):
    """Whole model, one or several targets and heads the native call does not take, against the oracle."""
    cfg = default_params(num_layers=2, adaptive_cutoff_sigma=0.0, **options)
    model = scaled(cfg)
    b = batch_of([3, 1, 40, 17])
    with torch.no_grad():
        if "pre_pooling_op" in options or len(cfg.embedding_dim) > 1:
            got = model.to(dev).eval()(b.to(dev))
            model.encoder.register_forward_hook(lambda m, i, o: None)
            want = model(b.to(dev)).cpu()
        else:
            want = om.latticeformer_forward({k: v.detach() for k, v in model.state_dict().items()}, cfg, b,
                                            training=False)
            got = model.to(dev).eval()(b.to(dev))
    assert_close(got, want, "model", rtol=RTOL)


# rows: one work-group's tile of 4, 8 and 16 rows less one, exactly, plus one; either side of the row counts at
# which the tile grows (four and eight rows per CU, one full round of sixteen)
ROW_TILES = [1, 3, 4, 5, 1023, 1025, 2047, 2049, 3480, 3490, 4097]


@pytest.mark.parametrize("atoms", ROW_TILES)
def test_row_kernel_tiles_and_head(dev, atoms):
    """Embedding, tail and head of the 128-wide blocks on crystals of up to 16 atoms against the module path, pooling and
    the regression head on the encoder's output against float64."""
    torch.manual_seed(atoms)
    sizes = [16] * (atoms // 16) + ([atoms % 16] if atoms % 16 else [])
    model = scaled(default_params(num_layers=2, value_pe_dist_real=0)).to(dev).eval()
    b = batch_of(sizes).to(dev)
    native, modules = both_ways(model, b)
    assert_close(native, modules, "encoder", rtol=RTOL, atol=atol_rows(modules))
    with torch.no_grad():
        y = model(b)
        last = {}
        hooks = [m.register_forward_hook(lambda m, i, o, k=k: last.__setitem__(k, o)) for k, m in
                 (("encoder", model.encoder), ("pool", model.mlp))]
        want = model(b)
        for h in hooks:
            h.remove()
        pooled = torch.stack([e.double().mean(0) for e in last["encoder"].split(sizes)])
        ref = pooled
        for m in model.mlp:
            ref = torch.nn.functional.linear(ref, m.weight.double(), m.bias.double()) if hasattr(m, "weight") else m(ref)
    assert_close(y, want, "model", rtol=RTOL)
    assert_close(y, ref.float(), "head", rtol=RTOL)


@pytest.mark.parametrize("atoms", ROW_TILES)
def test_row_kernel_tiles_against_float64(dev, atoms):
    """Embedding, tail and head of the 128-wide blocks on crystals of up to 8 atoms: the encoder alone and the whole
    model against the oracle in float64, under the batch's statistics (every exponent is in them) and stored ones."""
    torch.manual_seed(atoms)
    sizes = [8] * (atoms // 8) + ([atoms % 8] if atoms % 8 else [])
    cfg = default_params(num_layers=2, value_pe_dist_real=0, adaptive_cutoff_sigma=0.0)
    model = scaled(cfg).eval()
    b = batch_of(sizes)
    b64 = CrystalBatch(b.x.double(), b.pos.double(), b.batch, b.trans_vec.double(), b.sizes)
    x = torch.nn.functional.linear(b.x, model.input_embeddings.weight.detach())
    on_gpu = b.to(dev)
    for stored in (False, True):
        if stored:
            for layer in model.encoder.layers:
                layer.self_attn.gauss_scale.data.copy_(torch.tensor([0.7, -0.2]))
        P = {k: v.detach().cpu().double() for k, v in model.state_dict().items()}
        want_y = om.latticeformer_forward(P, cfg, b64)
        want = om.encoder_forward(P, cfg, x.double(), b64.pos, b.batch, b64.trans_vec, b.sizes)
        model.to(dev)
        with torch.no_grad():
            got = executor.encode(model.encoder, x.to(dev), on_gpu.pos, on_gpu.batch, on_gpu.trans_vec, on_gpu.sizes)
            y = executor.forward(model, on_gpu)[0]
        assert_close(got, want, "encoder", rtol=RTOL, atol=atol_rows(want))
        assert_close(y, want_y, "model", rtol=RTOL)


@pytest.mark.parametrize("domain", ["real", "multihead"])
@pytest.mark.parametrize("atoms", [2040, 2048, 2049, 2100, 5000])   # 64 groups of 256 exponents are kept in registers
def test_batch_statistics_of_many_atoms(dev, atoms, domain):
    """Exponents under the batch's own statistics, finished by one work-group or by a launch of their own."""
    sizes = [8] * (atoms // 8) + ([atoms % 8] if atoms % 8 else [])
    model = scaled(default_params(num_layers=3, value_pe_dist_real=0, domain=domain, adaptive_cutoff_sigma=0.0))
    model = model.to(dev).eval()
    b = batch_of(sizes).to(dev)
    native, modules = both_ways(model, b)
    assert_close(native, modules, "encoder", rtol=RTOL, atol=atol_rows(modules))


# tiles of 4, 8 and 16 rows against groups of 256 values; the last group short; capacities below and above the one from
# which the map is a launch of its own
@pytest.mark.parametrize("heads,domain", [(4, "real"), (8, "real"), (16, "real"), (8, "multihead")])
@pytest.mark.parametrize("atoms", [4095, 4096, 4098, 5601, 9001])
def test_spread_statistics(dev, atoms, heads, domain):
    """Statistics of groups formed by whichever work-group completes them: the module path's results, the same bits for
    every pass over the same batch, and from a capacity graph those of the eager call."""
    sizes = [8] * (atoms // 8) + ([atoms % 8] if atoms % 8 else [])
    model = scaled(default_params(num_layers=3, value_pe_dist_real=0, domain=domain, head_num=heads,
                                  adaptive_cutoff_sigma=0.0)).to(dev).eval()
    b = batch_of(sizes).to(dev)
    native, modules = both_ways(model, b)
    assert_close(native, modules, "encoder", rtol=RTOL, atol=atol_rows(modules))
    again, _ = both_ways(model, b)
    assert torch.equal(native, again)
    if domain == "real":
        with torch.no_grad():
            eager = model(b)
        for capacity in (atoms + 8, 33000):
            graph = GraphedForward(model, b, capacity=(len(sizes) + 4, capacity, 8 * capacity))
            for _ in range(3):
                assert torch.equal(graph(b), eager)
    stored = []
    for native_call in (True, False):
        m = scaled(default_params(num_layers=1, value_pe_dist_real=0, domain=domain, head_num=heads,
                                  adaptive_cutoff_sigma=0.0)).to(dev).train()
        if not native_call:
            m.encoder.layers[0].register_forward_hook(lambda *args: None)
        with torch.no_grad():
            m(b)
        stored.append(m.encoder.layers[0].self_attn.gauss_scale.clone())
    # (raw values summed in another order by the two paths' projections)
    assert_close(stored[0], stored[1], "statistics", rtol=RTOL)


def test_training_mode_without_gradients_stores_the_statistics(dev):
    cfg = default_params(num_layers=2)
    one, two = scaled(cfg).to(dev).train(), scaled(cfg).to(dev).train()
    b = batch_of([9, 20]).to(dev)
    handle = two.encoder.layers[0].register_forward_hook(lambda m, i, o: None)
    with torch.no_grad():
        y1, y2 = one(b), two(b)
    handle.remove()
    assert_close(y1, y2, "first pass")
    for l1, l2 in zip(one.encoder.layers, two.encoder.layers):
        assert float(l1.self_attn.gauss_scale[0]) > 0
        assert_close(l1.self_attn.gauss_scale, l2.self_attn.gauss_scale, "statistics")
    stored = [layer.self_attn.gauss_scale.clone() for layer in one.encoder.layers]
    with torch.no_grad():
        one(batch_of([4, 31], seed=8).to(dev))
    for layer, s in zip(one.encoder.layers, stored):
        assert torch.equal(layer.self_attn.gauss_scale, s)         # written once


def test_native_forward_leaves_other_models_to_the_modules(dev):
    b = batch_of([4, 6]).to(dev)
    for options in (dict(domain="reci"), dict(domain="multihead", gauss_lb_reci=0.3), dict(value_pe_condproj="i"), dict(gauss_state="1"),
                    dict(t_fixup_init=False), dict(norm_func_mode=2), dict(use_low_memory=False),
                    dict(t_activation="gelu")):
        model = scaled(default_params(num_layers=1, **options)).to(dev).eval()
        x = torch.nn.functional.linear(b.x, model.input_embeddings.weight)
        with torch.no_grad():
            assert executor.encode(model.encoder, x, b.pos, b.batch, b.trans_vec, b.sizes) is None, options
            assert torch.isfinite(model(b)).all()
    model = scaled(default_params(num_layers=1)).to(dev).eval()
    x = torch.nn.functional.linear(b.x, model.input_embeddings.weight)
    assert executor.encode(model.encoder, x, b.pos, b.batch, b.trans_vec, b.sizes) is None      # gradients wanted
    hip_funcs.KernelManager.DENSE_EDGE_BLOCKS = False
    try:
        with torch.no_grad():
            assert executor.encode(model.encoder, x, b.pos, b.batch, b.trans_vec, b.sizes) is None
    finally:
        hip_funcs.KernelManager.DENSE_EDGE_BLOCKS = True
