"""Which models, batches and settings the native inference call is chosen for, on the CPU (the call itself is
replaced by a marker), and on the GPU that everything it leaves alone computes what its modules say."""
import ctypes
import dataclasses
import types

import pytest
import torch
from torch import nn

from crystalformer_amd import executor, lib, ops
from crystalformer_amd.encoder import CrystalformerEncoderCUDA
from crystalformer_amd.lib import CrystalformerHipError
from crystalformer_amd.latticeformer import Latticeformer, default_params
from crystalformer_amd.synthetic import make_batch
from crystalformer_amd.training import fused_training_step, training_step
from tests.helpers import RTOL, assert_close


def small_model(**options):
    torch.manual_seed(2)
    model = Latticeformer(default_params(num_layers=2, **options)).eval()
    with torch.no_grad():
        model.input_embeddings.weight.normal_()            # (the initialisation's features are near zero)
        for layer in model.encoder.layers:                 # trained: stored statistics
            layer.self_attn.gauss_scale.copy_(torch.tensor([0.7, -0.2]))
    return model


def small_batch():
    return make_batch(3, (4, 9), False, (3.0, 11.0), (65.0, 115.0), seed=3)


@pytest.fixture
def natively(monkeypatch):
    """Whether a model's forward would take the native call: ``_run`` answers with a marker."""
    marker = torch.zeros(())
    monkeypatch.setattr(executor, "_run", lambda *args: None if args[6] is None else marker)

    def ask(model):
        with torch.no_grad():
            return executor.forward(model, small_batch())[0] is marker
    assert ask(small_model())
    return ask


def same_with_and_without_gradients(model, dev):
    """Under ``no_grad`` the model computes what it computes with gradients enabled, which is module by module."""
    model, b = model.to(dev), small_batch().to(dev)
    with torch.no_grad():
        got = model(b)
    assert_close(got, model(b).detach(), "model", rtol=RTOL)
    return got


class HalvingEncoder(CrystalformerEncoderCUDA):
    def forward(self, *args):
        return super().forward(*args) * 0.5


class ForeignEncoder(nn.Module):                           # (no layers, no d_model)
    def __init__(self, width=128):
        super().__init__()
        self.proj = nn.Linear(width, width)

    def forward(self, src, pos, batch, trans, sizes, onehot=None):
        return self.proj(src)


def subclassed_encoder(model):
    model.encoder.__class__ = HalvingEncoder


def foreign_encoder(model):
    model.encoder = ForeignEncoder()


def replaced_forward(model):
    plain = model.encoder.forward
    model.encoder.forward = lambda *args: plain(*args) * 0.5


@pytest.mark.parametrize("change", [subclassed_encoder, foreign_encoder, replaced_forward])
def test_encoders_of_the_users_own(natively, change):
    model = small_model()
    change(model)
    assert not natively(model)


@pytest.mark.gpu
@pytest.mark.parametrize("change", [subclassed_encoder, foreign_encoder, replaced_forward])
def test_encoders_of_the_users_own_are_called(dev, change):
    model = small_model()
    plain = same_with_and_without_gradients(small_model(), dev)
    change(model)
    assert not torch.equal(same_with_and_without_gradients(model, dev), plain)


class Residual(nn.Module):                                 # (the children of the usual head, used differently)
    def __init__(self):
        super().__init__()
        torch.manual_seed(4)
        self.a, self.r, self.b = nn.Linear(128, 128), nn.ReLU(), nn.Linear(128, 1)

    def forward(self, x):
        return self.b(x + self.r(self.a(x)))


class ResidualSequential(nn.Sequential):
    def __init__(self):
        torch.manual_seed(4)
        super().__init__(nn.Linear(128, 128), nn.ReLU(), nn.Linear(128, 1))

    def forward(self, x):
        return self[2](x + self[1](self[0](x)))


class DoublingModel(Latticeformer):
    def _head(self, x):
        return super()._head(x) * 2.0


def residual_head(model):
    model.mlp = Residual()


def residual_sequential_head(model):
    model.mlp = ResidualSequential()


def residual_instance_head(model):
    model.mlp = nn.Sequential(*ResidualSequential())
    model.mlp.forward = ResidualSequential.forward.__get__(model.mlp)


def overridden_head(model):
    model.__class__ = DoublingModel


HEADS = [residual_head, residual_sequential_head, residual_instance_head, overridden_head]


@pytest.mark.parametrize("change", HEADS)
def test_heads_of_the_users_own(natively, change):
    model = small_model()
    change(model)
    assert not natively(model)


@pytest.mark.gpu
@pytest.mark.parametrize("change", HEADS)
def test_heads_of_the_users_own_are_called(dev, change):
    model = small_model()
    b = small_batch().to(dev)
    change(model)
    got = same_with_and_without_gradients(model, dev)
    with torch.no_grad():
        x = torch.nn.functional.linear(b.x, model.input_embeddings.weight)
        x = model.encoder(x, b.pos, b.batch, b.trans_vec, b.sizes)
        pooled = torch.stack([p.double().mean(0) for p in x.split(b.sizes.tolist())]).float()
        want = 2.0 * model.mlp(pooled) if change is overridden_head else model.mlp(pooled)
    assert_close(got, want, "head", rtol=RTOL)


def weight_norm(module):
    torch.nn.utils.parametrizations.weight_norm(module)


def plain_attributes(module):
    """Weight and bias worked out elsewhere and set as plain tensors, as reparametrising code does."""
    for name in ("weight", "bias"):
        value = getattr(module, name).detach().clone() * 1.5 + 0.01
        delattr(module, name)
        setattr(module, name, value)


MODULES = [lambda m: m.encoder.layers[1].self_attn.out_proj, lambda m: m.encoder.layers[0].linear1,
           lambda m: m.encoder.layers[1].linear2, lambda m: m.mlp[0], lambda m: m.mlp[-1]]


@pytest.mark.parametrize("where", range(len(MODULES)))
@pytest.mark.parametrize("change", [weight_norm, plain_attributes])
def test_blocks_with_parameters_worked_out_are_declined(where, change):
    model = small_model()
    change(MODULES[where](model))
    blocks = [executor._block(layer, 128, -1) for layer in model.encoder.layers]
    head = executor._head(model.mlp, 128, -1)
    assert [blocks[1], blocks[0], blocks[1], head, head][where] is None
    assert sum(b is None for b in blocks) + (head is None) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("where", range(len(MODULES)))
@pytest.mark.parametrize("change", [weight_norm, plain_attributes])
def test_blocks_with_parameters_worked_out(dev, where, change):
    model = small_model().to(dev)
    change(MODULES[where](model))
    same_with_and_without_gradients(model, dev)


class PlainSGD:
    """An optimiser with the interface the training steps use, which leaves the parameters alone."""
    def __init__(self, model):
        self.params = list(model.parameters())

    def zero_grad(self, set_to_none=True):
        for p in self.params:
            p.grad = None

    def step(self):
        pass


def step_gradients(model, dev, fused):
    """Loss and gradients of one training step: from the fused step, or of the plain one."""
    b = make_batch(3, (4, 9), False, (3.0, 11.0), (65.0, 115.0), seed=3, with_targets=True).to(dev)
    opt = PlainSGD(model)
    loss = fused_training_step(model, b, opt) if fused else training_step(model, b, opt, clip_norm=0)
    return [loss] + [p.grad for p in opt.params if p.requires_grad]


def fused_step_equals_the_plain_one(model, dev):
    model = model.to(dev)
    plain = step_gradients(model, dev, False)
    for got, want in zip(step_gradients(model, dev, True), plain):
        # (sums over the atoms in another order: relative to the whole tensor)
        assert float((got - want).norm()) <= RTOL * float(want.norm().clamp_min(1e-12))


@pytest.mark.gpu
@pytest.mark.parametrize("where", range(3))
def test_training_with_parameters_worked_out(dev, where):
    model = small_model()
    weight_norm(MODULES[where](model))
    fused_step_equals_the_plain_one(model, dev)


# as many numbers in another shape: what the operators refuse one by one
SHAPES = {"pos": lambda b: dict(pos=b.pos.T.contiguous()), "pos_flat": lambda b: dict(pos=b.pos.reshape(-1)),
          "trans": lambda b: dict(trans_vec=b.trans_vec.reshape(-1, 9)),
          "trans_one": lambda b: dict(trans_vec=b.trans_vec.reshape(1, -1, 3)),
          "trans_rows": lambda b: dict(trans_vec=b.trans_vec.reshape(-1, 1, 9))}


def test_shapes_are_looked_at(monkeypatch):
    """Every batch of these shapes is declined before anything is laid out for it."""
    monkeypatch.setattr(torch.Tensor, "get_device", lambda t: 0)
    monkeypatch.setattr(executor.ops, "batch_layout", lambda *args: pytest.fail("accepted"))
    model, b = small_model(), small_batch()
    for change in SHAPES.values():
        c = dataclasses.replace(b, **change(b))
        with torch.no_grad():
            assert executor.encode(model.encoder, b.x @ model.input_embeddings.weight.T, c.pos, c.batch, c.trans_vec,
                                   c.sizes) is None


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_shapes_are_refused(dev, shape):
    model, b = small_model().to(dev), small_batch().to(dev)
    c = dataclasses.replace(b, **SHAPES[shape](b))
    with torch.no_grad(), pytest.raises(CrystalformerHipError):
        model(c)
    with pytest.raises(CrystalformerHipError):
        model(c)


def accepted(model):
    """Blocks that the native call takes, with whether they store statistics."""
    blocks = [executor._block(layer, 128, -1) for layer in model.encoder.layers]
    return [b and b[3] for b in blocks]


def test_modes_are_each_modules_own():
    model = small_model()
    assert accepted(model) == [False, False]
    assert accepted(model.train()) == [True, True]
    model.encoder.layers[0].eval()                         # (a frozen block)
    assert accepted(model) == [False, True]
    model.encoder.eval().training = True
    assert accepted(model) == [False, False]
    model = small_model(dropout=0.2)
    assert accepted(model) == [False, False]
    assert accepted(model.train()) == [None, None]
    model.eval().encoder.layers[1].self_attn.train()       # dropout on the weights only
    assert accepted(model) == [False, None]
    model.eval().encoder.layers[1].dropout2.train()
    assert accepted(model) == [False, None]
    model = small_model(normalize_gauss=False)
    model.encoder.layers[0].train()
    assert accepted(model) == [False, False]


@pytest.mark.gpu
@pytest.mark.parametrize("frozen", [[0], [1], [0, 1]])
def test_frozen_blocks_keep_their_statistics(dev, frozen):
    model = small_model().to(dev).train()
    for i, layer in enumerate(model.encoder.layers):
        layer.self_attn.gauss_scale.data.zero_()
        if i in frozen:
            layer.eval()
    with torch.no_grad():
        model(small_batch().to(dev))
    for i, layer in enumerate(model.encoder.layers):
        assert bool(layer.self_attn.gauss_scale[0] > 0) == (i not in frozen)


@pytest.mark.gpu
def test_dropout_follows_the_modules_modes(dev):
    """Dropout of an attention in training mode inside a block in evaluation mode, at inference; of a feed-forward
    in training mode, in a fused training step."""
    model, b = small_model(dropout=0.5).to(dev), small_batch().to(dev)
    with torch.no_grad():
        assert torch.equal(model(b), model(b))
        model.encoder.layers[0].self_attn.train()
        assert not torch.equal(model(b), model(b))
    model.eval()
    one, two = (step_gradients(model, dev, True)[0] for _ in range(2))
    assert torch.equal(one, two)
    model.encoder.layers[0].dropout2.train()
    one, two = (step_gradients(model, dev, True)[0] for _ in range(2))
    assert not torch.equal(one, two)


def halved_offsets(attn):
    """An attention whose offsets p_j - p_i are halved."""
    plain = attn.forward
    attn.forward = lambda *args, **kwargs: plain(*args[:6], 0.5 * args[6], *args[7:], **kwargs)


def halved_output(layer):
    plain = layer.forward
    layer.forward = lambda src, *args, **kwargs: 0.5 * plain(src, *args, **kwargs)


INNER = {"attention": lambda m: halved_offsets(m.encoder.layers[1].self_attn),
         "layer": lambda m: halved_output(m.encoder.layers[0])}
HOOKED = {"attention": lambda m: m.encoder.layers[1].self_attn, "layer": lambda m: m.encoder.layers[0]}


@pytest.mark.parametrize("where", INNER)
def test_forwards_replaced_below_the_encoder(where):
    model = small_model()
    assert not executor._touched(model.encoder)
    INNER[where](model)
    assert executor._touched(model.encoder)
    model = small_model()
    HOOKED[where](model).register_full_backward_hook(lambda *args: None)
    assert not executor._touched(model.encoder) and executor._touched(model.encoder, backward=True)


@pytest.mark.gpu
@pytest.mark.parametrize("where", INNER)
def test_forwards_replaced_below_the_encoder_are_called(dev, where):
    """At inference and in a fused training step."""
    model = small_model()
    plain = same_with_and_without_gradients(small_model(), dev)
    INNER[where](model)
    assert not torch.equal(same_with_and_without_gradients(model, dev), plain)
    fused_step_equals_the_plain_one(model, dev)


@pytest.mark.gpu
def test_hooks_of_a_layer_in_a_fused_step(dev):
    """A hook may hand on what the row kernels do not take, rows that are not contiguous here."""
    model = small_model()
    model.encoder.layers[0].register_forward_hook(lambda m, args, out: (0.5 * out.T.contiguous()).T)
    fused_step_equals_the_plain_one(model, dev)


def test_declined_models_are_hardly_looked_at(monkeypatch):
    """Options decide before anything is walked or counted: a model of another kind is asked at every forward."""
    looked = []
    monkeypatch.setattr(executor, "_touched", lambda *args: looked.append(args) or False)
    monkeypatch.setattr(executor, "_ready", lambda *args: looked.append(args) or True)
    for options in (dict(domain="reci"), dict(t_fixup_init=False), dict(t_activation="gelu"),
                    dict(value_pe_condproj="i")):
        model, b = small_model(**options), small_batch()
        with torch.no_grad():
            assert executor.forward(model, b) == (None, None)
            assert executor.encode(model.encoder, b.x, b.pos, b.batch, b.trans_vec, b.sizes) is None
        assert not looked, options


@pytest.mark.parametrize("rows, served", [(0, True), (1, False), (-1, False)])
def test_a_training_block_has_a_row_an_atom(rows, served):
    """A row too many or too few is left to the operators, which say what is wrong, before anything is launched: the
    native call has the batch's index structure and takes the row count from the features."""
    model, b = small_model().train(), small_batch()
    N, E, B = len(b.batch), int((b.sizes ** 2).sum()), len(b.sizes)
    layout = ops.BatchLayout()
    layout.batch, layout.pairs, layout.num_atoms, layout.num_edges = b.batch, torch.zeros((E + N) // 2, 5), N, E
    layout.atom_start = torch.zeros(B + 1, dtype=torch.int64)
    pack = types.SimpleNamespace(settings=[([0] * 26, 8, True)] * 2)
    got = executor.native_training(model.encoder, torch.zeros(N + rows, 128), pack, layout, torch.zeros(E, 3),
                                   b.trans_vec, torch.zeros(B, 3))
    assert (got is not None) == served
    need = (ctypes.c_int64 * 5)()
    args = lib.BlockTrain(N + rows, E, B, (E + N) // 2, 8, 64)
    assert (lib.load().cf_block_train_bytes(ctypes.byref(args), need) == 0) == served
