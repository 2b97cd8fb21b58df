"""A training block as one call each way (``hip_funcs.BlockTrainHIP``) against its operators one by one: the same bits,
whatever is trained, frozen, deferred or brought back by a saved-tensor hook."""
import pytest
import torch

from crystalformer_amd import executor, hip_funcs, ops
from crystalformer_amd.graphs import GraphedTrainStep
from crystalformer_amd.latticeformer import default_params
from crystalformer_amd.lib import CrystalformerHipError
from tests.test_gpu_forward import batch_of, scaled

pytestmark = pytest.mark.gpu


def labelled(sizes, dev):
    b = batch_of(sizes)
    b.y = torch.randn(len(sizes), generator=torch.Generator().manual_seed(7))
    return b.to(dev)


def nodes(loss):
    seen, todo = set(), [loss.grad_fn]
    while todo:
        f = todo.pop()
        if f is not None and f not in seen:
            seen.add(f)
            todo += [g for g, _ in f.next_functions]
    return [type(f).__name__ for f in seen]


def both(model, b, monkeypatch, deferred=True, step=None):
    """(loss, gradients, statistics) as one call a block and operator by operator, from the same state."""
    got = []
    start = [layer.self_attn.gauss_scale.clone() for layer in model.encoder.layers]
    for native in (True, False):
        with monkeypatch.context() as m:
            if not native:
                m.setattr(executor, "native_training", lambda *a: None)
            m.setattr(hip_funcs, "USE_LINEAR_FUNCTION", True)
            for layer, g in zip(model.encoder.layers, start):
                layer.self_attn.gauss_scale.data.copy_(g)
            model.zero_grad(set_to_none=True)
            loss = (model(b)[:, 0] - b.y).abs().mean()
            assert ("BlockTrainHIPBackward" in nodes(loss)) == native
            if deferred:
                with hip_funcs.deferred_weight_grads():
                    loss.backward()
            else:
                loss.backward()
            got.append([loss.detach()] + [p.grad for p in model.parameters()]
                       + [layer.self_attn.gauss_scale.detach().clone() for layer in model.encoder.layers])
    return got


def same(one, two):
    for a, b in zip(one, two):
        assert (a is None) == (b is None)
        if a is not None:
            assert torch.equal(a, b)


@pytest.mark.parametrize("sizes", [[2], [1, 2, 30], [5, 1, 64, 3], [200, 7]])
@pytest.mark.parametrize("options", [dict(), dict(adaptive_cutoff_sigma=0.0), dict(value_pe_dist_real=0), dict(head_num=4),
                                     dict(head_num=16, value_pe_dist_real=33), dict(value_pe_dist_real=128),
                                     dict(normalize_gauss=False), dict(adaptive_cutoff_sigma=2.0)])
def test_same_bits_as_the_operators(dev, sizes, options, monkeypatch):
    model = scaled(default_params(num_layers=2, **options)).to(dev).train()
    same(*both(model, labelled(sizes, dev), monkeypatch))


@pytest.mark.parametrize("rings", [True, False])
def test_without_rings_and_without_deferral(dev, rings, monkeypatch):
    monkeypatch.setattr(hip_funcs.KernelManager, "STAGED_RINGS", rings)
    model = scaled(default_params(num_layers=2)).to(dev).train()
    same(*both(model, labelled([9, 20], dev), monkeypatch, deferred=False))


@pytest.mark.parametrize("frozen", ["in_proj_bias", "q_proj", "linear1.bias", "linear2.weight", "pe_dist_proj", "lattice_pos",
                                    "out_proj", "input_embeddings", "layers.0"])
@pytest.mark.parametrize("deferred", [True, False])
def test_frozen_parameters(dev, frozen, deferred, monkeypatch):
    model = scaled(default_params(num_layers=2)).to(dev).train()
    for name, p in model.named_parameters():
        if frozen in name or "gauss_scale" in name:
            p.requires_grad_(False)
    same(*both(model, labelled([9, 20], dev), monkeypatch, deferred=deferred))


def test_blocks_nobody_differentiates_through(dev, monkeypatch):
    """Only the last layer trained: its own backward launch and no other."""
    model = scaled(default_params(num_layers=2)).to(dev).train()
    for name, p in model.named_parameters():
        p.requires_grad_(name.startswith("encoder.layers.1.linear2"))
    monkeypatch.setattr(hip_funcs, "USE_LINEAR_FUNCTION", True)
    b = labelled([9, 20], dev)
    loss = (model(b)[:, 0] - b.y).abs().mean()
    found = nodes(loss)
    assert "BlockTrainHIPBackward" not in found and "FusedDotProductAttentionCUDABackward" not in found


def test_saved_tensor_hooks_and_a_second_backward(dev, monkeypatch):
    model = scaled(default_params(num_layers=2)).to(dev).train()
    b = labelled([9, 20], dev)
    monkeypatch.setattr(hip_funcs, "USE_LINEAR_FUNCTION", True)
    plain = (model(b)[:, 0] - b.y).abs().mean()
    params = [p for p in model.parameters() if p.requires_grad]
    first = torch.autograd.grad(plain, params, retain_graph=True)
    same(first, torch.autograd.grad(plain, params))
    with torch.autograd.graph.save_on_cpu():
        loss = (model(b)[:, 0] - b.y).abs().mean()
    same(first, torch.autograd.grad(loss, params))
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t[:-1] if t.dim() == 1 and t.numel() > 40000 else t, lambda t: t):
        loss = (model(b)[:, 0] - b.y).abs().mean()
    with pytest.raises(CrystalformerHipError):
        torch.autograd.grad(loss, params)


def test_a_parameter_changed_in_between_is_noticed(dev, monkeypatch):
    model = scaled(default_params(num_layers=1)).to(dev).train()
    b = labelled([9, 20], dev)
    monkeypatch.setattr(hip_funcs, "USE_LINEAR_FUNCTION", True)
    loss = (model(b)[:, 0] - b.y).abs().mean()
    with torch.no_grad():
        model.encoder.layers[0].linear1.weight.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()


def test_what_outlives_a_block(dev, monkeypatch):
    """A gradient holds its own memory alone, and what deferred weight gradients wait with is rows, not edges."""
    b = labelled([60, 60], dev)
    model = scaled(default_params(num_layers=2)).to(dev).train()
    monkeypatch.setattr(hip_funcs, "USE_LINEAR_FUNCTION", True)
    with hip_funcs.deferred_weight_grads():
        (model(b)[:, 0] - b.y).abs().mean().backward()
        waiting = {t.untyped_storage().data_ptr(): t.untyped_storage().nbytes()
                   for entry in hip_funcs._deferred for t in entry[:2]}
    atoms, rows = 120, 128 * 4
    # (per block: att, s, h and gq, gk, gv, gs, gx, gh; the block inputs and the gradient behind the last block)
    assert sum(waiting.values()) < (2 * (6 + 9) + 4) * atoms * rows, waiting
    for name, p in model.named_parameters():
        if p.grad is not None and "lattice_pos_weights" in name:
            assert p.grad.untyped_storage().nbytes() == rows


def test_graph_replays_and_eager_steps(dev, monkeypatch):
    """The captured step, replayed with eager work in between, has the eager step's bits."""
    b = labelled([9, 20, 3], dev)
    model = scaled(default_params(num_layers=2)).to(dev).train()
    step = GraphedTrainStep(model, b)                      # (leaves the exponents' statistics stored)
    for _ in range(3):                                     # (every replay changes the parameters)
        native, operators = both(model, b, monkeypatch)
        same(native, operators)
        assert torch.equal(step(b), native[0])


def test_instrumented_runs_take_the_operators(dev, monkeypatch):
    model = scaled(default_params(num_layers=1)).to(dev).train()
    b = labelled([9, 20], dev)
    monkeypatch.setattr(hip_funcs, "USE_LINEAR_FUNCTION", True)
    monkeypatch.setattr(ops, "_event_log", [])
    assert "BlockTrainHIPBackward" not in nodes(model(b).sum())
