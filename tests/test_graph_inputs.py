"""Refreshing a graph's inputs: destinations keep the strides of the batch that was captured."""
import dataclasses

import pytest
import torch

from crystalformer_amd import graphs
from tests.test_executor_dispatch import small_batch, small_model


def strided(t):
    """The values of ``t`` with its last two dimensions the other way round in memory."""
    return t.transpose(-2, -1).contiguous().transpose(-2, -1)


def test_strided_destinations():
    src = torch.randn(3, 3, 3)
    dst = strided(torch.zeros(3, 3, 3)).clone()
    assert not dst.is_contiguous()
    graphs._refresh(((dst, src),))
    assert torch.equal(dst, src)


@pytest.mark.gpu
@pytest.mark.parametrize("field", ["trans_vec", "pos", "x"])
def test_replay_after_a_capture_of_strided_inputs(dev, field):
    model, b = small_model().to(dev), small_batch().to(dev)
    captured = dataclasses.replace(b, **{field: strided(getattr(b, field))})
    graph = graphs.GraphedForward(model, captured)
    other = dataclasses.replace(b, pos=b.pos.flip(0).contiguous(), trans_vec=b.trans_vec * 1.1, x=b.x.flip(0))
    for batch in (other, b, other):
        with torch.no_grad():
            want = model(batch)
        got = graph(batch)
        # (strided inputs go through the modules, whose sums are ordered differently)
        assert float((got - want).abs().max()) <= 1e-5 * float(want.abs().max())
