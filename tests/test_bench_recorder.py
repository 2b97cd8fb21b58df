"""bench.py times the kernels of a forward by re-issuing the operator calls it records: every block's are there,
whichever way the forward itself is issued."""
import pytest
import torch

import bench
from crystalformer_amd import executor, hip_funcs, ops
from tests.test_executor_dispatch import small_batch, small_model


def test_nothing_recorded_is_an_error():
    nothing = {"real_enc_fwd": [], "real_enc_fwd_rings": [], "fused_dpa_fwd": [1]}
    with pytest.raises(SystemExit):
        bench.require_encodings(nothing, "real")
    with pytest.raises(SystemExit):
        bench.require_encodings({"real_enc_bwd": []}, "multihead")
    bench.require_encodings(nothing, "reci")
    bench.require_encodings(dict(nothing, real_enc_fwd_rings=[1]), "real")


@pytest.mark.gpu
@pytest.mark.parametrize("options", [dict(), dict(adaptive_cutoff_sigma=0.0), dict(value_pe_dist_real=0),
                                     dict(domain="multihead")])
def test_every_block_is_recorded(dev, options):
    model, b = small_model(**options).to(dev), small_batch().to(dev)
    names = ("real_enc_fwd", "real_enc_fwd_rings", "fused_dpa_fwd", "staged_rings")
    before = [getattr(ops, name) for name in names]
    with torch.no_grad():
        assert executor.forward(model, b)[0] is not None       # (the forward itself goes past the operators)
        calls = bench.record_calls(ops, names, lambda: model(b))
    assert len(calls["real_enc_fwd"]) + len(calls["real_enc_fwd_rings"]) == len(model.encoder.layers)
    assert len(calls["fused_dpa_fwd"]) == len(model.encoder.layers)
    assert [getattr(ops, name) for name in names] == before
    assert not ops.instrumented() and hip_funcs.KernelManager.FUSE_ENCODING_ATTENTION
