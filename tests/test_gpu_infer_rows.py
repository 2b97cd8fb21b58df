"""The row kernel of an inference forward (``csrc/block_rows.hip``: split matrix products, tiles of 16 and 32 rows) against
the modules, over rows and columns of any magnitude, and against itself where its tiles change."""
import pytest
import torch

from crystalformer_amd.latticeformer import default_params
from crystalformer_amd.synthetic import CrystalBatch
from tests.helpers import RTOL, assert_close, atol_rows
from tests.test_gpu_forward import batch_of, both_ways, scaled

pytestmark = pytest.mark.gpu


def prepared(dev, **options):
    """A model with stored statistics: an atom's result is then its crystal's alone."""
    model = scaled(default_params(num_layers=2, **options))
    with torch.no_grad():
        for layer in model.encoder.layers:
            layer.self_attn.gauss_scale.copy_(torch.tensor([0.8, -0.1]))
    return model.to(dev).eval()


def head_of(b, crystals):
    n = int(b.sizes[:crystals].sum())
    return CrystalBatch(b.x[:n], b.pos[:n], b.batch[:n], b.trans_vec[:crystals], b.sizes[:crystals])


# a CU's share of 16 rows is full at 4096: tiles of 32 beyond, for up to eight heads; tiles less one, exactly, plus one
@pytest.mark.parametrize("heads", [8, 16])
@pytest.mark.parametrize("atoms", [4095, 4097, 4127, 8193])
def test_a_row_does_not_depend_on_its_tile(dev, atoms, heads):
    sizes = [7] * (atoms // 7) + ([atoms % 7] if atoms % 7 else [])
    model = prepared(dev, head_num=heads)
    b = batch_of(sizes)
    few = head_of(b, 5)
    native, modules = both_ways(model, b.to(dev))
    assert_close(native, modules, "encoder", rtol=RTOL, atol=atol_rows(modules))
    alone, _ = both_ways(model, few.to(dev))
    assert torch.equal(native[:35], alone)
    assert torch.equal(native, both_ways(model, b.to(dev))[0])


# Weights of a column's own magnitude, columns and rows of zeros.  A half's last bit is 2^-24 and a row's (a column's)
# largest value 2^14 to 2^15: what is taken from a value is at most 2^-22 of itself or 2^-38 of the largest, so hidden units
# 2^spread apart either way, which meet weights apart the other way, lose 2^(2 spread - 38) of a term of ordinary size;
# twice that for the two factors, and twice for the two blocks.
@pytest.mark.parametrize("spread", [0, 4, 12])
def test_columns_and_rows_of_any_magnitude(dev, spread):
    model = prepared(dev)
    g = torch.Generator().manual_seed(spread)
    with torch.no_grad():
        for layer in model.encoder.layers:
            powers = torch.exp2(torch.randint(-spread, spread + 1, (512,), generator=g).float()).to(dev)
            layer.linear1.weight.mul_(powers[:, None])            # (the reduction takes the power out again)
            layer.linear1.bias.mul_(powers)
            layer.linear2.weight.div_(powers[None, :])
            layer.linear1.weight[3].zero_()
            layer.self_attn.out_proj.weight[5].zero_()
            layer.linear2.weight[7].zero_()
    b = batch_of([1, 5, 40])
    b.x[2:4] = 0.0                                                # atoms without features
    native, modules = both_ways(model, b.to(dev))
    assert_close(native, modules, "encoder", rtol=RTOL, atol=atol_rows(modules, RTOL + 2.0 ** (2 * spread - 36)))


@pytest.mark.parametrize("value", [float("inf"), float("nan"), 1e38, 1e-38, 1e-42])
def test_features_at_the_ends_of_the_range(dev, value):
    """A crystal with such a feature has the modules' kind of result; its neighbours in the tile their own."""
    model = prepared(dev)
    b = batch_of([3, 4, 5])
    clean, _ = both_ways(model, b.to(dev))
    b.x[4, 0] = value
    native, modules = both_ways(model, b.to(dev))
    assert torch.equal(native[:3], clean[:3]) and torch.equal(native[7:], clean[7:])
    if 1e-40 < value < 1:
        assert_close(native, modules, "encoder", rtol=RTOL, atol=atol_rows(modules))
    elif value < 1e-40:
        assert torch.isfinite(native).all()
    else:
        assert torch.equal(torch.isfinite(native).all(1), torch.isfinite(modules).all(1))
