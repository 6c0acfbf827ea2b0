"""The eval-mode BatchNorm's scale and shift, kept by the memory layer, follow what they are made from."""
import pytest
import torch

from smlm_hip.pkm import ProductKeyMemory


@torch.no_grad()
@pytest.mark.parametrize("what", ["statistics", "weight", "bias", "loaded"])
def test_the_affine_follows_the_batch_norm(what):
    torch.manual_seed(0)
    m = ProductKeyMemory(8, 8, n_keys=8, heads=2, knn=2, k_dim=8).eval()
    bn, x = m.query_norm, torch.randn(30, 16) * 2 + 3
    m._bn_affine()
    if what == "statistics":              # a training pass without an optimizer step
        bn.train()
        bn(x)
        bn.eval()
    elif what == "loaded":
        bn.load_state_dict({k: v + 1 for k, v in bn.state_dict().items()})
    else:
        getattr(bn, what).add_(1.0)
    scale, shift = m._bn_affine()
    torch.testing.assert_close(x * scale + shift, bn(x))
    assert m._bn_affine()[0] is scale
