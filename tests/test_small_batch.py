"""Up to how many rows the memory layer's projections run on the decode step's kernel."""
import pytest

from smlm_hip.pkm import ProductKeyMemory


@pytest.mark.parametrize("width,v_dim,heads,k_dim,rows", [
    (384, 384, 4, 256, 64), (64, 64, 1, 16, 64), (1024, 1024, 4, 512, 64), (1024, 1024, 8, 512, 64), (384, 2048, 4, 512, 64),
    (1024, 1024, 8, 528, 16), (1536, 1536, 4, 512, 16), (1024, 1024, 8, 1024, 16), (2048, 2048, 4, 512, 16),
    (2048, 2048, 8, 1024, 16), (2048, 2048, 8, 1040, 0)])
def test_rows_by_the_weights_of_the_layer(width, v_dim, heads, k_dim, rows):
    m = ProductKeyMemory(width, width, n_keys=4, heads=heads, knn=2, k_dim=k_dim, v_dim=v_dim)
    assert m._small_batch_rows() == rows
    m.SMALL_BATCH = 5
    assert m._small_batch_rows() == min(5, rows)
