"""The training and Engram entry points' argument checks, without a GPU: the documented status codes before anything is
launched, and host rules that ask for no more than the entry points take."""
import ctypes

import pytest

from smlm_hip import _lib, kernels

FAKE = 256                    # a 16-byte aligned address that is never read: the checks fail first


@pytest.mark.parametrize("N,H,NK,half", [(1, 32769, 8, 8), (4, 2, 12, 8), (4, 2, 8, 12), (1 << 20, 4, 1024, 256), (0, 2, 8, 8)])
def test_the_keys_gradient_is_asked_for_what_it_takes(N, H, NK, half):
    """Shapes that smlm_score_keys_grad refuses go through the library's products."""
    assert not kernels.score_keys_grad_supported(N, H, NK, half)
    lib = _lib.lib()
    assert lib.smlm_score_keys_grad(FAKE, FAKE, FAKE, N, H, NK, half, FAKE, _lib.F32, None) == _lib.EUNSUPPORTED
    assert kernels.score_keys_grad_supported(4096, 4, 1024, 256)


def test_the_scores_are_asked_for_what_they_take():
    lib, most = _lib.lib(), kernels.SCORE_MAX_HEADS
    assert lib.smlm_pkm_score(FAKE, 16 * (most + 1), FAKE, _lib.BF16, 0, most + 1, 8, 8, FAKE, FAKE, None) == _lib.EINVAL
    assert lib.smlm_pkm_score(FAKE, 16 * most, FAKE, _lib.BF16, 0, most, 8, 8, FAKE, FAKE, None) == _lib.OK    # no rows


@pytest.mark.parametrize("N,C", [(2, (1 << 20) + 8), (1, 8), (2, 12), (2, 0)])
def test_the_query_norm_gradient_is_asked_for_what_it_takes(N, C):
    """Shapes that smlm_query_norm_backward refuses go through torch's batch norm."""
    assert not kernels.query_norm_supported(N, C)
    lib = _lib.lib()
    assert lib.smlm_query_norm_backward(*[FAKE] * 5, N, C, *[FAKE] * 6, None) == _lib.EUNSUPPORTED
    assert kernels.query_norm_supported(2, 8) and kernels.query_norm_supported(4096, 1 << 20)
