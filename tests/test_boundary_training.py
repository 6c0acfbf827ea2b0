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


@pytest.mark.parametrize("N,H,NK,half,taken", [(16384, 1, 128, 32, True), (16385, 1, 128, 32, False), (16384, 8, 1024, 248, True),
                                               (65536, 4, 128, 248, False), (131072, 4, 256, 256, True),
                                               (131073, 4, 256, 256, False)])
def test_long_walks_of_the_keys_gradient_go_through_the_library(N, H, NK, half, taken):
    """More tokens than its few workgroups walk faster than the library's split products."""
    assert kernels.score_keys_grad_supported(N, H, NK, half) == taken


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


@pytest.mark.parametrize("N,C,taken", [(16384, 8, True), (16385, 8, False), (131072, 64, True), (131073, 64, False),
                                       (246000, 120, False), (1 << 20, 128, True)])
def test_tall_narrow_query_norms_go_through_torch(N, C, taken):
    """Few columns leave most lanes of the kernel idle."""
    assert kernels.query_norm_supported(N, C) == taken


def _strides(*s):
    return (ctypes.c_int64 * 3)(*s)


def test_attention_train_refusals():
    lib = _lib.lib()
    H, T, hd = 2, 100, 64
    ok = dict(q=FAKE, k=FAKE, v=FAKE, vs=_strides(T * 384, 64, 384), y=FAKE, ys=_strides(T * 128, 64, 128), lse=FAKE,
              ls=128, B=1, H=H, T=T, hd=hd)

    def call(**kw):
        return lib.smlm_attention_train(*dict(ok, **kw).values(), None)

    for name in ("q", "k", "v", "vs", "y", "ys", "lse"):
        assert call(**{name: None}) == _lib.EINVAL and "null" in _lib.last_error(), name
    for name in ("q", "k", "v"):
        assert call(**{name: FAKE + 8}) == _lib.EINVAL and "aligned" in _lib.last_error(), name
    assert call(y=FAKE + 4) == _lib.EINVAL and "aligned" in _lib.last_error()
    assert call(hd=48) == call(hd=256) == _lib.EUNSUPPORTED and "head_dim" in _lib.last_error()
    assert call(vs=_strides(T * 384, 64, 380)) == call(ys=_strides(-4, 64, 128)) == _lib.EINVAL
    assert call(B=-1) == call(H=0) == call(T=-1) == call(ls=T - 1) == _lib.EINVAL
    assert call(T=1 << 23, ls=1 << 23) == _lib.EUNSUPPORTED and "2 GB" in _lib.last_error()
    assert call(B=1 << 30) == _lib.EINVAL and "workgroups" in _lib.last_error()
    assert call(B=0) == call(T=0) == _lib.OK                                    # nothing to do


def test_attention_backward_refusals():
    lib = _lib.lib()
    T = 100
    ok = dict(q=FAKE, k=FAKE, v=FAKE, vs=_strides(T * 384, 64, 384), y=FAKE, dy=FAKE, ys=_strides(T * 128, 64, 128), lse=FAKE,
              delta=FAKE, stride=128, cos=FAKE, sin=FAKE, dtype=_lib.F32, rope_len=T + 5, pos0=5, dqkv=FAKE, B=1, H=2, T=T,
              hd=64)

    def call(**kw):
        return lib.smlm_attention_backward(*dict(ok, **kw).values(), None)

    for name in ("q", "k", "v", "vs", "y", "dy", "ys", "lse", "delta", "cos", "sin", "dqkv"):
        assert call(**{name: None}) == _lib.EINVAL and "null" in _lib.last_error(), name
    for name in ("q", "k", "v", "y", "dy", "lse", "delta"):
        assert call(**{name: FAKE + 8}) == _lib.EINVAL and "aligned" in _lib.last_error(), name
    assert call(dqkv=FAKE + 4) == _lib.EINVAL
    assert call(dtype=_lib.I8) == _lib.EINVAL and "rope" in _lib.last_error()
    assert call(pos0=-1) == call(pos0=6) == call(rope_len=T) == _lib.EINVAL      # positions outside the table
    assert call(stride=100) == call(stride=64) == _lib.EINVAL                   # no multiple of 64, below T
    assert call(hd=16) == _lib.EUNSUPPORTED
    assert call(vs=_strides(T * 384, 60, 384)) == call(ys=_strides(T * 128, 64, 124)) == _lib.EINVAL
    big = 1 << 23
    assert call(T=big, stride=big, rope_len=big + 5) == _lib.EUNSUPPORTED and "2 GB" in _lib.last_error()
    assert call(B=1 << 30) == _lib.EINVAL
    assert call(B=0) == call(T=0) == _lib.OK


def test_engram_mix_refusals():
    lib = _lib.lib()
    shape = dict(B=1, T=40, d=64, taps=4, dilation=3, eps=1e-5)
    ok = dict(h=FAKE, k=FAKE, v=FAKE, wh=FAKE, wk=FAKE, wv=FAKE, conv=FAKE, dtype=_lib.F32, left=None, tail=None, **shape, y=FAKE)
    grad = dict(gy=FAKE, h=FAKE, k=FAKE, v=FAKE, wh=FAKE, wk=FAKE, wv=FAKE, conv=FAKE, **shape, dh=FAKE, dk=FAKE, dv=FAKE,
                dwh=FAKE, dwk=FAKE, dwv=FAKE, dconv=FAKE, parts=FAKE)

    def forward(**kw):
        return lib.smlm_engram_mix(*dict(ok, **kw).values(), None)

    def backward(**kw):
        return lib.smlm_engram_mix_backward(*dict(grad, **kw).values(), None)

    for name in ("h", "k", "v", "wh", "wk", "wv", "conv", "y"):
        assert forward(**{name: None}) == _lib.EINVAL, name
    for name in ("h", "k", "v", "wh", "wk", "wv", "left", "tail", "y"):
        assert forward(**{name: FAKE + 8}) == _lib.EINVAL and "aligned" in _lib.last_error(), name
    for name in set(grad) - set(shape):
        assert backward(**{name: None}) == _lib.EINVAL, name
    for name in ("gy", "h", "k", "v", "wh", "wk", "wv", "dh", "dk", "dv"):
        assert backward(**{name: FAKE + 8}) == _lib.EINVAL and "aligned" in _lib.last_error(), name
    assert forward(dtype=_lib.I8) == _lib.EINVAL
    for call in (forward, backward):
        for bad in (dict(B=0), dict(T=0), dict(d=0), dict(d=12), dict(d=520), dict(taps=0), dict(taps=5), dict(dilation=0),
                    dict(dilation=11), dict(B=1 << 31), dict(B=1 << 20, T=1 << 20)):
            assert call(**bad) == _lib.EUNSUPPORTED, bad
    assert kernels.ENGRAM_MIX_MAX_D == 512 and kernels.ENGRAM_MIX_MAX_TAPS == 4 and kernels.ENGRAM_MIX_MAX_PAST == 32
    assert lib.smlm_engram_mix_parts(3, 33, 64, 4) == 3 * 2 * 7 * 64


def test_score_keys_grad_refusals():
    lib = _lib.lib()
    ok = dict(g1=FAKE, g2=FAKE, q=FAKE, N=5, H=2, NK=64, half=32, dk=FAKE, dtype=_lib.F32)

    def call(**kw):
        return lib.smlm_score_keys_grad(*dict(ok, **kw).values(), None)

    assert call(q=None) == call(dk=None) == _lib.EINVAL and "null" in _lib.last_error()
    for name in ("g1", "g2", "q", "dk"):
        assert call(**{name: FAKE + 8}) == _lib.EINVAL and "aligned" in _lib.last_error(), name
    assert call(dtype=_lib.I8) == _lib.EINVAL


def test_query_norm_backward_refusals():
    lib = _lib.lib()
    names = ("g", "x", "weight", "mean", "invstd", "N", "C", "parts", "k", "dx", "dweight", "dbias")
    ok = dict.fromkeys(names, FAKE) | dict(N=4, C=16)

    def call(**kw):
        return lib.smlm_query_norm_backward(*dict(ok, **kw).values(), None)

    for name in set(names) - {"N", "C"}:
        assert call(**{name: None}) == _lib.EINVAL, name
    for name in ("g", "x", "dx", "parts"):
        assert call(**{name: FAKE + 8}) == _lib.EINVAL and "aligned" in _lib.last_error(), name
    assert lib.smlm_query_norm_parts(0, 8) == lib.smlm_query_norm_parts(8, 0) == 0 < lib.smlm_query_norm_parts(2, 8)


def test_flagged_norm_refusals():
    lib = _lib.lib()
    ok = dict(acc=FAKE, touched=FAKE, rows=4, D=8, max_norm=1.0, parts=FAKE, out=FAKE)

    def call(**kw):
        return lib.smlm_flagged_norm(*dict(ok, **kw).values(), None)

    for name in ("acc", "touched", "parts", "out"):
        assert call(**{name: None}) == _lib.EINVAL and "null" in _lib.last_error(), name
    assert call(rows=-1) == call(D=0) == _lib.EINVAL
    assert lib.smlm_flagged_norm_parts() >= 1


def test_decode_linear_pair_refusals():
    lib = _lib.lib()

    def call(w2=FAKE, **kw):
        a = _lib.LinearArgs()
        for name, value in dict(dict(M=4, N=64, K=64, prologue=_lib.LIN_PLAIN, epilogue=_lib.LIN_STORE, x=FAKE, x_stride=64,
                                     w=FAKE, out=FAKE, out_stride=32, out2=FAKE, out2_stride=32, n_split=32), **kw).items():
            assert hasattr(a, name), name
            setattr(a, name, value)
        return lib.smlm_decode_linear_pair(ctypes.byref(a), w2, None, None)

    assert call(M=0) == _lib.OK                                                 # valid, and nothing to do
    assert lib.smlm_decode_linear_pair(None, FAKE, None, None) == _lib.EINVAL
    assert call(w2=None, M=0) == call(w2=FAKE + 8, M=0) == _lib.EINVAL
    assert call(n_split=0, M=0) == call(n_split=64, M=0, out_stride=64) == call(n_split=24, M=0) == _lib.EINVAL
    assert call(epilogue=_lib.LIN_SWIGLU, M=0) != _lib.OK and call(epilogue=_lib.LIN_ARGMAX, M=0) != _lib.OK
