"""The recorded sub-key scores' backward around its kernels (smlm_hip.pkm._SubkeyScores), with the kernels restated in
PyTorch: which gradients reach them, and what it returns."""
import pytest
import torch

from smlm_hip import kernels
from smlm_hip.pkm import _score_ops, _SubkeyScores


@pytest.fixture
def keys_grads(monkeypatch):
    """Restates the two kernels; collects which of score_keys_grad's halves came with a gradient."""
    seen = []

    def score_keys_grad(g1, g2, q, keys_shape, dtype):
        seen.append((g1 is not None, g2 is not None))
        half = keys_shape[3]
        return torch.stack([torch.zeros(keys_shape[0], *keys_shape[2:], dtype=dtype) if g is None
                            else torch.einsum("nhk,nhd->hkd", g, q[..., p * half:(p + 1) * half]).to(dtype)
                            for p, g in enumerate((g1, g2))], 1)

    monkeypatch.setattr(kernels, "pk_scores", _score_ops)
    monkeypatch.setattr(kernels, "score_keys_grad", score_keys_grad)
    return seen


def _inputs(n_keys):
    g = torch.Generator().manual_seed(n_keys)
    q, keys = (torch.randn(*s, generator=g, dtype=torch.float64).requires_grad_()
               for s in ((5, 2, 16), (2, 2, n_keys, 8)))
    return q, keys, [torch.randn(5, 2, n_keys, generator=g, dtype=torch.float64) for _ in range(2)]


@pytest.mark.parametrize("n_keys", [16, 12], ids=["kernel", "products"])
@pytest.mark.parametrize("halves", [(0,), (1,), (0, 1)])
def test_only_the_halves_that_were_used_have_a_gradient(keys_grads, halves, n_keys):
    q, keys, grads = _inputs(n_keys)
    got, ref = _SubkeyScores.apply(q, keys), _score_ops(q, keys)
    chosen = [[t[p] for p in halves] for t in (got, ref, grads)]
    for a, b in zip(torch.autograd.grad(chosen[0], (q, keys), chosen[2], retain_graph=True),
                    torch.autograd.grad(chosen[1], (q, keys), chosen[2], retain_graph=True)):
        torch.testing.assert_close(a, b)
    assert keys_grads == ([] if n_keys % 8 else [(0 in halves, 1 in halves)])
    for wanted in ((q,), (keys,), (q, keys)):                   # recorded: the einsum's
        for a, b in zip(torch.autograd.grad(chosen[0], wanted, chosen[2], create_graph=True),
                        torch.autograd.grad(chosen[1], wanted, chosen[2], create_graph=True)):
            torch.testing.assert_close(a, b)
            assert a.requires_grad


class _NoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, a, b):
        return a + b

    @staticmethod
    def backward(ctx, g):
        return None, None


@pytest.mark.parametrize("create_graph", [False, True])
def test_no_gradient_at_all(keys_grads, create_graph):
    q, keys, _ = _inputs(16)
    for scores in (_SubkeyScores.apply, _score_ops):
        out = _NoGradient.apply(*scores(q, keys)).sum()
        got = torch.autograd.grad(out, (q, keys), create_graph=create_graph, allow_unused=True)
        assert all(g is None for g in got)
    assert keys_grads == []
