"""Engram n-gram memory on the GPU (smlm_hip.engram): the hash kernel bit-exact against the oracle, the row gather
bit-exact against indexing, the module against the fp64 oracle (fp32 within 1e-5 of the output scale, bf16 within
2e-2), the model's cached / chunked decode against its full forward, and the row-sparse training path against fp64
autograd (1e-5)."""
import numpy as np
import pytest
import torch

import oracle.engram_oracle as E
from smlm_hip import kernels as K
from smlm_hip.engram import EngramMemory, NgramHash
from smlm_hip.model import ModelConfig, Transformer

pytestmark = pytest.mark.gpu
DEV = "cuda"
VOCAB = 1000


def note(msg):
    print(msg, flush=True)


@pytest.mark.parametrize("orders,heads,rows,B,T", [((2, 3), 8, 524287, 4, 300), ((2, 3), 2, 101, 3, 1),
                                                   ((1, 2, 4), 3, 97, 2, 33)])
def test_hash_bit_exact(orders, heads, rows, B, T):
    note(f"engram hash orders={orders} heads={heads} rows={rows} B={B} T={T}")
    h = NgramHash(VOCAB, orders, heads, rows, seed=0, canon=torch.arange(VOCAB)).to(DEV)
    g = torch.Generator().manual_seed(T)
    c = torch.randint(0, h.pad + 1, (B, h.history + T), generator=g)
    got = h(c.to(DEV)).cpu().numpy()
    np.testing.assert_array_equal(got, E.ngram_rows(c.numpy(), h.mult.cpu().numpy(), orders, heads, rows))
    big = torch.randint(2 ** 40, 2 ** 62, (1, h.history + 7), generator=g)   # wrap-around products
    np.testing.assert_array_equal(h(big.to(DEV)).cpu().numpy(),
                                  E.ngram_rows(big.numpy(), h.mult.cpu().numpy(), orders, heads, rows))


@pytest.mark.parametrize("dtype,D", [(torch.float32, 24), (torch.bfloat16, 24), (torch.float32, 5),
                                     (torch.bfloat16, 13), (torch.bfloat16, 8)])
def test_row_gather_bit_exact(dtype, D):
    note(f"row gather {dtype} D={D}")
    g = torch.Generator().manual_seed(D)
    table = torch.randn(777, D, generator=g).to(DEV, dtype)
    rows = torch.randint(0, 777, (5, 9, 16), generator=g).to(DEV)
    out = K.row_gather(rows, table)
    assert out.shape == (5, 9, 16, D) and torch.equal(out, table[rows])
    bad = torch.tensor([3, 777, -1], device=DEV)
    o2 = K.row_gather(bad, table).float().cpu()
    assert torch.equal(o2[0], table[3].float().cpu()) and torch.isnan(o2[1:]).all()


def _module_params(m):
    return {"values": m.values.weight, "w_k": m.w_k.weight, "w_v": m.w_v.weight, "h_norm": m.h_norm.weight,
            "k_norm": m.k_norm.weight, "v_norm": m.v_norm.weight, "conv": m.conv.weight}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@torch.no_grad()
def test_module_forward_against_fp64_oracle(dtype):
    note(f"engram module {dtype}")
    torch.manual_seed(1)
    m = EngramMemory(64, 16, 24, 53, conv_kernel=4, dilation=3).to(DEV)
    m.conv.weight.normal_(std=0.3)
    m = m.to(dtype)
    p = {k: v.detach().double().cpu() for k, v in _module_params(m).items()}
    g = torch.Generator().manual_seed(2)
    h = torch.randn(2, 21, 64, generator=g)
    rows = torch.randint(0, 53, (2, 21, 16), generator=g) + torch.arange(16) * 53
    ref, _ = E.engram_forward(p, h.to(dtype).double(), rows, 1e-5, 3)
    cache = {}
    got = torch.cat([m(h[:, a:a + n].to(DEV, dtype), rows[:, a:a + n].to(DEV), cache)
                     for a, n in ((0, 9), (9, 1), (10, 11))], 1)
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    err = float((got.double().cpu() - ref).abs().max())
    assert err <= tol * float(ref.abs().max()), err


def _tiny(value_grad="row_sparse", seed=0, head_dim=24):
    cfg = ModelConfig(vocab_size=VOCAB, d_model=32, n_layers=4, n_heads=4, ffn_hidden=64, max_seq_len=64,
                      eng_layers=[0, 2], eng_heads=2, eng_head_dim=head_dim, eng_rows=101, eng_value_grad=value_grad)
    torch.manual_seed(seed)
    m = Transformer(cfg, ngram_canon=torch.arange(VOCAB))
    with torch.no_grad():
        for e in m.engram_layers():
            e.conv.weight.normal_(std=0.3)
    return m.to(DEV)


@torch.no_grad()
def test_model_cached_chunks_match_full_forward_and_causal():
    """tests/test_engram.py:58-78 on the GPU: cached chunks (hash history and conv past in the caches) give the
    full forward; changing later tokens leaves earlier logits alone."""
    note("engram model chunks")
    m = _tiny().eval()
    x = torch.randint(0, VOCAB, (2, 30), generator=torch.Generator().manual_seed(3)).to(DEV)
    full = m(x)
    caches = [dict() for _ in range(m.cfg.n_layers)]
    steps = [m(x[:, a:a + n], kv_caches=caches, pos0=a) for a, n in ((0, 7), (7, 1), (8, 1), (9, 12), (21, 9))]
    torch.testing.assert_close(torch.cat(steps, 1), full, rtol=1e-4, atol=1e-4)
    y = x.clone()
    y[:, 20:] = (y[:, 20:] + 1) % VOCAB
    torch.testing.assert_close(m(y)[:, :20], full[:, :20], rtol=0, atol=0)
    ids = m.generate(x[:, :9], 6)                           # eager steps (Engram decodes without graphs)
    assert ids.shape == (2, 7)
    cur = x[:, :9]
    for t in range(7):                                      # greedy tokens = argmax of full forwards
        nxt = m(cur)[:, -1].argmax(-1)
        assert torch.equal(nxt, ids[:, t])
        cur = torch.cat([cur, nxt[:, None]], 1)


def test_row_sparse_training_matches_fp64_autograd():
    """loss.backward() through the hash rows: the value tables' RowStore accumulators equal fp64 autograd of the
    oracle module (1e-5), touched flags are exactly the read rows, w_k's gradient too; value_grad="dense" gives
    the same table gradient as a dense .grad."""
    note("engram training")
    m = _tiny()
    e = m.engram_layers()[0]
    B, T = 2, 17
    g = torch.Generator().manual_seed(5)
    h = torch.randn(B, T, 32, generator=g)
    c = torch.randint(0, VOCAB, (B, 2 + T), generator=g)
    rows = m.ngram(c.to(DEV))
    G = torch.randn(B, T, 32, generator=g)
    (e(h.to(DEV), rows) * G.to(DEV)).sum().backward()
    p = {k: v.detach().double().cpu().requires_grad_(True) for k, v in _module_params(e).items()}
    y, _ = E.engram_forward(p, h.double(), rows.cpu(), 1e-5, 3)
    (y * G.double()).sum().backward()
    st = e.values.weight.row_store
    scale = float(p["values"].grad.abs().max())
    assert float((st.acc.double().cpu() - p["values"].grad).abs().max()) <= 1e-5 * scale
    read = torch.zeros(e.values.weight.shape[0], dtype=torch.bool)
    read[rows.reshape(-1).cpu()] = True
    assert torch.equal(st.touched.cpu(), read)
    assert e.values.weight.grad is None
    gk = float(p["w_k"].grad.abs().max())
    assert float((e.w_k.weight.grad.double().cpu() - p["w_k"].grad).abs().max()) <= 1e-5 * gk
    md = _tiny("dense")
    ed = md.engram_layers()[0]
    (ed(h.to(DEV), rows) * G.to(DEV)).sum().backward()
    assert float((ed.values.weight.grad.double().cpu() - p["values"].grad).abs().max()) <= 1e-5 * scale


# ---------------------------------------------------------------------------------------- gate and convolution kernel
MIX_SHAPES = [(1, 1, 8, 4, 3), (2, 31, 64, 4, 3), (3, 32, 384, 4, 3), (1, 33, 384, 4, 3), (2, 70, 512, 4, 10), (2, 41, 120, 1, 1),
              (2, 100, 72, 2, 32), (1, 8, 512, 3, 16)]


def _mix_inputs(B, T, d, taps, dtype, seed=0):
    g = torch.Generator().manual_seed(seed + T + d)
    h, k, v = (torch.randn(B, T, d, generator=g) for _ in range(3))
    w = [torch.rand(d, generator=g) + 0.5 for _ in range(3)] + [torch.randn(d, 1, taps, generator=g) * 0.4]
    return ([h.to(DEV, dtype)] + [t.to(DEV, torch.bfloat16) for t in (k, v)] + [t.to(DEV, dtype) for t in w])


def _mix64(h, k, v, wh, wk, wv, conv, dilation, eps, left=None):
    """(y, u of left and sequence, sum of |tap x u|) in fp64 on the CPU."""
    B, T, d = h.shape
    a = torch.sigmoid((E.rms_norm(h, wh, eps) * E.rms_norm(k, wk, eps)).sum(-1, keepdim=True) / d ** 0.5)
    past = (conv.shape[2] - 1) * dilation
    full = torch.cat([h.new_zeros(B, past, d) if left is None else left, E.rms_norm(a * v, wv, eps)], 1)
    mass = E.causal_depthwise_conv(full.abs(), conv.abs(), dilation, T)
    return torch.nn.functional.silu(E.causal_depthwise_conv(full, conv, dilation, T)) + a * v, full, mass


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,T,d,taps,dilation", MIX_SHAPES)
@pytest.mark.parametrize("cached", [False, True])
def test_engram_mix_against_fp64(B, T, d, taps, dilation, cached, dtype):
    """Per element: u is rounded to bf16 (8 bits: within 2^-8 of each tap's term, and silu's slope is below 1.1), the result to its
    type, and the fp32 arithmetic between (1e-5 of the largest value, a few hundred roundings of sums over d)."""
    note(f"engram mix B={B} T={T} d={d} taps={taps} dilation={dilation} cached={cached} {dtype}")
    args = _mix_inputs(B, T, d, taps, dtype)
    past = (taps - 1) * dilation
    left = torch.randn(B, past, d).to(DEV, torch.bfloat16) if cached else None
    y, tail = K.engram_mix(*args, dilation, 1e-5, left, keep_tail=True)
    assert torch.equal(K.engram_mix(*args, dilation, 1e-5, left), y) and y.dtype == dtype
    ref, full, mass = _mix64(*(t.double().cpu() for t in args), dilation, 1e-5,
                             None if left is None else left.double().cpu())
    bound = 1.1 * 2 ** -8 * mass + 1e-5 * ref.abs().max() + (2 ** -8 * ref.abs() if dtype == torch.bfloat16 else 0)
    assert bool(((y.double().cpu() - ref).abs() <= bound).all())
    want = full[:, full.shape[1] - past:] if past else full[:, :0]
    assert tail.shape == want.shape
    assert bool(((tail.double().cpu() - want).abs() <= 2 ** -8 * want.abs() + 1e-5).all())


@pytest.mark.parametrize("B,T,d,taps,dilation", MIX_SHAPES)
def test_engram_mix_gradient_against_fp64(B, T, d, taps, dilation):
    """Through the recorded node: bf16 roundings of u, of the convolution's output gradient and of dk and dv, each within
    2^-8 of its value and below 2^-9 in the mean, so 2^-7 of each gradient's norm; the same bits on every call; a gradient of the gradient."""
    note(f"engram mix gradient B={B} T={T} d={d} taps={taps} dilation={dilation}")
    from smlm_hip.engram import _Mix
    args = [t.requires_grad_() for t in _mix_inputs(B, T, d, taps, torch.float32, 5)]
    gy = torch.randn(B, T, d, generator=torch.Generator().manual_seed(9)).to(DEV)
    ref_args = [t.detach().double().cpu().requires_grad_() for t in args]
    ref = torch.autograd.grad(_mix64(*ref_args, dilation, 1e-5)[0], ref_args, gy.double().cpu())
    got = torch.autograd.grad(_Mix.apply(*args, dilation, 1e-5), args, gy)
    for name, a, b, x in zip(("h", "k", "v", "wh", "wk", "wv", "conv"), got, ref, args):
        assert a.dtype == x.dtype and a.shape == x.shape
        err = float((a.double().cpu() - b).norm() / b.norm())
        assert err <= 2 ** -7, (name, err)
    again = torch.autograd.grad(_Mix.apply(*args, dilation, 1e-5), args, gy)
    assert all(torch.equal(a, b) for a, b in zip(got, again))
    first = torch.autograd.grad(_Mix.apply(*args, dilation, 1e-5), args[0], gy, create_graph=True)[0]
    second = torch.autograd.grad(first.square().sum(), args[1])[0]
    f64 = torch.autograd.grad(_mix64(*ref_args, dilation, 1e-5)[0], ref_args[0], gy.double().cpu(), create_graph=True)[0]
    s64 = torch.autograd.grad(f64.square().sum(), ref_args[1])[0]
    assert float((second.double().cpu() - s64).norm()) <= 2 ** -4 * float(s64.norm())   # twice through bf16 ops


def test_engram_module_takes_the_kernel_or_the_ops():
    """The module's forward with and without the kernel: the same numbers within bf16, its results' types and cache; hooks,
    other autocast types, forward-mode and recorded bf16 weights keep the PyTorch ops."""
    note("engram module routes")
    torch.manual_seed(3)
    m = EngramMemory(64, 16, 24, 53).to(DEV)
    m.conv.weight.data.normal_(std=0.3)
    h, rows = torch.randn(2, 40, 64, device=DEV), torch.randint(0, 53, (2, 40, 16), device=DEV)
    calls = []
    real = K.engram_mix
    ops = EngramMemory.gated_value

    def count(f, *a):
        K.engram_mix = lambda *x, **kw: (calls.append(1), real(*x, **kw))[1]
        try:
            calls.clear()
            return f(*a), len(calls)
        finally:
            K.engram_mix = real

    with torch.autocast("cuda", dtype=torch.bfloat16):
        (y, n), hook = count(m, h, rows), m.k_norm.register_forward_hook(lambda *a: None)
        (z, n2) = count(m, h, rows)
        hook.remove()
    assert (n, n2) == (1, 0) and y.dtype == z.dtype and y.requires_grad and z.requires_grad
    assert float((y - z).norm()) <= 2 ** -6 * float(z.norm())
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16):
        assert count(m, h, rows)[1] == 0
    assert count(m, h, rows)[1] == 0                                        # fp32 without autocast
    b = EngramMemory(64, 16, 24, 53).to(DEV)
    b.load_state_dict(m.state_dict())
    b = b.to(torch.bfloat16)
    assert count(b, h.bfloat16(), rows)[1] == 0                             # its weights record
    with torch.no_grad():
        caches = {}, {}
        outs = []
        for cache, kernel in zip(caches, (True, False)):
            hook = None if kernel else b.v_norm.register_forward_hook(lambda *a: None)
            parts = [count(b, h[:, s:e].bfloat16(), rows[:, s:e], cache) for s, e in ((0, 3), (3, 4), (4, 40))]
            assert [c for _, c in parts] == ([1] * 3 if kernel else [0] * 3)
            outs.append(torch.cat([p for p, _ in parts], 1))
            hook and hook.remove()
        assert outs[0].dtype == outs[1].dtype
        assert float((outs[0] - outs[1]).float().norm()) <= 2 ** -6 * float(outs[1].float().norm())
        assert caches[0]["eng_u"].shape == caches[1]["eng_u"].shape and caches[0]["eng_u"].dtype == caches[1]["eng_u"].dtype
        with torch.autograd.forward_ad.dual_level():
            assert count(b, h.bfloat16(), rows)[1] == 0
    assert EngramMemory.gated_value is ops


def test_engram_module_under_a_global_hook():
    """A hook on every module sees the norms and the convolution."""
    note("engram module under a global hook")
    from torch.nn.modules.module import register_module_forward_hook
    m = EngramMemory(64, 16, 24, 53).to(DEV)
    h, rows, seen = torch.randn(2, 40, 64, device=DEV), torch.randint(0, 53, (2, 40, 16), device=DEV), []
    handle = register_module_forward_hook(lambda mod, args, out: seen.append(mod))
    try:
        with torch.autocast("cuda", dtype=torch.bfloat16):
            m(h, rows)
    finally:
        handle.remove()
    assert {m.h_norm, m.k_norm, m.v_norm, m.conv} <= set(seen)


class _Subclass(torch.Tensor):
    pass


@torch.no_grad()
@pytest.mark.parametrize("name", ["w_k", "w_v"])
def test_engram_module_with_subclassed_projection_weights(name):
    """A projection whose weight is a tensor subclass (which may hold its values elsewhere) is called as a module."""
    note(f"engram module with a subclassed {name}")
    m = EngramMemory(128, 16, 24, 53).to(DEV, torch.bfloat16)
    lin, seen = getattr(m, name), []
    lin.weight = torch.nn.Parameter(lin.weight.detach().as_subclass(_Subclass))
    assert type(lin.weight) is _Subclass
    real = K.prompt_linear
    K.prompt_linear = lambda x, w, *a: (seen.append(type(w)), real(x, w, *a))[1]
    try:
        m(torch.randn(2, 128, 128, device=DEV).bfloat16(), torch.randint(0, 53, (2, 128, 16), device=DEV))
    finally:
        K.prompt_linear = real
    assert _Subclass not in seen


class _Doubled(torch.nn.Linear):
    def forward(self, x):
        return 2 * super().forward(x)


@torch.no_grad()
@pytest.mark.parametrize("how", ["class", "instance"])
def test_engram_module_with_a_projection_of_its_own(how):
    """A projection with another forward than nn.Linear's, by its class or put on the module, is called: the result of
    the doubled weight, up to bf16."""
    note(f"engram module with a projection of its own: {how}")
    torch.manual_seed(2)
    m = EngramMemory(128, 16, 24, 53).to(DEV, torch.bfloat16)
    m.conv.weight.normal_(std=0.3)
    h, rows = torch.randn(2, 128, 128, device=DEV).bfloat16(), torch.randint(0, 53, (2, 128, 16), device=DEV)
    plain, w = m.w_v, m.w_v.weight.detach().clone()
    plain.weight.mul_(2)
    ref = m(h, rows).float()
    plain.weight.copy_(w)
    if how == "class":
        m.w_v = _Doubled(384, 128, bias=False).to(DEV, torch.bfloat16)
        m.w_v.weight.copy_(w)
    else:
        plain.forward = lambda x: 2 * torch.nn.Linear.forward(plain, x)
    assert float((m(h, rows).float() - ref).norm()) <= 2 ** -6 * float(ref.norm())
