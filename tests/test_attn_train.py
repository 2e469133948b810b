"""SelectiveMHA's training attention on the fp32 kernels (sa_gated_attn_train_fwd
/ _bwd): outputs and gradients against the dense form in fp64 (the formula of
modules/selective_attention.py:86-95, 125-144) at the edges of the 64-row
tiles, with dropped keys, for strided and misaligned inputs; the dispatch
between kernels and the dense form; second derivatives.

Tolerance: every output is a sum of at most n products of fp32 values with
fp32 rounding, and each softmax weight carries the rounding of its score
(|s| <= 32 here, so 32 * 2^-24 = 1.9e-6 relative); the 2-norm over a tensor
stays below 4 * 1.9e-6 < 1e-5.
"""
import pytest
import torch

from selective_attention.ops import gated_attention_train
from selective_attention.ops import selective_mha as M

REL = 1e-5


def inputs(b, H, L, D, dtype=torch.float32, device="cuda", seed=0):
    g = torch.Generator().manual_seed(seed)
    q, k, v, do = (torch.randn(b, H, L, D, generator=g).to(dtype).to(device) for _ in range(4))
    lg = torch.log(torch.sigmoid(torch.randn(b, H, L, generator=g) + 2.0))
    lg = lg.masked_fill(torch.rand(b, H, L, generator=g) < 0.2, float("-inf")).to(device)
    return q, k, v, lg, do.float()


def grads(fn, ts, do, dtype=None):
    leaves = [(t if dtype is None else t.to(dtype)).detach().requires_grad_(True) for t in ts]
    out = fn(*leaves)
    return (out,) + torch.autograd.grad(out, leaves, do.to(out.dtype))


def check(got, want, rel=REL):
    for name, a, e in zip(("out", "dq", "dk", "dv", "dlog_gate"), got, want):
        a, e = a.detach().double(), e.detach().double()
        assert torch.isfinite(a).all(), name
        err = float((a - e).norm() / e.norm().clamp(min=1e-30)) if float(e.norm()) else float(a.norm())
        assert err < rel, (name, err)


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("b,H,L,D", [(1, 1, 1, 64), (2, 3, 63, 64), (1, 2, 64, 32), (2, 2, 65, 96),
                                     (1, 2, 129, 128), (3, 5, 200, 64), (2, 4, 577, 64)])
def test_kernels_match_fp64(b, H, L, D, causal):
    *ts, do = inputs(b, H, L, D, seed=L)
    assert M._train_kernel_ok(*ts)
    got = grads(lambda *t: gated_attention_train(*t, causal), ts, do)
    want = grads(lambda *t: M._gated_attention_dense(*t, causal), ts, do, torch.float64)
    check(got, want)
    again = grads(lambda *t: gated_attention_train(*t, causal), ts, do)
    assert all(torch.equal(a, e) for a, e in zip(got, again))


@pytest.mark.gpu
def test_strides_dtypes_and_alignment():
    b, H, L, D = 2, 3, 70, 64
    q, k, v, lg, do = inputs(b, H, L, D, seed=9)
    want = grads(lambda *t: M._gated_attention_dense(*t, True), (q, k, v, lg), do, torch.float64)
    swap = lambda t: t.transpose(1, 2).contiguous().transpose(1, 2)      # (b, L, H, D) memory
    odd = torch.empty(b * H * L * D + 1, device="cuda")[1:].view(b, H, L, D).copy_(k)
    check(grads(gated_attention_train, (swap(q), odd, swap(v), lg), swap(do)), want)
    # an upstream gradient of stride 0 (a plain sum) and rows past alignment
    ones = torch.ones((), device="cuda").expand(b, H, L, D)
    wide = torch.zeros(b, H, L, D + 1, device="cuda")
    wide[..., :D] = v
    check(grads(gated_attention_train, (q, k, wide[..., :D], lg), ones),
          grads(lambda *t: M._gated_attention_dense(*t, True), (q, k, v, lg), ones, torch.float64))
    # bf16 inputs: fp32 inside, gradients rounded once to bf16
    qb = [t.bfloat16() for t in (q, k, v)]
    want = grads(lambda *t: M._gated_attention_dense(*t, True), (*qb, lg), do, torch.float64)
    got = grads(gated_attention_train, (*qb, lg), do)
    assert got[0].dtype == torch.float32 and got[1].dtype == torch.bfloat16
    check(got[:1] + got[4:], want[:1] + want[4:])
    check(got, want, 2 ** -8)


@pytest.mark.gpu
def test_dense_form_where_the_kernels_do_not_apply():
    q, k, v, lg, do = inputs(2, 2, 40, 64, seed=3)
    want = M._gated_attention_dense(q, k, v, lg, True)
    # broadcast gates, an unsupported head_dim, vmap, forward mode
    assert not M._train_kernel_ok(q, k, v, lg[:1])
    torch.testing.assert_close(gated_attention_train(q, k, v, lg[:1])[:1], want[:1])
    assert not M._train_kernel_ok(q[..., :48], k[..., :48], v[..., :48], lg)
    assert torch.isfinite(gated_attention_train(q[..., :48], k[..., :48], v[..., :48], lg)).all()
    vm = torch.vmap(gated_attention_train)(*(t[None] for t in (q, k, v, lg)))
    torch.testing.assert_close(vm[0], want, rtol=1e-5, atol=1e-5)
    _, jvp = torch.func.jvp(lambda x: gated_attention_train(x, k, v, lg), (q,), (do,))
    eps = 1e-3
    f = lambda x: M._gated_attention_dense(x.double(), k.double(), v.double(), lg.double(), True)
    torch.testing.assert_close(jvp.double(), (f(q + eps * do) - f(q - eps * do)) / (2 * eps),
                               rtol=1e-2, atol=1e-2)


@pytest.mark.gpu
def test_second_derivative_matches_dense():
    q, k, v, lg, do = inputs(1, 2, 30, 64, seed=5)

    def second(fn, dtype):
        ts = [t.to(dtype).requires_grad_(True) for t in (q, k, v, lg)]
        out = fn(*ts)
        g = torch.autograd.grad(out, ts[:3], do.to(out.dtype), create_graph=True)
        return torch.autograd.grad(sum((x * x).sum() for x in g), ts)
    got = second(gated_attention_train, torch.float32)
    want = second(lambda *t: M._gated_attention_dense(*t, True), torch.float64)
    for a, e in zip(got, want):
        assert float((a.double() - e).norm() / e.norm()) < 1e-4


def test_dense_form_on_the_cpu():
    q, k, v, lg, do = inputs(1, 2, 20, 64, device="cpu", seed=6)
    assert not M._train_kernel_ok(q, k, v, lg)
    check(grads(gated_attention_train, (q, k, v, lg), do),
          grads(lambda *t: M._gated_attention_dense(*t, True), (q, k, v, lg), do, torch.float64))
