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


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,b,H,Lq,Lk,D,causal,ql,kl", [
    (torch.float32, 2, 2, 1, 1, 64, True, None, None),
    (torch.float32, 2, 3, 255, 255, 64, True, [255, 130], [255, 130]),
    (torch.float32, 1, 2, 257, 257, 128, True, None, None),
    (torch.bfloat16, 3, 2, 600, 600, 64, True, [600, 256, 0], [600, 256, 0]),
    (torch.float32, 2, 2, 2500, 2500, 32, True, [2500, 1030], [2400, 1100]),
    (torch.bfloat16, 2, 2, 70, 300, 96, False, None, [300, 17]),
    (torch.float32, 1, 3, 530, 65, 64, False, [400], [65]),
])
def test_score_std_through_gram_matrices(dtype, b, H, Lq, Lk, D, causal, ql, kl):
    """Counts exact; std and its gradient against the fp64 oracle at the edges of
    the 64-row tiles and 256-row chunks, on vectors that share little (for what
    cancels see test_score_std_with_common_components).  The scores are fp32
    products of at most 128 terms, (128 / 4)^0.5 * 2^-24 = 3e-7 of the score,
    and a tile's gradient sum the same; 1e-5 leaves room for single entries."""
    from oracle import attn as ref
    g = torch.Generator().manual_seed(Lq)
    q = (torch.randn(b, H, Lq, D, generator=g) + 0.2).to(dtype)
    k = (torch.randn(b, H, Lk, D, generator=g) + 0.1).to(dtype)
    go = torch.randn(H, generator=g)
    lens = [None if x is None else torch.tensor(x) for x in (ql, kl)]
    dev = [None if x is None else x.cuda() for x in lens]
    qd, kd = q.cuda().requires_grad_(True), k.cuda().requires_grad_(True)
    std = M.ScoreStdFn.apply(qd, kd, *dev, causal)
    stats, _ = M.score_moments(qd.detach(), kd.detach(), *dev, causal)
    got = torch.autograd.grad(std, (qd, kd), go.cuda(), retain_graph=True)
    q64, k64 = q.double().requires_grad_(True), k.double().requires_grad_(True)
    want_stats = ref.score_stats(q64, k64, D ** -0.5, *lens, causal)
    want = ref.score_std(want_stats)
    assert torch.equal(stats[:, 0].cpu(), want_stats[:, 0].detach())
    torch.testing.assert_close(std.detach().cpu().double(), want.detach(), rtol=1e-5, atol=1e-6)
    wg = torch.autograd.grad(want, (q64, k64), go.double())
    rel = 1e-5 if dtype == torch.float32 else 2 ** -8
    if float(want.detach().min()) > 1e-3:      # (a single pair has std 0: no gradient)
        for a, e in zip(got, wg):
            assert float((a.double().cpu() - e).norm() / e.norm()) < rel
    else:
        assert all(float(a.abs().max()) < 1e-3 for a in got)
    # a recorded backward takes the torch form: the same gradients
    rec = torch.autograd.grad(std, (qd, kd), go.cuda(), create_graph=True)
    for a, e in zip(got, rec):
        assert rec[0].requires_grad
        torch.testing.assert_close(a.float(), e.detach().float(), rtol=2 * rel, atol=1e-6)


def test_dense_form_on_the_cpu():
    q, k, v, lg, do = inputs(1, 2, 20, 64, device="cpu", seed=6)
    assert not M._train_kernel_ok(q, k, v, lg)
    check(grads(gated_attention_train, (q, k, v, lg), do),
          grads(lambda *t: M._gated_attention_dense(*t, True), (q, k, v, lg), do, torch.float64))


def _dependent(kind):
    """Calls of gated_attention_train in which one input is made of another."""
    if kind == "gate of q and k":
        return lambda fn, q, k, v, lg: fn(q, k, v, lg + (q * k).sum(-1))
    if kind == "one tensor for q, k and v":
        return lambda fn, q, k, v, lg: fn(q, q, q, lg)
    # (0.1 q keeps a query's own score near the others: at 2 q its weight is 1 to
    # within 1e-4, and dq, a difference of such weights, loses four digits in the
    # dense fp32 form too)
    return lambda fn, q, k, v, lg: fn(q, 0.1 * q, v + k, lg)


@pytest.mark.parametrize("kind", ["gate of q and k", "one tensor for q, k and v", "k of q"])
@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_recorded_backward_of_dependent_inputs(kind, device, monkeypatch):
    """First and second gradients where the inputs depend on each other, against
    the dense form: a recorded backward differentiates with respect to the
    inputs of this call alone.  On the CPU the function runs with the dense form
    in the place of the kernels."""
    q, k, v, lg, do = inputs(1, 2, 24, 64, device=device, seed=11)
    lg = lg.clamp(min=-20.0)
    fn = gated_attention_train
    if device == "cpu":
        def forward(q, k, v, lg, causal):
            return M._gated_attention_dense(q, k, v, lg, causal), torch.zeros(2, *lg.shape)
        monkeypatch.setattr(M, "gated_attn_train_forward", forward)
        fn = lambda *t: M.GatedAttnTrainFn.apply(*t, True)

    def both(fn, dtype):
        ts = [t.to(dtype).requires_grad_(True) for t in (q, k, v, lg)]
        out = _dependent(kind)(fn, *ts)
        first = torch.autograd.grad(out, ts, do.to(dtype), create_graph=True, allow_unused=True)
        first = [g for g in first if g is not None]
        second = torch.autograd.grad(sum((g * g).sum() for g in first), ts, allow_unused=True)
        return first + [g for g in second if g is not None]
    got = both(fn, torch.float32)
    want = both(lambda *t: M._gated_attention_dense(*t, True), torch.float64)
    assert len(got) == len(want)
    for a, e in zip(got, want):
        assert float(((a.double() - e).norm() / e.norm()).detach()) < 1e-4


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_batched_and_dual_upstream_gradients(device, monkeypatch):
    """A backward that is vectorised over upstream gradients, or run with a
    forward-mode tangent on one, sees the dense form's ops."""
    q, k, v, lg, do = inputs(1, 2, 24, 64, device=device, seed=12)
    lg = lg.clamp(min=-20.0)
    fn = gated_attention_train
    if device == "cpu":
        def forward(q, k, v, lg, causal):
            return M._gated_attention_dense(q, k, v, lg, causal), torch.zeros(2, *lg.shape)

        def backward(q, k, v, lg, out, stats, dout, causal):
            dout.data_ptr()
            return tuple(torch.zeros_like(t) for t in (q, k, v, lg))
        monkeypatch.setattr(M, "gated_attn_train_forward", forward)
        monkeypatch.setattr(M, "gated_attn_train_backward", backward)
        fn = lambda *t: M.GatedAttnTrainFn.apply(*t, True)
    G = torch.stack([do, 2.0 * do.flip(2), torch.zeros_like(do)])

    def run(fn, how):
        ts = [t.detach().requires_grad_(True) for t in (q, k, v, lg)]
        out = fn(*ts)
        if how == "is_grads_batched":
            return torch.autograd.grad(out, ts, G, is_grads_batched=True)
        if how == "vmap":
            return torch.vmap(lambda g: torch.autograd.grad(out, ts, g, retain_graph=True))(G)
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(G[0], G[1])
            pairs = [torch.autograd.forward_ad.unpack_dual(g) for g in torch.autograd.grad(out, ts, dual)]
            return [t for p in pairs for t in (p.primal, p.tangent)]
    for how in ("is_grads_batched", "vmap", "dual"):
        got, want = run(fn, how), run(lambda *t: M._gated_attention_dense(*t, True), how)
        for a, e in zip(got, want):
            torch.testing.assert_close(a, e, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_score_std_dual_upstream_gradient(device, monkeypatch):
    """The std's backward is linear in the upstream gradient: its tangent is the
    backward of the tangent."""
    from oracle import attn as ref
    q, k, *_ = inputs(1, 2, 24, 64, device=device, seed=13)
    if device == "cpu":
        def moments(q, k, ql, kl, causal):
            st = ref.score_stats(q.double(), k.double(), 64 ** -0.5, ql, kl, causal)
            return st, ref.score_std(st).float()
        monkeypatch.setattr(M, "score_moments", moments)
        monkeypatch.setattr(M, "score_std_backward", lambda q, k, *a: (torch.zeros_like(q), torch.zeros_like(k)))
    ts = [t.requires_grad_(True) for t in (q, k)]
    std = M.ScoreStdFn.apply(*ts)
    g, tangent = torch.tensor([1.0, -2.0], device=device), torch.tensor([0.5, 3.0], device=device)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(g, tangent)
        got = [torch.autograd.forward_ad.unpack_dual(x)
               for x in torch.autograd.grad(std, ts, dual, retain_graph=True)]
        got = [(x.primal.clone(), x.tangent.clone()) for x in got]
    for i, up in enumerate((g, tangent)):
        want = torch.autograd.grad(std, ts, up, create_graph=True)
        for x, e in zip(got, want):
            torch.testing.assert_close(x[i], e.detach(), rtol=1e-5, atol=1e-7)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D,L,causal", [(32, 600, True), (64, 2048, True), (96, 700, False),
                                        (128, 1100, True)])
@pytest.mark.parametrize("q_off,k_off,orthogonal", [(0, 0, False), (4, 4, False), (10, 10, False),
                                                    (0, 100, True), (100, 0, True)])
def test_score_std_with_common_components(q_off, k_off, orthogonal, D, L, causal, dtype):
    """Vectors with a common part, which cancels in the variance, or meets nothing
    on the other side: the std and its gradient against fp64 are no further off
    than by the pass over every pair and the dense gradient, whose sums over the
    pairs do not cancel before fp64 (or than one rounding to fp32 and the
    products' own, 4 * 2^-24; bf16 gradients 2^-8)."""
    from oracle import attn as ref
    from selective_attention.kernels.attention import score_stats
    g = torch.Generator().manual_seed(D + L)
    q, k = (torch.randn(1, 2, L, D, generator=g) for _ in range(2))
    if orthogonal:      # the other side has nothing along the common vector
        e = torch.nn.functional.normalize(torch.randn(D, generator=g), dim=0)
        q, k = (t - (t @ e)[..., None] * e for t in (q, k))
        q, k = q + q_off * e, k + k_off * e
    else:
        q, k = q + q_off * torch.randn(D, generator=g).sign(), k + k_off * torch.randn(D, generator=g).sign()
    q, k = q.to(dtype).cuda().requires_grad_(True), k.to(dtype).cuda().requires_grad_(True)
    go = torch.randn(2, generator=g).cuda()
    q64, k64 = (t.detach().cpu().double().requires_grad_(True) for t in (q, k))
    std64 = ref.score_std(ref.score_stats(q64, k64, D ** -0.5, None, None, causal))
    want = [std64] + list(torch.autograd.grad(std64, (q64, k64), go.cpu().double()))
    std = M.ScoreStdFn.apply(q, k, None, None, causal)
    got = [std] + list(torch.autograd.grad(std, (q, k), go, retain_graph=True))
    pairs = ref.score_std(score_stats(q.detach(), k.detach(), None, None, causal)).float()
    dense = [pairs] + list(torch.autograd.grad(std, (q, k), go, create_graph=True))
    errs = [[float(((a.detach().cpu().double() - e).norm() / e.norm()).detach()) for a, e in zip(x, want)]
            for x in (got, dense)]
    print([f"{x:.1e}" for x in sum(errs, [])], flush=True)
    for i, (mine, other) in enumerate(zip(*errs)):
        one = 4 * 2.0 ** -24 if dtype == torch.float32 or i == 0 else 2.0 ** -8
        assert mine <= max(1.1 * other, one), (("std", "dq", "dk")[i], mine, other)


@pytest.mark.gpu
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_score_std_past_the_lengths(value):
    """Rows outside the valid pairs hold anything: past their length, and for the
    std (whose gradient multiplies them by 0) keys that no query sees."""
    from selective_attention.kernels.attention import score_stats
    b, H, L, D = 3, 2, 900, 64
    g = torch.Generator().manual_seed(1)
    q, k = (torch.randn(b, H, L, D, generator=g).cuda() for _ in range(2))
    ql, kl = torch.tensor([900, 300, 0]).cuda(), torch.tensor([700, 600, 0]).cuda()

    def fill(x, q_len, k_len):
        a, e = q.clone(), k.clone()
        for i in range(b):
            a[i, :, int(q_len[i]):] = x
            e[i, :, int(k_len[i]):] = x
        return a.requires_grad_(True), e.requires_grad_(True)
    want = M.ScoreStdFn.apply(*fill(0.0, ql, kl), ql, kl)
    unseen = fill(value, ql, torch.minimum(ql, kl))
    assert torch.equal(M.ScoreStdFn.apply(*unseen, ql, kl), want) and torch.isfinite(want).all()
    torch.testing.assert_close(M.score_moments(*unseen, ql, kl)[0], score_stats(*unseen, ql, kl),
                               rtol=1e-6, atol=1e-2)
    grads = []
    for x in (0.0, value):
        ts = fill(x, ql, kl)
        grads.append(torch.autograd.grad(M.ScoreStdFn.apply(*ts, ql, kl).sum(), ts))
    for a, e in zip(*grads):
        assert torch.isfinite(a).all() and torch.equal(a, e)


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("L,D", [(500, 128), (2048, 64), (4096, 32)])
def test_no_further_off_than_the_dense_form(L, D, causal):
    """Long sums: every output's error against fp64 is that of the dense fp32 form
    (torch's own sums over queries and keys), within the 5 % by which one draw's
    error scatters."""
    *ts, do = inputs(1, 4, L, D, seed=L + 1)
    want = grads(lambda *t: M._gated_attention_dense(*t, causal), ts, do, torch.float64)
    errs = []
    for fn in (gated_attention_train, M._gated_attention_dense):
        got = grads(lambda *t: fn(*t, causal), ts, do)
        errs.append([float((a.detach().double() - e.detach()).norm() / e.detach().norm()) for a, e in zip(got, want)])
    print([f"{x:.2e}" for x in sum(errs, [])], flush=True)
    for name, mine, dense in zip(("out", "dq", "dk", "dv", "dlog_gate"), *errs):
        assert mine <= 1.05 * dense, (name, mine, dense)


@pytest.mark.gpu
def test_another_current_device_takes_the_dense_form(monkeypatch):
    *ts, _ = inputs(1, 2, 40, 64, seed=4)
    assert M._train_kernel_ok(*ts)
    want = M._gated_attention_dense(*ts, True)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    assert not M._train_kernel_ok(*ts)
    assert torch.equal(gated_attention_train(*ts), want)
