"""Dense prefill attention on 128-query blocks (attention_dense.hip): the three
modes of attn_varlen at sizes past its dispatch line, and SelectiveMHA's prefill
over batch rows with 64- and 128-query blocks, against the attention formula in
fp64 (computed per head on the GPU).  bf16 outputs: the stated rtol / atol 2e-2."""
import pytest
import torch

from selective_attention.ops import attn_varlen, selective_mha_prefill
from tests.helpers import assert_parity


def attend(q, k, v, bias, mode):
    """fp64 (Lq, D) attention of one head; key j of `bias` is not applied on the
    query's own key ("cross": on key 0)."""
    s = q.double() @ k.double().T * q.shape[-1] ** -0.5
    if bias is not None:
        b = bias.double()[None, :].expand(s.shape).clone()
        if mode == "cross":
            b[:, :1] = 0.0
        else:
            b.fill_diagonal_(0.0)
        s = s + b
    if mode == "causal":
        s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), float("-inf"))
    return torch.softmax(s, -1) @ v.double() if k.shape[0] else torch.zeros_like(q, dtype=torch.float64)


def cu_of(lens):
    return torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("mode", ["causal", "full", "cross"])
@pytest.mark.parametrize("biased", [False, True])
def test_packed_modes(mode, D, biased):
    H, lens = 4, [16000, 1, 127, 128, 129, 65, 0, 63, 200]
    klens = [300, 1, 0, 64, 65, 31, 5, 33, 129] if mode == "cross" else lens
    g = torch.Generator(device="cuda").manual_seed(D)
    r = lambda n: torch.randn(n, H, D, generator=g, device="cuda").bfloat16()
    q, k, v = r(sum(lens)), r(sum(klens)), r(sum(klens))
    bias = None
    if biased:
        bias = 2.0 * torch.randn(H, sum(klens), generator=g, device="cuda")
        bias = bias.masked_fill(torch.rand(bias.shape, generator=g, device="cuda") < 0.1, float("-inf"))
    cu, cuk = cu_of(lens), cu_of(klens)
    o = attn_varlen(q, k, v, cu, mode, cuk if mode == "cross" else None, bias)
    a = e = 0
    for n, m in zip(lens, klens):
        for h in range(H if n < 1000 else 1):
            # the long sequence: its first, middle and last query blocks
            for i in ([0] if n < 1000 else [0, 7936, n - 130]):
                j = min(n, i + 300)
                hi = j if mode == "causal" else m
                qs = torch.zeros(hi, D, device="cuda", dtype=torch.bfloat16)
                if mode == "cross":
                    want = attend(q[a + i:a + j, h], k[e:e + m, h], v[e:e + m, h],
                                  None if bias is None else bias[h, e:e + m], mode)
                else:
                    qs[:min(hi, n)] = q[a:a + min(hi, n), h]
                    want = attend(qs, k[e:e + hi, h], v[e:e + hi, h],
                                  None if bias is None else bias[h, e:e + hi], mode)[i:j]
                assert_parity(o[a + i:a + j, h], want.cpu(), torch.bfloat16, f"{mode} n={n} h={h} i={i}")
        a, e = a + n, e + m
    assert torch.equal(o, attn_varlen(q, k, v, cu, mode, cuk if mode == "cross" else None, bias))


@pytest.mark.gpu
@pytest.mark.parametrize("b,H,L,D,lens", [
    (1, 2, 1, 64, None), (2, 2, 64, 64, [64, 63]), (3, 2, 130, 128, [130, 0, 129]),
    (2, 3, 200, 64, [1, 128]), (2, 16, 2100, 64, [2100, 1999]), (4, 32, 515, 128, [515, 130, 257, 64]),
])
def test_rows(b, H, L, D, lens):
    """The last two take 128-query blocks, the others 64."""
    g = torch.Generator(device="cuda").manual_seed(L)
    q, k, v = (torch.randn(b, L, H, D, generator=g, device="cuda").bfloat16().transpose(1, 2)
               for _ in range(3))
    lg = torch.log(torch.sigmoid(torch.randn(b, H, L, generator=g, device="cuda") + 1))
    lg = lg.masked_fill(torch.rand(b, H, L, generator=g, device="cuda") < 0.2, float("-inf"))
    lt = None if lens is None else torch.tensor(lens).cuda()
    o = selective_mha_prefill(q, k, v, lg, lt)
    assert o.shape == (b, H, L, D) and o.transpose(1, 2).is_contiguous()
    for i in range(b):
        n = L if lens is None else lens[i]
        assert not o[i, :, n:].any()
        for h in range(0, H, max(1, H // 4)):
            if n:
                want = attend(q[i, h, :n], k[i, h, :n], v[i, h, :n], lg[i, h, :n], "causal")
                assert_parity(o[i, h, :n], want.cpu(), torch.bfloat16, f"row {i} head {h}")
    # any other layout is copied: the same bits
    assert torch.equal(o, selective_mha_prefill(q.contiguous(), k, v.contiguous(), lg, lt))


def test_prefill_entry_refuses_misaligned_rows():
    """The kernel moves rows 16 bytes at a time; an odd pointer is an error, not a
    launch (the addresses are never read: the checks come first)."""
    from selective_attention import _lib
    lib = _lib.load()
    for bad in range(5):
        p = [0x1000 * (i + 1) for i in range(5)]   # q, k, v, log_gate, o
        p[bad] += 2
        q, k, v, lg, o = p
        rc = lib.sa_mha_prefill_fwd(_lib.DTYPE_BF16, q, k, v, lg, None, 0, 64, 4, 64, -1.0, o, None)
        assert (rc != 0) == (bad != 3), bad
        if rc:
            assert b"aligned" in lib.sa_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("off", [1, 4, 8])
def test_rows_off_a_16_byte_boundary(off):
    """Contiguous views `off` elements into a buffer: the aligned call's bits."""
    b, H, L, D = 2, 3, 150, 64
    g = torch.Generator(device="cuda").manual_seed(off)

    def odd(t):
        return torch.empty(t.numel() + off, device="cuda", dtype=t.dtype)[off:].view(t.shape).copy_(t)
    q, k, v = (torch.randn(b, L, H, D, generator=g, device="cuda").bfloat16() for _ in range(3))
    lg = -torch.rand(b, H, L, generator=g, device="cuda")
    want = selective_mha_prefill(*(t.transpose(1, 2) for t in (q, k, v)), lg)
    assert torch.equal(want, selective_mha_prefill(*(odd(t).transpose(1, 2) for t in (q, k, v)), odd(lg)))
    n, Hn = 4200, 16      # a packed launch of the same kernel
    q, k, v = (torch.randn(n, Hn, D, generator=g, device="cuda").bfloat16() for _ in range(3))
    bias = -torch.rand(Hn, n, generator=g, device="cuda")
    assert torch.equal(attn_varlen(q, k, v, cu_of([n]), "full", None, bias),
                       attn_varlen(odd(q), odd(k), odd(v), cu_of([n]), "full", None, odd(bias)))


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
def test_nan_and_infinite_rows(D):
    """A query, key or value that is not a number shows in every row that meets
    it and in no other: rows of one half tile (0, 5, 31) and of several."""
    b, H, L = 1, 4, 200
    g = torch.Generator(device="cuda").manual_seed(D)
    base = [torch.randn(b, L, H, D, generator=g, device="cuda").bfloat16() for _ in range(3)]
    lg = -torch.rand(b, H, L, generator=g, device="cuda")
    run = lambda q, k, v: selective_mha_prefill(*(t.transpose(1, 2) for t in (q, k, v)), lg).transpose(1, 2)
    clean = run(*base)
    for row in (0, 5, 31, 32, 130):
        q = base[0].clone()
        q[0, row, 1, 3] = float("nan")
        o = run(q, *base[1:])
        assert o[0, row, 1].isnan().all()
        o[0, row, 1] = clean[0, row, 1]
        torch.testing.assert_close(o, clean, rtol=2e-2, atol=2e-2)
        for value in (float("nan"), float("inf")):   # (inf - inf in the softmax)
            k = base[1].clone()
            k[0, row, 1, 3] = value
            o = run(base[0], k, base[2])
            hit = base[0][0, row:, 1, 3] > 0 if value > 0 else torch.ones(L - row, dtype=torch.bool, device="cuda")
            assert o[0, row:, 1][hit].isnan().all()
            torch.testing.assert_close(o[0, :row], clean[0, :row], rtol=2e-2, atol=2e-2)
    # packed: a sequence of one half tile, and a cross range of few keys
    n, Hn = 4200, 16
    q, k, v = (torch.randn(n, Hn, D, generator=g, device="cuda").bfloat16() for _ in range(3))
    q[4100, 2, 0] = float("nan")
    cu = cu_of([4096, 20, 84])
    for mode, cuk in (("causal", None), ("full", None), ("cross", cu_of([4096, 20, 84]))):
        o = attn_varlen(q, k, v, cu, mode, cuk)
        assert o[4100, 2].isnan().all() and int(o.isnan().any(-1).sum()) == 1, mode


@pytest.mark.gpu
@pytest.mark.parametrize("low", [torch.finfo(torch.float32).min, -1e30])
def test_biases_of_the_lowest_value(low):
    """A mask written as a huge finite bias drops its keys as -inf does."""
    b, H, L, D = 2, 2, 150, 64
    g = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (torch.randn(b, L, H, D, generator=g, device="cuda").bfloat16().transpose(1, 2) for _ in range(3))
    drop = torch.rand(b, H, L, generator=g, device="cuda") < 0.5
    lg = -torch.rand(b, H, L, generator=g, device="cuda")
    want = selective_mha_prefill(q, k, v, lg.masked_fill(drop, float("-inf")))
    assert torch.equal(selective_mha_prefill(q, k, v, lg.masked_fill(drop, low)), want)


@pytest.mark.gpu
@pytest.mark.parametrize("D,L,H", [(64, 300, 4), (128, 300, 4), (64, 4200, 16)])
def test_a_row_does_not_see_its_neighbours(D, L, H):
    """Other queries of the same tile, whose scores rise far above theirs (or are
    no numbers), leave a row's bits alone."""
    g = torch.Generator(device="cuda").manual_seed(L)
    q, k, v = (torch.randn(1, L, H, D, generator=g, device="cuda").bfloat16() for _ in range(3))
    lg = -torch.rand(1, H, L, generator=g, device="cuda")
    run = lambda q: selective_mha_prefill(*(t.transpose(1, 2) for t in (q, k, v)), lg).transpose(1, 2)
    clean, rows = run(q), torch.arange(3, L, 7, device="cuda")
    keep = torch.ones(L, dtype=torch.bool, device="cuda").index_fill(0, rows, False)
    for other in (20.0 * q[:, rows], -20.0 * q[:, rows], float("nan") * q[:, rows]):
        mixed = q.clone()
        mixed[:, rows] = other
        assert torch.equal(run(mixed)[:, keep], clean[:, keep])


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1e-39, 1e-36, 1e-6, 1.0])
def test_any_softmax_scale(scale):
    """Down to scales whose reciprocal leaves the range: only the biases count."""
    H, n, D = 16, 4200, 64
    g = torch.Generator(device="cuda").manual_seed(5)
    q, k, v = (torch.randn(n, H, D, generator=g, device="cuda").bfloat16() for _ in range(3))
    bias = 300.0 * torch.rand(H, n, generator=g, device="cuda")
    o = attn_varlen(q, k, v, cu_of([n]), "full", None, bias, scale)
    for h in (0, 9):
        s = q[:200, h].double() @ k[:, h].double().T * scale + bias[h].double()
        i = torch.arange(200, device="cuda")
        s[i, i] -= bias[h, :200].double()
        assert_parity(o[:200, h], (torch.softmax(s, -1) @ v[:, h].double()).cpu(), torch.bfloat16, f"head {h}")
