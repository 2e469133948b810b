"""The fp32 scan on 64-row tiles (ssd_f32.hip): forward and backward against the
fp64 oracle at the edges of its sizes (head_dim and state_dim instances, one
to four tiles a chunk, ragged rows, lengths inside and at tile boundaries,
heads per group that split into one or several shares), and the dispatch:
operands off a 16-byte boundary and sizes it does not take give the general
kernels' results."""
import pytest
import torch

from oracle import ssd as ref
from selective_attention.ops import SSDScanFn
from tests.helpers import assert_parity

F64 = torch.float64


def make(b, L, H, P, N, G, lens, init, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g)
    return dict(u=r(b, L, H, P), A=-torch.exp(torch.rand(H, generator=g) * 2.7), B=r(b, L, G, N) / 8,
                C=r(b, L, G, N) / 8, dr=r(b, L, H) - 3.0, bias=0.3 * r(H),
                h0=0.2 * r(b, H, P, N) if init else None,
                lens=None if lens is None else torch.tensor(lens), dy=r(b, L, H, P),
                dh=0.2 * r(b, H, P, N))


def run_gpu(x, chunk, move=lambda t: t.cuda()):
    names = [k for k in ("u", "A", "B", "C", "dr", "bias", "h0") if x[k] is not None]
    t = {k: move(x[k]).requires_grad_(True) for k in names}
    lens = None if x["lens"] is None else x["lens"].cuda()
    y, h = SSDScanFn.apply(t["u"], t["A"], t["B"], t["C"], t["dr"], t["bias"], t.get("h0"), lens,
                           chunk)
    gr = torch.autograd.grad((y, h), list(t.values()), (x["dy"].cuda(), x["dh"].cuda()))
    return {"y": y.detach(), "h": h.detach(), **{"d" + k: v for k, v in zip(names, gr)}}


def run_ref(x, chunk):
    b, L, H, _ = x["u"].shape
    lens = torch.full((b,), L) if x["lens"] is None else x["lens"]
    a = [x[k] if x[k] is None else x[k].to(F64) for k in ("u", "A", "B", "C", "dr", "bias", "h0")]
    y, h = ref.ssd_scan_forward(*a, lens, chunk_size=chunk)
    gr = ref.ssd_scan_backward(*a, x["dy"].to(F64), x["dh"].to(F64), lens, chunk)
    return {"y": y, "h": h, **{"d" + k: v for k, v in zip(
        ("u", "A", "B", "C", "dr", "bias", "h0"), gr) if v is not None}}


CASES = [
    # b, L, H, P, N, G, chunk, lens, init
    (1, 64, 1, 64, 64, 1, 64, None, False),
    (2, 1, 2, 64, 64, 1, 64, None, True),
    (2, 200, 4, 64, 128, 2, 128, [200, 129], True),
    (1, 333, 6, 64, 64, 2, 256, None, False),
    (2, 300, 5, 32, 32, 1, 64, [300, 64], False),
    (1, 260, 3, 128, 64, 3, 256, [255], True),
    (1, 130, 4, 128, 128, 1, 128, None, True),
    (3, 520, 16, 64, 32, 1, 256, [520, 0, 257], True),
    (1, 150, 2, 32, 128, 1, 64, [65], False),
    (2, 400, 8, 64, 64, 8, 192, [400, 383], False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("b,L,H,P,N,G,chunk,lens,init", CASES)
def test_tile_kernels_match_oracle(b, L, H, P, N, G, chunk, lens, init):
    x = make(b, L, H, P, N, G, lens, init, seed=L + H)
    got, want = run_gpu(x, chunk), run_ref(x, chunk)
    for k, v in want.items():
        assert_parity(got[k], v, torch.float32, k)
    again = run_gpu(x, chunk)
    assert all(torch.equal(got[k], again[k]) for k in got)


@pytest.mark.gpu
def test_two_heads_per_block_and_shares():
    """Sizes at which the scan takes two heads a block and dCB, dB / dC one share."""
    x = make(4, 1100, 16, 64, 64, 8, [1100, 900, 1024, 3], True, seed=3)
    got, want = run_gpu(x, 256), run_ref(x, 256)
    for k, v in want.items():
        assert_parity(got[k], v, torch.float32, k)


@pytest.mark.gpu
@pytest.mark.parametrize("P,N,chunk", [(64, 64, 128), (64, 128, 64)])
def test_misaligned_operands_take_the_general_kernels(P, N, chunk):
    x = make(2, 190, 4, P, N, 2, [190, 100], True, seed=8)

    def off(t):   # the same values one element past a 16-byte boundary
        return torch.empty(t.numel() + 1, device="cuda")[1:].view(t.shape).copy_(t)
    got, want = run_gpu(x, chunk, off), run_gpu(x, chunk)
    for k, v in want.items():
        assert_parity(got[k], v.cpu().to(F64), torch.float32, k)


@pytest.mark.gpu
@pytest.mark.parametrize("P,N,chunk", [(48, 64, 64), (64, 48, 64), (64, 64, 96), (96, 128, 50)])
def test_other_sizes_keep_the_general_kernels(P, N, chunk):
    x = make(1, 120, 2, P, N, 1, None, False, seed=4)
    got, want = run_gpu(x, chunk), run_ref(x, chunk)
    for k, v in want.items():
        assert_parity(got[k], v, torch.float32, k)


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("b,L", [(0, 64), (2, 0), (0, 0), (1, 1)])
@pytest.mark.parametrize("P,N", [(64, 64), (32, 128), (48, 64)])
def test_workspace_of_empty_sizes(dtype, b, L, P, N):
    """The workspace queries take an empty batch or sequence on every path (the
    fp32 path divides a block count of the launch among the heads)."""
    from selective_attention import _lib
    lib = _lib.load()
    nbytes = lib.sa_ssd_bwd_workspace_size(dtype, b, L, 2, P, 1, N, 64)
    lib.sa_ssd_bwd_gated_workspace_size(dtype, b, L, 2, P, 1, N, 64)
    assert (nbytes > 0) == (b * L > 0)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_empty_scans(dtype):
    """An empty sequence passes the state and its gradient through; an empty
    batch is refused, forward and backward, with an exception."""
    from selective_attention.kernels.ssd_scan import ssd_scan_backward
    x = make(2, 0, 4, 64, 64, 2, None, True, 0)
    for k in ("u", "B", "C", "dr"):
        x[k] = x[k].to(dtype)
    out = run_gpu(x, 64)
    assert not out["dA"].any() and not out["dbias"].any()
    assert torch.equal(out["h"].cpu(), x["h0"]) and torch.equal(out["dh0"].cpu(), x["dh"])
    x = make(0, 70, 4, 64, 64, 2, None, False, 0)
    t = [x[k].to(dtype if k in ("u", "B", "C", "dr") else torch.float32).cuda()
         for k in ("u", "A", "B", "C", "dr", "bias")]
    with pytest.raises(RuntimeError):
        SSDScanFn.apply(*t, None, None, 64)
    saved = [torch.empty(s, device="cuda") for s in ((0, 4, 2, 64), (0, 4, 2, 64), (0, 2, 4, 64, 64))]
    with pytest.raises(RuntimeError):
        ssd_scan_backward(*t, None, x["dy"].cuda(), None, None, 64, saved=saved)
