"""Routes the entry points choose by size: each against the general path or the oracle."""
import pytest
import torch

from conftest import announce
from dkv import gpu_ops
from dkv.gpu_cache import GPUCache
from dkv.workloads import frame_chunk_case

pytestmark = pytest.mark.gpu


def filled(case, cuda, heads, extra=64, precision='bf16'):
    past = case['k_hist'].shape[1]
    c = GPUCache(None, layers=1, heads=heads, max_tokens=past + case['q'].shape[1] + extra, precision=precision)
    lengths = [min(64, past - t) for t in range(0, past, 64)]
    c.append_batch(case['k_hist'][None].to(cuda), case['v_hist'][None].to(cuda), case['bits'], lengths)
    return c, past


@pytest.mark.parametrize('nq,past', [(1, 999), (5, 130), (64, 1000), (78, 64)])
@pytest.mark.parametrize('precision', ['fp32', 'bf16'])
def test_attend_argument_bytes(cuda, nq, past, precision):
    """attend() of one causal chunk packs the argument block as bytes; with segments=[0, nq], the same
    mask, it fills the Structure. Same launches, same bits; strided q, k and v rows included."""
    announce(f'routes: argument bytes nq={nq} past={past} precision={precision}')
    case = frame_chunk_case(past, seed=nq + past, nq=nq)
    c, past = filled(case, cuda, 5, precision=precision)
    q, k, v = (case[x].to(cuda).transpose(0, 1).contiguous().transpose(0, 1)[None] for x in ('q', 'k_new', 'v_new'))
    for dtype in (None, torch.float32):
        a = c.attend(q, k, v, 0, past, out_dtype=dtype)
        b = c.attend(q, k, v, 0, past, out_dtype=dtype, segments=[0, nq])
        assert a.dtype == b.dtype and torch.equal(a, b)


def test_attend_calls_share_no_workspace(cuda):
    """Split calls of one cache on two streams at once: each has its own partials, so every output
    equals the one computed alone."""
    announce('routes: concurrent attends of one cache')
    case = frame_chunk_case(4000, seed=3, nq=64)
    c, past = filled(case, cuda, 5)
    g = torch.Generator().manual_seed(1)
    qs = [torch.randn((1, 15, 64, 64), generator=g).to(torch.bfloat16).to(cuda) for _ in range(8)]
    k, v = case['k_new'][None].to(cuda), case['v_new'][None].to(cuda)
    want = [c.attend(q, k, v, 0, past) for q in qs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    got = []
    for i, q in enumerate(qs):
        with torch.cuda.stream(streams[i % 2]):
            got.append(c.attend(q, k, v, 0, past))
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize('rows,k,n,norm,epi', [
    (4481, 64, 64, True, 'plain'), (4417, 128, 64, False, 'residual'), (1201, 448, 256, True, 'plain'),
    (700, 512, 448, False, 'plain'), (4500, 576, 64, True, 'plain'), (321, 960, 960, False, 'residual'),
    (385, 960, 1600, True, 'plain'), (97, 960, 5120, True, 'silu'), (130, 960, 5120, False, 'silu'),
    (2071, 1024, 256, True, 'silu'), (577, 2560, 960, False, 'residual'), (3000, 2560, 192, False, 'plain'),
])
def test_many_row_projections_equal_few_row_ones(cuda, rows, k, n, norm, epi):
    """From some hundred rows on linear() runs 64 x 64 tiles (and the norm as a launch of its own).
    Both kernels form a row's sums in one order, so every row equals the one a 64-row call gives, bit
    for bit, in every operand layout; ragged last tiles, one to forty pairs of k."""
    announce(f'routes: projection rows={rows} k={k} n={n} norm={norm} epi={epi}')
    assert gpu_ops._lib.load().dkv_linear_prenorm(rows, n, k, {'plain': 0, 'residual': 1, 'silu': 2}[epi]) or k > 1024
    g = torch.Generator().manual_seed(rows + k)
    bf = torch.bfloat16
    x = (torch.randn(rows, k, generator=g) * 2).to(bf).to(cuda)
    w = (torch.randn(n, k, generator=g) / k ** 0.5).to(bf).to(cuda)
    nw = (torch.rand(k, generator=g) + 0.5).to(bf).to(cuda) if norm else None
    n_out = n // 2 if epi == 'silu' else n
    res = torch.randn(rows, n_out, generator=g).to(bf).to(cuda) if epi == 'residual' else None
    kw = dict(norm=nw, eps=1e-5, silu_mul=epi == 'silu')
    want = torch.cat([gpu_ops.linear(x[t:t + 64], w, residual=None if res is None else res[t:t + 64], **kw)
                      for t in range(0, rows, 64)])
    assert torch.equal(gpu_ops.linear(x, w, residual=res, **kw), want)
    wt, xt = gpu_ops.mfma_tiled(w), gpu_ops.mfma_tiled(x)
    assert torch.equal(gpu_ops.linear(x, w, residual=res, weight_tiled=wt, **kw), want)
    assert torch.equal(gpu_ops.linear(xt, w, residual=res, x_tiled=True, rows=rows, **kw), want)
    wide = torch.empty(rows, k + 64, dtype=bf, device=cuda)
    wide[:, :k] = x  # rows further apart than k
    assert torch.equal(gpu_ops.linear(wide[:, :k], w, residual=res, weight_tiled=wt, **kw), want)
    if n_out % 64 == 0:
        rt = None if res is None else gpu_ops.mfma_tiled(res)
        got = gpu_ops.linear(xt, w, residual=rt, weight_tiled=wt, x_tiled=True, rows=rows, out_tiled=True,
                             residual_tiled=res is not None, **kw)
        assert torch.equal(gpu_ops.mfma_untiled(got, rows), want)


def test_tiled_x_ends_with_its_last_block(cuda):
    """A tiled x holds its rows rounded up to 16; gate/up takes 32 rows at a time and must not read the
    16 after them (here NaN, in the same allocation)."""
    announce('routes: tiled x at the end of its buffer')
    g = torch.Generator().manual_seed(2)
    w = (torch.randn(1536, 384, generator=g) / 20).to(torch.bfloat16).to(cuda)
    buf = torch.full((32, 384), float('nan'), dtype=torch.bfloat16, device=cuda)
    x = torch.randn(9, 384, generator=g).to(torch.bfloat16).to(cuda)
    buf[:16] = gpu_ops.mfma_tiled(x)
    got = gpu_ops.linear(buf[:16], w, silu_mul=True, x_tiled=True, rows=9)
    assert torch.equal(got, gpu_ops.linear(x, w, silu_mul=True))
