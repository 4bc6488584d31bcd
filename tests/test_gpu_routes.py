"""Routes the entry points choose by size: each against the general path or the oracle."""
import pytest
import torch

from conftest import announce
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
