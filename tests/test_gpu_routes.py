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
    (2071, 1024, 256, True, 'silu'),
    (1000, 960, 5120, True, 'silu'), (2049, 512, 2112, False, 'silu'), (8200, 64, 576, False, 'silu'), (577, 2560, 960, False, 'residual'), (3000, 2560, 192, False, 'plain'),
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


def _dense(c, case, past, starts, dtype):
    """(output, attention over |v|) [nq, Hq, 64] in float64 from the cache's own dequantized history,
    K and V rounded to `dtype` as the kernel's precision does."""
    k, v = (x[0, :, :past].double() for x in c.materialize(0, dtype))
    q, kn, vn = (case[x].to(k.device).double() for x in ('q', 'k_new', 'v_new'))
    k, v = torch.cat((k, kn), 1), torch.cat((v, vn), 1)
    n, group = q.shape[1], q.shape[0] // k.shape[0]
    rows = torch.arange(n, device=k.device)
    mask = torch.ones(n, past + n, dtype=torch.bool, device=k.device)
    mask[:, past:] = (rows[None] <= rows[:, None]) & (rows[None] >= starts.to(k.device)[:, None])
    out, mag = (torch.empty(n, q.shape[0], 64, dtype=torch.float64, device=k.device) for _ in range(2))
    for h in range(q.shape[0]):
        p = (q[h] @ k[h // group].t().contiguous() / 8).masked_fill_(~mask, float('-inf')).softmax(-1)
        out[:, h], mag[:, h] = p @ v[h // group], p @ v[h // group].abs()
    return out, mag


@pytest.mark.parametrize('heads,group,nq,past,tiles', [
    (5, 3, 400, 0, 'none'),         # no history; the first row sees one key
    (5, 3, 401, 1, 'frames'),       # one key of history, an odd chunk
    (5, 3, 608, 999, 'frames'),     # past not a multiple of 64
    (8, 4, 256, 4096, 'frames'),    # the history ends on a unit
    (8, 2, 378, 700, 'ones'),       # one-token tiles (decode steps), 700 of them: past the table window
    (1, 1, 6010, 77, 'frames'),     # one head; the last group of rows is partly empty
    (2, 8, 379, 5000, 'mixed'),     # tiles of 1 to 64 rows
    (3, 3, 669, 64, 'frames'),
])
@pytest.mark.parametrize('precision', ['bf16', 'fp32'])
def test_long_chunks_match_dense_attention(cuda, heads, group, nq, past, tiles, precision):
    """Long chunks (unpacked keys, causal ranges, merge) against dense float64 attention. bf16: p is
    rounded to bf16 (8 significant bits: at most 2^-8 of each term) and partial outputs to fp16 (11
    bits: 2^-11), so an output is within 2^-8 + 2^-10 of the attention over |v| (fp32 sums and
    exponentials take the rest of 2^-10); fp32: within 1e-3, as every fp32 path. The frame-chunk kernel
    (path='mfma') must agree with the same bounds, and two calls bit for bit."""
    announce(f'routes: long chunk heads={heads} group={group} nq={nq} past={past} tiles={tiles} {precision}')
    assert heads * group * nq >= 6000 and group * nq >= 256
    case = frame_chunk_case(past, seed=nq + past, heads=heads, q_heads=heads * group, nq=nq)
    c = GPUCache(None, layers=2, heads=heads, max_tokens=past + nq + 64, precision=precision)
    g = torch.Generator().manual_seed(past)
    lengths, t = [], 0
    while t < past:
        n = {'ones': 1, 'mixed': int(torch.randint(1, 65, (1,), generator=g))}.get(tiles, 64)
        lengths.append(min(n, past - t))
        t += lengths[-1]
    if past:
        k, v = (case[x][None].expand(2, -1, -1, -1).contiguous().to(cuda) for x in ('k_hist', 'v_hist'))
        c.append_batch(k, v, [(4, 8, 16)[i % 3] for i in range(len(lengths))], lengths)
    q, k, v = (case[x].to(cuda).transpose(0, 1).contiguous().transpose(0, 1)[None] for x in ('q', 'k_new', 'v_new'))
    starts = torch.zeros(nq, dtype=torch.long)
    for segments in (None, [0, nq // 3, nq // 3 + 1, nq]):
        if segments:
            for b in segments[:-1]:
                starts[b:] = b
        ref, mag = _dense(c, case, past, starts, torch.bfloat16 if precision == 'bf16' else torch.float32)
        bound = mag * (2.0 ** -8 + 2.0 ** -10) + 1e-5 if precision == 'bf16' else torch.full_like(mag, 1e-3)
        got = c.attend(q, k, v, 0, past, out_dtype=torch.float32, segments=segments)
        assert bool(((got[0].double() - ref).abs() <= bound).all()), ((got[0].double() - ref).abs() - bound).max()
        assert torch.equal(got, c.attend(q, k, v, 0, past, out_dtype=torch.float32, segments=segments))
        assert torch.equal(got.to(torch.bfloat16), c.attend(q, k, v, 0, past, segments=segments))
        frame = c.attend(q, k, v, 0, past, out_dtype=torch.float32, segments=segments, path='mfma')
        assert bool(((frame[0].double() - ref).abs() <= bound).all())


@pytest.mark.parametrize('heads,group,nq,past', [(5, 3, 420, 1024), (5, 3, 1700, 300), (5, 3, 2048, 1000), (8, 4, 900, 500)])
def test_long_chunks_are_as_accurate_as_frame_chunks(cuda, heads, group, nq, past):
    """At fp32 precision the long-chunk kernels are no further from dense float64 attention than the
    frame-chunk kernel (path='mfma'), in the 2-norm over some hundred thousand outputs (whose own scatter is
    under 0.5%)."""
    announce(f'routes: long chunk accuracy heads={heads} group={group} nq={nq} past={past}')
    case = frame_chunk_case(past, seed=nq, heads=heads, q_heads=heads * group, nq=nq)
    c = GPUCache(None, layers=1, heads=heads, max_tokens=past + nq, precision='fp32')
    lengths = [min(64, past - t) for t in range(0, past, 64)]
    c.append_batch(case['k_hist'][None].to(cuda), case['v_hist'][None].to(cuda), case['bits'], lengths)
    q, k, v = (case[x][None].to(cuda) for x in ('q', 'k_new', 'v_new'))
    ref, _ = _dense(c, case, past, torch.zeros(nq, dtype=torch.long), torch.float32)
    err = [(c.attend(q, k, v, 0, past, out_dtype=torch.float32, path=path)[0].double() - ref).norm().item()
           for path in ('auto', 'mfma')]
    assert err[0] <= 1.005 * err[1], err


@pytest.mark.parametrize('heads,group,nq,past,tiles', [
    (32, 3, 1, 2500, 'frames'),    # 41 units at 32 KV heads: two per workgroup by default, descriptors in the arguments
    (5, 3, 10, 1999, 'mixed'),     # 30 rows; tiles of 1 to 64 rows
    (8, 2, 1, 700, 'ones'),        # 700 tiles: the device table, more units in a range than its window of 64
    (1, 8, 4, 64, 'frames'),       # one tile and the chunk
])
def test_decode_workgroups_of_several_units(cuda, heads, group, nq, past, tiles):
    """Few query rows at precision 0 when a workgroup walks several units (each loaded while the one
    before it is worked on), by default and at given split counts: within the bounds of
    test_long_chunks_match_dense_attention of dense float64 attention."""
    announce(f'routes: decode units heads={heads} group={group} nq={nq} past={past} tiles={tiles}')
    assert group * nq <= 32
    case = frame_chunk_case(past, seed=past, heads=heads, q_heads=heads * group, nq=nq)
    c = GPUCache(None, layers=1, heads=heads, max_tokens=past + nq + 64, precision='bf16')
    g = torch.Generator().manual_seed(past)
    lengths, t = [], 0
    while t < past:
        n = {'ones': 1, 'mixed': int(torch.randint(1, 65, (1,), generator=g))}.get(tiles, 64)
        lengths.append(min(n, past - t))
        t += lengths[-1]
    c.append_batch(case['k_hist'][None].to(cuda), case['v_hist'][None].to(cuda),
                   [(4, 8, 16)[i % 3] for i in range(len(lengths))], lengths)
    q, k, v = (case[x][None].to(cuda) for x in ('q', 'k_new', 'v_new'))
    ref, mag = _dense(c, case, past, torch.zeros(nq, dtype=torch.long), torch.bfloat16)
    bound = mag * (2.0 ** -8 + 2.0 ** -10) + 1e-5
    for splits in (0, 1, 2, 7, len(lengths)):
        got = c.attend(q, k, v, 0, past, out_dtype=torch.float32, splits=splits)
        assert bool(((got[0].double() - ref).abs() <= bound).all()), splits


@pytest.mark.parametrize('heads,group,nq,past', [(5, 3, 2048, 1000), (2, 8, 1601, 130), (8, 4, 900, 500)])
def test_long_chunk_sums_stay_in_32_bits(cuda, heads, group, nq, past):
    """Chunks so long that the frame-chunk kernel runs one history split keep O in fp32 to the end, so
    the long-chunk kernels' partials must too. With K = 0 every p is 1 and with small whole numbers as V
    every sum is exact, so an fp32 output is off by the reciprocal and one product: 2^-22 of it (fp16
    partials: 2^-12)."""
    announce(f'routes: long chunk sums heads={heads} group={group} nq={nq} past={past}')
    g = torch.Generator().manual_seed(nq)
    c = GPUCache(None, layers=1, heads=heads, max_tokens=past + nq)
    hist = torch.randint(-8, 9, (1, heads, past, 64), generator=g).to(torch.bfloat16).to(cuda)
    c.append_batch(torch.zeros_like(hist), hist, [16] * ((past + 63) // 64), [min(64, past - t) for t in range(0, past, 64)])
    q = torch.randn((1, heads * group, nq, 64), generator=g).to(torch.bfloat16).to(cuda)
    v = torch.randint(-8, 9, (1, heads, nq, 64), generator=g).to(torch.bfloat16).to(cuda)
    got = c.attend(q, torch.zeros_like(v), v, 0, past, out_dtype=torch.float32)[0].double()
    seen = torch.arange(past + 1, past + nq + 1, device=cuda, dtype=torch.float64)[:, None, None]
    ref = ((hist[0].double().sum(1, keepdim=True) + v[0].double().cumsum(1)).transpose(0, 1) / seen)
    ref = ref.repeat_interleave(group, 1)
    assert bool(((got - ref).abs() <= 2.0 ** -22 * ref.abs()).all())


def test_long_chunk_partials_keep_large_values(cuda):
    """|V| near the top of bf16: the fp16 partial outputs are stored scaled by a power of two. V and V * 2^20
    give outputs that differ by exactly that factor, up to the bits a scaled sum may lose: under 2^-15 of a
    partial's weight, in the sum of the weights too, so 2^-14 of the attention over |v|; and half a step of
    fp16 below its normal range, 2^-25, in the unscaled ones."""
    announce('routes: long chunk, large values')
    case = frame_chunk_case(2000, seed=9, nq=420)
    outs, mag = [], None
    for scale in (1.0, 2.0 ** 20):
        c = GPUCache(None, layers=1, heads=5, max_tokens=2500)
        k, v = case['k_hist'][None].to(cuda), (case['v_hist'].float() * scale).to(torch.bfloat16)[None].to(cuda)
        c.append_batch(k, v, [16] * 32, [64] * 31 + [16])
        if mag is None:
            _, mag = _dense(c, case, 2000, torch.zeros(420, dtype=torch.long), torch.bfloat16)
        q, kn, vn = (case[x][None].to(cuda) for x in ('q', 'k_new', 'v_new'))
        outs.append(c.attend(q, kn, (vn.float() * scale).to(torch.bfloat16), 0, 2000, out_dtype=torch.float32))
    a, b = outs[0][0].double(), outs[1][0].double() / 2.0 ** 20
    assert torch.isfinite(b).all()
    assert bool(((a - b).abs() <= 2.0 ** -14 * mag + 2.0 ** -24).all()), ((a - b).abs() / mag).max().item()


@pytest.mark.parametrize('precision', ['fp32', 'bf16'])
@pytest.mark.parametrize('past,nq', [(0, 500), (700, 420)])
def test_long_chunk_replays_equal_calls_as_replayed(cuda, past, nq, precision):
    """A long chunk recorded with graph steps runs the frame-chunk kernel: bit for bit what ordinary calls
    give with as_replayed set or path='mfma', over every replay. The default call differs by rounding: p to bf16 twice, 2^-8 of each term at most
    and random over rows of hundreds of keys, so under 1% of the outputs' norm."""
    announce(f'routes: long chunk replay past={past} nq={nq} {precision}')
    case = frame_chunk_case(max(past, 64), seed=nq, nq=nq)
    g = torch.Generator().manual_seed(nq)
    chunks = [[torch.randn((1, h, nq, 64), generator=g).to(torch.bfloat16).to(cuda) for h in (15, 5, 5)] for _ in range(3)]

    def cache():
        if past:
            return filled(case, cuda, 5, extra=3 * nq, precision=precision)[0]
        return GPUCache(None, layers=1, heads=5, max_tokens=3 * nq, precision=precision)

    plain, c = cache(), cache()
    c.select(8, 1)
    plain.select(8, 1)
    steps = c.begin_graph_steps(nq, q_heads=15)
    past0 = c.graph_step()
    static = [t.clone() for t in chunks[0]]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        c.append(static[1], static[2], 0)
        out = c.attend(static[0], static[1], static[2], 0, past0)
    steps.upload()
    for i, (q, k, v) in enumerate(chunks):
        if i:
            c.graph_step()
            for dst, src in zip(static, (q, k, v)):
                dst.copy_(src)
        graph.replay()
        at = plain.append(k, v, 0)
        auto = plain.attend(q, k, v, 0, at)
        assert torch.equal(out, plain.attend(q, k, v, 0, at, path='mfma'))
        plain.as_replayed = True
        assert torch.equal(out, plain.attend(q, k, v, 0, at))
        plain.as_replayed = False
        assert (out.float() - auto.float()).norm() <= 0.01 * out.float().norm()
    c.end_graph_steps()


def test_long_chunk_replay_over_a_shorter_table(cuda):
    """A captured long chunk whose cache was reset and refilled with shorter tiles reads the device table of
    that time: the ten tiles it was captured for now hold 100 of its 640 history tokens, and the rest count
    as zeros, in every replay. Within the bounds of test_long_chunks_match_dense_attention."""
    announce('routes: long chunk replay over a shorter table')
    nq, past = 420, 640
    case = frame_chunk_case(past, seed=8, nq=nq)
    c, _ = filled(case, cuda, 5, precision='fp32')
    q, k, v = (case[x][None].to(cuda) for x in ('q', 'k_new', 'v_new'))
    c.attend(q, k, v, 0, past, out_dtype=torch.float32)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = c.attend(q, k, v, 0, past, out_dtype=torch.float32)
    hist_k, hist_v = case['k_hist'][None].to(cuda), case['v_hist'][None].to(cuda)
    for bits in (4, 8, 16):
        c.reset()
        c.append_batch(hist_k, hist_v, [bits] * 64, [10] * 64)
        graph.replay()
        full_k, full_v = (x.clone() for x in c.materialize(0, torch.float32))
        full_k[:, :, 100:], full_v[:, :, 100:] = 0, 0

        class Held:
            @staticmethod
            def materialize(layer, dtype):
                return full_k, full_v

        ref, _ = _dense(Held, case, past, torch.zeros(nq, dtype=torch.long), torch.float32)
        assert (out[0].double() - ref).abs().max() <= 1e-3, bits


def test_long_chunk_without_scratch_for_its_keys(cuda):
    """dkv_attend_noalloc: the same call as dkv_attend where the unpacked keys and partials fit its
    scratch buffer; where they do not, the frame-chunk kernel's output instead of a refusal."""
    import ctypes

    from dkv import _lib
    announce('routes: long chunk through dkv_attend_noalloc')
    lib = _lib.load()
    for nq, past, fits in ((420, 1000, True), (2048, 30000, False)):
        case = frame_chunk_case(past, seed=nq, nq=nq)
        c, past = filled(case, cuda, 5)
        q, k, v = (case[x][None].to(cuda) for x in ('q', 'k_new', 'v_new'))
        out = torch.empty(1, nq, 15, 64, dtype=torch.float32, device=cuda)
        a = c.attend_args(q, k, v, 0, past, out)
        assert (lib.dkv_attend_workspace_bytes(ctypes.byref(a)) <= _lib.DKV_NOALLOC_SCRATCH_BYTES) == fits
        _lib.check(lib.dkv_attend_noalloc(ctypes.byref(a), _lib.stream_handle(cuda)), 'dkv_attend_noalloc')
        want = c.attend(q, k, v, 0, past, out_dtype=torch.float32, path='auto' if fits else 'mfma')
        assert torch.equal(out, want)


@pytest.mark.parametrize('n,k,q_heads,heads,bits', [
    (1, 960, 15, 5, 16), (15, 64, 1, 1, 4), (16, 512, 3, 3, 8), (17, 576, 9, 3, 4), (64, 960, 15, 5, 4),
    (78, 1024, 16, 8, 8), (200, 960, 15, 5, 8), (100, 960, 15, 5, 16), (353, 960, 15, 5, 4), (1000, 128, 9, 3, 16),
])
@pytest.mark.parametrize('tiled', [False, True])
def test_projection_that_packs_equals_its_parts(cuda, n, k, q_heads, heads, bits, tiled):
    """dkv_linear_rope_pack against linear() and append_projection() (themselves checked against torch and
    the quantizer): q, k, v, the packed bytes and the tile table, bit for bit, with the norm in the launch
    and apart (64 x 64 tiles); one to sixty row blocks with ragged last ones, one and two pairs of k per wave, behind another segment, with the job in the argument block and in device memory."""
    import ctypes

    from dkv import _lib
    announce(f'routes: projection and pack n={n} k={k} heads={q_heads}/{heads} bits={bits} tiled={tiled}')
    g = torch.Generator().manual_seed(n + k)
    bf = torch.bfloat16
    x = (torch.randn(n, k + 8, generator=g) * 2).to(bf).to(cuda)[:, :k]
    w = (torch.randn((q_heads + 2 * heads) * 64, k, generator=g) / k ** 0.5).to(bf).to(cuda)
    nw = (torch.rand(k, generator=g) + 0.5).to(bf).to(cuda)
    angle = torch.rand(n, 64, generator=g) * 6
    cos, sin = angle.cos().to(bf).to(cuda), angle.sin().to(bf).to(cuda)
    wt = gpu_ops.mfma_tiled(w) if tiled else None
    a, b, c, d, e = (GPUCache(None, layers=2, heads=heads, max_tokens=n + 9) for _ in range(5))
    lead = torch.randn(1, heads, 9, 64, generator=g).to(bf).to(cuda)
    for cache in (a, b, c, d, e):
        cache.arena.zero_()
        cache.tiles.zero_()
        cache.select(8, 0)
        cache.append(lead, lead, 0)
        cache.select(bits, 1)
    qkv = gpu_ops.linear(x, w, norm=nw, eps=1e-5, weight_tiled=wt)
    want = a.append_projection(qkv[None], cos[None], sin[None], q_heads, 0)
    xn = torch.empty((n + 15) // 16 * 16, k, dtype=bf, device=cuda)
    _lib.check(_lib.load().dkv_rms_norm_tiled(x.data_ptr(), x.stride(0), nw.data_ptr(), xn.data_ptr(), n, k, 1e-5, 0,
                                              _lib.stream_handle(cuda)), 'dkv_rms_norm_tiled')
    for cache, on_device, apart in ((b, 0, 0), (c, 1, 0), (d, 0, 1), (e, 1, 1)):
        past, seg, write_tiles = cache._claim(0, n)
        q, kn, v = (torch.full_like(t, float('nan')) for t in want[:3])
        job = cache._job(kn, v, 0, past, n, seg, write_tiles)
        dev = torch.frombuffer(bytearray(bytes(job)), dtype=torch.uint8).to(cuda)
        src = w if wt is None else wt
        _lib.check(_lib.load().dkv_linear_rope_pack(
            (xn if apart else x).data_ptr(), x.stride(0), src.data_ptr(), src.stride(0), n, k,
            None if apart else nw.data_ptr(), 1e-5,
            (gpu_ops.LINEAR_W_TILED if tiled else 0) | (gpu_ops.LINEAR_X_TILED if apart else 0), cos.data_ptr(),
            sin.data_ptr(), 64, q_heads, q.data_ptr(), kn.data_ptr(), v.data_ptr(),
            dev.data_ptr() if on_device else ctypes.byref(job), on_device, cache.arena.data_ptr(), cache.arena_bytes,
            cache.tiles.data_ptr(), 2, heads, _lib.stream_handle(cuda)), 'dkv_linear_rope_pack')
        for got, ref in zip((q, kn, v), want):
            assert torch.equal(got, ref)
        assert torch.equal(cache.arena, a.arena) and torch.equal(cache.tiles, a.tiles)


@pytest.mark.parametrize('layers,heads,lengths', [
    (3, 5, [64, 64, 64]), (2, 3, [1, 63, 65, 130, 7]), (1, 1, [64] * 128 + [5]), (2, 2, [1] * 300),
    (4, 8, [200]),
])
@pytest.mark.parametrize('strided', [False, True])
def test_volume_append_equals_appends(cuda, layers, heads, lengths, strided):
    """append_batch of an online cache (descriptors in the launch's argument block, 128 tiles a launch)
    writes the bytes, the tile table and the bookkeeping that an append per layer and segment writes,
    also behind earlier segments and for K/V whose tokens or heads are further apart."""
    announce(f'routes: volume append layers={layers} heads={heads} segments={len(lengths)} strided={strided}')
    n = sum(lengths)
    bits = [(4, 8, 16)[i % 3] for i in range(len(lengths))]
    g = torch.Generator().manual_seed(n + heads)
    k, v = (torch.randn((layers, heads, n + 3, 64), generator=g).to(torch.bfloat16).to(cuda) for _ in range(2))
    if strided:
        k = k.permute(2, 0, 1, 3).contiguous().permute(1, 2, 0, 3)  # tokens outermost
        v = torch.cat((v, v), -1)[..., :64]
    a, b = (GPUCache(None, layers=layers, heads=heads, max_tokens=n + 3) for _ in range(2))
    for c in (a, b):
        c.arena.zero_()
        for layer in range(layers):
            c.select(8, 4)
            c.append(k[None, layer, :, :3], v[None, layer, :, :3], layer)
    batch = a.append_batch(k[:, :, 3:], v[:, :, 3:], bits, lengths)
    t = 3
    for w, m in zip(bits, lengths):
        b.select(w, 4)
        for layer in range(layers):
            b.append(k[None, layer, :, t:t + m], v[None, layer, :, t:t + m], layer)
        t += m
    assert a.seen == b.seen and a.plan == b.plan and a.arena_used == b.arena_used
    used = a.arena_used
    assert torch.equal(a.arena[:used], b.arena[:used])
    tiles = len(a.tile_starts)
    assert torch.equal(a.tiles[:tiles], b.tiles[:tiles]) and a.tiles_host[:tiles].tobytes() == \
        a.tiles[:tiles].cpu().numpy().tobytes()
    a.arena[a.segments[1].offset:].zero_()
    batch.run()
    assert torch.equal(a.arena[:used], b.arena[:used])


def test_volume_append_takes_arrays(cuda):
    """lengths and bits as numpy arrays are what the same lists are, plain ints in the bookkeeping."""
    import numpy as np
    announce('routes: volume append, array arguments')
    g = torch.Generator().manual_seed(5)
    k, v = (torch.randn((2, 3, 200, 64), generator=g).to(torch.bfloat16).to(cuda) for _ in range(2))
    a, b = (GPUCache(None, layers=2, heads=3, max_tokens=200) for _ in range(2))
    for c in (a, b):
        c.arena.zero_()
    a.append_batch(k, v, [4, 8, 16], [64, 130, 6])
    b.append_batch(k, v, np.array([4, 8, 16]), np.array([64, 130, 6]))
    assert torch.equal(a.arena, b.arena) and a.plan == b.plan and a.seen == b.seen
    assert all(type(x) is int for entry in b.plan for x in entry)


def test_attend_holds_little_workspace(cuda):
    """The workspace of a call goes back to the allocator with it when it is large (a long chunk's unpacked
    keys); of a smaller one the cache holds the last, at most WORKSPACE_KEPT bytes."""
    from dkv.gpu_cache import WORKSPACE_KEPT
    announce('routes: workspace given back')
    for past, nq in ((52000, 1000), (1000, 1000)):
        case = frame_chunk_case(past, seed=4, nq=nq)
        c, past = filled(case, cuda, 5, precision='fp32')
        q, k, v = (case[x][None].to(cuda) for x in ('q', 'k_new', 'v_new'))
        assert (5 * (past + nq) * 512 > WORKSPACE_KEPT) == (past > 20000)
        held = torch.cuda.memory_allocated()
        for _ in range(3):
            out = c.attend(q, k, v, 0, past)
        kept = torch.cuda.memory_allocated() - held - out.numel() * 2
        # (torch's allocator leaves up to 1 MiB of a block unsplit: of the output's, of the one held)
        assert kept <= (0 if past > 20000 else WORKSPACE_KEPT + 2 ** 20) + 2 ** 20
