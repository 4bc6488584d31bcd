"""The work a user of this framework has it do, as cases that can be timed and checked.

A case is a dict of plain values; `kind` picks the entry point:

  attend       GPUCache.attend of one layer: a chunk of queries over a packed history and the
               chunk's own K/V (decode steps, frames, prompts);
  branch       the candidate protocol of one layer: fork the cache, append the candidates' K/V at
               16 bits, attend with block-diagonal chunk segments;
  pack         GPUCache.append_batch of a whole volume, every layer and frame;
  materialize  GPUCache.materialize of one layer's history;
  layer        gpu_ops.fused_decoder_layer on a fork: one decoder layer of the 960-wide decoder;
  request      StreamingDecoder: ingest a prefix and frames, then score a question (whole call).

Histories are a 16-bit text prefix followed by 64-token frames at the widths of `bits` (0: the
40/40/20 mix of 4/8/16 bits that dkv.workloads schedules), the last frame cut to fit `past`.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'dynamic-kv-cache_amd')
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from dkv import gpu_ops  # noqa: E402
from dkv.gpu_cache import GPUCache  # noqa: E402
from dkv.streaming import StreamingDecoder, build_decoder  # noqa: E402
from dkv.workloads import bit_schedule  # noqa: E402

DIM, TILE = 64, 64
ROW_BYTES = {4: 40, 8: 72, 16: 128}  # payload and (offset, scale) of one 64-element row
HIDDEN, INTER, HEADS, Q_HEADS = 960, 2560, 5, 15  # the decoder of dkv.streaming.build_decoder
DEVICE = 'cuda'


def listed():
    return [
        # one generated token over a short conversation: the smallest call, launches and latency
        dict(name='decode_short', kind='attend', heads=5, q_heads=15, nq=1, past=999, prefix=39, bits=0,
             precision='bf16'),
        # one generated token over the default cache's full history (96 frames and more)
        dict(name='decode_full', kind='attend', heads=5, q_heads=15, nq=1, past=8128, prefix=64, bits=0,
             precision='bf16'),
        # one generated token over a long video, past what a launch's argument block describes
        dict(name='decode_long', kind='attend', heads=8, q_heads=16, nq=1, past=33957, prefix=64, bits=0,
             precision='bf16'),
        # a 64-token frame attends over the default cache's full history
        dict(name='frame_full', kind='attend', heads=5, q_heads=15, nq=64, past=8128, prefix=64, bits=0,
             precision='bf16'),
        # the small model's 78-token chunk (3 KV heads) over uniform 4-bit history, fp32 accurate
        dict(name='frame_accurate', kind='attend', heads=3, q_heads=9, nq=78, past=6144, prefix=0, bits=4,
             precision='fp32'),
        # four candidate answers of 8-24 tokens share one 8-bit history
        dict(name='candidates', kind='branch', heads=5, q_heads=15, lengths='13,24,8,17', past=6144, prefix=0, bits=8,
             precision='bf16'),
        # a long prompt after a few frames: one attention call over two thousand query tokens
        dict(name='prompt', kind='attend', heads=5, q_heads=15, nq=2048, past=1000, prefix=40, bits=0,
             precision='bf16'),
        # prefill of 96 frames into a 32-layer cache
        dict(name='pack_volume', kind='pack', layers=32, heads=5, frames=96, last=64),
        # one layer's history for code that wants plain K/V (Cache.update, checks, other attention)
        dict(name='materialize', kind='materialize', heads=5, past=8128, prefix=64, bits=0, out='bf16'),
        # one decoder layer on a 64-token frame in the middle of a video
        dict(name='layer_frame', kind='layer', nq=64, past=4096, prefix=64, bits=0),
        # one decoder layer on a long prompt of odd length
        dict(name='layer_prompt', kind='layer', nq=1000, past=640, prefix=64, bits=0),
        # a whole request on a served (graph-replayed) decoder of eight layers
        dict(name='request', kind='request', layers=8, prefix=30, frames=16, question=21, vocab=49280),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(['attend', 'attend', 'attend', 'attend', 'branch', 'pack', 'materialize', 'layer', 'layer'])
    heads, q_heads = rng.choice([(5, 15), (5, 15), (3, 9), (8, 16), (4, 12), (8, 32), (1, 3)])
    bits = rng.choice([0, 0, 0, 4, 8, 16])
    prefix = rng.choice([0, 0, 64, rng.randint(1, 200)])
    if kind == 'pack':
        return dict(kind=kind, layers=rng.randint(1, 32), heads=rng.choice([3, 5, 8]), frames=_log_int(rng, 1, 60),
                    last=rng.randint(1, 64))
    if kind == 'materialize':
        past = _log_int(rng, 1, 30000)
        return dict(kind=kind, heads=heads, past=past, prefix=min(prefix, past), bits=bits,
                    out=rng.choice(['bf16', 'fp32']))
    if kind == 'layer':
        past = _log_int(rng, 1, 6000)
        return dict(kind=kind, nq=_log_int(rng, 1, 1000), past=past, prefix=min(prefix, past), bits=bits)
    precision = rng.choice(['bf16', 'bf16', 'fp32'])
    if kind == 'branch':
        past = _log_int(rng, 64, 8000)
        lengths = ','.join(str(rng.randint(1, 40)) for _ in range(rng.randint(2, 8)))
        return dict(kind=kind, heads=heads, q_heads=q_heads, lengths=lengths, past=past, prefix=min(prefix, past),
                    bits=bits, precision=precision)
    nq = _log_int(rng, 1, 2000)
    # no more products than the listed prompt has
    most = max(64, min(33000, 2048 * 3048 * 15 // (nq * q_heads) - nq))
    past = _log_int(rng, 32, most)
    return dict(kind=kind, heads=heads, q_heads=q_heads, nq=nq, past=past, prefix=min(prefix, past), bits=bits,
                precision=precision)


# -- inputs ---------------------------------------------------------------------------------------
def _segments(case):
    """(widths, lengths) of the history's segments."""
    past, prefix = case['past'], case['prefix']
    lengths = [prefix] if prefix else []
    while sum(lengths) < past:
        lengths.append(min(TILE, past - sum(lengths)))
    frames = len(lengths) - (1 if prefix else 0)
    widths = [case['bits']] * frames if case['bits'] else bit_schedule(past, frames)
    return ([16] if prefix else []) + widths, lengths


def _values(shape, gen, head_axis):
    """bf16 N(0, 1) with four outlier channels per head scaled by 8, as dkv.workloads draws them."""
    x = torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32)
    gain = torch.ones(shape[head_axis], DIM, device=DEVICE)
    order = torch.rand(shape[head_axis], DIM, generator=gen, device=DEVICE).argsort(1)[:, :4]
    gain.scatter_(1, order, 8.0)
    view = [1] * len(shape)
    view[head_axis], view[-1] = shape[head_axis], DIM
    return (x * gain.view(view)).to(torch.bfloat16)


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _history(case, gen, heads):
    return _values((heads, case['past'], DIM), gen, 0), _values((heads, case['past'], DIM), gen, 0)


def _filled_cache(case, hist, heads, tokens, layers=2, precision='bf16'):
    cache = GPUCache(None, layers=layers, heads=heads, max_tokens=case['past'] + tokens + TILE, precision=precision)
    widths, lengths = _segments(case)
    k, v = (x[None].expand(layers, -1, -1, -1).contiguous() for x in hist)
    cache.append_batch(k, v, widths, lengths)
    return cache


def _chunk(case, gen, heads, q_heads, nq):
    q = _values((q_heads, nq, DIM), gen, 0)[None]
    k = _values((heads, nq, DIM), gen, 0)[None]
    v = _values((heads, nq, DIM), gen, 0)[None]
    return q, k, v


def _lengths(case):
    return [int(n) for n in case['lengths'].split(',')]


def _bounds(case):
    bounds = [0]
    for n in _lengths(case):
        bounds.append(bounds[-1] + n)
    return bounds


def _layer_inputs(case, gen):
    hidden = torch.randn((1, case['nq'], HIDDEN), generator=gen, device=DEVICE).to(torch.bfloat16)
    pos = torch.arange(case['past'], case['past'] + case['nq'], device=DEVICE, dtype=torch.float32)
    freq = 100000.0 ** (-torch.arange(0, DIM, 2, device=DEVICE, dtype=torch.float32) / DIM)
    angle = torch.cat((pos[:, None] * freq, pos[:, None] * freq), -1)
    return hidden, angle.cos().to(torch.bfloat16)[None], angle.sin().to(torch.bfloat16)[None]


def _decoder(layers, vocab, seed):
    return build_decoder(layers=layers, hidden=HIDDEN, heads=Q_HEADS, kv_heads=HEADS, intermediate=INTER,
                         vocab=vocab, seed=seed)


def prepare(case, seed):
    kind, gen = case['kind'], _generator(seed)
    if kind in ('attend', 'branch'):
        heads, q_heads = case['heads'], case['q_heads']
        nq = case['nq'] if kind == 'attend' else sum(_lengths(case))
        hist = _history(case, gen, heads)
        q, k, v = _chunk(case, gen, heads, q_heads, nq)
        cache = _filled_cache(case, hist, heads, nq, precision=case['precision'])
        return dict(kind=kind, cache=cache, q=q, k=k, v=v, past=case['past'],
                    segments=_bounds(case) if kind == 'branch' else None)
    if kind == 'pack':
        tokens = (case['frames'] - 1) * TILE + case['last']
        shape = (case['layers'], case['heads'], tokens, DIM)
        k, v = _values(shape, gen, 1), _values(shape, gen, 1)
        cache = GPUCache(None, layers=case['layers'], heads=case['heads'], max_tokens=tokens)
        cache.arena.zero_()  # the few bytes that round a ragged frame's blocks up are never written
        return dict(kind=kind, cache=cache, k=k, v=v, bits=bit_schedule(tokens, case['frames']),
                    lengths=[TILE] * (case['frames'] - 1) + [case['last']])
    if kind == 'materialize':
        cache = _filled_cache(case, _history(case, gen, case['heads']), case['heads'], 0)
        return dict(kind=kind, cache=cache, out=torch.float32 if case['out'] == 'fp32' else torch.bfloat16)
    if kind == 'layer':
        hist = _history(case, gen, HEADS)
        hidden, cos, sin = _layer_inputs(case, gen)
        decoder = StreamingDecoder(_decoder(1, 64, seed))
        cache = _filled_cache(case, hist, HEADS, case['nq'], layers=1)
        return dict(kind=kind, cache=cache, decoder=decoder, hidden=hidden, cos=cos, sin=sin)
    decoder = StreamingDecoder(_decoder(case['layers'], case['vocab'], seed), graphs=True)
    ids = torch.randint(0, case['vocab'], (1, case['prefix'] + case['question']), generator=gen, device=DEVICE)
    frames = [torch.randn((1, TILE, HIDDEN), generator=gen, device=DEVICE).mul_(0.02).to(torch.bfloat16)
              for _ in range(case['frames'])]
    state = dict(kind=kind, decoder=decoder, prefix=ids[:, :case['prefix']], question=ids[:, case['prefix']:],
                 frames=frames, bits=bit_schedule(case['frames'], case['frames']))
    for _ in range(2):  # a server's decoder has captured its graphs before a request arrives
        run(state)
    return state


def run(state):
    kind = state['kind']
    if kind == 'attend':
        return state['cache'].attend(state['q'], state['k'], state['v'], 0, state['past'])
    if kind == 'branch':
        branch = state['cache'].fork()
        branch.select(16)
        past = branch.append(state['k'], state['v'], 0)
        return branch.attend(state['q'], state['k'], state['v'], 0, past, segments=state['segments'])
    if kind == 'pack':
        cache = state['cache']
        cache.reset()
        cache.append_batch(state['k'], state['v'], state['bits'], state['lengths'])
        return cache.arena[:cache.arena_used]
    if kind == 'materialize':
        return state['cache'].materialize(0, state['out'])
    if kind == 'layer':
        branch = state['cache'].fork()
        branch.select(16)
        used = branch.arena_used
        out = gpu_ops.fused_decoder_layer(state['decoder'].text.layers[0], state['hidden'], branch,
                                          (state['cos'], state['sin']))
        return out, branch.arena[used:branch.arena_used].view(torch.bfloat16)
    decoder = state['decoder']
    cache = decoder.ingest(state['prefix'], state['frames'], state['bits'])
    return decoder.forward(cache.fork(), ids=state['question'], logits=state['question'].shape[1])


# -- what a pass cannot do without ----------------------------------------------------------------
def _history_bytes(case, heads):
    widths, lengths = _segments(case)
    return sum(2 * heads * n * ROW_BYTES[b] for b, n in zip(widths, lengths))


def _attend_work(case, heads, q_heads, nq, pairs):
    native = 2 * DIM * (2 * heads * nq + q_heads * nq)  # chunk K, V and Q, bf16
    out = 2 * DIM * q_heads * nq
    return _history_bytes(case, heads) + native + out, 4 * DIM * q_heads * pairs


def _projection_work(rows, layers):
    cols = (Q_HEADS + 2 * HEADS) * DIM + HIDDEN + 2 * INTER
    weights = layers * (HIDDEN * cols + INTER * HIDDEN)
    return 2 * weights, 2 * rows * weights


def work(case):
    kind = case['kind']
    if kind == 'attend':
        nq = case['nq']
        b, f = _attend_work(case, case['heads'], case['q_heads'], nq, nq * case['past'] + nq * (nq + 1) // 2)
        return dict(bytes=b, flops=f)
    if kind == 'branch':
        ns = _lengths(case)
        pairs = sum(n * case['past'] + n * (n + 1) // 2 for n in ns)
        b, f = _attend_work(case, case['heads'], case['q_heads'], sum(ns), pairs)
        return dict(bytes=b + 2 * case['heads'] * sum(ns) * ROW_BYTES[16], flops=f)
    if kind == 'pack':
        tokens = (case['frames'] - 1) * TILE + case['last']
        lengths = [TILE] * (case['frames'] - 1) + [case['last']]
        rows = 2 * case['layers'] * case['heads']
        out = sum(rows * n * ROW_BYTES[b] for b, n in zip(bit_schedule(tokens, case['frames']), lengths))
        return dict(bytes=rows * tokens * 2 * DIM + out, flops=0)
    if kind == 'materialize':
        wide = 4 if case['out'] == 'fp32' else 2
        rows = 2 * case['heads'] * case['past']
        return dict(bytes=_history_bytes(case, case['heads']) + rows * DIM * wide, flops=2 * rows * DIM)
    if kind == 'layer':
        nq = case['nq']
        pw, pf = _projection_work(nq, 1)
        _, af = _attend_work(case, HEADS, Q_HEADS, nq, nq * case['past'] + nq * (nq + 1) // 2)
        moved = _history_bytes(case, HEADS) + 2 * 2 * nq * HIDDEN + 2 * HEADS * nq * ROW_BYTES[16]
        return dict(bytes=pw + moved, flops=pf + af)
    layers = case['layers']
    tokens = case['prefix'] + TILE * case['frames'] + case['question']
    pw, pf = _projection_work(tokens, layers)
    pairs = tokens * (tokens + 1) // 2
    head = case['vocab'] * HIDDEN
    return dict(bytes=pw + 2 * head + 4 * case['vocab'] * case['question'],
                flops=pf + layers * 4 * DIM * Q_HEADS * pairs + 2 * head * case['question'])


# -- what another correct implementation may differ by -----------------------------------------------
def tolerance(case):
    kind = case['kind']
    if kind in ('pack', 'materialize'):
        return 'exact'
    if kind in ('attend', 'branch'):
        # four times what other split counts and the vector path differ by: at fp32 8.5e-5 (sums that
        # end in a bf16 output), at bf16 2.2e-3 (one decode row; p is rounded to bf16 as well)
        return {'rel': 0.0005} if case['precision'] == 'fp32' else {'rel': 0.01}
    if kind == 'layer':
        return {'rel': 0.004}  # the layer's library projections and attention differ by 5e-4 to 1e-3
    return {'rel': 0.05}  # other split counts and library projections, over eight layers: 0.011


# -- the same values in 64 bits -------------------------------------------------------------------
def _divide32(a, b):
    """The correctly rounded 32-bit quotient (a 64-bit one rounds to it), which decides a code's ties."""
    return (a.double() / b.double()).float()


def _dequantized(x, bits):
    """What a width keeps of bf16 rows [..., 64]: codes from the 32-bit quantizer, values in 64 bits."""
    x = x.float()
    if bits == 16:
        return x.double()
    levels = 2 ** bits - 1
    low, high = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
    span = high - low
    scale = torch.where(span > 0, _divide32(span, torch.full_like(span, levels)), torch.ones_like(span))
    code = _divide32(x - low, scale).round().clamp(0, levels)
    return code.double() * scale.double() + low.double()


def _exact_history(case, hist):
    out = []
    for x in hist:
        parts, t = [], 0
        for b, n in zip(*_segments(case)):
            parts.append(_dequantized(x[:, t:t + n], b))
            t += n
        out.append(torch.cat(parts, 1))
    return out


def _exact_attention(q, k, v, past, starts):
    """q [Hq, n, 64], k and v [H, past + n, 64], all fp64 -> [n, Hq, 64]; chunk row m sees chunk rows
    starts[m]..m and every history token."""
    n, group = q.shape[1], q.shape[0] // k.shape[0]
    rows = torch.arange(n, device=q.device)
    chunk = torch.arange(n, device=q.device)
    seen = (chunk[None] <= rows[:, None]) & (chunk[None] >= starts[:, None])
    mask = torch.cat((torch.ones(n, past, dtype=torch.bool, device=q.device), seen), 1)
    out = torch.empty(n, q.shape[0], DIM, dtype=torch.float64, device=q.device)
    for h in range(q.shape[0]):
        s = q[h] @ k[h // group].t().contiguous() / 8.0
        out[:, h] = s.masked_fill_(~mask, -math.inf).softmax(-1) @ v[h // group]
    return out


def exact(case, seed):
    kind, gen = case['kind'], _generator(seed)
    if kind in ('pack', 'request'):
        return None
    if kind == 'materialize':
        k, v = _exact_history(case, _history(case, gen, case['heads']))
        return k[None], v[None]
    if kind in ('attend', 'branch'):
        heads, q_heads = case['heads'], case['q_heads']
        nq = case['nq'] if kind == 'attend' else sum(_lengths(case))
        hist = _exact_history(case, _history(case, gen, heads))
        q, k, v = (x[0].double() for x in _chunk(case, gen, heads, q_heads, nq))
        starts = torch.zeros(nq, dtype=torch.long, device=DEVICE)
        if kind == 'branch':
            for b in _bounds(case)[:-1]:
                starts[b:] = b
        return _exact_attention(q, torch.cat((hist[0], k), 1), torch.cat((hist[1], v), 1), case['past'], starts)[None]
    nq = case['nq']
    hist = _exact_history(case, _history(case, gen, HEADS))
    hidden, cos, sin = (x[0].double() for x in _layer_inputs(case, gen))
    layer = _decoder(1, 64, seed).model.layers[0].double()
    norm1, norm2, attn, mlp = layer.input_layernorm, layer.post_attention_layernorm, layer.self_attn, layer.mlp

    def rms(x, m):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + m.variance_epsilon) * m.weight

    def heads(x):
        return x.view(nq, -1, DIM).transpose(0, 1)

    def rope(x):
        return x * cos + torch.cat((-x[..., DIM // 2:], x[..., :DIM // 2]), -1) * sin

    with torch.no_grad():
        x = rms(hidden, norm1)
        q, k, v = (heads(x @ m.weight.t().contiguous()) for m in (attn.q_proj, attn.k_proj, attn.v_proj))
        q, k = rope(q), rope(k)
        starts = torch.zeros(nq, dtype=torch.long, device=DEVICE)
        o = _exact_attention(q, torch.cat((hist[0], k), 1), torch.cat((hist[1], v), 1), case['past'], starts)
        h = hidden + o.reshape(nq, -1) @ attn.o_proj.weight.t().contiguous()
        y = rms(h, norm2)
        gate, up = (y @ m.weight.t().contiguous() for m in (mlp.gate_proj, mlp.up_proj))
        out = h + (torch.nn.functional.silu(gate) * up) @ mlp.down_proj.weight.t().contiguous()
    # the appended rows as a 16-bit segment holds them: per 64-token tile K then V of every head
    tiles = [torch.stack((k[:, t:t + TILE], v[:, t:t + TILE])).flatten() for t in range(0, nq, TILE)]
    return out[None], torch.cat(tiles)
