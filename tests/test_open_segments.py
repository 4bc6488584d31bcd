"""GPUCache._open_segments (the batch form append_batch uses) against _open_segment, one by one."""
import random

import numpy as np
import pytest

from dkv.gpu_cache import GPUCache


@pytest.mark.parametrize('seed', range(20))
def test_batch_bookkeeping_equals_one_by_one(seed):
    """Plan, tile table, counts, segments and the arena's growth, over several batches of segments of
    1 to 300 tokens; every recorded number a plain int."""
    rng = random.Random(seed)
    kw = dict(layers=rng.randint(1, 4), heads=rng.randint(1, 5), device='cpu', max_tokens=3000,
              arena_bytes=rng.choice([None, 256, 5000]))
    one, batch = GPUCache(None, **kw), GPUCache(None, **kw)
    start = 0
    for _ in range(rng.randint(1, 3)):
        lengths = [rng.choice([64, 1, 63, 65, 128, rng.randint(1, 300)]) for _ in range(rng.randint(1, 4))]
        bits = [rng.choice([4, 8, 16]) for _ in lengths]
        frame, tile0, at = rng.randint(-1, 3), len(one.tile_starts), start
        for n, b in zip(lengths, bits):
            one._open_segment(at, n, b, frame)
            at += n
        if seed % 2:  # arrays are what the same lists are
            lengths, bits = np.array(lengths), np.array(bits)
        assert batch._open_segments(start, lengths, bits, frame) == tile0
        start = at
    for name in ('plan', 'tile_starts', 'host_counts', 'arena_used', 'arena_bytes'):
        assert getattr(one, name) == getattr(batch, name), name
    assert one.tiles_host.tobytes() == batch.tiles_host.tobytes()
    fields = ('start', 'rows', 'bits', 'offset', 'tile0', 'frame')
    assert [[getattr(s, f) for f in fields] for s in one.segments] == \
        [[getattr(s, f) for f in fields] for s in batch.segments]
    assert all(type(x) is int for entry in batch.plan for x in entry)
    assert all(type(getattr(s, f)) is int for s in batch.segments for f in fields)


def test_batch_past_the_tile_table_changes_nothing():
    c = GPUCache(None, layers=1, heads=1, device='cpu', max_tokens=4)
    with pytest.raises(ValueError, match='context limit'):
        c._open_segments(0, [1] * 5, [4] * 5)
    assert not c.segments and not c.plan and not c.tile_starts and c.arena_used == 0
