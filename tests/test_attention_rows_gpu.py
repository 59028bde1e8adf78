"""Attention of many rows (the group kernel of attention_decode.hip): bit-exact
with the oracle's chunk-and-merge restatement over the group sizes, workgroup
sizes, chunk counts and span lengths at which its launch and its rounds change;
invalid spans give zeros."""
import numpy as np
import pytest

from test_attention_decode_gpu import Cache, bit_equal, oracle_decode, queries, run_decode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,qk", [(12, 2, 48), (3, 1, 64), (4, 1, 64), (5, 1, 48), (16, 1, 64), (8, 8, 64)])
@pytest.mark.parametrize("rows,capacity,max_chunks", [
    (65, 300, 1), (65, 600, 2), (65, 1000, 8), (70, 530, 64), (45, 1100, 64), (66, 4096, 64), (65, 2100, 100),
])
def test_many_rows_bit_exact(hip, orc, heads, kv_heads, qk, rows, capacity, max_chunks):
    cache = Cache(orc, hip, 3 + heads + capacity + max_chunks, 3, capacity, kv_heads, qk)
    rng = np.random.default_rng(rows + capacity + heads)
    edge = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 64, 127, 128, 257, capacity - 1, capacity]
    spec = [(k % 3, 0, c) for k, c in enumerate(edge)] + [(1, 5, 40), (2, capacity - 1, 1), (0, capacity - 33, 33)]
    while len(spec) < rows:
        first = int(rng.integers(0, capacity))
        spec.append((int(rng.integers(0, 3)), first, int(rng.integers(1, capacity - first + 1))))
    q, qs = queries(orc, cache.st, rows, heads, qk)
    got, _ = run_decode(hip, cache, q, qs, heads, spec, max_chunks)
    assert bit_equal(got, oracle_decode(orc, cache, q, qs, heads, spec, max_chunks))


@pytest.mark.parametrize("heads,kv_heads,capacity", [(16, 8, 300), (16, 8, 500), (32, 8, 513)])
def test_many_rows_short_caches_and_invalid_spans(hip, orc, heads, kv_heads, capacity):
    rows = 80
    cache = Cache(orc, hip, heads + capacity, 2, capacity, kv_heads, 64)
    spec = [(r % 2, 0, 1 + (r * 37) % capacity) for r in range(rows)]
    bad = {1: (2, 0, 10), 2: (1, -1, 5), 3: (0, 0, 0), 4: (1, capacity - 10, 25), 5: (-1, 0, 3)}
    for k, v in bad.items():
        spec[k] = v
    q, qs = queries(orc, cache.st, rows, heads, 64)
    got, _ = run_decode(hip, cache, q, qs, heads, spec, 8)
    good = [k for k in range(rows) if k not in bad]
    want = oracle_decode(orc, cache, q, qs, heads, [spec[k] if k not in bad else (0, 0, 0) for k in range(rows)], 8)
    assert bit_equal(got[good], want[good])
    assert np.all(got[list(bad)] == 0.0)
