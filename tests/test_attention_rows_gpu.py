"""Attention of many rows: bit-exact with the oracle's chunk-and-merge
restatement on both sides of the group kernel's dispatch (attention_decode.hip),
in each of its forms (workgroup threads, heads a thread), over chunk counts and
span lengths at which its rounds change; invalid spans give zeros."""
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


# the group kernel's forms, (threads, heads a thread)
FORMS = [
    ((256, 1), 4, 4, 64, 100, 600, 16), ((256, 1), 16, 8, 64, 140, 500, 8), ((256, 2), 32, 8, 64, 66, 300, 8),
    ((256, 3), 12, 2, 48, 300, 300, 8), ((512, 1), 8, 8, 64, 100, 1000, 64), ((512, 1), 8, 4, 48, 70, 800, 16),
    ((512, 2), 12, 2, 48, 400, 500, 8), ((512, 2), 4, 2, 64, 200, 2300, 64), ((512, 3), 12, 4, 48, 65, 700, 32),
    ((512, 3), 12, 2, 64, 300, 1000, 64), ((1024, 1), 5, 1, 64, 66, 1024, 64), ((1024, 1), 12, 2, 48, 100, 2048, 8),
    ((1024, 2), 4, 1, 48, 70, 530, 64), ((1024, 2), 16, 1, 64, 100, 600, 8), ((1024, 3), 12, 2, 64, 70, 1020, 64),
]


@pytest.mark.parametrize("form,heads,kv_heads,qk,rows,capacity,max_chunks", FORMS)
def test_group_forms_bit_exact(hip, orc, form, heads, kv_heads, qk, rows, capacity, max_chunks):
    cache = Cache(orc, hip, sum(form) + heads + capacity, 2, capacity, kv_heads, qk)
    rng = np.random.default_rng(rows + capacity + heads)
    edge = [1, 2, 16, 17, 31, 33, 48, capacity // 2 + 1, capacity - 1, capacity]
    spec = [(k % 2, 0, c) for k, c in enumerate(edge)] + [(1, 5, 40), (0, capacity - 1, 1), (1, capacity - 33, 33)]
    while len(spec) < rows:
        first = int(rng.integers(0, capacity))
        spec.append((int(rng.integers(0, 2)), first, int(rng.integers(1, capacity - first + 1))))
    bad = {20: (2, 0, 10), 21: (1, -1, 5), 40: (0, 0, 0), 41: (1, capacity - 10, 25), rows - 1: (-1, 0, 3)}
    for k, v in bad.items():
        spec[k] = v
    q, qs = queries(orc, cache.st, rows, heads, qk)
    got, _ = run_decode(hip, cache, q, qs, heads, spec, max_chunks)
    good = [k for k in range(rows) if k not in bad]
    want = oracle_decode(orc, cache, q, qs, heads, [spec[k] if k not in bad else (0, 0, 0) for k in range(rows)],
                         max_chunks)
    assert bit_equal(got[good], want[good])
    assert np.all(got[list(bad)] == 0.0)
