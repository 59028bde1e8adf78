"""FeedSlot's long steps: a prompt longer than the context's chunk reaches the
bits of the same prompt fed chunk by chunk, over the edges of a step (512 rows,
after a history of 3), in several steps and at the context's end, with decode
steps after it; feeds of a captured step's rows between decode steps; and a
token out of range leaves what the chunk-by-chunk feed leaves."""
import numpy as np
import pytest

from test_needle3_step_gpu import archive, gpu_engine, model, same_bits, tokens  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count,capacity", [(17, 64), (130, 160), (512, 560), (513, 560), (90, 91),
                                            (515, 560), (516, 560), (1100, 1150)])
def test_long_feed_equals_chunks(hip, model, count, capacity):  # noqa: F811
    p = tokens(1000 + count, count)
    a = gpu_engine(model, slots=2, capacity=capacity, chunk=16)
    b = gpu_engine(model, slots=2, capacity=capacity, chunk=16)
    try:
        a.feed_slot(1, p[:3], compute_logits=False)  # a history before the prompt
        b.feed_slot(1, p[:3], compute_logits=False)
        got = a.feed_slot(1, p[3:])
        for start in range(3, count, 16):
            n = min(16, count - start)
            last = start + n == count
            want = b.forward_batch(p[start:start + n], [1] * n, [n - 1] if last else [])[0]
        assert same_bits(got, want[0])
        assert a.slot_length(1) == count
        for t in tokens(7, min(3, capacity - count)):
            assert same_bits(a.forward_batch([t], [1], [0])[0], b.forward_batch([t], [1], [0])[0])
    finally:
        a.close()
        b.close()


def test_short_feeds_between_decode_steps(hip, model):  # noqa: F811
    """A chunk of 4: feeds of 10 rows are one captured step over the long steps'
    inputs, replayed between decode steps over the short ones'."""
    a = gpu_engine(model, slots=3, capacity=96, chunk=4)
    b = gpu_engine(model, slots=3, capacity=96, chunk=4)
    try:
        for rep in range(4):
            for slot in (0, 2):
                p = tokens(60 + 3 * rep + slot, 10)
                got = a.feed_slot(slot, p)
                for start in range(0, 10, 4):
                    n = min(4, 10 - start)
                    last = start + n == 10
                    want = b.forward_batch(p[start:start + n], [slot] * n, [n - 1] if last else [])[0]
                assert same_bits(got, want[0]), (rep, slot)
            t = tokens(90 + rep, 3)
            assert same_bits(a.forward_batch(t, [0, 1, 2], [0, 1, 2])[0], b.forward_batch(t, [0, 1, 2], [0, 1, 2])[0]), rep
    finally:
        a.close()
        b.close()


def test_bad_token_feeds_the_chunks_before_it(hip, model):  # noqa: F811
    from needle_cs_amd import NeedleHipError
    p = np.array(tokens(5, 60))
    p[40] = 10**8  # past the vocabulary
    g = gpu_engine(model, slots=1, capacity=96, chunk=16)
    try:
        with pytest.raises(NeedleHipError, match="row 8: token"):
            g.feed_slot(0, p)
        assert g.slot_length(0) == 32
    finally:
        g.close()
