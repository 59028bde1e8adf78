"""Engines whose capacity is past 512 positions while their spans are not: the
decode steps up to position 511 take the short spans' attention launches, later
ones the general kernels.  Both engines cross that line with the bits of the
same text in steps of several rows, which never take the one-launch forms."""
import numpy as np
import pytest

from test_needle3_step_gpu import archive, gpu_engine, model, same_bits, tokens  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("start", [60, 506])
@pytest.mark.parametrize("slots", [1, 3, 7])
def test_needle3_steps_across_the_short_span(hip, model, start, slots):  # noqa: F811
    a = gpu_engine(model, slots=slots, capacity=640, chunk=64)
    b = gpu_engine(model, slots=slots, capacity=640, chunk=64)
    text = [np.array(tokens(40 + s, start + 12)) for s in range(slots)]
    every = list(range(slots))
    try:
        for e in (a, b):
            for s in every:
                e.feed_slot(s, text[s][:start], compute_logits=False)
        for step in range(0, 12, 2):
            got = [a.forward_batch([text[s][start + step + k] for s in every], every, every)[0] for k in (0, 1)]
            pairs = np.concatenate([text[s][start + step:start + step + 2] for s in every])
            want = b.forward_batch(pairs, np.repeat(every, 2), list(range(2 * slots)))[0]
            for k in (0, 1):
                assert same_bits(got[k], want[k::2]), (step, k)
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("start", [100, 508])
def test_decoder_steps_across_the_short_span(hip, start):
    from needle_cs_amd.decoder import CONFIG4, GpuDecoder, synthetic_model
    model_ = synthetic_model(dict(CONFIG4, layers=1), 5)
    rng = np.random.default_rng(9)
    text = rng.integers(4, CONFIG4["vocab"], start + 8, dtype=np.int32)
    one, many = GpuDecoder(model_, slots=2, capacity=700, max_rows=600), GpuDecoder(model_, slots=2, capacity=700,
                                                                                    max_rows=600)
    for d in (one, many):
        d.step(text[:start], [1] * start, [], logits=False)
    want = many.step(text[start:], [1] * 8, list(range(8)), k=1)[0]
    for i in range(8):
        got = one.step(text[start + i:start + i + 1], [1], [0], k=1)[0]
        assert np.array_equal(got.view(np.uint32), want[i:i + 1].view(np.uint32)), i
