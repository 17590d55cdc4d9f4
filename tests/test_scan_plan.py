"""How the chunked recurrences divide a batch among workgroups (chunk_scan.h), without a GPU."""
import random

import pytest

from agentic_traffic_testing_amd.ops import mixers as mx

RETENTION, FORGET, STATE_SPACE, DELTA, DELTA_CHANNEL = range(5)


@pytest.fixture(scope="module")
def plan():
    if not mx.load_native(build_if_missing=False):
        pytest.skip("mixer library not built")
    names = ("route", "waves", "heads", "cols", "chunks", "states", "floats")
    return lambda *a: dict(zip(names, mx._native().scan_plan(*a)))


def segments(n, chunks):
    """Segments of a portion of n chunks (scan_segment_chunks)."""
    P = (4 * n + chunks) // (4 * chunks)
    return 1 if P < 2 else -(-n // -(-n // P))


def test_segment_states_hold_any_batch(plan):
    """The scratch has room for the segments of every batch with these sums, whatever the portions' lengths are."""
    rng = random.Random(5)
    for _ in range(20000):
        S = rng.choice((1, 1, 2, 3, 5, 8, 30))
        lens = [rng.choice((1, 7, 16 * rng.randint(1, 40) + rng.choice((-1, 0, 1)), rng.randint(1, 4000))) for _ in range(S)]
        H, dk, dv = rng.choice((1, 2, 8, 32, 96)), rng.choice((64, 128)), rng.choice((40, 64, 128, 256))
        mode = rng.choice((RETENTION, FORGET, STATE_SPACE))
        p = plan(sum(lens), S, H, H, dk, dv, mode)
        if p["states"]:
            n = [segments(-(-x // 16), p["chunks"]) for x in lens]
            assert sum(x for x in n if x > 1) <= p["states"], (lens, H, dv, p)


@pytest.mark.parametrize("mode", [RETENTION, FORGET, STATE_SPACE])
@pytest.mark.parametrize("H,G,dv,T,S", [(32, 8, 128, 1400, 4), (32, 8, 128, 8000, 4), (8, 8, 128, 8192, 16), (16, 16, 256, 1400, 4),
                                        (96, 8, 64, 2000, 2), (64, 64, 64, 8000, 4)])
def test_portions_that_fill_the_chip(plan, mode, H, G, dv, T, S):
    """192 - 256 units of 64 columns fill the chip, and uncut if they are of one length: narrow workgroups, and no segments
    that such portions are cut into."""
    p = plan(T, S, H, G, 128, dv, mode)
    assert (p["waves"], p["heads"], p["cols"]) == (4, 1, 64)
    assert p["states"] == 0 or segments(-(-T // S // 16), p["chunks"]) == 1


@pytest.mark.parametrize("H,G,dk,dv,T,mode,most", [
    (64, 64, 64, 64, 2048, RETENTION, 256), (64, 64, 128, 64, 2048, FORGET, 256), (48, 48, 128, 64, 4096, STATE_SPACE, 256),
    (64, 64, 64, 64, 2048, FORGET, 512), (96, 8, 128, 64, 2048, RETENTION, 512), (96, 32, 128, 64, 1500, STATE_SPACE, 512)])
def test_segments_fill_the_workgroups_that_run(plan, H, G, dk, dv, T, mode, most):
    """One long prompt in workgroups of 64 columns: as many as run at once (256, the forget gate's of keys of 64 twice), or
    twice where the heads do not divide that; at least 3 / 4 of them."""
    p = plan(T, 1, H, G, dk, dv, mode)
    assert p["waves"] == 4 and 0.75 * most <= H * segments(-(-T // 16), p["chunks"]) <= most


@pytest.mark.parametrize("H,G,dv,T,S,shape", [
    (32, 8, 128, 2048, 1, (8, 1, 128)), (96, 8, 64, 1023, 1, (8, 2, 64)), (96, 32, 64, 1023, 1, (4, 1, 64)),
    (8, 8, 128, 8192, 1, (4, 1, 64)), (32, 8, 128, 4096, 8, (8, 1, 128)), (32, 8, 128, 191, 64, (4, 1, 64))])
def test_shapes_of_the_walk(plan, H, G, dv, T, S, shape):
    p = plan(T, S, H, G, 128, dv, STATE_SPACE)
    assert (p["waves"], p["heads"], p["cols"]) == shape
    for mode in (DELTA, DELTA_CHANNEL):
        q = plan(T, S, H, G, 128, dv, mode)
        assert (q["waves"], q["states"]) == (4, 0)


@pytest.mark.parametrize("mode,dk,floats", [(RETENTION, 64, 320), (STATE_SPACE, 128, 320), (DELTA, 64, 576), (FORGET, 13, 320 + 16 * 64),
                                            (FORGET, 64, 320 + 16 * 64), (FORGET, 72, 320 + 16 * 128),
                                            (DELTA_CHANNEL, 64, 576 + 16 * 64), (DELTA_CHANNEL, 128, 576 + 16 * 128)])
def test_scratch_per_chunk(plan, mode, dk, floats):
    """A chunk's record holds the decays that the recurrence keeps, at the width of its keys, and nothing for others."""
    H, dv, T, S = 4, 64, 800, 3
    p = plan(T, S, H, H, dk, dv, mode)
    assert p["floats"] == (T // 16 + S) * H * floats + p["states"] * H * (dk * dv + 128)
