"""The attention forms that make q and the new K / V rows in the blocks that read them: bit-equal to
the split form with its own prep launch, outputs and appended cache rows, at the slots where the
patched K fragments and segment borders lie (first and last slot of a 16-slot tile, a 64-slot
slice, a 128-slot part, a 256-slot chunk), and with a lane named twice (no folding there)."""
import numpy as np
import pytest

from test_gpu_attn_op import Harness, LAYER

pytestmark = pytest.mark.gpu
EDGES = [0, 1, 14, 15, 16, 17, 62, 63, 64, 65, 126, 127, 128, 254, 255, 256, 257, 510, 511, 512, 513, 1020, 1021]


@pytest.fixture(scope="module")
def harness():
    h = Harness(1024, 768)
    yield h
    h.s.close()
    h.e.close()


def rows_at(h, lane, p, T):
    return [np.asarray(h.s.read(lane, n, p + T))[LAYER][:, p:p + T].copy() for n in "kv"]


@pytest.mark.parametrize("T", [1, 2, 3])
@pytest.mark.parametrize("B", [2, 63, 64, 96, 128, 129, 256])
def test_folded_prep_equals_split(harness, B, T):
    h = harness
    rng = np.random.default_rng(B * 4 + T)
    pos = [EDGES[i % len(EDGES)] if i < 2 * len(EDGES) else int(rng.integers(0, 1024 - T)) for i in range(B)]
    pos = [min(p, 1024 - T) for p in rng.permutation(pos).tolist()]
    lanes = rng.permutation(256)[:B].tolist()
    want = h.run(lanes, pos, T, 1)
    check = list(range(0, B, max(1, B // 16)))
    kv = [rows_at(h, lanes[i], pos[i], T) for i in check]
    for i in check:                        # the appended rows must come from the next call
        for n in "kv":
            full = np.asarray(h.s.read(lanes[i], n, pos[i] + T))
            full[LAYER][:, pos[i]:pos[i] + T] = 0
            h.s.write(lanes[i], n, full, pos[i] + T)
    got = h.run(lanes, pos, T, 0)
    assert np.array_equal(got, want)
    for i, (k, v) in zip(check, kv):
        k2, v2 = rows_at(h, lanes[i], pos[i], T)
        assert np.array_equal(k2, k) and np.array_equal(v2, v), (lanes[i], pos[i])


@pytest.mark.parametrize("B, T", [(64, 1), (130, 1), (128, 3)])
def test_lane_named_twice(harness, B, T):
    """Two row groups of one lane, the second right after the first: every row reads both."""
    h = harness
    lanes = list(range(B - 1)) + [0]
    pos = [40] * (B - 1) + [40 + T]
    assert np.array_equal(h.run(lanes, pos, T, 0)[:T * (B - 1)], h.run(lanes, pos, T, 3)[:T * (B - 1)])
