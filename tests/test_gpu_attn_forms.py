"""The attention forms that make q and the new K / V rows in the blocks that read them: bit-equal to
the split form with its own prep launch, outputs and appended cache rows, at the slots where the
patched K fragments and segment borders lie (first and last slot of a 16-slot tile, a 64-slot
slice, a 128-slot part, a 256-slot chunk), and with a lane named twice (no folding there)."""
import numpy as np
import pytest

from test_gpu_attn_op import Harness, LAYER, bf16_val

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


def clear_slots(h, lane, p, n):
    """Zero K and V in slots p .. p + n: the rows a call appends there must be its own."""
    for kv in "kv":
        full = np.asarray(h.s.read(lane, kv, p + n))
        full[LAYER][:, p:p + n] = 0
        h.s.write(lane, kv, full, p + n)


def run_from(h, row, lanes, pos, T, form):
    """Harness.run on the projection rows from `row` on."""
    h.out.fill_(0)
    h.e.op_attn_decode(h.s, LAYER, lanes, pos, T, h.proj[row:].data_ptr(), h.qn.data_ptr(), h.kn.data_ptr(),
                       h.out.data_ptr(), form)
    return h.out[:len(lanes) * T].view(h.torch.int16).cpu().numpy().view(np.uint16).copy()


def prepared_q(h):
    """Row 0's q at position 500 in the q scratch (four rows of a lane always take the prep launch): a
    later call's prep launch writes its own over it, a form that makes q in its blocks leaves it."""
    h.run([1], [500], 4, 1)
    return h.e.read_scratch("q", (2048,), np.float32)


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


@pytest.mark.parametrize("T", [2, 3])
def test_segments_equal_split(T):
    """Verify rows of 31 lanes (the segment form) at the borders of its chunks (256 slots) and P.V
    segments (512), rows that straddle them, a lane of one segment and an empty one, some of 7,000
    slots and more, and with a lane named twice (q and K / V rows from the prep launch)."""
    h = Harness(8192, 128)
    try:
        pos = [0, 1, 62, 126, 253, 254, 255, 256, 509, 510, 511, 512, 513, 1022, 1023, 1024, 1535, 2047, 2048, 2303,
               2558, 2815, 4095, 8192 - T]
        pos += [int(p) for p in np.random.default_rng(T).integers(7000, 8190, 7)]
        lanes = np.random.default_rng(T).permutation(256)[:31].tolist()
        want = h.run(lanes, pos, T, 1)
        for i in range(31):
            clear_slots(h, lanes[i], pos[i], T)
        before = prepared_q(h)
        assert np.array_equal(h.run(lanes, pos, T, 0), want)
        assert np.array_equal(h.e.read_scratch("q", (2048,), np.float32), before)
        for i in (0, 6, 11, 23):
            h.check_lane(i, lanes[i], pos[i], T, want)
        lanes[5] = lanes[6]                 # a second group of the lane, right after the first
        pos[5] = pos[6] + T
        rest = [i for i in range(31) if i != 5]
        clear_slots(h, lanes[6], pos[6], 2 * T)
        first = h.run(lanes, [p if i != 5 else 8000 for i, p in enumerate(pos)], T, 1)   # group 5 elsewhere for now
        last = run_from(h, 5 * T, [lanes[5]], [pos[5]], T, 1)
        clear_slots(h, lanes[6], pos[6], 2 * T)
        before = prepared_q(h)
        got = h.run(lanes, pos, T, 0).reshape(31, T, 2048)
        assert not np.array_equal(h.e.read_scratch("q", (2048,), np.float32), before)
        assert np.array_equal(got[rest], first.reshape(31, T, 2048)[rest])
        assert np.array_equal(got[5], last)
    finally:
        h.s.close()
        h.e.close()


@pytest.mark.parametrize("T", [2, 3])
def test_few_long_lanes_equal_split(T):
    """100 lanes of which one has 8,000 slots and the others at most 1,000: by segments (in the rows
    form the long lane's block would run alone), the same bits as the split form and the rows form."""
    h = Harness(8192, 300)
    try:
        pos = [8000] + [int(p) for p in np.random.default_rng(T).integers(0, 1000, 99)]
        lanes = np.random.default_rng(T).permutation(256)[:100].tolist()
        want = h.run(lanes, pos, T, 1)
        for form in (0, 5):
            for i in range(0, 100, 9):
                clear_slots(h, lanes[i], pos[i], T)
            assert np.array_equal(h.run(lanes, pos, T, form), want), form
    finally:
        h.s.close()
        h.e.close()


@pytest.mark.parametrize("lanes, ctx, T, segments", [
    (1, 500, 3, False), (1, 4096, 3, False), (3, 500, 3, False), (3, 4096, 2, False), (8, 500, 3, False), (8, 4096, 3, True),
    (4, 16000, 2, True), (24, 500, 2, False)])
def test_form_by_context_not_capacity(lanes, ctx, T, segments):
    """A state of 16,384 slots per lane: verify rows go by the slots in use (segments make q in their
    blocks; the split path's comes from the prep launch), and the bits are the split path's."""
    h = Harness(16384, 128)
    try:
        pos = [ctx - T - 7 * i for i in range(lanes)]
        before = prepared_q(h)
        got = h.run(list(range(lanes)), pos, T, 0)
        assert np.array_equal(h.e.read_scratch("q", (2048,), np.float32), before) == segments
        assert np.array_equal(got, h.run(list(range(lanes)), pos, T, 1))
    finally:
        h.s.close()
        h.e.close()


@pytest.mark.parametrize("T", [2, 3])
@pytest.mark.parametrize("form, rows", [(5, 1), (5, 2), (0, 2)])
def test_later_rows_stay_out_of_earlier_ones(T, form, rows):
    """A non-finite row (its V infinite, or all of its projection NaN) is cached behind the lane's
    earlier rows only: those keep the split form's bits, which attends over slots 0 .. p + t. Rows that
    lie in one part (128 slots), end one and straddle two; the rows form in both block sizes and,
    through auto, the segments (whose P.V segments are 512 slots: a lane of one, lanes of several)."""
    h = Harness(8192, 192)
    try:
        h.e.set_option("attn_rows", rows)
        pos = [0, 1, 5, 63, 124, 125, 126, 127, 128, 254, 255, 256, 509, 510, 511, 512, 1021, 1022, 1023, 1024]
        pos += [8000 - 131 * i for i in range(20)]                     # enough slots in all for the segments
        n = len(pos)
        lanes = np.random.default_rng(T).permutation(256)[:n].tolist()
        bits = h.proj.view(h.torch.int16)
        good = bits.clone()
        for bad in range(1, T):
            for cols, value in ((slice(4608, 5120), 0x7F80), (slice(0, 5120), 0x7FC0)):
                bits.copy_(good)
                bits[bad:n * T:T, cols] = value
                want = h.run(lanes, pos, T, 1).reshape(n, T, 2048)
                got = h.run(lanes, pos, T, form).reshape(n, T, 2048)
                assert np.isfinite(bf16_val(want[:, :bad])).all()
                assert np.array_equal(got[:, :bad], want[:, :bad]), (bad, hex(value), np.argwhere(
                    (got[:, :bad] != want[:, :bad]).any(-1))[:8].tolist())
                assert np.array_equal(np.isfinite(bf16_val(got)), np.isfinite(bf16_val(want)))
    finally:
        h.s.close()
        h.e.close()


@pytest.mark.parametrize("B, T, form", [(2, 1, 0), (2, 1, 1), (2, 1, 2), (63, 1, 0), (64, 1, 0), (64, 1, 3), (130, 1, 0),
                                         (130, 1, 4), (2, 3, 0), (2, 2, 5), (96, 2, 5), (128, 3, 0)])
def test_lane_named_twice(harness, B, T, form):
    """Two row groups of one lane, the second right after the first and reading its rows: every row
    equals the two groups' calls one after the other (slots to be appended cleared before each), and
    q comes from the prep launch, which appends every K / V row before any block reads one."""
    h = harness
    lanes = list(range(B - 1)) + [0]
    pos = [40] * (B - 1) + [40 + T]
    clear_slots(h, 0, 40, 2 * T)
    want = [run_from(h, 0, lanes[:-1], pos[:-1], T, 1), run_from(h, (B - 1) * T, lanes[-1:], pos[-1:], T, 1)]
    clear_slots(h, 0, 40, 2 * T)
    before = prepared_q(h)
    got = h.run(lanes, pos, T, form)
    assert np.array_equal(got, np.concatenate(want))
    assert not np.array_equal(h.e.read_scratch("q", (2048,), np.float32), before)
