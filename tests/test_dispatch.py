"""The library's choice of kernel for a call, pinned as a table (csrc/vc_dispatch.h compiled for the CPU): from the rank
count and what the last forwarded call on the communicator looked like to lanes per pair of ranks (0 = through the
work-item list, 256 / 64 / 16 = a workgroup / a wavefront / a quarter of one per pair, 1 = a batch of pairs per wavefront)
and whether the call is first tried as one launch on fixed-stride staging.  Every entry point decides through this one
function; a changed threshold shows here."""
import pytest

from tests import emulator as E

LIST, BATCH, QUARTER, WAVE, GROUP = 0, 1, 16, 64, 256
# the last call: (average piece, most pieces of a block, longest block), one piece per pair of ranks
HINTS = {"100 B": (100, 1, 300), "500 B": (500, 1, 1500), "1 KB": (1000, 2, 5000), "2 KB": (2000, 3, 9000),
         "4 KB": (4000, 4, 16000), "4 KB, a block of 20 pieces": (4000, 20, 100000)}
# rank count -> per hint (lanes, fixed stride tried first), radix-2 Bruck
TABLE = {
    16: [(WAVE, True), (WAVE, True), (WAVE, True), (WAVE, True), (GROUP, True), (LIST, False)],       # up to 32 ranks never a quarter
    32: [(WAVE, True), (WAVE, True), (WAVE, True), (WAVE, True), (GROUP, True), (LIST, False)],
    64: [(QUARTER, True), (QUARTER, True), (QUARTER, True), (WAVE, True), (GROUP, False), (LIST, False)],   # a quarter below 1.75 KiB
    128: [(QUARTER, True), (QUARTER, True), (QUARTER, False), (QUARTER, False), (GROUP, False), (LIST, False)],   # ... below 3 KiB; 256 MiB of slots at most
    160: [(BATCH, True), (QUARTER, False), (LIST, False), (LIST, False), (LIST, False), (LIST, False)],     # above 128 ranks: short blocks only
    192: [(BATCH, True), (QUARTER, False), (LIST, False), (LIST, False), (LIST, False), (LIST, False)],
    256: [(BATCH, False), (QUARTER, False), (LIST, False), (LIST, False), (LIST, False), (LIST, False)],    # above 192 ranks no fixed stride
    1024: [(BATCH, False), (QUARTER, False), (LIST, False), (LIST, False), (LIST, False), (LIST, False)],
}


def _hint(P, average, max_pieces, max_len):
    return (1, P * P, average * P * P, max_pieces, max_len)


@pytest.mark.parametrize("P", sorted(TABLE))
def test_default_mode_decision_table(P):
    for (name, h), (lanes, strided) in zip(HINTS.items(), TABLE[P]):
        d = E.dispatch(E.F_TWOPHASE, P, _hint(P, *h), mode=1, r=2)
        assert (d["lanes"], d["stride"] > 0) == (lanes, strided), (P, name, d)
        if strided:
            # slots hold the last call's longest block at any cache-line phase; the batches become quarters there
            assert d["stride"] % 128 == 0 and d["stride"] >= h[2] + 127 and d["max_len"] == d["stride"] - 127
            assert d["stride_lanes"] == (QUARTER if lanes == BATCH else lanes)
        if lanes:
            # the hint is a guess: what the kernel checks on the device before it moves anything
            short = lanes in (BATCH, QUARTER)
            assert (d["max_pieces"], d["max_items"], d["max_average"]) == ((8, 0, 4096) if short else (16, 32768, 0)), (P, name, d)


def test_without_a_hint_and_in_the_forced_modes():
    for P in (8, 64, 1024):
        assert E.dispatch(E.F_TWOPHASE, P, (0, 0, 0, 0, 0), mode=1)["lanes"] == LIST            # the first call on a communicator
        short = _hint(P, 100, 1, 300)
        assert E.dispatch(E.F_TWOPHASE, P, short, mode=0)["lanes"] == LIST                        # launch per digit
        assert E.dispatch(E.F_TWOPHASE, P, short, mode=2)["lanes"] == LIST                        # the list was asked for
        for mode, lanes in ((3, GROUP), (4, QUARTER), (5, BATCH)):
            d = E.dispatch(E.F_TWOPHASE, P, (0, 0, 0, 0, 0), mode=mode)
            assert d == dict(lanes=lanes, stride=0, stride_lanes=0, max_pieces=0, max_items=0, max_average=0, max_len=0)


def test_calls_that_cannot_wait_for_a_list():
    """The _async twins and the entry point that allocates nothing never go through the list and never guard: short blocks by
    the same rule as the blocking calls, everything else a workgroup per pair."""
    for P, expect in ((64, [QUARTER, QUARTER, QUARTER, GROUP, GROUP, GROUP]), (1024, [BATCH, QUARTER, GROUP, GROUP, GROUP, GROUP])):
        for h, lanes in zip(HINTS.values(), expect):
            for mode in (0, 1, 2):
                d = E.dispatch(E.F_TWOPHASE, P, _hint(P, *h), mode=mode, call_kind=1)
                assert d == dict(lanes=lanes, stride=0, stride_lanes=0, max_pieces=0, max_items=0, max_average=0, max_len=0), (P, h, d)
        assert E.dispatch(E.F_TWOPHASE, P, (0, 0, 0, 0, 0), mode=1, call_kind=1)["lanes"] == GROUP


def test_many_digits_and_two_layers():
    # a staging region per digit: 7 regions of 128 x 128 slots of 1.6 KB are 184 MiB, of 5.1 KB more than the 256 MiB allowed
    assert E.dispatch(E.F_TWOPHASE, 128, _hint(128, 500, 1, 1500), r=2)["stride"] == 1664
    assert E.dispatch(E.F_TWOPHASE, 128, _hint(128, 1000, 2, 5000), r=2)["stride"] == 0
    assert E.dispatch(E.F_TWOPHASE, 128, _hint(128, 1000, 2, 5000), r=16)["stride"] == 5248       # two regions
    # the two-layer functions, forwarded, carry every block on its own (no organized region): same rule
    for f in (E.F_TTPL, E.F_TTPL_S1):
        d = E.dispatch(f, 64, _hint(64, 100, 1, 300), n=8, r=2)
        assert (d["lanes"], d["stride"]) == (QUARTER, 512)


def test_lanes_per_work_item_of_the_list_kernels():
    for average, lanes in ((16, QUARTER), (447, QUARTER), (448, WAVE), (3071, WAVE), (3072, GROUP), (4096, GROUP)):
        assert E.lanes_for_items(average * 1000, 1000) == lanes
    assert E.lanes_for_items(0, 0) == GROUP


# calls that stage in a window: a wavefront per pair from 46 ranks up, whatever the average, instead of the list and of workgroups (up to 192 ranks in
# one launch with any room for the slots); batches further up from 512 ranks
WINDOW_TABLE = {
    32: [(WAVE, True), (WAVE, True), (WAVE, True), (WAVE, True), (GROUP, True), (LIST, False)],
    45: [(QUARTER, True), (QUARTER, True), (WAVE, True), (WAVE, True), (GROUP, True), (LIST, False)],
    46: [(QUARTER, True), (QUARTER, True), (WAVE, True), (WAVE, True), (WAVE, True), (LIST, False)],
    64: [(QUARTER, True), (QUARTER, True), (WAVE, True), (WAVE, True), (WAVE, True), (LIST, False)],
    128: [(QUARTER, True), (QUARTER, True), (QUARTER, True), (WAVE, True), (WAVE, True), (LIST, False)],
    192: [(BATCH, True), (QUARTER, True), (QUARTER, True), (WAVE, True), (WAVE, True), (LIST, False)],
    256: [(BATCH, False), (QUARTER, False), (QUARTER, False), (WAVE, False), (WAVE, False), (LIST, False)],
    1024: [(BATCH, False), (BATCH, False), (QUARTER, False), (WAVE, False), (WAVE, False), (LIST, False)],
}


@pytest.mark.parametrize("P", sorted(WINDOW_TABLE))
def test_decision_table_of_calls_that_stage_in_a_window(P):
    for (name, h), (lanes, strided) in zip(HINTS.items(), WINDOW_TABLE[P]):
        d = E.dispatch(E.F_TWOPHASE, P, _hint(P, *h), mode=1, r=2, window=True)
        assert (d["lanes"], d["stride"] > 0) == (lanes, strided), (P, name, d)
        if lanes == WAVE and P >= 46:
            assert (d["max_pieces"], d["max_items"], d["max_average"]) == (16, 0, 0)
        assert E.dispatch(E.F_TWOPHASE, P, _hint(P, *h), window=True, batch=True) == (64 if h[2] <= 128 else 16)
        # a direct function stages nothing: the same with and without
        assert E.dispatch(E.F_SPREADOUT, P, _hint(P, *h), window=True) == E.dispatch(E.F_SPREADOUT, P, _hint(P, *h)), (P, name)
    assert [E.dispatch(E.F_TWOPHASE, P, _hint(P, 60, 1, longest), window=True, batch=True) for longest in (128, 129)] == [64, 16]


@pytest.mark.parametrize("func,P,lines", [(E.F_TWOPHASE, 90, [(0, QUARTER), (960, WAVE)]), (E.F_TWOPHASE, 128, [(768, QUARTER), (1280, WAVE)]),
                                          (E.F_TWOPHASE, 192, [(768, QUARTER), (1024, WAVE)]), (E.F_TWOPHASE, 362, [(768, QUARTER), (1280, LIST), (1344, WAVE)]),
                                          (E.F_TWOPHASE, 363, [(768, QUARTER), (1280, LIST), (1664, WAVE)]), (E.F_SPREADOUT, 64, [(0, QUARTER), (960, WAVE)]),
                                          (E.F_SPREADOUT, 192, [(768, QUARTER), (1664, WAVE)]), (E.F_SPREADOUT, 362, [(768, QUARTER), (1664, WAVE), (3072, LIST)]),
                                          (E.F_SPREADOUT, 363, [(384, QUARTER), (768, LIST), (1920, WAVE), (3072, LIST)])])
def test_lines_of_calls_with_slots_in_closed_form(func, P, lines):
    """A quarter of a wavefront, the list, a wavefront per pair: by the average piece, and by nothing else while no block is more than 8 pieces."""
    for (line, lanes), before in zip(lines, [None] + [lanes for _, lanes in lines]):
        if before is not None:
            assert E.dispatch(func, P, _hint(P, line - 1, 8, 30000), window=True)["lanes"] == before, line
        assert E.dispatch(func, P, _hint(P, line, 8, 30000), window=True)["lanes"] == lanes, line
        if lanes == WAVE:                                 # rows of ranks: the same blocks, most pairs empty
            kept = E.dispatch(func, P, (1, P * P // 8, line * (P * P // 8), 8, 30000), window=True)["lanes"]
            assert kept == (QUARTER if line < (1792 if P < 91 else 3072 if P <= 192 or (func == E.F_SPREADOUT and P <= 362) else 1280) else LIST), line
    # the _async twins, which never use the list
    for average, pieces, lanes in ((2000, 16, WAVE), (2000, 17, GROUP), (3071, 16, WAVE), (3072, 16, GROUP)):
        assert E.dispatch(func, P, _hint(P, average, pieces, 60000), window=True, call_kind=1)["lanes"] == lanes, (average, pieces)


def test_input_that_the_memory_side_cache_holds_is_read_with_ordinary_loads():
    for mode, kind in ((0, 0), (1, 0), (2, 0), (3, 0), (5, 0), (1, 1)):
        for func, limit in ((E.F_TWOPHASE, 24 << 20), (E.F_TTPL, 24 << 20), (E.F_SPREADOUT, 32 << 20)):
            at = lambda payload, valid=1: E.dispatch(func, 64, (valid, 8192, payload, 2, 1 << 13), mode=mode, call_kind=kind, n=8, window=True, cached=True)
            assert [at(0), at(limit), at(limit + 1), at(limit, valid=0)] == [True, True, False, False], (mode, func)


def test_no_single_launch_is_chosen_that_the_launcher_refuses():
    """Only instances without a window signal their own end: who signals and who stages in a window is decided in one place."""
    chosen = set()
    for P in range(3, 33):
        for r in range(2, P):
            digits = next(w for w in range(1, 6) if r ** w >= P)
            for length in list(range(1 << 10, 65537, 3 << 10)) + [50_000, 61_000]:
                pieces = 1 if length <= 8064 else length // 4096 + 2
                for payload in sorted({min(share * P * P * length // 8, 64 << 20) for share in (1, 5, 8)}):
                    hint = (1, max(1, payload // length) * pieces, payload, pieces, length)
                    for window in (False, True):
                        d = E.dispatch(E.F_TWOPHASE, P, hint, r=r, window=window, single=True)
                        assert not d["refused"] and not (d["window"] and not window), (P, r, length, payload, d)
                        assert d["window"] or d["stride"] * P * P * digits <= 256 << 20, (P, r, length, payload, d)
                        chosen.add((d["stride"] > 0, d["self"], d["window"]))
    W = 32 << 20
    assert chosen == {(False, False, 0), (True, True, 0), (True, False, 0), (True, False, W)}
    # above 12 MiB on 16 - 32 ranks: in a window, and then without a signal; and slots that have no room of their own
    for P, r, length in ((32, 4, 16384), (32, 8, 16384), (24, 6, 32768), (16, 2, 50_000)):
        hint = (1, P * P * 5, P * P * length, length // 4096 + 2, length)
        d = E.dispatch(E.F_TWOPHASE, P, hint, r=r, window=True, single=True)
        assert (d["self"], d["window"]) == (False, W), (P, r, length, d)
        assert E.dispatch(E.F_TWOPHASE, P, hint, r=r, single=True)["self"]
    d = E.dispatch(E.F_TWOPHASE, 31, (1, 31 * 31 * 2, 31 * 31 * 6000, 16, 60_000), r=2, window=True, single=True)
    assert (d["self"], d["window"]) == (False, W)


def test_a_call_like_the_last_one_passes_the_guard_of_its_own_shape():
    """What the device refuses is dispatched once more on what it is: that shape must take it."""
    lanes = set()
    for f, P, n in ((E.F_TWOPHASE, 12, 0), (E.F_TWOPHASE, 60, 0), (E.F_TWOPHASE, 128, 0), (E.F_TTPL, 160, 16), (E.F_TWOPHASE, 200, 0), (E.F_TTPL, 352, 32), (E.F_TWOPHASE, 400, 0),
                    (E.F_TTPL_S1, 1024, 32), (E.F_SPREADOUT, 60, 0), (E.F_SPREADOUT, 200, 0), (E.F_SPREADOUT, 362, 0), (E.F_SPREADOUT, 500, 0)):
        for window in (False, True):
            for share in (1, 2, 5, 50):                   # one pair in so many has a block
                for length in [1, 60, 128, 129, 200, 383, 384, 511, 513, 600, 767, 900, 1000, 1100, 1279, 1300, 1400, 1700, 1900, 2040, 2050, 2500, 3071, 3100, 5000, 9000, 20000, 40000]:
                    for uneven in (1, 4):
                        blocks = P * P // share
                        pieces = 1 if length <= 8064 else length // 4096 + 2
                        h = (1, blocks * pieces, blocks * length, pieces * uneven, length * uneven)
                        assert E.dispatch(f, P, h, n=n, window=window, single=True)["passes"], (f, P, window, h)
                        lanes.add(E.dispatch(f, P, h, n=n, window=window)["lanes"])
    assert lanes == {LIST, BATCH, QUARTER, WAVE, GROUP}


def test_runs_only_where_wavefronts_can_move_them():
    """A call that stages outside a window (an allowance of its own, the forced batches, the entry point that allocates nothing) has a tile with a block of two
    hops moved a lane a block: below a radix of a quarter of the ranks, where nearly every tile has one, it gets the instance without runs.  One that stages
    nothing needs no window."""
    for longest, vectors in ((16, 1), (32, 2), (64, 4)):
        hint = _hint(512, longest // 2, 1, longest)
        for mode, kind in ((1, 0), (1, 1), (5, 0)):
            at = lambda func, window, n=16, r=2: E.dispatch(func, 512, hint, mode=mode, call_kind=kind, n=n, r=r, window=window, run=True)
            assert [at(E.F_TWOPHASE, window, r=r) for r in (23, 127, 128, 511) for window in (True, False)] == [vectors, 0] * 2 + [vectors] * 4, (longest, mode, kind)
            assert [at(E.F_TTPL, False, n, r) for n, r in ((16, 16), (128, 127), (256, 127), (256, 255))] == [0, 0, 0, vectors], (longest, mode, kind)
            assert [at(E.F_SPREADOUT, window) for window in (True, False)] == [vectors] * 2, (longest, mode, kind)


def _run(P, longest, esz=1, r=2, func=E.F_TWOPHASE, payload=None):
    """Vectors of a run of a call in a window behind one of blocks of `longest` bytes; payload: half of `longest` for every pair."""
    return E.dispatch(func, P, (1, P * P, longest * P * P // 2 if payload is None else payload, 1, longest), r=r, esz=esz, window=True, run=True)


def test_vectors_of_a_run():
    """vc_run_vectors on both sides of each of its lines.  Hop slots of the Bruck functions here: digits of the ranks and one; of the direct ones, one."""
    direct = lambda P, longest, esz=1: _run(P, longest, esz, func=E.F_SPREADOUT)
    lengths = (4, 5, 16, 17, 32, 33, 64, 65)
    # 512 ranks, two digits (three slots): by the longest block and the element
    for esz, vectors in ((1, [0, 1, 1, 2, 2, 4, 4, 0]), (3, [0, 1, 1, 2, 2, 4, 4, 0]), (2, [0, 1, 1, 2, 2, 0, 0, 0]), (4, [0, 1, 1, 2, 2, 0, 0, 0]), (8, [0] * 8), (16, [0] * 8)):
        assert [_run(512, longest, esz, r=23) for longest in lengths] == vectors, esz
        assert [_run(511, longest, esz, r=23) for longest in lengths] == [0] * 8, esz          # too few ranks
        # nothing staged: one slot
        assert [direct(1000, longest, esz) for longest in lengths] == vectors, esz
        assert [direct(511, longest, esz) for longest in lengths] == [0] * 8, esz
    # runs of one and two vectors: routes of up to seven slots (six digits), from 2048 ranks on of any number
    assert [_run(729, 16, r=3), _run(730, 16, r=3), _run(729, 32, r=3), _run(730, 32, r=3)] == [1, 0, 2, 0]
    assert [_run(2047, 16), _run(2048, 16), _run(2047, 32), _run(2048, 32)] == [0, 1, 0, 2]
    assert [_run(P, 64) for P in (512, 2047, 2048)] == [4] * 3
    # elements of two and four bytes: two vectors with up to four slots; four where there is staging and 2^19 pairs
    for esz in (2, 4):
        assert [_run(512, 32, esz, r=r) for r in (8, 7)] == [2, 0], esz
        assert [_run(P, 64, esz, r=32) for P in (724, 725)] == [0, 4] and direct(1000, 64, esz) == 0, esz
    # more than one vector: blocks that average an eighth of the longest
    for longest, vectors in ((16, 1), (17, 2), (32, 2), (64, 4)):
        least = -(-512 * 512 * longest // 8)
        assert [_run(512, longest, r=23, payload=p) for p in (least, least - 1)] == [vectors, 1 if longest == 16 else 0], longest
    assert E.dispatch(E.F_TWOPHASE, 512, (0, 0, 0, 0, 0), r=23, window=True, run=True) == 0       # no hint
