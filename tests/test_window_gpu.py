"""Staging in a window (the default mode): layouts below, at and beyond it, through every kind of copy kernel, against the definition."""
import numpy as np
import pytest
import torch

from rbruck_alltoallv_amd import workloads as W

pytestmark = pytest.mark.gpu
WINDOW, CHUNK = 32 << 20, 8192


def _equal(P, length):
    return np.full((P, P), length, dtype=np.int32)


def _mixed(P, hi, seed=5):
    counts = np.random.default_rng(seed).integers(0, hi, (P, P)).astype(np.int32)
    counts[::5, ::7] = min(10 * hi, 150_001)
    return counts


# function, tunables, counts, element size, layout of the arenas.  Four ranks at radix 2 stage four blocks: 8 MiB blocks fill the window exactly.
CASES = {
    "at the window": ("twophase_rbruck_alltoallv", (2,), _equal(4, 8 << 20), 1, 0),
    "one line beyond": ("twophase_rbruck_alltoallv_om", (2,), _equal(4, (8 << 20) + 128), 1, 0),
    "below": ("twophase_rbruck_alltoallv", (3,), _equal(4, 1 << 20), 1, 1),
    "workgroups, odd addresses": ("tuna_algorithm", (2, 0), _mixed(40, 60_000), 1, 1),
    "wavefronts": ("TTPL_rbruck_alltoallv", (8, 2), _mixed(160, 2_100), 1, 1),
    "quarters from the list": ("TTPL_BT_alltoallv_s1", (64, 2, 0), np.where(_mixed(512, 60) > 60, 2_000, _mixed(512, 60)).astype(np.int32), 4, 1),
    "quarters": ("TTPL_BT_alltoallv", (30, 2, 0), np.random.default_rng(1).integers(0, 1100, (300, 300)).astype(np.int32), 1, 0),
    "batches, a lane a block": ("tuna_algorithm", (2, 0), np.random.default_rng(2).integers(0, 17, (512, 512)).astype(np.int32), 1, 0),
    "batches, a quarter a block": ("twophase_rbruck_alltoallv", (4,), np.random.default_rng(3).integers(0, 300, (512, 512)).astype(np.int32), 1, 1),
    "a lane a block, every length": ("TTPL_BT_alltoallv_s1", (26, 5, 0), (np.arange(260 * 260).reshape(260, 260) % 129).astype(np.int32), 1, 1),
    "one byte too long for a lane": ("twophase_rbruck_alltoallv", (3,), (np.arange(260 * 260).reshape(260, 260) % 130).astype(np.int32), 1, 1),
    "direct, a lane a block": ("spreadout_alltoallv", (), (np.arange(260 * 260).reshape(260, 260) % 43).astype(np.int32), 3, 1),
    "a wavefront a pair, no list": ("TTPL_BT_alltoallv", (23, 3, 0), np.random.default_rng(9).integers(0, 6_000, (207, 207)).astype(np.int32), 1, 0),
    "a wavefront a pair, no list, up to 16 pieces": ("twophase_rbruck_alltoallv", (14,), np.where(np.arange(196 * 196).reshape(196, 196) % 61 == 0, 61_000, 3_001).astype(np.int32), 1, 1),
    "a wavefront a pair, one launch, whole pieces": ("tuna_algorithm", (4, 0), _equal(46, 16384), 1, 0),
    "a wavefront a pair, one launch, odd addresses": ("TTPL_BT_alltoallv_s1", (12, 3, 0), np.random.default_rng(10).integers(0, 20_000, (180, 180)).astype(np.int32), 1, 1),
    "direct, a wavefront a pair": ("MPICH_intra_scattered", (0,), np.random.default_rng(11).integers(0, 4_500, (210, 210)).astype(np.int32), 1, 1),
    "nearly all of one hop, whole pieces": ("tuna_algorithm", (63, 0), _equal(64, 100_000), 1, 0),
    "nearly all of one hop, odd addresses": ("twophase_rbruck_alltoallv", (100,), np.random.default_rng(12).integers(0, 12_000, (110, 110)).astype(np.int32), 1, 1),
    "one launch": ("twophase_rbruck_alltoallv", (2,), np.random.default_rng(4).integers(0, 2500, (100, 100)).astype(np.int32), 1, 1),
    "one launch, workgroups in a window": ("twophase_rbruck_alltoallv", (2,), np.random.default_rng(6).integers(0, 30_000, (41, 41)).astype(np.int32), 1, 1),
    "one launch, wavefronts in a window": ("tuna_algorithm", (2, 0), np.random.default_rng(7).integers(0, 1700, (100, 100)).astype(np.int32), 3, 1),
    "one launch, quarters": ("TTPL_BT_alltoallv", (48, 2, 0), np.random.default_rng(8).integers(0, 1200, (192, 192)).astype(np.int32), 4, 0),
    "one launch that signals its end": ("twophase_rbruck_alltoallv_om", (2,), np.random.default_rng(4).integers(0, 12_000, (31, 31)).astype(np.int32), 1, 1),
}


@pytest.mark.parametrize("case", CASES)
def test_staging_window(case):
    from rbruck_alltoallv_amd import api
    name, tun, counts, esz, layout = CASES[case]
    packed = name == "TTPL_BT_alltoallv"
    prob = W.make_problem(counts, esz, layout, 0 if packed else layout)
    dp = api.DeviceProblem(prob)
    fn = getattr(api, name)
    ds, dr = dp.new_send_arena(), dp.new_recv_arena()
    dp.fill_payload(0, 9, ds)
    dp.comm.set_forwarding(2)
    dp.comm.set_staging_bound(0)
    assert fn(*tun, dp, ds, dr) == 0 and dp.verify(ds, dr, packed) == 0, dp.comm.error()
    want, slots = dr.clone(), dp.comm.last_stats().staging_bytes      # every slot in a place of its own
    dp.comm.free()
    dp = api.DeviceProblem(prob)
    dp.comm.set_forwarding(1)
    ran = []
    for _ in range(4):                                    # through the list, then on the hint of the call before
        dr.fill_(0xEE)
        assert fn(*tun, dp, ds, dr) == 0, dp.comm.error()
        assert torch.equal(dr, want), (case, ran)
        st = dp.comm.last_stats()
        ran.append((int(st.execution), int(st.lanes_per_item), int(st.staging_bytes)))
        assert st.execution == 3 or st.staging_bytes <= WINDOW + CHUNK
        if st.execution == 1:                             # (slots of a fixed stride take more)
            assert st.staging_bytes == (slots if slots <= WINDOW else WINDOW + CHUNK), (ran, slots)
    print(case, slots, ran, flush=True)
    plan = api.Plan(name, dp, dr, n=tun[0] if "TTPL" in name else 0, r=tun[1] if "TTPL" in name else (tun + (2,))[0])
    assert plan.rc == 0, dp.comm.error()
    for _ in range(2):
        dr.fill_(0xEE)
        assert plan.execute(ds, dr) == 0 and torch.equal(dr, want)
    plan.free()
    if name in ("twophase_rbruck_alltoallv", "twophase_rbruck_alltoallv_om", "tuna_algorithm", "TTPL_BT_alltoallv", "TTPL_BT_alltoallv_s1"):
        for _ in range(2):
            dr.fill_(0xEE)
            assert api.call_async(name, tun, dp, ds, dr, torch.cuda.current_stream()) == 0 and dp.comm.wait() == 0, dp.comm.error()
            assert torch.equal(dr, want)
    dp.comm.free()


@pytest.mark.parametrize("limit,name,tun,P", [(24, "twophase_rbruck_alltoallv", (2,), 16), (24, "tuna_algorithm", (2, 0), 40), (24, "twophase_rbruck_alltoallv", (4,), 110),
                                              (24, "TTPL_BT_alltoallv_s1", (10, 2, 0), 190), (24, "TTPL_BT_alltoallv", (32, 4, 0), 256), (24, "TTPL_rbruck_alltoallv", (12, 3), 300),
                                              (24, "twophase_rbruck_alltoallv_om", (8,), 520), (32, "spreadout_alltoallv", (), 100), (32, "MPICH_intra_scattered", (0,), 310)])
def test_calls_at_the_limit_of_ordinary_loads(limit, name, tun, P):
    """Payloads just below and just above the limit, the input rewritten between the calls."""
    from rbruck_alltoallv_amd import api
    for payload in ((limit << 20) * 63 // 64, (limit << 20) * 65 // 64):
        mean = payload // P ** 2
        counts = np.random.default_rng(P).integers(mean - mean // 8, mean + mean // 8 + 1, (P, P)).astype(np.int32)
        assert (int(counts.sum()) > limit << 20) == (payload > limit << 20)
        prob = W.make_problem(counts, 1, 1, 0 if name == "TTPL_BT_alltoallv" else 1)
        dp = api.DeviceProblem(prob)
        ds, dr = dp.new_send_arena(), dp.new_recv_arena()
        for turn in range(4):
            dp.fill_payload(0, turn, ds)
            dr.fill_(0xEE)
            assert getattr(api, name)(*tun, dp, ds, dr) == 0, dp.comm.error()
            assert dp.verify(ds, dr, name == "TTPL_BT_alltoallv") == 0, (payload, turn)
        if name in ("tuna_algorithm", "TTPL_BT_alltoallv"):
            plan = api.Plan(name, dp, dr, n=tun[0] if "TTPL" in name else 0, r=tun[1] if "TTPL" in name else tun[0])
            dr.fill_(0xEE)
            assert plan.rc == 0 and plan.execute(ds, dr) == 0 and dp.verify(ds, dr, name == "TTPL_BT_alltoallv") == 0
            plan.free()
        dp.comm.free()


def test_plan_with_a_window_in_a_graph():
    """Replays of a captured plan, with another call on the communicator between them, leave what an eager call leaves."""
    from rbruck_alltoallv_amd import api
    prob = W.make_problem(_mixed(64, 9_000), 4, 1, 1)
    dp = api.DeviceProblem(prob)
    ds, dr = dp.new_send_arena(), dp.new_recv_arena()
    dp.fill_payload(0, 4, ds)
    plan = api.Plan("tuna_algorithm", dp, dr, r=2)
    assert plan.rc == 0 and plan.execute(ds, dr) == 0 and dp.comm.last_stats().staging_bytes == WINDOW + CHUNK
    want = dr.clone()
    assert dp.verify(ds, dr) == 0
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        dp.comm.use_current_stream()
        assert plan.execute_async(ds, dr) == 0
    dp.comm.use_current_stream()
    for _ in range(4):
        dr.fill_(0xEE)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(dr, want)
        dr.fill_(0xEE)
        assert api.twophase_rbruck_alltoallv(8, dp, ds, dr) == 0 and torch.equal(dr, want)
    del graph
    plan.free()
    dp.comm.free()


@pytest.mark.parametrize("P,name,tun", [(193, "tuna_algorithm", (3, 0)), (256, "twophase_rbruck_alltoallv", (2,)), (510, "TTPL_BT_alltoallv", (30, 4, 0)),
                                        (513, "TTPL_rbruck_alltoallv", (27, 3)), (1024, "TTPL_BT_alltoallv_s1", (32, 32, 0)),
                                        (1027, "twophase_rbruck_alltoallv_om", (32,)), (1030, "TTPL_BT_alltoallv", (103, 103, 0)), (201, "spreadout_alltoallv", ())])
def test_the_check_counts_what_the_planner_counts(P, name, tun):
    """Calls without a list are checked and counted by a kernel of their own: same totals, same verdict, same bytes as through the list."""
    from rbruck_alltoallv_amd import api
    packed = name == "TTPL_BT_alltoallv"
    counts = np.random.default_rng(P).integers(0, 250, (P, P)).astype(np.int32)
    counts[::7, ::3] = 0
    counts[P - 1, P - 1], counts[3, P - 2] = 9_001, 20_003
    prob = W.make_problem(counts, 1, 1, 0 if packed else 1)
    dp = api.DeviceProblem(prob)
    fn = getattr(api, name)
    ds, dr = dp.new_send_arena(), dp.new_recv_arena()
    dp.fill_payload(0, 9, ds)

    def totals(mode, rc=0):
        dp.comm.set_forwarding(mode)
        dr.fill_(0xEE)
        assert fn(*tun, dp, ds, dr) == rc, dp.comm.error()
        assert bool((dr == 0xEE).all()) if rc else dp.verify(ds, dr, packed) == 0
        st = dp.comm.last_stats()
        return int(st.execution), (st.payload_bytes, st.moved_bytes, st.block_pieces, st.max_block_pieces, st.max_block_bytes, st.bad_table_entries)

    listed, checked = totals(2), totals(1)
    assert (listed[0], checked[0]) == (1, 2) and checked[1] == listed[1]
    for table, at, value in (("recvcounts", (P - 1, 0), 77), ("sdispls", (P - 2, 5), -3), ("sendcounts", (0, P - 1), -1)) + (() if packed else (("rdispls", (5, P - 1), -9),)):
        t = getattr(dp, table)
        keep = int(t[at])
        t[at] = value
        want = totals(2, -7)[1][-1]
        assert totals(1, -7)[1][-1] == want > 0, table
        t[at] = keep
    assert totals(1) == checked                           # (the hint is still that of the last good call)
    dp.comm.free()


@pytest.mark.parametrize("P,esz", [(21, 1), (20, 24), (130, 8)])
def test_the_check_on_long_blocks(P, esz):
    """Blocks beyond the check's 32-bit sums, through the _async twin of a communicator's first call, which has nothing to choose a shape by."""
    from rbruck_alltoallv_amd import api
    counts = np.random.default_rng(P).integers(0, 40_000 // esz, (P, P)).astype(np.int32)
    counts[1::5, ::4] = 300_001 // esz
    counts[P - 1, 0] = 20_000_011 // esz
    prob = W.make_problem(counts, esz, 0, 1)
    dp = api.DeviceProblem(prob)
    ds, dr = dp.new_send_arena(), dp.new_recv_arena()
    dp.fill_payload(0, 9, ds)
    dp.comm.set_forwarding(2)
    assert api.twophase_rbruck_alltoallv(2, dp, ds, dr) == 0
    want, st = dr.clone(), dp.comm.last_stats()
    listed = (st.payload_bytes, st.moved_bytes, st.block_pieces, st.max_block_pieces, st.max_block_bytes)
    dp.comm.free()
    dp = api.DeviceProblem(prob)
    for _ in range(2):
        dr.fill_(0xEE)
        assert api.call_async("twophase_rbruck_alltoallv", (2,), dp, ds, dr, torch.cuda.current_stream()) == 0 and dp.comm.wait() == 0, dp.comm.error()
        st = dp.comm.last_stats()
        assert torch.equal(dr, want) and st.execution == 2
        assert (st.payload_bytes, st.moved_bytes, st.block_pieces, st.max_block_pieces, st.max_block_bytes) == listed
    dp.comm.free()


def _few_long(P, length, longest):
    counts = _equal(P, length)
    counts[1, P - 1] = counts[P - 2, 0] = longest
    return counts


@pytest.mark.parametrize("r,counts", [(4, _equal(32, 16384)), (8, _equal(32, 16384)), (6, _equal(24, 32768)), (16, _equal(24, 32768)), (4, _equal(20, 32768)),
                                      (2, _equal(16, 50_000)), (5, _mixed(27, 30_000, 3).clip(0, 60_000)), (5, _mixed(27, 40_000, 3).clip(0, 60_000)),
                                      (2, _few_long(31, 8_000, 60_000)), (2, _few_long(20, 8_000, 60_000))])
def test_single_launch_on_few_ranks_with_long_blocks(r, counts):
    """Up to 32 ranks: one launch that signals its own end has no window; one of more than 12 MiB, or whose slots have no room of their own,
    stages in the window and is waited for."""
    from rbruck_alltoallv_amd import api
    prob = W.make_problem(counts, 1, 1, 1)
    dp = api.DeviceProblem(prob)
    ds, dr = dp.new_send_arena(), dp.new_recv_arena()
    for turn in range(3):
        dp.fill_payload(0, turn, ds)
        dr.fill_(0xEE)
        assert api.twophase_rbruck_alltoallv(r, dp, ds, dr) == 0, (turn, dp.comm.error())
        assert dp.verify(ds, dr) == 0
        st = dp.comm.last_stats()
        assert st.execution == (3 if turn else 1), turn
    P, stride = len(counts), -(-(int(counts.max()) + 127) // 128) * 128
    slots = next(w for w in range(1, 6) if r ** w >= P) * P * P * stride
    assert st.staging_bytes == (slots if int(counts.sum()) <= 12 << 20 and slots <= 256 << 20 else min(slots, WINDOW + CHUNK))
    dp.comm.free()


@pytest.mark.parametrize("P,name,tun,hi,execution", [(1024, "TTPL_BT_alltoallv", (32, 32, 0), 40, 2), (530, "twophase_rbruck_alltoallv", (9,), 700, 2), (256, "tuna_algorithm", (4, 0), 1500, 2),
                                                     (210, "TTPL_BT_alltoallv_s1", (30, 5, 0), 90, 2), (194, "TTPL_BT_alltoallv", (97, 97, 0), 3, 2), (150, "twophase_rbruck_alltoallv_om", (3,), 500, 3),
                                                     (40, "tuna_algorithm", (2, 0), 60, 3), (101, "twophase_rbruck_alltoallv", (2,), 4_000, 3)])
def test_a_longest_block_that_grows_from_call_to_call(P, name, tun, hi, execution):
    """Slots in a window have no limit of length: the next call's longer blocks, at the ends of the window too, are delivered by the first launch, that of
    an _async call before it is waited for."""
    from rbruck_alltoallv_amd import api
    packed = name == "TTPL_BT_alltoallv"
    counts = np.random.default_rng(P).integers(0, hi + 1, (P, P)).astype(np.int32)
    comm = api.VirtualComm(P)
    longest = hi
    for turn in range(7):
        if turn > 1:
            longest = longest * 3 // 2 + 200              # (up to 8 pieces, what a quarter of a wavefront takes)
            at = np.random.default_rng(turn).integers(0, P, (2, 5))
            counts[at[0], at[1]] = min(longest, 28_000)
            counts[P - 1, :3] = counts[:3, P - 1] = min(longest, 28_000)
        prob = W.make_problem(counts, 1, 1, 0 if packed else 1)
        dp = api.DeviceProblem(prob, comm=comm)
        ds, dr = dp.new_send_arena(), dp.new_recv_arena()
        dp.fill_payload(0, turn, ds)
        assert getattr(api, name)(*tun, dp, ds, dr) == 0, (turn, comm.error())
        st = comm.last_stats()
        assert dp.verify(ds, dr, packed) == 0, turn
        if turn:
            assert (st.execution, st.host_waits, st.staging_bytes) == (execution, 1, WINDOW + CHUNK), (turn, st.lanes_per_item)
        if turn < 2 or name not in ("twophase_rbruck_alltoallv", "twophase_rbruck_alltoallv_om", "tuna_algorithm", "TTPL_BT_alltoallv", "TTPL_BT_alltoallv_s1"):
            continue
        counts[at[0], at[1] - 1] = min(longest + 300, 28_000)
        prob = W.make_problem(counts, 1, 1, 0 if packed else 1)
        dp = api.DeviceProblem(prob, comm=comm)
        ds, dr = dp.new_send_arena(), dp.new_recv_arena()
        dp.fill_payload(0, turn, ds)
        assert api.call_async(name, tun, dp, ds, dr, torch.cuda.current_stream()) == 0, comm.error()
        torch.cuda.synchronize()
        early = dr.clone()
        assert comm.wait() == 0 and dp.verify(ds, dr, packed) == 0, turn
        assert torch.equal(early, dr), turn
    comm.free()


@pytest.mark.parametrize("P", [40, 128])
def test_a_call_of_another_kind_goes_straight_to_the_list(P):
    """What the single launch is refused for, but for the length of a block, the other kernels without a list would be refused for too."""
    from rbruck_alltoallv_amd import api
    comm = api.VirtualComm(P)
    waits = []
    for turn, hi in enumerate((600, 600, 90_000, 600, 600)):      # 90 000 bytes are at least 21 pieces; no shape without a list takes more than 16
        dp = api.DeviceProblem(W.make_problem(np.random.default_rng(turn).integers(0, hi + 1, (P, P)).astype(np.int32), 1, 1, 1), comm=comm)
        ds, dr = dp.new_send_arena(), dp.new_recv_arena()
        dp.fill_payload(0, turn, ds)
        assert api.twophase_rbruck_alltoallv(4, dp, ds, dr) == 0, comm.error()
        st = comm.last_stats()
        waits.append((int(st.execution), int(st.host_waits)))
        assert dp.verify(ds, dr) == 0, turn
    # the first call; one launch; refused, then planned for the list and copied; a list again, as the blocks of the last call were long; one launch
    assert [e for e, _ in waits] == [1, 3, 1, 1, 3] and waits[1][1] == waits[4][1] == 1 and waits[2][1] == 3, waits
    comm.free()


@pytest.mark.parametrize("P,name,tun,kinds", [(230, "twophase_rbruck_alltoallv", (4,), [(100, 1), (5_000, 64)]), (300, "TTPL_BT_alltoallv", (30, 30, 0), [(300, 1), (9_000, 64)]),
                                              (150, "tuna_algorithm", (4, 0), [(80, 16), (20_000, 64)]), (256, "spreadout_alltoallv", (), [(90, 1), (5_000, 64)])])
def test_a_refused_call_gets_the_shape_of_its_own_blocks(P, name, tun, kinds):
    """Calls of short and of long blocks in turn: what the device refuses goes out once more, in no shape of the call before."""
    from rbruck_alltoallv_amd import api
    packed = name == "TTPL_BT_alltoallv"
    comm = api.VirtualComm(P)
    seen = []
    for turn in range(6):
        hi, lanes = kinds[turn > 1 and turn % 2]
        dp = api.DeviceProblem(W.make_problem(np.random.default_rng(turn).integers(0, hi + 1, (P, P)).astype(np.int32), 1, 1, 0 if packed else 1), comm=comm)
        ds, dr = dp.new_send_arena(), dp.new_recv_arena()
        dp.fill_payload(0, turn, ds)
        assert getattr(api, name)(*tun, dp, ds, dr) == 0, comm.error()
        st = comm.last_stats()
        assert dp.verify(ds, dr, packed) == 0, turn
        seen.append((int(st.lanes_per_item), int(st.host_waits)))
        # (the single launch takes short blocks in any shape: no pair knows the payload of the call)
        assert turn == 0 or (seen[-1][0] == lanes and seen[-1][1] <= 2) or (P <= 192 and hi < 100), (turn, seen)
    comm.free()
