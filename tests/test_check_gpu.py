"""The kernel that checks the tables of calls without a list and plan tables, against the planner's header: payload, hop-weighted bytes, pieces, longest block and
bad entries are the same words, at the edges of its paths (blocks of one piece wherever they lie, 32-bit sums, 64-bit sums), of its tiles and rounds."""
import numpy as np
import pytest
import torch

from rbruck_alltoallv_amd import _lib, workloads as W

pytestmark = pytest.mark.gpu

WHOLE, BRIEF = 8192 - 127, 1 << 18                        # bytes: one piece at any phase; sums of a wavefront in 32 bits
LONG = {"short": [], "one piece": [WHOLE - 1, WHOLE], "two pieces": [WHOLE + 1, 8192, 12289], "32 bits": [BRIEF - 5, BRIEF], "64 bits": [BRIEF + 9, 3_000_001]}


@pytest.mark.parametrize("long", LONG)
@pytest.mark.parametrize("P,name,args,esz", [(193, "twophase_rbruck_alltoallv", (3,), 1), (255, "tuna_algorithm", (254, 0), 1), (256, "TTPL_BT_alltoallv", (16, 2, 0), 4),
                                             (300, "TTPL_BT_alltoallv_s1", (20, 5, 0), 3), (514, "twophase_rbruck_alltoallv_om", (2,), 8),
                                             (1026, "tuna_algorithm", (7, 0), 1), (1032, "TTPL_BT_alltoallv", (24, 3, 0), 1)])
def test_header_of_the_check(P, name, args, esz, long):
    from rbruck_alltoallv_amd import api
    rng = np.random.default_rng(P)
    counts = rng.integers(0, 60, (P, P)).astype(np.int32)
    counts[rng.random((P, P)) < 0.1] = 0
    for k, length in enumerate(LONG[long] * 3):           # in the first, a middle and the last tile
        counts[[0, P // 2, P - 1][k % 3], [P - 1, 1, P // 3][k // 3 % 3]] = (length + esz - 1) // esz if long != "one piece" else length // esz
    packed = name == "TTPL_BT_alltoallv"
    prob = W.make_problem(counts, esz, 1, 0 if packed else 1)
    dp = api.DeviceProblem(prob)
    ds, want, got = dp.new_send_arena(), dp.new_recv_arena(), dp.new_recv_arena()
    dp.fill_payload(0, 9, ds)
    want.fill_(0xA5)

    def words(rc):
        st = dp.comm.last_stats()
        return rc, (int(st.payload_bytes), int(st.moved_bytes), int(st.block_pieces), int(st.max_block_pieces), int(st.max_block_bytes), int(st.bad_table_entries))

    def by_list(out):
        dp.comm.set_forwarding(2)
        return words(getattr(api, name)(*args, dp, ds, out))

    def by_check(out):
        dp.comm.set_forwarding(1)
        print("running", P, name, long, flush=True)
        rc = api.call_async(name, args, dp, ds, out, torch.cuda.current_stream())
        return words(rc or dp.comm.wait())

    by_list(want)
    rc, planner = by_list(got)                            # (long blocks are cut where their place in `got` says)
    assert rc == 0 and planner[0] == prob.payload_bytes, dp.comm.error()
    for _ in range(2):
        got.fill_(0xA5)
        rc, checked = by_check(got)
        assert rc == 0 and checked == planner, dp.comm.error()
        assert int(dp.comm.last_stats().execution) == 2
        assert torch.equal(got, want)
    # bad tables: negative entries of every table, and receivers that expect something else than is sent
    picks = rng.choice(P * P, size=9, replace=False)
    for k, at in enumerate(picks):
        t, s = int(at // P), int(at % P)
        if k < 2:
            dp.sendcounts[t, s] = -5
        elif k < 4:
            dp.sdispls[t, s] = -1
        elif k < 6 and not packed:
            dp.rdispls[t, s] = -7
        else:
            dp.recvcounts[t, s] += 3 if k < 8 else -600
    rc, planner = by_list(got)
    assert rc == _lib.VC_ERR_TABLES
    got.fill_(0x11)
    rc, checked = by_check(got)
    assert rc == _lib.VC_ERR_TABLES and checked[5] == planner[5] >= 9
    assert bool((got == 0x11).all())
    dp.comm.free()


@pytest.mark.parametrize("P,n", [(200, 20), (514, 257), (1030, 10)])
def test_packed_layouts_past_an_int(P, n):
    """Receivers whose packed layout passes INT_MAX elements are counted apart from the bad entries, each once: the first one, neighbours of one workgroup, the last one, entries in
    the first and the last wavefront of the sources.  One that ends at INT_MAX is none of them."""
    from rbruck_alltoallv_amd import api
    prob = W.make_problem(np.random.default_rng(P).integers(0, 60, (P, P)).astype(np.int32), 1)
    dp = api.DeviceProblem(prob)
    ds, got = dp.new_send_arena(), dp.new_recv_arena()
    dp.fill_payload(0, 9, ds)
    for _ in range(2):
        assert api.call_async("TTPL_BT_alltoallv", (n, 2, 0), dp, ds, got, torch.cuda.current_stream()) == 0 and dp.comm.wait() == 0, dp.comm.error()
    assert int(dp.comm.last_stats().execution) == 2 and dp.verify(ds, got, True) == 0
    top, over = 2 ** 31 - 1, [0, 101, 102, P - 1]
    for t, total in [(t, top + 1) for t in over] + [(7, top)]:
        dp.recvcounts[t] = 0
        dp.recvcounts[t, 0], dp.recvcounts[t, P - 1] = 2 ** 30, total - 2 ** 30
        dp.sendcounts[:, t] = dp.recvcounts[t]
    dp.recvcounts[50, 50] += 1                            # and one bad entry
    got.fill_(0x11)
    for forwarding in (2, 1):                             # the planner, the check
        dp.comm.set_forwarding(forwarding)
        print("running", P, n, forwarding, flush=True)
        if forwarding == 2:
            rc = api.TTPL_BT_alltoallv(n, 2, 0, dp, ds, got)
        else:
            rc = api.call_async("TTPL_BT_alltoallv", (n, 2, 0), dp, ds, got, torch.cuda.current_stream()) or dp.comm.wait()
        assert rc == _lib.VC_ERR_OVERFLOW and int(dp.comm.last_stats().bad_table_entries) == (len(over) << 40) + 1, forwarding
    assert bool((got == 0x11).all())
    dp.comm.free()
