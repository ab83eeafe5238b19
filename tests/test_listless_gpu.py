"""Calls served without a work-item list, at the edges of what their kernels do: blocks moved by one lane (up to 32 bytes), by a quarter
of a wavefront or by a wavefront, rank counts that fill no tile of sources x receivers, blocks cut into pieces, whole aligned pieces."""
import numpy as np
import pytest
import torch

from rbruck_alltoallv_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    from rbruck_alltoallv_amd import api
    return api


# ranks, longest block in bytes, radix, executions allowed after the first call (2: listless, 3: fixed-stride staging)
@pytest.mark.parametrize("P,top,r,kinds", [(5, 33, 2, {3}), (64, 2050, 2, {3}), (127, 1500, 3, {3}), (191, 700, 8, {2, 3}), (197, 16, 2, {2}),
                                           (321, 33, 4, {2}), (363, 200, 3, {2}), (725, 17, 3, {2}), (1021, 48, 32, {2})])
def test_short_blocks_at_every_length(api, P, top, r, kinds):
    rng = np.random.default_rng(P)
    counts = rng.integers(0, top + 1, (P, P)).astype(np.int32)
    counts[: min(P, 8), : min(P, 34)] = np.arange(min(P, 34))[None] * (np.arange(min(P, 34)) <= top)      # every short length
    prob = W.make_problem(counts, 1, 1, 1)
    dp = api.DeviceProblem(prob)
    ds, want, got = dp.new_send_arena(), dp.new_recv_arena(), dp.new_recv_arena()
    dp.fill_payload(0, P, ds)
    want.fill_(0xA5)
    dp.comm.set_forwarding(0)
    assert api.twophase_rbruck_alltoallv(r, dp, ds, want) == 0 and dp.verify(ds, want) == 0
    dp.comm.set_forwarding(1)
    for call in range(3):
        got.fill_(0xA5)
        assert api.twophase_rbruck_alltoallv(r, dp, ds, got) == 0, dp.comm.error()
        assert torch.equal(got, want), (P, top, call)
        assert call == 0 or dp.comm.last_stats().execution in kinds
    dp.comm.free()


@pytest.mark.parametrize("P,length", [(16, 4096), (16, 20000), (48, 8191)])
def test_whole_pieces_on_fixed_stride_staging(api, P, length):
    counts = np.full((P, P), length, dtype=np.int32)
    counts[::3, ::2] -= 1
    prob = W.make_problem(counts, 1, 0, 0)
    dp = api.DeviceProblem(prob)
    ds, dr = dp.new_send_arena(), dp.new_recv_arena()
    dp.fill_payload(0, 9, ds)
    for _ in range(3):
        dr.zero_()
        assert api.twophase_rbruck_alltoallv(2, dp, ds, dr) == 0 and dp.verify(ds, dr) == 0
    dp.comm.free()


# ranks, block length around which the lengths lie, execution after the first call: the list beyond 362 ranks or 3 KiB
@pytest.mark.parametrize("P,around,execution", [(150, 1000, 3), (150, 2900, 3), (200, 2000, 2), (363, 2000, 1), (200, 3500, 1)])
def test_direct_functions(api, P, around, execution):
    counts = np.random.default_rng(P).integers(around - 900, around + 100, (P, P)).astype(np.int32)
    prob = W.make_problem(counts, 1, 1, 1)
    dp = api.DeviceProblem(prob)
    ds, dr = dp.new_send_arena(), dp.new_recv_arena()
    dp.fill_payload(0, 4, ds)
    for call in range(3):
        dr.zero_()
        assert api.spreadout_alltoallv(dp, ds, dr) == 0 and dp.verify(ds, dr) == 0, dp.comm.error()
        assert call == 0 or dp.comm.last_stats().execution == execution
    dp.comm.free()


# up to 32 ranks the launch stores past the caches and signals its own end: what it wrote is read at once from another stream
@pytest.mark.parametrize("P,top", [(2, 40), (9, 3000), (16, 70000), (32, 6000), (32, 30000), (33, 6000)])
def test_everything_is_there_when_the_call_returns(api, P, top):
    counts = np.random.default_rng(P).integers(top // 2, top + 1, (P, P)).astype(np.int32)
    prob = W.make_problem(counts, 1, 1, 1)
    dp = api.DeviceProblem(prob)
    ds, want, got = dp.new_send_arena(), dp.new_recv_arena(), dp.new_recv_arena()
    other = torch.cuda.Stream()
    for call in range(4):
        dp.fill_payload(0, call, ds)
        want.fill_(0xA5)
        got.fill_(0xA5)
        dp.comm.set_forwarding(0)
        assert api.twophase_rbruck_alltoallv(3, dp, ds, want) == 0 and dp.verify(ds, want) == 0
        dp.comm.set_forwarding(1)
        torch.cuda.synchronize()
        assert api.twophase_rbruck_alltoallv(3, dp, ds, got) == 0, dp.comm.error()
        with torch.cuda.stream(other):
            assert torch.equal(got.cpu(), want.cpu()), (P, top, call)
    dp.comm.free()


# ranks, longest block in bytes, radix, lanes per pair of the copy kernel (1: batches) of a communicator's first _async call: what its plan
# asks for, not a shape chosen before there is a plan; with one hop per block (radix = ranks) nothing is staged and the copy goes out at once
@pytest.mark.parametrize("timing", [False, True])
@pytest.mark.parametrize("P,top,r,lanes", [(300, 500, 4, 1), (300, 1300, 4, 16), (64, 1500, 2, 16), (64, 20000, 2, 256), (40, 900, 40, 256)])
def test_first_async_call(api, P, top, r, lanes, timing):
    prob = W.make_problem(W.counts_uniform_random(P, top, seed=P), 1, 1, 1)
    dp = api.DeviceProblem(prob)
    dp.comm.set_timing(timing)
    side = torch.cuda.Stream()
    ds, dr = dp.new_send_arena(), dp.new_recv_arena()
    dp.fill_payload(0, P, ds)
    torch.cuda.synchronize()
    for call in range(3):
        dr.fill_(0xA5)
        torch.cuda.synchronize()
        assert api.call_async("twophase_rbruck_alltoallv", (r,), dp, ds, dr, side) == 0, dp.comm.error()
        if r == P:
            side.synchronize()
            assert dp.verify(ds, dr) == 0
        assert dp.comm.wait() == 0 and dp.verify(ds, dr) == 0, dp.comm.error()
        st = dp.comm.last_stats()
        assert call or (st.execution, st.lanes_per_item, st.host_waits) == (2, lanes, 1 if r == P else 2)
        assert (st.total_ms > 0) == (st.launch_ms[0] > 0) == timing
    # a longer call than the arena holds: its own plan decides again
    counts = np.full((P, P), 40000, dtype=np.int32)
    longer = W.make_problem(counts, 1, 0, 0)
    dl = api.DeviceProblem(longer, comm=dp.comm)
    ls, lr = dl.new_send_arena(), dl.new_recv_arena()
    dl.fill_payload(0, 3, ls)
    torch.cuda.synchronize()
    assert api.call_async("twophase_rbruck_alltoallv", (2,), dl, ls, lr, side) == 0 and dl.comm.wait() == 0, dl.comm.error()
    assert dl.verify(ls, lr) == 0 and dl.comm.last_stats().lanes_per_item == 256
    dp.comm.free()
