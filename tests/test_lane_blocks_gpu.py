"""Blocks of one lane each or of four, staged in a window: every hop of every block of every length leaves the block where its slot starts (the slots of 200 ranks at
radix 15 do not wrap); and wavefronts that choose between a lane, four and sixteen by their longest block."""
import numpy as np
import pytest
import torch

from rbruck_alltoallv_amd import workloads as W

pytestmark = pytest.mark.gpu
P, R, STRIDE = 200, 15, 384                               # stride of slots for blocks of 1 .. 128 bytes: an odd number of lines


@pytest.mark.parametrize("longest", [1, 7, 16, 17, 31, 128])
def test_staged_blocks(longest):
    from rbruck_alltoallv_amd import api
    counts = (np.arange(P * P).reshape(P, P) * 7 % (longest + 1)).astype(np.int32)
    prob = W.make_problem(counts, 1, 1, 1)
    dp = api.DeviceProblem(prob)
    ds, dr, want = dp.new_send_arena(), dp.new_recv_arena(0xEE), dp.new_recv_arena(0xEE)
    dp.fill_payload(0, 9, ds)
    dp.comm.set_forwarding(0)
    assert api.twophase_rbruck_alltoallv(R, dp, ds, want) == 0 and dp.verify(ds, want) == 0
    dp.comm.set_forwarding(1)
    for _ in range(2):                                    # the second call on the hint of the first
        assert api.call_async("twophase_rbruck_alltoallv", (R,), dp, ds, dr, torch.cuda.current_stream()) == 0 and dp.comm.wait() == 0, dp.comm.error()
    st = dp.comm.last_stats()
    assert st.execution == 2 and st.lanes_per_item == 1 and torch.equal(dr, want)
    address, size = dp.comm.staging()
    staged = torch.empty((size + 15) // 16 * 16, dtype=torch.uint8, device="cuda:0")
    assert dp.comm.lib.vc_calibration_copy(staged.data_ptr(), address, staged.numel(), dp.comm.handle) == 0
    staged, sent = staged.cpu().numpy(), ds.cpu().numpy().view(np.uint8).reshape(-1)
    hops = 0
    for s in range(P):
        for t in range(P):
            j, n = (s - t) % P, int(counts[s, t])
            if n == 0 or j < R or j % R == 0:             # a single digit that is not zero: straight to the receiver
                continue
            holder = (s - j // R * R) % P                 # after the most significant digit
            place = ((P + holder) * P + (j + holder) % P) * STRIDE
            at = int(prob.sbase[s]) + int(prob.sdispls[s, t])
            assert np.array_equal(staged[place:place + n], sent[at:at + n]), (s, t, n)
            hops += 1
    assert hops > P * P // 2 * longest // (longest + 1)
    dp.comm.free()


# wavefronts of 64 pairs are tiles of 8 x 8 ranks: their longest block is one of `longest`
@pytest.mark.parametrize("ranks,name,args", [(512, "tuna_algorithm", (3, 0)), (516, "TTPL_BT_alltoallv", (43, 2, 0)), (520, "twophase_rbruck_alltoallv", (519,))])
@pytest.mark.parametrize("longest", [(80, 81, 15, 128, 16, 160), (129, 255, 256, 257, 600, 64)])
def test_lanes_by_the_longest_block(ranks, name, args, longest):
    from rbruck_alltoallv_amd import api
    rng = np.random.default_rng(ranks)
    tile = np.arange(ranks) // 8
    top = np.array(longest)[(tile[:, None] + 5 * tile[None, :]) % len(longest)]
    counts = np.minimum(rng.integers(0, 161, (ranks, ranks)), top).astype(np.int32)
    if max(longest) > 160:
        counts[::8, ::8] = top[::8, ::8]
        counts = np.where(rng.random((ranks, ranks)) < 0.5, 0, counts).astype(np.int32)
    packed = name == "TTPL_BT_alltoallv"
    dp = api.DeviceProblem(W.make_problem(counts, 1, 1, 0 if packed else 1))
    ds, got, want = dp.new_send_arena(), dp.new_recv_arena(0xEE), dp.new_recv_arena(0xEE)
    dp.fill_payload(0, 9, ds)
    dp.comm.set_forwarding(0)
    assert getattr(api, name)(*args, dp, ds, want) == 0 and dp.verify(ds, want, packed) == 0
    for first in (128, 700):                              # the hint: batches of 64, then of 16 and quarters
        hint = counts.copy()
        hint[0, 0] = first
        hp = api.DeviceProblem(W.make_problem(np.minimum(hint, first).astype(np.int32), 1, 1, 0 if packed else 1), comm=dp.comm)
        hs, hr = hp.new_send_arena(), hp.new_recv_arena()
        dp.comm.set_forwarding(1)
        for _ in range(2):
            assert getattr(api, name)(*args, hp, hs, hr) == 0, dp.comm.error()
        dp.comm.set_bases(dp.sbase, dp.rbase)
        got.fill_(0xEE)
        print("running", ranks, name, longest, first, flush=True)
        assert getattr(api, name)(*args, dp, ds, got) == 0, dp.comm.error()
        st = dp.comm.last_stats()
        assert torch.equal(got, want) and (st.execution, st.lanes_per_item) == (2, 1), (first, int(st.execution), int(st.lanes_per_item))
    dp.comm.free()
