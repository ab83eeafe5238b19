"""The metadata steps do not refuse to run beside a call on the same communicator (only vc_displs_from_counts does): neither may disturb the
other's workgroup counts, nor end the other's wait."""
import threading

import numpy as np
import pytest
import torch

from rbruck_alltoallv_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    from rbruck_alltoallv_amd import api
    return api


# up to 64 workgroups count themselves on one word (200 ranks: 49 of the transpose), more on several (520 ranks: 289)
@pytest.mark.parametrize("P", [200, 520])
def test_metadata_steps_beside_calls(api, P):
    prob = W.make_problem(W.counts_uniform_random(P, 300, seed=P), 1, 0, 0)
    dp = api.DeviceProblem(prob)
    lib, h, side = dp.comm.lib, dp.comm.handle, torch.cuda.Stream()
    ds, dr = dp.new_send_arena(), dp.new_recv_arena()
    dp.fill_payload(0, 5, ds)
    turned, top = torch.zeros_like(dp.recvcounts), torch.zeros(1, dtype=torch.int32, device="cuda")
    extent = torch.from_numpy(prob.sendcounts.sum(axis=1, dtype=np.int64)).cuda()
    base, total = torch.zeros(P, dtype=torch.int64, device="cuda"), torch.zeros(1, dtype=torch.int64, device="cuda")
    want_base = np.concatenate([[0], np.cumsum((prob.sendcounts.sum(axis=1, dtype=np.int64) + 255) // 256 * 256)])
    torch.cuda.synchronize()
    wrong, over = [], threading.Event()

    def steps():
        own = torch.cuda.Stream()
        n = 0
        while not over.is_set() or n < 50:
            with torch.cuda.stream(own):
                turned.zero_(), top.zero_(), base.zero_()
                own.synchronize()
                rcs = (lib.vc_alltoall_counts(dp.sendcounts.data_ptr(), turned.data_ptr(), h), lib.vc_allreduce_max_count(dp.sendcounts.data_ptr(), top.data_ptr(), h),
                       lib.vc_bases_from_extents(extent.data_ptr(), 1, 256, base.data_ptr(), total.data_ptr(), h))
                if rcs != (0, 0, 0) or not torch.equal(turned, dp.recvcounts) or int(top) != prob.sendcounts.max() or \
                        not np.array_equal(base.cpu().numpy(), want_base[:-1]) or int(total) != want_base[-1]:
                    wrong.append((n, rcs))
            n += 1

    t = threading.Thread(target=steps)
    t.start()
    try:
        for k in range(100):
            dr.fill_(0xEE)
            torch.cuda.synchronize()
            assert api.call_async("tuna_algorithm", (4, 0), dp, ds, dr, side) == 0 and dp.comm.wait() == 0, dp.comm.error()
            assert dp.verify(ds, dr) == 0, k
            dr.fill_(0xEE)
            torch.cuda.synchronize()
            assert api.tuna_algorithm(4, 0, dp, ds, dr) == 0 and dp.verify(ds, dr) == 0, k
    finally:
        over.set()
        t.join()
    assert not wrong, wrong[:3]
    dp.comm.free()


@pytest.mark.parametrize("step", ["counts", "wait"])
def test_a_wait_is_not_ended_by_a_call_on_another_stream(api, step):
    prob = W.make_problem(W.counts_uniform_random(64, 300, seed=1), 1, 0, 0)
    dp = api.DeviceProblem(prob)
    lib, h, own, side = dp.comm.lib, dp.comm.handle, torch.cuda.Stream(), torch.cuda.Stream()
    ds, dr = dp.new_send_arena(), dp.new_recv_arena()
    dp.fill_payload(0, 5, ds)
    turned = torch.zeros_like(dp.recvcounts)
    lib.vc_comm_set_stream(h, own.cuda_stream)
    for _ in range(2):                                     # (the second call allocates nothing: hipMalloc may wait for the device)
        assert api.call_async("tuna_algorithm", (4, 0), dp, ds, dr, side) == 0 and dp.comm.wait() == 0
    cycles, begin, end = 1 << 20, torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    begin.record(own)
    with torch.cuda.stream(own):
        torch.cuda._sleep(cycles)
    end.record(own)
    own.synchronize()
    cycles = int(cycles * 60 / begin.elapsed_time(end))    # 60 ms
    early = False
    for _ in range(4):                                     # (two streams may share a hardware queue: then the call waits for the sleep)
        side = torch.cuda.Stream()
        dr.fill_(0xEE)
        torch.cuda.synchronize()
        seen = []

        def on_own():
            rc = lib.vc_alltoall_counts(dp.sendcounts.data_ptr(), turned.data_ptr(), h) if step == "counts" else lib.vc_comm_wait(h)
            seen.append((rc, slept.query()))

        slept = torch.cuda.Event()
        with torch.cuda.stream(own):
            torch.cuda._sleep(cycles)
        slept.record(own)
        t = threading.Thread(target=on_own)
        t.start()
        t.join(0.005)                                      # its launch has gone out, its stream is asleep
        assert api.call_async("tuna_algorithm", (4, 0), dp, ds, dr, side) == 0 and dp.comm.wait() == 0
        early = not slept.query()
        t.join()
        assert seen == [(0, True)]
        if early:
            break
    else:
        pytest.skip("no call ran while the other stream was asleep")
    torch.cuda.synchronize()
    assert dp.verify(ds, dr) == 0 and (step == "wait" or torch.equal(turned, dp.recvcounts))
    dp.comm.free()
