"""Calls out of the staging bound in the default mode: batches of receivers on one staging arena, or a launch per digit."""
import numpy as np
import pytest

from rbruck_alltoallv_amd import workloads as W

pytestmark = pytest.mark.gpu


def _counts(P, kind):
    counts = np.random.default_rng(7).integers(0, 500, (P, P)).astype(np.int32)
    counts[::7, ::31] = 70_001                            # 18 pieces
    counts[3, P - 1] = 2_000_003                          # 489: two units of the list's writers
    if kind == "skewed":
        counts[:, P - 1] = 150_000                        # most of the payload ends on one rank
    return counts


@pytest.mark.parametrize("kind,mib,batched", [("even", 300, True), ("even", 100, True), ("skewed", 256, False), ("even", 16, False)])
def test_batches_of_receivers(kind, mib, batched):
    from rbruck_alltoallv_amd import api
    P = 512
    prob = W.make_problem(_counts(P, kind), 1, 0, 1)
    dp = api.DeviceProblem(prob)
    dp.comm.set_forwarding(1)
    ds, dr = dp.new_send_arena(), dp.new_recv_arena()
    dp.fill_payload(0, 3, ds)
    dp.comm.set_staging_bound(0)
    assert api.tuna_algorithm(2, 0, dp, ds, dr) == 0
    launches = -(-dp.comm.last_stats().staging_bytes // (mib << 20)) if batched else 9
    dp.comm.set_staging_bound(mib)
    for timing in (False, True):
        dp.comm.set_timing(timing)
        for _ in range(2):
            dr.fill_(0xEE)
            assert api.tuna_algorithm(2, 0, dp, ds, dr) == 0 and dp.verify(ds, dr) == 0, dp.comm.error()
            st = dp.comm.last_stats()
            assert (st.execution, st.n_launches) == (int(batched), launches), (st.execution, st.n_launches)
            assert st.payload_bytes == prob.payload_bytes and st.moved_bytes == sum(st.launch_bytes[:launches])
            assert 2 * st.moved_bytes == W.algorithmic_bytes(prob.sendcounts, 1, W.hops_flat(P, 2))
            if batched:
                assert st.staging_bytes < 1.25 * (mib << 20)
            assert (st.total_ms > 0) == timing
    # a smaller call on the same communicator is an ordinary one
    assert api.tuna_algorithm(32, 0, dp, ds, dr) == 0 and dp.verify(ds, dr) == 0 and dp.comm.last_stats().n_launches == 1
    dp.comm.free()
