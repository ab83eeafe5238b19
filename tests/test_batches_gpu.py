"""Calls out of the staging bound in the default mode: batches of receivers on one staging arena, or a launch per digit."""
import numpy as np
import pytest
import torch

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


# function, tunables before the problem, ranks, element size, allowance in MiB: most significant digit first; two layers, packed and not; a
# Bruck over the nodes too; more ranks than a planning workgroup takes in one round
@pytest.mark.parametrize("name,tun,P,esz,mib", [("twophase_rbruck_alltoallv", (2,), 640, 1, 128), ("TTPL_BT_alltoallv", (160, 2, 0), 640, 1, 128),
                                                ("TTPL_BT_alltoallv_s1", (160, 2, 0), 640, 8, 900), ("TTPL_rbruck_alltoallv", (160, 2), 640, 4, 512),
                                                ("tuna_algorithm", (2, 0), 1030, 1, 200)])
def test_batches_of_every_kind_of_schedule(name, tun, P, esz, mib):
    from rbruck_alltoallv_amd import api
    packed = name == "TTPL_BT_alltoallv"
    counts = np.random.default_rng(P).integers(0, 500 if P < 1000 else 90, (P, P)).astype(np.int32)
    counts[::9, ::53] = 9_001
    counts[5, P - 2] = 300_001
    prob = W.make_problem(counts, esz, 0, 0 if packed else 1)
    dp = api.DeviceProblem(prob)
    fn = getattr(api, name)
    ds, dr = dp.new_send_arena(), dp.new_recv_arena()
    dp.fill_payload(0, 3, ds)
    dp.comm.set_staging_bound(0)
    assert fn(*tun, dp, ds, dr) == 0
    whole = dp.comm.last_stats()
    want = dr.clone()
    assert dp.verify(ds, dr, packed) == 0 and whole.staging_bytes > 3 * prob.payload_bytes
    dp.comm.set_staging_bound(mib)
    for _ in range(2):
        dr.fill_(0xEE)
        assert fn(*tun, dp, ds, dr) == 0, dp.comm.error()
        assert torch.equal(dr, want)
        st = dp.comm.last_stats()
        assert (st.execution, st.n_launches) == (1, -(-whole.staging_bytes // (mib << 20))) and st.n_launches > 1
        assert st.moved_bytes == whole.moved_bytes and st.staging_bytes < 1.25 * (mib << 20)
    # bad tables are found by the plan of the whole call
    keep = int(dp.recvcounts[P - 1, 7])
    dp.recvcounts[P - 1, 7] = keep + 1
    dr.fill_(0xEE)
    assert fn(*tun, dp, ds, dr) == -7 and bool((dr == 0xEE).all())
    dp.recvcounts[P - 1, 7] = keep
    assert fn(*tun, dp, ds, dr) == 0 and torch.equal(dr, want)
    dp.comm.free()


def test_uneven_receivers_are_seen_before_anything_is_copied():
    """No batch is planned, listed or copied of a call that ends one launch per digit: it waits for the plan of the whole call, for what its
    receivers take, for the plan on reused staging and for its end."""
    from rbruck_alltoallv_amd import api
    P = 512
    prob = W.make_problem(_counts(P, "skewed"), 1, 0, 1)
    dp = api.DeviceProblem(prob)
    ds, dr = dp.new_send_arena(), dp.new_recv_arena()
    dp.fill_payload(0, 3, ds)
    dp.comm.set_staging_bound(256)
    for _ in range(2):
        dr.fill_(0xEE)
        assert api.tuna_algorithm(2, 0, dp, ds, dr) == 0 and dp.verify(ds, dr) == 0, dp.comm.error()
        st = dp.comm.last_stats()
        assert (st.execution, st.n_launches, st.host_waits) == (0, 9, 4)
    dp.comm.free()
