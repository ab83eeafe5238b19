"""Blocks of up to 64 bytes on 512 ranks and more: a tile of 8 x 8 pairs whose blocks lie side by side moves as runs, every other one (a tile at the edge, gaps, a run
shorter than a vector, a block that is longer) a lane a block.  Packed and with gaps on either side, runs that start and end anywhere in a vector, staged and direct."""
import numpy as np
import pytest
import torch

from rbruck_alltoallv_amd import workloads as W

pytestmark = pytest.mark.gpu


def counts_of(ranks, most, esz):
    rng = np.random.default_rng(ranks + most)
    counts = rng.integers(0, most + 1, (ranks, ranks))
    tile = np.arange(ranks) // 8
    kind = (tile[:, None] + 3 * tile[None, :]) % 7
    counts = np.where(kind == 1, most, counts)                                        # the longest runs
    counts = np.where(kind == 2, counts * (rng.random((ranks, ranks)) < 0.2), counts)  # empty runs, runs shorter than a vector
    counts = np.where(kind == 3, np.minimum(counts, -(-5 // esz)), counts)             # just long enough
    counts[::40, ::24] = most + 1                                                      # just too long, or a vector more
    return counts.astype(np.int32)


@pytest.mark.parametrize("layouts", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("ranks,name,args", [(512, "tuna_algorithm", (3, 0)), (736, "tuna_algorithm", (27, 0)), (515, "TTPL_BT_alltoallv", (5, 2, 0)), (520, "twophase_rbruck_alltoallv", (519,)), (516, "spreadout_alltoallv", ())])
@pytest.mark.parametrize("most,esz", [(16, 1), (15, 1), (5, 1), (7, 2), (4, 4), (2, 8), (31, 1), (32, 1), (15, 2), (8, 4), (63, 1), (64, 1), (31, 2), (15, 4), (16, 4)])
def test_tiles_as_runs(most, esz, ranks, name, args, layouts):
    from rbruck_alltoallv_amd import api
    packed = name == "TTPL_BT_alltoallv"
    dp = api.DeviceProblem(W.make_problem(counts_of(ranks, most, esz), esz, layouts[0], 0 if packed else layouts[1], align=8 if esz == 8 else 4 if esz == 4 else 2 * esz - 1))
    ds, got, want = dp.new_send_arena(), dp.new_recv_arena(0xEE), dp.new_recv_arena(0xEE)
    dp.fill_payload(0, 9, ds)
    dp.comm.set_forwarding(0)
    assert getattr(api, name)(*args, dp, ds, want) == 0 and dp.verify(ds, want, packed) == 0
    dp.comm.set_forwarding(1)
    hint = counts_of(ranks, most, esz)
    hint[::40, ::24] = most                               # ... of calls whose longest block is `most`: one longer than its wavefront takes
    hp = api.DeviceProblem(W.make_problem(hint, esz), comm=dp.comm)
    hs, hr = hp.new_send_arena(), hp.new_recv_arena()
    for hinted in (False, True):                          # the second call on the hint of the first
        for _ in range(2):
            got.fill_(0xEE)
            if hinted:
                dp.comm.set_bases(hp.sbase, hp.rbase)
                assert getattr(api, name)(*args, hp, hs, hr) == 0, dp.comm.error()
            dp.comm.set_bases(dp.sbase, dp.rbase)
            assert getattr(api, name)(*args, dp, ds, got) == 0, dp.comm.error()
        st = dp.comm.last_stats()
        assert st.execution == 2 and st.lanes_per_item == 1 and torch.equal(got, want)
    dp.comm.free()


@pytest.mark.parametrize("how", ["forced", "allowance", "noalloc"])
@pytest.mark.parametrize("most", [16, 32, 64])
@pytest.mark.parametrize("r", [23, 300])
def test_short_blocks_staged_outside_a_window(r, most, how):
    """512 ranks, two digits: batches that give every slot a place of its own, forced, with an allowance of the caller's, and out of the static scratch array.  At
    radix 23 a lane a block, at 300 tiles whose blocks have one hop as runs."""
    from rbruck_alltoallv_amd import api
    ranks = 512
    dp = api.DeviceProblem(W.make_problem(counts_of(ranks, most - 1, 1), 1))
    ds, got, want = dp.new_send_arena(), dp.new_recv_arena(0xEE), dp.new_recv_arena(0xEE)
    dp.fill_payload(0, 9, ds)
    dp.comm.set_forwarding(0)
    assert api.twophase_rbruck_alltoallv(r, dp, ds, want) == 0 and dp.verify(ds, want) == 0
    dp.comm.set_forwarding(5 if how == "forced" else 1)
    if how == "allowance":
        dp.comm.set_staging_bound(4096)
    call = api.twophase_rbruck_alltoallv_noalloc if how == "noalloc" else api.twophase_rbruck_alltoallv
    for turn in range(3):                                 # the later ones on the hint of the first
        got.fill_(0xEE)
        assert (call if turn else api.twophase_rbruck_alltoallv)(r, dp, ds, got) == 0, dp.comm.error()
        assert torch.equal(got, want)
    st = dp.comm.last_stats()
    assert st.execution == 2 and st.lanes_per_item == 1 and st.staging_bytes > 0
    dp.comm.free()
