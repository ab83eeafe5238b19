"""Blocks of up to 64 bytes on 512 ranks and more: a tile of 8 x 8 pairs whose blocks lie side by side moves as runs, every other one (a tile at the edge, gaps, a run
shorter than a vector, a block that is longer) a lane a block.  Packed and with gaps on either side, runs that start and end anywhere in a vector, staged and direct."""
import numpy as np
import pytest
import torch

from rbruck_alltoallv_amd import workloads as W
from tests import emulator as E

pytestmark = pytest.mark.gpu

SIZES = [(16, 1), (15, 1), (5, 1), (7, 2), (4, 4), (2, 8), (31, 1), (32, 1), (15, 2), (8, 4), (63, 1), (64, 1), (31, 2), (15, 4), (16, 4)]
# vectors of a run behind a call whose longest block is `most` elements, by the entry of SIZES
VECTORS = {512: [1, 1, 1, 1, 1, 0, 2, 2, 0, 0, 4, 4, 0, 0, 0], 736: [1, 1, 1, 1, 1, 0, 2, 2, 2, 2, 4, 4, 4, 4, 4]}
OTHERS = [1, 1, 1, 1, 1, 0, 2, 2, 2, 2, 4, 4, 0, 0, 0]
FUNCTION = {"tuna_algorithm": E.F_TUNA, "TTPL_BT_alltoallv": E.F_TTPL, "twophase_rbruck_alltoallv": E.F_TWOPHASE, "spreadout_alltoallv": E.F_SPREADOUT}


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
@pytest.mark.parametrize("most,esz", SIZES)
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
                # the instance that the call behind this one gets
                st, n, r = dp.comm.last_stats(), args[0] if packed else 0, args[1] if packed else (args or (2,))[0]
                last = (1, int(st.block_pieces), int(st.payload_bytes), int(st.max_block_pieces), int(st.max_block_bytes))
                assert E.dispatch(FUNCTION[name], ranks, last, n=n, r=r, esz=esz, window=True, run=True) == VECTORS.get(ranks, OTHERS)[SIZES.index((most, esz))]
            dp.comm.set_bases(dp.sbase, dp.rbase)
            assert getattr(api, name)(*args, dp, ds, got) == 0, dp.comm.error()
        st = dp.comm.last_stats()
        assert st.execution == 2 and st.lanes_per_item == 1 and torch.equal(got, want)
    dp.comm.free()


@pytest.mark.parametrize("longest,vectors", [(16, 1), (32, 2), (64, 4), (128, 0)])
def test_staged_hops_of_runs_lanes_and_four_lanes(longest, vectors):
    """512 ranks, two digits, behind a call whose longest block is `longest`: every staged hop is where its slot starts (the slots of one region are 2^18 places of the window, all
    different), and what is behind a block of less than a vector there says how its tile of 8 x 8 pairs moved: in a run the bytes that follow it, of a lane of its own
    zeros (behind 4 and 8 bytes the block again), by four lanes what was there before."""
    from rbruck_alltoallv_amd import api
    P, R, STRIDE, WINDOW, BEFORE = 512, 23, 384, 32 << 20, 0xAB
    rng = np.random.default_rng(longest)
    tile = np.arange(P) // 8
    kind = (tile[:, None] + 3 * tile[None, :]) % 5
    counts = rng.integers(1, 17, (P, P))                  # (runs of 8 blocks of at least 2 bytes: a vector or more)
    counts = np.where(counts == 1, 2, counts)
    counts = np.where((kind == 1) | (kind == 2), np.minimum(rng.integers(2, 65, (P, P)), max(16 * vectors, 16)), counts)
    counts[1::8, 2::8] = np.where(kind[1::8, 2::8] == 3, 80, counts[1::8, 2::8])           # too long for any run
    counts[6::8, 7::8] = np.where(kind[6::8, 7::8] == 4, rng.integers(81, 129, kind[6::8, 7::8].shape), counts[6::8, 7::8])
    dp = api.DeviceProblem(W.make_problem(counts.astype(np.int32), 1, align=1))
    ds, dr = dp.new_send_arena(), dp.new_recv_arena()
    dp.fill_payload(0, 9, ds)                             # (while the communicator has the bases of these arenas)
    hp = api.DeviceProblem(W.make_problem(np.minimum(np.where(kind == 0, longest, counts), longest).astype(np.int32), 1), comm=dp.comm)
    hs, hr = hp.new_send_arena(), hp.new_recv_arena()
    for _ in range(3):
        assert api.twophase_rbruck_alltoallv(R, hp, hs, hr) == 0, dp.comm.error()
    address, size = dp.comm.staging()
    assert size >= WINDOW
    staged = torch.full((WINDOW,), BEFORE, dtype=torch.uint8, device="cuda:0")
    assert dp.comm.lib.vc_calibration_copy(address, staged.data_ptr(), WINDOW, dp.comm.handle) == 0
    dp.comm.set_bases(dp.sbase, dp.rbase)
    assert api.twophase_rbruck_alltoallv(R, dp, ds, dr) == 0 and dp.verify(ds, dr) == 0, dp.comm.error()
    st = dp.comm.last_stats()
    assert st.execution == 2 and st.lanes_per_item == 1 and dp.comm.staging() == (address, size)
    assert dp.comm.lib.vc_calibration_copy(staged.data_ptr(), address, WINDOW, dp.comm.handle) == 0
    staged, sent = staged.cpu().numpy(), np.concatenate([ds.cpu().numpy().view(np.uint8).reshape(-1), np.zeros(128, np.uint8)])
    s, t = np.divmod(np.arange(P * P), P)
    j = (s - t) % P
    s, t, j = (a[(j >= R) & (j % R != 0)] for a in (s, t, j))                              # two digits that are not zero
    holder = (s - j // R * R) % P                         # after the most significant one
    place = ((P + holder) * P + (j + holder) % P) * STRIDE % WINDOW
    assert len(np.unique(place)) == len(place) > P * P * 9 // 10
    n, at = counts[s, t], dp.host.sbase[s] + dp.host.sdispls[s, t]
    k = np.arange(128)
    got, follows = staged[place[:, None] + k], sent[at[:, None] + k]
    assert np.array_equal(got[k < n[:, None]], follows[k < n[:, None]])
    by_tile = counts.reshape(P // 8, 8, P // 8, 8).max((1, 3))[s // 8, t // 8]
    runs, four = by_tile <= 16 * vectors, by_tile > 80
    assert four.any() and runs.any() == (vectors > 0) and (~runs & ~four).any()
    end = counts.reshape(P, P // 8, 8)[:, :, ::-1].cumsum(2)[:, :, ::-1].reshape(P, P)[s, t]      # bytes to the end of the run
    behind = (k < 16) & (k >= n[:, None])
    for moved, where, what in (("in runs", runs[:, None] & (k < end[:, None]), follows), ("a lane", (~runs & ~four & (n != 4) & (n != 8))[:, None], np.zeros_like(got)),
                               ("four lanes", four[:, None], np.full_like(got, BEFORE))):
        assert np.array_equal(got[where & behind], what[where & behind]), moved
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
