"""Block lengths at the edges of what the copy kernels do in one go (a lane's widths, 16-byte vectors, a lane's share of a block, one work item, several pieces),
at every byte phase of source and destination, in every shape of the kernels without a list: nothing but the blocks is written."""
import numpy as np
import pytest
import torch

from rbruck_alltoallv_amd import workloads as W

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 18, 31, 32, 33, 47, 48, 49, 63, 112, 113, 127, 128, 129, 239, 255, 256, 257, 511, 513, 767, 769, 897, 1023, 1025,
         1919, 1921, 2047, 2049, 4095, 4096, 4097, 8063, 8064, 8065, 8066, 8191, 8192, 8193, 12289, 28000]


def _counts(P, fill, seed):
    """About `fill` bytes a pair, every edge length in two rows and two columns of pairs that lie far apart."""
    rng = np.random.default_rng(seed)
    counts = rng.integers(fill // 2, fill + fill // 2 + 1, (P, P)).astype(np.int32)
    n = len(EDGES)
    for k in range(2 * n):
        counts[(k * 7 + 1) % P, (k * 5 + k // P) % P] = EDGES[k % n]
    return counts


# ranks, radix, bytes a pair, name, size of an element; what the default mode runs from the second call on (execution, lanes).  Elements of 4 bytes make blocks of 28 pieces, which
# go through the list there and without it in the forced modes.
@pytest.mark.parametrize("P,r,fill,name,element,default", [
    (24, 2, 40, "twophase_rbruck_alltoallv", 1, (3, 64)), (64, 2, 90, "twophase_rbruck_alltoallv", 1, (3, 16)), (64, 4, 2600, "tuna_algorithm", 1, (3, 64)),
    (130, 3, 700, "twophase_rbruck_alltoallv_om", 1, (3, 16)), (130, 3, 2500, "twophase_rbruck_alltoallv", 1, (3, 64)), (220, 5, 60, "twophase_rbruck_alltoallv", 1, (2, 1)),
    (220, 5, 900, "tuna_algorithm", 1, (2, 16)), (220, 15, 3000, "twophase_rbruck_alltoallv", 1, (2, 64)), (150, 2, 3100, "spreadout_alltoallv", 1, (3, 64)),
    (130, 4, 150, "twophase_rbruck_alltoallv", 4, (1, 64)), (220, 15, 800, "twophase_rbruck_alltoallv", 4, (1, 256))])
def test_lengths_at_the_edges(P, r, fill, name, element, default):
    from rbruck_alltoallv_amd import api
    args = {"tuna_algorithm": (r, 0), "spreadout_alltoallv": ()}.get(name, (r,))
    fn = getattr(api, name)
    prob = W.make_problem(_counts(P, fill, P + fill), element, 1, 1)
    dp = api.DeviceProblem(prob)
    ds, want, got = dp.new_send_arena(), dp.new_recv_arena(), dp.new_recv_arena()
    dp.fill_payload(0, P, ds)
    want.fill_(0xA5)
    dp.comm.set_forwarding(0)
    assert fn(*args, dp, ds, want) == 0 and dp.verify(ds, want) == 0
    for mode in (1, 3, 4, 5):
        dp.comm.set_forwarding(mode)
        for call in range(3 if mode == 1 else 2):
            got.fill_(0xA5)
            print("running", P, fill, name, "mode", mode, "call", call, flush=True)
            assert fn(*args, dp, ds, got) == 0, dp.comm.error()
            assert torch.equal(got, want), (mode, call)
            st = dp.comm.last_stats()
            if call or mode != 1:
                assert (st.execution, st.lanes_per_item) == {1: default, 3: (2, 256), 4: (2, 16), 5: (2, 1)}[mode], (mode, call)
    dp.comm.set_forwarding(1)
    if name != "spreadout_alltoallv":
        for _ in range(2):
            got.fill_(0xA5)
            assert api.call_async(name, args, dp, ds, got, torch.cuda.current_stream()) == 0 and dp.comm.wait() == 0, dp.comm.error()
            assert torch.equal(got, want)
    dp.comm.free()
