"""The branch-free forms of the route arithmetic the forwarded planner and the copy kernels use (csrc/vc_plan_math.h compiled for
the CPU): division of ranks by the call's constants, the block a staging slot keeps (vc_slot_block against
vc_region_slot_size), and a block's hops one after the other (vc_walk_step against vc_hop_place), over every slot and pair of
schedules with remainders, one rank per node, one node, radices that do and do not divide."""
import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "rbruck_alltoallv_amd", "csrc")

SOURCE = r"""
#include <vector>
#include "vc_sched.h"
#include "vc_plan_math.h"

extern "C" int rank_division_mismatches(int d_lo, int d_hi) {
    int wrong = 0;
    for (int d = d_lo; d <= d_hi; d++) {
        const VcRankDivisor v = vc_make_rank_divisor(d);
        for (int x = 0; x < 65536; x += 1 + (d > 64 && x % d > 1 && x % d < d - 2)) wrong += vc_div(x, v) != x / d || vc_mod(x, v) != x % d;
    }
    return wrong;
}

extern "C" int route_mismatches(int func, int P, int n, int r) {
    VcSched S;
    std::vector<VcLaunchInfo> L;
    if (vc_make_schedule((VcFunc)func, P, n, r, 0, 1, func == VC_F_UNIFORM_SPREADOUT || func == VC_F_UNIFORM_ISPLIT, S, L, 0, true)) return -1;
    std::vector<int> one((size_t)P * P, 1), zero((size_t)P * P, 0);
    std::vector<int64_t> base(P, 0);
    VcTables T = {one.data(), zero.data(), one.data(), zero.data(), base.data(), base.data(), zero.data()};
    int wrong = 0;
    for (int y = 0; y < S.w + S.w2; y++)
        for (int to = 0; to < P; to++)
            for (int id = 0; id < P; id++) {
                int st[2] = {-1, -1}, s = -1, t = -1;
                const bool there = vc_region_slot_size(S, T, y, to, id, nullptr, st) != 0;
                wrong += vc_slot_block(S, y, to, id, s, t) != there || s < 0 || s >= P || t < 0 || t >= P;
                if (there) {
                    wrong += s != st[0] || t != st[1];
                    const VcHop h = vc_hop_place(S, s, t, y);
                    wrong += !h.moves || !h.staged || h.row != y * P + to || h.id != id;
                }
            }
    for (int s = 0; s < P; s++)
        for (int t = 0; t < P; t++) {
            VcWalk w = vc_walk_start(S, s, t);
            int hops = 0, ends = 0;
            for (int k = 0; k < vc_hop_slots(S); k++) {
                const VcHop a = vc_walk_step(S, w, s, t, k), b = vc_hop_place(S, s, t, k);
                wrong += a.moves != b.moves || a.staged != b.staged || a.row != b.row || a.id != b.id;
                wrong += a.row < 0 || a.row >= (S.w + S.w2 > 0 ? S.w + S.w2 : 1) * P || a.id < 0 || a.id >= P;
                wrong += (a.moves != 0) != vc_block_moves(S, s, t, k);
                hops += a.moves != 0;
                ends += a.moves && !a.staged;
            }
            wrong += hops != vc_block_hops(S, s, t) || ends != 1;
        }
    return wrong;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("route")
    src, out = d / "route.cpp", d / "libroute.so"
    src.write_text(SOURCE)
    subprocess.run(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-fPIC", "-shared", "-I", CSRC, "-o", str(out), str(src)], check=True, capture_output=True)
    return C.CDLL(str(out))


@pytest.mark.parametrize("d_lo,d_hi", [(1, 40), (255, 258), (1023, 1026), (32760, 32768)])
def test_division_of_ranks(lib, d_lo, d_hi):
    assert lib.rank_division_mismatches(d_lo, d_hi) == 0


@pytest.mark.parametrize("func,P,n,r", [(0, 1, 0, 2), (0, 2, 0, 2), (0, 33, 0, 2), (1, 64, 0, 8), (0, 50, 0, 7), (2, 65, 0, 64), (2, 96, 0, 3), (4, 60, 12, 5),
                                        (3, 64, 64, 4), (4, 12, 1, 2), (15, 72, 6, 2), (15, 48, 4, 4), (6, 40, 8, 3), (7, 31, 0, 2), (13, 24, 6, 2)])
def test_slots_and_hops(lib, func, P, n, r):
    assert lib.route_mismatches(func, P, n, r) == 0
