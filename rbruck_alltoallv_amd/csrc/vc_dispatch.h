// vc_dispatch.h — which kernel a call gets: every threshold and the one function that applies them.
//
// Host code only, no device state: the library calls vc_dispatch() from every entry point (blocking calls, the _async
// twins, the entry point that allocates nothing), and the CPU tests compile this header to pin the decision table.
//
// The choices, measured on MI355X with blocking calls (microseconds per call unless noted):
//  * through the work-item list (lanes = 0): a planning kernel writes one item per block piece after the host has learnt
//    how many there are.  Right for long blocks; the list and the wait for its size cost more than they save below.
//  * without the list, a quarter of a wavefront per pair of ranks: blocks of a few hundred bytes, any number of ranks.
//    Average piece below 768 B: 26 - 30 at 64 ranks (through the list 42), 42 - 73 at 256 (51 - 88), 300 - 900 at 1024
//    (330 - 990); at 1 KiB the two ways are even.  On at most 128 ranks the alternative is a workgroup per pair, and the
//    quarter wins only further down: never up to 32 ranks (1024 pairs leave room for as many workgroups: 26 either way,
//    the workgroup up to 1.3 x faster on KiB blocks), below 1.75 KiB up to 90 ranks (64 ranks: 27 - 33 against 34 - 38),
//    below 3 KiB above (128 ranks: 30 - 70 against 64 - 84).
//  * ... a batch of 16 or 64 pairs per wavefront when the blocks are so short that working out the routes costs more than
//    moving the bytes: on 192 - 2048 ranks 5 - 40 % faster than the quarter up to an average block of 256 bytes, even at
//    512, 3 - 16 % slower beyond.  Not on at most 128 ranks, where batches would leave most of the chip without a wavefront.
//  * ... for calls that stage in a window, or nothing, a wavefront per pair on 46 ranks and more instead of the list, whatever the average
//    block, while none is more than 16 pieces (vc_closed_wave_from); direct calls on up to 362 ranks a quarter below that.
//  * ... else a wavefront (average piece below 3 KiB) or a workgroup per pair: at most 128 ranks and 32768 pieces (26 - 42
//    against 40 - 57 through the list at 16 and 64 ranks with blocks up to 8 KB, 31 - 77 against 48 - 92 up to 32 KB; a few
//    per cent at 128 ranks; at 256 ranks the list wins).
//  * never without the list after a call with a block of more than 8 (quarter, batch) / 16 (wavefront, workgroup) pieces:
//    one group of lanes moves the pieces of a block in turn.
//  * on fixed-stride staging in ONE launch (stride > 0): the reference's own staging layout, every slot as long as the
//    longest block (src/twophase_tunable_rbruckv.cpp:59), makes slot addresses closed forms, so the call needs no planner
//    at all.  64 ranks with blocks of 0 - 4 KiB 41 -> 24.6; 128 ranks, 0 - 512 B: 41 -> 25.6; 160 ranks: 31 - 42 -> 26 - 34;
//    192 ranks: 31 - 50 -> 30 - 42; but 256 ranks 34 - 68 -> 44 - 68 and 384 ranks 2 x slower (the atomics of the totals
//    and the arena grow with the square of the ranks): only up to 192 ranks and, where the slots do not lie in a window, 256 MiB of arena.
//    In a window, list or planner and copy / one launch: 64 ranks, 0 - 16 KB 53 / 48; 100 ranks, 0 - 8 KB 56 / 52; 128 ranks, 0 - 3 KB 47 / 43; 40 ranks,
//    0 - 30 KB 45 / 39; 150 ranks, power law up to 4 KB 44 / 37.
#pragma once

#include "vc_common.h"
#include "vc_plan_math.h"
#include "vc_scan.h"

#define VC_LISTLESS_MAX_PAIRS 16384           // "small communicator": at most 128 ranks
#define VC_LISTLESS_MAX_ITEMS 32768           // pieces of a call for a wavefront or a workgroup per pair
#define VC_LISTLESS_MAX_PIECES 8              // pieces of one block: quarter of a wavefront per pair, batches
#define VC_LISTLESS_WG_MAX_PIECES 16          // pieces of one block: wavefront or workgroup per pair
#define VC_LISTLESS_QUARTER_BELOW 768         // average piece below which pairs get a quarter of a wavefront, more than 128 ranks
// ... of calls that stage in a window, which need no plan tables then (vc_plan_check), more than 192 ranks.  Calls, list / quarters, by average
// block: 512 ranks, 1 KB 203 / 185, 1.5 KB 262 / 262; 1024 ranks, 1 KB 593 / 572, 1.5 KB 808 / 819; 256 ranks, 1 KB 61 / 61, 1.5 KB 74 / 77.
#define VC_WINDOW_QUARTER_BELOW 1280
// ... and batches from 512 ranks up: quarters / batches, 1024 ranks, 500 B 354 / 326, 700 B 435 / 439; 512 ranks, 500 B 129 / 121; 256 ranks, 700 B 51 / 49
#define VC_WINDOW_BATCH_BELOW 640
#define VC_WINDOW_BATCH_PAIRS (1 << 18)
#define VC_LISTLESS_BATCH_BELOW 384           // average piece below which a wavefront takes a batch of pairs
#define VC_LISTLESS_DIRECT_PAIRS (1 << 17)    // 362 ranks
#define VC_LISTLESS_WAVE_BELOW 3072           // average piece below which a pair gets a wavefront instead of a workgroup
#define VC_LISTLESS_MAX_AVERAGE 4096          // a call the short-block kernels were chosen for must stay below this average
// ... and without plan tables on more than 192 ranks, where the check in front of the copy kernel says what the call is and another shape is two launches
// away: quarters and batches that find an average above VC_CLOSED_MAX_AVERAGE, batches of 64 pairs (a lane a block) on up to 362 ranks one above
// VC_CLOSED_LANE_MAX_AVERAGE, and wavefronts that find fewer bytes for every pair than VC_CLOSED_WAVE_MIN_PER_PAIR leave the call to the shape it asks for.
// Microseconds a call, two kinds in turn, refused from 4096 / 2048 / 1024 / (64 pairs) 512 on: 256 ranks, 0 - 100 and 0 - 1500 B 61 / 61 / 61 / 54, 0 - 100 and 0 - 5000 142 / 93 / 93 / 93,
// 0 - 300 and 0 - 5000 97 / 93 / 93, 0 - 300 and 0 - 3000 78 / 79 / 85; 512, 0 - 100 and 0 - 3000 207 / 206 / 249 / 250, 0 - 300 and 0 - 20000 860 / 770 / 775.  The call
// of 0 - x bytes behind one of long blocks, wavefronts / refused below 320 bytes a pair / 480: 256 ranks, x = 100 69 / 62 / 62, 600 71 / 75 / 74, 900 71 / 71 / 81;
// 350, 100 116 / 91 / 91; 512, 300 233 / 168 / 169; 1024, 300 894 / 565 / 562.
#define VC_CLOSED_MAX_AVERAGE 2048
#define VC_CLOSED_LANE_MAX_AVERAGE 512
#define VC_CLOSED_WAVE_MIN_PER_PAIR 320
#define VC_STRIDED_MAX_BYTES ((int64_t)256 << 20)
// Payload up to which a single launch of wavefronts or workgroups that could use a window does without, where there is room: what little data stages is
// stored past the caches.  64 ranks, 1.2 KB 17.9 us, in a window 18.9; 48 ranks, 4 KB 18.5 / 19.3; but 64 ranks, 4 KB 25.4 / 23.2, 128 ranks, 2 KiB
// 33.2 / 31.3.  Up to 32 ranks the line also decides who signals its own end (VC_SELF_MAX_PAIRS).  Above it, signalled on slots of their own / in a window and
// waited for: 16 ranks, 48 KB 25.7 / 25.5; 20 ranks, 32 KB 23.5 / 21.1, 0 - 68 KB 28.9 / 25.8; 24 ranks, 22 KB 21.4 / 20.3, 32 KB 25.8 / 23.2; 28 ranks, 12.5 KB 21.9 / 21.6;
// 32 ranks, 13 KB 21.3 / 20.9, 16 KiB at radix 4 22.6 / 21.7, 8 20.5 / 20.5, 31 20.5 / 19.1.
#define VC_STRIDED_PAST_CACHES ((int64_t)12 << 20)
#define VC_STRIDED_MAX_PAIRS 36864            // 192 ranks
// In a window a slot may hold more than its stride (vc_window_arena): a single launch there takes blocks of up to this many times the last call's longest, so
// that one that grows a little from call to call does not have every call go out twice (100 ranks, 0 - 600 B, 256 B longer each call 37.1 us -> 18.1).
#define VC_WINDOW_GROWTH 4
// the launch signals its own end: gains up to 32 ranks (32 ranks of 0 - 2 KiB 14.0 us -> 13.5, 24 ranks of 0 - 32 KiB 26.6 -> 22.3), is even
// on 48 (0 - 4 KiB 17.0), and on 64 loses with cold caches what it gains with warm ones (0 - 4 KiB 23.2 -> 25.1, 21.5 -> 19.9): stores past
// the caches fill a memory queue that the L2s would have filled later
#define VC_SELF_MAX_PAIRS 1024
#define VC_SELF_MAX_BYTES ((int64_t)64 << 20)
// list-driven copy kernels: lanes per work item by the average piece of the launch
#define VC_ITEM_QUARTER_BELOW 448
#define VC_ITEM_WAVE_BELOW 3072

// What the last forwarded call on a communicator looked like: the guess about the next one.
struct VcHint {
    int valid;
    int64_t items;        // block pieces
    int64_t payload;      // bytes
    int64_t max_pieces;   // most pieces of one block
    int64_t max_len;      // longest block, bytes
};

// Who asks.  A blocking call may go through the list (it can wait for the list's size in mid-call); the _async twins and
// the entry point that allocates nothing enqueue everything at once and always run without it.
#define VC_CALL_BLOCKING 0
#define VC_CALL_LISTLESS_ONLY 1

struct VcDispatch {
    int lanes;               // 0: through the work-item list; else lanes per pair of ranks of the listless copy kernel:
                             // VC_THREADS, VC_WAVE, VC_QUARTER, or VC_BATCHED (a batch of pairs per wavefront)
    int stride;              // > 0: first try one launch on fixed-stride staging with slots of this many bytes ...
    int stride_lanes;        // ... with this many lanes per pair (the batches come without the totals: a quarter of a wavefront)
    int stride_window;       // ... in a window of this many bytes (VcSched::window), or with a place of its own for every slot (0)
    bool self;               // ... that tells the host itself when it is done
    int batch;               // VC_BATCHED: pairs per wavefront
    int run;                 // ... of 64 pairs: vc_run_vectors
    bool cached;             // vc_reads_cached
    VcListlessGuard guard;   // what the call must look like for the listless kernel to move anything, checked on the device
                             // against the plan (the hint is only a guess); stage_cap is the caller's to fill in
};

// Which single launches can tell the host that they are done: only instances without a window, with a wavefront or a workgroup per pair, store
// past the caches (vc_copy_blocks_kernel).  vc_launch_copy_blocks refuses any other.
VC_HD bool vc_may_signal(int lanes, int window) { return !window && (lanes == VC_WAVE || lanes == VC_THREADS); }

// Pairs per wavefront of the batched listless kernel.  Where a lane moves a block each, all 64 lanes have one; where quarters of the wavefront
// carry the blocks one after the other, short wavefronts keep the chip fuller.  Microseconds a call with 64 / 32 / 16 pairs, blocks of 0 .. x bytes: 1024 ranks, x = 32 53 / 60 / 75, 64 82 (a lane a block)
// / - / 102, 128 120 / - / 151; 256 174 / 165 / 157, 512 224 / 212 / 202, 700 270 / 256 / 245; 512 ranks, 16 30 / 32 / 36, 64 35 / - / 43, 256 82 / 75 / 65, 512
// 91 / 92 / 81; 800 ranks, 512 232 / 223 / 219; 256 ranks, 16 23.5 / 23.5 / 25.3, 100 28 / 28 / 30.
VC_HD int vc_batch_pairs(int64_t longest) { return longest > VC_LANE_BLOCK ? 16 : 64; }

// Batches of 64 pairs: blocks of up to this many vectors of 16 bytes, 1, 2 or 4, move as runs of 8 (vc_copy_runs); 0: a lane, or four lanes, a block.
// Calls, lanes / runs: 1024 ranks of 0 - 16 B 36.5 us / 32.1, 0 - 32 B 44.3 / 36.4, 0 - 64 B 71.5 / 56.3; 2048 at radix 2 of 0 - 16 B 356 / 277, 0 - 60 B 681 / 585; 512 at
// radix 3 of 0 - 30 B 30.7 / 29.8, 0 - 60 B 36.3 / 34.0; 1000, direct, of 0 - 12 B 30.5 / 27.6, 0 - 30 B 36.7 / 30.3, 0 - 60 B 44.4 / 38.6, but 0 - 100 B (8 vectors) 65.8 / 81.5.
// Up to two vectors a route of more than VC_RUN_SLOTS slots leaves nothing to gain but on very many ranks (radix 2, 0 - 20 B: 560 ranks 37.6 / 40.2, 1000 73.3 / 75.9, 1500
// 146 / 152; 0 - 12 B even).
// Nothing is gained where a block is one or two words anyway (elements of 8 bytes: 1000 ranks of 0 - 16 B, direct, 25.8 / 27.7; up to 4 bytes: 0 - 3 B 27.7 / 28.5), nor
// below 512 ranks (300, direct, 17.9 / 18.7).  Elements of 2 and 4 bytes have fewer widths: runs of two vectors gain while the routes take little LDS beside them (1024 ranks, two
// hops, of 0 - 32 B 38.0 / 35.3; at radix 3 800 ranks 45.2 / 46.3), of four where there is staging and pairs enough (0 - 64 B: 1024 63.6 / 55.1; 1000 at
// radix 3 132 / 118, 600 38.7 / 39.0; 1000, direct, 36.4 / 38.0).  Runs of more than one vector take LDS that wavefronts without any miss: calls whose blocks average less than
// a VC_RUN_FILLth of the longest do without (900 ranks in rows of 60 that exchange 50 B among themselves 28.3 / 30.2).  Layouts with gaps, whose wavefronts fall back to
// lanes, lose up to 1 % (1024 ranks of 0 - 60 B 70.8 / 71.2); with runs of 8 vectors, 11 KB a wavefront, it would be 9 % (0 - 100 B 90.8 / 100.3; packed 85.6 / 78.5).
// Where a call stages outside a window, a tile with a block of two hops moves a lane a block (vc_copy_blocks_batch_kernel).  The tiles without are those of neighbouring
// offsets below the radix, of one node: about r of P.  Runs for them / none, blocks of 0 - 60 B, every slot with a place of its own: 1000 ranks at radix 999 60.4 / 66.6, 500 92.2 / 96.0,
// 250 103.6 / 105.2; 512 at 256 34.0 / 34.8, 128 36.5 / 36.1, 23 36.5 / 36.0; 1024 at 32 113.6 / 112.8 (0 - 32 B 33.6 / 33.2 at 23, 53.2 / 59.0 at 999; 0 - 16 B 50.7 / 53.4 at 999).
#define VC_RUN_PAIRS (1 << 18)
#define VC_RUN_ABOVE 4                        // bytes
#define VC_RUN_SLOTS 7
#define VC_RUN_MANY_PAIRS (1 << 22)           // 2048 ranks
#define VC_RUN_WORD_SLOTS 4
#define VC_RUN_WORD_PAIRS (1 << 19)
#define VC_RUN_FILL 8
#define VC_RUN_DIRECT_SHARE 4
VC_HD int vc_run_vectors(const VcSched &S, int64_t longest, int64_t payload) {
    const int64_t pairs = (int64_t)S.P * S.P;
    if (vc_may_stage(S) && !S.window && S.r * VC_RUN_DIRECT_SHARE < S.P) return 0;
    if (pairs < VC_RUN_PAIRS || S.esz % 8 == 0 || longest <= VC_RUN_ABOVE || longest > 64) return 0;
    if (longest <= 32 && vc_hop_slots(S) > VC_RUN_SLOTS && pairs < VC_RUN_MANY_PAIRS) return 0;
    if (longest <= 16) return 1;
    if (payload * VC_RUN_FILL < pairs * longest) return 0;
    if (longest <= 32) return S.esz % 2 || vc_hop_slots(S) <= VC_RUN_WORD_SLOTS ? 2 : 0;
    return S.esz % 2 || (vc_may_stage(S) && pairs >= VC_RUN_WORD_PAIRS) ? 4 : 0;
}

// Fixed stride of a call that stages in a window without being the single launch: the last call's longest block at any cache-line phase, and an odd
// number of lines, so that slots whose blocks are much shorter do not all start at the same few places of the window.  0: blocks too long for it.
#define VC_STRIDE_MAX_LEN ((int64_t)1 << 30)
VC_HD int vc_window_stride(int64_t longest) {
    return longest > VC_STRIDE_MAX_LEN ? 0 : (int)((((longest + 2 * VC_LINE - 1) / VC_LINE) | 1) * VC_LINE);
}

VC_HD int64_t vc_small_quarter_below(int64_t pairs) { return pairs <= 1024 ? 0 : (pairs < 8192 ? 1792 : 3072); }

// Calls whose slots have closed-form places (they stage in a window, or nothing) need no plan tables, and then a wavefront per pair of ranks
// beats the list wherever there are pairs enough to fill the chip, as long as no block is many pieces: it takes up to 8 KiB of a block
// at once, reads no items, and nothing has to be planned and written down before it.  Average pieces from vc_closed_wave_from on get one, below
// vc_closed_quarter_below a quarter or less.  Microseconds a call by average block, before (list, workgroups or quarters) / a wavefront per pair:
//   48 ranks, 4 KB 21.6 / 18.4, 10 KB 31.4 / 28.8;  64, 1.7 KB 21.0 / 18.2, 9 KB 50.6 / 44.8;  100, 2.5 KB 32.1 / 29.1, 9 KB 94 / 75;
//   128, 4 KB 83 / 63, 20 KB 265 / 237;  160, 1.2 KB 49.8 / 44.1, 12 KB 189 / 173;  256, 2 KB 103 / 93, 12 KB 436 / 410;
//   512, 2 KB 326 / 308, 7 KB 1037 / 955;  1024, 4 KB 1980 / 1949;  nothing staged: 128, 5 KB 70 / 47;  300, 2 KB 105 / 87;  800, 2.5 KB 660 / 598.
// Fewer ranks: 34 ranks, 12 KB 24.0 / 30.3, 40 27.0 / 30.5 (but 4 KB 18.9 / 15.6); blocks of up to 40 pieces on 64 ranks 230 / 261.
// The lines: a quarter / a wavefront, 64 ranks, 800 B 17.2 / 17.9, 1.2 KB 19.6 / 18.0; 128, 1.2 KB 30.3 / 31.7, 1.5 KB 33.5 / 31.9; 150, 1030 B 33.1 / 37.6, and
// past what vc_reads_cached holds 1130 B 43.9 / 40.4; 192, 1030 B 58.7 / 57.5; blocks of 0 - 2 x the average, below that limit 95, 1030 B 21.8 / 21.7, 1275 B 22.9 / 21.8; 120,
// 1030 B 25.1 / 28.2, 1275 B 27.0 / 28.4; 140, 1275 B 30.4 / 33.4; beyond it 150, 1150 B 40.8 / 38.7; 160, 1030 B 42.5 / 41.2, 1275 B 46.1 / 42.5; 175, 1030 B 46.9 / 47.4, 1150 B 49.8 / 47.9;
// 190, 1030 B 51.0 / 52.4, 1150 B 54.4 / 52.9; nothing staged 160,
// 1.5 KB 35.9 / 34.8; a list / a wavefront 256, 1.3 KB 77.3 / 79.4; 350, 1.5 KB 150 / 135; 512, 1.65 KB 282 / 281; 800, 1.5 KB 532 / 583; nothing staged 512,
// 1.5 KB 174 / 201, 2.4 KB 274 / 245.  What stages on more than 192 ranks has the list between its two lines: even with quarters on blocks of 0 - 2 x the average (above), slower than them on normal
// ones from 300 ranks up (quarters / list / wavefronts: 256, 1330 B 71.9 / 69.2 / 74.4; 350, 1290 B 113 / 123 / 126; 400, 1450 B 153 / 167 / 161; 512, 1450 B 234 / 248 / 256; 700, 1450 B 420 / 455 / 467; 1024, 1600 B 853 / 867 / 920).
// Beyond 192 ranks direct calls of longer pieces stay with the list (256 ranks, 4 KB 119 / 115, 512 407 / 398).
#define VC_CLOSED_WAVE_PAIRS 2048             // 46 ranks
// Both lines are for calls of at least VC_CLOSED_WAVE_PER_PAIR bytes for every pair of ranks, the empty ones included: a wavefront that starts to find an
// empty block costs as much as any (before / a wavefront per pair, rows of ranks that exchange among themselves: 128 ranks, 750 B a pair in blocks of 6 KB 39 / 23;
// 400, 600 B 93 / 89; 600, 400 B 135 / 159; 1000, 300 B 271 / 401; 64 ranks, 375 B in blocks of 1.5 KB 15.8 / 16.7; nothing staged 100, 660 B 26 / 18; 256,
// 660 B 39 / 39; 600, 730 B 126 / 139).
#define VC_CLOSED_WAVE_PER_PAIR 640
#define VC_CLOSED_DIRECT_PER_PAIR 1920        // more than 362 ranks, nothing staged
VC_HD int64_t vc_closed_sparse_quarter_below(int64_t pairs, bool stages) {
    if (pairs <= VC_LISTLESS_MAX_PAIRS) return vc_small_quarter_below(pairs);
    if (pairs <= (stages ? VC_STRIDED_MAX_PAIRS : VC_LISTLESS_DIRECT_PAIRS)) return VC_LISTLESS_WAVE_BELOW;
    return stages ? VC_WINDOW_QUARTER_BELOW : VC_LISTLESS_QUARTER_BELOW;
}
VC_HD int64_t vc_closed_quarter_below(int64_t pairs, bool stages, bool cached) {
    if (pairs > VC_STRIDED_MAX_PAIRS) return stages ? VC_WINDOW_QUARTER_BELOW : (pairs <= VC_LISTLESS_DIRECT_PAIRS ? 1664 : VC_LISTLESS_QUARTER_BELOW);
    return pairs <= 1024 ? 0 : (pairs < 8192 ? 960 : (stages ? (cached ? 1280 : 1024) : 1664));
}
VC_HD int64_t vc_closed_wave_from(int64_t pairs, bool stages, bool cached) {
    if (pairs <= VC_STRIDED_MAX_PAIRS) return vc_closed_quarter_below(pairs, stages, cached);
    return pairs <= VC_LISTLESS_DIRECT_PAIRS ? (stages ? 1344 : 1664) : (stages ? 1664 : 1920);
}

// mode: vc_comm_set_forwarding (0 launch per digit, 1 the library's choice, 2 the list, 3 / 4 / 5 listless with a workgroup / a
// quarter of a wavefront per pair / batches).  S: the call's schedule (ranks, digits, whether it has an organized region).
inline VcDispatch vc_dispatch(int mode, int call_kind, const VcHint &h, const VcSched &S) {
    VcDispatch d = VcDispatch();
    d.batch = vc_batch_pairs(h.valid ? h.max_len : VC_LANE_BLOCK + 1);
    d.run = vc_run_vectors(S, h.valid ? h.max_len : VC_LANE_BLOCK + 1, h.payload);
    d.cached = h.valid && vc_reads_cached(S, h.payload);
    if (mode == 3) { d.lanes = VC_THREADS; return d; }
    if (mode == 4) { d.lanes = VC_QUARTER; return d; }
    if (mode == 5) { d.lanes = VC_BATCHED; return d; }
    const bool listless_only = call_kind == VC_CALL_LISTLESS_ONLY;
    if (!listless_only && mode != 1) return d;            // per digit, or the list was asked for
    const int64_t pairs = (int64_t)S.P * S.P;
    const bool small_comm = pairs <= VC_LISTLESS_MAX_PAIRS;
    const int64_t average = h.payload / (h.items > 0 ? h.items : 1);
    const bool stages = vc_may_stage(S), closed = S.window || !stages;      // closed: no plan tables, whatever the shape
    const bool dense = h.payload >= (stages || pairs <= VC_LISTLESS_DIRECT_PAIRS ? VC_CLOSED_WAVE_PER_PAIR : VC_CLOSED_DIRECT_PER_PAIR) * pairs;
    const int64_t quarter_below = closed ? (dense ? vc_closed_quarter_below(pairs, stages, d.cached) : vc_closed_sparse_quarter_below(pairs, stages))
                                         : (small_comm ? vc_small_quarter_below(pairs) : VC_LISTLESS_QUARTER_BELOW);
    const bool wave = closed && dense && h.valid && pairs >= VC_CLOSED_WAVE_PAIRS && h.max_pieces <= VC_LISTLESS_WG_MAX_PIECES &&
                      average >= vc_closed_wave_from(pairs, stages, d.cached) && (stages || pairs <= VC_STRIDED_MAX_PAIRS || average < VC_LISTLESS_WAVE_BELOW);
    const bool short_blocks = h.valid && h.max_pieces <= VC_LISTLESS_MAX_PIECES && average < quarter_below;
    if (short_blocks)
        d.lanes = !small_comm && average < (S.window && pairs >= VC_WINDOW_BATCH_PAIRS ? VC_WINDOW_BATCH_BELOW : VC_LISTLESS_BATCH_BELOW) ? VC_BATCHED : VC_QUARTER;
    else if (listless_only)
        d.lanes = wave && average < VC_LISTLESS_WAVE_BELOW ? VC_WAVE : VC_THREADS;
    else if (wave)
        d.lanes = VC_WAVE;
    else if (h.valid && small_comm && h.max_pieces <= VC_LISTLESS_WG_MAX_PIECES && h.items <= VC_LISTLESS_MAX_ITEMS)
        d.lanes = average < VC_LISTLESS_WAVE_BELOW ? VC_WAVE : VC_THREADS;
    else
        return d;                                         // no hint yet, or long blocks: the list
    if (listless_only) return d;                          // nothing to fall back to: whatever the call turns out to be, it runs
    // the hint may be wrong about this call: the kernel leaves a call of another kind alone and the host takes the list
    const bool quarter = d.lanes == VC_QUARTER || d.lanes == VC_BATCHED;
    d.guard.max_pieces = quarter ? VC_LISTLESS_MAX_PIECES : VC_LISTLESS_WG_MAX_PIECES;
    d.guard.max_items = quarter || wave ? 0 : VC_LISTLESS_MAX_ITEMS;
    d.guard.max_average = !quarter ? 0 : (!closed || pairs <= VC_STRIDED_MAX_PAIRS ? VC_LISTLESS_MAX_AVERAGE :
                                          (d.lanes == VC_BATCHED && d.batch == 64 && pairs <= VC_LISTLESS_DIRECT_PAIRS ? VC_CLOSED_LANE_MAX_AVERAGE :
                                           (quarter_below > VC_CLOSED_MAX_AVERAGE ? VC_LISTLESS_MAX_AVERAGE : VC_CLOSED_MAX_AVERAGE)));
    d.guard.min_payload = wave ? VC_CLOSED_WAVE_MIN_PER_PAIR * pairs : 0;
    // one launch on fixed-stride staging: the stride from the last call's longest block, at any cache-line phase
    if (!S.coalesce && vc_hop_slots(S) <= VC_MAX_HOP_SLOTS && pairs <= VC_STRIDED_MAX_PAIRS) {
        const int64_t stride = (h.max_len + 2 * VC_LINE - 1) & ~(int64_t)(VC_LINE - 1);
        VcSched strided = S;
        strided.stride = (int)stride;
        // (in a window the slots may take any room)
        const bool room = vc_strided_stage_bytes(strided) <= VC_STRIDED_MAX_BYTES;
        if (stride <= 0x7FFFFF80 && (S.window || room)) {
            d.stride = (int)stride;
            d.stride_lanes = d.lanes == VC_BATCHED ? VC_QUARTER : d.lanes;
            d.stride_window = room && vc_may_signal(d.stride_lanes, 0) && h.payload <= VC_STRIDED_PAST_CACHES ? 0 : S.window;
            d.self = vc_may_signal(d.stride_lanes, d.stride_window) && pairs <= VC_SELF_MAX_PAIRS && h.payload * vc_hop_slots(S) <= VC_SELF_MAX_BYTES;
            d.guard.max_len = (d.stride_window ? VC_WINDOW_GROWTH : 1) * (stride - VC_LINE + 1);
        }
    }
    return d;
}

// Lanes per work item of the list-driven copy kernels, from the average piece of the launch.  Short pieces leave most of a
// workgroup idle, and what bounds the launch is then the number of items in flight: a wavefront per item keeps four times as
// many as a workgroup, a quarter of a wavefront sixteen times.  Measured on 1 Mi items (1024 ranks, times of the copy kernel,
// workgroup / wavefront / quarter): pieces uniform in 0..16 B 830 / 269 / 67 us, 0..256 B 882 / 351 / 189, 0..1 KiB
// 926 / 455 / 431, 0..2 KiB 1105 / 693 / 770, 0..4 KiB 1449 / 1311 / 1462; around 4 KiB and above the workgroup is 5 - 8 %
// faster than the wavefront.
VC_HD int vc_lanes_for_items(int64_t bytes, int64_t items) {
    if (items <= 0) return VC_THREADS;
    const int64_t average = bytes / items;
    return average < VC_ITEM_QUARTER_BELOW ? VC_QUARTER : (average < VC_ITEM_WAVE_BELOW ? VC_WAVE : VC_THREADS);
}

// Groups of four items in a row per wavefront of the quarter kernels: as many as leave every SIMD of the chip a few wavefronts.
VC_HD int vc_quarter_rounds(int64_t items) { return items >= ((int64_t)1 << 19) ? 4 : (items >= ((int64_t)1 << 17) ? 2 : 1); }
