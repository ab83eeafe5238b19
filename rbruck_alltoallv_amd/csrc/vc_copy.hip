// vc_copy.hip — the data mover.  A Bruck round on P virtual ranks is a set of
// independent block copies inside HBM: the reference's pack (memcpy into
// temp_send_buffer), MPI_Sendrecv and unpack (memcpy out of temp_recv_buffer)
// (src/twophase_tunable_rbruckv.cpp:90-100,119,126-139) collapse into one read of
// the block where the sender holds it and one write where the receiver wants it.
//
// Shape of the kernels, chosen by measurement on MI355X: one work item = a piece of one block that fits a window of
// VC_CHUNK = 8 KiB; every lane moves 16-byte vectors whose loads are all issued before the stores, non-temporal on both
// sides (the data is touched once per hop).  For pieces of several KiB a 256-lane workgroup per item is fastest (many
// small workgroups beat persistent or wider ones for a plain copy on this chip, and the same holds for the scattered
// variable-size blocks of an alltoallv); lists of short pieces are bound by the number of items in flight and get a
// wavefront, or a quarter of one, per item.  The host chooses per launch (vc_lanes_for_items in vc_dispatch.h).
//
// Workgroups are handed to the 8 XCDs of the chip in turn (workgroup b runs on XCD
// b mod 8) and every XCD has its own L2.  Work items that follow each other in the
// list are neighbours in memory (pieces of one block, blocks of one run), so each
// XCD takes a contiguous eighth of the list instead of every eighth item: cache
// lines shared by two neighbouring items then meet in one L2, and every XCD streams
// through its own range of addresses.  Measured: +3 % on 4 KiB blocks, +15 % on
// 1 MiB blocks cut into pieces.
#include "vc_common.h"
#include "vc_dispatch.h"
#include "vc_plan_math.h"
#include "vc_scan.h"

#include <type_traits>

typedef unsigned int vc_u32x4 __attribute__((ext_vector_type(4)));
struct __attribute__((packed, aligned(1))) VcU128 { vc_u32x4 v; };

// 16-byte load from any byte address (one global_load_dwordx4; the hardware handles the misalignment).  CACHED: an ordinary one, served by the
// memory-side cache when the caller, or the last call, has left the input there, and leaving it there; see vc_reads_cached.
template <bool CACHED> __device__ __forceinline__ vc_u32x4 vc_load16(const char *p) {
    const vc_u32x4 *const v = &reinterpret_cast<const VcU128 *>(p)->v;
    return CACHED ? reinterpret_cast<const VcU128 *>(p)->v : __builtin_nontemporal_load(v);
}

// 16-byte store to a 16-byte aligned address
__device__ __forceinline__ void vc_store16(char *p, vc_u32x4 v) {
    __builtin_nontemporal_store(v, reinterpret_cast<vc_u32x4 *>(p));
}

// ... past the caches (THROUGH: for a kernel that signals its own end, vc_signal), to any byte address.  The wait states behind the store: a vector
// instruction must not write the registers of a store of more than 8 bytes right behind it, and the compiler, which keeps them apart
// for its own stores, does not see this one.
__device__ __forceinline__ void vc_store16_through(char *p, vc_u32x4 v) {
    asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 3" ::"v"(p), "v"(v) : "memory");
}

// ... of a call that stages in a window: an ordinary store, so that the window stays in the caches.  What goes to recvbuf is stored the same
// way (non-temporal: 1024 ranks, 4 KiB 1993 us -> 2066; 256 ranks, Zipf 148 -> 181), but not in calls that stage nothing (512 ranks, 1 KiB
// 200 -> 191).  Calls with and without a window have kernels of their own: of two branches that only differ in the kind of their
// stores the compiler makes one, with ordinary stores.
template <bool WINDOW> __device__ __forceinline__ void vc_store16_of(char *p, vc_u32x4 v) {
    if (WINDOW) *reinterpret_cast<vc_u32x4 *>(p) = v; else vc_store16(p, v);
}

// ... to recvbuf, of a piece that goes nowhere else, in a call that stages in a window: as in calls that stage nothing.  As an
// instruction, so that it stays the kind of store it is next to the ordinary ones; wait states as above.  512 ranks, radix 511, 1 MiB blocks, nearly all
// of one hop 5988 us with ordinary stores, 5437 so; 64 ranks, radix 63, planned 1440 / 1345; 256 ranks, radix 255, 4 KB 125 / 117.
__device__ __forceinline__ void vc_store16_alone(char *p, vc_u32x4 v) {
    asm volatile("global_store_dwordx4 %0, %1, off nt\n\ts_nop 3" ::"v"(p), "v"(v) : "memory");
}

// mask: vc_window_mask of the call, for the place of a piece in the staging arena
__device__ __forceinline__ char *vc_resolve(int64_t loc, const char *sendbuf, char *recvbuf, char *stage, int64_t mask = -1) {
    const int space = (int)(loc >> VC_SPACE_SHIFT);
    const int64_t off = loc & VC_OFFSET_MASK & (space >= 2 ? mask : -1);
    char *base = space == 0 ? const_cast<char *>(sendbuf) : (space == 1 ? recvbuf : stage);
    return base + off;
}

#define VC_XCDS 8
// Workgroups of one launch: a dispatch counts its grid in work-items in 32 bits, so gridDim.x * VC_THREADS must stay
// below 2^32 (a larger grid is not refused: it runs truncated); longer lists go out in several launches.  A multiple of
// VC_XCDS.
#define VC_MAX_GRID ((int64_t)((1ull << 32) / VC_THREADS) - VC_XCDS)

// One workgroup (or one wavefront) of LANES lanes moves one piece.  Lane t owns the t-th, (t + LANES)-th, ... 16-byte vector
// of the window that starts at the 128-byte boundary at or below dst, so every wave stores whole cache lines whatever
// the byte phase of the block (measured: +4 % over counting vectors from the first 16-byte boundary of dst).  Vectors
// that lie fully inside the block are moved by (possibly unaligned) 16-byte loads and aligned stores; the < 16 bytes
// before the first and after the last of them are moved byte-wise (lanes 0..15 the head, lanes 16..31 the tail: one byte
// load and one byte store each).  The planner guarantees len + (dst & 127) <= VC_CHUNK.
// With nhop > 1 this is forwarded execution: the piece is read once, from sendbuf, and every hop stores the same
// registers (all destinations of a block share the offset inside their cache line, `w`, so one mapping of lanes to window
// vectors serves them all).  next_dst() is where the next hop puts the piece.
// WINDOW: the call stages in a window (vc_store16_of).
// go() is asked once, after the loads have been issued and before the first store: false leaves the piece where it is.
#define VC_WAIT_VMCNT0 0x0F70              // s_waitcnt vmcnt(0): loads have arrived and stores have been acknowledged
struct VcAlwaysGo { __device__ __forceinline__ bool operator()() const { return true; } };

template <int LANES, bool THROUGH, bool WINDOW, bool CACHED, class NextDst, class Go = VcAlwaysGo>
__device__ __forceinline__ void vc_forward_piece(const char *src, int64_t len, int nhop, int w, NextDst next_dst, Go go = Go()) {
    constexpr int VECS = VC_CHUNK / 16 / LANES;           // window vectors per lane: 2 for a workgroup of 256, 8 for one wavefront
    const int t = threadIdx.x;
    const int n = (int)len;                               // (a piece fits the window)
    if (!THROUGH && n == VC_PIECE && w == 0) {
        // A whole aligned piece, the inside of a long block: no vector to leave out and no edge.  Without a window a wavefront waits for each
        // of its stores before the next one: on lists of these the memory runs a few per cent faster with fewer writes in flight
        // (64 ranks, 1.3 MB blocks, two hops, builds in turn in one process, quartiles within 0.4 %: without this path 2430 us, with it but
        // without the waits 2407, so 2349; 512 ranks, 1 MiB blocks 6527 / 6494 / 6474).
        constexpr int WHOLE = VC_PIECE / 16 / LANES;
        vc_u32x4 v[WHOLE];
#pragma unroll
        for (int i = 0; i < WHOLE; i++) v[i] = vc_load16<CACHED>(src + ((t + i * LANES) << 4));
        if (!go()) return;
        if (WINDOW && nhop == 1) {
            char *dst = next_dst();
#pragma unroll
            for (int i = 0; i < WHOLE; i++) {
                if (i) __builtin_amdgcn_s_waitcnt(VC_WAIT_VMCNT0);
                vc_store16_alone(dst + ((t + i * LANES) << 4), v[i]);
            }
            return;
        }
        for (int k = 0; k < nhop; k++) {
            char *dst = next_dst();
#pragma unroll
            for (int i = 0; i < WHOLE; i++) {
                if (!WINDOW && (k || i)) __builtin_amdgcn_s_waitcnt(VC_WAIT_VMCNT0);
                vc_store16_of<WINDOW>(dst + ((t + i * LANES) << 4), v[i]);
            }
        }
        return;
    }
    const int first_full = (w + 15) >> 4, end_full = (w + n) >> 4;
    const char *sw = src - w;
    vc_u32x4 v[VECS];
    bool has[VECS];
#pragma unroll
    for (int i = 0; i < VECS; i++) {
        const int j = t + i * LANES;
        has[i] = (i > 0 || j >= first_full) && j < end_full;
        if (has[i]) v[i] = vc_load16<CACHED>(sw + (j << 4));
    }
    int head = (first_full << 4) - w;
    if (head > n) head = n;
    int done = (end_full << 4) - w;
    if (done < head) done = head;
    const int edge = t < 16 ? (t < head ? t : -1) : (t < 32 && done + (t - 16) < n ? done + (t - 16) : -1);
    char edge_byte = 0;
    if (edge >= 0) edge_byte = src[edge];
    if (!go()) return;
    // all at once and after the last load has arrived, so that the writes of one line reach the L2 together (calls, builds in turn in one
    // process: 512 ranks, 1 KiB 197 us -> 188; 1024 ranks, 4 KiB 2486 -> 2453; 256 ranks, Zipf 165.0 -> 166.2)
    __builtin_amdgcn_s_waitcnt(VC_WAIT_VMCNT0);
    if (WINDOW && nhop == 1) {
        char *dst = next_dst(), *dw = dst - w;
        if (edge >= 0) dst[edge] = edge_byte;
#pragma unroll
        for (int i = 0; i < VECS; i++)
            if (has[i]) vc_store16_alone(dw + ((t + i * LANES) << 4), v[i]);
        return;
    }
    for (int k = 0; k < nhop; k++) {
        char *dst = next_dst(), *dw = dst - w;
        if (edge >= 0) { if (THROUGH) vc_store_through(dst + edge, edge_byte); else dst[edge] = edge_byte; }
#pragma unroll
        for (int i = 0; i < VECS; i++)
            if (has[i]) { if (THROUGH) vc_store16_through(dw + ((t + i * LANES) << 4), v[i]); else vc_store16_of<WINDOW>(dw + ((t + i * LANES) << 4), v[i]); }
    }
}

// LANES = VC_THREADS: one workgroup of four wavefronts per item, the shape that moves blocks of several KiB fastest.
// LANES = VC_WAVE: one wavefront per item, for lists of short pieces: four times as many items in flight per compute
// unit, and no wavefronts that start only to find nothing left for them in a piece of a few hundred bytes.
// GUARDED: the launch was enqueued before the host had seen the plan (see VcChainGuard): `nitems` is a guess, header[2] the
// truth, and nothing moves unless the plan is one this launch can serve.
// WINDOW: the plan stages in a window of `window` bytes.
template <int LANES, bool GUARDED, bool WINDOW, bool CACHED>
__global__ __launch_bounds__(LANES) void vc_copy_chains_kernel(const int64_t *__restrict__ items, int stride, unsigned nitems,
                                                               const char *__restrict__ sendbuf, char *__restrict__ recvbuf,
                                                               char *__restrict__ stage, const int64_t *__restrict__ header,
                                                               VcChainGuard guard, int window) {
    const unsigned per = gridDim.x / VC_XCDS;
    const unsigned idx = (blockIdx.x % VC_XCDS) * per + blockIdx.x / VC_XCDS;
    if (idx >= nitems) return;
    const int64_t *it = items + (int64_t)idx * stride;    // (there is room for nitems items, whatever is in them)
    const int64_t len = it[VC_CHAIN_LEN];
    const int nhop = (int)it[VC_CHAIN_NHOP];
    bool ok = (len > 0) & (nhop > 0);                     // (one condition: item and header are read together)
    if (GUARDED) ok = ok & vc_chain_guard_ok(header, guard) & ((int64_t)idx < header[2]);
    if (!ok) return;
    const char *src = vc_resolve(it[VC_CHAIN_SRC], sendbuf, recvbuf, stage);
    const int64_t mask = WINDOW ? vc_window_mask(window) : -1;
    char *dst = vc_resolve(it[VC_CHAIN_HEAD], sendbuf, recvbuf, stage, mask);
    const int w = (int)((uintptr_t)dst & (VC_LINE - 1)), lane = threadIdx.x % VC_WAVE;
    // the hops after the first in one read, a word per lane: a load between the stores would wait for the stores before it
    int64_t word = 0;
    if (lane < nhop) word = it[VC_CHAIN_HEAD + lane];
    int at = 0;
    vc_forward_piece<LANES, false, WINDOW, CACHED>(src, len, nhop, w, [&]() {
        const unsigned lo = __builtin_amdgcn_readlane((int)word, at), hi = __builtin_amdgcn_readlane((int)(word >> 32), at);
        return at++ ? vc_resolve((int64_t)hi << 32 | lo, sendbuf, recvbuf, stage, mask) : dst;
    });
}

// Launch-per-digit execution: one hop of one piece per item.
template <int LANES>
__global__ __launch_bounds__(LANES) void vc_copy_items_kernel(const VcDesc *__restrict__ items, unsigned nitems,
                                                              const char *__restrict__ sendbuf, char *__restrict__ recvbuf,
                                                              char *__restrict__ stage) {
    // gridDim.x is a multiple of VC_XCDS; XCD k = blockIdx.x % VC_XCDS works through items [k * per, (k + 1) * per)
    const unsigned per = gridDim.x / VC_XCDS;
    const unsigned idx = (blockIdx.x % VC_XCDS) * per + blockIdx.x / VC_XCDS;
    if (idx >= nitems) return;
    const VcDesc d = items[idx];
    if (d.len <= 0) return;
    char *dst = vc_resolve(d.dst, sendbuf, recvbuf, stage);
    vc_forward_piece<LANES, false, false, false>(vc_resolve(d.src, sendbuf, recvbuf, stage), d.len, 1, (int)((uintptr_t)dst & (VC_LINE - 1)), [&]() { return dst; });
}

// A quarter of a wavefront (16 lanes) per item, four items per wavefront, for lists of pieces of a few hundred bytes:
// such a launch is bound by how many items are in flight, not by HBM, and a piece of 100 bytes has work for 7 lanes.
// Every group of 16 lanes reads its own item; lane t of the group owns window vectors t, t + 16 of every 512-byte pass
// (most items need one pass; longer ones loop), and moves head byte t and tail byte t.
template <bool WINDOW, bool CACHED, class DstOf>
__device__ __forceinline__ void vc_forward_piece_quarter(const char *src, int64_t len, int nhop, DstOf dst_of) {
    const int t = threadIdx.x & 15;
    char *dst = dst_of(0);
    const int64_t w = (int64_t)((uintptr_t)dst & (VC_LINE - 1));
    const int64_t first_full = (w + 15) >> 4, end_full = (w + len) >> 4;
    int64_t head = (first_full << 4) - w;
    if (head > len) head = len;
    int64_t done = (end_full << 4) - w;
    if (done < head) done = head;
    const bool has_head = t < head, has_tail = done + t < len;
    char head_byte = 0, tail_byte = 0;
    if (has_head) head_byte = src[t];
    if (has_tail) tail_byte = src[done + t];
    const char *sw = src - w;
    bool first_pass = true;                               // the pass that also stores the head and tail bytes: there is
    for (int64_t j = t; first_pass || j < end_full; j += 32) {     // always one, also for a block without a full vector
        const bool has0 = j >= first_full && j < end_full, has1 = j + 16 >= first_full && j + 16 < end_full;
        vc_u32x4 v0, v1;
        if (has0) v0 = vc_load16<CACHED>(sw + (j << 4));
        if (has1) v1 = vc_load16<CACHED>(sw + ((j + 16) << 4));
        for (int k = 0; k < nhop; k++) {
            if (k || !first_pass) dst = dst_of(k);
            char *dw = dst - w;
            if (first_pass && has_head) dst[t] = head_byte;
            if (first_pass && has_tail) dst[done + t] = tail_byte;
            if (has0) vc_store16_of<WINDOW>(dw + (j << 4), v0);
            if (has1) vc_store16_of<WINDOW>(dw + ((j + 16) << 4), v1);
        }
        first_pass = false;
    }
}

// ---- blocks of a few hundred bytes, without byte-wise edges ----
// What bounds these is the number of requests the copying sends to the L2 (72 - 85 per ns on this chip by the kernel's mix of reads and writes: a
// request writes at most 64 bytes), so every byte-wise head and tail counts as much as a whole vector.  Edges are moved as
// 16-byte vectors that start or end with the block and overlap the aligned ones (the same bytes, twice).
struct __attribute__((packed, aligned(1))) VcU64 { unsigned long long v; };
struct __attribute__((packed, aligned(1))) VcU32 { unsigned v; };
struct __attribute__((packed, aligned(1))) VcU16 { unsigned short v; };

// A block of 1 .. VC_LANE_BLOCK bytes in one lane's registers: its first and its last 16 (8, 4, 2, 1) bytes, which overlap, and the
// vectors between them.  Every width is an instruction of its own for the lanes that have it, and these are what such a call is bound by (the address units, 29 clocks an
// instruction of a wavefront whose lanes go to 64 places, busy for nearly 0.9 of the time): 16 bytes are two of 8, so that shorter blocks have one width less beside
// them, and in a window the staged hops of a block of up to 16 bytes are one vector (vc_lane_vector).  Calls, before / after: 1024 ranks of 0 - 16 B 44.2 us / 36.9, of 0 - 32 B at
// radix 2 67.3 / 52.0; 512 of 0 - 60 B 46.7 / 41.0; 1024 of 0 - 128 B 116.6 / 108.5 (there it is the slot's start, fewer lines a block); 256 of 0 - 40 B 24.1 / 23.4.
#define VC_LANE_MIDDLE (VC_LANE_BLOCK / 16 - 2)
struct VcLaneBlock { vc_u32x4 first, last, middle[VC_LANE_MIDDLE]; };

__device__ __forceinline__ VcLaneBlock vc_lane_load(const char *src, int len) {
    VcLaneBlock b;
    b.first = b.last = vc_u32x4{0, 0, 0, 0};
    if (len > 16) {
        b.first = reinterpret_cast<const VcU128 *>(src)->v;
        b.last = reinterpret_cast<const VcU128 *>(src + len - 16)->v;
#pragma unroll
        for (int k = 0; k < VC_LANE_MIDDLE; k++)
            if (len > 32 + 16 * k) b.middle[k] = reinterpret_cast<const VcU128 *>(src + 16 + 16 * k)->v;
    } else if (len >= 8) {
        const unsigned long long x = reinterpret_cast<const VcU64 *>(src)->v, y = reinterpret_cast<const VcU64 *>(src + len - 8)->v;
        b.first.x = (unsigned)x; b.first.y = (unsigned)(x >> 32); b.last.x = (unsigned)y; b.last.y = (unsigned)(y >> 32);
    } else if (len >= 4) {
        b.first.x = reinterpret_cast<const VcU32 *>(src)->v;
        b.last.x = reinterpret_cast<const VcU32 *>(src + len - 4)->v;
    } else if (len >= 2) {
        b.first.x = reinterpret_cast<const VcU16 *>(src)->v;
        b.last.x = reinterpret_cast<const VcU16 *>(src + len - 2)->v;
    } else {
        b.first.x = *reinterpret_cast<const unsigned char *>(src);
    }
    return b;
}

__device__ __forceinline__ void vc_lane_store(const VcLaneBlock &b, char *dst, int len) {
    if (len > 16) {
        reinterpret_cast<VcU128 *>(dst)->v = b.first;
#pragma unroll
        for (int k = 0; k < VC_LANE_MIDDLE; k++)
            if (len > 32 + 16 * k) reinterpret_cast<VcU128 *>(dst + 16 + 16 * k)->v = b.middle[k];
        reinterpret_cast<VcU128 *>(dst + len - 16)->v = b.last;
    } else if (len >= 8) {
        reinterpret_cast<VcU64 *>(dst)->v = (unsigned long long)b.first.y << 32 | b.first.x;
        reinterpret_cast<VcU64 *>(dst + len - 8)->v = (unsigned long long)b.last.y << 32 | b.last.x;
    } else if (len >= 4) {
        reinterpret_cast<VcU32 *>(dst)->v = b.first.x;
        reinterpret_cast<VcU32 *>(dst + len - 4)->v = b.last.x;
    } else if (len >= 2) {
        reinterpret_cast<VcU16 *>(dst)->v = (unsigned short)b.first.x;
        reinterpret_cast<VcU16 *>(dst + len - 2)->v = (unsigned short)b.last.x;
    } else {
        *dst = (char)b.first.x;
    }
}

// The same block for the start of a slot in a window: one of no more than 16 bytes is one vector there, one instruction for all lanes whatever their widths.  What the
// vector has behind the block is in no one's way: a slot is at least a line, and nothing reads it.  (Shifts of a whole word, lengths 8 and 4, leave nothing
// of the block behind it.)
__device__ __forceinline__ vc_u32x4 vc_lane_vector(const VcLaneBlock &b, int len) {
    vc_u32x4 v = b.first;
    if (len >= 8) {
        const unsigned long long y = ((unsigned long long)b.last.y << 32 | b.last.x) >> (8 * (16 - len) & 63);
        v.z = (unsigned)y; v.w = (unsigned)(y >> 32);
    } else if (len >= 4) {
        v.y = b.last.x >> (8 * (8 - len) & 31);
    } else if (len == 3) {
        v.x = b.first.x | b.last.x << 8;
    }
    return v;
}

// Where a hop puts a block, and where it puts the piece that starts `lo` bytes into it: in a window the place wraps.  at_start: at the slot's start instead of at
// the line phase of the block in recvbuf.
template <bool WINDOW>
__device__ __forceinline__ char *vc_hop_at(const VcSched &S, const VcHop &h, int64_t slot, int64_t recv_off, char *recvbuf, char *stage, bool at_start = false) {
    if (WINDOW) slot &= vc_window_mask(S.window);
    return h.staged ? stage + slot + (at_start ? 0 : ((int)recv_off + S.recv_lo & (VC_LINE - 1))) : recvbuf + recv_off;
}
template <bool WINDOW> __device__ __forceinline__ char *vc_piece_at(const VcSched &S, char *dst, int64_t lo, char *stage) {
    const uint64_t place = dst - stage;
    return WINDOW && place < (uint64_t)S.window ? stage + ((place + lo) & vc_window_mask(S.window)) : dst + lo;
}

// A piece of a block (it fits VC_CHUNK) moved by GROUP neighbouring lanes, a quarter of a wavefront or fewer: lane t owns window vectors t, t + GROUP, ... (the window starts at the
// cache line of the destination, `w` bytes before it), VECS of them in flight at once.  Staging without a window is stored past the
// caches (nothing reads it again); recvbuf is not: a line that two neighbouring blocks share is then put together in the L2.
// Instructions count here as much as requests: with 8 wavefronts a SIMD the vector ALUs were busy more than half of the time while places were decoded
// for every hop (vc_resolve) and pieces counted in 64 bits.  Destinations that are pointers, clamped 32-bit offsets and one copy of this code per kernel
// (a second one for whole blocks made single launches 2 - 7 % slower: code is fetched anew by every launch): calls, before / after, 1024 ranks of 0 - 256 B 149 us / 131,
// 0 - 512 B 197 / 193, 0 - 1400 B 426 / 391; 512 ranks of 0 - 256 B 64.1 / 60.2.
template <int GROUP, int VECS, bool WINDOW, bool CACHED, class DstOf, class Go = VcAlwaysGo>
__device__ __forceinline__ void vc_forward_short(const char *src, int len, int nhop, int w, DstOf dst_of, Go go = Go()) {
    const int t = threadIdx.x % GROUP;
    if (len < 16) {
        VcLaneBlock b;
        if (t == 0) b = vc_lane_load(src, len);
        if (!go()) return;
        if (t == 0)
            for (int k = 0; k < nhop; k++) vc_lane_store(b, dst_of(k), len);
        return;
    }
    for (int base = -w; base < len; base += VECS * GROUP * 16) {
        vc_u32x4 v[VECS];
        unsigned at[VECS];                                // where the vector starts inside the block
        bool has[VECS];
#pragma unroll
        for (int i = 0; i < VECS; i++) {
            const int lo = base + (t << 4) + i * GROUP * 16;
            has[i] = (unsigned)(lo + 15) < (unsigned)(len + 15);
            at[i] = lo < 0 ? 0 : (lo > len - 16 ? len - 16 : lo);
            if (has[i]) v[i] = vc_load16<CACHED>(src + at[i]);
        }
        if (base == -w && !go()) return;
        for (int k = 0; k < nhop; k++) {
            char *dst = dst_of(k);
            if (WINDOW || k == nhop - 1) {
#pragma unroll
                for (int i = 0; i < VECS; i++)
                    if (has[i]) reinterpret_cast<VcU128 *>(dst + at[i])->v = v[i];
            } else {
#pragma unroll
                for (int i = 0; i < VECS; i++)
                    if (has[i]) __builtin_nontemporal_store(v[i], &reinterpret_cast<VcU128 *>(dst + at[i])->v);
            }
        }
    }
}

// A whole block: the route's destinations are `dsts`.  Only a block of several pieces is cut.
template <int GROUP, int VECS, bool WINDOW, bool CACHED, class Go = VcAlwaysGo>
__device__ __forceinline__ void vc_forward_block(const VcSched &S, const char *src, int64_t len, int nhop, int cut, char *const *dsts, char *stage, Go go = Go()) {
    const int phase = cut & (VC_LINE - 1);
    const bool one = vc_fits_one_item(len, phase);
    int64_t lo = 0;
    do {                                                  // the same cuts as the chain items of this block
        const int64_t hi = one || lo + VC_PIECE >= len + (lo ? 0 : cut) ? len : (lo ? lo : -cut) + VC_PIECE;
        vc_forward_short<GROUP, VECS, WINDOW, CACHED>(src + lo, (int)(hi - lo), nhop, lo ? 0 : phase, [&](int k) { return lo ? vc_piece_at<WINDOW>(S, dsts[k], lo, stage) : dsts[k]; }, go);
        lo = hi;
    } while (lo < len);
}

#define VC_ITEMS_PER_WAVE (VC_WAVE / VC_QUARTER)

// gridDim.x wavefronts, a multiple of VC_XCDS; XCD k works through the k-th eighth of them, each taking four items in a row
// `rounds`: groups of four items in a row a wavefront takes, one after the other (long lists of very short pieces: fewer
// wavefronts, each paying its start-up once for more items)
template <bool GUARDED, bool WINDOW, bool CACHED>
__global__ __launch_bounds__(VC_WAVE) void vc_copy_chains_quarter_kernel(const int64_t *__restrict__ items, int stride, unsigned nitems,
                                                                         int rounds, const char *__restrict__ sendbuf,
                                                                         char *__restrict__ recvbuf, char *__restrict__ stage,
                                                                         const int64_t *__restrict__ header,
                                                                         VcChainGuard guard, int window) {
    const unsigned per = gridDim.x / VC_XCDS;
    const unsigned wave = (blockIdx.x % VC_XCDS) * per + blockIdx.x / VC_XCDS;
    if (GUARDED && !vc_chain_guard_ok(header, guard)) return;
    for (int round = 0; round < rounds; round++) {
        const int64_t idx = ((int64_t)wave * rounds + round) * VC_ITEMS_PER_WAVE + threadIdx.x / VC_QUARTER;
        if (idx >= nitems || (GUARDED && idx >= header[2])) continue;
        const int64_t *it = items + idx * stride;
        const int64_t len = it[VC_CHAIN_LEN];
        const int nhop = (int)it[VC_CHAIN_NHOP];
        if (len <= 0 || nhop <= 0) continue;
        const int64_t mask = WINDOW ? vc_window_mask(window) : -1;
        vc_forward_piece_quarter<WINDOW, CACHED>(vc_resolve(it[VC_CHAIN_SRC], sendbuf, recvbuf, stage), len, nhop,
                                         [&](int k) { return vc_resolve(it[VC_CHAIN_HEAD + k], sendbuf, recvbuf, stage, mask); });
    }
}

__global__ __launch_bounds__(VC_WAVE) void vc_copy_items_quarter_kernel(const VcDesc *__restrict__ items, unsigned nitems, int rounds,
                                                                        const char *__restrict__ sendbuf, char *__restrict__ recvbuf,
                                                                        char *__restrict__ stage) {
    const unsigned per = gridDim.x / VC_XCDS;
    const unsigned wave = (blockIdx.x % VC_XCDS) * per + blockIdx.x / VC_XCDS;
    for (int round = 0; round < rounds; round++) {
        const int64_t idx = ((int64_t)wave * rounds + round) * VC_ITEMS_PER_WAVE + threadIdx.x / VC_QUARTER;
        if (idx >= nitems) continue;
        const VcDesc d = items[idx];
        if (d.len <= 0) continue;
        char *dst = vc_resolve(d.dst, sendbuf, recvbuf, stage);
        vc_forward_piece_quarter<false, false>(vc_resolve(d.src, sendbuf, recvbuf, stage), d.len, 1, [&](int) { return dst; });
    }
}

// ---- fixed-stride staging in one launch (the `verdict` of vc_launch_copy_blocks) ----
// The wavefronts of the first vc_totals_blocks workgroups of the grid: four pairs of ranks per lane (by receiver, then
// source).  Each puts its sums and maxima into a slot of its own in host memory, and the host adds the slots up when the launch
// is over; their verdict goes into VC_VERDICTS copies of one word, and every copying wavefront looks at one of them.  (With an atomic
// per wavefront on each of six shared words, and one verdict word that all wavefronts polled, these were what the launch waited for:
// atomics on one address follow each other at about 10 ns.  Kernel times with warm caches: 128 ranks, 2 KiB blocks 27.6 us -> 24.5; 64 ranks
// of 0 - 4 KiB 14.3 -> 12.8.)
// lanes: of the workgroup.
__device__ __forceinline__ void vc_add_totals(const VcSched &S, const VcTables &T, unsigned long long *verdict, int64_t *totals, int lanes) {
    const int P = S.P, pairs = P * P, per_wave = VC_TOTALS_PER_WAVE, nwaves = (int)vc_totals_waves(P);      // P^2 <= VC_STRIDED_MAX_PAIRS
    const int wave = (int)blockIdx.x * (lanes / VC_WAVE) + (int)threadIdx.x / VC_WAVE;
    if (wave >= nwaves) return;
    const int lane = threadIdx.x & (VC_WAVE - 1);
    // The verdict on the tables first, with nothing but one round of reads in front of it (all of a lane's pairs together): the
    // copying wavefronts of this launch hold their stores back until every totalling wavefront has reported (VcVerdictGate).
    VcPairEntries e[VC_TOTALS_PER_LANE];
    unsigned rbase[VC_TOTALS_PER_LANE];                   // (its low 32 bits: they say where a block is cut)
    int src[VC_TOTALS_PER_LANE], dst[VC_TOTALS_PER_LANE];
#pragma unroll
    for (int u = 0; u < VC_TOTALS_PER_LANE; u++) {
        const int idx = wave * per_wave + u * VC_WAVE + lane, in = idx < pairs ? idx : 0;
        dst[u] = vc_div(in, S.dP);
        src[u] = in - dst[u] * P;
    }
#pragma unroll
    for (int u = 0; u < VC_TOTALS_PER_LANE; u++) {
        e[u] = vc_pair_entries(S, T, src[u], dst[u]);
        rbase[u] = *reinterpret_cast<const unsigned *>(T.rbase + dst[u]);
    }
    // All of them are on their way before the first one is waited for: left to itself the compiler reads the entries in three rounds, one of them behind a
    // condition (150 ranks, power law up to 4 KB 31.9 us a call -> 30.1; 192 ranks of 0 - 1200 B 32.0 / 29.8; direct, 150 ranks of 0 - 1.5 KB 22.9 / 21.4).
#pragma unroll
    for (int u = 0; u < VC_TOTALS_PER_LANE; u++) asm volatile("" : "+v"(e[u].sent), "+v"(e[u].expected), "+v"(e[u].rd), "+v"(e[u].own), "+v"(rbase[u]));
    int64_t bad = 0;
#pragma unroll
    for (int u = 0; u < VC_TOTALS_PER_LANE; u++) {
        if (wave * per_wave + u * VC_WAVE + lane >= pairs) continue;
        bad += vc_bad_entries(S, e[u]);                   // the same count the planner makes
        // (a packed receive layout past INT_MAX elements shows as a negative packed displacement of a later source)
        if (S.packed_recv && (e[u].rd < 0 || (src[u] == P - 1 && (int64_t)e[u].rd + e[u].expected > 0x7FFFFFFF))) bad += VC_BAD_OVERFLOW;
    }
    // one word says it all, so one atomic instruction publishes it in every copy: wavefronts that have reported in the low half,
    // wavefronts that found something wrong in the high half
    const unsigned long long report = __ballot(bad != 0) ? 1ull | 1ull << 32 : 1ull;
    if (lane < VC_VERDICTS) atomicAdd(verdict + lane * (VC_LINE / 8), report);
    bad = vc_wave_inclusive_scan(bad);                    // (lane 63 has the sum)
    int64_t payload = 0, items = 0, most = 0, moved = 0, longest = 0;
#pragma unroll
    for (int u = 0; u < VC_TOTALS_PER_LANE; u++) {
        if (wave * per_wave + u * VC_WAVE + lane >= pairs) continue;
        const int64_t len = (int64_t)e[u].sent * S.esz;
        const int cut = (int)((rbase[u] + (unsigned)e[u].rd * (unsigned)S.esz + (unsigned)S.recv_lo) & (VC_PIECE - 1));
        const int64_t cnt = vc_chunk_count(len, cut & (VC_LINE - 1), cut);
        payload += (int64_t)e[u].expected * S.esz;        // (what the receivers expect, as the planner counts it)
        items += cnt;
        moved += len * vc_block_hops(S, src[u], dst[u]);
        most = cnt > most ? cnt : most;
        longest = len > longest ? len : longest;
    }
    payload = vc_wave_inclusive_scan(payload);
    items = vc_wave_inclusive_scan(items);
    moved = vc_wave_inclusive_scan(moved);
    most = vc_wave_max_last(most);
    longest = vc_wave_max_last(longest);
    // six words in one store: each store past the caches is a write of its own to host memory (90 ranks of 4-byte blocks: one
    // store per word 21 us)
    const int64_t all[] = {vc_last_lane(payload), vc_last_lane(items), vc_last_lane(bad), vc_last_lane(most), vc_last_lane(moved), vc_last_lane(longest)};
    int64_t v = all[VC_TOTALS_PAYLOAD];
#pragma unroll
    for (int k = VC_TOTALS_PAYLOAD + 1; k <= VC_TOTALS_LONGEST; k++) v = lane == k ? all[k] : v;
    if (lane <= VC_TOTALS_LONGEST) vc_store_through(&totals[wave * VC_TOTALS_SLOT + lane], v);
}

// A copying wavefront of the single launch asks before its first store: have all totalling wavefronts checked their part of
// the tables, and did they find them in order?  The totalling workgroups are the first of the grid, so they are resident
// before any copying one; the wait is bounded all the same (VC_CHECK_SPINS polls, a few milliseconds): a wavefront that
// gives up moves nothing and says so in the first slot of the totals, and the host redoes the call the general way.
#define VC_CHECK_SPINS (1 << 15)
__device__ __forceinline__ unsigned long long vc_verdict_word(unsigned long long *verdict) {
    return __hip_atomic_load(verdict, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Asked by the piece movers between their loads and their stores (see vc_forward_piece).  Without `verdict` there is nothing
// to wait for (the planner's verdict was checked before the block's route was worked out).  look() reads the word once
// ahead of the block's loads, so that a verdict that is already in costs no round trip of its own.
struct VcVerdictGate {
    unsigned long long *verdict;
    int64_t *totals;
    unsigned long long nwaves, word;
    int state;                                            // 0 not known yet, 1 go, 2 leave everything where it is
    __device__ __forceinline__ void look() { if (verdict) word = vc_verdict_word(verdict); }
    __device__ __forceinline__ bool operator()() {
        if (!verdict) return true;
        for (int spin = 0; state == 0; spin++) {
            if ((word & 0xFFFFFFFFull) >= nwaves) state = (word >> 32) ? 2 : 1;
            else if (spin >= VC_CHECK_SPINS) { vc_store_through(&totals[VC_TOTALS_STALLED], (int64_t)1); state = 2; }
            else { __builtin_amdgcn_s_sleep(1); word = vc_verdict_word(verdict); }
        }
        return state == 1;
    }
};

// Workgroups at the head of the grid that only add up the totals (none without `verdict`): their round trips run beside the
// copying instead of in front of it.  A multiple of VC_XCDS, so that the workgroups behind them keep their XCDs.
__host__ __device__ __forceinline__ unsigned vc_totals_blocks(const VcSched &S, const void *verdict, int lanes) {
    if (!verdict) return 0;
    const int64_t waves = vc_totals_waves(S.P), per = lanes / VC_WAVE;
    return (unsigned)(((waves + per - 1) / per + VC_XCDS - 1) / VC_XCDS * VC_XCDS);
}

// Everything the addresses of a pair's block depend on, read at once.
struct VcPairRead { int sent, expected, sd, rd; int64_t sbase, rbase; };

__device__ __forceinline__ VcPairRead vc_pair_read(const VcSched &S, const VcTables &T, int s, int t) {
    VcPairRead p;
    p.sent = vc_sc(S, T, s, t); p.expected = vc_rc(S, T, t, s); p.sd = vc_sd(S, T, s, t); p.rd = vc_rd(S, T, t, s);
    p.sbase = T.sbase[s]; p.rbase = T.rbase[t];
    return p;
}

// Whether the pair's own table entries allow its block to be moved (the single launch has no planner that checked them):
// none negative, the receiver expecting what the source sends, the block no longer than a slot and cut into no more pieces
// than the kernel was chosen for.
__device__ __forceinline__ bool vc_pair_allowed(const VcSched &S, const VcPairRead &p, const VcListlessGuard &g) {
    const int64_t len = (int64_t)p.sent * S.esz;
    const int cut = (int)((p.rbase + (int64_t)p.rd * S.esz + S.recv_lo) & (VC_PIECE - 1));
    bool ok = (p.sent | p.sd | p.rd) >= 0 && p.expected == p.sent;
    ok = ok && !(S.packed_recv && (int64_t)p.rd + p.sent > 0x7FFFFFFF);
    ok = ok && !(g.max_len && len > g.max_len);
    return ok && !(g.max_pieces && vc_chunk_count(len, cut & (VC_LINE - 1), cut) > g.max_pieces);
}

// Forwarded execution without a work-item list, for calls whose planning would otherwise cost more than their copying:
// one workgroup (LANES = VC_THREADS) or one wavefront (VC_WAVE: blocks of a KiB or two) per (source, destination)
// pair, in the order of the chain items (by destination, then source, an eighth
// of the pairs per XCD).  Every wavefront works out the route of its block in closed form from the plan tables (lane k
// evaluates hop slot k) and carries the block through it piece by piece, taking one hop's destination after the other from
// its lane into scalar registers.  The kernel is enqueued right behind the
// planning kernel, before the host has seen its result, so it checks that result itself: nothing is touched when the
// plan needs more staging than there is, the tables hold negative entries, or the call is not of the kind the host
// expected when it chose this kernel (the host, which evaluates the same condition afterwards, then takes another path).
// Everything the block's addresses depend on is read before the planner's verdict is looked at: the reads are
// independent of each other and of the verdict (tables are always readable), so they travel together instead of one
// memory round trip after the other; nothing is stored before the verdict is known.
template <int LANES, bool SELF, bool WINDOW, bool CACHED>
__device__ __forceinline__ void vc_copy_pair(const VcSched &S, const VcTables &T, const uint32_t *__restrict__ slot_off,
                                             const int64_t *__restrict__ row_base,
                                             const int64_t *__restrict__ header, VcListlessGuard guard,
                                             int64_t first_pair, const char *__restrict__ sendbuf,
                                             char *__restrict__ recvbuf, char *__restrict__ stage,
                                             unsigned long long *verdict, unsigned long long *verdict_next,
                                             int64_t *totals) {
    const unsigned head = vc_totals_blocks(S, verdict, LANES);
    // Read from the launch where a workgroup has a pair and nothing is staged in a window: with a constant the compiler, short of scalar registers, there keeps 28 of the copying
    // workgroups' in lanes of a vector register and reads them back in 138 places (64 ranks of 0 - 1500 B 33.3 us a call / 32.4, 220 161.8 / 149.3, 700 1368 / 1234).  The other
    // instances take the constant, a read less in front of the verdict (wavefronts: 192 ranks of 2000 B 59.7 / 58.5, direct, 180 39.8 / 37.6; workgroups in a window, 8 registers in
    // lanes, 600 ranks of 3500 B at radix 599 965 / 947, but of 9000 B at 25 1999 / 2030).
    if (blockIdx.x < head) { vc_add_totals(S, T, verdict, totals, LANES == VC_WAVE || WINDOW ? LANES : (int)blockDim.x); return; }
    const unsigned block = blockIdx.x - head;
    const int64_t per = (gridDim.x - head) / VC_XCDS;
    const int64_t idx = first_pair + (int64_t)(block % VC_XCDS) * per + block / VC_XCDS;
    const bool inside = idx < (int64_t)S.P * S.P;
    const int t = inside ? vc_div((int)idx, S.dP) : 0, s = inside ? (int)idx - t * S.P : 0;       // (idx < P^2 <= 2^30)
    const VcPairRead p = vc_pair_read(S, T, s, t);
    const int lane = threadIdx.x % VC_WAVE, nslots = vc_hop_slots(S);
    const VcHop hop = vc_hop_place(S, s, t, lane < nslots ? lane : 0);
    const int64_t slot = vc_slot_addr(S, slot_off, row_base, hop);
    if (verdict && block == 0 && threadIdx.x < VC_VERDICTS) vc_store_through(&verdict_next[threadIdx.x * (VC_LINE / 8)], 0ull);      // the words of the next call
    const int64_t len = (int64_t)p.sent * S.esz;
    if (!inside || len <= 0) return;
    if (verdict ? !vc_pair_allowed(S, p, guard) : !vc_listless_ok(header, guard)) return;
    const int64_t recv_off = p.rbase + (int64_t)p.rd * S.esz;
    const int64_t dst = vc_hop_dst(S, hop, slot, recv_off);
    const unsigned long long moves = __ballot(lane < nslots && hop.moves);
    const char *src = sendbuf + p.sbase + (int64_t)p.sd * S.esz;
    const int cut = (int)((recv_off + S.recv_lo) & (VC_PIECE - 1)), phase = cut & (VC_LINE - 1);
    const int64_t pieces = vc_chunk_count(len, phase, cut);
    VcVerdictGate gate = {verdict ? verdict + block % VC_VERDICTS * (VC_LINE / 8) : nullptr, totals, (unsigned long long)vc_totals_waves(S.P), 0, 0};
    gate.look();
    for (int64_t c = 0; c < pieces; c++) {                // the same cuts as the chain items of this block
        int64_t lo, hi;
        vc_piece_range(len, phase, cut, c, lo, hi);
        unsigned long long left = moves;
        vc_forward_piece<LANES, SELF, WINDOW, CACHED>(src + lo, hi - lo, __popcll(moves), c ? 0 : phase,
                                [&]() {
                                    const int k = __ffsll(left) - 1;
                                    left &= left - 1;
                                    const unsigned d_lo = __builtin_amdgcn_readlane((int)dst, k), d_hi = __builtin_amdgcn_readlane((int)(dst >> 32), k);
                                    return vc_resolve(((int64_t)d_hi << 32 | d_lo) + lo, sendbuf, recvbuf, stage, WINDOW ? vc_window_mask(S.window) : -1);
                                },
                                [&]() { return gate(); });
    }
}

// SELF: one launch on fixed-stride staging that tells the host itself that it is done (vc_signal), with everything it stores stored past
// the caches.  A kernel behind this one that only does that costs the boundary between the two: 8 ranks of 0 - 64 ints 13.0 -> 12.8 us,
// 32 ranks of 0 - 2 KiB 14.0 -> 13.5, 24 ranks of 0 - 32 KiB 26.6 -> 22.3.  The quarter kernel has no such instance: its lanes' short stores past the caches each
// cost a write to memory (64 ranks, 1 KiB blocks: 16.6 -> 21.9 us).
// WINDOW: S.window.
template <int LANES, bool SELF, bool WINDOW, bool CACHED>
__global__ __launch_bounds__(LANES) void vc_copy_blocks_kernel(VcSched S, VcTables T, const uint32_t *__restrict__ slot_off,
                                                               const int64_t *__restrict__ row_base,
                                                               const int64_t *__restrict__ header, VcListlessGuard guard,
                                                               int64_t first_pair, const char *__restrict__ sendbuf,
                                                               char *__restrict__ recvbuf, char *__restrict__ stage,
                                                               unsigned long long *verdict, unsigned long long *verdict_next,
                                                               int64_t *totals, VcSignal sig) {
    vc_copy_pair<LANES, SELF, WINDOW, CACHED>(S, T, slot_off, row_base, header, guard, first_pair, sendbuf, recvbuf, stage, verdict, verdict_next, totals);
    if (SELF) vc_signal(sig);
}

// The same for pairs whose blocks are a few hundred bytes: a quarter of a wavefront per pair, four pairs in a row per
// wavefront.  Lane q of a group evaluates hop slots q and q + 16; the four routes of the wavefront go through LDS.
// Eight vectors of a lane in flight, 2 KiB a group: 85 VGPRs, 5 wavefronts per SIMD.  With four (62 VGPRs, 7) the loads of a second round
// wait for the stores of the first: calls of blocks of 512 B - 2.5 KiB on average on 64 - 200 ranks 3 - 5 % slower (128 ranks, 2 KiB 33.0
// us -> 34.2; 192 ranks, 600 B 38.3 -> 40.4), 1024 ranks, 700 B 596 -> 605, and only direct calls on 300 ranks faster (91.9 -> 89.9).
template <bool WINDOW, bool CACHED>
__global__ __launch_bounds__(VC_WAVE) void vc_copy_blocks_quarter_kernel(VcSched S, VcTables T, const uint32_t *__restrict__ slot_off,
                                                                         const int64_t *__restrict__ row_base,
                                                                         const int64_t *__restrict__ header, VcListlessGuard guard,
                                                                         int64_t first_pair, const char *__restrict__ sendbuf,
                                                                         char *__restrict__ recvbuf, char *__restrict__ stage,
                                                                         unsigned long long *verdict, unsigned long long *verdict_next,
                                                                         int64_t *totals) {
    __shared__ char *route[VC_ITEMS_PER_WAVE][VC_MAX_HOP_SLOTS];
    const unsigned head = vc_totals_blocks(S, verdict, VC_WAVE);
    if (blockIdx.x < head) { vc_add_totals(S, T, verdict, totals, VC_WAVE); return; }
    const unsigned block = blockIdx.x - head;
    const int64_t per = (gridDim.x - head) / VC_XCDS;
    const int64_t wave = (int64_t)(block % VC_XCDS) * per + block / VC_XCDS;
    const int g = threadIdx.x / VC_QUARTER, q = threadIdx.x % VC_QUARTER;
    const int64_t idx = first_pair + wave * VC_ITEMS_PER_WAVE + g;
    const bool inside = idx < (int64_t)S.P * S.P;
    const int t = inside ? vc_div((int)idx, S.dP) : 0, s = inside ? (int)idx - t * S.P : 0;       // (idx < P^2 <= 2^30)
    // all reads the addresses depend on go out before the planner's verdict is looked at (see vc_copy_blocks_kernel)
    const VcPairRead p = vc_pair_read(S, T, s, t);
    const int nslots = vc_hop_slots(S);
    const VcHop h0 = vc_hop_place(S, s, t, q < nslots ? q : 0);
    const int64_t slot0 = vc_slot_addr(S, slot_off, row_base, h0);
    if (verdict && block == 0 && threadIdx.x < VC_VERDICTS) vc_store_through(&verdict_next[threadIdx.x * (VC_LINE / 8)], 0ull);
    if (!verdict && !vc_listless_ok(header, guard)) return;      // the same for every lane of the grid
    const int64_t len = inside ? (int64_t)p.sent * S.esz : 0, recv_off = p.rbase + (int64_t)p.rd * S.esz;
    // no lane leaves before the barrier below
    const bool active = len > 0 && (!verdict || vc_pair_allowed(S, p, guard));
    const bool m0 = active && q < nslots && h0.moves;
    const unsigned g0 = (unsigned)(__ballot(m0) >> (g * VC_QUARTER)) & 0xFFFFu;      // the group's hops among slots 0..15
    if (m0) route[g][__popc(g0 & ((1u << q) - 1))] = vc_hop_at<WINDOW>(S, h0, slot0, recv_off, recvbuf, stage);
    int nhop = __popc(g0);
    if (nslots > VC_QUARTER) {                            // ... among slots 16..31
        const int k1 = q + VC_QUARTER;
        const VcHop h1 = vc_hop_place(S, s, t, k1 < nslots ? k1 : 0);
        const bool m1 = active && k1 < nslots && h1.moves;
        const unsigned g1 = (unsigned)(__ballot(m1) >> (g * VC_QUARTER)) & 0xFFFFu;
        if (m1) route[g][nhop + __popc(g1 & ((1u << q) - 1))] = vc_hop_at<WINDOW>(S, h1, h1.staged ? vc_slot_addr(S, slot_off, row_base, h1) : 0, recv_off, recvbuf, stage);
        nhop += __popc(g1);
    }
    __syncthreads();
    if (!active || nhop <= 0) return;
    const char *src = sendbuf + p.sbase + (int64_t)p.sd * S.esz;
    const int cut = (int)((recv_off + S.recv_lo) & (VC_PIECE - 1));
    VcVerdictGate gate = {verdict ? verdict + block % VC_VERDICTS * (VC_LINE / 8) : nullptr, totals, (unsigned long long)vc_totals_waves(S.P), 0, 0};
    gate.look();
    vc_forward_block<VC_QUARTER, 8, WINDOW, CACHED>(S, src, len, nhop, cut, route[g], stage, [&]() { return gate(); });
}

// ---- blocks of up to 64 bytes, by runs ----
// The 64 pairs of a wavefront are a tile of 8 sources x 8 receivers.  In a packed layout what a source sends to the 8 receivers is one run, and what a receiver
// gets from the 8 sources another one: a run is read, and written, as vectors by 8 lanes, and the blocks change hands in LDS.  A block of a lane takes up to five
// loads and stores of different widths, each to 64 places (the address units were busy most of the time); a run of blocks of 16 bytes one of each, and two for the ends of
// what is written.  For which calls, and what they gain: vc_run_vectors.  NV: vectors a block may take.
#define VC_RUN_ROW(nv) (32 + 144 * (nv))                  // bytes of a run in LDS: 16 in front of it, up to 15 + 128 nv; a block's read may start at its end
#define VC_RUN_BYTES(nv) (8 * VC_RUN_ROW(nv))

__device__ __forceinline__ int64_t vc_from_lane(int64_t v, int lane) {
    const int lo = __builtin_amdgcn_ds_bpermute(lane << 2, (int)v), hi = __builtin_amdgcn_ds_bpermute(lane << 2, (int)(v >> 32));
    return (int64_t)hi << 32 | (unsigned)lo;
}

// 16 bytes from any place in LDS.
__device__ __forceinline__ vc_u32x4 vc_lds_read16(const char *lds, int at) {
    const unsigned *const w = reinterpret_cast<const unsigned *>(lds + (at & ~3));
    const unsigned a = w[0], b = w[1], c = w[2], d = w[3], e = w[4];
    return vc_u32x4{__builtin_amdgcn_alignbyte(b, a, at & 3), __builtin_amdgcn_alignbyte(c, b, at & 3), __builtin_amdgcn_alignbyte(d, c, at & 3), __builtin_amdgcn_alignbyte(e, d, at & 3)};
}

// v, `bytes` (0 .. 15) bytes further down.
__device__ __forceinline__ vc_u32x4 vc_bytes_down(vc_u32x4 v, int bytes) {
    if (bytes & 4) { v.x = v.y; v.y = v.z; v.z = v.w; }
    if (bytes & 8) { v.x = v.z; v.y = v.w; }
    v.x = __builtin_amdgcn_alignbyte(v.y, v.x, bytes & 3);
    v.y = __builtin_amdgcn_alignbyte(v.z, v.y, bytes & 3);
    v.z = __builtin_amdgcn_alignbyte(v.w, v.z, bytes & 3);
    v.w = v.w >> 8 * (bytes & 3);
    return v;
}

__device__ __forceinline__ unsigned vc_first_bytes(unsigned v, int n) { return n >= 4 ? v : (n <= 0 ? 0 : v & ((1u << 8 * n) - 1)); }

__device__ __forceinline__ void vc_lds_settled() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// False (and nothing done): the blocks of the tile lie otherwise, or a run is shorter than a vector.  len: 0 .. 16 NV; all pairs exist.  route: the lane's
// hops, the last one into recvbuf, the others to the start of a slot.
template <int NV, bool WINDOW> __device__ __forceinline__ bool vc_copy_runs(const char *sendbuf, char *recvbuf, int64_t send_off, int64_t recv_off, int len, int nhop, char *const *route, char *lds) {
    int lane = threadIdx.x;
    asm("" : "+v"(lane));
    const int si = lane & 7, ti = lane >> 3;
    const int64_t before_s = vc_from_lane(send_off + len, lane - 8 & 63), before_t = vc_from_lane(recv_off + len, lane - 1 & 63);
    const int64_t run_t = vc_from_lane(recv_off, lane & ~7);
    const int pos_s = (int)send_off - __builtin_amdgcn_ds_bpermute(si << 2, (int)send_off);
    const int bytes_s = __builtin_amdgcn_ds_bpermute((56 + si) << 2, pos_s + len);
    const int pos_t = (int)(recv_off - run_t), bytes_t = __builtin_amdgcn_ds_bpermute((lane | 7) << 2, pos_t + len);
    const bool fits = (ti == 0 || before_s == send_off) && (si == 0 || before_t == recv_off) && (bytes_s == 0 || bytes_s >= 16) && (bytes_t == 0 || bytes_t >= 16);
    if (__ballot(!fits)) return false;
    constexpr int ROW = VC_RUN_ROW(NV);
    // the runs of the sources: lane l has vectors l % 8 and, of blocks of two vectors, l % 8 + 8 of source l / 8's
    const int64_t run_s = vc_from_lane(send_off, lane >> 3);
    const int run_bytes = __builtin_amdgcn_ds_bpermute(lane >> 3 << 2, bytes_s);
    vc_u32x4 in[NV];
#pragma unroll
    for (int q = 0; q < NV; q++) {
        const int at = ((lane & 7) << 4) + 128 * q, from = at < run_bytes - 16 ? at : run_bytes - 16;
        in[q] = vc_u32x4{0, 0, 0, 0};
        if (at < run_bytes) in[q] = vc_load16<true>(sendbuf + run_s + from);
    }
#pragma unroll
    for (int q = 0; q < NV; q++) {
        const int at = ((lane & 7) << 4) + 128 * q, over = at - (run_bytes - 16);
        *reinterpret_cast<vc_u32x4 *>(lds + (lane >> 3) * ROW + at) = over > 0 && over < 16 ? vc_bytes_down(in[q], over) : in[q];
    }
    vc_lds_settled();
    vc_u32x4 v[NV];                                       // the pair's block, and what lies behind it
#pragma unroll
    for (int q = 0; q < NV; q++) v[q] = vc_lds_read16(lds, si * ROW + pos_s + 16 * q);
    vc_lds_settled();
    for (int k = lane; k < VC_RUN_BYTES(NV) / 16; k += VC_WAVE) reinterpret_cast<vc_u32x4 *>(lds)[k] = vc_u32x4{0, 0, 0, 0};
    if (WINDOW && len > 0)
        for (int k = 0; k < nhop - 1; k++) {
            *reinterpret_cast<vc_u32x4 *>(route[k]) = v[0];
#pragma unroll
            for (int q = 1; q < NV; q++) if (len > 16 * q) *reinterpret_cast<vc_u32x4 *>(route[k] + 16 * q) = v[q];
        }
    vc_lds_settled();
    // the runs of the receivers, counted from the 16 bytes at or below the run's place: every block ORed into its own bytes
    const int phase = (int)((uintptr_t)(recvbuf + run_t) & 15), to = ti * ROW + 16 + phase + pos_t, up = (to + 3 & 3) + 1;
    unsigned *word = reinterpret_cast<unsigned *>(lds + (to - up));
    if (len > 0) {
        unsigned before = 0;
#pragma unroll
        for (int q = 0; q < NV; q++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const unsigned now = vc_first_bytes(v[q][c], len - 16 * q - 4 * c);
                atomicOr(word++, __builtin_amdgcn_alignbyte(now, before, 4 - up));
                before = now;
            }
        atomicOr(word, __builtin_amdgcn_alignbyte(0u, before, 4 - up));
    }
    vc_lds_settled();
    const char *const row = lds + ti * ROW + 16;
    char *const dst = recvbuf + run_t;
#pragma unroll
    for (int q = 0; q < NV; q++) {
        const int j = (si << 4) + 128 * q;                // the lane's vector, full or not
        if (j >= phase && j + 16 <= phase + bytes_t) *reinterpret_cast<vc_u32x4 *>(dst - phase + j) = *reinterpret_cast<const vc_u32x4 *>(row + j);
    }
    // the run's first and last 16 bytes where a vector is not full
    const int edge = si == 0 ? 0 : bytes_t - 16;
    if (bytes_t > 0 && (si == 0 ? phase != 0 : si == 1 && (phase + bytes_t & 15) != 0))
        reinterpret_cast<VcU128 *>(dst + edge)->v = vc_lds_read16(row, phase + edge);
    return true;
}

// The same again for calls of many short blocks, where the wavefronts above live for one pass over four blocks and the
// round trips and the arithmetic of working out a route, not the bytes, set the pace: a wavefront takes BATCH pairs, a tile of
// TS sources x TR receivers, so that its table entries, the blocks it reads (of one source, for neighbouring receivers) and
// the blocks it writes (of one receiver, from neighbouring sources) share cache lines.
// 64 / BATCH lanes per pair evaluate its hop slots and leave the route in LDS.  Blocks of no more than VC_LANE_BLOCK bytes are then moved by
// a lane each, when all blocks of the wavefront are that short; else every quarter of the wavefront carries BATCH / 4 of them, one
// after the other.  Measured on MI355X, 1024 ranks, two hops for most blocks: 0 - 16 bytes 76 us (pairs of one receiver
// in a row, every block a quarter of a wavefront) -> 28, as runs 15; 0 - 64 bytes, calls 144 -> 82 (blocks of up to 32 bytes a lane before), as runs 57.
// RUN: the vectors a block may take in a run (vc_run_vectors).  Instances, because every launch fetches its code anew and the longer runs take more registers: with runs of one and
// of four vectors in one kernel 1024 ranks of 0 - 16 B take 34.4 us a call instead of 32.1.
// In a window short blocks of a batch start where their slots start, and their vectors are counted from the block itself instead of from its line in recvbuf: fewer lines a
// staged hop, fewer passes over a block, and nothing lost in recvbuf, where the vectors at the edges make the address units take every store of short blocks apart
// anyway.  From VC_BATCH_START_BELOW bytes on the unaligned lines of recvbuf cost more.  Calls, before / after: 1024 ranks of 0 - 256 B 138.5 us / 130, of 0 - 512 B packed, async
// 201.8 / 195, of 0 - 400 B at radix 2 235 / 213; 512 of 0 - 400 B at radix 3 84 / 76.6; 1024 of about 600 B 347 / 347 (without the line 348.7).
// Two blocks of a quarter in flight at once make it slower (0 - 512 bytes, calls of 16 pairs a wavefront 202 us -> 240): the requests of a wavefront
// queue up in the memory.
#define VC_BATCH_START_BELOW 512
// Wavefronts of 64 pairs with a block of more than VC_LANE_GROUPS_ABOVE bytes, in a window, carry a block with four neighbouring lanes instead of one, 16 blocks at a time: an
// instruction goes to fewer lines, and there is one of them for every 64 bytes of a block instead of one for every width.  Calls, a lane / four: 1024 ranks of 0 - 128 B
// 109 us / 95.7, 0 - 90 B 89.6 / 82.6, 0 - 64 B 72.3 / 71.0; 512 of 0 - 120 B 55.0 / 47.1, 0 - 80 B 46.1 / 46.7, 0 - 60 B 41.0 / 43.3, at radix 511 0 - 120 B 30.9 / 28.5.  Too few wavefronts
// from 512 ranks down (256 of 0 - 120 B 28.3 / 29.7), and no gain with one hop a block (1000 ranks direct, 0 - 100 B 65.3 / 76.5).
#define VC_LANE_GROUP 4
#define VC_LANE_GROUPS_PAIRS (1 << 18)
#define VC_LANE_GROUPS_ABOVE 80
template <int BATCH, int RUN, bool WINDOW, bool CACHED>
__global__ __launch_bounds__(VC_WAVE) void vc_copy_blocks_batch_kernel(VcSched S, VcTables T, const uint32_t *__restrict__ slot_off,
                                                                       const int64_t *__restrict__ row_base,
                                                                       const int64_t *__restrict__ header, VcListlessGuard guard,
                                                                       int64_t first_wave, const char *__restrict__ sendbuf,
                                                                       char *__restrict__ recvbuf, char *__restrict__ stage) {
    constexpr int TS = BATCH == 16 ? 4 : 8, TR = BATCH / TS, SHARE = VC_WAVE / BATCH, AHEAD = WINDOW ? 1 : 4;
    extern __shared__ char *batch_lds[];
    const int nslots = vc_hop_slots(S), P = S.P;
    char **route = batch_lds;                             // [BATCH][nslots]
    int64_t *b_len = reinterpret_cast<int64_t *>(route + BATCH * nslots), *b_src = b_len + BATCH;
    int *b_nhop = reinterpret_cast<int *>(b_src + BATCH), *b_cut = b_nhop + BATCH;
    const unsigned per = gridDim.x / VC_XCDS, tiles_s = (unsigned)(P + TS - 1) / TS;
    const unsigned wave = (unsigned)first_wave + (blockIdx.x % VC_XCDS) * per + blockIdx.x / VC_XCDS;
    const unsigned tile_t = wave / tiles_s, tile_s = wave - tile_t * tiles_s;
    const int p = threadIdx.x % BATCH, kq = threadIdx.x / BATCH;
    const int s_at = (int)tile_s * TS + p % TS, t_at = (int)tile_t * TR + p / TS;
    const bool inside = s_at < P && t_at < P;
    const int s = inside ? s_at : 0, t = inside ? t_at : 0;
    // all reads the addresses depend on go out before the planner's verdict is looked at (see vc_copy_blocks_kernel)
    const int sent = vc_sc(S, T, s, t);
    const int64_t send_off = vc_send_offset(S, T, s, t), recv_off = vc_recv_offset(S, T, s, t);
    const bool ok = vc_listless_ok(header, guard);
    const int64_t len = inside ? (int64_t)sent * S.esz : 0;
    const bool starts = WINDOW && (SHARE == 1 || len < VC_BATCH_START_BELOW);
    int nhop = 0;
    if (SHARE == 1) {
        VcWalk walk = vc_walk_start(S, s, t);
        // Reads of the slot tables travel together, four slots at a time.  In a window there are none, and one slot after the other is 2.9 KB less code, which
        // every launch fetches anew; nor is the last slot, recvbuf, looked at, the only one of a direct call.  Calls, before / after: 1024 ranks of 0 - 2 B
        // 31.8 us / 30.2, of 0 - 16 B 37.0 / 36.5; 700 of 0 - 16 B at radix 3 39.5 / 37.2; 300 of 0 - 8 B at radix 2 24.3 / 23.2; 1000 of 0 - 3 B, direct, 27.7 / 25.2.
        for (int k0 = 0; k0 < nslots - 1; k0 += AHEAD) {
            VcHop hop[AHEAD];
            int64_t at_row[AHEAD];
            uint32_t at[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; u++) {
                hop[u].moves = 0; at_row[u] = 0; at[u] = 0;
                if (k0 + u >= nslots - 1) continue;
                hop[u] = vc_walk_step(S, walk, s, t, k0 + u);
                if (S.stride) { at_row[u] = vc_slot_addr(S, slot_off, row_base, hop[u]); continue; }
                at_row[u] = row_base[hop[u].row];
                at[u] = slot_off[(int64_t)hop[u].row * P + hop[u].id];
            }
#pragma unroll
            for (int u = 0; u < AHEAD; u++)
                if (hop[u].moves && hop[u].staged) route[p * nslots + nhop++] = vc_hop_at<WINDOW>(S, hop[u], at_row[u] + vc_slot_bytes(at[u]), recv_off, recvbuf, stage, starts);
        }
        route[p * nslots + nhop++] = recvbuf + recv_off;      // the one hop of every block that is not staged, whenever it is made
    } else {
        for (int k = kq; k < nslots; k += SHARE) {
            const VcHop hop = vc_hop_place(S, s, t, k);
            char *const d = vc_hop_at<WINDOW>(S, hop, vc_slot_addr(S, slot_off, row_base, hop), recv_off, recvbuf, stage, starts);
            route[p * nslots + k] = hop.moves ? d : nullptr;
        }
        __syncthreads();
        for (int k = 0; k < nslots; k++) {                // (every lane of the pair on its own copy of the count; one writes)
            char *const d = route[p * nslots + k];
            if (d) { if (kq == 0) route[p * nslots + nhop] = d; nhop++; }
        }
    }
    if (!ok) return;                                      // the same for every lane of the grid
    const bool active = len > 0 && nhop > 0;
    const bool grouped = WINDOW && BATCH == VC_WAVE && P * P >= VC_LANE_GROUPS_PAIRS;
    if (__ballot(active && len > (grouped ? VC_LANE_GROUPS_ABOVE : VC_LANE_BLOCK)) == 0) {
        __syncthreads();
        if constexpr (RUN > 0)
            if (__ballot(!inside || (active && (len > 16 * RUN || (!WINDOW && nhop > 1)))) == 0 && __ballot(active && len > VC_RUN_ABOVE) != 0 &&
                vc_copy_runs<RUN, WINDOW>(sendbuf, recvbuf, send_off, recv_off, active ? (int)len : 0, nhop, route + p * nslots, reinterpret_cast<char *>(b_len)))
                return;
        if (active && kq == 0) {
            const VcLaneBlock b = vc_lane_load(sendbuf + send_off, (int)len);
            int k = 0;                                    // (the last one of the route is recvbuf)
            if (WINDOW && SHARE == 1 && nhop > 1 && len <= 16) {
                const vc_u32x4 v = vc_lane_vector(b, (int)len);
                for (; k < nhop - 1; k++) *reinterpret_cast<vc_u32x4 *>(route[p * nslots + k]) = v;
            }
            for (; k < nhop; k++) vc_lane_store(b, route[p * nslots + k], (int)len);
        }
        return;
    }
    if (kq == 0) {
        b_len[p] = active ? len : 0;
        b_src[p] = send_off;
        b_nhop[p] = nhop;
        b_cut[p] = (int)((recv_off + S.recv_lo) & (starts ? VC_PIECE - VC_LINE : VC_PIECE - 1));      // (vectors counted from the block itself, or from its line)
    }
    __syncthreads();
    if (grouped && __ballot(active && len > 2 * VC_LANE_BLOCK) == 0) {
        for (int b = threadIdx.x / VC_LANE_GROUP; b < BATCH; b += VC_WAVE / VC_LANE_GROUP) {
            const int64_t blen = b_len[b];
            if (blen <= 0) continue;
            vc_forward_block<VC_LANE_GROUP, 2, WINDOW, CACHED>(S, sendbuf + b_src[b], blen, b_nhop[b], b_cut[b], route + b * nslots, stage);
        }
        return;
    }
    for (int it = 0; it < BATCH / VC_ITEMS_PER_WAVE; it++) {
        const int b = it * VC_ITEMS_PER_WAVE + threadIdx.x / VC_QUARTER;
        const int64_t blen = b_len[b];
        if (blen <= 0) continue;
        vc_forward_block<VC_QUARTER, 4, WINDOW, CACHED>(S, sendbuf + b_src[b], blen, b_nhop[b], b_cut[b], route + b * nslots, stage);
    }
}

// The instance of a kernel for calls with or without a window, with ordinary or non-temporal loads: `of` names it.
template <class Of> static auto vc_instance(bool window, bool cached, Of of) {
    const std::true_type yes;
    const std::false_type no;
    return window ? (cached ? of(yes, yes) : of(yes, no)) : (cached ? of(no, yes) : of(no, no));
}

template <int BATCH, int RUN>
static void vc_launch_batch(const VcSched &S, VcTables T, const uint32_t *slot_off, const int64_t *row_base, const int64_t *header,
                            VcListlessGuard guard, const char *sendbuf, char *recvbuf, char *stage, hipStream_t st, bool cached) {
    const int64_t ts = BATCH == 16 ? 4 : 8, waves = ((S.P + ts - 1) / ts) * ((S.P + BATCH / ts - 1) / (BATCH / ts));
    // (behind the routes the blocks' words, or the runs)
    const size_t words = (sizeof(int64_t) * 2 + sizeof(int) * 2) * BATCH, runs = RUN ? VC_RUN_BYTES(RUN) : 0;
    const size_t lds = sizeof(int64_t) * BATCH * vc_hop_slots(S) + (runs > words ? runs : words);
    for (int64_t done = 0; done < waves; done += VC_MAX_GRID) {
        const int64_t now = waves - done < VC_MAX_GRID ? waves - done : VC_MAX_GRID;
        const auto kernel = vc_instance(S.window, cached, [](auto w, auto k) { return vc_copy_blocks_batch_kernel<BATCH, RUN, w(), k()>; });
        hipLaunchKernelGGL(kernel, dim3((unsigned)((now + VC_XCDS - 1) / VC_XCDS * VC_XCDS)), dim3(VC_WAVE), lds, st, S,
                           T, slot_off, row_base, header, guard, done, sendbuf, recvbuf, stage);
    }
}

hipError_t vc_launch_copy_blocks(const VcSched &S, VcTables T, const uint32_t *slot_off, const int64_t *row_base, const int64_t *header,
                                 VcListlessGuard guard, int lanes, const char *sendbuf, char *recvbuf, char *stage, hipStream_t st,
                                 unsigned long long *verdict, unsigned long long *verdict_next, int64_t *totals, VcSignal sig, int batch, bool cached, int run) {
    const int64_t npairs = (int64_t)S.P * S.P;
    if (sig.word && (!verdict || !vc_may_signal(lanes, S.window))) return hipErrorInvalidValue;
    if (lanes == VC_BATCHED) {
        if (verdict) return hipErrorInvalidValue;         // the batches are for more pairs than one launch with totals takes
        (batch != 64 ? vc_launch_batch<16, 0> : run == 0 ? vc_launch_batch<64, 0> : run == 1 ? vc_launch_batch<64, 1> : run == 2 ? vc_launch_batch<64, 2> : vc_launch_batch<64, 4>)(
            S, T, slot_off, row_base, header, guard, sendbuf, recvbuf, stage, st, cached);
        return hipGetLastError();
    }
    const int64_t step = lanes == VC_QUARTER ? VC_MAX_GRID * VC_ITEMS_PER_WAVE : VC_MAX_GRID;
    for (int64_t done = 0; done < npairs; done += step) {
        const int64_t now = npairs - done < step ? npairs - done : step;
        const int64_t units = lanes == VC_QUARTER ? (now + VC_ITEMS_PER_WAVE - 1) / VC_ITEMS_PER_WAVE : now;
        if (verdict && done) return hipErrorInvalidValue;    // the totals belong to a call that one launch takes
        const dim3 grid((unsigned)((units + VC_XCDS - 1) / VC_XCDS * VC_XCDS) + vc_totals_blocks(S, verdict, lanes == VC_THREADS ? VC_THREADS : VC_WAVE));
        if (lanes == VC_QUARTER) {
            const auto kernel = vc_instance(S.window, cached, [](auto w, auto k) { return vc_copy_blocks_quarter_kernel<w(), k()>; });
            hipLaunchKernelGGL(kernel, grid, dim3(VC_WAVE), 0, st, S, T, slot_off, row_base, header, guard, done, sendbuf, recvbuf, stage, verdict,
                               verdict_next, totals);
            continue;
        }
        const bool self = sig.word != nullptr;
        const auto wave = self ? vc_copy_blocks_kernel<VC_WAVE, true, false, false> : vc_instance(S.window, cached, [](auto w, auto k) { return vc_copy_blocks_kernel<VC_WAVE, false, w(), k()>; });
        const auto workgroup = self ? vc_copy_blocks_kernel<VC_THREADS, true, false, false> : vc_instance(S.window, cached, [](auto w, auto k) { return vc_copy_blocks_kernel<VC_THREADS, false, w(), k()>; });
        const auto kernel = lanes == VC_WAVE ? wave : workgroup;
        hipLaunchKernelGGL(kernel, grid, dim3(lanes), 0, st, S, T, slot_off, row_base, header, guard, done, sendbuf, recvbuf, stage, verdict,
                           verdict_next, totals, sig);
    }
    return hipGetLastError();
}

// Items of one launch: as many as VC_MAX_GRID workgroups or wavefronts take.
static int64_t vc_items_per_launch(int lanes) { return lanes == VC_QUARTER ? VC_MAX_GRID * VC_ITEMS_PER_WAVE : VC_MAX_GRID; }

static unsigned vc_grid_for(int64_t items, int lanes) {
    const int64_t per = lanes == VC_QUARTER ? VC_ITEMS_PER_WAVE * vc_quarter_rounds(items) : 1;
    const int64_t units = (items + per - 1) / per;
    return (unsigned)((units + VC_XCDS - 1) / VC_XCDS * VC_XCDS);
}

// One launch of the list-driven kernel with LANES lanes per item, in the instance for calls with or without a window.
template <bool GUARDED>
static void vc_launch_chains_once(const int64_t *items, int stride, unsigned nitems, int lanes, const char *sendbuf, char *recvbuf, char *stage,
                                  hipStream_t st, const int64_t *header, VcChainGuard guard, int window, bool cached) {
    const dim3 grid(vc_grid_for(nitems, lanes));
    if (lanes == VC_QUARTER) {
        const auto kernel = vc_instance(window, cached, [](auto w, auto k) { return vc_copy_chains_quarter_kernel<GUARDED, w(), k()>; });
        hipLaunchKernelGGL(kernel, grid, dim3(VC_WAVE), 0, st, items, stride, nitems, vc_quarter_rounds(nitems), sendbuf, recvbuf, stage, header,
                           guard, window);
        return;
    }
    const auto wave = vc_instance(window, cached, [](auto w, auto k) { return vc_copy_chains_kernel<VC_WAVE, GUARDED, w(), k()>; });
    const auto workgroup = vc_instance(window, cached, [](auto w, auto k) { return vc_copy_chains_kernel<VC_THREADS, GUARDED, w(), k()>; });
    hipLaunchKernelGGL(lanes == VC_WAVE ? wave : workgroup, grid, dim3(lanes == VC_WAVE ? VC_WAVE : VC_THREADS), 0, st, items, stride, nitems, sendbuf,
                       recvbuf, stage, header, guard, window);
}

hipError_t vc_launch_copy_chains(const int64_t *items, int stride, int64_t nitems, int lanes, const char *sendbuf, char *recvbuf,
                                 char *stage, hipStream_t st, int window, bool cached) {
    const int64_t step = vc_items_per_launch(lanes);
    for (int64_t done = 0; done < nitems; done += step) {
        const int64_t now = nitems - done < step ? nitems - done : step;
        vc_launch_chains_once<false>(items + done * stride, stride, (unsigned)now, lanes, sendbuf, recvbuf, stage, st, nullptr, VcChainGuard(), window, cached);
    }
    return hipGetLastError();
}

// One launch (a guessed list longer than a launch holds is cut to what one holds; the rest is the caller's second launch).
hipError_t vc_launch_copy_chains_guarded(const int64_t *items, int stride, int64_t grid_items, int lanes, const char *sendbuf,
                                         char *recvbuf, char *stage, hipStream_t st, const int64_t *header, VcChainGuard guard, int64_t *covered,
                                         int window, bool cached) {
    const int64_t step = vc_items_per_launch(lanes);
    const int64_t now = grid_items < step ? grid_items : step;
    *covered = now > 0 ? now : 0;
    if (now <= 0) return hipSuccess;
    vc_launch_chains_once<true>(items, stride, (unsigned)now, lanes, sendbuf, recvbuf, stage, st, header, guard, window, cached);
    return hipGetLastError();
}

hipError_t vc_launch_copy_items(const VcDesc *items, int64_t nitems, int lanes, const char *sendbuf, char *recvbuf, char *stage,
                                hipStream_t st) {
    const int64_t step = vc_items_per_launch(lanes);
    for (int64_t done = 0; done < nitems; done += step) {
        const int64_t now = nitems - done < step ? nitems - done : step;
        const dim3 grid(vc_grid_for(now, lanes));
        if (lanes == VC_QUARTER)
            hipLaunchKernelGGL(vc_copy_items_quarter_kernel, grid, dim3(VC_WAVE), 0, st, items + done, (unsigned)now, vc_quarter_rounds(now),
                               sendbuf, recvbuf, stage);
        else if (lanes == VC_WAVE)
            hipLaunchKernelGGL(vc_copy_items_kernel<VC_WAVE>, grid, dim3(VC_WAVE), 0, st, items + done, (unsigned)now, sendbuf, recvbuf, stage);
        else
            hipLaunchKernelGGL(vc_copy_items_kernel<VC_THREADS>, grid, dim3(VC_THREADS), 0, st, items + done, (unsigned)now, sendbuf, recvbuf,
                               stage);
    }
    return hipGetLastError();
}

// Plain contiguous copy of a known size: one 16-byte vector per lane, 4 KiB per workgroup, WRITES stores per load.  It exists so
// that hardware counters (bytes fetched / written per dispatch) can be scaled against a transfer whose size is known, and as
// the ceiling the block movers are held against: WRITES = 1 for launch-per-digit execution (one read, one write per hop),
// WRITES = 2 for the forwarded kernel on two-hop routes (one read, two writes).
template <int WRITES>
__global__ __launch_bounds__(VC_THREADS) void vc_calibration_copy_kernel(const vc_u32x4 *__restrict__ src, vc_u32x4 *__restrict__ dst,
                                                                         vc_u32x4 *__restrict__ dst2, int64_t nvec) {
    const int64_t i = (int64_t)blockIdx.x * VC_THREADS + threadIdx.x;
    if (i >= nvec) return;
    const vc_u32x4 v = __builtin_nontemporal_load(&src[i]);
    __builtin_nontemporal_store(v, &dst[i]);
    if (WRITES == 2) __builtin_nontemporal_store(v, &dst2[i]);
}

hipError_t vc_launch_calibration_copy(const char *src, char *dst, char *dst2, int64_t nbytes, hipStream_t st) {
    const int64_t nvec = nbytes / 16;
    for (int64_t done = 0; done < nvec; done += VC_MAX_GRID * VC_THREADS) {
        const int64_t now = nvec - done < VC_MAX_GRID * VC_THREADS ? nvec - done : VC_MAX_GRID * VC_THREADS;
        const dim3 grid((unsigned)((now + VC_THREADS - 1) / VC_THREADS));
        if (dst2)
            hipLaunchKernelGGL(vc_calibration_copy_kernel<2>, grid, dim3(VC_THREADS), 0, st, reinterpret_cast<const vc_u32x4 *>(src) + done,
                               reinterpret_cast<vc_u32x4 *>(dst) + done, reinterpret_cast<vc_u32x4 *>(dst2) + done, now);
        else
            hipLaunchKernelGGL(vc_calibration_copy_kernel<1>, grid, dim3(VC_THREADS), 0, st, reinterpret_cast<const vc_u32x4 *>(src) + done,
                               reinterpret_cast<vc_u32x4 *>(dst) + done, static_cast<vc_u32x4 *>(nullptr), now);
    }
    return hipGetLastError();
}
