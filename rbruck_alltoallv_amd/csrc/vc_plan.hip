// vc_plan.hip — turns the count tables into the work items of every launch.
//
// The reference learns the size of each incoming block from a metadata
// MPI_Sendrecv before every data round ("two-phase", src/twophase_tunable_rbruckv.cpp:110).
// With all P ranks' tables in one address space the size of a block is simply
// sendcounts[s][t] of the (s, t) it belongs to, and which (s, t) sits in a slot
// follows from the residency invariant (vc_plan_math.h).  Staging offsets (the
// reference's fixed-stride extra_buffer, :59) become exclusive prefix sums over
// the blocks that arrive in a rank's staging area in a digit phase, so the
// staging arena is compact; a second family of prefix sums numbers the work
// items (block pieces of at most VC_CHUNK bytes) so that every launch gets a
// dense list with no empty entries.
#include <algorithm>
#include <cstring>

#include "vc_common.h"
#include "vc_scan.h"

#include "vc_plan_math.h"

// ---- launch-per-digit execution, pass 1: row-wise prefix sums ----
// grid (P, regions + nl).  Rows y < regions = w + w2: staging sizes of region y, slot_off[(y*P + to)*P + id] = offset of the slot
// inside the row.  Later rows: work-item count and moved bytes of launch y - regions; the first of them also sums the
// payload and counts negative table entries.
// row_bytes rows: [launch][P], then [payload][P], then [negative entries][P].
__global__ __launch_bounds__(VC_THREADS) void vc_plan_rows(VcSched S, VcLaunchPack pack, const VcLaunchInfo *__restrict__ launches, int nl, VcTables T,
                                                           int64_t *__restrict__ slot_off, int64_t *__restrict__ row_tot,
                                                           int64_t *__restrict__ item_row_tot, int64_t *__restrict__ row_bytes) {
    __shared__ int64_t lds[VC_WAVES_PER_BLOCK];
    const int to = blockIdx.x, P = S.P;
    const int nreg = S.w + S.w2;                          // the organized region is laid out by vc_plan_org_rows
    if ((int)blockIdx.y < nreg && S.recycle) {
        // reused staging: the slots of the region in one prefix sum per hop slot in which their blocks leave again
        __shared__ int64_t family_carry[VC_RECYCLE_MAX_SLOTS];
        const int y = blockIdx.y, ns = nreg + 1, t_arrive = vc_slot_time(S, y);
        if (threadIdx.x < VC_RECYCLE_MAX_SLOTS) family_carry[threadIdx.x] = 0;
        __syncthreads();
        for (int base = 0; base < P; base += VC_THREADS) {
            const int id = base + threadIdx.x;
            int st[2] = {0, 0};
            const int64_t v = (id < P) ? vc_region_slot_size(S, T, y, to, id, nullptr, st) : 0;
            const int leaves = v ? vc_next_hop(S, st[0], st[1], y) : -1;
            for (int time = t_arrive + 1; time < ns; time++) {
                const int kd = vc_slot_time(S, time);
                int64_t total;
                const int64_t ex = vc_block_exclusive_scan(leaves == kd ? v : 0, lds, total);
                if (leaves == kd) slot_off[((int64_t)y * P + to) * P + id] = family_carry[kd] + ex;
                __syncthreads();
                if (threadIdx.x == 0) family_carry[kd] += total;
                __syncthreads();
            }
            if (id < P && !v) slot_off[((int64_t)y * P + to) * P + id] = 0;
        }
        if ((int)threadIdx.x < ns) row_tot[(int64_t)(y * ns + threadIdx.x) * P + to] = vc_slot_time(S, threadIdx.x) > t_arrive ? family_carry[threadIdx.x] : 0;
        return;
    }
    if ((int)blockIdx.y < nreg) {
        const int y = blockIdx.y;
        int64_t carry = 0;
        for (int base0 = 0; base0 < P; base0 += 4 * VC_THREADS) {       // four chunks at a time: their table reads travel together
            int64_t v[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int id = base0 + u * VC_THREADS + threadIdx.x;
                v[u] = (id < P) ? vc_region_slot_size(S, T, y, to, id) : 0;
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int id = base0 + u * VC_THREADS + threadIdx.x;
                if (base0 + u * VC_THREADS >= P) break;
                int64_t total;
                const int64_t ex = vc_block_exclusive_scan(v[u], lds, total);
                if (id < P) slot_off[((int64_t)y * P + to) * P + id] = carry + ex;
                carry += total;
            }
        }
        if (threadIdx.x == 0) row_tot[(int64_t)y * P + to] = carry;
        return;
    }
    int64_t items = 0, bytes = 0, payload = 0;
    int64_t bad = 0;                                      // entries of this rank's rows no rank could have passed
    const int L = blockIdx.y - nreg;
    const VcLaunchInfo info = launches ? launches[L] : pack.info[L];     // a short launch table travels as a kernel argument
    const int nent = vc_entries_per_rank(S, info);
    for (int id = threadIdx.x; id < nent; id += VC_THREADS) {
        VcEntry e;
        if (vc_entry_block(S, info, to, id, e)) {
            const int64_t len = vc_entry_len(S, T, e);
            items += vc_chunk_count(len, vc_entry_phase(S, T, e), vc_entry_cut(S, T, e));
            bytes += len;
        }
    }
    if (L == 0)
        for (int id = threadIdx.x; id < P; id += VC_THREADS) {
            payload += (int64_t)vc_rc(S, T, to, id) * S.esz;
            bad += vc_pair_bad_entries(S, T, id, to);
        }
    items = vc_block_sum(items, lds);
    bytes = vc_block_sum(bytes, lds);
    if (L == 0) {
        payload = vc_block_sum(payload, lds);
        bad = vc_block_sum(bad, lds);
        // the packed receive layout is an int prefix sum of the rank's receive counts, like the reference's displacements
        if (S.packed_recv && payload > (int64_t)0x7FFFFFFF * S.esz) bad += VC_BAD_OVERFLOW;
    }
    if (threadIdx.x == 0) {
        item_row_tot[(int64_t)L * P + to] = items;
        row_bytes[(int64_t)L * P + to] = bytes;
        if (L == 0) { row_bytes[(int64_t)nl * P + to] = payload; row_bytes[(int64_t)(nl + 1) * P + to] = bad; }
    }
}

// ---- pass 1b (S.coalesce): layout of the organized region, one workgroup per rank ----
// Scan of the run sizes over the groups, then slot_off[(w*P + to)*P + id] for every slot; row_tot[w*P + to].
__global__ __launch_bounds__(VC_THREADS) void vc_plan_org_rows(VcSched S, VcTables T, int64_t *__restrict__ slot_off,
                                                               int64_t *__restrict__ row_tot, int64_t *__restrict__ org_run_base) {
    __shared__ int64_t lds[VC_WAVES_PER_BLOCK];
    const int to = blockIdx.x, P = S.P, G = S.G;
    int64_t carry = 0;
    for (int base = 0; base < G; base += VC_THREADS) {
        const int g = base + threadIdx.x;
        int64_t total;
        const int64_t v = (g < G) ? vc_org_run_size(S, T, to, g) : 0;
        const int64_t ex = vc_block_exclusive_scan(v, lds, total);
        if (g < G) org_run_base[(int64_t)to * G + g] = carry + ex;
        carry += total;
    }
    const int ns = S.w + S.w2 + 1;
    if (threadIdx.x == 0) row_tot[(int64_t)(S.recycle ? ns * ns : S.w) * P + to] = carry;
    __syncthreads();                                      // org_run_base of this rank is complete (same workgroup wrote it)
    for (int id = threadIdx.x; id < P; id += VC_THREADS)
        slot_off[((int64_t)S.w * P + to) * P + id] = org_run_base[(int64_t)to * G + vc_div(id, S.dn)] + vc_org_slot_rel(S, T, to, id);
}

// ---- launch-per-digit execution, pass 2: prefix sums over the rows ----
// grid (nl + 1).  Workgroup L < nl: item bases of launch L's rows (relative to the launch's first item), its item count and
// moved bytes.  Workgroup nl: staging row bases, staging bytes, payload bytes, negative table entries.
__global__ __launch_bounds__(VC_THREADS) void vc_plan_bases(VcSched S, int P, int w, int nreg, int nl, const int64_t *__restrict__ row_tot,
                                                            int64_t *__restrict__ row_base, const int64_t *__restrict__ item_row_tot,
                                                            int64_t *__restrict__ item_row_base, const int64_t *__restrict__ row_bytes,
                                                            int64_t *__restrict__ header, int64_t *__restrict__ header_host) {
    __shared__ int64_t lds[VC_WAVES_PER_BLOCK];
    const int L = blockIdx.x;
    const bool recycle = S.recycle != 0;
    int64_t carry = 0, bytes = 0;
    if (L == nl && recycle) {
        // reused staging: row offsets inside every sub-region, the sizes of the sub-regions' pieces (the rows of
        // vc_recycle_rows_per_segment(P) consecutive receivers each), their places in the arena
        __shared__ int64_t piece_size[VC_RECYCLE_MAX_PAIRS * VC_RECYCLE_SEGMENTS], piece_base[VC_RECYCLE_MAX_PAIRS * VC_RECYCLE_SEGMENTS],
            hole_lo[VC_RECYCLE_MAX_HOLES], hole_hi[VC_RECYCLE_MAX_HOLES];
        const int ns = nreg + 1, nfam = ns * ns + 1, nseg = VC_RECYCLE_SEGMENTS, rps = vc_recycle_rows_per_segment(P);
        for (int f = 0; f < nfam; f++) {
            const int ka = f / ns, kd = f % ns;
            const bool used = f == ns * ns ? w > nreg : (ka < nreg && vc_slot_time(S, kd) > vc_slot_time(S, ka));
            int64_t fam_carry = 0;
            if (used)
                for (int b0 = 0; b0 < P; b0 += VC_THREADS) {
                    const int i = b0 + threadIdx.x;
                    int64_t total;
                    const int64_t ex = vc_block_exclusive_scan((i < P) ? row_tot[(int64_t)f * P + i] : 0, lds, total);
                    if (i < P) {
                        row_base[(int64_t)f * P + i] = fam_carry + ex;
                        if (i % rps == 0) piece_base[f * nseg + i / rps] = fam_carry + ex;      // where the piece starts (for now)
                    }
                    fam_carry += total;
                }
            __syncthreads();
            if ((int)threadIdx.x < nseg) {
                const int g = threadIdx.x;
                const bool has = used && g * rps < P, more = g + 1 < nseg && (g + 1) * rps < P;
                piece_size[f * nseg + g] = has ? (more ? piece_base[f * nseg + g + 1] : fam_carry) - piece_base[f * nseg + g] : 0;
            }
            __syncthreads();
        }
        if (threadIdx.x == 0) carry = vc_allocate_staging(S, piece_size, piece_base, hole_lo, hole_hi);
        __syncthreads();
        for (int64_t i = threadIdx.x; i < (int64_t)nfam * P; i += VC_THREADS) {
            const int f = (int)(i / P), g = (int)(i % P) / rps;
            int64_t start = 0;                            // offset of the piece's first row inside the sub-region
            for (int k = 0; k < g; k++) start += piece_size[f * nseg + k];
            if (piece_size[f * nseg + g] > 0) row_base[i] += piece_base[f * nseg + g] - start;
        }
        int64_t bad = 0;
        for (int i = threadIdx.x; i < P; i += VC_THREADS) { bytes += row_bytes[(int64_t)nl * P + i]; bad += row_bytes[(int64_t)(nl + 1) * P + i]; }
        bytes = vc_block_sum(bytes, lds);
        bad = vc_block_sum(bad, lds);
        if (threadIdx.x == 0) {
            header[0] = carry; header[1] = bytes; header[VC_HEADER_BAD] = bad;
            if (header_host) { header_host[0] = carry; header_host[1] = bytes; header_host[VC_HEADER_BAD] = bad; }
        }
        return;
    }
    if (L == nl) {
        const int64_t nrows = (int64_t)w * P;                 // w = number of staging regions
        for (int64_t b0 = 0; b0 < nrows; b0 += VC_THREADS) {
            const int64_t i = b0 + threadIdx.x;
            int64_t total;
            const int64_t v = (i < nrows) ? row_tot[i] : 0;
            const int64_t ex = vc_block_exclusive_scan(v, lds, total);
            if (i < nrows) row_base[i] = carry + ex;
            carry += total;
        }
        int64_t bad = 0;
        for (int i = threadIdx.x; i < P; i += VC_THREADS) { bytes += row_bytes[(int64_t)nl * P + i]; bad += row_bytes[(int64_t)(nl + 1) * P + i]; }
        bytes = vc_block_sum(bytes, lds);
        bad = vc_block_sum(bad, lds);
        if (threadIdx.x == 0) {
            header[0] = carry; header[1] = bytes; header[VC_HEADER_BAD] = bad;
            if (header_host) { header_host[0] = carry; header_host[1] = bytes; header_host[VC_HEADER_BAD] = bad; }
        }
        return;
    }
    for (int b0 = 0; b0 < P; b0 += VC_THREADS) {
        const int i = b0 + threadIdx.x;
        int64_t total;
        const int64_t v = (i < P) ? item_row_tot[(int64_t)L * P + i] : 0;
        const int64_t ex = vc_block_exclusive_scan(v, lds, total);
        if (i < P) item_row_base[(int64_t)L * P + i] = carry + ex;
        carry += total;
        bytes += (i < P) ? row_bytes[(int64_t)L * P + i] : 0;
    }
    bytes = vc_block_sum(bytes, lds);
    if (threadIdx.x == 0) {
        header[VC_HEADER_FIXED + L] = bytes; header[VC_HEADER_FIXED + nl + L] = carry;
        if (header_host) { header_host[VC_HEADER_FIXED + L] = bytes; header_host[VC_HEADER_FIXED + nl + L] = carry; }      // pinned host memory: no copy back
    }
}

// ---- launch-per-digit execution, pass 3: the work items ----
// grid (P, nl, Z).  Repeats the row scan of pass 1 to place every block's pieces; Z workgroups share a receiver's entries
// when there are few ranks (their blocks are then huge and have many pieces).
__global__ __launch_bounds__(VC_THREADS) void vc_plan_emit(VcSched S, VcLaunchPack pack, const VcLaunchInfo *__restrict__ launches, VcTables T,
                                                           const int64_t *__restrict__ slot_off, const int64_t *__restrict__ row_base,
                                                           const int64_t *__restrict__ item_row_base, const int64_t *__restrict__ header,
                                                           int nl, VcDesc *__restrict__ items) {
    __shared__ int64_t lds[VC_WAVES_PER_BLOCK];
    const int to = blockIdx.x, L = blockIdx.y, P = S.P;
    const VcLaunchInfo info = launches ? launches[L] : pack.info[L];
    int64_t first = 0;                                    // items of the launches before this one
    for (int k = threadIdx.x; k < L; k += VC_THREADS) first += header[VC_HEADER_FIXED + nl + k];
    first = vc_block_sum(first, lds);
    int64_t carry = first + item_row_base[(int64_t)L * P + to];
    // copies of many pieces are written by the whole workgroup: their pieces are numbered by a second prefix sum and
    // every lane takes every 256th piece, finding the copy it belongs to by bisection
    __shared__ VcDesc big_whole[VC_THREADS];
    __shared__ int64_t big_at[VC_THREADS], big_pre[VC_THREADS];
    __shared__ int big_phase[VC_THREADS], big_cut[VC_THREADS];
    const int nent_all = vc_entries_per_rank(S, info);
    // workgroup (to, L, z) writes the z-th slice of the receiver's entries; the items of the slices before it come first
    const int per = (nent_all + (int)gridDim.z - 1) / (int)gridDim.z;
    const int e_lo = (int)blockIdx.z * per < nent_all ? (int)blockIdx.z * per : nent_all;
    const int nent = e_lo + per < nent_all ? e_lo + per : nent_all;
    int64_t before = 0;
    for (int id = threadIdx.x; id < e_lo; id += VC_THREADS) {
        VcEntry e;
        if (vc_entry_block(S, info, to, id, e))
            before += vc_chunk_count(vc_entry_len(S, T, e), vc_entry_phase(S, T, e), vc_entry_cut(S, T, e));
    }
    carry += vc_block_sum(before, lds);
    for (int base = e_lo; base < nent; base += VC_THREADS) {
        const int id = base + threadIdx.x;
        VcEntry e;
        const bool active = id < nent && vc_entry_block(S, info, to, id, e);
        const int64_t len = active ? vc_entry_len(S, T, e) : 0;
        const int phase = active ? vc_entry_phase(S, T, e) : 0, cut = active ? vc_entry_cut(S, T, e) : 0;
        const int64_t cnt = vc_chunk_count(len, phase, cut);
        int64_t total;
        const int64_t at = carry + vc_block_exclusive_scan(cnt, lds, total);
        const bool big = cnt > 4;
        if (cnt) {
            const VcDesc whole = vc_entry_desc(S, T, slot_off, row_base, e, to);
            if (!big)
                for (int64_t c = 0; c < cnt; c++) items[at + c] = vc_chunk_of(whole, c, phase, cut);
            else { big_whole[threadIdx.x] = whole; big_at[threadIdx.x] = at; big_phase[threadIdx.x] = phase; big_cut[threadIdx.x] = cut; }
        }
        if (__syncthreads_or(big)) {
            int64_t btotal;
            big_pre[threadIdx.x] = vc_block_exclusive_scan(big ? cnt : 0, lds, btotal);
            __syncthreads();
            for (int64_t q = threadIdx.x; q < btotal; q += VC_THREADS) {
                int lo = 0, hi = VC_THREADS - 1;              // last lane whose pieces start at or before q
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (big_pre[mid] <= q) lo = mid; else hi = mid - 1;
                }
                const int64_t c = q - big_pre[lo];
                items[big_at[lo] + c] = vc_chunk_of(big_whole[lo], c, big_phase[lo], big_cut[lo]);
            }
            __syncthreads();                              // the lists are reused by the next round
        }
        carry += total;
    }
}

// Workgroups that share one receiver's entries when items are emitted: one per ~2048 items of an average row, so that
// a few ranks with huge blocks (many pieces each) still fill the chip, and small problems stay one workgroup per row.
static int vc_emit_slices(int64_t nitems, int64_t rows) {
    const int64_t per_row = nitems / (rows > 0 ? rows : 1);
    const int64_t z = (per_row + 2047) / 2048;
    return (int)(z < 1 ? 1 : (z > 16 ? 16 : z));
}

static VcLaunchPack vc_pack_launches(const VcLaunchInfo *host, int nl) {
    VcLaunchPack pack;
    memset(&pack, 0, sizeof pack);
    for (int k = 0; k < nl && k < VC_LAUNCH_PACK; k++) pack.info[k] = host[k];
    return pack;
}

hipError_t vc_launch_plan_sizes(const VcSched &S, const VcLaunchInfo *launches_host, const VcLaunchInfo *launches_dev, int nl,
                                VcTables T, int64_t *slot_off,
                                int64_t *row_tot, int64_t *row_base, int64_t *org_run_base, int64_t *item_row_tot,
                                int64_t *item_row_base, int64_t *row_bytes, int64_t *header, int64_t *header_host, hipStream_t st) {
    const int nreg = S.w + S.w2;
    hipLaunchKernelGGL(vc_plan_rows, dim3(S.P, nreg + nl), dim3(VC_THREADS), 0, st, S, vc_pack_launches(launches_host, nl),
                       nl <= VC_LAUNCH_PACK ? nullptr : launches_dev, nl, T, slot_off, row_tot, item_row_tot, row_bytes);
    if (S.coalesce)
        hipLaunchKernelGGL(vc_plan_org_rows, dim3(S.P), dim3(VC_THREADS), 0, st, S, T, slot_off, row_tot, org_run_base);
    hipLaunchKernelGGL(vc_plan_bases, dim3(nl + 1), dim3(VC_THREADS), 0, st, S, S.P, vc_regions(S), nreg, nl, row_tot, row_base,
                       item_row_tot, item_row_base, row_bytes, header, header_host);
    return hipGetLastError();
}

hipError_t vc_launch_plan_emit(const VcSched &S, const VcLaunchInfo *launches_host, const VcLaunchInfo *launches_dev, int nlaunch,
                               VcTables T, const int64_t *slot_off,
                               const int64_t *row_base, const int64_t *item_row_base, const int64_t *header, VcDesc *items,
                               int64_t nitems, hipStream_t st) {
    const int slices = vc_emit_slices(nitems, (int64_t)S.P * nlaunch);
    hipLaunchKernelGGL(vc_plan_emit, dim3(S.P, nlaunch, slices), dim3(VC_THREADS), 0, st, S, vc_pack_launches(launches_host, nlaunch),
                       nlaunch <= VC_LAUNCH_PACK ? nullptr : launches_dev, T, slot_off, row_base, item_row_base, header, nlaunch, items);
    return hipGetLastError();
}

// ---- forwarded execution ----
#define VC_PLAN_XCDS 8
// Rows a kernel gives a workgroup each: workgroup b runs on XCD b mod 8, and XCD k takes the k-th eighth of the ranks, so that
// the table entries of neighbouring ranks, which share cache lines (the entries of a rank lie in a column), meet in one L2.
static unsigned vc_rank_grid(int P, int rows) { return (unsigned)((P + VC_PLAN_XCDS - 1) / VC_PLAN_XCDS) * VC_PLAN_XCDS * rows; }

// What the last workgroup of a grid reads is stored and loaded past the L2 of the storing and the loading XCD.
__device__ __forceinline__ void vc_share(int64_t *p, int64_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ int64_t vc_shared(const int64_t *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Everything that has to be known before the list or the blocks: grid vc_rank_grid(P, regions + 1).  Of the rows of rank `to`, row
// y < regions = w + w2 sums up the staging slots of region y (slot_off[(y*P + to)*P + id] = offset of slot id inside the row, in lines) and
// the bytes of the blocks in them (every staged block is one hop); the last row counts the chain items of the blocks that end
// on the rank (by tile of VC_TILE_RANKS sources for vc_chain_emit), the payload, the table entries no rank could have
// passed, the most pieces and the longest of its blocks.
// A call in batches counts the slots, items and bytes of the blocks for the receivers of the batch only, and checks all of the tables.
// row_bytes rows: [region][P] bytes of staged blocks, then [payload][P], [bad entries][P], [longest block][P].
// chain_row_tot: [P] items, [P] most pieces, [P][tiles] items per tile of sources.
// The workgroup that finishes last turns the row totals into first addresses (row_base, chain_row_base: exclusive sums) and
// the header: a kernel of its own for that is a kernel boundary (2.6 us) more.  It learns that it is the last one from a count; no
// release fence is needed (one per workgroup would write the XCD's L2 back each time: calls on 160 - 512 ranks took twice
// as long that way), because the totals are stored past the L2 and waited for before the workgroup counts itself.
// Latency bound below about 512 ranks.  Together with the prefix sums by data-parallel primitives and one reduction for
// all totals: 150 ranks, four digits, 7.2 + 5.8 us (two kernels) -> 9.0,
// 256 ranks, two digits, 7.2 + 4.8 -> 10.1, 1024 ranks in nodes of 32 27 + 7.5 -> 26.
// PER: consecutive slots or sources per thread and round, so that one round takes all of them up to 1024 ranks.
template <int PER>
__global__ __launch_bounds__(VC_THREADS) void vc_plan_forward(VcSched S, VcTables T, uint32_t *__restrict__ slot_off, int64_t *row_tot,
                                                              int64_t *__restrict__ row_base, int64_t *row_bytes, int64_t *chain_row_tot,
                                                              int64_t *__restrict__ chain_row_base, int64_t *__restrict__ header,
                                                              int64_t *__restrict__ header_host, unsigned *ticket) {
    __shared__ int64_t lds[5 * VC_WAVES_PER_BLOCK];
    __shared__ int is_last;
    const int P = S.P, nreg = S.w + S.w2, nrow = nreg + 1, ranks_per_xcd = (P + VC_PLAN_XCDS - 1) / VC_PLAN_XCDS;
    const int at = blockIdx.x / VC_PLAN_XCDS, y = at % nrow, to = (int)(blockIdx.x % VC_PLAN_XCDS) * ranks_per_xcd + at / nrow;
    if (to < P && y < nreg) {
        int64_t carry = 0, data = 0;
        uint32_t *const slots = slot_off + ((int64_t)y * P + to) * P;
        for (int base = 0; base < P; base += PER * VC_THREADS) {
            const int id0 = base + threadIdx.x * PER;
            int64_t v[PER], rbase[PER], round = 0, total;
            int count[PER], displ[PER];
            bool there[PER];
#pragma unroll
            for (int u = 0; u < PER; u++) {                 // all reads first: none depends on another
                int s, t;
                const bool inside = id0 + u < P;
                there[u] = vc_slot_block(S, y, to, inside ? id0 + u : 0, s, t) && inside && vc_receives_now(S, t);
                count[u] = vc_sc(S, T, s, t); displ[u] = vc_rd(S, T, t, s); rbase[u] = T.rbase[t];
            }
#pragma unroll
            for (int u = 0; u < PER; u++) {
                const int64_t len = there[u] ? (int64_t)count[u] * S.esz : 0, phase = (rbase[u] + (int64_t)displ[u] * S.esz + S.recv_lo) & (VC_LINE - 1);
                v[u] = len ? (len + phase + VC_LINE - 1) & ~(int64_t)(VC_LINE - 1) : 0;
                round += v[u];
                data += len;
            }
            int64_t off = carry + vc_block_exclusive_scan(round, lds, total);
#pragma unroll
            for (int u = 0; u < PER; u++) {
                if (id0 + u < P) slots[id0 + u] = (uint32_t)(off / VC_LINE);
                off += v[u];
            }
            carry += total;
        }
        data = vc_block_sum(data, lds);
        if (threadIdx.x == 0) { vc_share(&row_tot[(int64_t)y * P + to], carry); vc_share(&row_bytes[(int64_t)y * P + to], data); }
    } else if (to < P) {
        const int ntile = VC_TILES(P), lanes = VC_TILE_RANKS / PER;              // threads per tile of sources
        const bool now = vc_receives_now(S, to);
        int64_t sum[5] = {0, 0, 0, 0, 0};                 // items, payload, bad entries; most pieces, longest block
        for (int base = 0; base < P; base += PER * VC_THREADS) {
            const int s0 = base + threadIdx.x * PER;
            int64_t tile = 0;
            VcPairEntries e[PER];
#pragma unroll
            for (int u = 0; u < PER; u++) {                 // all reads first
                e[u] = vc_pair_entries(S, T, s0 + u < P ? s0 + u : 0, to);
            }
            const int64_t rbase = T.rbase[to];
#pragma unroll
            for (int u = 0; u < PER; u++) {
                if (s0 + u >= P) continue;
                const int64_t len = (int64_t)e[u].sent * S.esz;
                const int cut = (int)((rbase + (int64_t)e[u].rd * S.esz + S.recv_lo) & (VC_PIECE - 1));
                const int64_t cnt = now ? vc_chunk_count(len, cut & (VC_LINE - 1), cut) : 0;
                tile += cnt;
                sum[1] += now ? (int64_t)e[u].expected * S.esz : 0;
                sum[2] += vc_bad_entries(S, e[u]);
                sum[3] = cnt > sum[3] ? cnt : sum[3];
                sum[4] = len > sum[4] ? len : sum[4];
            }
            sum[0] += tile;
            for (int o = 1; o < lanes; o <<= 1) tile += __shfl_xor(tile, o, VC_WAVE);
            if (threadIdx.x % lanes == 0 && s0 < P) chain_row_tot[2 * (int64_t)P + (int64_t)to * ntile + s0 / VC_TILE_RANKS] = tile;
        }
        vc_block_totals(sum, lds);
        if (threadIdx.x == 0) {
            // the packed receive layout is an int prefix sum of the rank's receive counts, like the reference's displacements
            if (S.packed_recv && sum[1] > (int64_t)0x7FFFFFFF * S.esz) sum[2] += VC_BAD_OVERFLOW;
            vc_share(&chain_row_tot[to], sum[0]);
            vc_share(&chain_row_tot[P + to], sum[3]);
            vc_share(&row_bytes[(int64_t)nreg * P + to], sum[1]);
            vc_share(&row_bytes[(int64_t)(nreg + 1) * P + to], sum[2]);
            vc_share(&row_bytes[(int64_t)(nreg + 2) * P + to], sum[4]);
        }
    }
    if (threadIdx.x == 0) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this workgroup's totals are where the last one will look
        is_last = vc_last_workgroup(ticket);
    }
    __syncthreads();
    if (!is_last) return;
    // rows are summed up in blocks of 4 per thread
    int64_t carry = 0, items = 0, total;
    const int64_t nrows = (int64_t)nreg * P;
    int64_t sum[5] = {0, 0, 0, 0, 0};                     // payload, staged bytes, bad entries; most pieces, longest block
    int64_t row_v[4], row_d[4];                           // the first round of the second loop, read together with the first loop's
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int64_t i = threadIdx.x * 4 + u;
        row_v[u] = i < nrows ? vc_shared(&row_tot[i]) : 0;
        row_d[u] = i < nrows ? vc_shared(&row_bytes[i]) : 0;
    }
    for (int64_t base = 0; base < P; base += 4 * VC_THREADS) {
        int64_t v[4], pay[4], bad[4], most[4], longest[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int64_t i = base + threadIdx.x * 4 + u;
            const bool inside = i < P;
            v[u] = inside ? vc_shared(&chain_row_tot[i]) : 0;
            most[u] = inside ? vc_shared(&chain_row_tot[P + i]) : 0;
            pay[u] = inside ? vc_shared(&row_bytes[nreg * (int64_t)P + i]) : 0;
            bad[u] = inside ? vc_shared(&row_bytes[(nreg + 1) * (int64_t)P + i]) : 0;
            longest[u] = inside ? vc_shared(&row_bytes[(nreg + 2) * (int64_t)P + i]) : 0;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            sum[0] += pay[u];
            sum[2] += bad[u];
            sum[3] = most[u] > sum[3] ? most[u] : sum[3];
            sum[4] = longest[u] > sum[4] ? longest[u] : sum[4];
        }
        int64_t off = items + vc_block_exclusive_scan(v[0] + v[1] + v[2] + v[3], lds, total);
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int64_t i = base + threadIdx.x * 4 + u;
            if (i < P) chain_row_base[i] = off;
            off += v[u];
        }
        items += total;
    }
    for (int64_t base = 0; base < nrows; base += 4 * VC_THREADS) {
        sum[1] += row_d[0] + row_d[1] + row_d[2] + row_d[3];
        int64_t off = carry + vc_block_exclusive_scan(row_v[0] + row_v[1] + row_v[2] + row_v[3], lds, total);
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int64_t i = base + threadIdx.x * 4 + u, next = i + 4 * VC_THREADS;
            if (i < nrows) row_base[i] = off;
            off += row_v[u];
            row_v[u] = next < nrows ? vc_shared(&row_tot[next]) : 0;
            row_d[u] = next < nrows ? vc_shared(&row_bytes[next]) : 0;
        }
        carry += total;
    }
    __syncthreads();                                      // lds from the scans above
    vc_block_totals(sum, lds);
    if (threadIdx.x != 0) return;
    // every staged block is one hop, every block's last hop ends in recvbuf
    const int64_t words[VC_HEADER_MAX_LEN + 1] = {vc_window_bytes(carry, S.window), sum[0], items, sum[2], sum[3], sum[0] + sum[1], sum[4]};
#pragma unroll
    for (int k = 0; k <= VC_HEADER_MAX_LEN; k++) { header[k] = words[k]; header_host[k] = words[k]; }
}
static_assert(VC_HEADER_BAD == 3 && VC_HEADER_MAX_PIECES == 4 && VC_HEADER_FIXED == 5 && VC_HEADER_MAX_LEN == 6, "order of the words above");

hipError_t vc_launch_plan_forward(const VcSched &S, VcTables T, uint32_t *slot_off, int64_t *row_tot, int64_t *row_base, int64_t *row_bytes,
                                  int64_t *chain_row_tot, int64_t *chain_row_base, int64_t *header, int64_t *header_host, unsigned *ticket,
                                  hipStream_t st) {
    const auto kernel = S.P <= VC_THREADS ? vc_plan_forward<1> : (S.P <= 2 * VC_THREADS ? vc_plan_forward<2> : vc_plan_forward<4>);
    hipLaunchKernelGGL(kernel, dim3(vc_rank_grid(S.P, S.w + S.w2 + 1)), dim3(VC_THREADS), 0, st, S, T, slot_off, row_tot, row_base,
                       row_bytes, chain_row_tot, chain_row_base, header, header_host, ticket);
    return hipGetLastError();
}

// ---- calls without a list on slots of a fixed stride: nothing has to be summed up but what the header holds ----
#define VC_CHECK_RANKS 4
struct __attribute__((packed, aligned(4))) VcFour { int v[VC_CHECK_RANKS]; };
enum { VC_CHECK_PAYLOAD, VC_CHECK_MOVED, VC_CHECK_BAD, VC_CHECK_ITEMS, VC_CHECK_MOST, VC_CHECK_LONGEST, VC_CHECK_WORDS };

// Digits of x, of `digits`, that are not zero: the hops of a block with that offset inside the node, or between the nodes.
__device__ __forceinline__ int vc_offset_digits(const VcSched &S, int x, int digits) {
    int hops = 0;
    for (int k = 0; k < digits; k++) { const int q = vc_div(x, S.dr); hops += q * S.r != x; x = q; }
    return hops;
}

// A workgroup has four receivers, a thread one source at a time: what the source sends to the four is one read of 16 bytes (a column of the
// table, which costs a request per entry when it is read one at a time as in vc_plan_forward), the receivers' own rows are read along.
// PACKED (S.packed_recv): writes the packed receive displacements on the way (rd_packed), which took a kernel of their own before.
// Bound by the latency of one round of reads, all of a thread's at once, of the count of the workgroups and of the last one's read of their sums; on 1024 ranks, four
// wavefronts a SIMD, by instructions as well.  So the hops of an offset come from a table in LDS instead of its digits, pair by pair; a wavefront whose blocks are all of
// one piece wherever they lie (whole_elems) counts them in ballots and adds up three quantities in elements, one whose blocks are no longer than VC_CHECK_SHORT bytes in
// 32 bits; the wavefronts of a workgroup add to its sums by LDS atomics, and the last workgroup has a wavefront a word.  Kernel, before / after: 200 ranks 7.0 us / 6.3,
// 256 7.5 / 6.4, 512 9.4 / 7.0, 1024 13.3 / 10.0, there with packed displacements 19.4 / 15.2 (vc_plan_forward 24 - 29, and 6.8 for vc_row_scan_kernel).
// A thread with four sources, a tile of 4 x 4 entries: too few wavefronts (10, 12.1 and 14.6 where 7.0, 7.5 and 12.8 were).
// As the first wavefronts of the copy kernel instead (copying ones wait for a verdict): even at best, because registers of the check are the copying wavefronts' too and
// thousands of them poll (1024 ranks, 0 - 16 B 46.8 us a call / 47.3; 300, 400 B direct 38.9 / 50).
// group_tot: VC_CHECK_WORDS words per four receivers.  Header as vc_plan_forward leaves it, its first word `stage_bytes`.  short_elems:
// the elements of VC_CHECK_SHORT bytes.
#define VC_CHECK_SHORT (1u << 18)                         // (64 lanes x 4 blocks x 32 hops of them are 2^31 bytes)
template <int THREADS, bool PACKED>
__global__ __launch_bounds__(THREADS) void vc_plan_check(VcSched S, VcTables T, int *__restrict__ rd_packed, int64_t *group_tot, int64_t stage_bytes,
                                                         unsigned whole_elems, unsigned short_elems, int64_t *__restrict__ header, int64_t *__restrict__ header_host,
                                                         unsigned *ticket) {
    constexpr int R = VC_CHECK_RANKS, WAVES = THREADS / VC_WAVE;
    static_assert((uint64_t)VC_CHECK_SHORT * R * VC_WAVE * VC_MAX_HOP_SLOTS <= (uint64_t)1 << 31, "sums of a wavefront in 32 bits");
    __shared__ int64_t of_wave[WAVES][R];
    __shared__ unsigned long long of_group[VC_CHECK_WORDS];
    __shared__ int is_last;
    extern __shared__ unsigned char hops_of[];            // hops of the offsets inside the node, then of those between the nodes
    const int P = S.P, groups = (P + R - 1) / R, groups_per_xcd = (groups + VC_PLAN_XCDS - 1) / VC_PLAN_XCDS;
    const int group = (int)(blockIdx.x % VC_PLAN_XCDS) * groups_per_xcd + (int)blockIdx.x / VC_PLAN_XCDS;      // (grid: VC_PLAN_XCDS x groups_per_xcd)
    const int lane = threadIdx.x % VC_WAVE, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / VC_WAVE), t0 = group * R;
    int64_t sum[VC_CHECK_WORDS] = {0, 0, 0, 0, 0, 0};     // (of the wavefront, in its last lane)
    const auto look_up = [&]() {                          // once, with the first table entries on their way
        for (int i = (int)threadIdx.x; i < S.n + S.G; i += THREADS)
            hops_of[i] = (unsigned char)(i < S.n ? vc_offset_digits(S, i, S.w)
                                                 : vc_offset_digits(S, i - S.n, S.w2) + (S.last_hop == 2 || (S.last_hop == 1 && i != S.n)));
        if (threadIdx.x < VC_CHECK_WORDS) of_group[threadIdx.x] = 0;
        __syncthreads();
    };
    if (group < groups) {
        int64_t carry[R] = {0, 0, 0, 0};
        for (int base = 0; base < P; base += THREADS) {
            const bool live = base + (int)threadIdx.x < P;
            const int s = live ? base + (int)threadIdx.x : 0;
            VcPairEntries e[R];
            int64_t rbase[R];
            if (t0 + R <= P && S.table_mask) {            // (the same branch in every thread)
                const VcFour column = *reinterpret_cast<const VcFour *>(reinterpret_cast<const char *>(T.sc) + ((unsigned)(s * P + t0) << 2));
#pragma unroll
                for (int j = 0; j < R; j++) e[j].sent = column.v[j];
            } else {
#pragma unroll
                for (int j = 0; j < R; j++) e[j].sent = vc_sc(S, T, s, t0 + j < P ? t0 + j : 0);
            }
#pragma unroll
            for (int j = 0; j < R; j++) {
                const int t = t0 + j < P ? t0 + j : 0;
                e[j].expected = vc_rc(S, T, t, s);
                e[j].rd = PACKED ? 0 : vc_rd(S, T, t, s);
                e[j].own = vc_sc(S, T, t, s) | vc_sd(S, T, t, s);
                rbase[j] = T.rbase[t];
            }
            if (base == 0) look_up();
            if (base + wave * VC_WAVE + VC_WAVE > P || t0 + R > P)       // (the same branch in a wavefront)
#pragma unroll
                for (int j = 0; j < R; j++)
                    if (!live || t0 + j >= P) e[j] = {0, 0, 0, 0};
            unsigned largest = 0;
#pragma unroll
            for (int j = 0; j < R; j++) {
                largest = (unsigned)e[j].sent > largest ? (unsigned)e[j].sent : largest;
                largest = (unsigned)e[j].expected > largest ? (unsigned)e[j].expected : largest;
            }
            const bool all_whole = __ballot(largest > whole_elems) == 0, all_brief = __ballot(largest > short_elems) == 0;
            if (PACKED) {
                int64_t incl[R];
#pragma unroll
                for (int j = 0; j < R; j++) incl[j] = all_brief ? (int64_t)vc_wave_join_last<false>((unsigned)e[j].expected) : vc_wave_inclusive_scan(e[j].expected);
                if (base) __syncthreads();                // (of_wave is read no more)
                if (lane == VC_WAVE - 1)
#pragma unroll
                    for (int j = 0; j < R; j++) of_wave[wave][j] = incl[j];
                __syncthreads();
                // lane 16 j + q: of row j, wavefronts 0 .. q
                const int64_t upto = vc_row_inclusive_scan(lane % 16 < WAVES ? of_wave[lane % 16][lane / 16] : 0);
#pragma unroll
                for (int j = 0; j < R; j++) {
                    const int64_t before = wave ? vc_lane(upto, 16 * j + wave - 1) : 0;
                    e[j].rd = (int)(carry[j] + before + incl[j] - e[j].expected);
                    carry[j] += vc_lane(upto, 16 * j + 15);
                    if (live && t0 + j < P) rd_packed[(int64_t)(t0 + j) * P + s] = e[j].rd;
                }
            }
            const int gs = vc_div(s, S.dn), ls = s - gs * S.n;
            int hops[R];
#pragma unroll
            for (int j = 0; j < R; j++) {
                const int t = t0 + j < P ? t0 + j : 0, gt = vc_div(t, S.dn), lt = t - gt * S.n;
                hops[j] = hops_of[vc_wrap(ls - lt + S.n, S.n)] + hops_of[S.n + vc_wrap(gs - gt + S.G, S.G)] + (s == t && S.last_hop != 2);
            }
            int64_t wide[VC_CHECK_WORDS] = {0, 0, 0, 0, 0, 0};
            if (all_whole) {                              // (in elements)
                unsigned payload = 0, moved = 0, longest = 0;
#pragma unroll
                for (int j = 0; j < R; j++) {
                    wide[VC_CHECK_ITEMS] += __popcll(__ballot(e[j].sent != 0));
                    wide[VC_CHECK_BAD] += __popcll(__ballot(e[j].expected != e[j].sent)) + __popcll(__ballot((e[j].own | (PACKED ? 0 : e[j].rd)) < 0));
                    payload += (unsigned)e[j].expected;
                    moved += __umul24((unsigned)e[j].sent, (unsigned)hops[j]);
                    longest = (unsigned)e[j].sent > longest ? (unsigned)e[j].sent : longest;
                }
                wide[VC_CHECK_PAYLOAD] = (int64_t)vc_wave_join_last<false>(payload) * S.esz;
                wide[VC_CHECK_MOVED] = (int64_t)vc_wave_join_last<false>(moved) * S.esz;
                wide[VC_CHECK_LONGEST] = (int64_t)vc_wave_join_last<true>(longest) * S.esz;
                wide[VC_CHECK_MOST] = wide[VC_CHECK_ITEMS] > 0;
            } else {
                unsigned payload = 0, moved = 0, bad = 0, items = 0, most = 0, longest = 0;
#pragma unroll
                for (int j = 0; j < R; j++) {
                    // (a power of two of the byte address: 32 bits that wrap around do)
                    const unsigned cut = ((unsigned)rbase[j] + (unsigned)e[j].rd * (unsigned)S.esz + (unsigned)S.recv_lo) & (VC_PIECE - 1), phase = cut & (VC_LINE - 1);
                    bad += vc_bad_entries(S, e[j]);
                    if (all_brief) {
                        const unsigned len = (unsigned)e[j].sent * (unsigned)S.esz;
                        const unsigned cnt = len == 0 ? 0 : (len + phase <= VC_CHUNK ? 1 : (len + cut + VC_PIECE - 1) / VC_PIECE);
                        payload += (unsigned)e[j].expected * (unsigned)S.esz;
                        moved += len * hops[j];
                        items += cnt;
                        most = cnt > most ? cnt : most;
                        longest = len > longest ? len : longest;
                    } else {
                        const int64_t len = (int64_t)e[j].sent * S.esz, cnt = vc_chunk_count(len, (int)phase, (int)cut);
                        wide[VC_CHECK_PAYLOAD] += (int64_t)e[j].expected * S.esz;
                        wide[VC_CHECK_MOVED] += len * hops[j];
                        wide[VC_CHECK_ITEMS] += cnt;
                        wide[VC_CHECK_MOST] = cnt > wide[VC_CHECK_MOST] ? cnt : wide[VC_CHECK_MOST];
                        wide[VC_CHECK_LONGEST] = len > wide[VC_CHECK_LONGEST] ? len : wide[VC_CHECK_LONGEST];
                    }
                }
                if (all_brief) {
                    wide[VC_CHECK_PAYLOAD] = vc_wave_join_last<false>(payload);
                    wide[VC_CHECK_MOVED] = vc_wave_join_last<false>(moved);
                    wide[VC_CHECK_ITEMS] = vc_wave_join_last<false>(items);
                    wide[VC_CHECK_MOST] = vc_wave_join_last<true>(most);
                    wide[VC_CHECK_LONGEST] = vc_wave_join_last<true>(longest);
                } else {
                    wide[VC_CHECK_PAYLOAD] = vc_wave_inclusive_scan(wide[VC_CHECK_PAYLOAD]);
                    wide[VC_CHECK_MOVED] = vc_wave_inclusive_scan(wide[VC_CHECK_MOVED]);
                    wide[VC_CHECK_ITEMS] = vc_wave_inclusive_scan(wide[VC_CHECK_ITEMS]);
                    wide[VC_CHECK_MOST] = vc_wave_max_last(wide[VC_CHECK_MOST]);
                    wide[VC_CHECK_LONGEST] = vc_wave_max_last(wide[VC_CHECK_LONGEST]);
                }
                wide[VC_CHECK_BAD] = vc_wave_join_last<false>(bad);
            }
#pragma unroll
            for (int k = 0; k < VC_CHECK_WORDS; k++) sum[k] = k < VC_CHECK_MOST ? sum[k] + wide[k] : (wide[k] > sum[k] ? wide[k] : sum[k]);
        }
        // the packed receive layout is an int prefix sum of the rank's receive counts, like the reference's displacements
        if (PACKED && threadIdx.x == VC_WAVE - 1)
#pragma unroll
            for (int j = 0; j < R; j++)
                if (carry[j] > 0x7FFFFFFF && t0 + j < P) sum[VC_CHECK_BAD] += VC_BAD_OVERFLOW;
    }
    // the workgroup's, then, in the last workgroup, all of them: a wavefront adds up one of the words
    if (group < groups) {
        // (the last lane's sums are read by the whole wavefront: behind a branch that leaves that lane out they need not be complete)
        int64_t v = 0;
#pragma unroll
        for (int k = 0; k < VC_CHECK_WORDS; k++) { const int64_t x = vc_last_lane(sum[k]); v = lane == k ? x : v; }
        if (lane < VC_CHECK_MOST) atomicAdd(&of_group[lane], (unsigned long long)v);
        else if (lane < VC_CHECK_WORDS) atomicMax(&of_group[lane], (unsigned long long)v);
    }
    __syncthreads();
    if (group < groups && threadIdx.x < VC_CHECK_WORDS) vc_share(&group_tot[(int64_t)lane * groups + group], (int64_t)of_group[lane]);
    if (threadIdx.x < VC_WAVE) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the totals are where the last workgroup will look
    if (threadIdx.x == 0) is_last = vc_last_workgroup(ticket);
    __syncthreads();
    if (!is_last) return;
    for (int k = wave; k < VC_CHECK_WORDS; k += WAVES) {
        int64_t all = 0;
        for (int g0 = lane; g0 < groups; g0 += 4 * VC_WAVE) {      // (four reads on their way at once)
            int64_t v[4];
#pragma unroll
            for (int u = 0; u < 4; u++) v[u] = vc_shared(&group_tot[(int64_t)k * groups + (g0 + u * VC_WAVE < groups ? g0 + u * VC_WAVE : g0)]);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                if (g0 + u * VC_WAVE >= groups) v[u] = 0;
                all = k < VC_CHECK_MOST ? all + v[u] : (v[u] > all ? v[u] : all);
            }
        }
        all = k < VC_CHECK_MOST ? vc_wave_inclusive_scan(all) : vc_wave_max_last(all);
        // every staged block is one hop, every block's last hop ends in recvbuf
        const int to = k == VC_CHECK_PAYLOAD ? 1 : (k == VC_CHECK_MOVED ? VC_HEADER_FIXED : (k == VC_CHECK_BAD ? VC_HEADER_BAD :
                       (k == VC_CHECK_ITEMS ? 2 : (k == VC_CHECK_MOST ? VC_HEADER_MAX_PIECES : VC_HEADER_MAX_LEN))));
        if (lane == VC_WAVE - 1) { header[to] = all; header_host[to] = all; }
    }
    if (threadIdx.x == 0) { header[0] = stage_bytes; header_host[0] = stage_bytes; }
}

size_t vc_check_bytes(int P) { return sizeof(int64_t) * VC_CHECK_WORDS * (size_t)((P + VC_CHECK_RANKS - 1) / VC_CHECK_RANKS); }

hipError_t vc_launch_plan_check(const VcSched &S, VcTables T, int *rd_packed, int64_t *group_tot, int64_t stage_bytes, int64_t *header,
                                int64_t *header_host, unsigned *ticket, hipStream_t st) {
    const int groups = (S.P + VC_CHECK_RANKS - 1) / VC_CHECK_RANKS, grid = (groups + VC_PLAN_XCDS - 1) / VC_PLAN_XCDS * VC_PLAN_XCDS;
    // all sources in one round up to 1024 ranks
    const int threads = S.P <= 128 ? 128 : (S.P <= 256 ? 256 : (S.P <= 512 ? 512 : 1024));
    const auto packed = threads == 128 ? vc_plan_check<128, true> : (threads == 256 ? vc_plan_check<256, true> : (threads == 512 ? vc_plan_check<512, true> : vc_plan_check<1024, true>));
    const auto plain = threads == 128 ? vc_plan_check<128, false> : (threads == 256 ? vc_plan_check<256, false> : (threads == 512 ? vc_plan_check<512, false> : vc_plan_check<1024, false>));
    hipLaunchKernelGGL(S.packed_recv ? packed : plain, dim3(grid), dim3(threads), (size_t)(S.n + S.G), st, S, T, rd_packed, group_tot, stage_bytes,
                       (VC_CHUNK - VC_LINE + 1) / (unsigned)S.esz, VC_CHECK_SHORT / (unsigned)S.esz, header, header_host, ticket);
    return hipGetLastError();
}

// What a call that runs in batches of receivers has to know before the first of them: grid (P).
__global__ __launch_bounds__(VC_THREADS) void vc_receiver_staging_kernel(VcSched S, VcTables T, int64_t *__restrict__ staging) {
    __shared__ int64_t lds[VC_WAVES_PER_BLOCK];
    const int t = blockIdx.x;
    int64_t sum = 0;
    for (int s = threadIdx.x; s < S.P; s += VC_THREADS) sum += vc_block_staging(S, T, s, t);
    sum = vc_block_sum(sum, lds);
    if (threadIdx.x == 0) staging[t] = sum;
}

hipError_t vc_launch_receiver_staging(const VcSched &S, VcTables T, int64_t *staging, hipStream_t st) {
    hipLaunchKernelGGL(vc_receiver_staging_kernel, dim3(S.P), dim3(VC_THREADS), 0, st, S, T, staging);
    return hipGetLastError();
}

// The chain items: grid vc_rank_grid(P, chunks x slices).  The list is ordered in tiles of VC_TILE_RANKS receivers x VC_TILE_RANKS sources, receiver by
// receiver inside a tile; the sources come in chunks of VC_THREADS, and several workgroups share a chunk (each a whole number
// of tiles) when there are few ranks, which would otherwise leave most of the chip idle: the kernel is a chain of dependent
// table reads per workgroup, and one workgroup per compute unit hides none of them.
// The items of a tile's blocks are neighbours in the list: where there are no more than VC_EMIT_TILE_ITEMS of them they are put
// together in LDS and stored as whole cache lines (item by item a wavefront's store touches 64 places 40 bytes apart;
// 1 Mi items: 34 -> 26 us with that and the reads of all hops together).
// Blocks of many pieces are written by the whole workgroup, and `shares` workgroups share those of a slice.  512 ranks, 32 blocks of 256
// pieces each, nine hop slots, one of two batches: 460 us (an item a thread, its route worked out again for every piece) -> 86.
#define VC_EMIT_TILE_ITEMS 64
#define VC_EMIT_UNIT 256
#define VC_EMIT_GROUP 32
static_assert(VC_MAX_HOP_SLOTS <= VC_EMIT_GROUP, "a hop slot per lane");
// ROUTE: hop slots of a route kept in registers, 3 or 6 (two-layer calls and large radices have no more than 3, and the registers of 6
// would cost them a third of the wavefronts in flight); with more the route is worked out again for every piece.
#define VC_ROUTE_CACHE 6
static_assert(VC_TILE_RANKS * VC_ROUTE_CACHE <= VC_EMIT_TILE_ITEMS * (VC_CHAIN_HEAD + 1), "routes of a tile's big blocks in the place of its items");
// The last of VC_THREADS ascending numbers that is no larger than x (the first one is 0).
__device__ __forceinline__ int vc_last_at_or_below(const int64_t *of, int64_t x) {
    int lo = 0, hi = VC_THREADS - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (of[mid] <= x) lo = mid; else hi = mid - 1;
    }
    return lo;
}

template <int ROUTE>
__global__ __launch_bounds__(VC_THREADS) void vc_chain_emit(VcSched S, VcTables T, const uint32_t *__restrict__ slot_off,
                                                            const int64_t *__restrict__ row_base, const int64_t *__restrict__ chain_row_base,
                                                            const int64_t *__restrict__ tile_items, int nchunk, int slices,
                                                            int shares, int64_t *__restrict__ items, const int64_t *__restrict__ header,
                                                            int64_t cap_items) {
    // [tiles of the workgroup][VC_EMIT_TILE_ITEMS][stride]: a tile's items, or, in a tile with blocks of many pieces, the routes of
    // these, [VC_TILE_RANKS][ROUTE], while the whole workgroup writes their items
    extern __shared__ int64_t tile_lds[];
    __shared__ int64_t lds[VC_WAVES_PER_BLOCK];
    __shared__ int64_t big_at[VC_THREADS], big_pre[VC_THREADS];
    __shared__ int big_nhop[VC_THREADS];
    __shared__ int64_t field[VC_THREADS / VC_EMIT_GROUP][VC_CHAIN_HEAD + VC_MAX_HOP_SLOTS];
    const int P = S.P, ntile = VC_TILES(P), ranks_per_xcd = (P + VC_PLAN_XCDS - 1) / VC_PLAN_XCDS;
    // (part by part, the ranks of the XCD in each: ranks with work only in some of the parts keep every compute unit busy)
    const int at_xcd = blockIdx.x / VC_PLAN_XCDS, part = at_xcd / ranks_per_xcd, t = (int)(blockIdx.x % VC_PLAN_XCDS) * ranks_per_xcd + at_xcd % ranks_per_xcd;
    if (t >= P || !vc_receives_now(S, t)) return;
    const int stride = VC_CHAIN_HEAD + vc_hop_slots(S);
    const bool cached = vc_hop_slots(S) <= ROUTE;
    const int share_no = part / (nchunk * slices), chunk = part / slices % nchunk, z = part % slices;
    const int c_lo = chunk * VC_THREADS, c_hi = c_lo + VC_THREADS < P ? c_lo + VC_THREADS : P;
    const int slice = ((c_hi - c_lo + slices - 1) / slices + VC_TILE_RANKS - 1) / VC_TILE_RANKS * VC_TILE_RANKS;      // whole tiles
    const int s_lo = c_lo + z * slice < c_hi ? c_lo + z * slice : c_hi, s_hi = s_lo + slice < c_hi ? s_lo + slice : c_hi;
    if (s_lo >= s_hi) return;
    const int s = s_lo + threadIdx.x;                     // one source per lane: a slice has at most VC_THREADS of them
    // everything the items depend on is read before any of it is used: the pair's table entries, the slots of its hops (hop
    // slot k in slot[k], statically indexed), the tile counts below, the header
    const int64_t header_bad = header ? header[VC_HEADER_BAD] : 0, header_items = header ? header[2] : 0;
    const int nslots = vc_hop_slots(S), se = s < s_hi ? s : s_lo;
    const int count = vc_sc(S, T, se, t);
    const int64_t send_off = vc_send_offset(S, T, se, t), recv_off = vc_recv_offset(S, T, se, t);
    VcHop hop[ROUTE];
    int64_t slot_row[ROUTE];
    uint32_t slot_at[ROUTE];                              // added up later: a sum here would wait for its two reads
    VcWalk walk = vc_walk_start(S, se, t);
#pragma unroll
    for (int k = 0; k < ROUTE; k++) {
        slot_row[k] = slot_at[k] = 0;
        hop[k].moves = 0;
        if (!cached || k >= nslots) continue;
        hop[k] = vc_walk_step(S, walk, se, t, k);
        const int region_row = (k == nslots - 1 ? 0 : k) * P;      // (hop slot k's slots lie in region k; the last one has none)
        slot_row[k] = (row_base + region_row)[(unsigned)(hop[k].row - region_row)];
        slot_at[k] = (slot_off + (int64_t)region_row * P)[(unsigned)((hop[k].row - region_row) * P + hop[k].id)];
    }
    // first item of each of the workgroup's tiles: the items of all receivers before the tile row, of the tile row's tiles of
    // earlier sources, and of the receivers before t in the tile
    const int t0 = t / VC_TILE_RANKS * VC_TILE_RANKS, sb0 = s_lo / VC_TILE_RANKS, tiles = (s_hi - s_lo + VC_TILE_RANKS - 1) / VC_TILE_RANKS;
    constexpr int COLS = VC_THREADS / VC_TILE_RANKS;      // 8 tiles at most, a thread per (receiver of the tile row, tile)
    __shared__ int64_t share[VC_WAVES_PER_BLOCK][COLS];   // what a wavefront's receivers have before each of the workgroup's tiles
    const int64_t row_first = chain_row_base[t0];
    {
        const int row = threadIdx.x / COLS, col = threadIdx.x % COLS, lane = threadIdx.x % VC_WAVE;
        const bool there = t0 + row < P;
        const int64_t *of_row = tile_items + (int64_t)(t0 + row) * ntile;
        const int64_t here = there && col < tiles ? of_row[sb0 + col] : 0;
        int64_t earlier = 0;                              // (only with more than VC_THREADS ranks)
        for (int sb = col; sb < sb0; sb += COLS) earlier += there ? of_row[sb] : 0;
        int64_t whole = here, mine = t0 + row < t ? here : 0;
#pragma unroll
        for (int o = COLS; o < VC_WAVE; o <<= 1) {
            whole += __shfl_xor(whole, o, VC_WAVE);
            mine += __shfl_xor(mine, o, VC_WAVE);
            earlier += __shfl_xor(earlier, o, VC_WAVE);
        }
#pragma unroll
        for (int o = 1; o < COLS; o <<= 1) earlier += __shfl_xor(earlier, o, VC_WAVE);
        // lanes 0 .. COLS - 1: the tiles of the earlier columns
        int64_t before = vc_dpp_add<VC_DPP_SHR(1), 0xf>(whole);
        before = vc_dpp_add<VC_DPP_SHR(2), 0xf>(before);
        before = vc_dpp_add<VC_DPP_SHR(4), 0xf>(before) - whole;
        if (lane < COLS) share[threadIdx.x / VC_WAVE][lane] = before + mine + earlier;
    }
    __syncthreads();
    // a launch that was enqueued before the host had seen the plan: nothing is written unless the tables are in order
    // (their entries could point anywhere) and the list has room for every item
    if (header && (header_bad != 0 || header_items > cap_items)) return;
    const int64_t len = (int64_t)count * S.esz;
    const int cut = (int)((recv_off + S.recv_lo) & (VC_PIECE - 1)), phase = cut & (VC_LINE - 1);
    const int64_t cnt = s < s_hi ? vc_chunk_count(len, phase, cut) : 0;
    const int tile = threadIdx.x / VC_TILE_RANKS, lane_in_tile = threadIdx.x % VC_TILE_RANKS;
    const int64_t upto = vc_half_inclusive_scan(cnt), in_tile = __shfl(upto, VC_TILE_RANKS - 1, VC_TILE_RANKS);
    int64_t first = row_first;                            // the first item of the lane's tile
#pragma unroll
    for (int q = 0; q < VC_WAVES_PER_BLOCK; q++) first += share[q][tile];
    const int64_t at = first + upto - cnt;
    const bool big = cnt > 4;
    const bool any_big = (__ballot(big) >> (threadIdx.x % VC_WAVE / VC_TILE_RANKS * VC_TILE_RANKS) & 0xFFFFFFFFull) != 0;
    const bool together = cached && !any_big && in_tile <= VC_EMIT_TILE_ITEMS;
    int64_t *const tile_buf = tile_lds + (int64_t)tile * VC_EMIT_TILE_ITEMS * stride;
    const bool small = cnt > 0 && !big && share_no == 0;
    if (cached && (small || big)) {
        int64_t d[ROUTE];
        unsigned moves = 0;
#pragma unroll
        for (int k = 0; k < ROUTE; k++) {
            d[k] = vc_hop_dst(S, hop[k], slot_row[k] + vc_slot_bytes(slot_at[k]), recv_off);
            moves |= hop[k].moves ? 1u << k : 0u;
        }
        const int nhop = __popc(moves);
        if (!big) {
            const int64_t src = VC_SPACE_SEND | send_off;
            for (int64_t c = 0; c < cnt; c++) {
                int64_t lo, hi;
                vc_piece_range(len, phase, cut, c, lo, hi);
                int64_t *item = together ? tile_buf + (upto - cnt + c) * stride : items + (at + c) * stride;
                item[VC_CHAIN_SRC] = src + lo;
                item[VC_CHAIN_LEN] = hi - lo;
                item[VC_CHAIN_NHOP] = nhop;
                int n = 0;
#pragma unroll
                for (int k = 0; k < ROUTE; k++)
                    if (moves >> k & 1) item[VC_CHAIN_HEAD + n++] = d[k] + lo;
            }
        } else {
            big_nhop[threadIdx.x] = nhop;
            int n = 0;
#pragma unroll
            for (int k = 0; k < ROUTE; k++)
                if (moves >> k & 1) tile_buf[lane_in_tile * ROUTE + n++] = d[k];
        }
    } else if (small) {
        for (int64_t c = 0; c < cnt; c++) vc_chain_item(S, T, slot_off, row_base, s, t, c, items + (at + c) * stride);
    }
    big_at[threadIdx.x] = at;
    const bool wg_big = __syncthreads_or(big);            // (also: the tiles in LDS are complete)
    if (together && share_no == 0)
        for (int k = lane_in_tile; k < (int)in_tile * stride; k += VC_TILE_RANKS) items[first * stride + k] = tile_buf[k];
    if (!wg_big) return;
    if (cached) {                                         // an item a thread
        int64_t btotal;
        big_pre[threadIdx.x] = vc_block_exclusive_scan(big ? cnt : 0, lds, btotal);
        __syncthreads();
        for (int64_t q = share_no * VC_THREADS + threadIdx.x; q < btotal; q += shares * VC_THREADS) {
            const int b = vc_last_at_or_below(big_pre, q), sb = s_lo + b;
            vc_chain_piece(VC_SPACE_SEND | vc_send_offset(S, T, sb, t), (int64_t)vc_sc(S, T, sb, t) * S.esz, vc_phase(S, T, sb, t),
                           vc_chain_cut(S, T, sb, t), q - big_pre[b],
                           tile_lds + (int64_t)(b / VC_TILE_RANKS) * VC_EMIT_TILE_ITEMS * stride + b % VC_TILE_RANKS * ROUTE, big_nhop[b],
                           items + (big_at[b] + q - big_pre[b]) * stride);
        }
        return;
    }
    // With more hop slots than a thread keeps, half a wavefront takes VC_EMIT_UNIT pieces of a block at a time: a hop slot per lane, then
    // the items word by word, whole cache lines at once.
    int64_t units;
    big_pre[threadIdx.x] = vc_block_exclusive_scan(big ? (cnt + VC_EMIT_UNIT - 1) / VC_EMIT_UNIT : 0, lds, units);
    __syncthreads();
    const int lane = threadIdx.x % VC_EMIT_GROUP, group = threadIdx.x / VC_EMIT_GROUP, groups = VC_THREADS / VC_EMIT_GROUP;
    const int step_c = VC_EMIT_GROUP / stride, step_f = VC_EMIT_GROUP % stride;
    int64_t *const f_of = field[group];
    for (int64_t u = share_no * groups + group; u < units; u += shares * groups) {
        const int b = vc_last_at_or_below(big_pre, u), sb = s_lo + b;
        const int64_t to = vc_recv_offset(S, T, sb, t), from = vc_send_offset(S, T, sb, t), blen = (int64_t)vc_sc(S, T, sb, t) * S.esz;
        const VcHop h = vc_hop_place(S, sb, t, lane < nslots ? lane : 0);
        const int64_t dst = vc_hop_dst(S, h, vc_slot_addr(S, slot_off, row_base, h), to);
        const unsigned moves = (unsigned)(__ballot(lane < nslots && h.moves) >> (threadIdx.x % VC_WAVE - lane));
        const int bcut = (int)((to + S.recv_lo) & (VC_PIECE - 1)), nhop = __popc(moves), fields = VC_CHAIN_HEAD + nhop;
        if (lane == 0) { f_of[VC_CHAIN_SRC] = VC_SPACE_SEND | from; f_of[VC_CHAIN_LEN] = 0; f_of[VC_CHAIN_NHOP] = nhop; }
        if (moves >> lane & 1) f_of[VC_CHAIN_HEAD + __popc(moves & ((1u << lane) - 1))] = dst;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int64_t begin = (u - big_pre[b]) * VC_EMIT_UNIT, left = vc_chunk_count(blen, bcut & (VC_LINE - 1), bcut) - begin;
        const int words = (int)(left < VC_EMIT_UNIT ? left : VC_EMIT_UNIT) * stride;
        int64_t *const out = items + (big_at[b] + begin) * stride;
        int f = lane % stride;
        int64_t start = (begin + lane / stride) * VC_PIECE - bcut;      // of the piece inside the block (below 0: the first one's)
        for (int q = lane; q < words; q += VC_EMIT_GROUP) {
            const int64_t lo = start > 0 ? start : 0, hi = start + VC_PIECE < blen ? start + VC_PIECE : blen;
            if (f < fields) out[q] = f_of[f] + (f == VC_CHAIN_LEN ? hi - lo : (f == VC_CHAIN_NHOP ? 0 : lo));
            start += step_c * VC_PIECE; f += step_f;
            if (f >= stride) { f -= stride; start += VC_PIECE; }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();                  // (the fields are read before the next unit's take their place)
    }
}

hipError_t vc_launch_chain_plan(const VcSched &S, VcTables T, const uint32_t *slot_off, const int64_t *row_base,
                                const int64_t *chain_row_base, const int64_t *chain_row_tot, int64_t *items, int64_t nitems, hipStream_t st,
                                const int64_t *header, int64_t cap_items) {
    const int nchunk = (S.P + VC_THREADS - 1) / VC_THREADS;
    // at least ~1024 workgroups (four per compute unit), each a whole number of tiles of sources
    int slices = 1;
    while (nchunk == 1 && slices < 8 && (int64_t)S.P * slices < 1024 && S.P / (slices * 2) >= VC_TILE_RANKS) slices *= 2;
    // workgroups that share the long blocks of a slice: one per ~2048 items of an average slice, and of slices with 256 items or more as
    // many as bring the grid to that size
    const int64_t wgs = (int64_t)S.P * nchunk * slices, per_slice = nitems / wgs;
    const int shares = (int)std::min<int64_t>(64, std::max<int64_t>(1, std::max(per_slice / 2048, std::min(per_slice / 256, 1024 / wgs))));
    const int stride = VC_CHAIN_HEAD + vc_hop_slots(S), tiles = (std::min(S.P, VC_THREADS) + VC_TILE_RANKS - 1) / VC_TILE_RANKS;
    const size_t lds = vc_hop_slots(S) <= VC_ROUTE_CACHE ? sizeof(int64_t) * tiles * VC_EMIT_TILE_ITEMS * stride : 0;
    const auto kernel = vc_hop_slots(S) <= 3 ? vc_chain_emit<3> : vc_chain_emit<VC_ROUTE_CACHE>;
    hipLaunchKernelGGL(kernel, dim3(vc_rank_grid(S.P, nchunk * slices * shares)), dim3(VC_THREADS), lds, st, S, T, slot_off, row_base, chain_row_base,
                       chain_row_tot + 2 * (size_t)S.P, nchunk, slices, shares, items, header, cap_items);
    return hipGetLastError();
}

// ---- route inspection: bytes sent from every rank to every rank in one launch ----
__global__ __launch_bounds__(VC_THREADS) void vc_traffic_kernel(const VcDesc *__restrict__ desc, int64_t ndesc, int64_t *__restrict__ matrix, int P) {
    int64_t i = (int64_t)blockIdx.x * VC_THREADS + threadIdx.x;
    if (i >= ndesc) return;
    VcDesc d = desc[i];
    if (d.len > 0 && d.from >= 0)
        atomicAdd((unsigned long long *)&matrix[(int64_t)d.from * P + d.to], (unsigned long long)d.len);
}

hipError_t vc_launch_traffic(const VcDesc *desc, int64_t ndesc, int64_t *matrix, int P, hipStream_t st) {
    // a dispatch counts its grid in work-items in 32 bits: at most 2^24 - 1 workgroups of VC_THREADS per launch
    const int64_t step = (((int64_t)1 << 24) - 1) * VC_THREADS;
    for (int64_t done = 0; done < ndesc; done += step) {
        const int64_t now = ndesc - done < step ? ndesc - done : step;
        hipLaunchKernelGGL(vc_traffic_kernel, dim3((unsigned)((now + VC_THREADS - 1) / VC_THREADS)), dim3(VC_THREADS), 0, st, desc + done,
                           now, matrix, P);
    }
    return hipGetLastError();
}
