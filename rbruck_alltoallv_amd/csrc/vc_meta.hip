// vc_meta.hip — the caller-side metadata steps of the reference drivers as kernels
// (count-matrix exchange, displacement prefix sums, global maximum), plus the
// payload fill and the exact receiver-side check used by the harness.
#include <climits>

#include "vc_common.h"
#include "vc_scan.h"

// ---------------------------------------------------------------------------
// MPI_Alltoall of one int per pair (examples/rbruckv_example.cpp:76) is the
// transpose of the P x P count matrix.  32 x 32 tiles staged through LDS with a
// one-word pad so that both the row-wise load and the column-wise read are
// bank-conflict free; 256 threads move one tile (each 4 rows).
// ---------------------------------------------------------------------------
#define VC_TILE 32

__global__ __launch_bounds__(VC_THREADS) void vc_transpose_kernel(const int *__restrict__ in, int *__restrict__ out, int P, VcSignal sig) {
    __shared__ int tile[VC_TILE][VC_TILE + 1];
    const int tx = threadIdx.x % VC_TILE, ty = threadIdx.x / VC_TILE;   // ty in [0, 8)
    const int tiles = (P + VC_TILE - 1) / VC_TILE, c0 = (int)(blockIdx.x % tiles) * VC_TILE, r0 = (int)(blockIdx.x / tiles) * VC_TILE;
#pragma unroll
    for (int k = 0; k < VC_TILE; k += VC_THREADS / VC_TILE) {
        int r = r0 + ty + k, c = c0 + tx;
        if (r < P && c < P) tile[ty + k][tx] = in[(int64_t)r * P + c];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < VC_TILE; k += VC_THREADS / VC_TILE) {
        int r = c0 + ty + k, c = r0 + tx;                                // transposed coordinates
        if (r < P && c < P) vc_store_through(&out[(int64_t)r * P + c], tile[tx][ty + k]);
    }
    vc_signal(sig);
}

hipError_t vc_launch_transpose(const int *in, int *out, int P, hipStream_t st, VcSignal sig) {
    const unsigned t = (P + VC_TILE - 1) / VC_TILE;
    hipLaunchKernelGGL(vc_transpose_kernel, dim3(t * t), dim3(VC_THREADS), 0, st, in, out, P, sig);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Displacement prefix sums (examples/rbruckv_example.cpp:69-72,77-82): one
// workgroup per rank, wavefront scans combined through LDS, a running carry for
// rows longer than the workgroup.  Where the planner has them scanned (no signal) stores past the caches would not be needed; they cost
// nothing: 1024 ranks, 6 us either way.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(VC_THREADS) void vc_row_scan_kernel(const int *__restrict__ counts, int *__restrict__ displs,
                                                                 int64_t *__restrict__ extent, int *__restrict__ flags, int P, VcSignal sig) {
    __shared__ int64_t lds[VC_WAVES_PER_BLOCK];
    const int p = blockIdx.x;
    int64_t carry = 0;
    for (int base = 0; base < P; base += VC_THREADS) {
        int i = base + threadIdx.x;
        int64_t v = (i < P) ? counts[(int64_t)p * P + i] : 0, total;
        int64_t ex = vc_block_exclusive_scan(v, lds, total);
        if (i < P) vc_store_through(&displs[(int64_t)p * P + i], (int)(carry + ex));
        if (flags && v < 0) vc_store_through(&flags[1], 1);      // a negative count
        carry += total;
    }
    if (extent && threadIdx.x == 0) vc_store_through(&extent[p], carry);
    // the last displacement is the largest when no count is negative
    if (flags && threadIdx.x == 0 && carry > 0x7FFFFFFFll) vc_store_through(&flags[0], 1);
    if (sig.word) vc_signal(sig);
}

hipError_t vc_launch_row_scan(const int *counts, int *displs, int64_t *extent, int *flags, int P, hipStream_t st, VcSignal sig) {
    hipLaunchKernelGGL(vc_row_scan_kernel, dim3(P), dim3(VC_THREADS), 0, st, counts, displs, extent, flags, P, sig);
    return hipGetLastError();
}

// base[p] = sum_{q<p} roundup(extent[q]*esz, align); one workgroup.
__global__ __launch_bounds__(VC_THREADS) void vc_bases_kernel(const int64_t *__restrict__ extent, int esz, int64_t align,
                                                              int64_t *__restrict__ base, int64_t *__restrict__ total_out, int P, VcSignal sig) {
    __shared__ int64_t lds[VC_WAVES_PER_BLOCK];
    int64_t carry = 0;
    for (int b0 = 0; b0 < P; b0 += VC_THREADS) {
        int i = b0 + threadIdx.x;
        int64_t v = 0, total;
        if (i < P) v = (extent[i] * esz + align - 1) / align * align;
        int64_t ex = vc_block_exclusive_scan(v, lds, total);
        if (i < P) vc_store_through(&base[i], carry + ex);
        carry += total;
    }
    if (total_out && threadIdx.x == 0) vc_store_through(total_out, carry);
    vc_signal(sig);
}

hipError_t vc_launch_bases(const int64_t *extent, int esz, int64_t align, int64_t *base, int64_t *total, int P, hipStream_t st, VcSignal sig) {
    hipLaunchKernelGGL(vc_bases_kernel, dim3(1), dim3(VC_THREADS), 0, st, extent, esz, align, base, total, P, sig);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// MPI_Allreduce(MAX) of the block length (src/twophase_tunable_rbruckv.cpp:40-44).
// ---------------------------------------------------------------------------
// One launch: every workgroup leaves its maximum in state[1 + workgroup] and counts itself in state[0]; the last one takes
// the maximum of these and leaves the count at zero for the next call.  A clearing kernel in front of a maximum by atomics was
// one more launch, 4 us of a call of 18.  Atomics of many workgroups on one word go one after the other (256 of them twice: 4 us),
// so the workgroups are few and large.
#define VC_MAX_WORKGROUPS 64
#define VC_MAX_LANES 1024
__global__ __launch_bounds__(VC_MAX_LANES) void vc_max_kernel(const int *__restrict__ counts, int *__restrict__ out, int64_t n, int *state, VcSignal sig) {
    __shared__ int wave_max[VC_MAX_LANES / VC_WAVE];
    const int lane = threadIdx.x % VC_WAVE, wave = threadIdx.x / VC_WAVE;
    int m = INT_MIN;
#pragma unroll 8
    for (int64_t i = (int64_t)blockIdx.x * VC_MAX_LANES + threadIdx.x; i < n; i += (int64_t)gridDim.x * VC_MAX_LANES) m = max(m, counts[i]);
#pragma unroll
    for (int o = VC_WAVE / 2; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, VC_WAVE));
    if (lane == 0) wave_max[wave] = m;
    __syncthreads();
    if (wave != 0) return;
    m = lane < VC_MAX_LANES / VC_WAVE ? wave_max[lane] : INT_MIN;
#pragma unroll
    for (int o = VC_MAX_LANES / VC_WAVE / 2; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, VC_WAVE));
    int last = 0;
    if (lane == 0) {
        __hip_atomic_store(&state[1 + blockIdx.x], m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the store has been performed where the others will look
        last = __hip_atomic_fetch_add(&state[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1;
    }
    if (!__shfl(last, 0, VC_WAVE)) return;
    m = lane < (int)gridDim.x ? __hip_atomic_load(&state[1 + lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : INT_MIN;
#pragma unroll
    for (int o = VC_WAVE / 2; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, VC_WAVE));
    if (lane == 0) {
        vc_store_through(out, m);
        __hip_atomic_store(&state[0], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        vc_store_through(sig.word, sig.value);            // (this workgroup is the last one)
    }
}

hipError_t vc_launch_max(const int *counts, int *out, int64_t nelem, int *state, hipStream_t st, VcSignal sig) {
    int64_t blocks = (nelem + 4 * VC_MAX_LANES - 1) / (4 * VC_MAX_LANES);
    if (blocks > VC_MAX_WORKGROUPS) blocks = VC_MAX_WORKGROUPS;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(vc_max_kernel, dim3((unsigned)blocks), dim3(VC_MAX_LANES), 0, st, counts, out, nelem, state, sig);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Payload.  The reference drivers fill `i + rank*10` (examples/rbruckv_example.cpp:88-92);
// here every byte depends on source, destination and position.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t vc_splitmix64(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__device__ __forceinline__ uint64_t vc_hash4(uint64_t seed, uint64_t a, uint64_t b, uint64_t c) {
    uint64_t h = vc_splitmix64(seed + a);
    h = vc_splitmix64(h + b);
    return vc_splitmix64(h + c);
}

// gridDim.z workgroups per (source, destination) pair, each on its own slice of the block; a thread writes 8 bytes at
// a time.
static unsigned vc_slices_per_block(int P) {
    const int64_t z = (4ll << 20) / ((int64_t)P * P);      // about 4 Mi workgroups at most; many slices when P is small
    return (unsigned)(z < 1 ? 1 : (z > 64 ? 64 : z));
}

__global__ __launch_bounds__(VC_THREADS) void vc_fill_kernel(int mode, uint64_t seed, char *__restrict__ sendbuf,
                                                             const int *__restrict__ sc, const int *__restrict__ sd,
                                                             const int64_t *__restrict__ sbase, int esz, int P) {
    const int s = blockIdx.y, d = blockIdx.x;
    const int64_t len = (int64_t)sc[(int64_t)s * P + d] * esz;
    unsigned char *at = (unsigned char *)sendbuf + sbase[s] + (int64_t)sd[(int64_t)s * P + d] * esz;
    const int64_t nwords = (len + 7) >> 3;
    const int64_t per = (nwords + gridDim.z - 1) / gridDim.z;
    const int64_t kend = (blockIdx.z + 1) * per < nwords ? (blockIdx.z + 1) * per : nwords;
    for (int64_t k = blockIdx.z * per + threadIdx.x; k < kend; k += VC_THREADS) {
        uint64_t word;
        if (mode == 1) {
            uint64_t lo = ((uint64_t)s << 20) + ((uint64_t)d << 10) + (uint64_t)(2 * k);
            uint64_t hi = ((uint64_t)s << 20) + ((uint64_t)d << 10) + (uint64_t)(2 * k + 1);
            word = (lo & 0xFFFFFFFFull) | (hi << 32);
        } else {
            word = vc_hash4(seed, (uint64_t)s, (uint64_t)d, (uint64_t)k);
        }
        int64_t b0 = k << 3;
        int nb = (len - b0) < 8 ? (int)(len - b0) : 8;
        for (int q = 0; q < nb; q++) at[b0 + q] = (unsigned char)(word >> (8 * q));
    }
}

hipError_t vc_launch_fill_payload(int mode, uint64_t seed, char *sendbuf, const int *sc, const int *sd, const int64_t *sbase,
                                  int esz, int P, hipStream_t st) {
    hipLaunchKernelGGL(vc_fill_kernel, dim3(P, P, vc_slices_per_block(P)), dim3(VC_THREADS), 0, st, mode, seed, sendbuf, sc, sd, sbase, esz, P);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Exact check of the textbook definition recv_t[rdispls_t[s] + k] = send_s[sdispls_s[t] + k]
// (the reference's check, src/utils.cpp:31-46, only looks at a residue of each word).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(VC_THREADS) void vc_verify_kernel(const char *__restrict__ sendbuf, const char *__restrict__ recvbuf,
                                                               VcTables T, int esz, int P, int packed,
                                                               unsigned long long *__restrict__ mismatch) {
    __shared__ int64_t lds[VC_WAVES_PER_BLOCK];
    const int t = blockIdx.y, s = blockIdx.x;
    const int64_t len = (int64_t)T.sc[(int64_t)s * P + t] * esz;
    int64_t bad = 0;
    if (blockIdx.z == 0 && threadIdx.x == 0 && (int64_t)T.rc[(int64_t)t * P + s] * esz != len) bad = 1;     // the count exchange itself is wrong
    const int *rd = packed ? T.rd_packed : T.rd;
    const unsigned char *a = (const unsigned char *)sendbuf + T.sbase[s] + (int64_t)T.sd[(int64_t)s * P + t] * esz;
    const unsigned char *b = (const unsigned char *)recvbuf + T.rbase[t] + (int64_t)rd[(int64_t)t * P + s] * esz;
    const int64_t per = (len + gridDim.z - 1) / gridDim.z;
    const int64_t kend = (blockIdx.z + 1) * per < len ? (blockIdx.z + 1) * per : len;
    for (int64_t k = blockIdx.z * per + threadIdx.x; k < kend; k += VC_THREADS) bad += a[k] != b[k];
    bad = vc_block_sum(bad, lds);
    if (threadIdx.x == 0 && bad) atomicAdd(mismatch, (unsigned long long)bad);
}

hipError_t vc_launch_verify(const char *sendbuf, const char *recvbuf, VcTables t, int esz, int P, int packed,
                            unsigned long long *mismatch, hipStream_t st) {
    hipLaunchKernelGGL(vc_verify_kernel, dim3(P, P, vc_slices_per_block(P)), dim3(VC_THREADS), 0, st, sendbuf, recvbuf, t, esz, P, packed, mismatch);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Traffic model for choosing the radix.  For radix r = cand[c]: moved[c] = sum over all blocks of hops_r(s, t) *
// bytes(s, t) and moved[ncand + 1 + c] = sum of hops_r(s, t) * pieces(s, t), where hops = non-zero base-r digits of the
// (local) offset, plus one if the node differs, and 1 for a rank's block to itself; pieces = the 4 KiB work items a
// block is cut into.  moved[ncand] and moved[2 ncand + 1] receive the payload and the pieces of all blocks (one hop
// each).  grid (P, ncand + 1); the last row of workgroups adds up the radix-independent totals.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(VC_THREADS) void vc_hop_bytes_kernel(const int *__restrict__ sc, int esz, int P, int n, int ncand,
                                                                  const int *__restrict__ cand, unsigned long long *__restrict__ moved) {
    __shared__ int64_t lds[VC_WAVES_PER_BLOCK];
    const int s = blockIdx.x, c = blockIdx.y;
    const int r = c < ncand ? cand[c] : 0;                // r = 0: every block counts once
    int64_t acc = 0, items = 0;
    for (int t = threadIdx.x; t < P; t += VC_THREADS) {
        int hops = 1;
        if (r && s != t) {
            hops = (s / n != t / n) ? 1 : 0;
            for (int j = (s % n - t % n + n) % n; j; j /= r) hops += (j % r) != 0;
        }
        const int64_t len = (int64_t)sc[(int64_t)s * P + t] * esz;
        acc += hops * len;
        items += hops * (len <= VC_CHUNK ? (len > 0) : (len + VC_PIECE - 1) / VC_PIECE);
    }
    acc = vc_block_sum(acc, lds);
    items = vc_block_sum(items, lds);
    if (threadIdx.x == 0 && acc) atomicAdd(&moved[c], (unsigned long long)acc);
    if (threadIdx.x == 0 && items) atomicAdd(&moved[ncand + 1 + c], (unsigned long long)items);
}

hipError_t vc_launch_hop_bytes(const int *sc, int esz, int P, int n, const int *cand_dev, int ncand, unsigned long long *moved_dev,
                               hipStream_t st) {
    hipLaunchKernelGGL(vc_hop_bytes_kernel, dim3(P, ncand + 1), dim3(VC_THREADS), 0, st, sc, esz, P, n, ncand, cand_dev, moved_dev);
    return hipGetLastError();
}

// A kernel that does nothing: what one launch costs is measured with a row of these.
__global__ void vc_empty_kernel() {}

hipError_t vc_launch_empty(hipStream_t st) {
    hipLaunchKernelGGL(vc_empty_kernel, dim3(1), dim3(VC_WAVE), 0, st);
    return hipGetLastError();
}

// The last kernel of a blocking call: the kernels before it on the stream have ended, their stores released, when it runs.
// Waiting for its word in pinned host memory takes the host 4 us less than hipStreamSynchronize, which enqueues a barrier
// packet with a completion signal of its own behind the last kernel: a 5 us kernel launched and waited for 17.2 -> 13.2 us,
// three of them 30.6 -> 26.5 (a kernel launched with a stop event gained 1 - 2 us alone and lost as much behind another).
__global__ void vc_done_kernel(unsigned *word, unsigned value) {
    if (threadIdx.x == 0) __hip_atomic_store(word, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

hipError_t vc_launch_done(unsigned *word, unsigned value, hipStream_t st) {
    hipLaunchKernelGGL(vc_done_kernel, dim3(1), dim3(VC_WAVE), 0, st, word, value);
    return hipGetLastError();
}
