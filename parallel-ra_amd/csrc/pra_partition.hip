// Stable partition of device rows by bucket = tuple_hash(row[0:jcc]) % nb:
// the routing of input rows to their owner rank
// (buffer_data_to_hash_buffer_col, src/IO/parallel_io.cpp:239-297) and of the
// all-to-all tuple exchange (src/comm/all_to_allv_comm.cpp:64-142), as one
// on-device step: the output holds bucket 0's rows, then bucket 1's, ..., each
// bucket's rows in input order, and the bucket bounds.
//
// Three launches over tiles of PRA_PART_TILE rows:
//   k_part_hist     per tile, the rows of each bucket          -> H[b][tile]
//   k_part_scan     per bucket, exclusive prefix over tiles    -> H, T[b]
//   k_part_scatter  per tile, bucket starts (scan of T) + H, then every row to
//                   its place, through LDS in bucket order.
// Scratch: nb * tiles + nb u32 words (H then T); every word a call reads was
// written earlier in the same call, so the scratch carries no state between
// calls and needs no clearing.
//
// Algorithmic bytes per row: 8 * jcc (histogram) + 8 * (w + jcc) + 8 * w
// (scatter: key words again, the row read and written).
#include "pra_device.hpp"
#include "pra_partition.hpp"

#include <mutex>

namespace {

constexpr int kPartBlock = 256;
constexpr int kPartRounds = PRA_PART_TILE / kPartBlock;
constexpr int kScanBlock = 1024;
constexpr u32 kStreamRun = 1024;   // bytes

__device__ inline u32 part_bucket(const u64* __restrict__ row, int jcc, u32 nb)
{
    return pra_bucket(pra_fnv(row, jcc), nb);
}

__global__ __launch_bounds__(kPartBlock) void k_part_hist(const u64* __restrict__ rows, u64 n, int w, int jcc,
                                                           u32 nb, u32* __restrict__ H, u32 ntiles)
{
    __shared__ u32 h[PRA_RADIX];
    const u32 tid = threadIdx.x, tile = blockIdx.x;
    h[tid] = 0;
    __syncthreads();
    const u64 base = (u64)tile * PRA_PART_TILE;
    u32 b[kPartRounds];
#pragma unroll
    for (int r = 0; r < kPartRounds; r++) {
        const u64 i = base + (u64)r * kPartBlock + tid;
        b[r] = i < n ? part_bucket(rows + i * (u64)w, jcc, nb) : ~0u;
    }
#pragma unroll
    for (int r = 0; r < kPartRounds; r++) {
        // one LDS add per bucket and wave: a wave's lanes fall into few buckets
        const u64 peers = pra_match<PRA_RADIX_BITS>(b[r], __ballot(b[r] != ~0u));
        if (b[r] != ~0u && __lane_id() == (u32)(__ffsll((long long)peers) - 1)) atomicAdd(&h[b[r]], (u32)__popcll(peers));
    }
    __syncthreads();
    if (tid < nb) H[(u64)tid * ntiles + tile] = h[tid];
}

// block b: exclusive prefix of H[b][0..ntiles) in place, the total into T[b]
__global__ __launch_bounds__(kScanBlock) void k_part_scan(u32* __restrict__ H, u32 ntiles, u32* __restrict__ T)
{
    __shared__ u32 part[kScanBlock];
    const u32 tid = threadIdx.x;
    u32* h = H + (u64)blockIdx.x * ntiles;
    const u32 per = (ntiles + kScanBlock - 1) / kScanBlock;
    const u32 lo = tid * per, hi = min(ntiles, lo + per);
    u32 s = 0;
    for (u32 t = lo; t < hi; t++) s += h[t];
    part[tid] = s;
    __syncthreads();
    for (u32 d = 1; d < kScanBlock; d <<= 1) {   // inclusive Hillis-Steele scan of the chunk sums
        const u32 v = tid >= d ? part[tid - d] : 0;
        __syncthreads();
        part[tid] += v;
        __syncthreads();
    }
    u32 run = part[tid] - s;
    for (u32 t = lo; t < hi; t++) {
        const u32 v = h[t];
        h[t] = run;
        run += v;
    }
    if (tid == kScanBlock - 1) T[blockIdx.x] = part[tid];
}

// A tile's rows to their places, SUB rows at a time through LDS: the rows come
// in as consecutive words, are ranked in input order (inside each wave by
// matching bucket ballots, then over the waves), and go out in bucket order as
// consecutive words again, so both sides move whole cache lines where each
// lane's own row would touch several.  Tiles run from the last one back: the
// rows the histogram read last are still in the last-level cache.
// W: the row width, 0 = any (w).  NT: non-temporal stores.
// Whole partitions, queued one behind another, a lane to each row's words /
// this without the prefetch / with it: 24 M rows of 3 words into 8 buckets 482 /
// 360 / 345 us, 12 M of 6 into 64 739 / 463 / 419, 30 M of 2 into 200 800 / 560
// / 560, into 3 359 / 345 / 328, 1 M of 3 into 200 34.3 / 35.4 / 32.6; waited
// for, 300,000 of 5 into 3 42.4 / 45.4 / 36.5.  (A caller that waits for each
// has 10 us more: 356 us for the first.)  Large ones are bound by memory (the histogram reads every line, the
// scatter again: 24 bytes a word), those of less than a few tiles a compute
// unit by a tile's own chain of loads, ranks and stores, which the prefetch
// shortens.
// NT against plain stores: 377 / 402 us (8 buckets, runs of 1.5 KB), 483 / 463
// (64, 384 bytes), 854 / 561 (200, 41 bytes): kStreamRun lies in between.
template <int W, int SUB, bool NT>
__global__ __launch_bounds__(kPartBlock) void k_part_scatter(const u64* __restrict__ rows, u64 n, int w_, int jcc,
                                                              u32 nb, const u32* __restrict__ H,
                                                              const u32* __restrict__ T, u32 ntiles,
                                                              u64* __restrict__ out, u64* __restrict__ bounds)
{
    constexpr int IT = SUB / kPartBlock;
    extern __shared__ u64 stage[];   // SUB rows
    __shared__ u32 next[PRA_RADIX];        // where the bucket's next row goes
    __shared__ u32 wc[PRA_WAVES][PRA_RADIX];
    __shared__ u32 shift[PRA_RADIX];       // output row of a bucket's rows minus their place in the sub-tile
    __shared__ unsigned short perm[SUB];   // row of each place of the sub-tile
    __shared__ unsigned char pb[SUB];      // its bucket
    __shared__ u32 wsum[PRA_WAVES];
    const int w = W ? W : w_;
    const u32 tid = threadIdx.x, tile = gridDim.x - 1 - blockIdx.x;
    const u32 wave = tid / 64, lane = __lane_id();
    // exclusive scan over the buckets, a thread each
    auto scan = [&](u32 v) {
        u32 x = v;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const u32 y = __shfl_up(x, d, 64);
            if (lane >= (u32)d) x += y;
        }
        if (lane == 63) wsum[wave] = x;
        __syncthreads();
        for (u32 q = 0; q < wave; q++) x += wsum[q];
        __syncthreads();
        return x - v;
    };
    const u32 st = scan(tid < nb ? T[tid] : 0);
    if (tile == 0) {
        if (tid < nb) bounds[tid] = st;
        if (tid == 0) bounds[nb] = n;
    }
    next[tid] = tid < nb ? st + H[(u64)tid * ntiles + tile] : 0;
    const u64 t0 = (u64)tile * PRA_PART_TILE;
    const u32 trows = (u32)min((u64)PRA_PART_TILE, n - t0);
    // of a known width, the next sub-tile's words are loaded while this one's
    // rows are ranked and written
    constexpr int PF = W ? SUB * W / kPartBlock : 1;
    u64 pre[PF];
    auto fetch = [&](u32 s0) {
        const u32 words = s0 < trows ? min((u32)SUB, trows - s0) * W : 0;
        const u64* src = rows + (t0 + s0) * W;
#pragma unroll
        for (int k = 0; k < PF; k++) {
            const u32 i = tid + k * kPartBlock;
            pre[k] = i < words ? src[i] : 0;
        }
    };
    if (W) fetch(0);
    for (u32 s0 = 0; s0 < trows; s0 += SUB) {
        const u32 m = min((u32)SUB, trows - s0);
        if (W) {
#pragma unroll
            for (int k = 0; k < PF; k++)
                if (tid + k * kPartBlock < m * W) stage[tid + k * kPartBlock] = pre[k];
        } else {
            const u64* src = rows + (t0 + s0) * (u64)w;
            for (u32 i = tid; i < m * w; i += kPartBlock) stage[i] = src[i];
        }
#pragma unroll
        for (int q = 0; q < PRA_WAVES; q++) wc[q][tid] = 0;
        __syncthreads();
        if (W) fetch(s0 + SUB);
        // rows in input order: wave v holds rows [v * 64 * IT, (v + 1) * 64 * IT)
        u32 b[IT], rank[IT];
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const u32 i = wave * 64 * IT + k * 64 + lane;
            const bool valid = i < m;
            b[k] = valid ? part_bucket(stage + (size_t)i * w, jcc, nb) : 0;
            const u64 peers = pra_match<PRA_RADIX_BITS>(b[k], __ballot(valid));
            if (valid) {
                const u32 before = wc[wave][b[k]];
                rank[k] = before + (u32)__popcll(peers & pra_lanemask_lt());
                if ((peers >> lane) == 1ULL) wc[wave][b[k]] = before + (u32)__popcll(peers);
            }
        }
        __syncthreads();
        u32 tot = 0;
#pragma unroll
        for (int q = 0; q < PRA_WAVES; q++) {
            const u32 v = wc[q][tid];
            wc[q][tid] = tot;
            tot += v;
        }
        const u32 start = scan(tot);
        shift[tid] = next[tid] - start;
        next[tid] += tot;
#pragma unroll
        for (int q = 0; q < PRA_WAVES; q++) wc[q][tid] += start;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const u32 i = wave * 64 * IT + k * 64 + lane;
            if (i < m) {
                const u32 p = wc[wave][b[k]] + rank[k];
                perm[p] = (unsigned short)i;
                pb[p] = (unsigned char)b[k];
            }
        }
        __syncthreads();
        for (u32 i = tid; i < m * w; i += kPartBlock) {
            const u32 p = i / w, c = i - p * w;
            u64* dst = &out[(u64)(shift[pb[p]] + p) * w + c];
            const u64 v = stage[(u32)perm[p] * w + c];
            if (NT)
                __builtin_nontemporal_store(v, dst);
            else
                *dst = v;
        }
        __syncthreads();
    }
}

template <int W, int SUB>
void launch_scatter(hipStream_t st, const u64* rows, u64 n, int w, int jcc, u32 nb, const u32* H, const u32* T, u32 ntiles,
                    u64* out, u64* bounds)
{
    // a sub-tile's run of one bucket, at least kStreamRun bytes on average:
    // the runs are mostly whole lines, which need not stay in the caches
    const bool stream = (u64)SUB * w * 8 >= (u64)kStreamRun * nb;
    auto k = stream ? k_part_scatter<W, SUB, true> : k_part_scatter<W, SUB, false>;
    hipLaunchKernelGGL(k, dim3(ntiles), dim3(kPartBlock), (size_t)SUB * w * 8, st, rows, n, w, jcc, nb, H, T, ntiles, out,
                       bounds);
}

__global__ void k_part_empty(u64* bounds, u32 nb)
{
    const u32 t = threadIdx.x;
    if (t <= nb) bounds[t] = 0;
}

// The allocation-free entry point's scratch: one array per device, for the
// whole process, holding H and T of a partition of at most
// PRA_NOALLOC_MAX_ROWS rows into at most 256 buckets.
static __device__ __align__(256) u32 scratch[PRA_NOALLOC_SCRATCH_WORDS];

std::mutex g_scratch_mu;
u32* g_scratch_dev[PRA_MAX_DEVICES] = {};

} // namespace

u32 pra_partition_tiles(u64 n) { return (u32)((n + PRA_PART_TILE - 1) / PRA_PART_TILE); }

size_t pra_partition_scratch_words(u64 n, u32 nb) { return (size_t)nb * pra_partition_tiles(n) + nb; }

void pra_launch_partition(hipStream_t st, const u64* rows, u64 n, int w, int jcc, u32 nb, u64* out, u64* bounds,
                          u32* scratch_words)
{
    if (n == 0) {
        hipLaunchKernelGGL(k_part_empty, dim3(1), dim3(PRA_RADIX + 1), 0, st, bounds, nb);
        return;
    }
    const u32 ntiles = pra_partition_tiles(n);
    u32* H = scratch_words;
    u32* T = scratch_words + (size_t)nb * ntiles;
    hipLaunchKernelGGL(k_part_hist, dim3(ntiles), dim3(kPartBlock), 0, st, rows, n, w, jcc, nb, H, ntiles);
    hipLaunchKernelGGL(k_part_scan, dim3(nb), dim3(kScanBlock), 0, st, H, ntiles, T);
    // rows of a sub-tile: 512 (256, 1,024: 5 to 10 % slower at 2, 3 and 6
    // words a row), fewer where they would not leave room for two blocks a CU
    switch (w) {
    case 1: launch_scatter<1, 512>(st, rows, n, w, jcc, nb, H, T, ntiles, out, bounds); break;
    case 2: launch_scatter<2, 512>(st, rows, n, w, jcc, nb, H, T, ntiles, out, bounds); break;
    case 3: launch_scatter<3, 512>(st, rows, n, w, jcc, nb, H, T, ntiles, out, bounds); break;
    case 4: launch_scatter<4, 512>(st, rows, n, w, jcc, nb, H, T, ntiles, out, bounds); break;
    case 5: launch_scatter<5, 512>(st, rows, n, w, jcc, nb, H, T, ntiles, out, bounds); break;
    case 6: launch_scatter<6, 512>(st, rows, n, w, jcc, nb, H, T, ntiles, out, bounds); break;
    default:
        if (w <= 8)
            launch_scatter<0, 512>(st, rows, n, w, jcc, nb, H, T, ntiles, out, bounds);
        else
            launch_scatter<0, 256>(st, rows, n, w, jcc, nb, H, T, ntiles, out, bounds);
    }
}

// Once per device, with that device current: the device address of this
// device's copy of `scratch`.  Host code uses only this address, never the
// array's name (which names a host-side stand-in).
hipError_t pra_partition_scratch_init(int device)
{
    if (device < 0 || device >= PRA_MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_dev[device]) return hipSuccess;
    u32* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_dev[device] = ptr;
    return hipSuccess;
}

u32* pra_partition_scratch(int device)
{
    if (device < 0 || device >= PRA_MAX_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    return g_scratch_dev[device];
}
