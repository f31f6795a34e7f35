// HIP kernels of the semi-naive RA hot path for gfx950 (MI355X).
//
// Work is integer hashing, scanning, partitioning and sorting over rows of
// u64 words; it is HBM-bandwidth bound, so kernels stream rows in tiles of
// PRA_TILE rows per 256-thread workgroup (4 wave64s) and keep per-tile
// histograms in LDS.  Launch wrappers at the bottom are called by the host
// engine (pra_engine.cpp) on the context's stream.
#include "pra_device.hpp"
#include "pra_kernels.hpp"

// ------------------------------------------------------------------ utils --

__global__ void k_fill_u64(u64* p, u64 n, u64 v)
{
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 stride = (u64)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

// Table slots of `stride` words: [hash, minpos, key...]; empty = hash 0,
// minpos = all ones so that atomicMin by the first claimant wins.
__global__ void k_table_clear(u64* t, u64 cap, int stride)
{
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 step = (u64)gridDim.x * blockDim.x;
    for (; i < cap; i += step) {
        u64* s = t + i * stride;
        s[0] = 0;
        s[1] = ~0ULL;
        for (int c = 2; c < stride; c++) s[c] = 0;
    }
}

template <typename T, int NW = PRA_WAVES>
__device__ inline T block_exclusive_scan(T v, T* lds, T* total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    T x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        T y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) lds[wave] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        T acc = 0;
        for (int w = 0; w < NW; w++) {
            T t = lds[w];
            lds[w] = acc;
            acc += t;
        }
        lds[NW] = acc;
    }
    __syncthreads();
    T res = x - v + lds[wave];
    *total = lds[NW];
    __syncthreads();
    return res;
}

// ---------------------------------------------------- one-sweep LSD sort ---
//
// k_sort_hist counts the digits of every pass in one read of the rows;
// k_sort_scan turns them into per-pass digit offsets; one k_sort_scatter per
// pass then finds its tile's offset inside each digit by decoupled look-back
// over the preceding tiles' published counts (tiles are numbered in dispatch
// order, so a tile only ever waits on tiles that are already running).

__global__ void k_sort_hist(const u64* rows, u64 n, int w, PassList pl, u32* ghist)
{
    extern __shared__ u32 sh[];
    const int nbins = pl.np * PRA_RADIX;
    for (int i = threadIdx.x; i < nbins; i += PRA_BLOCK) sh[i] = 0;
    __syncthreads();
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 step = (u64)gridDim.x * blockDim.x;
    for (; i < n; i += step) {
        const u64* r = rows + i * w;
        for (int p = 0; p < pl.np; p++) atomicAdd(&sh[p * PRA_RADIX + pra_digit(r, pl.p[p])], 1u);
    }
    __syncthreads();
    for (int j = threadIdx.x; j < nbins; j += PRA_BLOCK)
        if (sh[j]) atomicAdd(&ghist[j], sh[j]);
}

// exclusive scan of each pass's digit counts; when `bnd` is given the last
// pass is the bucket digit and its offsets are the bucket bounds
__global__ void k_sort_scan(const u32* ghist, int np, u32* gofs, u64* bnd, u32 nb, u64 n)
{
    __shared__ u32 lds[PRA_WAVES + 1];
    for (int p = 0; p < np; p++) {
        u32 v = ghist[p * PRA_RADIX + threadIdx.x];
        u32 tot;
        u32 ex = block_exclusive_scan<u32>(v, lds, &tot);
        gofs[p * PRA_RADIX + threadIdx.x] = ex;
        if (bnd && p == np - 1) {
            if (threadIdx.x < nb) bnd[threadIdx.x] = ex;
            if (threadIdx.x == 0) bnd[nb] = n;
        }
    }
}

static_assert(PRA_BLOCK == PRA_RADIX, "look-back assigns one digit per thread");

__device__ inline u64 st_pack(u32 epoch, u64 flag, u64 cnt) { return ((u64)epoch << 48) | (flag << 46) | cnt; }

// Inclusive prefix of digit d over the tiles before `tile`: walks back over
// the predecessors' published counts, PRA_LOOKBACK predecessors per step with
// all their loads in flight, until an inclusive prefix is found.
__device__ inline u64 pra_lookback(const u64* status, u32 tile, int d, u32 epoch, u32* flags)
{
    u64 excl = 0;
    long long t = (long long)tile - 1;
    u32 spins = 0;
    while (t >= 0) {
        u64 v[PRA_LOOKBACK];
#pragma unroll
        for (int j = 0; j < PRA_LOOKBACK; j++)
            v[j] = t - j >= 0 ? __hip_atomic_load(status + (u64)(t - j) * PRA_RADIX + d, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT)
                              : 0;
        int used = 0;
        bool done = false, stall = false;
#pragma unroll
        for (int j = 0; j < PRA_LOOKBACK; j++) {
            if (done || stall || t - j < 0) continue;
            u64 fl = (v[j] >> 46) & 3ULL;
            if ((u32)(v[j] >> 48) != epoch || fl == 0) {
                stall = true;
                continue;
            }
            excl += v[j] & ((1ULL << 46) - 1);
            used = j + 1;
            if (fl == PRA_ST_INC) done = true;
        }
        if (done) break;
        t -= used;
        if (stall && ++spins > PRA_LOOKBACK_SPIN_LIMIT) {
            atomicOr(flags, PRA_FLAG_SORT_STALL);
            break;
        }
    }
    return excl;
}

template <bool IDX, int ITEMS>
__global__ void k_sort_scatter(const u64* in, u64* out, u64 n, int w, DigitSpec ds, const u32* gofs, u64* status,
                               u32* tile_ctr, u32 epoch, u32* flags, const u32* iin, u32* iout)
{
    constexpr u64 TILE = (u64)PRA_BLOCK * ITEMS;
    __shared__ u32 wh[PRA_WAVES][PRA_RADIX];
    __shared__ u32 s_base[PRA_RADIX];
    __shared__ u32 s_tile;
    if (threadIdx.x == 0) {
        // tiles are handed out in launch order; the block taking the last one
        // returns the counter to zero for the next launch
        u32 t = atomicAdd(tile_ctr, 1u);
        if (t == gridDim.x - 1) atomicExch(tile_ctr, 0u);
        s_tile = t;
    }
    for (int i = threadIdx.x; i < PRA_WAVES * PRA_RADIX; i += PRA_BLOCK) (&wh[0][0])[i] = 0;
    __syncthreads();
    const u32 tile = s_tile;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const u64 lt = pra_lanemask_lt();
    u64 base = (u64)tile * TILE + (u64)wave * (TILE / PRA_WAVES);
    u32 dg[ITEMS], lc[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
        u64 idx = base + (u64)k * 64 + lane;
        bool valid = idx < n;
        u32 d = valid ? pra_digit(in + idx * w, ds) : 0u;
        u64 act = __ballot(valid);
        u64 peers = pra_match<PRA_RADIX_BITS>(d, act);
        dg[k] = d;
        lc[k] = 0;
        if (valid) {
            u32 before = wh[wave][d];
            lc[k] = before + (u32)__popcll(peers & lt);
            if ((peers >> lane) == 1ULL) wh[wave][d] = before + (u32)__popcll(peers);
        }
    }
    __syncthreads();
    {
        const int d = threadIdx.x;   // PRA_BLOCK == PRA_RADIX: one digit per thread
        u32 acc = 0;
        for (int v = 0; v < PRA_WAVES; v++) {
            u32 t = wh[v][d];
            wh[v][d] = acc;
            acc += t;
        }
        u64* my = status + (u64)tile * PRA_RADIX + d;
        u64 excl = 0;
        if (tile == 0) {
            __hip_atomic_store(my, st_pack(epoch, PRA_ST_INC, acc), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            __hip_atomic_store(my, st_pack(epoch, PRA_ST_AGG, acc), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            excl = pra_lookback(status, tile, d, epoch, flags);
            __hip_atomic_store(my, st_pack(epoch, PRA_ST_INC, excl + acc), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
        s_base[d] = gofs[d] + (u32)excl;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
        u64 idx = base + (u64)k * 64 + lane;
        if (idx < n) {
            u64 pos = (u64)s_base[dg[k]] + wh[wave][dg[k]] + lc[k];
            const u64* src = in + idx * w;
            u64* dst = out + pos * w;
            pra_copy_row(dst, src, w);
            if (IDX) iout[pos] = iin ? iin[idx] : (u32)idx;
        }
    }
}

// ------------------------------------------------------ value dictionary ---
//
// An order-preserving dictionary of the values in the relations' key columns
// (rank(a) < rank(b) iff a < b) lets a newt row's sort key
// (bucket, col0, .., col[a-1]) be packed into one u64: the bucket and the
// column ranks as digits of radix D (the dictionary size), which the sort
// then orders in a few byte passes.
// Slots: [value, bucket-major rank << 32 | rank + 1]; 0 marks an empty slot.
// The bucket-major rank orders the values by (bucket of the value alone,
// value): as the leading digit of a relation keyed on its first column it puts
// rows in trie order, bucket first.

__device__ inline u64 pra_dict_slot(u64 v, u64 cap) { return pra_mix64(v ^ 0x5851F42D4C957F2DULL) & (cap - 1); }

// the slot word of a value, 0 when it has none
__device__ __forceinline__ u64 pra_dict_find(const u64* tab, u64 cap, u64 v)
{
    u64 m = cap - 1, s = pra_dict_slot(v, cap);
    for (u64 q = 0; q < cap; q++) {
        const ulonglong2 sl = *(const ulonglong2*)(tab + 2 * s);
        if (sl.y == 0 || sl.x == v) return sl.y;
        s = (s + 1) & m;
    }
    return 0;
}

__device__ inline bool pra_dict_rank(const u64* tab, u64 cap, u64 v, u64* rank)
{
    const u64 e = pra_dict_find(tab, cap, v);
    *rank = (u32)e - 1;
    return e != 0;
}

// ---------------------------------------------------------- LDS sorts ------

// LDS of a block that sorts up to BLOCK * IT (key, index) pairs
template <int BLOCK, int IT>
struct SortLds {
    u64 key[BLOCK * IT];
    u32 idx[BLOCK * IT];
    u32 wh[BLOCK / 64][PRA_RADIX];
    u32 wsum[PRA_RADIX / 64];
};

// One stable counting pass of the block's m pairs by the 8 key bits from
// `shift` up; thread t holds its pairs as items k of positions wave * 64 * IT
// + k * 64 + lane, before and after.  Leaves digit d's first position in
// L.wh[0][d] and the pairs in L.key / L.idx.
template <int BLOCK, int IT>
__device__ __forceinline__ void pra_lds_pass(SortLds<BLOCK, IT>& L, u64 (&key)[IT], u32 (&id)[IT], u32 m, int shift)
{
    constexpr int WAVES = BLOCK / 64;
    constexpr u32 PER_WAVE = 64 * IT;
    static_assert(BLOCK >= PRA_RADIX, "the digit scan takes a thread per digit");
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const u64 lt = pra_lanemask_lt();
    {
        for (int i = threadIdx.x; i < WAVES * PRA_RADIX; i += BLOCK) (&L.wh[0][0])[i] = 0;
        __syncthreads();
        // stable rank of every pair among the pairs of its digit: wave-local
        // counts in element order, then a scan over waves and digits
        u32 dg[IT], lc[IT];
#pragma unroll
        for (int k = 0; k < IT; k++) {
            u32 i = (u32)wave * PER_WAVE + (u32)k * 64 + lane;
            bool valid = i < m;
            dg[k] = 0;
            lc[k] = 0;
            // a wave skips the ranking of item rows wholly past the pairs
            if ((u32)wave * PER_WAVE + (u32)k * 64 >= m) continue;
            u32 d = valid ? (u32)(key[k] >> shift) & 255u : 0u;
            u64 peers = pra_match<PRA_RADIX_BITS>(d, __ballot(valid));
            dg[k] = d;
            if (valid) {
                u32 before = L.wh[wave][d];
                lc[k] = before + (u32)__popcll(peers & lt);
                if ((peers >> lane) == 1ULL) L.wh[wave][d] = before + (u32)__popcll(peers);
            }
        }
        __syncthreads();
        const int d = threadIdx.x;   // digit of this thread in the scan (threads < PRA_RADIX)
        u32 acc = 0;
        if (d < PRA_RADIX)
            for (int v = 0; v < WAVES; v++) {
                u32 t = L.wh[v][d];
                L.wh[v][d] = acc;
                acc += t;
            }
        u32 x = acc;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            u32 y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (d < PRA_RADIX && lane == 63) L.wsum[wave] = x;
        __syncthreads();
        if (d < PRA_RADIX) {
            u32 base = x - acc;
            for (int v = 0; v < wave; v++) base += L.wsum[v];
            for (int v = 0; v < WAVES; v++) L.wh[v][d] += base;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < IT; k++) {
            u32 i = (u32)wave * PER_WAVE + (u32)k * 64 + lane;
            if (i < m) {
                u32 pos = L.wh[wave][dg[k]] + lc[k];
                L.key[pos] = key[k];
                L.idx[pos] = id[k];
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < IT; k++) {
            u32 i = (u32)wave * PER_WAVE + (u32)k * 64 + lane;
            if (i < m) {
                key[k] = L.key[i];
                id[k] = L.idx[i];
            }
        }
        __syncthreads();
    }
}

// Pairs equal in the sixteen highest varying key bits are put in order by
// comparing each with its neighbours, up to this many to either side; a larger
// group leaves the block to LSD passes.
#define PRA_GROUP_MAX 32

// Stable LSD passes over the bytes set in `bytes` (bit p = byte p)
template <int BLOCK, int IT>
__device__ __forceinline__ void pra_lds_lsd(SortLds<BLOCK, IT>& L, u64 (&key)[IT], u32 (&id)[IT], u32 m, u32 bytes)
{
#pragma unroll 1
    for (int p = 0; p < 8; p++)
        if ((bytes >> p) & 1u) pra_lds_pass<BLOCK, IT>(L, key, id, m, 8 * p);
}

// The block's m pairs into key order, given the key bits in which they may
// differ: two counting passes over the sixteen highest of them, then every
// pair's place among its neighbours that share those bits (before(j, i): index
// j sorts before index i, their keys being equal).  The pairs of a block
// are few beside 2^16 digits, so most have no such neighbour: two passes (each
// five barriers and a digit scan, about 3 us) where LSD passes take one for
// each varying byte.  False, with the pairs permuted, when a group is over
// PRA_GROUP_MAX.
template <int BLOCK, int IT, typename F>
__device__ __forceinline__ bool pra_lds_group_sort(SortLds<BLOCK, IT>& L, u64 (&key)[IT], u32 (&id)[IT], u32 m,
                                                   u64 vary, u32* s_far, F before)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int hb = vary ? 63 - __clzll(vary) : 0, shift = hb > 15 ? hb - 15 : 0;
    if (threadIdx.x == 0) *s_far = 0;
    pra_lds_pass<BLOCK, IT>(L, key, id, m, shift);
    if (hb - shift >= 8) pra_lds_pass<BLOCK, IT>(L, key, id, m, shift + 8);
    int pos[IT];
    u32 far = 0, moved = 0;
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const int i = wave * 64 * IT + k * 64 + lane;
        pos[k] = i;
        if ((u32)i >= m) continue;
        const u64 g = key[k] >> shift;
        int r = i, steps = 0;
        for (int j = i - 1; j >= 0 && steps <= PRA_GROUP_MAX; j--, steps++) {
            const u64 kj = L.key[j];
            if ((kj >> shift) != g) break;
            if (kj > key[k] || (kj == key[k] && !before(L.idx[j], id[k], true))) r--;
        }
        far |= steps > PRA_GROUP_MAX;
        steps = 0;
        for (int j = i + 1; j < (int)m && steps <= PRA_GROUP_MAX; j++, steps++) {
            const u64 kj = L.key[j];
            if ((kj >> shift) != g) break;
            if (kj < key[k] || (kj == key[k] && before(L.idx[j], id[k], false))) r++;
        }
        far |= steps > PRA_GROUP_MAX;
        moved |= r != i;
        pos[k] = r;
    }
    if (far || moved) atomicOr(s_far, far ? 3u : 1u);
    __syncthreads();
    const u32 st = *s_far;
    if (st & 2) return false;
    if (!st) return true;
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const int i = wave * 64 * IT + k * 64 + lane;
        if ((u32)i < m) {
            L.key[pos[k]] = key[k];
            L.idx[pos[k]] = id[k];
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const int i = wave * 64 * IT + k * 64 + lane;
        if ((u32)i < m) {
            key[k] = L.key[i];
            id[k] = L.idx[i];
        }
    }
    __syncthreads();
    return true;
}

// Row sort keys: the varying bits of (bucket, col0, col1, ..) concatenated,
// most significant first, and cut into 64-bit words (word 0 the leading one,
// the last one padded with zeros below).  Comparing the words orders rows as
// comparing (bucket, columns) does, since the bits left out are the same in
// every row.
__device__ __forceinline__ u64 pra_key_word(const u64* row, const KeyLayout& L, int q, bool* miss)
{
    u64 out = 0;
    int at = 0;
    for (int j = 0; j < L.nf && at < 64 * (q + 1); j++) {
        const int bits = L.f[j].bits, end = at + bits - 64 * q;
        if (end > 0) {
            u64 v;
            if (L.f[j].col < 0)
                v = pra_bucket(pra_fnv(row, L.jcc), L.nb);
            else if (!L.f[j].rank)
                v = row[L.f[j].col] >> L.f[j].shift;
            else if (!pra_dict_rank(L.dict, L.dict_cap, row[L.f[j].col], &v))
                *miss = true;
            if (bits < 64) v &= (1ULL << bits) - 1;
            out |= end <= 64 ? v << (64 - end) : v >> (end - 64);
        }
        at += bits;
    }
    return out;
}

// bits in which the block's m keys differ
template <int BLOCK, int IT>
__device__ __forceinline__ u64 pra_block_vary(const u64 (&key)[IT], u32 m, u64* s_or, u64* s_and)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    u64 o = 0, a = ~0ULL;
#pragma unroll
    for (int k = 0; k < IT; k++)
        if ((u32)wave * 64 * IT + (u32)k * 64 + lane < m) {
            o |= key[k];
            a &= key[k];
        }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        o |= __shfl_xor(o, d, 64);
        a &= __shfl_xor(a, d, 64);
    }
    __syncthreads();
    if (lane == 0) {
        s_or[wave] = o;
        s_and[wave] = a;
    }
    __syncthreads();
    o = 0;
    a = ~0ULL;
    for (int v = 0; v < BLOCK / 64; v++) {
        o |= s_or[v];
        a &= s_and[v];
    }
    return m > 1 ? o ^ a : 0;
}

__device__ __forceinline__ u32 pra_vary_bytes(u64 vary)
{
    u32 bytes = 0;
    for (int p = 0; p < 8; p++)
        if ((vary >> (8 * p)) & 255) bytes |= 1u << p;
    return bytes;
}

// The block's m pairs (key word 0, row index) into the order of the rows'
// whole keys: by groups of word 0 when they are small, rows that share word 0
// compared by their later words; else by LSD passes over every word, the last
// word first.
// (later, when not null: words 1 .. nlater of row i's key at later[(q - 1) *
// BLOCK * IT + i]).  *dup, when not null, is set when two rows' keys are equal,
// and where the LSD passes did not look.
template <int BLOCK, int IT>
__device__ __forceinline__ void pra_lds_sort_rows(SortLds<BLOCK, IT>& S, const KeyLayout& L, const u64* rows, int w,
                                                  u64 (&key)[IT], u32 (&id)[IT], u32 m, u64* s_or, u64* s_and,
                                                  u32* s_max, u64* dup, const u64* later = nullptr, int nlater = 0)
{
    if (m < 2) return;
    bool same = false;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int words = (L.bits + 63) / 64;
    bool miss = false;   // ranks are used in keys of one word only
    const u64 vary = pra_block_vary<BLOCK, IT>(key, m, s_or, s_and);
    if (pra_lds_group_sort<BLOCK, IT>(S, key, id, m, vary, s_max, [&](u32 idj, u32 idi, bool equal_order) {
            for (int q = 1; q < words; q++) {
                const bool held = q <= nlater;
                const u64 a = held ? later[(q - 1) * BLOCK * IT + idj] : pra_key_word(rows + (u64)idj * w, L, q, &miss);
                const u64 b = held ? later[(q - 1) * BLOCK * IT + idi] : pra_key_word(rows + (u64)idi * w, L, q, &miss);
                if (a != b) return a < b;
            }
            same = true;
            return equal_order;   // equal rows keep their places
        })) {
        if (dup && same) *dup = 1;
        return;
    }
    if (dup && threadIdx.x == 0) *dup = 1;
    for (int q = words - 1; q >= 0; q--) {
        if (q || words > 1) {
#pragma unroll
            for (int k = 0; k < IT; k++)
                if ((u32)wave * 64 * IT + (u32)k * 64 + lane < m) key[k] = pra_key_word(rows + (u64)id[k] * w, L, q, &miss);
        }
        pra_lds_lsd<BLOCK, IT>(S, key, id, m, pra_vary_bytes(pra_block_vary<BLOCK, IT>(key, m, s_or, s_and)));
    }
}

// One block sorts n <= PRA_SMALL_SORT rows by (bucket, col0 .. col[kc-1]) (the
// bucket FNV(row[0:jcc]) % nb leads when `bucketed`; columns compare as
// unsigned words) and gathers them into `out`.  The key layout comes from the
// columns' varying bits, which the block collects first; equal rows keep
// their order.  With bnd (bucketed), bnd[s] = first row of bucket s, bnd[nb]
// = n.  BLOCK threads hold up to 2 * BLOCK rows.  Bound by barriers and the
// latency of a single block, so it takes two counting passes and a look at the
// neighbours instead of a network's log^2 steps, and 256 threads where they
// hold the rows.  1,300 edges of random 64-bit values in 8 buckets: 68 us as a
// bitonic network over multi-word keys, 32 us; 60 edges 16 -> 14 us.
template <int BLOCK>
__device__ __forceinline__ void pra_small_sort_block(const u64* rows, u64 n, int w, int jcc, int kc, u64 nb,
                                                     int bucketed, u64* out, u64* bnd, u64* dup)
{
    constexpr int IT = 2, LATER = 2;
    __shared__ SortLds<BLOCK, IT> S;
    __shared__ u64 later[LATER * BLOCK * IT];
    __shared__ KeyLayout L;
    __shared__ u64 s_or[BLOCK / 64], s_and[BLOCK / 64];
    __shared__ unsigned long long c_or[PRA_MAXW], c_and[PRA_MAXW];
    __shared__ u32 s_max;
    const u32 m = (u32)n;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x < PRA_MAXW) {
        c_or[threadIdx.x] = 0;
        c_and[threadIdx.x] = ~0ULL;
    }
    __syncthreads();
    for (int c = 0; c < kc; c++) {
        u64 o = 0, a = ~0ULL;
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const u32 i = (u32)wave * 64 * IT + (u32)k * 64 + lane;
            if (i < m) {
                const u64 v = rows[(u64)i * w + c];
                o |= v;
                a &= v;
            }
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            o |= __shfl_xor(o, d, 64);
            a &= __shfl_xor(a, d, 64);
        }
        if (lane == 0) {
            atomicOr(&c_or[c], (unsigned long long)o);
            atomicAnd(&c_and[c], (unsigned long long)a);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        L.nb = nb;
        L.jcc = jcc;
        L.nf = L.bits = 0;
        if (bucketed) pra_key_field(L, -1, 0, 64 - __clzll(nb - 1));
        for (int c = 0; c < kc; c++) {
            const u64 vary = c_or[c] ^ c_and[c];
            if (vary && m > 1) pra_key_field(L, c, __ffsll((long long)vary) - 1, 65 - __clzll(vary) - __ffsll((long long)vary));
        }
    }
    __syncthreads();
    u64 key[IT];
    u32 id[IT];
    bool miss = false;
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const u32 i = (u32)wave * 64 * IT + (u32)k * 64 + lane;
        key[k] = i < m ? pra_key_word(rows + (u64)i * w, L, 0, &miss) : 0;
        id[k] = i;
    }
    const int nlater = min(LATER, (L.bits + 63) / 64 - 1);
    for (int q = 1; q <= nlater; q++)
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const u32 i = (u32)wave * 64 * IT + (u32)k * 64 + lane;
            if (i < m) later[(q - 1) * BLOCK * IT + i] = pra_key_word(rows + (u64)i * w, L, q, &miss);
        }
    __syncthreads();
    pra_lds_sort_rows<BLOCK, IT>(S, L, rows, w, key, id, m, s_or, s_and, &s_max, dup, later, nlater);
    __syncthreads();
    const bool bounds = bnd && bucketed;
    const int bsh = 64 - (bucketed ? L.f[0].bits : 0);
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const u32 i = (u32)wave * 64 * IT + (u32)k * 64 + lane;
        if (i < m) {
            pra_copy_row(out + (u64)i * w, rows + (u64)id[k] * w, w);
            if (bounds) S.key[i] = key[k];
        }
    }
    if (bounds) {
        __syncthreads();
        for (u32 i = threadIdx.x; i <= m; i += BLOCK) {
            // buckets (prev, cur] start at row i
            const u64 prev = i == 0 ? 0 : (S.key[i - 1] >> bsh) + 1;
            const u64 cur = i == m ? nb : S.key[i] >> bsh;
            for (u64 s = prev; s <= cur && s <= nb; s++) bnd[s] = i;
        }
    }
}

template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_small_sort(const u64* rows, u64 n, int w, int jcc, int kc, u64 nb,
                                                      int bucketed, u64* out, u64* bnd, u64* dup)
{
    pra_small_sort_block<BLOCK>(rows, n, w, jcc, kc, nb, bucketed, out, bnd, dup);
}

// Independent small sorts (one per output relation of an iteration), one
// block each.
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_small_sort_many(SmallSortBatch b)
{
    const SmallSortJob& j = b.job[blockIdx.x];
    pra_small_sort_block<BLOCK>(j.rows, j.n, j.w, j.jcc, j.kc, b.nb, j.bucketed, j.out, j.bnd, nullptr);
}

// ------------------------------------------------------ keyed row sort -----
//
// Rows too many for one block: word 0 of every row's key and its index go
// through one or two counting passes over the key's top bytes, then each
// segment of equal top bits is sorted in LDS by its whole keys and its rows
// gathered.  A row is read once for its key and once by the gather (and again
// for later key words where rows of a segment share word 0), where byte
// passes over whole rows read and write it once per varying byte.  2 M rows of
// 4 words (19 varying bytes, 8 buckets): 1.77 ms of byte passes and
// histogram, 0.30 ms this way; 13,000 edges: 275 us in one block, 60 us.

// word 0 of the rows' keys, and the digit counts of its top np bytes (hist:
// np x 256, the pass over the lower byte first); a column value without a
// dictionary rank sets *missing
__global__ void k_sort_keys(const u64* rows, u64 n, int w, KeyLayout L, int np, u64* keys, u32* hist, u64* missing)
{
    bool miss = false;
    __shared__ u32 sh[2 * PRA_RADIX];
    for (int i = threadIdx.x; i < np * PRA_RADIX; i += PRA_BLOCK) sh[i] = 0;
    __syncthreads();
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    const u64 step = (u64)gridDim.x * blockDim.x;
    for (; i < n; i += step) {
        const u64 k = pra_key_word(rows + i * w, L, 0, &miss);
        keys[i] = k;
        atomicAdd(&sh[(np - 1) * PRA_RADIX + (u32)(k >> 56)], 1u);
        if (np == 2) atomicAdd(&sh[(u32)(k >> 48) & 255u], 1u);
    }
    if (miss) *missing = 1;
    __syncthreads();
    for (int j = threadIdx.x; j < np * PRA_RADIX; j += PRA_BLOCK)
        if (sh[j]) atomicAdd(&hist[j], sh[j]);
}

// Segment b of the pairs (seg: the segments' first positions, as
// k_seg_bounds leaves them, or the top byte's 256 digit offsets when seg is
// null) by a block of BLOCK threads.
template <int BLOCK>
__device__ __forceinline__ void pra_keyseg_sort(const u64* keys, const u32* idx, u64 start, u64 end, u64 n,
                                                const u64* rows, int w, const KeyLayout& L, u64* out, u64* bnd,
                                                u64* dup, const u32 b, const int top)
{
    constexpr int IT = PRA_BIN_ITEMS;
    __shared__ SortLds<BLOCK, IT> S;
    __shared__ u64 s_or[BLOCK / 64], s_and[BLOCK / 64];
    __shared__ u32 s_max, below;
    const int bbits = bnd ? L.f[0].bits : 0;
    const u64 nb = bnd ? L.nb : 1;
    if (bnd && b == 0 && threadIdx.x == 0) {
        bnd[0] = 0;
        bnd[nb] = n;
    }
    if (end <= start) {
        for (u64 s = 1 + threadIdx.x; s < nb; s += BLOCK)
            if (((s << (64 - bbits)) >> top) == b) bnd[s] = start;
        return;
    }
    const u32 m = (u32)(end - start);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    u64 key[IT];
    u32 id[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const u32 i = (u32)wave * 64 * IT + (u32)k * 64 + lane;
        key[k] = 0;
        id[k] = 0;
        if (i < m) {
            key[k] = keys[start + i];
            id[k] = idx[start + i];
        }
    }
    pra_lds_sort_rows<BLOCK, IT>(S, L, rows, w, key, id, m, s_or, s_and, &s_max, dup);
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const u32 i = (u32)wave * 64 * IT + (u32)k * 64 + lane;
        if (i < m) pra_copy_row(out + (start + i) * w, rows + (u64)id[k] * w, w);
    }
    for (u64 s = 1; s < nb; s++) {
        const u64 T = s << (64 - bbits);
        if ((T >> top) != b) continue;
        __syncthreads();
        if (threadIdx.x == 0) below = 0;
        __syncthreads();
        u32 cnt = 0;
#pragma unroll
        for (int k = 0; k < IT; k++)
            if ((u32)wave * 64 * IT + (u32)k * 64 + lane < m && key[k] < T) cnt++;
        if (cnt) atomicAdd(&below, cnt);
        __syncthreads();
        if (threadIdx.x == 0) bnd[s] = start + below;
    }
    __syncthreads();
}

// one block of 256 threads per segment of at most PRA_SEG_SMALL pairs
__global__ __launch_bounds__(PRA_BLOCK) void k_keyseg_small(const u64* keys, const u32* idx, const u64* seg,
                                                            const u32* gofs, int top, u64 n, const u64* rows, int w,
                                                            KeyLayout L, u64* out, u64* bnd, u64* status)
{
    const u32 b = blockIdx.x;
    const u64 start = seg ? seg[b] : gofs[b];
    const u64 end = seg ? seg[b + 1] : b + 1 < PRA_RADIX ? (u64)gofs[b + 1] : n;
    if (end - start > PRA_SEG_SMALL) return;
    pra_keyseg_sort<PRA_BLOCK>(keys, idx, start, end, n, rows, w, L, out, bnd, status + 1, b, top);
}

// the larger segments, by blocks that take every gridDim.x-th of them (list
// and count from k_seg_bounds; every segment in turn when seg is null); one
// over PRA_BIN_CAP pairs sets status[0] and is left unsorted
__global__ __launch_bounds__(PRA_BIN_BLOCK) void k_keyseg_large(const u64* keys, const u32* idx, const u64* seg,
                                                                const u32* gofs, const u32* list, const u64* stat,
                                                                int top, u64 n, const u64* rows, int w, KeyLayout L,
                                                                u64* out, u64* bnd, u64* status)
{
    const u64 cnt = seg ? stat[1] : PRA_RADIX;
    for (u64 i = blockIdx.x; i < cnt; i += gridDim.x) {
        const u32 b = seg ? list[i] : (u32)i;
        const u64 start = seg ? seg[b] : gofs[b];
        const u64 end = seg ? seg[b + 1] : b + 1 < PRA_RADIX ? (u64)gofs[b + 1] : n;
        if (end - start <= PRA_SEG_SMALL) continue;
        if (end - start > PRA_BIN_CAP) {
            if (threadIdx.x == 0) status[0] = 1;
            continue;
        }
        pra_keyseg_sort<PRA_BIN_BLOCK>(keys, idx, start, end, n, rows, w, L, out, bnd, status + 1, b, top);
    }
}

// One block sorts n <= PRA_BLOCK_SORT rows with all the LSD passes of `pl`
// (least significant first; digits from the rows, as k_sort_scatter's): the
// row indices stay in registers and LDS, every pass ranks them stably by
// wave-local counts and a scan over waves and digits, and the rows are
// gathered into `out` at the end.  With bnd, the last pass is the bucket
// digit and bnd[s] = first row of bucket s (FNV(row[0:jcc]) % nb), bnd[nb] = n.
__global__ __launch_bounds__(PRA_BIN_BLOCK) void k_block_sort(const u64* rows, u64 n, int w, PassList pl, u64* out,
                                                              u64* bnd, int jcc, u64 nb)
{
    constexpr int IT = PRA_BLOCK_SORT / PRA_BIN_BLOCK;
    constexpr int WAVES = PRA_BIN_BLOCK / 64;
    constexpr u32 PER_WAVE = PRA_BLOCK_SORT / WAVES;
    __shared__ u32 sidx[PRA_BLOCK_SORT];
    __shared__ u32 wh[WAVES][PRA_RADIX];
    __shared__ u32 wsum[PRA_RADIX / 64];
    const u32 m = (u32)n;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const u64 lt = pra_lanemask_lt();
    u32 id[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) id[k] = (u32)wave * PER_WAVE + (u32)k * 64 + lane;
#pragma unroll 1
    for (int p = 0; p < pl.np; p++) {
        const DigitSpec ds = pl.p[p];
        for (int i = threadIdx.x; i < WAVES * PRA_RADIX; i += PRA_BIN_BLOCK) (&wh[0][0])[i] = 0;
        __syncthreads();
        u32 dg[IT], lc[IT];
#pragma unroll
        for (int k = 0; k < IT; k++) {
            u32 i = (u32)wave * PER_WAVE + (u32)k * 64 + lane;
            bool valid = i < m;
            dg[k] = 0;
            lc[k] = 0;
            if ((u32)wave * PER_WAVE + (u32)k * 64 >= m) continue;   // item row wholly past the rows
            u32 d = valid ? pra_digit(rows + (u64)id[k] * w, ds) : 0u;
            u64 peers = pra_match<PRA_RADIX_BITS>(d, __ballot(valid));
            dg[k] = d;
            if (valid) {
                u32 before = wh[wave][d];
                lc[k] = before + (u32)__popcll(peers & lt);
                if ((peers >> lane) == 1ULL) wh[wave][d] = before + (u32)__popcll(peers);
            }
        }
        __syncthreads();
        const int d = threadIdx.x;   // digit of this thread in the scan (threads < PRA_RADIX)
        u32 acc = 0;
        if (d < PRA_RADIX)
            for (int v = 0; v < WAVES; v++) {
                u32 t = wh[v][d];
                wh[v][d] = acc;
                acc += t;
            }
        u32 x = acc;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            u32 y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (d < PRA_RADIX && lane == 63) wsum[wave] = x;
        __syncthreads();
        if (d < PRA_RADIX) {
            u32 base = x - acc;
            for (int v = 0; v < wave; v++) base += wsum[v];
            for (int v = 0; v < WAVES; v++) wh[v][d] += base;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < IT; k++) {
            u32 i = (u32)wave * PER_WAVE + (u32)k * 64 + lane;
            if (i < m) sidx[wh[wave][dg[k]] + lc[k]] = id[k];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < IT; k++) {
            u32 i = (u32)wave * PER_WAVE + (u32)k * 64 + lane;
            if (i < m) id[k] = sidx[i];
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < IT; k++) {
        u32 i = (u32)wave * PER_WAVE + (u32)k * 64 + lane;
        if (i < m) {
            const u64* src = rows + (u64)id[k] * w;
            u64* dst = out + (u64)i * w;
            pra_copy_row(dst, src, w);
        }
    }
    if (bnd) {
        // buckets (bucket of row i-1, bucket of row i] start at row i
        for (u32 i = threadIdx.x; i <= m; i += PRA_BIN_BLOCK) {
            const u64 prev = i == 0 ? 0 : pra_bucket(pra_fnv(rows + (u64)sidx[i - 1] * w, jcc), nb) + 1;
            const u64 cur = i == m ? nb : pra_bucket(pra_fnv(rows + (u64)sidx[i] * w, jcc), nb);
            for (u64 s = prev; s <= cur && s <= nb; s++) bnd[s] = i;
        }
    }
}

// bitwise OR and AND of column blockIdx.y over all rows, used to skip radix
// passes whose digit is the same for every row
__global__ void k_col_orand2(const u64* rows, u64 n, int w, u64* out /* [0..15] or, [16..31] and */)
{
    const int c = blockIdx.y;
    u64 o = 0, a = ~0ULL;
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 step = (u64)gridDim.x * blockDim.x;
    for (; i < n; i += step) {
        u64 v = rows[i * w + c];
        o |= v;
        a &= v;
    }
    for (int d = 32; d >= 1; d >>= 1) {
        o |= __shfl_xor(o, d, 64);
        a &= __shfl_xor(a, d, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicOr((unsigned long long*)&out[c], (unsigned long long)o);
        atomicAnd((unsigned long long*)&out[16 + c], (unsigned long long)a);
    }
}

// ------------------------------------------------- dictionary and views ---

__global__ void k_collect_cols(const u64* rows, u64 n, int w, int ncols, u64* out)
{
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    for (int c = 0; c < ncols; c++) out[i * ncols + c] = rows[i * w + c];
}

// keep[i] = 1 when row i falls in the same bucket under the hash of its first
// ja columns as under the hash of its first jb columns
__global__ void k_view_keep(const u64* rows, u64 n, int w, int ja, int jb, u64 nb, u32* keep)
{
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const u64* r = rows + i * w;
    keep[i] = pra_bucket(pra_fnv(r, ja), nb) == pra_bucket(pra_fnv(r, jb), nb) ? 1u : 0u;
}

// the kept rows, in order, at their exclusive-prefix positions
__global__ void k_view_compact(const u64* rows, u64 n, int w, const u32* keep, const u32* pos, u64* out)
{
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !keep[i]) return;
    const u64* r = rows + i * w;
    u64* o = out + (u64)pos[i] * w;
    for (int k = 0; k < w; k++) o[k] = r[k];
}

// values sorted and distinct: rank = position
__global__ void k_dict_insert(const u64* vals, u64 n, u64* tab, u64 cap, u32* flags)
{
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    u64 v = vals[i];
    u64 m = cap - 1, s = pra_dict_slot(v, cap);
    for (u64 q = 0; q < cap; q++) {
        u64* sl = tab + 2 * s;
        if (atomicCAS((unsigned long long*)(sl + 1), 0ULL, (unsigned long long)(i + 1)) == 0) {
            sl[0] = v;
            return;
        }
        s = (s + 1) & m;
    }
    atomicOr(flags, PRA_FLAG_TABLE_FULL);
}

// vals: the dictionary's values by (bucket, value); their places into the
// slots' high halves, the maps between places and ranks, and the places'
// buckets
__global__ void k_dict_bucket_rank(const u64* vals, u64 n, u64* tab, u64 cap, u32* rank_of, u32* lead_of, u64 nb,
                                   unsigned char* bucket)
{
    const u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const u64 v = vals[i], m = cap - 1;
    bucket[i] = (unsigned char)pra_bucket(pra_fnv_word(PRA_FNV_OFFSET, v), nb);
    u64 s = pra_dict_slot(v, cap);
    for (u64 q = 0; q < cap && tab[2 * s + 1]; q++) {
        if (tab[2 * s] == v) {
            const u32 r = (u32)tab[2 * s + 1] - 1;
            rank_of[i] = r;
            lead_of[r] = (u32)i;
            tab[2 * s + 1] |= i << 32;
            return;
        }
        s = (s + 1) & m;
    }
}

// The slot words of the rows' first a columns (a words a row), and, rows
// sorted by their leading digit, the first row of every digit value (D + 1
// words); a value without a rank is counted in *miss.
__device__ __forceinline__ void pra_rank_row(const RankRowsArgs& r, u64 i)
{
    if (i >= r.n) return;
    bool ok = true;
    u64 e0 = 0;
    for (int c = 0; c < r.a; c++) {
        const u64 e = pra_dict_find(r.dict, r.dict_cap, r.rows[i * r.w + c]);
        ok = ok && e != 0;
        r.words[i * r.a + c] = e;
        if (c == 0) e0 = e;
    }
    const u64 p0 = i ? pra_dict_find(r.dict, r.dict_cap, r.rows[(i - 1) * r.w]) : 0;
    if (!ok || (i && !p0)) {
        atomicAdd((unsigned long long*)r.miss, 1ULL);
        return;
    }
    const u64 mine = r.by_bucket ? e0 >> 32 : (u64)((u32)e0 - 1);
    const u64 prev = !i ? 0 : 1 + (r.by_bucket ? p0 >> 32 : (u64)((u32)p0 - 1));
    for (u64 d = prev; d <= mine; d++) r.first[d] = (u32)i;
    if (i + 1 == r.n)
        for (u64 d = mine + 1; d <= r.D; d++) r.first[d] = (u32)r.n;
}

__global__ void k_rank_rows(RankRowsArgs r) { pra_rank_row(r, (u64)blockIdx.x * blockDim.x + threadIdx.x); }

// out[i] = in[idx[i]] for rows of w words
__global__ void k_gather_rows(const u64* in, const u32* idx, u64 n, int w, u64* out)
{
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const u64* src = in + (u64)idx[i] * w;
    u64* dst = out + i * w;
    pra_copy_row(dst, src, w);
}

// Packed-key sort of the newt rows.  The newt scatter has put every row's
// (key, newt position) pair into the bin of the key's top byte (bin b holds
// its pairs, in no particular order, at bin_keys / bin_idx + b * bin_cap, and
// its rows go to [bofs[b], bofs[b + 1]) of the sorted order); block b orders
// its bin by the key's lower varying bytes (bit p of `bytes` = byte p varies,
// p < 7) with LSD passes in LDS, then gathers the rows into `out` in that
// order.  Keys are distinct, so the result is the total order.  A bin holds
// at most min(bin_cap, PRA_BIN_CAP) pairs; the host checks the largest bin
// before it launches this kernel (a larger one raises PRA_FLAG_BIN_OVERFLOW
// and is left unsorted).  Bucket s starts at the first key >= (s * bmul) <<
// ls (the key is bucket * bmul + column ranks, shifted left by ls); the block
// whose bin holds that value counts its keys below it.
// The sort of one bin (or segment) b by a block of BLOCK threads (at most
// BLOCK * PRA_BIN_ITEMS pairs): its pairs are keys[0..end-start) /
// idx[0..end-start), all with the same key bits from bit `top` up (the bin's
// value b), and its rows go to [start, end) of the sorted order.
template <int BLOCK>
__device__ __forceinline__ void pra_bin_sort_range(const u64* keys, const u32* idx, u64 start, u64 end, u32 cap, u64 n,
                                                   u32 bytes, const u64* rows, int w, u64* out, u64 bmul, int ls,
                                                   u64 nb, u64* bnd, u32* flags, const u32 b, const int top)
{
    constexpr int IT = PRA_BIN_ITEMS;
    constexpr u32 CAP = BLOCK * PRA_BIN_ITEMS;
    constexpr int WAVES = BLOCK / 64;
    constexpr u32 PER_WAVE = CAP / WAVES;
    __shared__ SortLds<BLOCK, IT> L;
    __shared__ u32 below;
    if (b == 0 && threadIdx.x == 0) {
        bnd[0] = 0;
        bnd[nb] = n;
    }
    if (end <= start) {
        for (u64 s = 1 + threadIdx.x; s < nb; s += BLOCK)
            if ((((s * bmul) << ls) >> top) == b) bnd[s] = start;
        return;
    }
    if (end - start > CAP || end - start > cap) {
        if (threadIdx.x == 0) atomicOr(flags, PRA_FLAG_BIN_OVERFLOW);
        return;
    }
    const u32 m = (u32)(end - start);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    u64 key[IT];
    u32 id[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        u32 i = (u32)wave * PER_WAVE + (u32)k * 64 + lane;
        key[k] = 0;
        id[k] = 0;
        if (i < m) {
            key[k] = keys[i];
            id[k] = idx[i];
        }
    }
    pra_lds_lsd<BLOCK, IT>(L, key, id, m, bytes);
    for (u64 s = 1; s < nb; s++) {
        const u64 T = (s * bmul) << ls;
        if ((T >> top) != b) continue;
        if (threadIdx.x == 0) below = 0;
        __syncthreads();
        u32 cnt = 0;
#pragma unroll
        for (int k = 0; k < IT; k++) {
            u32 i = (u32)wave * PER_WAVE + (u32)k * 64 + lane;
            if (i < m && key[k] < T) cnt++;
        }
        if (cnt) atomicAdd(&below, cnt);
        __syncthreads();
        if (threadIdx.x == 0) bnd[s] = start + below;
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < IT; k++) {
        u32 i = (u32)wave * PER_WAVE + (u32)k * 64 + lane;
        if (i < m) {
            const u64* src = rows + (u64)id[k] * w;
            u64* dst = out + (start + i) * w;
            pra_copy_row(dst, src, w);
        }
    }
}

// bin b of the newt scatter's top-byte bins (bofs = the bins' first sorted
// positions) by a block of BLOCK threads
template <int BLOCK>
__device__ __forceinline__ void pra_bin_sort_block(const u64* bin_keys, const u32* bin_idx, u32 bin_cap, u64 n,
                                                   const u32* bofs, u32 bytes, const u64* rows, int w, u64* out,
                                                   u64 bmul, int ls, u64 nb, u64* bnd, u32* flags, const u32 b)
{
    const u64 start = bofs[b], end = b + 1 < PRA_RADIX ? bofs[b + 1] : n;
    pra_bin_sort_range<BLOCK>(bin_keys + (u64)b * bin_cap, bin_idx + (u64)b * bin_cap, start, end, bin_cap, n,
                              bytes & 0x7Fu, rows, w, out, bmul, ls, nb, bnd, flags, b, 56);
}

// BLOCK threads per bin: the narrowest of 256, 512 and PRA_BIN_BLOCK whose
// BLOCK * PRA_BIN_ITEMS pairs hold the largest bin (a wave holds 512 of a
// bin's pairs, so small bins leave most waves of a wide block without items,
// and every wave still takes part in each pass's barriers and digit scan)
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_bin_sort(const u64* bin_keys, const u32* bin_idx, u32 bin_cap, u64 n,
                                                    const u32* bofs, u32 bytes, const u64* rows, int w, u64* out,
                                                    u64 bmul, int ls, u64 nb, u64* bnd, u32* flags)
{
    pra_bin_sort_block<BLOCK>(bin_keys, bin_idx, bin_cap, n, bofs, bytes, rows, w, out, bmul, ls, nb, bnd, flags,
                              blockIdx.x);
}

// The bin sorts of several outputs in one launch: block b sorts bin b % 256
// of job b / 256 (job table in device memory).
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_bin_sort_many(const BinSortJob* jobs, u32* flags)
{
    const BinSortJob& j = jobs[blockIdx.x / PRA_RADIX];
    pra_bin_sort_block<BLOCK>(j.bin_keys, j.bin_idx, j.bin_cap, j.n, j.bofs, j.bytes, j.rows, j.w, j.out, j.bmul, j.ls,
                              j.nb, j.bnd, flags, blockIdx.x % PRA_RADIX);
}

// Segmented form for newts too large for the top-byte bins: the pairs are
// already ordered by the keys' top 16 bits (two counting passes), segment b
// is the pairs whose key bits from `top` up equal b ([seg[b], seg[b + 1])),
// and block b sorts it by the varying bytes below (bit p of `bytes`).
// Block i sorts segment list[i] (list null: segment i, skipping a segment
// of more than skip_above pairs, which a launch over the list sorts).
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_seg_sort(const u64* keys, const u32* idx, const u64* seg, int top, u64 n,
                                                    u32 bytes, const u64* rows, int w, u64* out, u64 bmul, int ls,
                                                    u64 nb, u64* bnd, u32* flags, const u32* list, u32 skip_above)
{
    const u32 b = list ? list[blockIdx.x] : blockIdx.x;
    const u64 start = seg[b], end = seg[b + 1];
    if (end - start > skip_above) return;
    pra_bin_sort_range<BLOCK>(keys + start, idx + start, start, end, BLOCK * PRA_BIN_ITEMS, n, bytes, rows, w, out,
                              bmul, ls, nb, bnd, flags, b, top);
}

// seg[v] = first position of a sorted key array whose bits from `top` up are
// >= v, for v in [0, nseg] (seg[nseg] = n); stat[0] = the largest segment,
// and the stat[1] segments of more than PRA_SEG_SMALL pairs are listed in
// large (in no particular order)
__global__ void k_seg_bounds(const u64* keys, u64 n, int top, u32 nseg, u64* seg, u64* stat, u32* large)
{
    const u64 v = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nseg) return;
    u64 b2[2];
    for (int k = 0; k < 2; k++) {
        const u64 t = v + (u64)k;
        if (t >= nseg) {
            b2[k] = n;
            continue;
        }
        u64 lo = 0, hi = n;
        while (lo < hi) {
            const u64 mid = (lo + hi) >> 1;
            if ((keys[mid] >> top) < t) lo = mid + 1; else hi = mid;
        }
        b2[k] = lo;
    }
    seg[v] = b2[0];
    if (v + 1 == nseg) seg[nseg] = n;
    const u64 size = b2[1] - b2[0];
    atomicMax((unsigned long long*)stat, (unsigned long long)size);
    if (size > PRA_SEG_SMALL) large[atomicAdd((unsigned long long*)(stat + 1), 1ULL)] = (u32)v;
}

// bnd[s] = first position whose key is >= (s * bmul) << ls (the key is
// bucket * bmul + column ranks, shifted left by ls)
__global__ void k_key_bounds(const u64* keys, u64 n, u64 bmul, int ls, u64 nb, u64* bnd)
{
    u64 s = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (s > nb) return;
    if (s == nb) {
        bnd[s] = n;
        return;
    }
    const u64 T = (s * bmul) << ls;
    u64 lo = 0, hi = n;
    while (lo < hi) {
        u64 mid = (lo + hi) >> 1;
        if (keys[mid] < T) lo = mid + 1; else hi = mid;
    }
    bnd[s] = lo;
}

// order-sensitive checksum of rows: sum over i of hash(row i, i)
__global__ void k_rows_checksum(const u64* rows, u64 n, int w, u64* out)
{
    __shared__ u64 red[PRA_WAVES];
    u64 acc = 0;
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 step = (u64)gridDim.x * blockDim.x;
    for (; i < n; i += step) acc += pra_mix64(pra_keyhash(rows + i * w, w) ^ pra_mix64(i + 0x2545F4914F6CDD1DULL));
    for (int d = 32; d >= 1; d >>= 1) acc += __shfl_xor(acc, d, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        u64 t = 0;
        for (int v = 0; v < PRA_WAVES; v++) t += red[v];
        atomicAdd((unsigned long long*)out, (unsigned long long)t);
    }
}

// bstart[s] = first row whose bucket is >= s, for s in [0, nb]
__global__ void k_bucket_bounds(const u64* rows, u64 n, int w, int jcc, u64 nb, u64* bstart)
{
    u64 s = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (s > nb) return;
    u64 lo = 0, hi = n;
    while (lo < hi) {
        u64 mid = (lo + hi) >> 1;
        u64 b = pra_bucket(pra_fnv(rows + mid * w, jcc), nb);
        if (b < s) lo = mid + 1; else hi = mid;
    }
    bstart[s] = lo;
}

// keep rows whose flag is set, in order
__global__ void k_compact_rows(const u64* in, u64 n, int w, const u64* flags, const u64* pos, u64* out)
{
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !flags[i]) return;
    const u64* src = in + i * w;
    u64* dst = out + pos[i] * w;
    pra_copy_row(dst, src, w);
}

// ------------------------------------------------------- join index --------

__global__ void k_group_flags(const u64* rows, u64 n, int w, int jcc, u64* flags)
{
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    u64 f = 1;
    if (i > 0) {
        f = 0;
        const u64* a = rows + i * w;
        const u64* b = a - w;
        for (int c = 0; c < jcc; c++)
            if (a[c] != b[c]) { f = 1; break; }
    }
    flags[i] = f;
}

__global__ void k_group_compact(const u64* flags, const u64* gpos, u64 n, u64* gstart)
{
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i > n) return;
    if (i == n) {
        gstart[n == 0 ? 0 : gpos[n - 1] + flags[n - 1]] = n;
        return;
    }
    if (flags[i]) gstart[gpos[i]] = i;
}

// longest group (largest number of rows sharing a key) of a sorted version
__global__ void k_group_maxlen(const u64* flags, const u64* gpos, const u64* gstart, u64 n, u64* maxlen)
{
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !flags[i]) return;
    u64 len = gstart[gpos[i] + 1] - i;
    atomicMax((unsigned long long*)maxlen, (unsigned long long)len);
}

// index slots: [hash, start row, row count]
__global__ void k_index_insert(const u64* rows, int w, int jcc, const u64* gstart, u64 ng, u64* table, u64 cap,
                               u32* flags)
{
    u64 g = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    u64 i0 = gstart[g], cnt = gstart[g + 1] - i0;
    u64 h = pra_keyhash(rows + i0 * w, jcc);
    u64 m = cap - 1, s = h & m;
    for (u64 p = 0; p < cap; p++) {
        u64* slot = table + s * 3;
        u64 prev = atomicCAS((unsigned long long*)slot, 0ULL, (unsigned long long)h);
        if (prev == 0) {
            slot[1] = i0;
            slot[2] = cnt;
            return;
        }
        if (prev == h) {
            atomicOr(flags, PRA_FLAG_INDEX_COLLISION);
            return;
        }
        s = (s + 1) & m;
    }
    atomicOr(flags, PRA_FLAG_TABLE_FULL);
}

// ------------------------------------------------- setup in one block ------

// Sort an array of P words (a power of two) in LDS, in place (bitonic network).
// Lane l of wave v exchanges within words 128 v .. 128 v + 127 (and the same
// 2,048 further on, block after block) while the distance is below 128, so
// only longer exchanges, and the step into one, meet at a barrier: 18 barriers
// instead of 78 at 4,096 words.
template <typename T>
__device__ __forceinline__ void pra_lds_bitonic(T* a, u32 P)
{
    for (u32 k = 2; k <= P; k <<= 1)
        for (u32 j = k >> 1; j; j >>= 1) {
            for (u32 t = threadIdx.x; t < P / 2; t += blockDim.x) {
                const u32 i = ((t & ~(j - 1)) << 1) | (t & (j - 1)), o = i | j;
                const T x = a[i], y = a[o];
                if ((x > y) == ((i & k) == 0)) {
                    a[i] = y;
                    a[o] = x;
                }
            }
            if (j >= 128 || (j == 1 && k >= 128)) {
                __syncthreads();
            } else {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
    __syncthreads();
}

__device__ __forceinline__ void pra_publish_words(const u64* src, u64 words, const u32* flags, u64* host, u64 seq);

// An instance's dictionary in one launch: the distinct values of the columns
// (an LDS table), sorted, with their bucket-major order (a second LDS sort of
// bucket << 16 | rank), into the maps and the probed table, and the number of
// values to the host.  ~0 when there are more than PRA_DICT_SMALL, with
// nothing written: the general build then sorts all of them.
// Bound by the latency of its LDS sorts; one compute unit works, but the
// general build is a dozen dependent launches and two waits: with this, the
// one-block index (k_index_small) and waits on published words, 60 programs of
// 200-1,500 vertices in one context took 28.5 ms instead of 36.1; one block an
// instance in one launch and one wait for all of them (k_dict_small_many,
// k_index_small_many), 16.3.
__device__ __forceinline__ void pra_dict_small(const DictSmallArgs& a)
{
    __shared__ u64 tab[2 * PRA_DICT_SMALL];
    __shared__ u64 sv[PRA_DICT_SMALL];
    __shared__ u32 lk[PRA_DICT_SMALL];
    __shared__ u32 count, top, kept;
    __shared__ u64 result;
    constexpr u32 M = 2 * PRA_DICT_SMALL - 1;
    const u32 t = threadIdx.x;
    for (u32 i = t; i <= M; i += 1024) tab[i] = ~0ULL;
    if (t == 0) count = top = kept = 0;
    for (u64 i = t; i < 2 * a.cap; i += 1024) a.dict[i] = 0;
    __syncthreads();
    // distinct values (~0 marks an empty slot; that value is kept aside).
    // Insertions end when more than PRA_DICT_SMALL are counted: at most one
    // more a thread, so an empty slot is always left.
    for (int s = 0; s < a.k; s++) {
        const u64* rows = a.rows[s];
        const u32 ar = (u32)a.arity[s], total = a.n[s] * ar;
        for (u32 j = t; j < total; j += 1024) {
            const u64 v = rows[(u64)(j / ar) * (u64)a.w[s] + j % ar];
            if (v == ~0ULL) {
                top = 1;
                continue;
            }
            u32 h = (u32)pra_dict_slot(v, M + 1);
            for (u32 q = 0; q <= M; q++, h = (h + 1) & M) {
                u64 cur = ((volatile u64*)tab)[h];
                if (cur == ~0ULL) {
                    if (*(volatile u32*)&count > PRA_DICT_SMALL) break;
                    cur = atomicCAS((unsigned long long*)&tab[h], ~0ULL, (unsigned long long)v);
                    if (cur == ~0ULL) {
                        atomicAdd(&count, 1u);
                        break;
                    }
                }
                if (cur == v) break;
            }
        }
    }
    __syncthreads();
    const u32 U = count + top;
    if (t == 0) result = U > PRA_DICT_SMALL ? ~0ULL : U;
    if (U <= PRA_DICT_SMALL) {
        u32 P = 2;
        while (P < U) P <<= 1;
        for (u32 i = t; i < P; i += 1024) sv[i] = ~0ULL;
        __syncthreads();
        for (u32 i = t; i <= M; i += 1024)
            if (tab[i] != ~0ULL) sv[atomicAdd(&kept, 1u)] = tab[i];
        __syncthreads();
        pra_lds_bitonic(sv, P);
        u32* lead = (u32*)tab;   // bucket-major rank of every rank
        if (a.nb > 1) {
            for (u32 i = t; i < P; i += 1024)
                lk[i] = i < U ? (u32)pra_bucket(pra_fnv_word(PRA_FNV_OFFSET, sv[i]), a.nb) << 16 | i : ~0u;
            __syncthreads();
            pra_lds_bitonic(lk, P);
            for (u32 i = t; i < U; i += 1024) {
                const u32 r = lk[i] & 0xFFFF;
                lead[r] = i;
                a.rank_of[i] = r;
                a.lead_of[r] = i;
                a.lead_vals[i] = sv[r];
                a.lead_bucket[i] = (unsigned char)(lk[i] >> 16);
            }
            __syncthreads();
        }
        for (u32 r = t; r < U; r += 1024) {
            const u64 v = sv[r], word = (a.nb > 1 ? (u64)lead[r] << 32 : 0) | (r + 1);
            a.vals[r] = v;
            const u64 m = a.cap - 1;
            u64 s = pra_dict_slot(v, a.cap), q = 0;
            for (; q < a.cap; q++, s = (s + 1) & m)
                if (atomicCAS((unsigned long long*)(a.dict + 2 * s + 1), 0ULL, (unsigned long long)word) == 0) {
                    a.dict[2 * s] = v;
                    break;
                }
            if (q == a.cap) atomicOr(a.err, PRA_FLAG_TABLE_FULL);
        }
    }
    __threadfence();
    __syncthreads();
    if (a.host)
        pra_publish_words(&result, 1, a.err, a.host, a.seq);
    else if (t == 0)
        *a.out = result;
}

__global__ __launch_bounds__(1024) void k_dict_small(DictSmallArgs a) { pra_dict_small(a); }

__global__ __launch_bounds__(1024) void k_dict_small_many(const DictSmallArgs* jobs) { pra_dict_small(jobs[blockIdx.x]); }

// The join index of a sorted version of at most PRA_INDEX_SMALL rows in one
// launch: the runs of equal keys, their longest, and the table, sized for the
// runs as the general build sizes it (longest run and number of runs to the
// host).  The general build is eight launches and two waits.
__device__ __forceinline__ void pra_index_small(const IndexSmallArgs& a)
{
    __shared__ u32 gstart[PRA_INDEX_SMALL + 1];
    __shared__ u32 wsum[16];
    __shared__ u32 longest;
    __shared__ u64 result[2];
    const u32 t = threadIdx.x, lane = t & 63, wv = t >> 6;
    if (t == 0) longest = 0;
    u32 ng = 0;
    for (u32 base = 0; base < a.n; base += 1024) {
        const u32 i = base + t;
        bool head = i < a.n;
        if (head && i > 0) {
            const u64* r = a.rows + (u64)i * a.w;
            int c = 0;
            while (c < a.jcc && r[c] == r[c - a.w]) c++;
            head = c < a.jcc;
        }
        const u64 mask = __ballot(head);
        if (lane == 0) wsum[wv] = (u32)__popcll(mask);
        __syncthreads();
        u32 at = ng, all = 0;
        for (u32 x = 0; x < 16; x++) {
            if (x == wv) at += all;
            all += wsum[x];
        }
        if (head) gstart[at + (u32)__popcll(mask & ((1ULL << lane) - 1))] = i;
        ng += all;
        __syncthreads();
    }
    if (t == 0) gstart[ng] = a.n;
    u64 cap = 64;
    while (cap < 2ULL * ng) cap <<= 1;
    for (u64 i = t; i < 3 * cap; i += 1024) a.table[i] = 0;
    __threadfence();
    __syncthreads();
    for (u32 g = t; g < ng; g += 1024) {
        const u32 i0 = gstart[g], cnt = gstart[g + 1] - i0;
        atomicMax(&longest, cnt);
        const u64 h = pra_keyhash(a.rows + (u64)i0 * a.w, a.jcc), m = cap - 1;
        u64 s = h & m, q = 0;
        for (; q < cap; q++, s = (s + 1) & m) {
            const u64 prev = atomicCAS((unsigned long long*)(a.table + 3 * s), 0ULL, (unsigned long long)h);
            if (prev == 0) {
                a.table[3 * s + 1] = i0;
                a.table[3 * s + 2] = cnt;
                break;
            }
            if (prev == h) {
                atomicOr(a.err, PRA_FLAG_INDEX_COLLISION);
                break;
            }
        }
        if (q == cap) atomicOr(a.err, PRA_FLAG_TABLE_FULL);
    }
    __threadfence();
    __syncthreads();
    if (t == 0) {
        result[0] = longest;
        result[1] = ng;
    }
    __syncthreads();
    if (a.host)
        pra_publish_words(result, 2, a.err, a.host, a.seq);
    else if (t < 2)
        a.out[t] = result[t];
}

__global__ __launch_bounds__(1024) void k_index_small(IndexSmallArgs a) { pra_index_small(a); }

__global__ __launch_bounds__(1024) void k_index_small_many(const IndexSmallArgs* jobs)
{
    pra_index_small(jobs[blockIdx.x]);
}

// --------------------------------------------------------------- join ------

// lexicographic comparison of the first n words of two rows
__device__ inline int pra_row_cmp(const u64* a, const u64* b, int n)
{
    for (int x = 0; x < n; x++)
        if (a[x] != b[x]) return a[x] < b[x] ? -1 : 1;
    return 0;
}

// First row of the sorted rows [a, z) whose first n > 0 columns are >= key
// (upper: > key).  Three probes a step, their loads in flight together, so a search
// takes half the dependent loads of a binary one; rows that differ from the
// key in column 0 need no more than that.  With one row a thread and runs
// found by four parallel compares, the points-to analysis' counts took 21 us a
// launch instead of 30.
__device__ inline u64 pra_row_bound(const u64* rows, int w, const u64* key, int n, u64 a, u64 z, bool upper)
{
    const u64 k0 = key[0];
    auto below = [&](u64 v, u64 m) {
        if (v != k0) return v < k0;
        const int c = n == 1 ? 0 : pra_row_cmp(rows + m * w + 1, key + 1, n - 1);
        return upper ? c <= 0 : c < 0;
    };
    while (z - a >= 4) {
        const u64 q = (z - a) / 4, m1 = a + q, m2 = m1 + q, m3 = m2 + q;
        const u64 v1 = rows[m1 * w], v2 = rows[m2 * w], v3 = rows[m3 * w];
        if (below(v2, m2)) {
            if (below(v3, m3)) {
                a = m3 + 1;
            } else {
                a = m2 + 1;
                z = m3;
            }
        } else if (below(v1, m1)) {
            a = m1 + 1;
            z = m2;
        } else {
            z = m1;
        }
    }
    while (a < z) {
        const u64 m = (a + z) >> 1;
        if (below(rows[m * w], m)) a = m + 1; else z = m;
    }
    return a;
}

// Run of inner rows matching an outer key, in an inner version kept sorted by
// (bucket, columns): one run inside the key's bucket, found by two searches
// (used for inner relations that change every iteration,
// where a hash index would be rebuilt each time).  Returns its length.
__device__ inline u64 pra_sorted_run(const u64* key, int jcc, const u64* inner, int wi, const u64* ibnd, u64 nb,
                                     u64* first_out)
{
    u64 b = nb == 1 ? 0 : pra_bucket(pra_fnv(key, jcc), nb);
    u64 lo = ibnd[b], hi = ibnd[b + 1];
    if (jcc == 0) {   // every row matches
        *first_out = lo;
        return hi - lo;
    }
    const u64 first = pra_row_bound(inner, wi, key, jcc, lo, hi, false);   // first row >= key
    // first row > key: most runs end within four rows, whose loads go out
    // together; the others are searched for
    u32 eq = 0;
#pragma unroll
    for (u32 q = 0; q < 4; q++)
        if (first + q < hi && pra_row_cmp(inner + (first + q) * wi, key, jcc) == 0) eq |= 1u << q;
    const u64 a = eq != 15u ? first + (u64)__popc(eq) : pra_row_bound(inner, wi, key, jcc, first + 4, hi, true);
    *first_out = first;
    return a - first;
}

// Merges of sorted deltas into sorted fulls (both ordered by (bucket, all w
// columns), disjoint), several relations in one launch each: rank[j] = number
// of full rows before delta row j, searched inside delta row j's bucket; then
// delta row j goes to j + rank[j], and full row i after the delta rows ranked
// at or before it (rank is non-decreasing).  Small merges are all launch and
// search latency: the points-to analysis' 221 merges took 9.3 + 4.5 us each, in
// 61 launches of each kernel 12.8 + 6.4 us.
__device__ inline int pra_merge_job(const MergeBatch& b, const u32* base)
{
    int k = 0;
    while (k + 1 < b.njobs && base[k + 1] <= blockIdx.x) k++;
    return k;
}

__global__ void k_merge_rank(MergeBatch b)
{
    const int k = pra_merge_job(b, b.rank_base);
    const MergeJob& m = b.job[k];
    const u64 j = (u64)(blockIdx.x - b.rank_base[k]) * blockDim.x + threadIdx.x;
    if (j >= m.nd) return;
    u64 lo = 0, hi = b.nb;   // bucket of row j: last b with dbnd[b] <= j
    while (lo + 1 < hi) {
        const u64 mid = (lo + hi) >> 1;
        if (m.dbnd[mid] <= j) lo = mid; else hi = mid;
    }
    m.rank[j] = pra_row_bound(m.F, m.w, m.D + j * m.w, m.w, m.fbnd[lo], m.fbnd[lo + 1], false);
}

// (the first block of a job also adds delta's bucket bounds to full's, the
// bounds of the merged version; k_merge_rank has read full's before)
__global__ void k_merge_scatter(MergeBatch b)
{
    const int k = pra_merge_job(b, b.scatter_base);
    const MergeJob& m = b.job[k];
    const u32 bid = blockIdx.x - b.scatter_base[k];
    if (bid == 0)
        for (u64 i = threadIdx.x; i <= b.nb; i += blockDim.x) m.add_to[i] += m.dbnd[i];
    const u64 t = (u64)bid * blockDim.x + threadIdx.x;
    if (t >= m.nf + m.nd) return;
    const u64* src;
    u64 pos;
    if (t < m.nf) {
        src = m.F + t * m.w;
        pos = t + pra_row_bound(m.rank, 1, &t, 1, 0, m.nd, true);   // delta rows with rank <= t
    } else {
        const u64 j = t - m.nf;
        src = m.D + j * m.w;
        pos = j + m.rank[j];
    }
    pra_copy_row(m.out + pos * m.w, src, m.w);
}

// One thread per join pair: locate the outer row by binary search over the
// exclusive offsets, build the projection of (outer ++ inner[jcc:]) (LEFT) or
// (inner ++ outer[jcc:]) (RIGHT), and write it at its arrival position.
// largest i in [lo, hi] with off[i] <= x (off[lo] <= x holds)
__device__ inline u64 pra_row_of(const u64* off, u64 lo, u64 hi, u64 x)
{
    while (lo < hi) {
        u64 mid = (lo + hi + 1) >> 1;
        if (off[mid] <= x) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// Row of output o0 for the whole block: the largest i in [0, n] with off[i]
// <= o0 (off[0] <= o0 holds), found with PRA_BLOCK probes per step, so the
// range shrinks PRA_BLOCK-fold per dependent load.
__device__ inline u64 pra_block_row_of(const u64* off, u64 n, u64 o0, u32* s_cnt)
{
    u64 lo = 0, hi = n + 1;   // answer in [lo, hi)
    while (hi - lo > 1) {
        const u64 span = hi - lo;
        const u64 idx = lo + (span * threadIdx.x) / PRA_BLOCK;
        const bool pred = off[idx] <= o0;   // true for a prefix of the threads
        if (threadIdx.x == 0) *s_cnt = 0;
        __syncthreads();
        const u64 b = __ballot(pred);
        if ((threadIdx.x & 63) == 0 && b) atomicAdd(s_cnt, (u32)__popcll(b));
        __syncthreads();
        const u32 cnt = *s_cnt;
        __syncthreads();
        const u64 nlo = lo + (span * (cnt - 1)) / PRA_BLOCK;
        hi = cnt < PRA_BLOCK ? lo + (span * cnt) / PRA_BLOCK : hi;
        lo = nlo;
    }
    return lo;
}

// block `bid` of `gdim` of one rule's join expansion
__device__ __forceinline__ void pra_join_expand_block(const JoinExpandArgs& a, u32 bid, u32 gdim)
{
    if (a.ctl[1]) return;
    const u64 first = a.off[0], total = a.off[a.n_outer];   // first > 0 for a window of rows
    __shared__ u64 s_off[PRA_BLOCK + 1];
    __shared__ u32 s_cnt;
    const u64 step = (u64)gdim * blockDim.x;
    for (u64 o0 = first + (u64)bid * blockDim.x; o0 < total; o0 += step) {
        __syncthreads();
        // the block's first row, then the offsets of the next PRA_BLOCK rows
        // in LDS, where each output finds its row
        const u64 r0 = pra_block_row_of(a.off, a.n_outer, o0, &s_cnt);
        s_off[threadIdx.x] = r0 + threadIdx.x <= a.n_outer ? a.off[r0 + threadIdx.x] : ~0ULL;
        if (threadIdx.x == 0) s_off[PRA_BLOCK] = r0 + PRA_BLOCK <= a.n_outer ? a.off[r0 + PRA_BLOCK] : ~0ULL;
        __syncthreads();
        u64 o = o0 + threadIdx.x;
        if (o >= total) continue;
        u64 i;
        if (o < s_off[PRA_BLOCK]) {
            u32 lo = 0, hi = PRA_BLOCK;   // largest j in [lo, hi] with s_off[j] <= o
            while (lo < hi) {
                u32 mid = (lo + hi + 1) >> 1;
                if (s_off[mid] <= o) lo = mid; else hi = mid - 1;
            }
            i = r0 + lo;
        } else {
            i = pra_row_of(a.off, r0 + PRA_BLOCK, a.n_outer, o);
        }
        const u64* d = a.outer + i * a.wo;
        const u64* f = a.inner + (a.istart[i] + (o - a.off[i])) * a.wi;
        u64 s = a.nb == 1 ? 0 : pra_bucket(pra_fnv(d, a.jcc), a.nb);
        u64 pos = a.posadj[s] + o;
        u64* dst = a.cand + pos * a.cw;
        // the destination bucket hashes the output's first out_jcc columns
        // as they are written
        u64 h = PRA_FNV_OFFSET;
        for (int c = 0; c < a.cw; c++) {
            int m = a.map[c];
            u64 v;
            if (a.left)
                v = m < a.wo ? d[m] : f[a.jcc + (m - a.wo)];
            else
                v = m < a.wi ? f[m] : d[a.jcc + (m - a.wi)];
            dst[c] = v;
            if (c < a.out_jcc) h = pra_fnv_word(h, v);
        }
        a.dest[pos] = a.nb == 1 ? 0u : pra_bucket(h, a.nb);
    }
}

__global__ void k_join_expand(JoinExpandArgs a)
{
    pra_join_expand_block(a, blockIdx.x, gridDim.x);
}

// job of block `bid` in a device job table (block bases after the njobs
// arguments): the number of later jobs' bases at or below it, 64 bases per
// load round
__device__ inline int pra_job_of(const u32* block_base, int njobs, u32 bid)
{
    int k = 0;
    for (int j0 = 1; j0 < njobs; j0 += 64) {
        const int j = j0 + (int)(threadIdx.x & 63);
        k += __popcll(__ballot(j < njobs && block_base[j] <= bid));
    }
    return k;
}

// The rank rows of several versions in one launch: bound by the launches (5.7
// us each for the 260-2,000 rows of 60 instances) and the waits behind them.
// 60 closures of 200-1,500 vertices: 15.1 -> 14.1 ms.
__global__ void k_rank_rows_many(const RankRowsArgs* jobs, int njobs)
{
    const u32* base = (const u32*)(jobs + njobs);
    const int k = pra_job_of(base, njobs, blockIdx.x);
    pra_rank_row(jobs[k], (u64)(blockIdx.x - base[k]) * PRA_BLOCK + threadIdx.x);
}

// Join expansions of several rules in one launch (job table in device
// memory); a block whose job has no outputs left for it leaves before it
// reads the job's arguments.
__global__ void k_join_expand_many(const JoinExpandArgs* jobs, int njobs)
{
    const u32* block_base = (const u32*)(jobs + njobs);
    const int k = pra_job_of(block_base, njobs, blockIdx.x);
    const u32 bid = blockIdx.x - block_base[k];
    const JoinExpandArgs* jp = jobs + k;
    if (jp->ctl[1] || jp->off[0] + (u64)bid * PRA_BLOCK >= jp->off[jp->n_outer]) return;
    const JoinExpandArgs a = *jp;
    pra_join_expand_block(a, bid, block_base[k + 1] - block_base[k]);
}

__device__ inline bool pra_filter(int op, u64 x, u64 y)
{
    switch (op) {
    case PRA_F_EQ: return x == y;
    case PRA_F_NEQ: return x != y;
    case PRA_F_LT: return x < y;
    case PRA_F_LE: return x <= y;
    case PRA_F_GT: return x > y;
    case PRA_F_GE: return x >= y;
    case PRA_F_TRUE: return true;
    default: return false;
    }
}

// outer row i of one rule's copy expansion
__device__ __forceinline__ void pra_copy_expand_row(const CopyExpandArgs& a, u64 i)
{
    if (a.ctl[1]) return;
    if (i >= a.n) return;
    if (a.off[i + 1] == a.off[i]) return;
    const u64* r = a.rows + i * a.w;
    u64 s = a.nb == 1 ? 0 : pra_bucket(pra_fnv(r, a.in_jcc), a.nb);
    u64 pos = a.posadj[s] + a.off[i];
    u64* dst = a.cand + pos * a.cw;
    u64 h = PRA_FNV_OFFSET;
    for (int c = 0; c < a.cw; c++) {
        u64 v = r[a.map[c]];
        dst[c] = v;
        if (c < a.out_jcc) h = pra_fnv_word(h, v);
    }
    a.dest[pos] = a.nb == 1 ? 0u : pra_bucket(h, a.nb);
}

__global__ void k_copy_expand(CopyExpandArgs a)
{
    pra_copy_expand_row(a, (u64)blockIdx.x * blockDim.x + threadIdx.x);
}

// Copy expansions of several rules in one launch (job table as
// k_join_expand_many's; every block has rows)
__global__ void k_copy_expand_many(const CopyExpandArgs* jobs, int njobs)
{
    const u32* block_base = (const u32*)(jobs + njobs);
    const int k = pra_job_of(block_base, njobs, blockIdx.x);
    const CopyExpandArgs a = jobs[k];
    pra_copy_expand_row(a, (u64)(blockIdx.x - block_base[k]) * blockDim.x + threadIdx.x);
}

// Arrival plan of one output relation, computed on the device: for source
// bucket s and the RAs producing the relation (in RA order), the position of
// their outputs in the arrival order source-major, RA-minor
// (src/comm/all_to_allv_comm.cpp:64-142), the candidate count, whether it
// exceeds the allocated capacity, and the join pairs.  RA j emits the outer
// rows [lo[j][s], hi[j][s]) of source s (whole buckets, or one round's rows).
// With rounds_check, a join call with more than `thresh` outputs from one
// source (src/RA/parallel_join.cpp:196-201, src/RAM/RA_tasks.cpp:312) marks
// the output for threshold rounds (ctl[1] = 2) instead of emitting.
__global__ void k_plan(PlanArgs a)
{
    const int nb = a.nb;
    for (int e = threadIdx.x; e < a.nr * nb; e += blockDim.x) {
        int j = e / nb, s = e % nb;
        u64 lo = a.off[j][a.lo[j][s]], hi = a.off[j][a.hi[j][s]];
        a.srcoff[(u64)a.ras[j] * 2 * nb + s] = lo;
        a.srcoff[(u64)a.ras[j] * 2 * nb + nb + s] = hi - lo;
    }
    __threadfence_block();
    __syncthreads();
    if (threadIdx.x != 0) return;
    u64 tot = 0, jtot = 0;
    bool rounds = false;
    for (int s = 0; s < nb; s++)
        for (int j = 0; j < a.nr; j++) {
            const u64* so = a.srcoff + (u64)a.ras[j] * 2 * nb;
            a.posadj[(u64)a.ras[j] * nb + s] = tot - so[s];
            u64 cnt = so[nb + s];
            if (a.is_join[j]) {
                if (a.rounds_check && (long long)cnt > a.thresh) rounds = true;
                jtot += cnt;
            }
            tot += cnt;
        }
    a.ctl[0] = tot;
    a.ctl[1] = rounds ? 2 : tot > a.cap ? 1 : 0;
    if (a.count_joined && (rounds || tot <= a.cap)) *a.joined += jtot;
}

// k_plan for every output of an iteration at once: block b plans output
// outs[b] over its active rules in rule order (source-major, rule-minor
// arrival, as k_plan).
__global__ void k_plan_all(PlanAllArgs a)
{
    const int oi = a.outs[blockIdx.x];
    const int nb = a.nb;
    __shared__ unsigned char lr[PRA_MAXRA];
    __shared__ int nlr;
    if (threadIdx.x == 0) {
        int k = 0;
        for (int r = 0; r < a.nra; r++)
            if (a.rout[r] == oi) lr[k++] = (unsigned char)r;
        nlr = k;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < nlr * nb; e += blockDim.x) {
        const int r = lr[e / nb], s = e % nb;
        const u64 lo = a.off[r][a.bnd[r][s]], hi = a.off[r][a.bnd[r][s + 1]];
        a.srcoff[(u64)r * 2 * nb + s] = lo;
        a.srcoff[(u64)r * 2 * nb + nb + s] = hi - lo;
    }
    __threadfence_block();
    __syncthreads();
    if (threadIdx.x != 0) return;
    u64 tot = 0, jtot = 0;
    bool rounds = false;
    for (int s = 0; s < nb; s++)
        for (int k = 0; k < nlr; k++) {
            const int r = lr[k];
            const u64* so = a.srcoff + (u64)r * 2 * nb;
            a.posadj[(u64)r * nb + s] = tot - so[s];
            const u64 cnt = so[nb + s];
            if (a.is_join[r]) {
                if ((long long)cnt > a.thresh) rounds = true;
                jtot += cnt;
            }
            tot += cnt;
        }
    u64* ctl = a.stage2 + (u64)oi * a.sw + 4;
    ctl[0] = tot;
    ctl[1] = rounds ? 2 : tot > a.cap[oi] ? 1 : 0;
    if ((rounds || tot <= a.cap[oi]) && jtot) atomicAdd((unsigned long long*)a.joined[oi], (unsigned long long)jtot);
}

__global__ void k_plan_tab(PlanTabArgs a)
{
    const PlanOut o = a.outs[blockIdx.x];
    const int nb = a.nb;
    for (u32 e = threadIdx.x; e < o.count * (u32)nb; e += blockDim.x) {
        const u32 r = a.rule_ids[o.first + e / nb];
        const int s = (int)(e % nb);
        const PlanRule& pr = a.rules[r];
        const u64 lo = pr.off[pr.bnd[s]], hi = pr.off[pr.bnd[s + 1]];
        a.srcoff[(u64)r * 2 * nb + s] = lo;
        a.srcoff[(u64)r * 2 * nb + nb + s] = hi - lo;
    }
    __threadfence_block();
    __syncthreads();
    if (threadIdx.x != 0) return;
    u64 tot = 0, jtot = 0;
    bool rounds = false;
    for (int s = 0; s < nb; s++)
        for (u32 k = 0; k < o.count; k++) {
            const u32 r = a.rule_ids[o.first + k];
            const u64* so = a.srcoff + (u64)r * 2 * nb;
            a.posadj[(u64)r * nb + s] = tot - so[s];
            const u64 cnt = so[nb + s];
            if (a.rules[r].is_join) {
                if ((long long)cnt > a.thresh) rounds = true;
                jtot += cnt;
            }
            tot += cnt;
        }
    u64* ctl = a.stage2 + (u64)o.oi * a.sw + 4;
    ctl[0] = tot;
    ctl[1] = rounds ? 2 : tot > o.cap ? 1 : 0;
    if ((rounds || tot <= o.cap) && jtot) atomicAdd((unsigned long long*)o.joined, (unsigned long long)jtot);
}

// Split of one threshold round: the first outer row i (of n, offsets off
// relative to base = off[0]) such that the call's distinct outputs through
// row i, kp[off[i + 1] - base] (exclusive prefix of first-occurrence flags),
// exceed thresh; n when there is none.
__global__ void k_find_split(const u64* off, u64 n, const u32* kp, long long thresh, u64* out)
{
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const u64 base = off[0];
    u64 a = 0, z = n;
    while (a < z) {
        u64 m = (a + z) >> 1;
        if ((long long)kp[off[m + 1] - base] > thresh) z = m; else a = m + 1;
    }
    *out = a;
}

// Copy `words` summary words and then the error flags into pinned host
// memory; the host reads them once the kernel has completed.
// The summary words and the error flags into pinned host memory, then
// host[-1] = seq once every word is visible to the host (each thread's
// system-scope release before the barrier, then one system-scope store), so
// the host can start on the summary before the kernel's completion is
// signalled.  host[-1] is written by publications only, so a sequence number
// never meets a stale summary word there.
__device__ __forceinline__ void pra_publish_words(const u64* src, u64 words, const u32* flags, u64* host, u64 seq)
{
    for (u64 i = threadIdx.x; i < words; i += blockDim.x) host[i] = src[i];
    if (threadIdx.x == 0) host[words] = *flags;
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(host - 1, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void k_publish(const u64* src, u64 words, const u32* flags, u64* host, u64 seq)
{
    pra_publish_words(src, words, flags, host, seq);
}

// ---------------------------------------------------- dedup / newt ---------

// Count this lane in LDS counter h[d] when `on`, adding once per group of
// lanes of the wave with the same d (d < 256): a tile's candidates fall into
// few destination buckets, and one LDS atomic per lane would serialise on
// them.  Every lane of the wave must call it.
__device__ __forceinline__ void pra_wave_count(u32* h, u32 d, bool on)
{
    const u64 act = __ballot(on);
    if (!act) return;
    const u64 peers = pra_match<PRA_RADIX_BITS>(on ? d : 0u, act);
    if (on && __lane_id() == (u32)(__ffsll((long long)peers) - 1)) atomicAdd(&h[d], (u32)__popcll(peers));
}


// Claim (or find) the slot of candidate p's key (p < the candidate count).
// The first claimant stores the key; every candidate then lowers the slot's
// arrival mark to (epoch << 40 | p+1), so the earliest arrival of this
// iteration wins, while a mark from an earlier iteration (key already in full
// or delta) always wins.  MAXKW > 0: keys of at most MAXKW words (exactly
// MAXKW with EXACT), loaded once into registers with every word in flight
// together; MAXKW == 0: any key width, read from the row as needed.
template <int MAXKW, bool EXACT>
__device__ __forceinline__ void pra_claim_one(const u64* cand, int cw, int kw_, u64* table, u64 cap, u64* slot_of,
                                              u64 epoch, u32* flags, u64 p)
{
    const int kw = EXACT ? MAXKW : kw_;
    const u64* key = cand + p * cw;
    u64 kr[MAXKW > 0 ? MAXKW : 1];
    u64 h;
    if (MAXKW > 0) {
#pragma unroll
        for (int c = 0; c < MAXKW; c++) kr[c] = c < kw ? key[c] : 0;
        // pra_keyhash over the register copy
        h = 0x9E3779B97F4A7C15ULL ^ (u64)kw;
#pragma unroll
        for (int c = 0; c < MAXKW; c++)
            if (c < kw) h = pra_mix64(h ^ (kr[c] + 0x632BE59BD9B4E019ULL * (u64)(c + 1)));
        h = h ? h : 1;
    } else {
        h = pra_keyhash(key, kw);
    }
    const int stride = 2 + kw;
    const u64 mark = (epoch << 40) | (p + 1);
    u64 m = cap - 1, s = h & m;
    for (u64 q = 0; q < cap; q++) {
        u64* slot = table + s * stride;
        u64 cur = slot[0];
        bool mine = false;
        if (cur == 0) {
            cur = atomicCAS((unsigned long long*)slot, 0ULL, (unsigned long long)h);
            if (cur == 0) {
                mine = true;
                if (MAXKW > 0) {
#pragma unroll
                    for (int c = 0; c < MAXKW; c++)
                        if (c < kw) slot[2 + c] = kr[c];
                } else {
                    for (int c = 0; c < kw; c++) slot[2 + c] = key[c];
                }
            }
        }
        if (mine || cur == h) {
            // the claimant lowers the mark at once; a later candidate first
            // reads it: a mark from an earlier iteration (key already present)
            // or an earlier arrival of this one already beats ours
            if (mine) {
                atomicMin((unsigned long long*)(slot + 1), (unsigned long long)mark);
            } else {
                u64 old = slot[1];
                if (old > mark && old >= (epoch << 40))
                    atomicMin((unsigned long long*)(slot + 1), (unsigned long long)mark);
            }
            slot_of[p] = s;
            return;
        }
        s = (s + 1) & m;
    }
    slot_of[p] = ~0ULL;
    atomicOr(flags, PRA_FLAG_TABLE_FULL);
}

// One output's claims: one thread per candidate.
template <int MAXKW, bool EXACT>
__global__ void k_dedup_claim2(const u64* cand, const u64* ctl, int cw, int kw_, u64* table, u64 cap, u64* slot_of,
                               u64 epoch, u32* flags)
{
    if (ctl[1]) return;
    const u64 p = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= ctl[0]) return;
    pra_claim_one<MAXKW, EXACT>(cand, cw, kw_, table, cap, slot_of, epoch, flags, p);
}

// Claims of several outputs in one launch: a block serves the job whose
// block range holds it, as k_dedup_claim2 serves its one output.
template <int MAXKW, bool EXACT>
__global__ void k_dedup_claim_many(ClaimBatch b, u32* flags)
{
    int k = 0;
    while (k + 1 < b.njobs && b.block_base[k + 1] <= blockIdx.x) k++;
    const ClaimJob& j = b.job[k];
    if (j.ctl[1]) return;
    const u64 p = (u64)(blockIdx.x - b.block_base[k]) * blockDim.x + threadIdx.x;
    if (p >= j.ctl[0]) return;
    pra_claim_one<MAXKW, EXACT>(j.cand, j.cw, j.kw, j.table, j.cap, j.slot_of, j.epoch, flags, p);
}

// Keep the winners, verify every key against its slot (a 64-bit hash
// collision between distinct keys is reported, never merged) and count kept
// candidates per destination bucket per tile.
// MAXKW > 0: keys of at most MAXKW words (exactly MAXKW with EXACT; the
// slot's words and the candidate's are loaded together); MAXKW == 0: any key
// width.
// Tile `tile` of PRA_TILE candidates (h, sl: the block's LDS counters and
// scan words).
template <int MAXKW, bool EXACT>
__device__ __forceinline__ void pra_decide_tile(const u64* cand, u64 n, int cw, int kw_, const u64* table,
                                                const u64* slot_of, u64 epoch, u32* keep, const u32* dest, u32 nb,
                                                u32* hist, u32 nblocks, u32* flags, u32* offs1, u32 tile, u32* h,
                                                u32* sl)
{
    const int kw = EXACT ? MAXKW : kw_;
    u64 base = (u64)tile * PRA_TILE;
    if (base >= n) {
        // a tile past the candidates keeps nothing
        for (u32 i = threadIdx.x; i < nb; i += PRA_DECIDE_BLOCK) hist[(u64)i * nblocks + tile] = 0;
        if (offs1)
            for (u32 i = threadIdx.x; i <= nb; i += PRA_DECIDE_BLOCK) offs1[i] = 0;
        return;
    }
    for (int i = threadIdx.x; i < PRA_RADIX; i += PRA_DECIDE_BLOCK) h[i] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PRA_TILE / PRA_DECIDE_BLOCK; k++) {
        u64 p = base + (u64)k * PRA_DECIDE_BLOCK + threadIdx.x;
        u32 kp = 0;
        if (p < n) {
            u64 s = slot_of[p];
            if (s != ~0ULL) {
                const u64* slot = table + s * (2 + kw);
                const u64* key = cand + p * cw;
                bool eq = true;
                if (MAXKW > 0) {
                    u64 x[MAXKW > 0 ? MAXKW : 1], y[MAXKW > 0 ? MAXKW : 1];
#pragma unroll
                    for (int c = 0; c < MAXKW; c++) {
                        x[c] = c < kw ? slot[2 + c] : 0;
                        y[c] = c < kw ? key[c] : 0;
                    }
#pragma unroll
                    for (int c = 0; c < MAXKW; c++) eq = eq && x[c] == y[c];
                } else {
                    for (int c = 0; c < kw; c++)
                        if (slot[2 + c] != key[c]) { eq = false; break; }
                }
                if (!eq) atomicOr(flags, PRA_FLAG_COLLISION);
                if (slot[1] == ((epoch << 40) | (p + 1))) kp = 1;
            }
            keep[p] = kp;
        }
        pra_wave_count(h, kp ? dest[p] : 0u, kp != 0);
    }
    __syncthreads();
    if (offs1) {
        // a single tile: its counts are the whole histogram, whose
        // exclusive offsets (and total, offs1[nb]) go out directly
        u32 tot;
        const u32 v = threadIdx.x < nb ? h[threadIdx.x] : 0u;
        const u32 ex = block_exclusive_scan<u32, PRA_DECIDE_BLOCK / 64>(v, sl, &tot);
        if (threadIdx.x < nb) offs1[threadIdx.x] = ex;
        if (threadIdx.x == 0) offs1[nb] = tot;
    } else {
        for (u32 i = threadIdx.x; i < nb; i += PRA_DECIDE_BLOCK) hist[(u64)i * nblocks + tile] = h[i];
    }
    __syncthreads();
}

// One output's decisions: blocks of PRA_DECIDE_BLOCK threads take tiles of
// PRA_TILE candidates in turn (each candidate is a chain of dependent loads,
// so many waves per tile hide them).
template <int MAXKW, bool EXACT>
__global__ __launch_bounds__(PRA_DECIDE_BLOCK) void k_dedup_decide_hist(const u64* cand, const u64* ctl, int cw,
                                                                        int kw_, const u64* table,
                                                                        const u64* slot_of, u64 epoch, u32* keep,
                                                                        const u32* dest, u32 nb, u32* hist,
                                                                        u32 nblocks, u32* flags, u32* offs1)
{
    if (ctl[1]) return;
    const u64 n = ctl[0];
    __shared__ u32 h[PRA_RADIX];
    __shared__ u32 sl[PRA_DECIDE_BLOCK / 64 + 1];
    for (u32 tile = blockIdx.x; tile < nblocks; tile += gridDim.x)
        pra_decide_tile<MAXKW, EXACT>(cand, n, cw, kw_, table, slot_of, epoch, keep, dest, nb, hist, nblocks, flags,
                                      offs1, tile, h, sl);
}

// Decisions of several outputs in one launch: block -> (job, tile) by the
// jobs' block ranges; no stride, every tile has its block.
template <int MAXKW, bool EXACT>
__global__ __launch_bounds__(PRA_DECIDE_BLOCK) void k_dedup_decide_many(DecideBatch b, u32* flags)
{
    __shared__ u32 h[PRA_RADIX];
    __shared__ u32 sl[PRA_DECIDE_BLOCK / 64 + 1];
    int k = 0;
    while (k + 1 < b.njobs && b.block_base[k + 1] <= blockIdx.x) k++;
    const DecideJob& j = b.job[k];
    if (j.ctl[1]) return;
    pra_decide_tile<MAXKW, EXACT>(j.cand, j.ctl[0], j.cw, j.kw, j.table, j.slot_of, j.epoch, j.keep, j.dest, b.nb,
                                  j.hist, j.nblocks, flags, j.offs1, blockIdx.x - b.block_base[k], h, sl);
}

// ----------------------------------------------------- dense membership ---

// rank index of a key of KW words (its leading digit the bucket-major rank
// when by_bucket), false when a value has no dictionary rank
template <int KW>
__device__ __forceinline__ bool pra_dense_index(const u64* key, const u64* dict, u64 dcap, u64 D, int by_bucket,
                                                u64* idx)
{
    u64 v[KW], e[KW];
#pragma unroll
    for (int c = 0; c < KW; c++) v[c] = key[c];
#pragma unroll
    for (int c = 0; c < KW; c++) e[c] = pra_dict_find(dict, dcap, v[c]);
    u64 x = 0;
    bool ok = true;
#pragma unroll
    for (int c = 0; c < KW; c++) {
        ok = ok && e[c] != 0;
        x = x * D + (c == 0 && by_bucket ? e[c] >> 32 : (u64)((u32)e[c] - 1));
    }
    *idx = x;
    return ok;
}

__device__ __forceinline__ bool pra_dense_index_n(int kw, const u64* key, const u64* dict, u64 dcap, u64 D,
                                                  int by_bucket, u64* idx)
{
    switch (kw) {
    case 1: return pra_dense_index<1>(key, dict, dcap, D, by_bucket, idx);
    case 2: return pra_dense_index<2>(key, dict, dcap, D, by_bucket, idx);
    case 3: return pra_dense_index<3>(key, dict, dcap, D, by_bucket, idx);
    default: return pra_dense_index<4>(key, dict, dcap, D, by_bucket, idx);
    }
}

// a slot written in this iteration (the others count as empty)
__device__ __forceinline__ bool pra_dense_live(u64 v, const DenseArgs& a) { return v != 0 && (v & a.emask) == a.stamp; }

// A candidate whose key is a member (bit set) is dropped at once
// (slot_of = ~0); any other claims or finds the slot holding x + 1 and lowers
// the slot's arrival to its own position, so the earliest arrival wins.  A
// slot is one word, epoch | (x + 1) << PRA_DENSE_PBITS | arrival: the first
// candidate of a key claims an empty slot with one compare-and-swap, a later
// one reads it and swaps only while its own arrival is earlier.
template <int KW>
__device__ __forceinline__ void pra_dense_claim_one(const DenseArgs& a, u64 p, u32* flags)
{
    u64 x;
    if (!pra_dense_index<KW>(a.cand + p * a.cw, a.dict, a.dict_cap, a.D, a.by_bucket, &x)) {
        atomicCAS((unsigned long long*)(a.ctl + 1), 0ULL, 3ULL);
        return;
    }
    if ((a.bitmap[x >> 5] >> (x & 31)) & 1u) {
        a.slot_of[p] = ~0ULL;
        return;
    }
    const u64 key = x + 1, m = a.cap - 1, mine = a.stamp | (key << PRA_DENSE_PBITS) | p;
    u64 s = pra_mix64(key) & m;
    for (u64 q = 0; q < a.cap; q++) {
        unsigned long long* slot = (unsigned long long*)(a.table + s);
        // a plain load first: a slot held by another key then costs no
        // atomic (swapping straight away measured slower)
        u64 cur = *slot;
        if (!pra_dense_live(cur, a)) {
            // empty: every other write in this launch leaves a live slot, so
            // a failed swap returns one
            const u64 prev = atomicCAS(slot, (unsigned long long)cur, (unsigned long long)mine);
            if (prev == cur) {
                a.slot_of[p] = s;
                return;
            }
            cur = prev;
        }
        if (((cur & ~a.emask) >> PRA_DENSE_PBITS) == key) {
            // the key's slot: lower its arrival while ours is earlier (the
            // key bits never change once set); a candidate that never got in
            // has lost to an earlier arrival for good, and the decision skips it
            bool in = false;
            while ((cur & PRA_DENSE_PMASK) > p) {
                const u64 prev = atomicCAS(slot, (unsigned long long)cur, (unsigned long long)mine);
                if (prev == cur) {
                    in = true;
                    break;
                }
                cur = prev;
            }
            a.slot_of[p] = in ? s : ~0ULL;
            return;
        }
        s = (s + 1) & m;
    }
    a.slot_of[p] = ~0ULL;
    atomicOr(flags, PRA_FLAG_TABLE_FULL);
}

template <int KW>
__global__ void k_dense_claim(DenseArgs a, u32* flags)
{
    if (a.ctl[1]) return;
    const u64 p = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= a.ctl[0]) return;
    pra_dense_claim_one<KW>(a, p, flags);
}

// Dense claims of several outputs (of one key width) in one launch; the job
// table in device memory is followed by the claim blocks' and the decision
// blocks' first block per job (njobs + 1 words each).
template <int KW>
__global__ void k_dense_claim_many(const DenseArgs* jobs, int njobs, u32* flags)
{
    const u32* cbase = (const u32*)(jobs + njobs);
    const int k = pra_job_of(cbase, njobs, blockIdx.x);
    const DenseArgs* jp = jobs + k;
    if (jp->ctl[1]) return;
    const u64 p = (u64)(blockIdx.x - cbase[k]) * blockDim.x + threadIdx.x;
    if (p >= jp->ctl[0]) return;
    pra_dense_claim_one<KW>(*jp, p, flags);
}

// Tile `tile` of the dense decision: the earliest arrival of each claimed key
// keeps it, sets its membership bit and returns its slot to empty; kept
// candidates are counted per destination bucket as in pra_decide_tile.
__device__ __forceinline__ void pra_dense_decide_tile(const DenseArgs& a, u64 n, u32 tile, u32* h, u32* sl)
{
    const u64 base = (u64)tile * PRA_TILE;
    if (base >= n) {
        for (u32 i = threadIdx.x; i < a.nb; i += PRA_DECIDE_BLOCK) a.hist[(u64)i * a.nblocks + tile] = 0;
        if (a.offs1)
            for (u32 i = threadIdx.x; i <= a.nb; i += PRA_DECIDE_BLOCK) a.offs1[i] = 0;
        return;
    }
    for (int i = threadIdx.x; i < PRA_RADIX; i += PRA_DECIDE_BLOCK) h[i] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PRA_TILE / PRA_DECIDE_BLOCK; k++) {
        const u64 p = base + (u64)k * PRA_DECIDE_BLOCK + threadIdx.x;
        u32 kp = 0, d = 0;
        if (p < n) {
            const u64 s = a.slot_of[p];
            if (s != ~0ULL) {
                u64* slot = a.table + s;
                const u64 v = *slot;
                // the earliest arrival of the key keeps it; without epochs
                // the slot returns to empty, which no later arrival's
                // position matches
                if (pra_dense_live(v, a) && (v & PRA_DENSE_PMASK) == p) {
                    kp = 1;
                    d = a.dest[p];
                    const u64 x = ((v & ~a.emask) >> PRA_DENSE_PBITS) - 1;
                    atomicOr(&a.bitmap[x >> 5], 1u << (x & 31));
                    if (!a.emask) *slot = 0;
                    // the rank index, for the newt scatter's packed key (which
                    // leads with the bucket, so its digits are plain ranks)
                    a.slot_of[p] = a.by_bucket ? a.rank_of[x / a.lead] * a.lead + x % a.lead : x;
                }
            }
            a.keep[p] = kp;
        }
        pra_wave_count(h, d, kp != 0);
    }
    __syncthreads();
    if (a.offs1) {
        u32 tot;
        const u32 v = threadIdx.x < a.nb ? h[threadIdx.x] : 0u;
        const u32 ex = block_exclusive_scan<u32, PRA_DECIDE_BLOCK / 64>(v, sl, &tot);
        if (threadIdx.x < a.nb) a.offs1[threadIdx.x] = ex;
        if (threadIdx.x == 0) a.offs1[a.nb] = tot;
    } else {
        for (u32 i = threadIdx.x; i < a.nb; i += PRA_DECIDE_BLOCK) a.hist[(u64)i * a.nblocks + tile] = h[i];
    }
    __syncthreads();
}

__global__ __launch_bounds__(PRA_DECIDE_BLOCK) void k_dense_decide(DenseArgs a)
{
    if (a.ctl[1]) return;
    const u64 n = a.ctl[0];
    __shared__ u32 h[PRA_RADIX];
    __shared__ u32 sl[PRA_DECIDE_BLOCK / 64 + 1];
    for (u32 tile = blockIdx.x; tile < a.nblocks; tile += gridDim.x) pra_dense_decide_tile(a, n, tile, h, sl);
}

// Dense decisions of several outputs in one launch: one block per tile of
// each job (table as k_dense_claim_many).
__global__ __launch_bounds__(PRA_DECIDE_BLOCK) void k_dense_decide_many(const DenseArgs* jobs, int njobs)
{
    __shared__ u32 h[PRA_RADIX];
    __shared__ u32 sl[PRA_DECIDE_BLOCK / 64 + 1];
    const u32* dbase = (const u32*)(jobs + njobs) + njobs + 1;
    const int k = pra_job_of(dbase, njobs, blockIdx.x);
    const DenseArgs a = jobs[k];
    if (a.ctl[1]) return;
    pra_dense_decide_tile(a, a.ctl[0], blockIdx.x - dbase[k], h, sl);
}

// the membership bits of n rows (key = their first kw columns)
template <int KW>
__global__ void k_dense_build(const u64* rows, u64 n, int w, const u64* dict, u64 dcap, u64 D, int by_bucket, u32* bitmap,
                              u64* miss)
{
    const u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    u64 x;
    if (!pra_dense_index<KW>(rows + i * w, dict, dcap, D, by_bucket, &x)) {
        atomicAdd((unsigned long long*)miss, 1ULL);
        return;
    }
    atomicOr(&bitmap[x >> 5], 1u << (x & 31));
}

// Order of a relation from its membership bitmap.  Bit x of the bitmap is the
// key of rank index x, and rank indexes order as the rows do, so a key's place
// among all keys is the number of set bits below x: the exclusive prefix of
// the 256-bit blocks' counts, plus the bits below x in its block.
#define PRA_BM_BLOCK_WORDS 4   // u64 words per counted block

// set bits below bit x; nblk blocks of u64 words, prefix[nblk] the total
__device__ __forceinline__ u32 pra_bm_rank(const u64* bm, u64 words, const u32* prefix, u64 x)
{
    const u64 b = x >> 8, w0 = b * PRA_BM_BLOCK_WORDS;
    u32 r = prefix[b];
    if (w0 >= words) return r;
    const u32 bit = (u32)(x & 255), wi = bit >> 6;
    u64 v[PRA_BM_BLOCK_WORDS];
#pragma unroll
    for (u32 k = 0; k < PRA_BM_BLOCK_WORDS; k++) v[k] = w0 + k < words ? bm[w0 + k] : 0;
#pragma unroll
    for (u32 k = 0; k < PRA_BM_BLOCK_WORDS; k++) {
        const u64 m = k < wi ? ~0ULL : k == wi ? (1ULL << (bit & 63)) - 1 : 0;
        r += (u32)__popcll(v[k] & m);
    }
    return r;
}

__global__ void k_bm_count(const u64* bm, u64 words, u64 nblk, u32* cnt)
{
    const u64 b = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nblk) return;
    u32 c = 0;
#pragma unroll
    for (u32 k = 0; k < PRA_BM_BLOCK_WORDS; k++) {
        const u64 i = b * PRA_BM_BLOCK_WORDS + k;
        c += i < words ? (u32)__popcll(bm[i]) : 0;
    }
    cnt[b] = c;
}

// Every row (all of them members) to its place.  Bound by the rows' own
// bytes and by the lines of 24-byte writes: runs of a delta log walk the
// bitmap in order, so its words, the prefix and the dictionary hit in cache.
template <int KW>
__global__ void k_bm_place(const u64* rows, u64 n, int w, const u64* dict, u64 dcap, u64 D, int by_bucket,
                           const u64* bm, u64 words, const u32* prefix, u64* out)
{
    const u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    u64 x;
    if (!pra_dense_index<KW>(rows + i * w, dict, dcap, D, by_bucket, &x)) return;
    const u32 pos = pra_bm_rank(bm, words, prefix, x);
    if (pos < n) pra_copy_row(out + (u64)pos * w, rows + i * w, w);
}

// Exclusive prefix of `tile` over its predecessors' published values (digit
// 0 of the status words, `stride` apart), walked by the 64 lanes of one wave: each step reads
// the 64 nearest unconsumed predecessors at once and adds the ready ones up to
// the nearest inclusive prefix.  Every lane returns the same value.
__device__ inline u64 pra_lookback_wave(const u64* status, u32 tile, u32 epoch, u32* flags, u32 stride = PRA_RADIX)
{
    constexpr u64 VAL = (1ULL << 46) - 1;
    const int lane = __lane_id();
    u64 excl = 0;
    long long t = (long long)tile - 1;
    u32 spins = 0;
    while (t >= 0) {
        long long j = t - lane;
        u64 v = j >= 0 ? __hip_atomic_load(status + (u64)j * stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                       : st_pack(epoch, PRA_ST_INC, 0);
        u64 fl = (v >> 46) & 3ULL;
        bool ready = (u32)(v >> 48) == epoch && fl != 0;
        u64 notready = __ballot(!ready);
        u64 inc = __ballot(ready && fl == PRA_ST_INC);
        int first_nr = notready ? __ffsll((unsigned long long)notready) - 1 : 64;
        int first_inc = inc ? __ffsll((unsigned long long)inc) - 1 : 64;
        bool stop = first_inc < first_nr;
        int take = stop ? first_inc + 1 : first_nr;
        u64 x = lane < take ? (v & VAL) : 0;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) x += __shfl_xor(x, d, 64);
        excl += x;
        if (stop) break;
        t -= take;
        if (take == 0 && ++spins > PRA_LOOKBACK_SPIN_LIMIT) {
            if (lane == 0) atomicOr(flags, PRA_FLAG_SORT_STALL);
            break;
        }
    }
    return excl;
}

// ---------------------------------------------------- ranked membership ---
//
// The whole newt step of a dense output without a hash slot or a sort.  A
// candidate that is no member sets its key's bit in a second bitmap, `fresh`;
// the fresh keys' places are the numbers of fresh bits below them, so each
// fresh key has a word of the dense array `first`, where the earliest arrival
// wins by atomicMin, and each kept row goes straight to its sorted place.
//   claim   rank index, member bit, fresh bit         (xs[p], fresh, dirty)
//   scan    fresh bits per line and superblock, scanned over the dirty
//           superblocks                               (linep, sbpre)
//   first   place of the key, earliest arrival        (pos[p], first)
//   place   kept rows counted by bucket in arrival order (look-back), ids, rows
//           at their places; fresh, dirty and first are left as they were
// Why: scattered atomics run at about 23 G/s on the device whatever they do
// (36 us for 846 K of them), but lanes that share a cache line share the
// transaction (14 us), and keys of neighbouring candidates are neighbours in
// a bitmap and in `first`, while their hash slots are not.  The hash form
// (claim, decision, scan, scatter and bin sort of the 150x150 grid, 846 K
// candidates an iteration) took 118 us, this form 88 us.

// fresh bits below bit x
__device__ __forceinline__ u32 pra_fresh_rank(const RankArgs& a, u64 x)
{
    u32 r = a.sbpre[x >> PRA_SB_BITS] + a.linep[x >> PRA_LINE_BITS];
    const ulonglong2* line = (const ulonglong2*)a.fresh + (x >> PRA_LINE_BITS) * 4;
    const u32 bit = (u32)(x & ((1u << PRA_LINE_BITS) - 1)), wi = bit >> 6;
    ulonglong2 v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = line[k];
#pragma unroll
    for (u32 k = 0; k < 8; k++) {
        const u64 m = k < wi ? ~0ULL : k == wi ? (1ULL << (bit & 63)) - 1 : 0;
        r += (u32)__popcll((k & 1 ? v[k >> 1].y : v[k >> 1].x) & m);
    }
    return r;
}

__device__ __forceinline__ void pra_rank_claim_key(const RankArgs& a, u64 p, u64 x)
{
    const u32 bit = 1u << (x & 31);
    if (a.member[x >> 5] & bit) {
        a.xs[p] = ~0ULL;
        return;
    }
    a.xs[p] = x;
    if (!(a.fresh[x >> 5] & bit)) {
        atomicOr(a.fresh + (x >> 5), bit);
        u32* d = a.dirty + (x >> PRA_SB_BITS);
        if (!*d) *d = 1;
    }
}

__device__ __forceinline__ void pra_rank_claim_one(const RankArgs& a, u64 p)
{
    u64 x;
    if (!pra_dense_index_n(a.kw, a.cand + p * a.kw, a.dict, a.dict_cap, a.D, a.by_bucket, &x))
        atomicCAS((unsigned long long*)(a.ctl + 1), 0ULL, 3ULL);
    else
        pra_rank_claim_key(a, p, x);
}

// digits of a rank index x < 2^35 in radix D < 2^32: x = q * D + rest
__device__ __forceinline__ void pra_digit_split(u64 x, u64 D, double inv, u64* q, u32* rest)
{
    u64 k = (u64)((double)x * inv);   // within one of the quotient
    long long r = (long long)(x - k * D);
    if (r < 0) {
        k--;
        r += (long long)D;
    } else if (r >= (long long)D) {
        k++;
        r -= (long long)D;
    }
    *q = k;
    *rest = (u32)r;
}

// Emission and claims of a ranked output with one rule, a join of a delta
// whose rows' rank indexes are known with a static inner relation whose rows
// are ranked (RankArgs::EmitArgs), in one launch: tiles of outer rows in ticket
// order find their offsets by look-back over the tiles' match counts, and each
// match's rank index is put together from digits, without a hash, a value or
// a candidate row.  With one rule the arrival position of an output is its
// emission offset.  The last tile leaves the candidate count, the capacity
// flag (1: over the capacity; 4: over the join threshold, so the arrival plan
// decides) and the join pairs.  A tile past the capacity claims nothing; the
// bits of the tiles before it are those the re-run sets again.
// Why: count, plan, expansion and claim as four launches took 69 us on the
// 150x150 grid's 430 K rows and 846 K matches, mostly key hashes, dictionary
// probes and candidate rows written and read back; this takes 30 us, bound by
// the lines of the two bitmaps (63 MB each).
#define PRA_EMIT_MLP 4   // 1, 2, 4: 10,000-vertex graph 6.03, 5.91, 5.84 ms, 150x150 grid 41.6, 42.2, 42.1 ms
__device__ __forceinline__ void pra_rank_emit_tile(const RankArgs& a, u64* status, u32 tile, u32 ntiles, u32 epoch,
                                                   u32* flags)
{
    constexpr int SW = PRA_EMIT_BLOCK / 64;
    __shared__ u32 lds[SW + 1];
    __shared__ u64 s_excl;
    const EmitArgs& em = a.emit;
    const u64 i = (u64)tile * PRA_EMIT_BLOCK + threadIdx.x;
    u32 digit[4] = {0, 0, 0, 0};
    u32 i0 = 0, cnt = 0;
    if (i < em.n) {
        u64 x = em.dx[i];
#pragma unroll
        for (int c = 3; c > 0; c--)
            if (c < em.kwo) pra_digit_split(x, a.D, em.inv, &x, &digit[c]);
        digit[0] = (u32)x;
        i0 = em.first[digit[0]];
        cnt = em.first[digit[0] + 1] - i0;
    }
    u32 tot;
    const u32 ex = block_exclusive_scan<u32, SW>(cnt, lds, &tot);
    if (threadIdx.x < 64) {
        u64 excl = 0;
        if (threadIdx.x == 0)
            __hip_atomic_store(status + tile, st_pack(epoch, tile == 0 ? PRA_ST_INC : PRA_ST_AGG, tot), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        if (tile != 0) {
            excl = pra_lookback_wave(status, tile, epoch, flags, 1);
            if (threadIdx.x == 0)
                __hip_atomic_store(status + tile, st_pack(epoch, PRA_ST_INC, excl + tot), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        if (threadIdx.x == 0) {
            s_excl = excl;
            if (tile == ntiles - 1) {
                const u64 total = excl + tot;
                const u64 st = total > em.cap ? 1 : (long long)total > em.thresh ? 4 : 0;
                a.ctl[0] = total;
                a.ctl[1] = st;
                if (!st && total) atomicAdd((unsigned long long*)em.joined, (unsigned long long)total);
            }
        }
    }
    __syncthreads();
    if (s_excl + tot > em.cap) return;
    // the digits that come from the outer row
    u64 base = 0;
    for (int c = 0; c < a.kw; c++) {
        u32 d = 0;
        if (em.side[c] == 0) {
            const int q = em.col[c];
            d = q == 0 ? digit[0] : q == 1 ? digit[1] : q == 2 ? digit[2] : digit[3];
            if (em.conv[c] == 1) d = em.rank_of[d];        // leading digit -> rank
            else if (em.conv[c] == 2) d = em.lead_of[d];   // rank -> leading digit
        }
        base = base * a.D + d;
    }
    // the row's matches, PRA_EMIT_MLP at a time with their loads in flight
    // together (a match's chain is inner words, member word, fresh word, atomic)
    const u64 p0 = s_excl + ex;
    for (u32 j0 = 0; j0 < cnt; j0 += PRA_EMIT_MLP) {
        u64 x[PRA_EMIT_MLP];
        u32 mw[PRA_EMIT_MLP], fw[PRA_EMIT_MLP];
#pragma unroll
        for (int q = 0; q < PRA_EMIT_MLP; q++) {
            x[q] = 0;
            if (j0 + q < cnt)
                for (int c = 0; c < a.kw; c++) {
                    u32 d = 0;
                    if (em.side[c] == 1) {
                        const u64 e = em.words[(u64)(i0 + j0 + q) * em.ia + em.col[c]];
                        d = c == 0 && a.by_bucket ? (u32)(e >> 32) : (u32)e - 1;
                    }
                    x[q] = x[q] * a.D + d;
                }
            x[q] += base;
        }
#pragma unroll
        for (int q = 0; q < PRA_EMIT_MLP; q++) {
            mw[q] = fw[q] = ~0u;
            if (j0 + q < cnt) {
                mw[q] = a.member[x[q] >> 5];
                fw[q] = a.fresh[x[q] >> 5];
            }
        }
#pragma unroll
        for (int q = 0; q < PRA_EMIT_MLP; q++) {
            if (j0 + q >= cnt) continue;
            const u32 bit = 1u << (x[q] & 31);
            const bool member = mw[q] & bit;
            a.xs[p0 + j0 + q] = member ? ~0ULL : x[q];
            if (!member && !(fw[q] & bit)) {
                atomicOr(a.fresh + (x[q] >> 5), bit);
                u32* d = a.dirty + (x[q] >> PRA_SB_BITS);
                if (!*d) *d = 1;
            }
        }
    }
}

__global__ void k_rank_claim(RankArgs a)
{
    if (a.ctl[1]) return;
    const u64 p = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (p < a.ctl[0]) pra_rank_claim_one(a, p);
}

// Chunk `chunk` of the scan: an equal share of the superblocks, a wave to each
// dirty one, a lane to each of its 512-bit lines.  A clean superblock costs its
// flag, so large rank spaces with few new keys stay cheap; there are at most
// PRA_SCAN_CHUNKS chunks, since the tickets of a launch are atomics on one
// word (about 10 ns each) and a look-back step reads 64 of them.
__device__ __forceinline__ void pra_rank_scan_chunk(const RankArgs& a, u64* status, u32 chunk, u32 epoch, u32* flags)
{
    constexpr int SB = PRA_SCAN_BLOCK, SW = SB / 64, PER = 4, MAX = PRA_SCAN_CHUNK_MAX / SB;
    __shared__ u32 cnt[PRA_SCAN_CHUNK_MAX];
    __shared__ unsigned short list[PRA_SCAN_CHUNK_MAX];
    __shared__ u32 lds[SW + 1], s_n, s_excl;
    const u32 per = (a.sbs + a.chunks - 1) / a.chunks;
    const u32 c0 = chunk * per, size = c0 < a.sbs ? min(per, a.sbs - c0) : 0;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    for (u32 i = threadIdx.x; i < size; i += SB) {
        cnt[i] = 0;
        if (a.dirty[c0 + i]) {
            list[atomicAdd(&s_n, 1u)] = (unsigned short)i;
            a.dirty[c0 + i] = 0;
        }
    }
    __syncthreads();
    const u32 nd = s_n;
    for (u32 j0 = (u32)wave * PER; j0 < nd; j0 += SW * PER) {
        u32 c[PER];
#pragma unroll
        for (int q = 0; q < PER; q++) {
            c[q] = 0;
            if (j0 + q < nd) {
                const u64 sb = c0 + list[j0 + q];
                const ulonglong2* line = (const ulonglong2*)a.fresh + (sb * 64 + lane) * 4;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const ulonglong2 v = line[k];
                    c[q] += (u32)(__popcll(v.x) + __popcll(v.y));
                }
            }
        }
#pragma unroll
        for (int q = 0; q < PER; q++) {
            if (j0 + q >= nd) break;
            u32 x = c[q];
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const u32 y = __shfl_up(x, d, 64);
                if (lane >= d) x += y;
            }
            const u32 i = list[j0 + q];
            a.linep[(u64)(c0 + i) * 64 + lane] = (unsigned short)(x - c[q]);
            if (lane == 63) cnt[i] = x;
        }
    }
    __syncthreads();
    // MAX consecutive superblocks a thread
    u32 v[MAX], sum = 0, tot;
#pragma unroll
    for (int k = 0; k < MAX; k++) {
        const u32 i = threadIdx.x * MAX + k;
        v[k] = i < size ? cnt[i] : 0;
        sum += v[k];
    }
    const u32 ex = block_exclusive_scan<u32, SW>(sum, lds, &tot);
    if (wave == 0) {
        u64 excl = 0;
        if (lane == 0)
            __hip_atomic_store(status + chunk, st_pack(epoch, chunk == 0 ? PRA_ST_INC : PRA_ST_AGG, tot),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (chunk != 0) {
            excl = pra_lookback_wave(status, chunk, epoch, flags, 1);
            if (lane == 0)
                __hip_atomic_store(status + chunk, st_pack(epoch, PRA_ST_INC, excl + tot), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        if (lane == 0) s_excl = (u32)excl;
    }
    __syncthreads();
    u32 run = s_excl + ex;
#pragma unroll
    for (int k = 0; k < MAX; k++) {
        const u32 i = threadIdx.x * MAX + k;
        if (i < size) a.sbpre[c0 + i] = run;
        run += v[k];
    }
}

// a block's place in launch order among the `takers` blocks that take one; the
// block taking the last returns the counter to zero
__device__ __forceinline__ u32 pra_ticket(u32* ctr, u32 takers)
{
    __shared__ u32 s_ticket;
    if (threadIdx.x == 0) {
        const u32 t = atomicAdd(ctr, 1u);
        if (t == takers - 1) atomicExch(ctr, 0u);
        s_ticket = t;
    }
    __syncthreads();
    return s_ticket;
}

__global__ __launch_bounds__(PRA_EMIT_BLOCK) void k_rank_emit(RankArgs a, u64* status, u32* ctr, u32 epoch, u32* flags)
{
    const u32 t = pra_ticket(ctr, gridDim.x);
    pra_rank_emit_tile(a, status, t, gridDim.x, epoch, flags);
}

__global__ __launch_bounds__(PRA_SCAN_BLOCK) void k_rank_scan(RankArgs a, u64* status, u32* ctr, u32 epoch,
                                                              u32* flags)
{
    const u32 t = pra_ticket(ctr, gridDim.x);
    if (a.ctl[1]) return;
    pra_rank_scan_chunk(a, status, t, epoch, flags);
}

__device__ __forceinline__ void pra_rank_first_one(const RankArgs& a, u64 p)
{
    const u64 x = a.xs[p];
    u32 r = ~0u;
    if (x != ~0ULL) {
        r = pra_fresh_rank(a, x);
        if (a.first[r] > (u32)p) atomicMin(a.first + r, (u32)p);
    }
    a.pos[p] = r;
}

__global__ void k_rank_first(RankArgs a)
{
    if (a.ctl[1]) return;
    const u64 p = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (p < a.ctl[0]) pra_rank_first_one(a, p);
}

// The summary of an iteration of one ranked output, to the host as
// pra_publish_words does it, by one thread: the words the host reads of it.
__device__ __forceinline__ void pra_publish_ranked(const RankArgs& a, u64 new_rows)
{
    a.host[0] = new_rows;
    a.host[4] = a.ctl[0];
    a.host[5] = a.ctl[1];
    a.host[a.host_words] = *a.err;
    __threadfence_system();
    __hip_atomic_store(a.host - 1, a.host_seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Tile `tile` of the placement (PRA_TILE candidates by PRA_PLACE_BLOCK
// threads).  The tile of the last candidate also writes the output's totals:
// its new tuples, the advanced seq counters (into the copy the next iteration
// reads) and the bucket bounds of the new rows.
__device__ __forceinline__ void pra_rank_place_tile(const RankArgs& a, u64* status, u32 tile, u32 epoch, u32* flags)
{
    constexpr int SB = PRA_PLACE_BLOCK, SW = SB / 64, IT = PRA_TILE / SB;
    __shared__ u32 wh[SW][PRA_RADIX];
    __shared__ u32 s_base[PRA_RADIX];
    __shared__ u32 lds[SW + 1];
    const u64 n = a.ctl[0];
    const u32 last = n ? (u32)((n - 1) / PRA_TILE) : 0;
    const u32 nb = a.nb;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const u64 lt = pra_lanemask_lt();
    const u64 base = (u64)tile * PRA_TILE + (u64)wave * 64 * IT;
    u32 pos[IT], dg[IT], lc[IT];
    bool kept[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const u64 p = base + (u64)k * 64 + lane;
        pos[k] = p < n ? a.pos[p] : ~0u;
    }
#pragma unroll
    for (int k = 0; k < IT; k++)
        kept[k] = pos[k] != ~0u && a.first[pos[k]] == (u32)(base + (u64)k * 64 + lane);
    // the kept rows' values, by their digits, and buckets (of the leading digit,
    // or, with more join columns, the candidate's), loaded before the barriers
    u64 x[IT], row[IT][4];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const u64 p = base + (u64)k * 64 + lane;
        x[k] = kept[k] ? a.xs[p] : 0;
    }
#pragma unroll
    for (int k = 0; k < IT; k++) {
        dg[k] = 0;
        if (!kept[k]) continue;
        u64 q = x[k];
#pragma unroll
        for (int c = 3; c > 0; c--)
            if (c < a.kw) {
                u32 d;
                pra_digit_split(q, a.D, a.inv, &q, &d);
                row[k][c] = a.vals[d];
            }
        row[k][0] = a.lead_vals[q];
        if (nb > 1) dg[k] = a.by_bucket ? (u32)a.bucket[q] : a.dest[base + (u64)k * 64 + lane];
    }
    for (u32 i = lane; i < nb; i += 64) wh[wave][i] = 0;
    // (a wave counts in its own row of wh, in lane order within each item)
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const u64 act = __ballot(kept[k]);
        const u64 peers = nb > 1 ? pra_match<PRA_RADIX_BITS>(dg[k], act) : act;
        lc[k] = 0;
        if (kept[k]) {
            const u32 before = wh[wave][dg[k]];
            lc[k] = before + (u32)__popcll(peers & lt);
            if ((peers >> lane) == 1ULL) wh[wave][dg[k]] = before + (u32)__popcll(peers);
        }
    }
    __syncthreads();
    u32 acc = 0;
    const u32 d0 = threadIdx.x;
    if (d0 < nb) {
        for (int v = 0; v < SW; v++) {
            const u32 t = wh[v][d0];
            wh[v][d0] = acc;
            acc += t;
        }
        __hip_atomic_store(status + (u64)tile * PRA_RADIX + d0, st_pack(epoch, tile == 0 ? PRA_ST_INC : PRA_ST_AGG, acc),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (nb <= 2 * SW) {
        // few buckets: a wave looks back for each, 64 tiles a step
        for (u32 d = wave; d < nb; d += SW) {
            const u32 e = tile ? (u32)pra_lookback_wave(status + d, tile, epoch, flags) : 0u;
            if (lane == 0) s_base[d] = e;
        }
    } else if (d0 < nb) {
        s_base[d0] = tile ? (u32)pra_lookback(status, tile, (int)d0, epoch, flags) : 0u;
    }
    __syncthreads();
    if (d0 < nb && tile)
        __hip_atomic_store(status + (u64)tile * PRA_RADIX + d0, st_pack(epoch, PRA_ST_INC, (u64)s_base[d0] + acc),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int k = 0; k < IT; k++) {
        if (!kept[k]) continue;
        const u32 d = dg[k];
        const u64 seq = a.seq[d] + s_base[d] + wh[wave][d] + lc[k];
        u64* dst = a.newt + (u64)pos[k] * a.wn;
#pragma unroll
        for (int c = 0; c < 4; c++)
            if (c < a.kw) dst[c] = row[k][c];
        dst[a.kw] = ((u64)a.tag << 46) | ((u64)d << 28) | seq;
        if (a.nx) a.nx[pos[k]] = x[k];
        atomicOr(a.member + (x[k] >> 5), 1u << (x[k] & 31));
        // back to the state between iterations: the word's fresh bits are all
        // of this iteration, and no other arrival equals ~0
        a.fresh[x[k] >> 5] = 0;
        a.first[pos[k]] = ~0u;
    }
    if (tile != last) return;
    u32 tot;
    const u32 mine = d0 < nb ? s_base[d0] + acc : 0u;
    const u32 ex = block_exclusive_scan<u32, SW>(mine, lds, &tot);
    if (d0 < nb) {
        a.seq_next[d0] = a.seq[d0] + mine;
        if (a.bnd) a.bnd[d0] = ex;
    }
    if (d0 == 0) {
        if (a.bnd) a.bnd[nb] = tot;
        a.stat[0] = tot;
        if (a.host) pra_publish_ranked(a, tot);
    }
}

__global__ __launch_bounds__(PRA_PLACE_BLOCK) void k_rank_place(RankArgs a, u64* status, u32* ctr, u32 epoch,
                                                                u32* flags)
{
    // only the blocks that have candidates (and the first) take a ticket
    if (a.ctl[1]) {
        if (a.host && blockIdx.x == 0 && threadIdx.x == 0) pra_publish_ranked(a, 0);
        return;
    }
    const u64 n = a.ctl[0];
    const u32 tiles = n ? (u32)((n + PRA_TILE - 1) / PRA_TILE) : 1;
    if (blockIdx.x >= tiles) return;
    const u32 t = pra_ticket(ctr, tiles);
    pra_rank_place_tile(a, status, t, epoch, flags);
}

// exclusive prefix of one value a thread over the block's SW waves; every wave
// adds up the others' totals itself (two barriers)
template <int SW>
__device__ __forceinline__ u32 pra_block_prefix(u32 v, u32* lds, u32* total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    u32 x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const u32 y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) lds[wave] = x;
    __syncthreads();
    u32 w = lds[lane & (SW - 1)];
#pragma unroll
    for (int d = 1; d < SW; d <<= 1) {
        const u32 y = __shfl_up(w, d, SW);
        if ((lane & (SW - 1)) >= d) w += y;
    }
    *total = __shfl(w, SW - 1, SW);
    const u32 before = wave ? __shfl(w, wave - 1, SW) : 0u;
    __syncthreads();
    return before + x - v;
}

// x = q * D + rest for x < 2^25: M = ceil(2^32 / D) puts the quotient at most
// one too high (x * M / 2^32 < x / D + 2^-7)
__device__ __forceinline__ u32 pra_split32(u32 x, u32 D, u32 M, u32* rest)
{
    u32 q = __umulhi(x, M), r = x - q * D;
    if ((int)r < 0) {
        q--;
        r += D;
    }
    *rest = r;
    return q;
}

// Whole iterations of a small ranked output that emits in digits from its own
// delta, one after another, by one block: what k_rank_emit .. k_rank_place do,
// with the delta's rank indexes, the candidates, the earliest arrivals and the
// seq counters in LDS, so that an iteration has neither a launch nor a wait of
// the host.  The loop ends at an empty iteration (the caller's fixed point),
// after max_iters, or, with nothing of it done, before an iteration of more
// than max_cand candidates, over the join threshold, or without room for its
// rows; the general steps take that one.
// A compute unit has one random access in flight after another (about three
// cycles a lane), which bounds it, so a candidate costs two: it sets its bit
// in the fresh bitmap without a look at the members, and finds its place in
// `places`, a 64-bit word for each 32 bits of a dirty superblock (the bits that
// are new, and their count before them).  One pass over the dirty superblocks
// in between takes the members out, adds the new keys to them, clears the
// fresh bits and leaves those words.  Digits are 32-bit here, and a row's
// matches are spread over the block before anything is looked up.  New rows
// are written in trie order, each iteration's after the last's, where the full
// log will have them.
// A closure of 1,000 vertices, 49 iterations of 3,700 rows and 4,400
// candidates on average: 45 us an iteration by the general launches and the
// readback, 24 us here (14 us of it the passes over bitmaps and `places`);
// one of 40 vertices 45 against 9 us.
__device__ __forceinline__ void pra_rank_loop(const LoopArgs& a)
{
    constexpr int SB = PRA_LOOP_BLOCK, SW = SB / 64, IT = PRA_LOOP_ROWS / SB, MLP = 4;
    __shared__ u32 va[PRA_LOOP_ROWS];   // the delta's rank indexes; inner rows; earliest arrivals; the new rank indexes
    __shared__ u32 vb[PRA_LOOP_ROWS];   // outer digits, then rank indexes of the candidates; the new rows' seq offsets
    __shared__ u32 wh[SW][PRA_RADIX];
    __shared__ u32 sbpre[PRA_LOOP_SBS];
    __shared__ unsigned short list[PRA_LOOP_SBS];
    __shared__ u32 dirty[PRA_LOOP_SBS / 32];
    __shared__ u32 lds[SW], s_run[PRA_RADIX], s_nd;
    __shared__ u64 s_seq[PRA_RADIX];
    __shared__ unsigned char s_bucket[PRA_LOOP_LEADS];   // of each leading digit (several buckets)
    const EmitArgs& em = a.emit;
    const u32 t = threadIdx.x, nb = a.nb, D = (u32)a.D, M = 0xFFFFFFFFu / D + 1;
    const int lane = t & 63, wave = t >> 6, kw = a.kw, wn = a.wn, ia = em.ia;
    const u64 lt = pra_lanemask_lt();
    const int dbits = nb > 1 ? 32 - __clz(nb - 1) : 0;
    u64* const dx = (u64*)em.dx;
    const u32* const first = em.first;
    const u64 *const words = em.words, *const vals = a.vals, *const lead_vals = a.lead_vals;
    const u32 *const rank_of = em.rank_of, *const lead_of = em.lead_of;
    u32* const fresh = a.fresh;
    u64* const places = a.places;
    // what each digit of the outer row adds to an output's rank index: as it
    // is, its leading digit as a rank, one of its ranks as a leading digit;
    // and each column of the inner row
    u32 wo[4] = {0, 0, 0, 0}, wrank = 0, wlead = 0, wi[4], ci[4];
    int qlead = 0;
    {
        u32 w = 1;
#pragma unroll
        for (int c = 3; c >= 0; c--) {
            wi[c] = 0;
            ci[c] = 0;
            if (c >= kw) continue;
            const int q = em.col[c];
            if (em.side[c] == 1) {
                wi[c] = w;
                ci[c] = q;
            } else if (em.conv[c] == 1) {
                wrank += w;
            } else if (em.conv[c] == 2) {   // (of output column 0)
                wlead = w;
                qlead = q;
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++) wo[k] += q == k ? w : 0;
            }
            w *= D;
        }
    }
    const bool inner_lead = a.by_bucket && wi[0];
    u32 n = (u32)em.n, it = 0, cand = 0;
    u64 written = 0, joined = 0;
    bool too_many = false;
    for (u32 r = t; r < n; r += SB) va[r] = (u32)dx[r];
    for (u32 i = t; nb > 1 && i < D; i += SB) s_bucket[i] = a.bucket[i];
    if (t < nb) {
        s_seq[t] = a.seq[t];
        s_run[t] = 0;
    }
    __syncthreads();
    while (it < a.max_iters && n) {
        // each row's inner run and the digits it gives: consecutive rows a
        // thread, so that threads in order are rows in order
        const u32 per = (n + SB - 1) / SB, r0 = t * per;
        u32 base[IT], run[IT];   // run: first inner row, then in the top bits how many
        u32 cnt = 0;
#pragma unroll
        for (int k0 = 0; k0 < IT; k0 += MLP) {
            u32 f[MLP], e[MLP];
#pragma unroll
            for (int q = 0; q < MLP; q++) base[k0 + q] = run[k0 + q] = f[q] = e[q] = 0;
            if ((u32)k0 >= per) continue;
#pragma unroll
            for (int q = 0; q < MLP; q++) {
                // (past the last row: row 0 again, counted as none)
                const bool in = (u32)(k0 + q) < per && r0 + k0 + q < n;
                u32 digit[4] = {0, 0, 0, 0}, x = va[in ? r0 + k0 + q : 0];
#pragma unroll
                for (int c = 3; c > 0; c--)
                    if (c < kw) x = pra_split32(x, D, M, &digit[c]);
                digit[0] = x;
                f[q] = first[x];
                e[q] = first[in ? x + 1 : x];
                u32 b = 0;
#pragma unroll
                for (int c = 0; c < 4; c++)
                    if (c < kw) b += digit[c] * wo[c];
                if (wrank) b += rank_of[digit[0]] * wrank;
                if (wlead) {
                    const u32 d = qlead == 0 ? digit[0] : qlead == 1 ? digit[1] : qlead == 2 ? digit[2] : digit[3];
                    b += lead_of[d] * wlead;
                }
                base[k0 + q] = b;
            }
#pragma unroll
            for (int q = 0; q < MLP; q++) {
                run[k0 + q] = f[q] | (e[q] - f[q]) << PRA_LOOP_RUN_SHIFT;
                cnt += e[q] - f[q];
            }
        }
        if (t < PRA_LOOP_SBS / 32) dirty[t] = 0;
        if (t == 0) s_nd = 0;
        u32 tot, p = pra_block_prefix<SW>(cnt, lds, &tot);
        if (tot > a.max_cand || (long long)tot > em.thresh) {
            too_many = true;
            break;
        }
        if (written + tot > a.room) break;
        // the candidates in arrival order: outer digits and inner row
#pragma unroll
        for (int k = 0; k < IT; k++) {
            if ((u32)k >= per) continue;
            const u32 len = run[k] >> PRA_LOOP_RUN_SHIFT, i0 = run[k] & ((1u << PRA_LOOP_RUN_SHIFT) - 1);
            for (u32 j = 0; j < len; j++, p++) {
                va[p] = i0 + j;
                vb[p] = base[k];
            }
        }
        __syncthreads();
        // claims: the candidates' bits
        for (u32 p0 = t; p0 < tot; p0 += SB * MLP) {
            u32 x[MLP];
#pragma unroll
            for (int q = 0; q < MLP; q++) {
                const u32 pq = p0 + q * SB < tot ? p0 + q * SB : p0;   // (past the last: its own first again)
                const u64* w = words + (u64)va[pq] * ia;
                x[q] = vb[pq];
#pragma unroll
                for (int c = 0; c < 4; c++)
                    if (wi[c]) {
                        const u64 e = w[ci[c]];
                        x[q] += (c == 0 && inner_lead ? (u32)(e >> 32) : (u32)e - 1) * wi[c];
                    }
            }
#pragma unroll
            for (int q = 0; q < MLP; q++) {
                const u32 pq = p0 + q * SB, sb = x[q] >> PRA_SB_BITS;
                if (pq >= tot) continue;
                __hip_atomic_fetch_or(fresh + (x[q] >> 5), 1u << (x[q] & 31), __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_WORKGROUP);
                if (!(*(volatile u32*)(dirty + (sb >> 5)) >> (sb & 31) & 1)) atomicOr(dirty + (sb >> 5), 1u << (sb & 31));
                va[pq] = ~0u;
                vb[pq] = x[q];
            }
        }
        __syncthreads();
        // a wave to each dirty superblock, in four steps of whole lines: its
        // new keys, into the members, and their places
        if (t < a.sbs) {
            sbpre[t] = 0;
            if (dirty[t >> 5] >> (t & 31) & 1) list[atomicAdd(&s_nd, 1u)] = (unsigned short)t;
        }
        __syncthreads();
        const u32 nd = s_nd;
        for (u32 j = wave; j < nd; j += SW) {
            const u32 sb = list[j];
            uint4* const fw = (uint4*)fresh + (u64)sb * 256 + lane;
            uint4* const mw = (uint4*)a.member + (u64)sb * 256 + lane;
            uint4 v[4], m[4];
            u32 c[4];
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = fw[k * 64];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                c[k] = v[k].x | v[k].y | v[k].z | v[k].w;
                m[k] = make_uint4(0, 0, 0, 0);
                if (c[k]) m[k] = mw[k * 64];
            }
            u32 x01, x23;   // counts of the steps, two to a register: a step's 64 lanes hold at most 8,192 bits
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if (c[k]) {
                    fw[k * 64] = make_uint4(0, 0, 0, 0);
                    v[k].x &= ~m[k].x;
                    v[k].y &= ~m[k].y;
                    v[k].z &= ~m[k].z;
                    v[k].w &= ~m[k].w;
                    mw[k * 64] = make_uint4(m[k].x | v[k].x, m[k].y | v[k].y, m[k].z | v[k].z, m[k].w | v[k].w);
                }
            }
            u32 cnt4[4];
#pragma unroll
            for (int k = 0; k < 4; k++)
                cnt4[k] = (u32)(__popc(v[k].x) + __popc(v[k].y) + __popc(v[k].z) + __popc(v[k].w));
            x01 = cnt4[0] | cnt4[1] << 16;
            x23 = cnt4[2] | cnt4[3] << 16;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const u32 y01 = __shfl_up(x01, d, 64), y23 = __shfl_up(x23, d, 64);
                if (lane >= d) {
                    x01 += y01;
                    x23 += y23;
                }
            }
            const u32 t01 = __shfl(x01, 63, 64), t23 = __shfl(x23, 63, 64);
            const u32 s1 = t01 & 0xFFFF, s2 = s1 + (t01 >> 16), s3 = s2 + (t23 & 0xFFFF);
            const u32 o[4] = {(x01 & 0xFFFF) - cnt4[0], s1 + (x01 >> 16) - cnt4[1], s2 + (x23 & 0xFFFF) - cnt4[2],
                              s3 + (x23 >> 16) - cnt4[3]};
            uint4* const pw = (uint4*)places + ((u64)sb * 256 + lane) * 2;
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (c[k]) {
                    const u32 o1 = o[k] + (u32)__popc(v[k].x), o2 = o1 + (u32)__popc(v[k].y),
                              o3 = o2 + (u32)__popc(v[k].z);
                    pw[k * 128] = make_uint4(v[k].x, o[k], v[k].y, o1);
                    pw[k * 128 + 1] = make_uint4(v[k].z, o2, v[k].w, o3);
                }
            if (lane == 0) sbpre[sb] = s3 + (t23 >> 16);
        }
        __syncthreads();
        u32 fresh_rows;
        const u32 sbex = pra_block_prefix<SW>(t < a.sbs ? sbpre[t] : 0u, lds, &fresh_rows);
        if (t < a.sbs) sbpre[t] = sbex;
        __syncthreads();
        // the earliest arrival of each key: consecutive candidates a wave
        const u32 items = (tot + SB - 1) / SB, p1 = (u32)wave * 64 * items + lane;
        u32 xk[IT], pos[IT];
#pragma unroll
        for (int k0 = 0; k0 < IT; k0 += 2 * MLP) {
            uint2 w[2 * MLP];
#pragma unroll
            for (int q = 0; q < 2 * MLP; q++) xk[k0 + q] = pos[k0 + q] = ~0u;
            if ((u32)k0 >= items) continue;
#pragma unroll
            for (int q = 0; q < 2 * MLP; q++) {
                w[q] = make_uint2(0, 0);
                const u32 pk = p1 + (k0 + q) * 64;
                if ((u32)(k0 + q) < items && pk < tot) {
                    xk[k0 + q] = vb[pk];
                    w[q] = ((const uint2*)places)[xk[k0 + q] >> 5];
                }
            }
#pragma unroll
            for (int q = 0; q < 2 * MLP; q++) {
                const u32 x = xk[k0 + q], bit = 1u << (x & 31);
                if (w[q].x & bit) {   // (else a member, or no candidate)
                    pos[k0 + q] = sbpre[x >> PRA_SB_BITS] + w[q].y + (u32)__popc(w[q].x & (bit - 1));
                    atomicMin(va + pos[k0 + q], p1 + (k0 + q) * 64);
                }
            }
        }
        for (u32 i = lane; i < nb; i += 64) wh[wave][i] = 0;
        __syncthreads();
        // seq offsets of the kept candidates: per wave in arrival order, then
        // over the waves
        u32 dl[IT];   // bucket, and the kept candidates of it before this one in the wave
#pragma unroll
        for (int k = 0; k < IT; k++) {
            dl[k] = ~0u;
            if ((u32)k >= items) continue;
            if (pos[k] != ~0u && va[pos[k]] == p1 + k * 64) {
                dl[k] = 0;
                if (nb > 1) {
                    u32 x = xk[k], rest;
#pragma unroll
                    for (int c = 3; c > 0; c--)
                        if (c < kw) x = pra_split32(x, D, M, &rest);
                    dl[k] = s_bucket[x];
                }
            }
        }
#pragma unroll
        for (int k = 0; k < IT; k++) {
            if ((u32)k >= items) continue;
            const bool kept = dl[k] != ~0u;
            u64 peers = __ballot(kept);
            for (int b = 0; b < dbits; b++) {
                const u64 set = __ballot(dl[k] >> b & 1);
                peers &= dl[k] >> b & 1 ? set : ~set;
            }
            if (kept) {
                const u32 d = dl[k], before = wh[wave][d];
                dl[k] = d | (before + (u32)__popcll(peers & lt)) << 8;
                if ((peers >> lane) == 1ULL) wh[wave][d] = before + (u32)__popcll(peers);
            }
        }
        __syncthreads();
        if (t < nb) {
            u32 c[SW], acc = s_run[t];
#pragma unroll
            for (int v = 0; v < SW; v++) c[v] = wh[v][t];
#pragma unroll
            for (int v = 0; v < SW; v++) {
                wh[v][t] = acc;
                acc += c[v];
            }
            s_run[t] = acc;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < IT; k++)
            if (dl[k] != ~0u) {
                va[pos[k]] = xk[k];
                vb[pos[k]] = wh[wave][dl[k] & 255] + (dl[k] >> 8);
            }
        __syncthreads();
        // the new rows, in order
        for (u32 rr = t; rr < fresh_rows; rr += SB * MLP) {
            u32 lead[MLP];
            u64 row[MLP][4];
#pragma unroll
            for (int q = 0; q < MLP; q++) {
                const u32 r = rr + q * SB;
                u32 y = va[r < fresh_rows ? r : 0];   // (past the last: row 0 again, not written)
#pragma unroll
                for (int c = 3; c > 0; c--)
                    if (c < kw) {
                        u32 d;
                        y = pra_split32(y, D, M, &d);
                        row[q][c] = vals[d];
                    }
                lead[q] = y;
                row[q][0] = lead_vals[y];
            }
#pragma unroll
            for (int q = 0; q < MLP; q++) {
                const u32 r = rr + q * SB;
                if (r >= fresh_rows) continue;
                const u32 d = nb > 1 ? s_bucket[lead[q]] : 0;
                u64* dst = a.rows + (written + r) * wn;
#pragma unroll
                for (int c = 0; c < 4; c++)
                    if (c < kw) dst[c] = row[q][c];
                dst[kw] = ((u64)a.tag << 46) | ((u64)d << 28) | (s_seq[d] + vb[r]);
            }
        }
        written += fresh_rows;
        joined += tot;
        cand = tot;
        n = fresh_rows;
        if (t == 0) ((u32*)(a.out + 4))[it] = n;
        it++;
    }
    // the last iteration's rank indexes are in `va`
    __syncthreads();
    if (it)
        for (u32 r = t; r < n; r += SB) dx[r] = va[r];
    if (t < nb) a.seq[t] = s_seq[t] + s_run[t];
    if (t == 0) {
        a.out[0] = it;
        a.out[1] = written;
        a.out[2] = n;
        a.out[3] = (u64)too_many << 32 | cand;
        if (joined) atomicAdd((unsigned long long*)em.joined, (unsigned long long)joined);
    }
    if (!a.host) return;
    __syncthreads();
    if (t == 0) a.host[a.host_words] = *a.err;
    pra_publish_words(a.out, 4 + (it + 1) / 2, a.err, a.host, a.host_seq);
}

__global__ __launch_bounds__(PRA_LOOP_BLOCK) void k_rank_loop(LoopArgs a) { pra_rank_loop(a); }
__global__ __launch_bounds__(PRA_LOOP_BLOCK) void k_rank_loop_many(const LoopArgs* jobs) { pra_rank_loop(jobs[blockIdx.x]); }

// Several outputs in one launch each: `jobs` (device memory) holds njobs
// RankArgs, then five tables of njobs + 1 first blocks, one a step (outputs
// that emit have no claim blocks, the others no emission tiles).
__global__ __launch_bounds__(PRA_EMIT_BLOCK) void k_rank_emit_many(const RankArgs* jobs, int njobs, u64* status,
                                                                   u32* ctr, u32 epoch, u32* flags)
{
    const u32* base = (const u32*)(jobs + njobs) + PRA_RANK_EMIT * (njobs + 1);
    const u32 t = pra_ticket(ctr, gridDim.x);
    const int k = pra_job_of(base, njobs, t);
    const RankArgs a = jobs[k];
    pra_rank_emit_tile(a, status + base[k], t - base[k], base[k + 1] - base[k], epoch, flags);
}

__global__ void k_rank_claim_many(const RankArgs* jobs, int njobs)
{
    const u32* base = (const u32*)(jobs + njobs) + PRA_RANK_CLAIM * (njobs + 1);
    const int k = pra_job_of(base, njobs, blockIdx.x);
    const RankArgs* jp = jobs + k;
    const u64 p = (u64)(blockIdx.x - base[k]) * blockDim.x + threadIdx.x;
    if (jp->ctl[1] || p >= jp->ctl[0]) return;
    pra_rank_claim_one(*jp, p);
}

__global__ __launch_bounds__(PRA_SCAN_BLOCK) void k_rank_scan_many(const RankArgs* jobs, int njobs, u64* status,
                                                                   u32* ctr, u32 epoch, u32* flags)
{
    const u32* base = (const u32*)(jobs + njobs) + PRA_RANK_SCAN * (njobs + 1);
    const u32 t = pra_ticket(ctr, gridDim.x);
    const int k = pra_job_of(base, njobs, t);
    const RankArgs* jp = jobs + k;
    if (jp->ctl[1]) return;
    pra_rank_scan_chunk(*jp, status + base[k], t - base[k], epoch, flags);
}

__global__ void k_rank_first_many(const RankArgs* jobs, int njobs)
{
    const u32* base = (const u32*)(jobs + njobs) + PRA_RANK_FIRST * (njobs + 1);
    const int k = pra_job_of(base, njobs, blockIdx.x);
    const RankArgs* jp = jobs + k;
    const u64 p = (u64)(blockIdx.x - base[k]) * blockDim.x + threadIdx.x;
    if (jp->ctl[1] || p >= jp->ctl[0]) return;
    pra_rank_first_one(*jp, p);
}

__global__ __launch_bounds__(PRA_PLACE_BLOCK) void k_rank_place_many(const RankArgs* jobs, int njobs, u64* status,
                                                                     u32* ctr, u32 epoch, u32* flags)
{
    const u32* base = (const u32*)(jobs + njobs) + PRA_RANK_PLACE * (njobs + 1);
    const u32 t = pra_ticket(ctr, gridDim.x);
    const int k = pra_job_of(base, njobs, t);
    const RankArgs a = jobs[k];
    const u32 tile = t - base[k];
    if (a.ctl[1] || (tile && (u64)tile * PRA_TILE >= a.ctl[0])) return;
    pra_rank_place_tile(a, status + (u64)base[k] * PRA_RADIX, tile, epoch, flags);
}

// Combine the PRA_NREP replicas of the scatter summaries and reset them to
// their identity values for the next scatter.  Part 0 (packed keys): the
// top-byte bin counters, whose exclusive offsets go to kgofs and whose
// largest count goes to stat[6]; the counters return to zero.  Part 1:
// summary words -> stat[1..3] (packed key OR / AND / dictionary miss) and
// stat[8..39] (key column OR / AND).  Part 2: the kept total -> stat[0], and
// the seq counters advance by the new tuples of each bucket (bucket d's rows
// start at offs[d * nblocks]).  PRA_BLOCK threads; counters and replicas are
// read by atomic exchange, so the scatter's own block may run it too.
// NW waves, at least PRA_WAVES; threads past PRA_BLOCK only keep the barriers.
template <int NW = PRA_WAVES>
__device__ inline void pra_newt_fold_part(const NewtFoldArgs& a, u32 y, u32 t, u32* lds, u32* mx)
{
    if (y == 0) {
        if (!a.packed) return;
        const u32 v = t < PRA_BLOCK ? atomicExch(&a.bin_cur[t], 0u) : 0u;
        u32 tot;
        const u32 ex = block_exclusive_scan<u32, NW>(v, lds, &tot);
        if (t < PRA_BLOCK) a.kgofs[t] = ex;
        if (t == 0) *mx = 0;
        __syncthreads();
        if (v) atomicMax(mx, v);
        __syncthreads();
        if (t == 0) a.stat[6] = *mx;
    } else if (y == 1) {
        if (t < PRA_PART_WORDS && !(t >= 3 && t < 8)) {
            const bool is_and = pra_summary_is_and(t);
            const u64 id = is_and ? ~0ULL : 0;
            u64 v = id;
            for (int r = 0; r < PRA_NREP; r++) {
                unsigned long long* p = (unsigned long long*)(a.rep_words + (u64)r * PRA_PART_WORDS + t);
                const u64 x = atomicExch(p, (unsigned long long)id);
                v = is_and ? (v & x) : (v | x);
            }
            a.stat[t < 3 ? t + 1 : t] = v;
        }
    } else {
        if (t == 0) a.stat[0] = *a.total;
        if (t < a.nb && a.intern) {
            const u32 start = a.offs[(u64)t * a.nblocks];
            const u32 end = t + 1 < a.nb ? a.offs[(u64)(t + 1) * a.nblocks] : *a.total;
            a.seqbase[t] += (u64)(end - start);
        }
    }
}

// k_newt_fold's three parts in one block after the scatter of a single tile
template <int NW>
__device__ inline void pra_scatter_fold_tail(const NewtFoldArgs& f)
{
    __shared__ u32 flds[NW + 1];
    __shared__ u32 fmx;
    __syncthreads();
    for (u32 y = 0; y < 3; y++) {
        pra_newt_fold_part<NW>(f, y, threadIdx.x, flds, &fmx);
        __syncthreads();
    }
}

// Stable partition of the kept candidates by destination bucket; JOIN-type
// rows get their intern id tag<<46 | bucket<<28 | seq, seq counted per
// (tag, bucket) in arrival order (src/RAM/RA_tasks.cpp:858-875).
template <bool PACKED, int SB>
__device__ __forceinline__ void pra_scatter_block(NewtScatterArgs& a, const u32 bid)
{
    // PRA_TILE candidates per block: SB threads of IT items, SW waves
    constexpr int SW = SB / 64, IT = PRA_TILE / SB;
    if (a.ctl[1]) return;
    a.n = a.ctl[0];
    // blocks past the candidates hold nothing; the summary reduce skips them
    if ((u64)bid * PRA_TILE >= a.n) {
        if (a.fold_here) pra_scatter_fold_tail<SW>(a.fold);
        return;
    }
    __shared__ u32 wh[SW][PRA_RADIX];
    for (int i = threadIdx.x; i < SW * PRA_RADIX; i += SB) (&wh[0][0])[i] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const u64 lt = pra_lanemask_lt();
    u64 base = (u64)bid * PRA_TILE + (u64)wave * (PRA_TILE / SW);
    u32 dg[IT], lc[IT], kept = 0;
#pragma unroll
    for (int k = 0; k < IT; k++) {
        u64 p = base + (u64)k * 64 + lane;
        bool valid = p < a.n && a.keep[p];
        kept |= (valid ? 1u : 0u) << k;
        u32 d = valid ? a.dest[p] : 0u;
        u64 act = __ballot(valid);
        u64 peers = pra_match<PRA_RADIX_BITS>(d, act);
        dg[k] = d;
        lc[k] = 0;
        if (valid) {
            u32 before = wh[wave][d];
            lc[k] = before + (u32)__popcll(peers & lt);
            if ((peers >> lane) == 1ULL) wh[wave][d] = before + (u32)__popcll(peers);
        }
    }
    // the wide form loads the kept rows' words (up to PW) and rank indexes
    // now, so that they arrive while the block forms its offsets and bin
    // counts (loads are not moved across the barriers in between)
    constexpr int PW = SB == PRA_SCATTER_BLOCK ? 2 : 0;
    const bool pre_rows = PW > 0 && a.cw <= PW;
    u64 prow[IT][PW > 0 ? PW : 1], pxk[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const u64 p = base + (u64)k * 64 + lane;
        pxk[k] = 0;
        if ((kept >> k) & 1u) {
            if (PACKED && PW > 0 && a.xk) pxk[k] = a.xk[p];
            if (pre_rows)
#pragma unroll
                for (int c = 0; c < (PW > 0 ? PW : 1); c++)
                    if (c < a.cw) prow[k][c] = a.cand[p * a.cw + c];
        }
    }
    __syncthreads();
    for (u32 d = threadIdx.x; d < a.nb; d += SB) {
        u32 acc = a.offs[(u64)d * a.nblocks + bid];
        for (int v = 0; v < SW; v++) {
            u32 t = wh[v][d];
            wh[v][d] = acc;
            acc += t;
        }
    }
    __syncthreads();
    // per-block summaries: the packed key's OR / AND / dictionary miss and the
    // block's share of each top-byte bin (packed mode), or the key columns'
    // OR / AND
    __shared__ u32 khist[PRA_RADIX];
    __shared__ u64 red[SW][PRA_PART_WORDS];
    constexpr bool packed = PACKED;
    if (packed)
        for (int i = threadIdx.x; i < PRA_RADIX; i += SB) khist[i] = 0;
    __syncthreads();
    // key columns summarised (unpacked, when asked): the first 16; later ones
    // report the identity values (OR 0, AND all ones), which the host reads as
    // "varies"
    constexpr int NC = PACKED ? 1 : 16;
    const int kc = !a.summarize ? 0 : a.cw < NC ? a.cw : NC;
    u64 kor = 0, kand = ~0ULL, kmiss = 0;
    u64 o[NC], an[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) { o[c] = 0; an[c] = ~0ULL; }
    // packed keys: from the rank index the dense decision left, or else the
    // column ranks of all items are looked up column by column with every
    // item's first probe in flight at once (a dictionary slot resolves at its
    // first probe unless its chain is longer)
    u64 K[PACKED ? IT : 1];
    u32 lr[PACKED ? IT : 1];
    if (packed) {
        if (a.xk) {
#pragma unroll
            for (int k = 0; k < IT; k++) {
                K[k] = 0;
                if ((kept >> k) & 1u)
                    K[k] = (u64)dg[k] * a.xk_scale + (PW > 0 ? pxk[k] : a.xk[base + (u64)k * 64 + lane]);
            }
        } else {
#pragma unroll
            for (int k = 0; k < IT; k++) K[k] = dg[k];
            for (int c = 0; c < a.cw; c++) {
                u64 v[IT], e[IT], r1[IT];
#pragma unroll
                for (int k = 0; k < IT; k++) {
                    v[k] = e[k] = r1[k] = 0;
                    if ((kept >> k) & 1u) v[k] = a.cand[(base + (u64)k * 64 + lane) * a.cw + c];
                }
#pragma unroll
                for (int k = 0; k < IT; k++)
                    if ((kept >> k) & 1u) {
                        const u64* sl = a.dict + 2 * pra_dict_slot(v[k], a.dict_cap);
                        e[k] = sl[0];
                        r1[k] = sl[1];
                    }
#pragma unroll
                for (int k = 0; k < IT; k++)
                    if ((kept >> k) & 1u) {
                        u64 r = 0;
                        if (r1[k] != 0 && e[k] == v[k])
                            r = (u32)r1[k] - 1;
                        else if (!pra_dict_rank(a.dict, a.dict_cap, v[k], &r))
                            kmiss = 1;
                        K[k] = K[k] * a.rank_radix + r;
                    }
            }
        }
        // every row's (key, newt position) goes to the bin of the key's top
        // byte: a rank inside the block's share of the bin, then one counter
        // reservation per bin and block
#pragma unroll
        for (int k = 0; k < IT; k++) {
            K[k] <<= a.key_lshift;
            if ((kept >> k) & 1u) lr[k] = atomicAdd(&khist[K[k] >> 56], 1u);
        }
        __syncthreads();
        for (int i = threadIdx.x; i < PRA_RADIX; i += SB)
            if (khist[i]) khist[i] = atomicAdd(a.bin_cur + i, khist[i]);
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < IT; k++) {
        u64 p = base + (u64)k * 64 + lane;
        if ((kept >> k) & 1u) {
            u32 d = dg[k];
            u64 pos = (u64)wh[wave][d] + lc[k];
            const u64* src = a.cand + p * a.cw;
            u64* dst = a.newt + pos * a.wn;
            if (pre_rows) {
#pragma unroll
                for (int c = 0; c < (PW > 0 ? PW : 1); c++)
                    if (c < a.cw) dst[c] = prow[k][c];
            } else {
                pra_copy_row(dst, src, a.cw);
            }
            if (a.intern) {
                u64 rank = pos - a.offs[(u64)d * a.nblocks];
                u64 key = ((u64)a.tag << 46) | ((u64)d << 28);
                dst[a.cw] = key | (a.seqbase[d] + rank);
            }
            if (packed) {
                const u64 Kk = K[PACKED ? k : 0];
                a.keys[pos] = Kk;
                kor |= Kk;
                kand &= Kk;
                const u32 bin = (u32)(Kk >> 56), slot = khist[bin] + lr[PACKED ? k : 0];
                if (slot < a.bin_cap) {
                    a.bin_keys[(u64)bin * a.bin_cap + slot] = Kk;
                    a.bin_idx[(u64)bin * a.bin_cap + slot] = (u32)pos;
                }
            } else {
#pragma unroll
                for (int c = 0; c < NC; c++)
                    if (c < kc) { o[c] |= src[c]; an[c] &= src[c]; }
            }
        }
    }
#pragma unroll
    for (int dd = 32; dd >= 1; dd >>= 1) {
        kor |= __shfl_xor(kor, dd, 64);
        kand &= __shfl_xor(kand, dd, 64);
        kmiss |= __shfl_xor(kmiss, dd, 64);
    }
    if (!packed) {
#pragma unroll
        for (int c = 0; c < NC; c++) {
            if (c < kc) {
#pragma unroll
                for (int dd = 32; dd >= 1; dd >>= 1) {
                    o[c] |= __shfl_xor(o[c], dd, 64);
                    an[c] &= __shfl_xor(an[c], dd, 64);
                }
            }
        }
    }
    if (lane == 0) {
        red[wave][0] = kor;
        red[wave][1] = kand;
        red[wave][2] = kmiss;
#pragma unroll
        for (int c = 0; c < 16; c++) {
            red[wave][8 + c] = (!packed && c < kc) ? o[c < NC ? c : 0] : 0;
            red[wave][24 + c] = (!packed && c < kc) ? an[c < NC ? c : 0] : ~0ULL;
        }
    }
    __syncthreads();
    // fold into replica bid % PRA_NREP of the summaries (identity
    // values are not sent); k_newt_fold combines and resets the replicas
    const u32 rep = bid % PRA_NREP;
    if (threadIdx.x < PRA_PART_WORDS) {
        const int j = threadIdx.x;
        if (j < 3 || j >= 8) {
            u64 v = red[0][j];
            bool is_and = pra_summary_is_and(j);
            for (int w2 = 1; w2 < SW; w2++) v = is_and ? (v & red[w2][j]) : (v | red[w2][j]);
            unsigned long long* dst = (unsigned long long*)(a.rep_words + (u64)rep * PRA_PART_WORDS + j);
            if (is_and && v != ~0ULL) atomicAnd(dst, (unsigned long long)v);
            if (!is_and && v != 0) atomicOr(dst, (unsigned long long)v);
        }
    }
    if (a.fold_here) pra_scatter_fold_tail<SW>(a.fold);
}

template <bool PACKED, int SB>
__global__ __launch_bounds__(SB) void k_dedup_scatter(NewtScatterArgs a)
{
    pra_scatter_block<PACKED, SB>(a, blockIdx.x);
}

// Partitions of several outputs' candidates in one launch (tiles of few items a
// thread: points-to analysis, 256 threads of 8 items 22.9 us a launch, 1,024 of
// 2 items 15.5): the jobs' arguments and block ranges are read from device memory
// (njobs arguments, then njobs + 1 block bases), a block serving the job whose
// range holds it as k_dedup_scatter serves its one output.
template <bool PACKED>
__global__ __launch_bounds__(PRA_SCATTER_BLOCK) void k_dedup_scatter_many(const NewtScatterArgs* jobs, int njobs)
{
    const u32* block_base = (const u32*)(jobs + njobs);
    // the job: the number of later jobs' block bases at or below this block,
    // 64 bases per load round
    int k = 0;
    for (int j0 = 1; j0 < njobs; j0 += 64) {
        const int j = j0 + (int)(threadIdx.x & 63);
        k += __popcll(__ballot(j < njobs && block_base[j] <= blockIdx.x));
    }
    NewtScatterArgs a = jobs[k];
    pra_scatter_block<PACKED, PRA_SCATTER_BLOCK>(a, blockIdx.x - block_base[k]);
}

// The folds of several outputs in one launch: block b runs part b % 3 of job
// b / 3 (job table in device memory).
__global__ void k_newt_fold_many(const NewtFoldArgs* jobs)
{
    const NewtFoldArgs& a = jobs[blockIdx.x / 3];
    if (a.ctl[1]) return;
    __shared__ u32 lds[PRA_WAVES + 1];
    __shared__ u32 mx;
    pra_newt_fold_part(a, blockIdx.x % 3, threadIdx.x, lds, &mx);
}

// One block per part of pra_newt_fold_part.
__global__ void k_newt_fold(NewtFoldArgs a)
{
    if (a.ctl[1]) return;
    __shared__ u32 lds[PRA_WAVES + 1];
    __shared__ u32 mx;
    pra_newt_fold_part(a, blockIdx.x, threadIdx.x, lds, &mx);
}

// The last output's fold and then the iteration's summary publication
// (k_publish) in one block: the fold's parts run in turn (skipped, as in
// k_newt_fold, when the output overflowed its candidate capacity), then
// `words` summary words and the error flags go to pinned host memory.
__global__ void k_newt_fold_publish(NewtFoldArgs a, const u64* src, u64 words, const u32* flags, u64* host, u64 seq)
{
    __shared__ u32 lds[PRA_WAVES + 1];
    __shared__ u32 mx;
    if (!a.ctl[1])
        for (u32 y = 0; y < 3; y++) {
            pra_newt_fold_part(a, y, threadIdx.x, lds, &mx);
            __syncthreads();
        }
    pra_publish_words(src, words, flags, host, seq);
}

// identity values of the summary replicas (all counts 0, OR words 0, AND
// words all ones)
__global__ void k_newt_rep_init(u64* rep_words)
{
    u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < PRA_NREP * PRA_PART_WORDS) rep_words[i] = pra_summary_is_and(i % PRA_PART_WORDS) ? ~0ULL : 0;
}

// ----------------------------------------- membership table maintenance -----

// Insert keys of already-present rows (minpos 0).  Duplicate keys (rows that
// differ only after the key) land on the same slot and are skipped.
__global__ void k_table_insert_rows(const u64* rows, u64 n, int w, int kw, u64* table, u64 cap, u32* flags)
{
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const u64* key = rows + i * w;
    const int stride = 2 + kw;
    u64 h = pra_keyhash(key, kw);
    u64 m = cap - 1, s = h & m;
    for (u64 q = 0; q < cap; q++) {
        u64* slot = table + s * stride;
        u64 cur = atomicCAS((unsigned long long*)slot, 0ULL, (unsigned long long)h);
        if (cur == 0) {
            slot[1] = 0;
            for (int c = 0; c < kw; c++) slot[2 + c] = key[c];
            return;
        }
        if (cur == h) return;
        s = (s + 1) & m;
    }
    atomicOr(flags, PRA_FLAG_TABLE_FULL);
}

__global__ void k_table_verify_rows(const u64* rows, u64 n, int w, int kw, const u64* table, u64 cap, u32* flags)
{
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const u64* key = rows + i * w;
    const int stride = 2 + kw;
    u64 h = pra_keyhash(key, kw);
    u64 m = cap - 1, s = h & m;
    for (u64 q = 0; q < cap; q++) {
        const u64* slot = table + s * stride;
        if (slot[0] == h) {
            for (int c = 0; c < kw; c++)
                if (slot[2 + c] != key[c]) { atomicOr(flags, PRA_FLAG_COLLISION); break; }
            return;
        }
        if (slot[0] == 0) { atomicOr(flags, PRA_FLAG_COLLISION); return; }
        s = (s + 1) & m;
    }
}

__global__ void k_table_rehash(const u64* old, u64 oldcap, u64* nt, u64 cap, int kw, u32* flags)
{
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= oldcap) return;
    const int stride = 2 + kw;
    const u64* os = old + i * stride;
    u64 h = os[0];
    if (h == 0) return;
    u64 m = cap - 1, s = h & m;
    for (u64 q = 0; q < cap; q++) {
        u64* slot = nt + s * stride;
        u64 cur = atomicCAS((unsigned long long*)slot, 0ULL, (unsigned long long)h);
        if (cur == 0) {
            slot[1] = 0;
            for (int c = 0; c < kw; c++) slot[2 + c] = os[2 + c];
            return;
        }
        s = (s + 1) & m;
    }
    atomicOr(flags, PRA_FLAG_TABLE_FULL);
}

// ------------------------------------------------------- launch wrappers ---

static inline unsigned grid_for(u64 n, unsigned bs = PRA_BLOCK)
{
    u64 g = (n + bs - 1) / bs;
    return (unsigned)(g ? g : 1);
}

void pra_launch_fill_u64(hipStream_t st, u64* p, u64 n, u64 v)
{
    if (!n) return;
    u64 g = (n + PRA_BLOCK - 1) / PRA_BLOCK;
    if (g > 65536) g = 65536;
    hipLaunchKernelGGL(k_fill_u64, dim3((unsigned)g), dim3(PRA_BLOCK), 0, st, p, n, v);
}

void pra_launch_table_clear(hipStream_t st, u64* t, u64 cap, int stride)
{
    u64 g = (cap + PRA_BLOCK - 1) / PRA_BLOCK;
    if (g > 65536) g = 65536;
    hipLaunchKernelGGL(k_table_clear, dim3((unsigned)(g ? g : 1)), dim3(PRA_BLOCK), 0, st, t, cap, stride);
}


// one block scans inputs of up to PRA_SMALL_SCAN elements, every thread
// holding a run of consecutive elements in registers
template <typename T>
__global__ void k_scan_small(const T* in, T* out, u64 n, T* total)
{
    constexpr int PER = PRA_SMALL_SCAN / PRA_BLOCK;
    __shared__ T lds[PRA_WAVES + 1];
    const u64 base = (u64)threadIdx.x * PER;
    T v[PER];
    T sum = 0;
#pragma unroll
    for (int k = 0; k < PER; k++) {
        v[k] = base + k < n ? in[base + k] : 0;
        sum += v[k];
    }
    T tot;
    T ex = block_exclusive_scan<T>(sum, lds, &tot);
#pragma unroll
    for (int k = 0; k < PER; k++) {
        if (base + k < n) out[base + k] = ex;
        ex += v[k];
    }
    if (threadIdx.x == 0 && total) *total = tot;
}

// Exclusive scans of several u32 arrays of at most PRA_SMALL_SCAN elements in
// one launch, one block each (job table in device memory).
__global__ void k_scan_small_many(const ScanJob* jobs)
{
    const ScanJob& j = jobs[blockIdx.x];
    constexpr int PER = PRA_SMALL_SCAN / PRA_BLOCK;
    __shared__ u32 lds[PRA_WAVES + 1];
    const u64 base = (u64)threadIdx.x * PER;
    u32 v[PER];
    u32 sum = 0;
#pragma unroll
    for (int k = 0; k < PER; k++) {
        v[k] = base + k < j.n ? j.in[base + k] : 0;
        sum += v[k];
    }
    u32 tot;
    u32 ex = block_exclusive_scan<u32>(sum, lds, &tot);
#pragma unroll
    for (int k = 0; k < PER; k++) {
        if (base + k < j.n) j.out[base + k] = ex;
        ex += v[k];
    }
    if (threadIdx.x == 0 && j.total) *j.total = tot;
}

// Word copies of several ranges in one launch: job k takes blocks
// [block_base[k], block_base[k + 1]), 8 words per thread (block_base follows
// the job table in device memory).
__global__ void k_copy_many(const CopyJob* jobs, int njobs)
{
    const u32* block_base = (const u32*)(jobs + njobs);
    const int k = pra_job_of(block_base, njobs, blockIdx.x);
    const CopyJob j = jobs[k];
    const u64 i0 = ((u64)(blockIdx.x - block_base[k]) * PRA_BLOCK + threadIdx.x) * 8;
    u64 t[8];
#pragma unroll
    for (int q = 0; q < 8; q++)
        if (i0 + q < j.words) t[q] = j.src[i0 + q];
#pragma unroll
    for (int q = 0; q < 8; q++)
        if (i0 + q < j.words) j.dst[i0 + q] = t[q];
}

// One-pass exclusive scan: tiles of PRA_TILE elements are taken in ticket
// order; each publishes its sum, finds the sum of the tiles before it by
// decoupled look-back (digit 0 of the sort's status words), publishes its
// inclusive prefix and writes its outputs.  Prefixes must stay below 2^46
// (PRA_FLAG_SCAN_OVERFLOW otherwise).
template <typename T>
__global__ void k_scan_lookback(const T* in, T* out, u64 n, u64* status, u32* tile_ctr, u32 epoch, u32* flags,
                                T* total)
{
    __shared__ T lds[PRA_WAVES + 1];
    __shared__ u32 s_tile;
    __shared__ u64 s_excl;
    if (threadIdx.x == 0) {
        u32 t = atomicAdd(tile_ctr, 1u);
        if (t == gridDim.x - 1) atomicExch(tile_ctr, 0u);
        s_tile = t;
    }
    __syncthreads();
    const u32 tile = s_tile;
    const u64 base = (u64)tile * PRA_TILE + (u64)threadIdx.x * PRA_ITEMS;
    T v[PRA_ITEMS];
    T sum = 0;
#pragma unroll
    for (int k = 0; k < PRA_ITEMS; k++) {
        v[k] = base + k < n ? in[base + k] : 0;
        sum += v[k];
    }
    T tot;
    T ex = block_exclusive_scan<T>(sum, lds, &tot);
    if (threadIdx.x < 64) {
        constexpr u64 LIM = 1ULL << 46;
        u64* my = status + (u64)tile * PRA_RADIX;
        const u64 agg = (u64)tot;
        u64 excl = 0;
        if (threadIdx.x == 0) {
            if (agg >= LIM) atomicOr(flags, PRA_FLAG_SCAN_OVERFLOW);
            __hip_atomic_store(my, st_pack(epoch, tile == 0 ? PRA_ST_INC : PRA_ST_AGG, agg & (LIM - 1)),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (tile != 0) {
            excl = pra_lookback_wave(status, tile, epoch, flags);
            if (threadIdx.x == 0) {
                if (excl + agg >= LIM) atomicOr(flags, PRA_FLAG_SCAN_OVERFLOW);
                __hip_atomic_store(my, st_pack(epoch, PRA_ST_INC, (excl + agg) & (LIM - 1)), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (threadIdx.x == 0) {
            s_excl = excl;
            if (tile == gridDim.x - 1 && total) *total = (T)(excl + agg);
        }
    }
    __syncthreads();
    T run = (T)s_excl + ex;
#pragma unroll
    for (int k = 0; k < PRA_ITEMS; k++) {
        if (base + k < n) out[base + k] = run;
        run += v[k];
    }
}

// One tile (`tile` of `ntiles`, status words from `status`) of one rule's
// per-row output counts and their exclusive prefix sums.  PRA_CS_INDEX
// (join): a row's count is the length of its key's run of inner rows, found
// in the static inner's key index (istart = the run's first row);
// PRA_CS_SORTED (join): the same run searched in the inner's sorted rows;
// PRA_CS_FILTER (copy, copy_filter): 1 for rows passing the filter `op`.  A tile holds PRA_COUNT_SCAN_TILE rows (one
// a thread: a second one's search would wait for the first's) and finds its offset by
// decoupled look-back over digit 0 of the status words, as k_scan_lookback
// does; the last tile writes off[n] = total.
template <int KIND>
__device__ inline void pra_count_scan_tile(const CountScanArgs& a, u64* status, u32 tile, u32 ntiles, u32 epoch,
                                           u32* flags, u64* lds, u64* s_excl)
{
    constexpr int IT = PRA_COUNT_SCAN_TILE / PRA_COUNT_SCAN_BLOCK;
    constexpr int NW = PRA_COUNT_SCAN_BLOCK / 64;
    const u64 base = (u64)tile * PRA_COUNT_SCAN_TILE + (u64)threadIdx.x * IT;
    u64 c[IT];
    if (KIND == PRA_CS_SORTED) {
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const u64 i = base + k;
            c[k] = 0;
            if (i < a.n) {
                u64 first;
                c[k] = pra_sorted_run(a.outer + i * a.wo, a.jcc, a.inner, a.wi, a.ibnd, a.nb, &first);
                a.istart[i] = first;
            }
        }
    } else if (KIND == PRA_CS_INDEX) {
        // every item's key hash and first index slot are loaded before any
        // item walks on (a probe mostly ends at its first slot)
        const u64 m = a.cap - 1;
        u64 h[IT], f0[IT], f1[IT], f2[IT];
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const u64 i = base + k;
            h[k] = i < a.n && a.cap ? pra_keyhash(a.outer + i * a.wo, a.jcc) : 0;
        }
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const u64* sl = a.table + (h[k] & m) * 3;
            f0[k] = h[k] ? sl[0] : 0;
            f1[k] = h[k] ? sl[1] : 0;
            f2[k] = h[k] ? sl[2] : 0;
        }
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const u64 i = base + k;
            u64 cnt = 0, st = 0;
            if (h[k]) {
                const u64* key = a.outer + i * a.wo;
                u64 s = h[k] & m, sh = f0[k], ss = f1[k], sc = f2[k];
                for (u64 q = 0; q < a.cap && sh != 0; q++) {
                    if (sh == h[k]) {
                        const u64* f = a.inner + ss * a.wi;
                        bool eq = true;
                        for (int x = 0; x < a.jcc; x++)
                            if (f[x] != key[x]) { eq = false; break; }
                        if (eq) { cnt = sc; st = ss; }
                        break;
                    }
                    s = (s + 1) & m;
                    const u64* sl = a.table + s * 3;
                    sh = sl[0];
                    ss = sl[1];
                    sc = sl[2];
                }
            }
            c[k] = cnt;
            if (i < a.n) a.istart[i] = st;
        }
    } else {
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const u64 i = base + k;
            const u64* r = a.outer + i * a.wo;
            c[k] = i < a.n && pra_filter(a.op, r[0], r[1]) ? 1 : 0;
        }
    }
    u64 sum = 0;
#pragma unroll
    for (int k = 0; k < IT; k++) sum += c[k];
    u64 tot;
    const u64 ex = block_exclusive_scan<u64, NW>(sum, lds, &tot);
    if (threadIdx.x < 64) {
        constexpr u64 LIM = 1ULL << 46;
        u64* my = status + (u64)tile * PRA_RADIX;
        u64 excl = 0;
        if (threadIdx.x == 0) {
            if (tot >= LIM) atomicOr(flags, PRA_FLAG_SCAN_OVERFLOW);
            __hip_atomic_store(my, st_pack(epoch, tile == 0 ? PRA_ST_INC : PRA_ST_AGG, tot & (LIM - 1)),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (tile != 0) {
            excl = pra_lookback_wave(status, tile, epoch, flags);
            if (threadIdx.x == 0) {
                if (excl + tot >= LIM) atomicOr(flags, PRA_FLAG_SCAN_OVERFLOW);
                __hip_atomic_store(my, st_pack(epoch, PRA_ST_INC, (excl + tot) & (LIM - 1)), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (threadIdx.x == 0) {
            *s_excl = excl;
            if (tile == ntiles - 1) a.off[a.n] = excl + tot;
        }
    }
    __syncthreads();
    u64 run = *s_excl + ex;
#pragma unroll
    for (int k = 0; k < IT; k++) {
        if (base + k < a.n) a.off[base + k] = run;
        run += c[k];
    }
}

// Counts and scans of several rules in one launch: tiles are taken in ticket
// order; a block's ticket names its rule (the job whose tile range holds it)
// and its tile within that rule, whose look-back covers that rule's tiles.
__global__ __launch_bounds__(PRA_COUNT_SCAN_BLOCK) void k_count_scan_many(CountScanBatch b, u64* status,
                                                                          u32* tile_ctr, u32 epoch, u32* flags)
{
    __shared__ u64 lds[PRA_COUNT_SCAN_BLOCK / 64 + 1];
    __shared__ u32 s_tile;
    __shared__ int s_job;
    __shared__ u64 s_excl;
    if (threadIdx.x == 0) {
        u32 t = atomicAdd(tile_ctr, 1u);
        if (t == gridDim.x - 1) atomicExch(tile_ctr, 0u);
        int k = 0;
        while (k + 1 < b.njobs && b.tile_base[k + 1] <= t) k++;
        s_job = k;
        s_tile = t;
    }
    __syncthreads();
    const int k = s_job;
    const CountScanJob& j = b.job[k];
    CountScanArgs a;
    a.outer = j.outer;
    a.table = j.table;
    a.inner = j.inner;
    a.off = j.off;
    a.istart = j.istart;
    a.n = j.n;
    a.cap = j.cap;
    a.wo = j.wo;
    a.wi = j.wi;
    a.jcc = j.jcc;
    a.op = j.op;
    a.ibnd = j.ibnd;
    a.nb = j.nb;
    const u32 t0 = b.tile_base[k], nt = b.tile_base[k + 1] - t0;
    u64* st = status + (u64)t0 * PRA_RADIX;
    if (j.kind == PRA_CS_INDEX)
        pra_count_scan_tile<PRA_CS_INDEX>(a, st, s_tile - t0, nt, epoch, flags, lds, &s_excl);
    else if (j.kind == PRA_CS_SORTED)
        pra_count_scan_tile<PRA_CS_SORTED>(a, st, s_tile - t0, nt, epoch, flags, lds, &s_excl);
    else
        pra_count_scan_tile<PRA_CS_FILTER>(a, st, s_tile - t0, nt, epoch, flags, lds, &s_excl);
}

// kernel arguments of one launch are limited to 4 KiB
static_assert(sizeof(CountScanBatch) + 4 * sizeof(void*) <= 4096, "count-scan batch exceeds the kernel arguments");
static_assert(sizeof(SmallSortBatch) <= 4096, "small-sort batch exceeds the kernel arguments");
static_assert(sizeof(PlanAllArgs) <= 4096, "plan batch exceeds the kernel arguments");

void pra_launch_count_scan_many(hipStream_t st, const CountScanBatch& b, u64* status, u32* tile_ctr, u32 epoch,
                                u32* flags)
{
    if (b.njobs <= 0 || !b.tile_base[b.njobs]) return;
    hipLaunchKernelGGL(k_count_scan_many, dim3(b.tile_base[b.njobs]), dim3(PRA_COUNT_SCAN_BLOCK), 0, st, b, status,
                       tile_ctr, epoch, flags);
}

template <typename T>
static void scan_impl(hipStream_t st, const T* in, T* out, u64 n, u64* status, u32* tile_ctr, u32 epoch, u32* flags,
                      T* total)
{
    if (n <= PRA_SMALL_SCAN) {
        hipLaunchKernelGGL(k_scan_small<T>, dim3(1), dim3(PRA_BLOCK), 0, st, in, out, n, total);
        return;
    }
    hipLaunchKernelGGL(k_scan_lookback<T>, dim3(pra_tiles(n)), dim3(PRA_BLOCK), 0, st, in, out, n, status, tile_ctr,
                       epoch, flags, total);
}

void pra_scan_u64(hipStream_t st, const u64* in, u64* out, u64 n, u64* status, u32* tile_ctr, u32 epoch, u32* flags,
                  u64* total)
{
    scan_impl<u64>(st, in, out, n, status, tile_ctr, epoch, flags, total);
}

void pra_scan_u32(hipStream_t st, const u32* in, u32* out, u64 n, u64* status, u32* tile_ctr, u32 epoch, u32* flags,
                  u32* total)
{
    scan_impl<u32>(st, in, out, n, status, tile_ctr, epoch, flags, total);
}

u32 pra_tiles(u64 n) { return (u32)((n + PRA_TILE - 1) / PRA_TILE); }

void pra_launch_bucket_bounds(hipStream_t st, const u64* rows, u64 n, int w, int jcc, u64 nb, u64* bstart)
{
    hipLaunchKernelGGL(k_bucket_bounds, dim3(grid_for(nb + 1)), dim3(PRA_BLOCK), 0, st, rows, n, w, jcc, nb, bstart);
}

void pra_launch_group_flags(hipStream_t st, const u64* rows, u64 n, int w, int jcc, u64* flags)
{
    hipLaunchKernelGGL(k_group_flags, dim3(grid_for(n)), dim3(PRA_BLOCK), 0, st, rows, n, w, jcc, flags);
}

void pra_launch_group_compact(hipStream_t st, const u64* flags, const u64* gpos, u64 n, u64* gstart)
{
    hipLaunchKernelGGL(k_group_compact, dim3(grid_for(n + 1)), dim3(PRA_BLOCK), 0, st, flags, gpos, n, gstart);
}

void pra_launch_compact_rows(hipStream_t st, const u64* in, u64 n, int w, const u64* flags, const u64* pos, u64* out)
{
    if (!n) return;
    hipLaunchKernelGGL(k_compact_rows, dim3(grid_for(n)), dim3(PRA_BLOCK), 0, st, in, n, w, flags, pos, out);
}

void pra_launch_index_insert(hipStream_t st, const u64* rows, int w, int jcc, const u64* gstart, u64 ng, u64* table,
                             u64 cap, u32* flags)
{
    if (!ng) return;
    hipLaunchKernelGGL(k_index_insert, dim3(grid_for(ng)), dim3(PRA_BLOCK), 0, st, rows, w, jcc, gstart, ng, table,
                       cap, flags);
}

u32 pra_join_expand_blocks(u64 cap)
{
    u64 g = (cap + PRA_BLOCK - 1) / PRA_BLOCK;
    return (u32)(g > 16384 ? 16384 : g);
}

void pra_launch_join_expand(hipStream_t st, const JoinExpandArgs& a, u64 cap)
{
    if (!cap) return;
    hipLaunchKernelGGL(k_join_expand, dim3(pra_join_expand_blocks(cap)), dim3(PRA_BLOCK), 0, st, a);
}

void pra_launch_expand_many(hipStream_t st, const void* jobs, int njobs, u32 nblocks, bool join)
{
    if (njobs <= 0 || !nblocks) return;
    if (join)
        hipLaunchKernelGGL(k_join_expand_many, dim3(nblocks), dim3(PRA_BLOCK), 0, st, (const JoinExpandArgs*)jobs,
                           njobs);
    else
        hipLaunchKernelGGL(k_copy_expand_many, dim3(nblocks), dim3(PRA_BLOCK), 0, st, (const CopyExpandArgs*)jobs,
                           njobs);
}

void pra_launch_plan(hipStream_t st, const PlanArgs& a)
{
    hipLaunchKernelGGL(k_plan, dim3(1), dim3(PRA_BLOCK), 0, st, a);
}

void pra_launch_plan_all(hipStream_t st, const PlanAllArgs& a, int nblocks)
{
    if (nblocks > 0) hipLaunchKernelGGL(k_plan_all, dim3(nblocks), dim3(PRA_BLOCK), 0, st, a);
}

void pra_launch_plan_tab(hipStream_t st, const PlanTabArgs& a, int nouts)
{
    if (nouts > 0) hipLaunchKernelGGL(k_plan_tab, dim3(nouts), dim3(PRA_BLOCK), 0, st, a);
}

void pra_launch_find_split(hipStream_t st, const u64* off, u64 n, const u32* kp, long long thresh, u64* out)
{
    hipLaunchKernelGGL(k_find_split, dim3(1), dim3(1), 0, st, off, n, kp, thresh, out);
}

void pra_launch_newt_fold_publish(hipStream_t st, const NewtFoldArgs& a, const u64* src, u64 words,
                                  const u32* flags, u64* host, u64 seq)
{
    hipLaunchKernelGGL(k_newt_fold_publish, dim3(1), dim3(PRA_BLOCK), 0, st, a, src, words, flags, host, seq);
}

void pra_launch_publish(hipStream_t st, const u64* src, u64 words, const u32* flags, u64* host, u64 seq)
{
    hipLaunchKernelGGL(k_publish, dim3(1), dim3(PRA_BLOCK), 0, st, src, words, flags, host, seq);
}

void pra_launch_copy_expand(hipStream_t st, const CopyExpandArgs& a)
{
    if (!a.n) return;
    hipLaunchKernelGGL(k_copy_expand, dim3(grid_for(a.n)), dim3(PRA_BLOCK), 0, st, a);
}


void pra_launch_dedup_scatter(hipStream_t st, const NewtScatterArgs& a, int wide_choice)
{
    // many tiles: wide blocks hide the per-candidate loads; few tiles: narrow
    // blocks keep the per-block scans short (the autotuner may choose instead)
    const bool wide = wide_choice < 0 ? a.nblocks >= PRA_SCATTER_WIDE_TILES : wide_choice != 0;
    if (a.dict && wide)
        hipLaunchKernelGGL((k_dedup_scatter<true, PRA_SCATTER_BLOCK>), dim3(a.nblocks), dim3(PRA_SCATTER_BLOCK), 0, st,
                           a);
    else if (a.dict)
        hipLaunchKernelGGL((k_dedup_scatter<true, PRA_BLOCK>), dim3(a.nblocks), dim3(PRA_BLOCK), 0, st, a);
    else if (wide)
        hipLaunchKernelGGL((k_dedup_scatter<false, PRA_SCATTER_BLOCK>), dim3(a.nblocks), dim3(PRA_SCATTER_BLOCK), 0,
                           st, a);
    else
        hipLaunchKernelGGL((k_dedup_scatter<false, PRA_BLOCK>), dim3(a.nblocks), dim3(PRA_BLOCK), 0, st, a);
}

void pra_launch_dedup_scatter_many(hipStream_t st, const NewtScatterArgs* jobs, int njobs, u32 nblocks, bool packed)
{
    if (njobs <= 0 || !nblocks) return;
    if (packed)
        hipLaunchKernelGGL(k_dedup_scatter_many<true>, dim3(nblocks), dim3(PRA_SCATTER_BLOCK), 0, st, jobs, njobs);
    else
        hipLaunchKernelGGL(k_dedup_scatter_many<false>, dim3(nblocks), dim3(PRA_SCATTER_BLOCK), 0, st, jobs, njobs);
}

void pra_launch_table_insert_rows(hipStream_t st, const u64* rows, u64 n, int w, int kw, u64* table, u64 cap,
                                  u32* flags)
{
    if (!n) return;
    hipLaunchKernelGGL(k_table_insert_rows, dim3(grid_for(n)), dim3(PRA_BLOCK), 0, st, rows, n, w, kw, table, cap,
                       flags);
}

void pra_launch_table_verify_rows(hipStream_t st, const u64* rows, u64 n, int w, int kw, const u64* table, u64 cap,
                                  u32* flags)
{
    if (!n) return;
    hipLaunchKernelGGL(k_table_verify_rows, dim3(grid_for(n)), dim3(PRA_BLOCK), 0, st, rows, n, w, kw, table, cap,
                       flags);
}

void pra_launch_table_rehash(hipStream_t st, const u64* old, u64 oldcap, u64* nt, u64 cap, int kw, u32* flags)
{
    if (!oldcap) return;
    hipLaunchKernelGGL(k_table_rehash, dim3(grid_for(oldcap)), dim3(PRA_BLOCK), 0, st, old, oldcap, nt, cap, kw,
                       flags);
}

void pra_launch_sort_hist(hipStream_t st, const u64* rows, u64 n, int w, const PassList& pl, u32* ghist)
{
    u64 g = (n + PRA_BLOCK * 4 - 1) / (PRA_BLOCK * 4);
    if (g > 2048) g = 2048;
    if (g == 0) g = 1;
    size_t lds = (size_t)pl.np * PRA_RADIX * sizeof(u32);
    hipLaunchKernelGGL(k_sort_hist, dim3((unsigned)g), dim3(PRA_BLOCK), lds, st, rows, n, w, pl, ghist);
}

void pra_launch_sort_scan(hipStream_t st, const u32* ghist, int np, u32* gofs, u64* bnd, u32 nb, u64 n)
{
    hipLaunchKernelGGL(k_sort_scan, dim3(1), dim3(PRA_BLOCK), 0, st, ghist, np, gofs, bnd, nb, n);
}

// rows are sorted in tiles of PRA_TILE; (key, index) pairs in tiles of 2 x PRA_TILE
void pra_launch_sort_scatter(hipStream_t st, const u64* in, u64* out, u64 n, int w, DigitSpec ds, const u32* gofs,
                             u64* status, u32* tile_ctr, u32 epoch, u32* flags, const u32* iin, u32* iout)
{
    if (iout) {
        u32 nt = pra_tiles(n);
        hipLaunchKernelGGL((k_sort_scatter<true, PRA_ITEMS>), dim3(nt ? nt : 1), dim3(PRA_BLOCK), 0, st, in, out, n, w, ds,
                           gofs, status, tile_ctr, epoch, flags, iin, iout);
    } else {
        u32 nt = pra_tiles(n);
        hipLaunchKernelGGL((k_sort_scatter<false, PRA_ITEMS>), dim3(nt ? nt : 1), dim3(PRA_BLOCK), 0, st, in, out, n, w, ds,
                           gofs, status, tile_ctr, epoch, flags, iin, iout);
    }
}

void pra_launch_seg_bounds(hipStream_t st, const u64* keys, u64 n, int top, u32 nseg, u64* seg, u64* stat, u32* large)
{
    hipLaunchKernelGGL(k_seg_bounds, dim3(grid_for(nseg)), dim3(PRA_BLOCK), 0, st, keys, n, top, nseg, seg, stat,
                       large);
}

void pra_launch_seg_sort(hipStream_t st, const u64* keys, const u32* idx, const u64* seg, int top, u32 nseg, u64 n,
                         u32 bytes, const u64* rows, int w, u64* out, u64 bmul, int ls, u64 nb, u64* bnd, u32* flags,
                         u64 maxseg, const u32* large, u64 nlarge)
{
#define PRA_SEG_SORT(B, G, L, S)                                                                                     \
    hipLaunchKernelGGL(k_seg_sort<B>, dim3(G), dim3(B), 0, st, keys, idx, seg, top, n, bytes, rows, w, out, bmul, ls, \
                       nb, bnd, flags, L, S)
    static_assert(PRA_SEG_SMALL == 256 * PRA_BIN_ITEMS, "the small segments fit the 256-thread blocks");
    // every segment that fits the 256-thread blocks, then the larger ones
    PRA_SEG_SORT(256, nseg, (const u32*)nullptr, maxseg <= PRA_SEG_SMALL ? ~0u : (u32)PRA_SEG_SMALL);
    if (maxseg > PRA_SEG_SMALL && nlarge > 0) {
        if (maxseg <= 512 * PRA_BIN_ITEMS)
            PRA_SEG_SORT(512, nlarge, large, ~0u);
        else
            PRA_SEG_SORT(PRA_BIN_BLOCK, nlarge, large, ~0u);
    }
#undef PRA_SEG_SORT
}

void pra_launch_bin_sort(hipStream_t st, const u64* bin_keys, const u32* bin_idx, u32 bin_cap, u64 n, const u32* bofs,
                         u32 bytes, const u64* rows, int w, u64* out, u64 bmul, int ls, u64 nb, u64* bnd, u32* flags,
                         u64 maxbin)
{
#define PRA_BIN_SORT(B)                                                                                              \
    hipLaunchKernelGGL(k_bin_sort<B>, dim3(PRA_RADIX), dim3(B), 0, st, bin_keys, bin_idx, bin_cap, n, bofs, bytes, rows, \
                       w, out, bmul, ls, nb, bnd, flags)
    if (maxbin <= 256 * PRA_BIN_ITEMS)
        PRA_BIN_SORT(256);
    else if (maxbin <= 512 * PRA_BIN_ITEMS)
        PRA_BIN_SORT(512);
    else
        PRA_BIN_SORT(PRA_BIN_BLOCK);
#undef PRA_BIN_SORT
}

void pra_launch_sort_keys(hipStream_t st, const u64* rows, u64 n, int w, const KeyLayout& L, int np, u64* keys, u32* hist,
                          u64* missing)
{
    hipLaunchKernelGGL(k_sort_keys, dim3(std::min<unsigned>(grid_for(n), 2048)), dim3(PRA_BLOCK), 0, st, rows, n, w, L,
                       np, keys, hist, missing);
}

void pra_launch_keyseg_sort(hipStream_t st, const u64* keys, const u32* idx, const u64* seg, const u32* gofs, u32 nseg,
                            const u32* list, const u64* stat, int top, u64 n, const u64* rows, int w,
                            const KeyLayout& L, u64* out, u64* bnd, u64* status)
{
    hipLaunchKernelGGL(k_keyseg_small, dim3(nseg), dim3(PRA_BLOCK), 0, st, keys, idx, seg, gofs, top, n, rows, w, L,
                       out, bnd, status);
    hipLaunchKernelGGL(k_keyseg_large, dim3(std::min<u32>(nseg, 256)), dim3(PRA_BIN_BLOCK), 0, st, keys, idx, seg, gofs,
                       list, stat, top, n, rows, w, L, out, bnd, status);
}

void pra_launch_small_sort(hipStream_t st, const u64* rows, u64 n, int w, int jcc, int kc, u64 nb, int bucketed,
                           u64* out, u64* bnd, u64* dup)
{
    if (n <= 2 * PRA_BLOCK)
        hipLaunchKernelGGL(k_small_sort<PRA_BLOCK>, dim3(1), dim3(PRA_BLOCK), 0, st, rows, n, w, jcc, kc, nb, bucketed,
                           out, bnd, dup);
    else
        hipLaunchKernelGGL(k_small_sort<PRA_SMALL_SORT / 2>, dim3(1), dim3(PRA_SMALL_SORT / 2), 0, st, rows, n, w, jcc,
                           kc, nb, bucketed, out, bnd, dup);
}

void pra_launch_small_sort_many(hipStream_t st, const SmallSortBatch& b, int njobs)
{
    if (njobs <= 0) return;
    u64 most = 0;
    for (int k = 0; k < njobs; k++) most = std::max(most, b.job[k].n);
    if (most <= 2 * PRA_BLOCK)
        hipLaunchKernelGGL(k_small_sort_many<PRA_BLOCK>, dim3(njobs), dim3(PRA_BLOCK), 0, st, b);
    else
        hipLaunchKernelGGL(k_small_sort_many<PRA_SMALL_SORT / 2>, dim3(njobs), dim3(PRA_SMALL_SORT / 2), 0, st, b);
}

void pra_launch_block_sort(hipStream_t st, const u64* rows, u64 n, int w, const PassList& pl, u64* out, u64* bnd,
                           int jcc, u64 nb)
{
    hipLaunchKernelGGL(k_block_sort, dim3(1), dim3(PRA_BIN_BLOCK), 0, st, rows, n, w, pl, out, bnd, jcc, nb);
}

void pra_launch_collect_cols(hipStream_t st, const u64* rows, u64 n, int w, int ncols, u64* out)
{
    if (!n) return;
    hipLaunchKernelGGL(k_collect_cols, dim3(grid_for(n)), dim3(PRA_BLOCK), 0, st, rows, n, w, ncols, out);
}

void pra_launch_view_keep(hipStream_t st, const u64* rows, u64 n, int w, int ja, int jb, u64 nb, u32* keep)
{
    if (!n) return;
    hipLaunchKernelGGL(k_view_keep, dim3(grid_for(n)), dim3(PRA_BLOCK), 0, st, rows, n, w, ja, jb, nb, keep);
}

void pra_launch_view_compact(hipStream_t st, const u64* rows, u64 n, int w, const u32* keep, const u32* pos, u64* out)
{
    if (!n) return;
    hipLaunchKernelGGL(k_view_compact, dim3(grid_for(n)), dim3(PRA_BLOCK), 0, st, rows, n, w, keep, pos, out);
}

void pra_launch_dict_insert(hipStream_t st, const u64* vals, u64 n, u64* tab, u64 cap, u32* flags)
{
    if (!n) return;
    hipLaunchKernelGGL(k_dict_insert, dim3(grid_for(n)), dim3(PRA_BLOCK), 0, st, vals, n, tab, cap, flags);
}

void pra_launch_dict_small(hipStream_t st, const DictSmallArgs& a)
{
    hipLaunchKernelGGL(k_dict_small, dim3(1), dim3(1024), 0, st, a);
}

void pra_launch_dict_small_many(hipStream_t st, const DictSmallArgs* jobs, int njobs)
{
    hipLaunchKernelGGL(k_dict_small_many, dim3(njobs), dim3(1024), 0, st, jobs);
}

void pra_launch_index_small_many(hipStream_t st, const IndexSmallArgs* jobs, int njobs)
{
    hipLaunchKernelGGL(k_index_small_many, dim3(njobs), dim3(1024), 0, st, jobs);
}

void pra_launch_index_small(hipStream_t st, const IndexSmallArgs& a)
{
    hipLaunchKernelGGL(k_index_small, dim3(1), dim3(1024), 0, st, a);
}

void pra_launch_gather_rows(hipStream_t st, const u64* in, const u32* idx, u64 n, int w, u64* out)
{
    if (!n) return;
    hipLaunchKernelGGL(k_gather_rows, dim3(grid_for(n)), dim3(PRA_BLOCK), 0, st, in, idx, n, w, out);
}

void pra_launch_key_bounds(hipStream_t st, const u64* keys, u64 n, u64 bmul, int ls, u64 nb, u64* bnd)
{
    hipLaunchKernelGGL(k_key_bounds, dim3(grid_for(nb + 1)), dim3(PRA_BLOCK), 0, st, keys, n, bmul, ls, nb, bnd);
}

void pra_launch_col_orand2(hipStream_t st, const u64* rows, u64 n, int w, int kc, u64* out)
{
    u64 g = (n + PRA_BLOCK - 1) / PRA_BLOCK;
    if (g > 512) g = 512;
    if (g == 0) g = 1;
    hipLaunchKernelGGL(k_col_orand2, dim3((unsigned)g, (unsigned)kc), dim3(PRA_BLOCK), 0, st, rows, n, w, out);
}

void pra_launch_dedup_claim2(hipStream_t st, const u64* cand, const u64* ctl, u64 capn, int cw, int kw, u64* table,
                             u64 cap, u64* slot_of, u64 epoch, u32* flags)
{
    if (!capn) return;
    const dim3 g(grid_for(capn)), b(PRA_BLOCK);
#define PRA_CLAIM(K, E)                                                                                                \
    hipLaunchKernelGGL((k_dedup_claim2<K, E>), g, b, 0, st, cand, ctl, cw, kw, table, cap, slot_of, epoch, flags)
    switch (kw) {
    case 1: PRA_CLAIM(1, true); break;
    case 2: PRA_CLAIM(2, true); break;
    case 3: PRA_CLAIM(3, true); break;
    case 4: PRA_CLAIM(4, true); break;
    default:
        if (kw <= 8)
            PRA_CLAIM(8, false);
        else if (kw <= 16)
            PRA_CLAIM(16, false);
        else
            PRA_CLAIM(0, false);
    }
#undef PRA_CLAIM
}

int pra_dedup_class(int kw)
{
    return kw >= 1 && kw <= 4 ? kw : kw <= 8 ? 5 : kw <= 16 ? 6 : 7;
}

#define PRA_DEDUP_DISPATCH(CLS, LAUNCH)                                                                                \
    switch (CLS) {                                                                                                     \
    case 1: LAUNCH(1, true); break;                                                                                    \
    case 2: LAUNCH(2, true); break;                                                                                    \
    case 3: LAUNCH(3, true); break;                                                                                    \
    case 4: LAUNCH(4, true); break;                                                                                    \
    case 5: LAUNCH(8, false); break;                                                                                   \
    case 6: LAUNCH(16, false); break;                                                                                  \
    default: LAUNCH(0, false);                                                                                         \
    }

void pra_launch_dense_claim(hipStream_t st, const DenseArgs& a, u64 capn, u32* flags)
{
    if (!capn) return;
    const dim3 g(grid_for(capn)), b(PRA_BLOCK);
    switch (a.kw) {
    case 1: hipLaunchKernelGGL(k_dense_claim<1>, g, b, 0, st, a, flags); break;
    case 2: hipLaunchKernelGGL(k_dense_claim<2>, g, b, 0, st, a, flags); break;
    case 3: hipLaunchKernelGGL(k_dense_claim<3>, g, b, 0, st, a, flags); break;
    default: hipLaunchKernelGGL(k_dense_claim<4>, g, b, 0, st, a, flags); break;
    }
}

void pra_launch_dense_many(hipStream_t st, const DenseArgs* jobs, int njobs, int kw, u32 claim_blocks,
                           u32 decide_blocks, u32* flags)
{
    if (njobs <= 0) return;
    if (claim_blocks) {
        const dim3 g(claim_blocks), b(PRA_BLOCK);
        switch (kw) {
        case 1: hipLaunchKernelGGL(k_dense_claim_many<1>, g, b, 0, st, jobs, njobs, flags); break;
        case 2: hipLaunchKernelGGL(k_dense_claim_many<2>, g, b, 0, st, jobs, njobs, flags); break;
        case 3: hipLaunchKernelGGL(k_dense_claim_many<3>, g, b, 0, st, jobs, njobs, flags); break;
        default: hipLaunchKernelGGL(k_dense_claim_many<4>, g, b, 0, st, jobs, njobs, flags); break;
        }
    }
    if (decide_blocks)
        hipLaunchKernelGGL(k_dense_decide_many, dim3(decide_blocks), dim3(PRA_DECIDE_BLOCK), 0, st, jobs, njobs);
}

void pra_launch_dense_decide(hipStream_t st, const DenseArgs& a, u32*)
{
    const dim3 g(std::min<u32>(a.nblocks, PRA_DECIDE_GRID)), b(PRA_DECIDE_BLOCK);
    hipLaunchKernelGGL(k_dense_decide, g, b, 0, st, a);
}

void pra_launch_dense_build(hipStream_t st, const u64* rows, u64 n, int w, int kw, const u64* dict, u64 dict_cap, u64 D,
                            int by_bucket, u32* bitmap, u64* miss)
{
    if (!n) return;
    const dim3 g(grid_for(n)), b(PRA_BLOCK);
    switch (kw) {
    case 1: hipLaunchKernelGGL(k_dense_build<1>, g, b, 0, st, rows, n, w, dict, dict_cap, D, by_bucket, bitmap, miss); break;
    case 2: hipLaunchKernelGGL(k_dense_build<2>, g, b, 0, st, rows, n, w, dict, dict_cap, D, by_bucket, bitmap, miss); break;
    case 3: hipLaunchKernelGGL(k_dense_build<3>, g, b, 0, st, rows, n, w, dict, dict_cap, D, by_bucket, bitmap, miss); break;
    default: hipLaunchKernelGGL(k_dense_build<4>, g, b, 0, st, rows, n, w, dict, dict_cap, D, by_bucket, bitmap, miss); break;
    }
}

void pra_launch_dict_bucket_rank(hipStream_t st, const u64* vals, u64 n, u64* tab, u64 cap, u32* rank_of, u32* lead_of,
                                 u64 nb, unsigned char* bucket)
{
    if (n)
        hipLaunchKernelGGL(k_dict_bucket_rank, dim3(grid_for(n)), dim3(PRA_BLOCK), 0, st, vals, n, tab, cap, rank_of,
                           lead_of, nb, bucket);
}

void pra_launch_rank_rows(hipStream_t st, const RankRowsArgs& a)
{
    if (a.n) hipLaunchKernelGGL(k_rank_rows, dim3(grid_for(a.n)), dim3(PRA_BLOCK), 0, st, a);
}

void pra_launch_rank_rows_many(hipStream_t st, const RankRowsArgs* jobs, int njobs, u32 blocks)
{
    if (blocks) hipLaunchKernelGGL(k_rank_rows_many, dim3(blocks), dim3(PRA_BLOCK), 0, st, jobs, njobs);
}

void pra_launch_rank(hipStream_t st, int step, const RankArgs& a, u64 cap, u64* status, u32* ctr, u32 epoch, u32* flags)
{
    switch (step) {
    case PRA_RANK_EMIT:
        hipLaunchKernelGGL(k_rank_emit, dim3((unsigned)((a.emit.n + PRA_EMIT_BLOCK - 1) / PRA_EMIT_BLOCK)),
                           dim3(PRA_EMIT_BLOCK), 0, st, a, status, ctr, epoch, flags);
        break;
    case PRA_RANK_CLAIM: hipLaunchKernelGGL(k_rank_claim, dim3(grid_for(cap)), dim3(PRA_BLOCK), 0, st, a); break;
    case PRA_RANK_SCAN:
        hipLaunchKernelGGL(k_rank_scan, dim3(a.chunks), dim3(PRA_SCAN_BLOCK), 0, st, a, status, ctr, epoch, flags);
        break;
    case PRA_RANK_FIRST: hipLaunchKernelGGL(k_rank_first, dim3(grid_for(cap)), dim3(PRA_BLOCK), 0, st, a); break;
    default:
        hipLaunchKernelGGL(k_rank_place, dim3(pra_tiles(cap)), dim3(PRA_PLACE_BLOCK), 0, st, a, status, ctr, epoch,
                           flags);
    }
}

void pra_launch_rank_loop(hipStream_t st, const LoopArgs& a)
{
    hipLaunchKernelGGL(k_rank_loop, dim3(1), dim3(PRA_LOOP_BLOCK), 0, st, a);
}

void pra_launch_rank_loop_many(hipStream_t st, const LoopArgs* jobs, int njobs)
{
    hipLaunchKernelGGL(k_rank_loop_many, dim3(njobs), dim3(PRA_LOOP_BLOCK), 0, st, jobs);
}

void pra_launch_rank_many(hipStream_t st, int step, const RankArgs* jobs, int njobs, u32 blocks, u64* status, u32* ctr,
                          u32 epoch, u32* flags)
{
    if (!blocks) return;
    switch (step) {
    case PRA_RANK_EMIT:
        hipLaunchKernelGGL(k_rank_emit_many, dim3(blocks), dim3(PRA_EMIT_BLOCK), 0, st, jobs, njobs, status, ctr, epoch,
                           flags);
        break;
    case PRA_RANK_CLAIM: hipLaunchKernelGGL(k_rank_claim_many, dim3(blocks), dim3(PRA_BLOCK), 0, st, jobs, njobs); break;
    case PRA_RANK_SCAN:
        hipLaunchKernelGGL(k_rank_scan_many, dim3(blocks), dim3(PRA_SCAN_BLOCK), 0, st, jobs, njobs, status, ctr, epoch,
                           flags);
        break;
    case PRA_RANK_FIRST: hipLaunchKernelGGL(k_rank_first_many, dim3(blocks), dim3(PRA_BLOCK), 0, st, jobs, njobs); break;
    default:
        hipLaunchKernelGGL(k_rank_place_many, dim3(blocks), dim3(PRA_PLACE_BLOCK), 0, st, jobs, njobs, status, ctr,
                           epoch, flags);
    }
}

void pra_launch_bm_count(hipStream_t st, const u64* bm, u64 words, u64 nblk, u32* cnt)
{
    hipLaunchKernelGGL(k_bm_count, dim3(grid_for(nblk)), dim3(PRA_BLOCK), 0, st, bm, words, nblk, cnt);
}

void pra_launch_bm_place(hipStream_t st, const u64* rows, u64 n, int w, int kw, const u64* dict, u64 dict_cap, u64 D,
                         int by_bucket, const u64* bm, u64 words, const u32* prefix, u64* out)
{
    if (!n) return;
    const dim3 g(grid_for(n)), b(PRA_BLOCK);
    auto k = kw == 1 ? k_bm_place<1> : kw == 2 ? k_bm_place<2> : kw == 3 ? k_bm_place<3> : k_bm_place<4>;
    hipLaunchKernelGGL(k, g, b, 0, st, rows, n, w, dict, dict_cap, D, by_bucket, bm, words, prefix, out);
}

void pra_launch_dense_table_clear(hipStream_t st, u64* table, u64 cap) { pra_launch_fill_u64(st, table, cap, 0); }

void pra_launch_dedup_claim_many(hipStream_t st, const ClaimBatch& b, int cls, u32* flags)
{
    if (b.njobs <= 0 || !b.block_base[b.njobs]) return;
    const dim3 g(b.block_base[b.njobs]), bl(PRA_BLOCK);
#define PRA_CLAIM_MANY(K, E) hipLaunchKernelGGL((k_dedup_claim_many<K, E>), g, bl, 0, st, b, flags)
    PRA_DEDUP_DISPATCH(cls, PRA_CLAIM_MANY)
#undef PRA_CLAIM_MANY
}

void pra_launch_dedup_decide_many(hipStream_t st, const DecideBatch& b, int cls, u32* flags)
{
    if (b.njobs <= 0 || !b.block_base[b.njobs]) return;
    const dim3 g(b.block_base[b.njobs]), bl(PRA_DECIDE_BLOCK);
#define PRA_DECIDE_MANY(K, E) hipLaunchKernelGGL((k_dedup_decide_many<K, E>), g, bl, 0, st, b, flags)
    PRA_DEDUP_DISPATCH(cls, PRA_DECIDE_MANY)
#undef PRA_DECIDE_MANY
}
#undef PRA_DEDUP_DISPATCH

static_assert(sizeof(ClaimBatch) + sizeof(void*) <= 4096, "claim batch exceeds the kernel arguments");
static_assert(sizeof(DecideBatch) + sizeof(void*) <= 4096, "decision batch exceeds the kernel arguments");

void pra_launch_dedup_decide_hist(hipStream_t st, const u64* cand, const u64* ctl, int cw, int kw, const u64* table,
                                  const u64* slot_of, u64 epoch, u32* keep, const u32* dest, u32 nb, u32* hist,
                                  u32 nblocks, u32* flags, u32* offs1)
{
    // tiles past the candidate count (known only on the device) cost a block
    // each, and a block fills a compute unit: a bounded grid strides over them
    const dim3 g(std::min<u32>(nblocks, PRA_DECIDE_GRID)), b(PRA_DECIDE_BLOCK);
#define PRA_DECIDE(K, E)                                                                                               \
    hipLaunchKernelGGL((k_dedup_decide_hist<K, E>), g, b, 0, st, cand, ctl, cw, kw, table, slot_of, epoch, keep, dest, \
                       nb, hist, nblocks, flags, offs1)
    switch (kw) {
    case 1: PRA_DECIDE(1, true); break;
    case 2: PRA_DECIDE(2, true); break;
    case 3: PRA_DECIDE(3, true); break;
    case 4: PRA_DECIDE(4, true); break;
    default:
        if (kw <= 8)
            PRA_DECIDE(8, false);
        else if (kw <= 16)
            PRA_DECIDE(16, false);
        else
            PRA_DECIDE(0, false);
    }
#undef PRA_DECIDE
}

void pra_launch_bin_sort_many(hipStream_t st, const BinSortJob* jobs, int njobs, u32* flags, u64 maxbin)
{
    if (njobs <= 0) return;
#define PRA_BIN_SORT(B) hipLaunchKernelGGL(k_bin_sort_many<B>, dim3(PRA_RADIX * njobs), dim3(B), 0, st, jobs, flags)
    if (maxbin <= 256 * PRA_BIN_ITEMS)
        PRA_BIN_SORT(256);
    else if (maxbin <= 512 * PRA_BIN_ITEMS)
        PRA_BIN_SORT(512);
    else
        PRA_BIN_SORT(PRA_BIN_BLOCK);
#undef PRA_BIN_SORT
}

void pra_launch_scan_small_many(hipStream_t st, const ScanJob* jobs, int njobs)
{
    if (njobs > 0) hipLaunchKernelGGL(k_scan_small_many, dim3(njobs), dim3(PRA_BLOCK), 0, st, jobs);
}

void pra_launch_copy_many(hipStream_t st, const CopyJob* jobs, int njobs, u32 nblocks)
{
    if (njobs > 0 && nblocks) hipLaunchKernelGGL(k_copy_many, dim3(nblocks), dim3(PRA_BLOCK), 0, st, jobs, njobs);
}

void pra_launch_newt_fold_many(hipStream_t st, const NewtFoldArgs* jobs, int njobs)
{
    if (njobs > 0) hipLaunchKernelGGL(k_newt_fold_many, dim3(3 * njobs), dim3(PRA_BLOCK), 0, st, jobs);
}

void pra_launch_newt_fold(hipStream_t st, const NewtFoldArgs& a)
{
    static_assert(PRA_RADIX == PRA_BLOCK && PRA_PART_WORDS <= PRA_BLOCK, "one thread per bin / word");
    hipLaunchKernelGGL(k_newt_fold, dim3(3), dim3(PRA_BLOCK), 0, st, a);
}

void pra_launch_newt_rep_init(hipStream_t st, u64* rep_words, int sets)
{
    for (int k = 0; k < sets; k++)
        hipLaunchKernelGGL(k_newt_rep_init, dim3((PRA_NREP * PRA_PART_WORDS + PRA_BLOCK - 1) / PRA_BLOCK),
                           dim3(PRA_BLOCK), 0, st, rep_words + (size_t)k * PRA_NREP * PRA_PART_WORDS);
}

void pra_launch_merge(hipStream_t st, const MergeBatch& b)
{
    if (b.njobs <= 0) return;
    hipLaunchKernelGGL(k_merge_rank, dim3(b.rank_base[b.njobs]), dim3(PRA_BLOCK), 0, st, b);
    hipLaunchKernelGGL(k_merge_scatter, dim3(b.scatter_base[b.njobs]), dim3(PRA_BLOCK), 0, st, b);
}

void pra_launch_rows_checksum(hipStream_t st, const u64* rows, u64 n, int w, u64* out)
{
    u64 g = (n + PRA_BLOCK - 1) / PRA_BLOCK;
    if (g > 1024) g = 1024;
    if (g == 0) g = 1;
    hipLaunchKernelGGL(k_rows_checksum, dim3((unsigned)g), dim3(PRA_BLOCK), 0, st, rows, n, w, out);
}

void pra_launch_group_maxlen(hipStream_t st, const u64* flags, const u64* gpos, const u64* gstart, u64 n, u64* maxlen)
{
    if (!n) return;
    hipLaunchKernelGGL(k_group_maxlen, dim3(grid_for(n)), dim3(PRA_BLOCK), 0, st, flags, gpos, gstart, n, maxlen);
}
