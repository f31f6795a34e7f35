// Host engine of the MI355X semi-naive RA backend: device-resident relation
// versions, the per-iteration pipeline (join / copy emit -> arrival-ordered
// candidates -> dedup + intern -> stable bucket partition -> LSD sort) and the
// LIE-style SCC scheduler, exported through the C ABI of include/pra.h.
//
// Layout in HBM: every version (full, delta, newt) of a relation is one array
// of rows of w = arity+1 u64 words.  delta and newt are kept sorted by
// (bucket, lexicographic row); full is an append log that is re-sorted only
// when an ordered walk of it is needed (copy from FULL, join probe side).
// Membership of full u delta is an open-addressing table keyed by the dedup
// columns; join probe sides get a (key -> first row, row count) index.
#include "../../include/pra.h"
#include "pra_blockcache.hpp"
#include "pra_tune.hpp"
#include "pra_kernels.hpp"
#include "pra_partition.hpp"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <thread>
#include <tuple>
#include <utility>
#include <vector>

namespace {

static bool yield_tables(pra_ctx* c);

enum { RA_COPY = 0, RA_COPY_FILTER = 1, RA_ACOPY = 3, RA_JOIN = 4 };

struct PraError : std::runtime_error {
    int code;
    PraError(int c, const std::string& m) : std::runtime_error(m), code(c) {}
    // device memory, or the context's share of it, is used up
    bool refused() const { return code == PRA_E_BUDGET || code == PRA_E_NOMEM; }
};

#define HIPCHK(x)                                                                                  \
    do {                                                                                           \
        hipError_t e_ = (x);                                                                       \
        if (e_ != hipSuccess)                                                                      \
            throw PraError(PRA_E_HIP, std::string(#x) + ": " + hipGetErrorString(e_));            \
    } while (0)

static void check_launch(const char* what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) throw PraError(PRA_E_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

// Large blocks (>= 64 MiB) go through the process-wide block cache of
// pra_blockcache.hpp (its ownership rule: a block released while its stream
// runs is reused only on that stream until a host synchronization of the
// stream declares it idle).  Out of memory: idle blocks are freed, oldest
// first, until the request fits; then the requesting stream is synchronized,
// its own blocks declared idle and the stream-ordered pool trimmed before one
// more attempt.
namespace {
constexpr size_t kBigBlock = 64ULL << 20;
pra::BlockCache g_big(kBigBlock);

void* hip_block_alloc(size_t bytes, void*)
{
    void* p = nullptr;
    if (hipMalloc(&p, bytes) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return p;
}
void hip_block_free(void* p, void*) { (void)hipFree(p); }
const pra::BlockAllocator kHipBlocks{hip_block_alloc, hip_block_free, nullptr};

// Device bytes held by each context, keyed by its stream (every buffer of a
// context is ordered on the context's stream): live bytes, their peak, the
// context's cap (0 = none), the stream's device, and the context.
struct MemAcct {
    long long live = 0, peak = 0;
    u64 budget = 0;
    int device = 0;
    pra_ctx* owner = nullptr;
};
std::mutex g_acct_mu;
std::map<hipStream_t, MemAcct> g_acct;

// the context of a stream gives back what it can do without
bool yield_for(hipStream_t s)
{
    pra_ctx* c;
    {
        std::lock_guard<std::mutex> lk(g_acct_mu);
        auto it = g_acct.find(s);
        c = it == g_acct.end() ? nullptr : it->second.owner;
    }
    return c && yield_tables(c);
}

// the device whose memory a stream's buffers are in; the calling thread's
// current device may be another one
int stream_device(hipStream_t s)
{
    std::lock_guard<std::mutex> lk(g_acct_mu);
    auto it = g_acct.find(s);
    return it == g_acct.end() ? 0 : it->second.device;
}

// charge `bytes` more to the context of stream s (fails past its budget while
// `check`), or credit them back when negative
void acct_charge(hipStream_t s, long long bytes, bool check)
{
    std::lock_guard<std::mutex> lk(g_acct_mu);
    auto it = g_acct.find(s);
    if (it == g_acct.end()) return;
    MemAcct& a = it->second;
    if (check && bytes > 0 && a.budget && (u64)(a.live + bytes) > a.budget)
        throw PraError(PRA_E_BUDGET, "device memory budget exceeded: " + std::to_string(a.live) + " bytes held + " +
                                         std::to_string(bytes) + " requested > budget " + std::to_string(a.budget));
    a.live += bytes;
    if (a.live > a.peak) a.peak = a.live;
}

// refuses when the context of stream s has not `bytes` left of its budget
void acct_need(hipStream_t s, long long bytes)
{
    std::lock_guard<std::mutex> lk(g_acct_mu);
    auto it = g_acct.find(s);
    if (it != g_acct.end() && it->second.budget && (u64)(it->second.live + bytes) > it->second.budget)
        throw PraError(PRA_E_BUDGET, "device memory budget exceeded: less than " + std::to_string(bytes) + " bytes left");
}

// the stream-ordered pool keeps freed memory for reuse; give it back
void trim_pool(int dev)
{
    hipMemPool_t pool = nullptr;
    if (hipDeviceGetDefaultMemPool(&pool, dev) == hipSuccess && pool) (void)hipMemPoolTrimTo(pool, 0);
}

void small_idle_flush(int dev, hipStream_t st);

void* big_get(size_t bytes, hipStream_t st, size_t* got)
{
    const int dev = stream_device(st);
    void* p = g_big.get(dev, st, bytes, got, kHipBlocks);
    if (!p) {
        small_idle_flush(dev, st);
        HIPCHK(hipStreamSynchronize(st));
        g_big.idle(st);
        trim_pool(dev);
        p = g_big.get(dev, st, bytes, got, kHipBlocks);
    }
    if (!p)
        throw PraError(PRA_E_NOMEM, "hipMalloc: out of memory (" + std::to_string(g_big.size_class(bytes)) + " bytes)");
    return p;
}

void big_put(void* p, size_t size, hipStream_t st)
{
    g_big.put(stream_device(st), st, p, size);
}

// every piece of work enqueued on st so far has completed
void stream_idle(hipStream_t st) { g_big.idle(st); }

// Small blocks (below 64 MiB) released by a buffer are kept for the stream
// they were released on and handed to later requests of the same
// quarter-octave class on that stream: work enqueued there after the release
// runs after every earlier use of the block, so stream order alone makes the
// reuse safe, and no hipFreeAsync / hipMallocAsync pair is paid per buffer
// (about 0.1 ms of host time each).  At most kSmallKeep bytes are kept per
// stream; the rest, and a stream's blocks when the device runs out of memory,
// are freed on their stream.  When a context goes away its stream has been
// waited for, so its blocks are idle: up to kSmallIdle bytes a device stay for
// whichever context asks next (a short-lived context used to spend more on
// freeing its sixty blocks than on solving: 0.65 ms of 1.3 on 40 vertices),
// and go back when the device runs out of memory.
constexpr size_t kSmallKeep = 2ULL << 30;
constexpr size_t kSmallIdle = 512ULL << 20;
struct SmallFree {
    std::map<size_t, std::vector<void*>> by_class;
    size_t bytes = 0;

    void* take(size_t cls)
    {
        auto c = by_class.find(cls);
        if (c == by_class.end() || c->second.empty()) return nullptr;
        void* p = c->second.back();
        c->second.pop_back();
        bytes -= cls;
        return p;
    }
    bool put(size_t cls, void* p, size_t limit)
    {
        if (bytes + cls > limit) return false;
        by_class[cls].push_back(p);
        bytes += cls;
        return true;
    }
};
std::mutex g_small_mu;
std::map<hipStream_t, SmallFree> g_small;
std::map<int, SmallFree> g_small_idle;   // per device
std::atomic<size_t> g_small_idle_limit{kSmallIdle};   // no more than the stream-ordered pool may keep

size_t small_class(size_t bytes)
{
    size_t oct = 256;
    while (oct * 2 <= bytes) oct <<= 1;
    for (size_t q = 4; q <= 8; q++)
        if (oct / 4 * q >= bytes) return oct / 4 * q;
    return oct * 2;
}

void* small_take(hipStream_t st, size_t cls)
{
    const int dev = stream_device(st);
    std::lock_guard<std::mutex> lk(g_small_mu);
    auto it = g_small.find(st);
    void* p = it == g_small.end() ? nullptr : it->second.take(cls);
    if (!p) {
        auto d = g_small_idle.find(dev);
        if (d != g_small_idle.end()) p = d->second.take(cls);
    }
    return p;
}

void small_put(hipStream_t st, void* p, size_t cls)
{
    {
        std::lock_guard<std::mutex> lk(g_small_mu);
        if (g_small[st].put(cls, p, kSmallKeep)) return;
    }
    (void)hipFreeAsync(p, st);
}

// free, on a stream, the idle small blocks of its device
void small_idle_flush(int dev, hipStream_t st)
{
    SmallFree f;
    {
        std::lock_guard<std::mutex> lk(g_small_mu);
        std::swap(f, g_small_idle[dev]);
    }
    for (auto& c : f.by_class)
        for (void* p : c.second) (void)hipFreeAsync(p, st);
}

// free the small blocks kept for a stream and the device's idle ones, on it
void small_flush(hipStream_t st)
{
    small_idle_flush(stream_device(st), st);
    SmallFree f;
    {
        std::lock_guard<std::mutex> lk(g_small_mu);
        auto it = g_small.find(st);
        if (it == g_small.end()) return;
        f = std::move(it->second);
        g_small.erase(it);
    }
    for (auto& c : f.by_class)
        for (void* p : c.second) (void)hipFreeAsync(p, st);
}

// The small blocks of a stream that has been waited for and goes away become
// idle.  Past the limit the largest idle blocks are freed first: a block costs
// the same to free and to make again whatever its size.
void small_retire(hipStream_t st)
{
    const int dev = stream_device(st);
    const size_t limit = g_small_idle_limit;
    std::vector<void*> drop;
    {
        std::lock_guard<std::mutex> lk(g_small_mu);
        auto it = g_small.find(st);
        if (it == g_small.end()) return;
        SmallFree& idle = g_small_idle[dev];
        for (auto& c : it->second.by_class)
            for (void* p : c.second) {
                while (idle.bytes + c.first > limit && !idle.by_class.empty() && idle.by_class.rbegin()->first > c.first) {
                    if (void* q = idle.take(idle.by_class.rbegin()->first))
                        drop.push_back(q);
                    else
                        idle.by_class.erase(std::prev(idle.by_class.end()));
                }
                if (!idle.put(c.first, p, limit)) drop.push_back(p);
            }
        g_small.erase(it);
    }
    for (void* p : drop) (void)hipFreeAsync(p, st);
}

// What a context needs of the driver beside device memory -- its stream and
// pinned host blocks -- kept idle for the next context, a few of each: making
// and freeing them costs from 0.05 to 0.4 ms apiece.
constexpr size_t kIdleStreams = 8, kIdlePinned = 32;
constexpr size_t kPinnedKeep = 256 << 10;   // larger pinned blocks are freed
struct IdleHost {
    std::map<int, std::vector<hipStream_t>> streams;         // per device
    std::map<std::pair<size_t, unsigned>, std::vector<void*>> pinned;   // by bytes and allocation flags
    size_t npinned = 0;
};
std::mutex g_idle_mu;
IdleHost g_idle;

hipStream_t stream_get(int dev)
{
    {
        std::lock_guard<std::mutex> lk(g_idle_mu);
        auto& v = g_idle.streams[dev];
        if (!v.empty()) {
            hipStream_t s = v.back();
            v.pop_back();
            return s;
        }
    }
    hipStream_t s = nullptr;
    HIPCHK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    return s;
}

// ok: everything enqueued on the stream has completed without an error
void stream_put(int dev, hipStream_t s, bool ok)
{
    if (ok) {
        std::lock_guard<std::mutex> lk(g_idle_mu);
        auto& v = g_idle.streams[dev];
        if (v.size() < kIdleStreams) {
            v.push_back(s);
            return;
        }
    }
    (void)hipStreamDestroy(s);
}

void* pinned_get(size_t bytes, unsigned flags)
{
    {
        std::lock_guard<std::mutex> lk(g_idle_mu);
        auto it = g_idle.pinned.find({bytes, flags});
        if (it != g_idle.pinned.end() && !it->second.empty()) {
            void* p = it->second.back();
            it->second.pop_back();
            g_idle.npinned--;
            return p;
        }
    }
    void* p = nullptr;
    HIPCHK(hipHostMalloc(&p, bytes, flags));
    return p;
}

// ok: no work that was enqueued can still touch the block
void pinned_put(void* p, size_t bytes, unsigned flags, bool ok)
{
    if (!p) return;
    if (ok && bytes <= kPinnedKeep) {
        std::lock_guard<std::mutex> lk(g_idle_mu);
        if (g_idle.npinned < kIdlePinned) {
            g_idle.pinned[{bytes, flags}].push_back(p);
            g_idle.npinned++;
            return;
        }
    }
    (void)hipHostFree(p);
}

// Autotuned knobs, per device and band of log2(work): the dense claim
// table's size (2, 4 or 8 slots per candidate of capacity, so a load of at
// most 1/2, 1/4 or 1/8), the newt scatter's block width (256 or 1,024
// threads), and whether a dense output takes the claim table (0) or ranked
// membership (1).  None changes a result: which arrival wins a key, and where
// every row and id goes, are the same under every variant.  Variants are
// timed with events on single-output iterations, per candidate.
enum { TUNE_DENSE_LOAD, TUNE_SCATTER_WIDE, TUNE_RANKED, TUNE_KNOBS };
const char* const kTuneNames[TUNE_KNOBS] = {"dense_table_slots_log2_minus_1", "newt_scatter_wide", "ranked_membership"};
const int kTuneVariants[TUNE_KNOBS] = {3, 2, 2};
constexpr u64 kTuneMinCandidates = 1ULL << 16;
// capacity from which a dense output takes ranked membership beside outputs of
// the general table
constexpr u64 kMixedRankedCandidates = 1ULL << 18;
// longest run of inner rows that an emission in digits walks in one thread
constexpr u64 kEmitRun = 32;
pra::Tuner g_tune(3);

// Tuning cache: with PRA_AUTOTUNE_FILE set, the settled choices are read from
// that file when the first context is created (those cells run without
// trials) and the file is rewritten whenever a cell settles.
std::once_flag g_tune_once;
std::mutex g_tune_file_mu;
std::string g_tune_file;

void tune_init()
{
    std::call_once(g_tune_once, [] {
        const char* f = getenv("PRA_AUTOTUNE_FILE");
        if (!f || !*f) return;
        g_tune_file = f;
        FILE* in = fopen(f, "r");
        if (!in) return;
        std::string text;
        char buf[4096];
        size_t got;
        while ((got = fread(buf, 1, sizeof(buf), in)) > 0) text.append(buf, got);
        fclose(in);
        g_tune.load(text, kTuneNames, TUNE_KNOBS);
    });
}

void tune_save()
{
    if (g_tune_file.empty()) return;
    const std::string r = g_tune.report(kTuneNames, TUNE_KNOBS);
    std::lock_guard<std::mutex> lk(g_tune_file_mu);
    FILE* out = fopen(g_tune_file.c_str(), "w");
    if (!out) return;
    fwrite(r.data(), 1, r.size(), out);
    fclose(out);
}

int band_of(u64 n)
{
    int b = 0;
    while (n > 1) {
        n >>= 1;
        b++;
    }
    return b;
}
} // namespace

// Device buffer owned by one context and ordered on its stream: small blocks
// come from the stream-ordered pool, large ones from the block cache above;
// growth and release never synchronize the device, so contexts driven from
// different host threads overlap.
struct DBuf {
    void* p = nullptr;
    size_t cap = 0;
    hipStream_t st = nullptr;
    bool big = false;
    DBuf() = default;
    DBuf(const DBuf&) = delete;
    DBuf& operator=(const DBuf&) = delete;
    DBuf(DBuf&& o) noexcept : p(o.p), cap(o.cap), st(o.st), big(o.big) { o.p = nullptr; o.cap = 0; }
    DBuf& operator=(DBuf&& o) noexcept
    {
        if (this != &o) {
            release();
            p = o.p;
            cap = o.cap;
            st = o.st;
            big = o.big;
            o.p = nullptr;
            o.cap = 0;
        }
        return *this;
    }
    ~DBuf() { release(); }
    void release()
    {
        if (p) {
            if (big)
                big_put(p, cap, st);
            else
                small_put(st, p, cap);
            acct_charge(st, -(long long)cap, false);
        }
        p = nullptr;
        cap = 0;
        big = false;
    }
    // grow to at least `bytes`, preserving the first `used` bytes; a refusal
    // is final only without the memory that the context can do without
    void reserve(size_t bytes, hipStream_t s, size_t used = 0)
    {
        if (bytes <= cap) return;
        try {
            grow(bytes, s, used);
        } catch (const PraError& e) {
            if (!e.refused() || !yield_for(s)) throw;
            grow(bytes, s, used);
        }
    }
    void grow(size_t bytes, hipStream_t s, size_t used)
    {
        // grow by doubling (fewer growth copies than growing by half, which
        // measured slower); the quarter-octave block classes keep the
        // rounding on top of that within 25 %
        size_t nc = std::max(bytes, 2 * cap);
        void* np = nullptr;
        bool nbig = nc >= kBigBlock;
        nc = nbig ? g_big.size_class(nc) : small_class(nc);
        acct_charge(s, (long long)nc, true);
        try {
            if (nbig) {
                const size_t want = nc;
                np = big_get(want, s, &nc);
                acct_charge(s, (long long)nc - (long long)want, false);   // a cached block of the next class
            } else if (!(np = small_take(s, nc)) && hipMallocAsync(&np, nc, s) != hipSuccess) {
                const int dev = stream_device(s);
                (void)hipGetLastError();
                small_flush(s);
                g_big.flush(dev, kHipBlocks, nc);
                if (hipMallocAsync(&np, nc, s) != hipSuccess) {
                    (void)hipGetLastError();
                    HIPCHK(hipStreamSynchronize(s));
                    g_big.idle(s);
                    g_big.flush(dev, kHipBlocks);
                    trim_pool(dev);
                    const hipError_t e = hipMallocAsync(&np, nc, s);
                    if (e == hipErrorOutOfMemory) {
                        (void)hipGetLastError();
                        throw PraError(PRA_E_NOMEM, "hipMallocAsync: out of memory (" + std::to_string(nc) + " bytes)");
                    }
                    HIPCHK(e);
                }
            }
        } catch (...) {
            acct_charge(s, -(long long)nc, false);
            throw;
        }
        if (p && used) HIPCHK(hipMemcpyAsync(np, p, used, hipMemcpyDeviceToDevice, s));
        if (p) {
            if (big)
                big_put(p, cap, s);
            else
                small_put(s, p, cap);
            acct_charge(st ? st : s, -(long long)cap, false);
        }
        p = np;
        cap = nc;
        st = s;
        big = nbig;
    }
    template <typename T> T* as() const { return static_cast<T*>(p); }
    void swap(DBuf& o)
    {
        std::swap(p, o.p);
        std::swap(cap, o.cap);
        std::swap(st, o.st);
        std::swap(big, o.big);
    }
};

struct Rows {
    DBuf buf;
    u64 n = 0;
    bool sorted = true;
    u64* d() { return buf.as<u64>(); }
};

static u64 pow2_at_least(u64 x)
{
    u64 c = 1;
    while (c < x) c <<= 1;
    return c;
}

} // namespace

struct pra_scc;

struct pra_rel {
    pra_ctx* ctx = nullptr;
    int group = 0;
    int arity = 0, jcc = 0, canonical = 1, w = 0;
    u32 tag = 0;
    Rows ver[3];  // PRA_DELTA, PRA_FULL, PRA_NEWT
    // membership table of full u delta keyed on mt_kw leading columns
    DBuf mt;
    u64 mt_cap = 0, mt_entries = 0;
    int mt_kw = -1;
    bool mt_valid = false;
    // dense membership (interned outputs with dictionary-ranked keys): bitmap
    // over the key's rank index, built for dictionary generation bm_gen and
    // kept current by the iterations that take the dense path; the
    // per-iteration claim table (empty between iterations)
    DBuf bm, dtab;
    // ranked membership: the new keys' bitmap (zero between iterations), its
    // superblocks' flags and prefixes, its lines' prefixes
    DBuf fresh, dirty, sbpre, linep;
    DBuf places;         // whole iterations in one block: the new keys' places
    u64 fresh_sbs = 0;   // superblocks of the zeroed bitmap (0: none)
    u64 sbs_use = 0;     // of them, those of the current rank space
    // rank indexes of the delta rows (valid for dictionary generation dx_gen)
    // and of the new rows
    DBuf dx, nx;
    u64 dx_gen = ~0ULL;
    // per version: the dictionary words of the rows' columns and the first row
    // of every leading digit (valid for dictionary generation rk_gen)
    DBuf rk_words[2], rk_first[2];
    u64 rk_gen[2] = {~0ULL, ~0ULL};
    bool rk_no[2] = {false, false};   // rows without ranks, or no room
    u64 bm_gen = ~0ULL, dtab_cap = 0, dtab_use = 0;   // slots allocated, slots in use this iteration
    int dtab_eb = -1;      // epoch bits of the claim table's slots (0: winners empty their slots)
    u32 dtab_epoch = 0;    // this iteration's epoch (slots of any other count as empty)
    int bm_kw = 0;
    bool bm_valid = false;
    // join index (key -> first row, count) per version
    DBuf idx[2];
    u64 idx_cap[2] = {0, 0};
    u64 idx_maxlen[2] = {0, 0};   // longest run of rows sharing a join key
    u64 jhint = 0;                // candidates of the previous iteration producing this relation
    bool idx_valid[2] = {false, false};
    // packed sort keys of newt rows, the offsets of their top-byte bins, and
    // the bins of (key, newt position) pairs the scatter fills
    DBuf nkeys, kgofs, bin_keys, bin_idx, bin_cur;
    u32 bin_cap = 0;
    // bucket bounds per version
    DBuf bnd[2];
    bool bnd_valid[2] = {false, false};
    DBuf next_bnd;   // the new rows' bounds, until they become the delta
    DBuf merged;     // the other buffer of a full version kept sorted by merges
    // set while an SCC runs: the relation is produced by one of its rules
    // (changes every iteration), and its full version is read by one of them
    // (so it is kept sorted by merging each delta into it)
    bool scc_changing = false, merge_full = false;
    // set while an SCC runs: a rule of it reads the relation's full version
    bool full_read = false;
    // set while an SCC runs whose iterations one block can run (loop_rule)
    bool loops = false;
    // changes of the delta and full versions so far
    u64 gen[2] = {0, 0};
    // a view: the rows of relation view_of that a join keyed on this
    // relation's jcc columns can match (built from view_of's versions of
    // generation view_gen)
    pra_rel* view_of = nullptr;
    u64 view_gen[2] = {~0ULL, ~0ULL};
    void touched(int v)
    {
        if (v == PRA_DELTA || v == PRA_FULL) {
            idx_valid[v] = false;
            bnd_valid[v] = false;
            rk_gen[v] = ~0ULL;
            rk_no[v] = false;
            if (v == PRA_DELTA) dx_gen = ~0ULL;
            gen[v]++;
        }
    }
};

namespace {

struct RADesc {
    int type = 0;
    pra_rel *out = nullptr, *in0 = nullptr, *in1 = nullptr;
    int v0 = 0, v1 = 0, op = PRA_F_TRUE;
    std::vector<int> map;
    // per-iteration state
    DBuf off, istart, posadj;
    u64 n_outer = 0;
    bool active = false;   // outer (and inner) non-empty this iteration
    bool sorted_probe = false;   // inner changes inside the SCC: binary search, no hash index
    pra_rel* outer = nullptr;
    int outer_v = 0;
    pra_rel* inner = nullptr;
    int inner_v = 0;
    int left = 1;
};

struct KStat {
    const char* name;
    uint64_t launches = 0;
    double ms = 0, bytes = 0;
};

enum {
    K_JOIN_COUNT, K_JOIN_EXPAND, K_COPY_EXPAND, K_DEDUP_CLAIM, K_DEDUP_DECIDE, K_DEDUP_VERIFY, K_DEDUP_SCATTER,
    K_RADIX_HIST, K_RADIX_SCATTER, K_TABLE_BUILD, K_INDEX_BUILD, K_SCAN, K_GATHER, K_MERGE, K_BIN_SORT, K_SMALL_SORT,
    K_BLOCK_SORT, K_RANK_EMIT, K_RANK_SCAN, K_RANK_FIRST, K_RANK_PLACE, K_RANK_LOOP, K_COUNT
};
static const char* kNames[K_COUNT] = {"join_count", "join_expand", "copy_expand", "dedup_claim", "dedup_decide",
                                      "dedup_verify_hist", "dedup_scatter", "radix_hist", "radix_scatter",
                                      "table_build", "index_build", "scan", "gather_rows", "merge_full",
                                      "bin_sort", "small_sort", "block_sort", "rank_emit", "rank_scan", "rank_first",
                                      "rank_place", "rank_loop"};

} // namespace

// One program instance (group) of a context.  A context holds one or more
// independent programs whose SCCs run in lock step (pra_ctx_set_group); each
// has its own intern counters (the reference keeps them per LIE,
// src/lie/lie.h:36), value dictionary, join-pair count and iteration count.
struct Group {
    // per intern tag: nb counters in two copies, of which `now` is current (a
    // ranked iteration reads one and writes the other)
    struct Seq {
        DBuf buf;
        int now = 0;
    };
    std::map<u32, std::unique_ptr<Seq>> seq;
    // order-preserving value dictionary for packed sort keys
    // value -> rank table; the values by rank; with several buckets, the values
    // by bucket-major rank, its maps to and from ranks, and its bucket
    DBuf dict, vals, lead_vals, rank_of, lead_of, lead_bucket;
    u64 dict_cap = 0, dict_n = 0;
    int dict_state = 0, dict_rebuilds = 0;   // state: 0 stale, 1 valid, 2 disabled
    u64 dict_gen = 0;                        // dictionary builds begun so far
    DBuf joined;                             // join pairs so far (one device word)
    u64 iterations = 0;
    // lock-step execution: the instance's SCC in progress and the iterations
    // of its current batch
    pra_scc* running = nullptr;
    u32 batch_it = 0;
};

struct pra_scc {
    pra_ctx* ctx = nullptr;
    int group = 0;
    int fixpoint = 1, id = 0;
    std::vector<pra_rel*> rels;
    std::vector<int> status;
    std::vector<RADesc> ras;
    bool done = false, running = false;
    std::vector<u64> hist;
    // delta rows at which an iteration last had too many candidates for one
    // block (~0: none had)
    u64 loop_stop = ~0ULL;
};

// Job-table staging slots.  A slot's pinned buffer is rewritten only after the
// host has waited for a kernel enqueued behind the slot's previous copy: every
// table but the early appends' is staged before an iteration's summary
// publication, or after its wait and before the next one's; the early appends
// are staged between a publication and its wait, so they alternate between
// two slots, and the wait of the iteration in between covers each copy.
enum { JOB_EXPAND, JOB_SCATTER, JOB_DENSE, JOB_SCAN, JOB_FOLD, JOB_SORT, JOB_EARLY_APPEND, JOB_EARLY_APPEND2,
       JOB_APPEND, JOB_PLAN, JOB_RANK, JOB_SETUP, JOB_LOOP, JOB_LOOP_FULL, JOB_LOOP_DELTA, PRA_JOB_SLOTS };

struct pra_ctx {
    int device = 0, nb = 1;
    hipStream_t st = nullptr;
    u64 budget = 0;
    u32 batch_size = 10;  // LIE::batch_size default (src/lie/lie.h:17)
    long long threshold = 20000000;
    std::vector<pra_rel*> rels;
    std::vector<pra_scc*> sccs;
    std::vector<std::pair<pra_scc*, pra_scc*>> deps;
    std::vector<std::unique_ptr<Group>> groups;   // program instances; relations and SCCs name theirs
    int cur_group = 0;                            // instance of the next pra_rel_create / pra_scc_create
    // scratch
    DBuf hist, offs, sort_tmp, flags_buf, stage, stage2, orand, tmp64a, tmp64b, tmp64c;
    DBuf cand, dest, slot_of, keep;
    DBuf first;              // ranked membership: earliest arrival per new key, all ones between iterations
    size_t first_words = 0;  // u32 words of it known to hold that
    DBuf ghist, gofs, lb_status, lb_ctr;
    DBuf part_scratch;   // pra_partition_rows
    // order-preserving value dictionary for packed sort keys
    DBuf ktmp, idxa, idxb, posadj_dev, rep_words, rctl, ttab, kp, jobtab[PRA_JOB_SLOTS];
    int rep_sets = 0;              // summary replica sets in rep_words (one per output of a batched partition)
    // pinned staging of batched kernels' job tables, one slot per table of an
    // iteration (expansions, partitions, dense claims, histogram scans, folds,
    // bin sorts, early appends, appends)
    char* job_stage[PRA_JOB_SLOTS] = {};
    size_t job_stage_cap[PRA_JOB_SLOTS] = {};
    int early_parity = 0;          // early appends' slot of the last iteration
    bool dense_on = true;        // dense membership for outputs that allow it
    bool tune_on = true;         // autotuned knobs (PRA_AUTOTUNE=0: the fixed defaults)
    bool loop_on = true;         // whole iterations in one block for small outputs (PRA_RANK_LOOP=0: never)
    // how often memory was refused since the last SCC began (yield_tables): from
    // once on no one-block iterations and second full buffers, from twice on no
    // ranked membership
    int lean = 0;
    int no_yield = 0;            // they are in use by launches under way (NoYield)
    bool merges_open = false;    // second full buffers are named by merges not yet launched
    bool seg_sort_on = true;     // segmented sort of newts too large for the bins (PRA_SEG_SORT=0: byte passes)
    u64 bin_cap_test = 0;        // PRA_SORT_TEST_BIN_CAP: a lower bin capacity, so tests reach the large-newt paths
    int dense_epoch_bits = 16;   // PRA_DENSE_EPOCH_BITS: at most this many epoch bits in claim slots (0: none)
    DBuf segb;                   // segment bounds of the segmented sort, then its largest segment
    // timed launches of an iteration, resolved per candidate after its readback
    struct TuneSample {
        int knob, band, var;
        hipEvent_t a, b;
        size_t oi;
        u64 cap;
    };
    std::vector<TuneSample> tune_pending;
    // samples whose events may not have completed when the iteration's summary
    // arrives (the placement publishes it before it ends), with their
    // candidates in `cap`.
    // A claim-table sample of the ranked-membership choice also has the events
    // of its sort, which ranked membership needs none of.
    struct LateSample {
        TuneSample s;
        bool sorts;
        hipEvent_t sort_a, sort_b;
    };
    std::vector<LateSample> tune_late;
    size_t lb_zeroed = 0;        // words of lb_status known to be zero-initialised
    u32 sort_epoch = 0;
    u64 dedup_epoch = 0;
    u64* host_stage = nullptr;  // pinned
    size_t host_stage_cap = 0;
    u64* mailbox = nullptr;     // pinned, written by the publish kernel
    size_t mailbox_cap = 0;
    u64 pub_seq = 0;            // sequence number of the last publication
    u64 pub_wait = 0;           // the one the host waits for
    bool pub_open = false;      // a publication is under way: the mailbox is taken
    hipEvent_t pub_ev = nullptr;
    std::string err;
    // profiling
    u32 prof_mask = 0;           // bit k: time kernel class k
    KStat kst[K_COUNT];
    struct Pending { int k; hipEvent_t a, b; double bytes; };
    std::vector<Pending> pending;
    // (index into pending, bytes per candidate, output index) to fix up once counts are read back
    std::vector<std::tuple<size_t, double, size_t>> per_candidate;
    std::vector<hipEvent_t> evpool;

    pra_ctx()
    {
        for (int i = 0; i < K_COUNT; i++) kst[i].name = kNames[i];
    }
    ~pra_ctx()
    {
        resolve_prof();
        // stream-ordered buffers are returned before their stream goes away
        if (st) (void)hipStreamSynchronize(st);
        groups.clear();
        for (DBuf* b : {&hist, &offs, &sort_tmp, &flags_buf, &stage, &stage2, &orand, &tmp64a, &tmp64b,
                        &tmp64c, &cand, &dest, &slot_of, &keep, &first, &ghist, &gofs, &lb_status, &lb_ctr, &ktmp,
                        &idxa, &idxb, &posadj_dev, &rep_words, &rctl, &ttab, &kp, &part_scratch, &segb})
            b->release();
        for (DBuf& b : jobtab) b.release();
        const bool ok = st && hipStreamSynchronize(st) == hipSuccess;
        if (ok)
            small_retire(st);
        else if (st)
            small_flush(st);
        for (auto& t : tune_late)
            for (hipEvent_t e : {t.s.a, t.s.b, t.sort_a, t.sort_b})
                if (e) evpool.push_back(e);
        for (auto e : evpool) (void)hipEventDestroy(e);
        if (st) {
            stream_idle(st);
            std::lock_guard<std::mutex> lk(g_acct_mu);
            g_acct.erase(st);
        }
        if (host_stage) (void)hipHostFree(host_stage);
        pinned_put(mailbox, mailbox_cap * sizeof(u64), hipHostMallocCoherent, ok);
        for (size_t i = 0; i < sizeof(job_stage) / sizeof(job_stage[0]); i++)
            pinned_put(job_stage[i], job_stage_cap[i], hipHostMallocDefault, ok);
        if (pub_ev) (void)hipEventDestroy(pub_ev);
        if (st) stream_put(device, st, ok);
    }

    hipEvent_t ev()
    {
        if (!evpool.empty()) {
            hipEvent_t e = evpool.back();
            evpool.pop_back();
            return e;
        }
        hipEvent_t e;
        HIPCHK(hipEventCreate(&e));
        return e;
    }
    int prof_begin(int k, hipEvent_t* a)
    {
        if (!(prof_mask & (1u << k))) return -1;
        *a = ev();
        HIPCHK(hipEventRecord(*a, st));
        return k;
    }
    // event opening a timed launch of a tuned knob, or null when not timing
    hipEvent_t tune_begin(bool timing)
    {
        if (!timing) return nullptr;
        hipEvent_t a = ev();
        HIPCHK(hipEventRecord(a, st));
        return a;
    }
    void tune_end(hipEvent_t a, int knob, int band, int var, size_t oi, u64 cap)
    {
        if (!a) return;
        hipEvent_t b = ev();
        HIPCHK(hipEventRecord(b, st));
        tune_pending.push_back({knob, band, var, a, b, oi, cap});
    }
    void prof_end(int k, hipEvent_t a, double bytes) noexcept
    {
        if (k < 0) return;
        hipEvent_t b = nullptr;
        if (!evpool.empty()) {
            b = evpool.back();
            evpool.pop_back();
        } else if (hipEventCreate(&b) != hipSuccess) {
            return;
        }
        if (hipEventRecord(b, st) != hipSuccess) return;
        pending.push_back({k, a, b, bytes});
    }
    void resolve_prof()
    {
        if (pending.empty()) return;
        if (hipStreamSynchronize(st) != hipSuccess) return;
        for (auto& p : pending) {
            float ms = 0;
            if (hipEventElapsedTime(&ms, p.a, p.b) == hipSuccess) {
                kst[p.k].ms += ms;
                kst[p.k].launches++;
                kst[p.k].bytes += p.bytes;
            }
            evpool.push_back(p.a);
            evpool.push_back(p.b);
        }
        pending.clear();
    }

    u64* host_buf(size_t words)
    {
        if (words > host_stage_cap) {
            if (host_stage) HIPCHK(hipHostFree(host_stage));
            host_stage = nullptr;
            size_t c = std::max<size_t>(words, 1024);
            HIPCHK(hipHostMalloc((void**)&host_stage, c * sizeof(u64)));
            host_stage_cap = c;
        }
        return host_stage;
    }
    // pinned staging for job tables copied to the device: a slot is rewritten
    // only after the host has waited for a kernel enqueued behind its previous
    // copy (see the slot list), and a larger buffer waits for the stream too
    char* job_stage_buf(int slot, size_t bytes)
    {
        if (bytes > job_stage_cap[slot]) {
            if (job_stage[slot]) {
                HIPCHK(hipStreamSynchronize(st));
                pinned_put(job_stage[slot], job_stage_cap[slot], hipHostMallocDefault, true);
            }
            job_stage[slot] = nullptr;
            const size_t c = std::max<size_t>(bytes, 64 << 10);
            job_stage[slot] = (char*)pinned_get(c, hipHostMallocDefault);
            job_stage_cap[slot] = c;
        }
        return job_stage[slot];
    }
    u64* mailbox_buf(size_t words)
    {
        if (words > mailbox_cap) {
            if (mailbox) HIPCHK(hipHostFree(mailbox));
            mailbox = nullptr;
            mailbox_cap = 0;
            size_t c = std::max<size_t>(words, 1024);
            mailbox = (u64*)pinned_get(c * sizeof(u64), hipHostMallocCoherent);
            memset(mailbox, 0, c * sizeof(u64));
            mailbox_cap = c;
        }
        return mailbox;
    }
    u32* dflags() { return flags_buf.as<u32>(); }
};

namespace {

// instance g of a context (created on first use)
static Group& grp(pra_ctx* c, int g)
{
    while ((int)c->groups.size() <= g) c->groups.emplace_back(new Group());
    return *c->groups[(size_t)g];
}

// Device memory that only speed needs -- the tables of ranked membership,
// emission in digits and one-block iterations, claim tables, second full
// buffers, tables that are out of date -- given back when a buffer that a
// program cannot do without is refused.  All of it is at rest, or used only by
// work already enqueued, outside of a NoYield's life.
static bool yield_tables(pra_ctx* c)
{
    if (c->no_yield) return false;
    bool any = false;
    auto drop = [&](DBuf& b) {
        any = any || b.p;
        b.release();
    };
    for (pra_rel* R : c->rels) {
        for (DBuf* b : {&R->fresh, &R->dirty, &R->sbpre, &R->linep, &R->places, &R->dtab, &R->rk_words[0],
                        &R->rk_words[1], &R->rk_first[0], &R->rk_first[1]})
            drop(*b);
        R->fresh_sbs = R->dtab_cap = 0;
        for (int v : {PRA_DELTA, PRA_FULL}) R->rk_gen[v] = ~0ULL;
        if (!c->merges_open) drop(R->merged);
        if (!R->mt_valid) drop(R->mt);
        if (!R->bm_valid) drop(R->bm);
    }
    drop(c->first);
    c->first_words = 0;
    c->lean++;
    return any;
}

struct NoYield {
    pra_ctx* c;
    explicit NoYield(pra_ctx* c_) : c(c_) { c->no_yield++; }
    ~NoYield() { end(); }
    void end()
    {
        if (c) c->no_yield--;
        c = nullptr;
    }
    NoYield(const NoYield&) = delete;
    NoYield& operator=(const NoYield&) = delete;
};

struct Prof {
    pra_ctx* c;
    int k;
    hipEvent_t a;
    double bytes;
    Prof(pra_ctx* c_, int k_, double b) : c(c_), k(-1), a(nullptr), bytes(b) { k = c->prof_begin(k_, &a); }
    ~Prof() { c->prof_end(k, a, bytes); }
};

// a timed launch whose byte count is (bytes per candidate) x (candidates of
// output `oi`), known only after the iteration's readback
struct ProfPerCand {
    pra_ctx* c;
    int k;
    hipEvent_t a;
    double per;
    size_t oi;
    ProfPerCand(pra_ctx* c_, int k_, double per_, size_t oi_) : c(c_), k(-1), a(nullptr), per(per_), oi(oi_)
    {
        k = c->prof_begin(k_, &a);
    }
    ~ProfPerCand()
    {
        if (k < 0) return;
        c->prof_end(k, a, 0.0);
        c->per_candidate.emplace_back(c->pending.size() - 1, per, oi);
    }
};

// room for a job table of up to `bytes`
static char* reserve_table(pra_ctx* c, int slot, size_t bytes)
{
    char* hs = c->job_stage_buf(slot, bytes);
    c->jobtab[slot].reserve(bytes, c->st);
    return hs;
}

// A batched launch's job table: through its pinned staging slot into device
// memory, ordered on the context stream; returns the device copy.
static char* stage_table(pra_ctx* c, int slot, const void* data, size_t bytes)
{
    char* hs = reserve_table(c, slot, bytes);
    memcpy(hs, data, bytes);
    HIPCHK(hipMemcpyAsync(c->jobtab[slot].p, hs, bytes, hipMemcpyHostToDevice, c->st));
    return c->jobtab[slot].as<char>();
}

// D2D copies of several ranges: one copy when there is one, else one launch
static void copy_ranges(pra_ctx* c, int slot, const std::vector<CopyJob>& jobs)
{
    if (jobs.empty()) return;
    if (jobs.size() == 1) {
        HIPCHK(hipMemcpyAsync(jobs[0].dst, jobs[0].src, jobs[0].words * 8, hipMemcpyDeviceToDevice, c->st));
        return;
    }
    std::vector<char> t(jobs.size() * sizeof(CopyJob) + (jobs.size() + 1) * 4);
    memcpy(t.data(), jobs.data(), jobs.size() * sizeof(CopyJob));
    u32* bb = (u32*)(t.data() + jobs.size() * sizeof(CopyJob));
    bb[0] = 0;
    for (size_t k = 0; k < jobs.size(); k++) bb[k + 1] = bb[k] + (u32)((jobs[k].words + 2047) / 2048);
    const char* d = stage_table(c, slot, t.data(), t.size());
    pra_launch_copy_many(c->st, (const CopyJob*)d, (int)jobs.size(), bb[jobs.size()]);
    check_launch("copy_many");
}

// ----------------------------------------------------------------- scans ---

static void prepare_lookback(pra_ctx* c, u64 n);
static u32 next_sort_epoch(pra_ctx* c);

// exclusive scans on the context stream (one-pass look-back above
// PRA_SMALL_SCAN elements, over the sort's status words)
static void scan_u64(pra_ctx* c, const u64* in, u64* out, u64 n, u64* total)
{
    Prof p(c, K_SCAN, 16.0 * n);
    u32 ep = 0;
    if (n > PRA_SMALL_SCAN) {
        prepare_lookback(c, n);
        ep = next_sort_epoch(c);
    }
    pra_scan_u64(c->st, in, out, n, c->lb_status.as<u64>(), c->lb_ctr.as<u32>(), ep, c->dflags(), total);
    check_launch("scan_u64");
}

static void scan_u32(pra_ctx* c, const u32* in, u32* out, u64 n, u32* total)
{
    Prof p(c, K_SCAN, 8.0 * n);
    u32 ep = 0;
    if (n > PRA_SMALL_SCAN) {
        prepare_lookback(c, n);
        ep = next_sort_epoch(c);
    }
    pra_scan_u32(c->st, in, out, n, c->lb_status.as<u64>(), c->lb_ctr.as<u32>(), ep, c->dflags(), total);
    check_launch("scan_u32");
}

static void check_flags(u32 f)
{
    if (f & (PRA_FLAG_COLLISION | PRA_FLAG_INDEX_COLLISION))
        throw PraError(PRA_E_COLLISION, "64-bit key hash collision between distinct keys");
    if (f & PRA_FLAG_TABLE_FULL) throw PraError(PRA_E_HIP, "hash table overflow");
    if (f & PRA_FLAG_SORT_STALL) throw PraError(PRA_E_HIP, "sort or scan look-back did not complete");
    if (f & PRA_FLAG_BIN_OVERFLOW) throw PraError(PRA_E_HIP, "sort bin exceeds its capacity");
    if (f & PRA_FLAG_SCAN_OVERFLOW) throw PraError(PRA_E_HIP, "prefix sum exceeds 2^46");
}

// Read back `words` u64 from device memory in one synchronization, together
// with the device error flags.  Flags are sticky: kernels only ever set them
// on a detected error, and every synchronization point checks them.
// A few words are published (below): a kernel and a spin cost about 10 us
// where two copies and a blocking wait cost about 25.
constexpr size_t kPublishWords = 256;
static u64* publish_readback(pra_ctx* c, const u64* src, size_t words);
static u64* readback(pra_ctx* c, const void* src, size_t words)
{
    if (words <= kPublishWords && !c->pub_open) {
        u64* h = publish_readback(c, (const u64*)src, words);
        stream_idle(c->st);
        return h;
    }
    u64* h = c->host_buf(words + 1);
    if (words) HIPCHK(hipMemcpyAsync(h, src, words * 8, hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipMemcpyAsync(h + words, c->flags_buf.p, 8, hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    stream_idle(c->st);
    check_flags((u32)h[words]);
    return h;
}

static void sync_check(pra_ctx* c) { readback(c, nullptr, 0); }

// The per-iteration readback: one kernel copies the summary words and the
// error flags into pinned host memory (no copy-engine transfers), then, once
// they are visible to the host, a sequence number in the word before them.  The host spins
// on that word instead of sleeping in a blocking synchronization or waiting
// for the kernel's completion to be signalled; an event recorded behind the
// kernel reports errors, and after a while the host falls back to a blocking
// wait on it.
// fold: a newt fold still to run, done by the publishing kernel itself
// by_kernel: a kernel given publish_take's mailbox publishes (the placement of
// the iteration's one ranked output, a one-block build), and this call only
// takes note of it
static u64* publish_take(pra_ctx* c, size_t words, u64* seq)
{
    // mailbox word 0: the sequence number; the summary and flags after it
    u64* h = c->mailbox_buf(words + 2) + 1;
    *seq = ++c->pub_seq;
    c->pub_open = true;
    return h;
}

static u64* publish_begin(pra_ctx* c, const u64* src, size_t words, const NewtFoldArgs* fold = nullptr,
                          bool by_kernel = false)
{
    u64 seq = c->pub_seq;
    u64* h = by_kernel ? c->mailbox + 1 : publish_take(c, words, &seq);
    c->pub_wait = seq;
    if (by_kernel) {
    } else if (fold)
        pra_launch_newt_fold_publish(c->st, *fold, src, words, c->flags_buf.as<u32>(), h, seq);
    else
        pra_launch_publish(c->st, src, words, c->flags_buf.as<u32>(), h, seq);
    check_launch("publish");
    if (!c->pub_ev) HIPCHK(hipEventCreateWithFlags(&c->pub_ev, hipEventDisableTiming));
    HIPCHK(hipEventRecord(c->pub_ev, c->st));
    return h;
}

// waits for the summary of publish_begin (work enqueued after it keeps the
// device busy meanwhile) and checks the error flags
static u64* publish_wait(pra_ctx* c, u64* h, size_t words)
{
    auto t0 = std::chrono::steady_clock::now();
    for (u32 k = 0;; k++) {
        if (__atomic_load_n(h - 1, __ATOMIC_ACQUIRE) == c->pub_wait) break;
        if ((k & 63) == 63) {
            const hipError_t q = hipEventQuery(c->pub_ev);
            if (q != hipSuccess && q != hipErrorNotReady) HIPCHK(q);
            if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(20)) {
                HIPCHK(hipEventSynchronize(c->pub_ev));
                break;
            }
        }
    }
    c->pub_open = false;
    check_flags((u32)h[words]);
    return h;
}

static u64* publish_readback(pra_ctx* c, const u64* src, size_t words)
{
    return publish_wait(c, publish_begin(c, src, words), words);
}

// ------------------------------------------------------------------ sort ---

// look-back status words for `n` rows, zero-initialised once per allocation
static void prepare_lookback(pra_ctx* c, u64 n)
{
    size_t need = (size_t)pra_tiles(n) * PRA_RADIX;
    if (need > c->lb_zeroed) {
        c->lb_status.reserve(need * 8, c->st);
        size_t words = c->lb_status.cap / 8;
        pra_launch_fill_u64(c->st, c->lb_status.as<u64>(), words, 0);
        c->lb_zeroed = words;
        c->sort_epoch = 0;
    }
    if (!c->lb_ctr.p) {   // per-pass tile counters; each sort pass returns its own to zero
        c->lb_ctr.reserve(PRA_MAXPASS * 4 + 8, c->st);
        pra_launch_fill_u64(c->st, c->lb_ctr.as<u64>(), (PRA_MAXPASS * 4 + 8) / 8, 0);
    }
    c->ghist.reserve(PRA_MAXPASS * PRA_RADIX * 4, c->st);
    c->gofs.reserve(PRA_MAXPASS * PRA_RADIX * 4, c->st);
}

static u32 next_sort_epoch(pra_ctx* c)
{
    if (++c->sort_epoch >= 0xFFFF) {
        pra_launch_fill_u64(c->st, c->lb_status.as<u64>(), c->lb_zeroed, 0);
        c->sort_epoch = 1;
    }
    return c->sort_epoch;
}

// Keyed sort of rows (more than one block holds): the varying bits of (bucket,
// columns) as a multi-word key, one or two counting passes over (word 0, row
// index) pairs, then an LDS sort and row gather per segment.  A pass moves 24
// bytes a row instead of 16 w, and there are two or three instead of one per
// varying byte.  False, with r untouched, when a segment is too large for one
// block (skewed keys) or there is no room for the pairs: the byte passes take
// any keys in no more than the rows' own bytes.  With bnd (bucketed), the
// bucket bounds are written too.
// One counting pass up to 2^18 rows (segments of at most 1,024 on average, 256
// blocks), two beyond.
// With a dictionary (G), keys of more than one word take the data columns'
// ranks instead of their bits when that makes them one word (a value without a
// rank: false).
// *dup (nullable): whether two rows' keys may be equal.
static bool sort_rows_keyed(pra_ctx* c, Rows& r, int w, int jcc, int keycols, const u64* orm, bool bucketed, u64* bnd,
                            const Group* G, bool* dup)
{
    const u64 n = r.n;
    KeyLayout L;
    memset(&L, 0, sizeof(L));
    L.jcc = jcc;
    L.nb = (u64)c->nb;
    auto bits_of = [](u64 x) { return x ? 64 - __builtin_clzll(x) : 0; };
    auto layout = [&](int rbits) {   // rbits: bits of a rank (0: no ranks)
        L.nf = L.bits = 0;
        if (bucketed) pra_key_field(L, -1, 0, bits_of(L.nb - 1));
        for (int col = 0; col < keycols; col++) {
            const u64 vary = (orm && col < 16) ? (orm[col] ^ orm[16 + col]) : ~0ULL;
            if (!vary) continue;
            const int lo = __builtin_ctzll(vary), bits = bits_of(vary) - lo;
            if (rbits && col < w - 1 && rbits < bits)
                pra_key_field(L, col, 0, rbits, 1);
            else
                pra_key_field(L, col, lo, bits);
        }
    };
    layout(0);
    if (L.bits > 64 && G && G->dict_state == 1 && G->dict_n > 1) {
        layout(bits_of(G->dict_n - 1));
        L.dict = G->dict.as<u64>();
        L.dict_cap = G->dict_cap;
        if (L.bits > 64) layout(0);
    }
    const int np = n <= (1ULL << 18) ? 1 : 2;
    const int sb = np == 1 ? 8 : std::min(16, std::max(9, bits_of((n - 1) / 2048)));
    const u32 nseg = 1u << sb;
    const int top = 64 - sb;
    DBuf *ka = &c->tmp64a, *kb = &c->ktmp;
    try {
        prepare_lookback(c, n);
        for (DBuf* b : {ka, kb}) b->reserve(n * 8, c->st);
        for (DBuf* b : {&c->idxa, &c->idxb}) b->reserve(n * 4, c->st);
        c->segb.reserve(((size_t)nseg + 5) * 8 + (size_t)nseg * 4, c->st);
        c->sort_tmp.reserve(n * w * 8, c->st);
    } catch (const PraError& e) {
        if (e.code != PRA_E_BUDGET && e.code != PRA_E_NOMEM) throw;
        for (DBuf* b : {ka, kb, &c->idxa, &c->idxb}) b->release();
        return false;
    }
    u64* seg = c->segb.as<u64>();
    u64* stat = seg + nseg + 1;   // largest segment, larger segments listed, overflow or missing rank, equal keys
    u32* list = (u32*)(seg + nseg + 5);
    pra_launch_fill_u64(c->st, c->ghist.as<u64>(), np * PRA_RADIX / 2, 0);
    pra_launch_fill_u64(c->st, stat, 4, 0);
    {
        Prof p(c, K_RADIX_HIST, 8.0 * n * (w + 1));
        pra_launch_sort_keys(c->st, r.d(), n, w, L, np, ka->as<u64>(), c->ghist.as<u32>(), stat + 2);
        check_launch("sort_keys");
    }
    pra_launch_sort_scan(c->st, c->ghist.as<u32>(), np, c->gofs.as<u32>(), nullptr, (u32)c->nb, n);
    check_launch("sort_scan");
    for (int i = 0; i < np; i++) {
        const u32 ep = next_sort_epoch(c);
        Prof p(c, K_RADIX_SCATTER, 24.0 * n);
        pra_launch_sort_scatter(c->st, ka->as<u64>(), kb->as<u64>(), n, 1,
                                DigitSpec{0, np == 2 && i == 0 ? 48 : 56, 0, 0, 0},
                                c->gofs.as<u32>() + (size_t)i * PRA_RADIX, c->lb_status.as<u64>(),
                                c->lb_ctr.as<u32>() + i, ep, c->dflags(), i ? c->idxa.as<u32>() : nullptr,
                                c->idxb.as<u32>());
        check_launch("key_sort_scatter");
        std::swap(ka, kb);
        c->idxa.swap(c->idxb);
    }
    if (np == 2) {
        pra_launch_seg_bounds(c->st, ka->as<u64>(), n, top, nseg, seg, stat, list);
        check_launch("seg_bounds");
    }
    {
        Prof p(c, K_BLOCK_SORT, 12.0 * n + 16.0 * n * w);
        pra_launch_keyseg_sort(c->st, ka->as<u64>(), c->idxa.as<u32>(), np == 2 ? seg : nullptr,
                               c->gofs.as<u32>(), nseg, list, stat, top, n, r.d(), w, L, c->sort_tmp.as<u64>(), bnd,
                               stat + 2);
        check_launch("keyseg_sort");
    }
    const u64* status = readback(c, stat + 2, 2);
    if (status[0]) return false;
    if (dup) *dup = status[1] != 0;
    r.buf.swap(c->sort_tmp);
    r.sorted = true;
    return true;
}

// One-sweep LSD radix sort of rows by (bucket, col0 .. col[keycols-1]).
// `orm` holds the OR (words 0..15) and AND (16..31) of the first 16 key
// columns: digits equal in every row are skipped.  When the bucket digit is
// sorted and nb <= 256, the bucket bounds are written to `bnd` (nb+1 words)
// and true is returned.
// G (nullable): the instance whose dictionary may shorten the keys.  dup
// (nullable): receives whether the sorted rows may hold equal keys.
// With `defer`, a sort that takes the one-block path is not launched: its job
// (into `defer_out`, which the caller swaps with r's buffer once the batch
// has been launched) is returned in *defer, with defer->n = 0 otherwise.
static bool sort_rows_masked(pra_ctx* c, Rows& r, int w, int jcc, int keycols, const u64* orm, u64* bnd,
                             bool by_bucket = true, SmallSortJob* defer = nullptr, DBuf* defer_out = nullptr,
                             const Group* G = nullptr, bool* dup = nullptr)
{
    if (defer) defer->n = 0;
    if (dup) *dup = r.n > 1;
    u64 n = r.n;
    if (n <= 1) {
        r.sorted = true;
        return false;
    }
    std::vector<DigitSpec> passes;
    for (int col = keycols - 1; col >= 0; col--) {
        u64 vary = (orm && col < 16) ? (orm[col] ^ orm[16 + col]) : ~0ULL;
        for (int sh = 0; sh < 64; sh += PRA_RADIX_BITS)
            if ((vary >> sh) & (PRA_RADIX - 1)) passes.push_back(DigitSpec{col, sh, 0, 0, 0});
    }
    bool bucket_last = false;
    if (c->nb > 1 && by_bucket) {
        for (int sh = 0; ((u64)(c->nb - 1) >> sh) != 0; sh += PRA_RADIX_BITS)
            passes.push_back(DigitSpec{-1, sh, jcc, 0, (u64)c->nb});
        bucket_last = c->nb <= PRA_RADIX;
    }
    if (passes.empty()) {
        r.sorted = true;
        return false;
    }
    // small inputs: one block sorts them in LDS
    const bool bucketed = c->nb > 1 && by_bucket;
    if (n <= PRA_SMALL_SORT) {
        u64* bout = (bnd && bucketed && bucket_last) ? bnd : nullptr;
        if (defer) {
            defer_out->reserve(n * w * 8, c->st);
            *defer = SmallSortJob{r.d(), defer_out->as<u64>(), bout, n, w, jcc, keycols, bucketed ? 1 : 0};
            r.sorted = true;
            return bout != nullptr;
        }
        c->sort_tmp.reserve(n * w * 8, c->st);
        u64* dup_dev = nullptr;
        if (dup) {
            c->orand.reserve(32 * 8, c->st);
            dup_dev = c->orand.as<u64>();
            pra_launch_fill_u64(c->st, dup_dev, 1, 0);
        }
        {
            Prof p(c, K_SMALL_SORT, 8.0 * n * (keycols + 1) + 16.0 * n * w);
            pra_launch_small_sort(c->st, r.d(), n, w, jcc, keycols, (u64)c->nb, bucketed ? 1 : 0,
                                  c->sort_tmp.as<u64>(), bout, dup_dev);
            check_launch("small_sort");
        }
        r.buf.swap(c->sort_tmp);
        r.sorted = true;
        if (dup) *dup = readback(c, dup_dev, 1)[0] != 0;
        return bout != nullptr;
    }
    // the keyed sort, from two passes saved on
    if (n < (1ULL << 32) && passes.size() >= 4) {
        u64* bout = (bnd && bucketed && bucket_last) ? bnd : nullptr;
        if (sort_rows_keyed(c, r, w, jcc, keycols, orm, bucketed, bout, G, dup)) return bout != nullptr;
    }
    // up to PRA_BLOCK_SORT rows: one block runs every pass in one launch
    if (n <= PRA_BLOCK_SORT && passes.size() >= 2 && passes.size() <= PRA_MAXPASS) {
        PassList pl;
        memset(&pl, 0, sizeof(pl));
        pl.np = (int)passes.size();
        for (size_t i = 0; i < passes.size(); i++) pl.p[i] = passes[i];
        c->sort_tmp.reserve(n * w * 8, c->st);
        u64* bout = (bnd && bucket_last) ? bnd : nullptr;
        {
            Prof p(c, K_BLOCK_SORT, 8.0 * n * pl.np + 16.0 * n * w);
            pra_launch_block_sort(c->st, r.d(), n, w, pl, c->sort_tmp.as<u64>(), bout, jcc, (u64)c->nb);
            check_launch("block_sort");
        }
        r.buf.swap(c->sort_tmp);
        r.sorted = true;
        return bout != nullptr;
    }
    prepare_lookback(c, n);
    c->sort_tmp.reserve(n * w * 8, c->st);
    bool wrote_bnd = false;
    for (size_t first = 0; first < passes.size(); first += PRA_MAXPASS) {
        size_t np = std::min<size_t>(PRA_MAXPASS, passes.size() - first);
        PassList pl;
        memset(&pl, 0, sizeof(pl));
        pl.np = (int)np;
        for (size_t i = 0; i < np; i++) pl.p[i] = passes[first + i];
        bool last_chunk = first + np == passes.size();
        pra_launch_fill_u64(c->st, c->ghist.as<u64>(), np * PRA_RADIX / 2, 0);
        {
            Prof p(c, K_RADIX_HIST, 8.0 * n * keycols);
            pra_launch_sort_hist(c->st, r.d(), n, w, pl, c->ghist.as<u32>());
            check_launch("sort_hist");
        }
        u64* bout = (bnd && bucket_last && last_chunk) ? bnd : nullptr;
        pra_launch_sort_scan(c->st, c->ghist.as<u32>(), (int)np, c->gofs.as<u32>(), bout, (u32)c->nb, n);
        check_launch("sort_scan");
        wrote_bnd = wrote_bnd || bout != nullptr;
        for (size_t i = 0; i < np; i++) {
            u32 ep = next_sort_epoch(c);
            Prof p(c, K_RADIX_SCATTER, 16.0 * n * w);
            pra_launch_sort_scatter(c->st, r.d(), c->sort_tmp.as<u64>(), n, w, pl.p[i],
                                    c->gofs.as<u32>() + i * PRA_RADIX, c->lb_status.as<u64>(),
                                    c->lb_ctr.as<u32>() + i, ep, c->dflags(), nullptr, nullptr);
            check_launch("sort_scatter");
            r.buf.swap(c->sort_tmp);
        }
    }
    r.sorted = true;
    return wrote_bnd;
}

static void sort_rows(pra_ctx* c, Rows& r, int w, int jcc, int keycols, bool by_bucket = true,
                      const Group* G = nullptr, bool* dup = nullptr)
{
    if (r.n <= 1) {
        r.sorted = true;
        if (dup) *dup = false;
        return;
    }
    // the one-block sort collects the columns' varying bits itself
    if (r.n <= PRA_SMALL_SORT) {
        sort_rows_masked(c, r, w, jcc, keycols, nullptr, nullptr, by_bucket, nullptr, nullptr, G, dup);
        return;
    }
    int kc = std::min(keycols, 16);
    c->orand.reserve(32 * 8, c->st);
    u64* om = c->orand.as<u64>();
    pra_launch_fill_u64(c->st, om, 16, 0);
    pra_launch_fill_u64(c->st, om + 16, 16, ~0ULL);
    pra_launch_col_orand2(c->st, r.d(), r.n, w, kc, om);
    check_launch("col_orand");
    u64* h = readback(c, om, 32);
    u64 m[32];
    std::copy(h, h + 32, m);
    sort_rows_masked(c, r, w, jcc, keycols, m, nullptr, by_bucket, nullptr, nullptr, G, dup);
}

static int ceil_log2(u64 x);

// Packed sort key of an interned relation's newt rows: bucket * D^arity + the
// column ranks as digits of radix D (the dictionary size), which orders rows
// by (bucket, col0, col1, ..), shifted left by ls so that its top bit is bit
// 63.  bmul = D^arity.  False when the key range does not fit 64 bits.
static bool packed_layout(u64 nb, u64 D, int arity, u64* bmul, int* ls)
{
    unsigned __int128 m = 1;
    for (int i = 0; i < arity; i++) {
        m *= D;
        if (m >> 64) return false;
    }
    unsigned __int128 range = m * nb;
    if (range >> 64) return false;
    int bits = ceil_log2((u64)range);
    *bmul = (u64)m;
    *ls = bits ? 64 - bits : 0;
    return true;
}

// Sort a relation's newt rows by their packed keys (all distinct; R->nkeys in
// newt order, R->kgofs the exclusive offsets of the keys' top-byte bins, and
// the bins of (key, position) pairs filled by the newt scatter).  When the
// largest bin fits its capacity and one block, k_bin_sort orders every bin in
// LDS, gathers the rows and writes the bucket bounds (nb + 1 words);
// otherwise every varying byte gets a one-sweep pass over R->nkeys, followed
// by a row gather and a bounds search.
// With `defer`, the bin sort is not launched: its job (writing into
// `defer_out`, which the caller swaps with newt's buffer once the batch is
// launched) goes to *defer and true is returned.
static bool sort_by_packed_key(pra_ctx* c, pra_rel* R, u64 kor, u64 kand, u64 maxbin, u64 bmul, int ls, u64* bnd,
                               BinSortJob* defer = nullptr, DBuf* defer_out = nullptr)
{
    Rows& r = R->ver[PRA_NEWT];
    const int w = R->w;
    DBuf& keys = R->nkeys;
    const u32* top_ofs = R->kgofs.as<u32>();
    u64 n = r.n;
    u64 vary = kor ^ kand;
    const u64 bin_limit = std::min<u64>(std::min<u64>(R->bin_cap, PRA_BIN_CAP), c->bin_cap_test ? c->bin_cap_test : ~0ULL);
    if (n > 1 && maxbin <= bin_limit) {
        u32 bytes = 0;
        for (int b = 0; b < 7; b++)
            if ((vary >> (8 * b)) & (PRA_RADIX - 1)) bytes |= 1u << b;
        if (defer) {
            defer_out->reserve(n * w * 8, c->st);
            *defer = BinSortJob{R->bin_keys.as<u64>(), R->bin_idx.as<u32>(), top_ofs, r.d(), defer_out->as<u64>(), bnd,
                                n, bmul, (u64)c->nb, R->bin_cap, bytes, w, ls};
            r.sorted = true;
            return true;
        }
        c->sort_tmp.reserve(n * w * 8, c->st);
        {
            Prof p(c, K_BIN_SORT, 12.0 * n + 16.0 * n * w);
            pra_launch_bin_sort(c->st, R->bin_keys.as<u64>(), R->bin_idx.as<u32>(), R->bin_cap, n, top_ofs, bytes,
                                r.d(), w, c->sort_tmp.as<u64>(), bmul, ls, (u64)c->nb, bnd, c->dflags(), maxbin);
            check_launch("bin_sort");
        }
        r.buf.swap(c->sort_tmp);
        r.sorted = true;
        return false;
    }
    // LSD passes over the keys (and the permutation in idxa, from `permuted`
    // on): the byte-pass sort, and the first stage of the segmented one
    bool permuted = false;
    auto run_passes = [&](const std::vector<DigitSpec>& ps) {
        if (ps.empty()) return;
        prepare_lookback(c, n);
        c->ktmp.reserve(n * 8, c->st);
        c->idxa.reserve(n * 4, c->st);
        c->idxb.reserve(n * 4, c->st);
        const int np = (int)ps.size();
        PassList pl;
        memset(&pl, 0, sizeof(pl));
        pl.np = np;
        for (int i = 0; i < np; i++) pl.p[i] = ps[i];
        pra_launch_fill_u64(c->st, c->ghist.as<u64>(), np * PRA_RADIX / 2, 0);
        {
            Prof p(c, K_RADIX_HIST, 8.0 * n);
            pra_launch_sort_hist(c->st, keys.as<u64>(), n, 1, pl, c->ghist.as<u32>());
            check_launch("sort_hist");
        }
        pra_launch_sort_scan(c->st, c->ghist.as<u32>(), np, c->gofs.as<u32>(), nullptr, (u32)c->nb, n);
        check_launch("sort_scan");
        for (int i = 0; i < np; i++) {
            u32 ep = next_sort_epoch(c);
            Prof p(c, K_RADIX_SCATTER, 24.0 * n);
            pra_launch_sort_scatter(c->st, keys.as<u64>(), c->ktmp.as<u64>(), n, 1, ps[i],
                                    c->gofs.as<u32>() + (size_t)i * PRA_RADIX, c->lb_status.as<u64>(),
                                    c->lb_ctr.as<u32>() + i, ep, c->dflags(), permuted ? c->idxa.as<u32>() : nullptr,
                                    c->idxb.as<u32>());
            check_launch("key_sort_scatter");
            keys.swap(c->ktmp);
            c->idxa.swap(c->idxb);
            permuted = true;
        }
    };
    // Segmented sort: two counting passes over the keys' top two bytes
    // order the pairs by their top 16 bits; then the segments of equal top
    // `sb` bits (sized to average 2,048 pairs) are each sorted in LDS by
    // their lower varying bytes, rows gathered in the same kernel.  A segment
    // over PRA_BIN_CAP pairs sends the sort on to the byte passes, which take
    // the permutation as it stands.
    const u64 seg_min = c->bin_cap_test ? 2 : (1ULL << 16);
    std::vector<DigitSpec> top2;
    for (int sh : {48, 56})
        if ((vary >> sh) & (PRA_RADIX - 1)) top2.push_back(DigitSpec{0, sh, 0, 0, 0});
    if (c->seg_sort_on && n >= seg_min && n < (1ULL << 32) && !top2.empty()) {
        run_passes(top2);
        // segments of about 2,048 pairs on average (the keys of one iteration
        // are skewed: with smaller segments the largest still overflows the
        // narrow blocks, and the wide ones then sort many tiny segments)
        const int sb = std::min(16, std::max(9, ceil_log2(std::max<u64>(1, n / 2048))));
        const int top = 64 - sb;
        const u32 nseg = 1u << sb;
        // segment bounds, then the largest segment and the number of those
        // over PRA_SEG_SMALL pairs, then their list
        c->segb.reserve(((size_t)nseg + 3) * 8 + (size_t)nseg * 4, c->st);
        u64* seg = c->segb.as<u64>();
        u64* sst = seg + nseg + 1;
        u32* large = (u32*)(seg + nseg + 3);
        pra_launch_fill_u64(c->st, sst, 2, 0);
        pra_launch_seg_bounds(c->st, keys.as<u64>(), n, top, nseg, seg, sst, large);
        check_launch("seg_bounds");
        const u64* sstat = readback(c, sst, 2);
        const u64 maxseg = sstat[0], nlarge = sstat[1];
        if (maxseg <= PRA_BIN_CAP) {
            const u64 low = vary & ((1ULL << top) - 1);
            u32 bytes = 0;
            for (int b = 0; b < 8; b++)
                if ((low >> (8 * b)) & (PRA_RADIX - 1)) bytes |= 1u << b;
            c->sort_tmp.reserve(n * w * 8, c->st);
            {
                Prof p(c, K_BIN_SORT, 12.0 * n + 16.0 * n * w);
                pra_launch_seg_sort(c->st, keys.as<u64>(), c->idxa.as<u32>(), seg, top, nseg, n, bytes, r.d(), w,
                                    c->sort_tmp.as<u64>(), bmul, ls, (u64)c->nb, bnd, c->dflags(), maxseg, large,
                                    nlarge);
                check_launch("seg_sort");
            }
            r.buf.swap(c->sort_tmp);
            r.sorted = true;
            return false;
        }
    }
    std::vector<DigitSpec> passes;
    for (int sh = 0; sh < 64; sh += PRA_RADIX_BITS)
        if ((vary >> sh) & (PRA_RADIX - 1)) passes.push_back(DigitSpec{0, sh, 0, 0, 0});
    if (n > 1 && !passes.empty()) {
        run_passes(passes);
        c->sort_tmp.reserve(n * w * 8, c->st);
        {
            Prof p(c, K_GATHER, 16.0 * n * w + 4.0 * n);
            pra_launch_gather_rows(c->st, r.d(), c->idxa.as<u32>(), n, w, c->sort_tmp.as<u64>());
            check_launch("gather_rows");
        }
        r.buf.swap(c->sort_tmp);
    }
    r.sorted = true;
    if (c->nb > 1) {
        pra_launch_key_bounds(c->st, keys.as<u64>(), n, bmul, ls, (u64)c->nb, bnd);
        check_launch("key_bounds");
    } else {
        pra_launch_fill_u64(c->st, bnd, 1, 0);
        pra_launch_fill_u64(c->st, bnd + 1, 1, n);
    }
    return false;
}

static int ceil_log2(u64 x)
{
    int b = 0;
    while (b < 64 && (1ULL << b) < x) b++;
    return b;
}

// remove rows equal (in all w columns) to their predecessor; rows sorted
static void unique_rows(pra_ctx* c, Rows& r, int w)
{
    u64 n = r.n;
    if (n <= 1) return;
    c->tmp64a.reserve(n * 8, c->st);
    c->tmp64b.reserve(n * 8 + 8, c->st);
    c->sort_tmp.reserve(n * w * 8, c->st);
    pra_launch_group_flags(c->st, r.d(), n, w, w, c->tmp64a.as<u64>());
    scan_u64(c, c->tmp64a.as<u64>(), c->tmp64b.as<u64>(), n, c->tmp64b.as<u64>() + n);
    pra_launch_compact_rows(c->st, r.d(), n, w, c->tmp64a.as<u64>(), c->tmp64b.as<u64>(), c->sort_tmp.as<u64>());
    check_launch("compact_rows");
    u64* h = readback(c, c->tmp64b.as<u64>() + n, 1);
    r.buf.swap(c->sort_tmp);
    r.n = h[0];
}

// rows in column order into trie order: a stable partition by bucket; bnd
// receives the bucket bounds
static void bucket_rows(pra_ctx* c, const u64* rows, u64 n, int w, int jcc, u64* out, u64* bnd)
{
    c->part_scratch.reserve(pra_partition_scratch_words(n, (u32)c->nb) * 4 + 256, c->st);
    pra_launch_partition(c->st, rows, n, w, jcc, (u32)c->nb, out, bnd, c->part_scratch.as<u32>());
    check_launch("bucket_rows");
}

// The arguments of a one-block dictionary of instance gi, and its tables: when
// at most PRA_DICT_SMALL_WORDS column values of at most PRA_DICT_SMALL_RELS
// versions may hold no more than PRA_DICT_SMALL distinct ones, what one compute
// unit reads and sorts in the time of two or three of the general build's dozen
// launches.  False when they do not, or there is no room for tables of that
// many values.
static bool small_dictionary_args(pra_ctx* c, int gi, DictSmallArgs* args)
{
    Group& G = grp(c, gi);
    DictSmallArgs a{};
    u64 total = 0;
    for (pra_rel* R : c->rels)
        for (int v : {PRA_FULL, PRA_DELTA}) {
            Rows& r = R->ver[v];
            if (R->group != gi || R->view_of || !r.n || !R->arity) continue;
            total += r.n * (u64)R->arity;
            if (a.k == PRA_DICT_SMALL_RELS || total > PRA_DICT_SMALL_WORDS) return false;
            a.rows[a.k] = r.d();
            a.n[a.k] = (u32)r.n;
            a.w[a.k] = R->w;
            a.arity[a.k++] = R->arity;
        }
    if (total == 0) return false;
    G.dict_gen++;   // the tables of the last build end here
    const u64 room = std::min<u64>(total, PRA_DICT_SMALL);
    a.cap = pow2_at_least(std::max<u64>(64, 2 * room));
    a.nb = (u64)c->nb;
    try {
        G.dict.reserve(a.cap * 16, c->st);
        G.vals.reserve(room * 8, c->st);
        if (c->nb > 1) {
            G.lead_vals.reserve(room * 8, c->st);
            G.rank_of.reserve(room * 4, c->st);
            G.lead_of.reserve(room * 4, c->st);
            G.lead_bucket.reserve(room, c->st);
        }
    } catch (const PraError& e) {
        if (e.code != PRA_E_BUDGET && e.code != PRA_E_NOMEM) throw;
        for (DBuf* b : {&G.dict, &G.vals, &G.lead_vals, &G.rank_of, &G.lead_of, &G.lead_bucket}) b->release();
        return false;
    }
    a.dict = G.dict.as<u64>();
    a.vals = G.vals.as<u64>();
    a.lead_vals = G.lead_vals.as<u64>();
    a.rank_of = G.rank_of.as<u32>();
    a.lead_of = G.lead_of.as<u32>();
    a.lead_bucket = G.lead_bucket.as<unsigned char>();
    a.err = c->dflags();
    *args = a;
    return true;
}

// Whether a one-block build of n words of results a job may publish them
// itself: one job does, the results of several are read back together.
static u64* small_jobs_host(pra_ctx* c, size_t njobs, size_t words, u64* seq)
{
    if (njobs == 1 && !c->pub_open) return publish_take(c, words, seq);
    c->tmp64a.reserve(njobs * words * 8, c->st);
    return nullptr;
}

static void build_dictionary(pra_ctx* c, int gi);

// (Re)build the value dictionaries of some instances: the small ones by one
// block each, in one launch.
static void build_dictionaries(pra_ctx* c, const std::vector<int>& groups)
{
    std::vector<DictSmallArgs> jobs;
    std::vector<int> of, general;
    for (int gi : groups) {
        DictSmallArgs a;
        if (small_dictionary_args(c, gi, &a)) {
            jobs.push_back(a);
            of.push_back(gi);
        } else {
            general.push_back(gi);
        }
    }
    if (!jobs.empty()) {
        const u64* n;
        u64 seq = 0;
        if (u64* host = small_jobs_host(c, jobs.size(), 1, &seq)) {
            jobs[0].host = host;
            jobs[0].seq = seq;
            pra_launch_dict_small(c->st, jobs[0]);
            check_launch("dict_small");
            n = publish_wait(c, publish_begin(c, nullptr, 1, nullptr, true), 1);
        } else {
            for (size_t k = 0; k < jobs.size(); k++) jobs[k].out = c->tmp64a.as<u64>() + k;
            const char* d = stage_table(c, JOB_SETUP, jobs.data(), jobs.size() * sizeof(DictSmallArgs));
            pra_launch_dict_small_many(c->st, (const DictSmallArgs*)d, (int)jobs.size());
            check_launch("dict_small_many");
            n = readback(c, c->tmp64a.p, jobs.size());
        }
        for (size_t k = 0; k < jobs.size(); k++) {
            Group& G = grp(c, of[k]);
            if (n[k] == ~0ULL) {
                general.push_back(of[k]);
                continue;
            }
            G.dict_cap = jobs[k].cap;
            G.dict_n = n[k];
            G.dict_state = 1;
        }
    }
    for (int gi : general) build_dictionary(c, gi);
}

// (Re)build instance gi's value dictionary from the key columns of every
// relation of that instance.
static void build_dictionary(pra_ctx* c, int gi)
{
    Group& G = grp(c, gi);
    u64 total = 0;
    for (pra_rel* R : c->rels)
        if (R->group == gi && !R->view_of)
            for (int v : {PRA_FULL, PRA_DELTA}) total += R->ver[v].n * (u64)R->arity;
    if (total == 0) return;
    G.dict_gen++;   // the tables of the last build end here, whether or not this one comes to its end
    Rows V;
    V.buf.reserve(total * 8, c->st);
    u64 off = 0;
    for (pra_rel* R : c->rels)
        for (int v : {PRA_FULL, PRA_DELTA}) {
            if (R->group != gi || R->view_of) continue;
            Rows& r = R->ver[v];
            pra_launch_collect_cols(c->st, r.d(), r.n, R->w, R->arity, V.d() + off);
            off += r.n * (u64)R->arity;
        }
    check_launch("collect_cols");
    V.n = total;
    sort_rows(c, V, 1, 0, 1, false);
    unique_rows(c, V, 1);
    u64 cap = pow2_at_least(std::max<u64>(64, 2 * V.n));
    G.dict.reserve(cap * 16, c->st);
    pra_launch_fill_u64(c->st, G.dict.as<u64>(), cap * 2, 0);
    pra_launch_dict_insert(c->st, V.d(), V.n, G.dict.as<u64>(), cap, c->dflags());
    check_launch("dict_insert");
    G.vals.reserve(V.n * 8, c->st);
    HIPCHK(hipMemcpyAsync(G.vals.p, V.d(), V.n * 8, hipMemcpyDeviceToDevice, c->st));
    if (c->nb > 1) {
        G.lead_vals.reserve(V.n * 8, c->st);
        G.rank_of.reserve(V.n * 4, c->st);
        G.lead_of.reserve(V.n * 4, c->st);
        G.lead_bucket.reserve(V.n, c->st);
        c->tmp64a.reserve((size_t)(c->nb + 1) * 8, c->st);
        bucket_rows(c, V.d(), V.n, 1, 1, G.lead_vals.as<u64>(), c->tmp64a.as<u64>());
        pra_launch_dict_bucket_rank(c->st, G.lead_vals.as<u64>(), V.n, G.dict.as<u64>(), cap, G.rank_of.as<u32>(),
                                    G.lead_of.as<u32>(), (u64)c->nb, G.lead_bucket.as<unsigned char>());
        check_launch("dict_bucket_rank");
    }
    sync_check(c);
    G.dict_cap = cap;
    G.dict_n = V.n;
    G.dict_state = 1;
}

// The bits of a dense output's rank indexes put rows in trie order when a
// row's bucket is a function of its first column (their leading digit is then
// the bucket-major rank); with more join columns and several buckets they put
// them in column order.
static bool by_bucket(const pra_ctx* c, const pra_rel* R) { return c->nb > 1 && R->jcc == 1; }
static bool bits_in_trie_order(const pra_ctx* c, const pra_rel* R) { return c->nb == 1 || R->jcc == 1; }

// Order an interned relation's full version through its membership bitmap
// (k_bm_place): one read and one write of the rows, where a sort moves them
// several times.  Taken when the bitmap holds exactly the keys of full --
// current for the dictionary, keyed on every column, no delta, as many set
// bits as rows.  The bitmap is read once more, so a rank space of more than 64
// words a row is left to the sort.
// Measured on the 150x150 grid (128 M rows of 24 bytes, 8 buckets), solve and
// ordered result: 132.0 ms with 26 byte passes over the rows, 63.8 ms this way;
// a 20,000-vertex random graph on one bucket (72 M rows) 66.3 -> 30.3 ms.
// False when the version is not of that kind, or there is no room.
static bool order_by_bitmap(pra_ctx* c, pra_rel* R)
{
    Group& G = grp(c, R->group);
    Rows& r = R->ver[PRA_FULL];
    const u64 n = r.n, D = G.dict_n;
    const int kw = R->bm_kw;
    if (!R->bm_valid || R->bm_gen != G.dict_gen || kw != R->arity || R->ver[PRA_DELTA].n || n < 2 || n >= (1ULL << 32))
        return false;
    u64 bits = 1;
    for (int i = 0; i < kw; i++) bits *= D;
    const u64 words = (bits + 63) / 64, nblk = (words * 64 + PRA_BM_BITS - 1) / PRA_BM_BITS;
    if (words > 64 * n + 4096) return false;
    try {
        c->tmp64a.reserve((nblk + 2) * 4, c->st);
    } catch (const PraError& e) {
        if (e.code != PRA_E_BUDGET && e.code != PRA_E_NOMEM) throw;
        c->tmp64a.release();
        return false;
    }
    u32* prefix = c->tmp64a.as<u32>();
    const u64* bm = R->bm.as<u64>();
    pra_launch_bm_count(c->st, bm, words, nblk, prefix);
    scan_u32(c, prefix, prefix, nblk, prefix + nblk);
    if ((u32)readback(c, prefix + nblk, 1)[0] != (u32)n) return false;
    c->sort_tmp.reserve(n * R->w * 8, c->st);
    {
        Prof p(c, K_GATHER, 16.0 * n * R->w);
        pra_launch_bm_place(c->st, r.d(), n, R->w, kw, G.dict.as<u64>(), G.dict_cap, D, by_bucket(c, R), bm, words,
                            prefix, c->sort_tmp.as<u64>());
        check_launch("bm_place");
    }
    R->touched(PRA_FULL);
    if (bits_in_trie_order(c, R)) {
        r.buf.swap(c->sort_tmp);
    } else {
        R->bnd[PRA_FULL].reserve((size_t)(c->nb + 1) * 8, c->st);
        bucket_rows(c, c->sort_tmp.as<u64>(), n, R->w, R->jcc, r.d(), R->bnd[PRA_FULL].as<u64>());
        R->bnd_valid[PRA_FULL] = true;
    }
    r.sorted = true;
    return true;
}

static void ensure_sorted(pra_ctx* c, pra_rel* R, int v)
{
    Rows& r = R->ver[v];
    if (r.sorted) return;
    if (v == PRA_FULL && order_by_bitmap(c, R)) return;
    sort_rows(c, r, R->w, R->jcc, R->w, true, &grp(c, R->group));
    R->touched(v);
}

static const u64* bucket_bounds(pra_ctx* c, pra_rel* R, int v)
{
    Rows& r = R->ver[v];
    R->bnd[v].reserve((size_t)(c->nb + 1) * 8, c->st);
    if (!R->bnd_valid[v]) {
        if (c->nb == 1) {
            pra_launch_fill_u64(c->st, R->bnd[v].as<u64>(), 1, 0);
            pra_launch_fill_u64(c->st, R->bnd[v].as<u64>() + 1, 1, r.n);
            check_launch("bucket_bounds");
        } else {
            pra_launch_bucket_bounds(c->st, r.d(), r.n, R->w, R->jcc, (u64)c->nb, R->bnd[v].as<u64>());
            check_launch("bucket_bounds");
        }
        R->bnd_valid[v] = true;
    }
    return R->bnd[v].as<u64>();
}

// The indexes of sorted versions of at most PRA_INDEX_SMALL rows that have none
// yet, by one block each, in one launch; a version with more rows, or without
// room for a table of that many runs, is left to ensure_index.
static void small_indexes(pra_ctx* c, const std::vector<std::pair<pra_rel*, int>>& versions)
{
    std::vector<IndexSmallArgs> jobs;
    std::vector<std::pair<pra_rel*, int>> of;
    for (auto& rv : versions) {
        pra_rel* R = rv.first;
        const int v = rv.second;
        Rows& r = R->ver[v];
        if (R->idx_valid[v] || !r.sorted || !r.n || r.n > PRA_INDEX_SMALL) continue;
        if (std::find(of.begin(), of.end(), rv) != of.end()) continue;
        try {
            R->idx[v].reserve(pow2_at_least(std::max<u64>(64, 2 * r.n)) * 3 * 8, c->st);
        } catch (const PraError& e) {
            if (e.code != PRA_E_BUDGET && e.code != PRA_E_NOMEM) throw;
            continue;
        }
        IndexSmallArgs a{};
        a.rows = r.d();
        a.n = (u32)r.n;
        a.w = R->w;
        a.jcc = R->jcc;
        a.table = R->idx[v].as<u64>();
        a.err = c->dflags();
        jobs.push_back(a);
        of.push_back(rv);
    }
    if (jobs.empty()) return;
    Prof p(c, K_INDEX_BUILD, 8.0 * jobs[0].n * jobs[0].jcc);
    const u64* h;
    u64 seq = 0;
    if (u64* host = small_jobs_host(c, jobs.size(), 2, &seq)) {
        jobs[0].host = host;
        jobs[0].seq = seq;
        pra_launch_index_small(c->st, jobs[0]);
        check_launch("index_small");
        h = publish_wait(c, publish_begin(c, nullptr, 2, nullptr, true), 2);
    } else {
        for (size_t k = 0; k < jobs.size(); k++) jobs[k].out = c->tmp64a.as<u64>() + 2 * k;
        const char* d = stage_table(c, JOB_SETUP, jobs.data(), jobs.size() * sizeof(IndexSmallArgs));
        pra_launch_index_small_many(c->st, (const IndexSmallArgs*)d, (int)jobs.size());
        check_launch("index_small_many");
        h = readback(c, c->tmp64a.p, 2 * jobs.size());
    }
    for (size_t k = 0; k < jobs.size(); k++) {
        pra_rel* R = of[k].first;
        const int v = of[k].second;
        R->idx_maxlen[v] = h[2 * k];
        R->idx_cap[v] = pow2_at_least(std::max<u64>(64, 2 * h[2 * k + 1]));
        R->idx_valid[v] = true;
    }
}

// (key -> first row, count) index over the sorted rows of a version
static void ensure_index(pra_ctx* c, pra_rel* R, int v)
{
    if (R->idx_valid[v]) return;
    ensure_sorted(c, R, v);
    small_indexes(c, {{R, v}});
    if (R->idx_valid[v]) return;
    Rows& r = R->ver[v];
    u64 n = r.n;
    if (n == 0) {
        R->idx_cap[v] = 0;
        R->idx_maxlen[v] = 0;
        R->idx_valid[v] = true;
        return;
    }
    Prof p(c, K_INDEX_BUILD, 8.0 * n * R->jcc);
    c->tmp64a.reserve(n * 8, c->st);
    c->tmp64b.reserve((n + 1) * 8, c->st);
    c->tmp64c.reserve((n + 1) * 8, c->st);
    pra_launch_group_flags(c->st, r.d(), n, R->w, R->jcc, c->tmp64a.as<u64>());
    scan_u64(c, c->tmp64a.as<u64>(), c->tmp64b.as<u64>(), n, c->tmp64b.as<u64>() + n);
    pra_launch_group_compact(c->st, c->tmp64a.as<u64>(), c->tmp64b.as<u64>(), n, c->tmp64c.as<u64>());
    check_launch("group_compact");
    c->orand.reserve(32 * 8, c->st);
    pra_launch_fill_u64(c->st, c->orand.as<u64>(), 1, 0);
    pra_launch_group_maxlen(c->st, c->tmp64a.as<u64>(), c->tmp64b.as<u64>(), c->tmp64c.as<u64>(), n,
                            c->orand.as<u64>());
    check_launch("group_maxlen");
    HIPCHK(hipMemcpyAsync(c->orand.as<u64>() + 1, c->tmp64b.as<u64>() + n, 8, hipMemcpyDeviceToDevice, c->st));
    u64* hm = readback(c, c->orand.p, 2);
    R->idx_maxlen[v] = hm[0];
    u64 ng = hm[1];
    u64 cap = pow2_at_least(std::max<u64>(64, 2 * ng));
    R->idx[v].reserve(cap * 3 * 8, c->st);
    pra_launch_table_clear(c->st, R->idx[v].as<u64>(), cap, 3);
    pra_launch_index_insert(c->st, r.d(), R->w, R->jcc, c->tmp64c.as<u64>(), ng, R->idx[v].as<u64>(), cap,
                            c->dflags());
    check_launch("index_insert");
    sync_check(c);
    R->idx_cap[v] = cap;
    R->idx_valid[v] = true;
}

// The dictionary words of sorted versions' columns and the first row of each
// leading digit, for emissions in digits, where they are missing.  A version
// stays without (rk_gen) when a value has no rank or there is no room for 8
// bytes a column.  One launch and one wait for all of them.
static void ensure_rank_rows(pra_ctx* c, const std::vector<std::pair<pra_rel*, int>>& versions)
{
    std::vector<std::pair<pra_rel*, int>> made;
    for (auto& rv : versions) {
        pra_rel* R = rv.first;
        const int v = rv.second;
        const Group& G = grp(c, R->group);
        Rows& r = R->ver[v];
        if (R->rk_gen[v] == G.dict_gen || R->rk_no[v] || R->jcc != 1 || !r.sorted || r.n >= (1ULL << 32) ||
            std::find(made.begin(), made.end(), rv) != made.end())
            continue;
        try {
            R->rk_words[v].reserve(r.n * (u64)R->arity * 8, c->st);
            R->rk_first[v].reserve((G.dict_n + 1) * 4, c->st);
        } catch (const PraError& e) {
            if (e.code != PRA_E_BUDGET && e.code != PRA_E_NOMEM) throw;
            R->rk_words[v].release();
            R->rk_no[v] = true;
            continue;
        }
        made.push_back(rv);
    }
    if (made.empty()) return;
    c->orand.reserve(std::max<size_t>(32, made.size()) * 8, c->st);
    pra_launch_fill_u64(c->st, c->orand.as<u64>(), made.size(), 0);
    const size_t n = made.size();
    std::vector<char> table(n * sizeof(RankRowsArgs) + (n + 1) * 4);
    RankRowsArgs* jobs = (RankRowsArgs*)table.data();
    u32* base = (u32*)(jobs + n);
    base[0] = 0;
    for (size_t k = 0; k < n; k++) {
        pra_rel* R = made[k].first;
        const int v = made[k].second;
        const Group& G = grp(c, R->group);
        Rows& r = R->ver[v];
        jobs[k] = RankRowsArgs{r.d(), G.dict.as<u64>(), r.n, G.dict_cap, G.dict_n, R->rk_words[v].as<u64>(),
                               R->rk_first[v].as<u32>(), c->orand.as<u64>() + k, R->w, R->arity, c->nb > 1};
        base[k + 1] = base[k] + (u32)((r.n + PRA_BLOCK - 1) / PRA_BLOCK);
    }
    if (n == 1)
        pra_launch_rank_rows(c->st, jobs[0]);
    else
        pra_launch_rank_rows_many(c->st, (const RankRowsArgs*)stage_table(c, JOB_SETUP, table.data(), table.size()),
                                  (int)n, base[n]);
    check_launch("rank_rows");
    const u64* missing = readback(c, c->orand.p, made.size());
    for (size_t k = 0; k < made.size(); k++) {
        pra_rel* R = made[k].first;
        const int v = made[k].second;
        if (missing[k])
            R->rk_no[v] = true;
        else
            R->rk_gen[v] = grp(c, R->group).dict_gen;
    }
}

// membership table of full u delta keyed on kw leading columns, with room for
// `incoming` more keys at load factor <= 1/2
static void ensure_member_table(pra_ctx* c, pra_rel* R, int kw, u64 incoming)
{
    int stride = 2 + kw;
    if (!R->mt_valid || R->mt_kw != kw) {
        Prof p(c, K_TABLE_BUILD, 8.0 * (R->ver[PRA_FULL].n + R->ver[PRA_DELTA].n) * kw);
        u64 entries = R->ver[PRA_FULL].n + R->ver[PRA_DELTA].n;
        u64 cap = pow2_at_least(std::max<u64>(1024, 2 * (entries + incoming)));
        R->mt.reserve(cap * stride * 8, c->st);
        pra_launch_table_clear(c->st, R->mt.as<u64>(), cap, stride);
        for (int v : {PRA_FULL, PRA_DELTA}) {
            Rows& r = R->ver[v];
            pra_launch_table_insert_rows(c->st, r.d(), r.n, R->w, kw, R->mt.as<u64>(), cap, c->dflags());
            check_launch("table_insert_rows");
        }
        for (int v : {PRA_FULL, PRA_DELTA}) {
            Rows& r = R->ver[v];
            pra_launch_table_verify_rows(c->st, r.d(), r.n, R->w, kw, R->mt.as<u64>(), cap, c->dflags());
            check_launch("table_verify_rows");
        }
        sync_check(c);
        R->mt_cap = cap;
        R->mt_entries = entries;
        R->mt_kw = kw;
        R->mt_valid = true;
        return;
    }
    if (2 * (R->mt_entries + incoming) <= R->mt_cap) return;
    Prof p(c, K_TABLE_BUILD, 8.0 * R->mt_cap * stride);
    // grow 4x while the table is small, 2x beyond 2^28 slots
    u64 cap = pow2_at_least(2 * (R->mt_entries + incoming));
    if (cap < (1ULL << 28)) cap *= 2;
    DBuf nt;
    nt.reserve(cap * stride * 8, c->st);
    pra_launch_table_clear(c->st, nt.as<u64>(), cap, stride);
    pra_launch_table_rehash(c->st, R->mt.as<u64>(), R->mt_cap, nt.as<u64>(), cap, kw, c->dflags());
    check_launch("table_rehash");
    sync_check(c);
    R->mt.swap(nt);
    R->mt_cap = cap;
}

// Dense membership of interned output R keyed on kw columns: the bitmap of
// full u delta for the current dictionary (rebuilt when the dictionary or the
// relation changed since it was built); *bits receives its rank space.  False
// when the output does not allow it: more than 4 key columns, a rank space
// over 2^35 bits, 2^28 or more candidates, or a value of full u delta without
// a rank.
static bool ensure_bitmap(pra_ctx* c, pra_rel* R, int kw, u64 C, u64* bits_out)
{
    Group& G = grp(c, R->group);
    if (!c->dense_on || G.dict_state != 1 || kw < 1 || kw > 4 || G.dict_n == 0 || C >= (1ULL << PRA_DENSE_PBITS))
        return false;
    unsigned __int128 bits = 1;
    for (int i = 0; i < kw; i++) {
        bits *= G.dict_n;
        if (bits > ((unsigned __int128)1 << 35)) return false;
    }
    *bits_out = (u64)bits;
    if (!R->bm_valid || R->bm_gen != G.dict_gen || R->bm_kw != kw) {
        const u64 words = ((u64)bits + 63) / 64;
        Prof p(c, K_TABLE_BUILD, 8.0 * words + 8.0 * kw * (R->ver[PRA_FULL].n + R->ver[PRA_DELTA].n));
        R->bm.reserve((words + 1) / 2 * 16, c->st);   // (one block reads and writes it by 16 bytes)
        pra_launch_fill_u64(c->st, R->bm.as<u64>(), words, 0);
        if (R->ver[PRA_FULL].n + R->ver[PRA_DELTA].n) {
            c->orand.reserve(32 * 8, c->st);
            pra_launch_fill_u64(c->st, c->orand.as<u64>(), 1, 0);
            for (int v : {PRA_FULL, PRA_DELTA}) {
                Rows& r = R->ver[v];
                pra_launch_dense_build(c->st, r.d(), r.n, R->w, kw, G.dict.as<u64>(), G.dict_cap, G.dict_n,
                                       by_bucket(c, R), R->bm.as<u32>(), c->orand.as<u64>());
                check_launch("dense_build");
            }
            if (readback(c, c->orand.p, 1)[0]) {
                R->bm_valid = false;
                return false;
            }
        }
        R->bm_valid = true;
        R->bm_gen = G.dict_gen;
        R->bm_kw = kw;
    }
    return true;
}

// c->first with room for `words` new keys, every word at rest
static void reserve_first(pra_ctx* c, u64 words)
{
    if (c->first_words >= words) return;
    c->first_words = 0;
    c->first.reserve(words * 4, c->st);
    const size_t w64 = c->first.cap / 8;
    pra_launch_fill_u64(c->st, c->first.as<u64>(), w64, ~0ULL);
    c->first_words = 2 * w64;
}

// Ranked membership over a bitmap of `bits` rank indexes, for up to C
// candidates whose words of c->first begin at `base`: the new keys' bitmap
// and its tables, at rest.  grow: c->first may move (no other output of the
// iteration points into it yet).  False when there is no room (the claim
// table needs less).
static bool ensure_ranked(pra_ctx* c, pra_rel* R, u64 bits, u64 base, u64 C, bool grow)
{
    if (!grow && c->first_words < base + C) return false;
    const u64 sbs = (bits + (1ULL << PRA_SB_BITS) - 1) >> PRA_SB_BITS;
    try {
        if (R->fresh_sbs < sbs) {
            R->fresh_sbs = 0;
            const u64 room = (sbs + 1) & ~1ULL;   // whole words of flags
            R->fresh.reserve((room << PRA_SB_BITS) / 8, c->st);
            R->dirty.reserve(room * 4, c->st);
            R->sbpre.reserve(room * 4, c->st);
            R->linep.reserve((room << (PRA_SB_BITS - PRA_LINE_BITS)) * 2, c->st);
            pra_launch_fill_u64(c->st, R->fresh.as<u64>(), (room << PRA_SB_BITS) / 64, 0);
            pra_launch_fill_u64(c->st, R->dirty.as<u64>(), room / 2, 0);
            R->fresh_sbs = room;
        }
        R->sbs_use = sbs;
        reserve_first(c, base + C);
        R->nx.reserve(C * 8, c->st);
        prepare_lookback(c, C);
    } catch (const PraError& e) {
        if (e.code != PRA_E_BUDGET && e.code != PRA_E_NOMEM) throw;
        for (DBuf* b : {&R->fresh, &R->dirty, &R->sbpre, &R->linep}) b->release();
        R->fresh_sbs = 0;
        return false;
    }
    check_launch("ranked");
    return true;
}

// the ranked tables of R back at rest, after claims that stopped at a
// dictionary miss
static void reset_ranked(pra_ctx* c, pra_rel* R)
{
    pra_launch_fill_u64(c->st, R->fresh.as<u64>(), (R->fresh_sbs << PRA_SB_BITS) / 64, 0);
    pra_launch_fill_u64(c->st, R->dirty.as<u64>(), R->fresh_sbs / 2, 0);
    check_launch("reset_ranked");
}

// A claim table of at least 2C slots over a bitmap of `bits` rank indexes.
static void ensure_claims(pra_ctx* c, pra_rel* R, u64 bits, u64 C, u64 slots_per_candidate)
{
    // slots in use: a power of two of at least slots_per_candidate x C; the
    // table is allocated for the largest use so far, and every slot is empty
    // between iterations, so a smaller use is a prefix of it
    const u64 cap = pow2_at_least(std::max<u64>(1024, slots_per_candidate * C));
    // the bits x + 1 <= D^kw needs leave the rest of its 36 bits to an epoch
    // tag (at most 16, or the context's setting): each use of the table takes
    // the next epoch, so the slots of earlier ones count as empty, and the
    // table is filled with zeros only when the epochs wrap
    int kbits = 0;
    while (kbits < 36 && (1ULL << kbits) <= bits) kbits++;
    const int eb = std::min(c->dense_epoch_bits, 36 - kbits);
    bool clear = false;
    if (cap > R->dtab_cap) {
        R->dtab.reserve(cap * 8, c->st);
        R->dtab_cap = cap;
        clear = true;
    }
    if (eb != R->dtab_eb) {
        R->dtab_eb = eb;
        clear = true;
    }
    if (eb > 0 && !clear && R->dtab_epoch + 1 >= (1u << eb)) clear = true;
    if (clear) {
        pra_launch_dense_table_clear(c->st, R->dtab.as<u64>(), R->dtab_cap);
        check_launch("dense_table_clear");
        R->dtab_epoch = 0;
    }
    if (eb > 0) R->dtab_epoch++;
    R->dtab_use = cap;
}

static Group::Seq& seq_counters(pra_ctx* c, int gi, u32 tag)
{
    Group& G = grp(c, gi);
    auto it = G.seq.find(tag);
    if (it != G.seq.end()) return *it->second;
    std::unique_ptr<Group::Seq> q(new Group::Seq());
    q->buf.reserve((size_t)c->nb * 16, c->st);
    pra_launch_fill_u64(c->st, q->buf.as<u64>(), 2 * (u64)c->nb, 0);
    Group::Seq& ref = *q;
    G.seq[tag] = std::move(q);
    return ref;
}

// append src rows (already on device) to a version; with `jobs`, the copy is
// left to the caller's batched copy (the version grows at once)
static void append_rows(pra_ctx* c, pra_rel* R, int v, const u64* src, u64 n, std::vector<CopyJob>* jobs = nullptr)
{
    if (!n) return;
    Rows& r = R->ver[v];
    size_t used = (size_t)r.n * R->w * 8;
    r.buf.reserve(used + (size_t)n * R->w * 8, c->st, used);
    if (jobs)
        jobs->push_back(CopyJob{src, r.d() + r.n * R->w, n * (u64)R->w});
    else
        HIPCHK(hipMemcpyAsync(r.d() + r.n * R->w, src, (size_t)n * R->w * 8, hipMemcpyDeviceToDevice, c->st));
    r.n += n;
    r.sorted = false;
    R->touched(v);
}

// full <- full u delta keeping full sorted, for several relations: both sides
// are sorted by (bucket, columns) and disjoint, so each delta row's place is a
// search inside its bucket and every row moves once, into the relation's other
// full buffer.  A relation whose sides are not both sorted is appended to; one
// without room for a second buffer is merged by itself, through the scratch
// that all share.
struct Merges {
    pra_ctx* c;
    MergeBatch b;
    std::vector<pra_rel*> rels;
    u64 rank_words = 0;
    double bytes = 0;
    explicit Merges(pra_ctx* c_) : c(c_) { memset(&b, 0, sizeof(b)); }
    ~Merges() { c->merges_open = false; }

    void add(pra_rel* R)
    {
        Rows &D = R->ver[PRA_DELTA], &F = R->ver[PRA_FULL];
        if (D.n == 0) return;
        if (F.n == 0 || !F.sorted || !D.sorted) {
            bool sorted = F.n == 0 && D.sorted;
            append_rows(c, R, PRA_FULL, D.d(), D.n);
            F.sorted = sorted;
            return;
        }
        bool own = !c->lean;
        if (own) {
            NoYield hold(c);
            try {
                R->merged.reserve((F.n + D.n) * R->w * 8, c->st);
            } catch (const PraError& e) {
                if (!e.refused()) throw;
                R->merged.release();
                own = false;
            }
        }
        if (own) c->merges_open = true;
        if (!own) run();
        MergeJob& m = b.job[b.njobs];
        m.F = F.d();
        m.nf = F.n;
        m.fbnd = bucket_bounds(c, R, PRA_FULL);
        m.add_to = R->bnd[PRA_FULL].as<u64>();
        m.D = D.d();
        m.nd = D.n;
        m.dbnd = bucket_bounds(c, R, PRA_DELTA);
        m.w = R->w;
        m.rank = (u64*)rank_words;   // its offset until the scratch is sized
        rank_words += D.n;
        if (!own) c->sort_tmp.reserve((F.n + D.n) * R->w * 8, c->st);
        m.out = (own ? R->merged : c->sort_tmp).as<u64>();
        b.rank_base[b.njobs + 1] = b.rank_base[b.njobs] + (u32)((D.n + PRA_BLOCK - 1) / PRA_BLOCK);
        b.scatter_base[b.njobs + 1] = b.scatter_base[b.njobs] + (u32)((F.n + D.n + PRA_BLOCK - 1) / PRA_BLOCK);
        b.njobs++;
        bytes += 16.0 * R->w * (F.n + D.n);
        rels.push_back(R);
        if (!own || b.njobs == PRA_MERGE_JOBS) run(own ? nullptr : &c->sort_tmp);
    }

    // the merges so far; shared: the one job's output, in place of the
    // relation's own second buffer
    void run(DBuf* shared = nullptr)
    {
        if (!b.njobs) return;
        c->tmp64a.reserve(rank_words * 8, c->st);
        for (int k = 0; k < b.njobs; k++) b.job[k].rank = c->tmp64a.as<u64>() + (size_t)b.job[k].rank;
        b.nb = (u64)c->nb;
        {
            Prof p(c, K_MERGE, bytes);
            pra_launch_merge(c->st, b);
            check_launch("merge");
        }
        for (pra_rel* R : rels) {
            Rows& F = R->ver[PRA_FULL];
            F.buf.swap(shared ? *shared : R->merged);
            F.n += R->ver[PRA_DELTA].n;
            F.sorted = true;
            // the merged bucket s holds full's and delta's rows of bucket s
            R->touched(PRA_FULL);
            R->bnd_valid[PRA_FULL] = true;
        }
        rels.clear();
        memset(&b, 0, sizeof(b));
        c->merges_open = false;
        rank_words = 0;
        bytes = 0;
    }
};

// The SCCs of one lock-step iteration seen as one: the rules of every member
// in member order, then rule order, and every member's relations.  Members
// come from different instances of the context and share no relation.
struct RAView {
    std::vector<RADesc*> v;
    RADesc& operator[](size_t i) const { return *v[i]; }
    size_t size() const { return v.size(); }
    struct It {
        RADesc* const* p;
        RADesc& operator*() const { return **p; }
        It& operator++()
        {
            ++p;
            return *this;
        }
        bool operator!=(const It& o) const { return p != o.p; }
    };
    It begin() const { return It{v.data()}; }
    It end() const { return It{v.data() + v.size()}; }
};
struct Merged {
    pra_ctx* ctx = nullptr;
    RAView ras;
    std::vector<pra_rel*> rels;
    explicit Merged(pra_ctx* c, const std::vector<pra_scc*>& members) : ctx(c)
    {
        for (pra_scc* m : members) {
            for (auto& ra : m->ras) ras.v.push_back(&ra);
            rels.insert(rels.end(), m->rels.begin(), m->rels.end());
        }
    }
};

// One threshold round of an output relation: the rules emitting (RA index
// order) and, per listed rule, the outer rows [lo, hi) of every source.
struct RoundSpec {
    std::vector<int> ras;
    std::vector<u64> lo, hi;   // per listed rule, nb each
    DBuf* bounds = nullptr;    // the same on the device: per listed rule lo[nb] then hi[nb]
    u64 nt_base = 0;           // newt rows written by earlier rounds
    u64 cap = 0;               // candidates of this round
};

static u64 read_word(pra_ctx* c, const u64* p) { return readback(c, p, 1)[0]; }

// Where the reference's local_join call over outer rows [start, end) of rule r
// stops (src/RA/parallel_join.cpp:157-230): its outputs are deduplicated per
// call, and the call returns after the first row through which it emitted
// more than the threshold.  Returns that row relative to start, or end-start.
static u64 find_split(pra_ctx* c, Merged* S, int r, u64 start, u64 end, int cw)
{
    RADesc& ra = S->ras[r];
    const int nb = c->nb;
    const u64 n = end - start;
    const u64 base = read_word(c, ra.off.as<u64>() + start);
    const u64 raw = read_word(c, ra.off.as<u64>() + end) - base;
    c->rctl.reserve((size_t)(nb + 4) * 8, c->st);
    u64* tctl = c->rctl.as<u64>();        // [0] candidates, [1] overflow
    u64* tout = tctl + 2;                  // split row
    u64* tposadj = tctl + 4;               // per source: -base
    pra_launch_fill_u64(c->st, tctl, 1, raw);
    pra_launch_fill_u64(c->st, tctl + 1, 1, 0);
    pra_launch_fill_u64(c->st, tposadj, (u64)nb, (u64)0 - base);
    c->cand.reserve(raw * cw * 8, c->st);
    c->dest.reserve(raw * 4, c->st);
    c->slot_of.reserve(raw * 8, c->st);
    c->keep.reserve(raw * 4, c->st);
    {
        JoinExpandArgs a;
        memset(&a, 0, sizeof(a));
        a.ctl = tctl;
        a.outer = ra.outer->ver[ra.outer_v].d() + start * ra.outer->w;
        a.inner = ra.inner->ver[ra.inner_v].d();
        a.off = ra.off.as<u64>() + start;
        a.istart = ra.istart.as<u64>() + start;
        a.posadj = tposadj;
        a.cand = c->cand.as<u64>();
        a.dest = c->dest.as<u32>();
        a.n_outer = n;
        a.nb = (u64)nb;
        a.wo = ra.outer->w;
        a.wi = ra.inner->w;
        a.jcc = ra.in0->jcc;
        a.left = ra.left;
        a.cw = cw;
        a.out_jcc = ra.out->jcc;
        for (int i = 0; i < cw; i++) a.map[i] = ra.map[i];
        pra_launch_join_expand(c->st, a, raw);
        check_launch("split_expand");
    }
    // first occurrences inside the call: a fresh table keyed on whole outputs
    const u64 tcap = pow2_at_least(std::max<u64>(1024, 2 * raw));
    c->ttab.reserve(tcap * (2 + cw) * 8, c->st);
    pra_launch_table_clear(c->st, c->ttab.as<u64>(), tcap, 2 + cw);
    pra_launch_dedup_claim2(c->st, c->cand.as<u64>(), tctl, raw, cw, cw, c->ttab.as<u64>(), tcap,
                            c->slot_of.as<u64>(), 1, c->dflags());
    const u32 nblocks = pra_tiles(raw);
    c->hist.reserve((size_t)nb * nblocks * 4, c->st);
    pra_launch_dedup_decide_hist(c->st, c->cand.as<u64>(), tctl, cw, cw, c->ttab.as<u64>(), c->slot_of.as<u64>(), 1,
                                 c->keep.as<u32>(), c->dest.as<u32>(), (u32)nb, c->hist.as<u32>(), nblocks,
                                 c->dflags());
    check_launch("split_dedup");
    c->kp.reserve((raw + 1) * 4, c->st);
    scan_u32(c, c->keep.as<u32>(), c->kp.as<u32>(), raw, c->kp.as<u32>() + raw);
    pra_launch_find_split(c->st, ra.off.as<u64>() + start, n, c->kp.as<u32>(), c->threshold, tout);
    check_launch("find_split");
    return read_word(c, tout);
}

// The round loop of RAM::execute_in_batches for one output relation whose
// join calls exceed the local-join threshold (src/RAM/RA_tasks.cpp:1121-1269):
// round k emits, per source and rule, the rows from where that call stopped
// in round k-1 to where it stops now; copies and finished calls would only
// re-emit tuples that already arrived, so they emit in the first round only.
// Interning and first-arrival dedup run per round, rounds in order.  Returns
// the new tuples of all rounds.
template <class F>
static u64 run_rounds(Merged* S, pra_rel* R, F&& run_round, u64* st2o_dev)
{
    pra_ctx* c = S->ctx;
    const int nb = c->nb;
    const int cw = R->arity;   // rounds happen for join outputs, which are interned
    struct Call {
        int r;
        std::vector<u64> bst, start;
        std::vector<char> done;
    };
    std::vector<Call> joins;
    std::vector<int> copies;
    for (int r = 0; r < (int)S->ras.size(); r++) {
        RADesc& ra = S->ras[r];
        if (ra.out != R || !ra.active) continue;
        if (ra.type != RA_JOIN) {
            copies.push_back(r);
            continue;
        }
        Call cl;
        cl.r = r;
        u64* hb = readback(c, ra.outer->bnd[ra.outer_v].p, (size_t)nb + 1);
        cl.bst.assign(hb, hb + nb + 1);
        cl.start.assign(cl.bst.begin(), cl.bst.begin() + nb);
        cl.done.resize(nb);
        for (int s = 0; s < nb; s++) cl.done[s] = cl.start[s] == cl.bst[s + 1];
        joins.push_back(std::move(cl));
    }
    DBuf bounds;
    u64 total = 0;
    for (int round = 0;; round++) {
        // (rule, lo, hi) of this round, in rule order
        std::vector<std::tuple<int, std::vector<u64>, std::vector<u64>>> rules;
        u64 cap = 0;
        for (auto& cl : joins) {
            RADesc& ra = S->ras[cl.r];
            std::vector<u64> lo(cl.start), hi(cl.start);
            bool any = false;
            for (int s = 0; s < nb; s++) {
                if (cl.done[s]) continue;
                u64 end = cl.bst[s + 1];
                u64 o0 = read_word(c, ra.off.as<u64>() + cl.start[s]);
                u64 stop = end;
                if ((long long)(read_word(c, ra.off.as<u64>() + end) - o0) > c->threshold)
                    stop = std::min(end, cl.start[s] + find_split(c, S, cl.r, cl.start[s], end, cw) + 1);
                hi[s] = stop;
                cap += read_word(c, ra.off.as<u64>() + stop) - o0;
                any = true;
            }
            if (any) rules.emplace_back(cl.r, lo, hi);
        }
        if (round == 0)
            for (int r : copies) {
                RADesc& ra = S->ras[r];
                u64* hb = readback(c, ra.outer->bnd[ra.outer_v].p, (size_t)nb + 1);
                std::vector<u64> lo(hb, hb + nb), hi(hb + 1, hb + nb + 1);
                cap += read_word(c, ra.off.as<u64>() + ra.n_outer);
                rules.emplace_back(r, lo, hi);
            }
        if (rules.empty()) break;
        std::sort(rules.begin(), rules.end(),
                  [](const auto& a, const auto& b) { return std::get<0>(a) < std::get<0>(b); });
        RoundSpec rs;
        rs.bounds = &bounds;
        rs.nt_base = total;
        rs.cap = cap;
        std::vector<u64> dev;
        for (auto& t : rules) {
            rs.ras.push_back(std::get<0>(t));
            rs.lo.insert(rs.lo.end(), std::get<1>(t).begin(), std::get<1>(t).end());
            rs.hi.insert(rs.hi.end(), std::get<2>(t).begin(), std::get<2>(t).end());
            dev.insert(dev.end(), std::get<1>(t).begin(), std::get<1>(t).end());
            dev.insert(dev.end(), std::get<2>(t).begin(), std::get<2>(t).end());
        }
        bounds.reserve(dev.size() * 8, c->st);
        HIPCHK(hipMemcpyAsync(bounds.p, dev.data(), dev.size() * 8, hipMemcpyHostToDevice, c->st));
        HIPCHK(hipStreamSynchronize(c->st));
        if (cap) {
            run_round(&rs);
            u64 cnt = publish_readback(c, st2o_dev, 8)[0];
            total += cnt;
            R->mt_entries += cnt;
        }
        bool all = true;
        for (auto& cl : joins) {
            for (auto& t : rules)
                if (std::get<0>(t) == cl.r)
                    for (int s = 0; s < nb; s++)
                        if (!cl.done[s]) {
                            cl.start[s] = std::get<2>(t)[s];
                            cl.done[s] = cl.start[s] == cl.bst[s + 1];
                        }
            for (int s = 0; s < nb; s++) all = all && cl.done[s];
        }
        if (all) break;
    }
    return total;
}

// ------------------------------------------------------------ iteration ---

static bool is_intern_type(int type) { return type != RA_ACOPY; }

// One semi-naive iteration (src/RAM/RA_tasks.cpp:1121-1269) of one SCC, or
// of the current SCCs of several instances in lock step: their rules, outputs
// and per-phase launches are taken together, while dedup, intern ids and
// dictionaries stay per instance.
// A join whose inputs have different join column counts matches on input 0's
// count (src/RAM/RA_tasks.cpp:448 passes input0->get_join_column_count() to
// local_join) and reads input 1 through a view keyed on that count.
// local_join probes input 1 in the bucket of the jcc0-column prefix
// (src/RA/parallel_join.cpp:180-186), and a rank holds only the rows of its own
// buckets, so a row of input 1 takes part only when its bucket under its first
// jcc0 columns equals its own bucket; for a RIGHT join it is the outer row
// whose bucket is checked the same way.  The view holds exactly those rows.
// Input 1's version is sorted by (bucket, columns), so the kept rows are in
// the view's order already.
static void refresh_view(pra_ctx* c, pra_rel* V, int v)
{
    pra_rel* src = V->view_of;
    ensure_sorted(c, src, v);
    if (V->view_gen[v] == src->gen[v]) return;
    Rows& S = src->ver[v];
    Rows& D = V->ver[v];
    const u64 n = S.n;
    if (n >= (1ULL << 32)) throw PraError(PRA_E_UNSUPPORTED, "join view of 2^32 rows or more");
    u64 kept = 0;
    if (n) {
        c->keep.reserve(n * 4, c->st);
        c->kp.reserve(n * 4, c->st);
        c->tmp64a.reserve(8, c->st);
        pra_launch_fill_u64(c->st, c->tmp64a.as<u64>(), 1, 0);
        pra_launch_view_keep(c->st, S.d(), n, src->w, V->jcc, src->jcc, (u64)c->nb, c->keep.as<u32>());
        check_launch("view_keep");
        scan_u32(c, c->keep.as<u32>(), c->kp.as<u32>(), n, c->tmp64a.as<u32>());
        kept = readback(c, c->tmp64a.p, 1)[0] & 0xFFFFFFFFULL;
        D.buf.reserve(std::max<u64>(1, kept) * src->w * 8, c->st);
        pra_launch_view_compact(c->st, S.d(), n, src->w, c->keep.as<u32>(), c->kp.as<u32>(), D.d());
        check_launch("view_compact");
    }
    D.n = kept;
    D.sorted = true;
    V->touched(v);
    V->view_gen[v] = src->gen[v];
}

// whether a join's output columns are all data columns of its inputs
static bool projects_data(const RADesc& ra)
{
    for (int m : ra.map) {
        const int first = ra.left ? ra.outer->w : ra.inner->w;
        const int w = m < first ? first : ra.left ? ra.inner->w : ra.outer->w;
        const int col = m < first ? m : ra.in0->jcc + (m - first);
        if (col >= w - 1) return false;
    }
    return true;
}

// the arguments of a join's emission in digits over its whole outer version
static EmitArgs emit_args(pra_ctx* c, const RADesc& rule)
{
    Group& G = grp(c, rule.out->group);
    const bool lead = by_bucket(c, rule.out);
    EmitArgs em;
    memset(&em, 0, sizeof(em));
    em.dx = rule.outer->dx.as<u64>();
    em.n = rule.outer->ver[rule.outer_v].n;
    em.thresh = c->threshold;
    em.joined = G.joined.as<u64>();
    em.first = rule.inner->rk_first[rule.inner_v].as<u32>();
    em.words = rule.inner->rk_words[rule.inner_v].as<u64>();
    em.rank_of = G.rank_of.as<u32>();
    em.lead_of = G.lead_of.as<u32>();
    em.inv = 1.0 / (double)G.dict_n;
    em.kwo = rule.outer->arity;
    em.ia = rule.inner->arity;
    for (int i = 0; i < rule.out->arity; i++) {
        const int m = rule.map[i], first = rule.left ? rule.outer->w : rule.inner->w;
        const bool outer = (m < first) == (rule.left != 0);
        const int col = m < first ? m : rule.in0->jcc + (m - first);
        em.side[i] = outer ? 0 : 1;
        em.col[i] = (signed char)col;
        // outer digits: the first is a leading digit (with several buckets),
        // the others are ranks
        const bool have = outer && c->nb > 1 && col == 0, want = i == 0 && lead;
        em.conv[i] = !outer || have == want ? 0 : have ? 1 : 2;
    }
    return em;
}

// rank spaces that one block's superblock flags cover
static bool loop_space(u64 bits) { return bits <= (u64)PRA_LOOP_SBS << PRA_SB_BITS; }

static void run_iteration(pra_ctx* c, const std::vector<pra_scc*>& members)
{
    for (pra_scc* m : members)
        for (auto& ra : m->ras)
            if (ra.type == RA_JOIN && ra.in1->view_of) refresh_view(c, ra.in1, ra.v1);
    Merged merged(c, members);
    Merged* S = &merged;
    const int nb = c->nb;
    const int nra = (int)S->ras.size();

    // 0. inputs ready: sorted versions, join indexes.  Rules whose outer (or
    //    inner) version is empty emit nothing and launch nothing.
    std::vector<std::pair<pra_rel*, int>> indexed;
    for (auto& ra : S->ras) {
        if (ra.type == RA_JOIN) {
            if (ra.v0 == PRA_DELTA) {
                ra.outer = ra.in0; ra.outer_v = PRA_DELTA; ra.inner = ra.in1; ra.inner_v = ra.v1; ra.left = 1;
            } else {
                ra.outer = ra.in1; ra.outer_v = ra.v1; ra.inner = ra.in0; ra.inner_v = PRA_FULL; ra.left = 0;
            }
            ra.active = ra.outer->ver[ra.outer_v].n > 0 && ra.inner->ver[ra.inner_v].n > 0;
            ra.sorted_probe = ra.inner->scc_changing;
            if (!ra.active) continue;
            ensure_sorted(c, ra.outer, ra.outer_v);
            ensure_sorted(c, ra.inner, ra.inner_v);
            if (ra.sorted_probe)
                bucket_bounds(c, ra.inner, ra.inner_v);
            else if (!ra.inner->idx_valid[ra.inner_v])
                indexed.push_back({ra.inner, ra.inner_v});
        } else {
            ra.outer = ra.in0; ra.outer_v = ra.v0; ra.inner = nullptr; ra.left = 1;
            ra.active = ra.outer->ver[ra.outer_v].n > 0;
            if (ra.active) ensure_sorted(c, ra.outer, ra.outer_v);
        }
    }
    small_indexes(c, indexed);
    for (auto& rv : indexed) ensure_index(c, rv.first, rv.second);
    for (auto& ra : S->ras) ra.n_outer = ra.active ? ra.outer->ver[ra.outer_v].n : 0;

    // 1. output relations, their rule kinds, and candidate capacities: the
    //    previous iteration's count with headroom, else an upper bound from the
    //    outer sizes and the inner index's longest key run.  No host
    //    synchronization: the arrival plan is computed on the device and an
    //    output whose candidates exceed its capacity is re-run.
    std::vector<pra_rel*> outs;
    for (auto& ra : S->ras)
        if (std::find(outs.begin(), outs.end(), ra.out) == outs.end()) outs.push_back(ra.out);
    const size_t no = outs.size();
    std::vector<size_t> out_of((size_t)nra);   // each rule's output
    for (int r = 0; r < nra; r++) out_of[(size_t)r] = std::find(outs.begin(), outs.end(), S->ras[r].out) - outs.begin();
    std::vector<int> out_intern(no, 1);
    std::vector<u64> ub(no, 0), cap(no, 0);
    for (size_t oi = 0; oi < no; oi++) {
        int type0 = -1, nr = 0;
        for (auto& ra : S->ras)
            if (ra.out == outs[oi]) {
                nr++;
                if (type0 < 0) type0 = is_intern_type(ra.type);
                else if (type0 != (int)is_intern_type(ra.type))
                    throw PraError(PRA_E_UNSUPPORTED, "relation is the target of both acopy and join/copy rules");
                if (!ra.active) continue;
                if (ra.type != RA_JOIN)
                    ub[oi] += ra.n_outer;
                else if (ra.sorted_probe)   // no run-length bound without an index: outer x inner
                    ub[oi] += ra.inner->ver[ra.inner_v].n > (~0ULL >> 8) / ra.n_outer
                                  ? (~0ULL >> 8)
                                  : ra.n_outer * ra.inner->ver[ra.inner_v].n;
                else
                    ub[oi] += ra.n_outer * ra.inner->idx_maxlen[ra.inner_v];
            }
        if (nr > PRA_MAXRA) throw PraError(PRA_E_UNSUPPORTED, "too many rules produce one relation");
        out_intern[oi] = type0;
        pra_rel* R = outs[oi];
        cap[oi] = R->jhint ? std::max<u64>(2 * R->jhint, 65536) : std::min<u64>(ub[oi], 1ULL << 22);
        cap[oi] = std::min(cap[oi], ub[oi]);
    }
    for (size_t i = 0; i < no; i++)
        for (size_t j = i + 1; j < no; j++)
            if (out_intern[i] && out_intern[j] && outs[i]->tag == outs[j]->tag && outs[i]->group == outs[j]->group)
                throw PraError(PRA_E_UNSUPPORTED, "two interned relations of one SCC share an intern tag");

    // per output relation: [0] new tuples, [1] packed-key OR, [2] AND, [3] dictionary miss,
    // [4] candidates, [5] capacity overflow, [6] largest top-byte bin of the packed keys,
    // [8..23] key-column OR, [24..39] AND
    const size_t SW = 40;
    c->stage2.reserve(std::max<size_t>(1, no) * SW * 8, c->st);
    c->posadj_dev.reserve((size_t)std::max(1, nra) * nb * 8, c->st);
    for (size_t oi = 0; oi < no; oi++) {
        Group& G = grp(c, outs[oi]->group);
        if (!G.joined.p) {
            G.joined.reserve(8, c->st);
            pra_launch_fill_u64(c->st, G.joined.as<u64>(), 1, 0);
        }
    }
    // packed sort keys need the instance's value dictionary (rebuilt after a
    // miss, given up after repeated misses)
    std::vector<int> stale;
    for (size_t oi = 0; oi < no; oi++) {
        const int gi = outs[oi]->group;
        if (out_intern[oi] && ub[oi] && grp(c, gi).dict_state == 0 &&
            std::find(stale.begin(), stale.end(), gi) == stale.end())
            stale.push_back(gi);
    }
    build_dictionaries(c, stale);
    std::vector<char> packed(no, 0);
    std::vector<u64> pk_mul(no, 0);
    std::vector<int> pk_ls(no, 0);
    for (size_t oi = 0; oi < no; oi++) {
        const Group& G = grp(c, outs[oi]->group);
        packed[oi] = G.dict_state == 1 && out_intern[oi] && ub[oi] &&
                     packed_layout((u64)nb, G.dict_n, outs[oi]->arity, &pk_mul[oi], &pk_ls[oi]);
    }

    // some output of the iteration takes the general membership table
    bool mixed = false;
    for (size_t oi = 0; oi < no; oi++) {
        if (!cap[oi]) continue;
        unsigned __int128 bits = packed[oi] && outs[oi]->arity <= 4 ? 1 : (unsigned __int128)1 << 36;
        for (int i = 0; packed[oi] && i < outs[oi]->arity && bits < ((unsigned __int128)1 << 36); i++)
            bits *= grp(c, outs[oi]->group).dict_n;
        mixed = mixed || bits > ((unsigned __int128)1 << 35);
    }

    size_t nactive = 0;
    for (size_t oi = 0; oi < no; oi++) nactive += cap[oi] ? 1 : 0;
    // per output: its rows (dest, slot_of, keep), candidate words and
    // histogram words in the shared buffers when its claim and decision are
    // batched with other outputs
    struct OutRegion {
        u64 rb = 0, cb = 0, hb = 0;
    };
    std::vector<OutRegion> reg(no);
    u64 region_rows = 0;
    if (nactive >= 2)
        for (size_t oi = 0; oi < no; oi++) {
            reg[oi].rb = region_rows;
            region_rows += cap[oi];
        }

    // dense membership of an output with C candidates of capacity: 0 = the
    // general table, 1 = the claim table, 2 = ranked.  Ranked membership
    // moves each candidate through a few light launches and needs no sort;
    // the claim table needs less memory.  From kTuneMinCandidates candidates
    // of capacity on, single-output iterations time both (the claim table's
    // sizes first) and the band's cheaper one is kept; below that, and
    // untimed, ranked (150x150 grid, 846 K candidates an iteration:
    // membership, new rows and their sort 118 us by the claim table, 88 us
    // ranked).
    struct Choice {
        int mode = 0, dvar = 0;
        bool dtime = false, rtime = false;
    };
    std::vector<char> dense_off(no, 0);   // redone the general way in this iteration
    auto decide = [&](size_t oi, u64 C, int phase, u64 rb) {
        Choice ch;
        pra_rel* R = outs[oi];
        u64 bits = 0;
        if (dense_off[oi] || !packed[oi] || !ensure_bitmap(c, R, R->arity, C, &bits)) return ch;
        ch.mode = 2;
        // (an output that one block can run is not tuned: its iterations
        // would go to the claim table, which that block does not know)
        const bool small = phase == 0 && R->loops && loop_space(bits) && R->jhint <= PRA_LOOP_ROWS &&
                           R->ver[PRA_DELTA].n <= PRA_LOOP_ROWS;
        if (c->tune_on && C >= kTuneMinCandidates && !small) {
            const int band = band_of(C), load = g_tune.settled(c->device, TUNE_DENSE_LOAD, band);
            ch.dvar = std::max(0, load);
            if (phase != 0) {
                // outputs of a batched iteration share their launches and are
                // not timed
            } else if (load < 0) {
                ch.dvar = g_tune.pick(c->device, TUNE_DENSE_LOAD, band, kTuneVariants[TUNE_DENSE_LOAD]);
                ch.dtime = true;
                ch.mode = 1;
            } else {
                ch.mode = 1 + g_tune.pick(c->device, TUNE_RANKED, band, kTuneVariants[TUNE_RANKED]);
                ch.rtime = g_tune.settled(c->device, TUNE_RANKED, band) < 0;
            }
        }
        // next to outputs that take the general table, the claim table
        // shares the partition and sort launches they need anyway: two
        // launches more, where ranked membership is four (points-to
        // analysis, 62 iterations: 15.04 against 15.60 ms)
        if (c->lean > 1 || (phase == 1 && mixed && C < kMixedRankedCandidates)) {
            ch.mode = 1;
            ch.rtime = false;
        }
        if (ch.mode == 2 && !ensure_ranked(c, R, bits, rb, C, phase == 0)) {
            ch.mode = 1;
            ch.rtime = false;
        }
        if (ch.mode == 1) ensure_claims(c, R, bits, C, 2ULL << ch.dvar);
        return ch;
    };
    // the rule of a ranked output that can be emitted in digits (k_rank_emit):
    // its only active one, a join on one column of a delta whose rank indexes
    // are at hand with an inner version that stays as it is, projecting data
    // columns.  A thread walks its row's matches, so joins with a run of more
    // than kEmitRun inner rows take the expansion that balances outputs.
    // -1: none.
    std::vector<char> emit_off(no, 0);
    auto emit_shape = [&](size_t oi) {   // but for the inner rows' ranks

        pra_rel* R = outs[oi];
        if (emit_off[oi] || !bits_in_trie_order(c, R)) return -1;
        int rule = -1;
        for (int r = 0; r < nra; r++)
            if (S->ras[r].active && S->ras[r].out == R) {
                if (rule >= 0) return -1;
                rule = r;
            }
        if (rule < 0) return -1;
        RADesc& ra = S->ras[rule];
        const Group& G = grp(c, R->group);
        if (ra.type != RA_JOIN || ra.sorted_probe || ra.outer_v != PRA_DELTA || ra.outer->dx_gen != G.dict_gen ||
            ra.outer->jcc != 1 || ra.inner->jcc != 1 || ra.outer->arity > 4 || ra.inner->view_of || ra.outer->view_of ||
            ra.inner->idx_maxlen[ra.inner_v] > kEmitRun || ra.n_outer >= (1ULL << 32))
            return -1;
        return projects_data(ra) ? rule : -1;   // no intern id
    };
    auto emit_ranked = [&](size_t oi, int rule) {
        const RADesc& ra = S->ras[rule];
        return ra.inner->rk_gen[ra.inner_v] == grp(c, outs[oi]->group).dict_gen ? rule : -1;
    };
    auto emit_rule_of = [&](size_t oi) {
        const int rule = emit_shape(oi);
        if (rule < 0) return -1;
        ensure_rank_rows(c, {{S->ras[rule].inner, S->ras[rule].inner_v}});
        return emit_ranked(oi, rule);
    };
    // taken per output; the rule an output emits (-1: the general expansions);
    // an emission that stopped left fresh bits that only another would set
    std::vector<Choice> choice(no);
    std::vector<int> emit_rule(no, -1);
    std::vector<char> use_dense(no, 0), fresh_left(no, 0);
    // the bins of an output's packed-key sort
    auto reserve_bins = [&](size_t oi, u64 C) {
        pra_rel* R = outs[oi];
        // bins of twice the average top-byte share (a fuller bin sends
        // the sort to its byte-pass fallback)
        const u32 bcap = (u32)std::min<u64>(PRA_BIN_CAP, pow2_at_least(std::max<u64>(256, 2 * C / 256 + 1)));
        if (bcap > R->bin_cap) {
            R->bin_keys.reserve((size_t)PRA_RADIX * bcap * 8, c->st);
            R->bin_idx.reserve((size_t)PRA_RADIX * bcap * 4, c->st);
            R->bin_cap = bcap;
        }
        if (!R->bin_cur.p) {
            R->bin_cur.reserve(PRA_RADIX * 4, c->st);
            pra_launch_fill_u64(c->st, R->bin_cur.as<u64>(), PRA_RADIX / 2, 0);
        }
        R->nkeys.reserve(C * 8, c->st);
    };
    // Room for what the launches of some outputs write, all of it before the
    // first of them: a refusal here can still be answered without the memory
    // that only speed needs, one between the launches could not.
    auto reserve_outputs = [&](const std::vector<size_t>& ois, const std::vector<Choice>& ch,
                               const std::vector<int>& er) {
        u64 ct = 0, rows = 0, ht = 0, ranked_tiles = 0;
        for (size_t oi : ois) {
            const u64 C = cap[oi];
            const int kw = out_intern[oi] == 1 ? outs[oi]->arity : outs[oi]->arity + 1;
            pra_rel* R = outs[oi];
            R->ver[PRA_NEWT].buf.reserve(C * R->w * 8, c->st);
            rows += C;
            if (er[oi] < 0) ct += C * (u64)kw;
            if (ch[oi].mode == 2) {
                ranked_tiles += pra_tiles(C);
                continue;
            }
            ht += (u64)nb * pra_tiles(C) + 2;
            if (packed[oi]) reserve_bins(oi, C);
            if (ch[oi].mode == 0) R->bm_valid = false, ensure_member_table(c, R, kw, C);
        }
        if (ct || ois.size() > 1) {
            c->cand.reserve(std::max<u64>(ct, 1) * 8, c->st);
            c->dest.reserve(rows * 4, c->st);
        }
        c->slot_of.reserve(rows * 8, c->st);
        c->keep.reserve(rows * 4, c->st);
        c->hist.reserve(ht * 4, c->st);
        c->offs.reserve(ht * 4 + 8, c->st);
        if (ranked_tiles) prepare_lookback(c, ranked_tiles * PRA_TILE);
        std::vector<char> in(no, 0);
        for (size_t oi : ois) in[oi] = er[oi] < 0;
        for (int r = 0; r < nra; r++) {
            RADesc& ra = S->ras[r];
            if (!ra.active || !in[out_of[(size_t)r]]) continue;
            ra.off.reserve((ra.n_outer + 1) * 8, c->st);
            ra.istart.reserve(std::max<u64>(1, ra.n_outer) * 8, c->st);
        }
        // (job tables, counters and bounds, a few KB, have their room below)
        if (c->lean < 2) acct_need(c->st, 64 << 10);
    };
    // f, and while it is refused memory, f again with less to speed it up
    // (nothing that f makes is named by a launch before it returns)
    auto or_lean = [&](bool first_pass, auto f) {
        for (;;) {
            try {
                NoYield hold(c);
                return f();
            } catch (const PraError& e) {
                if (!e.refused() || c->lean > 1) throw;
            }
            yield_tables(c);
            for (pra_rel* R : c->rels) {
                if (first_pass) R->nx.release();   // (else the new rows' indexes)
                if (c->lean < 2) continue;
                R->dx.release();
                R->dx_gen = ~0ULL;
            }
        }
    };
    or_lean(true, [&]() {
        choice.assign(no, Choice());
        emit_rule.assign(no, -1);
        if (nactive >= 2 && c->lean < 2) {
            try {
                reserve_first(c, region_rows);
            } catch (const PraError& e) {
                if (!e.refused()) throw;
            }
        }
        std::vector<std::pair<pra_rel*, int>> to_rank;
        std::vector<size_t> active;
        for (size_t oi = 0; oi < no; oi++) {
            if (!cap[oi]) continue;
            active.push_back(oi);
            choice[oi] = decide(oi, cap[oi], nactive >= 2 ? 1 : 0, reg[oi].rb);
            if (choice[oi].mode != 2) continue;
            emit_rule[oi] = emit_shape(oi);
            if (emit_rule[oi] >= 0) to_rank.push_back({S->ras[emit_rule[oi]].inner, S->ras[emit_rule[oi]].inner_v});
        }
        ensure_rank_rows(c, to_rank);
        for (size_t oi = 0; oi < no; oi++)
            if (emit_rule[oi] >= 0) emit_rule[oi] = emit_ranked(oi, emit_rule[oi]);
        reserve_outputs(active, choice, emit_rule);
    });
    NoYield tables_in_use(c);
    // both variants of the ranked-membership choice are timed from here:
    // emission in digits does the counts' and expansions' work too
    hipEvent_t rank_from = nullptr;
    for (size_t oi = 0; oi < no; oi++)
        if (cap[oi] && choice[oi].rtime) rank_from = c->tune_begin(true);

    // 2. per-RA output counts and their exclusive offsets (the arrival plan
    //    reads them at the source-bucket bounds); an output that emits in
    //    digits counts its rule itself
    c->stage.reserve((size_t)std::max(1, nra) * 2 * nb * 8, c->st);
    CountScanBatch csb;
    memset(&csb, 0, sizeof(csb));
    double cs_bytes = 0;
    auto flush_count_scans = [&]() {
        if (!csb.njobs) return;
        prepare_lookback(c, (u64)csb.tile_base[csb.njobs] * PRA_TILE);
        const u32 ep = next_sort_epoch(c);
        {
            Prof p(c, K_JOIN_COUNT, cs_bytes);
            pra_launch_count_scan_many(c->st, csb, c->lb_status.as<u64>(), c->lb_ctr.as<u32>(), ep, c->dflags());
            check_launch("count_scan_many");
        }
        memset(&csb, 0, sizeof(csb));
        cs_bytes = 0;
    };
    std::vector<char> counted((size_t)nra, 0);
    auto count_rule = [&](int r) {
        RADesc& ra = S->ras[r];
        if (!ra.active || counted[(size_t)r]) return;
        counted[(size_t)r] = 1;
        Rows& O = ra.outer->ver[ra.outer_v];
        u64 n = O.n;
        ra.off.reserve((n + 1) * 8, c->st);
        ra.istart.reserve(std::max<u64>(1, n) * 8, c->st);
        if (n == 0) {
            pra_launch_fill_u64(c->st, ra.off.as<u64>(), 1, 0);
        } else {
            // the counts and their offsets in one pass, batched over rules
            CountScanJob& j = csb.job[csb.njobs];
            memset(&j, 0, sizeof(j));
            j.outer = O.d();
            j.n = n;
            j.wo = ra.outer->w;
            j.off = ra.off.as<u64>();
            const bool join = ra.type == RA_JOIN;
            j.kind = !join ? PRA_CS_FILTER : ra.sorted_probe ? PRA_CS_SORTED : PRA_CS_INDEX;
            if (join) {
                j.inner = ra.inner->ver[ra.inner_v].d();
                j.wi = ra.inner->w;
                j.jcc = ra.in0->jcc;
                j.istart = ra.istart.as<u64>();
                if (ra.sorted_probe) {
                    j.ibnd = ra.inner->bnd[ra.inner_v].as<u64>();
                    j.nb = (u64)nb;
                } else {
                    j.table = ra.inner->idx[ra.inner_v].as<u64>();
                    j.cap = ra.inner->idx_cap[ra.inner_v];
                }
            } else {
                j.op = ra.type == RA_COPY_FILTER ? ra.op : PRA_F_TRUE;
            }
            csb.tile_base[csb.njobs + 1] =
                csb.tile_base[csb.njobs] + (u32)((n + PRA_COUNT_SCAN_TILE - 1) / PRA_COUNT_SCAN_TILE);
            cs_bytes += 8.0 * n * ra.outer->w + (join ? 24.0 : 8.0) * n;
            if (++csb.njobs == PRA_CS_JOBS) flush_count_scans();
        }
        bucket_bounds(c, ra.outer, ra.outer_v);
    };
    for (int r = 0; r < nra; r++)
        if (emit_rule[out_of[(size_t)r]] != r) count_rule(r);
    flush_count_scans();

    // 3+4. per output: arrival plan, emit candidates, deduplicate, partition
    //      and intern, summaries for the sort
    // rs == nullptr: the iteration's whole emission; else one threshold round
    // the last output of the main pass leaves its fold to the publication
    size_t last_oi = no;
    for (size_t oi = 0; oi < no; oi++)
        if (cap[oi]) last_oi = oi;
    NewtFoldArgs last_fold;
    bool have_last_fold = false;
    // batched partitions (unpacked, packed) and the folds that wait for them
    std::vector<NewtScatterArgs> scatter_jobs[2];
    std::vector<size_t> scatter_outs[2];
    std::vector<NewtFoldArgs> later_folds;
    // batched expansions: join (arguments, blocks, per-candidate bytes and
    // output) and copy (arguments, blocks, bytes)
    std::vector<JoinExpandArgs> jexp_jobs;
    std::vector<u32> jexp_blocks;
    std::vector<std::pair<double, size_t>> jexp_per;
    std::vector<CopyExpandArgs> cexp_jobs;
    std::vector<u32> cexp_blocks;
    double cexp_bytes = 0;
    static const int rank_kind[PRA_RANK_STEPS] = {K_RANK_EMIT, K_DEDUP_CLAIM, K_RANK_SCAN, K_RANK_FIRST, K_RANK_PLACE};
    auto rank_bytes = [](int step, int kw) {   // per candidate
        return step == PRA_RANK_EMIT    ? 24.0
               : step == PRA_RANK_CLAIM ? 8.0 * (kw + 1)
               : step == PRA_RANK_FIRST ? 16.0
               : step == PRA_RANK_PLACE ? 8.0 * (kw + 2) + 12.0
                                        : 0.0;
    };
    // an iteration of one ranked output: its placement publishes the summary
    const bool place_publishes = no == 1 && nactive == 1 && choice[0].mode == 2;
    // planned: the arrival plan was made by the iteration's batched plan
    std::vector<ClaimJob> claim_jobs(no);
    std::vector<DecideJob> decide_jobs(no);
    std::vector<ScanJob> scan_jobs;
    std::vector<std::pair<DenseArgs, size_t>> dense_jobs;
    std::vector<std::pair<RankArgs, size_t>> rank_jobs;
    // phase 0: one output start to end; 1: up to its candidates, 2: its
    // histogram scan, 3: from its partition on
    // kept counts on (the claims and decisions in between batched over the
    // outputs, each in its own region of the candidate buffers)
    auto run_output = [&](size_t oi, const RoundSpec* rs, bool planned = false, int phase = 0) {
        const OutRegion rg = phase ? reg[oi] : OutRegion{};
        pra_rel* R = outs[oi];
        const u64 C = rs ? rs->cap : cap[oi];
        const bool pk = packed[oi] && !rs;
        const u64 nt_base = rs ? rs->nt_base : 0;
        const bool intern = out_intern[oi] == 1;
        const int cw = intern ? R->arity : R->arity + 1;
        const int kw = cw;
        Rows& NT = R->ver[PRA_NEWT];
        u64* st2o = c->stage2.as<u64>() + oi * SW;
        u64* ctl = st2o + 4;
        // dense membership: the first pass as decided above, a re-run anew, a
        // threshold round by the general table
        Choice ch;
        if (phase >= 2)
            ch.mode = use_dense[oi];
        else if (planned)
            ch = choice[oi];
        else if (!rs)
            ch = decide(oi, C, 0, 0);
        const int mode = ch.mode, dvar = ch.dvar;
        const bool dtime = ch.dtime;
        const bool dn = mode != 0, ranked = mode == 2;
        use_dense[oi] = (char)mode;
        if (phase >= 2 && ranked) return;   // its new rows are in place
        const int er = !ranked ? -1 : planned ? emit_rule[oi] : emit_rule_of(oi);
        if (phase < 2 && fresh_left[oi]) {
            if (er < 0) reset_ranked(c, R);
            fresh_left[oi] = 0;
        }
        if (!planned && er < 0) {
            for (int r = 0; r < nra; r++)
                if (S->ras[r].out == R) count_rule(r);
            flush_count_scans();
        }
        if (dn)
            R->mt_valid = false;   // the general table is not kept current meanwhile
        else
            R->bm_valid = false, ensure_member_table(c, R, kw, C);
        if (er < 0) {
            c->cand.reserve(C * cw * 8, c->st);
            c->dest.reserve(C * 4, c->st);
        }
        c->slot_of.reserve(C * 8, c->st);
        c->keep.reserve(C * 4, c->st);
        NT.buf.reserve((nt_base + C) * R->w * 8, c->st, nt_base * R->w * 8);
        const u32 nblocks = pra_tiles(C);
        if (!ranked) {
            c->hist.reserve((size_t)nb * nblocks * 4, c->st);
            c->offs.reserve((size_t)nb * nblocks * 4 + 8, c->st);
        }
        u64* cand0 = c->cand.as<u64>() + rg.cb;
        u32* dest0 = c->dest.as<u32>() + rg.rb;
        u64* slot0 = c->slot_of.as<u64>() + rg.rb;
        u32* keep0 = c->keep.as<u32>() + rg.rb;
        u32* hist0 = c->hist.as<u32>() + rg.hb;
        u32* offs0 = c->offs.as<u32>() + rg.hb;
        if (phase < 2) {
            if (!planned && er < 0) {
                PlanArgs pa;
                memset(&pa, 0, sizeof(pa));
                pa.srcoff = c->stage.as<u64>();
                pa.posadj = c->posadj_dev.as<u64>();
                pa.ctl = ctl;
                pa.joined = grp(c, R->group).joined.as<u64>();
                pa.flags = c->dflags();
                pa.cap = C;
                pa.thresh = c->threshold;
                pa.nb = nb;
                pa.rounds_check = rs ? 0 : 1;
                pa.count_joined = rs ? 0 : 1;
                if (rs) {
                    for (size_t k = 0; k < rs->ras.size(); k++) {
                        RADesc& ra = S->ras[rs->ras[k]];
                        pa.ras[pa.nr] = rs->ras[k];
                        pa.is_join[pa.nr] = ra.type == RA_JOIN;
                        pa.off[pa.nr] = ra.off.as<u64>();
                        pa.lo[pa.nr] = rs->bounds->as<u64>() + k * 2 * nb;
                        pa.hi[pa.nr] = rs->bounds->as<u64>() + k * 2 * nb + nb;
                        pa.nr++;
                    }
                } else {
                    for (int r = 0; r < nra; r++) {
                        RADesc& ra = S->ras[r];
                        if (ra.out != R || !ra.active) continue;
                        pa.ras[pa.nr] = r;
                        pa.is_join[pa.nr] = ra.type == RA_JOIN;
                        pa.off[pa.nr] = ra.off.as<u64>();
                        pa.lo[pa.nr] = ra.outer->bnd[ra.outer_v].as<u64>();
                        pa.hi[pa.nr] = ra.outer->bnd[ra.outer_v].as<u64>() + 1;
                        pa.nr++;
                    }
                }
                pra_launch_plan(c->st, pa);
                check_launch("plan");
            }
            for (int r = 0; r < nra; r++) {
                RADesc& ra = S->ras[r];
                if (ra.out != R || !ra.active || er >= 0) continue;
                size_t k = 0;   // position in the round's rule list
                if (rs) {
                    while (k < rs->ras.size() && rs->ras[k] != r) k++;
                    if (k == rs->ras.size()) continue;
                }
                Rows& O = ra.outer->ver[ra.outer_v];
                if (ra.type == RA_JOIN) {
                    // a round emits one window of rows per source; otherwise all rows at once
                    const int nwin = rs ? nb : 1;
                    for (int s = 0; s < nwin; s++) {
                    u64 lo = rs ? rs->lo[k * nb + s] : 0, hi = rs ? rs->hi[k * nb + s] : ra.n_outer;
                    if (hi <= lo) continue;
                    JoinExpandArgs a;
                    memset(&a, 0, sizeof(a));
                    a.ctl = ctl;
                    a.outer = O.d() + lo * ra.outer->w;
                    a.inner = ra.inner->ver[ra.inner_v].d();
                    a.off = ra.off.as<u64>() + lo;
                    a.istart = ra.istart.as<u64>() + lo;
                    a.posadj = c->posadj_dev.as<u64>() + (size_t)r * nb;
                    a.cand = cand0;
                    a.dest = dest0;
                    a.n_outer = hi - lo;
                    a.nb = (u64)nb;
                    a.wo = ra.outer->w;
                    a.wi = ra.inner->w;
                    a.jcc = ra.in0->jcc;
                    a.left = ra.left;
                    a.cw = cw;
                    a.out_jcc = R->jcc;
                    for (int i = 0; i < cw; i++) a.map[i] = ra.map[i];
                    if (phase == 1) {
                        jexp_jobs.push_back(a);
                        jexp_blocks.push_back(pra_join_expand_blocks(std::min<u64>(C, ub[oi])));
                        jexp_per.emplace_back(8.0 * ra.inner->w + 8.0 * cw, oi);
                        continue;
                    }
                    ProfPerCand p(c, K_JOIN_EXPAND, 8.0 * ra.inner->w + 8.0 * cw, oi);
                    pra_launch_join_expand(c->st, a, std::min<u64>(C, ub[oi]));
                    check_launch("join_expand");
                    }
                } else {
                    CopyExpandArgs a;
                    memset(&a, 0, sizeof(a));
                    a.ctl = ctl;
                    a.rows = O.d();
                    a.off = ra.off.as<u64>();
                    a.posadj = c->posadj_dev.as<u64>() + (size_t)r * nb;
                    a.cand = cand0;
                    a.dest = dest0;
                    a.n = ra.n_outer;
                    a.nb = (u64)nb;
                    a.w = ra.outer->w;
                    a.in_jcc = ra.outer->jcc;
                    a.cw = cw;
                    a.out_jcc = R->jcc;
                    for (int i = 0; i < cw; i++) a.map[i] = ra.map[i];
                    if (phase == 1) {
                        if (a.n) {
                            cexp_jobs.push_back(a);
                            cexp_blocks.push_back((u32)((a.n + PRA_BLOCK - 1) / PRA_BLOCK));
                            cexp_bytes += (double)ra.n_outer * 8.0 * (ra.outer->w + cw);
                        }
                        continue;
                    }
                    Prof p(c, K_COPY_EXPAND, (double)ra.n_outer * 8.0 * (ra.outer->w + cw));
                    pra_launch_copy_expand(c->st, a);
                    check_launch("copy_expand");
                }
            }
            if (ranked) {
                RankArgs ra;
                memset(&ra, 0, sizeof(ra));
                Group& G = grp(c, R->group);
                Group::Seq& sq = seq_counters(c, R->group, R->tag);
                const bool lead = by_bucket(c, R);
                ra.cand = cand0;
                ra.ctl = ctl;
                ra.xs = slot0;
                ra.pos = keep0;
                ra.dest = dest0;
                ra.dict = G.dict.as<u64>();
                ra.dict_cap = G.dict_cap;
                ra.D = G.dict_n;
                ra.inv = 1.0 / (double)G.dict_n;
                ra.member = R->bm.as<u32>();
                ra.fresh = R->fresh.as<u32>();
                ra.dirty = R->dirty.as<u32>();
                ra.sbpre = R->sbpre.as<u32>();
                ra.linep = R->linep.as<unsigned short>();
                ra.first = c->first.as<u32>() + rg.rb;
                ra.vals = G.vals.as<u64>();
                ra.lead_vals = (lead ? G.lead_vals : G.vals).as<u64>();
                ra.bucket = G.lead_bucket.as<unsigned char>();
                ra.newt = NT.d();
                if (bits_in_trie_order(c, R)) {
                    R->next_bnd.reserve((size_t)(nb + 1) * 8, c->st);
                    ra.bnd = R->next_bnd.as<u64>();
                    ra.nx = R->nx.as<u64>();
                }
                ra.stat = st2o;
                ra.seq = sq.buf.as<u64>() + sq.now * nb;
                ra.seq_next = sq.buf.as<u64>() + (sq.now ^ 1) * nb;
                ra.sbs = (u32)R->sbs_use;
                ra.chunks = std::min<u32>(PRA_SCAN_CHUNKS, (ra.sbs + 15) / 16);
                ra.nb = (u32)nb;
                ra.tag = R->tag;
                ra.kw = kw;
                ra.wn = R->w;
                ra.by_bucket = lead;
                if (planned && place_publishes) {
                    ra.host = publish_take(c, no * SW, &ra.host_seq);
                    ra.host_words = (u32)(no * SW);
                    ra.err = c->dflags();
                }
                if (er >= 0) {
                    ra.emit = emit_args(c, S->ras[er]);
                    ra.emit.cap = C;
                }
                if (phase == 1) {
                    // launched after the batched expansions
                    rank_jobs.emplace_back(ra, oi);
                    return;
                }
                const u64 etiles = er >= 0 ? (ra.emit.n + PRA_EMIT_BLOCK - 1) / PRA_EMIT_BLOCK : 0;
                prepare_lookback(c, std::max<u64>(C, (etiles + PRA_RADIX - 1) / PRA_RADIX * PRA_TILE));
                for (int step = 0; step < PRA_RANK_STEPS; step++) {
                    if (step == (er >= 0 ? PRA_RANK_CLAIM : PRA_RANK_EMIT)) continue;
                    const u32 ep = next_sort_epoch(c);
                    ProfPerCand p(c, rank_kind[step], rank_bytes(step, kw), oi);
                    pra_launch_rank(c->st, step, ra, C, c->lb_status.as<u64>(), c->lb_ctr.as<u32>(), ep, c->dflags());
                    check_launch("rank");
                }
                if (planned) c->tune_end(rank_from, TUNE_RANKED, band_of(C), 1, oi, C);
                fresh_left[oi] = er >= 0;
                return;
            }
            if (dn) {
                DenseArgs da;
                memset(&da, 0, sizeof(da));
                da.cand = cand0;
                da.ctl = ctl;
                da.slot_of = slot0;
                da.keep = keep0;
                da.dest = dest0;
                da.hist = hist0;
                da.offs1 = nblocks == 1 ? offs0 : nullptr;
                Group& G = grp(c, R->group);
                da.dict = G.dict.as<u64>();
                da.dict_cap = G.dict_cap;
                da.D = G.dict_n;
                da.bitmap = R->bm.as<u32>();
                da.table = R->dtab.as<u64>();
                da.cap = R->dtab_use;
                if (R->dtab_eb > 0) {
                    da.emask = ~0ULL << (64 - R->dtab_eb);
                    da.stamp = (u64)R->dtab_epoch << (64 - R->dtab_eb);
                }
                da.nblocks = nblocks;
                da.nb = (u32)nb;
                da.cw = cw;
                da.kw = kw;
                da.by_bucket = by_bucket(c, R);
                da.rank_of = G.rank_of.as<u32>();
                da.lead = 1;
                for (int i = 1; i < kw; i++) da.lead *= G.dict_n;
                if (phase == 1) {
                    // launched after the batched expansions
                    dense_jobs.emplace_back(da, oi);
                    return;
                }
                hipEvent_t ta = c->tune_begin(dtime);
                {
                    ProfPerCand p(c, K_DEDUP_CLAIM, 8.0 * (kw + 1), oi);
                    pra_launch_dense_claim(c->st, da, C, c->dflags());
                    check_launch("dense_claim");
                }
                {
                    ProfPerCand p(c, K_DEDUP_VERIFY, 16.0, oi);
                    pra_launch_dense_decide(c->st, da, c->dflags());
                    check_launch("dense_decide");
                }
                c->tune_end(ta, TUNE_DENSE_LOAD, band_of(C), dvar, oi, C);
            }
        }
        if (phase < 2 && !dn) {
            u64* tab = R->mt.as<u64>();
            const u64 epoch = ++c->dedup_epoch;
            if (phase == 1) {
                // the batched claim and decision take it from here
                ClaimJob& cj = claim_jobs[oi];
                cj = ClaimJob{cand0, ctl, tab, slot0, R->mt_cap, epoch, cw, kw};
                DecideJob& dj = decide_jobs[oi];
                dj = DecideJob{cand0, ctl, tab, slot0, keep0, dest0, hist0, nblocks == 1 ? offs0 : nullptr, epoch,
                               nblocks, cw, kw};
                return;
            }
            {
                ProfPerCand p(c, K_DEDUP_CLAIM, 8.0 * (kw + 1), oi);
                pra_launch_dedup_claim2(c->st, cand0, ctl, C, cw, kw, tab, R->mt_cap, slot0, epoch, c->dflags());
                check_launch("dedup_claim");
            }
            {
                ProfPerCand p(c, K_DEDUP_VERIFY, 8.0 * kw + 16.0, oi);
                // one tile: the decision writes the offsets itself
                pra_launch_dedup_decide_hist(c->st, cand0, ctl, cw, kw, tab, slot0, epoch, keep0, dest0, (u32)nb, hist0,
                                             nblocks, c->dflags(), nblocks == 1 ? offs0 : nullptr);
                check_launch("dedup_decide_hist");
            }
        }
        u32* total_dev = offs0 + (size_t)nb * nblocks;
        if (phase == 2) {
            // the small histogram scans of a batched iteration go out together
            if (nblocks > 1) {
                if ((u64)nb * nblocks <= PRA_SMALL_SCAN)
                    scan_jobs.push_back(ScanJob{hist0, offs0, total_dev, (u64)nb * nblocks});
                else
                    scan_u32(c, hist0, offs0, (u64)nb * nblocks, total_dev);
            }
            return;
        }
        if (phase == 0 && nblocks > 1) scan_u32(c, hist0, offs0, (u64)nb * nblocks, total_dev);
        Group::Seq* sq = intern ? &seq_counters(c, R->group, R->tag) : nullptr;
        u64* seq_now = sq ? sq->buf.as<u64>() + sq->now * nb : nullptr;
        R->kgofs.reserve(PRA_RADIX * 4, c->st);
        NewtFoldArgs f;   // bin_cur: set with the scatter's bins
        memset(&f, 0, sizeof(f));
        // batched partitions: one summary replica set per output
        u64* rep0 = c->rep_words.as<u64>() + (phase ? oi : 0) * (size_t)PRA_NREP * PRA_PART_WORDS;
        f.rep_words = rep0;
        f.ctl = ctl;
        f.stat = st2o;
        f.kgofs = R->kgofs.as<u32>();
        f.seqbase = seq_now;
        f.offs = offs0;
        f.total = total_dev;
        f.nblocks = nblocks;
        f.nb = (u32)nb;
        f.packed = pk ? 1 : 0;
        f.intern = intern ? 1 : 0;
        // one tile: the scatter's block folds the summaries itself
        const bool fold_here = nblocks == 1;
        bool batched = false;
        {
            NewtScatterArgs a;
            memset(&a, 0, sizeof(a));
            a.ctl = ctl;
            a.cand = cand0;
            a.keep = keep0;
            a.dest = dest0;
            a.offs = offs0;
            a.seqbase = seq_now;
            a.newt = NT.d() + nt_base * R->w;
            a.nblocks = nblocks;
            a.nb = (u32)nb;
            a.cw = cw;
            a.wn = R->w;
            a.intern = intern ? 1 : 0;
            a.tag = R->tag;
            a.rep_words = rep0;
            if (pk) {
                reserve_bins(oi, C);
                a.bin_cap = R->bin_cap;
                a.bin_keys = R->bin_keys.as<u64>();
                a.bin_idx = R->bin_idx.as<u32>();
                a.bin_cur = R->bin_cur.as<u32>();
                f.bin_cur = a.bin_cur;
                Group& G = grp(c, R->group);
                a.dict = G.dict.as<u64>();
                a.dict_cap = G.dict_cap;
                a.keys = R->nkeys.as<u64>();
                a.rank_radix = G.dict_n;
                a.key_lshift = pk_ls[oi];
                if (dn) {
                    // the dense decision leaves each kept candidate's rank
                    // index in its slot_of word
                    u64 scale = 1;
                    for (int i = 0; i < cw; i++) scale *= G.dict_n;
                    a.xk = slot0;
                    a.xk_scale = scale;
                }
            }
            a.fold_here = fold_here ? 1 : 0;
            a.fold = f;
            // column masks only pick the sort passes of outputs too large for
            // the one-block sort, which compares whole key words
            a.summarize = C > PRA_SMALL_SORT;
            if (phase == 3 && nblocks < PRA_SCATTER_WIDE_TILES) {
                // narrow partitions of a batched iteration go out together
                scatter_jobs[pk ? 1 : 0].push_back(a);
                scatter_outs[pk ? 1 : 0].push_back(oi);
                batched = true;
            } else {
                // block width: tuned (timed) on single-output iterations of
                // at least two tiles
                int wide = -1;
                bool stime = false;
                const int sband = band_of(nblocks);
                if (c->tune_on && nblocks >= 2) {
                    if (phase == 0) {
                        wide = g_tune.pick(c->device, TUNE_SCATTER_WIDE, sband, kTuneVariants[TUNE_SCATTER_WIDE]);
                        stime = g_tune.settled(c->device, TUNE_SCATTER_WIDE, sband) < 0;
                    } else {
                        wide = g_tune.settled(c->device, TUNE_SCATTER_WIDE, sband);
                    }
                }
                hipEvent_t ta = c->tune_begin(stime);
                ProfPerCand p(c, K_DEDUP_SCATTER, 8.0 * cw + 8.0, oi);
                pra_launch_dedup_scatter(c->st, a, wide);
                check_launch("dedup_scatter");
                c->tune_end(ta, TUNE_SCATTER_WIDE, sband, wide, oi, C);
                if (planned) c->tune_end(rank_from, TUNE_RANKED, band_of(C), 0, oi, C);
            }
        }
        if (!fold_here && planned && oi == last_oi) {
            // the iteration's last output: folded by the summary's publication
            last_fold = f;
            have_last_fold = true;
        } else if (!fold_here && batched) {
            later_folds.push_back(f);
        } else if (!fold_here) {
            pra_launch_newt_fold(c->st, f);
            check_launch("newt_fold");
        }
    };
    // every output's arrival plan in one launch: its per-rule tables as kernel
    // arguments, or, past their size, from tables in device memory
    const bool plan_all = true;
    if (nra > PRA_MAXRA || no > PRA_MAXRA) {
        std::vector<PlanRule> rules((size_t)nra);
        std::vector<u32> ids;
        std::vector<PlanOut> pouts;
        for (int r = 0; r < nra; r++) {
            RADesc& ra = S->ras[r];
            if (ra.active && counted[(size_t)r])
                rules[(size_t)r] = PlanRule{ra.off.as<u64>(), ra.outer->bnd[ra.outer_v].as<u64>(),
                                            ra.type == RA_JOIN ? 1u : 0u, 0u};
        }
        for (size_t oi = 0; oi < no; oi++) {
            if (!cap[oi] || emit_rule[oi] >= 0) continue;
            PlanOut po{cap[oi], grp(c, outs[oi]->group).joined.as<u64>(), (u32)ids.size(), 0, (u32)oi, 0};
            for (int r = 0; r < nra; r++)
                if (S->ras[r].active && S->ras[r].out == outs[oi]) ids.push_back((u32)r);
            po.count = (u32)ids.size() - po.first;
            pouts.push_back(po);
        }
        const size_t rb = (rules.size() * sizeof(PlanRule) + 255) / 256 * 256;
        const size_t ib = (ids.size() * 4 + 255) / 256 * 256;
        std::vector<char> t(rb + ib + pouts.size() * sizeof(PlanOut));
        memcpy(t.data(), rules.data(), rules.size() * sizeof(PlanRule));
        memcpy(t.data() + rb, ids.data(), ids.size() * 4);
        memcpy(t.data() + rb + ib, pouts.data(), pouts.size() * sizeof(PlanOut));
        const char* d = stage_table(c, JOB_PLAN, t.data(), t.size());
        PlanTabArgs pa{c->stage.as<u64>(), c->posadj_dev.as<u64>(), c->stage2.as<u64>(), c->threshold, nb, (int)SW,
                       (const PlanRule*)d, (const u32*)(d + rb), (const PlanOut*)(d + rb + ib)};
        if (!pouts.empty()) pra_launch_plan_tab(c->st, pa, (int)pouts.size());
        check_launch("plan_tab");
    } else {
        PlanAllArgs pl;
        memset(&pl, 0, sizeof(pl));
        pl.srcoff = c->stage.as<u64>();
        pl.posadj = c->posadj_dev.as<u64>();
        pl.stage2 = c->stage2.as<u64>();
        for (size_t oi = 0; oi < no; oi++) pl.joined[oi] = grp(c, outs[oi]->group).joined.as<u64>();
        pl.thresh = c->threshold;
        pl.nb = nb;
        pl.nra = nra;
        pl.sw = (int)SW;
        int nblk = 0;
        for (size_t oi = 0; oi < no; oi++) {
            pl.cap[oi] = cap[oi];
            if (cap[oi] && emit_rule[oi] < 0) pl.outs[nblk++] = (unsigned char)oi;
        }
        for (int r = 0; r < nra; r++) {
            RADesc& ra = S->ras[r];
            pl.rout[r] = 0xFF;
            if (!ra.active || !counted[(size_t)r]) continue;
            pl.rout[r] = (unsigned char)out_of[(size_t)r];
            pl.is_join[r] = ra.type == RA_JOIN;
            pl.off[r] = ra.off.as<u64>();
            pl.bnd[r] = ra.outer->bnd[ra.outer_v].as<u64>();
        }
        pra_launch_plan_all(c->st, pl, nblk);
        check_launch("plan_all");
    }
    if (plan_all && nactive >= 2) {
        // every output's candidates in its own region; their claims and
        // decisions batched by key width
        u64 ct = 0, ht = 0;
        for (size_t oi = 0; oi < no; oi++) {
            if (!cap[oi]) continue;
            const int cwo = out_intern[oi] == 1 ? outs[oi]->arity : outs[oi]->arity + 1;
            reg[oi].cb = ct;
            reg[oi].hb = ht;
            if (emit_rule[oi] < 0) ct += cap[oi] * (u64)cwo;
            if (choice[oi].mode != 2) ht += (u64)nb * pra_tiles(cap[oi]) + 2;
        }
        c->cand.reserve(std::max<u64>(ct, 1) * 8, c->st);
        c->dest.reserve(region_rows * 4, c->st);
        c->slot_of.reserve(region_rows * 8, c->st);
        c->keep.reserve(region_rows * 4, c->st);
        c->hist.reserve(ht * 4, c->st);
        c->offs.reserve(ht * 4 + 8, c->st);
        for (size_t oi = 0; oi < no; oi++)
            if (cap[oi]) run_output(oi, nullptr, true, 1);
        // the expansions of all rules: job tables through pinned staging into
        // device memory, one launch per kind
        {
            auto table_bytes = [](size_t n, size_t sz) { return n * sz + ((n + 1) * 4 + 255) / 256 * 256; };
            const size_t jb = jexp_jobs.empty() ? 0 : table_bytes(jexp_jobs.size(), sizeof(JoinExpandArgs));
            const size_t cb = cexp_jobs.empty() ? 0 : table_bytes(cexp_jobs.size(), sizeof(CopyExpandArgs));
            if (jb + cb) {
                char* hs = c->job_stage_buf(0, jb + cb);
                c->jobtab[0].reserve(jb + cb, c->st);
                char* dv = c->jobtab[0].as<char>();
                auto put = [&](size_t at, const void* jobs, size_t n, size_t sz, const std::vector<u32>& blocks) {
                    memcpy(hs + at, jobs, n * sz);
                    u32* bb = (u32*)(hs + at + n * sz);
                    bb[0] = 0;
                    for (size_t k = 0; k < n; k++) bb[k + 1] = bb[k] + blocks[k];
                    HIPCHK(hipMemcpyAsync(dv + at, hs + at, table_bytes(n, sz), hipMemcpyHostToDevice, c->st));
                    return bb[n];
                };
                if (jb) {
                    const u32 nbk = put(0, jexp_jobs.data(), jexp_jobs.size(), sizeof(JoinExpandArgs), jexp_blocks);
                    const size_t before = c->pending.size();
                    {
                        Prof p(c, K_JOIN_EXPAND, 0.0);
                        pra_launch_expand_many(c->st, dv, (int)jexp_jobs.size(), nbk, true);
                        check_launch("join_expand_many");
                    }
                    if (c->pending.size() == before + 1)
                        for (auto& pe : jexp_per) c->per_candidate.emplace_back(before, pe.first, pe.second);
                }
                if (cb) {
                    const u32 nbk = put(jb, cexp_jobs.data(), cexp_jobs.size(), sizeof(CopyExpandArgs), cexp_blocks);
                    Prof p(c, K_COPY_EXPAND, cexp_bytes);
                    pra_launch_expand_many(c->st, dv + jb, (int)cexp_jobs.size(), nbk, false);
                    check_launch("copy_expand_many");
                }
            }
        }
        // the ranked outputs: one table through pinned staging, one launch a step
        if (!rank_jobs.empty()) {
            const size_t n = rank_jobs.size();
            std::vector<char> t(n * sizeof(RankArgs) + PRA_RANK_STEPS * (n + 1) * 4);
            RankArgs* J = (RankArgs*)t.data();
            u32* base[PRA_RANK_STEPS];
            for (int q = 0; q < PRA_RANK_STEPS; q++) {
                base[q] = (u32*)(t.data() + n * sizeof(RankArgs)) + q * (n + 1);
                base[q][0] = 0;
            }
            for (size_t k = 0; k < n; k++) {
                const size_t oi = rank_jobs[k].second;
                const u64 C = cap[oi];
                J[k] = rank_jobs[k].first;
                const bool em = emit_rule[oi] >= 0;
                const u32 cb = (u32)((C + PRA_BLOCK - 1) / PRA_BLOCK);
                const u32 blocks[PRA_RANK_STEPS] = {
                    em ? (u32)((J[k].emit.n + PRA_EMIT_BLOCK - 1) / PRA_EMIT_BLOCK) : 0, em ? 0 : cb, J[k].chunks, cb,
                    pra_tiles(C)};
                for (int q = 0; q < PRA_RANK_STEPS; q++) base[q][k + 1] = base[q][k] + blocks[q];
                fresh_left[oi] = em;
            }
            const u64 words = std::max(base[PRA_RANK_EMIT][n], base[PRA_RANK_SCAN][n]);
            prepare_lookback(c, std::max<u64>(base[PRA_RANK_PLACE][n], (words + PRA_RADIX - 1) / PRA_RADIX) * PRA_TILE);
            const RankArgs* d = (const RankArgs*)stage_table(c, JOB_RANK, t.data(), t.size());
            for (int step = 0; step < PRA_RANK_STEPS; step++) {
                if (!base[step][n]) continue;
                const u32 ep = next_sort_epoch(c);
                const size_t before = c->pending.size();
                {
                    Prof p(c, rank_kind[step], 0.0);
                    pra_launch_rank_many(c->st, step, d, (int)n, base[step][n], c->lb_status.as<u64>(),
                                         c->lb_ctr.as<u32>(), ep, c->dflags());
                    check_launch("rank_many");
                }
                if (c->pending.size() == before + 1)
                    for (auto& j : rank_jobs) c->per_candidate.emplace_back(before, rank_bytes(step, j.first.kw), j.second);
            }
        }
        // the dense claims and decisions: one table per key width through
        // pinned staging, one launch each
        if (!dense_jobs.empty()) {
            auto tbytes = [](size_t n) { return (n * sizeof(DenseArgs) + 2 * (n + 1) * 4 + 255) / 256 * 256; };
            size_t total = 0;
            for (int kw = 1; kw <= 4; kw++) {
                size_t n = 0;
                for (auto& dj : dense_jobs) n += dj.first.kw == kw;
                if (n) total += tbytes(n);
            }
            char* hs = c->job_stage_buf(2, total);
            c->jobtab[2].reserve(total, c->st);
            size_t at = 0;
            for (int kw = 1; kw <= 4; kw++) {
                std::vector<size_t> members;
                for (size_t k = 0; k < dense_jobs.size(); k++)
                    if (dense_jobs[k].first.kw == kw) members.push_back(k);
                if (members.empty()) continue;
                const size_t n = members.size();
                DenseArgs* J = (DenseArgs*)(hs + at);
                u32* cb = (u32*)(J + n);
                u32* db = cb + n + 1;
                cb[0] = db[0] = 0;
                for (size_t k = 0; k < n; k++) {
                    const DenseArgs& a = dense_jobs[members[k]].first;
                    const size_t oi = dense_jobs[members[k]].second;
                    J[k] = a;
                    cb[k + 1] = cb[k] + (u32)((cap[oi] + PRA_BLOCK - 1) / PRA_BLOCK);
                    db[k + 1] = db[k] + a.nblocks;
                }
                HIPCHK(hipMemcpyAsync(c->jobtab[2].as<char>() + at, hs + at, tbytes(n), hipMemcpyHostToDevice, c->st));
                const size_t before = c->pending.size();
                {
                    Prof p(c, K_DEDUP_CLAIM, 0.0);
                    pra_launch_dense_many(c->st, (const DenseArgs*)(c->jobtab[2].as<char>() + at), (int)n, kw, cb[n], 0,
                                          c->dflags());
                    check_launch("dense_claim_many");
                }
                if (c->pending.size() == before + 1)
                    for (size_t k : members)
                        c->per_candidate.emplace_back(before, 8.0 * (kw + 1), dense_jobs[k].second);
                const size_t before2 = c->pending.size();
                {
                    Prof p(c, K_DEDUP_VERIFY, 0.0);
                    pra_launch_dense_many(c->st, (const DenseArgs*)(c->jobtab[2].as<char>() + at), (int)n, kw, 0, db[n],
                                          c->dflags());
                    check_launch("dense_decide_many");
                }
                if (c->pending.size() == before2 + 1)
                    for (size_t k : members) c->per_candidate.emplace_back(before2, 16.0, dense_jobs[k].second);
                at += tbytes(n);
            }
        }
        for (int cls = 1; cls <= 7; cls++) {
            ClaimBatch cb;
            DecideBatch db;
            memset(&cb, 0, sizeof(cb));
            memset(&db, 0, sizeof(db));
            db.nb = (u32)nb;
            std::vector<size_t> members;
            auto flush = [&]() {
                if (!cb.njobs) return;
                // timed launches: bytes per candidate of every member output
                size_t before = c->pending.size();
                {
                    Prof p(c, K_DEDUP_CLAIM, 0.0);
                    pra_launch_dedup_claim_many(c->st, cb, cls, c->dflags());
                    check_launch("dedup_claim_many");
                }
                if (c->pending.size() == before + 1)
                    for (size_t oi : members) c->per_candidate.emplace_back(before, 8.0 * (claim_jobs[oi].kw + 1), oi);
                before = c->pending.size();
                {
                    Prof p(c, K_DEDUP_VERIFY, 0.0);
                    pra_launch_dedup_decide_many(c->st, db, cls, c->dflags());
                    check_launch("dedup_decide_many");
                }
                if (c->pending.size() == before + 1)
                    for (size_t oi : members)
                        c->per_candidate.emplace_back(before, 8.0 * decide_jobs[oi].kw + 16.0, oi);
                memset(&cb, 0, sizeof(cb));
                memset(&db, 0, sizeof(db));
                db.nb = (u32)nb;
                members.clear();
            };
            for (size_t oi = 0; oi < no; oi++) {
                if (!cap[oi] || use_dense[oi] || pra_dedup_class(claim_jobs[oi].kw) != cls) continue;
                const int k = cb.njobs;
                cb.job[k] = claim_jobs[oi];
                cb.block_base[k + 1] = cb.block_base[k] + (u32)((cap[oi] + PRA_BLOCK - 1) / PRA_BLOCK);
                cb.njobs++;
                db.job[k] = decide_jobs[oi];
                db.block_base[k + 1] = db.block_base[k] + decide_jobs[oi].nblocks;
                db.njobs++;
                members.push_back(oi);
                if (cb.njobs == PRA_DEDUP_JOBS) flush();
            }
            flush();
        }
        if (c->rep_sets < (int)no) {
            // every set at its identity values (sets at rest always are)
            c->rep_words.reserve(no * (size_t)PRA_NREP * PRA_PART_WORDS * 8, c->st);
            pra_launch_newt_rep_init(c->st, c->rep_words.as<u64>(), (int)no);
            check_launch("newt_rep_init");
            c->rep_sets = (int)no;
        }
        for (size_t oi = 0; oi < no; oi++)
            if (cap[oi]) run_output(oi, nullptr, true, 2);
        if (!scan_jobs.empty()) {
            Prof p(c, K_SCAN, 0.0);
            const char* d = stage_table(c, JOB_SCAN, scan_jobs.data(), scan_jobs.size() * sizeof(ScanJob));
            pra_launch_scan_small_many(c->st, (const ScanJob*)d, (int)scan_jobs.size());
            check_launch("scan_small_many");
        }
        for (size_t oi = 0; oi < no; oi++)
            if (cap[oi]) run_output(oi, nullptr, true, 3);
        // the batched partitions: job tables through pinned staging into
        // device memory, one launch per key kind
        size_t stage_bytes = 0;
        for (int pk = 0; pk < 2; pk++)
            if (!scatter_jobs[pk].empty())
                stage_bytes += scatter_jobs[pk].size() * sizeof(NewtScatterArgs) +
                               ((scatter_jobs[pk].size() + 1) * 4 + 255) / 256 * 256;
        if (stage_bytes) {
            char* hs = c->job_stage_buf(1, stage_bytes);
            c->jobtab[1].reserve(stage_bytes, c->st);
            size_t at = 0;
            for (int pk = 0; pk < 2; pk++) {
                const auto& J = scatter_jobs[pk];
                if (J.empty()) continue;
                const size_t bytes = J.size() * sizeof(NewtScatterArgs) + ((J.size() + 1) * 4 + 255) / 256 * 256;
                memcpy(hs + at, J.data(), J.size() * sizeof(NewtScatterArgs));
                u32* bb = (u32*)(hs + at + J.size() * sizeof(NewtScatterArgs));
                bb[0] = 0;
                for (size_t k = 0; k < J.size(); k++) bb[k + 1] = bb[k] + J[k].nblocks;
                HIPCHK(hipMemcpyAsync(c->jobtab[1].as<char>() + at, hs + at, bytes, hipMemcpyHostToDevice, c->st));
                const size_t before = c->pending.size();
                {
                    Prof p(c, K_DEDUP_SCATTER, 0.0);
                    pra_launch_dedup_scatter_many(c->st, (const NewtScatterArgs*)(c->jobtab[1].as<char>() + at),
                                                  (int)J.size(), bb[J.size()], pk == 1);
                    check_launch("dedup_scatter_many");
                }
                if (c->pending.size() == before + 1)
                    for (size_t k = 0; k < J.size(); k++)
                        c->per_candidate.emplace_back(before, 8.0 * J[k].cw + 8.0, scatter_outs[pk][k]);
                at += bytes;
            }
        }
        if (later_folds.size() == 1) {
            pra_launch_newt_fold(c->st, later_folds[0]);
            check_launch("newt_fold");
        } else if (!later_folds.empty()) {
            const char* d = stage_table(c, JOB_FOLD, later_folds.data(), later_folds.size() * sizeof(NewtFoldArgs));
            pra_launch_newt_fold_many(c->st, (const NewtFoldArgs*)d, (int)later_folds.size());
            check_launch("newt_fold_many");
        }
    } else {
        for (size_t oi = 0; oi < no; oi++)
            if (cap[oi]) run_output(oi, nullptr, plan_all);
    }

    // 5. new-tuple counts, sort-key summaries and error flags: the
    //    per-iteration host readback (repeated once for outputs whose
    //    candidates overflowed their capacity, now sized exactly)
    std::vector<u64> st2(no * SW, 0);
    // deltas of relations whose full version no rule of the SCC reads go to
    // their full logs while the host waits for the first readback
    std::vector<char> early(S->rels.size(), 0), redone(no, 0);
    // pass 1 redoes outputs whose candidates overflowed their capacity (now
    // sized exactly) or whose dense claims met a value without a dictionary
    // rank (now the general way); pass 2 the few that needed both
    tables_in_use.end();
    for (int pass = 0; pass < 3; pass++) {
        u64* h = publish_begin(c, c->stage2.as<u64>(), no * SW, pass == 0 && have_last_fold ? &last_fold : nullptr,
                               pass == 0 && place_publishes);
        if (pass == 0) {
            std::vector<CopyJob> appends;
            for (size_t i = 0; i < S->rels.size(); i++) {
                pra_rel* R = S->rels[i];
                if (R->full_read || R->merge_full || !R->ver[PRA_DELTA].n) continue;
                append_rows(c, R, PRA_FULL, R->ver[PRA_DELTA].d(), R->ver[PRA_DELTA].n, &appends);
                early[i] = 1;
            }
            copy_ranges(c, (c->early_parity ^= 1) ? JOB_EARLY_APPEND2 : JOB_EARLY_APPEND, appends);
        }
        h = publish_wait(c, h, no * SW);
        std::vector<size_t> redo;
        for (size_t oi = 0; oi < no; oi++) {
            if (!cap[oi]) continue;
            std::copy(h + oi * SW, h + (oi + 1) * SW, st2.begin() + oi * SW);
            const u64 state = st2[oi * SW + 5];
            if (state == 1 || state == 3 || state == 4) redo.push_back(oi);
            if (state == 0) fresh_left[oi] = 0;
        }
        if (redo.empty()) break;
        if (pass == 2) throw PraError(PRA_E_HIP, "candidate capacity overflow after resizing");
        for (size_t oi : redo) {
            if (st2[oi * SW + 5] == 3) {
                // claims that stopped at the miss left slots behind
                pra_rel* R = outs[oi];
                if (use_dense[oi] == 2) {
                    reset_ranked(c, R);
                } else {
                    pra_launch_dense_table_clear(c->st, R->dtab.as<u64>(), R->dtab_cap);
                    check_launch("dense_table_clear");
                }
                dense_off[oi] = 1;
            }
            // an emission over the join threshold: by the arrival plan
            if (st2[oi * SW + 5] == 4) emit_off[oi] = 1;
            cap[oi] = st2[oi * SW + 4];
            redone[oi] = 1;
            or_lean(false, [&]() {
                std::vector<Choice> ch(no);
                std::vector<int> er(no, -1);
                ch[oi] = decide(oi, cap[oi], 0, 0);
                if (ch[oi].mode == 2) er[oi] = emit_rule_of(oi);
                reserve_outputs({oi}, ch, er);
            });
            NoYield in_use(c);
            run_output(oi, nullptr);
        }
    }
    // outputs with a join call over the local-join threshold: emitted in
    // rounds (src/RAM/RA_tasks.cpp:1121-1269, src/RA/parallel_join.cpp:157-230)
    std::vector<char> in_rounds(no, 0);
    for (size_t oi = 0; oi < no; oi++)
        if (cap[oi] && st2[oi * SW + 5] == 2) {
            st2[oi * SW] = run_rounds(S, outs[oi], [&](const RoundSpec* rs) { run_output(oi, rs); },
                                      c->stage2.as<u64>() + oi * SW);
            st2[oi * SW + 5] = 0;
            in_rounds[oi] = 1;
        }
    for (auto& pc : c->per_candidate)
        if (std::get<0>(pc) < c->pending.size())
            c->pending[std::get<0>(pc)].bytes += std::get<1>(pc) * (double)st2[std::get<2>(pc) * SW + 4];
    c->per_candidate.clear();
    // tuned launches: cost per candidate, read at the next iteration (the
    // launches may still be running); one whose candidates passed its capacity
    // did part of the work and is not counted
    std::vector<pra_ctx::LateSample> samples;
    samples.swap(c->tune_late);
    for (auto& l : samples) {
        const auto& t = l.s;
        float ms = 0, sort_ms = 0;
        hipError_t e = l.sorts && !l.sort_b ? hipErrorInvalidValue : hipEventElapsedTime(&ms, t.a, t.b);
        if (e == hipSuccess && l.sorts) e = hipEventElapsedTime(&sort_ms, l.sort_a, l.sort_b);
        if (e == hipErrorNotReady) {
            c->tune_late.push_back(l);
            continue;
        }
        if (e == hipSuccess && g_tune.record(c->device, t.knob, t.band, t.var, (double)(ms + sort_ms) / (double)t.cap,
                                             kTuneVariants[t.knob]))
            tune_save();
        for (hipEvent_t x : {t.a, t.b, l.sort_a, l.sort_b})
            if (x) c->evpool.push_back(x);
    }
    const size_t waiting = c->tune_late.size();   // samples of earlier iterations
    for (auto& t : c->tune_pending) {
        const u64 n = st2[t.oi * SW + 4];
        if (n > 0 && n <= t.cap && !in_rounds[t.oi] && !redone[t.oi]) {
            t.cap = n;
            c->tune_late.push_back({t, t.knob == TUNE_RANKED && t.var == 0, nullptr, nullptr});
        } else {
            c->evpool.push_back(t.a);
            c->evpool.push_back(t.b);
        }
    }
    c->tune_pending.clear();
    for (size_t oi = 0; oi < no; oi++) {
        pra_rel* R = outs[oi];
        u64 cnt = cap[oi] ? st2[oi * SW] : 0;
        R->jhint = cap[oi] ? st2[oi * SW + 4] : 0;
        R->ver[PRA_NEWT].n = cnt;
        R->ver[PRA_NEWT].sorted = false;
        // the counters a ranked iteration advanced are the current ones now
        if (cap[oi] && use_dense[oi] == 2 && !in_rounds[oi]) seq_counters(c, R->group, R->tag).now ^= 1;
        if (!in_rounds[oi]) R->mt_entries += cnt;   // rounds count their own
    }

    // 6. delta -> full, sort newt into trie order, newt -> delta
    //    (src/RAM/RA_tasks.cpp:1044-1058).  The old delta is folded into full
    //    first: the newt sort writes the next delta's bucket bounds.
    {
        std::vector<CopyJob> appends;
        Merges merges(c);
        for (size_t i = 0; i < S->rels.size(); i++) {
            pra_rel* R = S->rels[i];
            Rows& D = R->ver[PRA_DELTA];
            if (R->merge_full)
                merges.add(R);
            else if (!early[i])
                append_rows(c, R, PRA_FULL, D.d(), D.n, &appends);
        }
        merges.run();
        copy_ranges(c, JOB_APPEND, appends);
        for (pra_rel* R : S->rels) {
            R->ver[PRA_DELTA].n = 0;
            R->touched(PRA_DELTA);
        }
    }
    std::vector<char> bnd_ok(no, 0);
    // one-block sorts of all outputs go out together, into the emptied delta
    // buffers (swapped back with newt's below)
    SmallSortBatch ssb;
    memset(&ssb, 0, sizeof(ssb));
    ssb.nb = (u64)nb;
    std::vector<size_t> ss_out;
    // several outputs sorting by packed key: their bin sorts go out as one
    // launch, each into its emptied delta buffer; one sorts at once
    std::vector<BinSortJob> bin_jobs;
    std::vector<size_t> bin_out;
    u64 bins_max = 0;   // the largest bin of the deferred bin sorts
    size_t n_packed_sorts = 0;
    // outputs whose new rows are in place already
    auto placed = [&](size_t oi) { return cap[oi] && use_dense[oi] == 2 && !in_rounds[oi]; };
    for (size_t oi = 0; oi < no; oi++)
        n_packed_sorts += packed[oi] && !placed(oi) && !in_rounds[oi] && st2[oi * SW + 3] == 0;
    auto flush_small_sorts = [&]() {
        if (ss_out.empty()) return;
        double bytes = 0;
        for (size_t k = 0; k < ss_out.size(); k++) {
            const SmallSortJob& j = ssb.job[k];
            bytes += 8.0 * j.n * (j.kc + j.bucketed) + 16.0 * j.n * j.w;
        }
        {
            Prof p(c, K_SMALL_SORT, bytes);
            pra_launch_small_sort_many(c->st, ssb, (int)ss_out.size());
            check_launch("small_sort_many");
        }
        for (size_t oi2 : ss_out) outs[oi2]->ver[PRA_NEWT].buf.swap(outs[oi2]->ver[PRA_DELTA].buf);
        ss_out.clear();
    };
    for (size_t oi = 0; oi < no; oi++) {
        pra_rel* R = outs[oi];
        Rows& NT = R->ver[PRA_NEWT];
        R->bnd[PRA_DELTA].reserve((size_t)(nb + 1) * 8, c->st);
        u64* bnd = R->bnd[PRA_DELTA].as<u64>();
        if (placed(oi)) {
            if (bits_in_trie_order(c, R)) {
                R->bnd[PRA_DELTA].swap(R->next_bnd);
            } else {
                c->sort_tmp.reserve(NT.n * R->w * 8, c->st);
                bucket_rows(c, NT.d(), NT.n, R->w, R->jcc, c->sort_tmp.as<u64>(), bnd);
                NT.buf.swap(c->sort_tmp);
            }
            bnd_ok[oi] = 1;
            continue;
        }
        if (packed[oi] && !in_rounds[oi] && st2[oi * SW + 3] == 0) {
            BinSortJob job;
            auto late = std::find_if(c->tune_late.begin() + (long)waiting, c->tune_late.end(),
                                     [&](const pra_ctx::LateSample& l) { return l.sorts && l.s.oi == oi; });
            if (late != c->tune_late.end()) late->sort_a = c->tune_begin(true);
            if (sort_by_packed_key(c, R, st2[oi * SW + 1], st2[oi * SW + 2], st2[oi * SW + 6], pk_mul[oi], pk_ls[oi],
                                   bnd, n_packed_sorts > 1 ? &job : nullptr, &R->ver[PRA_DELTA].buf)) {
                bin_jobs.push_back(job);
                bin_out.push_back(oi);
                bins_max = std::max<u64>(bins_max, st2[oi * SW + 6]);
            }
            if (late != c->tune_late.end()) late->sort_b = c->tune_begin(true);
            bnd_ok[oi] = 1;
            continue;
        }
        // packed mode collects no column masks (a dictionary miss sorts every
        // digit), and a round's masks cover that round only
        const u64* masks = (packed[oi] || in_rounds[oi]) ? nullptr : &st2[oi * SW + 8];
        Group& G = grp(c, R->group);
        if (packed[oi] && !in_rounds[oi] && G.dict_state == 1) G.dict_state = ++G.dict_rebuilds > 3 ? 2 : 0;
        SmallSortJob job;
        bnd_ok[oi] = sort_rows_masked(c, NT, R->w, R->jcc, out_intern[oi] ? R->arity : R->w, masks, bnd, true, &job,
                                      &R->ver[PRA_DELTA].buf, &G);
        if (job.n) {
            ssb.job[ss_out.size()] = job;
            ss_out.push_back(oi);
            if (ss_out.size() == PRA_SORT_JOBS) flush_small_sorts();
        }
        if (!bnd_ok[oi] && nb == 1) {
            pra_launch_fill_u64(c->st, bnd, 1, 0);
            pra_launch_fill_u64(c->st, bnd + 1, 1, NT.n);
            bnd_ok[oi] = 1;
        }
    }
    flush_small_sorts();
    // the bin sorts of all packed outputs, into the emptied delta buffers
    if (!bin_jobs.empty()) {
        double bytes = 0;
        for (const BinSortJob& j : bin_jobs) bytes += 12.0 * j.n + 16.0 * j.n * j.w;
        Prof p(c, K_BIN_SORT, bytes);
        if (bin_jobs.size() == 1) {
            const BinSortJob& j = bin_jobs[0];
            pra_launch_bin_sort(c->st, j.bin_keys, j.bin_idx, j.bin_cap, j.n, j.bofs, j.bytes, j.rows, j.w, j.out,
                                j.bmul, j.ls, j.nb, j.bnd, c->dflags(), bins_max);
        } else {
            const char* d = stage_table(c, JOB_SORT, bin_jobs.data(), bin_jobs.size() * sizeof(BinSortJob));
            pra_launch_bin_sort_many(c->st, (const BinSortJob*)d, (int)bin_jobs.size(), c->dflags(), bins_max);
        }
        check_launch("bin_sort");
        for (size_t oi2 : bin_out) outs[oi2]->ver[PRA_NEWT].buf.swap(outs[oi2]->ver[PRA_DELTA].buf);
    }
    for (pra_rel* R : S->rels) {
        Rows& D = R->ver[PRA_DELTA];
        D.buf.swap(R->ver[PRA_NEWT].buf);
        D.n = R->ver[PRA_NEWT].n;
        D.sorted = true;
        R->ver[PRA_NEWT].n = 0;
        R->touched(PRA_DELTA);
        auto it = std::find(outs.begin(), outs.end(), R);
        if (it == outs.end()) continue;
        if (bnd_ok[it - outs.begin()]) R->bnd_valid[PRA_DELTA] = true;
        if (placed((size_t)(it - outs.begin())) && bits_in_trie_order(c, R)) {
            R->dx.swap(R->nx);
            R->dx_gen = grp(c, R->group).dict_gen;
        }
    }
    for (pra_scc* m : members) grp(c, m->group).iterations++;
}

static u64 delta_sum(pra_scc* S)
{
    u64 d = 0;
    for (pra_rel* R : S->rels) d += R->ver[PRA_DELTA].n;
    return d;
}

// ------------------------------------------- whole iterations in a block ---

// The rule of an SCC whose iterations one block can run (k_rank_loop), by its
// shape: its only rule, a join on one column of its own output's delta with
// the full version of a relation that stays as it is, projecting data
// columns, into an output whose full version is a log.  Null: none.
static RADesc* loop_rule(pra_scc* S)
{
    if (!S->fixpoint || S->ras.size() != 1) return nullptr;
    RADesc& ra = S->ras[0];
    if (ra.type != RA_JOIN) return nullptr;
    ra.left = ra.v0 == PRA_DELTA;
    ra.outer = ra.left ? ra.in0 : ra.in1;
    ra.inner = ra.left ? ra.in1 : ra.in0;
    ra.outer_v = ra.left ? ra.v0 : ra.v1;
    ra.inner_v = ra.left ? ra.v1 : ra.v0;
    if (ra.outer != ra.out || ra.outer_v != PRA_DELTA || ra.inner == ra.out || ra.inner_v != PRA_FULL ||
        ra.inner->view_of || ra.outer->jcc != 1 || ra.inner->jcc != 1 || ra.out->arity > 4 || ra.out->full_read ||
        ra.out->merge_full || !projects_data(ra))
        return nullptr;
    return &ra;
}

// Whether S's next iterations can be run by one block now: the output ranked,
// its delta's rank indexes at hand and small, and every table in place (the
// general iterations before have made them).
static bool loop_ready(pra_ctx* c, pra_scc* S, u32 max_cand)
{
    if (!c->loop_on || c->lean || !S->running || S->ras.size() != 1 || !S->ras[0].out->loops) return false;
    RADesc* ra = loop_rule(S);
    if (!ra) return false;
    pra_rel* R = ra->out;
    Group& G = grp(c, R->group);
    const u64 n = R->ver[PRA_DELTA].n;
    if (!n || n > max_cand || R->jhint > max_cand || n >= S->loop_stop) return false;
    if (c->nb > 1 && G.dict_n > PRA_LOOP_LEADS) return false;
    if (G.dict_state != 1 || R->dx_gen != G.dict_gen || !R->bm_valid || R->bm_gen != G.dict_gen ||
        R->bm_kw != R->arity || !G.joined.p)
        return false;
    u64 bits = 1;
    for (int i = 0; i < R->arity; i++) {
        bits *= G.dict_n;
        if (!loop_space(bits)) return false;
    }
    if (R->sbs_use != (bits + (1ULL << PRA_SB_BITS) - 1) >> PRA_SB_BITS || R->fresh_sbs < R->sbs_use) return false;
    if (!ra->inner->idx_valid[PRA_FULL] || ra->inner->idx_maxlen[PRA_FULL] > kEmitRun || !ra->inner->ver[PRA_FULL].n ||
        ra->inner->ver[PRA_FULL].n >= (1ULL << PRA_LOOP_RUN_SHIFT))
        return false;
    for (pra_rel* o : S->rels)
        if (o != R && o->ver[PRA_DELTA].n) return false;
    return ra->inner->rk_gen[PRA_FULL] == G.dict_gen;
}

// Up to `max` iterations of each of some SCCs that are ready for it, a block
// each, in one launch; rows[k] receives the new rows of each iteration that
// SCC k made (none: the general iteration takes its next one).
// The full log takes the delta first and the new rows behind it, in place; the
// last iteration's are copied out as the delta again.
static void run_loops(pra_ctx* c, const std::vector<pra_scc*>& sccs, u32 max, u32 max_cand,
                      std::vector<std::vector<u32>>& rows)
{
    NoYield hold(c);
    std::vector<LoopArgs> jobs;
    std::vector<size_t> of;
    std::vector<CopyJob> appends;
    for (size_t k = 0; k < sccs.size(); k++) {
        RADesc& ra = *loop_rule(sccs[k]);
        pra_rel* R = ra.out;
        Group& G = grp(c, R->group);
        Rows &F = R->ver[PRA_FULL], &D = R->ver[PRA_DELTA], &N = R->ver[PRA_NEWT];
        LoopArgs a;
        memset(&a, 0, sizeof(a));
        // room for what the rank space can still hold, or as much again as
        // there is, as the appends' growth would make; an iteration stops by
        // its candidates, so their most on top.  Under a budget the room that
        // the general iterations have left in the log and newt, and as
        // many candidates: what they hold is never larger than they make it.
        u64 bits = 1;
        for (int i = 0; i < R->arity; i++) bits *= G.dict_n;
        const u64 have = F.n + D.n;
        const u64 more = c->budget ? 0 : std::min<u64>(bits - std::min(bits, have), std::max<u64>(1 << 18, have)) + PRA_LOOP_ROWS;
        try {
            F.buf.reserve((have + more) * R->w * 8, c->st, (size_t)F.n * R->w * 8);
            a.room = F.buf.cap / ((size_t)R->w * 8) - have;
            if (a.room < R->jhint) continue;   // not for another iteration like the last
            R->places.reserve((R->sbs_use << (PRA_SB_BITS - 5)) * 8, c->st);
            // the delta that an iteration may leave (new keys of its candidates),
            // in newt's buffer, which is empty
            const u64 left = std::min<u64>(bits - std::min(bits, have), max_cand);
            if (!c->budget) {
                R->dx.reserve(left * 8, c->st, D.n * 8);
                N.buf.reserve(left * R->w * 8, c->st);
            }
            a.max_cand = (u32)std::min<u64>(max_cand, std::min(R->dx.cap, N.buf.cap / (size_t)R->w) / 8);
            if (left <= a.max_cand) a.max_cand = max_cand;
        } catch (const PraError& e) {
            if (e.code != PRA_E_BUDGET && e.code != PRA_E_NOMEM) throw;
            R->places.release();
            sccs[k]->loop_stop = 0;   // the general launches from here on
            continue;
        }
        appends.push_back(CopyJob{D.d(), F.d() + F.n * R->w, D.n * (u64)R->w});
        a.emit = emit_args(c, ra);
        a.vals = G.vals.as<u64>();
        a.lead_vals = (by_bucket(c, R) ? G.lead_vals : G.vals).as<u64>();
        a.bucket = G.lead_bucket.as<unsigned char>();
        a.member = R->bm.as<u32>();
        a.fresh = R->fresh.as<u32>();
        a.places = R->places.as<u64>();
        a.rows = F.d() + have * R->w;
        Group::Seq& sq = seq_counters(c, R->group, R->tag);
        a.seq = sq.buf.as<u64>() + sq.now * c->nb;
        a.D = G.dict_n;
        a.sbs = (u32)R->sbs_use;
        a.nb = (u32)c->nb;
        a.tag = R->tag;
        a.max_iters = std::min<u32>(max, PRA_LOOP_ITERS);
        a.kw = R->arity;
        a.wn = R->w;
        a.by_bucket = by_bucket(c, R);
        jobs.push_back(a);
        of.push_back(k);
    }
    if (jobs.empty()) return;
    // from the launch on nothing is allocated, so nothing can be refused
    // between the rows that it writes and the counts that take them in
    try {
        c->tmp64a.reserve(jobs.size() * PRA_LOOP_OUT * 8, c->st);
        if (jobs.size() > 1 || c->pub_open)
            for (int slot : {JOB_LOOP_FULL, JOB_LOOP_DELTA, JOB_LOOP})
                reserve_table(c, slot, jobs.size() * std::max(sizeof(LoopArgs), sizeof(CopyJob) + 4) + 4);
    } catch (const PraError& e) {
        if (e.code != PRA_E_BUDGET && e.code != PRA_E_NOMEM) throw;
        for (pra_scc* S : sccs) S->loop_stop = 0;
        return;
    }
    copy_ranges(c, JOB_LOOP_FULL, appends);
    for (size_t k = 0; k < jobs.size(); k++) jobs[k].out = c->tmp64a.as<u64>() + k * PRA_LOOP_OUT;
    const u64* out;
    if (jobs.size() == 1 && !c->pub_open) {
        LoopArgs& a = jobs[0];
        a.host = publish_take(c, PRA_LOOP_OUT, &a.host_seq);
        a.host_words = PRA_LOOP_OUT;
        a.err = c->dflags();
        {
            Prof p(c, K_RANK_LOOP, 0.0);
            pra_launch_rank_loop(c->st, a);
            check_launch("rank_loop");
        }
        out = publish_wait(c, publish_begin(c, nullptr, PRA_LOOP_OUT, nullptr, true), PRA_LOOP_OUT);
    } else {
        const char* d = stage_table(c, JOB_LOOP, jobs.data(), jobs.size() * sizeof(LoopArgs));
        {
            Prof p(c, K_RANK_LOOP, 0.0);
            pra_launch_rank_loop_many(c->st, (const LoopArgs*)d, (int)jobs.size());
            check_launch("rank_loop_many");
        }
        out = readback(c, c->tmp64a.p, jobs.size() * PRA_LOOP_OUT);
    }
    std::vector<CopyJob> deltas;
    for (size_t j = 0; j < jobs.size(); j++, out += PRA_LOOP_OUT) {
        pra_scc* S = sccs[of[j]];
        pra_rel* R = S->ras[0].out;
        Group& G = grp(c, R->group);
        Rows &F = R->ver[PRA_FULL], &D = R->ver[PRA_DELTA];
        const u64 its = out[0], written = out[1], last = out[2];
        if (out[3] >> 32) S->loop_stop = last;   // too many candidates for one block from this delta
        if (!its) continue;
        const u32* h = (const u32*)(out + 4);
        rows[of[j]].assign(h, h + its);
        F.n += D.n + written - last;
        F.sorted = false;
        R->touched(PRA_FULL);
        D.n = last;
        D.sorted = true;
        R->touched(PRA_DELTA);
        R->dx_gen = G.dict_gen;
        D.buf.swap(R->ver[PRA_NEWT].buf);
        if (last) deltas.push_back(CopyJob{F.d() + F.n * R->w, D.d(), last * (u64)R->w});
        R->jhint = (u32)out[3];
        R->mt_entries += written;
        G.iterations += its;
    }
    copy_ranges(c, JOB_LOOP_DELTA, deltas);
}

// The next iterations of some SCCs: all of them make up to `max` by one block
// each when all are ready for that, else one together.  rows[k]: the new rows
// of each iteration of SCC k (of the general one: its delta after it).
// One block takes about 3 us and 3 us per 1,024 candidates an iteration, the
// general launches 45 us for one SCC and 100 us for sixty.  So a few SCCs give
// an iteration of more than 8,192 candidates to the general launches, four and
// more only one of more than 16,384.  Transitive closure of random graphs,
// general against one block of at most 4,096, 8,192, 16,384 candidates: 200
// vertices 802 against 544, 541, 542 us, 1,000 vertices 2.27 against 1.84,
// 1.70, 1.61 ms, 3,000 vertices 3.14 against 2.99, 3.03, 3.26 ms.  Sixty of
// 200-1,500 vertices: 17.0 ms by the general launches, 15.3 with 8,192, 15.2
// with 16,384; 17.1 when half of them being ready was enough (the others wait
// meanwhile).
static void advance(pra_ctx* c, const std::vector<pra_scc*>& members, u32 max, std::vector<std::vector<u64>>& rows)
{
    const u32 max_cand = members.size() < 4 ? PRA_LOOP_ROWS / 2 : PRA_LOOP_ROWS;
    rows.assign(members.size(), {});
    bool loops = max > 1;
    for (size_t k = 0; loops && k < members.size(); k++) loops = loop_ready(c, members[k], max_cand);
    if (loops) {
        std::vector<std::vector<u32>> made(members.size());
        run_loops(c, members, max, max_cand, made);
        for (size_t k = 0; k < members.size(); k++) rows[k].assign(made[k].begin(), made[k].end());
    }
    std::vector<pra_scc*> rest;
    for (size_t k = 0; k < members.size(); k++)
        if (rows[k].empty()) rest.push_back(members[k]);
    if (rest.empty()) return;
    run_iteration(c, rest);
    for (size_t k = 0; k < members.size(); k++)
        if (rows[k].empty()) rows[k].push_back(delta_sum(members[k]));
}

// The batches that some iterations of S complete, *b of whose current batch
// are made: records the delta after each.  True when S ends: after its one
// iteration, or after a batch that leaves its delta at zero.  With `whole`
// (the caller takes more than one iteration at a time) an empty iteration ends
// the batch of an SCC that one block can run: those left of it would find
// nothing either.
static bool record(pra_scc* S, u32* b, const std::vector<u64>& rows, bool whole)
{
    pra_ctx* c = S->ctx;
    for (u64 n : rows) {
        if (S->fixpoint && ++*b < c->batch_size) continue;
        *b = 0;
        S->hist.push_back(n);
        if (!S->fixpoint || n == 0) return true;
    }
    if (!whole || *b == 0 || rows.back() != 0 || S->ras.size() != 1 || !S->ras[0].out->loops) return false;
    grp(c, S->group).iterations += c->batch_size - *b;
    *b = 0;
    S->hist.push_back(0);
    return true;
}

// full -> delta at SCC start (src/relation/balanced_hash_relation.cpp:1152-1179)
static void full_to_delta(pra_ctx* c, pra_rel* R)
{
    Rows& F = R->ver[PRA_FULL];
    Rows& D = R->ver[PRA_DELTA];
    if (F.n == 0) return;
    if (D.n == 0) {
        D.buf.swap(F.buf);
        D.n = F.n;
        D.sorted = F.sorted;
        F.n = 0;
        F.sorted = true;
        R->touched(PRA_FULL);
        R->touched(PRA_DELTA);
        ensure_sorted(c, R, PRA_DELTA);
        return;
    }
    append_rows(c, R, PRA_DELTA, F.d(), F.n);
    F.n = 0;
    F.sorted = true;
    R->touched(PRA_FULL);
    sort_rows(c, D, R->w, R->jcc, R->w);
    unique_rows(c, D, R->w);
    R->touched(PRA_DELTA);
}

// delta -> full (src/relation/balanced_hash_relation.cpp:1120-1148)
static void delta_to_full(pra_ctx* c, pra_rel* R)
{
    Rows& D = R->ver[PRA_DELTA];
    if (D.n == 0) return;
    Rows& F = R->ver[PRA_FULL];
    if (F.n == 0) {   // the rows move, and stay in order
        F.buf.swap(D.buf);
        F.n = D.n;
        F.sorted = D.sorted;
        R->touched(PRA_FULL);
    } else {
        append_rows(c, R, PRA_FULL, D.d(), D.n);
    }
    D.n = 0;
    R->touched(PRA_DELTA);
}

// SCC prologue (src/lie/lie.cpp:286-302): note which relations the rules
// produce and which full versions they read in order, then move full to delta
// for the relations added with status true (skipped when a restart loaded the
// deltas from a checkpoint instead)
static void scc_begin(pra_scc* S, bool move_status)
{
    pra_ctx* c = S->ctx;
    if (S->done || S->running) throw PraError(PRA_E_STATE, "SCC already started");
    for (pra_rel* R : S->rels) R->scc_changing = R->merge_full = R->full_read = false;
    for (auto& ra : S->ras) ra.out->scc_changing = true;
    for (auto& ra : S->ras) {
        if (ra.v0 == PRA_FULL) ra.in0->full_read = true;
        if (ra.type == RA_JOIN && ra.v1 == PRA_FULL) ra.in1->full_read = true;
    }
    // a view changes with its relation, and reading its full reads the relation's
    for (auto& ra : S->ras)
        if (ra.type == RA_JOIN && ra.in1->view_of) {
            ra.in1->scc_changing = ra.in1->view_of->scc_changing;
            if (ra.v1 == PRA_FULL) ra.in1->view_of->full_read = true;
        }
    for (auto& ra : S->ras)
        for (pra_rel* R : {ra.in0, ra.in1, ra.out})
            if (R) R->merge_full = R->full_read && R->scc_changing;
    for (auto& ra : S->ras)
        if (ra.type == RA_JOIN && ra.in1->view_of) {
            pra_rel* src = ra.in1->view_of;
            src->merge_full = src->full_read && src->scc_changing;
            ra.in1->merge_full = false;
        }
    if (move_status)
        for (size_t i = 0; i < S->rels.size(); i++)
            if (S->status[i]) full_to_delta(c, S->rels[i]);
    S->running = true;
    c->lean = 0;
    S->loop_stop = ~0ULL;
    for (pra_rel* R : S->rels) R->loops = false;
    if (RADesc* ra = c->loop_on ? loop_rule(S) : nullptr) ra->out->loops = true;
}

// one batch: a single iteration for an SCC that runs once, else batch_size
// iterations; records and returns the global delta after it
// (RAM::execute_in_batches, src/RAM/RA_tasks.cpp:1121-1269)
static u64 scc_step(pra_scc* S)
{
    pra_ctx* c = S->ctx;
    if (!S->running) throw PraError(PRA_E_STATE, "SCC not started");
    u32 iters = S->fixpoint ? c->batch_size : 1;
    for (u32 b = 0; b < iters; b++) run_iteration(c, {S});
    u64 d = delta_sum(S);
    S->hist.push_back(d);
    return d;
}

// SCC epilogue: delta folded into full for every relation of the SCC (then
// the error flags checked, unless the caller checks them for several SCCs)
static void scc_end(pra_scc* S, bool check = true)
{
    pra_ctx* c = S->ctx;
    if (!S->running) throw PraError(PRA_E_STATE, "SCC not started");
    for (pra_rel* R : S->rels) {
        delta_to_full(c, R);
        R->merged.release();
        R->scc_changing = R->merge_full = R->full_read = R->loops = false;
    }
    if (check) sync_check(c);
    S->running = false;
    S->done = true;
}

static void scc_run(pra_scc* S)
{
    scc_begin(S, true);
    std::vector<std::vector<u64>> rows;
    u32 b = 0;
    do advance(S->ctx, {S}, PRA_LOOP_ITERS, rows);
    while (!record(S, &b, rows[0], true));
    scc_end(S);
}

// first runnable SCC (of instance g, or of any instance when g < 0) in
// creation order (src/lie/lie.cpp:27-60)
static pra_scc* one_runnable(pra_ctx* c, int g = -1)
{
    for (pra_scc* s : c->sccs) {
        if (s->done || (g >= 0 && s->group != g)) continue;
        bool blocked = false;
        for (auto& d : c->deps)
            if (d.second == s && !d.first->done) blocked = true;
        if (!blocked) return s;
    }
    return nullptr;
}

// One lock-step iteration over every instance's LIE::execute
// (src/lie/lie.cpp:197-448): an instance without an SCC in progress starts
// its next runnable one; then one merged iteration runs over the SCCs in
// progress, and each SCC records its batch and ends where its own LIE would:
// after its one iteration, or after a batch that leaves its delta at zero.
// Returns the instances with work left.
// max > 1: an SCC that one block can run makes up to so many iterations.
static u64 lockstep_step(pra_ctx* c, u32 max = 1)
{
    std::vector<pra_scc*> members;
    for (size_t g = 0; g < c->groups.size(); g++) {
        Group& G = *c->groups[g];
        if (!G.running) {
            pra_scc* s = one_runnable(c, (int)g);
            if (!s) continue;
            scc_begin(s, true);
            G.running = s;
            G.batch_it = 0;
        }
        members.push_back(G.running);
    }
    if (members.empty()) return 0;
    std::vector<std::vector<u64>> rows;
    advance(c, members, max, rows);
    u64 left = 0;
    for (size_t k = 0; k < members.size(); k++) {
        Group& G = grp(c, members[k]->group);
        if (record(members[k], &G.batch_it, rows[k], max > 1)) {
            scc_end(members[k], false);
            G.running = nullptr;
        }
    }
    for (size_t g = 0; g < c->groups.size(); g++)
        if (c->groups[g]->running || one_runnable(c, (int)g)) left++;
    return left;
}

static void execute_lockstep(pra_ctx* c)
{
    while (lockstep_step(c, PRA_LOOP_ITERS)) {
    }
    sync_check(c);
}

static int fail(pra_ctx* c, int code, const std::string& m)
{
    if (c) c->err = m;
    return code;
}

// The context's device is the current one inside a call (allocations and
// launches go by it).  API_BEGIN puts the caller's back at its end; the calls
// that run programs or move an exchange's rows (API_BEGIN_ON) leave the
// context's current.
struct DeviceScope {
    int prev = -1;
    explicit DeviceScope(int device)
    {
        int cur = 0;
        HIPCHK(hipGetDevice(&cur));
        if (cur == device) return;
        HIPCHK(hipSetDevice(device));
        prev = cur;
    }
    ~DeviceScope()
    {
        if (prev >= 0) (void)hipSetDevice(prev);
    }
};

#define API_BEGIN(ctxexpr)                                                                         \
    pra_ctx* ctx_ = (ctxexpr);                                                                     \
    try {                                                                                          \
        DeviceScope device_scope_(ctx_->device);
#define API_BEGIN_ON(ctxexpr)                                                                      \
    pra_ctx* ctx_ = (ctxexpr);                                                                     \
    try {                                                                                          \
        HIPCHK(hipSetDevice(ctx_->device));
#define API_END                                                                                    \
    }                                                                                              \
    catch (const PraError& e) { return fail(ctx_, e.code, e.what()); }                           \
    catch (const std::bad_alloc&) { return fail(ctx_, PRA_E_HIP, "host out of memory"); }        \
    catch (const std::exception& e) { return fail(ctx_, PRA_E_HIP, e.what()); }                  \
    return PRA_OK;

static bool valid_ver(int v) { return v == PRA_DELTA || v == PRA_FULL || v == PRA_NEWT; }

} // namespace

// ----------------------------------------------------------------- C ABI ---

extern "C" {

int pra_ctx_create(int device, int nbuckets, uint64_t hbm_budget, pra_ctx** out)
{
    if (!out || nbuckets < 1 || nbuckets > 256) return PRA_E_ARG;
    *out = nullptr;
    std::unique_ptr<pra_ctx> c(new pra_ctx());
    try {
        int ndev = 0;
        HIPCHK(hipGetDeviceCount(&ndev));
        if (device < 0 || device >= ndev) return PRA_E_ARG;
        HIPCHK(hipSetDevice(device));
        HIPCHK(pra_partition_scratch_init(device));
        // freed stream-ordered allocations stay in the device's pool for reuse
        // (instead of going back to the driver at every synchronization) up to
        // a quarter of the device memory, so that many contexts in a row do
        // not hoard fragments until allocations fail
        hipMemPool_t pool = nullptr;
        size_t free_b = 0, total_b = 0;
        if (hipDeviceGetDefaultMemPool(&pool, device) == hipSuccess && pool &&
            hipMemGetInfo(&free_b, &total_b) == hipSuccess) {
            uint64_t keep = total_b / 4;
            const char* env = getenv("PRA_POOL_RELEASE_GB");   // bytes the pool keeps, in GiB
            if (env && *env) keep = (uint64_t)(atof(env) * (double)(1ULL << 30));
            HIPCHK(hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep));
            g_small_idle_limit = (size_t)std::min<uint64_t>(keep, kSmallIdle);
        }
        c->device = device;
        c->st = stream_get(device);
        {
            std::lock_guard<std::mutex> lk(g_acct_mu);
            MemAcct& a = g_acct[c->st];
            a.budget = hbm_budget;
            a.device = device;
            a.owner = c.get();
        }
        c->nb = nbuckets;
        c->budget = hbm_budget;
        grp(c.get(), 0);
        const char* dense_env = getenv("PRA_DENSE_MEMBERSHIP");   // "0": the general hash table for every output
        c->dense_on = !(dense_env && dense_env[0] == '0');
        const char* tune_env = getenv("PRA_AUTOTUNE");            // "0": the fixed defaults of every knob
        c->tune_on = !(tune_env && tune_env[0] == '0');
        tune_init();
        const char* seg_env = getenv("PRA_SEG_SORT");             // "0": byte passes for newts over the bins
        c->seg_sort_on = !(seg_env && seg_env[0] == '0');
        const char* loop_env = getenv("PRA_RANK_LOOP");
        c->loop_on = !(loop_env && loop_env[0] == '0');
        const char* cap_env = getenv("PRA_SORT_TEST_BIN_CAP");
        c->bin_cap_test = cap_env ? strtoull(cap_env, nullptr, 10) : 0;
        const char* eb_env = getenv("PRA_DENSE_EPOCH_BITS");
        if (eb_env) c->dense_epoch_bits = std::max(0, std::min(16, atoi(eb_env)));
        c->flags_buf.reserve(64, c->st);
        pra_launch_fill_u64(c->st, c->flags_buf.as<u64>(), 1, 0);
        c->rep_words.reserve((size_t)PRA_NREP * PRA_PART_WORDS * 8, c->st);
        pra_launch_newt_rep_init(c->st, c->rep_words.as<u64>());
        c->rep_sets = 1;
        check_launch("init");
        HIPCHK(hipStreamSynchronize(c->st));
    } catch (const PraError& e) {
        return e.code;
    }
    *out = c.release();
    return PRA_OK;
}

int pra_ctx_destroy(pra_ctx* ctx)
{
    if (!ctx) return PRA_E_ARG;
    (void)hipSetDevice(ctx->device);
    if (ctx->st) (void)hipStreamSynchronize(ctx->st);
    for (auto* s : ctx->sccs) delete s;
    for (auto* r : ctx->rels) delete r;
    ctx->sccs.clear();
    ctx->rels.clear();
    delete ctx;
    return PRA_OK;
}

const char* pra_last_error(pra_ctx* ctx) { return ctx ? ctx->err.c_str() : "null context"; }

int pra_ctx_set_batch_size(pra_ctx* ctx, uint32_t bs)
{
    if (!ctx || bs == 0) return PRA_E_ARG;
    ctx->batch_size = bs;
    return PRA_OK;
}

int pra_ctx_set_join_threshold(pra_ctx* ctx, int64_t t)
{
    if (!ctx || t < 0) return PRA_E_ARG;
    ctx->threshold = t;
    return PRA_OK;
}

int pra_ctx_joined_tuples(pra_ctx* ctx, uint64_t* out)
{
    if (!ctx || !out) return PRA_E_ARG;
    API_BEGIN(ctx)
    u64 t = 0;
    for (auto& g : ctx->groups)
        if (g->joined.p) t += readback(ctx, g->joined.p, 1)[0];
    *out = t;
    API_END
}

int pra_ctx_iterations(pra_ctx* ctx, uint64_t* out)
{
    if (!ctx || !out) return PRA_E_ARG;
    u64 t = 0;
    for (auto& g : ctx->groups) t += g->iterations;
    *out = t;
    return PRA_OK;
}

int pra_ctx_set_profiling(pra_ctx* ctx, int on)
{
    if (!ctx) return PRA_E_ARG;
    API_BEGIN(ctx)
    ctx->resolve_prof();
    ctx->prof_mask = (u32)on;
    if (on)
        for (auto& k : ctx->kst) { k.launches = 0; k.ms = 0; k.bytes = 0; }
    API_END
}

int pra_ctx_kernel_stat(pra_ctx* ctx, int idx, const char** name, uint64_t* launches, double* ms, double* bytes)
{
    if (!ctx || idx < 0 || idx >= K_COUNT) return PRA_E_ARG;
    ctx->resolve_prof();
    if (name) *name = ctx->kst[idx].name;
    if (launches) *launches = ctx->kst[idx].launches;
    if (ms) *ms = ctx->kst[idx].ms;
    if (bytes) *bytes = ctx->kst[idx].bytes;
    return PRA_OK;
}

static int partition_args(pra_ctx* ctx, const uint64_t* rows, uint64_t n, uint32_t w, uint32_t jcc,
                          uint64_t* out_rows, uint64_t* bucket_bounds)
{
    if (!ctx) return PRA_E_ARG;
    if (w < 1 || w > PRA_MAXW || jcc > w) return fail(ctx, PRA_E_ARG, "row width or join-column count out of range");
    if (n >> 32) return fail(ctx, PRA_E_ARG, "more than 2^32 - 1 rows");
    if (!bucket_bounds || (n && (!rows || !out_rows))) return fail(ctx, PRA_E_ARG, "null buffer");
    return PRA_OK;
}

int pra_partition_rows(pra_ctx* ctx, const uint64_t* rows, uint64_t n, uint32_t w, uint32_t jcc, uint64_t* out_rows,
                       uint64_t* bucket_bounds)
{
    const int rc = partition_args(ctx, rows, n, w, jcc, out_rows, bucket_bounds);
    if (rc != PRA_OK) return rc;
    API_BEGIN_ON(ctx)
    ctx->part_scratch.reserve(pra_partition_scratch_words(n, (u32)ctx->nb) * 4 + 256, ctx->st);
    pra_launch_partition(ctx->st, rows, n, (int)w, (int)jcc, (u32)ctx->nb, out_rows, bucket_bounds,
                         ctx->part_scratch.as<u32>());
    check_launch("partition");
    API_END
}

int pra_partition_rows_noalloc(pra_ctx* ctx, const uint64_t* rows, uint64_t n, uint32_t w, uint32_t jcc,
                               uint64_t* out_rows, uint64_t* bucket_bounds)
{
    if (ctx && n > PRA_NOALLOC_MAX_ROWS)
        return fail(ctx, PRA_E_ARG, "allocation-free partition takes at most " + std::to_string(PRA_NOALLOC_MAX_ROWS) +
                                        " rows, got " + std::to_string(n));
    const int rc = partition_args(ctx, rows, n, w, jcc, out_rows, bucket_bounds);
    if (rc != PRA_OK) return rc;
    API_BEGIN_ON(ctx)
    u32* scratch = pra_partition_scratch(ctx->device);
    if (!scratch) throw PraError(PRA_E_STATE, "allocation-free scratch of this device was not set up");
    pra_launch_partition(ctx->st, rows, n, (int)w, (int)jcc, (u32)ctx->nb, out_rows, bucket_bounds, scratch);
    check_launch("partition_noalloc");
    API_END
}

int pra_ctx_set_group(pra_ctx* ctx, int group)
{
    if (!ctx || group < 0 || group >= PRA_MAX_GROUPS) return PRA_E_ARG;
    API_BEGIN(ctx)
    grp(ctx, group);
    ctx->cur_group = group;
    API_END
}

int pra_ctx_group_joined(pra_ctx* ctx, int group, uint64_t* out)
{
    if (!ctx || !out || group < 0 || group >= (int)ctx->groups.size()) return PRA_E_ARG;
    API_BEGIN(ctx)
    Group& G = *ctx->groups[(size_t)group];
    *out = G.joined.p ? readback(ctx, G.joined.p, 1)[0] : 0;
    API_END
}

int pra_ctx_step(pra_ctx* ctx, uint64_t* active)
{
    if (!ctx || !active) return PRA_E_ARG;
    API_BEGIN_ON(ctx)
    *active = lockstep_step(ctx);
    if (!*active) sync_check(ctx);
    API_END
}

int pra_ctx_group_status(pra_ctx* ctx, int group, int* done, uint64_t* iterations, uint64_t* bytes)
{
    if (!ctx || group < 0 || group >= (int)ctx->groups.size()) return PRA_E_ARG;
    Group& G = *ctx->groups[(size_t)group];
    if (done) *done = !G.running && !one_runnable(ctx, group);
    if (iterations) *iterations = G.iterations;
    if (bytes) {
        u64 b = 0;
        for (pra_rel* R : ctx->rels) {
            if (R->group != group) continue;
            for (auto& v : R->ver) b += v.buf.cap;
            for (const DBuf* d : {&R->mt, &R->bm, &R->dtab, &R->fresh, &R->dirty, &R->sbpre, &R->linep, &R->places, &R->next_bnd, &R->merged, &R->dx, &R->nx,
                                  &R->rk_words[0], &R->rk_words[1], &R->rk_first[0], &R->rk_first[1], &R->idx[0], &R->idx[1], &R->nkeys, &R->kgofs,
                                  &R->bin_keys, &R->bin_idx, &R->bin_cur, &R->bnd[0], &R->bnd[1]})
                b += d->cap;
        }
        *bytes = b;
    }
    return PRA_OK;
}

int pra_ctx_release_group(pra_ctx* ctx, int group)
{
    if (!ctx || group < 0 || group >= (int)ctx->groups.size()) return PRA_E_ARG;
    API_BEGIN(ctx)
    auto& deps = ctx->deps;
    deps.erase(std::remove_if(deps.begin(), deps.end(),
                              [&](const std::pair<pra_scc*, pra_scc*>& d) { return d.first->group == group; }),
               deps.end());
    std::vector<pra_scc*> keep_s;
    for (pra_scc* s : ctx->sccs)
        if (s->group == group)
            delete s;
        else
            keep_s.push_back(s);
    ctx->sccs.swap(keep_s);
    std::vector<pra_rel*> keep_r;
    for (pra_rel* r : ctx->rels)
        if (r->group == group)
            delete r;
        else
            keep_r.push_back(r);
    ctx->rels.swap(keep_r);
    ctx->groups[(size_t)group].reset(new Group());
    API_END
}

int pra_autotune_report(char* buf, uint64_t cap, uint64_t* len)
{
    if (!len) return PRA_E_ARG;
    const std::string r = g_tune.report(kTuneNames, TUNE_KNOBS);
    *len = r.size();
    if (buf && cap) {
        const size_t n = std::min<size_t>(r.size(), cap - 1);
        memcpy(buf, r.data(), n);
        buf[n] = 0;
    }
    return PRA_OK;
}

// the scratch of a context between steps: written before it is read inside
// every iteration that uses it; released on the context's stream, so reuse
// stays ordered behind the work already enqueued
static void release_scratch(pra_ctx* ctx)
{
    for (DBuf* b : {&ctx->sort_tmp, &ctx->stage, &ctx->stage2, &ctx->tmp64a, &ctx->tmp64b, &ctx->tmp64c, &ctx->cand,
                    &ctx->dest, &ctx->slot_of, &ctx->keep, &ctx->hist, &ctx->offs, &ctx->ktmp, &ctx->idxa, &ctx->idxb,
                    &ctx->posadj_dev, &ctx->ttab, &ctx->kp, &ctx->lb_status, &ctx->first})
        b->release();
    ctx->first_words = 0;
    ctx->lb_zeroed = 0;   // look-back words are zeroed again on next use
}

int pra_ctx_trim(pra_ctx* ctx)
{
    if (!ctx) return PRA_E_ARG;
    API_BEGIN_ON(ctx)
    release_scratch(ctx);
    API_END
}

// a version in trie order, between steps: refused memory, again without the
// scratch, tables, sort bins and empty versions of the iterations before
static void sorted_between_steps(pra_ctx* c, pra_rel* R, int v)
{
    try {
        ensure_sorted(c, R, v);
    } catch (const PraError& e) {
        if (!e.refused()) throw;
        release_scratch(c);
        yield_tables(c);
        for (pra_rel* r : c->rels) {
            for (DBuf* b : {&r->nkeys, &r->bin_keys, &r->bin_idx, &r->nx, &r->dx}) b->release();
            r->bin_cap = 0;
            r->dx_gen = ~0ULL;
            for (int x : {PRA_DELTA, PRA_NEWT})
                if (!r->ver[x].n) r->ver[x].buf.release();
        }
        ensure_sorted(c, R, v);
    }
}

int pra_ctx_device_bytes(pra_ctx* ctx, uint64_t* live, uint64_t* peak)
{
    if (!ctx) return PRA_E_ARG;
    std::lock_guard<std::mutex> lk(g_acct_mu);
    auto it = g_acct.find(ctx->st);
    if (live) *live = it == g_acct.end() ? 0 : (uint64_t)it->second.live;
    if (peak) *peak = it == g_acct.end() ? 0 : (uint64_t)it->second.peak;
    return PRA_OK;
}

int pra_ctx_synchronize(pra_ctx* ctx)
{
    if (!ctx) return PRA_E_ARG;
    API_BEGIN(ctx)
    HIPCHK(hipStreamSynchronize(ctx->st));
    stream_idle(ctx->st);
    API_END
}

int pra_rel_create(pra_ctx* ctx, uint32_t arity, uint32_t jcc, uint32_t tag, int canonical, pra_rel** out)
{
    if (!ctx || !out) return PRA_E_ARG;
    if (arity < 1 || arity + 1 > PRA_MAXW || jcc > arity || tag >= (1u << 18))
        return fail(ctx, PRA_E_ARG, "relation shape out of range");
    pra_rel* r = new pra_rel();
    r->ctx = ctx;
    r->arity = (int)arity;
    r->jcc = (int)jcc;
    r->tag = tag;
    r->canonical = canonical;
    r->w = (int)arity + 1;
    r->group = ctx->cur_group;
    ctx->rels.push_back(r);
    *out = r;
    return PRA_OK;
}

int pra_rel_destroy(pra_rel* rel)
{
    if (!rel) return PRA_E_ARG;
    pra_ctx* c = rel->ctx;
    (void)hipStreamSynchronize(c->st);
    std::vector<pra_rel*> keep;
    for (pra_rel* r : c->rels)
        if (r == rel || r->view_of == rel) {
            if (r != rel) delete r;
        } else {
            keep.push_back(r);
        }
    c->rels.swap(keep);
    delete rel;
    return PRA_OK;
}

int pra_rel_load_rows(pra_rel* rel, const uint64_t* rows, uint64_t nrows, int version)
{
    if (!rel || (nrows && !rows) || (version != PRA_FULL && version != PRA_DELTA)) return PRA_E_ARG;
    API_BEGIN(rel->ctx)
    pra_ctx* c = rel->ctx;
    if (nrows) {
        Rows& r = rel->ver[version];
        const size_t used = (size_t)r.n * rel->w * 8, bytes = (size_t)nrows * rel->w * 8;
        r.buf.reserve(used + bytes, c->st, used);
        HIPCHK(hipMemcpyAsync(r.buf.as<char>() + used, rows, bytes, hipMemcpyHostToDevice, c->st));
        r.n += nrows;
        r.sorted = false;
        rel->touched(version);
        bool dup = false;   // a sort that saw no equal rows leaves none to remove
        sort_rows(c, r, rel->w, rel->jcc, rel->w, true, nullptr, &dup);
        if (dup) unique_rows(c, r, rel->w);
        HIPCHK(hipStreamSynchronize(c->st));
        rel->touched(version);
        rel->mt_valid = false;
        rel->bm_valid = false;
    }
    API_END
}

int pra_rel_load_bin(pra_rel* rel, const char* path, int version)
{
    if (!rel || !path) return PRA_E_ARG;
    pra_ctx* c = rel->ctx;
    std::string sp = std::string(path) + ".size";
    FILE* f = fopen(sp.c_str(), "r");
    if (!f) return fail(c, PRA_E_IO, "cannot open " + sp);
    long long rows = -1, cols = -1;
    int got = fscanf(f, "%lld\n%lld", &rows, &cols);
    fclose(f);
    if (got != 2 || rows < 0) return fail(c, PRA_E_IO, "malformed " + sp);
    if (cols != rel->w) return fail(c, PRA_E_IO, "column count in " + sp + " does not match arity+1");
    std::vector<u64> buf((size_t)rows * cols);
    if (rows) {
        FILE* d = fopen(path, "rb");
        if (!d) return fail(c, PRA_E_IO, std::string("cannot open ") + path);
        size_t n = fread(buf.data(), 8, buf.size(), d);
        fclose(d);
        if (n != buf.size()) return fail(c, PRA_E_IO, std::string("short read of ") + path);
    }
    return pra_rel_load_rows(rel, buf.data(), (uint64_t)rows, version);
}

int pra_rel_count(pra_rel* rel, int version, uint64_t* out)
{
    if (!rel || !out || !valid_ver(version)) return PRA_E_ARG;
    *out = rel->ver[version].n;
    return PRA_OK;
}

int pra_rel_device_rows(pra_rel* rel, int version, const uint64_t** rows, uint64_t* nrows)
{
    if (!rel || !rows || !nrows || !valid_ver(version)) return PRA_E_ARG;
    API_BEGIN(rel->ctx)
    pra_ctx* c = rel->ctx;
    if (version != PRA_NEWT) sorted_between_steps(c, rel, version);
    HIPCHK(hipStreamSynchronize(c->st));
    *rows = rel->ver[version].d();
    *nrows = rel->ver[version].n;
    API_END
}

int pra_rel_checksum(pra_rel* rel, int version, uint64_t* out)
{
    if (!rel || !out || !valid_ver(version)) return PRA_E_ARG;
    API_BEGIN(rel->ctx)
    pra_ctx* c = rel->ctx;
    if (version != PRA_NEWT) sorted_between_steps(c, rel, version);
    Rows& r = rel->ver[version];
    c->orand.reserve(32 * 8, c->st);
    pra_launch_fill_u64(c->st, c->orand.as<u64>(), 1, 0);
    pra_launch_rows_checksum(c->st, r.d(), r.n, rel->w, c->orand.as<u64>());
    check_launch("rows_checksum");
    *out = readback(c, c->orand.p, 1)[0];
    API_END
}

int pra_rel_download(pra_rel* rel, int version, uint64_t* rows, uint64_t cap, uint64_t* nrows)
{
    if (!rel || !nrows || !valid_ver(version)) return PRA_E_ARG;
    API_BEGIN(rel->ctx)
    pra_ctx* c = rel->ctx;
    if (version != PRA_NEWT) sorted_between_steps(c, rel, version);
    Rows& r = rel->ver[version];
    *nrows = r.n;
    u64 m = std::min<u64>(cap, r.n);
    if (m && rows) HIPCHK(hipMemcpyAsync(rows, r.d(), m * rel->w * 8, hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    API_END
}

int pra_rel_write_bin(pra_rel* rel, const char* path, int version)
{
    if (!rel || !path || !valid_ver(version)) return PRA_E_ARG;
    pra_ctx* c = rel->ctx;
    uint64_t n = 0, got = 0;
    int rc = pra_rel_count(rel, version, &n);
    if (rc != PRA_OK) return rc;
    std::vector<u64> buf((size_t)n * rel->w);
    rc = pra_rel_download(rel, version, buf.data(), n, &got);
    if (rc != PRA_OK) return rc;
    FILE* f = fopen(path, "wb");
    if (!f) return fail(c, PRA_E_IO, std::string("cannot create ") + path);
    size_t wrote = n ? fwrite(buf.data(), 8, buf.size(), f) : 0;
    int closed = fclose(f);
    if (wrote != buf.size() || closed != 0) return fail(c, PRA_E_IO, std::string("short write of ") + path);
    std::string sp = std::string(path) + ".size";
    FILE* m = fopen(sp.c_str(), "w");
    if (!m) return fail(c, PRA_E_IO, "cannot create " + sp);
    fprintf(m, "%llu\n%d", (unsigned long long)n, rel->w);
    if (fclose(m) != 0) return fail(c, PRA_E_IO, "short write of " + sp);
    return PRA_OK;
}

int pra_scc_create(pra_ctx* ctx, int fixpoint, int id, pra_scc** out)
{
    if (!ctx || !out) return PRA_E_ARG;
    pra_scc* s = new pra_scc();
    s->ctx = ctx;
    s->fixpoint = fixpoint != 0;
    s->id = id;
    s->group = ctx->cur_group;
    ctx->sccs.push_back(s);
    *out = s;
    return PRA_OK;
}

int pra_scc_destroy(pra_scc* scc)
{
    if (!scc) return PRA_E_ARG;
    pra_ctx* c = scc->ctx;
    c->sccs.erase(std::remove(c->sccs.begin(), c->sccs.end(), scc), c->sccs.end());
    c->deps.erase(std::remove_if(c->deps.begin(), c->deps.end(),
                                 [&](const std::pair<pra_scc*, pra_scc*>& d) {
                                     return d.first == scc || d.second == scc;
                                 }),
                  c->deps.end());
    delete scc;
    return PRA_OK;
}

int pra_scc_add_relation(pra_scc* scc, pra_rel* rel, int move_full_to_delta)
{
    if (!scc || !rel || rel->ctx != scc->ctx || rel->group != scc->group) return PRA_E_ARG;
    if (scc->rels.size() >= 64) return fail(scc->ctx, PRA_E_ARG, "at most 64 relations per SCC");
    scc->rels.push_back(rel);
    scc->status.push_back(move_full_to_delta != 0);
    return PRA_OK;
}

// the relations belong to the SCC's context and instance
static bool same_ctx(pra_scc* s, pra_rel* a, pra_rel* b = nullptr, pra_rel* d = nullptr)
{
    auto ok = [&](pra_rel* r) { return r->ctx == s->ctx && r->group == s->group; };
    return a && ok(a) && (!b || ok(b)) && (!d || ok(d));
}

int pra_scc_add_join(pra_scc* scc, pra_rel* out, pra_rel* in0, int ver0, pra_rel* in1, int ver1, const int* proj,
                     int nproj)
{
    if (!scc || !same_ctx(scc, out, in0, in1) || (nproj && !proj)) return PRA_E_ARG;
    pra_ctx* c = scc->ctx;
    if ((ver0 != PRA_DELTA && ver0 != PRA_FULL) || (ver1 != PRA_DELTA && ver1 != PRA_FULL))
        return fail(c, PRA_E_ARG, "join versions must be DELTA or FULL");
    if (nproj != out->arity) return fail(c, PRA_E_ARG, "projection width must equal the output arity");
    if (in0->jcc > in1->arity) return fail(c, PRA_E_ARG, "input 0's join column count exceeds input 1's arity");
    int span = in0->w + in1->w - in0->jcc;
    for (int i = 0; i < nproj; i++)
        if (proj[i] < 0 || proj[i] >= span) return fail(c, PRA_E_ARG, "projection index out of range");
    RADesc ra;
    ra.type = RA_JOIN;
    ra.out = out;
    ra.in0 = in0;
    ra.v0 = ver0;
    ra.in1 = in1;
    ra.v1 = ver1;
    if (in0->jcc != in1->jcc) {
        // input 1 seen through its view keyed on input 0's join column count
        pra_rel* view = nullptr;
        for (pra_rel* r : c->rels)
            if (r->view_of == in1 && r->jcc == in0->jcc) view = r;
        if (!view) {
            view = new pra_rel();
            view->ctx = c;
            view->group = in1->group;
            view->arity = in1->arity;
            view->jcc = in0->jcc;
            view->tag = in1->tag;
            view->canonical = in1->canonical;
            view->w = in1->w;
            view->view_of = in1;
            c->rels.push_back(view);
        }
        ra.in1 = view;
    }
    ra.map.assign(proj, proj + nproj);
    scc->ras.push_back(std::move(ra));
    return PRA_OK;
}

static int add_copylike(pra_scc* scc, int type, pra_rel* out, pra_rel* in, int ver, const int* map, int n, int op)
{
    if (!scc || !same_ctx(scc, out, in) || (n && !map)) return PRA_E_ARG;
    pra_ctx* c = scc->ctx;
    if (ver != PRA_DELTA && ver != PRA_FULL) return fail(c, PRA_E_ARG, "input version must be DELTA or FULL");
    int want = type == RA_ACOPY ? out->w : out->arity;
    if (n != want) return fail(c, PRA_E_ARG, "reorder width does not match the output relation");
    for (int i = 0; i < n; i++)
        if (map[i] < 0 || map[i] >= in->w) return fail(c, PRA_E_ARG, "reorder index out of range");
    if (type == RA_COPY_FILTER && (op < PRA_FILTER_EQ || op > PRA_FILTER_FALSE))
        return fail(c, PRA_E_ARG, "unknown filter predicate");
    if (type == RA_COPY_FILTER && in->w < 2) return fail(c, PRA_E_ARG, "filter reads two input columns");
    RADesc ra;
    ra.type = type;
    ra.out = out;
    ra.in0 = in;
    ra.v0 = ver;
    ra.op = op;
    ra.map.assign(map, map + n);
    scc->ras.push_back(std::move(ra));
    return PRA_OK;
}

int pra_scc_add_copy(pra_scc* scc, pra_rel* out, pra_rel* in, int ver, const int* reorder, int n)
{
    return add_copylike(scc, RA_COPY, out, in, ver, reorder, n, PRA_F_TRUE);
}

int pra_scc_add_acopy(pra_scc* scc, pra_rel* out, pra_rel* in, int ver, const int* reorder, int n)
{
    return add_copylike(scc, RA_ACOPY, out, in, ver, reorder, n, PRA_F_TRUE);
}

int pra_scc_add_copy_filter(pra_scc* scc, pra_rel* out, pra_rel* in, int ver, const int* reorder, int n, int op)
{
    return add_copylike(scc, RA_COPY_FILTER, out, in, ver, reorder, n, op);
}

int pra_scc_add_dependency(pra_scc* before, pra_scc* after)
{
    if (!before || !after || before->ctx != after->ctx || before->group != after->group) return PRA_E_ARG;
    before->ctx->deps.push_back({before, after});
    return PRA_OK;
}

int pra_scc_run(pra_scc* scc, uint64_t* delta_hist, uint64_t cap, uint64_t* nbatches)
{
    if (!scc) return PRA_E_ARG;
    API_BEGIN_ON(scc->ctx)
    size_t before = scc->hist.size();
    scc_run(scc);
    size_t nb = scc->hist.size() - before;
    if (nbatches) *nbatches = nb;
    for (size_t i = 0; delta_hist && i < nb && i < cap; i++) delta_hist[i] = scc->hist[before + i];
    API_END
}

int pra_scc_begin(pra_scc* scc, int move_full_to_delta)
{
    if (!scc) return PRA_E_ARG;
    API_BEGIN_ON(scc->ctx)
    scc_begin(scc, move_full_to_delta != 0);
    API_END
}

int pra_scc_step(pra_scc* scc, uint64_t* delta)
{
    if (!scc) return PRA_E_ARG;
    API_BEGIN_ON(scc->ctx)
    u64 d = scc_step(scc);
    if (delta) *delta = d;
    API_END
}

int pra_scc_end(pra_scc* scc)
{
    if (!scc) return PRA_E_ARG;
    API_BEGIN_ON(scc->ctx)
    scc_end(scc);
    API_END
}

int pra_scc_history(pra_scc* scc, uint64_t* out, uint64_t cap, uint64_t* n)
{
    if (!scc || !n) return PRA_E_ARG;
    *n = scc->hist.size();
    for (size_t i = 0; out && i < scc->hist.size() && i < cap; i++) out[i] = scc->hist[i];
    return PRA_OK;
}

int pra_execute(pra_ctx* ctx)
{
    if (!ctx) return PRA_E_ARG;
    API_BEGIN_ON(ctx)
    if (ctx->groups.size() > 1) {
        execute_lockstep(ctx);
    } else {
        pra_scc* s;
        while ((s = one_runnable(ctx)) != nullptr) scc_run(s);
    }
    API_END
}

int pra_execute_many(pra_ctx** ctxs, int n, int concurrency, int* rc)
{
    if (!ctxs || n < 0 || concurrency < 1) return PRA_E_ARG;
    for (int i = 0; i < n; i++)
        if (!ctxs[i]) return PRA_E_ARG;
    std::vector<int> status(n, PRA_OK);
    std::atomic<int> next(0);
    auto worker = [&]() {
        for (;;) {
            int i = next.fetch_add(1);
            if (i >= n) return;
            status[i] = pra_execute(ctxs[i]);
        }
    };
    int nt = std::min(concurrency, std::max(n, 1));
    std::vector<std::thread> pool;
    for (int t = 1; t < nt; t++) pool.emplace_back(worker);
    worker();
    for (auto& t : pool) t.join();
    int first = PRA_OK;
    for (int i = 0; i < n; i++) {
        if (rc) rc[i] = status[i];
        if (first == PRA_OK && status[i] != PRA_OK) first = status[i];
    }
    return first;
}

} // extern "C"
