// bj_tiles.h -- device bodies shared by the single-join kernels (bj_kernels.hip)
// and the batched kernels (bj_batch.hip).
//
// Each body works on one contiguous range (a histogram chunk, a scatter range,
// a filter segment, a probe work item); the kernels around them only decide
// which range a workgroup owns and where its results go.
#pragma once

#include "bj_device.h"

#include <type_traits>

namespace bj {

// 64-bit value that is the same in every lane, in scalar registers
__device__ __forceinline__ uint64_t uniform_u64(uint64_t v)
{
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// ---------------------------------------------------------------- histogram
// h[] (LDS, zeroed by the caller) += histogram of the top (32 - sh) bits of the
// radix hash over key[lo, hi).  8 loads in flight per thread.
template <int BLOCK>
__device__ __forceinline__ void hist_range(const uint32_t* __restrict__ key, uint64_t lo, uint64_t hi,
                                           int sh, uint32_t* h)
{
    constexpr int U = 8;
    uint64_t i = lo + threadIdx.x;
    for (; i + (uint64_t)(U - 1) * BLOCK < hi; i += (uint64_t)U * BLOCK) {
        uint32_t k[U];
#pragma unroll
        for (int u = 0; u < U; u++) k[u] = key[i + (uint64_t)u * BLOCK];
#pragma unroll
        for (int u = 0; u < U; u++) atomicAdd(&h[radix_hash(k[u]) >> sh], 1u);
    }
    for (; i < hi; i += BLOCK) atomicAdd(&h[radix_hash(key[i]) >> sh], 1u);
}

// ---------------------------------------------------------------- scatter
// LDS-staged scatter with write-combining carries.
//
// Each tile of T tuples is counting-sorted by bucket in LDS (rank from an LDS atomic,
// offsets from an LDS scan).  Bucket b's tuples go to consecutive global positions
// starting at cur[b].  Only whole CS-tuple chunks (CS * 8 bytes of whole tuples, CS * 4
// of each of two arrays) are written; the unaligned tail of every bucket (< CS tuples)
// is carried in LDS to the next tile, so every chunk of the output is written by one
// workgroup within one tile.  Partial chunks occur only where two workgroups' ranges of
// a bucket meet.  The next tile is loaded into registers while the current one is
// written out.
// A tuple as one 8-byte unit: key, then value.
typedef uint32_t Tuple __attribute__((ext_vector_type(2)));

// Where a scatter reads or writes: keys and values in two arrays (the caller's
// relations, the final sub-bucket layout) or whole tuples in one (the layout
// between two passes, and between S's first pass and the filter).
template <bool PAIR>
struct TupleIn;
template <>
struct TupleIn<false> {
    const uint32_t* __restrict__ key;
    const uint32_t* __restrict__ val;
    __device__ __forceinline__ Tuple load(uint32_t i) const
    {
        return Tuple{__builtin_nontemporal_load(&key[i]), __builtin_nontemporal_load(&val[i])};
    }
    __device__ __forceinline__ TupleIn from(uint64_t lo) const { return {key + lo, val + lo}; }
};
template <>
struct TupleIn<true> {
    const Tuple* __restrict__ t;
    __device__ __forceinline__ Tuple load(uint32_t i) const { return __builtin_nontemporal_load(&t[i]); }
    __device__ __forceinline__ TupleIn from(uint64_t lo) const { return {t + lo}; }
};
template <bool PAIR>
struct TupleOut;
template <>
struct TupleOut<false> {
    uint32_t* __restrict__ key;
    uint32_t* __restrict__ val;
    __device__ __forceinline__ void store(uint64_t i, Tuple x) const
    {
        key[i] = x.x;
        val[i] = x.y;
    }
};
template <>
struct TupleOut<true> {
    Tuple* __restrict__ t;
    __device__ __forceinline__ void store(uint64_t i, Tuple x) const { t[i] = x; }
};

struct ScatterLds {
    uint64_t* cur;   // [nbk] next global position
    uint64_t* dst;   // [nbk] position of the tile's tuple s: dst + s
    Tuple* carry;    // [nbk * cs] carried tuples
    Tuple* stage;    // [T] the tile, bucket by bucket
    uint32_t* cnt;   // [nbk] tile tuples (even tiles: low half, odd tiles: high half)
    uint32_t* ol;    // [nbk] staging offset | end of the staged tuples written this tile << 16
    uint32_t* nc;    // [nbk] tuples written this tile | carried tuples << 16
    uint32_t* wtmp;  // [BLOCK/64 + 1]
};
constexpr int SCATTER_BUCKET_BYTES = 28;  // cur, dst, cnt, ol, nc

// Carry chunk (log2 tuples) of an nbk-way pass.  big: one workgroup per CU, which
// has the CU's LDS to itself.  Whole tuples fill a 128-byte line with 16; two
// arrays need 32 for whole lines of each, affordable in big up to 256 buckets.
// Above 512 buckets smaller chunks keep the carry at 64 KB.
__host__ __device__ __forceinline__ int scatter_carry_log2(int nbk, bool big, bool opair)
{
    if (big && !opair && nbk <= 256) return 5;
    return nbk <= 512 ? 4 : (nbk <= 1024 ? 3 : 2);
}

template <int BLOCK, int ITEMS>
__device__ __forceinline__ ScatterLds scatter_lds(uint64_t* lds64, int nbk, int cs_log2)
{
    constexpr int T = BLOCK * ITEMS;
    static_assert(T <= 16384, "offsets and counts are kept in 16 bits");
    ScatterLds L;
    L.cur = lds64;
    L.dst = L.cur + nbk;
    L.carry = (Tuple*)(L.dst + nbk);
    L.stage = L.carry + (nbk << cs_log2);
    L.cnt = (uint32_t*)(L.stage + T);
    L.ol = L.cnt + nbk;
    L.nc = L.ol + nbk;
    L.wtmp = L.nc + nbk;
    return L;
}

// Buckets [b0, b0 + PER) of a thread after a tile's ranks: retire the previous
// tile (its nw tuples leave the carry, the others stay carried), then size this
// tile's writes from the bucket's count c and its staging offset.  scan turns a
// thread's sum of counts into its exclusive prefix; on: the thread owns buckets.
template <int PER, class Scan>
__device__ __forceinline__ void scatter_offsets(const ScatterLds& L, int b0, bool on, uint32_t par, uint32_t cs,
                                                Scan&& scan)
{
    uint32_t c[PER], cc[PER];
    uint64_t cur[PER];
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        c[j] = cc[j] = 0;
        cur[j] = 0;
        if (on) {
            const uint32_t cn = L.cnt[b0 + j], nc = L.nc[b0 + j], nw = nc & 0xFFFFu;
            const uint32_t lo = cn & 0xFFFFu, hi = cn >> 16;
            c[j] = par ? hi : lo;
            cc[j] = (nc >> 16) + (par ? lo : hi) - nw;
            cur[j] = L.cur[b0 + j] + nw;
            L.cnt[b0 + j] = par ? hi << 16 : lo;  // the next tile counts from zero
            sum += c[j];
        }
    }
    uint32_t ex = scan(sum);
#pragma unroll
    for (int j = 0; j < PER; j++) {
        if (on) {
            const uint32_t b = b0 + j;
            // written: up to the bucket's last whole chunk, then none of the carry
            // stays (a0 + carried < cs: one more chunk always covers it)
            const uint32_t a0 = (uint32_t)cur[j] & (cs - 1u);
            const uint32_t e = a0 + cc[j] + c[j];
            const uint32_t nw = e >= cs ? (e & ~(cs - 1u)) - a0 : 0u;
            L.cur[b] = cur[j];
            L.dst[b] = cur[j] + cc[j] - ex;
            L.ol[b] = ex | ((nw ? ex + nw - cc[j] : ex) << 16);
            L.nc[b] = nw | (cc[j] << 16);
            ex += c[j];
        }
    }
}

// Scatters in[0, len) by bucket (radix_hash(key) >> shift) & bmask into out at the
// cursors L.cur[] (initialised by the caller; this function begins with a
// barrier).  Writes are bounds-checked against out_cap; returns true on a
// violation.
//
// Per tile three barriers: (next tile's loads) ranks (LDS atomics) | offsets (scan of
// the counts, retiring the previous tile's buckets and sizing this tile's writes) |
// staging + (or here the loads) + carried tuples out | the tile's tuples out or into the carry
// (which runs into the next tile's ranks).  Counts alternate between the halves of
// a word so the next tile's ranks need no clearing barrier.
//
// A whole tile runs without per-tuple branches, every group of LDS or global
// accesses issued before the first of them is waited for, and the next tile's
// loads are unconditional (clamped to the last tuple): with a branch per tuple the
// compiler waited for each load, and for each LDS read, before it issued the next.
// HBM bandwidth bounds large passes: 640M tuples by 128 buckets into whole tuples
// 2.43 -> 2.24 ms (4.6 TB/s; a plain copy reaches 4.96), by 256 buckets 2.88 -> 2.41,
// a second pass 2.67 -> 2.43; 100M tuples 0.45 -> 0.33 ms.  Whole tuples halve a
// bucket's carry (16 tuples fill a 128-byte line) and the store instructions.
template <int BLOCK, int ITEMS, bool IPAIR, bool OPAIR>
__device__ __forceinline__ bool scatter_range(const ScatterLds& L, const TupleIn<IPAIR>& in, uint32_t len, int nbk,
                                              int shift, uint32_t bmask, int cs_log2, const TupleOut<OPAIR>& out,
                                              uint64_t out_cap)
{
    constexpr uint32_t T = BLOCK * ITEMS;
    constexpr int U = 4;  // tuples of a thread handled together on the way out
    static_assert(ITEMS % U == 0, "groups of U");
    const uint32_t cs = 1u << cs_log2;
    const uint32_t ncarry = (uint32_t)nbk << cs_log2;
    for (int b = threadIdx.x; b < nbk; b += BLOCK) {
        L.cnt[b] = 0u;
        L.nc[b] = 0u;
    }
    __syncthreads();  // cur is read by other threads
    if (len == 0) return false;

    Tuple kv[ITEMS], nx[ITEMS];
    auto load_tile = [&](Tuple* x, uint32_t at) {
#pragma unroll
        for (int it = 0; it < ITEMS; it++) x[it] = in.load(min(at + (uint32_t)it * BLOCK + threadIdx.x, len - 1u));
    };
    load_tile(kv, 0);
    bool bad = false;
    uint32_t par = 0;

    auto run_tile = [&](auto whole, uint32_t tile, uint32_t tn) {
        constexpr bool WHOLE = decltype(whole)::value;
        // one workgroup per CU: no other workgroup's loads fill the time until this
        // tile is staged, and there are registers for a second tile
        constexpr bool EARLY = WHOLE && ITEMS == 8 && BLOCK == 1024;
        if (EARLY) load_tile(nx, tile + T);
        uint32_t br[ITEMS];  // bucket | rank << 16
        const uint32_t one = par ? 1u << 16 : 1u, half = par ? 16u : 0u;
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            br[it] = (radix_hash(kv[it].x) >> shift) & bmask;
            if (WHOLE || (uint32_t)it * BLOCK + threadIdx.x < tn)
                br[it] |= ((atomicAdd(&L.cnt[br[it]], one) >> half) & 0xFFFFu) << 16;
        }
        __syncthreads();
        if (nbk <= 2 * WAVE) {
            // one wave, up to two buckets per lane
            if (threadIdx.x < WAVE) {
                auto scan = [&](uint32_t x) { return wave_inclusive_scan<uint32_t>(x) - x; };
                if (nbk <= WAVE) scatter_offsets<1>(L, threadIdx.x, (int)threadIdx.x < nbk, par, cs, scan);
                else scatter_offsets<2>(L, 2 * threadIdx.x, true, par, cs, scan);
            }
        } else {
            // the whole workgroup: from 3 buckets per lane on, one wave working
            // through them keeps the others waiting longer than the block scan's
            // barriers
            auto scan = [&](uint32_t x) {
                uint32_t tot;
                return block_exclusive_scan<BLOCK, uint32_t>(x, L.wtmp, &tot);
            };
            if (nbk <= BLOCK) scatter_offsets<1>(L, threadIdx.x, (int)threadIdx.x < nbk, par, cs, scan);
            else if (nbk == 2 * BLOCK) scatter_offsets<2>(L, 2 * threadIdx.x, true, par, cs, scan);
            else scatter_offsets<4>(L, 4 * threadIdx.x, 4 * (int)threadIdx.x < nbk, par, cs, scan);
        }
        __syncthreads();
        uint32_t q[ITEMS];
#pragma unroll
        for (int it = 0; it < ITEMS; it++) q[it] = (L.ol[br[it] & 0xFFFFu] & 0xFFFFu) + (br[it] >> 16);
#pragma unroll
        for (int it = 0; it < ITEMS; it++)
            if (WHOLE || (uint32_t)it * BLOCK + threadIdx.x < tn) L.stage[q[it]] = kv[it];
        // (two workgroups per CU: the next tile takes the registers of the staged one;
        // its own registers spill, 3M x 4.5M's second pass 33 -> 40 us)
        if (WHOLE && !EARLY && tile + T < len) load_tile(kv, tile + T);
        // carried tuples of the buckets that are written go out
        for (uint32_t i0 = threadIdx.x; i0 < ncarry; i0 += U * BLOCK) {
            uint32_t nc[U];
            uint64_t g[U];
            Tuple x[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t i = min(i0 + (uint32_t)u * BLOCK, ncarry - 1u);
                nc[u] = L.nc[i >> cs_log2];
                g[u] = L.cur[i >> cs_log2] + (i & (cs - 1u));
                x[u] = L.carry[i];
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t i = i0 + (uint32_t)u * BLOCK;
                if (i < ncarry && (nc[u] & 0xFFFFu) && (i & (cs - 1u)) < nc[u] >> 16) {
                    if (g[u] < out_cap) out.store(g[u], x[u]);
                    else bad = true;
                }
            }
        }
        __syncthreads();
        // the tile's tuples go out, or into the carry
#pragma unroll
        for (int h = 0; h < ITEMS; h += U) {
            Tuple x[U];
            uint32_t b[U], ol[U];
            uint64_t g[U];
#pragma unroll
            for (int u = 0; u < U; u++) x[u] = L.stage[(uint32_t)(h + u) * BLOCK + threadIdx.x];
#pragma unroll
            for (int u = 0; u < U; u++) {
                b[u] = (radix_hash(x[u].x) >> shift) & bmask;
                ol[u] = L.ol[b[u]];
                g[u] = L.dst[b[u]];
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t s = (uint32_t)(h + u) * BLOCK + threadIdx.x;
                if (!WHOLE && s >= tn) continue;
                if (s < ol[u] >> 16) {
                    g[u] += s;
                    if (g[u] < out_cap) out.store(g[u], x[u]);
                    else bad = true;
                } else {
                    // behind the carried tuples, or first where those were written
                    const uint32_t nc = L.nc[b[u]];
                    L.carry[(b[u] << cs_log2) + s - (ol[u] >> 16) + ((nc & 0xFFFFu) ? 0u : nc >> 16)] = x[u];
                }
            }
        }
        if (EARLY) {
#pragma unroll
            for (int it = 0; it < ITEMS; it++) kv[it] = nx[it];
        }
        par ^= 1u;
    };
    uint32_t tile = 0;
    for (; tile + T <= len; tile += T) run_tile(std::true_type{}, tile, T);
    if (tile < len) run_tile(std::false_type{}, tile, len - tile);
    __syncthreads();
    // retire the last tile: the remaining carries (partial chunks at the range ends)
    for (uint32_t i = threadIdx.x; i < ncarry; i += BLOCK) {
        const uint32_t b = i >> cs_log2, k = i & (cs - 1u);
        const uint32_t cn = L.cnt[b], nc = L.nc[b], nw = nc & 0xFFFFu;
        if (k < (nc >> 16) + (par ? cn & 0xFFFFu : cn >> 16) - nw) {
            const uint64_t g = L.cur[b] + nw + k;
            if (g < out_cap) out.store(g, L.carry[i]);
            else bad = true;
        }
    }
    return bad;
}

// ---------------------------------------------------------------- Bloom build
// seg[] (LDS, wps 64-bit blocks, zeroed by the caller) |= the block masks of
// rkey[lo, hi); all keys belong to the segment starting at block segbase.
template <int BLOCK>
__device__ __forceinline__ void bloom_build_range(const uint32_t* __restrict__ rkey, uint64_t lo,
                                                  uint64_t hi, const BloomGeom& g, uint64_t segbase,
                                                  unsigned long long* seg)
{
    constexpr int U = 8;
    for (uint64_t i = lo + threadIdx.x; i < hi; i += (uint64_t)U * BLOCK) {
        uint32_t kk[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint64_t j = i + (uint64_t)u * BLOCK;
            kk[u] = (j < hi) ? __builtin_nontemporal_load(&rkey[j]) : 0u;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (i + (uint64_t)u * BLOCK < hi) {
                const uint32_t w = (uint32_t)(bloom_block(kk[u], g) - segbase);
                atomicOr(&seg[w], (unsigned long long)bloom_mask(kk[u], g.k));
            }
        }
    }
}

// ---------------------------------------------------------------- Bloom filter S -> S'
// One tile of a filter run: its source (two arrays, or whole tuples at pair), its
// tuples, the filter, and where its survivors go (reserved on *count).
struct FilterTile {
    const uint32_t* key;
    const uint32_t* val;
    const Tuple* pair;  // not null: the source
    uint32_t n;         // 1 .. BLOCK * ITEMS
    const uint64_t* filter;
    BloomGeom g;
    uint32_t* okey;
    uint32_t* oval;
    uint64_t out_cap;
    uint64_t* count;
};

// Runs tiles through the filter: every key tests its 64-bit block; survivors are ranked
// by wave ballots per (item, wave) group and a scan of the group counts, staged in LDS
// and written, compacted, at places reserved with one global atomic per tile.  The
// reservation and the stores lag one tile behind (two staging buffers) and the next
// tile's tuples are loaded while this one is staged, so neither latency is on a tile's
// path.  Values are loaded with the keys: from some 10% survivors on their lines are
// touched anyway, and below that the requests for filter words bound the run, not the
// bytes (2.5M x 100M with 0 / 1 / 3 / 10% matches: 453 / 456 / 458 / 459 us; the
// form before, with the values of survivors only, 474 / 495 / 513 / 545).  Tile numbers run below end: next(t)
// is the number that follows the one it returned last (thread 0 requests it a tile
// ahead), desc(t) its tile.  stage: 2 * BLOCK * ITEMS tuples, gcnt: 64 counts, s_base /
// s_next: one word each.  Returns true if a write would pass its tile's out_cap.
template <int BLOCK, int ITEMS, class Next, class Desc>
__device__ __forceinline__ bool filter_run(uint32_t end, Next&& next, Desc&& desc, Tuple* stage, uint32_t* gcnt,
                                           uint64_t* s_base, uint32_t* s_next)
{
    constexpr int T = BLOCK * ITEMS;
    constexpr int NW = BLOCK / WAVE;
    static_assert(ITEMS * NW == WAVE, "one group count per lane");
    const int wid = threadIdx.x / WAVE;
    const uint32_t lane = lane_id();
    if (threadIdx.x == 0) {
        s_next[0] = next();
        s_next[1] = next();
    }
    __syncthreads();
    // (in scalar registers: so are the tiles' addresses then)
    const uint32_t t_first = __builtin_amdgcn_readfirstlane(s_next[0]);
    uint32_t t_next = __builtin_amdgcn_readfirstlane(s_next[1]);
    __syncthreads();  // s_next is rewritten
    if (t_first >= end) return false;
    FilterTile d = desc(t_first);
    Tuple nk[ITEMS];
    // clamped to the tile's last tuple rather than skipped past it: no branch per load
    auto load_tile = [&](const FilterTile& f) {
        if (f.pair) {
            const TupleIn<true> in{f.pair};
#pragma unroll
            for (int it = 0; it < ITEMS; it++) nk[it] = in.load(min((uint32_t)it * BLOCK + threadIdx.x, f.n - 1u));
        } else {
            const TupleIn<false> in{f.key, f.val};
#pragma unroll
            for (int it = 0; it < ITEMS; it++) nk[it] = in.load(min((uint32_t)it * BLOCK + threadIdx.x, f.n - 1u));
        }
    };
    load_tile(d);
    bool bad = false;
    uint32_t par = 0, last_n = 0;  // survivors of the last tile, staged and not yet written
    uint32_t *last_key = nullptr, *last_val = nullptr;
    uint64_t last_cap = 0, base = 0;  // base: thread 0, the last tile's reservation
    auto write_out = [&]() {
        const uint64_t b = uniform_u64(*s_base);
        const uint32_t nw = b >= last_cap ? 0u : (uint32_t)min<uint64_t>(last_n, last_cap - b);
        bad |= nw < last_n;
        const Tuple* src = stage + (par ^ 1u) * T;
        for (uint32_t q = threadIdx.x; q < nw; q += BLOCK) {
            const Tuple x = src[q];
            (last_key + b)[q] = x.x;
            (last_val + b)[q] = x.y;
        }
    };
    for (;;) {
        uint32_t t_after = end;
        if (threadIdx.x == 0) t_after = next();
        Tuple k[ITEMS];
#pragma unroll
        for (int it = 0; it < ITEMS; it++) k[it] = nk[it];
        // every filter word in flight before any is tested
        uint64_t fw[ITEMS];
#pragma unroll
        for (int it = 0; it < ITEMS; it++) fw[it] = d.filter[bloom_block(k[it].x, d.g)];
        uint32_t rank[ITEMS], pass = 0;
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            asm volatile("" : "+v"(fw[it]));  // used on every path: not sunk into a branch
            const uint64_t m = bloom_mask(k[it].x, d.g.k);
            const bool ok = (uint32_t)it * BLOCK + threadIdx.x < d.n && (fw[it] & m) == m;
            const uint64_t b = __ballot(ok);
            rank[it] = lanes_below(b);
            pass |= (ok ? 1u : 0u) << it;
            if (lane == 0) gcnt[it * NW + wid] = (uint32_t)__popcll(b);
        }
        __syncthreads();
        const uint32_t c = gcnt[lane];
        const uint32_t inc = wave_inclusive_scan<uint32_t>(c);
        const uint32_t total = __builtin_amdgcn_readlane(inc, WAVE - 1);
        if (threadIdx.x == 0) {
            *s_base = base;
            s_next[0] = t_after;
            base = total ? atomicAdd((unsigned long long*)d.count, (unsigned long long)total) : 0ull;
        }
        const bool more = t_next < end;  // uniform
        FilterTile dn = d;
        if (more) {
            dn = desc(t_next);
            load_tile(dn);
        }
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            const uint32_t o = __builtin_amdgcn_readlane(inc - c, it * NW + wid);
            if ((pass >> it) & 1u) stage[par * T + o + rank[it]] = k[it];
        }
        __syncthreads();
        t_next = __builtin_amdgcn_readfirstlane(s_next[0]);
        if (last_n) write_out();
        last_n = total;
        last_key = d.okey;
        last_val = d.oval;
        last_cap = d.out_cap;
        d = dn;
        par ^= 1u;
        if (!more) break;
    }
    if (last_n) {  // uniform: the last tile
        __syncthreads();  // s_base may still be read for the tile before
        if (threadIdx.x == 0) *s_base = base;
        __syncthreads();
        write_out();
    }
    return bad;
}

// ---------------------------------------------------------------- build + probe of one work item
// The build side's chunk (bn <= CAP tuples) is counting-sorted into an LDS
// table by the hash bits below the radix bits (up to two buckets per build
// tuple): bst[t] is the first slot of bucket t (bst[nbk] = bn), hkey[] holds the
// keys bucket by bucket and hidx[] their row in the chunk (8 bytes of LDS per
// build tuple).  A probe key reads its bucket's start and end, then scans a
// short contiguous run of keys: no pointer chasing.
// The probe side (pn keys) streams through in rounds of BLOCK*PITEMS keys (the
// next round is loaded while the current one is processed).  Each round counts
// its matches and block-scans the counts.  A round with at most STAGE rows
// stages them in LDS as (probe row, table slot) pairs, reserved together with
// those of the round before or after by one global atomic; the keys and values
// are loaded two rounds later, one or two rows per thread, and stored after the
// third round's count (stores by consecutive threads).  Larger rounds reserve and
// write from the lanes at once.  Both
// values of a row are read only for matches: the build side's from its
// (cache-resident) chunk, the probe side's from its slice.  Rows past out_cap
// are counted, not written.
template <int BLOCK, int CAP>
struct alignas(16) ProbeLds {
    static constexpr int STAGE = CAP / 8;  // rows of one round staged in LDS: one or two per thread
    // a round's rows, three rounds (first: short LDS offsets): probe-side row of the
    // round | table slot of the build tuple (its key and row) << 16
    uint32_t stage[3][STAGE];
    uint32_t hkey[CAP];        // keys by bucket (bucket counts while the table is built)
    uint16_t hidx[CAP];
    uint16_t bst[CAP + 2];     // bucket starts, CAP buckets at most
    uint32_t wtmp[BLOCK / WAVE + 1];
    unsigned long long s_base[3];  // reservations of staged rounds being stored
    unsigned long long s_direct;  // reservation of a round written from the lanes
};

// waves per SIMD of a probe kernel: 8192-tuple tables two to a CU, 4096-tuple ones four
constexpr int probe_waves(int block, int cap) { return block / WAVE * (cap == 8192 ? 2 : 4) / 4; }

// Probe phase timers (one accumulator per workgroup, kept by thread 0, in
// ticks of the constant-rate wall clock): fetching work items, clearing the
// table, building it, counting the rounds' matches (through the reservation),
// writing the rounds' rows.
enum { PT_ITEM = 0, PT_CLEAR, PT_BUILD, PT_COUNT, PT_WRITE, PT_N };

__device__ __forceinline__ uint64_t phase_clock() { return wall_clock64(); }

// thread 0 of a collecting workgroup: acc[ph] += now - mark, mark = now
template <bool COLLECT>
__device__ __forceinline__ void phase_tick(uint64_t* acc, uint64_t* mark, int ph)
{
    if (COLLECT && threadIdx.x == 0) {
        const uint64_t t = phase_clock();
        acc[ph] += t - *mark;
        *mark = t;
    }
}

// COLLECT: thread 0 adds the item's phase times to tacc[PT_CLEAR..PT_WRITE]
// (tmark: the time the item started; left at the item's end).
// WATCH: returns true, with nothing probed, when a bucket holds more than max_run
// build tuples (the same for all threads); false otherwise.
template <int BLOCK, int CAP, int PITEMS, bool COLLECT = false, bool WATCH = false>
__device__ __forceinline__ bool probe_item(ProbeLds<BLOCK, CAP>& L, const uint32_t* __restrict__ bkp,
                                           const uint32_t* __restrict__ bvp, int bn,
                                           const uint32_t* __restrict__ pkp, const uint32_t* __restrict__ pvp,
                                           uint32_t pn, bool build_r, int bits,
                                           uint64_t* __restrict__ out_count, uint64_t out_cap,
                                           uint32_t* __restrict__ o_key, uint32_t* __restrict__ o_rval,
                                           uint32_t* __restrict__ o_sval, uint64_t* tacc = nullptr,
                                           uint64_t* tmark = nullptr, uint32_t max_run = 0)
{
    constexpr int ROUND = BLOCK * PITEMS;
    constexpr int BPT = CAP / BLOCK;  // build tuples per thread
    constexpr int STAGE = ProbeLds<BLOCK, CAP>::STAGE;
    // a wave's mark in its round's row count (at most 16 waves, 2^27 rows)
    constexpr uint32_t DUPS = 1u << 27;
    static_assert((uint64_t)ROUND * CAP < DUPS && BLOCK / WAVE <= 16, "row count and waves' marks in one word");
    static_assert(CAP % BLOCK == 0 && CAP <= 32768, "bucket and rank pack into 16 bits each");
    if (pn == 0) return false;  // an empty slice (uniform)

    // table geometry: 2^tb buckets, about two per build tuple when the probe
    // side is at least as long as the build side (shorter runs per probe key:
    // 5-7% off the probe of sub-buckets with 1-4 times as many probe as build
    // tuples, against a threshold of 8 times), else one to two build tuples per
    // bucket (less table to clear and scan)
    int tb = 0;
    if (pn >= (uint32_t)bn) {
        while ((1 << tb) < 2 * bn && (1 << tb) < CAP) tb++;
    } else {
        while ((1 << (tb + 1)) < bn && (1 << (tb + 1)) <= CAP / 2) tb++;
    }
    const int nbk = 1 << tb;
    // bucket of a key: hash bits [32 - bits - tb, 32 - bits), just below the
    // radix bits (a field of width 0 is bucket 0)
    const uint32_t toff = (uint32_t)(32 - bits - tb);
    auto bucket = [&](uint32_t key) { return __builtin_amdgcn_ubfe(radix_hash(key), toff, (uint32_t)tb); };
    uint32_t* cnt = L.hkey;  // bucket counts until the keys are placed
    if (nbk >= 4) {
        for (int i = threadIdx.x * 4; i < nbk; i += BLOCK * 4) *(uint4*)&cnt[i] = make_uint4(0u, 0u, 0u, 0u);
    } else if (threadIdx.x < nbk) {
        cnt[threadIdx.x] = 0u;
    }
    if (WATCH && threadIdx.x == 0) L.s_direct = 0ull;  // here: whether a bucket is too long
    __syncthreads();
    phase_tick<COLLECT>(tacc, tmark, PT_CLEAR);
    // build: rank each tuple in its bucket, scan the counts, place;
    // bucket (< 2^15) and rank (< 2^16) of each build tuple, packed, then its slot
    uint32_t bkey[BPT], btr[BPT];
#pragma unroll
    for (int u = 0; u < BPT; u++) {
        const int i = u * BLOCK + threadIdx.x;
        bkey[u] = (i < bn) ? bkp[i] : 0u;
    }
#pragma unroll
    for (int u = 0; u < BPT; u++) {
        const int i = u * BLOCK + threadIdx.x;
        btr[u] = 0;
        if (i < bn) {
            const uint32_t t = bucket(bkey[u]);
            const uint32_t r = atomicAdd(&cnt[t], 1u);
            btr[u] = (r << 16) | t;
            if (WATCH && r == max_run) L.s_direct = 1ull;
        }
    }
    __syncthreads();
    if (WATCH && L.s_direct) return true;  // uniform
    {
        // exclusive scan of the counts into the bucket starts; a thread's run
        // of counts is a power of two, read and written four at a time from 4
        // counts on (16-byte reads, 8-byte writes of four 16-bit starts)
        const int per_t = (nbk + BLOCK - 1) / BLOCK;
        const int lo_t = min((int)threadIdx.x * per_t, nbk), hi_t = min(lo_t + per_t, nbk);
        uint32_t sum = 0;
        if (per_t >= 4) {
            for (int t = lo_t; t < hi_t; t += 4) {
                const uint4 q = *(const uint4*)&cnt[t];
                sum += q.x + q.y + q.z + q.w;
            }
        } else {
            for (int t = lo_t; t < hi_t; t++) sum += cnt[t];
        }
        uint32_t tot;
        uint32_t ex = block_exclusive_scan<BLOCK, uint32_t>(sum, L.wtmp, &tot);
        if (per_t >= 4) {
            for (int t = lo_t; t < hi_t; t += 4) {
                const uint4 q = *(const uint4*)&cnt[t];
                const uint32_t e1 = ex + q.x, e2 = e1 + q.y, e3 = e2 + q.z;
                *(uint2*)&L.bst[t] = make_uint2((ex & 0xFFFFu) | (e1 << 16), (e2 & 0xFFFFu) | (e3 << 16));
                ex = e3 + q.w;
            }
        } else {
            for (int t = lo_t; t < hi_t; t++) {
                L.bst[t] = (uint16_t)ex;
                ex += cnt[t];
            }
        }
        if (threadIdx.x == 0) L.bst[nbk] = (uint16_t)bn;
    }
    __syncthreads();
    // every tuple's bucket start is read before the first is placed (reads inside
    // the branches below would be waited for one by one)
#pragma unroll
    for (int u = 0; u < BPT; u++) btr[u] = (uint32_t)L.bst[btr[u] & 0xFFFFu] + (btr[u] >> 16);
#pragma unroll
    for (int u = 0; u < BPT; u++) {
        const int i = u * BLOCK + threadIdx.x;
        if (i < bn) {
            L.hkey[btr[u]] = bkey[u];
            L.hidx[btr[u]] = (uint16_t)i;
        }
    }
    __syncthreads();
    phase_tick<COLLECT>(tacc, tmark, PT_BUILD);

    // key loads clamped to the last key (pn >= 1): no branches around loads
    uint32_t nk[PITEMS];
#pragma unroll
    for (int it = 0; it < PITEMS; it++) nk[it] = pkp[min((uint32_t)it * BLOCK + threadIdx.x, pn - 1u)];
    // Rows are written three rounds late, with two barriers per round (those of the
    // count scan): round r stages the (probe row, table slot) pairs of its matches in
    // stage[r % 3]; round r + 2 loads the key and values of rows tid, tid + BLOCK, ...;
    // round r + 3 stores them after its count, at the place thread 0 published before
    // that round's scan.  The scan barriers of the rounds between separate every LDS
    // write from the reads of the same slot.  No wait for a reservation or a value
    // load is on a round's path.
    // One atomic reserves the rows of two rounds (an odd one and the one before): the
    // chip does about 70 atomics on one address per us, and one per round of 5120 keys
    // (512 threads of 10 keys) was as many (640M x 640M: 125K in 1.94 ms; rounds of 4096
    // keys took 2.24 ms, of 6144 keys 1.76).  One per two rounds: 1.69 ms, and 16M x 16M 100
    // -> 93 us; 1024 threads of 4 keys: 1.56 ms.
    constexpr int NR = STAGE / BLOCK;
    uint32_t wk[NR], wp[NR], wb[NR];  // loaded rows: key, probe / build value
    uint32_t n_loaded = 0;          // rows in the registers, stored this round (uniform)
    uint32_t n_last = 0, n_prev = 0;  // rows staged last round and in the one before (uniform)
    // thread 0: the reservations of the loaded rows and of those of the pairs of
    // rounds that the last two belong to; a pair's second round lies behind its first
    unsigned long long sb_loaded = 0, sb_pair = 0;
    uint32_t off_loaded = 0, off_prev = 0, off_last = 0;
    uint32_t r3 = 0;                // round number mod 3
    bool odd = false;               // of the round
    // The key and build row come from the table (LDS), the values from global
    // memory.  The four loads are issued in every round, also where nothing is
    // staged (row 0 of the probe side and table slot 0, unused): the loads in
    // flight at the top of a round are then the same on every path (the next
    // keys, then these four), so waiting for the keys never waits for these.
    auto load_rows = [&](uint32_t n, uint32_t buf, uint32_t base, uint32_t* wk, uint32_t* wp, uint32_t* wb) {
        uint32_t p[NR], q[NR], b[NR];
#pragma unroll
        for (int u = 0; u < NR; u++) {
            p[u] = q[u] = 0;
            if (n) {  // uniform; rows tid, tid + BLOCK, clamped to the last row
                const uint32_t j = min((uint32_t)(u * BLOCK) + threadIdx.x, n - 1u);
                const uint32_t x = L.stage[buf][j];
                p[u] = base + (x & 0xFFFFu);
                q[u] = x >> 16;
            }
        }
#pragma unroll
        for (int u = 0; u < NR; u++) {
            wk[u] = L.hkey[q[u]];
            b[u] = L.hidx[q[u]];
            // per-lane rows: vector loads on every path (a known row 0 would become
            // a scalar load, which the vector load counter does not see)
            asm volatile("" : "+v"(p[u]), "+v"(b[u]));
        }
#pragma unroll
        for (int u = 0; u < NR; u++) wp[u] = pvp[p[u]];
#pragma unroll
        for (int u = 0; u < NR; u++) wb[u] = bvp[b[u]];
    };
    auto flush = [&](uint32_t n, uint32_t slot, const uint32_t* wk, const uint32_t* wp, const uint32_t* wb) {  // after a barrier that published L.s_base[slot]
        const uint64_t sb = uniform_u64(L.s_base[slot]);
        const uint32_t nw = sb >= out_cap ? 0u : (uint32_t)min<uint64_t>(n, out_cap - sb);
#pragma unroll
        for (int u = 0; u < NR; u++) {
            const uint32_t j = (uint32_t)(u * BLOCK) + threadIdx.x;
            if (j < nw) {
                o_key[sb + j] = wk[u];
                o_rval[sb + j] = build_r ? wb[u] : wp[u];
                o_sval[sb + j] = build_r ? wp[u] : wb[u];
            }
        }
    };
    load_rows(0, 0, 0, wk, wp, wb);
    for (uint32_t base = 0; base < pn; base += ROUND, r3 = r3 == 2u ? 0u : r3 + 1u, odd = !odd) {
        uint32_t kk[PITEMS], qs[PITEMS], qe[PITEMS];
#pragma unroll
        for (int it = 0; it < PITEMS; it++) kk[it] = nk[it];
        // the next round's keys, issued before this round's value loads so that
        // the next round's wait for them does not cover those; clamped, and
        // issued in the last round too, so that every round has the same loads
        // in flight (the compiler's waits then count past them)
#pragma unroll
        for (int it = 0; it < PITEMS; it++)
            nk[it] = pkp[min(base + ROUND + (uint32_t)it * BLOCK + threadIdx.x, pn - 1u)];
#pragma unroll
        for (int it = 0; it < PITEMS; it++) {
            // two 16-bit reads: one 32-bit read at a 2-byte aligned address is
            // slower on this LDS than the pair (t + 1 <= nbk)
            const uint32_t t = bucket(kk[it]);
            qs[it] = L.bst[t];
            qe[it] = L.bst[t + 1];
        }
        if (base + ROUND > pn) {  // last round: keys past pn match nothing
#pragma unroll
            for (int it = 0; it < PITEMS; it++)
                if (base + (uint32_t)it * BLOCK + threadIdx.x >= pn) qe[it] = qs[it];
        }
        // count the matches of every key and note its first matching slot q0
        // (the run is scanned downwards, so the last match seen is the first)
        uint32_t c = 0, hitmask = 0, multi = 0, qm[PITEMS];  // first match | run end << 16
#pragma unroll
        for (int it = 0; it < PITEMS; it++) {
            uint32_t m = 0, f = 0;
            for (uint32_t q = qe[it]; q > qs[it];) {
                q--;
                const bool e = L.hkey[q] == kk[it];
                f = e ? q : f;
                m += e;
            }
            qm[it] = f | (qe[it] << 16);
            c += m;
            hitmask |= (m ? 1u : 0u) << it;
            multi |= (m > 1 ? 1u : 0u) << it;
        }
        // the place of the rows stored this round (the slot's last reader was the
        // store three rounds ago)
        if (threadIdx.x == 0 && n_loaded) L.s_base[r3] = sb_loaded + off_loaded;
        uint32_t total;
        uint32_t pre = block_exclusive_scan<BLOCK, uint32_t>(c, L.wtmp, &total, __ballot(multi != 0u) ? DUPS : 0u);
        pre &= DUPS - 1u;
        const bool dups = total >= DUPS;  // uniform: some key of the round has several matches
        total &= DUPS - 1u;
        phase_tick<COLLECT>(tacc, tmark, PT_COUNT);
        if (n_loaded) flush(n_loaded, r3, wk, wp, wb);
        // the rows of the round before the last into the registers (stage[r3 + 1 mod 3])
        load_rows(n_prev, r3 == 2u ? 0u : r3 + 1u, base - 2u * ROUND, wk, wp, wb);
        const bool wrote = n_loaded != 0u;
        n_loaded = n_prev;
        sb_loaded = sb_pair;
        off_loaded = off_prev;
        n_prev = n_last;
        off_prev = off_last;
        const bool large = total > (uint32_t)STAGE;  // uniform
        n_last = large ? 0u : total;
        off_last = odd ? n_prev : 0u;
        // this round's rows, and those of the round before where it opened a pair
        const uint32_t res = n_last + off_last;
        const bool last = pn - base <= (uint32_t)ROUND;
        if (threadIdx.x == 0 && (odd || last)) {
            // (a last round without a second: the round before belongs to the pair before)
            if (last && !odd) L.s_base[r3 == 0u ? 2u : r3 - 1u] = sb_pair + off_prev;
            if (res) sb_pair = atomicAdd((unsigned long long*)out_count, (unsigned long long)res);
        }
        if (total == 0) {  // uniform
            if (wrote) phase_tick<COLLECT>(tacc, tmark, PT_WRITE);
            continue;
        }
        if (!large) {
            uint32_t w = pre;
            uint32_t* const st = L.stage[r3];
#pragma unroll
            for (int it = 0; it < PITEMS; it++) {
                if (hitmask & (1u << it)) {
                    const uint32_t prow = (uint32_t)it * BLOCK + threadIdx.x;
                    st[w++] = prow | qm[it] << 16;
                    if (multi & (1u << it)) {
                        for (uint32_t q = (qm[it] & 0xFFFFu) + 1; q < qm[it] >> 16; q++)
                            if (L.hkey[q] == kk[it]) st[w++] = prow | q << 16;
                    }
                }
            }
            phase_tick<COLLECT>(tacc, tmark, PT_WRITE);
            continue;
        }
        // a round with more rows than the stage: every wave writes its own rows
        // (consecutive places from its first lane's prefix), after the reservation.
        // Bound by the latency of the value loads and by partly filled stores: with
        // every lane writing its own rows one match after the other, 6001 x 20M rows
        // took 0.29 ms in the direct join, now 0.16, and the probe of 9M x 24M with
        // four copies of each key (19.2M rows) 434 us, now 337.  The first values are
        // loaded while thread 0 waits for the reservation: 6001 x 20M 159 -> 149 us, 12M x
        // 50M with every tuple matching 461 -> 428.  Waves with duplicate matches write in
        // another form than waves without; a barrier only stands where the whole workgroup
        // goes the same way (dups), and a round without any keeps its loads ahead of it (one
        // barrier before a branch per wave, loads under that branch: 6001 x 20M 158 us, 12M x
        // 50M 455 against 151 and 418 so).
        unsigned long long sd = 0;
        if (threadIdx.x == 0) sd = atomicAdd((unsigned long long*)out_count, (unsigned long long)total);
        // rows that fit from place w on (uniform)
        auto room = [&](uint64_t w) { return w >= out_cap ? 0u : (uint32_t)min<uint64_t>(out_cap - w, 4u * WAVE); };
        // One row per matching key: key group by key group, so that the lanes of a
        // store write consecutive rows (in lane order a lane's keys would lie up to
        // PITEMS rows apart); the values of HALF groups in flight together (of all
        // groups: spills).
        constexpr int HALF = (PITEMS + 1) / 2;
        uint32_t pv[HALF], bv[HALF];
        auto load_values = [&](int h) {
#pragma unroll
            for (int u = 0; u < HALF; u++) {
                if (h + u >= PITEMS) continue;
                const bool hit = (hitmask >> (h + u)) & 1u;
                pv[u] = pvp[hit ? base + (uint32_t)(h + u) * BLOCK + threadIdx.x : 0u];
                bv[u] = bvp[L.hidx[qm[h + u] & 0xFFFFu]];
            }
        };
        auto write_single = [&](uint64_t w) {  // the values of the first HALF groups are loaded
#pragma unroll
            for (int h = 0; h < PITEMS; h += HALF) {
                if (h) {
                    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the stores of the groups before
                    load_values(h);
                }
#pragma unroll
                for (int u = 0; u < HALF; u++) {
                    if (h + u >= PITEMS) continue;
                    const bool hit = (hitmask >> (h + u)) & 1u;
                    const uint64_t m = __ballot(hit);
                    const uint64_t d = w + lanes_below(m);
                    if (hit && d < out_cap) {
                        o_key[d] = kk[h + u];
                        o_rval[d] = build_r ? bv[u] : pv[u];
                        o_sval[d] = build_r ? pv[u] : bv[u];
                    }
                    w += (uint32_t)__popcll(m);
                }
            }
        };
        if (!dups) {  // no key of the round has several matches (the same for all waves)
            load_values(0);  // under way while thread 0 waits for the reservation
            if (threadIdx.x == 0) L.s_direct = sd;
            __syncthreads();
            write_single(uniform_u64(L.s_direct + pre));
            phase_tick<COLLECT>(tacc, tmark, PT_WRITE);
            continue;
        }
        if (threadIdx.x == 0) L.s_direct = sd;
        __syncthreads();
        uint64_t w = uniform_u64(L.s_direct + pre);
        if (w >= out_cap) {
            // all of the wave's rows are past the capacity: counted, no more (7M x 7M with ten
            // rows per S tuple and room for one: 1640 -> 276 us)
        } else if (__ballot(multi != 0u) == 0ull) {  // this wave has none
            load_values(0);
            write_single(w);
        } else {
            // duplicate build keys: the wave's rows go through its share of the
            // round's stage (free: stage[r3] was last read a round ago), so the
            // values of all its rows are in flight instead of one per match of a lane.
            // Where a lane has a run of more than DEEP slots the whole wave reads the runs, one
            // after the other: with every lane adding its own matches few lanes are busy in a
            // window (3000 x 3000 with 50 copies of each key 553 us, now 99; 1M x 1.5M 1310 ->
            // 358), with short runs they are the faster ones (by the lanes / by the wave, 37K x
            // 394K with some 10 copies in a chunk 217 / 278 us, 50K x 227K 118 / 150).
            constexpr uint32_t DEEP = 24;
            constexpr uint32_t FIFO = STAGE / (BLOCK / WAVE);
            static_assert(FIFO == 2 * WAVE || FIFO == WAVE, "one or two rows per lane");
            const uint32_t lane = lane_id();
            uint32_t* fifo = &L.stage[r3][threadIdx.x / WAVE * FIFO];
            uint32_t n = 0;  // rows in the wave's FIFO (uniform)
            auto drain = [&]() {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                constexpr int NF = FIFO / WAVE;
                uint32_t k[NF], fp[NF], fb[NF];
#pragma unroll
                for (int u = 0; u < NF; u++) {
                    const uint32_t j = min(lane + u * WAVE, n - 1u);
                    const uint32_t x = fifo[j];
                    k[u] = L.hkey[x >> 16];
                    fp[u] = pvp[base + (x & 0xFFFFu)];
                    fb[u] = bvp[L.hidx[x >> 16]];
                }
                const uint32_t nw = min(n, room(w));
#pragma unroll
                for (int u = 0; u < NF; u++) {
                    const uint32_t j = lane + u * WAVE;
                    if (j < nw) {
                        (o_key + w)[j] = k[u];
                        (o_rval + w)[j] = build_r ? fb[u] : fp[u];
                        (o_sval + w)[j] = build_r ? fp[u] : fb[u];
                    }
                }
                w += n;
                n = 0;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            };
            uint32_t longest = 0;
#pragma unroll
            for (int it = 0; it < PITEMS; it++)
                if ((multi >> it) & 1u) longest = max(longest, (qm[it] >> 16) - (qm[it] & 0xFFFFu));
            if (__ballot(longest > DEEP) == 0ull) {
#pragma unroll
                for (int it = 0; it < PITEMS; it++) {
                    // this key's matches, places in the wave by a scan
                    const uint32_t prow = (uint32_t)it * BLOCK + threadIdx.x, qend = qm[it] >> 16;
                    uint32_t q = qm[it] & 0xFFFFu;
                    uint32_t left = (hitmask >> it) & 1u;
                    if ((multi >> it) & 1u)
                        for (uint32_t x = q + 1; x < qend; x++) left += L.hkey[x] == kk[it];
                    const uint32_t inc = wave_inclusive_scan<uint32_t>(left);
                    uint32_t pos = inc - left;  // of this lane's next row
                    const uint32_t rows = __builtin_amdgcn_readlane(inc, WAVE - 1);
                    // the FIFO takes the rows in windows of its free room
                    for (uint32_t w0 = 0; w0 < rows;) {
                        const uint32_t take = min(FIFO - n, rows - w0);
                        while (left && pos < w0 + take) {
                            fifo[n + pos - w0] = prow | q << 16;
                            pos++;
                            if (--left)
                                while (L.hkey[++q] != kk[it]) {}
                        }
                        n += take;
                        w0 += take;
                        if (n == FIFO) drain();
                    }
                }
            } else {
                // the wave reads one run after the other, 64 slots at a time
#pragma unroll 1
                for (int it = 0; it < PITEMS && w < out_cap; it++) {
                    uint32_t mine = kk[0], run = qm[0];
#pragma unroll
                    for (int u = 1; u < PITEMS; u++) {
                        mine = it == u ? kk[u] : mine;
                        run = it == u ? qm[u] : run;
                    }
                    for (uint64_t todo = __ballot((hitmask >> it) & 1u); todo && w < out_cap; todo &= todo - 1ull) {
                        const int l = __builtin_ctzll(todo);
                        const uint32_t key = __builtin_amdgcn_readlane(mine, l);
                        const uint32_t q0 = __builtin_amdgcn_readlane(run, l), q1 = q0 >> 16;
                        const uint32_t row = (uint32_t)it * BLOCK + (threadIdx.x & ~(WAVE - 1u)) + (uint32_t)l;
                        for (uint32_t x = q0 & 0xFFFFu; x < q1; x += WAVE) {
                            const uint32_t slot = x + lane;
                            const bool hit = slot < q1 && L.hkey[min(slot, q1 - 1u)] == key;
                            const uint64_t m = __ballot(hit);
                            const uint32_t cnt = (uint32_t)__popcll(m), take = min(FIFO - n, cnt), at = lanes_below(m);
                            if (hit && at < take) fifo[n + at] = row | slot << 16;
                            n += take;
                            if (n == FIFO) {
                                drain();
                                if (hit && at >= take) fifo[at - take] = row | slot << 16;
                                n = cnt - take;
                            }
                        }
                    }
                }
            }
            if (n) drain();
        }
        // L.s_direct is rewritten only after the next round's scan barriers
        phase_tick<COLLECT>(tacc, tmark, PT_WRITE);
    }
    // the rows still in flight: those in the registers and those staged by the last
    // two rounds (r3: the number of rounds mod 3)
    if (n_loaded || n_prev || n_last) {  // uniform
        const uint32_t s1 = r3 == 2u ? 0u : r3 + 1u, s2 = 3u - r3 - s1;  // stages of the last but one, the last
        const uint32_t base1 = (pn - 1u) / ROUND * ROUND;  // the last round's
        __syncthreads();  // the last round's rows are staged, its store has read s_base
        // the values are under way while thread 0 waits for the reservation
        uint32_t xk[NR], xp[NR], xb[NR], yk[NR], yp[NR], yb[NR];
        if (n_prev) load_rows(n_prev, s1, base1 - ROUND, xk, xp, xb);
        if (n_last) load_rows(n_last, s2, base1, yk, yp, yb);
        if (threadIdx.x == 0) {
            if (n_loaded) L.s_base[r3] = sb_loaded + off_loaded;
            // (odd: of the round after the last)
            if (n_prev && !odd) L.s_base[s1] = sb_pair + off_prev;
            if (n_last) L.s_base[s2] = sb_pair + off_last;
        }
        __syncthreads();
        if (n_loaded) flush(n_loaded, r3, wk, wp, wb);
        if (n_prev) flush(n_prev, s1, xk, xp, xb);
        if (n_last) flush(n_last, s2, yk, yp, yb);
        phase_tick<COLLECT>(tacc, tmark, PT_WRITE);
    }
    // the caller synchronises before the next item rebuilds the table
    return false;
}

// Work-item split of one sub-bucket (vlsplit).  A sub-bucket whose build side
// (build_from_r) fits one LDS tile and whose probe side fits one slice is
// "regular": one work item, indexed by the sub-bucket itself.  Larger ones are
// split: the build side into ceil(nb / tile) chunks, the probe side into
// min(ceil(np / slice), max_slices) slices, one explicit item per (chunk, slice).
__device__ __forceinline__ uint32_t plan_items(uint64_t nr, uint64_t ns, uint32_t tile, uint32_t slice,
                                               uint32_t max_slices, uint32_t& chunks, uint32_t& slices)
{
    chunks = slices = 0;
    if (nr == 0 || ns == 0) return 0;
    const bool br = build_from_r(nr, ns, tile);
    const uint64_t nb = br ? nr : ns, np = br ? ns : nr;
    if (nb <= tile && np <= slice) return 0;
    chunks = (uint32_t)((nb + tile - 1) / tile);
    slices = (uint32_t)min<uint64_t>((np + slice - 1) / slice, max_slices);
    return chunks * slices;
}

}  // namespace bj
