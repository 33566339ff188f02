// bj_kernels.hip -- gfx950 kernels of the radix hash join, and their launchers.
//
// Pipeline (one GPU; all integer, all exact):
//   R:  k_hist -> k_cols -> k_scatter(pass 1, sub-bucket starts) -> k_scatter(pass 2)
//   BF: k_bloom_build (one workgroup per filter segment, built in LDS)
//   S:  bf_stage 2: k_hist + pass 1 of S, then k_filter_l1 (per first-level
//       bucket, XCD-aware, filter slice L2-resident) places the survivors;
//       bf_stage 1: k_bloom_prefilter (S -> S') then the two-level partition
//   J:  k_plan (vlsplit work items; in S's second pass where that is last) ->
//       k_probe (persistent; LDS hash table on the build side, stream the other side)
//   Below 32M tuples per side one launch takes R and S together (Sides).
//
// Reference counterparts (Chanho-LEE-SNU/BRIG-Join):
//   k_hist / k_cols                  gpu_run_hist_for_both, gpu_make_simple_prefix,
//                                    gpu_run_hist_second_pass
//                                    (src/kernel_functions.cu:22-90, 461-492, 163-207)
//   k_scatter                        gpu_make_sorted_table_for_both, gpu_build_table_second_pass
//                                    (src/kernel_functions.cu:95-133, 210-281)
//   k_bloom_build                    insertKernelPartitioned (src/bloom.cu:698-722)
//   k_bloom_prefilter, k_filter_l1   queryAndCompactKernelPartitioned (src/bloom.cu:725-773)
//   k_probe                          gpu_probe_with_second_pass / gpu_fused_probe_transfer
//                                    local part (src/kernel_functions.cu:294-457, 612-789)
#include "bj_kernels.h"
#include "bj_device.h"
#include "bj_tiles.h"

#include <math.h>

#include <algorithm>

namespace bj {

// ============================================================== utilities
__global__ void k_zero_u64(uint64_t* __restrict__ p, int n)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0ull;
}

__global__ void k_add2_u64(const uint64_t* __restrict__ a, const uint64_t* __restrict__ b, uint64_t* __restrict__ acc)
{
    if (threadIdx.x == 0) {
        acc[0] += *a;
        acc[1] += *b;
    }
}

// ============================================================== generator
__global__ void k_gen_r(uint32_t* __restrict__ key, uint32_t* __restrict__ val, uint64_t n,
                        PermKeys K)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x) {
        key[i] = gen_r_key((uint32_t)i, K);
        if (val) val[i] = (uint32_t)i;
    }
}

// Zipf(s) rank in [1, n] by inverting the generalised harmonic number
// H_s(r) = sum_{i<=r} i^-s with an Euler-Maclaurin approximation; small ranks
// are summed exactly.
__device__ double zipf_H(double r, double s)
{
    if (r < 16.0) {
        double acc = 0.0;
        for (int i = 1; i <= (int)r; i++) acc += pow((double)i, -s);
        return acc;
    }
    // exact sum to 15, then the integral tail with end corrections
    double acc = 0.0;
    for (int i = 1; i <= 15; i++) acc += pow(15.0 + 1.0 - i, -s);  // sum 1..15
    const double a = 15.0;
    double tail;
    if (fabs(s - 1.0) < 1e-12) tail = log(r) - log(a);
    else tail = (pow(r, 1.0 - s) - pow(a, 1.0 - s)) / (1.0 - s);
    tail += 0.5 * (pow(r, -s) - pow(a, -s));
    tail -= s / 12.0 * (pow(r, -s - 1.0) - pow(a, -s - 1.0));
    return acc + tail;
}

__device__ uint32_t zipf_rank(double u, uint32_t n, double s, double Hn)
{
    const double t = u * Hn;
    // initial guess from the continuous inverse
    double g;
    if (fabs(s - 1.0) < 1e-12) g = exp(t - 0.5772156649015329);
    else g = pow(fmax(1e-300, (1.0 - s) * (t - 0.5772156649015329) + 1.0), 1.0 / (1.0 - s));
    double r = fmin(fmax(floor(g), 1.0), (double)n);
    // walk to the smallest r with H(r) >= t (a few steps)
    for (int it = 0; it < 64 && r < (double)n && zipf_H(r, s) < t; it++) r += 1.0;
    for (int it = 0; it < 64 && r > 1.0 && zipf_H(r - 1.0, s) >= t; it++) r -= 1.0;
    return (uint32_t)r;
}

__global__ void k_gen_s(uint32_t* __restrict__ key, uint32_t* __restrict__ val, uint64_t n_s,
                        uint64_t n_r, uint64_t m_s, int L, PermKeys KR, PermKeys KP,
                        PermKeys KN, uint32_t useed, double zipf_s, double zipf_Hn,
                        uint32_t zseed)
{
    for (uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n_s;
         j += (uint64_t)gridDim.x * blockDim.x) {
        uint32_t p = permw((uint32_t)j, L, KP);
        while ((uint64_t)p >= n_s) p = permw(p, L, KP);
        uint32_t k;
        if ((uint64_t)p < m_s) {
            uint32_t u;
            if (zipf_s > 0.0) {
                const uint32_t a = lowbias32((uint32_t)j ^ zseed);
                const uint32_t b = lowbias32(a ^ 0x68E31DA4u);
                const double uu = ((double)(((uint64_t)a << 21) ^ (uint64_t)(b >> 11)) + 0.5) *
                                  (1.0 / 9007199254740992.0);
                u = zipf_rank(uu, (uint32_t)n_r, zipf_s, zipf_Hn) - 1u;
            } else {
                u = (uint32_t)(((uint64_t)lowbias32((uint32_t)j ^ useed) * n_r) >> 32);
            }
            k = gen_r_key(u, KR);
        } else {
            k = 0x80000000u | permw((uint32_t)j, 31, KN);
        }
        key[j] = k;
        if (val) val[j] = (uint32_t)j;
    }
}

// The reference datagen's distribution (datagen/gen_dataset.cpp:172-220) on the
// device.  Before its shuffle, R is [0, k) then k + (i - k) mod (2^31 - 1 - k),
// and S is a run of matching keys (0, 1, ...) and S-only keys R + j mod
// (2^31 - 1 - R) per region; the reference shuffles each region with
// Fisher-Yates, here position i of a region takes the unshuffled element at a
// keyed permutation of i (cycle-walked onto the region), so each region holds
// the same key multiset in another random order.
__device__ __forceinline__ uint32_t perm_onto(uint64_t i, uint64_t n, int L, const PermKeys& K)
{
    uint32_t p = permw((uint32_t)i, L, K);
    while ((uint64_t)p >= n) p = permw(p, L, K);
    return p;
}

__global__ void k_gen_refdist_r(uint32_t* __restrict__ key, uint64_t n, uint64_t k, int L, PermKeys K)
{
    const uint64_t r_only = 0x7FFFFFFFull - k;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t t = perm_onto(i, n, L, K);
        key[i] = (uint32_t)(t < k ? t : k + (t - k) % r_only);
    }
}

// One region of S: positions [0, n) of key (already offset), the first m
// unshuffled elements matching keys mc0, mc0 + 1, ..., the rest S-only keys
// n_r + (sj0 + j) mod (2^31 - 1 - n_r).
__global__ void k_gen_refdist_s(uint32_t* __restrict__ key, uint64_t n, uint64_t m, uint64_t mc0,
                                uint64_t sj0, uint64_t n_r, int L, PermKeys K)
{
    const uint64_t s_only = 0x7FFFFFFFull - n_r;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t t = perm_onto(i, n, L, K);
        key[i] = (uint32_t)(t < m ? mc0 + t : n_r + (sj0 + (t - m)) % s_only);
    }
}

__global__ void k_zipf_Hn(double* out, uint32_t n, double s)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) out[0] = zipf_H((double)n, s);
}

// ============================================================== partition
// The launches of a partition take one side (R or S) or both: workgroups
// [0, na) belong to side a, the rest to side b.  Joins below some tens of
// millions of tuples per side spend as long between launches as in them.
struct Sides {
    PartSide a, b;
    int na;  // workgroups of side a
};
__device__ __forceinline__ PartSide side_of(const Sides& S, uint32_t& x)
{
    if ((int)x < S.na) return S.a;
    x -= (uint32_t)S.na;
    return S.b;
}
__device__ __forceinline__ uint64_t side_len(const PartSide& s) { return s.n_dev ? *s.n_dev : s.n; }

// Per-workgroup histogram of the full radix (2^bits bins) over a contiguous
// chunk.  Chunking: chunk = ceil(n / G), workgroup g owns [g*chunk, (g+1)*chunk).
// k_scatter pass 1 uses exactly the same chunks, so the per-(bucket, group)
// offsets derived from these histograms place every tuple without atomics.
// Also clears what the later launches accumulate into: the bin totals, the
// join's counters (ctr, in the first launch of a join) and zero32.
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_hist(Sides S, uint64_t* __restrict__ ctr, int n_ctr,
                                                uint32_t* __restrict__ zero32, int n_zero32)
{
    extern __shared__ uint32_t h[];
    if (ctr && blockIdx.x == 0 && (int)threadIdx.x < n_ctr) ctr[threadIdx.x] = 0ull;
    if (zero32)
        for (int i = blockIdx.x * BLOCK + threadIdx.x; i < n_zero32; i += gridDim.x * BLOCK) zero32[i] = 0u;
    uint32_t x = blockIdx.x;
    const PartSide s = side_of(S, x);
    const int nbins = 1 << s.bits;
    for (int i = threadIdx.x; i < nbins; i += BLOCK) h[i] = 0u;
    for (int i = x * BLOCK + threadIdx.x; i < nbins; i += s.G * BLOCK) s.totals[i] = 0u;
    __syncthreads();
    const uint64_t n = side_len(s);
    const uint64_t chunk = (n + (uint64_t)s.G - 1) / (uint64_t)s.G;
    const uint64_t lo = min((uint64_t)x * chunk, n);
    const uint64_t hi = min(lo + chunk, n);
    hist_range<BLOCK>(s.key, lo, hi, 32 - s.bits, h);
    __syncthreads();
    uint32_t* dst = s.part + (size_t)x * nbins;
    for (int b = threadIdx.x; b < nbins; b += BLOCK) dst[b] = h[b];
    // this chunk's first-level counts (two levels): thread b1 sums its 2^b2
    // bins from LDS, starting at a rotated offset so that threads hit different
    // banks at each step
    const int b2 = s.bits - s.p1;
    if (b2 > 0) {
        const int P1 = 1 << s.p1, seg = 1 << b2;
        for (int b1 = threadIdx.x; b1 < P1; b1 += BLOCK) {
            const uint32_t* hb = h + ((size_t)b1 << b2);
            uint32_t sum = 0;
            for (int j = 0; j < seg; j++) sum += hb[(j + b1) & (seg - 1)];
            s.l1h[(size_t)x * P1 + b1] = sum;
        }
    }
}

// k_cols, the column sums of a side's histograms, in two kinds of workgroups:
// - [0, ncb * W): column block cb (1024 bins) of the per-chunk histograms summed
//   over chunk group w (chunks [w*G/W, (w+1)*G/W)) into colsum[w][b] and, by
//   atomics, into totals[b] (zeroed by k_hist);
// - then ceil(2^p1 / L1_COLS): a column scan of the first-level counts,
//   l1rel[g][b1] = sum_{g' < g} l1h[g'][b1] and the column's total l1tot[b1].  Each
//   workgroup owns 16 columns; 64 row ranges per column are summed, scanned by
//   one wave per column, then rescanned row by row (short row ranges keep the
//   serial chains short when there are few columns).
constexpr int L1_COLS = 16, L1_ROWS = 1024 / L1_COLS;
static_assert(L1_ROWS == WAVE && 1024 / WAVE == L1_COLS, "one wave scans one column");

__host__ __device__ __forceinline__ int cols_sum_wgs(const PartSide& s) { return ((1 << s.bits) + 1023) / 1024 * s.W; }
__host__ __device__ __forceinline__ int cols_wgs(const PartSide& s)
{
    return cols_sum_wgs(s) + ((1 << s.p1) + L1_COLS - 1) / L1_COLS;
}

__global__ __launch_bounds__(1024) void k_cols(Sides S)
{
    __shared__ uint32_t part_sum[L1_ROWS][L1_COLS + 1];
    uint32_t x = blockIdx.x;
    const PartSide s = side_of(S, x);
    const int nbins = 1 << s.bits, nsum = cols_sum_wgs(s);
    if ((int)x < nsum) {
        const int ncb = (nbins + 1023) / 1024;
        const int cb = (int)x % ncb, w = (int)x / ncb;
        const int c = cb * 1024 + threadIdx.x;
        const int g0 = (int)((int64_t)w * s.G / s.W), g1 = (int)((int64_t)(w + 1) * s.G / s.W);
        if (c < nbins) {
            uint32_t sum = 0;
#pragma unroll 8
            for (int g = g0; g < g1; g++) sum += s.part[(size_t)g * nbins + c];
            s.colsum[(size_t)w * nbins + c] = sum;
            if (sum) atomicAdd(&s.totals[c], sum);
        }
        return;
    }
    x -= (uint32_t)nsum;
    const int P1 = 1 << s.p1;
    const uint32_t* l1h = s.p1 < s.bits ? s.l1h : s.part;
    const int c = threadIdx.x % L1_COLS, r = threadIdx.x / L1_COLS;
    const int b1 = (int)x * L1_COLS + c;
    const int rows = (s.G + L1_ROWS - 1) / L1_ROWS;
    const int g0 = min(r * rows, s.G), g1 = min(g0 + rows, s.G);
    uint32_t sum = 0;
    if (b1 < P1)
        for (int g = g0; g < g1; g++) sum += l1h[(size_t)g * P1 + b1];
    part_sum[r][c] = sum;
    __syncthreads();
    {
        // wave w: column w, lane = row range (the branch is uniform per wave)
        const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
        const int col = (int)x * L1_COLS + w;
        if (col < P1) {
            const uint32_t v = part_sum[lane][w];
            const uint32_t inc = wave_inclusive_scan<uint32_t>(v);
            part_sum[lane][w] = inc - v;
            if (lane == WAVE - 1) s.l1tot[col] = inc;
        }
    }
    __syncthreads();
    if (b1 < P1) {
        uint32_t acc = part_sum[r][c];
        for (int g = g0; g < g1; g++) {
            s.l1rel[(size_t)g * P1 + b1] = acc;
            acc += l1h[(size_t)g * P1 + b1];
        }
    }
}

// One workgroup: exclusive scan of v[0, n) (n a power of two) into out[0, n], as
// a thread's run of max(1, n / BLOCK) entries, read twice (the second time from
// the cache), 16 bytes at a time from 4 entries on.  lds: BLOCK/64 + 1 words.
template <int BLOCK>
__device__ __forceinline__ void starts_block(const uint32_t* __restrict__ v, int n, uint64_t* __restrict__ out,
                                             uint64_t* lds)
{
    const int per = max(1, n / BLOCK);
    const int b0 = (int)threadIdx.x * per;
    uint64_t sum = 0;
    if (per >= 4) {
        for (int j = 0; j < per; j += 4) {
            const uint4 q = *(const uint4*)&v[b0 + j];
            sum += (uint64_t)q.x + q.y + q.z + q.w;
        }
    } else {
        for (int j = 0; j < per; j++)
            if (b0 + j < n) sum += v[b0 + j];
    }
    uint64_t tot;
    uint64_t ex = block_exclusive_scan<BLOCK, uint64_t>(sum, lds, &tot);
    if (per >= 4) {
        for (int j = 0; j < per; j += 4) {
            const uint4 q = *(const uint4*)&v[b0 + j];
            ulonglong2* o = (ulonglong2*)(out + b0 + j);
            const uint64_t e1 = ex + q.x, e2 = e1 + q.y, e3 = e2 + q.z;
            o[0] = make_ulonglong2(ex, e1);
            o[1] = make_ulonglong2(e2, e3);
            ex = e3 + q.w;
        }
    } else {
        for (int j = 0; j < per; j++)
            if (b0 + j < n) {
                out[b0 + j] = ex;
                ex += v[b0 + j];
            }
    }
    if (threadIdx.x == 0) out[n] = tot;
}

// ============================================================== scan (u32 -> u64 exclusive)
// Reduce-then-scan over n entries; out has n + 1 entries, out[n] = total.
constexpr int SCAN_BLOCK = 256;
constexpr int SCAN_ITEMS = 16;
constexpr int SCAN_TILE = SCAN_BLOCK * SCAN_ITEMS;

__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_reduce(const uint32_t* __restrict__ in,
                                                            uint64_t n, uint64_t* __restrict__ partial)
{
    __shared__ uint64_t wtmp[SCAN_BLOCK / WAVE + 1];
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE;
    uint64_t s = 0;
    for (int it = 0; it < SCAN_ITEMS; it++) {
        const uint64_t i = base + (uint64_t)it * SCAN_BLOCK + threadIdx.x;
        if (i < n) s += in[i];
    }
    uint64_t tot;
    block_exclusive_scan<SCAN_BLOCK, uint64_t>(s, wtmp, &tot);
    if (threadIdx.x == 0) partial[blockIdx.x] = tot;
}

// single workgroup: exclusive scan of the W partials in place (W <= 1024*64)
__global__ __launch_bounds__(1024) void k_scan_top(uint64_t* __restrict__ partial, int W)
{
    __shared__ uint64_t wtmp[1024 / WAVE + 1];
    const int per = (W + 1023) / 1024;
    const int lo = min((int)threadIdx.x * per, W);
    const int hi = min(lo + per, W);
    uint64_t s = 0;
    for (int i = lo; i < hi; i++) s += partial[i];
    uint64_t tot;
    uint64_t ex = block_exclusive_scan<1024, uint64_t>(s, wtmp, &tot);
    for (int i = lo; i < hi; i++) {
        const uint64_t c = partial[i];
        partial[i] = ex;
        ex += c;
    }
    if (threadIdx.x == 0) partial[W] = tot;
}

__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_down(const uint32_t* __restrict__ in, uint64_t n,
                                                          const uint64_t* __restrict__ partial,
                                                          uint64_t* __restrict__ out, int W)
{
    __shared__ uint64_t wtmp[SCAN_BLOCK / WAVE + 1];
    // each thread owns SCAN_ITEMS consecutive entries
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
    uint32_t v[SCAN_ITEMS];
    uint64_t s = 0;
#pragma unroll
    for (int it = 0; it < SCAN_ITEMS; it++) {
        const uint64_t i = base + it;
        v[it] = (i < n) ? in[i] : 0u;
        s += v[it];
    }
    uint64_t tot;
    uint64_t ex = block_exclusive_scan<SCAN_BLOCK, uint64_t>(s, wtmp, &tot) + partial[blockIdx.x];
#pragma unroll
    for (int it = 0; it < SCAN_ITEMS; it++) {
        const uint64_t i = base + it;
        if (i < n) out[i] = ex;
        ex += v[it];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) out[n] = partial[W];
}

// ============================================================== probe planning
// A sub-bucket whose build side (build_from_r: R when it fits one LDS tile,
// else the smaller side) fits one LDS tile and whose probe side fits one slice
// is "regular": one work item, indexed by the sub-bucket itself.
// Larger ones are split (vlsplit): the build side into ceil(nb / tile) chunks,
// the probe side into min(ceil(np / slice), max_slices) slices, one explicit
// work item per (chunk, slice).  Count, scan, fill: no contention, and the
// item buffer bound max_slices * (sum ceil(nb / tile)) always holds.
__device__ __forceinline__ void sb_sizes(const uint64_t* r_start, const uint64_t* s_start,
                                         const uint32_t* s_cnt, int sb, uint64_t& r0, uint64_t& nr,
                                         uint64_t& s0, uint64_t& ns)
{
    r0 = r_start[sb];
    nr = r_start[sb + 1] - r0;
    s0 = s_start[sb];
    ns = s_cnt ? (uint64_t)s_cnt[sb] : (s_start[sb + 1] - s0);
}

// One workgroup: every thread takes sub-buckets t, t + BLOCK, ... in groups of
// PG, counts their items, and a block scan per group places them.  lds: BLOCK/64
// + 1 words.  In a launch of its own it is latency-bound; where both sides end in
// a second scatter pass it runs in that launch, whose other workgroups do not
// need it.
template <int BLOCK>
__device__ void plan_block(const PlanArgs& A, uint64_t* lds)
{
    constexpr int PG = 8;
    const int nbins = 1 << A.bits;
    uint64_t base = 0;
    bool over = false;
    for (int sb0 = 0; sb0 < nbins; sb0 += BLOCK * PG) {
        uint32_t v[PG], sum = 0;
#pragma unroll
        for (int j = 0; j < PG; j++) {
            const int sb = sb0 + j * BLOCK + (int)threadIdx.x;
            v[j] = 0;
            if (sb < nbins) {
                uint64_t r0, nr, s0, ns;
                sb_sizes(A.r_start, A.s_start, A.s_cnt, sb, r0, nr, s0, ns);
                uint32_t c, sl;
                v[j] = plan_items(nr, ns, A.tile, A.slice, A.max_slices, c, sl);
            }
            sum += v[j];
        }
        uint64_t tot;
        uint64_t at = base + block_exclusive_scan<BLOCK, uint64_t>((uint64_t)sum, lds, &tot);
        base += tot;
        if (tot == 0) continue;  // uniform: no split sub-bucket in the group
#pragma unroll
        for (int j = 0; j < PG; j++) {
            if (v[j] == 0) continue;
            const int sb = sb0 + j * BLOCK + (int)threadIdx.x;
            uint64_t r0, nr, s0, ns;
            sb_sizes(A.r_start, A.s_start, A.s_cnt, sb, r0, nr, s0, ns);
            uint32_t chunks, slices;
            plan_items(nr, ns, A.tile, A.slice, A.max_slices, chunks, slices);
            if (at + v[j] > A.item_cap) {
                over = true;
            } else {
                for (uint32_t c = 0; c < chunks; c++)
                    for (uint32_t q = 0; q < slices; q++) {
                        HeavyItem it;
                        it.sb = (uint32_t)sb;
                        it.chunk = c;
                        it.slice = q;
                        it.nslices = slices;
                        A.items[at + (uint64_t)c * slices + q] = it;
                    }
            }
            at += v[j];
        }
    }
    if (threadIdx.x == 0) *A.n_items = base;
    if (over) atomicOr((unsigned long long*)A.err, 4ull);
}

template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_plan(PlanArgs A)
{
    __shared__ uint64_t lds[BLOCK / WAVE + 1];
    plan_block<BLOCK>(A, lds);
}

// ============================================================== scatter
// Write-combining scatter of one range (scatter_range, bj_tiles.h).  What a
// workgroup of a side owns:
//   pass 1 (p1 bits): workgroup 1 + g owns the same chunk as k_hist's group g;
//       bucket = h >> (32 - p1); cur[b] = the bucket's start (a scan of l1tot) +
//       l1rel[g][b].  Workgroup 0 meanwhile turns the bin totals into the
//       sub-bucket starts, which only later launches read.
//   pass 2 (bits - p1 bits): workgroup (b1, w) of the bucket's A owns the pass-1 output
//       of bucket b1 written by pass-1 groups [w*G/A, (w+1)*G/A); bucket = (h >> (32 -
//       bits)) & (2^(bits-p1) - 1); cur[b] = start[sb] + what the chunks before hold of
//       sb = (b1 << (bits-p1)) + b.  A follows the bucket's size (second_share).
// IPAIR / OPAIR: whole tuples in one array (TupleIn / TupleOut) on that side:
// pass 1 writes them unless it is the only pass, pass 2 (IPAIR) reads them.
// Writes are bounds-checked against the capacity and flag err on violation.
// plan.items not null: workgroup 0 of the launch plans the probe (plan_block).
// Occupancy targets: two 1024-thread workgroups per CU for the 4096-tuple tile,
// one for the 8192-tuple tile (launched one per CU), three 512-thread ones.
constexpr int sc_min_waves(int block, int items) { return block == 1024 ? (items == 4 ? 8 : 4) : 6; }

// Workgroups launched for a side's second pass.
static int second_wgs(const PartSide& s) { return s.shared2 ? s.shared2 : s.W2 << s.p1; }

// Bucket b1 of workgroup x of a side's second pass, its place w among the bucket's A
// workgroups; false: there is none.  With shared2 a bucket of nb tuples takes ceil(nb /
// per), at least one and at most W2, per being such that the sum stays within shared2;
// every wave finds its place by itself, lane l adding up 2^p1 / 64 buckets.
// W2 workgroups each would be many for the work below some 16M tuples (3M x 4.5M: 58 us
// with 1024 per side, 35 so), but a fixed smaller number leaves a hot key's bucket to those
// few (eight there: half of S equal 365 us, so 110).
__device__ __forceinline__ bool second_place(const PartSide& s, uint32_t x, int& b1, int& w, int& A)
{
    A = s.W2;
    b1 = (int)x / s.W2;
    w = (int)x % s.W2;
    if (s.shared2 == 0) return true;
    const int P1 = 1 << s.p1, b2 = s.bits - s.p1;
    const uint32_t room = (uint32_t)(s.shared2 - P1);
    const uint32_t per = max(1u, (uint32_t)((side_len(s) + room - 1u) / room));
    auto share = [&](int b) {
        const uint32_t nb = (uint32_t)(s.start[(uint64_t)(b + 1) << b2] - s.start[(uint64_t)b << b2]);
        return min((uint32_t)s.W2, max(1u, (nb + per - 1u) / per));
    };
    const int np = (P1 + WAVE - 1) / WAVE, q0 = (int)lane_id() * np;
    uint32_t sum = 0;
    for (int j = 0; j < np; j++)
        if (q0 + j < P1) sum += share(q0 + j);
    const uint32_t inc = wave_inclusive_scan<uint32_t>(sum);
    if (x >= __builtin_amdgcn_readlane(inc, WAVE - 1)) return false;
    const int l = __popcll(__ballot(inc <= x));  // the lane whose buckets x falls into
    uint32_t at = l ? __builtin_amdgcn_readlane(inc, l - 1) : 0u;
    for (b1 = l * np;; b1++) {  // ends: x lies below the sum of the lane's shares
        A = (int)share(b1);
        if (x < at + (uint32_t)A) break;
        at += (uint32_t)A;
    }
    w = (int)(x - at);
    return true;
}

template <int BLOCK, int ITEMS, bool IPAIR, bool OPAIR>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(sc_min_waves(BLOCK, ITEMS), 8))) void k_scatter(
    Sides S, PlanArgs plan, uint64_t* __restrict__ err)
{
    extern __shared__ uint64_t lds64[];
    uint32_t x = blockIdx.x;
    if (IPAIR && plan.items) {
        if (x == 0) {
            plan_block<BLOCK>(plan, lds64);
            return;
        }
        x--;
    }
    const PartSide s = side_of(S, x);
    const int b2 = s.bits - s.p1;
    const int nbk = IPAIR ? (1 << b2) : (1 << s.p1);
    const int shift = IPAIR ? (32 - s.bits) : (32 - s.p1);
    const int cs_log2 = scatter_carry_log2(nbk, ITEMS == 8 && BLOCK == 1024, OPAIR);
    const ScatterLds L = scatter_lds<BLOCK, ITEMS>(lds64, nbk, cs_log2);
    const int P1 = 1 << s.p1;
    uint64_t lo, hi;
    TupleIn<IPAIR> in;
    TupleOut<OPAIR> out;
    uint64_t cap;
    if constexpr (!IPAIR) {
        if (x == 0) {
            starts_block<BLOCK>(s.totals, 1 << s.bits, s.start, lds64);
            return;
        }
        const uint32_t g = x - 1u;
        const uint64_t n = side_len(s);
        const uint64_t chunk = (n + (uint64_t)s.G - 1) / (uint64_t)s.G;
        lo = min((uint64_t)g * chunk, n);
        hi = min(lo + chunk, n);
        // the buckets' starts: thread t scans buckets [t * per, (t + 1) * per)
        const int per = max(1, nbk / BLOCK), q0 = (int)threadIdx.x * per;
        uint32_t sum = 0, tot;
        for (int j = 0; j < per; j++)
            if (q0 + j < nbk) sum += s.l1tot[q0 + j];
        uint32_t ex = block_exclusive_scan<BLOCK, uint32_t>(sum, L.wtmp, &tot);
        for (int j = 0; j < per; j++)
            if (q0 + j < nbk) {
                L.cur[q0 + j] = (uint64_t)ex + s.l1rel[(size_t)g * P1 + q0 + j];
                ex += s.l1tot[q0 + j];
            }
        in = {s.key, s.val};
    } else {
        int b1, w, A;
        if (!second_place(s, x, b1, w, A)) return;
        const int g0 = (int)(((int64_t)w * s.G) / A), g1 = (int)(((int64_t)(w + 1) * s.G) / A);
        const uint64_t b_lo = s.start[(uint64_t)b1 << b2], b_hi = s.start[(uint64_t)(b1 + 1) << b2];
        lo = (g0 < s.G) ? b_lo + s.l1rel[(size_t)g0 * P1 + b1] : b_hi;
        hi = (g1 < s.G) ? b_lo + s.l1rel[(size_t)g1 * P1 + b1] : b_hi;
        // cursor of sub-bucket sb: its start plus what the earlier chunks hold of it, those
        // of the column sums' groups before chunk g0's and the others of that group
        const int v0 = (int)(((int64_t)(g0 + 1) * s.W2 - 1) / s.G), gs = (int)(((int64_t)v0 * s.G) / s.W2);
        // (2^b2 threads take every K-th row of them, and the next 2^b2 the rows beside)
        const uint64_t nbins = 1ull << s.bits;
        for (int b = threadIdx.x; b < nbk; b += BLOCK) L.cur[b] = s.start[((uint64_t)b1 << b2) + b];
        __syncthreads();
        const int K = max(1, BLOCK >> b2), k = (int)threadIdx.x >> b2;
        for (int b = threadIdx.x & (nbk - 1); b < nbk; b += BLOCK) {
            const uint32_t* row = s.colsum + ((size_t)b1 << b2) + b;
            uint32_t sum = 0;
#pragma unroll 4
            for (int v = k; v < v0; v += K) sum += row[(size_t)v * nbins];
            row = s.part + ((size_t)b1 << b2) + b;
#pragma unroll 4
            for (int g = gs + k; g < g0; g += K) sum += row[(size_t)g * nbins];
            if (sum) atomicAdd((unsigned long long*)&L.cur[b], (unsigned long long)sum);
        }
        in = {(const Tuple*)s.tmp};
    }
    if constexpr (OPAIR) {
        out = {(Tuple*)s.tmp};
        cap = s.tmp_cap;
    } else {
        out = {s.okey, s.oval};
        cap = s.out_cap;
    }
    // ranges are below 2^31 tuples
    const bool bad = scatter_range<BLOCK, ITEMS, IPAIR, OPAIR>(L, in.from(lo), (uint32_t)(hi - lo), nbk, shift,
                                                               (uint32_t)nbk - 1u, cs_log2, out, cap);
    if (bad) atomicOr((unsigned long long*)err, 1ull);
}

// ============================================================== Bloom build
// One workgroup per filter segment: zero the segment in LDS, OR in the block
// of every R key of the segment's sub-buckets (one 64-bit LDS atomic per key),
// write the segment once.
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_bloom_build(const uint32_t* __restrict__ rkey,
                                                       const uint64_t* __restrict__ r_start, int bits,
                                                       BloomGeom g, uint64_t* __restrict__ filter)
{
    extern __shared__ unsigned long long seg[];
    const uint32_t wps = g.wps;
    for (uint32_t i = threadIdx.x; i < wps; i += BLOCK) seg[i] = 0ull;
    __syncthreads();
    const uint64_t s = blockIdx.x;
    const int d = bits - g.seg_bits;
    const uint64_t lo = r_start[s << d], hi = r_start[(s + 1) << d];
    const uint64_t segbase = s * (uint64_t)wps;
    bloom_build_range<BLOCK>(rkey, lo, hi, g, segbase, seg);
    __syncthreads();
    uint64_t* dst = filter + segbase;
    for (uint32_t i = threadIdx.x; i < wps; i += BLOCK) dst[i] = seg[i];
}

// ============================================================== Bloom filter S -> S' (before partitioning)
// The reference's order (queryAndCompactKernelPartitioned): S is filtered
// before it is partitioned.  Used when the filter fits an XCD's L2, since each key
// probes a random filter block.  Grid-stride over tiles (filter_run).
template <int BLOCK, int ITEMS>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_bloom_prefilter(
    const uint32_t* __restrict__ skey, const uint32_t* __restrict__ sval, uint64_t n,
    const uint64_t* __restrict__ filter, BloomGeom g, uint32_t* __restrict__ okey,
    uint32_t* __restrict__ oval, uint64_t out_cap, uint64_t* __restrict__ count,
    uint64_t* __restrict__ err)
{
    constexpr int T = BLOCK * ITEMS;
    __shared__ Tuple stage[2 * T];
    __shared__ uint32_t gcnt[WAVE], s_next[2];
    __shared__ uint64_t s_base;
    const uint32_t end = (uint32_t)((n + T - 1) / T);
    uint32_t at = blockIdx.x;
    auto next = [&]() {
        const uint32_t t = at;
        at += gridDim.x;
        return t;
    };
    auto desc = [&](uint32_t t) {
        const uint64_t lo = (uint64_t)t * T;
        return FilterTile{skey + lo, sval + lo, nullptr, (uint32_t)min((uint64_t)T, n - lo), filter, g,
                          okey, oval, out_cap, count};
    };
    if (filter_run<BLOCK, ITEMS>(end, next, desc, stage, gcnt, &s_base, s_next))
        atomicOr((unsigned long long*)err, 2ull);
}

// ============================================================== Bloom filter after pass 1
// S has been scattered by its first-pass bucket.  The filter slice of
// first-pass bucket p is contiguous (segments are the top radix bits), 1/P1 of
// the filter.  Workgroups are dealt to XCDs round-robin (workgroup i runs on
// XCD i % 8), so XCD x takes buckets x, x+8, ... as one sequence of tiles,
// handed out in order by the XCD's own counter (tile_ctr[x]): all its
// workgroups work on the same bucket, whose filter slice stays in the XCD's L2
// while its S tuples stream past (loaded non-temporally), and a workgroup that
// finishes early takes the next tile instead of running ahead into the next
// bucket.  Survivors are counting-sorted by sub-bucket in LDS per tile, reserved
// with one atomic per (tile, sub-bucket) and written, compacted, into their
// sub-bucket's region of the S layout (sub-bucket sb gets positions
// sb_start[sb] + [0, s_fill[sb])), so no second pass over S is needed.  S comes as
// whole tuples, so the values of tuples that fail are read too.
//
// Tile walk of one XCD: bucket p owns ceil(size / T) consecutive tile numbers
// starting at tb; a workgroup's tile numbers only grow, so it walks forward.
struct FilterWalk {
    int p;          // current bucket (>= P1: done)
    uint64_t tb;    // first tile number of bucket p
    uint64_t lo, hi;
};

__device__ __forceinline__ void filter_walk_to(FilterWalk& w, uint64_t t, const uint64_t* __restrict__ sb_start,
                                               int P1, int bits2, uint64_t T)
{
    while (w.p < P1) {
        const uint64_t nt = (w.hi - w.lo + T - 1) / T;
        if (t < w.tb + nt) return;
        w.tb += nt;
        w.p += 8;
        if (w.p < P1) {
            w.lo = sb_start[(uint64_t)w.p << bits2];
            w.hi = sb_start[(uint64_t)(w.p + 1) << bits2];
        }
    }
}

// A tile's reservations and stores lag one tile behind: tile t's places are
// requested (one atomic per sub-bucket) while it is staged in one of two LDS
// buffers, and read, published and used after tile t + 1's test, so neither their
// latency nor that of the values is on a tile's path.  The next tile's tuples are
// issued after the test, not behind this tile's filter words (3.66 against 3.39 ms).
// Bound by the XCD's L2, one request per key: 640M keys in 3 MB slices 3.53 -> 3.39
// ms, 1.28B keys in 0.75 MB slices 5.87 -> 5.63 ms (227 G keys/s).
//
// K: the filter's bits per key when fixed at compile time (3 or 4), 0 = g.k.
// PER: sub-buckets per thread of the offset scan; 0: at most one per lane of one
// wave (no block scan).
template <int BLOCK, int ITEMS, int K, int PER>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_filter_l1(
    TupleIn<true> in, const uint64_t* __restrict__ sb_start, int bits, int bits2, const uint64_t* __restrict__ filter,
    BloomGeom g, uint32_t* __restrict__ okey, uint32_t* __restrict__ oval, uint64_t out_cap,
    uint32_t* __restrict__ s_fill, uint64_t* __restrict__ count, uint64_t* __restrict__ tile_ctr,
    uint64_t* __restrict__ err)
{
    constexpr int T = BLOCK * ITEMS;
    constexpr int NXCD = 8;
    constexpr int NB = PER ? PER : 1;
    const int P1 = 1 << (bits - bits2), P2 = 1 << bits2;
    const int shift = 32 - bits;
    const uint32_t bmask = (uint32_t)P2 - 1u;
    extern __shared__ uint64_t lds64[];
    uint64_t* dst = lds64;                        // [P2] position of the last tile's tuple q: dst + q
    Tuple* stage = (Tuple*)(dst + P2);            // [2 * T] survivors, sub-bucket by sub-bucket (two tiles)
    uint32_t* cnt0 = (uint32_t*)(stage + 2 * T);  // [2 * P2] survivors per sub-bucket (two tiles)
    uint32_t* off = cnt0 + 2 * P2;                // [P2] staging offset
    uint32_t* wtmp = off + P2;                    // [BLOCK/64 + 1]
    __shared__ uint32_t s_total[2];
    __shared__ uint64_t s_tile, s_tile2;

    const int xcd = blockIdx.x % NXCD;
    unsigned long long* xctr = (unsigned long long*)tile_ctr + xcd;
    bool bad = false;
    uint32_t surv_total = 0;
    for (int b = threadIdx.x; b < 2 * P2; b += BLOCK) cnt0[b] = 0u;
    // tile numbers are taken one tile ahead: the current one and the next are
    // known, the one after that is requested while the current tile runs
    if (threadIdx.x == 0) {
        s_tile = atomicAdd(xctr, 1ull);
        s_tile2 = atomicAdd(xctr, 1ull);
    }
    __syncthreads();
    // (in scalar registers: so is the walk then)
    const uint64_t t_first = uniform_u64(s_tile);
    uint64_t t_next = uniform_u64(s_tile2);
    uint32_t par = 0;

    FilterWalk wk;
    wk.p = xcd;
    wk.tb = 0;
    wk.lo = wk.hi = 0;
    if (wk.p < P1) {
        wk.lo = sb_start[(uint64_t)wk.p << bits2];
        wk.hi = sb_start[(uint64_t)(wk.p + 1) << bits2];
    }
    filter_walk_to(wk, t_first, sb_start, P1, bits2, T);
    // the current tile [tile, chi) of bucket p; tuples are streamed once
    // (non-temporal, so the filter slice keeps the L2), a tile ahead
    int p = wk.p;
    uint64_t tile = wk.lo + (t_first - wk.tb) * (uint64_t)T;
    uint64_t chi = min(tile + (uint64_t)T, wk.hi);
    Tuple nk[ITEMS];
    // clamped to the tile's last tuple rather than skipped past it: no branches
    auto load_tile = [&](uint64_t at, uint64_t end) {
        const TupleIn<true> src = in.from(at);
        const uint32_t last = (uint32_t)(end - 1 - at);
#pragma unroll
        for (int it = 0; it < ITEMS; it++) nk[it] = src.load(min((uint32_t)it * BLOCK + threadIdx.x, last));
    };
    if (p < P1) load_tile(tile, chi);

    // this thread's sub-buckets [b0, b0 + NB) of the scan, and what it knows of
    // their last tile's reservations
    const int b0 = (int)threadIdx.x * NB;
    const bool own = b0 < P2;
    uint64_t rstart[NB];
    uint32_t rbase[NB], roff[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        rstart[j] = 0;
        rbase[j] = roff[j] = 0;
    }
    auto publish = [&]() {  // the last tile's places
        if (own)
#pragma unroll
            for (int j = 0; j < NB; j++) dst[b0 + j] = rstart[j] + rbase[j] - roff[j];
    };
    auto write_out = [&](uint32_t buf, uint32_t ts) {
        for (uint32_t q = threadIdx.x; q < ts; q += BLOCK) {
            const Tuple x = stage[buf * T + q];
            const uint64_t d = dst[(radix_hash(x.x) >> shift) & bmask] + q;
            if (d < out_cap) {
                okey[d] = x.x;
                oval[d] = x.y;
            } else {
                bad = true;
            }
        }
        surv_total += ts;
    };

    bool have_last = false;  // a tile is staged and not yet written (uniform)
    // Per tile two barriers (more with a block scan): test + rank | offsets,
    // reservations, the last tile's places | staging, the last tile out (runs into
    // the next tile's test).
    while (p < P1) {
        const int tn = (int)(chi - tile);
        uint32_t* cnt = cnt0 + (par ? P2 : 0);
        uint32_t* cnext = cnt0 + (par ? 0 : P2);
        // the tile number after the next one, in flight during this tile
        unsigned long long t_after = 0ull;
        if (threadIdx.x == 0) t_after = atomicAdd(xctr, 1ull);
        Tuple k[ITEMS];
#pragma unroll
        for (int it = 0; it < ITEMS; it++) k[it] = nk[it];
        // all filter words of the tile in flight before any is tested
        uint64_t fw[ITEMS];
#pragma unroll
        for (int it = 0; it < ITEMS; it++) fw[it] = filter[bloom_block(k[it].x, g)];
        // then the next tile's tuples, so that no wait for a filter word covers them
        // (on every path: after the last tile, this tile again, unused)
        filter_walk_to(wk, t_next, sb_start, P1, bits2, T);
        const int p_next = wk.p;
        const uint64_t tile_next = wk.lo + (t_next - wk.tb) * (uint64_t)T;
        const uint64_t chi_next = min(tile_next + (uint64_t)T, wk.hi);
        uint32_t br[ITEMS];  // sub-bucket | rank << 16
        uint32_t pass = 0;
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            // used here on every path: the load is not sunk into the branch below
            // (where it would wait for all loads before it)
            asm volatile("" : "+v"(fw[it]));
            const uint64_t m = K ? bloom_mask_k<(K ? K : 1)>(k[it].x) : bloom_mask(k[it].x, g.k);
            if (it * BLOCK + (int)threadIdx.x < tn && (fw[it] & m) == m) {
                const uint32_t b = (radix_hash(k[it].x) >> shift) & bmask;
                br[it] = b | (atomicAdd(&cnt[b], 1u) << 16);
                pass |= 1u << it;
            }
        }
        __syncthreads();
        if (PER || threadIdx.x < WAVE) {
            publish();
            uint32_t c[NB], sum = 0;
#pragma unroll
            for (int j = 0; j < NB; j++) {
                c[j] = own ? cnt[b0 + j] : 0u;
                sum += c[j];
            }
            uint32_t ex, tot;
            if constexpr (PER == 0) {
                const uint32_t inc = wave_inclusive_scan<uint32_t>(sum);
                ex = inc - sum;
                tot = __builtin_amdgcn_readlane(inc, WAVE - 1);
            } else {
                ex = block_exclusive_scan<BLOCK, uint32_t>(sum, wtmp, &tot);
            }
            if (own) {
#pragma unroll
                for (int j = 0; j < NB; j++) {
                    const uint64_t sb = ((uint64_t)p << bits2) + b0 + j;
                    off[b0 + j] = ex;
                    cnext[b0 + j] = 0u;
                    roff[j] = ex;
                    rstart[j] = sb_start[sb];
                    if (c[j]) rbase[j] = atomicAdd(&s_fill[sb], c[j]);
                    ex += c[j];
                }
            }
            if (threadIdx.x == 0) {
                s_total[par] = tot;
                s_tile = t_after;
            }
        }
        __syncthreads();
        load_tile(p_next < P1 ? tile_next : tile, p_next < P1 ? chi_next : chi);
#pragma unroll
        for (int it = 0; it < ITEMS; it++)
            if ((pass >> it) & 1u) stage[par * T + off[br[it] & 0xFFFFu] + (br[it] >> 16)] = k[it];
        t_next = uniform_u64(s_tile);
        if (have_last) write_out(par ^ 1u, s_total[par ^ 1u]);
        have_last = true;
        p = p_next;
        tile = tile_next;
        chi = chi_next;
        par ^= 1u;
    }
    if (have_last) {  // uniform: the last tile
        __syncthreads();
        if (PER || threadIdx.x < WAVE) publish();
        __syncthreads();
        write_out(par ^ 1u, s_total[par ^ 1u]);
    }
    if (threadIdx.x == 0 && surv_total)
        atomicAdd((unsigned long long*)count, (unsigned long long)surv_total);
    if (bad) atomicOr((unsigned long long*)err, 8ull);
}

// ============================================================== S' of the chunks of S
// With S in chunks, every chunk's S' (its surviving tuples, in sub-bucket
// regions) stays in its own region of a pool, and one probe runs after the
// last chunk on all of them, so R streams past the tables once instead of once
// per chunk.  Note: sub-bucket sb of the chunk whose region starts at base has
// its piece at base + s_start[sb], cnt[sb] tuples long (the chunk's row of the
// piece table); *total accumulates the tuples.
constexpr int POOL_BLOCK = 256;

__global__ __launch_bounds__(POOL_BLOCK) void k_pool_note(const uint64_t* __restrict__ s_start,
                                                          const uint32_t* __restrict__ s_cnt, int nbins, uint64_t base,
                                                          uint32_t* __restrict__ cnt, uint64_t* __restrict__ off,
                                                          uint64_t* __restrict__ total)
{
    const int sb = blockIdx.x * POOL_BLOCK + threadIdx.x;
    uint64_t n = 0;
    if (sb < nbins) {
        const uint64_t s0 = s_start[sb];
        n = s_cnt ? (uint64_t)s_cnt[sb] : s_start[sb + 1] - s0;
        cnt[sb] = (uint32_t)n;
        off[sb] = base + s0;
    }
    n = wave_sum<uint64_t>(n);
    if (lane_id() == 0 && n) atomicAdd((unsigned long long*)total, (unsigned long long)n);
}

// totals[sb] = the pieces of sub-bucket sb summed over the nch chunks.
__global__ void k_pool_totals(const uint32_t* __restrict__ cnt, int nch, int nbins, uint32_t* __restrict__ totals)
{
    const int sb = blockIdx.x * blockDim.x + threadIdx.x;
    if (sb >= nbins) return;
    uint32_t t = 0;
    for (int c = 0; c < nch; c++) t += cnt[(size_t)c * nbins + sb];
    totals[sb] = t;
}

// Sub-bucket sb (one workgroup) gathers its pieces, chunk by chunk, into
// [start[sb], start[sb + 1]) of ok / ov.
__global__ __launch_bounds__(POOL_BLOCK) void k_pool_merge(
    const uint32_t* __restrict__ pk, const uint32_t* __restrict__ pv, const uint32_t* __restrict__ cnt,
    const uint64_t* __restrict__ off, int nch, int nbins, const uint64_t* __restrict__ start,
    uint32_t* __restrict__ ok, uint32_t* __restrict__ ov, uint64_t out_cap, uint64_t* __restrict__ err)
{
    const int sb = blockIdx.x;
    uint64_t d = start[sb];
    if (start[sb + 1] > out_cap) {
        if (threadIdx.x == 0) atomicOr((unsigned long long*)err, 16ull);
        return;
    }
    for (int c = 0; c < nch; c++) {
        const uint32_t n = cnt[(size_t)c * nbins + sb];
        const uint64_t o = off[(size_t)c * nbins + sb];
        for (uint32_t i = threadIdx.x; i < n; i += POOL_BLOCK) {
            ok[d + i] = pk[o + i];
            ov[d + i] = pv[o + i];
        }
        d += n;
    }
}

// ============================================================== build + probe
// Persistent workgroups take work items in order, first the vlsplit items (the
// largest), then one item per regular sub-bucket: the first by workgroup number,
// the others from a global counter (claimed while the current one runs).  Each item builds the
// build side's chunk into an LDS table and streams the other side's slice
// past it (probe_item, bj_tiles.h).
// COLLECT (the reference's COLLECT / --fused_probe_breakdown): thread 0 of
// every workgroup adds its phase times (PT_*) to timers[blockIdx.x * PT_N + p].
#ifndef BJ_PROBE_GRAB
#define BJ_PROBE_GRAB 2
#endif
constexpr int PROBE_GRAB = BJ_PROBE_GRAB;

template <int BLOCK, int CAP, int PITEMS, bool COLLECT>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(probe_waves(BLOCK, CAP), 8))) void k_probe(
    const uint32_t* __restrict__ rk, const uint32_t* __restrict__ rv,
    const uint64_t* __restrict__ r_start, const uint32_t* __restrict__ sk,
    const uint32_t* __restrict__ sv, const uint64_t* __restrict__ s_start,
    const uint32_t* __restrict__ s_cnt, int bits, uint32_t slice,
    const HeavyItem* __restrict__ items, const uint64_t* __restrict__ n_items_p, uint64_t item_cap,
    uint64_t* __restrict__ work_ctr, uint64_t* __restrict__ out_count, uint64_t out_cap,
    uint32_t* __restrict__ o_key, uint32_t* __restrict__ o_rval, uint32_t* __restrict__ o_sval,
    uint64_t* __restrict__ timers)
{
    __shared__ ProbeLds<BLOCK, CAP> L;
    __shared__ uint64_t s_next;
    uint64_t tacc[PT_N] = {}, tmark = 0;
    if (COLLECT && threadIdx.x == 0) tmark = phase_clock();

    const int nbins = 1 << bits;
    const uint64_t n_heavy = min(*n_items_p, item_cap);
    const uint64_t n_work = n_heavy + (uint64_t)nbins;

    // Items are claimed PROBE_GRAB at a time (the counter's answer is waited for
    // once per claim), but one by one when there is no more than one claim for each
    // workgroup: 3M x 4.5M has 512 items, which pairs would give to half of the 512
    // workgroups (46.6 -> 32.2 us with the next line, by 512 threads per table; 16M x
    // 16M, 2048 items: 99-102 us in pairs, 105 us one by one).  The first claim is the workgroup's number: from
    // the counter, the last of 512 answers would be several us away.
    const int grab = n_work <= (uint64_t)gridDim.x * PROBE_GRAB ? 1 : PROBE_GRAB;
    uint64_t item = (uint64_t)blockIdx.x * grab;
    const uint64_t claimed = (uint64_t)gridDim.x * grab;
    int left = grab;  // items of the current claim, this one included

    while (item < n_work) {
        if (left == 1 && threadIdx.x == 0)
            s_next = atomicAdd((unsigned long long*)work_ctr, (unsigned long long)grab);

        uint32_t sb, chunk = 0, sl = 0, nsl = 1;
        const bool heavy = item < n_heavy;
        if (heavy) {
            const HeavyItem hi = items[item];
            sb = hi.sb; chunk = hi.chunk; sl = hi.slice; nsl = hi.nslices;
        } else {
            sb = (uint32_t)(item - n_heavy);
        }
        uint64_t r0, nr, s0, ns;
        sb_sizes(r_start, s_start, s_cnt, (int)sb, r0, nr, s0, ns);
        const bool build_r = build_from_r(nr, ns, (uint32_t)CAP);
        const uint64_t nb = build_r ? nr : ns, np = build_r ? ns : nr;
        // empty, or a regular index whose sub-bucket is on the vlsplit list: nothing to do
        const bool skip = nr == 0 || ns == 0 || (!heavy && (nb > (uint64_t)CAP || np > (uint64_t)slice));
        if (!skip) {
            const uint64_t b_lo = (uint64_t)chunk * CAP;
            const int bn = (int)min((uint64_t)CAP, nb - b_lo);
            const uint64_t per = (np + nsl - 1) / nsl;
            const uint64_t p_lo = min((uint64_t)sl * per, np);
            const uint32_t pn = (uint32_t)min(per, np - p_lo);
            const uint64_t brow0 = (build_r ? r0 : s0) + b_lo;
            const uint64_t prow0 = (build_r ? s0 : r0) + p_lo;
            phase_tick<COLLECT>(tacc, &tmark, PT_ITEM);
            probe_item<BLOCK, CAP, PITEMS, COLLECT>(L, (build_r ? rk : sk) + brow0, (build_r ? rv : sv) + brow0,
                                                    bn, (build_r ? sk : rk) + prow0, (build_r ? sv : rv) + prow0,
                                                    pn, build_r, bits, out_count, out_cap, o_key, o_rval, o_sval,
                                                    tacc, &tmark);
        }
        __syncthreads();  // the table is rebuilt by the next item; s_next is written
        if (left > 1) {
            item++;
            left--;
        } else {
            item = claimed + s_next;
            left = grab;
        }
        __syncthreads();
    }
    if (COLLECT && threadIdx.x == 0) {
        phase_tick<COLLECT>(tacc, &tmark, PT_ITEM);
        for (int p = 0; p < PT_N; p++) timers[(size_t)blockIdx.x * PT_N + p] += tacc[p];
    }
}

// ============================================================== direct join (small build side)
// Clears the join's counters and its filter in one launch.
__global__ void k_direct_begin(uint64_t* __restrict__ ctr, int n_ctr, uint64_t* __restrict__ filter, uint64_t nf)
{
    const uint64_t i0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i0 < (uint64_t)n_ctr) ctr[i0] = 0ull;
    for (uint64_t i = i0; i < nf; i += (uint64_t)gridDim.x * blockDim.x) filter[i] = 0ull;
}

// The filter of an unpartitioned R (cleared before); the same bits as k_bloom_build's.
// Every workgroup gathers its keys' bits block by block in an LDS hash table, then ORs
// each block into the filter with one 64-bit atomic: the chip does some 70 atomics on
// one address per us, so that with an atomic per key equal keys, or a filter of few
// blocks, set the pace (100K equal keys 1.14 ms, 2.5M 28.3 ms, 200K keys in 256 bits
// 1.08 ms; so 7, 116 and 9 us).  Distinct keys are bound by the atomics either way: 2.5M
// 97 -> 99 us, 200K 12 -> 13 (two or four keys per thread 16-19).
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_direct_bloom(const uint32_t* __restrict__ rkey, uint32_t n, BloomGeom g,
                                                        uint64_t* __restrict__ filter)
{
    constexpr uint32_t SLOTS = 2 * BLOCK, EMPTY = 0xFFFFFFFFu;  // at most half full
    static_assert((SLOTS & (SLOTS - 1)) == 0, "slots are found by a mask");
    __shared__ uint32_t blk[SLOTS];
    __shared__ unsigned long long bits[SLOTS];
    for (uint32_t i = threadIdx.x; i < SLOTS; i += BLOCK) {
        blk[i] = EMPTY;
        bits[i] = 0ull;
    }
    const uint32_t i = blockIdx.x * BLOCK + threadIdx.x;
    const uint32_t k = rkey[min(i, n - 1u)];
    __syncthreads();
    if (i < n) {
        const uint32_t b = (uint32_t)bloom_block(k, g);
        uint32_t s = b & (SLOTS - 1);
        for (;; s = (s + 1) & (SLOTS - 1)) {  // ends: there are more slots than keys
            const uint32_t was = atomicCAS(&blk[s], EMPTY, b);
            if (was == EMPTY || was == b) break;
        }
        atomicOr(&bits[s], (unsigned long long)bloom_mask(k, g.k));
    }
    __syncthreads();
    for (uint32_t s = threadIdx.x; s < SLOTS; s += BLOCK)
        if (blk[s] != EMPTY) atomicOr((unsigned long long*)&filter[blk[s]], bits[s]);
}

// Joins unpartitioned relations: the build side in C chunks of at most CAP tuples, the
// probe side in slices, one (chunk, slice) pair per workgroup and step.  Every chunk
// streams all of the probe side past its table, so the work is C * np probes where the
// partitioned path moves every tuple two to four times (sixteen or more launches when
// this was measured, five to twelve now).  Bound by launches and the build's latency
// for small relations (1500 x 2000: 124 -> 53 us a call, 200K x 300K with the filter
// 233 -> 115 us), by the probe's issue rate and row writes for long ones (6001 x 20M:
// 4.99 -> 0.42 ms a call; the partitioned path had 32 work items there).  ns_dev, when
// not null, is the device-side length of S (S' after the filter).  Workgroups of one
// slice run on one XCD (slices are dealt in multiples of 8), so its keys come from that
// XCD's L2 after the first chunk.
// WATCH (build sides of several chunks): every probe key of a bucket walks its whole
// run, so a key that fills a good part of every chunk costs far more than here is saved
// (300K x 200K with 90% of S equal: 1.8 ms), where the partitioned join builds the hot
// sub-bucket's table from the other side.  A workgroup whose table has a longer run than
// it may have sets *long_run and leaves; the host then joins by partitions (of bits
// radix bits).  With one chunk (C = 1) the partitioned join would build the same table.
// Otherwise a run may be DIRECT_MAX_RUN long, or as long as a key that has it in every
// chunk leaves its sub-bucket of the partitioned join smaller on this side than on the
// other, so that a C times longer run would be walked there.  Both sides of the line,
// direct against partitioned: 200K x 300K, 256 copies in a chunk 109 / 76 us (some 40
// us more after the attempt), 512 138 / 76, 1024 281 / 76; 300K x 100K 512 119 / 969,
// 1024 270 / 75; 100K x 1M 1024 398 / 660, 2M x 50K 4096 1582 / 2192.
constexpr uint32_t DIRECT_MAX_RUN = 320;

template <int BLOCK, int CAP, int PITEMS, bool WATCH>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(probe_waves(BLOCK, CAP), 8))) void k_join_direct(
    const uint32_t* __restrict__ rk, const uint32_t* __restrict__ rv, uint32_t nr,
    const uint32_t* __restrict__ sk, const uint32_t* __restrict__ sv, uint32_t ns_host,
    const uint64_t* __restrict__ ns_dev, bool build_r, uint32_t grain, int bits, uint64_t* __restrict__ long_run,
    uint64_t* __restrict__ out_count, uint64_t out_cap, uint32_t* __restrict__ o_key, uint32_t* __restrict__ o_rval, uint32_t* __restrict__ o_sval)
{
    __shared__ ProbeLds<BLOCK, CAP> L;
    const uint32_t ns = ns_dev ? (uint32_t)min(*ns_dev, (uint64_t)ns_host) : ns_host;
    const uint32_t nb = build_r ? nr : ns, np = build_r ? ns : nr;
    if (nb == 0 || np == 0) return;
    const uint32_t C = (nb + CAP - 1) / CAP;
    // longest run that a table may have
    const uint32_t per_b = nb >> bits, per_p = np >> bits;
    const uint32_t max_run = C == 1 ? 0xFFFFFFFFu : max(DIRECT_MAX_RUN, per_p > per_b ? (per_p - per_b) / C : 0u);
    const uint32_t cper = (nb + C - 1) / C;
    uint32_t S = max(1u, min(gridDim.x / C, (np + grain - 1) / grain));
    if (S > 8) S &= ~7u;
    const uint32_t sper = (np + S - 1) / S;
    const uint64_t items = (uint64_t)C * S;
    for (uint64_t item = blockIdx.x; item < items; item += gridDim.x) {
        const uint32_t c = (uint32_t)(item / S), sl = (uint32_t)(item % S);
        const uint32_t b0 = min(c * cper, nb), p0 = (uint32_t)min((uint64_t)sl * sper, (uint64_t)np);
        const int bn = (int)min(cper, nb - b0);
        const uint32_t pn = min(sper, np - p0);
        if (probe_item<BLOCK, CAP, PITEMS, false, WATCH>(
                L, (build_r ? rk : sk) + b0, (build_r ? rv : sv) + b0, bn, (build_r ? sk : rk) + p0,
                (build_r ? sv : rv) + p0, pn, build_r, 0, out_count, out_cap, o_key, o_rval, o_sval, nullptr, nullptr,
                max_run)) {
            if (threadIdx.x == 0) *long_run = 1ull;
            return;
        }
        __syncthreads();  // the table is rebuilt by the next item
    }
}

// ============================================================== launchers
static int ceil_div_i(uint64_t a, uint64_t b) { return (int)((a + b - 1) / b); }

hipError_t launch_add2_u64(const uint64_t* a, const uint64_t* b, uint64_t* acc, hipStream_t st)
{
    k_add2_u64<<<1, 64, 0, st>>>(a, b, acc);
    return hipGetLastError();
}

hipError_t launch_zero_u64(uint64_t* p, int n, hipStream_t st)
{
    k_zero_u64<<<1, 256, 0, st>>>(p, n);
    return hipGetLastError();
}

hipError_t launch_gen_r(uint32_t* key, uint32_t* val, uint64_t n, const PermKeys& K, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    const int grid = (int)std::min<uint64_t>(65536, (n + 255) / 256);
    k_gen_r<<<grid, 256, 0, st>>>(key, val, n, K);
    return hipGetLastError();
}

hipError_t launch_gen_s(uint32_t* key, uint32_t* val, uint64_t n_s, uint64_t n_r, uint64_t m_s,
                        int L, const PermKeys& KR, const PermKeys& KP, const PermKeys& KN,
                        uint32_t useed, double zipf_s, uint32_t zseed, double* d_tmp,
                        hipStream_t st)
{
    if (n_s == 0) return hipSuccess;
    double Hn = 0.0;
    if (zipf_s > 0.0) {
        k_zipf_Hn<<<1, 64, 0, st>>>(d_tmp, (uint32_t)n_r, zipf_s);
        hipError_t e = hipMemcpyAsync(&Hn, d_tmp, sizeof(double), hipMemcpyDeviceToHost, st);
        if (e != hipSuccess) return e;
        e = hipStreamSynchronize(st);
        if (e != hipSuccess) return e;
    }
    const int grid = (int)std::min<uint64_t>(65536, (n_s + 255) / 256);
    k_gen_s<<<grid, 256, 0, st>>>(key, val, n_s, n_r, m_s, L, KR, KP, KN, useed, zipf_s, Hn, zseed);
    return hipGetLastError();
}

static int log2_ceil_u64(uint64_t n)
{
    int l = 0;
    while ((1ull << l) < n) l++;
    return l;
}

hipError_t launch_gen_refdist_r(uint32_t* key, uint64_t n, uint64_t k, const PermKeys& K, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    const int grid = (int)std::min<uint64_t>(65536, (n + 255) / 256);
    k_gen_refdist_r<<<grid, 256, 0, st>>>(key, n, k, std::max(1, log2_ceil_u64(n)), K);
    return hipGetLastError();
}

hipError_t launch_gen_refdist_s(uint32_t* key, uint64_t n, uint64_t m, uint64_t mc0, uint64_t sj0, uint64_t n_r,
                                const PermKeys& K, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    const int grid = (int)std::min<uint64_t>(65536, (n + 255) / 256);
    k_gen_refdist_s<<<grid, 256, 0, st>>>(key, n, m, mc0, sj0, n_r, std::max(1, log2_ceil_u64(n)), K);
    return hipGetLastError();
}

constexpr int HIST_BLOCK = 1024;
constexpr int SC_BLOCK = 1024;
constexpr int SC_ITEMS = 4;
constexpr int SC_BIG_ITEMS = 8;  // 8192-tuple tiles for one-workgroup-per-CU launches
static size_t g_max_lds = 64 * 1024;
constexpr int FL_BLOCK = 512;
constexpr int FL_ITEMS = 8;

// Allow dynamic LDS up to the device limit minus the kernel's static LDS.
static hipError_t set_lds(const void* fn, size_t bytes)
{
    hipFuncAttributes attr;
    hipError_t e = hipFuncGetAttributes(&attr, fn);
    if (e != hipSuccess) return e;
    const size_t stat = attr.sharedSizeBytes;
    return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)(bytes > stat ? bytes - stat : 0));
}

template <int K>
static hipError_t set_filter_lds(int bytes)
{
    hipError_t e;
    if ((e = set_lds((const void*)k_filter_l1<FL_BLOCK, FL_ITEMS, K, 0>, bytes)) != hipSuccess) return e;
    if ((e = set_lds((const void*)k_filter_l1<FL_BLOCK, FL_ITEMS, K, 1>, bytes)) != hipSuccess) return e;
    return set_lds((const void*)k_filter_l1<FL_BLOCK, FL_ITEMS, K, 4>, bytes);
}

template <bool IPAIR, bool OPAIR>
static hipError_t set_scatter_lds(int bytes)
{
    hipError_t e;
    if ((e = set_lds((const void*)k_scatter<SC_BLOCK, SC_ITEMS, IPAIR, OPAIR>, bytes)) != hipSuccess) return e;
    if ((e = set_lds((const void*)k_scatter<SC_BLOCK / 2, SC_ITEMS * 2, IPAIR, OPAIR>, bytes)) != hipSuccess) return e;
    return set_lds((const void*)k_scatter<SC_BLOCK, SC_BIG_ITEMS, IPAIR, OPAIR>, bytes);
}

hipError_t kernels_init(int max_lds_bytes)
{
    hipError_t e;
    if ((e = set_lds((const void*)k_hist<HIST_BLOCK>, max_lds_bytes)) != hipSuccess) return e;
    if ((e = set_scatter_lds<false, false>(max_lds_bytes)) != hipSuccess) return e;
    if ((e = set_scatter_lds<false, true>(max_lds_bytes)) != hipSuccess) return e;
    if ((e = set_scatter_lds<true, false>(max_lds_bytes)) != hipSuccess) return e;
    g_max_lds = (size_t)max_lds_bytes;
    if ((e = set_lds((const void*)k_bloom_build<1024>, max_lds_bytes)) != hipSuccess) return e;
    if ((e = set_filter_lds<0>(max_lds_bytes)) != hipSuccess) return e;
    if ((e = set_filter_lds<3>(max_lds_bytes)) != hipSuccess) return e;
    if ((e = set_filter_lds<4>(max_lds_bytes)) != hipSuccess) return e;
    return hipSuccess;
}

static Sides sides_of(const PartSide* sides, int n, int (*wgs)(const PartSide&), int& grid)
{
    Sides S;
    S.a = sides[0];
    S.b = sides[n - 1];
    S.na = wgs(sides[0]);
    grid = S.na + (n > 1 ? wgs(sides[1]) : 0);
    return S;
}

hipError_t launch_hist(const PartSide* sides, int n, uint64_t* ctr, int n_ctr, uint32_t* zero32, int n_zero32,
                       hipStream_t st)
{
    int grid;
    const Sides S = sides_of(sides, n, [](const PartSide& s) { return s.G; }, grid);
    const size_t lds = sizeof(uint32_t) << std::max(S.a.bits, S.b.bits);
    k_hist<HIST_BLOCK><<<grid, HIST_BLOCK, lds, st>>>(S, ctr, n_ctr, zero32, n_zero32);
    return hipGetLastError();
}

hipError_t launch_cols(const PartSide* sides, int n, hipStream_t st)
{
    int grid;
    const Sides S = sides_of(sides, n, [](const PartSide& s) { return cols_wgs(s); }, grid);
    if (S.a.bits > 15 || S.b.bits > 15) return hipErrorInvalidValue;
    k_cols<<<grid, 1024, 0, st>>>(S);
    return hipGetLastError();
}

size_t scan_partials_needed(uint64_t n) { return (size_t)ceil_div_i(n ? n : 1, SCAN_TILE) + 1; }

hipError_t launch_scan(const uint32_t* in, uint64_t n, uint64_t* out, uint64_t* partial,
                       hipStream_t st)
{
    const int W = ceil_div_i(n ? n : 1, SCAN_TILE);
    if (W > 1024 * 64) return hipErrorInvalidValue;
    k_scan_reduce<<<W, SCAN_BLOCK, 0, st>>>(in, n, partial);
    k_scan_top<<<1, 1024, 0, st>>>(partial, W);
    k_scan_down<<<W, SCAN_BLOCK, 0, st>>>(in, n, partial, out, W);
    return hipGetLastError();
}

static size_t scatter_lds_tile(int nbk, int tile, int cs_log2)
{
    return (size_t)nbk * SCATTER_BUCKET_BYTES + ((size_t)nbk << cs_log2) * 8 + (size_t)tile * 8 +
           (SC_BLOCK / WAVE + 1) * 4;
}

size_t scatter_lds_bytes(int nbk)
{
    return scatter_lds_tile(nbk, SC_BLOCK * SC_ITEMS, scatter_carry_log2(nbk, false, false));
}

size_t scatter_lds_bytes_big(int nbk)
{
    return scatter_lds_tile(nbk, SC_BLOCK * SC_BIG_ITEMS, scatter_carry_log2(nbk, true, false));
}

template <bool IPAIR, bool OPAIR>
static hipError_t scatter_pass(const PartSide* sides, int n, const PlanArgs& plan, uint64_t* err, int wg,
                               size_t min_lds, hipStream_t st)
{
    int grid;
    const Sides S = sides_of(
        sides, n, [](const PartSide& s) { return IPAIR ? second_wgs(s) : s.G + 1; }, grid);
    if (IPAIR && plan.items) grid++;
    size_t lds = 0, lds_big = 0;
    for (int i = 0; i < n; i++) {
        const int nbk = IPAIR ? 1 << (sides[i].bits - sides[i].p1) : 1 << sides[i].p1;
        lds = std::max(lds, scatter_lds_tile(nbk, SC_BLOCK * SC_ITEMS, scatter_carry_log2(nbk, false, OPAIR)));
        lds_big =
            std::max(lds_big, scatter_lds_tile(nbk, SC_BLOCK * SC_BIG_ITEMS, scatter_carry_log2(nbk, true, OPAIR)));
    }
    lds = std::max(lds, min_lds);
    lds_big = std::max(lds_big, min_lds);
    if (wg != 512 && min_lds > 0 && lds_big <= g_max_lds) {
        // one workgroup per CU: twice the tile, twice the loads in flight, whole-line carries
        k_scatter<SC_BLOCK, SC_BIG_ITEMS, IPAIR, OPAIR><<<grid, SC_BLOCK, lds_big, st>>>(S, plan, err);
    } else if (wg == 512) {
        // same tile (4096 tuples), half the threads: more workgroups per CU
        k_scatter<SC_BLOCK / 2, SC_ITEMS * 2, IPAIR, OPAIR><<<grid, SC_BLOCK / 2, lds, st>>>(S, plan, err);
    } else {
        k_scatter<SC_BLOCK, SC_ITEMS, IPAIR, OPAIR><<<grid, SC_BLOCK, lds, st>>>(S, plan, err);
    }
    return hipGetLastError();
}

hipError_t launch_scatter(int pass, const PartSide* sides, int n, const PlanArgs* plan, uint64_t* err, int wg,
                          size_t min_lds, hipStream_t st)
{
    const PlanArgs p = plan ? *plan : PlanArgs{};
    switch (pass) {
    case SCATTER_ONLY: return scatter_pass<false, false>(sides, n, p, err, wg, min_lds, st);
    case SCATTER_FIRST: return scatter_pass<false, true>(sides, n, p, err, wg, min_lds, st);
    case SCATTER_SECOND: return scatter_pass<true, false>(sides, n, p, err, wg, min_lds, st);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_bloom_build(const uint32_t* rkey, const uint64_t* r_start, int bits,
                              const BloomGeom& g, uint64_t* filter, hipStream_t st)
{
    const int nseg = 1 << g.seg_bits;
    k_bloom_build<1024><<<nseg, 1024, (size_t)g.wps * 8, st>>>(rkey, r_start, bits, g, filter);
    return hipGetLastError();
}

hipError_t launch_bloom_prefilter(const uint32_t* skey, const uint32_t* sval, uint64_t n,
                                  const uint64_t* filter, const BloomGeom& g, uint32_t* okey,
                                  uint32_t* oval, uint64_t out_cap, uint64_t* count, uint64_t* err,
                                  int num_cu, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    constexpr int B = 512, I = 8;
    const int grid = (int)std::min<uint64_t>((uint64_t)num_cu * 2, (n + B * I - 1) / (B * I));
    k_bloom_prefilter<B, I><<<grid, B, 0, st>>>(skey, sval, n, filter, g, okey, oval, out_cap, count, err);
    return hipGetLastError();
}

hipError_t launch_filter_l1(const uint32_t* tuples, const uint64_t* sb_start, int bits,
                            int bits2, const uint64_t* filter, const BloomGeom& g, uint32_t* okey,
                            uint32_t* oval, uint64_t out_cap, uint32_t* s_fill, uint64_t* count,
                            uint64_t* tile_ctr, uint64_t* err, int num_cu, hipStream_t st)
{
    const int P2 = 1 << bits2;
    const size_t lds = (size_t)P2 * 8 + 2 * (size_t)FL_BLOCK * FL_ITEMS * 8 + (size_t)P2 * 12 +
                       (FL_BLOCK / WAVE + 1) * 4;
    const int W = std::max(1, num_cu / 8) * 2;  // workgroups per XCD
    static_assert((1 << 11) <= 4 * FL_BLOCK, "sub-buckets of one first-pass bucket: at most 4 per thread");
    if (bits2 > 11) return hipErrorInvalidValue;
#define BJ_FILTER_PER(K, PER)                                                                                \
    k_filter_l1<FL_BLOCK, FL_ITEMS, K, PER><<<8 * W, FL_BLOCK, lds, st>>>(                                   \
        {(const Tuple*)tuples}, sb_start, bits, bits2, filter, g, okey, oval, out_cap, s_fill, count, tile_ctr, err)
#define BJ_FILTER(K)                                    \
    do {                                                \
        if (P2 <= WAVE) BJ_FILTER_PER(K, 0);            \
        else if (P2 <= FL_BLOCK) BJ_FILTER_PER(K, 1);   \
        else BJ_FILTER_PER(K, 4);                       \
    } while (0)
    if (g.k == 3) BJ_FILTER(3);
    else if (g.k == 4) BJ_FILTER(4);
    else BJ_FILTER(0);
#undef BJ_FILTER
#undef BJ_FILTER_PER
    return hipGetLastError();
}

hipError_t launch_pool_note(const uint64_t* s_start, const uint32_t* s_cnt, int nbins, uint64_t base, uint32_t* cnt,
                            uint64_t* off, uint64_t* total, hipStream_t st)
{
    k_pool_note<<<ceil_div_i((uint64_t)nbins, POOL_BLOCK), POOL_BLOCK, 0, st>>>(s_start, s_cnt, nbins, base, cnt, off,
                                                                                total);
    return hipGetLastError();
}

hipError_t launch_pool_start(const uint32_t* cnt, int nch, int nbins, uint32_t* totals, uint64_t* start,
                             uint64_t* partials, hipStream_t st)
{
    k_pool_totals<<<ceil_div_i((uint64_t)nbins, 256), 256, 0, st>>>(cnt, nch, nbins, totals);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_scan(totals, (uint64_t)nbins, start, partials, st);
}

hipError_t launch_pool_merge(const uint32_t* pk, const uint32_t* pv, const uint32_t* cnt, const uint64_t* off,
                             int nch, int nbins, const uint64_t* start, uint32_t* ok, uint32_t* ov,
                             uint64_t out_cap, uint64_t* err, hipStream_t st)
{
    k_pool_merge<<<nbins, POOL_BLOCK, 0, st>>>(pk, pv, cnt, off, nch, nbins, start, ok, ov, out_cap, err);
    return hipGetLastError();
}

hipError_t launch_plan(const PlanArgs& plan, hipStream_t st)
{
    if (plan.bits > 15) return hipErrorInvalidValue;
    k_plan<1024><<<1, 1024, 0, st>>>(plan);
    return hipGetLastError();
}

int probe_grid(int tile, int num_cu) { return tile == 8192 ? num_cu * 2 : num_cu * 4; }

// Probe keys per thread per round of k_probe.  The rounds are chains of LDS latencies
// between barriers, so the CU's 160 KB of tables are worked on by as many waves as it
// holds: 1024 threads per 8192-tuple table (8 waves per SIMD, 64 registers) against
// 512 threads with 10 keys each: ids 100M x 130M 742 -> 678 us, 9M x 24M with four
// copies of each key 315 -> 259, 64M x 1.28B 289 -> 263, 3M x 4.5M 33.4 -> 29.7.  Rounds
// of 3 keys per thread leave less of a short probe side's last round empty (ids with 4:
// 693 us, 3M x 4.5M 35.2); from PROBE_LONG probe tuples per sub-bucket on 4 are better,
// with fewer reservations (640M x 640M, 39K per sub-bucket: 1.56 ms, 3 keys 1.74).
constexpr int PROBE_ITEMS = 3, PROBE_ITEMS_LONG = 4;
constexpr uint64_t PROBE_LONG = 16384;

static_assert(PT_N == PROBE_TIMER_SLOTS, "probe timer slots");

hipError_t launch_direct_begin(uint64_t* ctr, int n_ctr, uint64_t* filter, uint64_t blocks, hipStream_t st)
{
    const int grid = (int)std::max<uint64_t>(1, std::min<uint64_t>(1024, (blocks + 255) / 256));
    k_direct_begin<<<grid, 256, 0, st>>>(ctr, n_ctr, filter, blocks);
    return hipGetLastError();
}

hipError_t launch_direct_bloom(const uint32_t* rkey, uint64_t n, const BloomGeom& g, uint64_t* filter,
                               hipStream_t st)
{
    constexpr int B = 256;
    if (n == 0) return hipSuccess;
    if (((uint64_t)g.wps << g.seg_bits) >= 0xFFFFFFFFull) return hipErrorInvalidValue;  // block numbers in 32 bits
    k_direct_bloom<B><<<ceil_div_i(n, B), B, 0, st>>>(rkey, (uint32_t)n, g, filter);
    return hipGetLastError();
}

hipError_t launch_join_direct(const uint32_t* rk, const uint32_t* rv, uint64_t nr, const uint32_t* sk,
                              const uint32_t* sv, uint64_t ns, const uint64_t* ns_dev, int bits,
                              uint64_t* long_run, uint64_t* out_count, uint64_t out_cap, uint32_t* o_key,
                              uint32_t* o_rval, uint32_t* o_sval, int num_cu, hipStream_t st)
{
    constexpr int CAP = 8192, B = 512;
    if (nr == 0 || ns == 0) return hipSuccess;
    const bool build_r = build_from_r(nr, ns, CAP);
    const uint64_t nb = build_r ? nr : ns, np = build_r ? ns : nr;
    const uint64_t C = (nb + CAP - 1) / CAP;
    const uint64_t wgs = (uint64_t)probe_grid(CAP, num_cu);
    // one short round (2 keys per thread) per workgroup while that fills at most
    // one wave of workgroups, else rounds of DIRECT_ITEMS keys per thread
    // (1024 threads of 3 keys as in k_probe: 6001 x 20M 159 -> 162 us)
    constexpr int SMALL_ITEMS = 2, DIRECT_ITEMS = 10;
    const uint64_t small_slices = (np + B * SMALL_ITEMS - 1) / (B * SMALL_ITEMS);
    const bool small = C * small_slices <= wgs;
    const uint32_t grain = B * (small ? SMALL_ITEMS : DIRECT_ITEMS);
    const int grid = (int)std::min<uint64_t>(wgs, C * std::max<uint64_t>(1, (np + grain - 1) / grain));
#define BJ_DIRECT(I, W)                                                                                          \
    k_join_direct<B, CAP, I, W><<<grid, B, 0, st>>>(rk, rv, (uint32_t)nr, sk, sv, (uint32_t)ns, ns_dev, build_r, grain, \
                                                    bits, long_run, out_count, out_cap, o_key, o_rval, o_sval)
    if (small && C > 1) BJ_DIRECT(SMALL_ITEMS, true);
    else if (small) BJ_DIRECT(SMALL_ITEMS, false);
    else if (C > 1) BJ_DIRECT(DIRECT_ITEMS, true);
    else BJ_DIRECT(DIRECT_ITEMS, false);
#undef BJ_DIRECT
    return hipGetLastError();
}

hipError_t launch_probe(int tile, uint64_t probe_mean, const uint32_t* rk, const uint32_t* rv, const uint64_t* r_start,
                        const uint32_t* sk, const uint32_t* sv, const uint64_t* s_start,
                        const uint32_t* s_cnt, int bits, uint32_t slice, const HeavyItem* items,
                        const uint64_t* n_items, uint64_t item_cap, uint64_t* work_ctr, uint64_t* out_count,
                        uint64_t out_cap, uint32_t* o_key, uint32_t* o_rval, uint32_t* o_sval, int num_cu,
                        uint64_t* timers, hipStream_t st)
{
#define BJ_PROBE(B, C, I, G)                                                                               \
    do {                                                                                                 \
        if (timers)                                                                                      \
            k_probe<B, C, I, true><<<(G), B, 0, st>>>(rk, rv, r_start, sk, sv, s_start, s_cnt, bits, slice, \
                                                      items, n_items, item_cap, work_ctr, out_count,     \
                                                      out_cap, o_key, o_rval, o_sval, timers);           \
        else                                                                                             \
            k_probe<B, C, I, false><<<(G), B, 0, st>>>(rk, rv, r_start, sk, sv, s_start, s_cnt, bits,    \
                                                       slice, items, n_items, item_cap, work_ctr,        \
                                                       out_count, out_cap, o_key, o_rval, o_sval, nullptr); \
    } while (0)
    const bool long_probe = probe_mean >= PROBE_LONG;
    if (tile == 8192 && long_probe) BJ_PROBE(1024, 8192, PROBE_ITEMS_LONG, probe_grid(8192, num_cu));
    else if (tile == 8192) BJ_PROBE(1024, 8192, PROBE_ITEMS, probe_grid(8192, num_cu));
    else if (tile == 4096) BJ_PROBE(512, 4096, PROBE_ITEMS, probe_grid(4096, num_cu));
    else return hipErrorInvalidValue;
#undef BJ_PROBE
    return hipGetLastError();
}


}  // namespace bj
