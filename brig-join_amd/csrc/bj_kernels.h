// bj_kernels.h -- launchers of the gfx950 kernels (host side).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bj_device.h"

namespace bj {

// One explicit vlsplit work item of an oversized sub-bucket.
struct HeavyItem {
    uint32_t sb;       // sub-bucket
    uint32_t chunk;    // build-side chunk (tile tuples each)
    uint32_t slice;    // probe-side slice index
    uint32_t nslices;  // number of probe-side slices of this sub-bucket
};

hipError_t kernels_init(int max_lds_bytes);

hipError_t launch_zero_u64(uint64_t* p, int n, hipStream_t st);
// acc[0] += *a, acc[1] += *b (one thread): per-chunk counts summed on the device.
hipError_t launch_add2_u64(const uint64_t* a, const uint64_t* b, uint64_t* acc, hipStream_t st);
hipError_t launch_gen_r(uint32_t* key, uint32_t* val, uint64_t n, const PermKeys& K, hipStream_t st);
hipError_t launch_gen_s(uint32_t* key, uint32_t* val, uint64_t n_s, uint64_t n_r, uint64_t m_s,
                        int L, const PermKeys& KR, const PermKeys& KP, const PermKeys& KN,
                        uint32_t useed, double zipf_s, uint32_t zseed, double* d_tmp,
                        hipStream_t st);

// The reference datagen's distribution (datagen/gen_dataset.cpp:172-220) in a
// keyed random order: R of n keys with k matching ones; one region of S (n keys,
// m matching keys from mc0 on, S-only keys from offset sj0 of their sequence).
hipError_t launch_gen_refdist_r(uint32_t* key, uint64_t n, uint64_t k, const PermKeys& K, hipStream_t st);
hipError_t launch_gen_refdist_s(uint32_t* key, uint64_t n, uint64_t m, uint64_t mc0, uint64_t sj0, uint64_t n_r,
                                const PermKeys& K, hipStream_t st);

// One side of a partition launch: a relation and where its partition goes.
struct PartSide {
    const uint32_t *key, *val;  // source
    uint64_t n;                 // tuples, or n_dev (not null): on the device
    const uint64_t* n_dev;
    int G;                      // chunks (histogram and first-pass workgroups)
    int bits, p1;               // radix bits, and those of the first pass
    int W, W2;                  // chunk groups of the column sums, second-pass workgroups per bucket (W = W2)
    int shared2;                // not 0: so many in all (above 2^p1), shared by the buckets' sizes, at most W2 each
    uint32_t* part;             // [G][2^bits] chunk histograms
    uint32_t* l1h;              // [G][2^p1] first-level counts (p1 < bits)
    uint32_t* l1rel;            // [G][2^p1] first-level counts of the chunks before
    uint32_t* l1tot;            // [2^p1] first-level totals
    uint32_t* colsum;           // [W][2^bits]
    uint32_t* totals;           // [2^bits]
    uint64_t* start;            // [2^bits + 1] sub-bucket starts
    uint32_t* tmp;              // whole tuples between the passes (8-byte aligned)
    uint64_t tmp_cap;           // in tuples
    uint32_t *okey, *oval;      // the partitioned relation
    uint64_t out_cap;
};
// The launches of a partition, for one side or for two in one launch (the same
// radix bits): histograms (which also clear totals, the n_ctr counters at ctr and
// n_zero32 words at zero32, either may be null), column sums, the scatter passes.
hipError_t launch_hist(const PartSide* sides, int n, uint64_t* ctr, int n_ctr, uint32_t* zero32, int n_zero32,
                       hipStream_t st);
hipError_t launch_cols(const PartSide* sides, int n, hipStream_t st);
// The vlsplit work items of a probe (bits <= 15): items, and their number at *n_items.
struct PlanArgs {
    const uint64_t *r_start = nullptr, *s_start = nullptr;
    const uint32_t* s_cnt = nullptr;
    int bits = 0;
    uint32_t tile = 0, slice = 0, max_slices = 0;
    uint64_t* n_items = nullptr;
    HeavyItem* items = nullptr;
    uint64_t item_cap = 0;
    uint64_t* err = nullptr;
};
size_t scan_partials_needed(uint64_t n);
hipError_t launch_scan(const uint32_t* in, uint64_t n, uint64_t* out, uint64_t* partial,
                       hipStream_t st);
size_t scatter_lds_bytes(int nbk);
// LDS of a 1024-thread, 8192-tuple tile with whole-line carries
size_t scatter_lds_bytes_big(int nbk);
// One pass of a partition.  SCATTER_ONLY: the partition's only pass (p1 = bits),
// keys and values in two arrays on both sides.  SCATTER_FIRST: by the top p1
// bits, into whole 8-byte tuples (key, value) at tmp.  SCATTER_SECOND: those by the
// remaining bits, W2 workgroups per first-pass bucket, into two arrays.  The first
// two also write the sub-bucket starts; SCATTER_SECOND plans the probe when plan
// is not null (both sides' starts are known then).  The launch reserves at least
// min_lds bytes of LDS per workgroup (a way to cap workgroups per CU).
enum { SCATTER_ONLY = 0, SCATTER_FIRST, SCATTER_SECOND };
hipError_t launch_scatter(int pass, const PartSide* sides, int n, const PlanArgs* plan, uint64_t* err, int wg,
                          size_t min_lds, hipStream_t st);
hipError_t launch_bloom_build(const uint32_t* rkey, const uint64_t* r_start, int bits,
                              const BloomGeom& g, uint64_t* filter, hipStream_t st);
hipError_t launch_bloom_prefilter(const uint32_t* skey, const uint32_t* sval, uint64_t n,
                                  const uint64_t* filter, const BloomGeom& g, uint32_t* okey,
                                  uint32_t* oval, uint64_t out_cap, uint64_t* count, uint64_t* err,
                                  int num_cu, hipStream_t st);
// tile_ctr: 8 zeroed counters, one per XCD (the tile order of each XCD)
// (tuples: S after SCATTER_FIRST)
hipError_t launch_filter_l1(const uint32_t* tuples, const uint64_t* sb_start, int bits,
                            int bits2, const uint64_t* filter, const BloomGeom& g, uint32_t* okey,
                            uint32_t* oval, uint64_t out_cap, uint32_t* s_fill, uint64_t* count,
                            uint64_t* tile_ctr, uint64_t* err, int num_cu, hipStream_t st);
// S in chunks, one probe after the last chunk: each chunk's S' stays in its own
// region of a pool (starting at base); launch_pool_note records its pieces
// (sub-bucket sb: s_cnt[sb] tuples when not null, else the region's length, at
// base + s_start[sb]) in this chunk's row cnt / off of the piece table (nbins
// entries each) and adds them to *total.  launch_pool_start sums the table over
// nch chunks into totals and scans them into start (nbins + 1 entries);
// launch_pool_merge gathers every sub-bucket's pieces into
// [start[sb], start[sb + 1]) of ok / ov (err |= 16 past out_cap).
hipError_t launch_pool_note(const uint64_t* s_start, const uint32_t* s_cnt, int nbins, uint64_t base, uint32_t* cnt,
                            uint64_t* off, uint64_t* total, hipStream_t st);
hipError_t launch_pool_start(const uint32_t* cnt, int nch, int nbins, uint32_t* totals, uint64_t* start,
                             uint64_t* partials, hipStream_t st);
hipError_t launch_pool_merge(const uint32_t* pk, const uint32_t* pv, const uint32_t* cnt, const uint64_t* off,
                             int nch, int nbins, const uint64_t* start, uint32_t* ok, uint32_t* ov,
                             uint64_t out_cap, uint64_t* err, hipStream_t st);
hipError_t launch_plan(const PlanArgs& plan, hipStream_t st);
// probe_mean: probe tuples of a sub-bucket on average, as far as the host knows
hipError_t launch_probe(int tile, uint64_t probe_mean, const uint32_t* rk, const uint32_t* rv, const uint64_t* r_start,
                        const uint32_t* sk, const uint32_t* sv, const uint64_t* s_start,
                        const uint32_t* s_cnt, int bits, uint32_t slice, const HeavyItem* items,
                        const uint64_t* n_items, uint64_t item_cap, uint64_t* work_ctr, uint64_t* out_count,
                        uint64_t out_cap, uint32_t* o_key, uint32_t* o_rval, uint32_t* o_sval, int num_cu,
                        uint64_t* timers, hipStream_t st);
// Direct join of unpartitioned relations (small build sides): begin clears the
// join's counters and its filter (64-bit blocks), bloom fills the filter, join
// emits the rows.
// ns_dev (nullable): device-side length of S, at most ns.  *long_run is set, and the
// rows are not all there, when a table has a run of equal keys that makes the join by
// partitions (of bits radix bits) the faster one.
hipError_t launch_direct_begin(uint64_t* ctr, int n_ctr, uint64_t* filter, uint64_t blocks, hipStream_t st);
hipError_t launch_direct_bloom(const uint32_t* rkey, uint64_t n, const BloomGeom& g, uint64_t* filter,
                               hipStream_t st);
hipError_t launch_join_direct(const uint32_t* rk, const uint32_t* rv, uint64_t nr, const uint32_t* sk,
                              const uint32_t* sv, uint64_t ns, const uint64_t* ns_dev, int bits,
                              uint64_t* long_run, uint64_t* out_count, uint64_t out_cap, uint32_t* o_key,
                              uint32_t* o_rval, uint32_t* o_sval, int num_cu, hipStream_t st);
// Workgroups of a probe launch (persistent: a fixed number per CU).  With
// timers, every workgroup adds its phase times (ticks, PT_* order of bj_tiles.h,
// PT_N = 5 per workgroup) to its slots; the caller clears them.
int probe_grid(int tile, int num_cu);
constexpr int PROBE_TIMER_SLOTS = 5;

}  // namespace bj
