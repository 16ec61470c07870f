// eimp_internal.h -- types shared by the device kernels and the host engine.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace eimp {

// Elements of one condensed-reference block: 16 consecutive cref rows are
// stored transposed, one uint16 per conditioning haplotype (bit j = row
// 16*b + j).  The PBWT kernel carries these bits with each haplotype index
// so that a step needs no gather.
constexpr int kBlockRows = 16;

// Excluded haplotype (ignored target sample or second hap of a haploid
// reference sample) in the distance array: never selected.
constexpr uint32_t kExcluded = 0xFFFFFFFFu;

// Per-target flags
enum : uint32_t {
    TF_SELECT = 1u,    // K < Ncorr: top-K selection by (nerr, idx)
    TF_IDENTITY = 2u,  // bestHaps == 0..N_ad-1 (whole panel, no exclusions)
    TF_RAW = 4u,       // output rows hold data words only (raw layout)
};

// Output row layouts and their stride in uint32 per stored row
enum : uint32_t {
    LAYOUT_GPU = 0u,      // 4*Kwords: (data, cumulative zeros) pairs, tail pairs zero
    LAYOUT_COMPACT = 1u,  // 2*ceil(K/32) pairs, the CPU layout
    LAYOUT_RAW = 2u,      // roundToMultiple(K,512)/32 data words, tail words all ones
};
__host__ __device__ inline uint32_t row_stride(uint32_t K, uint32_t layout) {
    return layout == LAYOUT_COMPACT ? 2 * ((K + 31) / 32)
         : layout == LAYOUT_RAW     ? (K + 511) / 512 * 16
                                    : 4 * ((K + 511) / 512 * 8);
}

// Per-target record in device memory.  Filled by the host in two stages:
// the prep fields before phase A, the build fields (Mp, offsets) after the
// split counts are known.
struct TgtDev {
    // inputs
    const uint64_t *gt;    // window-relative genotype words (is0, is2 interleaved)
    uint64_t s0;           // window start (panel site)
    uint32_t W;            // window sites
    uint32_t K;            // conditioning haplotypes (<= Ncorr)
    int32_t ignore;        // sample whose haplotypes are skipped, -1 none
    uint32_t flags;        // TF_*
    float cMmaxSplit;
    uint32_t pad0;
    // phase A (prep) outputs / scratch
    uint32_t *nerr;        // N_ad   (TF_SELECT only)
    uint32_t *bh;          // K      bestHaps ascending
    uint64_t *bhflags;     // unit_words(N_ad)
    const uint64_t *mand;  // all-ones-at-site bits (window or panel coordinates)
    const uint64_t *mor;   // any-one-at-site bits
    uint64_t *mand_w;      // window-relative accumulators written by k_monos (TF_IDENTITY off)
    uint64_t *mor_w;
    uint64_t mono_off;     // bit offset of window site 0 in mand/mor
    uint32_t *splitsites;  // W
    uint64_t *splits;      // unit_words(W)
    float *cMdiffs;        // W + 1
    uint32_t *stats;       // [0] S, [1] ncalls, [2] deferred (stream contexts), [3] best haps set
    // phase B (build)
    uint16_t *cref;        // nblk x Kpad, transposed 16-row blocks
    int32_t *count0;       // Mp
    uint32_t *out;         // 2 x Mp x RS uint32 (forward rows, then backward rows)
    uint16_t *seg;         // 2 x nseg x 3 x Kpad: segments of the chains (nseg > 1)
    uint16_t *hdr;         // 2 x nblk: runs listed in a block's rows (forward, then backward blocks)
    uint64_t *digest;      // [0] pbwt words, [1] count0
    uint32_t Mp;
    uint32_t Kpad;         // K rounded up to 64
    uint32_t RS;           // output row stride in uint32
    uint32_t S;
    uint32_t nseg, seglen; // segments of each chain, blocks of a segment
};

// Device-side header of a batch run by a stream context (device-driven
// path: no host synchronisation between the phases).
struct BatchDev {
    uint32_t n;           // targets in this submission (written by the host)
    uint32_t ncref;       // cref blocks queued by k_plan: subset (gather) targets
    uint32_t npbwt[2];    // PBWT chain items queued by k_plan, by chain shape: rows
    uint32_t nfit;        // targets whose outputs fit the pools
    uint32_t cref_ctr;    // work-queue counters (zeroed by k_plan)
    uint32_t pbwt_ctr[2];
    uint32_t ncref_id;    // cref blocks of whole-panel (identity) targets
    uint32_t cref_id_ctr;
    // cref queue order per kind ([0] subset, [1] identity): 0 target-major
    // (prefix sums in blockpref), else block-major over the nrr targets listed
    // in blockpref (item i = block i / nrr of target i % nrr)
    uint32_t rr[2];
    uint32_t nrr[2];
    // subset cref items: blocks of a group, parts of the haplotypes, passes of a part
    uint32_t cref_grp, cref_parts, cref_per;
    // chain items of cut chains: ranks of the segments, then their combination
    uint32_t nrank[2], ncomb[2], rank_ctr[2], comb_ctr[2];
};

// 16-row blocks per work item of the subset cref kernel in a full batch
constexpr uint32_t kCrefGroup = 128;
constexpr uint32_t kCrefThreads = 256;

// cref work item: target t, blocks [b0, b1), passes [p0, p1) of kCrefThreads
// haplotypes
struct CrefItem {
    uint32_t t, b0, b1, p0, p1;
};

// Cut of a batch's subset cref work (n128 groups of kCrefGroup blocks, up to K
// haplotypes) into at least `want` items where it can be: first the
// haplotypes into parts, then groups of 32 blocks.  A batch with that many
// groups stays whole: smaller groups read more of each row's cache lines
// twice (96 targets on the 200,000-haplotype panel are 1.6 ms whole).
__host__ __device__ inline void cref_cut(uint32_t n128, uint32_t K, uint32_t want, uint32_t &grp,
                                         uint32_t &parts) {
    const uint32_t passes = (K + kCrefThreads - 1) / kCrefThreads;
    grp = kCrefGroup;
    parts = 1;
    if (n128 >= want || !n128) return;
    uint32_t groups = n128;
    if ((uint64_t)n128 * passes < want) {
        grp = 32;
        groups = 4 * n128;
    }
    parts = (want + groups - 1) / groups;
    if (parts > passes) parts = passes;
    if (parts < 1) parts = 1;
}

// 16-row blocks of a target's PBWT, both directions
__host__ __device__ inline uint32_t pbwt_blocks(uint32_t Mp) { return 2 * ((Mp + 15) / 16); }

// k_rows work item: block q of chain 2 t + direction, its runs; and the words
// that count the lists of items
struct RowItem {
    uint32_t chain, q, runs;
};
constexpr uint32_t kRowsCounters = 4;

// PBWT chain items (k_order): target t, direction (0 fwd, 1 bck), blocks
// [q0, q1) in processing order, segment seg
enum : uint32_t { CHAIN_ROWS, CHAIN_STARTS, CHAIN_RANK_UP, CHAIN_RANK_DOWN, CHAIN_COMBINE };
struct OrderItem {
    uint32_t t, dir, kind, seg, q0, q1;
};

// Cut of a chain of nblk blocks for segments of about L blocks (0: none).  A
// cut chain is three times the blocks (both rank passes and the rows), so its
// latency, 2 len + about 2 block times per segment for the combination, is
// least near sqrt(nblk) segments and no gain below 3.
__host__ __device__ inline uint32_t seg_isqrt(uint32_t x) {
    uint32_t r = 0;
    for (uint32_t b = 1u << 15; b; b >>= 1)
        if ((uint64_t)(r | b) * (r | b) <= x) r |= b;
    return r;
}
__host__ __device__ inline uint32_t seg_split(uint32_t nblk, uint32_t L, uint32_t &len) {
    len = nblk;
    if (!L) return 1;
    uint32_t s = (nblk + L - 1) / L;
    const uint32_t most = seg_isqrt(nblk);
    if (s > most) s = most;
    if (s < 3) return 1;
    len = (nblk + s - 1) / s;
    return (nblk + len - 1) / len;
}
// Time of a block of a chain that has its CU to itself, about 0.5 us (2.4 us
// at K = 1,000, 4.3 at 3,000, 6.7 at 10,000), and a chain's latency and work
// (one direction) in these units.
__host__ __device__ inline uint64_t seg_block_cost(uint32_t Kpad) { return 4 + Kpad / 1024; }
__host__ __device__ inline uint64_t seg_path(uint32_t nblk, uint32_t S, uint32_t len, uint32_t Kpad) {
    return seg_block_cost(Kpad) * (S > 1 ? 2 * ((uint64_t)len + S) : nblk);
}
__host__ __device__ inline uint64_t seg_work(uint32_t nblk, uint32_t S, uint32_t Kpad) {
    return seg_block_cost(Kpad) * (S > 1 ? 3 * (uint64_t)nblk + 2 * S : nblk);
}
// Expected time of a batch's chains for candidate L: the longest chain, or all
// work over par / 10 chains' worth of parallel work.
__host__ __device__ inline uint64_t seg_time(uint64_t path, uint64_t work, uint32_t par) {
    const uint64_t w = 20 * work / par;
    return path > w ? path : w;
}
// The longest chain takes longer than all work spread over the CUs, by a
// quarter: the shape with twice the threads, which moves a chain faster and
// holds fewer of them on a CU (K = 10,000, 1024 against 512 threads: one target
// of 45,000 rows 2.87 against 3.25 ms as a call, 192 chains 24.3 against 26.0,
// 512 of very different lengths 55.5 against 61.0; 384 equal ones 22.6 against
// 19.2).
__host__ __device__ inline bool seg_latency_bound(uint64_t path, uint64_t work, uint32_t ncu) {
    return 4 * path * ncu >= 5 * 2 * work;
}
// candidates: segments of 4 << c blocks, c < kSegCands, and none
constexpr int kSegCands = 14;
// uint16 words of a target's segments, both directions
__host__ __device__ inline uint64_t seg_words(uint32_t S, uint32_t Kpad) {
    return S > 1 ? 6ull * S * Kpad : 0ull;
}
// most segments of a batch (target, direction, segment)
constexpr uint32_t kMaxSegments = 8192;

// One item of the large-K PBWT kernel (order in global memory): one
// direction of one target, or the panel PBWT.
struct BigItem {
    const uint64_t *rows;    // row r of this item's rows (bit k = haplotype k) at rows + r * rstride
    uint64_t rstride;        // uint64 words per row
    uint32_t *out;           // 2 x Mp (or Mp) rows of RS uint32, this direction's first row
    int32_t *count0;         // Mp zero counts (forward items), else null
    int32_t *absperm;        // (Mp + 1) x K absolute orders (panel PBWT) or null
    uint32_t *ord0, *ord1;   // Kpad indexes each
    uint64_t *digest;        // [0] += digest of the rows, or null
    uint64_t gbase;          // global index of this direction's first logical word (digest)
    uint32_t K, Mp, RS, rev, raw, pad;
};

// Output pool and queues of a stream context, for k_plan.  Each target gets
// one contiguous region of the pool: cref blocks, count0, PBWT rows.
struct PlanArgs {
    char *pool;
    uint64_t pool_cap;
    uint64_t *dig_base;    // 2 words per target
    uint32_t *blockpref;     // nmax + 1 prefix sums of cref blocks (gather targets)
    uint32_t *blockpref_id;  // nmax + 1 prefix sums of cref blocks (identity targets)
    OrderItem *rows_items;   // 2 * nmax + kMaxSegments
    OrderItem *rank_items;   // 2 * kMaxSegments
    OrderItem *comb_items;   // 2 * nmax
    uint16_t *seg;           // seg_cap words for the segments of cut chains
    uint64_t seg_cap;
    uint32_t cref_want;      // subset cref items that fill the device
    uint32_t ncu, shapes;    // compute units; 2: the context has a latency shape too
    uint32_t seg_par;        // chains' worth of parallel work, times 10
    uint32_t *rowpref;       // kRowsCounters, then nmax + 1 prefix sums of pbwt_blocks
    uint32_t layout;         // LAYOUT_*
    uint32_t digest;
    uint32_t ident_ok;       // identity targets take the transpose kernel
    uint32_t pad;
};

// Bytes of a target's region in a stream context's pool (each part rounded
// to 256 bytes): cref blocks, count0, forward + backward PBWT rows.
__host__ __device__ inline uint64_t region_cref_bytes(uint32_t Mp, uint32_t Kpad) {
    return ((uint64_t)((Mp + 15) / 16) * Kpad * 2 + 255) / 256 * 256;
}
__host__ __device__ inline uint64_t region_c0_bytes(uint32_t Mp) {
    return ((uint64_t)Mp * 4 + 255) / 256 * 256;
}
__host__ __device__ inline uint64_t region_out_bytes(uint32_t Mp, uint32_t RS) {
    return (2ull * Mp * RS * 4 + 255) / 256 * 256;
}

// Panel in device memory (resident)
struct PanelDev {
    const uint64_t *hap;   // N_ad rows x hap_stride words (bit m = site m)
    const uint64_t *site;  // M rows x site_stride words (bit h = hap h)
    const float *cM;       // M
    const uint8_t *haploid; // N_ad/2 flags or null
    const uint64_t *pand;  // panel-level all-ones bits per site
    const uint64_t *por;   // panel-level any-one bits per site
    uint64_t hap_stride, site_stride;
    uint32_t N_ad, N_corr, M, pad;
};

// Output digest (the CPU oracle computes the same sums): over the PBWT words,
// sum of rotl32(v ^ g * 0x9E3779B1, g mod 32), g the word's global index;
// over count0, sum of fmix32(c0 + r * 0x7FEB352D + 0x68E31DA4).  Each term is
// a bijection of its word.
// 32-bit finaliser of MurmurHash3 (Appleby).
__host__ __device__ inline uint32_t fmix32(uint32_t h) {
    h ^= h >> 16;
    h *= 0x85EBCA6Bu;
    h ^= h >> 13;
    h *= 0xC2B2AE35u;
    h ^= h >> 16;
    return h;
}
constexpr uint32_t kDigKey = 0x9E3779B1u;
__host__ __device__ inline uint32_t dig_word(uint64_t g, uint32_t v) {
    const uint32_t x = v ^ ((uint32_t)g * kDigKey);
    const uint32_t r = (uint32_t)(g & 31);
    return r ? (x << r) | (x >> (32 - r)) : x;
}
__host__ __device__ inline uint32_t dig_count0(uint32_t r, int32_t c0) {
    return fmix32((uint32_t)c0 + r * 0x7FEB352Du + 0x68E31DA4u);
}

}  // namespace eimp
