// eimp_kernels.hip -- gfx950 kernels of the phasing pre-stage.
//
// Everything here is integer/bitwise work; wave64 ballots and LDS do the
// per-site and per-step partitions, HBM is streamed with coalesced loads.
//
//   k_site_to_hap    site-major -> hap-major panel (64x64 bit tiles via LDS)
//   k_panel_mono     per-site "all ones" / "any one" bits of the whole panel
//   k_distance       nerr(h) = sum popcount((is0 & h) | (is2 & ~h))
//                    (GenotypeVector::compare_withPreInit, src/Datatypes.cpp:107-116)
//   k_select         exact K smallest (nerr, h), ascending h
//                    (Target::findBestHaps, src/Target.cpp:779-875)
//   k_monos          AND / OR of the chosen rows per window word
//                    (Target::findMonos, src/Target.cpp:878-897)
//   k_splits         split / call sites, one wave per target
//                    (Target::findCallLocs, src/Target.cpp:900-950)
//   k_bits_to_list   bitmap -> ascending index list (drop-in inputs)
//   k_cref           condensed reference in 16-row transposed blocks
//                    (Target::condensedReferenceT, src/Target.cpp:953-1059)
#include <algorithm>
#include <map>
#include <mutex>

#include "eimp_device.h"
#include "eimp_launch.h"

namespace eimp {

// bits [bitoff, bitoff+64) of a bit row with `words` readable words
__device__ __forceinline__ uint64_t funnel(const uint64_t *__restrict__ row, uint64_t bitoff,
                                           uint64_t words) {
    uint64_t w = bitoff >> 6;
    uint32_t sh = (uint32_t)(bitoff & 63);
    uint64_t lo = w < words ? row[w] : 0ull;
    if (sh == 0) return lo;
    uint64_t hi = (w + 1) < words ? row[w + 1] : 0ull;
    return (lo >> sh) | (hi << (64 - sh));
}

__device__ __forceinline__ bool excluded_hap(const PanelDev &P, int32_t ignore, uint32_t h) {
    uint32_t nr = h >> 1;
    if ((int32_t)nr == ignore) return true;
    return (h & 1u) && P.haploid && P.haploid[nr];
}

// ---------------------------------------------------------------------------
// panel set-up
// ---------------------------------------------------------------------------
// grid (ceil(hap_stride/4), ceil(N_ad/64)), block 256: one 64-hap x 256-site tile
__global__ __launch_bounds__(256) void k_site_to_hap(PanelDev P, uint64_t *__restrict__ hap) {
    __shared__ uint64_t tile[256];
    const uint32_t tid = threadIdx.x, wave = tid >> 6, l = lane_id();
    const uint64_t hb = blockIdx.y;
    const uint64_t sw0 = (uint64_t)blockIdx.x * 4;
    const uint64_t m = sw0 * 64 + tid;
    tile[tid] = (m < P.M && hb < P.site_stride) ? P.site[m * P.site_stride + hb] : 0ull;
    __syncthreads();
    uint64_t out = 0;
#pragma unroll 8
    for (int j = 0; j < 64; j++) out |= ((tile[wave * 64 + j] >> l) & 1ull) << j;
    const uint64_t h = hb * 64 + l, sw = sw0 + wave;
    if (h < P.N_ad && sw < P.hap_stride) hap[h * P.hap_stride + sw] = out;
}

// grid ceil(M/4), block 256: one wave per site
__global__ __launch_bounds__(256) void k_panel_mono(PanelDev P, uint64_t *__restrict__ pand,
                                                   uint64_t *__restrict__ por) {
    const uint32_t wave = threadIdx.x >> 6, l = lane_id();
    const uint64_t m = (uint64_t)blockIdx.x * 4 + wave;
    if (m >= P.M) return;
    const uint64_t nw = (P.N_ad + 63) / 64;
    uint32_t c = 0;
    for (uint64_t w = l; w < nw; w += 64) c += __popcll(P.site[m * P.site_stride + w]);
    c = wave_sum(c);
    if (l == 0) {
        unsigned long long bit = 1ull << (m & 63);
        if (c == P.N_ad) atomicOr((unsigned long long *)&pand[m >> 6], bit);
        if (c > 0) atomicOr((unsigned long long *)&por[m >> 6], bit);
    }
}

// ---------------------------------------------------------------------------
// a3: distances for groups of DIST_G targets.  block 256: DIST_W haplotypes
// (DIST_H per wave) x DIST_G targets per workgroup.  Over the union of the
// group's windows, 64 panel words at a time, the group's genotype words are
// staged in LDS shifted to panel alignment (sites outside a target's window
// zero); each lane then reads one word of its DIST_H haplotype rows once for all
// targets of the group whose window reaches these words.  nerr = sum of
// popcount((is0 & h) | (is2 & ~h)) over the window (compare_withPreInit,
// src/Datatypes.cpp:107-116).
//
// Bound by vector instructions (four per word, haplotype and target) once the
// loads are out of the way: the next 64 words of haplotypes and genotypes are
// loaded while these are compared, the LDS words alternate between two halves
// (one barrier per 64), and the staging, whose cost per wave does not depend on
// DIST_H, is shared by eight haplotypes.  The grid is (8 target groups, groups
// of 8 haplotype blocks): workgroups go to the XCDs in turn, so that all target
// groups of a haplotype block run on one XCD and all but the first find its rows
// in that L2.
// 256 targets with 10,000 to 100,000 sites on 20,000 haplotypes: 2,275 us with
// four haplotypes per wave, loads after the barrier and one reduction per sum,
// 1,185 us so; 96 targets with 20,000 sites on 200,000 haplotypes: 2,415 and
// 1,513 us (three waves per SIMD; four spill and take longer).
// ---------------------------------------------------------------------------
constexpr int DIST_G = 8;
constexpr int DIST_H = 8;
constexpr uint32_t DIST_W = 4 * DIST_H;

// genotype words (is0, is2) around panel word p of a target, its window's words
// q and q + 1, as loaded and shifted to panel alignment, bits of sites outside
// [s0, s0 + W) zero
struct GtWords {
    uint64_t a0 = 0, b0 = 0, a1 = 0, b1 = 0;
};
__device__ __forceinline__ GtWords gt_load(gptr_t<const uint64_t> gt, uint64_t s0, uint64_t W, uint64_t p) {
    const int64_t nq = (int64_t)((W + 63) / 64), q = ((int64_t)(64 * p) - (int64_t)s0) >> 6;
    GtWords r;
    if (q >= 0 && q < nq) {
        r.a0 = gt[2 * q];
        r.b0 = gt[2 * q + 1];
    }
    if (q + 1 >= 0 && q + 1 < nq) {
        r.a1 = gt[2 * q + 2];
        r.b1 = gt[2 * q + 3];
    }
    return r;
}
__device__ __forceinline__ void gt_align(const GtWords &r, uint64_t s0, uint64_t W, uint64_t p, uint64_t &a,
                                         uint64_t &b) {
    const uint32_t sh = (uint32_t)(0u - (uint32_t)s0) & 63u;  // (64 p - s0) mod 64
    a = r.a0 >> sh;
    b = r.b0 >> sh;
    if (sh) {
        a |= r.a1 << (64 - sh);
        b |= r.b1 << (64 - sh);
    }
    // panel bits at or beyond the window end
    const int64_t end = (int64_t)s0 + (int64_t)W - (int64_t)(64 * p);
    const uint64_t keep = end >= 64 ? ~0ull : (end <= 0 ? 0ull : ((1ull << end) - 1));
    a &= keep;
    b &= keep;
}

// Sums of 64 values over the wave: lane l returns the sum of v[wave_sums_index(l)]
// over all lanes.  Each stage adds two halves of the lanes and halves the values
// that a lane carries: 32 and 16 by swapping rows, the rest by DPP.
__device__ __forceinline__ uint32_t wave_sums_index(uint32_t l) {
    return (l & 0x38u) | ((l & 1u) << 2) | (l & 2u) | ((l >> 2) & 1u);
}
__device__ __forceinline__ uint32_t wave_sums(uint32_t (&v)[64]) {
    const uint32_t l = lane_id();
#pragma unroll
    for (int k = 0; k < 32; k++) {
        const u32x2 s = __builtin_amdgcn_permlane32_swap(v[k], v[k + 32], false, false);
        v[k] = s.x + s.y;
    }
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const u32x2 s = __builtin_amdgcn_permlane16_swap(v[k], v[k + 16], false, false);
        v[k] = s.x + s.y;
    }
    auto fold = [&](auto ctrl, uint32_t bit, int k, int half) {
        const uint32_t keep = l & bit ? v[k + half] : v[k], give = l & bit ? v[k] : v[k + half];
        v[k] = keep + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)give, decltype(ctrl)::value, 0xF, 0xF, true);
    };
#pragma unroll
    for (int k = 0; k < 8; k++) fold(std::integral_constant<int, 0x128>{}, 8u, k, 8);  // lane ^ 8
#pragma unroll
    for (int k = 0; k < 4; k++) fold(std::integral_constant<int, 0xB1>{}, 1u, k, 4);   // lane ^ 1
#pragma unroll
    for (int k = 0; k < 2; k++) fold(std::integral_constant<int, 0x4E>{}, 2u, k, 2);   // lane ^ 2
    const uint32_t keep = l & 4u ? v[1] : v[0], give = l & 4u ? v[0] : v[1];
    return keep + (uint32_t)__shfl_xor((int)give, 4);
}

__global__ __launch_bounds__(256) void k_distance(PanelDev P, const TgtDev *__restrict__ tg,
                                                 const uint32_t *__restrict__ tlist, uint32_t nlist,
                                                 const uint32_t *__restrict__ d_n) {
    // tlist: targets that select (nlist of them); without it every target of the
    // batch (size *d_n), those that do not select are skipped
    __shared__ uint64_t sg[2][DIST_G][64][2];
    const uint32_t n = tlist ? nlist : *d_n;
    const uint32_t j0 = (blockIdx.x >> 3) * DIST_G;
    if (j0 >= n) return;
    // panel words of the targets' windows; empty for those left out
    uint32_t pb[DIST_G], pe[DIST_G];
    uint32_t plo = ~0u, phi = 0;
#pragma unroll
    for (int j = 0; j < DIST_G; j++) {
        const uint32_t q = min(j0 + (uint32_t)j, n - 1);
        const TgtDev &T = tg[tlist ? tlist[q] : q];
        pb[j] = pe[j] = 0;
        if (j0 + j < n && (T.flags & TF_SELECT)) {
            pb[j] = (uint32_t)(T.s0 / 64);
            pe[j] = (uint32_t)((T.s0 + T.W + 63) / 64);
            plo = min(plo, pb[j]);
            phi = max(phi, pe[j]);
        }
    }
    if (phi == 0) return;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), l = lane_id();
    // this wave stages the words of targets wave and wave + 4
    gptr_t<const uint64_t> sgt[2];
    uint64_t ss0[2], sW[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const uint32_t q = min(j0 + wave + 4u * (uint32_t)u, n - 1);
        const TgtDev &T = tg[tlist ? tlist[q] : q];
        sgt[u] = gmem(T.gt);
        ss0[u] = T.s0;
        sW[u] = T.W;
    }
    for (uint32_t hblk = blockIdx.y * 8 + (blockIdx.x & 7u); hblk * DIST_W < P.N_ad; hblk += gridDim.y * 8) {
        const uint32_t hb = hblk * DIST_W + wave * DIST_H;
        uint32_t e[64];
#pragma unroll
        for (int k = 0; k < 64; k++) e[k] = 0;
        uint64_t hv[DIST_H], hx[DIST_H];
        GtWords gw[2];
        const gptr_t<const uint64_t> row0 = gmem(P.hap) + (uint64_t)hb * P.hap_stride;
        auto load = [&](uint32_t c0) {
#pragma unroll
            for (int u = 0; u < 2; u++) gw[u] = gt_load(sgt[u], ss0[u], sW[u], c0 + l);
#pragma unroll
            for (int i = 0; i < DIST_H; i++)
                hx[i] = (hb + i < P.N_ad && c0 + l < phi) ? row0[i * P.hap_stride + c0 + l] : 0ull;
        };
        auto stage = [&](uint32_t c0, uint32_t half) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                uint64_t a, b;
                gt_align(gw[u], ss0[u], sW[u], c0 + l, a, b);
                sg[half][wave + 4 * u][l][0] = a;
                sg[half][wave + 4 * u][l][1] = b;
            }
        };
        load(plo);
        stage(plo, 0);
        uint32_t half = 0;
        for (uint32_t c0 = plo; c0 < phi; c0 += 64, half ^= 1u) {
#pragma unroll
            for (int i = 0; i < DIST_H; i++) hv[i] = hx[i];
            __syncthreads();  // half is written, and everyone is done with the other
            if (c0 + 64 < phi) load(c0 + 64);
#pragma unroll
            for (int j = 0; j < DIST_G; j++) {
                if (c0 >= pe[j] || c0 + 64 <= pb[j]) continue;
                const uint64_t g0 = sg[half][j][l][0], g2 = sg[half][j][l][1];
#pragma unroll
                for (int i = 0; i < DIST_H; i++)
                    e[j * DIST_H + i] += (uint32_t)__popcll((g0 & hv[i]) | (g2 & ~hv[i]));
            }
            if (c0 + 64 < phi) stage(c0 + 64, half ^ 1u);
        }
        __syncthreads();  // the next block's first words go to either half
        const uint32_t s = wave_sums(e), k = wave_sums_index(l), h = hb + k % DIST_H, q = j0 + k / DIST_H;
        if (q < n && h < P.N_ad) {
            const TgtDev &T = tg[tlist ? tlist[q] : q];
            if (T.flags & TF_SELECT) T.nerr[h] = excluded_hap(P, T.ignore, h) ? kExcluded : s;
        }
    }
}

// ---------------------------------------------------------------------------
// a4: exact top-K selection / take-all.  grid n, block SEL_NT.  Workgroups of
// 256 threads fit on CUs beside a PBWT workgroup, so a context's selection can
// run while another context's PBWT holds the device.
//
// One workgroup per target, so its time is what the loops over the N distances
// wait for: eight loads in flight in the radix passes, and a compaction that
// takes 2,048 haplotypes between two barriers, each wave counting and placing
// 512 neighbours by ballots (96 targets on 200,000 haplotypes: 1,735 us with a
// block scan per 256 and one load in flight, 574 us so; four on 20,000: 121 and
// 51 us).
// ---------------------------------------------------------------------------
constexpr int SEL_NT = 256;
constexpr int SEL_NW = SEL_NT / 64;
constexpr int SEL_BINS = 1024;                    // 10-bit digits
constexpr int SEL_BPT = SEL_BINS / SEL_NT;        // bins per thread in the bin scan

constexpr int SEL_SUB = 8;                        // 64-haplotype words per wave and tile
constexpr uint32_t SEL_TILE = SEL_NT * SEL_SUB;

// f(distance) for the haplotypes that are not excluded, in any order
template <class F>
__device__ __forceinline__ void sel_each(const uint32_t *__restrict__ nerr, uint32_t N, F &&f) {
    constexpr uint32_t U = 8;
    for (uint32_t h0 = threadIdx.x; h0 < N; h0 += U * SEL_NT) {
        uint32_t v[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            const uint32_t h = h0 + u * SEL_NT;
            v[u] = h < N ? nerr[h] : kExcluded;
        }
#pragma unroll
        for (uint32_t u = 0; u < U; u++)
            if (v[u] != kExcluded) f(v[u]);
    }
}

// block-wide exclusive scan of one value per thread; also returns the total
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t *s_w, uint32_t &total) {
    const uint32_t wave = threadIdx.x >> 6, l = lane_id();
    uint32_t inc = wave_scan_incl(v);
    if (l == 63) s_w[wave] = inc;
    __syncthreads();
    uint32_t before = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < SEL_NW; w++) {
        uint32_t x = s_w[w];
        tot += x;
        if (w < (int)wave) before += x;
    }
    __syncthreads();
    total = tot;
    return before + inc - v;
}

__global__ __launch_bounds__(SEL_NT) void k_select(PanelDev P, const TgtDev *__restrict__ tg,
                                                   const uint32_t *__restrict__ d_n) {
    if (d_n && blockIdx.x >= *d_n) return;
    const TgtDev &T = tg[blockIdx.x];
    __shared__ uint32_t hist[SEL_BINS];
    __shared__ uint32_t s_w[SEL_NW];
    __shared__ uint32_t s_bin, s_before;
    const uint32_t tid = threadIdx.x, wave = tid >> 6, l = lane_id();
    const uint32_t N = P.N_ad;
    const bool select = (T.flags & TF_SELECT) != 0;
    uint32_t thr = 0, need = 0;
    if (select) {
        const uint32_t *__restrict__ nerr = T.nerr;
        uint32_t mx = 0;
        sel_each(nerr, N, [&](uint32_t v) { mx = max(mx, v); });
        mx = wave_max(mx);
        if (l == 0) s_w[wave] = mx;
        __syncthreads();
        mx = 0;
        for (int w = 0; w < SEL_NW; w++) mx = max(mx, s_w[w]);
        __syncthreads();
        int hi = mx ? 32 - __clz(mx) : 0;
        uint32_t k = T.K;  // rank (1-based) of the threshold value
        uint64_t prefix = 0;
        while (hi > 0) {
            const int lo = hi > 10 ? hi - 10 : 0;
            const uint32_t nb = 1u << (hi - lo);
            for (uint32_t b = tid; b < nb; b += SEL_NT) hist[b] = 0;
            __syncthreads();
            sel_each(nerr, N, [&](uint32_t v) {
                if (((uint64_t)v >> hi) == (prefix >> hi)) atomicAdd(&hist[(v >> lo) & (nb - 1)], 1u);
            });
            __syncthreads();
            // thread tid scans bins SEL_BPT*tid .. SEL_BPT*tid + SEL_BPT-1
            uint32_t cb[SEL_BPT], c = 0, total;
#pragma unroll
            for (int q = 0; q < SEL_BPT; q++) {
                const uint32_t bin = SEL_BPT * tid + (uint32_t)q;
                cb[q] = bin < nb ? hist[bin] : 0u;
                c += cb[q];
            }
            uint32_t ex = block_excl_scan(c, s_w, total);
#pragma unroll
            for (int q = 0; q < SEL_BPT; q++) {
                const uint32_t bin = SEL_BPT * tid + (uint32_t)q;
                if (bin < nb && ex < k && k <= ex + cb[q]) {
                    s_bin = bin;
                    s_before = ex;
                }
                ex += cb[q];
            }
            __syncthreads();
            k -= s_before;
            prefix |= (uint64_t)s_bin << lo;
            hi = lo;
            __syncthreads();
        }
        thr = (uint32_t)prefix;
        need = k;
    }
    // compaction in index order: ties at the threshold value go to the lowest
    // indices.  Per tile wave w holds 64 SEL_SUB neighbours; the waves' counts
    // alternate between two halves, so a tile has one barrier.
    const uint32_t nwords = ((N + 511) / 512) * 8;
    __shared__ uint32_t s_lt[2][SEL_NW], s_eq[2][SEL_NW];
    uint32_t ties_before = 0, sel_before = 0, par = 0;
    auto load = [&](uint32_t base, uint32_t (&v)[SEL_SUB]) {
#pragma unroll
        for (int u = 0; u < SEL_SUB; u++) {
            const uint32_t h = base + (wave * SEL_SUB + (uint32_t)u) * 64 + l;
            v[u] = select && h < N ? T.nerr[h] : 0u;
        }
    };
    uint32_t nx[SEL_SUB];
    load(0, nx);
    for (uint32_t base = 0; base < nwords * 64; base += SEL_TILE, par ^= 1u) {
        uint32_t cur[SEL_SUB];
#pragma unroll
        for (int u = 0; u < SEL_SUB; u++) cur[u] = nx[u];
        load(base + SEL_TILE, nx);
        uint64_t ltm[SEL_SUB], eqm[SEL_SUB];
        uint32_t nlt = 0, neq = 0;
#pragma unroll
        for (int u = 0; u < SEL_SUB; u++) {
            const uint32_t h = base + (wave * SEL_SUB + (uint32_t)u) * 64 + l;
            const bool in = h < N;
            ltm[u] = __ballot(in && (select ? cur[u] < thr : !excluded_hap(P, T.ignore, h)));
            eqm[u] = __ballot(in && select && cur[u] == thr);
            nlt += (uint32_t)__popcll(ltm[u]);
            neq += (uint32_t)__popcll(eqm[u]);
        }
        if (l == 0) {
            s_lt[par][wave] = nlt;
            s_eq[par][wave] = neq;
        }
        __syncthreads();
        uint32_t tb = ties_before, sb = sel_before;
#pragma unroll
        for (int w = 0; w < SEL_NW; w++) {
            const uint32_t c = s_lt[par][w], q = s_eq[par][w];
            const uint32_t taken = min(q, need > ties_before ? need - ties_before : 0u);
            if (w < (int)wave) {
                tb += q;
                sb += c + taken;
            }
            ties_before += q;
            sel_before += c + taken;
        }
#pragma unroll
        for (int u = 0; u < SEL_SUB; u++) {
            const bool tie = (eqm[u] >> l) & 1ull;
            bool sel = ((ltm[u] >> l) & 1ull) || (tie && tb + mbcnt(eqm[u]) < need);
            tb += (uint32_t)__popcll(eqm[u]);
            const uint64_t m = __ballot(sel);
            const uint32_t pos = sb + mbcnt(m);
            sb += (uint32_t)__popcll(m);
            // exactly K when Ncorr is consistent; the bitmap always matches bh
            sel = sel && pos < T.K;
            const uint32_t word = base / 64 + wave * SEL_SUB + (uint32_t)u;
            if (sel) T.bh[pos] = word * 64 + l;
            const uint64_t sm = __ballot(sel);
            if (l == 0 && word < nwords) T.bhflags[word] = sm;
        }
    }
    if (tid == 0) T.stats[3] = sel_before;
    // k_monos starts from these
    if (!(T.flags & TF_IDENTITY)) {
        for (uint32_t w = tid; w < (T.W + 63) / 64; w += SEL_NT) {
            T.mand_w[w] = ~0ull;
            T.mor_w[w] = 0ull;
        }
    }
}

// ---------------------------------------------------------------------------
// a5: monos for targets that select a subset.  grid (ceil(Ww/64), n, parts),
// block MONO_NT: the waves split the part's share of the K chosen rows, lanes
// cover 64 window words (256 threads: they fit beside a PBWT workgroup, as the
// selection does).  A few targets have few word groups, so their rows are cut
// into parts (mono_parts) whose results meet in mand_w / mor_w by atomics; the
// selection has set those to ones and zeros (4 targets of up to 30,000 sites
// and 10,000 rows: 905 us in one part, 70 us in 16).
// ---------------------------------------------------------------------------
constexpr int MONO_NT = 256;
constexpr int MONO_NW = MONO_NT / 64;
// parts for a grid of `groups` workgroups per part
static uint32_t mono_parts(uint64_t groups, uint32_t ncu) {
    const uint64_t want = 4ull * ncu;
    return groups * 2 > want ? 1u : (uint32_t)std::min<uint64_t>(32, want / std::max<uint64_t>(groups, 1));
}

__global__ __launch_bounds__(MONO_NT) void k_monos(PanelDev P, const TgtDev *__restrict__ tg,
                                                   const uint32_t *__restrict__ tlist,
                                                   const uint32_t *__restrict__ d_n) {
    // tlist: targets that need monos; without it every target of the batch (size *d_n)
    if (!tlist && blockIdx.y >= *d_n) return;
    const TgtDev &T = tg[tlist ? tlist[blockIdx.y] : blockIdx.y];
    if (T.flags & TF_IDENTITY) return;
    const uint32_t per = (T.K + gridDim.z - 1) / gridDim.z;
    const uint32_t k0 = blockIdx.z * per, kend = min(T.K, k0 + per);
    if (k0 >= kend || (uint64_t)blockIdx.x * 64 * 64 >= T.W) return;
    __shared__ uint64_t s_and[MONO_NW][64], s_or[MONO_NW][64];
    const uint32_t wave = threadIdx.x >> 6, l = lane_id();
    const uint64_t Ww = (T.W + 63) / 64;
    const uint64_t i = (uint64_t)blockIdx.x * 64 + l;
    const bool valid = i < Ww;
    uint64_t a = ~0ull, o = 0ull;
    const uint64_t bitoff = T.s0 + 64 * i;
    if (valid) {
        uint32_t k = k0 + wave;
        for (; k + 3 * MONO_NW < kend; k += 4 * MONO_NW) {
            uint64_t v0 = funnel(P.hap + (uint64_t)T.bh[k] * P.hap_stride, bitoff, P.hap_stride);
            uint64_t v1 = funnel(P.hap + (uint64_t)T.bh[k + MONO_NW] * P.hap_stride, bitoff,
                                 P.hap_stride);
            uint64_t v2 = funnel(P.hap + (uint64_t)T.bh[k + 2 * MONO_NW] * P.hap_stride, bitoff,
                                 P.hap_stride);
            uint64_t v3 = funnel(P.hap + (uint64_t)T.bh[k + 3 * MONO_NW] * P.hap_stride, bitoff,
                                 P.hap_stride);
            a &= v0 & v1 & v2 & v3;
            o |= v0 | v1 | v2 | v3;
        }
        for (; k < kend; k += MONO_NW) {
            uint64_t v = funnel(P.hap + (uint64_t)T.bh[k] * P.hap_stride, bitoff, P.hap_stride);
            a &= v;
            o |= v;
        }
    }
    s_and[wave][l] = a;
    s_or[wave][l] = o;
    __syncthreads();
    if (wave == 0 && valid) {
        for (int w = 1; w < MONO_NW; w++) {
            a &= s_and[w][l];
            o |= s_or[w][l];
        }
        if (gridDim.z == 1) {
            T.mand_w[i] = a;
            T.mor_w[i] = o;
        } else {
            atomicAnd((unsigned long long *)&T.mand_w[i], (unsigned long long)a);
            atomicOr((unsigned long long *)&T.mor_w[i], (unsigned long long)o);
        }
    }
}

// ---------------------------------------------------------------------------
// a6: split and call sites.  grid n, block 64 (one wave per target).
// Sequential over 64-site chunks; within a chunk het candidates are always
// splits and hom candidates are resolved lowest-first against the cM of the
// previous split (see the comment in the loop).
//
// Only the cM of the last split and the running counts go from chunk to chunk,
// so everything else is kept off that chain: lane x works out the candidate
// masks of chunk x of 64 chunks at once (one coalesced load per array), and the
// positions' cM come in eight chunks ahead.  56,000 sites: 1,040 us with the
// chunk's words loaded in the chunk, 335 us so; 256 targets of 10,000 to
// 100,000 sites 1,320 and 532 us.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t readlane64(uint64_t v, uint32_t lane) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, (int)lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), (int)lane);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ float lane_float(float v, uint32_t lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), (int)lane));
}

__global__ __launch_bounds__(64) void k_splits(PanelDev P, const TgtDev *__restrict__ tg,
                                              const uint32_t *__restrict__ d_n) {
    if (d_n && blockIdx.x >= *d_n) return;
    const TgtDev &T = tg[blockIdx.x];
    const uint32_t l = lane_id();
    const uint32_t W = T.W;
    const uint32_t Ww = (W + 63) / 64;
    const float *__restrict__ cMw = P.cM + T.s0;
    const float thr = T.cMmaxSplit;
    const uint64_t lt = lanemask_lt();
    const uint64_t mono_words = T.mand == T.mand_w ? (uint64_t)((W + 511) / 512) * 8
                                                   : (uint64_t)((P.M + 511) / 512) * 8;
    float Lprev = cMw[0];
    bool started = false;
    uint32_t S = 0, ncalls = 0;
    int64_t lastcall = -1;      // index (in splitsites) of the last het split
    float lastcall_cm = 0.f;
    uint32_t lastcall_word = 0;
    uint64_t lastcall_mask = 0;
    const gptr_t<uint32_t> sites = gmem(T.splitsites);
    const gptr_t<float> diffs = gmem(T.cMdiffs);
    constexpr uint32_t AHEAD = 8;
    float cm[AHEAD], nx[AHEAD];
    auto load_cm = [&](uint32_t c, float (&v)[AHEAD]) {
#pragma unroll
        for (uint32_t u = 0; u < AHEAD; u++) v[u] = cMw[min((c + u) * 64 + l, W - 1)];
    };
    load_cm(0, nx);
    for (uint32_t cb = 0; cb < Ww; cb += 64) {
        // lane x: chunk cb + x
        const uint32_t cl = cb + l;
        uint64_t het = 0, hetc = 0, homc = 0;
        if (cl < Ww) {
            const uint64_t g0 = T.gt[2 * cl], g2 = T.gt[2 * cl + 1];
            const uint64_t ma = funnel(T.mand, T.mono_off + 64ull * cl, mono_words);
            const uint64_t mo = funnel(T.mor, T.mono_off + 64ull * cl, mono_words);
            const uint64_t valid = cl == Ww - 1 && (W & 63) ? (1ull << (W & 63)) - 1 : ~0ull;
            het = valid & ~g0 & ~g2;
            const uint64_t cand = valid & ~(ma | ~mo) & ~(g0 & g2);  // neither mono nor missing
            hetc = cand & het;
            homc = cand & ~het;
        }
        if (!started) {
            // the phasing starts at the first het (:907-913)
            const uint64_t any = __ballot(het != 0ull);
            const uint32_t first = any ? (uint32_t)__ffsll((unsigned long long)any) - 1 : 64u;
            started = any != 0ull;
            if (l < first) hetc = homc = 0ull;
            if (l == first) homc &= ~((het & (0 - het)) - 1);  // het itself has no earlier bit
        }
        const uint32_t cend = min(64u, Ww - cb);
        for (uint32_t i0 = 0; i0 < cend; i0 += AHEAD) {
#pragma unroll
            for (uint32_t u = 0; u < AHEAD; u++) cm[u] = nx[u];
            load_cm(min(cb + i0 + AHEAD, Ww - 1), nx);
#pragma unroll
            for (uint32_t u = 0; u < AHEAD; u++) {
                const uint32_t i = i0 + u, c = cb + i;
                if (i >= cend) break;
                const uint64_t hets = readlane64(hetc, i), homs = readlane64(homc, i);
                uint64_t splitm = hets, pending = homs;
                // Resolve hom candidates.  All splits fixed so far are true splits
                // and L (cM of the previous split) only grows as splits are added,
                // so a pending candidate failing now fails for good, and the
                // lowest one passing now has exactly the true L: accept it and
                // repeat.
                uint64_t below;
                float L;  // cM of the last split before this lane's site
                auto previous = [&]() {
                    below = splitm & lt;
                    const float Ls = __shfl(cm[u], below ? 63 - __clzll((long long)below) : (int)l);
                    L = below ? Ls : Lprev;
                };
                if (!(splitm | pending)) continue;  // hetc is zero already
                previous();
                while (pending) {
                    const uint64_t passm = __ballot(((pending >> l) & 1ull) && (cm[u] - L > thr));
                    if (!passm) break;
                    const uint64_t p = passm & (~passm + 1);  // lowest passing lane
                    splitm |= p;
                    pending = passm & ~p;
                    previous();
                }
                if (splitm) {
                    // emit split sites and their cM differences (src/Target.cpp:943-947)
                    if ((splitm >> l) & 1ull) {
                        const uint32_t idx = S + (uint32_t)__popcll(below);
                        sites[idx] = c * 64 + l;
                        diffs[idx] = cm[u] - L;
                    }
                    if (hets) {
                        const uint32_t top = 63 - (uint32_t)__clzll((long long)hets);
                        const uint64_t upto = top == 63 ? ~0ull : ((1ull << (top + 1)) - 1);
                        lastcall = (int64_t)S + __popcll(splitm & upto) - 1;
                        lastcall_cm = lane_float(cm[u], top);
                        lastcall_word = c;
                        lastcall_mask = splitm & upto;
                        ncalls += (uint32_t)__popcll(hets);
                    }
                    S += (uint32_t)__popcll(splitm);
                    Lprev = lane_float(cm[u], 63 - (uint32_t)__clzll((long long)splitm));
                }
                if (l == i) hetc = splitm;  // this lane's chunk is done: keep its splits
            }
        }
        if (cl < Ww) T.splits[cl] = hetc;
    }
    // no split, or no call: S = 0 (:927-935); else truncate after the last call (:939-940)
    uint32_t Sfin = (S == 0 || ncalls == 0) ? 0u : (uint32_t)(lastcall + 1);
    const uint32_t nwords = ((W + 511) / 512) * 8;
    const uint32_t keep_to = Sfin ? lastcall_word : 0u;
    // words below keep_to hold the loop's values
    for (uint32_t w = (Sfin ? keep_to : 0u) + l; w < nwords; w += 64)
        T.splits[w] = Sfin && w == keep_to ? lastcall_mask : 0ull;
    if (l == 0) {
        if (Sfin) T.cMdiffs[Sfin] = cMw[W - 1] - lastcall_cm;
        T.stats[0] = Sfin;
        T.stats[1] = Sfin ? ncalls : 0u;
    }
}

// ---------------------------------------------------------------------------
// bitmap -> ascending index list (drop-in path: best-haps flags, split
// bitmap).  grid n, block SEL_NT.  which: 0 best haps, 1 split sites.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(SEL_NT) void k_bits_to_list(const TgtDev *__restrict__ tg,
                                                        uint32_t nbits_bh, int which) {
    const TgtDev &T = tg[blockIdx.x];
    __shared__ uint32_t s_w[SEL_NW];
    const uint32_t tid = threadIdx.x;
    const uint64_t *bits = which == 0 ? T.bhflags : T.splits;
    uint32_t *out = which == 0 ? T.bh : T.splitsites;
    const uint32_t nbits = which == 0 ? nbits_bh : T.W;
    const uint32_t cap = which == 0 ? T.K : T.W;  // list capacity; the host rejects a mismatch
    uint32_t before = 0;
    for (uint32_t base = 0; base < nbits; base += SEL_NT) {
        const uint32_t i = base + tid;
        const bool set = i < nbits && ((bits[i >> 6] >> (i & 63)) & 1ull);
        uint32_t total;
        uint32_t pos = before + block_excl_scan(set ? 1u : 0u, s_w, total);
        if (set && pos < cap) out[pos] = i;
        before += total;
    }
    if (tid == 0 && which == 1) T.stats[0] = before;
    if (tid == 0 && which == 0) T.stats[3] = before;
}

// ---------------------------------------------------------------------------
// a7: condensed reference, in 16-row blocks (segments 8b..8b+7): row 2s is the
// OR of the inconsistencies of segment s (mergeInconsistencies,
// src/Target.cpp:1040-1059), row 2s+1 the haplotypes at split s (:986-1003);
// one uint16 per haplotype holds a block's 16 rows.  Two kernels:
//  - whole-panel targets (all N haplotypes in panel order): one work item =
//    one block, its rows built in LDS from the site-major panel (every thread
//    streaming two words through all the block's site rows, 8 independent
//    loads in flight) and transposed in registers;
//  - the others: one work item = a group of blocks and a range of the chosen
//    haplotypes, from the haplotype-major panel, reading only the K chosen
//    rows.  A batch that fills the device takes groups of 128 blocks and all
//    haplotypes in one item (neighbouring groups share cache lines of the
//    rows); one that does not is cut finer (cref_cut).
// count0 (zeros per row) is written by the forward PBWT pass.
// ---------------------------------------------------------------------------
constexpr int CREF_NT = (int)kCrefThreads;
constexpr uint32_t CREF_TW = 512;  // words of the haplotype axis per tile (16 rows: 64 KB)

__host__ __device__ inline uint32_t cref_tile_words(uint32_t nw) {
    return nw < CREF_TW ? nw : CREF_TW;
}

// The rows of block b over words [w0, w0 + tw) into srow[row * tw + (w - w0)]
// (row 2(s-8b)+1 only for s < S).
__device__ __forceinline__ void cref_fill(const PanelDev &P, const TgtDev &T, uint32_t b,
                                          uint32_t w0, uint32_t tw, uint32_t nw, uint64_t *srow) {
    const uint64_t *__restrict__ site = P.site + T.s0 * P.site_stride;
    const uint64_t ss = P.site_stride;
    const uint32_t S = T.S, W = T.W;
    const gptr_t<const uint32_t> splitsites = gmem((const uint32_t *)T.splitsites);
    const gptr_t<const uint64_t> splits = gmem((const uint64_t *)T.splits);
    const gptr_t<const uint64_t> gt = gmem((const uint64_t *)T.gt);
    const uint32_t sa = 8 * b, sb = min(8 * b + 8, S + 1);
    const uint64_t lastmask = (P.N_ad & 63) ? ((1ull << (P.N_ad & 63)) - 1) : ~0ull;
    // sites of the block: after split sa-1 up to split sb-1 (or the window end)
    const uint32_t m0 = sa == 0 ? 0u : splitsites[sa - 1] + 1;
    const uint32_t m1 = sb <= S ? splitsites[sb - 1] + 1 : W;
    for (uint32_t wi = threadIdx.x; wi < tw; wi += 2 * CREF_NT) {
        const uint32_t wj = wi + CREF_NT;  // this thread's second word
        const bool two = wj < tw;
        const uint32_t w = w0 + wi, w2 = w0 + (two ? wj : wi);
        const uint64_t mask0 = (w == nw - 1) ? lastmask : ~0ull;
        const uint64_t mask1 = (w2 == nw - 1) ? lastmask : ~0ull;
        uint32_t s = sa;
        uint64_t a0 = 0, a1 = 0;
        // one pass over the sites; per group of 4 sites the site-row words, the
        // genotype bits and the split bits are independent loads
        for (uint32_t mb = m0; mb < m1; mb += 4) {
            uint64_t v0[4], v1[4];
            uint32_t sp[4], is0[4], is2[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const uint32_t m = mb + u;
                const bool in = m < m1;
                const uint32_t mw = in ? m : m0;
                v0[u] = in ? site[(uint64_t)m * ss + w] : 0ull;
                v1[u] = in ? site[(uint64_t)m * ss + w2] : 0ull;
                sp[u] = (uint32_t)(splits[mw >> 6] >> (mw & 63)) & 1u;
                is0[u] = (uint32_t)(gt[2 * (mw >> 6)] >> (mw & 63)) & 1u;
                is2[u] = (uint32_t)(gt[2 * (mw >> 6) + 1] >> (mw & 63)) & 1u;
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const uint32_t m = mb + u;
                if (m >= m1) break;
                if (sp[u]) {  // split: close segment s, its haplotypes are row 2s+1
                    const uint32_t r0 = 2 * (s - sa);
                    srow[(uint64_t)r0 * tw + wi] = a0 & mask0;
                    srow[(uint64_t)(r0 + 1) * tw + wi] = v0[u];
                    if (two) {
                        srow[(uint64_t)r0 * tw + wj] = a1 & mask1;
                        srow[(uint64_t)(r0 + 1) * tw + wj] = v1[u];
                    }
                    a0 = a1 = 0;
                    s++;
                } else {
                    // HomRef: the ones are inconsistent; HomAlt: the zeros; het/missing: none
                    const uint64_t flip = is2[u] ? ~0ull : 0ull;
                    const uint64_t keep = (is0[u] ^ is2[u]) ? ~0ull : 0ull;
                    a0 |= (v0[u] ^ flip) & keep;
                    a1 |= (v1[u] ^ flip) & keep;
                }
            }
        }
        if (sb == S + 1) {  // the last segment has no split row
            const uint32_t r0 = 2 * (S - sa);
            srow[(uint64_t)r0 * tw + wi] = a0 & mask0;
            if (two) srow[(uint64_t)r0 * tw + wj] = a1 & mask1;
        }
    }
}

// Blocks [b0, b1) of a subset target from the haplotype-major panel, passes
// [p0, p1) of CREF_NT haplotypes.  A wave takes 64 H chosen haplotypes at a
// time, H per lane, and streams their rows over the sites of the blocks, 32
// window sites per step:
//   inc = (v & HomRef) | (~v & HomAlt)  (HomRef = is0 & ~is2, HomAlt =
//                                        is2 & ~is0; split sites and sites
//                                        outside the range masked out)
//   C   = carries of ~splits + inc + cin
// A split kills the carry chain, any other site propagates it and an
// inconsistency generates it, so bit p of C says whether the segment ending
// at split p has an inconsistency (row 2s, mergeInconsistencies,
// src/Target.cpp:1040-1059) and bit p of v is row 2s+1 (src/Target.cpp:986-1003);
// the carry out of bit 31 goes into the next word, and after the last word it
// is the final segment's row 2S.  The split positions are the same for every
// haplotype: a wave-uniform loop over them packs two bits per split into the
// block's uint16.  Only the K chosen rows are read (the site-major layout
// would need all N bits of every site).  Haplotypes K..Kpad-1 get all-ones
// values (the PBWT kernel's padding); count0 comes from the PBWT kernel.
//
// Bound by instruction issue: the loop over the splits takes four vector
// instructions per split and haplotype and six scalar ones per split and wave.
// Where a part has two passes or more a lane takes two haplotypes, which halves
// the scalar ones (256 targets, windows of 10,000 to 100,000 sites, K of 2,000
// to 10,000: 8,784 us with one, 5,803 us with two; 96 targets on the
// 200,000-haplotype panel: 2,763 and 1,611 us); a part of one pass would leave
// half of its waves idle.
template <int H>
__device__ __forceinline__ void cref_range_h(const PanelDev &P, const TgtDev &T, uint32_t b0,
                                               uint32_t b1, uint32_t p0, uint32_t p1) {
    const uint32_t tid = threadIdx.x;
    const uint32_t K = T.K, S = T.S, Kpad = T.Kpad, W = T.W;
    const bool ident = (T.flags & TF_IDENTITY) != 0;
    // the target's arrays, written by earlier kernels and read-only here
    const cptr_t<uint32_t> splitsites = cmem((const uint32_t *)T.splitsites);
    const cptr_t<uint32_t> sp32 = cmem((const uint32_t *)T.splits);
    const cptr_t<uint32_t> gt32 = cmem((const uint32_t *)T.gt);
    const gptr_t<const uint32_t> bh = gmem((const uint32_t *)T.bh);
    const gptr_t<uint16_t> dst = gmem(T.cref);
    const uint32_t sa = 8 * b0, sb = min(8 * b1, S + 1);
    const bool last = sb == S + 1;  // the range ends with the final segment (no split row)
    // window sites [m0, m1): after split sa-1, up to split sb-1 or the window end
    const uint32_t m0 = sa == 0 ? 0u : splitsites[sa - 1] + 1;
    const uint32_t m1 = last ? W : splitsites[sb - 1] + 1;
    const uint32_t i0 = m0 >> 5, i1 = (m1 + 31) >> 5;  // 32-site window words
    if (p0 == 0)
        for (uint32_t k = K + tid; k < Kpad; k += CREF_NT)
            for (uint32_t b = b0; b < b1; b++) dst[(uint64_t)b * Kpad + k] = 0xFFFFu;
    // window word i of a row = bits sh.. of row words q0 + i, q0 + i + 1
    const uint64_t rowlen = 2 * P.hap_stride;  // uint32 words per haplotype row
    const uint64_t q0 = T.s0 >> 5;
    const uint32_t sh = (uint32_t)T.s0 & 31;
    const uint32_t kend = min(K, p1 * CREF_NT), wave = tid >> 6, l = lane_id();
    for (uint32_t kb = p0 * CREF_NT + 64 * H * wave; kb < kend; kb += H * CREF_NT) {
        uint32_t k[H], cin[H], acc[H];
        gptr_t<const uint32_t> row[H];
#pragma unroll
        for (int e = 0; e < H; e++) {
            k[e] = kb + 64 * e + l;
            const uint32_t h = k[e] < kend ? (ident ? k[e] : bh[k[e]]) : 0u;
            row[e] = gmem((const uint32_t *)P.hap) + (uint64_t)h * rowlen;
            cin[e] = acc[e] = 0;
        }
        uint32_t room = 8, b = b0;  // pairs until block b is full
        auto store = [&](uint32_t shift) {
#pragma unroll
            for (int e = 0; e < H; e++)
                if (k[e] < kend) dst[(uint64_t)b * Kpad + k[e]] = (uint16_t)(acc[e] >> shift);
        };
        // The row is read in chunks of 16 words (64 bytes) aligned in the row
        // (rows start on 64-byte boundaries), each as four 16-byte loads, one
        // chunk ahead of the words being processed.  Window word i is bits
        // sh.. of row words q0 + i and q0 + i + 1.
        auto chunk = [&](int e, uint64_t R, uint32_t (&c)[16]) {
            if (R + 16 <= rowlen) {
                const gptr_t<const u32x4> r4 = (gptr_t<const u32x4>)(row[e] + R);
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const u32x4 x = r4[u];
                    c[4 * u] = x[0];
                    c[4 * u + 1] = x[1];
                    c[4 * u + 2] = x[2];
                    c[4 * u + 3] = x[3];
                }
            } else {
#pragma unroll
                for (int u = 0; u < 16; u++) c[u] = R + u < rowlen ? row[e][R + u] : 0u;
            }
        };
        const uint64_t R0 = (q0 + i0) & ~15ull;  // the first chunk
        uint32_t nx[H][16];
#pragma unroll
        for (int e = 0; e < H; e++) chunk(e, R0, nx[e]);
        for (uint64_t R = R0; R < q0 + i1; R += 16) {
            uint32_t w[H][16];
#pragma unroll
            for (int e = 0; e < H; e++) {
#pragma unroll
                for (int u = 0; u < 16; u++) w[e][u] = nx[e][u];
                chunk(e, R + 16, nx[e]);
            }
            // window word of the chunk's first word (below i0 for the first
            // chunk: those words are skipped)
            const int64_t ib = (int64_t)R - (int64_t)q0;
#pragma unroll
            for (int u = 0; u < 16; u++) {
                if (ib + u < (int64_t)i0) continue;
                const uint32_t i = (uint32_t)(ib + u);
                if (i >= i1) break;
                uint32_t rng = ~0u;
                if (i == i0) rng &= ~0u << (m0 & 31);
                if (i == i1 - 1 && (m1 & 31)) rng &= (1u << (m1 & 31)) - 1;
                // the target's words are the same for every lane; a missing
                // genotype sets both is0 and is2 and is no inconsistency
                const uint32_t spw = __builtin_amdgcn_readfirstlane(sp32[i] & rng);
                const uint32_t g0 = gt32[4 * (i >> 1) + (i & 1)], g2 = gt32[4 * (i >> 1) + 2 + (i & 1)];
                const uint32_t hr = __builtin_amdgcn_readfirstlane(g0 & ~g2 & ~spw & rng);
                const uint32_t ha = __builtin_amdgcn_readfirstlane(g2 & ~g0 & ~spw & rng);
                uint32_t v[H], C[H];
#pragma unroll
                for (int e = 0; e < H; e++) {
                    v[e] = __builtin_amdgcn_alignbit(u < 15 ? w[e][(u + 1) & 15] : nx[e][0], w[e][u], sh);
                    const uint32_t inc = (v[e] & hr) | (~v[e] & ha), pr = ~spw;
                    const uint64_t sum = (uint64_t)pr + inc + cin[e];
                    C[e] = (uint32_t)sum ^ pr ^ inc;
                    cin[e] = (uint32_t)(sum >> 32);
                }
                // the splits up to the end of the word or of the block: their
                // rows, inconsistency and allele, enter acc from the top
                for (uint32_t sl = spw; sl;) {
                    uint32_t m = min((uint32_t)__builtin_popcount(sl), room);
                    room -= m;
                    do {
                        const uint32_t p = (uint32_t)__builtin_ctz(sl);
                        sl &= sl - 1;
#pragma unroll
                        for (int e = 0; e < H; e++) {
                            acc[e] = __builtin_amdgcn_alignbit(C[e] >> p, acc[e], 1u);
                            acc[e] = __builtin_amdgcn_alignbit(v[e] >> p, acc[e], 1u);
                        }
                    } while (--m);
                    if (!room) {
                        store(16u);
                        room = 8;
                        b++;
                    }
                }
            }
        }
        if (last) {  // row 2S: an inconsistency after the last split
#pragma unroll
            for (int e = 0; e < H; e++)  // the pairs come down to bit 0, the row above them
                acc[e] = room == 8 ? cin[e] : (acc[e] >> (16 + 2 * room)) | (cin[e] << (16 - 2 * room));
            store(0u);
        }
    }
}

__device__ __forceinline__ void cref_range_hap(const PanelDev &P, const TgtDev &T, uint32_t b0,
                                               uint32_t b1, uint32_t p0, uint32_t p1) {
    if (p1 - p0 > 1) cref_range_h<2>(P, T, b0, b1, p0, p1);
    else cref_range_h<1>(P, T, b0, b1, p0, p1);
}

// In-register transpose of two 16x16 bit blocks side by side: on entry bit c
// of a[r] is (row r, column c) for c < 16 and (row r, column 16 + c') at bit
// 16 + c'; on exit bit r of a[c] is (row r, column c) and bit 16 + r is
// (row r, column 16 + c).  Four rounds of masked block swaps (bits of one
// 16-bit half never move into the other: the masks repeat per half).
__device__ __forceinline__ void transpose16x2(uint32_t (&a)[16]) {
    static_for<0, 4>([&](auto ji) {
        constexpr int j = 8 >> decltype(ji)::value;
        constexpr uint32_t m = j == 8 ? 0x00FF00FFu : j == 4 ? 0x0F0F0F0Fu : j == 2 ? 0x33333333u
                                                                                     : 0x55555555u;
#pragma unroll
        for (int k = 0; k < 16; k++) {
            if (k & j) continue;
            const uint32_t t = ((a[k] >> j) ^ a[k + j]) & m;
            a[k + j] ^= t;
            a[k] ^= t << j;
        }
    });
}

// Block b of a target taking all N haplotypes in panel order (TF_IDENTITY):
// no gather.  Each thread owns GPT groups of 64 haplotypes: it reads their
// word of the 16 staged rows, transposes the low and the high halves as two
// pairs of 16x16 bit blocks, and writes the 64 uint16 values as 128
// contiguous bytes.
template <int GPT>
__device__ __forceinline__ void cref_block_ident(const PanelDev &P, const TgtDev &T, uint32_t b,
                                                 uint64_t *srow) {
    const uint32_t tid = threadIdx.x;
    const uint32_t K = T.K, S = T.S, Kpad = T.Kpad;
    const uint32_t nw = (P.N_ad + 63) / 64;  // == Kpad / 64 (K == N_ad), at most CREF_TW
    const uint32_t sb = min(8 * b + 8, S + 1);
    cref_fill(P, T, b, 0, nw, nw, srow);
    __syncthreads();
    const uint32_t nrows = 2 * (sb - 8 * b) - (sb == S + 1 ? 1u : 0u);
    uint32_t V[GPT][32];  // two uint16 values per register: haplotypes 2i, 2i+1
#pragma unroll
    for (int e = 0; e < GPT; e++) {
        const uint32_t q = tid + CREF_NT * e;
        uint32_t lo[16], hi[16];
#pragma unroll
        for (int rr = 0; rr < 16; rr++) {
            const uint64_t wv = (q < nw && (uint32_t)rr < nrows) ? srow[(uint64_t)rr * nw + q] : 0ull;
            lo[rr] = (uint32_t)wv;
            hi[rr] = (uint32_t)(wv >> 32);
        }
        transpose16x2(lo);
        transpose16x2(hi);
        // lo[c]: haplotype c in the low half, 16 + c in the high half
#pragma unroll
        for (int i = 0; i < 8; i++) {
            V[e][i] = __builtin_amdgcn_perm(lo[2 * i + 1], lo[2 * i], 0x05040100u);
            V[e][8 + i] = __builtin_amdgcn_perm(lo[2 * i + 1], lo[2 * i], 0x07060302u);
            V[e][16 + i] = __builtin_amdgcn_perm(hi[2 * i + 1], hi[2 * i], 0x05040100u);
            V[e][24 + i] = __builtin_amdgcn_perm(hi[2 * i + 1], hi[2 * i], 0x07060302u);
        }
    }
    __syncthreads();  // the staged rows are free for the next block
    const gptr_t<uint16_t> dst = gmem(T.cref) + (uint64_t)b * Kpad;
#pragma unroll
    for (int e = 0; e < GPT; e++) {
        const uint32_t q = tid + CREF_NT * e;
        if (q < nw) {
            if (64 * q + 64 > K) {  // last group: haplotypes >= K are padding
#pragma unroll
                for (int i = 0; i < 32; i++) {
                    const uint32_t k0 = 64 * q + 2 * i;
                    if (k0 >= K) V[e][i] |= 0xFFFFu;
                    if (k0 + 1 >= K) V[e][i] |= 0xFFFF0000u;
                }
            }
            const gptr_t<u32x4> d4 = (gptr_t<u32x4>)(dst + 64 * q);
#pragma unroll
            for (int i = 0; i < 8; i++)
                d4[i] = u32x4{V[e][4 * i], V[e][4 * i + 1], V[e][4 * i + 2], V[e][4 * i + 3]};
        }
    }
}

__global__ __launch_bounds__(CREF_NT) void k_cref(PanelDev P, const TgtDev *__restrict__ tg,
                                                 const CrefItem *__restrict__ items) {
    const CrefItem it = items[blockIdx.x];
    cref_range_hap(P, tg[it.t], it.b0, it.b1, it.p0, it.p1);
}

template <int GPT>
__global__ __launch_bounds__(CREF_NT) void k_cref_ident(PanelDev P, const TgtDev *__restrict__ tg,
                                                       const CrefItem *__restrict__ items) {
    extern __shared__ uint64_t srow[];
    const CrefItem it = items[blockIdx.x];
    for (uint32_t b = it.b0; b < it.b1; b++) cref_block_ident<GPT>(P, tg[it.t], b, srow);
}

// Site rows [m0, m0 + nsites) of the panel as 16-row blocks, one uint16 per
// haplotype (bit j = site m0 + 16b + j), haplotypes N..Kpad-1 all ones.
// grid (nblk, ceil(nw/256)), block 256: a thread transposes one 64-haplotype word.
__global__ __launch_bounds__(256) void k_site_blocks(PanelDev P, uint64_t m0, uint32_t nsites,
                                                    uint16_t *__restrict__ blocks, uint32_t Kpad) {
    const uint32_t b = blockIdx.x, q = blockIdx.y * 256 + threadIdx.x;
    const uint32_t nw = (P.N_ad + 63) / 64;
    if (q >= nw) return;
    uint32_t V[32];  // two uint16 values per register: haplotypes 2i, 2i+1 of the low word etc.
#pragma unroll
    for (int i = 0; i < 32; i++) V[i] = 0;
    for (uint32_t r = 0; r < 16; r++) {
        const uint32_t j = 16 * b + r;
        const uint64_t wv = j < nsites ? P.site[(m0 + j) * P.site_stride + q] : 0ull;
        const uint32_t lo = (uint32_t)wv, hi = (uint32_t)(wv >> 32);
#pragma unroll
        for (int i = 0; i < 16; i++) {
            V[i] |= (((lo >> (2 * i)) & 1u) << r) | (((lo >> (2 * i + 1)) & 1u) << (16 + r));
            V[16 + i] |= (((hi >> (2 * i)) & 1u) << r) | (((hi >> (2 * i + 1)) & 1u) << (16 + r));
        }
    }
    if (64 * q + 64 > P.N_ad) {
#pragma unroll
        for (int i = 0; i < 32; i++) {
            const uint32_t k0 = 64 * q + 2 * i;
            if (k0 >= P.N_ad) V[i] |= 0xFFFFu;
            if (k0 + 1 >= P.N_ad) V[i] |= 0xFFFF0000u;
        }
    }
    uint4 *d4 = (uint4 *)(blocks + (uint64_t)b * Kpad + 64 * q);
#pragma unroll
    for (int i = 0; i < 8; i++) d4[i] = make_uint4(V[4 * i], V[4 * i + 1], V[4 * i + 2], V[4 * i + 3]);
}

// ---------------------------------------------------------------------------
// Device-driven batch (stream contexts): k_plan sizes every target's outputs
// from its split count, lays them out in the context's pools (targets that do
// not fit are deferred), and queues cref blocks and PBWT items (largest
// first) for the persistent kernels below.  One workgroup, n <= 1024.
// ---------------------------------------------------------------------------
constexpr int PLAN_NT = 1024;

__device__ __forceinline__ uint64_t wave_scan_incl64(uint64_t v) {
    const uint32_t l = lane_id();
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint64_t u = __shfl_up(v, o);
        if (l >= (uint32_t)o) v += u;
    }
    return v;
}

// block-wide exclusive scan of 64-bit values (PLAN_NT threads); total returned
__device__ __forceinline__ uint64_t block_excl_scan64(uint64_t v, uint64_t *s_w, uint64_t &total) {
    const uint32_t wave = threadIdx.x >> 6, l = lane_id();
    const uint64_t inc = wave_scan_incl64(v);
    if (l == 63) s_w[wave] = inc;
    __syncthreads();
    uint64_t before = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < PLAN_NT / 64; w++) {
        const uint64_t x = s_w[w];
        tot += x;
        if (w < (int)wave) before += x;
    }
    __syncthreads();
    total = tot;
    return before + inc - v;
}

// block-wide maximum (PLAN_NT threads)
__device__ __forceinline__ uint64_t block_max64(uint64_t v, uint64_t *s_w) {
    const uint32_t wave = threadIdx.x >> 6, l = lane_id();
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint64_t u = __shfl_xor(v, o);
        v = u > v ? u : v;
    }
    if (l == 0) s_w[wave] = v;
    __syncthreads();
    uint64_t m = 0;
#pragma unroll
    for (int w = 0; w < PLAN_NT / 64; w++) m = s_w[w] > m ? s_w[w] : m;
    __syncthreads();
    return m;
}

__global__ __launch_bounds__(PLAN_NT) void k_plan(TgtDev *__restrict__ tg, BatchDev *__restrict__ B,
                                                 PlanArgs A) {
    __shared__ uint64_t s_w[PLAN_NT / 64];
    __shared__ uint64_t keys[2 * PLAN_NT];
    const uint32_t t = threadIdx.x;
    const uint32_t n = B->n;
    const bool valid = t < n;
    uint32_t Mp = 0, Kpad = 0, RS = 0, nblk = 0, S = 0, K = 0;
    uint64_t cb = 0, c0b = 0, ob = 0;
    if (valid) {
        const TgtDev &T = tg[t];
        S = T.stats[0];
        K = T.K;
        Mp = 2 * S + 1;
        Kpad = (K + 63) / 64 * 64;
        RS = row_stride(K, A.layout);
        nblk = (Mp + 15) / 16;
        cb = region_cref_bytes(Mp, Kpad);
        c0b = region_c0_bytes(Mp);
        ob = region_out_bytes(Mp, RS);
    }
    uint64_t tot;
    const uint64_t off = block_excl_scan64(cb + c0b + ob, s_w, tot);
    // prefix sums grow with t, so the targets that fit are a prefix of the batch
    const bool fit = valid && off + cb + c0b + ob <= A.pool_cap;
    if (valid) {
        TgtDev &T = tg[t];
        T.S = S;
        T.stats[2] = fit ? 0u : 1u;  // 1: deferred, outputs not built
        if (fit) {
            T.Mp = Mp;
            T.Kpad = Kpad;
            T.RS = RS;
            T.cref = (uint16_t *)(A.pool + off);
            T.count0 = (int32_t *)(A.pool + off + cb);
            T.out = (uint32_t *)(A.pool + off + cb + c0b);
            T.digest = A.digest ? A.dig_base + 2 * t : nullptr;
            if (A.digest) {
                A.dig_base[2 * t] = 0;
                A.dig_base[2 * t + 1] = 0;
            }
        } else {
            T.Mp = 0;
            T.digest = nullptr;
        }
    }
    // two cref queues: whole-panel targets (transpose kernel) and the others.
    // Block-major order (block b of every target before block b+1) when it
    // costs few empty items: targets with similar windows then read the same
    // panel rows at the same time, from the cache.
    const bool idk = fit && A.ident_ok && (tg[t].flags & TF_IDENTITY);
    const bool gk = fit && !idk;
    // subset targets are queued in items of a group of blocks and a part of the
    // haplotypes, cut alike for the batch
    uint64_t nb128, nb_tot, nb_id, ng, ni, mxg, mxi;
    (void)block_excl_scan64(gk ? (nblk + kCrefGroup - 1) / kCrefGroup : 0u, s_w, nb128);
    const uint32_t Kg = (uint32_t)block_max64(gk ? K : 0u, s_w);
    uint32_t grp, parts;
    cref_cut((uint32_t)nb128, Kg, A.cref_want, grp, parts);
    const uint32_t ngrp = (nblk + grp - 1) / grp;
    const uint64_t bp = block_excl_scan64(gk ? ngrp : 0u, s_w, nb_tot);
    const uint64_t bpi = block_excl_scan64(idk ? nblk : 0u, s_w, nb_id);
    const uint64_t pg = block_excl_scan64(gk ? 1u : 0u, s_w, ng);
    const uint64_t pi = block_excl_scan64(idk ? 1u : 0u, s_w, ni);
    mxg = block_max64(gk ? ngrp : 0u, s_w);
    mxi = block_max64(idk ? nblk : 0u, s_w);
    const bool rrg = ng > 1 && ng * mxg * 4 <= nb_tot * 5;
    const bool rri = ni > 1 && ni * mxi * 4 <= nb_id * 5;
    if (valid) {
        if (rrg) {
            if (gk) A.blockpref[pg] = t;
        } else {
            A.blockpref[t] = (uint32_t)bp;
        }
        if (rri) {
            if (idk) A.blockpref_id[pi] = t;
        } else {
            A.blockpref_id[t] = (uint32_t)bpi;
        }
    }
    uint64_t nfit, nrow;
    (void)block_excl_scan64(fit ? 1u : 0u, s_w, nfit);
    const uint64_t rp = block_excl_scan64(fit ? pbwt_blocks(Mp) : 0u, s_w, nrow);
    if (t < kRowsCounters) A.rowpref[t] = 0;
    if (valid) A.rowpref[kRowsCounters + t] = (uint32_t)rp;
    if (t == 0) A.rowpref[kRowsCounters + n] = (uint32_t)nrow;
    if (t == 0) {
        if (!rrg) A.blockpref[n] = (uint32_t)nb_tot;
        if (!rri) A.blockpref_id[n] = (uint32_t)nb_id;
        B->ncref = (uint32_t)(rrg ? ng * mxg : nb_tot) * parts;
        B->cref_grp = grp;
        B->cref_parts = parts;
        B->cref_per = ((Kg + CREF_NT - 1) / CREF_NT + parts - 1) / parts;
        B->ncref_id = (uint32_t)(rri ? ni * mxi : nb_id);
        B->rr[0] = rrg ? 1u : 0u;
        B->rr[1] = rri ? 1u : 0u;
        B->nrr[0] = (uint32_t)ng;
        B->nrr[1] = (uint32_t)ni;
        B->nfit = (uint32_t)nfit;
        B->cref_ctr = 0;
        B->cref_id_ctr = 0;
    }
    // Chains: cut into segments where that shortens the batch.  Wave w works out
    // the expected time of candidate w (the last one: no cut).
    __shared__ uint32_t s_nb[PLAN_NT], s_kp[PLAN_NT];
    __shared__ uint64_t s_time[kSegCands + 1], s_path[kSegCands + 1], s_work[kSegCands + 1];
    __shared__ uint32_t s_L, s_shape;
    s_nb[t] = fit ? nblk : 0u;
    s_kp[t] = Kpad;
    __syncthreads();
    {
        const uint32_t w = t >> 6;
        if (w <= (uint32_t)kSegCands) {
            const uint32_t L = w < (uint32_t)kSegCands ? 4u << w : 0u;
            uint64_t path = 0, work = 0, words = 0, segs = 0;
            for (uint32_t i = t & 63; i < n; i += 64) {
                const uint32_t nb = s_nb[i], kp = s_kp[i];
                if (!nb) continue;
                uint32_t len;
                const uint32_t Sg = seg_split(nb, L, len);
                const uint64_t p = seg_path(nb, Sg, len, kp);
                path = p > path ? p : path;
                work += seg_work(nb, Sg, kp);
                words += seg_words(Sg, kp);
                segs += Sg > 1 ? 2 * Sg : 0;
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                const uint64_t p = __shfl_xor(path, o);
                path = p > path ? p : path;
            }
            work = wave_sum64(work);
            words = wave_sum64(words);
            segs = wave_sum64(segs);
            if ((t & 63) == 0) {
                s_path[w] = path;
                s_work[w] = work;
            }
            if ((t & 63) == 0)
                s_time[w] = words > A.seg_cap || segs > kMaxSegments ? ~0ull
                                                                    : seg_time(path, work, A.seg_par);
        }
    }
    __syncthreads();
    if (t == 0) {
        // the least expected time, the longer segments of equals; a cut must
        // be worth a quarter (256 windowed targets: cut where a tenth was
        // expected, 32.1 ms of chains, uncut 31.5)
        int best = kSegCands;
        for (int c = kSegCands - 1; c >= 0; c--)
            if (s_time[c] < s_time[best] && s_time[c] != ~0ull &&
                s_time[c] < s_time[kSegCands] - s_time[kSegCands] / 4)
                best = c;
        s_L = best < kSegCands ? 4u << best : 0u;
        s_shape = seg_latency_bound(s_path[best], s_work[best], A.ncu) ? 1u : 0u;
    }
    __syncthreads();
    uint32_t seglen = nblk;
    const uint32_t nseg = fit ? seg_split(nblk, s_L, seglen) : 1u;
    uint64_t seg_tot;
    const uint64_t seg_off = block_excl_scan64(fit ? seg_words(nseg, Kpad) : 0u, s_w, seg_tot);
    if (valid) {
        tg[t].nseg = nseg;
        tg[t].seglen = seglen;
        tg[t].seg = A.seg + seg_off;
    }
    __syncthreads();
    s_nb[t] = nseg;  // now the segments of target t
    s_kp[t] = seglen;
    // PBWT chains 2t (forward) and 2t+1 (backward), most work first:
    // key = (~(Mp * Kpad) & 40 bits) << 24 | item; unused slots sort last
    const uint64_t wk = fit ? ((~((uint64_t)Mp * Kpad)) & 0xFFFFFFFFFFull) << 24 : ~0ull;
    keys[2 * t] = fit ? (wk | (2 * t)) : ~0ull;
    keys[2 * t + 1] = fit ? (wk | (2 * t + 1)) : ~0ull;
    __syncthreads();
    // bitonic sort of 2*PLAN_NT keys, ascending
    for (uint32_t k = 2; k <= 2 * PLAN_NT; k <<= 1) {
        for (uint32_t jj = k >> 1; jj > 0; jj >>= 1) {
            for (uint32_t i = t; i < 2 * PLAN_NT; i += PLAN_NT) {
                const uint32_t ixj = i ^ jj;
                if (ixj > i) {
                    const uint64_t a = keys[i], b = keys[ixj];
                    const bool up = (i & k) == 0;
                    if ((a > b) == up) {
                        keys[i] = b;
                        keys[ixj] = a;
                    }
                }
            }
            __syncthreads();
        }
    }
    // thread t writes the items of the sorted chains 2t and 2t + 1
    uint32_t ch[2], cs[2];
    uint64_t nr = 0, nk = 0, nc = 0;
    for (uint32_t e = 0; e < 2; e++) {
        const uint32_t i = 2 * t + e;
        ch[e] = i < 2 * (uint32_t)nfit ? (uint32_t)(keys[i] & 0xFFFFFFu) : ~0u;
        cs[e] = ch[e] != ~0u ? s_nb[ch[e] >> 1] : 0u;
        nr += cs[e];
        nk += cs[e] > 1 ? 2 * (cs[e] - 1) : 0;
        nc += cs[e] > 1 ? 1 : 0;
    }
    uint64_t nr_tot, nk_tot, nc_tot;
    uint64_t r0 = block_excl_scan64(nr, s_w, nr_tot), k0 = block_excl_scan64(nk, s_w, nk_tot),
             c0 = block_excl_scan64(nc, s_w, nc_tot);
    for (uint32_t e = 0; e < 2; e++) {
        if (ch[e] == ~0u) continue;
        const uint32_t tt = ch[e] >> 1, dir = ch[e] & 1u, len = s_kp[tt];
        const uint32_t nb = (tg[tt].Mp + 15) / 16;
        for (uint32_t s = 0; s < cs[e]; s++) {
            const uint32_t q0 = s * len, q1 = min(nb, q0 + len);
            A.rows_items[r0++] = OrderItem{tt, dir, CHAIN_ROWS, s, q0, q1};
            if (s + 1 < cs[e]) {
                A.rank_items[k0++] = OrderItem{tt, dir, CHAIN_RANK_UP, s, q0, q1};
                A.rank_items[k0++] = OrderItem{tt, dir, CHAIN_RANK_DOWN, s, q0, q1};
            }
        }
        if (cs[e] > 1) A.comb_items[c0++] = OrderItem{tt, dir, CHAIN_COMBINE, 0, 0, cs[e]};
    }
    if (t == 0) {
        for (uint32_t v = 0; v < 2; v++) {
            const bool on = v == (A.shapes > 1 ? s_shape : 0u);
            B->pbwt_ctr[v] = B->rank_ctr[v] = B->comb_ctr[v] = 0;
            B->npbwt[v] = on ? (uint32_t)nr_tot : 0u;
            B->nrank[v] = on ? (uint32_t)nk_tot : 0u;
            B->ncomb[v] = on ? (uint32_t)nc_tot : 0u;
        }
    }
}

// next cref item from a queue of nq, `parts` to an entry: position i (i >= nq ends), target t,
// item b of t (items of `unit` 16-row blocks); b = ~0u for an empty item of a
// block-major queue
__device__ __forceinline__ void cref_pop(uint32_t *ctr, uint32_t nq, uint32_t parts, uint32_t n,
                                         uint32_t rr, uint32_t nrr, const TgtDev *__restrict__ tg,
                                         const uint32_t *__restrict__ pref, uint32_t unit,
                                         uint32_t &i, uint32_t &t, uint32_t &b) {
    __shared__ uint32_t s_i, s_t, s_b;
    if (threadIdx.x == 0) {
        const uint32_t at = atomicAdd(ctr, 1u), ii = at / parts;
        uint32_t tt = 0, bb = 0;
        if (at < nq) {
            if (rr) {  // block-major: block ii / nrr of the (ii % nrr)-th listed target
                tt = pref[ii % nrr];
                bb = ii / nrr;
                if (bb >= ((tg[tt].Mp + 15) / 16 + unit - 1) / unit) bb = ~0u;
            } else {  // last target whose first block is <= ii (it owns block ii)
                uint32_t lo = 0, hi = n;
                while (hi - lo > 1) {
                    const uint32_t mid = (lo + hi) >> 1;
                    if (pref[mid] <= ii) lo = mid; else hi = mid;
                }
                tt = lo;
                bb = ii - pref[lo];
            }
        }
        s_i = at;
        s_t = tt;
        s_b = bb;
    }
    __syncthreads();
    // the same for every lane: scalar registers, so the target's fields load
    // through the scalar cache
    i = __builtin_amdgcn_readfirstlane(s_i);
    t = __builtin_amdgcn_readfirstlane(s_t);
    b = __builtin_amdgcn_readfirstlane(s_b);
    __syncthreads();
}

// cref items of subset targets from their queue: entry i / parts of the queue
// of block groups, part i % parts of the haplotypes
__global__ __launch_bounds__(CREF_NT) void k_cref_persist(PanelDev P, const TgtDev *__restrict__ tg,
                                                         BatchDev *__restrict__ B,
                                                         const uint32_t *__restrict__ blockpref) {
    const uint32_t nq = B->ncref, n = B->n, rr = B->rr[0], nrr = B->nrr[0];
    const uint32_t grp = B->cref_grp, parts = B->cref_parts, per = B->cref_per;
    for (;;) {
        uint32_t i, t, g;
        cref_pop(&B->cref_ctr, nq, parts, n, rr, nrr, tg, blockpref, grp, i, t, g);
        if (i >= nq) break;
        if (g != ~0u) {
            const uint32_t nblk = (tg[t].Mp + 15) / 16, part = i % parts;
            cref_range_hap(P, tg[t], g * grp, min(nblk, (g + 1) * grp), part * per, (part + 1) * per);
        }
    }
}

// cref blocks of whole-panel targets from their queue
template <int GPT>
__global__ __launch_bounds__(CREF_NT, 4) void k_cref_persist_ident(PanelDev P,
                                                               const TgtDev *__restrict__ tg,
                                                               BatchDev *__restrict__ B,
                                                               const uint32_t *__restrict__ blockpref) {
    extern __shared__ uint64_t srow[];
    const uint32_t nq = B->ncref_id, n = B->n, rr = B->rr[1], nrr = B->nrr[1];
    for (;;) {
        uint32_t i, t, b;
        cref_pop(&B->cref_id_ctr, nq, 1u, n, rr, nrr, tg, blockpref, 1u, i, t, b);
        if (i >= nq) break;
        if (b != ~0u) cref_block_ident<GPT>(P, tg[t], b, srow);
    }
}

// count0 digest (grid n, block 256)
__global__ __launch_bounds__(256) void k_digest_count0(const TgtDev *__restrict__ tg,
                                                      const uint32_t *__restrict__ d_n) {
    if (d_n && blockIdx.x >= *d_n) return;
    const TgtDev &T = tg[blockIdx.x];
    if (!T.digest || T.Mp == 0) return;
    uint64_t s = 0;
    for (uint32_t r = threadIdx.x; r < T.Mp; r += 256) s += dig_count0(r, T.count0[r]);
    s = wave_sum64(s);
    if (lane_id() == 0) atomicAdd((unsigned long long *)&T.digest[1], (unsigned long long)s);
}

// Digests recomputed from stored rows (data / cumulative-zero pairs, the
// drop-in and compact layouts) and count0: the same sums as the in-kernel
// digest, for outputs built without it.  grid (DIGR_G, n), block 256: row
// group x of target y; dig receives 2 words per target (zeroed beforehand).
constexpr uint32_t DIGR_G = 64;
__global__ __launch_bounds__(256) void k_digest_rows(const TgtDev *__restrict__ tg,
                                                    const uint32_t *__restrict__ d_n,
                                                    uint64_t *__restrict__ dig) {
    if (blockIdx.y >= *d_n) return;
    const TgtDev &T = tg[blockIdx.y];
    if (T.Mp == 0 || !T.out) return;
    const uint32_t KW = 2 * ((T.K + 31) / 32), RS = T.RS;
    const uint64_t rows = 2ull * T.Mp;
    const uint64_t per = (rows + DIGR_G - 1) / DIGR_G;
    const uint64_t r0 = per * blockIdx.x, r1 = min(rows, r0 + per);
    uint64_t sp = 0, sc = 0;
    for (uint64_t r = r0; r < r1; r++) {
        const uint32_t *row = T.out + r * RS;
        for (uint32_t w = threadIdx.x; w < KW; w += 256) sp += dig_word(r * KW + w, row[w]);
    }
    if (blockIdx.x == 0)
        for (uint32_t r = threadIdx.x; r < T.Mp; r += 256) sc += dig_count0(r, T.count0[r]);
    sp = wave_sum64(sp);
    sc = wave_sum64(sc);
    if (lane_id() == 0) {
        atomicAdd((unsigned long long *)&dig[2 * blockIdx.y], (unsigned long long)sp);
        if (blockIdx.x == 0) atomicAdd((unsigned long long *)&dig[2 * blockIdx.y + 1], (unsigned long long)sc);
    }
}

// cref blocks -> condensed reference rows (for inspection).  grid (Mp, 1), block 256
__global__ __launch_bounds__(256) void k_cref_rows(const TgtDev *__restrict__ tg, uint32_t t,
                                                  uint64_t *__restrict__ rows, uint32_t rw) {
    const TgtDev &T = tg[t];
    const uint32_t r = blockIdx.x;
    const uint16_t *blk = T.cref + (uint64_t)(r >> 4) * T.Kpad;
    for (uint32_t w = threadIdx.x; w < rw; w += 256) {
        uint64_t v = 0;
        for (uint32_t q = 0; q < 64; q++) {
            const uint32_t k = w * 64 + q;
            if (k < T.K) v |= (uint64_t)((blk[k] >> (r & 15)) & 1u) << q;
        }
        rows[(uint64_t)r * rw + w] = v;
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// The dynamic-LDS limit of a kernel is process-wide: contexts of different
// sizes (and engines with different panels) only ever raise it.
hipError_t raise_lds_limit(const void *fn, size_t lds) {
    static std::mutex mu;
    static std::map<const void *, size_t> limit;
    std::lock_guard<std::mutex> lk(mu);
    size_t &cur = limit[fn];
    if (lds <= cur) return hipSuccess;
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e == hipSuccess) cur = lds;
    return e;
}

// Pieces of device arrays into one pinned host buffer (grid x pieces).  Bound by
// the link to the host; 16 bytes a thread keep its writes whole.  One wave per
// workgroup: it finds a place beside other contexts' kernels where four at once
// would not.
constexpr uint32_t GATHER_NT = 64;
__global__ __launch_bounds__(GATHER_NT) void k_gather(GatherArgs A, char *__restrict__ dst) {
    const uint32_t i = blockIdx.y, bytes = A.bytes[i], n16 = bytes / 16;
    const gptr_t<const uint32_t> src = (gptr_t<const uint32_t>)(const uint32_t *)A.src[i];
    const gptr_t<uint32_t> out = (gptr_t<uint32_t>)(uint32_t *)(dst + A.off[i]);
    for (uint32_t q = blockIdx.x * GATHER_NT + threadIdx.x; q < n16; q += gridDim.x * GATHER_NT) {
        // the arrays are aligned to their elements only
        const u32x4 v = u32x4{src[4 * q], src[4 * q + 1], src[4 * q + 2], src[4 * q + 3]};
        *(gptr_t<u32x4>)(out + 4 * q) = v;
    }
    const uint32_t tail = 4 * n16 + threadIdx.x;
    if (blockIdx.x == 0 && tail < bytes / 4) out[tail] = src[tail];
}
hipError_t launch_gather(const GatherArgs &a, void *dst, hipStream_t s) {
    uint32_t most = 0;
    for (uint32_t i = 0; i < a.n; i++) most = std::max(most, a.bytes[i]);
    const uint32_t wgs = std::min((most + 1023) / 1024, 512u);
    hipLaunchKernelGGL(k_gather, dim3(std::max(wgs, 1u), a.n), dim3(GATHER_NT), 0, s, a, static_cast<char *>(dst));
    return hipGetLastError();
}
hipError_t launch_site_to_hap(const PanelDev &P, uint64_t *hap, hipStream_t s) {
    dim3 grid((unsigned)((P.hap_stride + 3) / 4), (P.N_ad + 63) / 64);
    hipLaunchKernelGGL(k_site_to_hap, grid, dim3(256), 0, s, P, hap);
    return hipGetLastError();
}
hipError_t launch_panel_mono(const PanelDev &P, uint64_t *pand, uint64_t *por, hipStream_t s) {
    hipLaunchKernelGGL(k_panel_mono, dim3((P.M + 3) / 4), dim3(256), 0, s, P, pand, por);
    return hipGetLastError();
}
static dim3 distance_grid(const PanelDev &P, uint32_t n) {
    const uint32_t nhb = (P.N_ad + DIST_W - 1) / DIST_W;
    return dim3(8 * ((n + DIST_G - 1) / DIST_G), std::min((nhb + 7) / 8, 65535u));
}
hipError_t launch_distance(const PanelDev &P, const TgtDev *tg, const uint32_t *tlist,
                           uint32_t nsel, hipStream_t s) {
    if (!nsel) return hipSuccess;
    hipLaunchKernelGGL(k_distance, distance_grid(P, nsel), dim3(256), 0, s, P, tg, tlist, nsel, (const uint32_t *)nullptr);
    return hipGetLastError();
}
hipError_t launch_select(const PanelDev &P, const TgtDev *tg, uint32_t n, hipStream_t s) {
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_select, dim3(n), dim3(SEL_NT), 0, s, P, tg, (const uint32_t *)nullptr);
    return hipGetLastError();
}
hipError_t launch_monos(const PanelDev &P, const TgtDev *tg, const uint32_t *tlist, uint32_t n,
                        uint32_t max_ww, uint32_t ncu, hipStream_t s) {
    if (!n) return hipSuccess;
    const uint32_t gx = (max_ww + 63) / 64;
    hipLaunchKernelGGL(k_monos, dim3(gx, n, mono_parts((uint64_t)gx * n, ncu)), dim3(MONO_NT), 0, s, P, tg, tlist,
                       (const uint32_t *)nullptr);
    return hipGetLastError();
}
hipError_t launch_splits(const PanelDev &P, const TgtDev *tg, uint32_t n, hipStream_t s) {
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_splits, dim3(n), dim3(64), 0, s, P, tg, (const uint32_t *)nullptr);
    return hipGetLastError();
}
hipError_t launch_bits_to_list(const TgtDev *tg, uint32_t n, uint32_t nbits_bh, int which,
                               hipStream_t s) {
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_bits_to_list, dim3(n), dim3(SEL_NT), 0, s, tg, nbits_bh, which);
    return hipGetLastError();
}

// dynamic LDS of the cref kernels: the 16 staged rows of one tile
size_t cref_lds_bytes(const PanelDev &P, uint32_t maxK) {
    (void)maxK;
    return (size_t)16 * cref_tile_words((P.N_ad + 63) / 64) * sizeof(uint64_t);
}

hipError_t launch_cref(const PanelDev &P, const TgtDev *tg, const CrefItem *items, uint32_t nitems,
                       uint32_t maxK, bool ident, hipStream_t s) {
    if (!nitems) return hipSuccess;
    const uint32_t nw = (P.N_ad + 63) / 64;
    const size_t lds = cref_lds_bytes(P, maxK);
    if (ident) {
        const uint32_t gpt = (nw + CREF_NT - 1) / CREF_NT;
        if (gpt <= 2) {
            const void *fn = gpt <= 1 ? (const void *)k_cref_ident<1> : (const void *)k_cref_ident<2>;
            hipError_t e = raise_lds_limit(fn, lds);
            if (e != hipSuccess) return e;
            if (gpt <= 1)
                hipLaunchKernelGGL(k_cref_ident<1>, dim3(nitems), dim3(CREF_NT), lds, s, P, tg, items);
            else
                hipLaunchKernelGGL(k_cref_ident<2>, dim3(nitems), dim3(CREF_NT), lds, s, P, tg, items);
            return hipGetLastError();
        }
    }
    if (!P.hap || !P.hap_stride) return hipErrorInvalidValue;  // the haplotype-major panel is needed
    hipLaunchKernelGGL(k_cref, dim3(nitems), dim3(CREF_NT), 0, s, P, tg, items);
    return hipGetLastError();
}

// haplotype positions are 16-bit in the PBWT payload
uint32_t cref_max_k() { return 65536 - 64; }

hipError_t launch_digest_count0(const TgtDev *tg, uint32_t n, hipStream_t s) {
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_digest_count0, dim3(n), dim3(256), 0, s, tg, (const uint32_t *)nullptr);
    return hipGetLastError();
}
hipError_t launch_digest_rows(const TgtDev *tg, const uint32_t *d_n, uint32_t nmax, uint64_t *dig,
                              hipStream_t s) {
    if (!nmax) return hipSuccess;
    hipLaunchKernelGGL(k_digest_rows, dim3(DIGR_G, nmax), dim3(256), 0, s, tg, d_n, dig);
    return hipGetLastError();
}
hipError_t launch_cref_rows(const TgtDev *tg, uint32_t t, uint32_t Mp, uint64_t *rows, uint32_t rw,
                            hipStream_t s) {
    hipLaunchKernelGGL(k_cref_rows, dim3(Mp), dim3(256), 0, s, tg, t, rows, rw);
    return hipGetLastError();
}

hipError_t launch_site_blocks(const PanelDev &P, uint64_t m0, uint32_t nsites, uint16_t *blocks,
                              hipStream_t s) {
    const uint32_t nw = (P.N_ad + 63) / 64;
    hipLaunchKernelGGL(k_site_blocks, dim3((nsites + 15) / 16, (nw + 255) / 256), dim3(256), 0, s, P,
                       m0, nsites, blocks, (P.N_ad + 63) / 64 * 64);
    return hipGetLastError();
}

// ---- device-driven batch (stream contexts)

// Prep phase over a batch of *d_n <= nmax targets, one kernel class per call
// (0 distances, 1 top-K, 2 monos, 3 split sites); grids cover nmax targets.
hipError_t launch_prep_dev(int cls, const PanelDev &P, const TgtDev *tg, const uint32_t *d_n,
                           uint32_t nmax, uint32_t max_ww, uint32_t ncu, hipStream_t s) {
    switch (cls) {
    case 0:
        hipLaunchKernelGGL(k_distance, distance_grid(P, nmax), dim3(256), 0, s, P, tg, (const uint32_t *)nullptr, 0u, d_n);
        break;
    case 1:
        hipLaunchKernelGGL(k_select, dim3(nmax), dim3(SEL_NT), 0, s, P, tg, d_n);
        break;
    case 2:
        hipLaunchKernelGGL(k_monos,
                           dim3((max_ww + 63) / 64, nmax, mono_parts((uint64_t)((max_ww + 63) / 64) * nmax, ncu)),
                           dim3(MONO_NT), 0, s, P, tg,
                           (const uint32_t *)nullptr, d_n);
        break;
    default:
        hipLaunchKernelGGL(k_splits, dim3(nmax), dim3(64), 0, s, P, tg, d_n);
        break;
    }
    return hipGetLastError();
}
hipError_t launch_plan(TgtDev *tg, BatchDev *B, const PlanArgs &A, hipStream_t s) {
    hipLaunchKernelGGL(k_plan, dim3(1), dim3(PLAN_NT), 0, s, tg, B, A);
    return hipGetLastError();
}
hipError_t launch_digest_count0_dev(const TgtDev *tg, const uint32_t *d_n, uint32_t nmax,
                                    hipStream_t s) {
    hipLaunchKernelGGL(k_digest_count0, dim3(nmax), dim3(256), 0, s, tg, d_n);
    return hipGetLastError();
}

using CrefPersistFn = void (*)(PanelDev, const TgtDev *, BatchDev *, const uint32_t *);
static CrefPersistFn cref_persist_fn(const PanelDev &P, bool ident) {
    if (!ident) return k_cref_persist;
    const uint32_t gpt = ((P.N_ad + 63) / 64 + CREF_NT - 1) / CREF_NT;
    return gpt <= 1 ? k_cref_persist_ident<1> : k_cref_persist_ident<2>;
}

// identity targets take the transpose path when every 64-haplotype group
// fits two per thread
bool cref_ident_ok(const PanelDev &P) { return (P.N_ad + 63) / 64 <= 2u * CREF_NT; }

// sets the dynamic LDS limit; occ[0], occ[1] = resident workgroups per CU of
// the subset and identity kernels
hipError_t cref_persist_prepare(const PanelDev &P, uint32_t maxK, int *occ) {
    for (int k = 0; k < 2; k++) {
        occ[k] = 0;
        if (k == 1 && !cref_ident_ok(P)) continue;
        // the subset kernel stages nothing in LDS
        const size_t lds = k == 1 ? cref_lds_bytes(P, maxK) : 0;
        const void *fn = (const void *)cref_persist_fn(P, k == 1);
        hipError_t e = raise_lds_limit(fn, lds);
        if (e != hipSuccess) return e;
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ[k], fn, CREF_NT, lds);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
// grid[0], grid[1]: workgroups of the subset and identity kernels (0: none)
hipError_t launch_cref_persist(const PanelDev &P, const TgtDev *tg, BatchDev *B,
                               const uint32_t *blockpref, const uint32_t *blockpref_id,
                               uint32_t maxK, const uint32_t *grid, hipStream_t s) {
    const size_t lds = cref_lds_bytes(P, maxK);
    if (grid[0] && (!P.hap || !P.hap_stride)) return hipErrorInvalidValue;
    if (grid[0])
        hipLaunchKernelGGL(cref_persist_fn(P, false), dim3(grid[0]), dim3(CREF_NT), 0, s, P, tg,
                           B, blockpref);
    if (grid[1] && cref_ident_ok(P))
        hipLaunchKernelGGL(cref_persist_fn(P, true), dim3(grid[1]), dim3(CREF_NT), lds, s, P, tg, B,
                           blockpref_id);
    return hipGetLastError();
}
}  // namespace eimp
