// eimp_pbwt.hip -- compressed forward / backward PBWT on gfx950
// (PBWT::buildComprPBWT, src/PBWT.cpp:207-285).
//
// A row's step is a stable partition of the order by the row's bit, zeros
// first; 16 rows in a row are one stable sort of the order by the 16-bit key
// of each haplotype's bits (first row lowest).  The work is cut there:
//
//   k_order  the chain.  One workgroup per (target, direction) carries the
//            order from one 16-row block of the condensed reference to the
//            next: it looks up every position's key, finds the runs of equal
//            keys (neighbours in the order share long matches, so a block has
//            far fewer runs than haplotypes), sorts the runs by key and moves
//            each run's haplotypes to its new place.  Per block it leaves the
//            run list (key, first position) in the block's own rows.
//   k_rows   the rows.  One wave per block, all blocks of all targets
//            independent: 16 one-bit partitions of the run list give the
//            block's 16 rows.
//
// Carrying every haplotype through every row (two barriers and 5 vector
// instructions per 64 haplotypes and row, one workgroup per chain for all
// rows) took 32.3 ms for 192 targets of 15,000 rows at K = 10,000; the chain
// now takes 9.1 ms and the rows 5.6 ms.  One target of 45,000 rows:
// 61.3 and 2.8 ms for the whole call (its chain cut into segments).
//
// Blocks with more runs than k_rows takes and the last block of a target when
// it has fewer than 16 rows are done row by row in k_order (order_dense).
// Where the order after every row is asked for (panel PBWT), k_order only
// leaves the order at the start of every block and k_dense does the blocks row
// by row, all of them independent.
#include <algorithm>

#include "eimp_launch.h"
#include "eimp_order.h"

namespace eimp {

namespace {

// ---------------------------------------------------------------------------
// k_rows: the 16 rows of a block from its run list, one wave per block.
//
// An entry is key << 16 | length.  Behind the R runs stand empty runs of ones
// up to 64 E entries, E odd (no two lanes on one LDS bank) and fixed for the
// block; under the stable partition they stay there.  Per row, lane x takes
// entries [x E, x E + E):
//   one packed sum {length, ones} per lane and its prefix sum over the wave give
//       the position and the ones before a lane's first entry; inside the lane
//       both run along
//   where the row's bit differs from the previous entry's, position P is marked
//       in the row's bit map: -2^P where ones begin, +2^P where they end (LDS
//       add on the word)
//   the entry is written to its new place: zeros from entry 0, ones behind all
//       zeros (every entry is in a register before)
// then the row's words come from the marks: a word's sum, one less where a run
// goes on into it (run_states), a scan of the words' zeros for the offsets.
// Bound by vector instructions: 13 per 64 entries and row and about 40 per 64
// word pairs and row; one wave per block because two barriers a row cost a
// workgroup more than the wave's own latency.  Entries with their first position
// instead of the length, neighbours with equal remaining bits merged row by row,
// took 28: the merging (2,400 entries of a block become 1,700 by its twelfth
// row) cost more than it saved.  96 targets on the 200,000-haplotype panel
// (2,750 runs a block): 8,106 us so, 5,021 us now; 192 whole-panel targets at
// K = 10,000 (1,050 runs): 6,757 and 5,630 us; 256 windows: 12.3 and 9.8 ms.
// ---------------------------------------------------------------------------
// Lanes entered inside a run of ones, from what every lane does with that
// state: f0 / f1 = lanes left inside a run when entered outside / inside one.
// Where entering does not matter or only passes through, that is a carry chain
// (generate f0 & f1, propagate f1 & ~f0), one 64-bit addition; a lane that
// inverts the state (f0 & ~f1: its only mark is on its last bit) is settled
// before the lanes above it.  in: state before lane 0, replaced by the state
// after lane 63.
__device__ __forceinline__ uint64_t run_states(uint64_t f0, uint64_t f1, uint32_t &in) {
    uint64_t g = f0 & f1, p = f0 | f1, x = f0 & ~f1;  // p: generate or propagate
    p &= ~x;
    for (;;) {
        const uint64_t lo = g + p, sum = lo + in;
        const uint64_t entered = sum ^ g ^ p;
        if (x == 0) {
            // carry out of lane 63
            in = (uint32_t)((lo < g) || (sum < lo));
            return entered;
        }
        const uint64_t b = x & (0 - x);
        x ^= b;
        if (!(entered & b)) {
            g |= b;
            p |= b;
        }
    }
}

// LDS of k_rows: entries from byte kRowsBias on (what a store address may lie
// below its immediate offset), then the marks.
constexpr uint32_t kRowsBias = 128;

// Row of key bit `bit` (an entry's bit 16 + bit, bit < 8) on E entries per lane,
// partitioned in place.
template <int E>
__device__ __forceinline__ void rows_step(const uint32_t bit, const bool halve, const lds_ptr_t<uint32_t> tog) {
    const uint32_t ln = opaque(lane_id());
    const lds_ptr_t<uint32_t> mine = lds_at(kRowsBias) + ln * E;
    uint32_t p[E];
#pragma unroll
    for (int e = 0; e < E; e++) p[e] = mine[e];
    if (halve) {  // rows 8..15: their bits come down
#pragma unroll
        for (int e = 0; e < E; e++) p[e] = __builtin_amdgcn_perm(p[e], p[e], 0x0C030100u);
    }
    // {length, ones} of my entries: no more than 61 ones above a length of at
    // most 32,768
    uint32_t bm = opaque_s(0x10000u << bit), acc = 0;
    const uint32_t am = bm | 0xFFFFu;
    static_for<0, E>([&](auto ei) { acc += p[decltype(ei)::value] & am; });
    const uint32_t sum = (acc & 0xFFFFu) | (acc >> (16 + bit) << 16);
    const uint32_t ex = lane_scan_excl<64>(sum);
    const uint32_t nz = 64u * E - ((uint32_t)__builtin_amdgcn_readlane((int)(ex + sum), 63) >> 16);
    uint64_t before = __ballot((p[E - 1] & bm) != 0u) << 1;  // the entry before each lane's first
    wave_order();
    // y ones before the entry: a one goes to entry nz + y, a zero to (E ln + e) -
    // y; in bytes less 2 e, the store's immediate offset, that is x and V - x,
    // and x grows by 2 behind a one and falls by 2 behind a zero
    uint32_t x = 4u * ((ex >> 16) + nz) + kRowsBias, P = ex & 0xFFFFu;
    const uint32_t V = 4u * (E * ln + nz) + 2u * kRowsBias;
    static_for<0, E>([&](auto ei) {
        constexpr int e = decltype(ei)::value;
        const uint64_t one = __ballot((p[e] & bm) != 0u);
        const uint64_t changed = one ^ before;
        before = one;
        const bool o = __builtin_amdgcn_inverse_ballot_w64(one);
        const uint32_t to = o ? x : V - x;
        *(lds_ptr_t<uint32_t>)(size_t)(to + 2u * e) = p[e];
        x += o ? 2u : ~1u;
        if (__builtin_amdgcn_inverse_ballot_w64(changed))
            __hip_atomic_fetch_add(&tog[P >> 5], (o ? ~0u : 1u) << (P & 31), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WAVEFRONT);
        P += p[e] & 0xFFFFu;
        if constexpr (e % 4 == 3) asm volatile("" : "+v"(x), "+v"(P), "+s"(bm));
    });
    wave_order();
}

// Entries per lane instantiated, all odd: 1, 3, .. 17, then 21, 25, .. 61
__host__ __device__ constexpr int row_entries_at(int i) { return i <= 8 ? 2 * i + 1 : 17 + 4 * (i - 8); }
// the index of the fewest that hold n entries
__device__ __forceinline__ uint32_t row_entries_index(uint32_t n) {
    const uint32_t need = (n + 63) / 64;
    return need <= 17 ? need / 2 : 8 + (need - 17 + 3) / 4;
}
// f(integral_constant i) for run-time i in [B, E): a tree of uniform branches
template <int B, int E, class F>
__device__ __forceinline__ void dispatch(uint32_t i, F &&f) {
    if constexpr (E - B == 1) {
        f(std::integral_constant<int, B>{});
    } else {
        constexpr int M = (B + E) / 2;
        if (i < (uint32_t)M) dispatch<B, M>(i, f);
        else dispatch<M, E>(i, f);
    }
}

template <int E>
__device__ __forceinline__ void rows_block(const TgtDev &T, const bool rev, const uint32_t q,
                                           const uint32_t R, const lds_ptr_t<uint32_t> tog, uint64_t &dsum) {
    const uint32_t ln = lane_id();
    const uint32_t K = T.K, Mp = T.Mp, Kpad = T.Kpad, RS = T.RS;
    const uint32_t nblk = (Mp + 15) / 16, nch = Kpad / 64, npairs = (K + 31) / 32, KW = 2 * npairs;
    const BlockGeo geo = block_geo(q, Mp, nblk, rev);
    const bool raw = (T.flags & TF_RAW) != 0;
    const bool dig = T.digest != nullptr;
    const gptr_t<uint32_t> outrow = gmem(T.out) + ((rev ? (uint64_t)Mp : 0ull) + geo.s0) * RS;
    // run list (key, first position) to entries (key, length); behind them
    // empty runs of ones, which stay there
    const lds_ptr_t<uint32_t> ent = lds_at(kRowsBias);
    constexpr int B = 8;  // slots whose loads are in flight together
    static_for<0, (E + B - 1) / B>([&](auto bi) {
        constexpr int e0 = decltype(bi)::value * B, e1 = e0 + B < E ? e0 + B : E;
        uint32_t here[B], next[B];
#pragma unroll
        for (int e = e0; e < e1; e++) {
            const uint32_t i = 64 * e + ln;
            here[e - e0] = outrow[min(i, R - 1)];
            next[e - e0] = outrow[min(i + 1, R - 1)];
        }
#pragma unroll
        for (int e = e0; e < e1; e++) {
            const uint32_t i = 64 * e + ln, h = here[e - e0], len = (i + 1 < R ? next[e - e0] : Kpad) - h;
            ent[i] = i < R ? (h & 0xFFFF0000u) | (len & 0xFFFFu) : 0xFFFF0000u;
        }
    });
    const uint32_t pw0 = raw ? 2 * nch : 2 * npairs, tw = (RS - pw0) / 2;  // padding pairs of a row
    const uint32_t fw = raw ? ~0u : 0u;
    uint32_t g0 = (rev ? Mp * KW : 0u) + geo.s0 * KW;
    uint32_t c0acc = 0;
    wave_order();
#pragma unroll 1
    for (uint32_t j = 0; j < 16; j++) {
        rows_step<E>(j & 7u, j == 8, tog);
        // the row's words: 64 positions per lane
        const gptr_t<uint32_t> row = outrow + (uint64_t)j * RS;
        uint32_t zrun = 0, state = 0;
        for (uint32_t c0 = 0; c0 < nch; c0 += 64) {
            const uint32_t ch = c0 + ln;
            const bool in = ch < nch;
            u32x2 t = u32x2{0u, 0u};
            if (in) {
                const lds_ptr_t<u32x2> w = (lds_ptr_t<u32x2>)(tog + 2 * ch);
                t = *w;
                *w = u32x2{0u, 0u};
            }
            // a word with marks +2^e at the ends and -2^s at the starts of
            // its one-runs is their sum, less one if a run goes on into it;
            // its top bit then says whether one goes on into the next
            const uint64_t f0 = __ballot((int32_t)(t[1] + ((int32_t)t[0] >> 31)) < 0);
            const uint64_t f1 = __ballot((int32_t)(t[1] + ((int32_t)(t[0] - 1) >> 31)) < 0);
            const uint64_t entered = run_states(f0, f1, state);
            const uint32_t lo = t[0] - (__builtin_amdgcn_inverse_ballot_w64(entered) ? 1u : 0u);
            const uint32_t hi = t[1] + (uint32_t)((int32_t)lo >> 31);
            const uint32_t z0 = 32u - (uint32_t)__popc(lo);
            const uint32_t zl = in ? z0 + 32u - (uint32_t)__popc(hi) : 0u;
            const uint32_t zex = lane_scan_excl<64>(zl);
            const uint32_t o1 = zrun + zex + z0, o3 = zrun + zex + zl;
            zrun += (uint32_t)__builtin_amdgcn_readlane((int)(zex + zl), 63);
            if (in) {
                const bool second = 2 * ch + 1 < npairs;
                if (raw) {
                    *(gptr_t<u32x2>)(row + 2 * ch) = u32x2{lo, hi};
                } else {
                    *(gptr_t<u32x2>)(row + 4 * ch) = u32x2{lo, o1};
                    if (second) *(gptr_t<u32x2>)(row + 4 * ch + 2) = u32x2{hi, o3};
                }
                if (dig) {
                    const uint32_t g = g0 + 4u * ch;
                    const uint32_t dkey = g * kDigKey, dneg = 0u - g;
                    dsum += __builtin_amdgcn_alignbit(lo ^ dkey, lo ^ dkey, dneg);
                    const uint32_t x1 = o1 ^ (dkey + kDigKey);
                    dsum += __builtin_amdgcn_alignbit(x1, x1, dneg - 1u);
                    if (second) {
                        const uint32_t x2 = hi ^ (dkey + 2u * kDigKey), x3 = o3 ^ (dkey + 3u * kDigKey);
                        dsum += __builtin_amdgcn_alignbit(x2, x2, dneg - 2u);
                        dsum += __builtin_amdgcn_alignbit(x3, x3, dneg - 3u);
                    }
                }
            }
        }
        c0acc = eimp_llvm_writelane(zrun, j, c0acc);
        if (ln < tw) *(gptr_t<u32x2>)(row + pw0 + 2 * ln) = u32x2{fw, fw};
        g0 += KW;
        if (ln == 0) tog[Kpad / 32] = 0;  // the end of ones before the empty runs
        wave_order();
    }
    if (!rev && ln < 16) gmem(T.count0)[geo.s0 + ln] = (int32_t)c0acc;
    wave_order();
}

// k_rows kernels by entries per lane: LDS and registers go with the most
// entries of a wave, and one kernel for all blocks would have two waves per
// SIMD.  Kernel k does the blocks of R + 1 <= 64 kRowsEntries[k] entries that
// the kernel before it does not.
constexpr int kRowsKernels = 4;
constexpr int kRowsEntries[kRowsKernels] = {17, 33, 49, 61};

// Sorts the blocks into one list per k_rows kernel (their order within a list
// does not matter).  pref: per target (of *d_n, or n) its first block, both
// directions, pref[n] their number; cnt: kRowsKernels list lengths, zero
// beforehand.  The lists of kernels 0 and 1 share `total` entries from both
// ends, those of kernels 2 and 3 the `total` after them.
__device__ __forceinline__ uint64_t list_at(int kernel, uint32_t total, uint32_t i) {
    return (kernel >= 2 ? (uint64_t)total : 0ull) + (kernel & 1 ? total - 1 - i : i);
}
constexpr uint32_t LIST_NT = 1024;
__global__ __launch_bounds__(LIST_NT) void k_rows_list(const TgtDev *__restrict__ tg,
                                                   const uint32_t *__restrict__ d_n, uint32_t n,
                                                   const uint32_t *__restrict__ pref,
                                                   RowItem *__restrict__ list,
                                                   uint32_t *__restrict__ cnt) {
    // one atomic per list and LIST_NT blocks: on one address they queue up
    __shared__ uint32_t s_cnt[kRowsKernels][LIST_NT / 64], s_base[kRowsKernels];
    const uint32_t wave = threadIdx.x >> 6;
    if (d_n) n = *d_n;
    const uint32_t total = pref[n];
    for (uint32_t i0 = blockIdx.x * LIST_NT; i0 < total; i0 += gridDim.x * LIST_NT) {
        const uint32_t i = i0 + threadIdx.x;
        const bool in = i < total;
        uint32_t t = 0, hi = n;  // last target whose first block is <= i
        while (hi - t > 1) {
            const uint32_t mid = (t + hi) >> 1;
            if (pref[mid] <= i) t = mid; else hi = mid;
        }
        const uint32_t nblk = (tg[t].Mp + 15) / 16, b = i - pref[t];
        const uint32_t R = in ? (uint32_t)tg[t].hdr[b] : kDense;
        const bool rev = b >= nblk;
        const RowItem item{2 * t + (rev ? 1u : 0u), rev ? b - nblk : b, R};
        int mine = -1;  // the first kernel that takes R + 1 entries
        if (R != kDense) {
#pragma unroll
            for (int k = kRowsKernels - 1; k >= 0; k--)
                if (R + 1 <= 64u * kRowsEntries[k]) mine = k;
        }
        uint32_t rank = 0;
#pragma unroll
        for (int k = 0; k < kRowsKernels; k++) {
            const uint64_t m = __ballot(mine == k);
            if (mine == k) rank = mbcnt(m);
            if (lane_id() == 0) s_cnt[k][wave] = (uint32_t)__popcll(m);
        }
        __syncthreads();
        if (threadIdx.x < kRowsKernels) {
            uint32_t sum = 0;
            for (uint32_t w = 0; w < LIST_NT / 64; w++) {
                const uint32_t c = s_cnt[threadIdx.x][w];
                s_cnt[threadIdx.x][w] = sum;
                sum += c;
            }
            s_base[threadIdx.x] = sum ? atomicAdd(&cnt[threadIdx.x], sum) : 0u;
        }
        __syncthreads();
        if (mine >= 0) {
            const uint32_t at = s_base[mine] + s_cnt[mine][wave] + rank;
            list[list_at(mine, total, at)] = item;
        }
        __syncthreads();
    }
}

template <int KERNEL>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(KERNEL == 0 ? 6 : (KERNEL == 1 ? 4 : (KERNEL == 2 ? 3 : 2))))) void k_rows(
    const TgtDev *__restrict__ tg, const uint32_t *__restrict__ d_n, uint32_t n,
    const uint32_t *__restrict__ pref, const RowItem *__restrict__ list,
    const uint32_t *__restrict__ cnt, uint32_t ntog) {
    constexpr int EMAX = kRowsEntries[KERNEL];
    // the indexes of the sizes of this kernel
    constexpr int top = EMAX <= 17 ? EMAX / 2 : 8 + (EMAX - 17) / 4;
    constexpr int low = KERNEL == 0 ? 0 : 8 + (kRowsEntries[KERNEL ? KERNEL - 1 : 0] - 17) / 4 + 1;
    const lds_ptr_t<uint32_t> tog = lds_at(kRowsBias) + 64 * EMAX;
    const uint32_t items = cnt[KERNEL];
    if (blockIdx.x >= items) return;
    const uint32_t total = pref[d_n ? *d_n : n];
    for (uint32_t i = lane_id(); i < ntog; i += 64) tog[i] = 0;
    wave_order();
    for (uint32_t i = blockIdx.x; i < items; i += gridDim.x) {
        const RowItem it = list[list_at(KERNEL, total, i)];
        const TgtDev &T = tg[it.chain >> 1];
        uint64_t dsum = 0;
        dispatch<low, top + 1>(row_entries_index(it.runs + 1), [&](auto ii) {
            rows_block<row_entries_at(decltype(ii)::value)>(T, (it.chain & 1u) != 0, it.q, it.runs, tog, dsum);
        });
        if (T.digest) {
            dsum = wave_sum64(dsum);
            if (lane_id() == 0)
                atomicAdd((unsigned long long *)&T.digest[0], (unsigned long long)dsum);
        }
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// Compressed PBWT for K beyond the LDS-resident kernels (src/PBWT.cpp:207-285,
// the same rows): the order lives in global memory (two arrays of Kpad
// haplotype indexes, swapped every step; L2-resident at these sizes) and only
// the current row's K bits are staged in LDS.  One workgroup of BIG_NT
// threads per item; wave w takes chunks w, w + NW, ... of 64 positions.  A
// step: stage row r; pass 1 counts the zeros of every chunk (ballots) into
// LDS; a block scan turns them into zeros-before-chunk; pass 2 recomputes
// each chunk's ballot, scatters every index to its place under the stable
// partition (zeros first) and writes the chunk's (data, cumulative zeros)
// pairs.  Positions K..Kpad-1 hold index K and read as ones (1-padding).
// ---------------------------------------------------------------------------
constexpr int BIG_NT = 1024;
constexpr uint32_t kBigMaxK = 1u << 19;  // LDS: K/8 bytes of row + K/16 of chunk counts


__device__ __forceinline__ uint32_t big_bit(const uint32_t *rowb, uint32_t idx, uint32_t K) {
    return idx < K ? (rowb[idx >> 5] >> (idx & 31)) & 1u : 1u;
}

__global__ __launch_bounds__(BIG_NT) void k_pbwt_big(const BigItem *__restrict__ items) {
    extern __shared__ uint32_t smem[];
    constexpr uint32_t NW = BIG_NT / 64;
    const BigItem I = items[blockIdx.x];
    const uint32_t K = I.K, Mp = I.Mp, RS = I.RS;
    const uint32_t Kpad = (K + 63) / 64 * 64, nch = Kpad / 64;
    const uint32_t nw32 = (K + 31) / 32, npairs = nw32, KW = 2 * npairs;
    uint32_t *rowb = smem;               // nw32 words: the current row
    uint32_t *cz = smem + (nw32 + 1) / 2 * 2;  // nch: zeros per chunk, then zeros before it
    __shared__ uint32_t s_part[NW + 1];
    const uint32_t tid = threadIdx.x, wave = tid >> 6, ln = lane_id();
    gptr_t<uint32_t> ordA = gmem(I.ord0), ordB = gmem(I.ord1);
    for (uint32_t q = tid; q < Kpad; q += BIG_NT) {
        ordA[q] = q < K ? q : K;
        if (I.absperm && q < K) gmem(I.absperm)[q] = (int32_t)q;
    }
    {
        // the padding words of every row, stored once
        const uint32_t pw0 = I.raw ? 2 * nch : 2 * npairs;
        const uint32_t fw = I.raw ? ~0u : 0u;
        for (uint32_t rr = tid; rr < Mp; rr += BIG_NT) {
            gptr_t<uint32_t> prow = gmem(I.out) + (uint64_t)rr * RS;
            for (uint32_t w = pw0; w < RS; w++) prow[w] = fw;
        }
    }
    uint64_t dsum = 0;
    __syncthreads();
    for (uint32_t step = 0; step < Mp; step++) {
        const uint32_t r = I.rev ? Mp - 1 - step : step;
        const gptr_t<const uint32_t> src = (gptr_t<const uint32_t>)(I.rows + (uint64_t)r * I.rstride);
        for (uint32_t q = tid; q < nw32; q += BIG_NT) rowb[q] = src[q];
        __syncthreads();
        // pass 1: zeros of every chunk
        for (uint32_t ch = wave; ch < nch; ch += NW) {
            const uint32_t idx = ordA[ch * 64 + ln];
            const uint64_t m = __ballot(big_bit(rowb, idx, K));
            if (ln == 0) cz[ch] = 64u - (uint32_t)__popcll(m);
        }
        __syncthreads();
        // exclusive scan of cz over the chunks: thread tid owns a contiguous run
        const uint32_t per = (nch + BIG_NT - 1) / BIG_NT;
        const uint32_t c0 = min(nch, tid * per), c1 = min(nch, c0 + per);
        uint32_t mine = 0;
        for (uint32_t c = c0; c < c1; c++) mine += cz[c];
        const uint32_t incl = wave_scan_incl(mine);
        if (ln == 63) s_part[wave] = incl;
        __syncthreads();
        uint32_t before = 0, total = 0;
        for (uint32_t w = 0; w < NW; w++) {
            const uint32_t v = s_part[w];
            total += v;
            before += w < wave ? v : 0u;
        }
        uint32_t run = before + incl - mine;
        for (uint32_t c = c0; c < c1; c++) {
            const uint32_t z = cz[c];
            cz[c] = run;
            run += z;
        }
        __syncthreads();
        if (tid == 0) {
            if (I.count0) gmem(I.count0)[r] = (int32_t)total;
        }
        // pass 2: scatter the order, write the row's pairs
        const gptr_t<uint32_t> row = gmem(I.out) + (uint64_t)step * RS;
        for (uint32_t ch = wave; ch < nch; ch += NW) {
            const uint32_t pos = ch * 64 + ln;
            const uint32_t idx = ordA[pos];
            const uint32_t b = big_bit(rowb, idx, K);
            const uint64_t m = __ballot(b);
            const uint32_t zb = __builtin_amdgcn_readfirstlane(cz[ch]);
            const uint32_t t = mbcnt(m);  // ones below me in the chunk
            const uint32_t dest = b ? total + (ch * 64u - zb) + t : zb + (ln - t);
            ordB[dest] = idx;
            if (I.absperm && dest < K) gmem(I.absperm)[(uint64_t)(step + 1) * K + dest] = (int32_t)idx;
            const uint32_t lo = (uint32_t)m, hi = (uint32_t)(m >> 32);
            const uint32_t o1 = zb + 32u - (uint32_t)__popc(lo);
            const uint32_t o3 = zb + 64u - (uint32_t)__popcll(m);
            const bool second = 2 * ch + 1 < npairs;
            if (ln == 0) {
                if (I.raw) {
                    row[2 * ch] = lo;
                    row[2 * ch + 1] = hi;
                } else {
                    row[4 * ch] = lo;
                    row[4 * ch + 1] = o1;
                    if (second) {
                        row[4 * ch + 2] = hi;
                        row[4 * ch + 3] = o3;
                    }
                }
                if (I.digest) {
                    const uint64_t g = I.gbase + (uint64_t)step * KW + 4ull * ch;
                    dsum += (uint64_t)dig_word(g, lo) + dig_word(g + 1, o1);
                    if (second) dsum += (uint64_t)dig_word(g + 2, hi) + dig_word(g + 3, o3);
                }
            }
        }
        __syncthreads();  // the new order is complete (and cz free) before the next step
        const gptr_t<uint32_t> tmp = ordA;
        ordA = ordB;
        ordB = tmp;
    }
    if (I.digest && ln == 0) atomicAdd((unsigned long long *)I.digest, (unsigned long long)dsum);
}


size_t pbwt_big_lds_bytes(uint32_t K) {
    const uint32_t nw32 = (K + 31) / 32, nch = (K + 63) / 64;
    return (size_t)((nw32 + 1) / 2 * 2 + nch) * 4;
}
uint32_t pbwt_big_max_k() { return kBigMaxK; }

hipError_t launch_pbwt_big(const BigItem *items, uint32_t nitems, uint32_t maxK, hipStream_t s) {
    if (!nitems) return hipSuccess;
    const size_t lds = pbwt_big_lds_bytes(maxK);
    hipError_t e = raise_lds_limit((const void *)k_pbwt_big, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_pbwt_big, dim3(nitems), dim3(BIG_NT), lds, s, items);
    return hipGetLastError();
}


// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// The chains address their row-by-row payloads from LDS byte 0: no static LDS
// may lie ahead of the dynamic buffer.
static hipError_t order_lds_at_zero(const void *fn) {
    hipFuncAttributes a{};
    hipError_t e = hipFuncGetAttributes(&a, fn);
    if (e != hipSuccess) return e;
    return a.sharedSizeBytes == 0 ? hipSuccess : hipErrorInvalidKernelFile;
}

// numbers 5 and 6 name the shapes of 2 and 4
static const PbwtVariant kPbwtVariants[] = {variant_256x8(),  variant_256x16(),  variant_512x20(),
                                            variant_512x32(), variant_1024x24(), variant_512x20(),
                                            variant_1024x24()};
constexpr int kNumPbwtVariants = sizeof(kPbwtVariants) / sizeof(kPbwtVariants[0]);

int pbwt_variant_count() { return kNumPbwtVariants; }
int pbwt_variant_threads(int v) { return kPbwtVariants[v].nt; }
int pbwt_variant_cpw(int v) { return kPbwtVariants[v].cpw; }
uint32_t pbwt_variant_maxk(int v) { return (uint32_t)(kPbwtVariants[v].nt * kPbwtVariants[v].cpw); }

size_t pbwt_lds_bytes(int v, uint32_t Kpad) {
    const int nt = kPbwtVariants[v].nt;
    const int ns = pbwt_slots_for(Kpad, nt);
    if (ns < 0 || ns > kPbwtVariants[v].cpw) return ~(size_t)0;
    return order_lds(nt, ns);
}
hipError_t pbwt_prepare(int v, size_t lds, int *occ) {
    const PbwtVariant &k = kPbwtVariants[v];
    for (const void *fn : {(const void *)k.rows, (const void *)k.aux, (const void *)k.dense}) {
        hipError_t e = order_lds_at_zero(fn);
        if (e == hipSuccess) e = raise_lds_limit(fn, lds);
        if (e != hipSuccess) return e;
    }
    if (!occ) return hipSuccess;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(occ, (const void *)k.rows, k.nt, lds);
}

hipError_t launch_order(int v, const TgtDev *tg, const OrderItem *items, bool rows, uint32_t grid,
                        const uint32_t *d_items, uint32_t *ctr, uint16_t *starts, size_t lds,
                        hipStream_t s) {
    if (!grid) return hipSuccess;
    hipLaunchKernelGGL(rows ? kPbwtVariants[v].rows : kPbwtVariants[v].aux, dim3(grid),
                       dim3(kPbwtVariants[v].nt), lds, s, tg, items, d_items, ctr, kMaxRuns, starts);
    return hipGetLastError();
}
hipError_t launch_dense(int v, const TgtDev *tg, uint32_t nblk, const uint16_t *starts, int32_t *absperm,
                        size_t lds, hipStream_t s) {
    hipLaunchKernelGGL(kPbwtVariants[v].dense, dim3(nblk), dim3(kPbwtVariants[v].nt), lds, s, tg, starts,
                       absperm);
    return hipGetLastError();
}

// Waves of a k_rows kernel: eight times what the device holds, each ending after
// its share, so that places come free all the time and other contexts' kernels get
// some.  With waves that stay to the end nothing else ran where they took all
// registers: 10 MB copied beside the blocks of 128 targets up to 13.5 ms instead
// of 0.3, now 2.3.  (Waves that end late also cost less so: the build takes 70.2
// instead of 71.5 ms, with four times 70.7, with twice 71.4.)
constexpr uint64_t kRowsRounds = 8;

// blocks: of the batch, or an upper bound; Kpad: the largest of the batch; ncu:
// compute units.  A batch launches the kernels that half of Kpad (the most
// runs of a block that a chain hands over) can reach.
hipError_t launch_rows(const TgtDev *tg, const uint32_t *d_n, uint32_t n, const uint32_t *pref,
                       RowItem *list, uint32_t *cnt, uint32_t Kpad, uint64_t blocks, uint32_t ncu,
                       hipStream_t s) {
    if (!blocks) return hipSuccess;
    using Fn = void (*)(const TgtDev *, const uint32_t *, uint32_t, const uint32_t *, const RowItem *,
                        const uint32_t *, uint32_t);
    static const Fn fns[kRowsKernels] = {k_rows<0>, k_rows<1>, k_rows<2>, k_rows<3>};
    hipLaunchKernelGGL(k_rows_list, dim3((uint32_t)std::min<uint64_t>((blocks + LIST_NT - 1) / LIST_NT, 2 * ncu)),
                       dim3(LIST_NT), 0, s, tg, d_n, n, pref, list, cnt);
    for (int k = 0; k < kRowsKernels; k++) {
        if (k && Kpad / 2 + 1 <= 64u * (uint32_t)kRowsEntries[k - 1]) break;
        const uint32_t ntog = Kpad / 32 + 2;
        const size_t lds = kRowsBias + (64 * (size_t)kRowsEntries[k] + ntog) * 4;
        int occ = 0;
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, (const void *)fns[k], 64, lds);
        if (e != hipSuccess) return e;
        const uint32_t grid = (uint32_t)std::min<uint64_t>(blocks, kRowsRounds * ncu * (uint64_t)std::max(occ, 1));
        hipLaunchKernelGGL(fns[k], dim3(grid), dim3(64), lds, s, tg, d_n, n, pref, list, cnt, ntog);
    }
    return hipGetLastError();
}

}  // namespace eimp
