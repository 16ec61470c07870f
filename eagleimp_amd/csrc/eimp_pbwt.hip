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
// now takes 8.7 ms and the rows 6.9 ms.  One target of 45,000 rows: 60.1 ms
// before, 19.0 + 0.3 ms now.
//
// Blocks with more runs than k_rows takes and the last block of a target when
// it has fewer than 16 rows are done row by row in k_order (order_dense).
// Where the order after every row is asked for (panel PBWT), k_order only
// leaves the order at the start of every block and k_dense does the blocks row
// by row, all of them independent.
#include <algorithm>

#include "eimp_device.h"
#include "eimp_launch.h"

namespace eimp {

namespace {

// header of a block done row by row (its rows are final)
constexpr uint32_t kDense = 0xFFFFu;

// Block q of a direction in processing order: cref block b, rows r0..r0+nrows-1
// of it, first output row s0 of the direction.  Backward blocks run from the
// last row down.
struct BlockGeo {
    uint32_t b, nrows, s0;
};
__device__ __forceinline__ BlockGeo block_geo(uint32_t q, uint32_t Mp, uint32_t nblk, bool rev) {
    BlockGeo g;
    g.b = rev ? nblk - 1 - q : q;
    g.nrows = min(16u, Mp - 16 * g.b);
    g.s0 = rev ? Mp - 16 * g.b - g.nrows : 16 * g.b;
    return g;
}

// Two haplotypes' keys from two cref values: bit j = the block's j-th row in
// processing order.
__device__ __forceinline__ uint32_t key_pair(uint32_t v, bool rev, uint32_t nrows) {
    if (!rev) return v;
    v = __builtin_bitreverse32(v);
    v = __builtin_amdgcn_alignbit(v, v, 16);
    const uint32_t sh = 16u - nrows;
    return (v >> sh) & ((0xFFFFu >> sh) * 0x10001u);
}

// A value the compiler cannot see through: what is computed from it inside a
// loop is computed there instead of being kept in registers across the loop.
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

__device__ __forceinline__ void hold(uint32_t &v) { asm volatile("" : "+v"(v)); }

// Gives registers that only some paths of a loop body write a (meaningless)
// definition inside the loop, at no cost: without one they would count as
// carried from turn to turn.
template <int N>
__device__ __forceinline__ void begin_life(uint32_t (&a)[N]) {
#pragma unroll
    for (int i = 0; i < N; i++) asm volatile("" : "=v"(a[i]));
}

// LDS accesses of one wave to memory that only this wave uses: the hardware
// keeps their order, the compiler must too
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Exclusive prefix sum over the workgroup's threads; total returned.  One
// barrier; red (NW words) must not be reused before the next one.
template <int NT>
__device__ __forceinline__ uint32_t wg_scan_excl(uint32_t v, uint32_t *red, uint32_t &total) {
    constexpr int NW = NT / 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = lane_id();
    const uint32_t ex = lane_scan_excl<64>(v);
    red[wave] = (uint32_t)__builtin_amdgcn_readlane((int)(ex + v), 63);
    __syncthreads();
    const uint32_t wv = red[ln & (NW - 1)];
    const uint32_t wex = lane_scan_excl<NW>(wv);
    total = (uint32_t)__builtin_amdgcn_readlane((int)(wex + wv), NW - 1);
    return ex + (uint32_t)__builtin_amdgcn_readlane((int)wex, (int)wave);
}

// LDS bytes before the row-by-row payloads: 32 (NS - 1) words, the largest
// amount a slot's store address sits below its destination (order_dense).
__host__ __device__ constexpr uint32_t dense_bias(int ns) { return 128u * (uint32_t)(ns - 1); }

// Most runs of a block that k_rows takes (62 entries per lane, one of them
// closing the list); with it three 512-thread chains of 10,240 positions fit a
// CU's LDS.
constexpr uint32_t kMaxRuns = 64 * 62 - 1;
// Run starts (uint16) a chain keeps room for: at most one run per two positions
// goes to k_rows, and the positions past Kpad may count as one more.
__host__ __device__ constexpr uint32_t order_starts(int nt, int e) {
    const uint32_t half = (uint32_t)(nt * e) / 2;
    return ((half < kMaxRuns ? half : kMaxRuns) + 2 + 3) / 4 * 4;
}
// LDS of one chain: order and keys (uint16 per position each), run starts,
// per-wave digit counts, digit bases, wave totals of three scans.
__host__ __device__ constexpr uint32_t order_lds(int nt, int e) {
    return 4u * (uint32_t)(nt * e) + 2u * order_starts(nt, e) + 512u * (uint32_t)(nt / 64) + 512u +
           16u * (uint32_t)(nt / 64);
}

// ---------------------------------------------------------------------------
// One block row by row, from the order in LDS.  Wave w holds chunks
// [w*NS, w*NS+NS) of 64 positions, one position per lane, as a 32-bit payload:
// doubled haplotype index << 16 | key.  Positions K..Kpad-1 (and whole padding
// chunks) carry all-ones bits: under the stable partition they never move, and
// they give the 1-padding of the last word.  A step:
//   pass 1  ballot of the row bit per slot: the slot's two data words go to
//           output lane c; the wave's zero count (scalar) to LDS
//   (barrier) zeros before the wave's first chunk and in the row (count0)
//   pass 2  per slot: the ones before the chunk are a scalar running sum, so
//           mbcnt of the ballot plus that base gives a one's destination and
//           a lane constant minus it a zero's; payloads scattered into LDS;
//           output lanes store their data / cumulative-zero pairs
//   (barrier)
//   pass 3  read back the payloads of my positions.
// A row whose K bits are all equal keeps the order: pass 2, the second
// barrier and pass 3 are skipped (the wave counts alternate between two LDS
// halves, so the next step's counts never overwrite ones still being read).
// Order and keys are read from ord and xs (over which the payloads then lie)
// and the new order is written to ord.  Not inlined: the chain's registers are
// sized by its other path, which nearly all blocks take.
// The kernels use dynamic LDS only (the host checks it), so LDS byte addresses
// are plain offsets from 0: pay[] starts at byte dense_bias(NS).
// ---------------------------------------------------------------------------
template <int NT, int NS>
__device__ __attribute__((noinline)) void order_dense(const TgtDev &T, const bool rev,
                                                      const BlockGeo geo, const bool emit,
                                                      uint32_t *smem, uint32_t *wzero2,
                                                      int32_t *__restrict__ absperm) {
    constexpr int NW = NT / 64;
    uint16_t *ord = (uint16_t *)smem;
    const uint16_t *xs = ord + NT * NS;
    uint64_t dsum = 0;
    const uint32_t K = T.K, Kpad = T.Kpad, RS = T.RS;
    const uint32_t nch = Kpad / 64;
    const uint32_t npairs = (K + 31) / 32;
    const uint32_t KW = 2 * npairs;
    uint32_t *pay = smem + dense_bias(NS) / 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = lane_id();
    const uint32_t ch0 = wave * NS;  // first chunk of this wave
    const uint32_t vbase4 = 4u * (ch0 * 64u + ln + 64u * (NS - 1));
    uint32_t p[NS];
#pragma unroll
    for (int c = 0; c < NS; c++) {
        const uint32_t id2 = ord[(ch0 + (uint32_t)c) * 64 + ln];
        p[c] = (id2 << 16) | *(const uint16_t *)((const char *)xs + id2);
    }
    __syncthreads();
    const bool dig = emit && __builtin_amdgcn_readfirstlane(T.digest != nullptr ? 1u : 0u) != 0;
    const bool raw = (__builtin_amdgcn_readfirstlane(T.flags) & TF_RAW) != 0;
    const uint32_t och = ch0 + ln;  // chunk stored by this lane
    const bool ostore = emit && ln < (uint32_t)NS && och < nch;
    // the raw layout has one word pair per chunk, the others two
    const bool second = !raw && 2 * och + 1 < npairs;
    const gptr_t<uint32_t> outrow =
        gmem(T.out) + ((rev ? (uint64_t)T.Mp : 0ull) + geo.s0) * RS;
    // global index of this lane's first word (digest): key g * kDigKey, rotation -g
    uint32_t g = (rev ? T.Mp * KW : 0u) + geo.s0 * KW + 4u * och;
    if (emit) {
        // the padding words of the block's rows: after the logical pairs zero,
        // in the raw layout all ones after the data words
        const uint32_t pw0 = raw ? 2 * nch : 2 * npairs, tw = (RS - pw0) / 2;
        const uint32_t fw = raw ? ~0u : 0u;
        for (uint32_t i = threadIdx.x; i < geo.nrows * tw; i += NT) {
            const uint32_t rr = i / tw, w = i - rr * tw;
            *(gptr_t<u32x2>)(outrow + (uint64_t)rr * RS + pw0 + 2 * w) = u32x2{fw, fw};
        }
    }
    uint32_t obyte;  // this lane's byte offset of its chunk's words within a row
    asm("" : "=v"(obyte) : "0"((raw ? 8u : 16u) * och));
    uint64_t rowaddr = (uint64_t)(size_t)outrow;
    uint32_t c0acc = 0;  // count0 of the block, lane = row
    for (uint32_t j = 0; j < geo.nrows; j++) {
        const uint32_t jbit = 1u << j;
        uint32_t olo, ohi;
        asm volatile("" : "=v"(olo), "=v"(ohi));  // lanes >= NS are never read
        uint64_t mk[NS];
        static_for<0, NS>([&](auto ci) {
            constexpr int c = decltype(ci)::value;
            const uint64_t m = __ballot((p[c] & jbit) != 0u);
            mk[c] = m;
            olo = writelane<c>(olo, (uint32_t)m);
            ohi = writelane<c>(ohi, (uint32_t)(m >> 32));
        });
        const uint32_t zl = 64u - (uint32_t)__popc(olo) - (uint32_t)__popc(ohi);
        const uint32_t zex = lane_scan_excl<NS>(zl);
        uint32_t *wzero = wzero2 + (j & 1u) * (uint32_t)NW;
        wzero[wave] = (uint32_t)__builtin_amdgcn_readlane((int)(zex + zl), NS - 1);
        __syncthreads();
        const uint32_t wv = wzero[ln & (NW - 1)];
        const uint32_t wex = lane_scan_excl<NW>(wv);
        const uint32_t run = (uint32_t)__builtin_amdgcn_readlane((int)wex, (int)wave);
        const uint32_t cnt0 = (uint32_t)__builtin_amdgcn_readlane((int)(wex + wv), NW - 1);
        c0acc = eimp_llvm_writelane(cnt0, j, c0acc);
        const uint32_t zbv = run + zex;
        if (cnt0 != 0u && cnt0 != K) {
            // For slot c let ob_c / run_c be the destinations of the row's
            // first one / zero at or after the chunk and t the ones below me
            // in the chunk: a one goes to ob_c + t, a zero to run_c + ln - t.
            // With x = ob_c + t + 32 (NS - 1 - c), dest + 32 (NS - 1 - c) is x
            // for a one and V - x for a zero, V = cnt0 + 64 ch0 + ln +
            // 64 (NS - 1) the same for every slot; 128 c is the store's
            // immediate offset.
            uint32_t a4 = (cnt0 + ch0 * 64u - run + 32u * (NS - 1)) * 4u;
            const uint32_t V4 = vbase4 + cnt0 * 4u;
            static_for<0, NS>([&](auto ci) {
                constexpr int c = decltype(ci)::value;
                const uint64_t m = mk[c];
                const uint32_t x4 = mbcnt(m) * 4u + a4;
                const uint32_t sel4 = __builtin_amdgcn_inverse_ballot_w64(m) ? x4 : V4 - x4;
                *(lds_ptr_t<uint32_t>)(size_t)(sel4 + 128u * (uint32_t)c) = p[c];
                a4 += (uint32_t)__popcll(m) * 4u - 128u;
                asm volatile("" : "+s"(a4));  // keeps the running sum in bytes
            });
            __syncthreads();
#pragma unroll
            for (int c = 0; c < NS; c++) p[c] = pay[(ch0 + (uint32_t)c) * 64 + ln];
        }
        if (absperm) {
            const gptr_t<int32_t> ap = gmem(absperm) + (uint64_t)(geo.s0 + j + 1) * K;
#pragma unroll
            for (int c = 0; c < NS; c++) {
                const uint32_t pos = (ch0 + (uint32_t)c) * 64 + opaque(ln);
                if (pos < K) ap[pos] = (int32_t)(p[c] >> 17);
            }
        }
        const uint32_t o1 = zbv + 32u - (uint32_t)__popc(olo);
        const uint32_t o3 = o1 + 32u - (uint32_t)__popc(ohi);
        if (ostore) {
            const gptr_t<char> rowb = (gptr_t<char>)(size_t)rowaddr;
            *(gptr_t<u32x2>)(rowb + obyte) = u32x2{olo, raw ? ohi : o1};
            if (second) *(gptr_t<u32x2>)(rowb + obyte + 8u) = u32x2{ohi, o3};
        }
        if (dig && ostore) {
            // rotl(v ^ key, g mod 32) == rotr by -g: one v_alignbit each
            const uint32_t dkey = g * kDigKey, dneg = 0u - g;
            dsum += __builtin_amdgcn_alignbit(olo ^ dkey, olo ^ dkey, dneg);
            const uint32_t x1 = o1 ^ (dkey + kDigKey);
            dsum += __builtin_amdgcn_alignbit(x1, x1, dneg - 1u);
            if (2 * och + 1 < npairs) {
                const uint32_t x2 = ohi ^ (dkey + 2u * kDigKey), x3 = o3 ^ (dkey + 3u * kDigKey);
                dsum += __builtin_amdgcn_alignbit(x2, x2, dneg - 2u);
                dsum += __builtin_amdgcn_alignbit(x3, x3, dneg - 3u);
            }
        }
        g += KW;
        rowaddr += RS * 4u;
    }
    if (emit && !rev && wave == 0 && ln < geo.nrows)
        gmem(T.count0)[geo.s0 + ln] = (int32_t)c0acc;
    __syncthreads();  // every wave has read back its payloads
#pragma unroll
    for (int c = 0; c < NS; c++) ord[(ch0 + (uint32_t)c) * 64 + ln] = (uint16_t)(p[c] >> 16);
    if (dig) {
        dsum = wave_sum64(dsum);
        if (ln == 0) atomicAdd((unsigned long long *)&T.digest[0], (unsigned long long)dsum);
    }
}

// Lanes of the wave (among those in `valid`) whose 8-bit digit (bits sh.. of v)
// equals mine: per bit the ballot of the bit, complemented where mine is zero,
// ands in (four vector instructions; the empty asm statements keep the compiler
// from splitting them).
__device__ __forceinline__ uint64_t match8(uint32_t v, uint32_t sh, uint64_t valid) {
    uint32_t lo = (uint32_t)valid, hi = (uint32_t)(valid >> 32);
    const uint32_t d = v >> sh;
    static_for<0, 8>([&](auto bi) {
        uint32_t s = (uint32_t)__builtin_amdgcn_sbfe((int)d, decltype(bi)::value, 1);
        asm("" : "+v"(s));
        const uint64_t B = __ballot(s != 0u);
        lo &= ~((uint32_t)B ^ s);
        hi &= ~((uint32_t)(B >> 32) ^ s);
        asm("" : "+v"(lo), "+v"(hi));
    });
    return ((uint64_t)hi << 32) | lo;
}

// One pass of the stable sort of R run entries by the 8-bit digit at bits sh:
// wave w holds entries [w SL 64, (w + 1) SL 64) in ev, 64 per slot, and writes
// them to their places in ent.  A slot's ranks come from match8 and the wave's
// running digit counts; one wave then turns the counts of all waves into
// bases.  Every wave holds its entries before the first barrier, so ent may be
// where they were read from.  between(): run by every thread after that
// barrier.
template <int NT, int EH, class F>
__device__ __forceinline__ void sort_pass(const uint32_t (&ev)[EH], uint32_t SL, uint32_t R,
                                          uint32_t sh, uint32_t *ent, uint16_t *hist, uint16_t *base,
                                          F &&between) {
    constexpr int NW = NT / 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = lane_id();
    const uint32_t i0 = wave * SL * 64 + opaque(ln);
    uint16_t *hw = hist + 256 * wave;
    uint32_t rk[EH];
    begin_life(rk);
    ((uint32_t *)hw)[ln] = 0;
    ((uint32_t *)hw)[64 + ln] = 0;
    wave_order();
    static_for<0, EH>([&](auto si) {
        constexpr int s = decltype(si)::value;
        if ((uint32_t)s < SL) {
            const bool valid = i0 + 64 * s < R;
            const uint64_t m = match8(ev[s], sh, __ballot(valid));
            uint16_t *h = hw + ((ev[s] >> sh) & 255u);
            const uint32_t before = *h, below = mbcnt(m);
            wave_order();
            rk[s] = before + below;
            if (valid && below == 0) *h = (uint16_t)(before + (uint32_t)__popcll(m));
            wave_order();
        }
    });
    __syncthreads();
    if (wave == 0) {
        // digits 4 ln .. 4 ln + 3: counts of earlier waves, then the base
        uint32_t a0 = 0, a1 = 0;  // two uint16 each; no count exceeds 65535
#pragma unroll
        for (int w = 0; w < NW; w++) {
            u32x2 *h = (u32x2 *)(hist + 256 * w + 4 * ln);
            const u32x2 v = *h;
            *h = u32x2{a0, a1};
            a0 += v[0];
            a1 += v[1];
        }
        const uint32_t t0 = a0 & 0xFFFFu, t1 = a0 >> 16, t2 = a1 & 0xFFFFu, t3 = a1 >> 16;
        const uint32_t ex = lane_scan_excl<64>(t0 + t1 + t2 + t3);
        *(u32x2 *)(base + 4 * ln) =
            u32x2{ex | ((ex + t0) << 16), (ex + t0 + t1) | ((ex + t0 + t1 + t2) << 16)};
    }
    between();
    __syncthreads();
    static_for<0, EH>([&](auto si) {
        constexpr int s = decltype(si)::value;
        if ((uint32_t)s < SL) {
            const uint32_t d = (ev[s] >> sh) & 255u;
            if (i0 + 64 * s < R) ent[(uint32_t)base[d] + hw[d] + rk[s]] = ev[s];
        }
    });
    __syncthreads();
}

// The chain of one (target, direction) over its 16-row blocks.  E positions
// per thread: thread x holds positions [x E, x E + E).  LDS: ord (doubled
// haplotype index per position), xs (the block's keys by haplotype), st (first
// position of each run, then the run's displacement).  The run entries being
// sorted (key << 16 | run) take ord's place: its indexes are in registers
// until the runs have moved.  xs is free once the entries are built, and takes
// the next block's keys then.
// rcap: most runs k_rows takes.  ROWS: the run lists are left for k_rows, other
// blocks' rows written; else starts receives Kpad (doubled) indexes per block,
// the order at its start.
template <int NT, int E, bool ROWS>
__device__ __forceinline__ void order_chain(const TgtDev &T, const bool rev, uint32_t *smem,
                                            const uint32_t rcap, uint16_t *__restrict__ starts) {
    constexpr int NW = NT / 64, EH = E / 2;
    constexpr uint32_t NPOS = (uint32_t)(NT * E);
    static_assert(E % 2 == 0 && E <= 32, "positions go in pairs, their flags into one register");
    uint16_t *ord = (uint16_t *)smem;
    uint16_t *xs = ord + NPOS;
    uint16_t *st = xs + NPOS;
    uint16_t *hist = st + order_starts(NT, E);
    uint16_t *base = hist + 256 * NW;
    uint32_t *red = (uint32_t *)(base + 256);
    uint32_t *ent = smem;
    const uint32_t tid = threadIdx.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), ln = lane_id();
    const uint32_t Mp = T.Mp, Kpad = T.Kpad, RS = T.RS;
    const uint32_t nblk = (Mp + 15) / 16;
    const uint32_t rmax = min(rcap, Kpad / 2);
    const gptr_t<const uint16_t> cref = gmem((const uint16_t *)T.cref);
    const gptr_t<uint16_t> hdr = gmem(T.hdr) + (rev ? nblk : 0u);
    uint32_t pf[EH];  // the next block's keys, loaded one block ahead
    auto fetch = [&](uint32_t q) {
        const BlockGeo g = block_geo(q, Mp, nblk, rev);
        const gptr_t<const uint32_t> src = (gptr_t<const uint32_t>)(cref + (uint64_t)g.b * Kpad);
#pragma unroll
        for (int i = 0; i < EH; i++) {
            const uint32_t w = opaque(tid) + (uint32_t)i * NT;
            pf[i] = src[min(w, Kpad / 2 - 1)];
        }
    };
    // xs = keys of block q, then the block after it is fetched
    auto stage = [&](uint32_t q) {
        const BlockGeo g = block_geo(q, Mp, nblk, rev);
#pragma unroll
        for (int i = 0; i < EH; i++) {
            const uint32_t w = opaque(tid) + (uint32_t)i * NT;
            ((uint32_t *)xs)[w] = w < Kpad / 2 ? key_pair(pf[i], rev, g.nrows) : ~0u;
        }
        if (q + 1 < nblk) fetch(q + 1);
    };
    // panel order; positions past Kpad hold index Kpad, whose key is all ones
    // (they never move)
#pragma unroll
    for (int i = 0; i < EH; i++) {
        const uint32_t w = tid + (uint32_t)i * NT;
        const uint32_t a = min(2 * w, Kpad), b = min(2 * w + 1, Kpad);
        ((uint32_t *)ord)[w] = 2 * a | (2 * b << 16);
    }
    fetch(0);
    stage(0);
    __syncthreads();
    auto key_at = [&](uint32_t id2) { return (uint32_t)*(const uint16_t *)((const char *)xs + id2); };
    for (uint32_t q = 0; q < nblk; q++) {
        const BlockGeo geo = block_geo(q, Mp, nblk, rev);
        const uint32_t tq = opaque(tid), pos0 = tq * E;
        // keys of my positions and where a run of equal keys begins: flag of
        // position pos0 + e at bit e/2 (e even) or 16 + e/2 (e odd)
        uint32_t idp[EH];
#pragma unroll
        for (int i = 0; i < EH; i++) idp[i] = ((const uint32_t *)ord)[tq * EH + i];
        if constexpr (!ROWS) {
            const gptr_t<uint32_t> so = (gptr_t<uint32_t>)(gmem(starts) + (uint64_t)q * Kpad);
#pragma unroll
            for (int i = 0; i < EH; i++)
                if (pos0 + 2 * i < Kpad) so[tq * EH + i] = idp[i];
        }
        uint32_t flags = 0;
        {
            uint32_t prev = tid ? key_at(ord[pos0 - 1]) << 16 : 0u;
#pragma unroll
            for (int i = 0; i < EH; i++) {
                const uint32_t kk = key_at(idp[i] & 0xFFFFu) | (key_at(idp[i] >> 16) << 16);
                const uint32_t x = kk ^ __builtin_amdgcn_alignbit(kk, prev, 16);
                typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
                const u16x2 f = __builtin_elementwise_min(__builtin_bit_cast(u16x2, x), u16x2{1, 1});
                flags |= __builtin_bit_cast(uint32_t, f) << i;
                prev = kk;
                if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
        }
        // position 0 begins the first run; the positions past Kpad are a run
        // of their own that is not sorted and stays where it is
        if (tid == 0) flags |= 1u;
        if (Kpad - pos0 < (uint32_t)E) flags |= 1u << ((Kpad - pos0) / 2);
        uint32_t R;
        const uint32_t rbase = wg_scan_excl<NT>((uint32_t)__popc(flags), red, R);
        R = __builtin_amdgcn_readfirstlane(R) - (Kpad < NPOS ? 1u : 0u);
        if (R <= rmax && (!ROWS || geo.nrows == 16)) {
            auto flag = [&](auto ei) {
                constexpr int e = decltype(ei)::value;
                return (flags >> (e / 2 + 16 * (e & 1))) & 1u;
            };
            {
                uint16_t *w = st + rbase;
                static_for<0, E>([&](auto ei) {
                    if (flag(ei)) *w++ = (uint16_t)(pos0 + decltype(ei)::value);
                });
                if (tid == 0) st[R] = (uint16_t)Kpad;
            }
            __syncthreads();
            // the runs' entries, and the run list for k_rows in the block's rows
            const uint32_t SL = (R + NT - 1) / NT;  // slots of 64 entries per wave, <= EH
            {
                uint32_t ev[EH];
                begin_life(ev);
                const gptr_t<uint32_t> list =
                    gmem(T.out) + ((rev ? (uint64_t)Mp : 0ull) + geo.s0) * RS;
                static_for<0, EH>([&](auto si) {
                    constexpr int s = decltype(si)::value;
                    if ((uint32_t)s < SL) {
                        const uint32_t i = wave * SL * 64 + opaque(ln) + 64 * s;
                        const uint32_t a = st[min(i, R - 1)];
                        const uint32_t k = key_at(ord[a]) << 16;
                        ev[s] = k | i;
                        if (ROWS && i < R) list[i] = k | a;
                    }
                });
                if (ROWS && tid == 0) hdr[q] = (uint16_t)R;
                sort_pass<NT, EH>(ev, SL, R, 16, ent, hist, base, [&]() {
                    if (q + 1 < nblk) stage(q + 1);
                });
            }
            {
                uint32_t ev[EH];
                begin_life(ev);
                static_for<0, EH>([&](auto si) {
                    constexpr int s = decltype(si)::value;
                    if ((uint32_t)s < SL)
                        ev[s] = ent[min(wave * SL * 64 + opaque(ln) + 64 * s, R - 1)];
                });
                sort_pass<NT, EH>(ev, SL, R, 24, ent, hist, base, []() {});
            }
            // new start of every run: prefix sum of the lengths in key order,
            // SL consecutive sorted runs per thread
            uint32_t ra[EH], rl[EH];
            begin_life(ra);
            begin_life(rl);
            uint32_t sum = 0;
            static_for<0, EH>([&](auto si) {
                constexpr int s = decltype(si)::value;
                if ((uint32_t)s < SL) {
                    const uint32_t i = tq * SL + s;
                    const uint32_t run = ent[min(i, R - 1)] & 0xFFFFu;
                    const uint32_t a = st[run], b = st[run + 1];
                    ra[s] = (run << 16) | a;
                    rl[s] = i < R ? b - a : 0u;
                    sum += rl[s];
                }
            });
            uint32_t tot;
            uint32_t at = wg_scan_excl<NT>(sum, red + NW, tot);
            static_for<0, EH>([&](auto si) {
                constexpr int s = decltype(si)::value;
                if ((uint32_t)s < SL) {
                    if (tq * SL + s < R) st[ra[s] >> 16] = (uint16_t)(at - (ra[s] & 0xFFFFu));
                    at += rl[s];
                }
            });
            if (tid == 0) st[R] = 0;
            __syncthreads();
            // every haplotype moves with its run (displacements are signed 16-
            // bit: Kpad < 32768)
            const int16_t *d = (const int16_t *)st + (int32_t)rbase - 1;
            uint16_t *me = ord + pos0;
            static_for<0, E>([&](auto ei) {
                constexpr int e = decltype(ei)::value;
                d += flag(ei);
                me[(int32_t)*d + e] = (uint16_t)((e & 1) ? idp[e / 2] >> 16 : idp[e / 2]);
                // few lookups in flight at a time: registers, and other
                // workgroups' waves fill the gaps
                if constexpr (e % 8 == 7) __builtin_amdgcn_sched_barrier(0);
            });
        } else {
            order_dense<NT, E>(T, rev, geo, ROWS, smem, red + 2 * NW, nullptr);
            if (ROWS && tid == 0) hdr[q] = (uint16_t)kDense;
            if (q + 1 < nblk) {
                fetch(q + 1);  // again: registers are not kept across the call
                stage(q + 1);
            }
        }
        __syncthreads();
    }
}

// Waves per SIMD that one workgroup's LDS allows at the variant's capacity: the
// register budget is capped so that VGPRs do not lower it (512 x 20: three
// workgroups, 80 registers; 8.65 ms for 384 chains of 941 blocks at K = 10,000
// against 9.36 ms with two workgroups and 128 registers).
constexpr int order_waves_hint(int NT, int CPW) {
    const int w = (163840 / (int)order_lds(NT, CPW)) * (NT / 256);
    return w < 1 ? 1 : (w > 6 ? 6 : w);
}

// positions per thread instantiated; a target uses the smallest that holds Kpad
constexpr int kSlotCounts[] = {2, 4, 6, 8, 10, 12, 14, 16, 20, 24, 28, 32};
constexpr int kNumSlotCounts = sizeof(kSlotCounts) / sizeof(kSlotCounts[0]);

__host__ __device__ inline int pbwt_slots_for(uint32_t Kpad, int nt) {
    const uint32_t need = (Kpad + nt - 1) / nt;
    for (int i = 0; i < kNumSlotCounts; i++)
        if ((uint32_t)kSlotCounts[i] >= need) return kSlotCounts[i];
    return -1;
}

// Chains, one per item; with a counter the workgroups take items from it in
// turn until *d_items is reached, else workgroup x does item x.
template <int NT, int CPW, bool ROWS>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(order_waves_hint(NT, CPW))))
void k_order(const TgtDev *__restrict__ tg, const PbwtItem *__restrict__ items,
             const uint32_t *__restrict__ d_items, uint32_t *__restrict__ ctr, uint32_t rcap,
             uint16_t *__restrict__ starts) {
    // dynamic LDS only; the next item's index passes through smem[0], which no
    // item uses between two items
    extern __shared__ uint32_t smem[];
    // highest wave priority for instruction issue: the chains bound the
    // launch, and other contexts' kernels may share these CUs
    __builtin_amdgcn_s_setprio(3);
    for (uint32_t once = 0;; once++) {
        uint32_t i = blockIdx.x;
        if (ctr) {
            if (threadIdx.x == 0) smem[0] = atomicAdd(ctr, 1u);
            __syncthreads();
            i = __builtin_amdgcn_readfirstlane(smem[0]);
            __syncthreads();
            if (i >= *d_items) break;
        } else if (once) {
            break;
        }
        const PbwtItem it = items[i];
        const TgtDev &T = tg[it.t];
        const int ns = pbwt_slots_for(T.Kpad, NT);
        static_for<0, kNumSlotCounts>([&](auto ii) {
            constexpr int NSv = kSlotCounts[decltype(ii)::value];
            if constexpr (NSv <= CPW) {
                if (ns == NSv) order_chain<NT, NSv, ROWS>(T, it.dir != 0, smem, rcap, starts);
            }
        });
        __syncthreads();
    }
}

// Block x of a forward chain row by row from the order at its start (k_order's
// starts), with the order after every row in absperm (row 0: the panel order).
template <int NT, int E>
__device__ __forceinline__ void dense_block(const TgtDev &T, uint32_t q, const uint16_t *starts,
                                            int32_t *absperm, uint32_t *smem) {
    constexpr uint32_t NPOS = (uint32_t)(NT * E);
    constexpr int NW = NT / 64;
    uint32_t *ord = smem, *xs = smem + NPOS / 2;
    uint32_t *red = smem + order_lds(NT, E) / 4 - 4 * NW;
    const uint32_t Kpad = T.Kpad, K = T.K;
    const BlockGeo geo = block_geo(q, T.Mp, (T.Mp + 15) / 16, false);
    const gptr_t<const uint32_t> src = (gptr_t<const uint32_t>)(gmem(starts) + (uint64_t)q * Kpad);
    const gptr_t<const uint32_t> key =
        (gptr_t<const uint32_t>)(gmem((const uint16_t *)T.cref) + (uint64_t)geo.b * Kpad);
    for (uint32_t w = threadIdx.x; w < NPOS / 2; w += NT) {
        const bool in = w < Kpad / 2;
        ord[w] = in ? src[w] : 2 * Kpad * 0x10001u;  // past Kpad: index Kpad, all-ones key
        xs[w] = in ? key[w] : ~0u;
    }
    if (q == 0)
        for (uint32_t k = threadIdx.x; k < K; k += NT) gmem(absperm)[k] = (int32_t)k;
    __syncthreads();
    order_dense<NT, E>(T, false, geo, true, smem, red + 2 * NW, absperm);
}
// (order_dense's register budget is that of all kernels that call it)
template <int NT, int CPW>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(order_waves_hint(NT, CPW))))
void k_dense(const TgtDev *__restrict__ tg,
                                              const uint16_t *__restrict__ starts,
                                              int32_t *__restrict__ absperm) {
    extern __shared__ uint32_t smem[];
    const int ns = pbwt_slots_for(tg->Kpad, NT);
    static_for<0, kNumSlotCounts>([&](auto ii) {
        constexpr int NSv = kSlotCounts[decltype(ii)::value];
        if constexpr (NSv <= CPW) {
            if (ns == NSv) dense_block<NT, NSv>(*tg, blockIdx.x, starts, absperm, smem);
        }
    });
}

// ---------------------------------------------------------------------------
// k_rows: the 16 rows of a block from its run list, one wave per block.
//
// An entry is key << 16 | first position; entry i's run ends where entry i+1's
// begins.  A last entry (all-ones key, position Kpad, no length) stands after
// them; under the stable partition it stays last.  Per row j, lane x takes
// entries [x Ej, x Ej + Ej) (Ej odd: no two lanes on one LDS bank):
//   x = entry ^ previous entry; bit j of x: the row's bits change here, so
//       position P is marked in the row's bit map: -2^P where ones begin, +2^P
//       where they end (LDS add on the word)
//   bits j.. of x all zero: the two runs stay together from here on; the
//       entry is dropped (its length stays with the previous one)
//   one packed prefix sum over the wave, {4 x entries kept, length} of the
//       zeros, and one of 4 x entries kept give every entry's new index and
//       first position: zeros in order from 0, ones after all zeros
// then the entries are scattered (read into registers before), and the row's
// words come from the marks: a word's sum, one less where a run goes on into
// it (run_states), a scan of the words' zeros for the offsets.
// Bound by vector instructions: about 18 per 64 entries and row and 40 per 64
// word pairs and row; one wave per block because two barriers a row cost a
// workgroup more than the wave's own latency.
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

// Row of bit bm (in the key's half of an entry) on n entries: returns its zero
// count, leaves the next row's entries and their number in n.
template <int E>
__device__ __forceinline__ uint32_t rows_step(const uint32_t bm, uint32_t &n, uint32_t *ent,
                                              uint32_t *tog) {
    const uint32_t ln = opaque(lane_id());
    const uint32_t first = ln * E;
    uint32_t p[E + 1], dst[E];
    const uint32_t pv = ent[ln ? first - 1 : 0];
#pragma unroll
    for (int e = 0; e <= E; e++) p[e] = ent[first + e];
    // packed {4 x entries kept, length} prefix sums of my zeros (zacc) and my
    // ones (oacc); an entry notes the sum of its own kind before it
    uint32_t zacc = 0, oacc = 0, prev = ln ? pv : 0u;
    // the conditions fit the scalar registers up to here; beyond, they are
    // computed again
    constexpr bool keep = E <= 17;
    uint64_t kept[E], one[E];
    uint32_t b = bm;
    static_for<0, E>([&](auto ei) {
        constexpr int e = decltype(ei)::value;
        const uint32_t x = p[e] ^ prev;
        prev = p[e];
        one[e] = __ballot((p[e] & b) != 0u);
        kept[e] = __ballot(x >= b) | (e == 0 ? 1ull : 0ull);
        const uint64_t changed = e == 0 ? __ballot((x & b) != 0u) : one[e] ^ one[e ? e - 1 : 0];
        if (__builtin_amdgcn_inverse_ballot_w64(changed)) {
            const uint32_t P = p[e] & 0xFFFFu;
            const uint32_t sign = __builtin_amdgcn_inverse_ballot_w64(one[e]) ? ~0u : 1u;
            __hip_atomic_fetch_add(&tog[P >> 5], sign << (P & 31), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WAVEFRONT);
        }
        const uint32_t c = __builtin_amdgcn_inverse_ballot_w64(kept[e]) ? 0x40000u : 0u;
        const uint32_t w = ((p[e + 1] - p[e]) & 0xFFFFu) | c;
        const bool o = __builtin_amdgcn_inverse_ballot_w64(one[e]);
        dst[e] = o ? oacc : zacc;
        const uint32_t wz = o ? 0u : w;
        zacc += wz;
        oacc += w - wz;
        // four entries at a time: the next ones wait for these sums
        if constexpr (e % 4 == 3) {
            asm volatile("" : "+v"(zacc), "+v"(oacc), "+s"(b));
            static_for<e + 2, (e + 6 < E + 1 ? e + 6 : E + 1)>(
                [&](auto k) { hold(p[decltype(k)::value]); });
        }
    });
    const uint32_t zx = lane_scan_excl<64>(zacc), ox = lane_scan_excl<64>(oacc);
    const uint32_t ztot = (uint32_t)__builtin_amdgcn_readlane((int)(zx + zacc), 63);
    const uint32_t otot = (uint32_t)__builtin_amdgcn_readlane((int)(ox + oacc), 63);
    wave_order();
    // zeros from index and position 0, ones behind them all
    const uint32_t ob = ox + ztot;
    if constexpr (!keep) {
        b = bm;
        asm volatile("" : "+s"(b) : "s"(ztot));
        prev = ln ? pv : 0u;
    }
    static_for<0, E>([&](auto ei) {
        constexpr int e = decltype(ei)::value;
        if constexpr (!keep) {
            one[e] = __ballot((p[e] & b) != 0u);
            kept[e] = __ballot((p[e] ^ prev) >= b) | (e == 0 ? 1ull : 0ull);
            prev = p[e];
        }
        const uint32_t to = dst[e] + (__builtin_amdgcn_inverse_ballot_w64(one[e]) ? ob : zx);
        if (__builtin_amdgcn_inverse_ballot_w64(kept[e]))
            *(uint32_t *)((char *)ent + (to >> 16)) = (p[e] & 0xFFFF0000u) | (to & 0xFFFFu);
        if constexpr (!keep && e % 4 == 3) {
            asm volatile("" : "+s"(b)::"memory");
            static_for<e + 1, (e + 5 < E ? e + 5 : E)>(
                [&](auto k) { hold(p[decltype(k)::value]); });
        }
    });
    n = (ztot + otot) >> 18;
    return ztot & 0xFFFFu;
}

// entries per lane instantiated: odd
constexpr int kRowEntries[] = {1, 3, 5, 7, 9, 11, 13, 17, 21, 25, 33, 41, 49, 63};
constexpr int kNumRowEntries = sizeof(kRowEntries) / sizeof(kRowEntries[0]);
__device__ __forceinline__ uint32_t row_entries(uint32_t n) {
    const uint32_t need = (n + 63) / 64;
    uint32_t r = kRowEntries[kNumRowEntries - 1];
#pragma unroll
    for (int i = kNumRowEntries - 2; i >= 0; i--)
        if (need <= (uint32_t)kRowEntries[i]) r = kRowEntries[i];
    return r;
}

template <int EMAX>
__device__ __forceinline__ void rows_block(const TgtDev &T, const bool rev, const uint32_t q,
                                           const uint32_t R, uint32_t *ent, uint32_t *tog,
                                           uint64_t &dsum) {
    const uint32_t ln = lane_id();
    const uint32_t K = T.K, Mp = T.Mp, Kpad = T.Kpad, RS = T.RS;
    const uint32_t nblk = (Mp + 15) / 16, nch = Kpad / 64, npairs = (K + 31) / 32, KW = 2 * npairs;
    const BlockGeo geo = block_geo(q, Mp, nblk, rev);
    const bool raw = (T.flags & TF_RAW) != 0;
    const bool dig = T.digest != nullptr;
    const gptr_t<uint32_t> outrow = gmem(T.out) + ((rev ? (uint64_t)Mp : 0ull) + geo.s0) * RS;
    const uint32_t endv = 0xFFFF0000u | Kpad;
    for (uint32_t i = ln; i < R; i += 64) ent[i] = outrow[i];
    uint32_t n = R + 1;  // entries, the last one included
    uint32_t Ej = row_entries(n);
    for (uint32_t i = R + ln; i <= 64u * Ej; i += 64) ent[i] = endv;
    const uint32_t pw0 = raw ? 2 * nch : 2 * npairs, tw = (RS - pw0) / 2;  // padding pairs of a row
    const uint32_t fw = raw ? ~0u : 0u;
    uint32_t g0 = (rev ? Mp * KW : 0u) + geo.s0 * KW;
    uint32_t c0acc = 0;
    wave_order();
#pragma unroll 1
    for (uint32_t j = 0; j < 16; j++) {
        uint32_t cnt0 = 0;
        static_for<0, kNumRowEntries>([&](auto ii) {
            constexpr int E = kRowEntries[decltype(ii)::value];
            if constexpr (E <= EMAX) {
                if (Ej == (uint32_t)E) cnt0 = rows_step<E>(0x10000u << j, n, ent, tog);
            }
        });
        c0acc = eimp_llvm_writelane(cnt0, j, c0acc);
        Ej = row_entries(n);
        // entries past the last one: no length, never kept
        for (uint32_t i = n + ln; i <= 64u * Ej; i += 64) ent[i] = endv;
        wave_order();
        // the row's words: 64 positions per lane
        const gptr_t<uint32_t> row = outrow + (uint64_t)j * RS;
        uint32_t zrun = 0, state = 0;
        for (uint32_t c0 = 0; c0 < nch; c0 += 64) {
            const uint32_t ch = c0 + ln;
            const bool in = ch < nch;
            u32x2 t = u32x2{0u, 0u};
            if (in) {
                t = *(u32x2 *)(tog + 2 * ch);
                *(u32x2 *)(tog + 2 * ch) = u32x2{0u, 0u};
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
            const uint32_t zl = z0 + 32u - (uint32_t)__popc(hi);
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
        if (ln < tw) *(gptr_t<u32x2>)(row + pw0 + 2 * ln) = u32x2{fw, fw};
        g0 += KW;
        wave_order();
    }
    if (ln == 0) tog[Kpad / 32] = 0;  // the last entry's toggle
    if (!rev && ln < 16) gmem(T.count0)[geo.s0 + ln] = (int32_t)c0acc;
    wave_order();
}

// k_rows kernels by entries per lane: LDS and registers go with the most
// entries of a wave, and one kernel for all blocks would have two waves per
// SIMD.  Kernel k does the blocks of R + 1 <= 64 kRowsEntries[k] entries that
// the kernel before it does not.
constexpr int kRowsKernels = 3;
constexpr int kRowsEntries[kRowsKernels] = {17, 33, 63};

// Sorts the blocks into one list per k_rows kernel (their order within a list
// does not matter).  pref: per target (of *d_n, or n) its first block, both
// directions, pref[n] their number; cnt: kRowsKernels list lengths, zero
// beforehand.  The lists of kernels 0 and 1 share `total` entries from both
// ends, kernel 2's follows them.
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
            list[mine == 1 ? total - 1 - at : (mine == 2 ? total + at : at)] = item;
        }
        __syncthreads();
    }
}

template <int KERNEL>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(KERNEL == 0 ? 6 : (KERNEL == 1 ? 4 : 2)))) void k_rows(
    const TgtDev *__restrict__ tg, const uint32_t *__restrict__ d_n, uint32_t n,
    const uint32_t *__restrict__ pref, const RowItem *__restrict__ list,
    const uint32_t *__restrict__ cnt, uint32_t ntog) {
    extern __shared__ uint32_t smem[];
    constexpr int EMAX = kRowsEntries[KERNEL];
    uint32_t *ent = smem, *tog = smem + 64 * EMAX + 2;
    const uint32_t items = cnt[KERNEL];
    if (blockIdx.x >= items) return;
    const uint32_t total = pref[d_n ? *d_n : n];
    for (uint32_t i = lane_id(); i < ntog; i += 64) tog[i] = 0;
    wave_order();
    for (uint32_t i = blockIdx.x; i < items; i += gridDim.x) {
        const RowItem it = list[KERNEL == 1 ? total - 1 - i : (KERNEL == 2 ? total + i : i)];
        const TgtDev &T = tg[it.chain >> 1];
        uint64_t dsum = 0;
        rows_block<EMAX>(T, (it.chain & 1u) != 0, it.q, it.runs, ent, tog, dsum);
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
        // the padding words of every row, stored once (as pbwt_steps)
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

// Variants of the chain kernel: (threads, most positions per thread).
struct PbwtVariant {
    int nt, cpw;
    // chains for k_rows; chains that leave the order at every block's start
    void (*fn)(const TgtDev *, const PbwtItem *, const uint32_t *, uint32_t *, uint32_t, uint16_t *);
    void (*starts)(const TgtDev *, const PbwtItem *, const uint32_t *, uint32_t *, uint32_t, uint16_t *);
    void (*dense)(const TgtDev *, const uint16_t *, int32_t *);
};
#define PBWT_VARIANT(NT, CPW) {NT, CPW, k_order<NT, CPW, true>, k_order<NT, CPW, false>, k_dense<NT, CPW>}
static const PbwtVariant kPbwtVariants[] = {
    PBWT_VARIANT(256, 8),  PBWT_VARIANT(256, 16),  PBWT_VARIANT(512, 20),
    PBWT_VARIANT(512, 32), PBWT_VARIANT(1024, 24),
    // numbers 5 and 6 name the shapes of 2 and 4
    PBWT_VARIANT(512, 20), PBWT_VARIANT(1024, 24),
};
#undef PBWT_VARIANT
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
    for (const void *fn : {(const void *)k.fn, (const void *)k.starts, (const void *)k.dense}) {
        hipError_t e = order_lds_at_zero(fn);
        if (e == hipSuccess) e = raise_lds_limit(fn, lds);
        if (e != hipSuccess) return e;
    }
    if (!occ) return hipSuccess;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(occ, (const void *)k.fn, k.nt, lds);
}

hipError_t launch_order(int v, const TgtDev *tg, const PbwtItem *items, uint32_t nitems,
                        const uint32_t *d_items, uint32_t *ctr, uint16_t *starts, size_t lds,
                        hipStream_t s) {
    if (!nitems) return hipSuccess;
    hipLaunchKernelGGL(starts ? kPbwtVariants[v].starts : kPbwtVariants[v].fn, dim3(nitems),
                       dim3(kPbwtVariants[v].nt), lds, s, tg, items, d_items, ctr, kMaxRuns, starts);
    return hipGetLastError();
}
hipError_t launch_dense(int v, const TgtDev *tg, uint32_t nblk, const uint16_t *starts, int32_t *absperm,
                        size_t lds, hipStream_t s) {
    hipLaunchKernelGGL(kPbwtVariants[v].dense, dim3(nblk), dim3(kPbwtVariants[v].nt), lds, s, tg, starts,
                       absperm);
    return hipGetLastError();
}

// blocks: of the batch, or an upper bound; Kpad: the largest of the batch; ncu:
// compute units.  A batch launches the kernels that half of Kpad (the most
// runs of a block that a chain hands over) can reach.
hipError_t launch_rows(const TgtDev *tg, const uint32_t *d_n, uint32_t n, const uint32_t *pref,
                       RowItem *list, uint32_t *cnt, uint32_t Kpad, uint64_t blocks, uint32_t ncu,
                       hipStream_t s) {
    if (!blocks) return hipSuccess;
    using Fn = void (*)(const TgtDev *, const uint32_t *, uint32_t, const uint32_t *, const RowItem *,
                        const uint32_t *, uint32_t);
    static const Fn fns[kRowsKernels] = {k_rows<0>, k_rows<1>, k_rows<2>};
    hipLaunchKernelGGL(k_rows_list, dim3((uint32_t)std::min<uint64_t>((blocks + LIST_NT - 1) / LIST_NT, 2 * ncu)),
                       dim3(LIST_NT), 0, s, tg, d_n, n, pref, list, cnt);
    for (int k = 0; k < kRowsKernels; k++) {
        if (k && Kpad / 2 + 1 <= 64u * (uint32_t)kRowsEntries[k - 1]) break;
        const uint32_t ntog = Kpad / 32 + 2;
        const size_t lds = (64 * (size_t)kRowsEntries[k] + 2 + ntog) * 4;
        int occ = 0;
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, (const void *)fns[k], 64, lds);
        if (e != hipSuccess) return e;
        const uint32_t grid = (uint32_t)std::min<uint64_t>(blocks, ncu * (uint64_t)std::max(occ, 1));
        hipLaunchKernelGGL(fns[k], dim3(grid), dim3(64), lds, s, tg, d_n, n, pref, list, cnt, ntog);
    }
    return hipGetLastError();
}

}  // namespace eimp
