// eimp_order.h -- the order chain of the compressed PBWT (overview in
// eimp_pbwt.hip); one translation unit per shape instantiates it.
#pragma once

#include "eimp_device.h"

namespace eimp {

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

// Arguments of a called function arrive in vector registers: wave-uniform ones
// are taken back into scalar registers on entry.
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
template <class T>
__device__ __forceinline__ T *uniform(T *p) {
    const uint64_t v = (uint64_t)(size_t)p;
    return (T *)(size_t)(((uint64_t)uniform((uint32_t)(v >> 32)) << 32) | uniform((uint32_t)v));
}
// LDS byte address b of the workgroup's dynamic LDS (the kernels have no other,
// so it begins at 0): offsets from it stay immediate offsets
__device__ __forceinline__ lds_ptr_t<uint32_t> lds_at(uint32_t b) {
    return (lds_ptr_t<uint32_t>)(size_t)b;
}
using TgtConst = const __attribute__((address_space(4))) TgtDev;

// a wave-uniform value the compiler cannot see through
__device__ __forceinline__ uint32_t opaque_s(uint32_t v) {
    v = __builtin_amdgcn_readfirstlane(v);
    asm volatile("" : "+s"(v));
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
__device__ __forceinline__ uint32_t wg_scan_excl(uint32_t v, lds_ptr_t<uint32_t> red, uint32_t &total) {
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

// Most runs of a block that k_rows takes (61 entries per lane, one of them
// closing the list); with it three 512-thread chains of 10,240 positions fit a
// CU's LDS.
constexpr uint32_t kMaxRuns = 64 * 61 - 1;
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
__device__ __attribute__((noinline)) void order_dense(const TgtDev *tgt, uint32_t rev_, BlockGeo geo,
                                                      uint32_t emit_, int32_t *absperm) {
    TgtConst &T = *cmem(uniform(tgt));
    const bool rev = uniform(rev_) != 0, emit = uniform(emit_) != 0;
    geo = BlockGeo{uniform(geo.b), uniform(geo.nrows), uniform(geo.s0)};
    absperm = uniform(absperm);
    const lds_ptr_t<uint32_t> smem = lds_at(0);
    // 2 x NW: zeros of each wave's chunks, by step parity
    const lds_ptr_t<uint32_t> wzero2 = lds_at(order_lds(NT, NS) - 8u * (NT / 64));
    constexpr int NW = NT / 64;
    const lds_ptr_t<uint16_t> ord = (lds_ptr_t<uint16_t>)smem, xs = ord + NT * NS;
    uint64_t dsum = 0;
    const uint32_t K = T.K, Kpad = T.Kpad, RS = T.RS;
    const uint32_t nch = Kpad / 64;
    const uint32_t npairs = (K + 31) / 32;
    const uint32_t KW = 2 * npairs;
    const lds_ptr_t<uint32_t> pay = smem + dense_bias(NS) / 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = lane_id();
    const uint32_t ch0 = wave * NS;  // first chunk of this wave
    const uint32_t vbase4 = 4u * (ch0 * 64u + ln + 64u * (NS - 1));
    uint32_t p[NS];
#pragma unroll
    for (int c = 0; c < NS; c++) {
        const uint32_t id2 = ord[(ch0 + (uint32_t)c) * 64 + ln];
        p[c] = (id2 << 16) | *(lds_ptr_t<uint16_t>)((lds_ptr_t<char>)xs + id2);
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
        const lds_ptr_t<uint32_t> wzero = wzero2 + (j & 1u) * (uint32_t)NW;
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
// a wave holds the entries from slot s0 of 64 on in ev, SL slots, and writes
// them to their places in ent.  A slot's ranks come from match8 and the wave's
// running digit counts; one wave then turns the counts of all waves into
// bases.  Every wave holds its entries before the first barrier, so ent may be
// where they were read from.
template <int NT, int EH>
__device__ __forceinline__ void sort_pass(const uint32_t (&ev)[EH], uint32_t s0, uint32_t SL, uint32_t R,
                                          uint32_t sh, lds_ptr_t<uint32_t> ent,
                                          lds_ptr_t<uint16_t> hist, lds_ptr_t<uint16_t> base) {
    constexpr int NW = NT / 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = lane_id();
    const lds_ptr_t<uint16_t> hw = hist + 256 * wave;
    // the conditions of the slots are worked out anew in each loop over them:
    // kept, they would fill the scalar registers
    uint32_t sl = opaque_s(SL), i0 = s0 * 64 + opaque(ln);
    uint32_t rk[EH];
    begin_life(rk);
    ((lds_ptr_t<uint32_t>)hw)[ln] = 0;
    ((lds_ptr_t<uint32_t>)hw)[64 + ln] = 0;
    wave_order();
    static_for<0, EH>([&](auto si) {
        constexpr int s = decltype(si)::value;
        if ((uint32_t)s < sl) {
            const bool valid = i0 + 64 * s < R;
            const uint64_t m = match8(ev[s], sh, __ballot(valid));
            const lds_ptr_t<uint16_t> h = hw + ((ev[s] >> sh) & 255u);
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
            const lds_ptr_t<u32x2> h = (lds_ptr_t<u32x2>)(hist + 256 * w + 4 * ln);
            const u32x2 v = *h;
            *h = u32x2{a0, a1};
            a0 += v[0];
            a1 += v[1];
        }
        const uint32_t t0 = a0 & 0xFFFFu, t1 = a0 >> 16, t2 = a1 & 0xFFFFu, t3 = a1 >> 16;
        const uint32_t ex = lane_scan_excl<64>(t0 + t1 + t2 + t3);
        *(lds_ptr_t<u32x2>)(base + 4 * ln) =
            u32x2{ex | ((ex + t0) << 16), (ex + t0 + t1) | ((ex + t0 + t1 + t2) << 16)};
    }
    __syncthreads();
    sl = opaque_s(SL);
    i0 = s0 * 64 + opaque(ln);
    static_for<0, EH>([&](auto si) {
        constexpr int s = decltype(si)::value;
        if ((uint32_t)s < sl) {
            const uint32_t d = (ev[s] >> sh) & 255u;
            if (i0 + 64 * s < R) ent[(uint32_t)base[d] + hw[d] + rk[s]] = ev[s];
        }
    });
    __syncthreads();
}

// One item of the chain: (target, direction) over the 16-row blocks
// [it.q0, it.q1), by it.kind:
//   CHAIN_ROWS     from the order at the segment's start; the run lists are left
//                  for k_rows, other blocks' rows written
//   CHAIN_STARTS   the same chain, but only the order (doubled indexes) at the
//                  start of every block is left, in starts
//   CHAIN_RANK     from the panel order (CHAIN_RANK_UP) or its reverse
//                  (CHAIN_RANK_DOWN); at the end every haplotype's position
//   CHAIN_COMBINE  q counts segments: keys are the sums of a segment's two
//                  positions; leaves the order at the start of every segment
// ROWS: the kernel of CHAIN_ROWS items; the other kinds share one.
//
// Segments cut a chain's latency: haplotypes that no row of a segment tells
// apart keep their order, the others are sorted, so a segment acts on any
// order as a stable sort by rank.  A class of k haplotypes at positions r ..
// r + k - 1 comes out of the panel order and of its reverse in opposite
// orders, so the sum of a haplotype's two positions is 2 r + k - 1 for the
// whole class, and grows from class to class: that is the rank.
//
// E positions per thread: thread x holds positions [x E, x E + E).  LDS: ord
// (doubled haplotype index per position), xs (the block's keys by haplotype),
// st (first position of each run, then the run's displacement).  The run
// entries being sorted (key << 16 | run) take xs's place once they are built;
// when they are sorted and read, xs takes the next block's keys.
// rcap: most runs k_rows takes.
// A call of its own for each E: the registers of one shape are not mixed with
// another's (inlined into one kernel, spills of the most used shape cost 45%).
template <int NT, int E, bool ROWS>
__device__ __attribute__((noinline)) void order_chain(const TgtDev *tgt, OrderItem it,
                                                      uint32_t rcap, uint16_t *starts) {
    tgt = uniform(tgt);
    TgtConst &T = *cmem(tgt);
    it = OrderItem{0, uniform(it.dir), uniform(it.kind), uniform(it.seg), uniform(it.q0), uniform(it.q1)};
    const lds_ptr_t<uint32_t> smem = lds_at(0);
    rcap = uniform(rcap);
    starts = uniform(starts);
    constexpr int NW = NT / 64, EH = E / 2;
    constexpr uint32_t NPOS = (uint32_t)(NT * E);
    static_assert(E % 2 == 0 && E <= 32, "positions go in pairs, their flags into one register");
    const lds_ptr_t<uint16_t> ord = (lds_ptr_t<uint16_t>)smem;
    const lds_ptr_t<uint32_t> ord32 = smem;
    const lds_ptr_t<uint16_t> xs = ord + NPOS;
    const lds_ptr_t<uint32_t> xs32 = (lds_ptr_t<uint32_t>)xs;
    const lds_ptr_t<uint16_t> st = xs + NPOS;
    const lds_ptr_t<uint16_t> hist = st + order_starts(NT, E);
    const lds_ptr_t<uint16_t> base = hist + 256 * NW;
    const lds_ptr_t<uint32_t> red = (lds_ptr_t<uint32_t>)(base + 256);
    const lds_ptr_t<uint32_t> ent = xs32;
    const uint32_t tid = threadIdx.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), ln = lane_id();
    const uint32_t K = T.K, Mp = T.Mp, Kpad = T.Kpad, RS = T.RS;
    const uint32_t nblk = (Mp + 15) / 16, q1 = it.q1;
    const bool rev = it.dir != 0;
    const bool combine = !ROWS && it.kind == CHAIN_COMBINE;
    const bool rank = !ROWS && (it.kind == CHAIN_RANK_UP || it.kind == CHAIN_RANK_DOWN);
    // this chain's segments: {positions up, positions down, order at the start}
    const gptr_t<uint16_t> seg = gmem(T.seg) + (uint64_t)(rev ? T.nseg : 0u) * 3 * Kpad;
    const uint32_t rmax = min(rcap, Kpad / 2);
    const gptr_t<const uint16_t> cref = gmem((const uint16_t *)T.cref);
    const gptr_t<uint16_t> hdr = gmem(T.hdr) + (rev ? nblk : 0u);
    uint32_t pf[EH];  // the next block's keys, loaded one block ahead
    auto fetch = [&](uint32_t q) {
        const BlockGeo g = block_geo(q, Mp, nblk, rev);
        gptr_t<const uint32_t> src = (gptr_t<const uint32_t>)(cref + (uint64_t)g.b * Kpad);
        if (combine) src = (gptr_t<const uint32_t>)(seg + (uint64_t)q * 3 * Kpad);
#pragma unroll
        for (int i = 0; i < EH; i++) {
            const uint32_t w = min(opaque(tid) + (uint32_t)i * NT, Kpad / 2 - 1);
            pf[i] = src[w];
            if (combine) pf[i] += src[Kpad / 2 + w];  // below 65536 each
        }
    };
    // a segment's ranks have the bits of 2 K - 2
    auto geo_of = [&](uint32_t q) {
        BlockGeo g = block_geo(q, Mp, nblk, rev);
        if (combine) g.nrows = K > 1 ? 32u - (uint32_t)__clz(2 * K - 2) : 1u;
        return g;
    };
    // xs = keys of block q, then the block after it is fetched
    auto stage = [&](uint32_t q) {
        const BlockGeo g = geo_of(q);
#pragma unroll
        for (int i = 0; i < EH; i++) {
            const uint32_t w = opaque(tid) + (uint32_t)i * NT;
            xs32[w] = w < Kpad / 2 ? key_pair(pf[i], rev && !combine, g.nrows) : ~0u;
        }
        if (q + 1 < q1) fetch(q + 1);
    };
    // the order at the start; positions past Kpad hold index Kpad, whose key is
    // all ones (they never move)
    {
        const bool given = it.seg != 0 && !rank && !combine;
        const gptr_t<const uint32_t> so = (gptr_t<const uint32_t>)(seg + (uint64_t)(3 * it.seg + 2) * Kpad);
#pragma unroll
        for (int i = 0; i < EH; i++) {
            const uint32_t w = tid + (uint32_t)i * NT;
            uint32_t a = min(2 * w, Kpad), b = min(2 * w + 1, Kpad);
            if (!ROWS && it.kind == CHAIN_RANK_DOWN) {
                if (a < K) a = K - 1 - a;
                if (b < K) b = K - 1 - b;
            }
            uint32_t v = 2 * a | (2 * b << 16);
            if (given && w < Kpad / 2) v = so[w];
            ord32[w] = v;
        }
    }
    fetch(it.q0);
    stage(it.q0);
    __syncthreads();
    auto key_at = [&](uint32_t id2) { return (uint32_t)*(lds_ptr_t<uint16_t>)((lds_ptr_t<char>)xs + id2); };
    for (uint32_t q = it.q0; q < q1; q++) {
        const BlockGeo geo = geo_of(q);
        const uint32_t tq = opaque(tid), pos0 = tq * E;
        // keys of my positions and where a run of equal keys begins: flag of
        // position pos0 + e at bit e/2 (e even) or 16 + e/2 (e odd)
        uint32_t idp[EH];
#pragma unroll
        for (int i = 0; i < EH; i++) idp[i] = ord32[tq * EH + i];
        if constexpr (!ROWS) {
            if (it.kind == CHAIN_STARTS || (combine && q)) {
                const gptr_t<uint32_t> so =
                    combine ? (gptr_t<uint32_t>)(seg + (uint64_t)(3 * q + 2) * Kpad)
                            : (gptr_t<uint32_t>)(gmem(starts) + (uint64_t)q * Kpad);
#pragma unroll
                for (int i = 0; i < EH; i++)
                    if (pos0 + 2 * i < Kpad) so[tq * EH + i] = idp[i];
            }
            if (combine && q + 1 == q1) break;  // the last segment needs its start only
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
                lds_ptr_t<uint16_t> w = st + rbase;
                static_for<0, E>([&](auto ei) {
                    if (flag(ei)) *w++ = (uint16_t)(pos0 + decltype(ei)::value);
                });
                if (tid == 0) st[R] = (uint16_t)Kpad;
            }
            __syncthreads();
            // the runs' entries, and the run list for k_rows in the block's rows
            // slots of 64 entries, spread evenly over the waves (at most EH each)
            const uint32_t nslot = (R + 63) / 64;
            const uint32_t s0 = wave * nslot / NW, SL = (wave + 1) * nslot / NW - s0;
            {
                uint32_t ev[EH];
                begin_life(ev);
                const gptr_t<uint32_t> list =
                    gmem(T.out) + ((rev ? (uint64_t)Mp : 0ull) + geo.s0) * RS;
                const uint32_t sl = opaque_s(SL), i0 = s0 * 64 + opaque(ln);
                static_for<0, EH>([&](auto si) {
                    constexpr int s = decltype(si)::value;
                    if ((uint32_t)s < sl) {
                        const uint32_t i = i0 + 64 * s;
                        const uint32_t a = st[min(i, R - 1)];
                        const uint32_t k = key_at(ord[a]) << 16;
                        ev[s] = k | i;
                        if (ROWS && i < R) list[i] = k | a;
                    }
                });
                if (ROWS && tid == 0) hdr[q] = (uint16_t)R;
                sort_pass<NT, EH>(ev, s0, SL, R, 16, ent, hist, base);
            }
            {
                uint32_t ev[EH];
                begin_life(ev);
                const uint32_t sl = opaque_s(SL), i0 = s0 * 64 + opaque(ln);
                static_for<0, EH>([&](auto si) {
                    constexpr int s = decltype(si)::value;
                    if ((uint32_t)s < sl) ev[s] = ent[min(i0 + 64 * s, R - 1)];
                });
                sort_pass<NT, EH>(ev, s0, SL, R, 24, ent, hist, base);
            }
            // new start of every run: prefix sum of the lengths in key order,
            // per consecutive sorted runs per thread
            const uint32_t per = (R + NT - 1) / NT;
            uint32_t ra[EH], rl[EH];
            begin_life(ra);
            begin_life(rl);
            uint32_t sum = 0;
            // (waves past the last run skip)
            const uint32_t mine = wave * 64 * per < R ? per : 0u;
            uint32_t sl = opaque_s(mine), i0 = opaque(tid) * per;
            static_for<0, EH>([&](auto si) {
                constexpr int s = decltype(si)::value;
                if ((uint32_t)s < sl) {
                    const uint32_t i = i0 + s;
                    const uint32_t run = ent[min(i, R - 1)] & 0xFFFFu;
                    const uint32_t a = st[run], b = st[run + 1];
                    ra[s] = (run << 16) | a;
                    rl[s] = i < R ? b - a : 0u;
                    sum += rl[s];
                }
            });
            uint32_t tot;
            uint32_t at = wg_scan_excl<NT>(sum, red + NW, tot);
            sl = opaque_s(mine);
            i0 = opaque(tid) * per;
            static_for<0, EH>([&](auto si) {
                constexpr int s = decltype(si)::value;
                if ((uint32_t)s < sl) {
                    if (i0 + s < R) st[ra[s] >> 16] = (uint16_t)(at - (ra[s] & 0xFFFFu));
                    at += rl[s];
                }
            });
            if (tid == 0) st[R] = 0;
            // my haplotypes again (not kept through the sort: registers), and
            // the next block's keys
            uint32_t id[EH];
#pragma unroll
            for (int i = 0; i < EH; i++) id[i] = ord32[tq * EH + i];
            if (q + 1 < q1) stage(q + 1);
            __syncthreads();
            // every haplotype moves with its run (displacements are signed 16-
            // bit: Kpad < 32768)
            lds_ptr_t<int16_t> d = (lds_ptr_t<int16_t>)st + (int32_t)rbase - 1;
            const lds_ptr_t<uint16_t> me = ord + pos0;
            static_for<0, E>([&](auto ei) {
                constexpr int e = decltype(ei)::value;
                d += flag(ei);
                me[(int32_t)*d + e] = (uint16_t)((e & 1) ? id[e / 2] >> 16 : id[e / 2]);
                // few lookups in flight at a time: registers, and other
                // workgroups' waves fill the gaps
                if constexpr (e % 8 == 7) __builtin_amdgcn_sched_barrier(0);
            });
        } else {
            order_dense<NT, E>(tgt, rev, geo, ROWS, nullptr);
            if (ROWS && tid == 0) hdr[q] = (uint16_t)kDense;
            if (q + 1 < q1) {
                fetch(q + 1);  // again: registers are not kept across the call
                stage(q + 1);
            }
        }
        __syncthreads();
    }
    if (rank) {
        // positions by haplotype, through xs; the padding gets all ones in sum
#pragma unroll
        for (int i = 0; i < EH; i++) {
            const uint32_t p = tid * E + 2 * i, v = ord32[tid * EH + i];
            if (p < Kpad) {
                *(lds_ptr_t<uint16_t>)((lds_ptr_t<char>)xs + (v & 0xFFFFu)) = (uint16_t)p;
                *(lds_ptr_t<uint16_t>)((lds_ptr_t<char>)xs + (v >> 16)) = (uint16_t)(p + 1);
            }
        }
        __syncthreads();
        const bool up = it.kind == CHAIN_RANK_UP;
        const gptr_t<uint32_t> dst =
            (gptr_t<uint32_t>)(seg + (uint64_t)(3 * it.seg + (up ? 0u : 1u)) * Kpad);
        for (uint32_t w = tid; w < Kpad / 2; w += NT) {
            uint32_t v = xs32[w];
            const uint32_t pad = (2 * w >= K ? 0xFFFFu : 0u) | (2 * w + 1 >= K ? 0xFFFF0000u : 0u);
            v = up ? v | pad : v & ~pad;
            dst[w] = v;
        }
    }
}

// Waves per SIMD that one workgroup's LDS allows at the variant's capacity: the
// register budget is capped so that VGPRs do not lower it (512 x 20: three
// workgroups, 80 registers; 8.65 ms for 384 chains of 941 blocks at K = 10,000
// against 9.36 ms with two workgroups and 128 registers).  No fewer than five
// waves, 96 registers: 1024 x 24 and 512 x 32 hold four waves per SIMD, which at
// 128 registers are all there are, and nothing else then runs on a CU until its
// chains end, not even the copies and the selection of another context (380 KB
// copied beside 256 chains of 1,024 threads: up to 30 ms so, 2 ms with 96
// registers; their build takes 66.6 ms either way.  The sizes above 12 positions
// per thread spill a few registers more: two targets at K = 16,000 in 512 x 32
// 3.27 and 3.42 ms, in 1024 x 24, which the automatic choice takes there, 2.66
// and 2.64; one target of 45,000 rows at K = 10,000, 10 positions per thread,
// 2.77 and 2.79).
constexpr int order_waves_hint(int NT, int CPW) {
    const int w = (163840 / (int)order_lds(NT, CPW)) * (NT / 256);
    return w < 5 ? 5 : (w > 6 ? 6 : w);
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
void k_order(const TgtDev *__restrict__ tg, const OrderItem *__restrict__ items,
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
        const OrderItem it = items[i];
        const TgtDev &T = tg[it.t];
        const int ns = pbwt_slots_for(T.Kpad, NT);
        static_for<0, kNumSlotCounts>([&](auto ii) {
            constexpr int NSv = kSlotCounts[decltype(ii)::value];
            if constexpr (NSv <= CPW) {
                if (ns == NSv)
                    order_chain<NT, NSv, ROWS>(&T, it, rcap, starts);
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
    uint32_t *ord = smem, *xs = smem + NPOS / 2;
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
    order_dense<NT, E>(&T, 0, geo, 1, absperm);
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

// Variants of the chain kernel: (threads, most positions per thread).
struct PbwtVariant {
    int nt, cpw;
    // CHAIN_ROWS items; items of the other kinds; rows with the order after each
    void (*rows)(const TgtDev *, const OrderItem *, const uint32_t *, uint32_t *, uint32_t, uint16_t *);
    void (*aux)(const TgtDev *, const OrderItem *, const uint32_t *, uint32_t *, uint32_t, uint16_t *);
    void (*dense)(const TgtDev *, const uint16_t *, int32_t *);
};
template <int NT, int CPW>
PbwtVariant make_variant() {
    return {NT, CPW, k_order<NT, CPW, true>, k_order<NT, CPW, false>, k_dense<NT, CPW>};
}
PbwtVariant variant_256x8();
PbwtVariant variant_256x16();
PbwtVariant variant_512x20();
PbwtVariant variant_512x32();
PbwtVariant variant_1024x24();

}  // namespace eimp
