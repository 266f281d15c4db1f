// kv_prefill.hip -- causal prefill flash attention on f16 MFMA, split-K over positions.
//
// Replaces q_f16 + attn_fa_mx + attn_fd_combine of the reference's prefill (fa_mx.wgsl:19-115, 313-319;
// engine.rs:1215-1236). Token t of the block (0-based) sees positions [start, n + t).
//
// Work-group = (32 or 16 tokens of the block, key split, kv head): 8 waves (two per SIMD, so one wave's softmax overlaps
// the other's matrix work), each owns 4 tokens x the kv head's 8 query heads = 32 query rows (row = token*8 + head) and,
// with two key groups (PfGeom), every other tile. The split's 32-key tiles (a 16 KB K block and four 4 KB V groups,
// contiguous in HBM) stream through an LDS ring filled by direct global->LDS loads, shared by the waves. Per tile and wave:
//   S^T[32 keys][32 rows] = K . Q^T    16 x v_mfma_f32_32x32x16_f16 (A = K rows in key_perm order from LDS,
//                                      B = Q rounded to f16, held in registers for the whole split)
//   online softmax of the 32 rows in registers, lazy reference max (moves when first or when the tile max exceeds
//   it by more than 8), row sums from the f32 P (as attn_fa_mx), P rounded to f16 for the matrix units
//   O[32 rows][256] += P . V           16 x v_mfma_f32_32x32x16_f16 (A = P straight from the S registers,
//                                      B = V from LDS)
// One partial [m, l, acc[256]] per row; launch_merge combines the splits (and applies the gate).
#include <climits>
#include <type_traits>

#include "mkv_device.h"

namespace mkv {
namespace {

constexpr int NW = 8;                         // waves per work-group
constexpr int TILE_BYTES = 32 * HD * 2;       // one 32-key K block (or its 4 V groups), f16
constexpr int RING_BYTES = 8 * TILE_BYTES;    // LDS ring

// KS: key groups of a work-group. KS = 1: its 8 waves hold 32 tokens and take every tile. KS = 2: waves 0-3 hold 16 tokens
// and take the even tiles, waves 4-7 the same tokens and the odd tiles, and the two states of a row meet in LDS at the
// end: half the split partials (and half of Q's reads) for the same work-groups, twice the tiles read from L2.
template <int KS>
struct PfGeom {
    static constexpr int RW = NW / KS;                  // waves over the rows
    static constexpr int PT = 4 * RW;                   // tokens per work-group
    static constexpr int STEP_BYTES = 2 * KS * TILE_BYTES;  // K and V of a step's KS tiles
    static constexpr int NSLOT = RING_BYTES / STEP_BYTES;   // ring slots: NSLOT - 1 steps in flight while one is computed
    static constexpr int PART_BYTES = TILE_BYTES / RW;  // of its key group's K block (or V groups) a wave copies
    static constexpr int LPT = 2 * PART_BYTES / 1024;   // direct loads per step and wave
};

template <int KS>
__device__ inline void wait_steps(int later) {  // at most `later` steps (LPT direct loads each per wave) pending
    if constexpr (KS == 2) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else {
        static_assert(PfGeom<1>::LPT == 4 && PfGeom<1>::NSLOT == 4, "wait counts");
        if (later >= 2) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        else if (later == 1) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
}

template <int KS>
__global__ void __launch_bounds__(NW * 64) prefill_f16(const _Float16* __restrict__ kplane,
                                                   const _Float16* __restrict__ vplane, size_t plane_elems,
                                                   const float* __restrict__ q, int T, int n, int start, float scale2,
                                                   int span, int nch, float* __restrict__ part) {
    // XCD-aware order with the token blocks of one (split, kv head) -- the work-groups that stream the same keys --
    // neighbours: each key is fetched into one L2 instead of eight. For every grid: 200 tokens at 9,000 positions (252
    // work-groups) took 66.2 us while only multiples of 8 were ordered, 62.7 since (one key group both times).
    const int G = gridDim.x, L = blockIdx.x;
    const int W = xcd_order(L, G);
    using Gm = PfGeom<KS>;
    constexpr int PT = Gm::PT, PART_BYTES = Gm::PART_BYTES, NSLOT = Gm::NSLOT;
    const int nblk = (T + PT - 1) / PT;
    const int rb = W % nblk, sp = (W / nblk) % nch, kvh = W / nblk / nch, tid = threadIdx.x;
    const int lane = tid & 63, w = tid >> 6;
    const int wr = w % Gm::RW, kg = __builtin_amdgcn_readfirstlane(w / Gm::RW);  // row wave, key group
    const int h = lane >> 5, r = lane & 31;
    const int t0 = rb * PT + 4 * wr;         // this wave's first token
    const int tlast = min(T - 1, rb * PT + PT - 1);
    const int kend = n + T - 1;              // positions written for this block
    const int cs = chunk_lo(sp, span, nch), ce = min(sp + 1 < nch ? chunk_lo(sp + 1, span, nch) : span, n + tlast);
    if (cs >= ce) return;                    // no key of this split is seen by these tokens: never merged
    const _Float16* K = kplane + (size_t)kvh * plane_elems;
    const _Float16* V = vplane + (size_t)kvh * plane_elems;

    __shared__ __attribute__((aligned(16))) unsigned char ring[RING_BYTES];
    __shared__ __attribute__((aligned(16))) float cfs[NW][32];  // rescale factors of a wave's rows
    const int ntiles = (ce - cs + 31) / 32, nsteps = (ntiles + KS - 1) / KS;
    // step j is tiles KS j .. KS j + KS - 1; this wave copies a part of tile KS j + kg, the one it computes: a per-lane
    // offset fixed for the kernel; the tile's base and LDS slot are wave-uniform
    const unsigned voff = wr * PART_BYTES + lane * 16;
    const unsigned wlds = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(lds_void*)ring + kg * 2 * TILE_BYTES + wr * PART_BYTES);
    auto kof = [&](int j) { return (j % NSLOT) * Gm::STEP_BYTES + kg * 2 * TILE_BYTES; };  // this key group's K of step j
    // V rows past the written length may hold anything: each wave zeroes them in the part of the tile it copied itself,
    // after its own copies have landed and before the barrier that hands the tile to every wave (no barrier of its own)
    auto zero_own_tail = [&](int j) {
        const int k0 = cs + 32 * (KS * j + kg);
        if (k0 + 32 <= kend) return;
        unsigned char* Vw = ring + kof(j) + TILE_BYTES;
#pragma unroll
        for (int i = 0; i < PART_BYTES / 1024; i++) {
            const unsigned off = voff + i * 1024;  // 8 consecutive positions of one dim: group off / 4096
            const int key = k0 + (int)(off / 4096) * 8;
            if (key + 8 > kend) {
                half8 x = *(const half8*)(Vw + off);
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (key + e >= kend) x[e] = (_Float16)0.f;
                *(half8*)(Vw + off) = x;
            }
        }
    };
    auto issue = [&](int j) {  // this wave's part of its tile's K block and V groups into slot j % NSLOT
        const int k0 = cs + 32 * (KS * j + kg);
        if (KS > 1 && KS * j + kg >= ntiles) return;
        const unsigned char* ks = (const unsigned char*)(K + (size_t)(k0 / KBLK) * (KBLK * HD));
        const unsigned char* vs = (const unsigned char*)(V + (size_t)(k0 / VGRP) * (VGRP * HD));
        const unsigned dst = wlds + (j % NSLOT) * Gm::STEP_BYTES;
#pragma unroll
        for (int i = 0; i < PART_BYTES / 1024; i++) dma16s(ks + i * 1024, voff, dst + i * 1024);
#pragma unroll
        for (int i = 0; i < PART_BYTES / 1024; i++) dma16s(vs + i * 1024, voff, dst + TILE_BYTES + i * 1024);
    };
    for (int j = 0; j < NSLOT - 1 && j < nsteps; j++) issue(j);

    // Q as the B operand of S^T: lane (r, h) holds row r (token t0 + r/8, head r%8), dims 16s + 8h .. +7 for step s, rounded
    // to f16 (q_f16); rows of tokens past the block are zero
    half8 qb[16];
    const int tr = t0 + (r >> 3);
    const int vis = tr < T ? n + tr : 0;  // row r sees keys [start, vis)
    // key - start < seen, unsigned: both bounds in one comparison. With two the compiler chained each pair through vcc (16
    // round trips to the scalar unit per masked tile): 448 tokens at 60,000 positions, half of them below start, 440 us
    // against 407 without the chain, now 0.98 of that; 300 tokens there (waves without tokens mask every tile) 328 / 315
    const unsigned seen = max(vis - start, 0);
    // through the ring's last slot, which no load fills before the first tile's barrier
    stage_q16(q + (size_t)kvh * GQA * HD, QH * HD, HD, T, t0, lane, ring + (NSLOT - 1) * Gm::STEP_BYTES + w * 4096, qb);
    __builtin_amdgcn_sched_barrier(0);  // the loads' registers are free before O takes its own
    const int kaddr = h * 512 + key_perm(r) * 16;
    // the smallest window end of the wave's rows (its first token's; 0 when they run past T): a tile with every key below
    // it, and none below start, needs no mask (a wave-uniform test)
    const int tf = __builtin_amdgcn_readfirstlane(t0), vmin = tf + 3 < T ? n + tf : 0;
    float m = NEG_INF, lsum = 0.f;
    f32x16 O[8];
#pragma unroll
    for (int nb = 0; nb < 8; nb++) O[nb] = f32x16{};
    // O's rows times the factor of each, which lane (row) holds: register i of O holds row 8(i/4) + 4h + i%4, so the 32
    // factors pass through this wave's LDS row (constant offsets, no per-register lane index to keep)
    auto scale_rows = [&](float cf) {
        if (h == 0) cfs[w][r] = cf;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const f32x4 f = *(const f32x4*)&cfs[w][8 * a + 4 * h];
#pragma unroll
            for (int nb = 0; nb < 8; nb++) {
#pragma unroll
                for (int q = 0; q < 4; q++) O[nb][4 * a + q] *= f[q];
            }
        }
    };

    // S of this wave's tile of step j, the mask where it crosses a row's window, the online softmax (lazy reference max, O
    // rescaled when a finite reference moved) and P into pa
    auto s_mfma = [&](int j, f32x16& S) {
        const unsigned char* Ks = ring + kof(j);
        S = f32x16{};
        constexpr int KP = 3;  // K operands in flight ahead of the S chain (LDS latency; 4 to 6 measured no faster)
        half8 kbuf[KP];
#pragma unroll
        for (int s = 0; s < KP; s++) kbuf[s] = *(const half8*)(Ks + kaddr + s * 1024);
#pragma unroll
        for (int s = 0; s < 16; s++) {
            const half8 ka = kbuf[s % KP];
            if (s + KP < 16) kbuf[s % KP] = *(const half8*)(Ks + kaddr + (s + KP) * 1024);
            S = mfma32(ka, qb[s], S);
        }
        // schedule: KP LDS reads (mask 0x100), then alternately one MFMA (0x008) and the next LDS read
        __builtin_amdgcn_sched_group_barrier(0x100, KP, 0);
#pragma unroll
        for (int s = 0; s < 16 - KP; s++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, KP, 0);
    };
    auto softmax = [&](int j, f32x16& S, half8(&pa)[2]) {
        const int k0 = cs + 32 * (KS * j + kg);
        // the causal / start mask only where this tile crosses a row's window (raw scores; the scale, log2 units, is
        // applied to the max and inside the exponent's FMA)
        if (!(k0 >= start && k0 + 32 <= vmin)) {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int key = k0 + 8 * h + i + (i >= 8 ? 8 : 0);
                S[i] = (unsigned)(key - start) < seen ? S[i] : NEG_INF;
            }
        }
        // the first maximum is the compiler's: it reads the MFMA results and so carries the wait states a vector read of
        // them needs, which inline assembly would not get; the rest follows it
        float mt = fmaxf(S[0], S[1]);
#pragma unroll
        for (int i = 2; i < 16; i += 2) mt = vmax3(mt, S[i], S[i + 1]);
        mt = max_xor32(mt);
        mt *= scale2;  // scale2 > 0: the max of the scaled scores is the scaled max
        // the reference max moves when first or when the tile max exceeds it by more than 8; O and the sum are rescaled
        // only when a finite reference moved (rare: the exponential is not evaluated otherwise)
        const bool rescale = m != NEG_INF && mt > m + LAZY2;
        const float mr = m == NEG_INF || rescale ? fmaxf(m, mt) : m;
        float cf = 1.f;
        if (__any(rescale)) {
            cf = rescale ? fast_exp2(m - mr) : 1.f;
            scale_rows(cf);
        }
        m = mr;
        // P = 2^(s * scale2 - m) (one FMA): masked scores are -inf and give 0 (the reference is 0 while a row has seen no
        // key); the row sum takes the f32 P, as attn_fa_mx does, the P.V operand its f16 rounding
        const float base = mr == NEG_INF ? 0.f : mr;
        float ls;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const float p = fast_exp2(__builtin_fmaf(S[i], scale2, -base));
            ls = i == 0 ? p : ls + p;  // 0 + p0 is p0: the same sum without the first add
            pa[i >> 3][i & 7] = (_Float16)p;
        }
        lsum = lsum * cf + ls;
    };
    // O += P . V of this wave's tile of step j
    auto pv_tile = [&](int j, const half8(&pa)[2]) {
        const unsigned char* Vs = ring + kof(j) + TILE_BYTES;
        constexpr int VP = 3;  // V operands in flight ahead of the P.V MFMAs
        half8 vbuf[VP];
        auto vaddr = [&](int i) { return Vs + (2 * (i >> 3) + h) * 4096 + (32 * (i & 7) + r) * 16; };
#pragma unroll
        for (int i = 0; i < VP; i++) vbuf[i] = *(const half8*)vaddr(i);
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const half8 vb = vbuf[i % VP];
            if (i + VP < 16) vbuf[i % VP] = *(const half8*)vaddr(i + VP);
            O[i & 7] = mfma32(pa[i >> 3], vb, O[i & 7]);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, VP, 0);
#pragma unroll
        for (int i = 0; i < 16 - VP; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, VP, 0);
    };
    for (int j = 0; j < nsteps; j++) {
        wait_steps<KS>(min(nsteps - 1 - j, NSLOT - 2));
        zero_own_tail(j);
        lds_barrier();  // step j is in LDS for every wave; every wave is done with step j - 1
        if (j + NSLOT - 1 < nsteps) issue(j + NSLOT - 1);  // into the slot of step j - 1
        if (KS > 1 && KS * j + kg >= ntiles) break;        // no odd tile in the last step
        f32x16 S;
        half8 pa[2];
        s_mfma(j, S);
        softmax(j, S, pa);
        pv_tile(j, pa);
    }
    lsum += __shfl_xor(lsum, 32);

    // partials of this wave's rows of present tokens: row index t*8 + head of the kv head, rows per kv head = 8T
    const size_t rpk = (size_t)T * GQA;
    auto row_part = [&](int ri) { return part + ((kvh * rpk + (size_t)t0 * GQA + ri) * nch + sp) * PART; };
    auto store_o = [&](auto nb0, auto cnt) {  // dim blocks nb0 .. nb0 + cnt - 1 of O
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int ri = 8 * (i >> 2) + 4 * h + (i & 3);
            if (t0 + (ri >> 3) < T) {
                float* p = row_part(ri) + PACC + r;
#pragma unroll
                for (int nb = 0; nb < cnt; nb++) p[32 * (nb0 + nb)] = O[nb0 + nb][i];
            }
        }
    };
    using std::integral_constant;
    if constexpr (KS == 1) {
        store_o(integral_constant<int, 0>{}, integral_constant<int, 8>{});
    } else {
        // the row's two states, waves w and w ^ 4: both scaled to the common maximum, each wave then takes over half of the
        // dims (its partner's half of them through the ring, which no wave reads any more behind the first barrier)
        __shared__ __attribute__((aligned(16))) float ml[NW][2][32];
        if (h == 0) {
            ml[w][0][r] = m;
            ml[w][1][r] = lsum;
        }
        __syncthreads();
        const float mo = ml[w ^ Gm::RW][0][r], lo = ml[w ^ Gm::RW][1][r];
        const float M = fmaxf(m, mo);
        const float f = m == NEG_INF ? 0.f : fast_exp2(m - M), fo = mo == NEG_INF ? 0.f : fast_exp2(mo - M);
        scale_rows(f);
        f32x4* const mine = (f32x4*)ring + w * 1024 + lane;
        const f32x4* const other = (const f32x4*)ring + (w ^ Gm::RW) * 1024 + lane;
        auto give = [&](auto nb0) {
#pragma unroll
            for (int nb = 0; nb < 4; nb++)
#pragma unroll
                for (int a = 0; a < 4; a++)
                    mine[(nb * 4 + a) * 64] = f32x4{O[nb0 + nb][4 * a], O[nb0 + nb][4 * a + 1], O[nb0 + nb][4 * a + 2],
                                                    O[nb0 + nb][4 * a + 3]};
        };
        auto take = [&](auto nb0) {
#pragma unroll
            for (int nb = 0; nb < 4; nb++)
#pragma unroll
                for (int a = 0; a < 4; a++) {
                    const f32x4 x = other[(nb * 4 + a) * 64];
#pragma unroll
                    for (int e = 0; e < 4; e++) O[nb0 + nb][4 * a + e] += x[e];
                }
            store_o(nb0, integral_constant<int, 4>{});
        };
        const integral_constant<int, 0> low{};
        const integral_constant<int, 4> high{};
        if (kg == 0) give(high);
        else give(low);
        __syncthreads();
        if (kg == 0) take(low);
        else take(high);
        m = M;
        lsum = lsum * f + lo * fo;
    }
    if (kg == 0 && h == 0 && t0 + (r >> 3) < T) {
        float* p = row_part(r);
        p[0] = m;
        p[1] = lsum;
    }
}


// ---- f32 store: causal prefill with f32-class arithmetic (attn_fa, ops.wgsl:540-651) ----
// Work-group = (16 tokens of the block, key split, kv head), 8 waves: wave w takes row block w / 2 (4 tokens x 8
// heads = 32 rows) and dim half w % 2 (128 dims). The split's 32-key tiles (32 KB of K, 32 KB of V) stream through a
// 2-slot LDS ring filled by direct global->LDS loads and shared by the 8 waves, so a key is fetched once per 16
// tokens. f32 operands are split into f16 hi + lo (hi.hi + hi.lo + lo.hi on v_mfma_f32_32x32x16_f16). Per tile and
// wave:
//   partial S^T[32 keys][32 rows] over the wave's 128 dims: 8 dim steps x 3 passes (A = K rows in key_perm order,
//   the tile's K and V split into hi + lo once, in place in the ring, by the whole work-group; B = Q split once, in
//   registers); the two halves are exchanged through LDS and added
//   (a + b in both waves, so both hold the same S)
//   online softmax with a lazy reference max, redundantly in both waves of the pair
//   O[32 rows][the wave's 128 dims] += P . V: 2 key steps x 4 dim blocks x 3 passes
// Registers hold Q's hi and lo for 128 dims and O for 128 dims; LDS is 128 KB of ring and 32 KB of S exchange.
constexpr int P32_NW = 8;
constexpr int P32_PT = 16;                    // tokens per work-group
constexpr int P32_TILE = 32 * HD * 4;         // f32 K (or V) bytes of 32 positions: 32 KB
constexpr int P32_SLOT = 2 * P32_TILE;
constexpr int P32_LPT = P32_SLOT / P32_NW / 1024;  // direct loads per wave and slot: 8

__global__ void __launch_bounds__(P32_NW * 64) prefill_f32(const float* __restrict__ kplane,
                                                          const float* __restrict__ vplane, size_t plane_elems,
                                                          const float* __restrict__ q, int T, int n, int start,
                                                          float scale2, int span, int nch, float* __restrict__ part) {
    const int G = gridDim.x, Lb = blockIdx.x;
    const int W = xcd_order(Lb, G);
    const int nblk = (T + P32_PT - 1) / P32_PT;
    const int rb = W % nblk, sp = (W / nblk) % nch, kvh = W / nblk / nch, tid = threadIdx.x;
    const int lane = tid & 63, w = tid >> 6, h = lane >> 5, r = lane & 31, blk = w >> 1, dh = w & 1;
    const int t0 = rb * P32_PT + 4 * blk;  // this wave's first token
    const int tlast = min(T - 1, rb * P32_PT + P32_PT - 1);
    const int kend = n + T - 1;            // positions written for this block
    const int cs = chunk_lo(sp, span, nch), ce = min(sp + 1 < nch ? chunk_lo(sp + 1, span, nch) : span, n + tlast);
    const int ntiles = ce > cs ? (ce - cs + 31) / 32 : 0;
    const unsigned char* K = (const unsigned char*)(kplane + (size_t)kvh * plane_elems);
    const unsigned char* V = (const unsigned char*)(vplane + (size_t)kvh * plane_elems);

    __shared__ __attribute__((aligned(16))) unsigned char ring[2 * P32_SLOT];
    __shared__ __attribute__((aligned(16))) f32x4 xs[P32_NW][4][64];  // each wave's partial S^T
    // Each wave copies 1/8 of tile j's K and V into slot j % 2, chosen so that the 16-byte chunk pairs it later splits
    // (below) are all its own: K bytes [4 KB w, +4 KB) (chunks d/4 = 8w .. 8w + 7 of every key), V dims
    // [128 (w % 2), +128) of groups 2 (w / 2) and 2 (w / 2) + 1 (2 KB each).
    const unsigned kreg = w * (P32_TILE / P32_NW);
    const unsigned vreg0 = (2 * (w >> 1)) * (HD * 16) + (w & 1) * (HD / 2 * 16), vreg1 = vreg0 + HD * 16;
    static_assert(P32_TILE / P32_NW == 4096 && HD / 2 * 16 == 2048, "4 KB of K and 2 x 2 KB of V per wave");
    // per-lane offsets of the wave's regions, fixed for the kernel; the tile's base and LDS slot are wave-uniform
    const unsigned vk = kreg + lane * 16, v0 = vreg0 + lane * 16, v1 = vreg1 + lane * 16;
    const unsigned lk = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(lds_void*)ring + kreg);
    const unsigned l0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(lds_void*)ring + P32_TILE + vreg0);
    const unsigned l1 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(lds_void*)ring + P32_TILE + vreg1);
    auto issue = [&](int j) {
        const size_t off = (size_t)(cs + 32 * j) * HD * 4;
        const unsigned slot = (j & 1) * P32_SLOT;
#pragma unroll
        for (int d = 0; d < 4; d++) dma16s(K + off + d * 1024, vk, lk + slot + d * 1024);
#pragma unroll
        for (int d = 0; d < 2; d++) {
            dma16s(V + off + d * 1024, v0, l0 + slot + d * 1024);
            dma16s(V + off + d * 1024, v1, l1 + slot + d * 1024);
        }
    };
    if (ntiles > 0) issue(0);

    // Q: lane (r, h) holds row r (token t0 + r / 8, head r % 8), dims 128dh + 16s + 8h .. +7 of step s, split
    const int tr = t0 + (r >> 3);
    const int vis = tr < T ? n + tr : 0;  // row r sees keys [start, vis)
    const unsigned seen = max(vis - start, 0);  // as prefill_f16
    half8 qh[8], ql[8];  // through the ring's second slot, which no load fills before the first tile's barrier
    stage_q32(q + (size_t)kvh * GQA * HD + 128 * dh, QH * HD, HD, T, t0, lane, ring + P32_SLOT + w * 4096, qh, ql);
    const int kaddr = (32 * dh + 2 * h) * 512 + key_perm(r) * 16;  // K chunk (dims / 4) 32dh + 4s + 2h, +1
    float m = NEG_INF, lsum = 0.f;
    f32x16 O[4];
#pragma unroll
    for (int nb = 0; nb < 4; nb++) O[nb] = f32x16{};

    for (int j = 0; j < ntiles; j++) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's copies of tile j have landed
        const int k0 = cs + 32 * j;
        unsigned char* Ks = ring + (j & 1) * P32_SLOT;
        unsigned char* Vs = Ks + P32_TILE;
        // This wave's part of tile j split once, in place, into f16 hi + lo (the 4 row blocks' waves then read split
        // operands instead of each splitting the same tile): a pair of 16-byte chunks holds 8 consecutive dims of one
        // key (K chunks d/4 = 2g, 2g + 1) or 8 consecutive keys of one dim (V groups 2g, 2g + 1); hi goes over the
        // first chunk and lo over the second, where the operand reads below find them. The pairs are the ones this
        // wave copied, so no barrier comes between its copies and its split. V rows past the written length are
        // zeroed on the way (0 * V stays finite).
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int pk = lane + 64 * u;  // K pair pk: chunk 8w + 2 (pk / 32) of key pk % 32
            unsigned char* a = Ks + ((8 * w + 2 * (pk >> 5)) * 32 + (pk & 31)) * 16;
            half8 hi, lo;
            split8(*(const f32x4*)a, *(const f32x4*)(a + 512), hi, lo);
            unsigned char* b = Vs + vreg0 + (lane + 64 * u) * 16;  // V pair: dim 128 (w % 2) + lane + 64u
            f32x4 v0 = *(const f32x4*)b, v1 = *(const f32x4*)(b + HD * 16);
            if (k0 + 32 > kend) {
                const int key = k0 + 8 * (w >> 1);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v0[e] = key + e < kend ? v0[e] : 0.f;
                    v1[e] = key + 4 + e < kend ? v1[e] : 0.f;
                }
            }
            half8 vh, vl;
            split8(v0, v1, vh, vl);
            *(half8*)a = hi;
            *(half8*)(a + 512) = lo;
            *(half8*)b = vh;
            *(half8*)(b + HD * 16) = vl;
        }
        lds_barrier();  // tile j is in LDS, split, for every wave; every wave is done with tile j - 1 and its exchange
        if (j + 1 < ntiles) issue(j + 1);  // into the slot of tile j - 1
        f32x16 Sh = f32x16{}, Sl = f32x16{};
        constexpr int KP = 2;
        half8 kb[KP][2];
#pragma unroll
        for (int s = 0; s < KP; s++) {
            kb[s][0] = *(const half8*)(Ks + kaddr + s * 2048);
            kb[s][1] = *(const half8*)(Ks + kaddr + s * 2048 + 512);
        }
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const half8 kh = kb[s % KP][0], kl = kb[s % KP][1];
            if (s + KP < 8) {
                kb[s % KP][0] = *(const half8*)(Ks + kaddr + (s + KP) * 2048);
                kb[s % KP][1] = *(const half8*)(Ks + kaddr + (s + KP) * 2048 + 512);
            }
            Sh = mfma32(kh, qh[s], Sh);
            Sl = mfma32(kh, ql[s], Sl);
            Sl = mfma32(kl, qh[s], Sl);
        }
        f32x16 S = Sh + Sl;
#pragma unroll
        for (int a = 0; a < 4; a++) xs[w][a][lane] = f32x4{S[4 * a], S[4 * a + 1], S[4 * a + 2], S[4 * a + 3]};
        lds_barrier();
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const f32x4 o = xs[w ^ 1][a][lane];
#pragma unroll
            for (int b = 0; b < 4; b++) S[4 * a + b] += o[b];  // a + b == b + a: both waves hold the same S
        }
        // register i of lane (r, h) is key 8h + i (i < 8) or 16 + 8h + i - 8 of the tile for row r
        if (!__all(k0 >= start && k0 + 32 <= vis)) {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int key = k0 + 8 * h + i + (i >= 8 ? 8 : 0);
                S[i] = (unsigned)(key - start) < seen ? S[i] : NEG_INF;
            }
        }
        float mt = vmax(S[0], S[1]);  // masked scores are -inf, never NaN: single-instruction maxima
#pragma unroll
        for (int i = 2; i < 16; i += 2) mt = vmax3(mt, S[i], S[i + 1]);
        mt = max_xor32(mt);
        mt *= scale2;  // scale2 > 0
        const bool rescale = m != NEG_INF && mt > m + LAZY2;
        const float mr = m == NEG_INF || rescale ? fmaxf(m, mt) : m;
        float cf = 1.f;
        if (__any(rescale)) {  // register i of O holds row 8(i/4) + 4h + i%4, whose factor that row's lanes hold
            cf = rescale ? fast_exp2(m - mr) : 1.f;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const float f = __shfl(cf, 8 * (i >> 2) + 4 * h + (i & 3));
#pragma unroll
                for (int nb = 0; nb < 4; nb++) O[nb][i] *= f;
            }
        }
        m = mr;
        const float base = mr == NEG_INF ? 0.f : mr;
        float p[16], ls = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            p[i] = fast_exp2(__builtin_fmaf(S[i], scale2, -base));
            ls += p[i];
        }
        lsum = lsum * cf + ls;
        half8 ph[2], pl[2];
#pragma unroll
        for (int k = 0; k < 2; k++)
            split8(f32x4{p[8 * k], p[8 * k + 1], p[8 * k + 2], p[8 * k + 3]},
                   f32x4{p[8 * k + 4], p[8 * k + 5], p[8 * k + 6], p[8 * k + 7]}, ph[k], pl[k]);
        // key step k: keys 16k + 8h .. +7 = V groups 4k + 2h, +1; dim block nb: dims 128dh + 32nb + r
        auto vaddr = [&](int i) { return Vs + ((4 * (i >> 2) + 2 * h) * HD + 128 * dh + 32 * (i & 3) + r) * 16; };
        constexpr int VP = 2;
        half8 vb[VP][2];
#pragma unroll
        for (int i = 0; i < VP; i++) {
            vb[i][0] = *(const half8*)vaddr(i);
            vb[i][1] = *(const half8*)(vaddr(i) + HD * 16);
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const half8 vh = vb[i % VP][0], vl = vb[i % VP][1];
            if (i + VP < 8) {
                vb[i % VP][0] = *(const half8*)vaddr(i + VP);
                vb[i % VP][1] = *(const half8*)(vaddr(i + VP) + HD * 16);
            }
            O[i & 3] = mfma32(pl[i >> 2], vh, mfma32(ph[i >> 2], vl, mfma32(ph[i >> 2], vh, O[i & 3])));
        }
    }

    // partials of this wave's rows of present tokens: its 128 dims; m and l from the dim-half-0 wave
    lsum += __shfl_xor(lsum, 32);
    const size_t rpk = (size_t)T * GQA;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int ri = 8 * (i >> 2) + 4 * h + (i & 3);
        if (t0 + (ri >> 3) < T) {
            float* pp = part + ((kvh * rpk + (size_t)t0 * GQA + ri) * nch + sp) * PART + PACC + 128 * dh + r;
#pragma unroll
            for (int nb = 0; nb < 4; nb++) pp[32 * nb] = O[nb][i];
        }
    }
    if (dh == 0 && h == 0 && tr < T) {
        float* pp = part + ((kvh * rpk + (size_t)t0 * GQA + r) * nch + sp) * PART;
        pp[0] = m;
        pp[1] = lsum;
    }
}

}  // namespace

// Splits per f16 plan at most: about one work-group per CU down to blocks of 64 tokens; with at most 16, a 64-token block
// at 28,000 positions took 95 us on 64 work-groups, 64 us on 256. The workspace bound is tokens x splits <= 4,096.
constexpr int PF_MAXCH = 64;
// The cheapest split count of one work-group shape by a model of the call (0.01 us): what does not depend on the splits,
// a wave's tiles, and what each split adds in partials written (20 of 55) and read back by the merge, which takes the
// splits with keys from start on; from 32 splits on a split costs half.
static PrefillPlan best_splits(int T, int kend, int start, int ks, int& cost) {
    const int pt = 32 / ks, blocks = (T + pt - 1) / pt, tiles = (kend + 31) / 32;
    int most = 128 / blocks;  // at most about one work-group per CU
    most = most > PF_MAXCH ? PF_MAXCH : most < 1 ? 1 : most;
    const int below = (int)(100LL * start / kend);  // of 100 tiles, the masked ones below the window
    const int per = T * (55 - 35 * below / 100) + 2000;
    PrefillPlan p{kend, 1, ks};
    cost = INT_MAX;
    for (int nch = 1; nch <= most && (nch == 1 || nch * ks <= tiles); nch++) {
        const int s = (tiles + nch * ks - 1) / (nch * ks);  // tiles of a wave
        const int c = (ks == 1 ? 1100 + 135 * s : 1230 + 145 * s) + (nch <= 32 ? nch : 16 + nch / 2) * per / 100;
        if (c < cost) {
            cost = c;
            p.nch = nch;
        }
    }
    // The card is power limited on long calls. One group: a block of 32 tokens computes up to 16 absent ones more than
    // blocks of 16. Two groups: each tile read for half as many rows, and a masked tile costs more.
    const int s = (tiles + p.nch * ks - 1) / (p.nch * ks);
    if (ks == 1) cost += (blocks * 32 - (T + 15) / 16 * 16) * tiles * 40 / 1000;
    else cost += s * below * 40 / 100 + (T > 256 ? s * (T - 256) * 24 / 512 : 0) + (s > 32 ? 60 * (s - 32) : 0);
    return p;
}

PrefillPlan prefill_plan(int T, int n, int start, int* us100) {
    // Two key groups save half the partials and read each tile for half as many rows, which tells on long splits, where the
    // card is power limited, and sooner where the keys come from HBM. Time of two groups over one, per call with the merge,
    // keys from HBM (as many layers in turn as 640 MB hold) / from the last-level cache:
    //   512 tokens at 1,000, 4,000, 7,500, 9,000, 12,000, 28,000 positions .92 .95 1.02 1.08 1.08 1.10 / .91 .93 .97 .98 1.00 1.05
    //   256 tokens at 1,000, 9,000, 16,000, 20,000, 24,000, 28,000         .91 .95 .98 1.02 1.05 1.07 / .91 .91 .96 .97 .99 1.00
    //   200 tokens at 2,000, 9,000, 20,000, 28,000, 36,000                 .91 .82 .93 .96 1.00       / .90 .81 .90 .94
    //   128 tokens at 2,000, 9,000, 28,000, 45,000, 60,000                 .89 .90 .94 1.00 1.05      / .88 .88 .92
    //    64 tokens at 3,000, 28,000, 60,000, 90,000, 120,000               .88 .99 1.01 1.07 1.11     / .87 .97
    // The line lies between the two crossings. Over 570 such pairs (64-512 tokens) the plan loses 0.1% on average against
    // the faster group count, 4.4% at most from HBM and 6% from the cache. Splits, two groups: 64 tokens at 4,000 positions
    // on 32 / 16 / 8 splits 32.7 / 26.4 / 26.2 us, at 9,000 34.4 / 31.5 / 38.7, 128 tokens at 2,000 on 16 / 8 32.5 / 26.0.
    const int kend = n + T - 1;
    int c1, c2;
    const PrefillPlan p1 = best_splits(T, kend, start, 1, c1), p2 = best_splits(T, kend, start, 2, c2);
    if (us100) *us100 = c2 <= c1 ? c2 : c1;
    return c2 <= c1 ? p2 : p1;
}

PrefillPlan prefill32_plan(int T, int n, int start) {
    // As best_splits (0.01 us): 2.55 us per tile of a work-group against the partials and the merge, whose kernel for more
    // than 16 splits in the window takes about 3 us longer. 5 tokens at 1,000 / 9,000 / 20,000 positions 17.9 / 27.6 / 44.5
    // us on at most 64 splits of at least 64 positions, 14.4 / 21.7 / 32.7 on these; 64 tokens at 1,000 positions on 8 / 16 /
    // 32 splits 26.1 / 24.6 / 31.4, at 4,000 59.5 / 41.6 / 38.4 us; at 2,000 with a window of 500 on 16 / 20 / 32 27.0 / 24.6 /
    // 22.6.
    const int kend = n + T - 1, tiles = (kend + 31) / 32;
    int most = 256 / (KVH * ((T + P32_PT - 1) / P32_PT));  // at most about one work-group per CU
    most = most < 1 ? 1 : most;
    int best = INT_MAX, nch = 1;
    // The merge reads the splits with keys of the window, and the stores of the others cost nothing measurable; with a window
    // the mean of a split's longest and average tiles fits best (121 windows of 5-256 tokens at 64-9,000 positions, each on
    // 10 split counts: 1.5% on average behind the best of them; splits as without a window 2-3%, up to 17%)
    const long long seen = kend - start;
    const int per = (int)((T < 64 ? T * 45 : T * 55 + 800) * seen / kend);
    for (int k = 1; k <= most && k <= tiles; k++) {
        const int len = start > 0 ? 255 * tiles / k / 2 + 255 * ((tiles + k - 1) / k) / 2 : 255 * tiles / k;
        const int c = len + k * per / 100 + (k * seen > 16LL * kend ? 300 : 0);
        if (c < best) {
            best = c;
            nch = k;
        }
    }
    return PrefillPlan{kend, nch, 1};
}

size_t prefill_ws_floats(int T, int nch) { return (size_t)KVH * T * GQA * nch * PART; }

hipError_t launch_prefill(const Geom& g, const void* base, int layer, const float* q, int T, int n, int start,
                          float scale, const PrefillPlan& p, float* ws, const Launch& L) {
    if (g.fmt != 0) return hipErrorNotSupported;
    const char* b = (const char*)base;
    const void* kp = b + g.plane(layer, 0, 0) * g.plane_bytes();
    const void* vp = b + g.plane(layer, 1, 0) * g.plane_bytes();
    const int pt = p.ks == 2 ? PfGeom<2>::PT : PfGeom<1>::PT;
    return launch(p.ks == 2 ? prefill_f16<2> : prefill_f16<1>, dim3((T + pt - 1) / pt * p.nch * KVH), dim3(NW * 64), L, kp,
                  vp, g.plane_elems, q, T, n, start, scale * LOG2E, p.span, p.nch, ws);
}

hipError_t launch_prefill_f32(const Geom& g, const void* base, int layer, const float* q, int T, int n, int start,
                              float scale, const PrefillPlan& p, float* ws, const Launch& L) {
    if (g.fmt != 1) return hipErrorNotSupported;
    const char* b = (const char*)base;
    const float* kp = (const float*)(b + g.plane(layer, 0, 0) * g.plane_bytes());
    const float* vp = (const float*)(b + g.plane(layer, 1, 0) * g.plane_bytes());
    dim3 grid((T + P32_PT - 1) / P32_PT * p.nch * KVH);
    return launch(prefill_f32, grid, dim3(P32_NW * 64), L, kp, vp, g.plane_elems, q, T, n, start, scale * LOG2E,
                  p.span, p.nch, ws);
}

}  // namespace mkv
