// kvd_gemm.hip -- the OK_Q4B GEMM over a token batch (prefill passes, batched
// decode) with the block scales folded into int8 weight digits, on
// v_mfma_i32_16x16x64_i8 (gfx950).
//
// The exact integer of the decode GEMV, one rounding (RNE) per output:
//   x side: xq = rne(x 2^sh) per token as three balanced base-256 digits
//     a0 + 2^8 a1 + 2^16 a2 (k_stage);
//   weight side: code * f16 scale = V 2^(top - 9), top = the row's largest
//     block exponent: an integer V = code * Ms, Ms = f16 2^(9 - top) < 2^20 for
//     blocks at most 9 exponents below top, and V = R + 2^8 L + 2^16 H in
//     balanced base-256 digits.  R is zero unless the block's exponent is below
//     top - 1 and Ms has a low byte.
//   The digit products meet in int32 sums by their weight, S_k = sum over
//     a_i, digit_j with i + j = k (|S_k| < 3 K 2^14 < 2^31), and the output is
//     RNE(sum_k 2^(8k) S_k 2^(top-9-sh)).
// Tensors with few such low bytes (DevW::fold = 2) run six products, L and H,
// and add the listed blocks' low bytes at the end; the others (fold = 3) run
// all nine.
// No arithmetic is left per 32-column block: k_gemm_q4b (kvd_prefill.hip), which
// adds d * Ms per block and output in int64, is bound by exactly that (two
// quarter-rate multiply-adds and the digit recombination per block and output)
// and now serves only tensors whose rows spread over more than 9 exponents.
#include "kvd_internal.h"
#include "kvd_exact.h"
#include "kvd_vec.h"
#include "kvd_pass.h"
#include <algorithm>

namespace kvd {

namespace {

typedef short s2 __attribute__((ext_vector_type(2)));

// all but this wave's youngest N loads have arrived and its LDS reads are done,
// then the workgroup's barrier
template <int N> __device__ __forceinline__ void arrive_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}

// The int16 weight words code * m of a dword's 8 columns, pairs (0,4) (1,5)
// (2,6) (3,7), then their low and high balanced digits as bytes in the column
// order 0 1 4 5 2 3 6 7 (k_stage writes the activation digits in that order).
__device__ __forceinline__ void codes16(int w, s2 c[4]) {
    const s2 v = __builtin_bit_cast(s2, w);
    c[0] = (s2)(v << 12) >> 12; c[1] = (s2)(v << 8) >> 12; c[2] = (s2)(v << 4) >> 12; c[3] = v >> 12;
}
__device__ __forceinline__ void lo_bytes(const s2 w[4], int &a, int &b) {
    a = (int)__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, w[1]), __builtin_bit_cast(uint32_t, w[0]), 0x06020400u);
    b = (int)__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, w[3]), __builtin_bit_cast(uint32_t, w[2]), 0x06020400u);
}
__device__ __forceinline__ void hi_bytes(const s2 w[4], int &a, int &b) {
    a = (int)__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, w[1]), __builtin_bit_cast(uint32_t, w[0]), 0x07030501u);
    b = (int)__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, w[3]), __builtin_bit_cast(uint32_t, w[2]), 0x07030501u);
}
__device__ __forceinline__ s2 both(int v) { s2 r; r.x = (short)v; r.y = (short)v; return r; }

// the digits of one dword's 8 columns, as two dwords each: V = code (256 m16 + m8)
struct Dig { int l0, l1, h0, h1, r0, r1; };
template <int ND> __device__ __forceinline__ Dig fold8(int w, int m16, int m8) {
    const s2 m = both(m16), half = both(128);
    s2 c[4], v[4], h[4];
    Dig d;
    codes16(w, c);
    if constexpr (ND == 3) {
        const s2 mr = both(m8);                        // |code m8| <= 2040
        s2 r[4];
        #pragma unroll
        for (int k = 0; k < 4; k++) { r[k] = c[k] * mr; v[k] = c[k] * m + ((s2)(r[k] + half) >> 8); }
        lo_bytes(r, d.r0, d.r1);
    } else {
        #pragma unroll
        for (int k = 0; k < 4; k++) v[k] = c[k] * m;
    }
    #pragma unroll
    for (int k = 0; k < 4; k++) h[k] = v[k] + half;
    lo_bytes(v, d.l0, d.l1);
    hi_bytes(h, d.h0, d.h1);
    return d;
}

constexpr int FOLD_WAVES = 8;
constexpr int FOLD_LDS = 156 * 1024;      // ring bytes a workgroup may take (one per CU)

// LDS rings: per K group the activation digits of a super-step (2 halves x 3
// planes x TT tiles x 1 KiB), D slots; per wave the codes (1 KiB) and scales
// (256 bytes) of its two row tiles, D + 1 slots; as deep as fits, up to 6
constexpr int fold_planes(int WK, int TT) { return WK * 6 * TT * 1024; }
constexpr int FOLD_CODES = FOLD_WAVES * 2 * (1024 + 256);
constexpr int fold_depth(int WK, int TT) {
    const int d = (FOLD_LDS - FOLD_CODES) / (fold_planes(WK, TT) + FOLD_CODES);
    return d < 6 ? d : 6;
}

}  // namespace

// A workgroup's 8 waves are WR = 8 / WK row groups x WK K groups; it owns TT
// 16-token tiles and 32 rows per row group (PAIRED: 16 gate rows and the same
// up rows).  K runs in super-steps of 128 columns = 4 blocks, a K group's own
// share of them: lane (row n = lane % 16, g = lane / 16) takes its row's block
// 4 s + g -- 16 bytes of codes and one f16 -- so a wave's load covers 64
// contiguous bytes of each row and no lane exchange is needed; the two 64-column
// halves of those 16 bytes are one MFMA step each.  The activation digits are
// the A operand (16 tokens), stored by k_stage in operand order.
//
// Everything a super-step reads goes straight into LDS rings, super-steps ahead
// (no registers held by loads in flight; with loads through registers the
// accumulators left room for one step ahead, less than the latency of the
// weights, and the kernel ran at a fifth of the MFMA rate).  One barrier per
// super-step: before it each wave waits for its own loads of that step, after it
// the slots read in the step before are free for the next loads.  The weights
// run one super-step ahead of the activations: their digits for the next half
// are formed between this half's MFMAs (vector and matrix pipes both busy; one
// dword of codes per token tile at TT = 4).
//
// The waves of a K group share the staged digits (each 1 KiB operand serves 4
// MFMAs of each wave); K groups trade that sharing for a smaller output tile
// where rows x tokens alone would leave CUs idle, and meet in LDS at the end.
// ND = 2: the low bytes of the listed blocks (DevW::exl, 4 blocks of a row
// tile per pass, one per lane group: r = code * low byte = Rlo + 256 Rhi) are
// added to the sums after the loop.  In the loop, skipped where no scale of the
// super-step has one, they cost more than their share: 15% of a tile's steps,
// but nearly every step of some wave, for which the others wait at the barrier.
template <bool PAIRED, int ND, int WK, int TT, bool SPLIT>
__global__ __launch_bounds__(64 * FOLD_WAVES, 2) void k_gemm_fold(GemmArgs a) {
    constexpr int WR = FOLD_WAVES / WK, RT = 2, D = fold_depth(WK, TT), DC = D + 1;
    constexpr int PU = 6 * TT, PL = (PU + WR - 1) / WR, NL = PL + 2 * RT;   // 1 KiB operands, loads per wave and step
    constexpr int PLANES = fold_planes(WK, TT), CODES = D * PLANES, SCALES = FOLD_WAVES * RT * 1024;
    constexpr int LDS = CODES + DC * FOLD_CODES;
    static_assert(D >= 2 && LDS <= FOLD_LDS && (D - 1) * NL + 2 * RT < 63, "ring slots and load counts");
    __shared__ __align__(1024) uint8_t ring[LDS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave % WR, kg = wave / WR, n16 = lane & 15, g = lane >> 4;
    const int NT = a.TP / 16, S = a.cols / 128;        // token tiles, super-steps
    // this K group's super-steps [sk, sk + ns), ns <= kper
    const int kper = (S + (int)gridDim.z * WK - 1) / ((int)gridDim.z * WK);
    const int sk = ((int)blockIdx.z * WK + kg) * kper;
    const int ns = S - sk < kper ? (S - sk > 0 ? S - sk : 0) : kper;
    const int tile0 = (int)blockIdx.y * TT;
    // the wave's row tiles: segment and row base within it; tiles past the
    // launch's rows repeat the last one and store nothing
    const int total = PAIRED ? a.arows / 2 : a.arows;
    int seg[RT], rb0[RT], grow[RT], voc[RT], vos[RT], scs[RT], top[RT];
    bool live[RT];
    v4i rc[RT], rs[RT];
    float sc[RT];
    #pragma unroll
    for (int r = 0; r < RT; r++) {
        int row = PAIRED ? ((int)blockIdx.x * WR + wr) * 16 : (((int)blockIdx.x * WR + wr) * RT + r) * 16;
        live[r] = row < total;
        if (!live[r]) row = total - 16;
        grow[r] = row;
        int s = PAIRED ? r : 0;
        if (!PAIRED) while (s < a.nseg - 1 && row >= a.seg[s].w.rows) { row -= a.seg[s].w.rows; s++; }
        seg[r] = s; rb0[r] = row;
        const DevW &w = a.seg[s].w;
        const int rb = w.cols / 2;
        rc[r] = rsrc_of(w.codes + (size_t)row * rb, 16u * rb);
        // the scales' interleaved copy: il rows per group, [group][block][il]
        rs[r] = rsrc_of(w.bs8 + (size_t)row * w.nblk, 32u * w.nblk);
        voc[r] = n16 * rb + 16 * g;
        vos[r] = ((n16 / w.il) * w.nblk * w.il + g * w.il + n16 % w.il) * 2;
        scs[r] = __builtin_amdgcn_readfirstlane(8 * w.il);   // bytes of a super-step's scales (4 blocks x il x 2)
        top[r] = w.etop[row + n16];
        sc[r] = ldexpf(1.0f, 9 - top[r]);
    }
    const v4i rpl = rsrc_of(a.planes, 3u * S * 2 * NT * 1024);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)ring;
    // local super-step s in the tensor (past the last: the last again)
    auto step_at = [&](int s) -> int {
        const int sl = sk + (s < ns ? s : ns - 1);
        return __builtin_amdgcn_readfirstlane(sl < S ? sl : S - 1);
    };
    // load n of the NL this wave issues for a step: the codes and scales of
    // local super-step s + 1 into codes slot dc, then its share of the
    // activation operands of s into slot d
    auto load = [&](int n, int s, int d, int dc) {
        if (n < 2 * RT) {
            const int r = n >> 1, sx = step_at(s + 1);
            const uint32_t b = lds0 + CODES + dc * FOLD_CODES;
            if (n & 1) dma2(b + SCALES + (wave * RT + r) * 256, vos[r], rs[r], sx * scs[r]);
            else dma16(b + (wave * RT + r) * 1024, voc[r], rc[r], sx * 64);
            return;
        }
        // operand q = (half m, plane p, tile j) of the super-step; token tiles
        // past the batch's repeat its last
        const int sx = step_at(s), k = n - 2 * RT, q = wr * PL + k < PU ? wr * PL + k : PU - 1;
        const int m = q / (3 * TT), p = q / TT % 3, j = q % TT, tl = tile0 + j < NT ? tile0 + j : NT - 1;
        const int so = __builtin_amdgcn_readfirstlane((((p * S + sx) * 2 + m) * NT + tl) * 1024);
        dma16(lds0 + d * PLANES + kg * (PU * 1024) + q * 1024, lane * 16, rpl, so);
    };
    constexpr int NS = ND + 2, O = ND - 2;             // sums S_(3-ND) .. S_4; acc[k + O] is S_(k+1)
    v4i acc[NS][RT][TT];
    #pragma unroll
    for (int k = 0; k < NS; k++)
        #pragma unroll
        for (int r = 0; r < RT; r++)
            #pragma unroll
            for (int j = 0; j < TT; j++) acc[k][r][j] = (v4i){0, 0, 0, 0};
    struct Wd { v4i L, H, R; };                        // weight digits of one half
    auto put = [](Wd &w, int d, const Dig &g) {
        w.L[2 * d] = g.l0; w.L[2 * d + 1] = g.l1; w.H[2 * d] = g.h0; w.H[2 * d + 1] = g.h1;
        if constexpr (ND == 3) { w.R[2 * d] = g.r0; w.R[2 * d + 1] = g.r1; }
    };
    // the products of one 64-column half (operands at b, weight digits w); the
    // next half's digits nw are formed on the way from its code dwords and
    // scale integers ms
    auto half = [&](const v4i *b, const Wd (&w)[RT], const int2 (&xy)[RT], const int (&ms)[RT], Wd (&nw)[RT], auto between) {
        v4i a0 = b[0], a1 = b[TT * 64], a2 = b[2 * TT * 64];
        #pragma unroll
        for (int j = 0; j < TT; j++) {
            v4i n0, n1, n2;
            if (j + 1 < TT) { n0 = b[(j + 1) * 64]; n1 = b[(TT + j + 1) * 64]; n2 = b[(2 * TT + j + 1) * 64]; }
            #pragma unroll
            for (int k = 0; k < 2 * RT; k++)
                if (k * TT / (2 * RT) == j) put(nw[k >> 1], k & 1, fold8<ND>(k & 1 ? xy[k >> 1].y : xy[k >> 1].x, ms[k >> 1] >> 8, ms[k >> 1] & 255));
            #pragma unroll
            for (int r = 0; r < RT; r++) {
                acc[O + 0][r][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, w[r].L, acc[O + 0][r][j], 0, 0, 0);
                acc[O + 3][r][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a2, w[r].H, acc[O + 3][r][j], 0, 0, 0);
                acc[O + 1][r][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, w[r].H, acc[O + 1][r][j], 0, 0, 0);
                acc[O + 2][r][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a2, w[r].L, acc[O + 2][r][j], 0, 0, 0);
            }
            if constexpr (ND == 3) {
                #pragma unroll
                for (int r = 0; r < RT; r++) {
                    acc[0][r][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, w[r].R, acc[0][r][j], 0, 0, 0);
                    acc[1][r][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, w[r].R, acc[1][r][j], 0, 0, 0);
                    acc[2][r][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a2, w[r].R, acc[2][r][j], 0, 0, 0);
                }
            }
            #pragma unroll
            for (int r = 0; r < RT; r++) {
                acc[O + 1][r][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, w[r].L, acc[O + 1][r][j], 0, 0, 0);
                acc[O + 2][r][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, w[r].H, acc[O + 2][r][j], 0, 0, 0);
            }
            // the next tile's operands first, then vector instructions between the MFMAs
            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
            #pragma unroll
            for (int k = 0; k < 3 * ND * RT; k++) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, TT >= 3 ? 2 : 4, 0);
            }
            if (j + 1 < TT) { a0 = n0; a1 = n1; a2 = n2; }
            __builtin_amdgcn_sched_barrier(0);
            between(j);
        }
    };
    auto codes_of = [&](int d, int r) { return (const int2 *)(ring + CODES + d * FOLD_CODES + (wave * RT + r) * 1024 + lane * 16); };
    auto ms_of = [&](int d, int r) {
        const uint32_t h = ((const uint32_t *)(ring + CODES + d * FOLD_CODES + SCALES))[(wave * RT + r) * 64 + lane];
        return (int)((float)__builtin_bit_cast(_Float16, (unsigned short)h) * sc[r]);
    };
    // every K group runs the same number of barriers (kper); one with fewer
    // super-steps (ns) repeats its last load and computes nothing
    #pragma unroll
    for (int n = 0; n < 2 * RT; n++) load(n, -1, 0, 0);
    #pragma unroll
    for (int d = 0; d < D - 1; d++)
        #pragma unroll
        for (int n = 0; n < NL; n++) load(n, d, d, d + 1);
    int d = 0, dc = 0;                                 // ring slots of super-step s
    Wd wa[RT], wb[RT];
    int ms[RT];
    for (int s = 0; s < kper; s++) {
        arrive_barrier<(D - 2) * NL>();                // planes of s, codes of s + 1
        // the step's loads go into the slots of step s - 1, a few after each
        // token tile's products (all at once they take ~600 clocks to issue)
        const int dp = d == 0 ? D - 1 : d - 1, dcp = dc == 0 ? DC - 1 : dc - 1;
        auto issue = [&](int i) {
            #pragma unroll
            for (int n = 0; n < NL; n++) if (n * 2 * TT / NL == i) load(n, s + D - 1, dp, dcp);
        };
        const int dn = dc == DC - 1 ? 0 : dc + 1;
        const v4i *ops = (const v4i *)(ring + d * PLANES + kg * (PU * 1024)) + lane;
        if (s == 0) {
            #pragma unroll
            for (int r = 0; r < RT; r++) {
                ms[r] = ms_of(0, r);
                const int2 xy = codes_of(0, r)[0];
                put(wa[r], 0, fold8<ND>(xy.x, ms[r] >> 8, ms[r] & 255));
                put(wa[r], 1, fold8<ND>(xy.y, ms[r] >> 8, ms[r] & 255));
            }
        }
        if (s < ns) {
            int2 zw[RT], xy[RT];
            int mn[RT];
            #pragma unroll
            for (int r = 0; r < RT; r++) { zw[r] = codes_of(dc, r)[1]; xy[r] = codes_of(dn, r)[0]; mn[r] = ms_of(dn, r); }
            half(ops, wa, zw, ms, wb, [&](int j) { issue(j); });
            half(ops + 3 * TT * 64, wb, xy, mn, wa, [&](int j) { issue(TT + j); });
            #pragma unroll
            for (int r = 0; r < RT; r++) ms[r] = mn[r];
        } else {
            #pragma unroll
            for (int i = 0; i < 2 * TT; i++) issue(i);
        }
        d = d == D - 1 ? 0 : d + 1;
        dc = dn;
    }
    arrive_barrier<0>();                               // no load in flight, the ring is free
    // S_0 .. S_4 -> the exact sum
    int64_t tot[RT][TT][4];
    #pragma unroll
    for (int r = 0; r < RT; r++)
        #pragma unroll
        for (int j = 0; j < TT; j++)
            #pragma unroll
            for (int i = 0; i < 4; i++) {
                tot[r][j][i] = 0;
                #pragma unroll
                for (int k = 0; k < NS; k++) tot[r][j][i] += (int64_t)acc[k][r][j][i] << (8 * (k + 1 - O));
            }
    if constexpr (ND == 2) {
        // the listed blocks' low bytes, four blocks a pass; the K groups and
        // splits take the passes in turn
        #pragma unroll
        for (int r = 0; r < RT; r++) {
            const DevW &w = a.seg[seg[r]].w;
            const int e0 = w.exo[rb0[r] / 16], e1 = w.exo[rb0[r] / 16 + 1];
            for (int e = e0 + 4 * ((int)blockIdx.z * WK + kg); e < e1; e += 4 * (int)gridDim.z * WK) {
                const uint32_t x = e + g < e1 ? w.exl[e + g] : 0;   // row | block << 4 | low byte << 24
                const int b = (x >> 4) & 0xFFFF, m8 = n16 == (int)(x & 15) ? (int)(x >> 24) : 0;
                const int4 cw = *(const int4 *)(w.codes + (size_t)(rb0[r] + (x & 15)) * (w.cols / 2) + 16 * b);
                v4i L[2], H[2];
                #pragma unroll
                for (int m = 0; m < 2; m++)
                    #pragma unroll
                    for (int k = 0; k < 2; k++) {
                        const Dig q = fold8<2>(m ? (k ? cw.w : cw.z) : (k ? cw.y : cw.x), m8, 0);
                        L[m][2 * k] = q.l0; L[m][2 * k + 1] = q.l1; H[m][2 * k] = q.h0; H[m][2 * k + 1] = q.h1;
                    }
                #pragma unroll
                for (int j = 0; j < TT; j++) {
                    const int tl = tile0 + j < NT ? tile0 + j : NT - 1;
                    v4i u[4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
                    #pragma unroll
                    for (int m = 0; m < 2; m++) {
                        v4i o[3];
                        #pragma unroll
                        for (int p = 0; p < 3; p++)
                            o[p] = *(const v4i *)(a.planes + ((((size_t)p * S + (b >> 2)) * 2 + m) * NT + tl) * 1024 + ((b & 3) * 16 + n16) * 16);
                        u[0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(o[0], L[m], u[0], 0, 0, 0);
                        u[1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(o[1], L[m], u[1], 0, 0, 0);
                        u[2] = __builtin_amdgcn_mfma_i32_16x16x64_i8(o[2], L[m], u[2], 0, 0, 0);
                        u[3] = __builtin_amdgcn_mfma_i32_16x16x64_i8(o[2], H[m], u[3], 0, 0, 0);
                        u[1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(o[0], H[m], u[1], 0, 0, 0);
                        u[2] = __builtin_amdgcn_mfma_i32_16x16x64_i8(o[1], H[m], u[2], 0, 0, 0);
                    }
                    #pragma unroll
                    for (int i = 0; i < 4; i++)
                        tot[r][j][i] += (int64_t)u[0][i] + ((int64_t)u[1][i] << 8) + ((int64_t)u[2][i] << 16) + ((int64_t)u[3][i] << 24);
                }
            }
        }
    }
    // The sums go through LDS, [(K group, row group, tile r, j, i)][lane]: the K
    // groups meet there, each finishing every WK-th (j, i), in loops that stay
    // rolled (unrolled, the rounding and the activation of 32 outputs per lane
    // are more code than the rest).
    constexpr int ITEMS = TT * 4;
    static_assert(FOLD_WAVES * RT * ITEMS * 64 * 8 <= LDS, "the sums fit the rings");
    int64_t *const ex = (int64_t *)ring + lane;
    auto at = [&](int k, int r, int it) { return (((k * WR + wr) * RT + r) * ITEMS + it) * 64; };
    #pragma unroll
    for (int r = 0; r < RT; r++)
        #pragma unroll
        for (int it = 0; it < ITEMS; it++) ex[at(kg, r, it)] = tot[r][it >> 2][it & 3];
    __syncthreads();
    auto sum_of = [&](int r, int it) {
        int64_t v = 0;
        #pragma unroll
        for (int k = 0; k < WK; k++) v += ex[at(k, r, it)];
        return v;
    };
    const int t0 = tile0 * 16 + 4 * g;                 // lane's tokens: t0 + 16 (it / 4) + it % 4
    // where a split keeps its partial of (r, token t)
    auto slot = [&](int r, int t) { return (size_t)t * a.arows + (PAIRED && r ? a.arows / 2 : 0) + grow[r] + n16; };
    const size_t zs = (size_t)a.TP * a.arows;
    if constexpr (SPLIT) {
        // every split stores its exact partials in its own slice (agent-scope
        // stores, coherent across the XCDs' L2s); the tile's last split adds
        // the others' to its own
        #pragma unroll 1
        for (int it = kg; it < ITEMS; it += WK) {
            const int t = t0 + 16 * (it >> 2) + (it & 3);
            #pragma unroll
            for (int r = 0; r < RT; r++)
                if (live[r] && t < a.TP) st_agent(&a.part[blockIdx.z * zs + slot(r, t)], sum_of(r, it));
        }
        mem_complete();
        __shared__ int last;
        __syncthreads();
        int *cnt = a.cnt + blockIdx.y * gridDim.x + blockIdx.x;
        if (tid == 0) last = arrive(cnt) == (int)gridDim.z - 1;
        __syncthreads();
        if (!last) return;
        if (tid == 0) reset_counter(cnt);
    }
    #pragma unroll 1
    for (int it = kg; it < ITEMS; it += WK) {
        const int t = t0 + 16 * (it >> 2) + (it & 3);
        if (t >= a.T) continue;
        const int sh = a.sh[t];
        float y[RT];
        #pragma unroll
        for (int r = 0; r < RT; r++) {
            int64_t v = sum_of(r, it);
            if constexpr (SPLIT)
                for (int z = 0; z < (int)gridDim.z; z++)
                    if (z != (int)blockIdx.z) v += ld_agent(&a.part[z * zs + slot(r, t)]);
            y[r] = sh == SH_ZERO ? 0.0f : rne_i64_scaled(v, top[r] - 9 - sh);
            if (!PAIRED && live[r]) a.seg[seg[r]].out[(size_t)t * a.seg[seg[r]].w.rows + rb0[r] + n16] = y[r];
        }
        if constexpr (PAIRED)
            if (live[0]) a.act_out[(size_t)t * a.seg[0].w.rows + rb0[0] + n16] = act_apply(y[0], y[1], a.act, a.mode);
    }
}

// the digits a tensor's GEMM runs (0: not this GEMM): scales that fold, whole super-steps
int gemm_folds(const DevW &w) { return w.rows % 64 == 0 && w.cols % 128 == 0 && w.cols <= 32768 ? w.fold : 0; }

template <bool PAIRED, int ND, int WK, int TT>
static void fold_go(const GemmArgs &g, dim3 grid, hipStream_t s) {
    const dim3 wg(64 * FOLD_WAVES);
    if (grid.z > 1) hipLaunchKernelGGL((k_gemm_fold<PAIRED, ND, WK, TT, true>), grid, wg, 0, s, g);
    else hipLaunchKernelGGL((k_gemm_fold<PAIRED, ND, WK, TT, false>), grid, wg, 0, s, g);
}
template <bool PAIRED>
static void fold_pick(const GemmArgs &g, int nd, int wk, int tt, dim3 grid, hipStream_t s) {
    switch (nd * 100 + wk * 10 + tt) {
    case 211: fold_go<PAIRED, 2, 1, 1>(g, grid, s); break;
    case 212: fold_go<PAIRED, 2, 1, 2>(g, grid, s); break;
    case 214: fold_go<PAIRED, 2, 1, 4>(g, grid, s); break;
    case 222: fold_go<PAIRED, 2, 2, 2>(g, grid, s); break;
    case 224: fold_go<PAIRED, 2, 2, 4>(g, grid, s); break;
    case 241: fold_go<PAIRED, 2, 4, 1>(g, grid, s); break;
    case 242: fold_go<PAIRED, 2, 4, 2>(g, grid, s); break;
    case 281: fold_go<PAIRED, 2, 8, 1>(g, grid, s); break;
    case 311: fold_go<PAIRED, 3, 1, 1>(g, grid, s); break;
    case 312: fold_go<PAIRED, 3, 1, 2>(g, grid, s); break;
    case 322: fold_go<PAIRED, 3, 2, 2>(g, grid, s); break;
    case 341: fold_go<PAIRED, 3, 4, 1>(g, grid, s); break;
    case 342: fold_go<PAIRED, 3, 4, 2>(g, grid, s); break;
    default: fold_go<PAIRED, 3, 8, 1>(g, grid, s); break;
    }
}

// The shape of a launch: K groups, token tiles per workgroup and K splits with
// the least estimated time (us).  Over 60 launches of three served layer shapes
// at 16 to 512 tokens the pick is within 5% of the best shape's time in 53 and
// within 13% in all (the others: a second split that pays at 16 tokens, and
// down at 256, 134 us against 121); 84% of 2 024 timed shapes are within 25% of
// the estimate.  A super-step takes 1.0 +
// 0.21 us per token tile and digit, a quarter more where the ring holds only
// two slots, 10% more on a full chip; a workgroup 5 us around its steps, more
// with the activation; a split 3 us and its share of the partial sums.
static const int FOLD_SHAPES[][2] = {{1, 1}, {1, 2}, {1, 4}, {2, 2}, {2, 4}, {4, 1}, {4, 2}, {8, 1}};
bool gemm_fold_built(int wk, int tt) {
    for (const auto &sh : FOLD_SHAPES) if (sh[0] == wk && sh[1] == tt) return true;
    return false;
}
// whether k splits of S super-steps each have some (of `slice` partial sums each)
static bool split_ok(int k, int wk, int S, size_t slice, int wgs, size_t part_cap, int cnt_cap) {
    if (k == 1) return true;
    const int steps = (S + k * wk - 1) / (k * wk);
    return k * wk <= S && slice * k <= part_cap && wgs <= cnt_cap && (S + steps * wk - 1) / (steps * wk) == k;
}
void fold_plan(int rows, int tiles, int S, bool paired, int nd, size_t slice, size_t part_cap, int cnt_cap, int &wk, int &tt, int &ks) {
    double best = 1e30;
    wk = 1; tt = 1; ks = 1;
    for (const auto &sh : FOLD_SHAPES) {
        const int WK = sh[0], TT = sh[1];
        if (nd == 3 && TT == 4) continue;              // its accumulators don't fit the registers
        const int rows_wg = FOLD_WAVES / WK * (paired ? 16 : 32);
        const int wgs = ((rows + rows_wg - 1) / rows_wg) * ((tiles + TT - 1) / TT);
        const double outs = (double)FOLD_WAVES / WK * 32 * 16 * TT;
        for (int k = 1; k <= 16; k++) {
            if (!split_ok(k, WK, S, slice, wgs, part_cap, cnt_cap)) continue;
            const int steps = (S + k * WK - 1) / (k * WK);
            const double full = wgs * k < 256 ? wgs * k / 256.0 : 1.0;
            const double step = (1.0 + 0.21 * nd * TT) * (fold_depth(WK, TT) > 2 ? 1.0 : 1.25) * (1.0 + 0.1 * full);
            const double fixed = 5.0 + (paired ? 1.0 + 2.0 * TT / WK : 0.0);
            const double t = (double)((wgs * k + 255) / 256) * (steps * step + fixed) + (k > 1 ? 3.0 + k * (1.0 + outs / 2000.0) : 0.0);
            if (t < best) { best = t; wk = WK; tt = TT; ks = k; }
        }
    }
}

void launch_gemm_fold(const GemmArgs &a, int nrows_total, hipStream_t s) {
    const bool paired = a.act != ACT_NONE;
    if (a.TP % 16 || a.T > a.TP || nrows_total % 64 || (size_t)3 * a.cols * a.TP >= ((size_t)1 << 31))
        return launch_fail("folded GEMM: rows or token count outside the kernel's limits");
    GemmArgs g = a;
    g.arows = nrows_total * (paired ? 2 : 1);
    int nd = 2, wk, tt, ks;
    for (int i = 0; i < a.nseg; i++) nd = std::max(nd, a.seg[i].w.fold);
    const bool can = a.part && a.cnt;
    const int S = a.cols / 128, tiles = a.TP / 16;
    const size_t slice = (size_t)a.TP * g.arows, part_cap = can ? a.part_cap : 0;
    const int cnt_cap = can ? a.cnt_cap : 0;
    auto grid_of = [&] {
        const int rows_wg = FOLD_WAVES / wk * (paired ? 16 : 32);
        return dim3((nrows_total + rows_wg - 1) / rows_wg, (tiles + tt - 1) / tt, ks);
    };
    if (a.shape.wk) {
        wk = a.shape.wk; tt = a.shape.tt; ks = 1;
        if (!gemm_fold_built(wk, tt) || (nd == 3 && tt == 4)) return launch_fail("folded GEMM: no kernel of the shape that was set");
        const dim3 one = grid_of();
        for (int k = 2; k <= a.shape.ks; k++)          // the most splits up to those set
            if (split_ok(k, wk, S, slice, (int)(one.x * one.y), part_cap, cnt_cap)) ks = k;
    } else fold_plan(nrows_total, tiles, S, paired, nd, slice, part_cap, cnt_cap, wk, tt, ks);
    const dim3 grid = grid_of();
    if (paired) fold_pick<true>(g, nd, wk, tt, grid, s);
    else fold_pick<false>(g, nd, wk, tt, grid, s);
}

}  // namespace kvd
