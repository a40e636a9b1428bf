// kvd_pfloat.hip -- float-mode attention of one session's batched prefill: the
// batch's token-heads share every K and V row they read, on the f32 matrix
// cores (v_mfma_f32_16x16x4_f32: f32 products and f32 sums, as on the vector
// units).
//
// A workgroup (8 waves) takes 128 token-heads of one kv head (128 / G tokens x
// its G q heads, 16 per wave) over a range of positions, 32 at a time, in two
// LDS buffers that rows enter without passing through registers (16-byte pieces
// in an order that spreads a column over the banks).  Spinor code rows keep the
// per-token kernel: their codec turns another order of the sums into other codes.
//
// Scores are formed transposed, S^T = K Q^T: lane l then holds token-head l % 16
// and positions 4 (l / 16) + i -- the A operand of the V product, so the weights
// go from the softmax into the second product without leaving their registers.
// Softmax is online (running maximum and sum per token-head), as the decode
// kernel's merge of chunks; workgroups of one token tile split the positions
// where tiles x kv heads leave CUs idle, and k_pfloat_merge joins the parts.
//
// The per-token kernel (k_attn_float with a token grid) streamed the whole span
// once per token: 870 us for 128 tokens at 8 192 positions (Qwen3-8B shape).
#include "kvd_internal.h"
#include "kvd_vec.h"
#include "kvd_spinor.h"
#include "kvd_pass.h"
#include <algorithm>

namespace kvd {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int PF_WAVES = 8, PF_ROWS = 16 * PF_WAVES;   // token-heads per workgroup
constexpr int PF_POS = 32;                             // positions per tile (within one page)

__device__ __forceinline__ bool finite4(const v4f &v) {
    const v4i b = __builtin_bit_cast(v4i, v) & 0x7F800000;
    return b.x != 0x7F800000 && b.y != 0x7F800000 && b.z != 0x7F800000 && b.w != 0x7F800000;
}

}  // namespace

// grid: (kv heads, token tiles, position splits); with 8 kv heads each XCD
// (workgroups go to the 8 of them in turn) reads one head's rows
template <int EPL, int G>
__global__ __launch_bounds__(64 * PF_WAVES, 2) void k_pfloat(AttnArgs a, int nsplit) {
    constexpr int HD = EPL * 64, CPR = HD / 16, TOK = PF_ROWS / G;     // CPR: 16-float groups of a row
    constexpr int PIECES = PF_POS * HD / 4;                            // 16-byte pieces of a K or V tile
    __shared__ __align__(1024) v4f kv[2][2][PIECES];                   // [buffer][K, V][position][piece ^ position % 16]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, g = lane >> 4, h = blockIdx.x;
    const int t0 = (int)blockIdx.y * TOK, tend = t0 + TOK < a.nt ? t0 + TOK : a.nt;
    // this split's tiles of the token tile's span [start, last]
    const int last = a.pos0 + tend - 1, lo = win_start(a, t0) / PF_POS, hi = last / PF_POS + 1;
    const int per = (hi - lo + nsplit - 1) / nsplit, b0 = lo + (int)blockIdx.z * per, b1 = b0 + per < hi ? b0 + per : hi;
    // this lane's token-head, and the wave's token range
    const int row = wave * 16 + l16, tq = t0 + row / G, head = h * G + row % G;
    const bool live = tq < tend;
    const int wt0 = t0 + wave * 16 / G, wt1 = t0 + (wave * 16 + 15) / G < tend ? t0 + (wave * 16 + 15) / G : tend - 1;
    const int my_lo = win_start(a, tq), my_hi = live ? a.pos0 + tq : -1;     // positions this token-head attends
    const int w_lo = win_start(a, wt0), w_hi = a.pos0 + wt1;                 // ... any of the wave's
    const int w_lo1 = win_start(a, wt1), w_hi0 = a.pos0 + wt0;               // ... all of them
    const bool wlive = wt0 < tend;
    const size_t QD = (size_t)a.NH * HD;
    v4f Q[CPR];                                                        // dims 16 s + 4 g ..
    {
        const float *qp = a.qr + (size_t)(live ? tq : t0) * QD + (size_t)head * HD + 4 * g;
        #pragma unroll
        for (int s = 0; s < CPR; s++) Q[s] = *(const v4f *)(qp + 16 * s);
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) v4f *)&kv[0][0][0];
    // K and V of a tile into LDS buffer buf: piece i = position p, 16 bytes c ^
    // (p % 16); rows past the batch's last position repeat it
    auto load = [&](int tile, int buf) {
        constexpr int N = PIECES / 64 / PF_WAVES;      // 1 KiB loads per wave of K, and of V
        const uint8_t *page = (const uint8_t *)page_at(a, __builtin_amdgcn_readfirstlane(tile * PF_POS));
        const int lp = last - tile * PF_POS, q0 = (tile * PF_POS) & (PAGE - 1);
        #pragma unroll
        for (int v = 0; v < 2; v++) {
            const v4i rs = rsrc_of(page + ((size_t)v * a.NKV + h) * PAGE * HD * 4, PAGE * HD * 4);
            #pragma unroll
            for (int k = 0; k < N; k++) {
                const int i = (wave * N + k) * 64 + lane, p = i / (HD / 4), c = (i % (HD / 4)) ^ (p & 15);
                dma16(lds0 + (uint32_t)(((buf * 2 + v) * PIECES + (wave * N + k) * 64) * 16), (q0 + (p < lp ? p : lp)) * HD * 4 + 16 * c, rs);
            }
        }
    };
    // this lane's operand places in a tile, up to constants: K piece 4 s + g of
    // position l % 16 (+ 16), V piece 16 u + l % 16 of position 4 g + e (+ 16)
    int kb[4], vb[4];
    #pragma unroll
    for (int e = 0; e < 4; e++) {
        kb[e] = l16 * (HD / 4) + ((4 * e + g) ^ l16);
        vb[e] = (4 * g + e) * (HD / 4) + (l16 ^ (4 * g + e));
    }
    v4f O[CPR];                                                        // column 64 u + 4 (l % 16) + w of rows 4 g + i: O[4 u + w][i]
    #pragma unroll
    for (int s = 0; s < CPR; s++) O[s] = (v4f){0, 0, 0, 0};
    float m = -INFINITY, l = 0.0f;                                     // of this lane's token-head
    if (b0 < b1) load(b0, 0);
    for (int tile = b0; tile < b1; tile++) {
        const int buf = (tile - b0) & 1;
        // this tile has arrived for every wave, and nobody reads the other buffer
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
        if (tile + 1 < b1) load(tile + 1, buf ^ 1);
        const int p0 = tile * PF_POS;
        if (wlive && p0 <= w_hi && p0 + PF_POS > w_lo) {
            const v4f *K = kv[buf][0], *V = kv[buf][1];
            const bool whole = p0 >= w_lo1 && p0 + PF_POS - 1 <= w_hi0 && wt0 + 15 / G < tend;
            v4f S[2];
            #pragma unroll
            for (int s2 = 0; s2 < 2; s2++) S[s2] = (v4f){0, 0, 0, 0};
            #pragma unroll
            for (int s = 0; s < CPR; s++) {
                v4f kx[2];
                #pragma unroll
                for (int s2 = 0; s2 < 2; s2++) kx[s2] = K[kb[s & 3] + 16 * (s >> 2) + 4 * HD * s2];
                #pragma unroll
                for (int e = 0; e < 4; e++)
                    #pragma unroll
                    for (int s2 = 0; s2 < 2; s2++) S[s2] = __builtin_amdgcn_mfma_f32_16x16x4f32(kx[s2][e], Q[s][e], S[s2], 0, 0, 0);
                // few reads ahead at a time (all at once they would spill at head_dim 256)
                if (EPL == 4 && s % 2) __builtin_amdgcn_sched_barrier(0);
            }
            float mx = -INFINITY;
            #pragma unroll
            for (int s2 = 0; s2 < 2; s2++)
                #pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int p = p0 + 16 * s2 + 4 * g + i;
                    S[s2][i] = p >= my_lo && p <= my_hi ? S[s2][i] * a.ascale : -INFINITY;
                    mx = fmaxf(mx, S[s2][i]);
                }
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float mn = fmaxf(m, mx), ms = mn == -INFINITY ? 0.0f : mn;   // no position yet: weights 0
            const float al = expf(m - ms);
            float sum = 0.0f;
            #pragma unroll
            for (int s2 = 0; s2 < 2; s2++)
                #pragma unroll
                for (int i = 0; i < 4; i++) { S[s2][i] = expf(S[s2][i] - ms); sum += S[s2][i]; }
            sum += __shfl_xor(sum, 16, 64);
            sum += __shfl_xor(sum, 32, 64);
            l = l * al + sum;
            m = mn;
            if (__any(al != 1.0f)) {                                   // O's rows are 4 g + i
                #pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float f = __shfl(al, 4 * g + i, 64);
                    #pragma unroll
                    for (int s = 0; s < CPR; s++) O[s][i] *= f;
                }
            }
            // a masked position's weight is 0, which a V row that is not finite
            // would turn into NaN: such tiles add their positions one by one
            bool bad = false;
            if (!whole)
                for (int i = lane; i < PIECES; i += 64) bad |= !finite4(V[i]);
            if (__any(bad)) {
                for (int p = 0; p < PF_POS; p++) {
                    #pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int src = 16 * ((p & 15) >> 2) + 4 * g + i;
                        const v4f sv = S[0], sw = S[1];
                        float w = 0.0f;
                        #pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const float x = __shfl(p < 16 ? sv[e] : sw[e], src, 64);
                            if (e == (p & 3)) w = x;
                        }
                        const int lo_i = __shfl(my_lo, 4 * g + i, 64), hi_i = __shfl(my_hi, 4 * g + i, 64);
                        if (p0 + p >= lo_i && p0 + p <= hi_i) {
                            #pragma unroll
                            for (int u = 0; u < HD / 64; u++) {
                                const v4f x = V[p * (HD / 4) + ((16 * u + l16) ^ (p & 15))];
                                #pragma unroll
                                for (int e = 0; e < 4; e++) O[4 * u + e][i] += w * x[e];
                            }
                        }
                    }
                }
            } else {
                #pragma unroll
                for (int s2 = 0; s2 < 2; s2++)
                    #pragma unroll
                    for (int e = 0; e < 4; e++) {
                        #pragma unroll
                        for (int u = 0; u < HD / 64; u++) {
                            const v4f x = V[vb[e] + 16 * u + 4 * HD * s2];
                            #pragma unroll
                            for (int w = 0; w < 4; w++) O[4 * u + w] = __builtin_amdgcn_mfma_f32_16x16x4f32(S[s2][e], x[w], O[4 * u + w], 0, 0, 0);
                        }
                        if (EPL == 4 && e % 2) __builtin_amdgcn_sched_barrier(0);
                    }
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    // rows 4 g + i of the wave: one part of nsplit, or the result
    #pragma unroll
    for (int i = 0; i < 4; i++) {
        const int r = wave * 16 + 4 * g + i, t = t0 + r / G, hd = h * G + r % G;
        const float lr = __shfl(l, 4 * g + i, 64), mr = __shfl(m, 4 * g + i, 64);
        if (t >= tend) continue;
        const size_t at = ((size_t)t * a.NH + hd) * nsplit + blockIdx.z;
        float *out = nsplit > 1 ? a.part + at * HD : a.ao + (size_t)t * QD + (size_t)hd * HD;
        #pragma unroll
        for (int u = 0; u < HD / 64; u++) {
            v4f x = {O[4 * u][i], O[4 * u + 1][i], O[4 * u + 2][i], O[4 * u + 3][i]};
            if (nsplit == 1) x /= lr;
            *(v4f *)(out + 64 * u + 4 * l16) = x;
        }
        __builtin_amdgcn_sched_barrier(0);
        if (nsplit > 1 && l16 == 0) { a.part_ml[2 * at] = mr; a.part_ml[2 * at + 1] = lr; }
    }
}

// out = sum_c e^(m_c - M) O_c / sum_c e^(m_c - M) l_c; grid (tokens x q heads), HD threads
__global__ __launch_bounds__(256) void k_pfloat_merge(AttnArgs a, int nsplit) {
    const size_t at = blockIdx.x;
    const float *ml = a.part_ml + 2 * at * nsplit, *po = a.part + at * nsplit * a.HD;
    float M = -INFINITY;
    for (int c = 0; c < nsplit; c++) M = fmaxf(M, ml[2 * c]);
    float L = 0.0f, o = 0.0f;
    for (int c = 0; c < nsplit; c++) {
        if (ml[2 * c] == -INFINITY) continue;          // a part without a position of this token
        const float w = expf(ml[2 * c] - M);
        L += w * ml[2 * c + 1];
        o += w * po[(size_t)c * a.HD + threadIdx.x];
    }
    a.ao[at * a.HD + threadIdx.x] = o / L;
}

template <int EPL, int G>
static void pfloat_go(const AttnArgs &a, hipStream_t s) {
    constexpr int TOK = PF_ROWS / G;
    const int tiles = (a.nt + TOK - 1) / TOK;
    // splits: two workgroups' worth of positions per CU, at least two tiles
    // each, as many as the parts' buffers hold.  They are cut by this launch's
    // tokens, so another cut of the same prompt adds its float sums in another
    // order (up to 2e-6 of K, V and logits).
    const int span = (a.pos0 + a.nt - 1) / PF_POS - win_start(a, a.nt > TOK ? a.nt - TOK : 0) / PF_POS + 1;
    const int room = std::min(a.part_slots / a.nt, 64);
    int n = (512 + tiles * a.NKV - 1) / (tiles * a.NKV);
    n = std::max(1, std::min(std::min(n, span / 2), room));
    const dim3 grid(a.NKV, tiles, n), wg(64 * PF_WAVES);
    hipLaunchKernelGGL((k_pfloat<EPL, G>), grid, wg, 0, s, a, n);
    if (n > 1) hipLaunchKernelGGL(k_pfloat_merge, dim3(a.nt * a.NH), dim3(a.HD), 0, s, a, n);
}

bool prefill_attention_float(const AttnArgs &a) {
    const int G = a.NH / a.NKV;
    return a.mode == FLOAT && a.kvc == KVC_PLAIN && a.nt > 0 && !a.tpages && !a.tpos && a.part_slots > 0 &&
           (a.HD == 64 || a.HD == 128 || a.HD == 256) && (G == 2 || G == 4);
}

void launch_prefill_float(const AttnArgs &a, hipStream_t s) {
    const int G = a.NH / a.NKV;
    if (!prefill_attention_float(a)) return launch_fail("float prefill attention: arguments outside the kernel's limits");
    if (a.HD == 256 && G == 2) pfloat_go<4, 2>(a, s);
    else if (a.HD == 256) pfloat_go<4, 4>(a, s);
    else if (a.HD == 128 && G == 2) pfloat_go<2, 2>(a, s);
    else if (a.HD == 128) pfloat_go<2, 4>(a, s);
    else if (G == 2) pfloat_go<1, 2>(a, s);
    else pfloat_go<1, 4>(a, s);
}

}  // namespace kvd
