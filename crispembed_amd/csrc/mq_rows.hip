// mq_rows.hip -- the layers of a Q8_0 BERT encoder for a few rows (one query, a short batch).
//
// A few dozen rows are bound by neither memory nor arithmetic but by the chain of dependent
// launches: the GEMM path takes seven or eight a layer and the GEMV path seventeen, at 4-8 us
// each on MI355X however little they do.  Here a layer is five:
//   qkv        [residual + LN2 of the layer before,] quantize, product
//   attention  storing its rows quantized
//   o          product of those
//   fc1        residual + LN1, quantize, product, GELU-erf, storing its rows quantized
//   fc2        product of those
// A LayerNorm needs whole rows, so the workgroups of a row tile (one per 32 output columns) each
// form and quantize the tile's rows for themselves, while their weights are in flight; what a
// workgroup can quantize for the next kernel (its 32 columns are one Q8_0 block of each row) it
// does in its store.  Every value rounds as on the general path (mq_gemv.hip, mq_gemm.hip,
// mq_encoder.hip, mq_quant.hip), whose results these layers give bit for bit: a quantized encoder
// turns one other rounding of an activation, 1e-7, into 1e-3 of its output wherever that moves an
// 8-bit value.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "mq_internal.h"
#include "mq_act.h"
#include "mq_q8k.h"
#include "mq_rows.h"
#include "mq_wave.h"

namespace mq {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));

// what a wave's lanes wrote to its own LDS is there for its other lanes
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One value of 32 lanes (a half wave) as a Q8_0 block of row `row` and chunk kc of a GEMM-layout
// activation; l32 the value's place in the block
__device__ __forceinline__ void rows_store_q8_0(float x, int8_t *qo, float *qd, int kch, int64_t m_pad, int64_t row,
                                                int kc, int l32, int variant, bool live) {
    float amax = max8(fabsf(x));
    amax = fmaxf(amax, dpp_f<0x140>(amax));
    amax = fmaxf(amax, __shfl_xor(amax, 16));
    float d, id;
    q8_0_scale(amax, variant, d, id);
    if (live) {
        qo[(((row >> 5) * kch + kc) << 10) + ((((l32 >> 4) << 5) + (row & 31)) << 4) + (l32 & 15)] =
            (int8_t)q8_0_quant(x, id, variant);
        if (l32 == 0) qd[kc * m_pad + row] = d;
    }
}

// rows_tree<KP, I, S>: the sum of steps I, I + S, I + 2 S, ... < min(KP, 8), as the GEMV's lanes meet
// (a step that is not there is +0 in the GEMV, and no step's sum is -0: it drops out)
template <int KP, int I, int S, class F>
__device__ __forceinline__ v16f rows_tree(F &&leaf) {
    if constexpr (S == 8) {
        return leaf(std::integral_constant<int, I>{});
    } else {
        v16f t = rows_tree<KP, I, 2 * S>(leaf);
        if constexpr (I + S < (KP < 8 ? KP : 8)) t += rows_tree<KP, I + S, 2 * S>(leaf);
        return t;
    }
}

// The few-row product.  8 waves; wave w multiplies the 32-value blocks w, w + 8, ... of K (one
// v_mfma_i32_32x32x32_i8 and a scaled add each), and the eight partial tiles meet in LDS.  The sums
// are the GEMV's, in its order, so the results are its results bit for bit: there lane l of a wave
// adds up blocks l and l + 64 and the lanes meet in a tree over lane ^ 32, 16, 8, 4, 2, 1; here block
// l = w + 8 i is step i of wave w, so the tree's first three levels join steps i ^ 4, 2, 1 of a wave
// and the last three join waves w ^ 4, 2, 1.
// PRO: the rows.  ROWS_Q: quantized already (GEMM layout), fragments straight to registers.
// ROWS_F32, ROWS_LN: wave w forms rows w, w + 8, w + 16, w + 24 (lane l values 256 p + 4 l .. + 3, p < KP =
// ceil(K / 256)), as they are or as layer_norm(x + res), quantizes them and leaves them in LDS
// as fragments; the first column tile's workgroups store the normed rows to xout (neither x nor
// res: the other workgroups still read those).  Rows past M are skipped: their fragment bytes are
// whatever LDS holds, and so are output rows that are never stored.
// RQ: the output, after GELU, leaves as the Q8_0 activation of the next product.
template <int KP, int PRO, bool RQ>
__global__ __launch_bounds__(512) void k_rows(const RowsArgs a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int l32 = lane & 31, half = lane >> 5;
    const int n0 = blockIdx.x * 32, m0 = blockIdx.y * 32;
    const int nblk = a.K >> 5;
    char *frag = smem;                                   // nblk fragments of 1 KB
    float *sd = (float *)(smem + ((size_t)nblk << 10));  // nblk x 32 row scales

    v4i wf[KP], af[KP];
    float dw[KP], dx[KP];
    auto weights = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < KP; i++) {
            const int kc = min(wave + 8 * i, nblk - 1);
            wf[i] = *(const v4i *)(a.wq + (((int64_t)blockIdx.x * a.kch + kc) << 10) + lane * 16);
            dw[i] = a.wd[(int64_t)kc * a.n_pad + n0 + l32];
        }
    };
    if constexpr (PRO == ROWS_Q) {
#pragma unroll
        for (int i = 0; i < KP; i++) {
            const int kc = min(wave + 8 * i, nblk - 1);
            af[i] = *(const v4i *)(a.xq + (((int64_t)blockIdx.y * a.kch + kc) << 10) + lane * 16);
            dx[i] = a.xd[(int64_t)kc * a.m_pad + m0 + l32];
        }
        weights();
    } else {
        const int nr = min((a.M - m0 - wave + 7) >> 3, 4);  // live rows of this wave
        if (nr > 0) {
            float4 v[4][KP], res[4][KP], lw[KP], lb[KP];
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int p = 0; p < KP; p++) {
                    const int c = 256 * p + 4 * lane;
                    const int64_t row = m0 + wave + 8 * min(r, nr - 1);
                    v[r][p] = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (c < a.K) v[r][p] = *(const float4 *)(a.x + row * a.K + c);
                    if constexpr (PRO == ROWS_LN) {
                        res[r][p] = make_float4(0.f, 0.f, 0.f, 0.f);
                        if (c < a.K) res[r][p] = *(const float4 *)(a.res + row * a.K + c);
                    }
                }
            if constexpr (PRO == ROWS_LN)
#pragma unroll
                for (int p = 0; p < KP; p++) {
                    const int c = 256 * p + 4 * lane;
                    lw[p] = lb[p] = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (c < a.K) lw[p] = *(const float4 *)(a.lw + c), lb[p] = *(const float4 *)(a.lb + c);
                }
            weights();
            if constexpr (PRO == ROWS_LN) {
                // x + res here holds 4 values of a column step a lane, the statistics sum lane by
                // lane over columns 64 apart (ln_stats): RB rows at a time change hands through LDS
                constexpr int RB = KP <= 2 ? 4 : 2, V = 4 * KP;
                float *xr = (float *)(smem + (size_t)nblk * (1024 + 128)) + wave * RB * a.K;
#pragma unroll
                for (int r0 = 0; r0 < 4; r0 += RB) {
#pragma unroll
                    for (int r = r0; r < r0 + RB; r++) {
                        if (r >= nr) continue;  // uniform
#pragma unroll
                        for (int p = 0; p < KP; p++) {
                            float4 &t = v[r][p];
                            const float4 u = res[r][p];
                            t.x = u.x + t.x, t.y = u.y + t.y, t.z = u.z + t.z, t.w = u.w + t.w;
                            const int c = 256 * p + 4 * lane;
                            if (c < a.K) *(float4 *)(xr + (r - r0) * a.K + c) = t;
                        }
                    }
                    wave_lds_sync();
#pragma unroll
                    for (int r = r0; r < r0 + RB; r++) {
                        if (r >= nr) continue;
                        float t[V], mean, rstd;
#pragma unroll
                        for (int e = 0; e < V; e++) t[e] = lane + 64 * e < a.K ? xr[(r - r0) * a.K + lane + 64 * e] : 0.f;
                        ln_stats(t, a.K, lane, a.eps, mean, rstd);
#pragma unroll
                        for (int p = 0; p < KP; p++) {
                            float4 &x = v[r][p];
                            x.x = ln_value(x.x, mean, rstd, lw[p].x, lb[p].x), x.y = ln_value(x.y, mean, rstd, lw[p].y, lb[p].y);
                            x.z = ln_value(x.z, mean, rstd, lw[p].z, lb[p].z), x.w = ln_value(x.w, mean, rstd, lw[p].w, lb[p].w);
                            const int c = 256 * p + 4 * lane;
                            if (blockIdx.x == 0 && c < a.K)
                                *(float4 *)(a.xout + (int64_t)(m0 + wave + 8 * r) * a.K + c) = x;
                        }
                    }
                    wave_lds_sync();
                }
            }
            float am[4 * KP];
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int p = 0; p < KP; p++) {
                    const float4 t = v[r][p];
                    am[4 * p + r] = max8(fmaxf(fmaxf(fabsf(t.x), fabsf(t.y)), fmaxf(fabsf(t.z), fabsf(t.w))));
                }
            // the 8-lane groups hold one block each of every (r, p); lane g of a group divides for
            // block g of eight
            const int sub = lane & 7;
#pragma unroll
            for (int g0 = 0; g0 < 4 * KP; g0 += 8) {
                float mine = am[g0];
#pragma unroll
                for (int g = 1; g < 8; g++) mine = sub == g ? am[g0 + g] : mine;
                float d, id;
                q8_0_scale(mine, a.variant, d, id);
                const int pd = (g0 + sub) >> 2, kd = 8 * pd + (lane >> 3);
                if (kd < nblk) sd[kd * 32 + wave + 8 * (sub & 3)] = d;
#pragma unroll
                for (int g = 0; g < 8; g++) {
                    const int r = g & 3, p = (g0 + g) >> 2, kc = 8 * p + (lane >> 3), w0 = 4 * sub;
                    if (r >= nr) continue;  // uniform
                    const float ig = __shfl(id, (lane & 56) + g);
                    const float4 t = v[r][p];
                    const uint32_t q = pack4_i8(q8_0_quant(t.x, ig, a.variant), q8_0_quant(t.y, ig, a.variant),
                                                q8_0_quant(t.z, ig, a.variant), q8_0_quant(t.w, ig, a.variant));
                    if (kc < nblk)
                        *(uint32_t *)(frag + (kc << 10) + (((w0 >> 4) << 5) + wave + 8 * r) * 16 + (w0 & 15)) = q;
                }
            }
        } else {
            weights();
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < KP; i++) {
            const int kc = min(wave + 8 * i, nblk - 1);
            af[i] = *(const v4i *)(frag + (kc << 10) + lane * 16);
            dx[i] = sd[kc * 32 + l32];
        }
    }

    // steps i and i + 8: the exact dot times the exact product of the two fp16 scales
    auto leaf = [&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        v16f t = (v16f){};
#pragma unroll
        for (int u = i; u < KP; u += 8)
            if (wave + 8 * u < nblk) {  // uniform
                const v16i I = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[u], wf[u], (v16i){}, 0, 0, 0);
                // the tile of d_x d_w, a rank-1 product
                const v16f P = __builtin_amdgcn_mfma_f32_32x32x2f32(half ? 0.f : dx[u], half ? 0.f : dw[u], (v16f){}, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; r++) t[r] = __builtin_fmaf((float)I[r], P[r], t[r]);
            }
        return t;
    };
    const v16f acc = rows_tree<KP, 0, 1>(leaf);
    if constexpr (PRO != ROWS_Q) __syncthreads();  // the fragments' space takes the partial tiles
    float *part = (float *)smem;
#pragma unroll
    for (int r = 0; r < 16; r++) part[(wave * 16 + r) * 64 + lane] = acc[r];
    const int col = n0 + l32;
    const float bias = a.bias && col < a.N ? a.bias[col] : 0.f;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int r = 2 * wave + u, row = m0 + 8 * (r / 4) + 4 * half + r % 4;
        float w[8];
#pragma unroll
        for (int v = 0; v < 8; v++) w[v] = part[(v * 16 + r) * 64 + lane];
        float s = ((w[0] + w[4]) + (w[2] + w[6])) + ((w[1] + w[5]) + (w[3] + w[7]));
        if (a.bias) s += bias;
        if constexpr (RQ) {
            rows_store_q8_0(gelu_erf_f32(s), a.qo, a.qd, a.q_kch, a.q_m_pad, row, blockIdx.x, l32, a.variant, row < a.M);
        } else {
            if (row < a.M && col < a.N) a.y[(int64_t)row * a.ldy + col] = s;
        }
    }
}

// The FFN-down product of 9 - 32 rows, which the general path gives to the GEMM: its sums, bit for bit
// (the K-group form's: group g of four adds up blocks g, g + 4, ... in turn, the groups meet in
// order, then the bias).  4 waves, wave g the group, over quantized rows; a round of PF blocks in
// flight while the one before is summed.  What bounds it is its chain of K / 128 dependent steps and
// the launch: 384 x 1536 at 16 rows 5.8 us (the GEMM 7.6; the eight-wave tree, other sums, 4.7).
__global__ __launch_bounds__(256) void k_rows_groups(const RowsArgs a) {
    constexpr int PF = 12;
    __shared__ float part[4][16][64];
    const int g = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int l32 = lane & 31, half = lane >> 5;
    const int n0 = blockIdx.x * 32, m0 = blockIdx.y * 32;
    const int nblk = a.K >> 5;
    struct Step {
        v4i w, x;
        float dw, dx;
    } ra[PF], rb[PF];
    auto load = [&](Step (&s)[PF], int kc0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PF; i++) {
            const int kc = min(kc0 + 4 * i, nblk - 1);
            s[i].w = *(const v4i *)(a.wq + (((int64_t)blockIdx.x * a.kch + kc) << 10) + lane * 16);
            s[i].x = *(const v4i *)(a.xq + (((int64_t)blockIdx.y * a.kch + kc) << 10) + lane * 16);
            s[i].dw = a.wd[(int64_t)kc * a.n_pad + n0 + l32];
            s[i].dx = a.xd[(int64_t)kc * a.m_pad + m0 + l32];
        }
    };
    v16f acc = (v16f){};
    auto compute = [&](const Step (&s)[PF], int kc0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PF; i++)
            if (kc0 + 4 * i < nblk) {  // uniform
                const v16i I = __builtin_amdgcn_mfma_i32_32x32x32_i8(s[i].x, s[i].w, (v16i){}, 0, 0, 0);
                const v16f P = __builtin_amdgcn_mfma_f32_32x32x2f32(half ? 0.f : s[i].dx, half ? 0.f : s[i].dw, (v16f){}, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; r++) acc[r] = __builtin_fmaf((float)I[r], P[r], acc[r]);
            }
    };
    constexpr int D = 4 * PF;  // blocks a round
    load(ra, g);
    for (int kc0 = g; kc0 < nblk; kc0 += 2 * D) {
        if (kc0 + D < nblk) load(rb, kc0 + D);
        compute(ra, kc0);
        if (kc0 + 2 * D < nblk) load(ra, kc0 + 2 * D);
        if (kc0 + D < nblk) compute(rb, kc0 + D);
    }
#pragma unroll
    for (int r = 0; r < 16; r++) part[g][r][lane] = acc[r];
    const int col = n0 + l32;
    const float bias = a.bias && col < a.N ? a.bias[col] : 0.f;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int r = 4 * g + u, row = m0 + 8 * g + 4 * half + u;
        float s = ((part[0][r][lane] + part[1][r][lane]) + part[2][r][lane]) + part[3][r][lane];
        if (a.bias) s += bias;
        if (row < a.M && col < a.N) a.y[(int64_t)row * a.ldy + col] = s;
    }
}

// Attention of one (sequence, head) of at most ROWS_MAX_T tokens: k_attention's values bit for bit
// (its key ranges, key blocks and order of sums), with a wave per query row instead of a thread.
// q (scaled), k, v (bias added) go to LDS; lane j takes key j: score, largest score so far of its key
// range, probability; then lane d takes head dim d (and d + 64 at HD 128, which k_attention does
// not have) and sums the ranges side by side.  At HD 32 the two lane halves take half of the ranges
// each.  The rows leave as the Q8_0 activation of the o product (32 head dims a block).
template <int HD, int KS>
__global__ __launch_bounds__(1024) void k_rows_attn(const float *__restrict__ qkv, int8_t *__restrict__ qo,
                                                    float *__restrict__ qd, int kch, int64_t m_pad, int variant, int T,
                                                    int H, int nh, float scale) {
    constexpr int ST = HD + 4;  // row stride: float4 reads of 8 consecutive rows hit all banks
    constexpr int NG = HD == 32 && KS > 1 ? 2 : 1, NR = KS / NG;  // lane groups, ranges a lane
    constexpr int DL = HD > 64 ? HD / 64 : 1;                            // dims a lane
    extern __shared__ __attribute__((aligned(16))) float sm[];
    float *Q = sm, *K = Q + T * ST, *V = K + T * ST;
    __shared__ float ps[16][ROWS_MAX_T], ms[16][4];  // scores, then probabilities; maxima of ranges or blocks
    const int b = blockIdx.x / nh, h = blockIdx.x % nh;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const float *base = qkv + (int64_t)b * T * 3 * H + h * HD;
    for (int e = threadIdx.x; e < 3 * T * (HD / 4); e += 1024) {
        const int d4 = e % (HD / 4), rest = e / (HD / 4), t = rest % T, w = rest / T;
        float4 x = *(const float4 *)(base + (int64_t)t * 3 * H + w * H + 4 * d4);
        if (w == 0) x = make_float4(x.x * scale, x.y * scale, x.z * scale, x.w * scale);
        *(float4 *)(Q + (w * T + t) * ST + 4 * d4) = x;
    }
    __syncthreads();
    const int span = T / KS;                             // keys a range
    const int jr = min(lane, T - 1) / span, j0 = jr * span;  // this lane's range and its first key
    const int jb = (min(lane, T - 1) - j0) / ATT_KB;      // and its block in the range
    const int d0 = lane % (HD < 64 ? HD : 64), g = NG > 1 ? lane / HD : 0;
    for (int i = wave; i < T; i += 16) {
        float s = 0.f;
        if (lane < T) {
#pragma unroll
            for (int d4 = 0; d4 < HD / 4; d4++)
                s = score4(s, *(const float4 *)(Q + i * ST + 4 * d4), *(const float4 *)(K + lane * ST + 4 * d4));
            ps[wave][lane] = s;
        }
        wave_lds_sync();
        float mx = -INFINITY;
        const int j1 = min(j0 + ATT_KB * (jb + 1), j0 + span);
        for (int c = j0; c < j1; c += 4)  // four reads in flight, the last key again past the end
#pragma unroll
            for (int u = 0; u < 4; u++) mx = fmaxf(mx, ps[wave][min(c + u, j1 - 1)]);
        wave_lds_sync();
        if (lane < T) {
            ps[wave][lane] = expf(s - mx);
            if (lane == j1 - 1) ms[wave][KS == 1 ? jb : jr] = mx;
        }
        wave_lds_sync();
        float l[KS], o[KS][DL], m[KS];
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int k0 = (g * NR + r) * span;
            l[r] = 0.f;
#pragma unroll
            for (int n = 0; n < DL; n++) o[r][n] = 0.f;
            m[r] = ms[wave][g * NR + r];
            for (int c = 0; c < span; c += 4) {
                if constexpr (KS == 1)  // one range of up to two blocks: the second rescales
                    if (c == ATT_KB) {
                        const float corr = expf(m[0] - ms[wave][1]);
                        m[0] = ms[wave][1];
                        l[0] *= corr;
#pragma unroll
                        for (int n = 0; n < DL; n++) o[0][n] *= corr;
                    }
                float p[4], v[4][DL];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int j = k0 + min(c + u, span - 1);
                    p[u] = ps[wave][j];
#pragma unroll
                    for (int n = 0; n < DL; n++) v[u][n] = V[j * ST + d0 + 64 * n];
                }
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const bool in = c + u < span;
                    l[r] = in ? l[r] + p[u] : l[r];
#pragma unroll
                    for (int n = 0; n < DL; n++) o[r][n] = in ? __builtin_fmaf(p[u], v[u][n], o[r][n]) : o[r][n];
                }
            }
        }
        if constexpr (NG > 1)
#pragma unroll
            for (int r = 0; r < NR; r++) {
                l[NR + r] = __shfl_xor(l[r], 32), o[NR + r][0] = __shfl_xor(o[r][0], 32), m[NR + r] = __shfl_xor(m[r], 32);
            }
        float lt = l[0];
        float (&ot)[DL] = o[0];
        if constexpr (KS > 1) {  // lanes of the other half (g = 1) compute values that are not stored
            float mt = m[0];
#pragma unroll
            for (int k = 1; k < KS; k++) mt = fmaxf(mt, m[k]);
            const float w0 = expf(m[0] - mt);
#pragma unroll
            for (int k = 1; k < KS; k++) {
                const float w = expf(m[k] - mt);
                lt = k == 1 ? __builtin_fmaf(lt, w0, l[k] * w) : __builtin_fmaf(l[k], w, lt);
#pragma unroll
                for (int n = 0; n < DL; n++)
                    ot[n] = k == 1 ? __builtin_fmaf(ot[n], w0, o[k][n] * w) : __builtin_fmaf(o[k][n], w, ot[n]);
            }
        }
        const float inv = 1.0f / lt;
#pragma unroll
        for (int n = 0; n < DL; n++)
            rows_store_q8_0(ot[n] * inv, qo, qd, kch, m_pad, (int64_t)b * T + i, (h * HD + d0 + 64 * n) >> 5, lane & 31,
                            variant, lane < HD);
        wave_lds_sync();
    }
}

template <int KP, int PRO, bool RQ = false>
static hipError_t rows_cfg(const RowsArgs &a, hipStream_t s) {
    // fragments and row scales, the LayerNorm's rows of each wave; then the partial tiles
    constexpr int RB = KP <= 2 ? 4 : 2;
    const size_t op = (PRO == ROWS_Q ? 0 : (size_t)(a.K / 32) * (1024 + 128)) + (PRO == ROWS_LN ? (size_t)8 * RB * a.K * 4 : 0);
    const size_t lds = op > 32768 ? op : 32768;
    if constexpr (PRO == ROWS_LN) {
        static std::atomic<bool> attr_set[MQ_MAX_DEVICES];
        constexpr int most = KP * 8 * (1024 + 128) + 8 * RB * KP * 256 * 4;
        static_assert(most <= 160 * 1024, "LDS budget");
        const hipError_t e = dyn_lds_once((const void *)k_rows<KP, PRO, RQ>, most, attr_set);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_rows<KP, PRO, RQ>), dim3((unsigned)((a.N + 31) / 32), (unsigned)((a.M + 31) / 32)), dim3(512), lds,
                       s, a);
    return hipGetLastError();
}

hipError_t launch_rows(const void *image, int64_t n, int64_t k, RowsArgs a, void *q_out, hipStream_t s) {
    if (a.M <= 0) return hipSuccess;
    const WeightPlanes p = weight_planes(MQ_TYPE_Q8_0, n, k);
    a.wq = (const int8_t *)image + p.tq;
    a.wd = (const float *)((const char *)image + p.tdw);
    a.n_pad = (int)p.n_pad;
    a.kch = (int)(p.kb_pad / 32);
    a.N = (int)n, a.K = (int)k;
    if (k % 32 || k > ROWS_MAX_K) return hipErrorInvalidValue;
    if (q_out) {
        if (n % 32) return hipErrorInvalidValue;
        const ActPlanes o = act_planes(MQ_TYPE_Q8_0, a.M, n, true);
        a.qo = (int8_t *)q_out + o.xq, a.qd = (float *)((char *)q_out + o.xd);
        a.q_kch = (int)(o.kb_pad / 32), a.q_m_pad = o.m_pad;
    }
    if (a.x_ws) {
        const ActPlanes x = act_planes(MQ_TYPE_Q8_0, a.M, k, true);
        a.xq = (const int8_t *)a.x_ws + x.xq, a.xd = (const float *)((const char *)a.x_ws + x.xd);
        a.m_pad = x.m_pad;
        if (a.qo) return hipErrorInvalidValue;
        // steps a wave: each one that is not there still costs its (clamped) loads
        if (k <= 512) return rows_cfg<2, ROWS_Q>(a, s);
        if (k <= 1024) return rows_cfg<4, ROWS_Q>(a, s);
        if (k <= 1536) return rows_cfg<6, ROWS_Q>(a, s);
        if (k <= 2048) return rows_cfg<8, ROWS_Q>(a, s);
        if (k <= 3072) return rows_cfg<12, ROWS_Q>(a, s);
        return rows_cfg<16, ROWS_Q>(a, s);
    }
    if (k > ROWS_MAX_LN || (a.res && (!a.xout || a.xout == a.res || a.xout == a.x)) ||
        ((uintptr_t)a.x | (uintptr_t)a.res | (uintptr_t)a.lw | (uintptr_t)a.lb | (uintptr_t)a.xout) % 16)
        return hipErrorInvalidValue;
    if (a.res && a.qo) return k <= 512 ? rows_cfg<2, ROWS_LN, true>(a, s) : rows_cfg<4, ROWS_LN, true>(a, s);
    if (a.res) return k <= 512 ? rows_cfg<2, ROWS_LN>(a, s) : rows_cfg<4, ROWS_LN>(a, s);
    if (a.qo) return hipErrorInvalidValue;
    return k <= 512 ? rows_cfg<2, ROWS_F32>(a, s) : rows_cfg<4, ROWS_F32>(a, s);
}

hipError_t launch_rows_groups(const void *image, int64_t n, int64_t k, RowsArgs a, hipStream_t s) {
    if (a.M <= 0) return hipSuccess;
    if (k % 32 || !a.x_ws) return hipErrorInvalidValue;
    const WeightPlanes p = weight_planes(MQ_TYPE_Q8_0, n, k);
    const ActPlanes x = act_planes(MQ_TYPE_Q8_0, a.M, k, true);
    a.wq = (const int8_t *)image + p.tq, a.wd = (const float *)((const char *)image + p.tdw);
    a.xq = (const int8_t *)a.x_ws + x.xq, a.xd = (const float *)((const char *)a.x_ws + x.xd);
    a.n_pad = (int)p.n_pad, a.m_pad = x.m_pad, a.kch = (int)(p.kb_pad / 32), a.N = (int)n, a.K = (int)k;
    hipLaunchKernelGGL(k_rows_groups, dim3((unsigned)((a.N + 31) / 32), (unsigned)((a.M + 31) / 32)), dim3(256), 0, s, a);
    return hipGetLastError();
}

template <int HD, int KS>
static hipError_t rows_attn_cfg(const float *qkv, void *q_out, int variant, int B, int T, int H, int nh, hipStream_t s) {
    const ActPlanes o = act_planes(MQ_TYPE_Q8_0, (int64_t)B * T, H, true);
    const size_t lds = (size_t)3 * T * (HD + 4) * sizeof(float);
    static_assert(3 * ROWS_MAX_T * (128 + 4) * 4 + 4096 <= 64 * 1024, "no raised LDS limit");
    hipLaunchKernelGGL((k_rows_attn<HD, KS>), dim3((unsigned)(B * nh)), dim3(1024), lds, s, qkv, (int8_t *)q_out + o.xq,
                       (float *)((char *)q_out + o.xd), (int)(o.kb_pad / 32), o.m_pad, variant, T, H, nh,
                       1.0f / sqrtf((float)HD));
    return hipGetLastError();
}

hipError_t launch_rows_attn(const float *qkv, void *q_out, int variant, int B, int T, int H, int nh, hipStream_t s) {
    if (T <= 0 || T > ROWS_MAX_T || B <= 0 || (uintptr_t)qkv % 16) return hipErrorInvalidValue;
    const int hd = H / nh, ks = T % 4 == 0 ? 4 : T % 2 == 0 ? 2 : 1;  // launch_attention's key ranges
    static_assert(ROWS_MAX_T / 2 <= ATT_KB && ROWS_MAX_T <= 2 * ATT_KB, "one block a range, two in a single one");
    switch (hd * 8 + ks) {
        case 32 * 8 + 4: return rows_attn_cfg<32, 4>(qkv, q_out, variant, B, T, H, nh, s);
        case 32 * 8 + 2: return rows_attn_cfg<32, 2>(qkv, q_out, variant, B, T, H, nh, s);
        case 32 * 8 + 1: return rows_attn_cfg<32, 1>(qkv, q_out, variant, B, T, H, nh, s);
        case 64 * 8 + 4: return rows_attn_cfg<64, 4>(qkv, q_out, variant, B, T, H, nh, s);
        case 64 * 8 + 2: return rows_attn_cfg<64, 2>(qkv, q_out, variant, B, T, H, nh, s);
        case 64 * 8 + 1: return rows_attn_cfg<64, 1>(qkv, q_out, variant, B, T, H, nh, s);
        case 128 * 8 + 4: return rows_attn_cfg<128, 4>(qkv, q_out, variant, B, T, H, nh, s);
        case 128 * 8 + 2: return rows_attn_cfg<128, 2>(qkv, q_out, variant, B, T, H, nh, s);
        case 128 * 8 + 1: return rows_attn_cfg<128, 1>(qkv, q_out, variant, B, T, H, nh, s);
        default: return hipErrorInvalidValue;
    }
}

// The few-row form takes the batches whose products the general path gives to the GEMV (at most
// GEMV_MAX_M rows) and whose attention is k_attention: those it computes bit for bit.  Up to 64 or 128
// rows it would still be the faster one at some sizes (H 384, 6 layers: 2 x 32 tokens 247 -> 222 us,
// 4 x 32 249 -> 225 us), but there the general path's sums are the GEMM's, and its attention the
// matrix cores'.  MI355X, microseconds a call, general path / few rows, tokens B x T:
//   H 384, F 1536, 6 layers:  1x5 302 / 152, 1x16 489 / 182, 1x32 804 / 225
//   H 768, F 3072, 3 layers:  1x16 335 / 142
//   H 1024, F 4096, 3 layers: 1x16 377 / 164
// Head_dim 128, which k_attention does not take: up to 64 rows (128 at H <= 512), where the runner
// has no other path (its fused GEMM path comes first).
// MQ_BERT_ROWS sets the most rows it takes (0: none; measurements, and comparing the two paths).
int64_t rows_path_limit(int64_t H, int64_t F, int hd) {
    if (H > ROWS_MAX_LN || F > ROWS_MAX_K || H % 32 || F % 32 || (hd != 32 && hd != 64 && hd != 128)) return 0;
    int64_t lim = hd < 128 ? GEMV_MAX_M : H > 512 ? 64 : 128;
    if (const char *e = getenv("MQ_BERT_ROWS"))
        if (*e) lim = std::min<int64_t>(lim, std::max(atoi(e), 0));
    return lim;
}
bool rows_path_fits(int64_t rows, int64_t T, int64_t H, int64_t F, int hd) {
    auto gemv = [&](int64_t n, int64_t k) { return mq_mul_mat_path(MQ_TYPE_Q8_0, n, k, rows) == MQ_PATH_GEMV; };
    return rows <= rows_path_limit(H, F, hd) && T <= ROWS_MAX_T &&
           (hd == 128 || (gemv(3 * H, H) && gemv(H, H) && gemv(F, H)));
}

}  // namespace mq
