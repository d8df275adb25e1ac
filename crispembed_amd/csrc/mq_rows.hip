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
// does in its store.
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

// ggml's Q8_0 scale and reciprocal of a block whose largest magnitude is amax, and one quant
__device__ __forceinline__ void rows_scale(float amax, int variant, float &d, float &id) {
#pragma clang fp contract(off)
    const float dd = amax / 127.f;
    if (variant == MQ_Q8_0_X86) id = (amax != 0.0f) ? 127.f / amax : 0.0f;
    else id = (dd != 0.0f) ? 1.0f / dd : 0.0f;
    d = f16_bits_to_f32(f32_to_f16_bits(dd));
}
__device__ __forceinline__ int rows_quant(float x, float id, int variant) {
#pragma clang fp contract(off)
    const float t = x * id;
    const float r = (variant == MQ_Q8_0_REF) ? roundf(t) : rintf(t);
    return (int)fminf(fmaxf(r, -128.f), 127.f);
}

// One value of 32 lanes (a half wave) as a Q8_0 block of row `row` and chunk kc of a GEMM-layout
// activation; l32 the value's place in the block
__device__ __forceinline__ void rows_store_q8_0(float x, int8_t *qo, float *qd, int kch, int64_t m_pad, int64_t row,
                                                int kc, int l32, int variant, bool live) {
    float amax = max8(fabsf(x));
    amax = fmaxf(amax, dpp_f<0x140>(amax));
    amax = fmaxf(amax, __shfl_xor(amax, 16));
    float d, id;
    rows_scale(amax, variant, d, id);
    if (live) {
        qo[(((row >> 5) * kch + kc) << 10) + ((((l32 >> 4) << 5) + (row & 31)) << 4) + (l32 & 15)] =
            (int8_t)rows_quant(x, id, variant);
        if (l32 == 0) qd[kc * m_pad + row] = d;
    }
}

// The few-row product.  8 waves; wave w multiplies the 32-value blocks w, w + 8, ... of K (one
// v_mfma_i32_32x32x32_i8 and a scaled add each), and the eight partial tiles meet in LDS.  The sums
// are the GEMV's, in its order, so the results are its results bit for bit: there lane l of a wave
// adds up blocks l and l + 64 and the lanes meet in a tree over lane ^ 32, 16, 8, 4, 2, 1; here block
// l = w + 8 i is step i of wave w, so the tree's first three levels join steps i ^ 4, 2, 1 of a wave
// and the last three join waves w ^ 4, 2, 1.
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
            float4 v[4][KP], res[PRO == ROWS_LN ? 4 : 1][KP], lw[KP], lb[KP];
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
            float am[4 * KP];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if (PRO == ROWS_LN && r < nr) {  // uniform
                    // the statistics in fp32 (their error scales a whole row, which its blocks' scales
                    // take up), the values in fp64 up to the one rounding of the result
                    float s = 0.f;
#pragma unroll
                    for (int p = 0; p < KP; p++) {
                        const float4 t = v[r][p], u = res[PRO == ROWS_LN ? r : 0][p];
                        s += ((t.x + u.x) + (t.y + u.y)) + ((t.z + u.z) + (t.w + u.w));
                    }
                    const float mean = wave_sum_f(s) / (float)a.K;
                    float s2 = 0.f;
#pragma unroll
                    for (int p = 0; p < KP; p++)
                        if (256 * p + 4 * lane < a.K) {
                            const float4 t = v[r][p], u = res[PRO == ROWS_LN ? r : 0][p];
                            const float x0 = (t.x + u.x) - mean, x1 = (t.y + u.y) - mean, x2 = (t.z + u.z) - mean,
                                        x3 = (t.w + u.w) - mean;
                            s2 += (x0 * x0 + x1 * x1) + (x2 * x2 + x3 * x3);
                        }
                    const double rstd = 1.0 / sqrt((double)wave_sum_f(s2) / (double)a.K + (double)a.eps);
#pragma unroll
                    for (int p = 0; p < KP; p++) {
                        float4 &t = v[r][p];
                        const float4 u = res[PRO == ROWS_LN ? r : 0][p];
                        auto norm = [&](float x, float y, float w, float b) {
                            return (float)(((double)x + (double)y - (double)mean) * rstd * (double)w + (double)b);
                        };
                        t.x = norm(t.x, u.x, lw[p].x, lb[p].x), t.y = norm(t.y, u.y, lw[p].y, lb[p].y);
                        t.z = norm(t.z, u.z, lw[p].z, lb[p].z), t.w = norm(t.w, u.w, lw[p].w, lb[p].w);
                        const int c = 256 * p + 4 * lane;
                        if (blockIdx.x == 0 && c < a.K) *(float4 *)(a.xout + (int64_t)(m0 + wave + 8 * r) * a.K + c) = t;
                    }
                }
#pragma unroll
                for (int p = 0; p < KP; p++) {
                    const float4 t = v[r][p];
                    am[4 * p + r] = max8(fmaxf(fmaxf(fabsf(t.x), fabsf(t.y)), fmaxf(fabsf(t.z), fabsf(t.w))));
                }
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
                rows_scale(mine, a.variant, d, id);
                const int pd = (g0 + sub) >> 2, kd = 8 * pd + (lane >> 3);
                if (kd < nblk) sd[kd * 32 + wave + 8 * (sub & 3)] = d;
#pragma unroll
                for (int g = 0; g < 8; g++) {
                    const int r = g & 3, p = (g0 + g) >> 2, kc = 8 * p + (lane >> 3), w0 = 4 * sub;
                    if (r >= nr) continue;  // uniform
                    const float ig = __shfl(id, (lane & 56) + g);
                    const float4 t = v[r][p];
                    const uint32_t q = pack4_i8(rows_quant(t.x, ig, a.variant), rows_quant(t.y, ig, a.variant),
                                                rows_quant(t.z, ig, a.variant), rows_quant(t.w, ig, a.variant));
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

// Attention of one (sequence, head) of at most ROWS_MAX_T tokens, fp32: q, k, v (bias added) to LDS, then
// a wave per query row, lane j key j: score, softmax over the lanes, and lanes as head dims for
// the weighted sum of V (64 / HD groups of keys side by side at HD < 64, HD / 64 dims a lane
// above).  The rows leave as the Q8_0 activation of the o product (32 head dims a block).
template <int HD>
__global__ __launch_bounds__(1024) void k_rows_attn(const float *__restrict__ qkv, int8_t *__restrict__ qo,
                                                    float *__restrict__ qd, int kch, int64_t m_pad, int variant, int T,
                                                    int H, int nh, float scale) {
    constexpr int ST = HD + 4;  // row stride: float4 reads of 8 consecutive rows hit all banks
    constexpr int DL = HD < 64 ? 1 : HD / 64, KG = HD < 64 ? 64 / HD : 1;
    extern __shared__ __attribute__((aligned(16))) float sm[];
    float *Q = sm, *K = Q + T * ST, *V = K + T * ST;
    __shared__ float ps[16][64];
    const int b = blockIdx.x / nh, h = blockIdx.x % nh;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const float *base = qkv + (int64_t)b * T * 3 * H + h * HD;
    for (int e = threadIdx.x; e < 3 * T * (HD / 4); e += 1024) {
        const int d4 = e % (HD / 4), rest = e / (HD / 4), t = rest % T, w = rest / T;
        *(float4 *)(Q + (w * T + t) * ST + 4 * d4) = *(const float4 *)(base + (int64_t)t * 3 * H + w * H + 4 * d4);
    }
    __syncthreads();
    for (int i = wave; i < T; i += 16) {
        float s = -INFINITY;
        if (lane < T) {
            float4 t = make_float4(0.f, 0.f, 0.f, 0.f), u = t;  // eight short chains
#pragma unroll
            for (int d = 0; d < HD; d += 8) {
                const float4 q = *(const float4 *)(Q + i * ST + d), k = *(const float4 *)(K + lane * ST + d);
                const float4 q2 = *(const float4 *)(Q + i * ST + d + 4), k2 = *(const float4 *)(K + lane * ST + d + 4);
                t.x += q.x * k.x, t.y += q.y * k.y, t.z += q.z * k.z, t.w += q.w * k.w;
                u.x += q2.x * k2.x, u.y += q2.y * k2.y, u.z += q2.z * k2.z, u.w += q2.w * k2.w;
            }
            s = (((t.x + t.y) + (t.z + t.w)) + ((u.x + u.y) + (u.z + u.w))) * scale;
        }
        const float mx = wave_max_f(s);
        const float p = lane < T ? expf(s - mx) : 0.f;
        const float sum = wave_sum_f(p);
        ps[wave][lane] = p;  // one wave writes and reads its row
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int d0 = lane % (HD < 64 ? HD : 64), g = KG > 1 ? lane / HD : 0;
        float o[DL], o2[DL];
#pragma unroll
        for (int n = 0; n < DL; n++) o[n] = o2[n] = 0.f;
        int j = g;
        for (; j + KG < T; j += 2 * KG) {
            const float pj = ps[wave][j], pk = ps[wave][j + KG];
#pragma unroll
            for (int n = 0; n < DL; n++) {
                o[n] += pj * V[j * ST + d0 + 64 * n];
                o2[n] += pk * V[(j + KG) * ST + d0 + 64 * n];
            }
        }
        if (j < T) {
            const float pj = ps[wave][j];
#pragma unroll
            for (int n = 0; n < DL; n++) o[n] += pj * V[j * ST + d0 + 64 * n];
        }
#pragma unroll
        for (int n = 0; n < DL; n++) o[n] += o2[n];
        if constexpr (KG > 1) o[0] += __shfl_xor(o[0], 32);
#pragma unroll
        for (int n = 0; n < DL; n++)
            rows_store_q8_0(o[n] / sum, qo, qd, kch, m_pad, (int64_t)b * T + i, (h * HD + d0 + 64 * n) >> 5, lane & 31,
                            variant, g == 0);
        __builtin_amdgcn_wave_barrier();
    }
}

template <int KP, int PRO, bool RQ = false>
static hipError_t rows_cfg(const RowsArgs &a, hipStream_t s) {
    const size_t op = PRO == ROWS_Q ? 0 : (size_t)(a.K / 32) * (1024 + 128), lds = op > 32768 ? op : 32768;
    static_assert(ROWS_MAX_LN / 32 * (1024 + 128) <= 64 * 1024, "no raised LDS limit");
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

hipError_t launch_rows_attn(const float *qkv, void *q_out, int variant, int B, int T, int H, int nh, hipStream_t s) {
    const int hd = H / nh;
    if (T <= 0 || T > ROWS_MAX_T || B <= 0 || (uintptr_t)qkv % 16) return hipErrorInvalidValue;
    const ActPlanes o = act_planes(MQ_TYPE_Q8_0, (int64_t)B * T, H, true);
    int8_t *qo = (int8_t *)q_out + o.xq;
    float *qd = (float *)((char *)q_out + o.xd);
    const int kch = (int)(o.kb_pad / 32);
    const dim3 g((unsigned)(B * nh));
    const size_t lds = (size_t)3 * T * (hd + 4) * sizeof(float);
    const float scale = 1.0f / sqrtf((float)hd);
    static_assert(3 * ROWS_MAX_T * (128 + 4) * 4 + 4096 <= 64 * 1024, "no raised LDS limit");
    switch (hd) {
        case 32:
            hipLaunchKernelGGL((k_rows_attn<32>), g, dim3(1024), lds, s, qkv, qo, qd, kch, o.m_pad, variant, T, H, nh, scale);
            break;
        case 64:
            hipLaunchKernelGGL((k_rows_attn<64>), g, dim3(1024), lds, s, qkv, qo, qd, kch, o.m_pad, variant, T, H, nh, scale);
            break;
        case 128:
            hipLaunchKernelGGL((k_rows_attn<128>), g, dim3(1024), lds, s, qkv, qo, qd, kch, o.m_pad, variant, T, H, nh, scale);
            break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// Where the few-row form ends: its workgroups repeat a row tile's LayerNorm and quantization per 32
// output columns, so it loses once a launch holds several of them per CU, sooner at wide rows; and
// its attention walks T / 16 query rows a wave.  MI355X, microseconds a call, GEMM path (GEMV
// path under 33 rows) / few rows, tokens B x T:
//   H 384, F 1536, 6 layers:  1x16 489 / 175, 1x32 799 / 214, 2x32 240 / 219, 1x64 243 / 248,
//                             4x32 243 / 222, 2x64 245 / 252, 16x16 277 / 270, 8x32 247 / 282
//   H 768, F 3072, 3 layers:  1x16 324 / 138, 2x32 181 / 175, 1x64 181 / 191, 4x32 184 / 248
//   H 1024, F 4096, 3 layers: 1x16 374 / 165, 2x32 214 / 204, 1x64 211 / 217, 4x32 216 / 283
// MQ_BERT_ROWS sets the most rows it takes (0: none; measurements).
bool rows_path_fits(int64_t rows, int64_t T, int64_t H, int64_t F, int hd) {
    int64_t lim = H > 512 ? 64 : 128;
    if (const char *e = getenv("MQ_BERT_ROWS"))
        if (*e) lim = atoi(e);
    return rows <= lim && T <= ROWS_MAX_T && H <= ROWS_MAX_LN && F <= ROWS_MAX_K && H % 32 == 0 && F % 32 == 0 &&
           (hd == 32 || hd == 64 || hd == 128);
}

}  // namespace mq
