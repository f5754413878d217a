/*
 * fno_layer.hip -- fused kernels of the pass surrogate's Fourier layers.
 *
 * k_column: everything between two layers' transverse transforms, one
 * transverse point (x, y) at a time with all its channels and times: inverse
 * t-DFT of the layer's mode coefficients, 1x1 channel map, bias, GELU, and
 * the next layer's forward t-DFT (or, after the last layer, the projection
 * head).  As separate kernels (k_gemm_bf16, k_pointwise_mf) these passes move
 * the activations through HBM five times per layer; here they are read once
 * and written once.
 *
 * k_dft / k_dft_t: a truncated complex DFT along y or x with the complex
 * recombination in its epilogue, and its transpose.  As k_gemm_bf16 and
 * k_combine the real-block products went through HBM between the two.
 *
 * The arithmetic is that of the separate kernels, in the same order: operands
 * of the DFT products are rounded to BF16 as they are staged and products
 * accumulate in FP32 along k in ascending order (the MFMA shapes
 * v_mfma_f32_16x16x16_bf16, 16x16x32 and 32x32x16 give the same bits for the
 * same order, checked on the device); the channel maps are FP32
 * (v_mfma_f32_32x32x2f32: a chain of fused multiply-adds in ascending channel
 * order, the same bits as the vector form).
 */
#include "internal.h"
#include "fno_device.h"
#include "../../include/mpc_fno.h"

namespace {

constexpr int CW = 8;                  /* waves per workgroup of k_column */
constexpr int CT_MAX = 256;            /* t points a workgroup covers: CW tiles of 32 */
constexpr int CN2_MAX = 64;            /* columns of the t-DFT (2 mt) */
constexpr int CG_MAX = 4096;           /* workgroups of k_column */
constexpr int CH_MAX = 64;             /* hidden channels of the head */

__device__ __forceinline__ f32x16 mfma_bf16(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
/*
 * The rows of a 32 x 32 product as the operand of an FP32 product that
 * contracts over them: step s takes rows 2 s (lower half-wave) and 2 s + 1
 * (upper), which lie in the registers of two lanes: pairs of registers swap
 * halves.
 */
__device__ __forceinline__ void operand_of(const f32x16 &d, float (&x)[16]) {
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
        const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(d[r]), __float_as_uint(d[r + 1]), false, false);
        const int s = 4 * (r / 4) + (r % 4) / 2;
        x[s] = __uint_as_float(p[0]);
        x[s + 2] = __uint_as_float(p[1]);
    }
}
/* row of a 32 x 32 product that register r of a lane in half-wave h holds */
__device__ __forceinline__ int drow(int r, int h) { return 8 * (r / 4) + 4 * h + r % 4; }

/* dW (oc x ic, of which no x ni are stored) += and db = the sums that nwg workgroups left in part; 32 entries a block, 32 threads an entry */
__global__ void __launch_bounds__(1024) k_wgrad_sum(const float *__restrict__ part, int nwg, int oc, int ic,
                                                    float *__restrict__ dW, float *__restrict__ db, int no, int ni) {
    __shared__ float red[32][33];
    const int ne = oc * (ic + 1), e = blockIdx.x * 32 + (threadIdx.x & 31), q = threadIdx.x >> 5;
    float s = 0.f;
    if (e < ne)
        for (int w = q; w < nwg; w += 32) s += part[(long)w * ne + e];
    red[q][threadIdx.x & 31] = s;
    __syncthreads();
    if (q != 0 || e >= ne) return;
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < 32; ++k) t += red[k][threadIdx.x];
    if (e < oc * ic) {
        const int o = e / ic, i = e % ic;
        if (o < no && i < ni) dW[(long)o * ni + i] += t;
    } else if (db && e - oc * ic < no) {
        db[e - oc * ic] = t;
    }
}
/*
 * k_column<W, CIN, KIND, ZS, CPI>: workgroups walk groups of CPI transverse
 * points (b, pos), grid-stride.  Wave u of a workgroup holds t tile u % ntile
 * (32 times) of point u / ntile of the group; a lane holds one time and, in
 * each product register, one channel (drow).
 *   KIND 0, lift:  z = Wm x + bias                        (no mode part)
 *   KIND 1, layer: z = V6 Gt + Wm v + bias; v' = GELU(z) if act; ZS (training):
 *           z is stored too and the GELU is the training path's
 *   KIND 2, last:  as KIND 1, then y = Q2 GELU(Q1 v' + q1) + q2 + x[:, :2]
 *   KIND 3, backward: dz' = (V6 Gt + Wm dz) GELU'(zin), with V6 the transposed
 *           mode path's result, Gt = Ft^T and Wm the transposed channel map of
 *           the layer above, zin this layer's pre-activation
 *   KIND 4, backward through the first layer: V6 Gt + Wm dz only
 *   KIND 5, backward through the head: its hidden layer formed again from v as
 *           KIND 2 does, dh = (Q2^T dpred) GELU'(hz) (stored for Q1's gradient),
 *           dz = Wm dh with Wm = Q1^T, and the sums of Q2's and q2's gradients
 * Training's KIND 2 (ZS) also stores v', and its GELU and order of summation
 * over the hidden channels are the separate kernels' (the products with Q2 go
 * through the matrix cores), so y keeps its bits.  The last layer, the head and
 * the way back to dz at batch 4 of 64 x 64 x 256 points, 32 and 64 channels:
 * 525 + 803 us, bound by the GELUs and the FP32 products; as separate kernels,
 * which store and read hz, h and dh between them, 2670.
 * Kinds 0, 1, 3 and 5 then form C1 = v' Ft (3: Ft = Gt^T), from v' rounded to BF16
 * in LDS (5: as 3).  Kind 3 at batch 4 of 64 x 64 x 256 points, width 32, moves 3 streams
 * of 0.54 GB in 395 us; the four kernels it stands for took 1100.
 * LDS at W = 32, T = 256: Ft 33 KB, v' 17 KB, V6 5 KB, Wm 4 KB: two workgroups
 * (four waves per SIMD) fit on a CU, so one's loads and stores run under the
 * other's products and GELUs.
 *
 * The next group's mode rows and channels are loaded while this one is worked
 * on.  Loads and stores share one in-order counter, so a wait for those loads
 * must not also wait for the stores behind them: the loop is straight-line
 * (in a branch the compiler has to assume the path without the stores).
 * Times past T, waves without a tile, rows past W and columns past n2
 * therefore work on the last valid one again and store the same value there.
 */
template <int W, int CIN, int KIND> struct ColCfg {
    static constexpr int MT = W <= 32 ? 1 : W / 32;            /* 32-row channel tiles */
    static constexpr int NR = W >= 32 ? 16 : W / 2;            /* product registers in use per tile */
    static constexpr int KS = (CIN + 1) / 2;                   /* FP32 product steps of the channel map */
    static constexpr int WP = (KIND == 5 ? CH_MAX : CIN) + 1;  /* LDS pitch of the weight rows */
    static constexpr int AP = CN2_MAX + 8;                     /* pitch of the staged V6 rows */
    static constexpr int M16 = (W + 15) / 16;                  /* 16-row tiles of the forward t-DFT */
};

template <int W, int CIN, int KIND, bool ZS, int CPI>
__global__ void __launch_bounds__(64 * CW, (W <= 32 && KIND != 5 ? 4 : 2)) k_column(mpc_fno_col a) {
    using C = ColCfg<W, CIN, KIND>;
    constexpr int MT = C::MT, NR = C::NR, KS = C::KS, WP = C::WP, AP = C::AP, M16 = C::M16;
    constexpr bool MODES = KIND != 0 && KIND != 5;             /* takes mode rows V6 */
    constexpr bool DFT = KIND != 2 && KIND != 4, BWD = KIND >= 3, HEAD = KIND == 2 || KIND == 5;
    const int T = a.nt, n2 = a.n2, npos = a.npos;
    const int ntile = (T + 31) / 32, tpad = 32 * ntile;
    const int tp = tpad + 8;                                   /* pitch of the v' and Ft rows (bf16) */
    const int n16 = (n2 + 15) / 16;
    extern __shared__ __align__(16) unsigned char smem[];
    /* bias | Wm | q1 and its weights (KIND 2) | V6 rows | v' rows | Ft rows */
    float *Bl = reinterpret_cast<float *>(smem);
    float *Wl = Bl + MT * 32;
    float *Ql = Wl + MT * 32 * WP;
    const int ht = HEAD ? (a.h + 31) / 32 : 0;
    short *A6 = reinterpret_cast<short *>(smem + ((MT * 32 * (WP + 1) + ht * 32 * (W + 4)) * 4 + 15) / 16 * 16);
    short *Vl = A6 + (MODES ? CPI * MT * 32 * AP : 0);
    short *Fl = Vl + CPI * M16 * 16 * tp;

    const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int unit = min(wave, CPI * ntile - 1);
    const int csub = unit / ntile, tile = unit % ntile;
    const int t = 32 * tile + col;

    if constexpr (!BWD)
        for (int i = tid; i < MT * 32; i += 64 * CW) Bl[i] = i < W ? a.bias[i] : 0.f;
    if constexpr (KIND == 5) {                                 /* Q1^T: W x h */
        for (int i = tid; i < MT * 32 * a.h; i += 64 * CW) {
            const int o = i / a.h, k = i % a.h;
            Wl[o * WP + k] = o < W ? a.w[o * a.h + k] : 0.f;
        }
    } else {
        for (int i = tid; i < MT * 32 * CIN; i += 64 * CW) {
            const int o = i / CIN, k = i % CIN;
            Wl[o * WP + k] = o < W ? a.w[o * CIN + k] : 0.f;
        }
    }
    /* q1 | the two rows of Q2 | Q1 */
    if constexpr (HEAD) {
        for (int i = tid; i < ht * 32 * W; i += 64 * CW) {
            const int o = i / W, k = i % W;
            Ql[ht * 96 + o * (W + 1) + k] = o < a.h ? a.q1w[o * W + k] : 0.f;
        }
        for (int o = tid; o < ht * 32; o += 64 * CW) {
            Ql[o] = o < a.h ? a.q1[o] : 0.f;
            Ql[ht * 32 + o] = o < a.h ? a.q2w[o] : 0.f;
            Ql[ht * 64 + o] = o < a.h ? a.q2w[a.h + o] : 0.f;
        }
    }
    if constexpr (MODES)
        for (int i = tid; i < CPI * MT * 32 * AP; i += 64 * CW) A6[i] = 0;
    if constexpr (DFT) {
        const int rq = tpad / 8;                               /* 16-byte pieces per row */
        for (int i = tid; i < n16 * 16 * rq; i += 64 * CW)
            *reinterpret_cast<bf16x8 *>(Fl + i / rq * tp + i % rq * 8) = reinterpret_cast<const bf16x8 *>(a.Ft)[i];
    }
    /* the wave's columns of Gt */
    bf16x8 gB[MODES ? 4 : 1];
    if constexpr (MODES) {
#pragma unroll
        for (int s = 0; s < 4; ++s) gB[s] = reinterpret_cast<const bf16x8 *>(a.Gt)[(tile * 4 + s) * 64 + lane];
    }

    const int stride = gridDim.x * CPI;
    const unsigned cs = (unsigned)npos * (unsigned)T;          /* channel stride of the activations */
    /* byte offsets of this lane's time from a sample's (b, pos), in channel row
     * half and channel row 4 half; a channel is c4 bytes */
    const unsigned to = 4u * (unsigned)min(t, T - 1);
    const unsigned xo = 4u * half * cs + to, lo = 16u * half * cs + to, c4 = 4u * cs;
    auto advance = [&](int &b, int &pos, int by) {
        pos += by;
        while (pos >= npos) { pos -= npos; ++b; }
    };
    /* point i of the group at (b0, pos0), or the last point there is */
    auto point = [&](int b0, int pos0, int i, int &b, int &pos) {
        b = b0;
        pos = pos0;
        advance(b, pos, i);
        if (b >= a.nb) { b = a.nb - 1; pos = npos - 1; }
    };
    /* V6 of a group: CPI x W rows of n2 floats (n2 even); 32 threads a row, two floats each */
    constexpr int RPP = 64 * CW / 32, NV = (CPI * W + RPP - 1) / RPP;
    float2 pre[MODES ? NV : 1];
    const int kp = min(tid & 31, n2 / 2 - 1), row0 = tid >> 5;
    const unsigned row4 = 4u * (unsigned)npos * (unsigned)n2;  /* bytes of a channel's mode rows */
    auto load_v6 = [&](int b0, int pos0) {
        if constexpr (MODES) {
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int r = min(row0 + RPP * i, CPI * W - 1);
                int b, pos;
                point(b0, pos0, CPI > 1 ? __builtin_amdgcn_readfirstlane(r / W) : 0, b, pos);   /* a wave's two rows are of one point */
                pre[i] = buf_ld2(buf_of(a.V6 + (long)b * W * npos * n2), (unsigned)(r % W) * row4 + 8u * kp, 4u * pos * n2);
            }
        }
    };
    float xv[KS], xn[KS];                                      /* this wave's channels of its time; the next group's */
    auto load_x = [&](int b0, int pos0) {
        int b, pos;
        point(b0, pos0, csub, b, pos);
        const rsrc_t xb = buf_of(a.v + b * a.v_bs);
#pragma unroll
        for (int s = 0; s < KS; ++s) xn[s] = buf_ld(xb, xo, 4u * pos * T + 2u * s * c4);
    };
    int b0 = 0, pos0 = 0;                                      /* the group's first point */
    advance(b0, pos0, blockIdx.x * CPI);
    __syncthreads();                                           /* the zeroed rows come before the staged ones */
    load_v6(b0, pos0);
    load_x(b0, pos0);
    /* the loads of the next group are waited for here, at the end of a
     * group's work, where the stores issued after them are known and need not
     * be waited for: at the top of the loop the wait would have to suit the
     * first round too, which has none */
    auto arrive = [&] {
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            asm volatile("" : "+v"(xn[s]));
            xv[s] = xn[s];
        }
        if constexpr (MODES) {
#pragma unroll
            for (int i = 0; i < NV; ++i) asm volatile("" : "+v"(pre[i].x), "+v"(pre[i].y));
        }
    };
    arrive();
    float s2[KIND == 5 ? 2 : 1][2][16] = {}, sb[2] = {};       /* KIND 5: sums of dpred h and dpred */
    while (b0 < a.nb) {
        if constexpr (MODES) {
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int r = min(row0 + RPP * i, CPI * W - 1);
                *reinterpret_cast<int *>(&A6[(r / W * MT * 32 + r % W) * AP + 2 * kp]) = bf16_pair(pre[i].x, pre[i].y);
            }
        }
        __syncthreads();
        int b, pos;
        point(b0, pos0, csub, b, pos);
        const long ob = (long)b * W * cs;
        const unsigned po = 4u * pos * T;
        float zq[KIND == 3 ? MT : 1][16];                      /* before the next group's loads, which it need not wait for */
        if constexpr (KIND == 3) {
            const rsrc_t zb = buf_of(a.zin + ob);
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int r = 0; r < NR; ++r) zq[m][r] = buf_ld(zb, lo, po + (32u * m + 8 * (r / 4) + r % 4) * c4);
        }
        float dp[2] = {};
        if constexpr (KIND == 5) {
            const rsrc_t db = buf_of(a.x + b * a.x_bs);
#pragma unroll
            for (int o = 0; o < 2; ++o) dp[o] = buf_ld(db, to, po + o * c4);
        }
        int bn = b0, pn = pos0;
        advance(bn, pn, stride);
        load_v6(bn, pn);
        load_x(bn, pn);
        float zr[KIND == 2 ? MT : 1][16];
        f32x16 dva[KIND == 5 ? MT : 1] = {};
        if constexpr (KIND == 5) {
            /* times, waves and points that are only repeated count once */
            const bool live = wave < CPI * ntile && t < T && (CPI == 1 || (long)b0 * npos + pos0 + csub < (long)a.nb * npos);
            const float dq0 = live ? bf16_round(dp[0]) : 0.f, dq1 = live ? bf16_round(dp[1]) : 0.f;
            sb[0] += live ? dp[0] : 0.f;
            sb[1] += live ? dp[1] : 0.f;
            const rsrc_t hb = buf_of(a.dh + (long)b * a.h * cs);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                if (q >= ht) break;
                f32x16 acc = {};
#pragma unroll
                for (int s = 0; s < KS; ++s)
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(Ql[ht * 96 + (32 * q + col) * (W + 1) + 2 * s + half], xv[s], acc, 0, 0, 0);
                float xb[16];
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int o = 32 * q + drow(r, half);
                    const float z = acc[r] + Ql[o], hv = bf16_round(gelu(z));
                    s2[q][0][r] = fmaf(dq0, hv, s2[q][0][r]);
                    s2[q][1][r] = fmaf(dq1, hv, s2[q][1][r]);
                    acc[r] = fmaf(Ql[ht * 64 + o], dp[1], Ql[ht * 32 + o] * dp[0]) * gelu_d(z);
                    buf_st(hb, lo, po + (32u * q + 8 * (r / 4) + r % 4) * c4, acc[r]);
                    if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                }
                operand_of(acc, xb);
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int s = 0; s < 16; ++s)
                        dva[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(Wl[(32 * m + col) * WP + 32 * q + 2 * s + half], xb[s], dva[m], 0, 0, 0);
            }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            f32x16 sp = {}, acc = {};
            if constexpr (KIND == 5) acc = dva[m];
            if constexpr (MODES) {
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    sp = mfma_bf16(*reinterpret_cast<const bf16x8 *>(&A6[((csub * MT + m) * 32 + col) * AP + 16 * s + 8 * half]),
                                   gB[s], sp);
            }
#pragma unroll
            for (int s = 0; s < (KIND == 5 ? 0 : KS); ++s)
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(Wl[(32 * m + col) * WP + 2 * s + half], xv[s], acc, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                if constexpr (MODES) acc[r] += sp[r];
                if constexpr (!BWD) acc[r] += Bl[32 * m + 4 * half + 8 * (r / 4) + r % 4];
                if constexpr (KIND == 3) {
                    acc[r] *= gelu_d(zq[m][r]);
                    if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);   /* four GELU' in flight: more spill */
                }
            }
            /* rows of the lower half-wave: 32 m + 8 (r / 4) + r % 4 */
            auto store = [&](float *base) {
                const rsrc_t rs = buf_of(base + ob);
#pragma unroll
                for (int r = 0; r < NR; ++r) buf_st(rs, lo, po + (32u * m + 8 * (r / 4) + r % 4) * c4, acc[r]);
            };
            if constexpr (ZS) store(a.zs);
            if constexpr (KIND == 2) {
#pragma unroll
                for (int r = 0; r < NR; ++r) zr[m][r] = acc[r];
            } else {
                if (!BWD && a.act) {
#pragma unroll
                    for (int r = 0; r < NR; ++r) acc[r] = ZS ? gelu(acc[r]) : gelu_fast(acc[r]);
                }
                store(a.out);
                if constexpr (DFT) {
                    short *vl = Vl + (csub * M16 * 16 + 32 * m + 4 * half) * tp + t;
#pragma unroll
                    for (int r = 0; r < NR; ++r) vl[(8 * (r / 4) + r % 4) * tp] = to_bf16(acc[r]);
                }
            }
        }
        if constexpr (KIND == 2) {
            /* the channels of a time lie in the registers of two lanes; as the
             * operand of the next channel map, step s takes channels 2s (lower
             * half-wave) and 2s + 1 (upper): pairs of registers swap halves */
            float xb2[MT * NR];
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int r = 0; r < NR; r += 2) {
                    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(zr[m][r]), __float_as_uint(zr[m][r + 1]), false, false);
                    const int s0 = 16 * m + 4 * (r / 4) + (r % 4) / 2;
                    xb2[s0] = __uint_as_float(p[0]);
                    xb2[s0 + 2] = __uint_as_float(p[1]);
                }
            float y0 = 0.f, y1 = 0.f;
            f32x16 ya = {};
            for (int q = 0; q < ht; ++q) {
                f32x16 acc = {};
#pragma unroll
                for (int s = 0; s < W / 2; ++s)
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(Ql[ht * 96 + (32 * q + col) * (W + 1) + 2 * s + half], xb2[s], acc, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int o = 32 * q + drow(r, half);
                    if constexpr (ZS) {
                        acc[r] = gelu(acc[r] + Ql[o]);
                    } else {
                        const float hv = gelu_fast(acc[r] + Ql[o]);
                        y0 = fmaf(Ql[ht * 32 + o], hv, y0);
                        y1 = fmaf(Ql[ht * 64 + o], hv, y1);
                    }
                    /* the rows' LDS operands load where they are used, not all ahead */
                    if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (ZS) {                            /* rows past the second repeat it */
                    float hb[16];
                    operand_of(acc, hb);
#pragma unroll
                    for (int s = 0; s < 16; ++s)
                        ya = __builtin_amdgcn_mfma_f32_32x32x2f32(Ql[ht * 32 * (1 + min(col, 1)) + 32 * q + 2 * s + half], hb[s], ya, 0, 0, 0);
                }
            }
            /* each half-wave summed its rows of both outputs (ZS: the lower one
             * all of them): the lower one finishes output 0, the upper output 1 */
            if constexpr (ZS) {
                y0 = ya[0];
                y1 = ya[1];
            }
            const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(y0), __float_as_uint(y1), false, false);
            const float ys = ZS ? __uint_as_float(p[0]) : __uint_as_float(p[0]) + __uint_as_float(p[1]);
            const float x0 = buf_ld(buf_of(a.x + b * a.x_bs), xo, po);
            buf_st(buf_of(a.y + b * 2L * cs), xo, po, ys + x0 + a.q2[half]);
        }
        __syncthreads();
        if constexpr (DFT) {
            constexpr int RND = (CPI * M16 * (CN2_MAX / 16) + CW - 1) / CW;
            const int nt16 = CPI * M16 * n16;
#pragma unroll
            for (int r = 0; r < RND; ++r) {
                const int i = min(wave + r * CW, nt16 - 1);
                const int n = i % n16, cm = i / n16, cc = cm / M16, m = cm % M16;
                int b2, p2;
                point(b0, pos0, cc, b2, p2);
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                const short *ap = Vl + ((cc * M16 + m) * 16 + (lane & (W < 16 ? 7 : 15))) * tp + 8 * (lane >> 4);
                const short *bp = Fl + (n * 16 + (lane & 15)) * tp + 8 * (lane >> 4);
                for (int k = 0; k < tpad; k += 32)
                    acc = mfma_bf16(*reinterpret_cast<const bf16x8 *>(ap + k), *reinterpret_cast<const bf16x8 *>(bp + k), acc);
                const int nn = min(n * 16 + (lane & 15), n2 - 1);
                const unsigned o = (unsigned)(4 * (lane >> 4) % W) * row4 + 4u * nn;
                const rsrc_t cp = buf_of(a.C1 + (long)b2 * W * npos * n2);
#pragma unroll
                for (int e = 0; e < 4; ++e) buf_st(cp, o, 4u * p2 * n2 + (16u * m + e) * row4, acc[e]);
            }
        }
        arrive();
        b0 = bn;
        pos0 = pn;
    }
    if constexpr (KIND == 5) {
        /* this workgroup's [2][h] sums and the two of dpred: over a half-wave's times, then the waves in order */
        float *red = reinterpret_cast<float *>(smem);          /* [CW][2 CH_MAX + 2]; the last products' barrier is behind */
        __syncthreads();
        constexpr int NE = 2 * CH_MAX + 2;
        auto lanes = [&](float v) {
#pragma unroll
            for (int k = 16; k > 0; k >>= 1) v += __shfl_xor(v, k);
            return v;
        };
#pragma unroll
        for (int o = 0; o < 2; ++o) {
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float v = lanes(s2[q][o][r]);
                    if (col == 0) red[wave * NE + o * CH_MAX + 32 * q + drow(r, half)] = v;
                }
            const float v = lanes(sb[o]);
            if (lane == 0) red[wave * NE + 2 * CH_MAX + o] = v;
        }
        __syncthreads();
        const int ne = 2 * (a.h + 1);
        for (int e = tid; e < ne; e += 64 * CW) {
            const int src = e < 2 * a.h ? e / a.h * CH_MAX + e % a.h : 2 * CH_MAX + e - 2 * a.h;
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < CW; ++w) v += red[w * NE + src];
            a.ws[(long)blockIdx.x * ne + e] = v;
        }
    }
}

template <int W, int CIN, int KIND, bool ZS, int CPI> int column_go(const mpc_fno_col *a, hipStream_t s) {
    using C = ColCfg<W, CIN, KIND>;
    const int tp = (a->nt + 31) / 32 * 32 + 8, ht = KIND == 2 || KIND == 5 ? (a->h + 31) / 32 : 0, n16 = (a->n2 + 15) / 16;
    size_t lds = ((size_t)(C::MT * 32 * (C::WP + 1) + ht * 32 * (W + 4)) * 4 + 15) / 16 * 16;
    if (KIND != 0 && KIND != 5) lds += (size_t)CPI * C::MT * 32 * C::AP * 2;
    if (KIND != 2 && KIND != 4) lds += (size_t)(CPI * C::M16 * 16 + n16 * 16) * tp * 2;
    int dev = 0, ncu = 0, per = 0;
    const void *k = (const void *)k_column<W, CIN, KIND, ZS, CPI>;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, 64 * CW, lds) != hipSuccess || per < 1)
        return MPC_EHIP;
    const long ngrp = ((long)a->nb * a->npos + CPI - 1) / CPI;
    const unsigned grid = (unsigned)std::min(ngrp, std::min((long)ncu * per, (long)CG_MAX));
    hipLaunchKernelGGL((k_column<W, CIN, KIND, ZS, CPI>), dim3(grid), dim3(64 * CW), lds, s, *a);
    if (KIND == 5)
        hipLaunchKernelGGL(k_wgrad_sum, dim3((2 * (a->h + 1) + 31) / 32), dim3(1024), 0, s, a->ws, (int)grid, 2, a->h,
                           a->dq2w, a->dq2, 2, a->h);
    return hipGetLastError() == hipSuccess ? 0 : MPC_EHIP;
}
/* short lines (at most CW/2 t tiles): two points at a time, so that no wave idles */
template <int W, int CIN, int KIND, bool ZS> int column_k(const mpc_fno_col *a, hipStream_t s) {
    return (a->nt + 31) / 32 <= CW / 2 ? column_go<W, CIN, KIND, ZS, 2>(a, s) : column_go<W, CIN, KIND, ZS, 1>(a, s);
}
template <int W> int column_w(const mpc_fno_col *a, hipStream_t s) {
    if constexpr (W <= 32) {
        if (a->dh) return column_k<W, W, 5, false>(a, s);
        if (a->y && a->zs) return column_k<W, W, 2, true>(a, s);
    }
    if (a->bwd) return a->zin ? column_k<W, W, 3, false>(a, s) : column_k<W, W, 4, false>(a, s);
    if (!a->V6) return column_k<W, 4, 0, false>(a, s);
    if (a->y) return column_k<W, W, 2, false>(a, s);
    return a->zs ? column_k<W, W, 1, true>(a, s) : column_k<W, W, 1, false>(a, s);
}

/* ---------------------------------------------------------------------- */
/* truncated DFT along y or x                                              */
/* ---------------------------------------------------------------------- */
/*
 * out[s][row][q][re(0..h) | im(0..h)], row < m, from in[s][k][q][re | im],
 * k < kk, and G = [cos (m x kk); sin (m x kk)]:
 *   out = (C in)_r - sg (S in)_i,  (C in)_i + sg (S in)_r.
 * A wave forms 16 rows x 32 columns of a block's re and im parts: its 32 x 32
 * product tile holds the 16 cos rows in registers 0-7 and the same 16 sin rows
 * in registers 8-15, so the recombination stays within a lane.  Inputs go
 * from memory to registers (an element is an operand of at most m / 16 waves)
 * and a wave walks slices with its rows of G in registers, so there is no
 * LDS and no barrier.  kk <= 16 KS.
 */
/* FULL: kk = 16 KS */
template <int KS, bool FULL>
__global__ void __launch_bounds__(256) k_dft(const bf16x8 *__restrict__ G, const float *__restrict__ in,
                                             float *__restrict__ out, long nunit, int m, int kk, int nq, int h, float sg) {
    const int lane = threadIdx.x & 63, col = lane & 31, half = lane >> 5;
    const int m0 = blockIdx.y * 16;
    bf16x8 ga[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) ga[s] = G[(blockIdx.y * KS + s) * 64 + lane];
    const int nh = (h + 31) / 32;
    const long rowl = (long)nq * 2 * h;                        /* floats per row of a slice */
    /* unit: (slice, block q, column tile) */
    for (long u = blockIdx.x * 4L + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); u < nunit; u += gridDim.x * 4L) {
        const int hc = (int)(u % nh);
        const long sq = u / nh;
        const int q = (int)(sq % nq);
        const long sl = sq / nq;
        const int c = hc * 32 + col;
        const bool cin = c < h;
        const rsrc_t ib = buf_of(in + sl * kk * rowl + q * 2 * h);
        f32x16 re = {}, im = {};
        float vr[KS][8], vi[KS][8];
        /* rows past kk meet zero columns of G: the last row stands in for them */
        const unsigned co = 4u * (unsigned)(cin ? c : h - 1), row4 = 4u * (unsigned)rowl;
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const unsigned o = FULL ? (unsigned)(8 * half) * row4 + co
                                        : (unsigned)min(16 * s + 8 * half + j, kk - 1) * row4 + co;
                const unsigned u0 = FULL ? (16 * s + j) * row4 : 0;
                vr[s][j] = buf_ld(ib, o, u0);
                vi[s][j] = buf_ld(ib, o, u0 + 4 * h);
            }
        if constexpr (KS <= 4) __builtin_amdgcn_sched_barrier(0);    /* all loads go out before the first wait */
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            re = mfma_bf16(ga[s], bf16_octet(vr[s]), re);
            im = mfma_bf16(ga[s], bf16_octet(vi[s]), im);
        }
        const rsrc_t ob = buf_of(out + (sl * m + m0) * rowl + q * 2 * h);
        const unsigned oo = (unsigned)(4 * half) * row4 + co;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int row = 8 * (r / 4) + r % 4;
            if (cin && m0 + row + 4 * half < m) {
                buf_st(ob, oo, row * row4, re[r] - sg * im[r + 8]);
                buf_st(ob, oo, row * row4 + 4 * h, im[r] + sg * re[r + 8]);
            }
        }
    }
}

/*
 * The transpose: out[s][k][q][re | im] = sum over the 2m real rows of G of
 * G[row][k] dP[row], dP the transposed recombination of in[s][row][q][re | im]
 * (row < m: (dVr, dVi); row >= m: (sg dVi, -sg dVr)).  A wave forms 32 k x 32
 * columns of re and im.  2 m <= 16 KS.
 */
template <int KS>
__global__ void __launch_bounds__(256) k_dft_t(const bf16x8 *__restrict__ G, const float *__restrict__ in,
                                               float *__restrict__ out, long nunit, int m, int kk, int nq, int h, float sg) {
    const int lane = threadIdx.x & 63, col = lane & 31, half = lane >> 5;
    const int k0 = blockIdx.y * 32;
    const int m2 = 2 * m;
    bf16x8 ga[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) ga[s] = G[(blockIdx.y * KS + s) * 64 + lane];
    const int nh = (h + 31) / 32;
    const long rowl = (long)nq * 2 * h;
    for (long u = blockIdx.x * 4L + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); u < nunit; u += gridDim.x * 4L) {
        const int hc = (int)(u % nh);
        const long sq = u / nh;
        const int q = (int)(sq % nq);
        const long sl = sq / nq;
        const int c = hc * 32 + col;
        const bool cin = c < h;
        const rsrc_t ib = buf_of(in + sl * m * rowl + q * 2 * h);
        f32x16 re = {}, im = {};
        const unsigned co = 4u * (unsigned)(cin ? c : h - 1), row4 = 4u * (unsigned)rowl;
        float vr[KS][8], vi[KS][8];
        /* rows past 2m meet zero columns: the last row stands in for them */
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int r = min(16 * s + 8 * half + j, m2 - 1);
                const bool sine = r >= m;
                const unsigned o = (unsigned)(sine ? r - m : r) * row4 + co;
                const float x = buf_ld(ib, o, 0), y = buf_ld(ib, o, 4 * h);
                vr[s][j] = sine ? sg * y : x;
                vi[s][j] = sine ? -sg * x : y;
            }
        if constexpr (KS <= 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            re = mfma_bf16(ga[s], bf16_octet(vr[s]), re);
            im = mfma_bf16(ga[s], bf16_octet(vi[s]), im);
        }
        const rsrc_t ob = buf_of(out + (sl * kk + k0) * rowl + q * 2 * h);
        const unsigned oo = (unsigned)(4 * half) * row4 + co;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int k = 8 * (r / 4) + r % 4;
            if (cin && k0 + k + 4 * half < kk) {
                buf_st(ob, oo, k * row4, re[r]);
                buf_st(ob, oo, k * row4 + 4 * h, im[r]);
            }
        }
    }
}

/* K steps a k_dft instantiation holds for a contraction over n */
int dft_steps(int n) { return n <= 16 ? 1 : n <= 32 ? 2 : n <= 64 ? 4 : 8; }
int dft_tiles(int m, int kk, bool tr) { return tr ? (kk + 31) / 32 : (m + 15) / 16; }

/*
 * The constant operands in the order the products read them, 8 BF16 per lane
 * and step, so a wave's rows load as 1 KB pieces.  Read as rows of the FP32
 * matrix, every lane of a load touches a cache line of its own, and those
 * accesses were most of a k_dft launch (28 us of which 20 at 64 x 64 x 256,
 * width 32).
 * kind 0: rows of G = [cos; sin] for k_dft (16 cos rows, the same 16 sin rows
 * per tile); 1: columns of G for k_dft_t; 2: Gt (n2 x nt) for k_column, 4
 * steps of 16 per 32-point t tile; 3: Ft (nt x n2), transposed, for k_column's
 * LDS.  Contracted indices past the end are zero; times past nt (kind 2) and
 * columns past n2 (3) repeat the last one.
 */
__global__ void k_pack(const float *__restrict__ G, short *__restrict__ out, long n, int kind, int m, int kk, int steps) {
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += gridDim.x * 256L) {
        const int j = (int)(i % 8), lane = (int)(i / 8 % 64), col = lane & 31, half = lane >> 5;
        const int step = (int)(i / 512 % steps), tile = (int)(i / 512 / steps);
        const int c = 16 * step + 8 * half + j;                /* contracted index */
        float v = 0.f;
        if (kind == 0) {
            const int row = tile * 16 + (col & 15);
            if (row < m && c < kk) v = G[(long)(col < 16 ? row : m + row) * kk + c];
        } else if (kind == 1) {
            const int k = tile * 32 + col;
            if (c < 2 * m && k < kk) v = G[(long)c * kk + k];
        } else if (kind == 2) {                                /* m = n2, kk = nt */
            const int t = min(tile * 32 + col, kk - 1);
            if (c < m) v = G[(long)c * kk + t];
        } else {                                               /* m = nt, kk = n2: rows of tpad */
            const int tpad = (m + 31) / 32 * 32;
            const int t = (int)(i % tpad), nn = min((int)(i / tpad), kk - 1);
            if (t < m) v = G[(long)t * kk + nn];
        }
        out[i] = to_bf16(v);
    }
}
long pack_elems(int kind, int m, int kk, int *steps) {
    *steps = 4;
    switch (kind) {
    case 0: *steps = dft_steps(kk); return (long)dft_tiles(m, kk, false) * *steps * 512;
    case 1: *steps = dft_steps(2 * m); return (long)dft_tiles(m, kk, true) * *steps * 512;
    case 2: return (long)((kk + 31) / 32) * 4 * 512;
    default: return (long)((kk + 15) / 16 * 16) * ((m + 31) / 32 * 32);
    }
}

template <int KS>
void dft_go(bool tr, const void *G, const float *in, float *out, long nunit, int m, int kk, int nq, int h, float sg,
            hipStream_t s) {
    const int tiles = dft_tiles(m, kk, tr);
    /* a wave keeps its rows of G for several units once the chip is full */
    const long blocks = std::max(1L, std::min((nunit + 3) / 4, 4096L / tiles));
    const dim3 grid((unsigned)blocks, (unsigned)tiles);
    const bf16x8 *g = (const bf16x8 *)G;
    if (tr) hipLaunchKernelGGL((k_dft_t<KS>), grid, dim3(256), 0, s, g, in, out, nunit, m, kk, nq, h, sg);
    else if (kk == 16 * KS)
        hipLaunchKernelGGL((k_dft<KS, true>), grid, dim3(256), 0, s, g, in, out, nunit, m, kk, nq, h, sg);
    else hipLaunchKernelGGL((k_dft<KS, false>), grid, dim3(256), 0, s, g, in, out, nunit, m, kk, nq, h, sg);
}

/* ---------------------------------------------------------------------- */
/* weight and bias gradients of a channel map                              */
/* ---------------------------------------------------------------------- */
/*
 * dW[o][i] = sum over samples and points of d[b][o][p] x[b][i][p] (operands
 * rounded to BF16, as k_gemm_bf16 does), db[o] = the FP32 sum of d[b][o][p].
 * Bound by reading d and x once.  Channels lie megabytes apart, so a wave reads
 * 1 KB of one channel at a time (4 points a lane); read in the operands' order
 * instead (128 bytes of 32 channels), without the pass through LDS, the same
 * sums ran at 3.0 TB/s.  At no = ni = 32 and 4.2 M points 206 us (5.2 TB/s); as
 * a product per sample and a bias kernel 515.
 * Workgroups walk chunks of 256 points; the next chunk loads under the
 * products, of which each wave forms 64 points' share.  Each workgroup leaves
 * its sums in part; k_wgrad_sum adds them.
 */
constexpr int WG_WAVES = 4, WG_GRID = 512, WG_MAX = 64, WG_PTS = 256, WG_PITCH = WG_PTS + 8;

template <int OT, int IT>
__global__ void __launch_bounds__(64 * WG_WAVES, OT + IT == 2 ? 4 : 2)
k_wgrad(const float *__restrict__ d, const float *__restrict__ x, float *__restrict__ part, int nb, int no, int ni, int np) {
    constexpr int NE = OT * 32 * (IT * 32 + 1);                /* a workgroup's sums: rows of IT * 32, then db */
    constexpr int NR = 8 * (OT + IT);                          /* channels a wave loads: wave, wave + 4, ... of d's, then x's */
    constexpr int BYTES = 32 * (OT + IT) * WG_PITCH * 2, RED = WG_WAVES * OT * IT * 1024 * 4;
    __shared__ __align__(16) unsigned char smem[BYTES > RED ? BYTES : RED];
    short *st = reinterpret_cast<short *>(smem);
    const int lane = threadIdx.x & 63, col = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    f32x16 acc[OT][IT] = {};
    float sum[8 * OT] = {};
    float4 v[NR];
    const unsigned np4 = 4u * (unsigned)np;
    /* channels past no and ni are nobody's: the last one stands in, and its sums are not read */
    auto load = [&](int b, int p0) {
        const rsrc_t db = buf_of(d + (long)b * no * np), xb = buf_of(x + (long)b * ni * np);
        const unsigned p = 4u * min(p0 + 4 * lane, np - 4);
#pragma unroll
        for (int i = 0; i < NR; ++i)
            v[i] = i < 8 * OT ? buf_ld4(db, p, min(wave + 4 * i, no - 1) * np4)
                              : buf_ld4(xb, p, min(wave + 4 * (i - 8 * OT), ni - 1) * np4);
    };
    const int step = WG_PTS * gridDim.x, pend = WG_PTS * ((np + WG_PTS - 1) / WG_PTS);
    int b = 0, p0 = WG_PTS * blockIdx.x;
    auto wrap = [&] {
        while (p0 >= pend) { p0 -= pend; ++b; }
    };
    wrap();
    load(min(b, nb - 1), p0);
    while (b < nb) {
        const bool in = p0 + 4 * lane < np;                    /* np is a multiple of 4 */
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            if (!in) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (i < 8 * OT) sum[i < 8 * OT ? i : 0] += (v[i].x + v[i].y) + (v[i].z + v[i].w);
            *reinterpret_cast<int2 *>(&st[(wave + 4 * i) * WG_PITCH + 4 * lane]) =
                make_int2(bf16_pair(v[i].x, v[i].y), bf16_pair(v[i].z, v[i].w));
        }
        p0 += step;
        wrap();
        load(min(b, nb - 1), p0);
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const short *at = st + col * WG_PITCH + 64 * wave + 16 * s + 8 * half;
            bf16x8 xo[IT];
#pragma unroll
            for (int j = 0; j < IT; ++j) xo[j] = *reinterpret_cast<const bf16x8 *>(at + 32 * (OT + j) * WG_PITCH);
#pragma unroll
            for (int o = 0; o < OT; ++o) {
                const bf16x8 dd = *reinterpret_cast<const bf16x8 *>(at + 32 * o * WG_PITCH);
#pragma unroll
                for (int j = 0; j < IT; ++j) acc[o][j] = mfma_bf16(dd, xo[j], acc[o][j]);
            }
        }
        __syncthreads();
    }
    float *red = reinterpret_cast<float *>(smem), *out = part + (long)blockIdx.x * NE;
    constexpr int NW = OT * IT * 1024;
#pragma unroll
    for (int o = 0; o < OT; ++o)
#pragma unroll
        for (int j = 0; j < IT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                red[wave * NW + (32 * o + drow(r, half)) * IT * 32 + 32 * j + col] = acc[o][j][r];
#pragma unroll
    for (int i = 0; i < 8 * OT; ++i) {
        float t = sum[i];
#pragma unroll
        for (int k = 32; k > 0; k >>= 1) t += __shfl_xor(t, k);
        if (lane == 0) out[NW + wave + 4 * i] = t;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < NW; e += 64 * WG_WAVES)
        out[e] = (red[e] + red[NW + e]) + (red[2 * NW + e] + red[3 * NW + e]);
}
template <int OT, int IT>
void wgrad_go(const float *d, const float *x, float *dW, float *db, float *ws, int nb, int no, int ni, long np,
              hipStream_t s) {
    const int nwg = (int)std::min((long)WG_GRID, nb * ((np + WG_PTS - 1) / WG_PTS));
    hipLaunchKernelGGL((k_wgrad<OT, IT>), dim3(nwg), dim3(64 * WG_WAVES), 0, s, d, x, ws, nb, no, ni, (int)np);
    hipLaunchKernelGGL(k_wgrad_sum, dim3(OT * (IT * 32 + 1)), dim3(1024), 0, s, ws, nwg, OT * 32, IT * 32, dW, db, no, ni);
}

} // namespace

extern "C" int mpc_sizeof_fno_col(void) { return (int)sizeof(mpc_fno_col); }

extern "C" int mpc_fno_column_fits(int w, int cin, int nt, int n2, int h) {
    return (w == 8 || w == 16 || w == 32 || w == 64) && cin == 4 && nt >= 1 && nt <= CT_MAX && n2 >= 2 && n2 % 2 == 0 &&
           n2 <= CN2_MAX && h >= 1 && h <= 64 && (h & (h - 1)) == 0;
}

/* dh is stored in whole tiles of 32 hidden channels; at width 64 the sums and
 * operands of kind 5 exceed the registers (61 spills) */
extern "C" long mpc_fno_head_ws(int w, int h) {
    return w > 32 || h < 1 || h > CH_MAX || h % 32 ? MPC_EUNSUPP : 4L * CG_MAX * 2 * (h + 1);
}

extern "C" int mpc_fno_column(const mpc_fno_col *a, void *stream) {
    if (!a || a->nb <= 0 || a->npos <= 0 || !a->v || !a->w || (!a->bias && !a->bwd)) return MPC_EINVAL;
    if (!mpc_fno_column_fits(a->width, 4, a->nt, a->n2, a->y || a->dh ? a->h : 1)) return MPC_EUNSUPP;
    /* byte offsets within a sample's activations and mode rows are 32-bit */
    if ((long)a->width * a->npos * std::max(a->nt, a->n2) > (1L << 29) || (long)a->nb * a->npos > (1L << 30))
        return MPC_EUNSUPP;
    if (a->zs && !a->V6) return MPC_EINVAL;
    if ((a->dh || (a->y && a->zs)) && mpc_fno_head_ws(a->width, a->h) < 0) return MPC_EUNSUPP;
    if (a->dh) {
        if ((long)a->h * a->npos * a->nt > (1L << 29)) return MPC_EUNSUPP;
        if (!a->bwd || a->V6 || a->zin || a->y || !a->q1w || !a->q1 || !a->q2w || !a->x || !a->out || !a->Ft || !a->C1 ||
            !a->ws || !a->dq2w || !a->dq2)
            return MPC_EINVAL;
    } else if (a->V6 && !a->Gt) {
        return MPC_EINVAL;
    } else if (a->bwd) {
        if (!a->V6 || !a->out || a->zs || a->y || (a->zin && (!a->Ft || !a->C1))) return MPC_EINVAL;
    } else if (a->y ? (!a->q1w || !a->q1 || !a->q2w || !a->q2 || !a->x || !a->V6) : (!a->Ft || !a->C1 || !a->out)) {
        return MPC_EINVAL;
    }
    hipStream_t s = (hipStream_t)stream;
    switch (a->width) {
    case 8:  return column_w<8>(a, s);
    case 16: return column_w<16>(a, s);
    case 32: return column_w<32>(a, s);
    default: return column_w<64>(a, s);
    }
}

extern "C" int mpc_fno_dft_fits(int m, int kk, int bwd) {
    return m >= 1 && kk >= 1 && (bwd ? 2 * m : kk) <= 128 && m <= (1 << 20) && kk <= (1 << 20);
}

extern "C" long mpc_fno_pack_bytes(int kind, int m, int kk) {
    if (kind < 0 || kind > 3 || m <= 0 || kk <= 0 || (kind < 2 && !mpc_fno_dft_fits(m, kk, kind)) ||
        (kind == 2 && (m > CN2_MAX || kk > CT_MAX)) || (kind == 3 && (kk > CN2_MAX || m > CT_MAX)))
        return MPC_EUNSUPP;
    int steps;
    return 2 * pack_elems(kind, m, kk, &steps);
}

extern "C" int mpc_fno_pack(const float *G, void *out, int kind, int m, int kk, void *stream) {
    if (!G || !out || mpc_fno_pack_bytes(kind, m, kk) <= 0) return MPC_EINVAL;
    int steps;
    const long n = pack_elems(kind, m, kk, &steps);
    hipLaunchKernelGGL(k_pack, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, G, (short *)out, n,
                       kind, m, kk, steps);
    return hipGetLastError() == hipSuccess ? 0 : MPC_EHIP;
}

extern "C" int mpc_fno_dft(const void *G, const float *in, float *out, long nslice, int m, int kk, int nq, int h,
                           int sign, int bwd, void *stream) {
    if (!G || !in || !out || in == out || nslice <= 0 || nq <= 0 || h <= 0 || (sign != 1 && sign != -1)) return MPC_EINVAL;
    /* byte offsets within a slice are 32-bit */
    if (!mpc_fno_dft_fits(m, kk, bwd) || (long)std::max(m, kk) * nq * 2 * h > (1L << 29)) return MPC_EUNSUPP;
    hipStream_t s = (hipStream_t)stream;
    const long nunit = nslice * nq * ((h + 31) / 32);
    const float sg = (float)sign;
    switch (dft_steps(bwd ? 2 * m : kk)) {
    case 1:  dft_go<1>(bwd != 0, G, in, out, nunit, m, kk, nq, h, sg, s); break;
    case 2:  dft_go<2>(bwd != 0, G, in, out, nunit, m, kk, nq, h, sg, s); break;
    case 4:  dft_go<4>(bwd != 0, G, in, out, nunit, m, kk, nq, h, sg, s); break;
    default: dft_go<8>(bwd != 0, G, in, out, nunit, m, kk, nq, h, sg, s); break;
    }
    return hipGetLastError() == hipSuccess ? 0 : MPC_EHIP;
}

extern "C" long mpc_fno_wgrad_ws(int no, int ni, long np) {
    /* a sample's byte offsets are 32-bit */
    if (no < 1 || ni < 1 || no > WG_MAX || ni > WG_MAX || np < 4 || np % 4 || np * std::max(no, ni) > (1L << 29))
        return MPC_EUNSUPP;
    const long oc = (no + 31) / 32 * 32, ic = (ni + 31) / 32 * 32;
    return 4 * WG_GRID * oc * (ic + 1);
}

extern "C" int mpc_fno_wgrad(const float *d, const float *x, float *dW, float *db, float *ws, int nb, int no, int ni,
                             long np, void *stream) {
    if (!d || !x || !dW || !ws || nb <= 0 || np <= 0) return MPC_EINVAL;
    if (mpc_fno_wgrad_ws(no, ni, np) < 0 || (((uintptr_t)d | (uintptr_t)x) & 15)) return MPC_EUNSUPP;
    hipStream_t s = (hipStream_t)stream;
    if (no <= 32 && ni <= 32) wgrad_go<1, 1>(d, x, dW, db, ws, nb, no, ni, np, s);
    else if (no <= 32) wgrad_go<1, 2>(d, x, dW, db, ws, nb, no, ni, np, s);
    else if (ni <= 32) wgrad_go<2, 1>(d, x, dW, db, ws, nb, no, ni, np, s);
    else wgrad_go<2, 2>(d, x, dW, db, ws, nb, no, ni, np, s);
    return hipGetLastError() == hipSuccess ? 0 : MPC_EHIP;
}
