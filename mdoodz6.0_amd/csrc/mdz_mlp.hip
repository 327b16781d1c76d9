/*
 * mdz_mlp.hip -- the surrogate network of the local visco-elastic iteration
 * on the matrix cores of gfx950: training-data generation with the FP64
 * reference rheology (Viscosity, RheologyDensity.c:44-707), forward /
 * backward / Adam kernels (BF16 operands of v_mfma_f32_16x16x16_bf16, FP32
 * accumulation), and the fused grid inference that writes the initial guess
 * of eta_ve for the rheology kernels.
 *
 * Tile convention of the 16x16x16 BF16 matrix instruction, lane l = 16 q + r
 * (r = l mod 16, q = l / 16):
 *   A (M x K):  lane holds A[r][4q .. 4q+3]
 *   B (K x N):  lane holds B[4q .. 4q+3][r]
 *   D (M x N):  lane holds D[4q .. 4q+3][r]
 * A layer's output tile in D layout (neurons x samples) is therefore, after
 * rounding to BF16, exactly the B operand of the next layer's K step: the
 * whole forward pass of 16 samples stays in registers.  One wave handles 16
 * samples; a training block of 4 waves handles 64, and the weight gradients
 * (K = samples) are formed from the block's activations staged in LDS.
 */
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "mdz_kernels.h"
#include "mdz_mlp.h"
#include "mdz_mlp_dev.h"
#include "mdz_viscosity.h"

#define TBLK 256 /* training / inference block: 4 waves x 16 samples */
#define TSAMP 64

/* LDS copies of the weights and activations use padded rows (16 -> 20 and
 * 64 -> 68 BF16 entries) so that the 16 rows one operand load touches fall
 * into different banks */
#define LS16 20
#define LS64 68
#define LDS_W1 0
#define LDS_W2 (LDS_W1 + 64 * LS16)
#define LDS_W3 (LDS_W2 + 64 * LS64)
#define LDS_W4 (LDS_W3 + 64 * LS64)
#define LDS_FWD (LDS_W4 + 16 * LS64) /* end of the forward weights */
#define LDS_W2T LDS_FWD
#define LDS_W3T (LDS_W2T + 64 * LS64)
#define LDS_W4T (LDS_W3T + 64 * LS64)
#define LDS_ALL (LDS_W4T + 64 * LS16)

/* z[mt] = W[16mt .. 16mt+15][:] * B (+ bias), NK K-steps of 16 inputs; W
 * row-major with leading dimension ldw (in LDS); NM output tiles. */
template <int NM, int NK, bool BIAS = true>
__device__ __forceinline__ void dense(const unsigned short *W, int ldw, const bf16x4 *b, const float *bias, f32x4 *z) {
    const int l = threadIdx.x & 63, r = l & 15, q = l >> 4;
#pragma unroll
    for (int mt = 0; mt < NM; mt++) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ks = 0; ks < NK; ks++) acc = mfma(lds4(W + (16 * mt + r) * ldw + 16 * ks + 4 * q), b[ks], acc);
#pragma unroll
        for (int i = 0; i < 4; i++) z[mt][i] = BIAS ? acc[i] + bias[16 * mt + 4 * q + i] : acc[i];
    }
}

/* forward pass of one wave's 16 samples (weights in the padded LDS layout);
 * x = the lane's 4 features (BF16).
 * Returns the pre-activations of the hidden layers and the two outputs in
 * lanes q == 0 (y[0], y[1]). */
__device__ __forceinline__ void mlp_forward(const unsigned short *W, const float *B, bf16x4 x, f32x4 *z1, f32x4 *z2,
                                            f32x4 *z3, f32x4 &y) {
    bf16x4 h[4];
    dense<4, 1>(W + LDS_W1, LS16, &x, B, z1);
#pragma unroll
    for (int t = 0; t < 4; t++) h[t] = pack4(silu4(z1[t]));
    dense<4, 4>(W + LDS_W2, LS64, h, B + 64, z2);
#pragma unroll
    for (int t = 0; t < 4; t++) h[t] = pack4(silu4(z2[t]));
    dense<4, 4>(W + LDS_W3, LS64, h, B + 128, z3);
#pragma unroll
    for (int t = 0; t < 4; t++) h[t] = pack4(silu4(z3[t]));
    dense<1, 4>(W + LDS_W4, LS64, h, B + 192, &y);
}

/* ------------------------------------------------------------------ */
/* features                                                             */
/* ------------------------------------------------------------------ */
__device__ __forceinline__ void mlp_features(double Eii_s, double T_K, double P_Pa, double tau0_Pa, double dt_s,
                                             int phase, double tauy_Pa, float *f) {
    f[0] = (float)((log10(fmax(Eii_s, 1e-30)) + 15.0) / 3.0);
    f[1] = (float)((T_K - 1123.0) / 850.0);
    f[2] = (float)((P_Pa * 1e-9 - 5.0) / 5.0);
    f[3] = (float)((tau0_Pa * 1e-6 - 250.0) / 250.0);
    f[4] = (float)(log10(fmax(dt_s, 1e-30)) - 11.0);
    f[5] = phase == 0 ? 1.0f : 0.0f;
    f[6] = phase == 1 ? 1.0f : 0.0f;
    f[7] = phase == 2 ? 1.0f : 0.0f;
    f[8] = (float)((log10(fmax(tauy_Pa * 1e-6, 1e-3)) - 1.5) / 1.5);
}

/* the lane's 4 features 4q .. 4q+3 (9 .. 15 are zero) */
__device__ __forceinline__ bf16x4 lane_features(const float *f) {
    const int q = (threadIdx.x & 63) >> 4;
    bf16x4 x;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        int k = 4 * q + j;
        x[j] = (short)f2bf(k < MLP_IN ? f[k] : 0.0f);
    }
    return x;
}

/* ------------------------------------------------------------------ */
/* parameter layout                                                     */
/* ------------------------------------------------------------------ */
__device__ __forceinline__ void pack_param(int p, float w, unsigned short *wp, float *bp) {
    unsigned short b = f2bf(w);
    if (p < MLP_OFF_B1) {
        int o = p / MLP_IN, i = p % MLP_IN;
        wp[MLP_WP_W1 + o * 16 + i] = b;
    } else if (p < MLP_OFF_W2) {
        bp[p - MLP_OFF_B1] = w;
    } else if (p < MLP_OFF_B2) {
        int o = (p - MLP_OFF_W2) / 64, i = (p - MLP_OFF_W2) % 64;
        wp[MLP_WP_W2 + o * 64 + i] = b;
        wp[MLP_WP_W2T + i * 64 + o] = b;
    } else if (p < MLP_OFF_W3) {
        bp[64 + p - MLP_OFF_B2] = w;
    } else if (p < MLP_OFF_B3) {
        int o = (p - MLP_OFF_W3) / 64, i = (p - MLP_OFF_W3) % 64;
        wp[MLP_WP_W3 + o * 64 + i] = b;
        wp[MLP_WP_W3T + i * 64 + o] = b;
    } else if (p < MLP_OFF_W4) {
        bp[128 + p - MLP_OFF_B3] = w;
    } else if (p < MLP_OFF_B4) {
        int o = (p - MLP_OFF_W4) / 64, i = (p - MLP_OFF_W4) % 64;
        wp[MLP_WP_W4 + o * 64 + i] = b;
        wp[MLP_WP_W4T + i * 16 + o] = b;
    } else {
        bp[192 + p - MLP_OFF_B4] = w;
    }
}

/* zero the padded buffers, then scatter the blob (one block of 256 threads
 * per part; launched as two kernels) */
__global__ void k_mlp_zero(unsigned short *wp, float *bp) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < MLP_WP_TOTAL; i += gridDim.x * 256) wp[i] = 0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < MLP_BP_TOTAL; i += gridDim.x * 256) bp[i] = 0.0f;
}
__global__ void k_mlp_scatter(const float *__restrict__ blob, unsigned short *wp, float *bp) {
    int p = blockIdx.x * 256 + threadIdx.x;
    if (p < MLP_NPARAMS) pack_param(p, blob[p], wp, bp);
}

void mdz_mlp_pack(const float *blob, unsigned short *wp, float *bp, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_zero, dim3(16), dim3(256), 0, s, wp, bp);
    hipLaunchKernelGGL(k_mlp_scatter, dim3(mdz_div_up(MLP_NPARAMS, 256)), dim3(256), 0, s, blob, wp, bp);
}

/* ------------------------------------------------------------------ */
/* inference form (mdz_mlp.h)                                           */
/* ------------------------------------------------------------------ */
#define LOG2E 1.4426950408889634

/* row position of input neuron n (0..63) within a K-permuted row */
__device__ __forceinline__ int kperm_pos(int n) {
    const int s = n >> 5, m = n & 31;
    return m < 16 ? 32 * s + 8 * (m >> 2) + (m & 3) : 32 * s + 8 * ((m - 16) >> 2) + 4 + (m & 3);
}

__global__ void k_mlp_zero_inf(unsigned short *wi, float *bi) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < MLI_TOTAL; i += gridDim.x * 256) wi[i] = 0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < MLI_B_TOTAL; i += gridDim.x * 256) bi[i] = 0.0f;
}

__global__ void k_mlp_scatter_inf(const float *__restrict__ blob, unsigned short *wi, float *bi) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= MLP_NPARAMS) return;
    const double w = blob[p];
    if (p < MLP_OFF_B1) {
        wi[MLI_W1 + (p / MLP_IN) * 16 + p % MLP_IN] = f2bf((float)(LOG2E * w));
    } else if (p < MLP_OFF_W2) {
        bi[p - MLP_OFF_B1] = (float)(LOG2E * w);
    } else if (p < MLP_OFF_B2) {
        const int o = (p - MLP_OFF_W2) / 64, i = (p - MLP_OFF_W2) % 64;
        wi[MLI_W2 + o * 64 + kperm_pos(i)] = f2bf((float)w);
    } else if (p < MLP_OFF_W3) {
        bi[64 + p - MLP_OFF_B2] = (float)(LOG2E * w);
    } else if (p < MLP_OFF_B3) {
        const int o = (p - MLP_OFF_W3) / 64, i = (p - MLP_OFF_W3) % 64;
        wi[MLI_W3 + o * 64 + kperm_pos(i)] = f2bf((float)w);
    } else if (p < MLP_OFF_W4) {
        bi[128 + p - MLP_OFF_B3] = (float)(LOG2E * w);
    } else if (p < MLP_OFF_B4) {
        const int o = (p - MLP_OFF_W4) / 64, i = (p - MLP_OFF_W4) % 64;
        wi[MLI_W4 + o * 64 + kperm_pos(i)] = f2bf((float)(w / LOG2E));
    } else {
        bi[192 + p - MLP_OFF_B4] = (float)w;
    }
}

void mdz_mlp_pack_inference(const float *blob, unsigned short *wi, float *bi, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_zero_inf, dim3(16), dim3(256), 0, s, wi, bi);
    hipLaunchKernelGGL(k_mlp_scatter_inf, dim3(mdz_div_up(MLP_NPARAMS, 256)), dim3(256), 0, s, blob, wi, bi);
}

/* LDS copy of the inference form: rows padded to 20 (W1) and 72 (W2..W4)
 * BF16 entries, so that the 16-byte operand loads of 8 consecutive rows fall
 * into distinct banks */
#define LI16 20
#define LI64 72
#define LDI_W1 0
#define LDI_W2 (LDI_W1 + 64 * LI16)
#define LDI_W3 (LDI_W2 + 64 * LI64)
#define LDI_W4 (LDI_W3 + 64 * LI64)
#define LDI_TOTAL (LDI_W4 + 16 * LI64)

__device__ __forceinline__ int lds_index_inf(int i) {
    if (i < MLI_W2) return LDI_W1 + (i / 16) * LI16 + i % 16;
    if (i < MLI_W3) { i -= MLI_W2; return LDI_W2 + (i / 64) * LI64 + i % 64; }
    if (i < MLI_W4) { i -= MLI_W3; return LDI_W3 + (i / 64) * LI64 + i % 64; }
    i -= MLI_W4;
    return LDI_W4 + (i / 64) * LI64 + i % 64;
}

/* the inference weights into LDS, two entries per thread and step */
__device__ __forceinline__ void load_weights_inf(DevMLPI w, unsigned short *sW, float *sB) {
    const unsigned *src = (const unsigned *)w.w;
    for (int i = threadIdx.x; i < MLI_TOTAL / 2; i += blockDim.x) *(unsigned *)(sW + lds_index_inf(2 * i)) = src[i];
    for (int i = threadIdx.x; i < MLI_B_TOTAL; i += blockDim.x) sB[i] = w.b[i];
}

/* dense kernel-layout index -> padded LDS index */
__device__ __forceinline__ int lds_index(int i) {
    if (i < MLP_WP_W2) return LDS_W1 + (i / 16) * LS16 + i % 16;
    if (i < MLP_WP_W3) { i -= MLP_WP_W2; return LDS_W2 + (i / 64) * LS64 + i % 64; }
    if (i < MLP_WP_W4) { i -= MLP_WP_W3; return LDS_W3 + (i / 64) * LS64 + i % 64; }
    if (i < MLP_WP_W2T) { i -= MLP_WP_W4; return LDS_W4 + (i / 64) * LS64 + i % 64; }
    if (i < MLP_WP_W3T) { i -= MLP_WP_W2T; return LDS_W2T + (i / 64) * LS64 + i % 64; }
    if (i < MLP_WP_W4T) { i -= MLP_WP_W3T; return LDS_W3T + (i / 64) * LS64 + i % 64; }
    i -= MLP_WP_W4T;
    return LDS_W4T + (i / 16) * LS16 + i % 16;
}

/* weights into LDS: the forward ones (nw = MLP_WP_W2T) or all (MLP_WP_TOTAL),
 * eight entries per thread and step (rows are 16 or 64 long: the eight share
 * one; padded rows start on 8 bytes) */
__device__ __forceinline__ void load_weights(DevMLPW w, unsigned short *sW, float *sB, int nw) {
    const uint4 *src = (const uint4 *)w.wp;
    for (int i = threadIdx.x; i < nw / 8; i += blockDim.x) {
        const uint4 v = src[i];
        uint2 *d = (uint2 *)(sW + lds_index(8 * i));
        d[0] = uint2{v.x, v.y};
        d[1] = uint2{v.z, v.w};
    }
    for (int i = threadIdx.x; i < MLP_BP_TOTAL; i += blockDim.x) sB[i] = w.bp[i];
}

/* ------------------------------------------------------------------ */
/* training step                                                        */
/* ------------------------------------------------------------------ */
__device__ __forceinline__ long long sample_index(long long j, long long n, unsigned long long mul,
                                                  unsigned long long add) {
    return (long long)((((unsigned long long)j % (unsigned long long)n) * mul + add) % (unsigned long long)n);
}

#define TWAVES 4                 /* waves of a training block, each on its own 32 samples at a time */
#define TBLOCKS 256              /* most training blocks: one per CU */
#define TSW 36                   /* row stride of 32 staged samples */
#define TWAVE_LDS (4 * 64 * TSW + 2 * 16 * TSW) /* H1 H2 H3 D, X D4 */

/* dense() of two groups of 16 samples, the weights read once */
template <int NM, int NK, bool BIAS>
__device__ __forceinline__ void dense_x2(const unsigned short *W, int ldw, const bf16x4 (*b)[NK], const float *bias,
                                         f32x4 (*z)[4]) {
    const int l = threadIdx.x & 63, r = l & 15, q = l >> 4;
#pragma unroll
    for (int mt = 0; mt < NM; mt++) {
        f32x4 acc[2] = {};
#pragma unroll
        for (int ks = 0; ks < NK; ks++) {
            const bf16x4 a = lds4(W + (16 * mt + r) * ldw + 16 * ks + 4 * q);
#pragma unroll
            for (int g = 0; g < 2; g++) acc[g] = mfma(a, b[g][ks], acc[g]);
        }
#pragma unroll
        for (int g = 0; g < 2; g++)
#pragma unroll
            for (int i = 0; i < 4; i++) z[g][mt][i] = BIAS ? acc[g][i] + bias[16 * mt + 4 * q + i] : acc[g][i];
    }
}

/* 8 staged samples of a row: the lane's operand of a 16 x 16 x 32 product */
__device__ __forceinline__ bf16x8 lds8(const unsigned short *p) {
    const bf16x4 a = lds4(p), b = lds4(p + 4);
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

/* a hidden layer's activations and (in z) their derivative, the activations
 * also staged [row][sample] for the weight gradient */
__device__ __forceinline__ void train_act(f32x4 (*z)[4], bf16x4 (*h)[4], unsigned short *Hs) {
    const int l = threadIdx.x & 63, r = l & 15, q = l >> 4;
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
        for (int t = 0; t < 4; t++) {
            f32x4 v;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float s = sigmoidf_(z[g][t][i]);
                v[i] = z[g][t][i] * s;
                z[g][t][i] = s * (1.0f + z[g][t][i] * (1.0f - s));
            }
            h[g][t] = pack4(v);
#pragma unroll
            for (int i = 0; i < 4; i++) Hs[(16 * t + 4 * q + i) * TSW + 16 * g + r] = (unsigned short)h[g][t][i];
        }
}

/* LDS ordering between the lanes of one wave.  DS instructions of a wave run
 * in the order they are issued, so that nothing has to be waited for; the
 * fence (no instruction at this scope) keeps the compiler from moving an
 * access across. */
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

/* sum of a staged row over its 32 samples */
__device__ __forceinline__ float row_sum(const unsigned short *row) {
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < 32; k += 4) {
        const bf16x4 v = lds4(row + k);
#pragma unroll
        for (int i = 0; i < 4; i++) sum += bf2f((unsigned short)v[i]);
    }
    return sum;
}

/* a hidden layer's output gradients d (times the activation's derivative),
 * rounded and staged */
__device__ __forceinline__ void train_grad(const f32x4 (*d)[4], const f32x4 (*dact)[4], bf16x4 (*bd)[4],
                                           unsigned short *Ds) {
    const int l = threadIdx.x & 63, r = l & 15, q = l >> 4;
    wave_lds_order();
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
        for (int t = 0; t < 4; t++) {
            bd[g][t] = pack4(d[g][t] * dact[g][t]);
#pragma unroll
            for (int i = 0; i < 4; i++) Ds[(16 * t + 4 * q + i) * TSW + 16 * g + r] = (unsigned short)bd[g][t][i];
        }
    wave_lds_order();
}

/* g[mt][nt] += D H^T over the 32 staged samples */
__device__ __forceinline__ void weight_grad(const unsigned short *Ds, const unsigned short *Hs, f32x4 (*g)[4]) {
    const int l = threadIdx.x & 63, r = l & 15, q = l >> 4;
    bf16x8 h[4];
#pragma unroll
    for (int nt = 0; nt < 4; nt++) h[nt] = lds8(Hs + (16 * nt + r) * TSW + 8 * q);
#pragma unroll
    for (int mt = 0; mt < 4; mt++) {
        const bf16x8 a = lds8(Ds + (16 * mt + r) * TSW + 8 * q);
#pragma unroll
        for (int nt = 0; nt < 4; nt++) g[mt][nt] = mfma32(a, h[nt], g[mt][nt]);
    }
}

/* Forward and backward pass of `tiles` tiles of 32 samples, one wave per
 * tile; partial[block][p]: the block's gradient of sum((y - t)^2) / (2
 * batch), loss[block]: its sum of squared errors.
 *
 * The matrix products of a tile are about 200 instructions; what bounds the
 * kernel is the chain through the layers and what surrounds the samples.
 * So the waves are independent (a tile's activations are transposed through
 * the wave's own LDS, no barrier), two groups of 16 samples run through the
 * layers side by side, four waves to a CU share one copy of the weights
 * (eight halve the registers and spill), and a wave keeps its weight
 * gradients in 160 accumulators over all of its tiles: 256 partial gradients
 * of 36 KB a step, whatever the batch.  The sums over the four waves rotate
 * through the parameters' eight parts, in an order that depends on nothing.
 * Measured, batch 65 536: a step 43 us with its reduction and Adam (47 with
 * one group a wave), against 105 for one block per 64 samples that wrote
 * 1024 partial gradients, a reduction of 37 MB and Adam.
 *
 * Up to a tile per CU (batches of 8192) a tile has a block to itself: its
 * other waves help to read the weights, and its gradient goes from the
 * registers to the partials, without the eight rounds and their barriers.
 * A step of 1024 samples takes 18 us, 26 with four tiles a block (25 for the
 * one block per 64 samples), one of 8192 26 against 28 (31). */
__global__ void __launch_bounds__(TWAVES * 64, 1) k_mlp_train_step(
    const float *__restrict__ X, const float *__restrict__ Y, long long n, long long first, unsigned long long mul,
    unsigned long long add, long long stride, int tiles, float inv_batch, DevMLPW w, float *__restrict__ partial,
    float *__restrict__ loss) {
    __shared__ __attribute__((aligned(16))) unsigned short sW[LDS_ALL];
    __shared__ float sB[MLP_BP_TOTAL];
    __shared__ __attribute__((aligned(16))) unsigned short sA[TWAVES * TWAVE_LDS];
    __shared__ float sLoss[TWAVES];
    static_assert(TWAVES == 4 && sizeof(unsigned short) * TWAVES * TWAVE_LDS >= sizeof(float) * MLP_NPARAMS,
                  "the gradients' sums");
    const int l = threadIdx.x & 63, r = l & 15, q = l >> 4, wv = threadIdx.x >> 6;
    /* (all reads of the weights and of the first samples in flight at once:
     * one round trip instead of ten) */
    constexpr int WL = (MLP_WP_TOTAL / 8 + TWAVES * 64 - 1) / (TWAVES * 64);
    uint4 wl[WL];
#pragma unroll
    for (int k = 0; k < WL; k++)
        wl[k] = ((const uint4 *)w.wp)[min((int)threadIdx.x + k * TWAVES * 64, MLP_WP_TOTAL / 8 - 1)];
    const float bl = w.bp[min((int)threadIdx.x, MLP_BP_TOTAL - 1)];
    unsigned short *H1s = sA + wv * TWAVE_LDS, *H2s = H1s + 64 * TSW, *H3s = H2s + 64 * TSW, *Ds = H3s + 64 * TSW,
                   *Xs = Ds + 64 * TSW, *D4s = Xs + 16 * TSW;
    f32x4 g1[4] = {}, g2[4][4] = {}, g3[4][4] = {}, g4[4] = {};
    float gb1 = 0.0f, gb2 = 0.0f, gb3 = 0.0f, gb4 = 0.0f, se = 0.0f;
    const bool solo = (int)gridDim.x >= tiles; /* a block for each tile */
    int tile = solo ? (wv == 0 ? (int)blockIdx.x : tiles) : blockIdx.x * TWAVES + wv;
    long long idx[2];
    float f[2][4], tgt[2][2] = {};
#pragma unroll
    for (int g = 0; g < 2; g++) idx[g] = sample_index(first + 32LL * tile + 16 * g + r, n, mul, add);
    auto fetch = [&] {
#pragma unroll
        for (int g = 0; g < 2; g++) {
#pragma unroll
            for (int j = 0; j < 4; j++) f[g][j] = 4 * q + j < MLP_IN ? X[idx[g] * MLP_IN + 4 * q + j] : 0.0f;
            if (q == 0) {
                tgt[g][0] = Y[idx[g] * 2];
                tgt[g][1] = Y[idx[g] * 2 + 1];
            }
        }
    };
    if (tile < tiles) fetch();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < WL; k++) {
        const int i = threadIdx.x + k * TWAVES * 64;
        if (i < MLP_WP_TOTAL / 8) {
            uint2 *o = (uint2 *)(sW + lds_index(8 * i));
            o[0] = uint2{wl[k].x, wl[k].y};
            o[1] = uint2{wl[k].z, wl[k].w};
        }
    }
    static_assert(MLP_BP_TOTAL <= TWAVES * 64, "one bias a thread");
    if (threadIdx.x < MLP_BP_TOTAL) sB[threadIdx.x] = bl;
    __syncthreads();
    if (solo && wv) return; /* (no barrier follows for the first wave) */
    for (; tile < tiles; tile += gridDim.x * TWAVES) {
        bf16x4 x[2][1];
        float t[2][2];
#pragma unroll
        for (int g = 0; g < 2; g++) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                x[g][0][j] = (short)f2bf(f[g][j]);
                Xs[(4 * q + j) * TSW + 16 * g + r] = (unsigned short)x[g][0][j];
            }
            t[g][0] = tgt[g][0];
            t[g][1] = tgt[g][1];
            idx[g] += stride; /* the wave's next tile, read ahead */
            if (idx[g] >= n) idx[g] -= n;
        }
        if (tile + (int)gridDim.x * TWAVES < tiles) fetch();

        /* forward; z1..z3 become the activations' derivatives */
        f32x4 z1[2][4], z2[2][4], z3[2][4], d[2][4];
        bf16x4 h[2][4];
        dense_x2<4, 1, true>(sW + LDS_W1, LS16, x, sB, z1);
        train_act(z1, h, H1s);
        dense_x2<4, 4, true>(sW + LDS_W2, LS64, h, sB + 64, z2);
        train_act(z2, h, H2s);
        dense_x2<4, 4, true>(sW + LDS_W3, LS64, h, sB + 128, z3);
        train_act(z3, h, H3s);
        dense_x2<1, 4, true>(sW + LDS_W4, LS64, h, sB + 192, d);

        /* loss and output gradient (rows 0, 1 in lanes q == 0) */
        bf16x4 b4[2][1], bd[2][4];
#pragma unroll
        for (int g = 0; g < 2; g++) {
            f32x4 e = {0.0f, 0.0f, 0.0f, 0.0f};
            if (q == 0) {
                const float e0 = d[g][0][0] - t[g][0], e1 = d[g][0][1] - t[g][1];
                se += e0 * e0 + e1 * e1;
                e[0] = e0 * inv_batch;
                e[1] = e1 * inv_batch;
            }
            b4[g][0] = pack4(e);
#pragma unroll
            for (int i = 0; i < 4; i++) D4s[(4 * q + i) * TSW + 16 * g + r] = (unsigned short)b4[g][0][i];
        }
        wave_lds_order();
        gb4 += row_sum(D4s + r * TSW);
        {
            const bf16x8 a = lds8(D4s + r * TSW + 8 * q);
#pragma unroll
            for (int nt = 0; nt < 4; nt++) g4[nt] = mfma32(a, lds8(H3s + (16 * nt + r) * TSW + 8 * q), g4[nt]);
        }
        /* backward through the hidden layers */
        dense_x2<4, 1, false>(sW + LDS_W4T, LS16, b4, nullptr, d);
        train_grad(d, z3, bd, Ds);
        gb3 += row_sum(Ds + l * TSW);
        weight_grad(Ds, H2s, g3);
        dense_x2<4, 4, false>(sW + LDS_W3T, LS64, bd, nullptr, d);
        train_grad(d, z2, bd, Ds);
        gb2 += row_sum(Ds + l * TSW);
        weight_grad(Ds, H1s, g2);
        dense_x2<4, 4, false>(sW + LDS_W2T, LS64, bd, nullptr, d);
        train_grad(d, z1, bd, Ds);
        gb1 += row_sum(Ds + l * TSW);
        const bf16x8 xt = lds8(Xs + r * TSW + 8 * q);
#pragma unroll
        for (int mt = 0; mt < 4; mt++) g1[mt] = mfma32(lds8(Ds + (16 * mt + r) * TSW + 8 * q), xt, g1[mt]);
        wave_lds_order();
    }

    float *P = partial + (size_t)blockIdx.x * MLP_NPARAMS;
    /* part 0..7 of the wave's gradient: put(parameter, value) */
    auto each = [&](int part, auto &&put) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
            if (part == c) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int row = 16 * c + 4 * q + i;
                    if (r < MLP_IN) put(MLP_OFF_W1 + row * MLP_IN + r, g1[c][i]);
#pragma unroll
                    for (int nt = 0; nt < 4; nt++) put(MLP_OFF_W2 + row * 64 + 16 * nt + r, g2[c][nt][i]);
                }
            }
            if (part == c + 4) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int row = 16 * c + 4 * q + i;
#pragma unroll
                    for (int nt = 0; nt < 4; nt++) put(MLP_OFF_W3 + row * 64 + 16 * nt + r, g3[c][nt][i]);
                }
                if (q == 0) {
                    put(MLP_OFF_W4 + 16 * c + r, g4[c][0]);
                    put(MLP_OFF_W4 + 64 + 16 * c + r, g4[c][1]);
                }
            }
        }
        if (part == 0) put(MLP_OFF_B1 + l, gb1);
        if (part == 1) put(MLP_OFF_B2 + l, gb2);
        if (part == 2) put(MLP_OFF_B3 + l, gb3);
        if (part == 3 && l < MLP_OUT) put(MLP_OFF_B4 + l, gb4);
    };
    for (int o = 32; o > 0; o >>= 1) se += __shfl_xor(se, o, 64);
    if (solo) {
#pragma unroll
        for (int part = 0; part < 8; part++) each(part, [&](int p, float v) { P[p] = v; });
        if (l == 0) loss[blockIdx.x] = se;
        return;
    }
    /* the block's gradient: wave wv adds part (2 wv + k) mod 8 in round k (the
     * first two rounds are the first to touch a part) */
    float *sum = (float *)sA;
#pragma unroll 1
    for (int k = 0; k < 8; k++) {
        __syncthreads();
        each((2 * wv + k) & 7, [&](int p, float v) { sum[p] = k > 1 ? sum[p] + v : v; });
    }
    if (l == 0) sLoss[wv] = se;
    __syncthreads();
    for (int p = threadIdx.x; p < MLP_NPARAMS; p += TWAVES * 64) P[p] = sum[p];
    if (threadIdx.x == 0) {
        float s = 0.0f;
        for (int i = 0; i < TWAVES; i++) s += sLoss[i];
        loss[blockIdx.x] = s;
    }
}

/* Adam (Kingma & Ba 2015) on an FP32 master weight; refreshes the BF16
 * kernel copies */
struct AdamStep {
    float *w, *m, *v;
    float lr, b1, b2, eps, c1, c2;
    unsigned short *wp;
    float *bp;
};
__device__ __forceinline__ void adam_param(const AdamStep &a, int p, float gp) {
    const float mp = a.b1 * a.m[p] + (1.0f - a.b1) * gp;
    const float vp = a.b2 * a.v[p] + (1.0f - a.b2) * gp * gp;
    a.m[p] = mp;
    a.v[p] = vp;
    const float wn = a.w[p] - a.lr * (mp / a.c1) / (sqrtf(vp / a.c2) + a.eps);
    a.w[p] = wn;
    pack_param(p, wn, a.wp, a.bp);
}

/* g[p] = sum over blocks of partial[block][p]; loss_acc += sum of the block
 * losses; with ADAM the parameters take their step at once.  A block reduces
 * 64 parameters: its eight waves take every eighth partial (four independent
 * accumulators each), then the slices are added in a fixed order, so the
 * result does not depend on scheduling. */
#define RED_P 64
#define RED_W 8
template <bool ADAM>
__global__ void __launch_bounds__(RED_P *RED_W) k_mlp_reduce(const float *__restrict__ partial, int nblocks,
                                                             float *__restrict__ g, const float *__restrict__ loss,
                                                             double *loss_acc, AdamStep adam) {
    __shared__ float sp[RED_W][RED_P];
    const int pl = threadIdx.x & (RED_P - 1), sl = threadIdx.x >> 6;
    const int p = blockIdx.x * RED_P + pl;
    float a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (p < MLP_NPARAMS) {
        int b = sl;
        for (; b + 7 * RED_W < nblocks; b += 8 * RED_W) {
            float x[8];
#pragma unroll
            for (int u = 0; u < 8; u++) x[u] = partial[(size_t)(b + u * RED_W) * MLP_NPARAMS + p];
#pragma unroll
            for (int u = 0; u < 8; u++) a[u & 3] += x[u];
        }
        for (; b < nblocks; b += RED_W) a[0] += partial[(size_t)b * MLP_NPARAMS + p];
    }
    sp[sl][pl] = (a[0] + a[1]) + (a[2] + a[3]);
    __syncthreads();
    if (sl == 0 && p < MLP_NPARAMS) {
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < RED_W; k++) s += sp[k][pl];
        g[p] = s;
        if (ADAM) adam_param(adam, p, s);
    }
    if (blockIdx.x == 0 && sl == 1 && loss_acc) {
        double s = 0.0;
        for (int b = pl; b < nblocks; b += 64) s += loss[b];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (pl == 0) *loss_acc += s;
    }
}

__global__ void k_mlp_adam(AdamStep a, const float *__restrict__ g) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p < MLP_NPARAMS) adam_param(a, p, g[p]);
}

/* forward pass over stored samples (outputs Y[n][2]) */
__global__ void __launch_bounds__(TBLK) k_mlp_predict(const float *__restrict__ X, long long first, long long count,
                                                      DevMLPW w, float *__restrict__ Yout) {
    __shared__ __attribute__((aligned(16))) unsigned short sW[LDS_FWD];
    __shared__ float sB[MLP_BP_TOTAL];
    load_weights(w, sW, sB, MLP_WP_W2T);
    __syncthreads();
    const int l = threadIdx.x & 63, r = l & 15, q = l >> 4, wv = threadIdx.x >> 6;
    const long long j = (long long)blockIdx.x * TSAMP + 16 * wv + r;
    float f[MLP_IN];
#pragma unroll
    for (int k = 0; k < MLP_IN; k++) f[k] = j < count ? X[(first + j) * MLP_IN + k] : 0.0f;
    f32x4 z1[4], z2[4], z3[4], y;
    mlp_forward(sW, sB, lane_features(f), z1, z2, z3, y);
    if (q == 0 && j < count) {
        Yout[j * 2] = y[0];
        Yout[j * 2 + 1] = y[1];
    }
}

/* ------------------------------------------------------------------ */
/* training data: the FP64 reference rheology on sampled inputs         */
/* ------------------------------------------------------------------ */
__device__ __forceinline__ unsigned long long splitmix(unsigned long long x) {
    x += 0x9e3779b97f4a7c15ULL;
    x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ULL;
    x = (x ^ (x >> 27)) * 0x94d049bb133111ebULL;
    return x ^ (x >> 31);
}
__device__ __forceinline__ double urand(unsigned long long seed, long long i, int k) {
    return (double)(splitmix(seed ^ splitmix((unsigned long long)i * 16ULL + (unsigned long long)k)) >> 11) *
           (1.0 / 9007199254740992.0);
}

__global__ void k_mlp_generate(long long first, long long count, unsigned long long seed, const mat_prop *mt,
                               DevParams prm, float *__restrict__ X, float *__restrict__ Y) {
    const long long j = (long long)blockIdx.x * 256 + threadIdx.x;
    if (j >= count) return;
    const long long i = first + j;
    /* SI draws */
    const double lE = -18.0 + 6.0 * urand(seed, i, 0);
    const double T_K = 273.0 + 1700.0 * urand(seed, i, 1);
    const double P_Pa = 10.0e9 * urand(seed, i, 2);
    const double tau0 = 500.0e6 * urand(seed, i, 3);
    const double dt_s = pow(10.0, 10.0 + 2.0 * urand(seed, i, 4));
    int phase = (int)(3.0 * urand(seed, i, 5));
    phase = phase > 2 ? 2 : phase;
    const double coh = 5.0e6 + 45.0e6 * urand(seed, i, 6);
    const double fric = (10.0 + 25.0 * urand(seed, i, 7)) * M_PI / 180.0;
    /* nondimensional local update (pure shear; the old stress enters the
     * effective strain rate already) */
    DevParams p = prm;
    p.dt = dt_s / prm.st;
    p.rheo_mode = MDZ_RHEO_FP64;
    const double E = pow(10.0, lE) / prm.sE;
    const double P = P_Pa / prm.sS, T = T_K / prm.sT, t0 = tau0 / prm.sS, C = coh / prm.sS;
    VGuess gs;
    gs.mode = MDZ_RHEO_FP64;
    gs.factor = 0.0;
    gs.gdot = 0.0;
    VOut o;
    mdz_viscosity(phase, mt->mu[phase], T, P, mt->gs_ref[phase], 0.0, 0.0, E, -E, 0.0, E, -E, 0.0, t0, -t0, 0.0, mt, p,
                  0.0, fric, C, P, mt->bet[phase], gs, o);
    float f[MLP_IN];
    mlp_features(pow(10.0, lE), T_K, P_Pa, tau0, dt_s, phase, coh * cos(fric) + P_Pa * sin(fric), f);
#pragma unroll
    for (int k = 0; k < MLP_IN; k++) X[j * MLP_IN + k] = f[k];
    Y[j * 2] = (float)(4.0 * log10(o.eta_ve / o.eta_up));
    /* the plastic multiplier relative to the return map's closed-form start
     * (0 without yielding, and for a linear return map, whose start is the root) */
    Y[j * 2 + 1] = o.gdot0 > 0.0 && o.gdot > 0.0 ? (float)fmin(fmax(4.0 * log10(o.gdot / o.gdot0), -8.0), 8.0) : 0.0f;
}

/* ------------------------------------------------------------------ */
/* grid inference: initial guess of eta_ve                              */
/* ------------------------------------------------------------------ */
#define GBLK 256 /* grid inference: 4 waves x 64 nodes */

/* One node's entries of the guess arrays: the factors for its phase ph,
 * 0 (the reference's guess) for the others. */
__device__ __forceinline__ void put_guess(float *guess, float *gguess, size_t n, int node, int nph, int ph, float y0,
                                          float y1) {
    const float fac = guess_factor(ph, y0), gd = guess_gdot(ph, y1);
    for (int p = 0; p < nph; p++) {
        guess[(size_t)p * n + node] = p == ph ? fac : 0.0f;
        gguess[(size_t)p * n + node] = p == ph ? gd : 0.0f;
    }
}

/* Grid inference at the centroids, 64 nodes per wave: one feature vector
 * per lane staged through LDS, four 16-sample groups sharing every weight
 * operand, the guesses of the dominant phase written per phase (factor on
 * the reference's eta_ve guess, then the initial plastic multiplier) and
 * the outputs kept for the vertices. */
__global__ void __launch_bounds__(GBLK) k_mlp_guess(DevGrid g, DevParams prm, DevMLPI w, const PhaseK *__restrict__ pk,
                                                   SpreadConst sc, float *__restrict__ guess) {
    __shared__ __attribute__((aligned(16))) unsigned short sW[LDI_TOTAL];
    __shared__ __attribute__((aligned(16))) float sB[MLI_B_TOTAL];
    __shared__ __attribute__((aligned(16))) unsigned short sX[4][64 * GS]; /* per wave: 64 samples x 16 features */
    __shared__ float sY0[4][64], sY1[4][64];                               /* per wave: network outputs */
    load_weights_inf(w, sW, sB);
    const int l = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int n = g.ncx * g.ncz;
    const int ntiles = (n + GBLK - 1) / GBLK;
    const int nph = min(prm.Nb_phases, g.nph);
    float *gguess = guess + (size_t)g.nph * n;
    /* grid-stride over tiles of 256 nodes: the weights are staged once per block */
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int node = tile * GBLK + threadIdx.x;
        const bool inside = node < n;
        float f[MLP_IN];
        int ph = -1;
        if (inside) ph = guess_features<true>(g, prm, pk, sc, node, n, f);
        else
#pragma unroll
            for (int k = 0; k < MLP_IN; k++) f[k] = 0.0f;
        stage_features(sX[wv], f);
        __syncthreads();
        /* a wave none of whose nodes takes the network's guess skips it */
        const bool run = __any(ph >= 0);
        if (run)
            net_infer64(sW + LDI_W1, LI16, sW + LDI_W2, sW + LDI_W3, sW + LDI_W4, LI64, sB, sX[wv], sY0[wv], sY1[wv]);
        __syncthreads();
        if (inside) {
            const float y0 = ph >= 0 ? sY0[wv][l] : 0.0f, y1 = ph >= 0 ? sY1[wv][l] : 0.0f;
            w.cn[node] = CellNet{y0, y1, ph, 0};
            put_guess(guess, gguess, (size_t)n, node, nph, ph, y0, y1);
        }
    }
}

/* The vertices' guess from the centroids' network outputs (vertex_net). */
__global__ void __launch_bounds__(256) k_guess_vertices(DevGrid g, DevParams prm, const CellNet *__restrict__ cn,
                                                        float *__restrict__ guess) {
    const int node = blockIdx.x * 256 + threadIdx.x;
    const int n = g.Nx * g.Nz;
    if (node >= n) return;
    const int nph = min(prm.Nb_phases, g.nph);
    float y0, y1;
    const int ph = vertex_net(g, prm, cn, node, y0, y1);
    put_guess(guess, guess + (size_t)g.nph * n, (size_t)n, node, nph, ph, y0, y1);
}

void mdz_launch_mlp_guess(const DevGrid &g, const DevParams &prm, DevMLPI w, const void *d_pk, double R,
                          float *guess_n, float *guess_s, hipStream_t s) {
    const SpreadConst sc = spread_const(R, prm.sT, prm.dt, prm.iselastic && prm.step != 0);
    const int nc = g.ncx * g.ncz, nv = g.Nx * g.Nz;
    const int cap = 1024; /* 4 blocks per CU */
    const int bc = mdz_div_up(nc, GBLK);
    hipLaunchKernelGGL(k_mlp_guess, dim3(bc < cap ? bc : cap), dim3(GBLK), 0, s, g, prm, w, (const PhaseK *)d_pk, sc,
                       guess_n);
    hipLaunchKernelGGL(k_guess_vertices, dim3(mdz_div_up(nv, 256)), dim3(256), 0, s, g, prm, (const CellNet *)w.cn,
                       guess_s);
}

/* The inference form on stored samples (features X[n][9]): outputs Y[n][2],
 * 64 samples per wave -- the grid guess's network on inputs a test chooses. */
__global__ void __launch_bounds__(GBLK) k_mlp_predict_inf(const float *__restrict__ X, long long first,
                                                          long long count, DevMLPI w, float *__restrict__ Yout) {
    __shared__ __attribute__((aligned(16))) unsigned short sW[LDI_TOTAL];
    __shared__ __attribute__((aligned(16))) float sB[MLI_B_TOTAL];
    __shared__ __attribute__((aligned(16))) unsigned short sX[4][64 * GS];
    __shared__ float sY0[4][64], sY1[4][64];
    load_weights_inf(w, sW, sB);
    const int l = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const long long j = (long long)blockIdx.x * GBLK + threadIdx.x;
    float f[MLP_IN];
#pragma unroll
    for (int k = 0; k < MLP_IN; k++) f[k] = j < count ? X[(first + j) * MLP_IN + k] : 0.0f;
    stage_features(sX[wv], f);
    __syncthreads();
    net_infer64(sW + LDI_W1, LI16, sW + LDI_W2, sW + LDI_W3, sW + LDI_W4, LI64, sB, sX[wv], sY0[wv], sY1[wv]);
    __syncthreads();
    if (j < count) {
        Yout[j * 2] = sY0[wv][l];
        Yout[j * 2 + 1] = sY1[wv][l];
    }
}

/* ------------------------------------------------------------------ */
/* host API                                                             */
/* ------------------------------------------------------------------ */
struct mdz_mlp {
    hipStream_t s;
    float *w, *m, *v, *g;           /* master weights, Adam moments, gradient */
    unsigned short *wp;
    float *bp;
    float *partial, *loss;          /* per-block gradient / loss */
    int partial_blocks;
    double *loss_acc;
    float *X, *Y;                   /* dataset */
    long long n, cap;
    mat_prop *d_mat;
    DevParams prm;
    int t;                          /* Adam step */
};

#define MCHK(x)                                                                                   \
    do {                                                                                          \
        if ((x) != hipSuccess) return mdz_error(MDZ_EHIP, "surrogate network: " #x " failed");    \
    } while (0)

extern "C" int mdz_mlp_create(mdz_mlp **out, const mat_prop *materials, const params *model, const scale *scaling) {
    if (!out || !materials || !model || !scaling) return mdz_error(MDZ_EINVAL, "mdz_mlp_create: NULL argument");
    if (materials->Nb_phases < 3 && model->Nb_phases < 3)
        return mdz_error(MDZ_EINVAL, "mdz_mlp_create: the network encodes three phases");
    mdz_mlp *n = (mdz_mlp *)calloc(1, sizeof(mdz_mlp));
    if (!n) return mdz_error(MDZ_ENOMEM, "mdz_mlp_create");
    *out = n;
    MCHK(hipStreamCreate(&n->s));
    MCHK(hipMalloc((void **)&n->w, MLP_NPARAMS * 4));
    MCHK(hipMalloc((void **)&n->m, MLP_NPARAMS * 4));
    MCHK(hipMalloc((void **)&n->v, MLP_NPARAMS * 4));
    MCHK(hipMalloc((void **)&n->g, MLP_NPARAMS * 4));
    MCHK(hipMalloc((void **)&n->wp, MLP_WP_TOTAL * 2));
    MCHK(hipMalloc((void **)&n->bp, MLP_BP_TOTAL * 4));
    MCHK(hipMalloc((void **)&n->loss_acc, 8));
    MCHK(hipMalloc((void **)&n->d_mat, sizeof(mat_prop)));
    MCHK(hipMemcpy(n->d_mat, materials, sizeof(mat_prop), hipMemcpyHostToDevice));
    DevParams &p = n->prm;
    memset(&p, 0, sizeof(p));
    p.dt = model->dt; p.mineta = model->mineta; p.maxeta = model->maxeta;
    p.sT = scaling->T; p.sE = scaling->E; p.seta = scaling->eta; p.sS = scaling->S; p.sL = scaling->L; p.st = scaling->t;
    p.step = 1; p.iselastic = 1; p.Nb_phases = 3;
    return MDZ_OK;
}

extern "C" void mdz_mlp_destroy(mdz_mlp *n) {
    if (!n) return;
    hipStreamSynchronize(n->s);
    hipFree(n->w); hipFree(n->m); hipFree(n->v); hipFree(n->g); hipFree(n->wp); hipFree(n->bp);
    hipFree(n->partial); hipFree(n->loss); hipFree(n->loss_acc); hipFree(n->X); hipFree(n->Y); hipFree(n->d_mat);
    hipStreamDestroy(n->s);
    free(n);
}

static int mlp_upload_weights(mdz_mlp *n, const float *w) {
    MCHK(hipMemcpyAsync(n->w, w, MLP_NPARAMS * 4, hipMemcpyHostToDevice, n->s));
    MCHK(hipMemsetAsync(n->m, 0, MLP_NPARAMS * 4, n->s));
    MCHK(hipMemsetAsync(n->v, 0, MLP_NPARAMS * 4, n->s));
    mdz_mlp_pack(n->w, n->wp, n->bp, n->s);
    MCHK(hipStreamSynchronize(n->s));
    n->t = 0;
    return MDZ_OK;
}

/* He-normal weights (std sqrt(2 / fan_in)), zero biases, from a splitmix64
 * stream of the seed (Box-Muller). */
extern "C" int mdz_mlp_init(mdz_mlp *n, unsigned long long seed) {
    if (!n) return mdz_error(MDZ_EINVAL, "NULL network");
    std::vector<float> w(MLP_NPARAMS, 0.0f);
    unsigned long long st = seed;
    auto next = [&]() {
        st += 0x9e3779b97f4a7c15ULL;
        unsigned long long x = st;
        x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ULL;
        x = (x ^ (x >> 27)) * 0x94d049bb133111ebULL;
        x ^= x >> 31;
        return ((x >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    };
    auto normal = [&]() { return sqrt(-2.0 * log(next())) * cos(2.0 * M_PI * next()); };
    const int offs[4] = {MLP_OFF_W1, MLP_OFF_W2, MLP_OFF_W3, MLP_OFF_W4};
    const int fan[4] = {MLP_IN, MLP_H, MLP_H, MLP_H}, cnt[4] = {MLP_H * MLP_IN, MLP_H * MLP_H, MLP_H * MLP_H, MLP_OUT * MLP_H};
    for (int L = 0; L < 4; L++)
        for (int i = 0; i < cnt[L]; i++) w[offs[L] + i] = (float)(normal() * sqrt(2.0 / fan[L]));
    return mlp_upload_weights(n, w.data());
}

extern "C" int mdz_mlp_set_weights(mdz_mlp *n, const float *w, size_t n_floats) {
    if (!n || !w || n_floats != MLP_NPARAMS) return mdz_error(MDZ_EINVAL, "mdz_mlp_set_weights: size");
    return mlp_upload_weights(n, w);
}

extern "C" int mdz_mlp_get_weights(mdz_mlp *n, float *w, size_t n_floats) {
    if (!n || !w || n_floats != MLP_NPARAMS) return mdz_error(MDZ_EINVAL, "mdz_mlp_get_weights: size");
    MCHK(hipMemcpyAsync(w, n->w, MLP_NPARAMS * 4, hipMemcpyDeviceToHost, n->s));
    MCHK(hipStreamSynchronize(n->s));
    return MDZ_OK;
}

static int mlp_reserve(mdz_mlp *n, long long count) {
    if (count <= n->cap) return MDZ_OK;
    hipFree(n->X);
    hipFree(n->Y);
    n->X = n->Y = nullptr;
    MCHK(hipMalloc((void **)&n->X, (size_t)count * MLP_IN * 4));
    MCHK(hipMalloc((void **)&n->Y, (size_t)count * 2 * 4));
    n->cap = count;
    return MDZ_OK;
}

extern "C" int mdz_mlp_generate(mdz_mlp *n, long long count, unsigned long long seed) {
    if (!n || count < TSAMP) return mdz_error(MDZ_EINVAL, "mdz_mlp_generate: count");
    int rc = mlp_reserve(n, count);
    if (rc) return rc;
    const long long chunk = 1LL << 22;
    for (long long f = 0; f < count; f += chunk) {
        long long c = count - f < chunk ? count - f : chunk;
        hipLaunchKernelGGL(k_mlp_generate, dim3((unsigned)((c + 255) / 256)), dim3(256), 0, n->s, f, c, seed,
                           (const mat_prop *)n->d_mat, n->prm, n->X + f * MLP_IN, n->Y + f * 2);
    }
    MCHK(hipGetLastError());
    MCHK(hipStreamSynchronize(n->s));
    n->n = count;
    return MDZ_OK;
}

extern "C" int mdz_mlp_upload_samples(mdz_mlp *n, long long count, const float *X, const float *Y) {
    if (!n || !X || !Y || count < 1) return mdz_error(MDZ_EINVAL, "mdz_mlp_upload_samples");
    int rc = mlp_reserve(n, count);
    if (rc) return rc;
    MCHK(hipMemcpyAsync(n->X, X, (size_t)count * MLP_IN * 4, hipMemcpyHostToDevice, n->s));
    MCHK(hipMemcpyAsync(n->Y, Y, (size_t)count * 2 * 4, hipMemcpyHostToDevice, n->s));
    MCHK(hipStreamSynchronize(n->s));
    n->n = count;
    return MDZ_OK;
}

extern "C" int mdz_mlp_download_samples(mdz_mlp *n, long long first, long long count, float *X, float *Y) {
    if (!n || first < 0 || count < 0 || first + count > n->n) return mdz_error(MDZ_EINVAL, "mdz_mlp_download_samples");
    if (X) MCHK(hipMemcpyAsync(X, n->X + first * MLP_IN, (size_t)count * MLP_IN * 4, hipMemcpyDeviceToHost, n->s));
    if (Y) MCHK(hipMemcpyAsync(Y, n->Y + first * 2, (size_t)count * 2 * 4, hipMemcpyDeviceToHost, n->s));
    MCHK(hipStreamSynchronize(n->s));
    return MDZ_OK;
}

/* the constants of the network's next Adam step */
static AdamStep adam_step(mdz_mlp *n, float lr) {
    n->t++;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    return AdamStep{n->w, n->m, n->v, lr, b1, b2, eps, 1.0f - powf(b1, (float)n->t), 1.0f - powf(b2, (float)n->t),
                    n->wp, n->bp};
}

/* gradient of sum((y-t)^2) / (2 * count) over the stored samples [first,
 * first + count), with an Adam step of rate *lr where lr is not null */
static int mlp_gradient(mdz_mlp *n, long long first, int count, unsigned long long mul, unsigned long long add,
                        double *loss_acc, const float *lr) {
    if (count < TSAMP || count % TSAMP) return mdz_error(MDZ_EINVAL, "batch must be a multiple of 64");
    const int tiles = count / 32, nb = tiles <= TBLOCKS ? tiles : std::min(TBLOCKS, mdz_div_up(tiles, TWAVES));
    if (nb > n->partial_blocks) {
        hipFree(n->partial);
        hipFree(n->loss);
        n->partial = nullptr;
        n->loss = nullptr;
        n->partial_blocks = 0;
        MCHK(hipMalloc((void **)&n->partial, (size_t)nb * MLP_NPARAMS * 4));
        MCHK(hipMalloc((void **)&n->loss, (size_t)nb * 4));
        n->partial_blocks = nb;
    }
    DevMLPW w{n->wp, n->bp};
    /* from one tile of a wave to its next: 32 nb TWAVES samples on */
    const unsigned long long un = (unsigned long long)n->n;
    const long long stride = (long long)(((unsigned long long)(32LL * nb * TWAVES) % un) * (mul % un) % un);
    hipLaunchKernelGGL(k_mlp_train_step, dim3(nb), dim3(TWAVES * 64), 0, n->s, (const float *)n->X, (const float *)n->Y,
                       n->n, first, mul, add, stride, tiles, 1.0f / (float)count, w, n->partial, n->loss);
    const dim3 grid(mdz_div_up(MLP_NPARAMS, RED_P)), blk(RED_P * RED_W);
    const AdamStep as = lr ? adam_step(n, *lr) : AdamStep{};
    if (lr)
        hipLaunchKernelGGL(k_mlp_reduce<true>, grid, blk, 0, n->s, (const float *)n->partial, nb, n->g,
                           (const float *)n->loss, loss_acc, as);
    else
        hipLaunchKernelGGL(k_mlp_reduce<false>, grid, blk, 0, n->s, (const float *)n->partial, nb, n->g,
                           (const float *)n->loss, loss_acc, as);
    MCHK(hipGetLastError());
    return MDZ_OK;
}

extern "C" int mdz_mlp_gradient(mdz_mlp *n, long long first, int count, float *grad, double *loss) {
    if (!n || first < 0 || first + count > n->n) return mdz_error(MDZ_EINVAL, "mdz_mlp_gradient: range");
    MCHK(hipMemsetAsync(n->loss_acc, 0, 8, n->s));
    int rc = mlp_gradient(n, first, count, 1ULL, 0ULL, n->loss_acc, nullptr);
    if (rc) return rc;
    if (grad) MCHK(hipMemcpyAsync(grad, n->g, MLP_NPARAMS * 4, hipMemcpyDeviceToHost, n->s));
    if (loss) MCHK(hipMemcpyAsync(loss, n->loss_acc, 8, hipMemcpyDeviceToHost, n->s));
    MCHK(hipStreamSynchronize(n->s));
    return MDZ_OK;
}

/* one Adam step with a caller-supplied gradient */
extern "C" int mdz_mlp_adam_step(mdz_mlp *n, const float *grad, float lr) {
    if (!n || !grad) return mdz_error(MDZ_EINVAL, "mdz_mlp_adam_step");
    MCHK(hipMemcpyAsync(n->g, grad, MLP_NPARAMS * 4, hipMemcpyHostToDevice, n->s));
    hipLaunchKernelGGL(k_mlp_adam, dim3(mdz_div_up(MLP_NPARAMS, 256)), dim3(256), 0, n->s, adam_step(n, lr),
                       (const float *)n->g);
    MCHK(hipGetLastError());
    MCHK(hipStreamSynchronize(n->s));
    return MDZ_OK;
}

/* epochs over the stored samples in batches (a multiple of 64); each epoch
 * visits the samples in the order i -> (i * a + c) mod n with a random odd
 * a coprime to n; loss_per_epoch[e] = mean squared error per output */
extern "C" int mdz_mlp_train(mdz_mlp *n, int epochs, int batch, float lr, unsigned long long seed,
                             double *loss_per_epoch) {
    if (!n || epochs < 1 || batch < TSAMP || batch % TSAMP || n->n < batch)
        return mdz_error(MDZ_EINVAL, "mdz_mlp_train: arguments");
    const long long steps = n->n / batch;
    unsigned long long st = seed;
    for (int e = 0; e < epochs; e++) {
        st = st * 6364136223846793005ULL + 1442695040888963407ULL;
        unsigned long long mul = (st >> 17) | 1ULL;
        while (true) { /* coprime to n */
            unsigned long long a = mul % (unsigned long long)n->n, b = (unsigned long long)n->n;
            while (b) { unsigned long long t = a % b; a = b; b = t; }
            if (a == 1) break;
            mul += 2;
        }
        mul %= (unsigned long long)n->n;
        const unsigned long long add = (st >> 7) % (unsigned long long)n->n;
        MCHK(hipMemsetAsync(n->loss_acc, 0, 8, n->s));
        for (long long k = 0; k < steps; k++) {
            int rc = mlp_gradient(n, k * batch, batch, mul, add, n->loss_acc, &lr);
            if (rc) return rc;
        }
        double acc = 0.0;
        MCHK(hipMemcpyAsync(&acc, n->loss_acc, 8, hipMemcpyDeviceToHost, n->s));
        MCHK(hipStreamSynchronize(n->s));
        if (loss_per_epoch) loss_per_epoch[e] = acc / (double)(steps * batch * 2);
    }
    return MDZ_OK;
}

extern "C" int mdz_mlp_predict(mdz_mlp *n, long long first, long long count, float *Yout) {
    if (!n || !Yout || first < 0 || count < 1 || first + count > n->n) return mdz_error(MDZ_EINVAL, "mdz_mlp_predict");
    float *d = nullptr;
    MCHK(hipMalloc((void **)&d, (size_t)count * 2 * 4));
    DevMLPW w{n->wp, n->bp};
    hipLaunchKernelGGL(k_mlp_predict, dim3((unsigned)((count + TSAMP - 1) / TSAMP)), dim3(TBLK), 0, n->s,
                       (const float *)n->X, first, count, w, d);
    hipError_t e = hipMemcpyAsync(Yout, d, (size_t)count * 2 * 4, hipMemcpyDeviceToHost, n->s);
    hipError_t e2 = hipStreamSynchronize(n->s);
    hipFree(d);
    if (e != hipSuccess || e2 != hipSuccess) return mdz_error(MDZ_EHIP, "mdz_mlp_predict");
    return MDZ_OK;
}

/* The same samples through the inference form of the current weights (the
 * network the grid guess evaluates): Y[count][2]. */
extern "C" int mdz_mlp_predict_inference(mdz_mlp *n, long long first, long long count, float *Yout) {
    if (!n || !Yout || first < 0 || count < 1 || first + count > n->n)
        return mdz_error(MDZ_EINVAL, "mdz_mlp_predict_inference");
    float *d = nullptr, *bi = nullptr;
    unsigned short *wi = nullptr;
    MCHK(hipMalloc((void **)&d, (size_t)count * 2 * 4));
    if (hipMalloc((void **)&wi, MLI_TOTAL * 2) != hipSuccess || hipMalloc((void **)&bi, MLI_B_TOTAL * 4) != hipSuccess) {
        hipFree(d); hipFree(wi);
        return mdz_error(MDZ_EHIP, "mdz_mlp_predict_inference: allocation");
    }
    mdz_mlp_pack_inference(n->w, wi, bi, n->s);
    hipLaunchKernelGGL(k_mlp_predict_inf, dim3((unsigned)((count + GBLK - 1) / GBLK)), dim3(GBLK), 0, n->s,
                       (const float *)n->X, first, count, DevMLPI{wi, bi, nullptr}, d);
    hipError_t e = hipMemcpyAsync(Yout, d, (size_t)count * 2 * 4, hipMemcpyDeviceToHost, n->s);
    hipError_t e2 = hipStreamSynchronize(n->s);
    hipFree(d); hipFree(wi); hipFree(bi);
    if (e != hipSuccess || e2 != hipSuccess) return mdz_error(MDZ_EHIP, "mdz_mlp_predict_inference");
    return MDZ_OK;
}
