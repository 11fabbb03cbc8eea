// mlp.hip - the learned cut proposal: a point-set network that ranks a part's
// candidate planes, trained on exact scores the library computes itself.
//
// No reference counterpart. Network (PointNet-style, conditioned on the
// plane): 256 area-stratified surface samples of a part in the part's box
// frame (center, half the largest extent); for a candidate plane (unit normal
// n, offset d in the same frame) every sample gets its signed distance
// s = n.p + d, and (x, y, z, s) goes through a shared point MLP
// 4 -> 128 -> 128 -> 128 (ReLU); the features are max-pooled separately over
// the samples on each side of the plane (g+, g-: the two halves' shapes) and a
// head [g+, g-, n, d] -> 128 -> 128 -> 1 (ReLU between) predicts the plane's
// exact cut score. BF16 operands, FP32 accumulation on v_mfma_f32_16x16x16_bf16.
// Inference and training run fused kernels whose activations stay in registers
// (see "Register chains"); a layer-by-layer GEMM path is kept for inference
// (tuning knob mlp_fused; the same scores). Training keeps FP32 master weights
// and Adam state on the device (mean squared error on the score).
//
// Parameter layout (FP32, padded to multiples of 16; the padding stays zero):
//   W1 [16 x 128] (rows 0..3 used), b1 [128], W2 [128 x 128], b2, W3, b3,
//   H1 [272 x 128] (rows 0..259 used), c1 [128], H2 [128 x 128], c2,
//   H3 [128 x 16] (column 0 used), c3 [16] (entry 0 used).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>
#include "kerr.h"
#include "mlp.hpp"
#include "wave.hpp"

// signed distances and sums round as written (the oracle repeats them)
#pragma clang fp contract(off)

using namespace cuacd;

namespace {

typedef unsigned short bf16_t;
typedef short s4v_t __attribute__((ext_vector_type(4)));
typedef float f4v_t __attribute__((ext_vector_type(4)));

constexpr int NS = MLP_SAMPLES;  // samples per part
constexpr int HD = 128;   // hidden width
constexpr int KIN = 16;   // padded point input width
constexpr int KH = 272;   // padded head input width (2 x 128 + 4)
constexpr int NO = 16;    // padded output width

// offsets of the parameter blocks (floats)
constexpr int P_W1 = 0, P_B1 = P_W1 + KIN * HD, P_W2 = P_B1 + HD, P_B2 = P_W2 + HD * HD, P_W3 = P_B2 + HD,
              P_B3 = P_W3 + HD * HD, P_H1 = P_B3 + HD, P_C1 = P_H1 + KH * HD, P_H2 = P_C1 + HD,
              P_C2 = P_H2 + HD * HD, P_H3 = P_C2 + HD, P_C3 = P_H3 + HD * NO, P_TOTAL = P_C3 + NO;

// FP32 -> BF16, round to nearest even (NaN kept quiet)
__host__ __device__ __forceinline__ bf16_t f2bf(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x7fffffu)) return (bf16_t)((u >> 16) | 0x40);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (bf16_t)(u >> 16);
}
__host__ __device__ __forceinline__ float bf2f(bf16_t b) {
    const uint32_t u = (uint32_t)b << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

// ---------------------------------------------------------------------------
// GEMM (the layer-by-layer path): C[M x N] = A[M x K] . B[K x N] (+ bias[n]) (ReLU)
// A(m, k) = A[m * sam + k * sak], B(k, n) = B[k * sbk + n * sbn] (BF16), so
// transposed operands are strides. 64 x 64 output tile per 256-thread
// workgroup, K in steps of 32 staged through LDS; each wave owns a 32 x 32
// quarter as 2 x 2 MFMA 16 x 16 x 16 tiles. Operand layout of the MFMA (lane
// l): A row l % 16, k 4 (l / 16) .. +3; B column l % 16, same k; D column
// l % 16, rows 4 (l / 16) .. +3.
// ---------------------------------------------------------------------------
struct GemmArgs {
    int M, N, K;
    const bf16_t* A;
    long long sam, sak;
    const bf16_t* B;
    long long sbk, sbn;
    const float* bias;  // [N] or null
    int relu;
    float* C;           // FP32 out (row stride ldc) or null
    long long ldc;
    bf16_t* Cb;         // BF16 out (row stride ldcb) or null
    long long ldcb;
};

constexpr int GM = 64, GN = 64, GK = 32, GKP = GK + 8;  // LDS rows padded by 16 bytes

__global__ __launch_bounds__(256) void mlp_gemm_kernel(GemmArgs g) {
    __shared__ __align__(16) bf16_t As[GM][GKP];
    __shared__ __align__(16) bf16_t Bt[GN][GKP];  // transposed: Bt[n][k]
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int m0 = blockIdx.y * GM, n0 = blockIdx.x * GN;
    const int wm = (wv >> 1) * 32, wn = (wv & 1) * 32;
    f4v_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f4v_t{0.f, 0.f, 0.f, 0.f};
    const int lr = tid >> 2, lk = (tid & 3) * 8;  // loader: one row (or column), 8 consecutive k
    for (int k0 = 0; k0 < g.K; k0 += GK) {
        {
            const int m = m0 + lr;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int k = k0 + lk + j;
                As[lr][lk + j] = (m < g.M && k < g.K) ? g.A[(long long)m * g.sam + (long long)k * g.sak] : (bf16_t)0;
            }
            const int n = n0 + lr;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int k = k0 + lk + j;
                Bt[lr][lk + j] = (n < g.N && k < g.K) ? g.B[(long long)k * g.sbk + (long long)n * g.sbn] : (bf16_t)0;
            }
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < GK; ks += 16) {
            const int kk = ks + 4 * (lane >> 4);
            s4v_t a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const bf16_t* pa = &As[wm + 16 * i + (lane & 15)][kk];
                a[i] = s4v_t{(short)pa[0], (short)pa[1], (short)pa[2], (short)pa[3]};
                const bf16_t* pb = &Bt[wn + 16 * i + (lane & 15)][kk];
                b[i] = s4v_t{(short)pb[0], (short)pb[1], (short)pb[2], (short)pb[3]};
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = n0 + wn + 16 * j + (lane & 15);
            if (n >= g.N) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
                if (m >= g.M) continue;
                float v = acc[i][j][r];
                if (g.bias) v += g.bias[n];
                if (g.relu) v = fmaxf(v, 0.0f);
                if (g.C) g.C[(long long)m * g.ldc + n] = v;
                if (g.Cb) g.Cb[(long long)m * g.ldcb + n] = f2bf(v);
            }
        }
}

// ---------------------------------------------------------------------------
// Register chains: a wave carries 16 rows (samples, candidates) per tile through
// consecutive layers without LDS or memory in between. With the weights as the
// MFMA's A operand (rows = output channels) and the activations as its B
// operand (columns = rows of the batch), lane l of the result holds output
// channels 4 (l / 16) .. +3 of row l % 16 - exactly the B operand of the next
// layer's product over those channels. The k order (16-wide steps, ascending),
// the epilogue (bias, ReLU, BF16 rounding) and so the results are those of
// mlp_gemm_kernel, bit for bit.
// ---------------------------------------------------------------------------
constexpr int FP = HD + 8;    // weight row pitch in LDS (bf16)
constexpr int FP1 = KIN + 8;  // pitch of the transposed first layer

typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
typedef float f2v_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ s4v_t ld_frag(const bf16_t* p) { return *reinterpret_cast<const s4v_t*>(p); }
__device__ __forceinline__ f4v_t mma(s4v_t a, s4v_t b, f4v_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
// round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ s4v_t pack4(float x, float y, float z, float w) {
    const bf2_t lo = __builtin_convertvector((f2v_t{x, y}), bf2_t), hi = __builtin_convertvector((f2v_t{z, w}), bf2_t);
    const uint2 u = make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
    return __builtin_bit_cast(s4v_t, u);
}
__device__ __forceinline__ s4v_t relu4(f4v_t a, f4v_t b) {
    return pack4(fmaxf(a[0] + b[0], 0.0f), fmaxf(a[1] + b[1], 0.0f), fmaxf(a[2] + b[2], 0.0f),
                 fmaxf(a[3] + b[3], 0.0f));
}
// the gradient where the activation is positive
__device__ __forceinline__ s4v_t mask4(f4v_t v, s4v_t act) {
    return pack4((act[0] & 0x7fff) ? v[0] : 0.0f, (act[1] & 0x7fff) ? v[1] : 0.0f, (act[2] & 0x7fff) ? v[2] : 0.0f,
                 (act[3] & 0x7fff) ? v[3] : 0.0f);
}
// First-layer operand of a sample: (x, y, z, s) in the lanes of channels 0..3.
__device__ __forceinline__ s4v_t point_frag(const float* p, float sd, bool on) {
    const s4v_t z = {0, 0, 0, 0};
    return on ? s4v_t{(short)f2bf(p[0]), (short)f2bf(p[1]), (short)f2bf(p[2]), (short)f2bf(sd)} : z;
}
// The transpose of a 16 x 16 tile as the same lane layout: a product with the
// identity (BF16 values pass through exactly).
__device__ __forceinline__ s4v_t identity_frag() {
    const int fr = lane_id() & 15, fk = 4 * (lane_id() >> 4);
    s4v_t r;
#pragma unroll
    for (int q = 0; q < 4; ++q) r[q] = (short)(fk + q == fr ? 0x3f80 : 0);
    return r;
}
__device__ __forceinline__ s4v_t transpose4(s4v_t a, s4v_t eye) {
    const f4v_t d = mma(a, eye, f4v_t{0.f, 0.f, 0.f, 0.f});
    return pack4(d[0], d[1], d[2], d[3]);
}

// rows x cols of a row-major BF16 matrix into LDS rows of `pitch` (16-byte pieces)
__device__ __forceinline__ void stage_rows(bf16_t* dst, int pitch, const bf16_t* src, int rows, int cols) {
    const int per = cols / 8;
    for (int i = threadIdx.x; i < rows * per; i += blockDim.x)
        *reinterpret_cast<uint4*>(dst + (i / per) * pitch + (i % per) * 8) =
            *reinterpret_cast<const uint4*>(src + (i / per) * cols + (i % per) * 8);
}

// Point layers and pooling: a persistent grid of 512-thread workgroups with the
// transposed point-layer weights in LDS; four waves take a candidate, each 64
// samples (4 tiles), and only the head's input row (Hin: pooled features, the
// plane, zeros) - and for training the pooled rows - reach memory. Two waves
// per SIMD: one's MFMAs cover the other's epilogue. An output tile's weight
// fragment (512 B of LDS) feeds four MFMAs. Pooling takes integer maxima of
// (BF16 bits, inverted sample), so ties go to the first sample. 12,032
// candidates: the activations in LDS, one wave per SIMD, took 0.87 ms.
constexpr unsigned ENC_LDS = 2 * HD * FP * 2 + HD * FP1 * 2 + 3 * HD * 4 + 2 * 2 * 4 * 2 * HD * 4;

template <int CTRL> __device__ __forceinline__ int row_max(int v) {
    return max(v, __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true));  // rotation in a row of 16
}

__global__ __launch_bounds__(512) void mlp_encode_kernel(const float* pts, const float* planes, const int* part_of,
                                                         int C, const bf16_t* Wt, const float* Wf, bf16_t* Hin,
                                                         uint8_t* arg) {
    extern __shared__ __align__(16) char fl[];
    bf16_t* W2t = (bf16_t*)fl;            // [HD][FP] W2t[n][k]
    bf16_t* W3t = W2t + HD * FP;          // [HD][FP]
    bf16_t* W1t = W3t + HD * FP;          // [HD][FP1]
    float* bs = (float*)(W1t + HD * FP1); // [3][HD] biases
    int* red = (int*)(bs + 3 * HD);       // [2 rounds][2 candidates][4 waves][2 sides x HD] keys
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    stage_rows(W2t, FP, Wt + P_W2, HD, HD);
    stage_rows(W3t, FP, Wt + P_W3, HD, HD);
    stage_rows(W1t, FP1, Wt + P_W1, HD, KIN);
    for (int i = tid; i < HD; i += 512) {
        bs[i] = Wf[P_B1 + i];
        bs[HD + i] = Wf[P_B2 + i];
        bs[2 * HD + i] = Wf[P_B3 + i];
    }
    __syncthreads();
    const int fr = lane & 15, fk = 4 * (lane >> 4);
    const int cw = wv >> 2, ws = wv & 3;
    const f4v_t zero = {0.f, 0.f, 0.f, 0.f};
    int round = 0;
    for (int pr = blockIdx.x; 2 * pr < C; pr += gridDim.x, round ^= 1) {
        const int c = min(2 * pr + cw, C - 1);
        const float* pl = planes + 4ll * c;
        const float* base = pts + (long long)part_of[c] * NS * 3;
        s4v_t x[4], a1[8][4], a2[8][4];
        bool pos[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float* pp = base + 3 * (64 * ws + 16 * j + fr);
            const float sd = pl[0] * pp[0] + pl[1] * pp[1] + pl[2] * pp[2] + pl[3];
            pos[j] = sd >= 0.0f;
            x[j] = point_frag(pp, sd, fk == 0);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const s4v_t a = ld_frag(W1t + (16 * i + fr) * FP1 + fk);
            const f4v_t b = *(const f4v_t*)(bs + 16 * i + fk);
#pragma unroll
            for (int j = 0; j < 4; ++j) a1[i][j] = relu4(mma(a, x[j], zero), b);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            f4v_t acc[4] = {zero, zero, zero, zero};
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const s4v_t a = ld_frag(W2t + (16 * i + fr) * FP + 16 * k + fk);
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[j] = mma(a, a1[k][j], acc[j]);
            }
            const f4v_t b = *(const f4v_t*)(bs + HD + 16 * i + fk);
#pragma unroll
            for (int j = 0; j < 4; ++j) a2[i][j] = relu4(acc[j], b);
        }
        int* rd = red + ((round * 2 + cw) * 4 + ws) * 2 * HD;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            f4v_t acc[4] = {zero, zero, zero, zero};
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const s4v_t a = ld_frag(W3t + (16 * i + fr) * FP + 16 * k + fk);
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[j] = mma(a, a2[k][j], acc[j]);
            }
            const f4v_t b = *(const f4v_t*)(bs + 2 * HD + 16 * i + fk);
            int kp[4] = {-1, -1, -1, -1}, kn[4] = {-1, -1, -1, -1};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint2 u = __builtin_bit_cast(uint2, relu4(acc[j], b));
                const int inv = 255 - (64 * ws + 16 * j + fr);
                const int key[4] = {(int)((u.x & 0x7fffu) << 8) | inv, (int)((u.x >> 8) & 0x7fff00u) | inv,
                                    (int)((u.y & 0x7fffu) << 8) | inv, (int)((u.y >> 8) & 0x7fff00u) | inv};
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    kp[r] = max(kp[r], pos[j] ? key[r] : -1);
                    kn[r] = max(kn[r], pos[j] ? -1 : key[r]);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                kp[r] = row_max<0x121>(row_max<0x122>(row_max<0x124>(row_max<0x128>(kp[r]))));
                kn[r] = row_max<0x121>(row_max<0x122>(row_max<0x124>(row_max<0x128>(kn[r]))));
            }
            if (fr == 0) {
                *(int4*)(rd + 16 * i + fk) = make_int4(kp[0], kp[1], kp[2], kp[3]);
                *(int4*)(rd + HD + 16 * i + fk) = make_int4(kn[0], kn[1], kn[2], kn[3]);
            }
        }
        __syncthreads();  // the next round writes the other half of red
        const int cd = tid >> 8, q = tid & 255;
        const long long co = 2ll * pr + cd;
        if (co < C) {
            const int* r0 = red + (round * 2 + cd) * 4 * 2 * HD + q;
            const int m = max(max(r0[0], r0[2 * HD]), max(r0[4 * HD], r0[6 * HD]));
            Hin[co * KH + q] = m >= 0 ? (bf16_t)(m >> 8) : (bf16_t)0;
            if (arg) arg[co * 2 * HD + q] = m >= 0 ? (uint8_t)(255 - (m & 255)) : (uint8_t)0;
            if (q < KH - 2 * HD) Hin[co * KH + 2 * HD + q] = q < 4 ? f2bf(planes[4 * co + q]) : (bf16_t)0;
        }
    }
}

// Operand tiles of the weight gradients, [group of 16 rows][tile][64 lanes]:
// lane l holds channel l % 16 of rows 4 (l / 16) .. +3.
constexpr int HT_HIN = 0, HT_B1 = 17, HT_B2 = 25, HT_D1 = 33, HT_D2 = 41, HT_DY = 49, HT_N = 50;      // head
constexpr int ET_X = 0, ET_A1 = 1, ET_A2 = 9, ET_D3 = 17, ET_D2 = 25, ET_D1 = 33, ET_N = 41;          // encoder

// Head, a wave per 16 candidates, weights from L2. Training adds the loss
// terms, the head's backward (gb: the pooled features' gradients, zero where
// the feature is) and the operand tiles. One launch instead of the three
// forward GEMMs and, in training, six backward ones with their column sums.
template <bool TRAIN>
__global__ __launch_bounds__(256) void mlp_head_kernel(const bf16_t* Hin, int C, const bf16_t* Wt, const bf16_t* W,
                                                       const float* Wf, float* Y, const float* target, float* err2,
                                                       bf16_t* gb, s4v_t* tiles) {
    const int lane = threadIdx.x & 63, grp = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (grp * 16 >= C) return;
    const int fr = lane & 15, fk = 4 * (lane >> 4);
    const long long c = 16ll * grp + fr;
    const bool on = c < C;
    const f4v_t zero = {0.f, 0.f, 0.f, 0.f};
    const s4v_t z4 = {0, 0, 0, 0};
    s4v_t h[17], b1[8], b2[8];
#pragma unroll
    for (int k = 0; k < 17; ++k) h[k] = on ? ld_frag(Hin + c * KH + 16 * k + fk) : z4;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        f4v_t acc = zero;
#pragma unroll
        for (int k = 0; k < 17; ++k) acc = mma(ld_frag(Wt + P_H1 + (16 * i + fr) * KH + 16 * k + fk), h[k], acc);
        b1[i] = relu4(acc, *(const f4v_t*)(Wf + P_C1 + 16 * i + fk));
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        f4v_t acc = zero;
#pragma unroll
        for (int k = 0; k < 8; ++k) acc = mma(ld_frag(Wt + P_H2 + (16 * i + fr) * HD + 16 * k + fk), b1[k], acc);
        b2[i] = relu4(acc, *(const f4v_t*)(Wf + P_C2 + 16 * i + fk));
    }
    f4v_t acc = zero;
#pragma unroll
    for (int k = 0; k < 8; ++k) acc = mma(ld_frag(Wt + P_H3 + fr * HD + 16 * k + fk), b2[k], acc);
    const float y = acc[0] + Wf[P_C3];  // output 0: lanes of channels 0..3
    if (fk == 0 && on) Y[c] = y;
    if constexpr (TRAIN) {
        s4v_t dy = z4;
        if (fk == 0 && on) {
            const float e = y - target[c];
            err2[c] = e * e;
            dy[0] = (short)f2bf(2.0f * e / (float)C);
        }
        s4v_t d2[8], d1[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) d2[i] = mask4(mma(ld_frag(W + P_H3 + (16 * i + fr) * NO + fk), dy, zero), b2[i]);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            f4v_t v = zero;
#pragma unroll
            for (int k = 0; k < 8; ++k) v = mma(ld_frag(W + P_H2 + (16 * i + fr) * HD + 16 * k + fk), d2[k], v);
            d1[i] = mask4(v, b1[i]);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            f4v_t v = zero;
#pragma unroll
            for (int k = 0; k < 8; ++k) v = mma(ld_frag(W + P_H1 + (16 * i + fr) * HD + 16 * k + fk), d1[k], v);
            if (on) *(s4v_t*)(gb + c * 2 * HD + 16 * i + fk) = mask4(v, h[i]);
        }
        const s4v_t eye = identity_frag();
        s4v_t* o = tiles + (long long)grp * HT_N * 64 + lane;
#pragma unroll
        for (int i = 0; i < 17; ++i) o[(HT_HIN + i) * 64] = transpose4(h[i], eye);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            o[(HT_B1 + i) * 64] = transpose4(b1[i], eye);
            o[(HT_B2 + i) * 64] = transpose4(b2[i], eye);
            o[(HT_D1 + i) * 64] = transpose4(d1[i], eye);
            o[(HT_D2 + i) * 64] = transpose4(d2[i], eye);
        }
        o[HT_DY * 64] = transpose4(dy, eye);
    }
}

// ---------------------------------------------------------------------------
// Encoder backward. The max-pool passes a gradient to one sample per side and
// channel, so of a candidate's 256 rows only the pooled ones - some 60 of them
// - have any: the rest contribute exact zeros to every gradient. The pooled
// rows of all candidates are listed (in order, by a scan, so sums do not
// depend on timing), their two layers recomputed, and their gradients formed
// densely over the list. Layer by layer over all 1.3 million rows of 5,056
// candidates a training step took 11.5 ms, most of it in GEMMs, column sums
// and the unpooling, all through memory.
// ---------------------------------------------------------------------------
// pooled rows of each candidate as a bit mask, and their number
__global__ __launch_bounds__(256) void mlp_rows_mark(const bf16_t* Hin, const uint8_t* arg,
                                                     unsigned long long* mask, int* cnt) {
    __shared__ uint8_t mark[NS];
    __shared__ int wc[4];
    const long long c = blockIdx.x;
    const int t = threadIdx.x;
    mark[t] = 0;
    __syncthreads();
    if (Hin[c * KH + t] & 0x7fff) mark[arg[c * 2 * HD + t]] = 1;
    __syncthreads();
    const unsigned long long m = ballot(mark[t] != 0);
    if ((t & 63) == 0) {
        mask[c * 4 + (t >> 6)] = m;
        wc[t >> 6] = __popcll(m);
    }
    __syncthreads();
    if (t == 0) cnt[c] = wc[0] + wc[1] + wc[2] + wc[3];
}

// exclusive prefix of cnt, in place; *total; the list's tail up to a whole
// pair of 16-row groups is empty rows
__global__ __launch_bounds__(1024) void mlp_rows_scan(int* cnt, int C, int* total, int* list) {
    __shared__ int ws[16];
    int carry = 0;
    const int t = threadIdx.x, wv = t >> 6;
    for (int b = 0; b < C; b += 1024) {
        const int v = b + t < C ? cnt[b + t] : 0;
        const int incl = wave_incl_scan(v);
        if ((t & 63) == 63) ws[wv] = incl;
        __syncthreads();
        int base = 0, all = 0;
        for (int q = 0; q < 16; ++q) {
            if (q < wv) base += ws[q];
            all += ws[q];
        }
        if (b + t < C) cnt[b + t] = carry + base + incl - v;
        carry += all;
        __syncthreads();
    }
    if (t == 0) *total = carry;
    const int end = (carry + 31) / 32 * 32;
    if (carry + t < end) list[carry + t] = -1;
}

__global__ __launch_bounds__(256) void mlp_rows_fill(const unsigned long long* mask, const int* off, int* list) {
    const long long c = blockIdx.x;
    const int t = threadIdx.x, wv = t >> 6;
    int o = off[c];
    for (int q = 0; q < wv; ++q) o += __popcll(mask[c * 4 + q]);
    const unsigned long long m = mask[c * 4 + wv];
    if ((m >> (t & 63)) & 1ull) list[o + mask_rank(m)] = (int)(c * NS + t);
}

constexpr unsigned ROWS_LDS = 3 * HD * FP * 2 + HD * FP1 * 2 + 2 * HD * 4;

// Recomputed layers and gradients of the listed rows: a persistent grid, two
// 16-row groups per wave, so each weight fragment read from LDS feeds two
// MFMAs. Writes the operand tiles.
__global__ __launch_bounds__(512) void mlp_rows_kernel(const float* pts, const float* planes, const int* part_of,
                                                       const bf16_t* Wt, const bf16_t* W, const float* Wf,
                                                       const uint8_t* arg, const bf16_t* gb, const int* list,
                                                       const int* total, s4v_t* tiles) {
    extern __shared__ __align__(16) char fl[];
    bf16_t* W2t = (bf16_t*)fl;      // [HD][FP] transposed
    bf16_t* W2n = W2t + HD * FP;    // [HD][FP] as stored
    bf16_t* W3n = W2n + HD * FP;    // [HD][FP] as stored
    bf16_t* W1t = W3n + HD * FP;    // [HD][FP1]
    float* bs = (float*)(W1t + HD * FP1);
    const int tid = threadIdx.x, lane = tid & 63;
    stage_rows(W2t, FP, Wt + P_W2, HD, HD);
    stage_rows(W2n, FP, W + P_W2, HD, HD);
    stage_rows(W3n, FP, W + P_W3, HD, HD);
    stage_rows(W1t, FP1, Wt + P_W1, HD, KIN);
    for (int i = tid; i < HD; i += 512) {
        bs[i] = Wf[P_B1 + i];
        bs[HD + i] = Wf[P_B2 + i];
    }
    __syncthreads();
    const int fr = lane & 15, fk = 4 * (lane >> 4);
    const f4v_t zero = {0.f, 0.f, 0.f, 0.f};
    const s4v_t eye = identity_frag();
    const int pairs = (*total + 31) / 32;
    for (int pr = blockIdx.x * 8 + (tid >> 6); pr < pairs; pr += gridDim.x * 8) {
        s4v_t x[2], a1[8][2], a2[8][2], d3[8][2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int row = list[32 * pr + 16 * j + fr];
            const bool on = row >= 0;
            const int c = on ? row / NS : 0, sm = on ? row % NS : 0;
            const float* pl = planes + 4ll * c;
            const float* pp = pts + ((long long)part_of[c] * NS + sm) * 3;
            const float sd = pl[0] * pp[0] + pl[1] * pp[1] + pl[2] * pp[2] + pl[3];
            x[j] = point_frag(pp, sd, on && fk == 0);
            const uint8_t* ar = arg + (long long)c * 2 * HD + fk;
            const bf16_t* gr = gb + (long long)c * 2 * HD + fk;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                // a side without the feature has gradient 0, whatever its row
                const uint32_t ap = *(const uint32_t*)(ar + 16 * k), an = *(const uint32_t*)(ar + HD + 16 * k);
                const s4v_t gp = ld_frag(gr + 16 * k), gn = ld_frag(gr + HD + 16 * k);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int vp = (int)((ap >> (8 * q)) & 255u) == sm ? gp[q] : 0;
                    const int vn = (int)((an >> (8 * q)) & 255u) == sm ? gn[q] : 0;
                    d3[k][j][q] = (short)(on ? vp | vn : 0);
                }
            }
        }
        s4v_t* o = tiles + 2ll * pr * ET_N * 64 + lane;
        auto put = [&](int tile, int j, s4v_t v) { o[(j * ET_N + tile) * 64] = transpose4(v, eye); };
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const s4v_t a = ld_frag(W1t + (16 * i + fr) * FP1 + fk);
            const f4v_t b = *(const f4v_t*)(bs + 16 * i + fk);
#pragma unroll
            for (int j = 0; j < 2; ++j) a1[i][j] = relu4(mma(a, x[j], zero), b);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            f4v_t acc[2] = {zero, zero};
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const s4v_t a = ld_frag(W2t + (16 * i + fr) * FP + 16 * k + fk);
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[j] = mma(a, a1[k][j], acc[j]);
            }
            const f4v_t b = *(const f4v_t*)(bs + HD + 16 * i + fk);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                a2[i][j] = relu4(acc[j], b);
                put(ET_A2 + i, j, a2[i][j]);
                put(ET_D3 + i, j, d3[i][j]);
            }
        }
        s4v_t d2[8][2];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            f4v_t acc[2] = {zero, zero};
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const s4v_t a = ld_frag(W3n + (16 * i + fr) * FP + 16 * k + fk);
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[j] = mma(a, d3[k][j], acc[j]);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                d2[i][j] = mask4(acc[j], a2[i][j]);
                put(ET_D2 + i, j, d2[i][j]);
                put(ET_A1 + i, j, a1[i][j]);
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            f4v_t acc[2] = {zero, zero};
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const s4v_t a = ld_frag(W2n + (16 * i + fr) * FP + 16 * k + fk);
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[j] = mma(a, d2[k][j], acc[j]);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) put(ET_D1 + i, j, mask4(acc[j], a1[i][j]));
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) put(ET_X, j, x[j]);
    }
}

// One weight gradient P^T Q over the rows of a tile table (np x nq tiles from
// p0 / q0), and the bias gradient (column sums of Q) as a product with ones.
// Workgroup z of nz takes groups z, z + nz, ...; a wave owns two of the P
// tiles and all of Q; FP32 partial sums, added in order by mlp_grad_reduce.
struct GradJob {
    const s4v_t* tiles;
    int stride;        // tiles per group
    int p0, np, q0, nq;
    const int* rows;   // rows on the device, or null
    int groups;        // else the group count
    int nz, block0;    // workgroups, the first one's index
    float* part;       // [nz][np*16 x nq*16 (+ nq*16)]
    int w_off, w_cols; // the gradient's place: w_off + row * w_cols + column
    int b_off;         // the bias's, or -1
};
constexpr int GRAD_JOBS = 8;
struct GradJobs {
    GradJob j[GRAD_JOBS];
};

__global__ __launch_bounds__(256) void mlp_grad_kernel(GradJobs jobs) {
    int ji = 0;
#pragma unroll
    for (int k = 1; k < GRAD_JOBS; ++k)
        if ((int)blockIdx.x >= jobs.j[k].block0) ji = k;
    const GradJob& J = jobs.j[ji];
    const int z = blockIdx.x - J.block0;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int i0 = 2 * wv;
    if (i0 >= J.np) return;
    const int groups = J.rows ? (*J.rows + 15) / 16 : J.groups;
    const bool two = i0 + 1 < J.np, bias = J.b_off >= 0 && wv == 0;
    const int nq = J.nq;
    const f4v_t zero = {0.f, 0.f, 0.f, 0.f};
    const s4v_t z4 = {0, 0, 0, 0};
    const s4v_t ones = {0x3f80, 0x3f80, 0x3f80, 0x3f80};
    f4v_t acc[2][8], ab[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[0][j] = acc[1][j] = ab[j] = zero;
    const s4v_t* src = J.tiles + lane;
    auto load = [&](int g, s4v_t (&p)[2], s4v_t (&q)[8]) {
        const s4v_t* b = src + (long long)g * J.stride * 64;
        p[0] = b[(J.p0 + i0) * 64];
        p[1] = two ? b[(J.p0 + i0 + 1) * 64] : z4;
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j] = j < nq ? b[(J.q0 + j) * 64] : z4;
    };
    s4v_t p[2], q[8];
    if (z < groups) load(z, p, q);
    for (int g = z; g < groups; g += J.nz) {
        s4v_t pn[2], qn[8];
        load(min(g + J.nz, groups - 1), pn, qn);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            acc[0][j] = mma(p[0], q[j], acc[0][j]);
            acc[1][j] = mma(p[1], q[j], acc[1][j]);
        }
        if (bias)
#pragma unroll
            for (int j = 0; j < 8; ++j) ab[j] = mma(ones, q[j], ab[j]);
        p[0] = pn[0];
        p[1] = pn[1];
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j] = qn[j];
    }
    const int fr = lane & 15, fk = 4 * (lane >> 4), cols = nq * 16, rows = J.np * 16;
    float* o = J.part + (long long)z * (rows * cols + (J.b_off >= 0 ? cols : 0));
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        if (a && !two) break;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (j < nq)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[(16 * (i0 + a) + fk + r) * cols + 16 * j + fr] = acc[a][j][r];
    }
    if (bias && fk == 0)
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (j < nq) o[rows * cols + 16 * j + fr] = ab[j][0];
}

// Sums the partial gradients in order; the last row of workgroups also forms
// the loss, the mean of the squared errors.
__global__ __launch_bounds__(256) void mlp_grad_reduce(GradJobs jobs, float* g, const float* err2, int C, float* loss) {
    const int tid = threadIdx.x;
    if (blockIdx.y == GRAD_JOBS) {
        __shared__ float red[4];
        if (blockIdx.x) return;
        float s = 0.0f;
        for (int c = tid; c < C; c += 256) s += err2[c];
        s = wave_sum_f(s);
        if ((tid & 63) == 0) red[tid >> 6] = s;
        __syncthreads();
        if (tid == 0) loss[0] = (red[0] + red[1] + red[2] + red[3]) / (float)C;
        return;
    }
    const GradJob& J = jobs.j[blockIdx.y];
    const int cols = J.nq * 16, rows = J.np * 16, n = rows * cols + (J.b_off >= 0 ? cols : 0);
    const int i = blockIdx.x * 256 + tid;
    if (i >= n) return;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    int z = 0;
    for (; z + 4 <= J.nz; z += 4)
#pragma unroll
        for (int u = 0; u < 4; ++u) s[u] += J.part[(long long)(z + u) * n + i];
    for (; z < J.nz; ++z) s[0] += J.part[(long long)z * n + i];
    const float v = (s[0] + s[1]) + (s[2] + s[3]);
    if (i < rows * cols) g[J.w_off + (i / cols) * J.w_cols + i % cols] = v;
    else g[J.b_off + i - rows * cols] = v;
}

// ---------------------------------------------------------------------------
// Elementwise / reduction kernels
// ---------------------------------------------------------------------------
// X [C*NS x 16] BF16: candidate c's rows are its part's samples with their
// signed distance to the plane (x, y, z, s, zeros); S [C*NS] the distances
__global__ void mlp_pack_points(const float* pts, const float* planes, const int* part_of, int C, bf16_t* X,
                                float* S) {
    const long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= (long long)C * NS) return;
    const long long c = r / NS;
    const int i = (int)(r % NS);
    const float* p = pts + ((long long)part_of[c] * NS + i) * 3;
    const float* pl = planes + 4 * c;
    const float sd = pl[0] * p[0] + pl[1] * p[1] + pl[2] * p[2] + pl[3];
    S[r] = sd;
    bf16_t* x = X + r * KIN;
    x[0] = f2bf(p[0]);
    x[1] = f2bf(p[1]);
    x[2] = f2bf(p[2]);
    x[3] = f2bf(sd);
    for (int j = 4; j < KIN; ++j) x[j] = 0;
}

// per candidate and channel: max of A [C*NS x 128] over its rows with s >= 0
// (G[c][j]) and with s < 0 (G[c][128 + j]); 0 when a side has no sample
__global__ __launch_bounds__(HD) void mlp_maxpool(const bf16_t* A, const float* S, int C, float* G) {
    const int c = blockIdx.x, j = threadIdx.x;
    if (c >= C) return;
    float bp = -1e30f, bn = -1e30f;
    for (int i = 0; i < NS; ++i) {
        const long long r = (long long)c * NS + i;
        const float v = bf2f(A[r * HD + j]);
        if (S[r] >= 0.0f) bp = fmaxf(bp, v);
        else bn = fmaxf(bn, v);
    }
    G[(long long)c * 2 * HD + j] = bp > -1e30f ? bp : 0.0f;
    G[(long long)c * 2 * HD + HD + j] = bn > -1e30f ? bn : 0.0f;
}

// head input [C x 272] BF16: g+, g-, plane (n, d), zeros
__global__ void mlp_head_input(const float* G, const float* planes, int C, bf16_t* Hin) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)C * KH) return;
    const long long c = i / KH;
    const int j = (int)(i % KH);
    float v = 0.0f;
    if (j < 2 * HD) v = G[c * 2 * HD + j];
    else if (j < 2 * HD + 4) v = planes[4 * c + (j - 2 * HD)];
    Hin[i] = f2bf(v);
}

// Place of parameter i in the transposed copy: each weight block [K x N] as
// [N x K], everything else where it is.
__device__ __forceinline__ int wt_index(int i) {
    const int off[6] = {P_W1, P_W2, P_W3, P_H1, P_H2, P_H3}, K[6] = {KIN, HD, HD, KH, HD, HD},
              N[6] = {HD, HD, HD, HD, HD, NO};
    int r = i;
#pragma unroll
    for (int b = 0; b < 6; ++b) {
        const int j = i - off[b];
        if (j >= 0 && j < K[b] * N[b]) r = off[b] + (j % N[b]) * K[b] + j / N[b];
    }
    return r;
}

// Adam (FP32 master weights), then the BF16 copies used by the products
__global__ void mlp_adam(float* w, const float* gr, float* m, float* v, bf16_t* wb, bf16_t* wt, int n, float lr,
                         float b1, float b2, float eps, float c1, float c2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float g = gr[i];
    const float mi = b1 * m[i] + (1.0f - b1) * g;
    const float vi = b2 * v[i] + (1.0f - b2) * g * g;
    m[i] = mi;
    v[i] = vi;
    const float upd = lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] -= upd;
    wb[i] = f2bf(w[i]);
    wt[wt_index(i)] = wb[i];
}

__global__ void mlp_to_bf16(const float* w, bf16_t* wb, bf16_t* wt, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    wb[i] = f2bf(w[i]);
    wt[wt_index(i)] = wb[i];
}

// ---------------------------------------------------------------------------
// Surface samples of a part: NS area-stratified points in the part's box
// frame. One workgroup per part; triangle areas are prefix-summed in chunks
// into `cum` (nt floats per part at cum_off[p]). Sample i takes the triangle
// holding u = (i + 1/2) / NS of the total area and a point of it from a hash
// of (part, i).
// ---------------------------------------------------------------------------
struct SampleTask {
    const float* v;
    const int* t;
    int nv, nt;
    long long cum_off;
    float lo[3], hi[3];  // part box (for the frame)
};

__device__ __forceinline__ uint32_t mlp_hash(uint32_t x) {
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}

__global__ __launch_bounds__(256) void mlp_sample_kernel(const SampleTask* tasks, int P, float* cum_all, float* out) {
    __shared__ float wsum[4];
    __shared__ float carry;
    const int p = blockIdx.x, tid = threadIdx.x;
    if (p >= P) return;
    const SampleTask T = tasks[p];
    float* cum = cum_all + T.cum_off;
    if (tid == 0) carry = 0.0f;
    __syncthreads();
    for (int b = 0; b < T.nt; b += 256) {
        const int i = b + tid;
        float a = 0.0f;
        if (i < T.nt) {
            const int i0 = T.t[3 * i], i1 = T.t[3 * i + 1], i2 = T.t[3 * i + 2];
            const float ux = T.v[3 * i1] - T.v[3 * i0], uy = T.v[3 * i1 + 1] - T.v[3 * i0 + 1],
                        uz = T.v[3 * i1 + 2] - T.v[3 * i0 + 2];
            const float wx = T.v[3 * i2] - T.v[3 * i0], wy = T.v[3 * i2 + 1] - T.v[3 * i0 + 1],
                        wz = T.v[3 * i2 + 2] - T.v[3 * i0 + 2];
            const float cx = uy * wz - uz * wy, cy = uz * wx - ux * wz, cz = ux * wy - uy * wx;
            a = 0.5f * sqrtf(cx * cx + cy * cy + cz * cz);
        }
        float s = a;  // inclusive wave scan
        for (int o = 1; o < 64; o <<= 1) {
            const float y = __shfl_up(s, o);
            if ((tid & 63) >= o) s += y;
        }
        if ((tid & 63) == 63) wsum[tid >> 6] = s;
        __syncthreads();
        float base = carry;
        for (int q = 0; q < (tid >> 6); ++q) base += wsum[q];
        if (i < T.nt) cum[i] = base + s;
        __syncthreads();
        if (tid == 0) carry += wsum[0] + wsum[1] + wsum[2] + wsum[3];
        __syncthreads();
    }
    const float total = carry;
    float c[3], sc = 0.0f;
    for (int j = 0; j < 3; ++j) {
        c[j] = 0.5f * (T.lo[j] + T.hi[j]);
        sc = fmaxf(sc, 0.5f * (T.hi[j] - T.lo[j]));
    }
    const float inv = sc > 0.0f ? 1.0f / sc : 0.0f;
    for (int i = tid; i < NS; i += 256) {
        float px = 0.f, py = 0.f, pz = 0.f;
        if (T.nt > 0 && total > 0.0f) {
            const float u = ((float)i + 0.5f) / (float)NS * total;
            int lo = 0, hi = T.nt - 1;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (cum[mid] > u) hi = mid;
                else lo = mid + 1;
            }
            const uint32_t h1 = mlp_hash((uint32_t)p * 0x9e3779b1u + (uint32_t)i * 0x85ebca6bu + 1u);
            const uint32_t h2 = mlp_hash(h1 ^ 0x68e31da4u);
            float r1 = (float)(h1 >> 8) * (1.0f / 16777216.0f), r2 = (float)(h2 >> 8) * (1.0f / 16777216.0f);
            if (r1 + r2 > 1.0f) { r1 = 1.0f - r1; r2 = 1.0f - r2; }
            const int i0 = T.t[3 * lo], i1 = T.t[3 * lo + 1], i2 = T.t[3 * lo + 2];
            const float* a = T.v + 3 * i0;
            const float* b = T.v + 3 * i1;
            const float* d = T.v + 3 * i2;
            px = a[0] + r1 * (b[0] - a[0]) + r2 * (d[0] - a[0]);
            py = a[1] + r1 * (b[1] - a[1]) + r2 * (d[1] - a[1]);
            pz = a[2] + r1 * (b[2] - a[2]) + r2 * (d[2] - a[2]);
        }
        float* o = out + ((long long)p * NS + i) * 3;
        o[0] = (px - c[0]) * inv;
        o[1] = (py - c[1]) * inv;
        o[2] = (pz - c[2]) * inv;
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
struct gpu_mlp {
    float* w;      // FP32 master weights [P_TOTAL]
    bf16_t* wb;    // BF16 copy
    bf16_t* wt;    // BF16 copy, every weight block transposed
    float* g;      // gradients
    float* m;      // Adam moments
    float* v;
    int step;
    // grow-only activations and partial sums
    char* act;
    size_t act_cap;
    float* part;
    size_t part_cap;
};

namespace {

template <class T> T* carve(char*& p, size_t n) {
    T* r = (T*)p;
    p += (n * sizeof(T) + 255) / 256 * 256;
    return r;
}

// workspace of at least n floats for the weight gradients' partial sums
// (grow-only; a growth waits for the stream so no launch still reads the old
// buffer)
float* part_ws(gpu_ctx_t ctx, gpu_mlp* mp, size_t n) {
    if (n > mp->part_cap) {
        if (hipStreamSynchronize(ctx->stream) != hipSuccess) return nullptr;
        if (mp->part) (void)hipFree(mp->part);
        mp->part = nullptr;
        mp->part_cap = 0;
        if (hipMalloc((void**)&mp->part, n * sizeof(float)) != hipSuccess) return nullptr;
        mp->part_cap = n;
    }
    return mp->part;
}

int gemm(gpu_ctx_t ctx, int M, int N, int K, const bf16_t* A, long long sam, long long sak, const bf16_t* B,
         long long sbk, long long sbn, const float* bias, int relu, float* C, long long ldc, bf16_t* Cb,
         long long ldcb) {
    if (M <= 0 || N <= 0) return 0;
    const GemmArgs g{M, N, K, A, sam, sak, B, sbk, sbn, bias, relu, C, ldc, Cb, ldcb};
    const int tm = (M + GM - 1) / GM, tn = (N + GN - 1) / GN;
    hipLaunchKernelGGL(mlp_gemm_kernel, dim3((unsigned)tn, (unsigned)tm), dim3(256), 0, ctx->stream, g);
    HIP_TRY(hipGetLastError());
    return 0;
}

struct Act {
    // layer by layer
    bf16_t *X, *A1, *A2, *A3, *B1, *B2;
    float *S, *G, *Yw;
    // fused
    bf16_t* Hin;
    float* Y;
    // training
    bf16_t* gb;
    uint8_t* arg;
    float *err2, *loss;
    unsigned long long* mask;
    int *off, *total, *list;
    s4v_t *htiles, *etiles;
};

enum ActKind { ACT_LAYERS, ACT_FUSED, ACT_TRAIN };

// Buffers of C candidates in the network's grow-only block. Training's largest
// part is the encoder's operand tiles, for as many rows as there could be.
int act_layout(gpu_ctx_t ctx, gpu_mlp* mp, int C, ActKind kind, Act* a) {
    const size_t n = (size_t)C, R = n * NS;
    auto carve_all = [&](char* p) -> size_t {
        char* const p0 = p;
        *a = Act{};
        a->Hin = carve<bf16_t>(p, n * KH);
        if (kind == ACT_LAYERS) {
            a->X = carve<bf16_t>(p, R * KIN);
            a->A1 = carve<bf16_t>(p, R * HD);
            a->A2 = carve<bf16_t>(p, R * HD);
            a->A3 = carve<bf16_t>(p, R * HD);
            a->B1 = carve<bf16_t>(p, n * HD);
            a->B2 = carve<bf16_t>(p, n * HD);
            a->S = carve<float>(p, R);
            a->G = carve<float>(p, n * 2 * HD);
            a->Yw = carve<float>(p, n * NO);
        } else {
            a->Y = carve<float>(p, n);
        }
        if (kind == ACT_TRAIN) {
            a->gb = carve<bf16_t>(p, n * 2 * HD);
            a->arg = carve<uint8_t>(p, n * 2 * HD);
            a->err2 = carve<float>(p, n);
            a->loss = carve<float>(p, 64);
            a->mask = carve<unsigned long long>(p, n * 4);
            a->off = carve<int>(p, n);
            a->total = carve<int>(p, 1);
            a->list = carve<int>(p, R + 32);
            a->htiles = carve<s4v_t>(p, (n + 15) / 16 * HT_N * 64);
            a->etiles = carve<s4v_t>(p, (R / 16 + 2) * ET_N * 64);
        }
        return (size_t)(p - p0);
    };
    const size_t need = carve_all(nullptr);
    if (need > mp->act_cap) {
        if (mp->act) HIP_TRY(hipFree(mp->act));
        mp->act = nullptr;
        mp->act_cap = 0;
        HIP_TRY(hipMalloc((void**)&mp->act, need));
        mp->act_cap = need;
    }
    (void)carve_all(mp->act);
    return 0;
}

// layer by layer over device inputs: points [P*NS x 3], planes [C x 4],
// part_of [C]; the scores in column 0 of Yw [C x NO]
int forward_layers(gpu_ctx_t ctx, gpu_mlp* mp, const float* d_pts, const float* d_planes, const int* d_part, int C,
            Act& a) {
    const int R = C * NS;
    const bf16_t* W = mp->wb;
    const float* Wf = mp->w;
    hipLaunchKernelGGL(mlp_pack_points, dim3((unsigned)((R + 255) / 256)), dim3(256), 0, ctx->stream, d_pts,
                       d_planes, d_part, C, a.X, a.S);
    HIP_TRY(hipGetLastError());
    if (int rc = gemm(ctx, R, HD, KIN, a.X, KIN, 1, W + P_W1, HD, 1, Wf + P_B1, 1, nullptr, 0, a.A1, HD))
        return rc;
    if (int rc = gemm(ctx, R, HD, HD, a.A1, HD, 1, W + P_W2, HD, 1, Wf + P_B2, 1, nullptr, 0, a.A2, HD))
        return rc;
    if (int rc = gemm(ctx, R, HD, HD, a.A2, HD, 1, W + P_W3, HD, 1, Wf + P_B3, 1, nullptr, 0, a.A3, HD))
        return rc;
    hipLaunchKernelGGL(mlp_maxpool, dim3((unsigned)C), dim3(HD), 0, ctx->stream, a.A3, a.S, C, a.G);
    HIP_TRY(hipGetLastError());
    {
        const long long n = (long long)C * KH;
        hipLaunchKernelGGL(mlp_head_input, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, a.G,
                           d_planes, C, a.Hin);
        HIP_TRY(hipGetLastError());
    }
    if (int rc = gemm(ctx, C, HD, KH, a.Hin, KH, 1, W + P_H1, HD, 1, Wf + P_C1, 1, nullptr, 0, a.B1, HD))
        return rc;
    if (int rc = gemm(ctx, C, HD, HD, a.B1, HD, 1, W + P_H2, HD, 1, Wf + P_C2, 1, nullptr, 0, a.B2, HD))
        return rc;
    return gemm(ctx, C, NO, HD, a.B2, HD, 1, W + P_H3, NO, 1, Wf + P_C3, 0, a.Yw, NO, nullptr, 0);
}

// point layers and pooling (arg: also the pooled rows)
int encode(gpu_ctx_t ctx, gpu_mlp* mp, const float* d_pts, const float* d_planes, const int* d_part, int C, Act& a) {
    HIP_TRY(hipFuncSetAttribute((const void*)mlp_encode_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)ENC_LDS));
    const int grid = std::max(1, std::min((C + 1) / 2, ctx->n_cu));
    hipLaunchKernelGGL(mlp_encode_kernel, dim3((unsigned)grid), dim3(512), ENC_LDS, ctx->stream, d_pts, d_planes,
                       d_part, C, (const bf16_t*)mp->wt, (const float*)mp->w, a.Hin, a.arg);
    HIP_TRY(hipGetLastError());
    return 0;
}

// inference through the fused kernels: the scores into d_out [C]
int forward_fused(gpu_ctx_t ctx, gpu_mlp* mp, const float* d_pts, const float* d_planes, const int* d_part, int C,
                  Act& a, float* d_out) {
    if (int rc = encode(ctx, mp, d_pts, d_planes, d_part, C, a)) return rc;
    hipLaunchKernelGGL(mlp_head_kernel<false>, dim3((unsigned)((C + 63) / 64)), dim3(256), 0, ctx->stream,
                       (const bf16_t*)a.Hin, C, (const bf16_t*)mp->wt, (const bf16_t*)mp->wb, (const float*)mp->w, d_out,
                       (const float*)nullptr, (float*)nullptr, (bf16_t*)nullptr, (s4v_t*)nullptr);
    HIP_TRY(hipGetLastError());
    return 0;
}

// forward, loss and gradients of the mean squared error (into mp->g)
int train_grads(gpu_ctx_t ctx, gpu_mlp* mp, const float* d_pts, const float* d_planes, const int* d_part,
                const float* d_t, int C, Act& a) {
    const bf16_t *wt = mp->wt, *wb = mp->wb;
    const float* wf = mp->w;
    if (int rc = encode(ctx, mp, d_pts, d_planes, d_part, C, a)) return rc;
    hipLaunchKernelGGL(mlp_head_kernel<true>, dim3((unsigned)((C + 63) / 64)), dim3(256), 0, ctx->stream,
                       (const bf16_t*)a.Hin, C, wt, wb, wf, a.Y, d_t, a.err2, a.gb, a.htiles);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(mlp_rows_mark, dim3((unsigned)C), dim3(256), 0, ctx->stream, (const bf16_t*)a.Hin,
                       (const uint8_t*)a.arg, a.mask, a.off);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(mlp_rows_scan, dim3(1), dim3(1024), 0, ctx->stream, a.off, C, a.total, a.list);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(mlp_rows_fill, dim3((unsigned)C), dim3(256), 0, ctx->stream,
                       (const unsigned long long*)a.mask, (const int*)a.off, a.list);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipFuncSetAttribute((const void*)mlp_rows_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)ROWS_LDS));
    const int grid = std::max(1, std::min((C * (NS / 32) + 7) / 8, ctx->n_cu));
    hipLaunchKernelGGL(mlp_rows_kernel, dim3((unsigned)grid), dim3(512), ROWS_LDS, ctx->stream, d_pts, d_planes, d_part,
                       wt, wb, wf, (const uint8_t*)a.arg, (const bf16_t*)a.gb, (const int*)a.list,
                       (const int*)a.total, a.etiles);
    HIP_TRY(hipGetLastError());
    // the weight gradients: enough workgroups per job that each sees a few
    // dozen groups at most (the loads of a group are its latency)
    const int hg = (C + 15) / 16, eg = C * (NS / 16);
    const int nzh = std::max(1, std::min(hg / 8, 32)), nze = std::max(1, std::min(eg / 16, 256));
    GradJobs jobs{};
    size_t floats = 0;
    int blocks = 0, most = 0;
    auto job = [&](int k, bool enc, int p0, int np, int q0, int nq, int w_off, int w_cols, int b_off) {
        GradJob& J = jobs.j[k];
        J.tiles = enc ? a.etiles : a.htiles;
        J.stride = enc ? ET_N : HT_N;
        J.p0 = p0; J.np = np; J.q0 = q0; J.nq = nq;
        J.rows = enc ? a.total : nullptr;
        J.groups = hg;
        J.nz = enc ? nze : nzh;
        J.block0 = blocks;
        J.w_off = w_off; J.w_cols = w_cols; J.b_off = b_off;
        blocks += J.nz;
        const int n = np * nq * 256 + (b_off >= 0 ? nq * 16 : 0);
        most = std::max(most, n);
        J.part = (float*)(uintptr_t)floats;  // its offset until the block is known
        floats += (size_t)J.nz * n;
    };
    job(0, true, ET_A2, 8, ET_D3, 8, P_W3, HD, P_B3);
    job(1, true, ET_A1, 8, ET_D2, 8, P_W2, HD, P_B2);
    job(2, true, ET_X, 1, ET_D1, 8, P_W1, HD, P_B1);
    job(3, false, HT_HIN, 8, HT_D1, 8, P_H1, HD, P_C1);
    job(4, false, HT_HIN + 8, 8, HT_D1, 8, P_H1 + 128 * HD, HD, -1);
    job(5, false, HT_HIN + 16, 1, HT_D1, 8, P_H1 + 256 * HD, HD, -1);
    job(6, false, HT_B1, 8, HT_D2, 8, P_H2, HD, P_C2);
    job(7, false, HT_B2, 8, HT_DY, 1, P_H3, NO, P_C3);
    float* part = part_ws(ctx, mp, floats);
    REQUIRE(part, "mlp: partial-sum workspace allocation failed");
    for (GradJob& J : jobs.j) J.part = part + (size_t)(uintptr_t)J.part;
    hipLaunchKernelGGL(mlp_grad_kernel, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, jobs);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(mlp_grad_reduce, dim3((unsigned)((most + 255) / 256), GRAD_JOBS + 1), dim3(256), 0, ctx->stream,
                       jobs, mp->g, (const float*)a.err2, C, a.loss);
    HIP_TRY(hipGetLastError());
    return 0;
}

// Inputs staged on the device (points [P*NS*3], planes [C*4], part_of,
// targets), for one call.
struct Staged {
    float* pts = nullptr;
    float* planes = nullptr;
    int* part = nullptr;
    float* t = nullptr;
    char* base = nullptr;
    gpu_ctx_t ctx = nullptr;
    ~Staged() {
        if (base) (void)hipFreeAsync(base, ctx->stream);
    }
    int load(gpu_ctx_t c, const float* h_pts, int P, const float* h_planes, const int* h_part, int C,
             const float* h_t) {
        ctx = c;
        for (int i = 0; i < C; ++i) {
            if (h_part[i] < 0 || h_part[i] >= P) return -2;
            if (i > 0 && h_part[i] < h_part[i - 1]) return -3;
        }
        const size_t b0 = ((size_t)P * NS * 12 + 255) / 256 * 256, b1 = ((size_t)C * 16 + 255) / 256 * 256,
                     b2 = ((size_t)C * 4 + 255) / 256 * 256;
        if (hipMallocAsync((void**)&base, b0 + b1 + 2 * b2 + 256, c->stream) != hipSuccess) return -1;
        pts = (float*)base;
        planes = (float*)(base + b0);
        part = (int*)(base + b0 + b1);
        t = (float*)(base + b0 + b1 + b2);
        if (hipMemcpyAsync(pts, h_pts, (size_t)P * NS * 12, hipMemcpyHostToDevice, c->stream) != hipSuccess ||
            hipMemcpyAsync(planes, h_planes, (size_t)C * 16, hipMemcpyHostToDevice, c->stream) != hipSuccess ||
            hipMemcpyAsync(part, h_part, (size_t)C * 4, hipMemcpyHostToDevice, c->stream) != hipSuccess)
            return -1;
        if (h_t && hipMemcpyAsync(t, h_t, (size_t)C * 4, hipMemcpyHostToDevice, c->stream) != hipSuccess) return -1;
        return 0;
    }
};

int stage_err(gpu_ctx_t ctx, int rc) {
    if (rc == -2) set_error(ctx, "mlp: part_of index out of range");
    else if (rc == -3) set_error(ctx, "mlp: candidates must be grouped by part (part_of ascending)");
    else set_error(ctx, "mlp: input staging failed");
    return -1;
}

}  // namespace

namespace cuacd {
int mlp_forward_dev(gpu_ctx_t ctx, gpu_mlp* mp, const float* d_pts, int P, const float* d_planes, const int* d_part,
                    int C, float* d_out) {
    // bounded activations: slices of at most 8192 candidates (2M encoder
    // rows) layer by layer; the fused kernel keeps those rows in registers
    (void)P;
    const bool fused = mlp_fused_on() != 0;
    const int slice = fused ? 65536 : 8192;
    Act a;
    if (int rc = act_layout(ctx, mp, std::min(slice, C), fused ? ACT_FUSED : ACT_LAYERS, &a)) return rc;
    for (int c0 = 0; c0 < C; c0 += slice) {
        const int n = std::min(slice, C - c0);
        if (fused) {
            if (int rc = forward_fused(ctx, mp, d_pts, d_planes + 4ll * c0, d_part + c0, n, a, d_out + c0)) return rc;
            continue;
        }
        if (int rc = forward_layers(ctx, mp, d_pts, d_planes + 4ll * c0, d_part + c0, n, a)) return rc;
        HIP_TRY(hipMemcpy2DAsync(d_out + c0, 4, a.Yw, 4 * NO, 4, n, hipMemcpyDeviceToDevice, ctx->stream));
    }
    return 0;
}

int mlp_sample_dev(gpu_ctx_t ctx, const MlpSamplePart* parts, int P, float* d_out) {
    if (P <= 0) return 0;
    std::vector<SampleTask> st(P);
    long long off = 0;
    for (int p = 0; p < P; ++p) {
        st[p].v = parts[p].v;
        st[p].t = parts[p].t;
        st[p].nv = parts[p].nv;
        st[p].nt = parts[p].nt;
        st[p].cum_off = off;
        for (int j = 0; j < 3; ++j) { st[p].lo[j] = parts[p].lo[j]; st[p].hi[j] = parts[p].hi[j]; }
        off += parts[p].nt;
    }
    SampleTask* d_st = nullptr;
    float* d_cum = nullptr;
    HIP_TRY(hipMallocAsync((void**)&d_st, sizeof(SampleTask) * P, ctx->stream));
    HIP_TRY(hipMallocAsync((void**)&d_cum, 4 * (size_t)(off + 1), ctx->stream));
    HIP_TRY(hipMemcpyAsync(d_st, st.data(), sizeof(SampleTask) * P, hipMemcpyHostToDevice, ctx->stream));
    hipLaunchKernelGGL(mlp_sample_kernel, dim3((unsigned)P), dim3(256), 0, ctx->stream, d_st, P, d_cum, d_out);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipFreeAsync(d_st, ctx->stream));
    HIP_TRY(hipFreeAsync(d_cum, ctx->stream));
    return 0;
}
}  // namespace cuacd

extern "C" {

int gpu_mlp_n_params(void) { return P_TOTAL; }

int gpu_mlp_create(gpu_ctx_t ctx, const float* params, int seed, gpu_mlp_t* out) {
    *out = nullptr;
    HIP_TRY(hipSetDevice(ctx->device));
    std::vector<float> w(P_TOTAL, 0.0f);
    if (params) {
        memcpy(w.data(), params, sizeof(float) * P_TOTAL);
    } else {
        // He-uniform weights on the used entries, zero biases and padding
        uint64_t s = 0x9E3779B97F4A7C15ull ^ (uint64_t)(uint32_t)seed;
        auto rnd = [&]() {
            s = s * 6364136223846793005ull + 1442695040888963407ull;
            return (double)(s >> 11) * (1.0 / 9007199254740992.0);
        };
        auto fill = [&](int off, int rows_used, int rows, int cols_used, int cols, int fan_in) {
            const double a = std::sqrt(6.0 / fan_in);
            for (int r = 0; r < rows; ++r)
                for (int c = 0; c < cols; ++c)
                    w[off + r * cols + c] = (r < rows_used && c < cols_used) ? (float)((2.0 * rnd() - 1.0) * a) : 0.0f;
        };
        fill(P_W1, 4, KIN, HD, HD, 4);
        fill(P_W2, HD, HD, HD, HD, HD);
        fill(P_W3, HD, HD, HD, HD, HD);
        fill(P_H1, 2 * HD + 4, KH, HD, HD, 2 * HD + 4);
        fill(P_H2, HD, HD, HD, HD, HD);
        fill(P_H3, HD, HD, 1, NO, HD);
    }
    gpu_mlp* m = (gpu_mlp*)calloc(1, sizeof(gpu_mlp));
    REQUIRE(m, "out of host memory");
    const size_t fb = sizeof(float) * P_TOTAL;
    if (hipMalloc((void**)&m->w, fb) != hipSuccess || hipMalloc((void**)&m->wb, 2 * P_TOTAL) != hipSuccess ||
        hipMalloc((void**)&m->wt, 2 * P_TOTAL) != hipSuccess ||
        hipMalloc((void**)&m->g, fb) != hipSuccess || hipMalloc((void**)&m->m, fb) != hipSuccess ||
        hipMalloc((void**)&m->v, fb) != hipSuccess) {
        gpu_mlp_destroy(ctx, m);
        set_error(ctx, "mlp: allocation failed");
        return -1;
    }
    HIP_TRY(hipMemcpyAsync(m->w, w.data(), fb, hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(hipMemsetAsync(m->g, 0, fb, ctx->stream));
    HIP_TRY(hipMemsetAsync(m->m, 0, fb, ctx->stream));
    HIP_TRY(hipMemsetAsync(m->v, 0, fb, ctx->stream));
    hipLaunchKernelGGL(mlp_to_bf16, dim3((P_TOTAL + 255) / 256), dim3(256), 0, ctx->stream, m->w, m->wb, m->wt, P_TOTAL);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    *out = m;
    return 0;
}

void gpu_mlp_destroy(gpu_ctx_t ctx, gpu_mlp_t m) {
    if (!m) return;
    if (ctx) (void)hipStreamSynchronize(ctx->stream);
    if (m->w) (void)hipFree(m->w);
    if (m->wb) (void)hipFree(m->wb);
    if (m->wt) (void)hipFree(m->wt);
    if (m->g) (void)hipFree(m->g);
    if (m->m) (void)hipFree(m->m);
    if (m->v) (void)hipFree(m->v);
    if (m->act) (void)hipFree(m->act);
    if (m->part) (void)hipFree(m->part);
    free(m);
}

int gpu_mlp_get_params(gpu_ctx_t ctx, gpu_mlp_t m, float* out) {
    REQUIRE(m, "null network");
    HIP_TRY(hipMemcpyAsync(out, m->w, sizeof(float) * P_TOTAL, hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    return 0;
}

int gpu_mlp_forward(gpu_ctx_t ctx, gpu_mlp_t m, const float* points, int n_parts, const float* planes,
                    const int* part_of, int n_cand, float* out_scores) {
    REQUIRE(m && n_parts >= 0 && n_cand >= 0, "mlp_forward: bad arguments");
    if (n_cand == 0) return 0;
    HIP_TRY(hipSetDevice(ctx->device));
    Staged s;
    if (int rc = s.load(ctx, points, n_parts, planes, part_of, n_cand, nullptr)) return stage_err(ctx, rc);
    float* d_out = nullptr;
    HIP_TRY(hipMallocAsync((void**)&d_out, 4ll * n_cand + 16, ctx->stream));
    int rc = mlp_forward_dev(ctx, m, s.pts, n_parts, s.planes, s.part, n_cand, d_out);
    if (rc == 0) {
        HIP_TRY(hipMemcpyAsync(out_scores, d_out, 4ll * n_cand, hipMemcpyDeviceToHost, ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));
    }
    (void)hipFreeAsync(d_out, ctx->stream);
    return rc;
}

int gpu_mlp_train_step(gpu_ctx_t ctx, gpu_mlp_t m, const float* points, int n_parts, const float* planes,
                       const int* part_of, int n_cand, const float* targets, float lr, int apply,
                       float* out_loss, float* out_grads) {
    REQUIRE(m && n_parts > 0 && n_cand > 0, "mlp_train_step: bad arguments");
    HIP_TRY(hipSetDevice(ctx->device));
    Staged s;
    if (int rc = s.load(ctx, points, n_parts, planes, part_of, n_cand, targets)) return stage_err(ctx, rc);
    Act a;
    if (int rc = act_layout(ctx, m, n_cand, ACT_TRAIN, &a)) return rc;
    if (int rc = train_grads(ctx, m, s.pts, s.planes, s.part, s.t, n_cand, a)) return rc;
    if (out_grads)
        HIP_TRY(hipMemcpyAsync(out_grads, m->g, sizeof(float) * P_TOTAL, hipMemcpyDeviceToHost, ctx->stream));
    if (apply) {
        m->step++;
        const float b1 = 0.9f, b2 = 0.999f;
        const float c1 = 1.0f - std::pow(b1, (float)m->step), c2 = 1.0f - std::pow(b2, (float)m->step);
        hipLaunchKernelGGL(mlp_adam, dim3((P_TOTAL + 255) / 256), dim3(256), 0, ctx->stream, m->w, m->g, m->m, m->v,
                           m->wb, m->wt, P_TOTAL, lr, b1, b2, 1e-8f, c1, c2);
        HIP_TRY(hipGetLastError());
    }
    float loss = 0.0f;
    HIP_TRY(hipMemcpyAsync(&loss, a.loss, 4, hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    if (out_loss) *out_loss = loss;
    return 0;
}

int gpu_mlp_sample_parts(gpu_ctx_t ctx, const float* verts, const int* vert_off, const int* tris, const int* tri_off,
                         int n_parts, float* out_points) {
    REQUIRE(n_parts >= 0, "sample_parts: bad arguments");
    if (n_parts == 0) return 0;
    HIP_TRY(hipSetDevice(ctx->device));
    const size_t tv = (size_t)vert_off[n_parts], tt = (size_t)tri_off[n_parts];
    float* dv = nullptr;
    int* dt = nullptr;
    float* dout = nullptr;
    HIP_TRY(hipMallocAsync((void**)&dv, 12 * tv + 16, ctx->stream));
    HIP_TRY(hipMallocAsync((void**)&dt, 12 * tt + 16, ctx->stream));
    HIP_TRY(hipMallocAsync((void**)&dout, 12ull * NS * n_parts, ctx->stream));
    HIP_TRY(hipMemcpyAsync(dv, verts, 12 * tv, hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(hipMemcpyAsync(dt, tris, 12 * tt, hipMemcpyHostToDevice, ctx->stream));
    std::vector<MlpSamplePart> ps(n_parts);
    for (int p = 0; p < n_parts; ++p) {
        const int v0 = vert_off[p], v1 = vert_off[p + 1];
        REQUIRE(v1 >= v0 && tri_off[p + 1] >= tri_off[p], "sample_parts: bad offsets");
        ps[p].v = dv + 3ll * v0;
        ps[p].t = dt + 3ll * tri_off[p];
        ps[p].nv = v1 - v0;
        ps[p].nt = tri_off[p + 1] - tri_off[p];
        for (int j = 0; j < 3; ++j) { ps[p].lo[j] = 1e30f; ps[p].hi[j] = -1e30f; }
        for (int i = v0; i < v1; ++i)
            for (int j = 0; j < 3; ++j) {
                ps[p].lo[j] = std::min(ps[p].lo[j], verts[3ll * i + j]);
                ps[p].hi[j] = std::max(ps[p].hi[j], verts[3ll * i + j]);
            }
        for (int i = tri_off[p]; i < tri_off[p + 1]; ++i)
            for (int j = 0; j < 3; ++j)
                REQUIRE(tris[3ll * i + j] >= 0 && tris[3ll * i + j] < v1 - v0, "sample_parts: triangle index out of range");
    }
    int rc = mlp_sample_dev(ctx, ps.data(), n_parts, dout);
    if (rc == 0) {
        HIP_TRY(hipMemcpyAsync(out_points, dout, 12ull * NS * n_parts, hipMemcpyDeviceToHost, ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));
    }
    (void)hipFreeAsync(dv, ctx->stream);
    (void)hipFreeAsync(dt, ctx->stream);
    (void)hipFreeAsync(dout, ctx->stream);
    return rc;
}

// GEMM through the C-ABI (tests of the MFMA tile layout): C [M x N] FP32 =
// A . B for BF16 host matrices with element strides.
int gpu_mlp_gemm_test(gpu_ctx_t ctx, int M, int N, int K, const unsigned short* A, long long sam, long long sak,
                      long long a_len, const unsigned short* B, long long sbk, long long sbn, long long b_len,
                      float* C) {
    HIP_TRY(hipSetDevice(ctx->device));
    REQUIRE(M > 0 && N > 0 && K > 0 && a_len > 0 && b_len > 0, "gemm_test: bad sizes");
    REQUIRE((M - 1) * sam + (K - 1) * sak < a_len && (K - 1) * sbk + (N - 1) * sbn < b_len,
            "gemm_test: strides exceed the operands");
    bf16_t *dA = nullptr, *dB = nullptr;
    float* dC = nullptr;
    HIP_TRY(hipMallocAsync((void**)&dA, 2 * a_len, ctx->stream));
    HIP_TRY(hipMallocAsync((void**)&dB, 2 * b_len, ctx->stream));
    HIP_TRY(hipMallocAsync((void**)&dC, 4ll * M * N, ctx->stream));
    HIP_TRY(hipMemcpyAsync(dA, A, 2 * a_len, hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(hipMemcpyAsync(dB, B, 2 * b_len, hipMemcpyHostToDevice, ctx->stream));
    int rc = gemm(ctx, M, N, K, dA, sam, sak, dB, sbk, sbn, nullptr, 0, dC, N, nullptr, 0);
    if (rc == 0) {
        HIP_TRY(hipMemcpyAsync(C, dC, 4ll * M * N, hipMemcpyDeviceToHost, ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));
    }
    (void)hipFreeAsync(dA, ctx->stream);
    (void)hipFreeAsync(dB, ctx->stream);
    (void)hipFreeAsync(dC, ctx->stream);
    (void)hipStreamSynchronize(ctx->stream);
    return rc;
}

}  // extern "C"
