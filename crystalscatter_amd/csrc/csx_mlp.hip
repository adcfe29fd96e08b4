// Surrogate network of the fits: a small MLP that maps a parameter set and a pixel's (qx, qy)
// to the normalised log-intensity of that pixel.  It has no counterpart in the reference; the
// fit driver uses it to propose starting simplices and to pre-screen vertices, and the exact
// kernels re-score every point it accepts.
//
//   input   6 normalised parameters + 64 Fourier features sin/cos(a_f), 32 phases
//           a_f = 2*pi*(F_f0*qx + F_f1*qy) + F_f2*|q|*v_f, where v_f is the physical value of
//           parameter pidx_f (offset + scale * normalised value) or 1 (pidx_f < 0)
//           (70 values, zero-padded to 128 columns)
//   hidden  4 x 256, SiLU
//   output  1 (linear)
//
// Precision: BF16 weights and activations on the matrix cores (v_mfma_f32_16x16x32_bf16),
// FP32 accumulation, FP32 master weights and Adam state.  One kernel takes kPM rows through the
// whole network with their activations in one LDS tile (k_mlp: inference, or forward and
// backward with Z kept in registers); for the weight gradients it also leaves H_{l-1}^T and
// dZ_l^T (bf16) behind, and dW_l = dZ_l^T . H_{l-1} is one NT product over the rows for all
// layers together (k_wgrad), whose split partials k_finish adds in a fixed order.  Each weight
// is kept in bf16 in both orientations.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "csx.h"

namespace csm {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kIn = CSX_MLP_IN_PAD;    // padded input width
constexpr int kUsed = CSX_MLP_IN;      // used inputs: 6 parameters + 64 Fourier features
constexpr int kH = CSX_MLP_HIDDEN;     // hidden width
constexpr int kL = CSX_MLP_LAYERS;     // hidden layers
constexpr int kNF = CSX_MLP_NFREQ;     // Fourier frequencies
constexpr int kNP = CSX_MLP_NPAR;      // parameters per set
constexpr int kBM = 128;               // max_batch is rounded up to a multiple of this

// Offsets of the FP32 master parameters (one buffer): hidden layer l has W_l [kH][in_l]
// (out x in) then b_l [kH]; then the output weights w [kH] and bias.
__host__ __device__ constexpr int in_of(int l) { return l == 0 ? kIn : kH; }
__host__ __device__ constexpr int64_t w_off(int l) {
    return l == 0 ? 0 : (int64_t)kH * kIn + kH + (int64_t)(l - 1) * ((int64_t)kH * kH + kH);
}
__host__ __device__ constexpr int64_t b_off(int l) { return w_off(l) + (int64_t)kH * in_of(l); }
constexpr int64_t kOutW = w_off(kL);
constexpr int64_t kOutB = kOutW + kH;
constexpr int64_t kNParams = kOutB + 1;

// Sigmoid 1 / (1 + e^-z): the reciprocal of the hardware, 1 ulp, with one Newton step, which
// rounds it correctly; an IEEE division here was a third of the inference's instructions.  The
// denominator is kept finite, so that the step of an infinite one gives 0 like the division.
__device__ __forceinline__ float sigm(float z) {
    const float x = fminf(1.0f + __expf(-z), 3.402823466e38f);
    const float r = __builtin_amdgcn_rcpf(x);
    return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
}
__device__ __forceinline__ float silu_grad(float z) {
    const float s = sigm(z);
    return s * (1.0f + z * (1.0f - s));
}

// Position of weight (row, k) of a [rows][K] matrix in its bf16 copy: MFMA A fragments of 16 rows
// x 32 k one after the other, rows first, each as the 64 lanes hold it (lane row % 16 +
// 16 (k % 32 / 8), 8 values), so a wave's fragment load is 1 KB in a row.  Row-major, it touched
// 16 cache lines of which it used half.
__host__ __device__ constexpr int frag_index(int row, int k, int rows) {
    return ((k / 32) * (rows / 16) + row / 16) * 512 + ((row % 16) + 16 * (k % 32 / 8)) * 8 + k % 8;
}

// ---- input features ----------------------------------------------------------------
// Feature phases (see the header comment): frequencies F [kNF][3], parameter index per
// phase, and the affine map normalised -> physical value per parameter.
struct Features {
    float f[kNF][3];
    int32_t pidx[kNF];
    float off[kNP], sc[kNP];
};

// ---- the network over kPM rows ---------------------------------------------------------
// NW waves; wave w owns 256 / NW consecutive features of every layer.  A layer is the product
// W . H^T (D[feature][row]): the weights are the A operand, read straight from the bf16
// [out][in] copies (L2-resident), the rows' activations the B operand, from LDS.  A lane then
// holds four consecutive features of one row, so the epilogue writes 8 bytes where the other
// orientation writes four 2-byte values.  The bias is added to the finished products.
// Bound: the vector unit -- per row 1024 SiLU values at about 60 cycles each per wave of 64
// (exp2 and reciprocal at quarter rate) and 32 sincosf, against 422 matrix cycles.  2.1 M rows of
// inference: 1.25 ms (2.75 ms with H . W^T, IEEE divisions and row-major weights).  1.10 ms with
// the bare reciprocal, hardware sines of the phase in turns and the bias as the accumulators'
// initial value, but then activations flip bf16 roundings and y moves by 8e-4 in norm.
// Training, 65,536 rows: 0.17-0.19 ms, its phases between barriers (4 waves at 2 per SIMD: 0.22 ms),
// for the 11 launches and 0.38 ms of the layer-by-layer passes.
constexpr int kPM = 64;        // rows per block
constexpr int kInferWaves = 4, kTrainWaves = 8;
constexpr int kPLd = kH + 8;   // LDS row stride (bf16): 16-byte aligned rows
static_assert(kPM == 64 && kH == 256, "one lane per row");

// Parameters of set[i] (already normalised by the caller; an index outside [0, nsets) is
// clamped, the host checks them), then sin and cos of the kNF phases, then zeros; rows >= n are
// zero.  Lane = row; each wave takes kNF / NW phases.
template <int NW>
__device__ __forceinline__ void embed_rows(int r0, int n, int nsets, const float* __restrict__ par,
                                           const int32_t* __restrict__ set, const float* __restrict__ q,
                                           const Features& ft, bf16* act) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = r0 + lane;
    const bool live = i < n;
    float v[kNP];
#pragma unroll
    for (int k = 0; k < kNP; ++k) v[k] = 0.0f;
    float qx = 0.0f, qy = 0.0f;
    if (live) {
        const float* pp = par + (size_t)min(max(set[i], 0), nsets - 1) * kNP;  // clamped: never out of bounds
#pragma unroll
        for (int k = 0; k < kNP; ++k) v[k] = pp[k];
        qx = q[2 * (size_t)i];
        qy = q[2 * (size_t)i + 1];
    }
    uint32_t* row = reinterpret_cast<uint32_t*>(act + lane * kPLd);
    auto pack = [](float a, float b) {
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        const bf16x2 p = {(bf16)a, (bf16)b};
        return __builtin_bit_cast(uint32_t, p);
    };
    static_assert(kNP % 2 == 0 && kNF % 8 == 0 && kIn % 2 == 0, "features in pairs");
    if (wave == 0)
#pragma unroll
        for (int k = 0; k < kNP; k += 2) row[k / 2] = pack(v[k], v[k + 1]);
    const float qa = sqrtf(qx * qx + qy * qy);
    constexpr int NF = kNF / NW;
#pragma unroll 1
    for (int f0 = 0; f0 < NF; f0 += 2) {
        float sn[2], cs[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int f = wave * NF + f0 + e;
            const int j = ft.pidx[f];
            float pv = 1.0f;
#pragma unroll
            for (int k = 0; k < kNP; ++k) pv = (k == j) ? ft.off[k] + ft.sc[k] * v[k] : pv;
            sincosf(6.283185307f * (ft.f[f][0] * qx + ft.f[f][1] * qy) + ft.f[f][2] * qa * pv, &sn[e], &cs[e]);
            if (!live) sn[e] = cs[e] = 0.0f;
        }
        row[(kNP + NF * wave + f0) / 2] = pack(sn[0], sn[1]);
        row[(kNP + kNF + NF * wave + f0) / 2] = pack(cs[0], cs[1]);
    }
    for (int k = kUsed / 2 + wave; k < kIn / 2; k += NW) row[k] = 0u;
}

// acc[i][j] += the wave's 16 NI features x kPM rows of W . act^T over k < K (W in fragment order,
// kH rows).
template <int K, int NI, bool PREFETCH>
__device__ __forceinline__ void layer_product(const bf16* __restrict__ W, const bf16* act, int wn,
                                              f32x4 (&acc)[NI][4]) {
    const int lane = threadIdx.x & 63, fr = lane & 15, fk = (lane >> 4) * 8;
    const bf16* wp = W + (size_t)(wn / 16) * 512 + lane * 8;
    if constexpr (PREFETCH) {
        bf16x8 a[NI], an[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) a[i] = *(const bf16x8*)(wp + i * 512);
#pragma unroll
        for (int ks = 0; ks < K; ks += 32) {
            if (ks + 32 < K)
#pragma unroll
                for (int i = 0; i < NI; ++i) an[i] = *(const bf16x8*)(wp + ((ks / 32 + 1) * (kH / 16) + i) * 512);
            bf16x8 b[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = *(const bf16x8*)&act[(j * 16 + fr) * kPLd + ks + fk];
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < NI; ++i) a[i] = an[i];
        }
    } else {
        // training: half of the registers hold Z, no room for a second set of fragments
#pragma unroll 1
        for (int ks = 0; ks < K; ks += 32, wp += (kH / 16) * 512) {
            bf16x8 a[NI], b[4];
#pragma unroll
            for (int i = 0; i < NI; ++i) a[i] = *(const bf16x8*)(wp + i * 512);
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = *(const bf16x8*)&act[(j * 16 + fr) * kPLd + ks + fk];
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
}

// Accumulator (i, j)[r] is feature wn + 16 i + 4 (lane / 16) + r of row 16 j + lane % 16.
__device__ __forceinline__ int acc_feature(int wn, int i) { return wn + i * 16 + ((threadIdx.x & 63) >> 4) * 4; }
__device__ __forceinline__ int acc_row(int j) { return j * 16 + (threadIdx.x & 15); }

// The LDS tile's transpose to outT, a [ncol][kPM] matrix in fragment order (frag_index), which is
// what k_wgrad's MFMAs take: a block's rows are contiguous (with all rows of a feature in a row, a
// tile's 256 pieces lay 128 KB apart and shared a few memory channels).  A thread takes two
// features and 2 / NW of the rows (b32 reads, conflict-free), one k octet of both in 32 bytes; with
// SUM the columns' sums over those rows as well.
// Partial sums per block of kPM rows: biases of the kL layers, output weights, output bias, loss.
constexpr int kPartB = (kL + 1) * kH + 2;
template <int NW, bool SUM>
__device__ __forceinline__ void store_columns(const bf16* act, bf16* __restrict__ outT, int ncol,
                                              float* __restrict__ sums) {
    constexpr int R = 2 * kPM / NW;
    const int c = (threadIdx.x & 127) * 2, h = (threadIdx.x >> 7) * R;
    if (c >= ncol) return;
    float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
    for (int g = 0; g < R; g += 8) {
        uint32_t x[8];
        uint4 lo, hi;
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = *(const uint32_t*)&act[(h + g + k) * kPLd + c];
        uint32_t* lp = reinterpret_cast<uint32_t*>(&lo);
        uint32_t* hp = reinterpret_cast<uint32_t*>(&hi);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            lp[k] = (x[2 * k] & 0xffffu) | (x[2 * k + 1] << 16);
            hp[k] = (x[2 * k] >> 16) | (x[2 * k + 1] & 0xffff0000u);
        }
        if constexpr (SUM) {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                s0 += __uint_as_float(x[k] << 16);
                s1 += __uint_as_float(x[k] & 0xffff0000u);
            }
        }
        *(uint4*)&outT[frag_index(c, h + g, ncol)] = lo;
        *(uint4*)&outT[frag_index(c + 1, h + g, ncol)] = hi;
    }
    if constexpr (SUM) *(float2*)&sums[(threadIdx.x >> 7) * kH + c] = make_float2(s0, s1);
}

// Training outputs of k_mlp.
struct TrainArgs {
    const float* tgt;     // targets
    bf16* xt;             // X^T, H_l^T, dZ_l^T: per block of kPM rows [features][kPM], fragments
    bf16* ht[kL - 1];
    bf16* dzt[kL];
    const bf16* wtb;      // weights [in][out]
    float* part;          // [blocks][kPartB]
};

// 4 waves per SIMD in both forms.  Training keeps Z in registers (64 of them with 8 waves), and
// with two waves per SIMD its phases between barriers did not hide each other.
template <bool TRAIN, int NW>
__global__ void __launch_bounds__(64 * NW, 4) k_mlp(int n, int nsets, const float* __restrict__ par,
                                             const int32_t* __restrict__ set, const float* __restrict__ q,
                                             const Features ft, const bf16* __restrict__ wb,
                                             const float* __restrict__ p, float* __restrict__ y, const TrainArgs tr) {
    __shared__ __attribute__((aligned(16))) bf16 act[kPM * kPLd];
    __shared__ float s_y[kPM];
    __shared__ __attribute__((aligned(16))) float s_sum[TRAIN ? NW / 2 : 1][kH];  // column sums of the row groups
    const int r0 = blockIdx.x * kPM;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    constexpr int NI = 16 / NW;  // 16-feature tiles per wave
    const int wn = wave * 16 * NI;
    constexpr int64_t kW1 = (int64_t)kH * kIn, kWl = (int64_t)kH * kH;
    bf16x4 z[TRAIN ? kL : 1][NI][4];  // pre-activations, kept for the backward pass
    embed_rows<NW>(r0, n, nsets, par, set, q, ft, act);
    __syncthreads();
    if constexpr (TRAIN) store_columns<NW, false>(act, tr.xt + (size_t)r0 * kIn, kIn, nullptr);
#pragma unroll
    for (int l = 0; l < kL; ++l) {
        f32x4 acc[NI][4];
        const float* b = p + b_off(l);
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (l == 0) layer_product<kIn, NI, !TRAIN>(wb, act, wn, acc);
        else layer_product<kH, NI, !TRAIN>(wb + kW1 + (l - 1) * kWl, act, wn, acc);
        __syncthreads();  // every wave has read the layer's input
        __builtin_amdgcn_sched_barrier(0);  // the bias loads would be moved up here and spill
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const float* bi = b + acc_feature(wn, i);
            const float bias[4] = {bi[0], bi[1], bi[2], bi[3]};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                bf16x4 h;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float zz = acc[i][j][r] + bias[r];
                    h[r] = (bf16)(zz * sigm(zz));
                    if constexpr (TRAIN) z[l][i][j][r] = (bf16)zz;
                }
                *(bf16x4*)&act[acc_row(j) * kPLd + acc_feature(wn, i)] = h;
            }
        }
        __syncthreads();
        if constexpr (TRAIN)
            if (l < kL - 1) store_columns<NW, false>(act, tr.ht[l] + (size_t)r0 * kH, kH, nullptr);
    }
    // output layer: one wave per row
    const float* w = p + kOutW;
    for (int rr = wave; rr < kPM; rr += NW) {
        const bf16* row = act + rr * kPLd + lane * 4;
        float sum = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; ++c) sum = fmaf((float)row[c], w[lane * 4 + c], sum);
        for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
        if (lane == 0) {
            sum += p[kOutB];
            if constexpr (TRAIN) s_y[rr] = sum;
            else if (r0 + rr < n) y[r0 + rr] = sum;
        }
    }
    if constexpr (TRAIN) {
        // loss 1/n sum (y - t)^2: dy = 2 (y - t) / n, 0 for rows >= n
        __syncthreads();
        float* part = tr.part + (size_t)blockIdx.x * kPartB;
        auto sum_groups = [&](float* out) {  // a barrier after the groups' sums
            if (t < kH) {
                float v = s_sum[0][t];
#pragma unroll
                for (int g = 1; g < NW / 2; ++g) v += s_sum[g][t];
                out[t] = v;
            }
        };
        if (t < kPM) {
            const float e = r0 + t < n ? s_y[t] - tr.tgt[r0 + t] : 0.0f;
            const float dy = 2.0f * e / (float)n;
            s_y[t] = dy;
            float db = dy, ls = e * e;
            for (int o = 32; o > 0; o >>= 1) {
                db += __shfl_xor(db, o, 64);
                ls += __shfl_xor(ls, o, 64);
            }
            if (t == 0) {
                part[(kL + 1) * kH] = db;
                part[(kL + 1) * kH + 1] = ls;
            }
        }
        __syncthreads();
        {
            // output weights: dw[c] = sum over the rows of dy H_kL[row][c], rows and features
            // split as in store_columns
            constexpr int R = 2 * kPM / NW;
            const int c = (t & 127) * 2, h = (t >> 7) * R;
            float s0 = 0.0f, s1 = 0.0f;
#pragma unroll 8
            for (int r = 0; r < R; ++r) {
                const uint32_t x = *(const uint32_t*)&act[(h + r) * kPLd + c];
                s0 = fmaf(__uint_as_float(x << 16), s_y[h + r], s0);
                s1 = fmaf(__uint_as_float(x & 0xffff0000u), s_y[h + r], s1);
            }
            *(float2*)&s_sum[t >> 7][c] = make_float2(s0, s1);
        }
        __syncthreads();  // the last activations are read
        sum_groups(part + kL * kH);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float dy = s_y[acc_row(j)];
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                bf16x4 dz;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    dz[r] = (bf16)(dy * w[acc_feature(wn, i) + r] * silu_grad((float)z[kL - 1][i][j][r]));
                *(bf16x4*)&act[acc_row(j) * kPLd + acc_feature(wn, i)] = dz;
            }
        }
        __syncthreads();
#pragma unroll
        for (int l = kL - 1; l >= 0; --l) {
            // dZ_l^T and the bias gradient's partials
            store_columns<NW, true>(act, tr.dzt[l] + (size_t)r0 * kH, kH, s_sum[0]);
            if (l == 0) {
                __syncthreads();
                sum_groups(part);
                break;
            }
            // dH_{l-1} = dZ_l . W_l, dZ_{l-1} = dH_{l-1} silu'(Z_{l-1})
            f32x4 acc[NI][4];
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            layer_product<kH, NI, false>(tr.wtb + kW1 + (l - 1) * kWl, act, wn, acc);
            __syncthreads();
            sum_groups(part + l * kH);
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    bf16x4 dz;
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        dz[r] = (bf16)(acc[i][j][r] * silu_grad((float)z[l - 1][i][j][r]));
                    *(bf16x4*)&act[acc_row(j) * kPLd + acc_feature(wn, i)] = dz;
                }
            __syncthreads();
        }
    }
}

// ---- weight gradients --------------------------------------------------------------------
// part_l[split][out][in] = sum over the split's rows of dZ_l[m][out] H_{l-1}[m][in]: block x
// takes layer x whole (256 outputs x its inputs), block y the split, so every operand byte is
// read by one block only.  8 waves, 4 x 2, each 64 outputs x half of the inputs; the operands lie
// in fragment order and go straight to registers, the next k step's while this one is
// multiplied.  Bound: the operands' bytes, 235 MB at 65,536 rows (50 us at 4.8 TB/s).  As 128 x 128
// tiles through LDS, per layer, each byte was read by two blocks, seldom on one XCD.
struct WgradArgs {
    const bf16* dzt[kL];
    const bf16* ht[kL];  // layer inputs: X^T, H_0^T, ...
    float* part[kL];     // [splits][kH][in]
    int nb, kchunk;      // row blocks of kPM, row blocks per split
};
template <int K>
__device__ __forceinline__ void wgrad_layer(const bf16* __restrict__ A, const bf16* __restrict__ B,
                                            float* __restrict__ out, int k0, int k1) {
    constexpr int NJ = K / 32;  // 16-column tiles per wave
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave & 3) * 64, wn = (wave >> 2) * (K / 2);
    const bf16* ap = A + (size_t)(wm / 16) * 512 + lane * 8;
    const bf16* bp = B + (size_t)(wn / 16) * 512 + lane * 8;
    // a block's kPM rows are two k steps of kH / 16 and K / 16 fragments each
    f32x4 acc[4][NJ];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    bf16x8 a[4], b[NJ], an[4], bn[NJ];
    const int s0 = 2 * k0, s1 = 2 * k1;
    auto fetch = [&](int st, bf16x8* fa, bf16x8* fb) {
#pragma unroll
        for (int i = 0; i < 4; ++i) fa[i] = *(const bf16x8*)(ap + ((size_t)st * (kH / 16) + i) * 512);
#pragma unroll
        for (int j = 0; j < NJ; ++j) fb[j] = *(const bf16x8*)(bp + ((size_t)st * (K / 16) + j) * 512);
    };
    auto multiply = [&](const bf16x8* fa, const bf16x8* fb) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    };
    fetch(s0, a, b);
#pragma unroll 1
    for (int st = s0; st < s1; st += 2) {  // an even number of steps
        fetch(st + 1, an, bn);
        multiply(a, b);
        fetch(min(st + 2, s1 - 2), a, b);
        multiply(an, bn);
    }
    // accumulator (i, j)[r] is C[wm + 16i + 4(lane/16) + r][wn + 16j + lane%16]
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m0 = wm + i * 16 + (lane >> 4) * 4;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int c = wn + j * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) out[(size_t)(m0 + r) * K + c] = acc[i][j][r];
        }
    }
}
__global__ void __launch_bounds__(512, 2) k_wgrad(const WgradArgs g) {
    const int l = blockIdx.x;
    const int k0 = blockIdx.y * g.kchunk, k1 = min(g.nb, k0 + g.kchunk);
    if (k0 >= k1) return;
    if (l == 0) wgrad_layer<kIn>(g.dzt[0], g.ht[0], g.part[0] + (size_t)blockIdx.y * kH * kIn, k0, k1);
    else wgrad_layer<kH>(g.dzt[l], g.ht[l], g.part[l] + (size_t)blockIdx.y * kH * kH, k0, k1);
}

// The packed gradient from the partials, each sum in a fixed order: blocks below kFinW take 1024
// weights each (four per thread, summed over the splits), the others 16 of the kPartB sums over
// the nr row blocks (16 threads per value, then a tree).
constexpr int kFinW = (int)((kH * kIn + (kL - 1) * (int64_t)kH * kH) / 1024);
constexpr int kFinB = (kPartB + 15) / 16;
struct FinishArgs {
    const float* part[kL];
    const float* pb;   // [nr][kPartB]
    float* g;          // packed gradient
    float* loss;       // sum of the squared errors
    int ns, nr;
};
__global__ void __launch_bounds__(256) k_finish(const FinishArgs a) {
    const int t = threadIdx.x;
    if ((int)blockIdx.x < kFinW) {
        int c = blockIdx.x * 1024 + t * 4, l = 0;
        if (c >= kH * kIn) {
            c -= kH * kIn;
            l = 1 + c / (kH * kH);
            c %= kH * kH;
        }
        const int sz = kH * in_of(l);
        float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 8
        for (int k = 0; k < a.ns; ++k) {
            const float4 v = *(const float4*)&a.part[l][(size_t)k * sz + c];
            s.x += v.x;
            s.y += v.y;
            s.z += v.z;
            s.w += v.w;
        }
        float* o = a.g + w_off(l) + c;
        o[0] = s.x;
        o[1] = s.y;
        o[2] = s.z;
        o[3] = s.w;
        return;
    }
    __shared__ float red[16][17];
    const int vi = t & 15, sg = t >> 4;
    const int v = ((int)blockIdx.x - kFinW) * 16 + vi;
    float s = 0.0f;
    if (v < kPartB)
#pragma unroll 8
        for (int k = sg; k < a.nr; k += 16) s += a.pb[(size_t)k * kPartB + v];
    red[sg][vi] = s;
    __syncthreads();
    for (int h = 8; h > 0; h >>= 1) {
        if (sg < h) red[sg][vi] += red[sg + h][vi];
        __syncthreads();
    }
    if (sg == 0 && v < kPartB) {
        const float r = red[0][vi];
        if (v < kL * kH) a.g[b_off(v / kH) + v % kH] = r;
        else if (v < (kL + 1) * kH) a.g[kOutW + v - kL * kH] = r;
        else if (v == (kL + 1) * kH) a.g[kOutB] = r;
        else *a.loss = r;
    }
}

// Adam on the FP32 master parameters, then the bf16 copies of the hidden weights in both
// orientations (W and W^T), in the order in which k_mlp's waves read them.
__global__ void __launch_bounds__(256) k_adam(int64_t np, float* __restrict__ p, const float* __restrict__ g,
                                              float* __restrict__ m1, float* __restrict__ m2, float lr, float b1,
                                              float b2, float eps, float c1, float c2) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= np) return;
    const float gi = g[i];
    const float a = b1 * m1[i] + (1.0f - b1) * gi;
    const float v = b2 * m2[i] + (1.0f - b2) * gi * gi;
    m1[i] = a;
    m2[i] = v;
    p[i] -= lr * (a * c1) / (sqrtf(v * c2) + eps);
}
__global__ void __launch_bounds__(256) k_cast_weights(const float* __restrict__ p, bf16* __restrict__ wb,
                                                      bf16* __restrict__ wtb) {
    // flat index over all hidden weights, layer by layer
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    for (int l = 0; l < kL; ++l) {
        const int64_t cnt = (int64_t)kH * in_of(l);
        if (i < cnt) {
            const int o = (int)(i / in_of(l)), k = (int)(i % in_of(l));
            const bf16 v = (bf16)p[w_off(l) + i];
            const int64_t base = l == 0 ? 0 : (int64_t)kH * kIn + (int64_t)(l - 1) * kH * kH;
            wb[base + frag_index(o, k, kH)] = v;
            wtb[base + frag_index(k, o, in_of(l))] = v;
            return;
        }
        i -= cnt;
    }
}

}  // namespace csm

// ===========================================================================
// C ABI
// ===========================================================================
using namespace csm;

struct csx_mlp {
    int device = 0;
    int max_batch = 0;  // rows, a multiple of 128
    hipStream_t stream = nullptr;
    bool own_stream = false;
    std::string err;
    Features feat;
    // parameters
    float *p = nullptr, *g = nullptr, *m1 = nullptr, *m2 = nullptr;
    bf16 *wb = nullptr, *wtb = nullptr;  // hidden weights, [out][in] and [in][out]
    int64_t adam_t = 0;
    // training buffers: the layers' inputs and dZ, transposed; partial sums
    bf16 *XT = nullptr, *HT[kL - 1] = {}, *dZT[kL] = {};
    float *part = nullptr, *pb = nullptr, *loss = nullptr;
    int splits = 0;
};

namespace {

int fail(csx_mlp* m, int code, const std::string& msg) {
    if (m) m->err = msg;
    return code;
}
#define MCHK(m, call)                                                                        \
    do {                                                                                     \
        hipError_t e_ = (call);                                                              \
        if (e_ != hipSuccess) return fail(m, CSX_E_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

// splitmix64 -> uniform doubles, Box-Muller normals (host-side initialisation only)
struct Rng {
    uint64_t s;
    uint64_t next() {
        uint64_t z = (s += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    }
    double uni() { return (double)(next() >> 11) * 0x1.0p-53; }
};

int cast_weights(csx_mlp* m) {
    const int64_t nw = (int64_t)kH * kIn + (int64_t)(kL - 1) * kH * kH;
    hipLaunchKernelGGL(k_cast_weights, dim3((unsigned)((nw + 255) / 256)), dim3(256), 0, m->stream, m->p, m->wb, m->wtb);
    MCHK(m, hipGetLastError());
    return CSX_OK;
}

int check_rows(csx_mlp* m, int n, int nsets) {
    if (n < 1 || n > m->max_batch) return fail(m, CSX_E_ARG, "row count must be in [1, max_batch]");
    if (nsets < 1) return fail(m, CSX_E_ARG, "need at least one parameter set");
    return CSX_OK;
}

int infer(csx_mlp* m, int n, int nsets, const float* d_par, const int32_t* d_set, const float* d_q, float* d_y) {
    hipLaunchKernelGGL((k_mlp<false, kInferWaves>), dim3((unsigned)((n + kPM - 1) / kPM)), dim3(64 * kInferWaves), 0,
                       m->stream, n, nsets, d_par, d_set, d_q, m->feat, m->wb, m->p, d_y, TrainArgs{});
    MCHK(m, hipGetLastError());
    return CSX_OK;
}

}  // namespace

extern "C" {

int64_t csx_mlp_nparams(void) { return kNParams; }

int csx_mlp_create(int device, int max_batch, uint64_t seed, csx_mlp** out) {
    if (!out || max_batch < 1 || max_batch > (1 << 24)) return CSX_E_ARG;
    *out = nullptr;
    if (hipSetDevice(device) != hipSuccess) return CSX_E_HIP;
    csx_mlp* m = new csx_mlp();
    m->device = device;
    m->max_batch = (max_batch + kBM - 1) / kBM * kBM;
    const size_t M = (size_t)m->max_batch;
    // weight-gradient splits over the rows, >= 512 rows each: 64 give one block per CU (4 layers);
    // every split writes and reads 0.9 MB of partials
    m->splits = (int)std::max<size_t>(1, std::min<size_t>(64, M / 512));
    auto alloc = [&](void** p, size_t bytes) { return hipMalloc(p, bytes) == hipSuccess; };
    bool ok = hipStreamCreate(&m->stream) == hipSuccess;
    m->own_stream = ok;
    const int64_t nw = (int64_t)kH * kIn + (int64_t)(kL - 1) * kH * kH;
    ok = ok && alloc((void**)&m->p, kNParams * 4) && alloc((void**)&m->g, kNParams * 4) &&
         alloc((void**)&m->m1, kNParams * 4) && alloc((void**)&m->m2, kNParams * 4) &&
         alloc((void**)&m->wb, nw * 2) && alloc((void**)&m->wtb, nw * 2) &&
         alloc((void**)&m->XT, M * kIn * 2) && alloc((void**)&m->part, (size_t)m->splits * nw * 4) &&
         alloc((void**)&m->pb, (M / kPM) * kPartB * 4) && alloc((void**)&m->loss, 4);
    for (int l = 0; l < kL - 1 && ok; ++l) ok = alloc((void**)&m->HT[l], M * kH * 2);
    for (int l = 0; l < kL && ok; ++l) ok = alloc((void**)&m->dZT[l], M * kH * 2);
    if (!ok) {
        csx_mlp_destroy(m);
        return CSX_E_NOMEM;
    }
    // Initialisation: He-uniform hidden weights (fan-in = used inputs), zero biases, a
    // small output layer; Fourier frequencies with log-uniform magnitude in [0.5, 16]
    // cycles per nm^-1 and uniform directions.
    std::vector<float> hp(kNParams, 0.0f);
    Rng r{seed};
    for (int l = 0; l < kL; ++l) {
        const int fan = l == 0 ? kUsed : kH;
        const double bound = std::sqrt(6.0 / fan);
        for (int o = 0; o < kH; ++o)
            for (int k = 0; k < in_of(l); ++k)
                hp[w_off(l) + (int64_t)o * in_of(l) + k] = (l == 0 && k >= kUsed) ? 0.0f : (float)((2 * r.uni() - 1) * bound);
    }
    for (int c = 0; c < kH; ++c) hp[kOutW + c] = (float)((2 * r.uni() - 1) * std::sqrt(3.0 / kH));
    // default phases: 2*pi*F.q with log-uniform magnitudes in [0.5, 16] and uniform directions
    std::memset(&m->feat, 0, sizeof m->feat);
    for (int f = 0; f < kNF; ++f) {
        const double mag = 0.5 * std::pow(32.0, r.uni()), ang = 2 * M_PI * r.uni();
        m->feat.f[f][0] = (float)(mag * std::cos(ang));
        m->feat.f[f][1] = (float)(mag * std::sin(ang));
        m->feat.pidx[f] = -1;
    }
    for (int j = 0; j < kNP; ++j) m->feat.sc[j] = 1.0f;
    ok = hipMemcpyAsync(m->p, hp.data(), kNParams * 4, hipMemcpyHostToDevice, m->stream) == hipSuccess &&
         hipMemsetAsync(m->m1, 0, kNParams * 4, m->stream) == hipSuccess &&
         hipMemsetAsync(m->m2, 0, kNParams * 4, m->stream) == hipSuccess &&
         hipMemsetAsync(m->g, 0, kNParams * 4, m->stream) == hipSuccess && cast_weights(m) == CSX_OK &&
         hipStreamSynchronize(m->stream) == hipSuccess;
    if (!ok) {
        csx_mlp_destroy(m);
        return CSX_E_HIP;
    }
    *out = m;
    return CSX_OK;
}

void csx_mlp_destroy(csx_mlp* m) {
    if (!m) return;
    (void)hipSetDevice(m->device);
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    for (void* q : {(void*)m->p, (void*)m->g, (void*)m->m1, (void*)m->m2, (void*)m->wb, (void*)m->wtb,
                    (void*)m->XT, (void*)m->part, (void*)m->pb, (void*)m->loss})
        if (q) (void)hipFree(q);
    for (bf16* q : m->HT)
        if (q) (void)hipFree(q);
    for (bf16* q : m->dZT)
        if (q) (void)hipFree(q);
    if (m->own_stream && m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
}

int csx_mlp_last_error(const csx_mlp* m, char* buf, int len) {
    if (!m || !buf || len <= 0) return CSX_E_ARG;
    std::snprintf(buf, (size_t)len, "%s", m->err.c_str());
    return CSX_OK;
}

int csx_mlp_set_stream(csx_mlp* m, void* stream) {
    if (!m) return CSX_E_ARG;
    MCHK(m, hipStreamSynchronize(m->stream));
    if (m->own_stream) (void)hipStreamDestroy(m->stream);
    m->own_stream = false;
    m->stream = (hipStream_t)stream;
    return CSX_OK;
}

int csx_mlp_get_params(csx_mlp* m, float* h_params) {
    if (!m || !h_params) return CSX_E_ARG;
    MCHK(m, hipSetDevice(m->device));
    MCHK(m, hipMemcpyAsync(h_params, m->p, kNParams * 4, hipMemcpyDeviceToHost, m->stream));
    MCHK(m, hipStreamSynchronize(m->stream));
    return CSX_OK;
}

int csx_mlp_get_features(const csx_mlp* m, float* h_freq, int32_t* h_pidx, float* h_affine) {
    if (!m) return CSX_E_ARG;
    for (int f = 0; f < kNF; ++f) {
        if (h_freq) for (int c = 0; c < 3; ++c) h_freq[3 * f + c] = m->feat.f[f][c];
        if (h_pidx) h_pidx[f] = m->feat.pidx[f];
    }
    if (h_affine)
        for (int j = 0; j < kNP; ++j) {
            h_affine[2 * j] = m->feat.off[j];
            h_affine[2 * j + 1] = m->feat.sc[j];
        }
    return CSX_OK;
}

int csx_mlp_set_features(csx_mlp* m, const float* h_freq, const int32_t* h_pidx, const float* h_affine) {
    if (!m || !h_freq || !h_pidx || !h_affine) return CSX_E_ARG;
    for (int f = 0; f < kNF; ++f)
        if (h_pidx[f] < -1 || h_pidx[f] >= kNP) return fail(m, CSX_E_ARG, "parameter index of a phase out of range");
    MCHK(m, hipStreamSynchronize(m->stream));  // launches already queued keep their copy
    for (int f = 0; f < kNF; ++f) {
        for (int c = 0; c < 3; ++c) m->feat.f[f][c] = h_freq[3 * f + c];
        m->feat.pidx[f] = h_pidx[f];
    }
    for (int j = 0; j < kNP; ++j) {
        m->feat.off[j] = h_affine[2 * j];
        m->feat.sc[j] = h_affine[2 * j + 1];
    }
    return CSX_OK;
}

int csx_mlp_set_params(csx_mlp* m, const float* h_params) {
    if (!m) return CSX_E_ARG;
    MCHK(m, hipSetDevice(m->device));
    if (h_params) {
        // the padded input columns of the first layer stay zero
        std::vector<float> hp(h_params, h_params + kNParams);
        for (int o = 0; o < kH; ++o)
            for (int k = kUsed; k < kIn; ++k) hp[w_off(0) + (int64_t)o * kIn + k] = 0.0f;
        MCHK(m, hipMemcpyAsync(m->p, hp.data(), kNParams * 4, hipMemcpyHostToDevice, m->stream));
        MCHK(m, hipStreamSynchronize(m->stream));
        int rc = cast_weights(m);
        if (rc) return rc;
    }
    m->adam_t = 0;
    MCHK(m, hipMemsetAsync(m->m1, 0, kNParams * 4, m->stream));
    MCHK(m, hipMemsetAsync(m->m2, 0, kNParams * 4, m->stream));
    MCHK(m, hipStreamSynchronize(m->stream));
    return CSX_OK;
}

int csx_mlp_forward(csx_mlp* m, int n, int nsets, const float* d_par, const int32_t* d_set, const float* d_q,
                    float* d_y) {
    if (!m || !d_par || !d_set || !d_q || !d_y) return CSX_E_ARG;
    int rc = check_rows(m, n, nsets);
    if (rc) return rc;
    MCHK(m, hipSetDevice(m->device));
    return infer(m, n, nsets, d_par, d_set, d_q, d_y);
}

int csx_mlp_predict(csx_mlp* m, int n, int nsets, const float* d_par, const int32_t* d_set, const float* d_q,
                    float* d_y) {
    if (!m || !d_par || !d_set || !d_q || !d_y || n < 1 || nsets < 1) return CSX_E_ARG;
    MCHK(m, hipSetDevice(m->device));
    return infer(m, n, nsets, d_par, d_set, d_q, d_y);
}

int csx_mlp_gradient(csx_mlp* m, int n, int nsets, const float* d_par, const int32_t* d_set, const float* d_q,
                     const float* d_t, float* h_loss) {
    if (!m || !d_par || !d_set || !d_q || !d_t) return CSX_E_ARG;
    int rc = check_rows(m, n, nsets);
    if (rc) return rc;
    MCHK(m, hipSetDevice(m->device));
    const int nb = (n + kPM - 1) / kPM;
    const int64_t w1 = (int64_t)kH * kIn, wl = (int64_t)kH * kH;
    TrainArgs tr{};
    WgradArgs wg{};
    FinishArgs fa{};
    tr.tgt = d_t;
    tr.xt = m->XT;
    tr.wtb = m->wtb;
    tr.part = m->pb;
    wg.nb = nb;
    for (int l = 0; l < kL; ++l) {
        if (l < kL - 1) tr.ht[l] = m->HT[l];
        tr.dzt[l] = m->dZT[l];
        wg.dzt[l] = m->dZT[l];
        wg.ht[l] = l == 0 ? m->XT : m->HT[l - 1];
        wg.part[l] = m->part + (l == 0 ? 0 : m->splits * (w1 + (l - 1) * wl));
        fa.part[l] = wg.part[l];
    }
    hipLaunchKernelGGL((k_mlp<true, kTrainWaves>), dim3(nb), dim3(64 * kTrainWaves), 0, m->stream, n, nsets, d_par,
                       d_set, d_q, m->feat, m->wb, m->p, (float*)nullptr, tr);
    MCHK(m, hipGetLastError());
    wg.kchunk = (nb + m->splits - 1) / m->splits;
    const int ns = (nb + wg.kchunk - 1) / wg.kchunk;
    hipLaunchKernelGGL(k_wgrad, dim3(kL, ns), dim3(512), 0, m->stream, wg);
    MCHK(m, hipGetLastError());
    fa.pb = m->pb;
    fa.g = m->g;
    fa.loss = m->loss;
    fa.ns = ns;
    fa.nr = nb;
    hipLaunchKernelGGL(k_finish, dim3(kFinW + kFinB), dim3(256), 0, m->stream, fa);
    MCHK(m, hipGetLastError());
    if (h_loss) {
        float ls = 0.0f;
        MCHK(m, hipMemcpyAsync(&ls, m->loss, 4, hipMemcpyDeviceToHost, m->stream));
        MCHK(m, hipStreamSynchronize(m->stream));
        *h_loss = ls / (float)n;
    }
    return CSX_OK;
}

int csx_mlp_get_grads(csx_mlp* m, float* h_grads) {
    if (!m || !h_grads) return CSX_E_ARG;
    MCHK(m, hipSetDevice(m->device));
    MCHK(m, hipMemcpyAsync(h_grads, m->g, kNParams * 4, hipMemcpyDeviceToHost, m->stream));
    MCHK(m, hipStreamSynchronize(m->stream));
    return CSX_OK;
}

int csx_mlp_adam(csx_mlp* m, float lr, float b1, float b2, float eps) {
    if (!m || !(lr >= 0) || !(b1 >= 0 && b1 < 1) || !(b2 >= 0 && b2 < 1)) return CSX_E_ARG;
    MCHK(m, hipSetDevice(m->device));
    ++m->adam_t;
    const float c1 = (float)(1.0 / (1.0 - std::pow((double)b1, (double)m->adam_t)));
    const float c2 = (float)(1.0 / (1.0 - std::pow((double)b2, (double)m->adam_t)));
    hipLaunchKernelGGL(k_adam, dim3((unsigned)((kNParams + 255) / 256)), dim3(256), 0, m->stream, kNParams, m->p, m->g,
                       m->m1, m->m2, lr, b1, b2, eps, c1, c2);
    MCHK(m, hipGetLastError());
    return cast_weights(m);
}

int csx_mlp_train_step(csx_mlp* m, int n, int nsets, const float* d_par, const int32_t* d_set, const float* d_q,
                       const float* d_t, float lr, float* h_loss) {
    int rc = csx_mlp_gradient(m, n, nsets, d_par, d_set, d_q, d_t, h_loss);
    if (rc) return rc;
    return csx_mlp_adam(m, lr, 0.9f, 0.999f, 1e-8f);
}

int csx_mlp_synchronize(csx_mlp* m) {
    if (!m) return CSX_E_ARG;
    MCHK(m, hipStreamSynchronize(m->stream));
    return CSX_OK;
}

}  // extern "C"
