// libnfx: MLP surrogate kernels (BF16 operands on MFMA, FP32 accumulation) -- forward, backward
// and Adam for a fully connected GELU network.  No reference counterpart: the surrogate maps cell
// and indentation parameters to the force-indentation curve for parameter fitting.
//
// Every GEMM is C[M x N] = A[M x K] * B[N x K]^T with A and B row-major BF16 (K contiguous), the
// operand layout v_mfma_f32_16x16x32_bf16 reads directly: lane l holds 8 consecutive k of row
// (l % 16) of A and of row (l % 16) of B at k offset 8 * (l / 16); the 16 x 16 FP32 result tile
// leaves row 4 * (l / 16) + r, column l % 16 in accumulator element r.  Both tile kernels stage their operands
// in LDS and add the products of an output in the order of k.
// Split-K (split_k > 1, for the weight-gradient GEMMs, whose M x N output is small and K the
// batch): workgroup z of the third grid dimension accumulates K-slice z into an FP32 workspace
// plane; a finish kernel sums the planes in slice order (deterministic) and applies the epilogue.
//
// Epilogues fuse the elementwise work into the GEMM that produces it:
//   STORE     C = acc (+ bias)
//   FWD_GELU  Z = acc + bias (FP32, kept for the backward pass), H = gelu(Z) as BF16 in [M x N] and
//             transposed [N x M] (the transposed copy feeds the weight-gradient GEMM)
//   BWD_GELU  dZ = acc * gelu'(Z) as BF16 in [M x N] and [N x M]
//   ADAM      acc is the weight gradient: Adam update of the FP32 master weights C (eps added to the
//             bias-corrected sqrt(v)), BF16 copies of the weights in [M x N] and [N x M]
#include <hip/hip_runtime.h>

#include <cmath>

#include "nfx_common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace nfx {

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }

__device__ __forceinline__ float gelu_grad(float z) {
    return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

__device__ __forceinline__ __bf16 to_bf16(float x) { return (__bf16)x; }

// What the epilogue of four outputs reads (rows row .. row + 3, row a multiple of 4, of column col).  The kernels load
// it for many outputs before they store the first: memory instructions are counted in order, so the use of a load behind
// stores waits for them.  With the bias loaded per output, the epilogue of 65 536 x 512 GELU outputs took 50 us, now 37
// (33 of them erff); the layer at K = 512 84.8 -> 74.5 us
struct EpilogueIn {
    float bias, z[4], m[4], v[4], w[4];
};

template <int EPI>
__device__ __forceinline__ EpilogueIn epilogue_in(const nfx_mlp_gemm_args& g, int row, int col) {
    EpilogueIn in;
    if constexpr (EPI == NFX_MLP_STORE || EPI == NFX_MLP_FWD_GELU) in.bias = g.bias ? g.bias[col] : 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int64_t o = (int64_t)(row + r) * g.N + col;
        if constexpr (EPI == NFX_MLP_BWD_GELU) in.z[r] = g.Z[o];
        if constexpr (EPI == NFX_MLP_ADAM) {
            in.m[r] = g.adam_m[o];
            in.v[r] = g.adam_v[o];
            in.w[r] = g.C[o];
        }
    }
    return in;
}

// The epilogue itself.  The transposed copy's four entries are neighbours: one 8-byte store where HT is 8-byte aligned
template <int EPI>
__device__ __forceinline__ void epilogue4(const nfx_mlp_gemm_args& g, int row, int col, f32x4 v, const EpilogueIn& in) {
    const int M = g.M, N = g.N;
    bf16x4 h;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int64_t o = (int64_t)(row + r) * N + col;
        if constexpr (EPI == NFX_MLP_STORE) {
            g.C[o] = g.bias ? v[r] + in.bias : v[r];
        } else if constexpr (EPI == NFX_MLP_FWD_GELU) {
            const float z = v[r] + in.bias;
            if (g.C) g.C[o] = z;
            h[r] = to_bf16(gelu(z));
            static_cast<__bf16*>(g.H)[o] = h[r];
        } else if constexpr (EPI == NFX_MLP_BWD_GELU) {
            h[r] = to_bf16(v[r] * gelu_grad(in.z[r]));
            static_cast<__bf16*>(g.H)[o] = h[r];
        } else {  // ADAM
            const float gr = v[r] * g.grad_scale;
            const float m = g.beta1 * in.m[r] + (1.0f - g.beta1) * gr;
            const float s = g.beta2 * in.v[r] + (1.0f - g.beta2) * gr * gr;
            g.adam_m[o] = m;
            g.adam_v[o] = s;
            const float w = in.w[r] - g.lr_t * m / (sqrtf(s) * g.bc2 + g.eps);
            g.C[o] = w;
            h[r] = to_bf16(w);
            static_cast<__bf16*>(g.H)[o] = h[r];
        }
    }
    if constexpr (EPI != NFX_MLP_STORE) {
        if (!g.HT) return;
        __bf16* t = static_cast<__bf16*>(g.HT) + (int64_t)col * M + row;
        if ((reinterpret_cast<uintptr_t>(g.HT) & 7) == 0) {
            *reinterpret_cast<bf16x4*>(t) = h;
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) t[r] = h[r];
        }
    }
}

// The product for smaller grids.  A workgroup of four wavefronts (2 x 2) computes a kTM x kTN tile, staged
// through LDS in k-steps of kKS, so that each operand row is read once per workgroup in full 128-byte lines
// (kKS = 64).  The next k-step's operands are loaded into registers before the step's products; past the end the
// last step is read again, at a valid address, so that the loop has no branch and the compiler waits for the loads
// where they are used only.  Two LDS buffers and one barrier per k-step: a wave that writes a buffer has passed the
// barrier that ended its last reads.  Rows are padded by 8 BF16: the 16 rows of a fragment start at 16 different
// multiples of four banks.  Times at K = 512 with the GELU epilogue, against 128 x 32 tiles read from memory by
// each wave: 4096 x 512 20.8 -> 11.0 us, 1024 x 512 12.3 -> 5.8 us, slices of 512 of the weight gradients
// 14.0 -> 8.5 us.  What is left is latency: eight times load, barrier and LDS.  64 x 64, 128 x 64 and 128 x 32 tiles
// and two or four k-steps in flight were no faster (4096 x 512: 12.4 us with 64 x 32, 13.6 with 64 x 64, 16.4 with
// 128 x 64; 13.2 with two steps in flight).
// PARTIAL: store the raw accumulator of K-slice blockIdx.z into workspace plane blockIdx.z
// (the host checks K % (32 * gridDim.z) == 0).
template <int EPI, bool PARTIAL, int kTM, int kTN, int kKS>
__global__ __launch_bounds__(256) void k_gemm_tile(nfx_mlp_gemm_args g) {
    constexpr int kPitch = kKS + 8, kChunks = kKS / 8;           // 16-byte chunks per row
    constexpr int kRows = kTM + kTN, kPer = kRows * kChunks / 256;  // chunks per thread and k-step
    static_assert(kRows * kChunks % 256 == 0 && kTM % 32 == 0 && kTN % 32 == 0, "tile");
    constexpr int kMi = kTM / 32, kNi = kTN / 32;
    __shared__ __align__(16) __bf16 S[2][kRows * kPitch];  // kTM rows of A, then kTN rows of B
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int nt = g.N / kTN;
    const int m0 = (int)blockIdx.x / nt * kTM, n0 = (int)blockIdx.x % nt * kTN;
    const int r16 = lane & 15, kq = 8 * (lane >> 4);
    const int wm = (wave >> 1) * (kTM / 2), wn = (wave & 1) * (kTN / 2);
    const int kspan = g.K / (int)gridDim.z;
    const int kb = (int)blockIdx.z * kspan, n = kspan / kKS;
    const __bf16* src[kPer];
    int dst[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int c = tid + 256 * i, row = c / kChunks, kc = c % kChunks * 8;
        src[i] = (row < kTM ? static_cast<const __bf16*>(g.A) + (int64_t)(m0 + row) * g.lda
                            : static_cast<const __bf16*>(g.B) + (int64_t)(n0 + row - kTM) * g.ldb) +
                 kb + kc;
        dst[i] = row * kPitch + kc;
    }
    bf16x8 q[kPer];
    auto gload = [&](int s) {
        const int k = kKS * (s < n ? s : n - 1);
#pragma unroll
        for (int i = 0; i < kPer; ++i) q[i] = *reinterpret_cast<const bf16x8*>(src[i] + k);
    };
    f32x4 acc[kMi][kNi];
#pragma unroll
    for (int i = 0; i < kMi; ++i)
#pragma unroll
        for (int j = 0; j < kNi; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    gload(0);
    for (int s = 0, buf = 0; s < n; ++s, buf ^= 1) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) *reinterpret_cast<bf16x8*>(&S[buf][dst[i]]) = q[i];
        gload(s + 1);
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < kKS; kk += 32) {
            bf16x8 a[kMi], b[kNi];
#pragma unroll
            for (int i = 0; i < kMi; ++i)
                a[i] = *reinterpret_cast<const bf16x8*>(&S[buf][(wm + 16 * i + r16) * kPitch + kk + kq]);
#pragma unroll
            for (int j = 0; j < kNi; ++j)
                b[j] = *reinterpret_cast<const bf16x8*>(&S[buf][(kTM + wn + 16 * j + r16) * kPitch + kk + kq]);
#pragma unroll
            for (int i = 0; i < kMi; ++i)
#pragma unroll
                for (int j = 0; j < kNi; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
    const int row0 = m0 + wm + 4 * (lane >> 4), col0 = n0 + wn + r16;
    if constexpr (PARTIAL) {
        float* ws = g.workspace + (int64_t)blockIdx.z * g.M * g.N;
#pragma unroll
        for (int i = 0; i < kMi; ++i)
#pragma unroll
            for (int j = 0; j < kNi; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) ws[(int64_t)(row0 + 16 * i + r) * g.N + col0 + 16 * j] = acc[i][j][r];
    } else {
        EpilogueIn in[kMi][kNi];
#pragma unroll
        for (int i = 0; i < kMi; ++i)
#pragma unroll
            for (int j = 0; j < kNi; ++j) in[i][j] = epilogue_in<EPI>(g, row0 + 16 * i, col0 + 16 * j);
#pragma unroll
        for (int i = 0; i < kMi; ++i)
#pragma unroll
            for (int j = 0; j < kNi; ++j) epilogue4<EPI>(g, row0 + 16 * i, col0 + 16 * j, acc[i][j], in[i][j]);
    }
}

// Workgroups go to the 8 XCDs in turn: each XCD takes a contiguous range of the output's tiles, so that the tiles of
// the same rows share the reads of A in its L2
__device__ __forceinline__ int xcd_tile(int b, int nb) {
    const int q = nb >> 3, r = nb & 7, x = b & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// The same product for grids that fill the chip (M a multiple of 128, N of kTN; one pass over K): a
// workgroup tile of 128 x kTN staged through LDS, each wave a 64 x 64 sub-tile (4 x 4 MFMA tiles,
// 16 MFMAs per k-step from 8 LDS fragment reads).  Double
// buffered: the next k-slice goes global -> registers during the MFMAs and registers -> the other
// LDS buffer after them, one barrier per k-step.  Rows are padded by 8 BF16 against bank
// conflicts.  Accumulator layout and epilogue as k_gemm_tile.  Four waves per SIMD (the accumulators
// then live in VGPRs; the LDS fits them): 13-30 % faster than the three the unbounded allocation gives.
// The products are bound by what the L2s deliver: the layer of 65 536 x 512 with K = 512 and GELU takes 74.5 us with
// 128 x 128 tiles in launch order, 66.5 with each XCD's tiles together, 64.3 (0.53 PFLOP/s; 37 us are the epilogue's) with
// 128 x 256 tiles too, which read a quarter less.  256 x 256 tiles, one workgroup of 16 waves per CU, took 69
constexpr int kLdsTile = 128, kLdsK = 32, kLdsPitch = kLdsK + 8;
template <int EPI, int kTN>
__global__ __launch_bounds__(2 * kTN, 4) void k_gemm_lds(nfx_mlp_gemm_args g) {
    constexpr int kThreads = 2 * kTN, kRows = kLdsTile + kTN, kPer = 4 * kRows / kThreads;
    __shared__ __align__(16) __bf16 S[2][kRows * kLdsPitch];  // the rows of A, then those of B
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wm = (wave & 1) * 64, wn = (wave >> 1) * 64;
    const int tile = xcd_tile((int)(blockIdx.y * gridDim.x + blockIdx.x), (int)(gridDim.x * gridDim.y));
    const int m0 = tile / (int)gridDim.x * kLdsTile, n0 = tile % (int)gridDim.x * kTN;
    const int r16 = lane & 15, kq = 8 * (lane >> 4);
    // copy assignment: 4 chunks of 8 BF16 per row
    const __bf16* src[kPer];
    int dst[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int c = tid + kThreads * i, row = c >> 2, kc = (c & 3) * 8;
        src[i] = (row < kLdsTile ? static_cast<const __bf16*>(g.A) + (int64_t)(m0 + row) * g.lda
                                 : static_cast<const __bf16*>(g.B) + (int64_t)(n0 + row - kLdsTile) * g.ldb) +
                 kc;
        dst[i] = row * kLdsPitch + kc;
    }
    bf16x8 q[kPer];
    auto gload = [&](int k0) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) q[i] = *reinterpret_cast<const bf16x8*>(src[i] + k0);
    };
    auto sstore = [&](int buf) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) *reinterpret_cast<bf16x8*>(&S[buf][dst[i]]) = q[i];
    };
    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    gload(0);
    sstore(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < g.K; k0 += kLdsK) {
        const bool more = k0 + kLdsK < g.K;
        if (more) gload(k0 + kLdsK);
        bf16x8 a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a[i] = *reinterpret_cast<const bf16x8*>(&S[buf][(wm + 16 * i + r16) * kLdsPitch + kq]);
            b[i] = *reinterpret_cast<const bf16x8*>(&S[buf][(kLdsTile + wn + 16 * i + r16) * kLdsPitch + kq]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        if (more) sstore(buf ^ 1);  // nobody reads buf ^ 1 now: the last barrier ended its reads
        __syncthreads();
        buf ^= 1;
    }
    const int row0 = m0 + wm + 4 * (lane >> 4), col0 = n0 + wn + r16;
    EpilogueIn in[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (EPI == NFX_MLP_BWD_GELU || (i == 0 && EPI != NFX_MLP_ADAM)) {  // the biases serve all rows
#pragma unroll
            for (int j = 0; j < 4; ++j) in[j] = epilogue_in<EPI>(g, row0 + 16 * i, col0 + 16 * j);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (EPI == NFX_MLP_ADAM) in[j] = epilogue_in<EPI>(g, row0 + 16 * i, col0 + 16 * j);  // more would spill
            epilogue4<EPI>(g, row0 + 16 * i, col0 + 16 * j, acc[i][j], in[j]);
        }
    }
}

// split-K finish: one thread per four rows of a column sums the split_k workspace planes in order (four
// planes' loads in flight: a thread per entry with one load in flight 8.9 us at 8 planes of 512 x 512, now 5.8), then
// the epilogue
template <int EPI>
__global__ __launch_bounds__(256) void k_splitk_finish(nfx_mlp_gemm_args g) {
    const int64_t MN = (int64_t)g.M * g.N;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= MN / 4) return;  // M is a multiple of 128
    const int col = (int)(i % g.N), row = 4 * (int)(i / g.N);
    const float* w = g.workspace + (int64_t)row * g.N + col;
    const EpilogueIn in = epilogue_in<EPI>(g, row, col);
    f32x4 v{0.f, 0.f, 0.f, 0.f};
    int s = 0;
    for (; s + 4 <= g.split_k; s += 4) {
        f32x4 q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) q[u][r] = w[(s + u) * MN + (int64_t)r * g.N];
#pragma unroll
        for (int u = 0; u < 4; ++u) v += q[u];
    }
    for (; s < g.split_k; ++s)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] += w[s * MN + (int64_t)r * g.N];
    epilogue4<EPI>(g, row, col, v, in);
}

// loss = sum_ij w_i (Y - T)^2 / (M N) (w_i = 1 without row weights); dZ = 2 w_i (Y - T) / (M N) as
// BF16 in [M x N] and [N x M].  One workgroup per tile of kRows x 32 (M a multiple of kRows, N of 32, checked on
// the host): the tile is staged in LDS so that both the row-major and the transposed copy are written along
// contiguous rows.  The workgroups' sums meet in one FP64 atomic each, which take their turns on the one address:
// with 128 rows a quarter of them (4096 x 256: 1024 atomics 16.0 us, 256 7.7 us)
template <int kRows>
__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ Y, const float* __restrict__ Tg,
                                             const float* __restrict__ w, int32_t M, int32_t N, __bf16* dZ,
                                             __bf16* dZT, double* loss_sum) {
    __shared__ __bf16 tile[kRows][34];
    __shared__ double ws[4];
    const int nt = N / 32, r0 = (int)blockIdx.x / nt * kRows, c0 = (int)blockIdx.x % nt * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8 threads
    const float sc = 2.0f / ((float)M * (float)N);
    float y[kRows / 8], t[kRows / 8], wr[kRows / 8];
#pragma unroll
    for (int j = 0; j < kRows / 8; ++j) {
        const int row = r0 + ty + 8 * j;
        const int64_t i = (int64_t)row * N + c0 + tx;
        y[j] = Y[i];
        t[j] = Tg[i];
        wr[j] = w ? w[row] : 1.0f;
    }
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < kRows / 8; ++j) {
        const int row = ty + 8 * j;
        const float d = y[j] - t[j];
        s += (double)wr[j] * d * d;
        const __bf16 b = to_bf16(sc * wr[j] * d);
        dZ[(int64_t)(r0 + row) * N + c0 + tx] = b;
        tile[row][tx] = b;
    }
    __syncthreads();
#pragma unroll
    for (int e0 = 0; e0 < 32 * kRows; e0 += 256) {
        const int e = e0 + threadIdx.x, col = e / kRows, row = e % kRows;
        dZT[(int64_t)(c0 + col) * M + r0 + row] = tile[row][col];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(loss_sum, (ws[0] + ws[1] + ws[2] + ws[3]) / ((double)M * (double)N));
}

// bias gradient (row sums of dZ^T) and its Adam update; one workgroup per output feature.  Eight entries per
// load where the rows are 16-byte aligned (512 rows of 4096: 6.0 -> 3.4 us)
__global__ __launch_bounds__(256) void k_bias_adam(const __bf16* __restrict__ dZT, int32_t M, float* b, float* m,
                                                   float* v, float lr_t, float bc2, float beta1, float beta2,
                                                   float eps, float grad_scale) {
    const int j = blockIdx.x;
    const __bf16* z = dZT + (int64_t)j * M;
    float s = 0.f;
    if ((reinterpret_cast<uintptr_t>(dZT) & 15) == 0 && (M & 7) == 0) {
        for (int i = 8 * threadIdx.x; i < M; i += 8 * 256) {
            const bf16x8 q = *reinterpret_cast<const bf16x8*>(z + i);
#pragma unroll
            for (int e = 0; e < 8; ++e) s += (float)q[e];
        }
    } else {
        for (int i = threadIdx.x; i < M; i += 256) s += (float)z[i];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    __shared__ float ws[4];
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        const float gr = (ws[0] + ws[1] + ws[2] + ws[3]) * grad_scale;
        const float mm = beta1 * m[j] + (1.0f - beta1) * gr;
        const float vv = beta2 * v[j] + (1.0f - beta2) * gr * gr;
        m[j] = mm;
        v[j] = vv;
        b[j] -= lr_t * mm / (sqrtf(vv) * bc2 + eps);
    }
}

template <int kTM, int kTN, int kKS>
static void launch_tile(const nfx_mlp_gemm_args& g, int split, hipStream_t s) {
    const dim3 grid((unsigned int)(g.N / kTN) * (unsigned int)(g.M / kTM), 1, split);
    if (split > 1) {
        k_gemm_tile<NFX_MLP_STORE, true, kTM, kTN, kKS><<<grid, 256, 0, s>>>(g);
        return;
    }
    switch (g.epilogue) {
        case NFX_MLP_STORE: k_gemm_tile<NFX_MLP_STORE, false, kTM, kTN, kKS><<<grid, 256, 0, s>>>(g); break;
        case NFX_MLP_FWD_GELU: k_gemm_tile<NFX_MLP_FWD_GELU, false, kTM, kTN, kKS><<<grid, 256, 0, s>>>(g); break;
        case NFX_MLP_BWD_GELU: k_gemm_tile<NFX_MLP_BWD_GELU, false, kTM, kTN, kKS><<<grid, 256, 0, s>>>(g); break;
        default: k_gemm_tile<NFX_MLP_ADAM, false, kTM, kTN, kKS><<<grid, 256, 0, s>>>(g); break;
    }
}

template <int kTN>
static void launch_lds(const nfx_mlp_gemm_args& g, hipStream_t s) {
    const dim3 grid(g.N / kTN, g.M / kLdsTile);
    switch (g.epilogue) {
        case NFX_MLP_STORE: k_gemm_lds<NFX_MLP_STORE, kTN><<<grid, 2 * kTN, 0, s>>>(g); break;
        case NFX_MLP_FWD_GELU: k_gemm_lds<NFX_MLP_FWD_GELU, kTN><<<grid, 2 * kTN, 0, s>>>(g); break;
        case NFX_MLP_BWD_GELU: k_gemm_lds<NFX_MLP_BWD_GELU, kTN><<<grid, 2 * kTN, 0, s>>>(g); break;
        default: k_gemm_lds<NFX_MLP_ADAM, kTN><<<grid, 2 * kTN, 0, s>>>(g); break;
    }
}

}  // namespace nfx

using namespace nfx;

extern "C" {

int nfx_mlp_gemm(nfx_ctx* c, const nfx_mlp_gemm_args* g) {
    NFX_ON_DEVICE(c);
    NFX_REQUIRE(c && g, "NULL argument");
    NFX_REQUIRE(g->M > 0 && g->N > 0 && g->K > 0 && g->M % 128 == 0 && g->N % 32 == 0 && g->K % 32 == 0,
                "mlp gemm: M must be a multiple of 128, N and K of 32 (got %d %d %d)", g->M, g->N, g->K);
    NFX_REQUIRE(g->A && g->B && g->lda >= g->K && g->ldb >= g->K && g->lda % 8 == 0 && g->ldb % 8 == 0,
                "mlp gemm: bad operands");
    switch (g->epilogue) {
        case NFX_MLP_STORE: NFX_REQUIRE(g->C, "STORE needs C"); break;
        case NFX_MLP_FWD_GELU: NFX_REQUIRE(g->bias && g->H, "FWD_GELU needs bias and H"); break;
        case NFX_MLP_BWD_GELU: NFX_REQUIRE(g->Z && g->H && g->HT, "BWD_GELU needs Z, H and HT"); break;
        case NFX_MLP_ADAM: NFX_REQUIRE(g->C && g->H && g->HT && g->adam_m && g->adam_v, "ADAM needs C, H, HT, m, v"); break;
        default: NFX_REQUIRE(false, "unknown epilogue %d", g->epilogue);
    }
    const int S = g->split_k > 1 ? g->split_k : 1;
    NFX_REQUIRE(g->split_k >= 0 && S <= 64 && g->K % (32 * S) == 0,
                "mlp gemm: split_k %d must be at most 64 and divide K / 32 (K %d)", g->split_k, g->K);
    NFX_REQUIRE(S == 1 || g->workspace, "mlp gemm: split_k > 1 needs a workspace of split_k * M * N floats");
    // the 128 x 128 tiles where they still give a full grid (>= 256 workgroups): less is read per product, but fewer
    // workgroups hide the latency (K 512, GELU: 512 tiles 24 us against 34 with the smaller tiles, 128 tiles 22
    // against 11)
    const bool lds = S == 1 && g->M % kLdsTile == 0 && g->N % kLdsTile == 0 &&
                     (int64_t)(g->M / kLdsTile) * (g->N / kLdsTile) >= 256;
    if (lds) {
        // the wide tiles where two workgroups per CU are left (K 512, GELU, us, wide against 128 x 128: 65 536 x 512
        // 64.3 / 66.5, 32 768 x 512 35.4 / 37.0, 65 536 x 256 36.4 / 37.8; 24 576 x 512 32.9 / 30.3, 16 384 x 256 21.7 / 19.0)
        if (g->N % 256 == 0 && (int64_t)(g->M / kLdsTile) * (g->N / 256) >= 512) launch_lds<256>(*g, c->stream);
        else launch_lds<128>(*g, c->stream);
    } else {
        // k-steps of 64 where they divide a slice; a 32 x 32 tile with k-steps of 32 elsewhere
        if (g->K / S % 64 == 0) launch_tile<64, 32, 64>(*g, S, c->stream);
        else launch_tile<32, 32, 32>(*g, S, c->stream);
    }
    if (S > 1) {
        NFX_CHECK_LAUNCH();
        const unsigned int nb = (unsigned int)(((int64_t)g->M * g->N / 4 + 255) / 256);
        switch (g->epilogue) {
            case NFX_MLP_STORE: k_splitk_finish<NFX_MLP_STORE><<<nb, 256, 0, c->stream>>>(*g); break;
            case NFX_MLP_FWD_GELU: k_splitk_finish<NFX_MLP_FWD_GELU><<<nb, 256, 0, c->stream>>>(*g); break;
            case NFX_MLP_BWD_GELU: k_splitk_finish<NFX_MLP_BWD_GELU><<<nb, 256, 0, c->stream>>>(*g); break;
            default: k_splitk_finish<NFX_MLP_ADAM><<<nb, 256, 0, c->stream>>>(*g); break;
        }
    }
    NFX_CHECK_LAUNCH();
    return NFX_OK;
}

int nfx_mlp_mse(nfx_ctx* c, const float* Y, const float* target, const float* row_weight, int32_t M, int32_t N,
                void* dZ, void* dZT, double* loss_sum) {
    NFX_ON_DEVICE(c);
    NFX_REQUIRE(c && Y && target && dZ && dZT && loss_sum, "NULL argument");
    NFX_REQUIRE(M > 0 && N > 0 && M % 32 == 0 && N % 32 == 0, "mlp mse: M and N must be multiples of 32 (got %d %d)",
                M, N);
    const unsigned int tiles = (unsigned int)(N / 32) * (unsigned int)(M / 32);
    if (M % 128 == 0)
        k_mse<128><<<tiles / 4, 256, 0, c->stream>>>(Y, target, row_weight, M, N, (__bf16*)dZ, (__bf16*)dZT, loss_sum);
    else
        k_mse<32><<<tiles, 256, 0, c->stream>>>(Y, target, row_weight, M, N, (__bf16*)dZ, (__bf16*)dZT, loss_sum);
    NFX_CHECK_LAUNCH();
    return NFX_OK;
}

int nfx_mlp_bias_adam(nfx_ctx* c, const void* dZT, int32_t M, int32_t N, float* b, float* m, float* v, float lr_t,
                      float bc2, float beta1, float beta2, float eps, float grad_scale) {
    NFX_ON_DEVICE(c);
    NFX_REQUIRE(c && dZT && b && m && v && M > 0 && N > 0, "bad argument");
    k_bias_adam<<<N, 256, 0, c->stream>>>((const __bf16*)dZT, M, b, m, v, lr_t, bc2, beta1, beta2, eps, grad_scale);
    NFX_CHECK_LAUNCH();
    return NFX_OK;
}

}  // extern "C"
