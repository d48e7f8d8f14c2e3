// lx_matmul.hip -- MatMul on gfx950 (Tensor<T>.MatMul, TensorOps.cs:504-806,
// via CPUExecutionProvider.MatMul, CPUExecutionProvider.cs:359-378).
//
// float : K ranges above 512, and of 256 and more over more than 256
//         tiles of 64x64, with N above 32 (but see f32_b3): every operand in three
//         bf16 parts on v_mfma_f32_32x32x16_bf16 (k_matmul_f32_b3), closer to
//         64 bits than float32 products and 2.2 times the rate.  The others,
//         and ranges of up to 1024 of a split product:
//         v_mfma_f32_32x32x2f32 (fp32 products, fp32 accumulation), summed in
//         one order by two kernels: K a multiple of 64 with aligned operands
//         through a ring of LDS stages filled by direct-to-LDS loads
//         (k_matmul_f32_dl), otherwise double-buffered LDS fed from registers
//         one K step ahead (k_matmul_f32).  Block tiles from 64x64 to 128x128
//         chosen per shape, K step 16, four waves.  Split products of at most
//         64 rows in ranges of 64: one launch on the VALU in that order
//         (k_matmul_small).
// double: v_mfma_f64_16x16x4f64, 64x64 block tile, four waves of 32x32.
// int32 : exact two's-complement products as ten int8 digit products on
//         v_mfma_i32_32x32x32_i8 (small products of K up to 96: on the VALU).
// Batches: the leading (broadcast) axes are decomposed per block with
// per-operand element strides, 0 on broadcast axes (no materialisation).
// Layout of the MFMA operands and results checked on the device:
//   32x32x2 f32: a lane l = A[l%32][l/32], b = B[l/32][l%32],
//                acc[r] = C[8*(r/4) + 4*(l/32) + r%4][l%32]
//   16x16x4 f64: a = A[l%16][l/16], b = B[l/16][l%16], acc[r] = C[l/16 + 4r][l%16]
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "lx_device.h"
#include "lx_kernels.h"

namespace lx {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// per-block batch offsets of A, B and C
__device__ __forceinline__ void batch_offsets(int64_t b, const MatMulArgs &p, int64_t *ao, int64_t *bo,
                                              int64_t *co) {
    int64_t a = 0, bb = 0, c = 0;
    for (int d = p.nbatch - 1; d >= 0; d--) {
        const int64_t i = b % p.bdims[d];
        b /= p.bdims[d];
        a += i * p.a_bstr[d];
        bb += i * p.b_bstr[d];
        c += i * p.c_bstr[d];
    }
    *ao = a;
    *bo = bb;
    *co = c;
}

// ---------------------------------------------------------------------------
// float: MFMA 32x32x2
// ---------------------------------------------------------------------------

// Bias / residual / GELU epilogue and store of a wave's MT x NT tiles of 32x32 results (rows r0.., columns
// c0..) into the batch's C at offset co.  The MFMA ran as B^T A^T, so acc[i][j][q] = C[r0 + 32 i + l % 32][c0 +
// 32 j + 8 (q / 4) + 4 (l / 32) + q % 4]: each lane holds four consecutive columns of one row per group of four
// results (one 16-byte store).  The residual and the bias rows are dense.
template <int MT, int NT, bool VEC, bool GELU>
__device__ __forceinline__ void mm_epilogue(const v16f (&acc)[MT][NT], float *__restrict__ C, const MatMulArgs &p,
                                            int64_t co, int r0, int c0, int l, const ExpTable &tab) {
    const int M = p.m, N = p.n;
    const int64_t bz = p.batch_base + blockIdx.z;
    float *Cb = C + co;
    const float *Rb = p.res ? p.res + bz * (int64_t)M * N : nullptr;
    const float *Bias = p.bias ? p.bias + bz * p.bias_bstr : nullptr;
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int row = r0 + 32 * i + (l % 32);
        if (row >= M) continue;
        float *Cr = Cb + (int64_t)row * p.ldc;
        const float *Rr = Rb ? Rb + (int64_t)row * N : nullptr;
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int c = c0 + 32 * j + 8 * q + 4 * (l / 32);
                float v[4] = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
                if (VEC && c + 3 < N) {
                    if (Bias) {
                        const float4 bc = *reinterpret_cast<const float4 *>(Bias + c);
                        v[0] = v[0] + bc.x; v[1] = v[1] + bc.y; v[2] = v[2] + bc.z; v[3] = v[3] + bc.w;
                    }
                    if (Rr) {
                        const float4 rc = *reinterpret_cast<const float4 *>(Rr + c);
                        v[0] = v[0] + rc.x; v[1] = v[1] + rc.y; v[2] = v[2] + rc.z; v[3] = v[3] + rc.w;
                    }
                    if constexpr (GELU) {
#pragma unroll
                        for (int e = 0; e < 4; e++) v[e] = gelu_erf_lx(v[e], tab);
                    }
                    *reinterpret_cast<float4 *>(Cr + c) = make_float4(v[0], v[1], v[2], v[3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        if (c + e >= N) break;
                        float x = v[e];
                        if (Bias) x = x + Bias[c + e];
                        if (Rr) x = x + Rr[c + e];
                        if constexpr (GELU) x = gelu_erf_lx(x, tab);
                        Cr[c + e] = x;
                    }
                }
            }
    }
}

// Store of a wave's raw accumulators (no epilogue) into the partial product P (a dense M x N matrix, N a multiple
// of 4), in mm_epilogue's layout.
template <int MT, int NT>
__device__ __forceinline__ void mm_store_part(const v16f (&acc)[MT][NT], float *__restrict__ P, int M, int N, int r0,
                                              int c0, int l) {
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int row = r0 + 32 * i + (l % 32);
        if (row >= M) continue;
        float *Pr = P + (int64_t)row * N;
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int c = c0 + 32 * j + 8 * q + 4 * (l / 32);
                if (c < N)
                    *reinterpret_cast<v4f *>(Pr + c) =
                        v4f{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
            }
    }
}

// C = epilogue(P[0] + P[1] + ... + P[split - 1]) over the split partial products of a launch's batches, summed in
// that order, then the bias, residual and GELU of mm_epilogue, each rounded as there: 16 bytes per lane.
template <bool GELU>
__global__ __launch_bounds__(256) void k_matmul_split_sum(float *__restrict__ C, MatMulArgs p) {
    __shared__ ExpTable tab;
    if constexpr (GELU) {
        exp_table_fill(tab);
        __syncthreads();
    }
    const int64_t mn = (int64_t)p.m * p.n, nq = mn / 4;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nq * p.batch) return;
    const int64_t zb = i / nq, e = (i - zb * nq) * 4;  // batch of this launch, element of its matrix
    const int64_t stride = p.batch * mn;                // between the partials of two K ranges
    const float *P = p.part + zb * mn + e;
    // the bias and residual loaded with the partials, one memory latency for all (added after them, as before)
    const int64_t bz = p.batch_base + zb;
    const float4 bc = p.bias ? *reinterpret_cast<const float4 *>(p.bias + bz * p.bias_bstr + e % p.n)
                             : make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 rc = p.res ? *reinterpret_cast<const float4 *>(p.res + bz * mn + e) : make_float4(0.f, 0.f, 0.f, 0.f);
    // the partials eight at a time, all eight loads in flight before the first add (one memory latency per
    // eight, not one per partial); the adds in range order
    constexpr int kChunk = 8;
    v4f v = *reinterpret_cast<const v4f *>(P);
    for (int s0 = 1; s0 < p.split; s0 += kChunk) {
        v4f x[kChunk];
#pragma unroll
        for (int c = 0; c < kChunk; c++)
            if (s0 + c < p.split) x[c] = *reinterpret_cast<const v4f *>(P + (s0 + c) * stride);
#pragma unroll
        for (int c = 0; c < kChunk; c++)
            if (s0 + c < p.split) {
                v[0] = v[0] + x[c][0]; v[1] = v[1] + x[c][1]; v[2] = v[2] + x[c][2]; v[3] = v[3] + x[c][3];
            }
    }
    if (p.bias) {
        v[0] = v[0] + bc.x; v[1] = v[1] + bc.y; v[2] = v[2] + bc.z; v[3] = v[3] + bc.w;
    }
    if (p.res) {
        v[0] = v[0] + rc.x; v[1] = v[1] + rc.y; v[2] = v[2] + rc.z; v[3] = v[3] + rc.w;
    }
    if constexpr (GELU) {
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = gelu_erf_lx(v[k], tab);
    }
    int64_t ao, bo, co;
    batch_offsets(bz, p, &ao, &bo, &co);
    const int64_t row = e / p.n;
    *reinterpret_cast<float4 *>(C + co + row * p.ldc + (e - row * p.n)) = make_float4(v[0], v[1], v[2], v[3]);
}

// k_matmul_split_sum for a product whose rows are then normalised (the decomposed LayerNorm after a projection and
// its residual): one wave per row, lane l holding the vectors c * 64 + l as k_layernorm does; each element summed
// over the partials in range order with the bias and residual exactly as in k_matmul_split_sum, then the row
// normalised by ln_row_finish into y (dense, the product's shape).  Bit for bit k_matmul_split_sum followed by
// k_layernorm, without the product's round trip through memory.
template <int NV>
__global__ __launch_bounds__(64) void k_matmul_split_sum_ln(const float *__restrict__ gamma, const float *__restrict__ beta,
                                                             float eps, float *__restrict__ y, MatMulArgs p) {
    const int lane = threadIdx.x;
    const int64_t rg = blockIdx.x, zb = rg / p.m, row = rg - zb * p.m;  // row of the launch's batch zb
    const int N = p.n;
    const int64_t mn = (int64_t)p.m * N, stride = p.batch * mn, bz = p.batch_base + zb;
    constexpr int kChunk = 8;
    // the bias, residual, gamma and beta vectors loaded with the partials, one memory latency for all
    Vec<float, 4> v[NV], gv[NV], bv[NV];
    float4 bcv[NV], rcv[NV];
#pragma unroll
    for (int c = 0; c < NV; c++) {
        const int col = (c * 64 + lane) * 4;
        if (col >= N) continue;
        gv[c] = vload<float, 4>(gamma + col);
        bv[c] = vload<float, 4>(beta + col);
        if (p.bias) bcv[c] = *reinterpret_cast<const float4 *>(p.bias + bz * p.bias_bstr + col);
        if (p.res) rcv[c] = *reinterpret_cast<const float4 *>(p.res + bz * mn + row * N + col);
    }
#pragma unroll
    for (int c = 0; c < NV; c++) {
        const int col = (c * 64 + lane) * 4;
        v[c] = Vec<float, 4>{{0.0f, 0.0f, 0.0f, 0.0f}};
        if (col >= N) continue;
        const float *P = p.part + zb * mn + row * N + col;
        v4f a = *reinterpret_cast<const v4f *>(P);
        for (int s0 = 1; s0 < p.split; s0 += kChunk) {
            v4f x[kChunk];
#pragma unroll
            for (int q = 0; q < kChunk; q++)
                if (s0 + q < p.split) x[q] = *reinterpret_cast<const v4f *>(P + (s0 + q) * stride);
#pragma unroll
            for (int q = 0; q < kChunk; q++)
                if (s0 + q < p.split) {
                    a[0] = a[0] + x[q][0]; a[1] = a[1] + x[q][1]; a[2] = a[2] + x[q][2]; a[3] = a[3] + x[q][3];
                }
        }
        if (p.bias) {
            const float4 bc = bcv[c];
            a[0] = a[0] + bc.x; a[1] = a[1] + bc.y; a[2] = a[2] + bc.z; a[3] = a[3] + bc.w;
        }
        if (p.res) {
            const float4 rc = rcv[c];
            a[0] = a[0] + rc.x; a[1] = a[1] + rc.y; a[2] = a[2] + rc.z; a[3] = a[3] + rc.w;
        }
        v[c] = Vec<float, 4>{{a[0], a[1], a[2], a[3]}};
    }
    ln_row_finish<NV>(v, N, lane, gamma, beta, eps, y + bz * mn + row * N, gv, bv);
}

// BM x BN block tile, four waves in a WM x WN grid, each wave (BM/WM) x (BN/WN)
// = MT x NT MFMA tiles of 32x32.  K steps of 16, double-buffered in LDS with k
// as the outer index (A transposed to [k][m], B as [k][n]), so the lanes of a
// fragment read 32 consecutive floats.  The kernel for K not a multiple of 64,
// unaligned operands, K <= 64, N <= 64 and 128x96 tiles beyond one per CU.
constexpr int kFBK = 16, kFPad = 4;

// BT: B stored by columns (element (k, n) at n * ldb + k: a transposed view), loaded as A is, along K, and
// written into the same LDS layout, so the MFMAs and their sums are those of a row-major B.
template <int BM, int BN, int WM, int WN, bool VEC, bool GELU, bool BT = false>
__global__ __launch_bounds__(WM * WN * 64) void k_matmul_f32(const float *__restrict__ A, const float *__restrict__ B,
                                                             float *__restrict__ C, MatMulArgs p) {
    constexpr int NTHR = WM * WN * 64;               // threads of the block
    constexpr int WTM = BM / WM, WTN = BN / WN;      // wave tile
    constexpr int MT = WTM / 32, NT = WTN / 32;      // MFMA tiles per wave
    static_assert((WM * WN == 4 || WM * WN == 8) && MT * 32 == WTM && NT * 32 == WTN, "waves of whole 32x32 tiles");
    constexpr int AV = BM * kFBK / 4, BV = BN * kFBK / 4;  // float4 of A and of B per K step
    constexpr int LA = (AV + NTHR - 1) / NTHR, LB = (BV + NTHR - 1) / NTHR;
    constexpr int BQ = BN / 4;                       // float4 per B row
    __shared__ float As[2][kFBK][BM + kFPad];
    __shared__ float Bs[2][kFBK][BN + kFPad];
    __shared__ ExpTable tab;  // the GELU epilogue's exponential (filled before the first barrier)
    if constexpr (GELU) exp_table_fill(tab);
    const int M = p.m, N = p.n, K = p.k;
    const int t = threadIdx.x, l = t & 63, w = t >> 6;
    const int row0 = blockIdx.y * BM, col0 = blockIdx.x * BN;
    int64_t ao, bo, co;
    batch_offsets(p.batch_base + blockIdx.z, p, &ao, &bo, &co);
    const float *Ab = A + ao;
    const float *Bb = B + bo;
    const int64_t lda = p.lda, ldb = p.ldb;

    // global -> register staging one K step ahead: float4 e = t + NTHR h of the step's
    // A tile (row e / KQ, k 4 (e % KQ)) and B tile (k row e / BQ, column 4 (e % BQ))
    constexpr int KQ = kFBK / 4;                     // float4 per A row of a K step
    float4 ra[LA], rb[LB];
    auto load = [&](int k0) {
#pragma unroll
        for (int h = 0; h < LA; h++) {
            const int e = t + NTHR * h;
            if (AV % NTHR != 0 && e >= AV) continue;
            const int r = row0 + e / KQ, kk = k0 + (e % KQ) * 4;
            if constexpr (VEC) {
                ra[h] = (r < M && kk < K) ? *reinterpret_cast<const float4 *>(Ab + (int64_t)r * lda + kk)
                                          : make_float4(0.f, 0.f, 0.f, 0.f);
            } else {
                float v[4];
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = (r < M && kk + q < K) ? Ab[(int64_t)r * lda + kk + q] : 0.f;
                ra[h] = make_float4(v[0], v[1], v[2], v[3]);
            }
        }
#pragma unroll
        for (int h = 0; h < LB; h++) {
            const int e = t + NTHR * h;
            if (BV % NTHR != 0 && e >= BV) continue;
            if constexpr (BT) {  // column col0 + e / KQ, k 4 (e % KQ) of the step
                const int c = col0 + e / KQ, kk = k0 + (e % KQ) * 4;
                if constexpr (VEC) {
                    rb[h] = (c < N && kk < K) ? *reinterpret_cast<const float4 *>(Bb + (int64_t)c * ldb + kk)
                                              : make_float4(0.f, 0.f, 0.f, 0.f);
                } else {
                    float v[4];
#pragma unroll
                    for (int q = 0; q < 4; q++) v[q] = (c < N && kk + q < K) ? Bb[(int64_t)c * ldb + kk + q] : 0.f;
                    rb[h] = make_float4(v[0], v[1], v[2], v[3]);
                }
                continue;
            }
            const int kb = k0 + e / BQ, c = col0 + (e % BQ) * 4;
            if constexpr (VEC) {
                rb[h] = (kb < K && c < N) ? *reinterpret_cast<const float4 *>(Bb + (int64_t)kb * ldb + c)
                                          : make_float4(0.f, 0.f, 0.f, 0.f);
            } else {
                float v[4];
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = (kb < K && c + q < N) ? Bb[(int64_t)kb * ldb + c + q] : 0.f;
                rb[h] = make_float4(v[0], v[1], v[2], v[3]);
            }
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int h = 0; h < LA; h++) {
            const int e = t + NTHR * h;
            if (AV % NTHR != 0 && e >= AV) continue;
            const int r = e / KQ, kk = (e % KQ) * 4;
            As[buf][kk + 0][r] = ra[h].x;
            As[buf][kk + 1][r] = ra[h].y;
            As[buf][kk + 2][r] = ra[h].z;
            As[buf][kk + 3][r] = ra[h].w;
        }
#pragma unroll
        for (int h = 0; h < LB; h++) {
            const int e = t + NTHR * h;
            if (BV % NTHR != 0 && e >= BV) continue;
            if constexpr (BT) {
                const int c = e / KQ, kk = (e % KQ) * 4;
                Bs[buf][kk + 0][c] = rb[h].x;
                Bs[buf][kk + 1][c] = rb[h].y;
                Bs[buf][kk + 2][c] = rb[h].z;
                Bs[buf][kk + 3][c] = rb[h].w;
            } else {
                *reinterpret_cast<float4 *>(&Bs[buf][e / BQ][(e % BQ) * 4]) = rb[h];
            }
        }
    };

    const int wr = (w / WN) * WTM, wc = (w % WN) * WTN;  // this wave's sub-tile
    v16f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    const int nk = (K + kFBK - 1) / kFBK;
    load(0);
    store(0);
    __syncthreads();
    int buf = 0;
    for (int kt = 0; kt < nk; kt++) {
        if (kt + 1 < nk) load((kt + 1) * kFBK);
        // MFMA j of the step takes k = j from lanes 0-31 and k = 8 + j from lanes 32-63, the order of the
        // direct-load kernel below: every float MatMul sums its products in one order, whichever kernel runs it
#pragma unroll
        for (int j = 0; j < kFBK / 2; j++) {
            const int kr = 8 * (l / 32) + j;
            float a[MT], b[NT];
#pragma unroll
            for (int i = 0; i < MT; i++) a[i] = As[buf][kr][wr + 32 * i + (l % 32)];
#pragma unroll
            for (int jn = 0; jn < NT; jn++) b[jn] = Bs[buf][kr][wc + 32 * jn + (l % 32)];
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int jn = 0; jn < NT; jn++)
                    acc[i][jn] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[jn], a[i], acc[i][jn], 0, 0, 0);
        }
        if (kt + 1 < nk) store(buf ^ 1);
        __syncthreads();
        buf ^= 1;
    }
    mm_epilogue<MT, NT, VEC, GELU>(acc, C, p, co, row0 + wr, col0 + wc, l, tab);
}

// Direct-to-LDS pipeline for K a multiple of 64 and 16-byte aligned operands.  Each K step of 16 is one stage of a
// four-stage ring in LDS, filled by global_load_lds_dwordx4 (16 bytes per lane straight into LDS, no register
// staging) three steps ahead of the MFMAs, with one barrier per step; each wave reads its fragments of a stage one
// step before it multiplies them.  Stage layout:
//   A: BM rows of the step's 16 floats (four 16-byte chunks per row, chunk c of row r at slot c ^ swz(r));
//   B: the step's rows 0-7, then 128 bytes on, rows 8-15, each row BN floats.
// The K order within a step is permuted: MFMA j (j = 0..7) takes k = j from lanes 0-31 and k = 8 + j from lanes
// 32-63, so a lane's A operands for the whole step are eight consecutive floats of its row (two 16-byte reads).
// Rows past M and columns past N read a clamped in-range address (their results are not stored).
__device__ __forceinline__ int dl_swz(int r) { return ((r >> 1) ^ (r >> 3)) & 3; }

// global_load_lds_dwordx4: the lane's 16 bytes at g land in LDS at lds + 16 * lane (lds uniform over the wave).
// Written as inline asm so that the compiler does not track these LDS writes: it would otherwise wait for every
// outstanding direct load before LDS reads of the other stages.  The kernel orders them itself: a stage is read
// only after an s_waitcnt vmcnt that covers its loads and a barrier.  (Loads the compiler does not count only
// make its own vmcnt waits longer.)  The LDS address goes in M0 (set by the compiler, an operand of the asm),
// which takes one wait state before the load.
__device__ __forceinline__ void load_to_lds16(const float *g, char *lds) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint32_t m0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)lds;
    __asm__ volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"{m0}"(m0), "v"(g) : "memory");
#else
    (void)g;
    (void)lds;
#endif
}
// no instruction is scheduled across this point
__device__ __forceinline__ void sched_fence() {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_sched_barrier(0);
#endif
}

// f(integral_constant<int, i>) for i = R0 .. R1 - 1, in order
template <int R0, typename F, int... Is>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, R0 + Is>()), ...);
}
template <int R0, int R1, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (R1 > R0) static_for_impl<R0>(f, std::make_integer_sequence<int, R1 - R0>());
}

// s_waitcnt vmcnt(n) lgkmcnt(0), then s_barrier: this wave's direct loads but the last n have landed and its LDS
// reads are done before any wave passes.  (A __syncthreads would wait for every outstanding direct load.)
template <int N>
__device__ __forceinline__ void wait_vmcnt_barrier() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
#if defined(__HIP_DEVICE_COMPILE__)
    __asm__ volatile("s_barrier" ::: "memory");
#endif
}

// SPLIT: block z = batch * p.split + r computes the partial product of the r-th of p.split equal K ranges (whole
// passes of four steps) into p.part, without the epilogue (k_matmul_split_sum applies it).
template <int BM, int BN, int WM, int WN, int S, int WMIN, int WMAX, bool GELU, bool SPLIT = false>
__global__ __launch_bounds__(WM * WN * 64) __attribute__((amdgpu_waves_per_eu(WMIN, WMAX))) void k_matmul_f32_dl(const float *__restrict__ A, const float *__restrict__ B,
                                                                float *__restrict__ C, MatMulArgs p) {
    constexpr int NW = WM * WN;
    constexpr int WTM = BM / WM, WTN = BN / WN, MT = WTM / 32, NT = WTN / 32;
    static_assert(MT * 32 == WTM && NT * 32 == WTN && S >= 2 && S <= 4, "waves of whole 32x32 tiles");
    constexpr int A_BYTES = BM * 64, B_HALF = BN * 32, B_HI = A_BYTES + B_HALF + 128;
    constexpr int STAGE = A_BYTES + 2 * B_HALF + 128;
    static_assert(A_BYTES % 1024 == 0 && B_HALF % 1024 == 0, "whole wave loads");
    constexpr int LA = A_BYTES / 1024, LBH = B_HALF / 1024, NL = LA + 2 * LBH;
    constexpr int L = (NL + NW - 1) / NW;  // wave loads per wave per stage (the last one repeated when uneven)
    // one LDS variable per stage: the compiler then knows that the reads of one stage do not wait for the
    // direct loads still landing in the others
    __shared__ __attribute__((aligned(1024))) char sm0[STAGE];
    __shared__ __attribute__((aligned(1024))) char sm1[STAGE];
    __shared__ __attribute__((aligned(1024))) char sm2[STAGE];
    __shared__ __attribute__((aligned(1024))) char sm3[STAGE];
    auto stage_mem = [&](auto sidx) -> char * {
        constexpr int sx = decltype(sidx)::value;
        if constexpr (sx == 0) return sm0;
        else if constexpr (sx == 1) return sm1;
        else if constexpr (sx == 2) return sm2;
        else return sm3;
    };
    __shared__ ExpTable tab;
    if constexpr (GELU) exp_table_fill(tab);
    const int M = p.m, N = p.n, K = p.k;
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = blockIdx.y * BM, col0 = blockIdx.x * BN;
    // the batch of this launch and, split, the K range: steps [k0, k0 + nk) of 16
    const int zb = SPLIT ? (int)blockIdx.z / p.split : (int)blockIdx.z;
    const int nk = SPLIT ? K / 16 / p.split : K / 16;
    const int k0 = SPLIT ? ((int)blockIdx.z - zb * p.split) * nk * 16 : 0;
    int64_t ao, bo, co;
    batch_offsets(p.batch_base + zb, p, &ao, &bo, &co);

    // this wave's loads: a per-lane source address (advanced by `inc` floats per step) and an LDS offset
    const float *src[L];
    int64_t inc[L];
    int dst[L];
#pragma unroll
    for (int j = 0; j < L; j++) {
        const int i = min(w + NW * j, NL - 1);
        if (i < LA) {
            const int q = 64 * i + l, r = q >> 2, c = (q & 3) ^ dl_swz(r);
            src[j] = A + ao + (int64_t)min(row0 + r, M - 1) * p.lda + k0 + 4 * c;
            inc[j] = 16;
            dst[j] = 1024 * i;
        } else {
            const int h = (i - LA) / LBH, wl = (i - LA) % LBH, q = 64 * wl + l;
            const int k = 8 * h + q / (BN / 4), c = col0 + 4 * (q % (BN / 4));
            src[j] = B + bo + (int64_t)(k0 + k) * p.ldb + min(c, N - 4);
            inc[j] = 16 * p.ldb;
            dst[j] = A_BYTES + h * (B_HALF + 128) + 1024 * wl;
        }
    }
    auto issue = [&](auto sidx, int kt) {
        char *base = stage_mem(sidx);
#pragma unroll
        for (int j = 0; j < L; j++)
            load_to_lds16(src[j] + kt * inc[j], base + dst[j]);
    };

    // fragment offsets within a stage
    const int wr = (w / WN) * WTM, wc = (w % WN) * WTN, h = l / 32;
    int aoff[MT][2], boff[NT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int r = wr + 32 * i + (l % 32);
#pragma unroll
        for (int e = 0; e < 2; e++) aoff[i][e] = r * 64 + 16 * ((2 * h + e) ^ dl_swz(r));
    }
#pragma unroll
    for (int j = 0; j < NT; j++) boff[j] = (h ? B_HI : A_BYTES) + 4 * (wc + 32 * j + (l % 32));

    v16f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    // Step t: wait for this wave's loads of step t + 1 (the S - 3 later steps' loads stay outstanding); barrier
    // (every wave's loads of step t + 1 are visible, and stage (t - 1) % S, read during step t - 2, is free);
    // issue step t + S - 1 into that stage; read step t + 1's fragments; run step t's MFMAs on the fragments read
    // during step t - 1.  No read latency lies between the barrier and the first MFMA.  The LDS reads are
    // ordinary loads, waited for by the compiler; the direct loads are invisible to it (load_to_lds16).
    // two fragment sets, the current step's and the next's, swapping roles from step to step (no copies)
    v4f af0[MT][2], af1[MT][2];
    float bf0[NT][8], bf1[NT][8];
    auto read_all = [&](auto sidx, v4f (&ra)[MT][2], float (&rb)[NT][8]) {
        const char *stg = stage_mem(sidx);
#pragma unroll
        for (int i = 0; i < MT; i++) {
            ra[i][0] = *reinterpret_cast<const v4f *>(stg + aoff[i][0]);
            ra[i][1] = *reinterpret_cast<const v4f *>(stg + aoff[i][1]);
        }
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int kk = 0; kk < 8; kk++) rb[j][kk] = *reinterpret_cast<const float *>(stg + boff[j] + kk * BN * 4);
    };
    auto step = [&](auto sidx, int t, const v4f (&caf)[MT][2], const float (&cbf)[NT][8], v4f (&naf)[MT][2],
                    float (&nbf)[NT][8]) {
        constexpr int sx = decltype(sidx)::value;
        wait_vmcnt_barrier<(S - 3) * L>();
        // the MFMAs of k pair kk, then a slice of the next stage's fragment reads (the direct loads after the first
        // pair): the reads' latency hides under the MFMAs that follow, and the fences keep this order
        const char *nst = stage_mem(std::integral_constant<int, (sx + 1) % S>());
        constexpr int R = 2 * MT + 8 * NT;  // fragment reads per stage
        auto read_one = [&](auto rc) {
            constexpr int r = decltype(rc)::value;
            if constexpr (r < 2 * MT) {
                naf[r / 2][r % 2] = *reinterpret_cast<const v4f *>(nst + aoff[r / 2][r % 2]);
            } else {
                constexpr int j = (r - 2 * MT) / 8, kk = (r - 2 * MT) % 8;
                nbf[j][kk] = *reinterpret_cast<const float *>(nst + boff[j] + kk * BN * 4);
            }
        };
        static_for<0, 8>([&](auto kc) {
            constexpr int kk = decltype(kc)::value;
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(cbf[j][kk], caf[i][kk / 4][kk % 4], acc[i][j], 0, 0, 0);
            sched_fence();
            if constexpr (kk == 0) {
                // past the last step the ring re-loads step nk - 1 into a stage no later step reads: every
                // step then issues the same loads, and the wait above is the same count everywhere
                issue(std::integral_constant<int, (sx + S - 1) % S>(), min(t + S - 1, nk - 1));
            } else if constexpr (kk <= 6) {
                static_for<(kk - 1) * R / 6, kk * R / 6>(read_one);
            }
            sched_fence();
        });
    };
    issue(std::integral_constant<int, 0>(), 0);
    issue(std::integral_constant<int, 1>(), min(1, nk - 1));
    issue(std::integral_constant<int, 2>(), min(2, nk - 1));
    static_assert(S == 4, "fragments a step ahead need the loads two steps ahead; four steps per loop pass");
    wait_vmcnt_barrier<(S - 2) * L>();
    read_all(std::integral_constant<int, 0>(), af0, bf0);
    // K is a multiple of 64: whole passes of four steps, each fragment set in the same registers on every pass
    for (int t = 0; t < nk; t += S) {
        step(std::integral_constant<int, 0>(), t, af0, bf0, af1, bf1);
        step(std::integral_constant<int, 1>(), t + 1, af1, bf1, af0, bf0);
        step(std::integral_constant<int, 2>(), t + 2, af0, bf0, af1, bf1);
        step(std::integral_constant<int, 3>(), t + 3, af1, bf1, af0, bf0);
    }
    // the ring's last loads land before the wave can end (the block's LDS is then handed to another block)
    __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));
    if constexpr (SPLIT)
        mm_store_part<MT, NT>(acc, p.part + ((int64_t)(blockIdx.z - zb * p.split) * p.batch + zb) * M * N, M, N,
                              row0 + wr, col0 + wc, l);
    else
        mm_epilogue<MT, NT, true, GELU>(acc, C, p, co, row0 + wr, col0 + wc, l, tab);
}

template <int BM, int BN, int WM, int WN, int WMIN, int WMAX>
static void launch_f32_dl(const float *a, const float *b, float *c, const MatMulArgs &p, hipStream_t s) {
    dim3 g((p.n + BN - 1) / BN, (p.m + BM - 1) / BM, (unsigned)p.batch);
    const dim3 blk(WM * WN * 64);
    if (p.gelu) hipLaunchKernelGGL((k_matmul_f32_dl<BM, BN, WM, WN, 4, WMIN, WMAX, true>), g, blk, 0, s, a, b, c, p);
    else hipLaunchKernelGGL((k_matmul_f32_dl<BM, BN, WM, WN, 4, WMIN, WMAX, false>), g, blk, 0, s, a, b, c, p);
}

// ---------------------------------------------------------------------------
// float, K ranges of 256 or more: every operand in three bf16 parts on the bf16 matrix unit
// ---------------------------------------------------------------------------
// x = p1 + p2 + p3 with p1 = bf16(x), p2 = bf16(x - p1), p3 = bf16(x - p1 - p2): three 8-bit significands hold all 24
// bits of a float32, so the parts of a value of 2^-109 or more are exact.  A product is the six part products of
// weight 2^-16 or more,
//   (a3 b1 + a1 b3 + a2 b2 + a2 b1 + a1 b2) + a1 b1
// (the three left out weigh 2^-25 |a b| at most), each exact in the MFMA and accumulated in float32: per step of 16
// six v_mfma_f32_32x32x16_bf16 of 32 cycles, where v_mfma_f32_32x32x2f32 takes eight of 64.  The five small ones have
// an accumulator of their own, added to the sum of the a1 b1 at the end: those have 16 significant bits, so that sum
// hardly rounds, and the others round at 2^-8 of its size.  In one accumulator every MFMA rounded at full size, up to
// twice as far off as a float32 chain where operands hold zeros (the chain does not round on a zero).  Relative error
// against 64 bits, the fp32 MFMA's in brackets: normal data K 384 1.1e-7 (3.5e-7), 768 1.6e-7 (5.0e-7), 3072 3.4e-7
// (9.9e-7); left operand 10% dense 4.6e-8 (1.1e-7), 6.1e-8 (1.6e-7), 1.2e-7 (3.2e-7), 2% dense 3.0e-8 (5.5e-8), 3.4e-8
// (7.5e-8), 5.7e-8 (1.4e-7).  Only rows of a single nonzero product are off a little more, 2.60e-8 (2.53e-8, the
// correctly rounded product), by the part products left out (none where one factor has 8 bits or fewer: a selection).
// Shorter ranges stay on the fp32 MFMA: they are bound by launches and loads ([667,384]x[384,384] in ranges of
// 128 ran slower in parts).  f32_b3 chooses by the K range, N, the row strides and f32_tiles, none of which depends on the
// block tile or on what is fused or folded: an unsplit product is the same bits in all of these forms.
//
// What the parts cannot hold goes to the fp32 MFMA, element by element: a result that is not finite (a value that is
// not, or rounds to an infinite bf16); a result smaller than 2^-96 of its column's largest operand where its row holds
// a nonzero value below 2^-109 (parts below 2^-133 are lost: 2^-134 of the operand per product), and the other way
// round; and a result below 2^-120 that is not zero or has no product of 2^-120 in its row and column (the small part
// products are lost below float32's range).  Each thread keeps the largest magnitude it loaded of its row and column
// and the smallest but zero; a wave holding such a result runs that 32x32 tile again from global memory (f32_tile) and
// takes those elements from it.  A zero or small result alone says nothing: products of integers, of sparse operands
// or of values of 1e-24 take the time of any others ([4096,768]x[768,768] of values -8..8 ran 186 us when every zero
// ran again, 33 now; the smallest magnitudes cost normal data 1 to 3%).
//
// Bound: the matrix unit (register-only, 340 TFLOP/s of float32 products at the clock it holds), then the issue slots
// of the splitting (15 VALU instructions per pair of elements) and of LDS, so each element is split once per block,
// on its way from global memory to LDS, and the splitting, the LDS accesses and the loads are dealt out between the
// MFMAs one by one (in runs they stalled the wave's MFMAs: [4096,3072]x[3072,768] 208 us with the phases one after
// another, 130 with fragments a step ahead, 112 dealt out evenly with eight waves; 118 since the small products have their
// own accumulator).  Stage layout: per 16-k sub-step
// and part, [k half][row] chunks of eight bf16, the halves 64 bytes apart modulo 256: the 16-byte fragment reads and
// the writes are free of bank conflicts.  Two stages: step t multiplies the fragments read during step t - 1, reads
// those of step t + 1, writes the parts of step t + 2 into the stage they left and loads step t + 4.
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t bf16_pair(float x0, float x1) {
    const v2f x = {x0, x1};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, v2bf));
}

// one 32x32 tile of the product over k in [k0, k1), rows row0.. and columns col0.. (clamped to M, N), straight from
// global memory on the fp32 MFMA in the fp32 kernels' order
template <bool BT>
__device__ __noinline__ v16f f32_tile(const float *A, const float *B, int M, int N, int64_t lda, int64_t ldb, int row0,
                                      int col0, int k0, int k1, int l) {
    const int h = l / 32;
    const float *ar = A + (int64_t)min(row0 + l % 32, M - 1) * lda;
    const int64_t col = min(col0 + l % 32, N - 1);
    v16f acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.f;
    for (int k = k0; k < k1; k += 16) {
        float a[8], b[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int kk = k + 8 * h + j;
            a[j] = kk < k1 ? ar[kk] : 0.f;
            b[j] = kk < k1 ? (BT ? B[col * ldb + kk] : B[(int64_t)kk * ldb + col]) : 0.f;
        }
#pragma unroll
        for (int j = 0; j < 8; j++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(b[j], a[j], acc, 0, 0, 0);
    }
    return acc;
}

// BM x BN tile, WM x WN multiplying waves, KS sub-steps of 16 per step, WE waves per SIMD.  PW: loading waves that
// load and split for them (0: every wave does both).  A block alone on its CU is bound by its waves' issue slots, not
// by the matrix unit: eight loading waves beside the four of a 64x64 tile take [788,3072]x[3072,768] (156 tiles) from
// 58 to 45 us; with 128x128 tiles both forms run alike ([4096,3072]x[3072,768] 118 in eight joint waves, 118 to 126 with
// eight or four loading ones).  VEC: 16-byte loads along K (the rows
// of A, and of B by columns, 16-byte aligned).  TAIL: the K range is no whole number of step pairs (past it the loads
// clamp to the last step's and their elements are zeroed).  vc: 16-byte epilogue.  SPLIT as in k_matmul_f32_dl.
template <int BM, int BN, int WM, int WN, int PW, int KS, int WE, bool VEC, bool TAIL, bool BT, bool GELU,
          bool SPLIT = false>
__global__ __launch_bounds__((WM * WN + PW) * 64) __attribute__((amdgpu_waves_per_eu(WE, WE))) void k_matmul_f32_b3(
    const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C, MatMulArgs p, int vc) {
    constexpr int NW = WM * WN, NTHR = (PW ? PW : NW) * 64, KB = 16 * KS;  // NTHR: the threads that load and split
    constexpr int MT = BM / WM / 32, NT = BN / WN / 32;
    static_assert(MT * WM * 32 == BM && NT * WN * 32 == BN, "waves of whole 32x32 tiles");
    constexpr int AH = BM * 16 + 64, BH = BN * 16 + 64;         // bytes of a k half of one part (64: the bank offset)
    constexpr int AP = 2 * AH, BP = 2 * BH, SUB = 3 * (AP + BP), STAGE = SUB * KS;
    constexpr int CA = BM * KB / NTHR >= 8 ? 8 : 4, NA = BM * KB / CA / NTHR;  // floats per chunk, chunks per thread
    constexpr int CB = BN * KB / NTHR >= 8 ? 8 : 4, NB = BN * KB / CB / NTHR;
    static_assert(NA * CA * NTHR == BM * KB && NB * CB * NTHR == BN * KB, "whole chunks");
    __shared__ __attribute__((aligned(1024))) char sm[2][STAGE];
    // of each row and column: the bits of its largest magnitude, and of its smallest but zero as (bits << 1) - 1
    __shared__ uint32_t amax[BM], bmax[BN], amin[BM], bmin[BN];
    __shared__ ExpTable tab;
    if constexpr (GELU) exp_table_fill(tab);
    const int M = p.m, N = p.n;
    const int l = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = (int)threadIdx.x - (PW ? NW * 64 : 0);  // index among the threads that load and split
    const int row0 = blockIdx.y * BM, col0 = blockIdx.x * BN;
    const int zb = SPLIT ? (int)blockIdx.z / p.split : (int)blockIdx.z;
    const int kr = SPLIT ? p.k / p.split : p.k;                       // length of the K range
    const int kbeg = SPLIT ? ((int)blockIdx.z - zb * p.split) * kr : 0;
    const int nk = 2 * ((kr + 2 * KB - 1) / (2 * KB));                // steps, in pairs
    int64_t ao, bo, co;
    batch_offsets(p.batch_base + zb, p, &ao, &bo, &co);
    for (int i = threadIdx.x; i < BM; i += blockDim.x) amax[i] = 0, amin[i] = ~0u;
    for (int i = threadIdx.x; i < BN; i += blockDim.x) bmax[i] = 0, bmin[i] = ~0u;

    // this thread's chunks: A chunk h is CA floats along K of one row (byte offset aoff, LDS offset ad); B chunk h is
    // CB k of one column (b by columns: as A's)
    int aoff[NA], ak[NA], ad[NA], ar[NA], boff[NB], bk[NB], bd[NB], bc[NB];
#pragma unroll
    for (int h = 0; h < NA; h++) {
        const int q = t + NTHR * h, r = q / (KB / CA), c = q % (KB / CA) * CA;
        ar[h] = r;
        ak[h] = c;
        aoff[h] = (int)(((int64_t)min(r, M - 1 - row0) * p.lda + c) * 4);
        ad[h] = c / 16 * SUB + c % 16 / 8 * AH + r * 16 + c % 8 * 2;
    }
#pragma unroll
    for (int h = 0; h < NB; h++) {
        const int q = t + NTHR * h;
        const int c = BT ? q / (KB / CB) : q % BN;
        int k = BT ? q % (KB / CB) * CB : q / BN * CB;
        if constexpr (!BT && BN >= 64) k = __builtin_amdgcn_readfirstlane(k);
        bc[h] = c;
        bk[h] = k;
        const int cc = min(c, N - 1 - col0);
        boff[h] = (int)((BT ? (int64_t)cc * p.ldb + k : (int64_t)k * p.ldb + cc) * 4);
        bd[h] = k / 16 * SUB + 3 * AP + k % 16 / 8 * BH + c * 16 + k % 8 * 2;
    }
    const char *Ab = (const char *)(A + ao + (int64_t)row0 * p.lda + kbeg);
    const char *Bb = (const char *)(B + bo + (BT ? (int64_t)col0 * p.ldb + kbeg : (int64_t)kbeg * p.ldb + col0));
    const int64_t bstep = BT ? (int64_t)KB * 4 : (int64_t)KB * p.ldb * 4;  // bytes per step
    const int ldb4 = BT ? 4 : (int)p.ldb * 4;                              // bytes between a B chunk's elements
    // buffer loads: a step's base in scalar registers, one 32-bit offset per lane (all in range: the host bounds the
    // strides, rows, columns and k are clamped)
    auto rsrc = [](const char *b) { return __builtin_amdgcn_make_buffer_rsrc((void *)b, 0, 0x7fffffff, 0x00027000); };
    // k index within the range of element e of a chunk at k c of step kt, clamped in the tail: offset back in bytes
    struct Set {
        float a[NA][CA], b[NB][CB];
    };
    // loads elements e .. e + n - 1 (n = 4 with VEC) of chunk h of step kt
    auto load_a = [&](Set &s, auto hc, auto ec, int kt) {
        constexpr int h = decltype(hc)::value, e = decltype(ec)::value;
        const auto rs = rsrc(Ab + (int64_t)kt * (KB * 4));
        const int lim = TAIL ? kr - kt * KB : 0;  // k left in the range at this step (may be below 1)
        if constexpr (VEC) {
            int o = aoff[h] + e * 4;
            if constexpr (TAIL) o -= max(0, ak[h] + e + 4 - lim) * 4;
            const v4f v = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0));
#pragma unroll
            for (int z = 0; z < 4; z++) s.a[h][e + z] = v[z];
        } else {
#pragma unroll
            for (int z = 0; z < 4; z++) {
                const int o = aoff[h] + (e + z) * 4 - max(0, ak[h] + e + z + 1 - lim) * 4;
                s.a[h][e + z] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, o, 0, 0));
            }
        }
    };
    auto load_b = [&](Set &s, auto hc, auto ec, int kt) {  // by columns: elements e .. e + 3; else e and e + 1
        constexpr int h = decltype(hc)::value, e = decltype(ec)::value;
        const auto rs = rsrc(Bb + kt * bstep);
        const int lim = TAIL ? kr - kt * KB : 0;
        if constexpr (BT && VEC) {
            int o = boff[h] + e * 4;
            if constexpr (TAIL) o -= max(0, bk[h] + e + 4 - lim) * 4;
            const v4f v = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0));
#pragma unroll
            for (int z = 0; z < 4; z++) s.b[h][e + z] = v[z];
        } else {
#pragma unroll
            for (int z = 0; z < (BT ? 4 : 2); z++) {
                int so = (e + z) * ldb4;
                int o = boff[h];
                if constexpr (TAIL) {
                    const int back = max(0, bk[h] + e + z + 1 - lim);
                    o += so - back * ldb4;
                    so = 0;
                }
                s.b[h][e + z] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, o, so, 0));
            }
        }
    };
    auto load_all = [&](Set &s, int kt) {
        static_for<0, NA>([&](auto h) {
            static_for<0, CA / 4>([&](auto e) { load_a(s, h, std::integral_constant<int, 4 * decltype(e)::value>(), kt); });
        });
        static_for<0, NB>([&](auto h) {
            constexpr int n = BT ? 4 : 2;
            static_for<0, CB / n>([&](auto e) { load_b(s, h, std::integral_constant<int, n * decltype(e)::value>(), kt); });
        });
    };

    // splitting: the pairs of a thread's chunks in units of four, twelve segments per unit, in each segment one
    // instruction (or two) per pair, so that neighbouring instructions are independent
    constexpr int PA = NA * CA / 2, PB = NB * CB / 2, PT = PA + PB, U = (PT + 3) / 4, SEGS = 12 * U;
    float mxa[NA], mxb[NB];
    uint32_t mna[NA], mnb[NB];
#pragma unroll
    for (int h = 0; h < NA; h++) mxa[h] = 0.f, mna[h] = ~0u;
#pragma unroll
    for (int h = 0; h < NB; h++) mxb[h] = 0.f, mnb[h] = ~0u;
    float res[8];
    uint32_t hi[8], pk[3][PT];
    // segment ic of the split of step kt's elements in s into stage ws; then loads step kl into s
    auto segment = [&](auto ic, Set &s, int kt, char *ws, int kl) {
        constexpr int i = decltype(ic)::value, un = i / 12, sg = i % 12, np = PT - 4 * un < 4 ? PT - 4 * un : 4;
        static_for<0, np>([&](auto qc) {
            constexpr int q = decltype(qc)::value, pr = 4 * un + q;
            constexpr bool isA = pr < PA;
            constexpr int CN = isA ? CA : CB, qq = isA ? pr : pr - PA, h = qq / (CN / 2), e = qq % (CN / 2) * 2;
            float *x;
            if constexpr (isA) x = &s.a[h][e];
            else x = &s.b[h][e];
            if constexpr (sg == 0) {
                if constexpr (TAIL) {
                    const int k = (isA ? ak[isA ? h : 0] : bk[isA ? 0 : h]) + e, lim = kr - kt * KB;
                    x[0] = k < lim ? x[0] : 0.f;
                    x[1] = k + 1 < lim ? x[1] : 0.f;
                }
                pk[0][pr] = bf16_pair(x[0], x[1]);
            }
            if constexpr (sg == 1 || sg == 6) hi[2 * q] = pk[sg / 6][pr] << 16;
            if constexpr (sg == 2 || sg == 7) hi[2 * q + 1] = pk[sg / 6][pr] & 0xffff0000u;
            if constexpr (sg == 3) res[2 * q] = x[0] - __builtin_bit_cast(float, hi[2 * q]);
            if constexpr (sg == 4) {
                res[2 * q + 1] = x[1] - __builtin_bit_cast(float, hi[2 * q + 1]);
                uint32_t &m = isA ? mna[isA ? h : 0] : mnb[isA ? 0 : h];
                m = min(min((__builtin_bit_cast(uint32_t, x[0]) << 1) - 1u, (__builtin_bit_cast(uint32_t, x[1]) << 1) - 1u), m);
            }
            if constexpr (sg == 5) {
                pk[1][pr] = bf16_pair(res[2 * q], res[2 * q + 1]);
                float &m = isA ? mxa[isA ? h : 0] : mxb[isA ? 0 : h];
                m = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), m);
            }
            if constexpr (sg == 8) res[2 * q] -= __builtin_bit_cast(float, hi[2 * q]);
            if constexpr (sg == 9) res[2 * q + 1] -= __builtin_bit_cast(float, hi[2 * q + 1]);
            if constexpr (sg == 10) pk[2][pr] = bf16_pair(res[2 * q], res[2 * q + 1]);
            if constexpr (e + 2 == CN && (sg == 1 || sg == 6 || sg == 11)) {  // part sg / 5 of the chunk is complete
                constexpr int z = sg / 5, p0 = pr + 1 - CN / 2;
                char *d = ws + (isA ? ad[isA ? h : 0] : bd[isA ? 0 : h]) + z * (isA ? AP : BP);
                if constexpr (CN == 8) *(v4u *)d = v4u{pk[z][p0], pk[z][p0 + 1], pk[z][p0 + 2], pk[z][p0 + 3]};
                else *(v2u *)d = v2u{pk[z][p0], pk[z][p0 + 1]};
            }
            // the elements are in parts: reload them
            if constexpr (isA) {
                if constexpr (e % 4 == 2 && sg == 7 + q / 2)
                    load_a(s, std::integral_constant<int, h>(), std::integral_constant<int, e - 2>(), kl);
            } else if constexpr (BT) {
                if constexpr (e % 4 == 2 && sg == 7 + q / 2)
                    load_b(s, std::integral_constant<int, h>(), std::integral_constant<int, e - 2>(), kl);
            } else if constexpr (sg == 6 + q) {
                load_b(s, std::integral_constant<int, h>(), std::integral_constant<int, e>(), kl);
            }
        });
    };

    // the largest and the smallest operand of each row and column
    auto store_max = [&]() {
#pragma unroll
        for (int h = 0; h < NA; h++) {
            atomicMax(&amax[ar[h]], __builtin_bit_cast(uint32_t, mxa[h]));
            atomicMin(&amin[ar[h]], mna[h]);
        }
#pragma unroll
        for (int h = 0; h < NB; h++) {
            atomicMax(&bmax[bc[h]], __builtin_bit_cast(uint32_t, mxb[h]));
            atomicMin(&bmin[bc[h]], mnb[h]);
        }
    };
    // parts of steps 0 and 1 into their stages, steps 2 and 3 loading
    Set s0, s1;
    auto prologue = [&]() {
        load_all(s0, 0);
        load_all(s1, 1);
        static_for<0, SEGS>([&](auto c) { segment(c, s0, 0, sm[0], min(2, nk - 1)); });
        static_for<0, SEGS>([&](auto c) { segment(c, s1, 1, sm[1], min(3, nk - 1)); });
        wait_vmcnt_barrier<63>();
    };
    if constexpr (PW > 0) {
        if (w >= NW) {  // a loading wave: step by step with the barriers of the multiplying ones
            prologue();
            wait_vmcnt_barrier<63>();
            auto produce = [&](int kt, Set &s) {
                static_for<0, SEGS>([&](auto c) { segment(c, s, kt + 2, sm[kt & 1], min(kt + 4, nk - 1)); });
                wait_vmcnt_barrier<63>();
            };
            for (int kt = 0; kt < nk; kt += 2) {
                produce(kt, s0);
                produce(kt + 1, s1);
            }
            store_max();
            __syncthreads();
            return;
        }
    }

    const int wr = (w / WN) * MT * 32, wc = (w % WN) * NT * 32;
    const int fa = (wr + (l & 31)) * 16 + AH * (l >> 5), fb = 3 * AP + (wc + (l & 31)) * 16 + BH * (l >> 5);
    struct Frag {
        v8bf a[KS][3][MT], b[KS][3][NT];
    };
    constexpr int RF = 3 * (MT + NT), R = RF * KS;  // fragment reads per step, in the order of their first use
    auto read_frag = [&](auto ic, const char *rs, Frag &f) {
        constexpr int i = decltype(ic)::value, u = i / RF, o = i % RF / (MT + NT), z = i % RF % (MT + NT);
        constexpr int pa = o == 0 ? 2 : o == 1 ? 0 : 1, pb = o == 0 ? 0 : o == 1 ? 2 : 1;
        if constexpr (z < MT) f.a[u][pa][z] = *(const v8bf *)(rs + u * SUB + pa * AP + fa + z * 512);
        else f.b[u][pb][z - MT] = *(const v8bf *)(rs + u * SUB + pb * BP + fb + (z - MT) * 512);
    };
    v16f acc[MT][NT], lo[MT][NT];  // the sums of a1 b1 and of the small part products
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = lo[i][j][r] = 0.f;
    constexpr int G = 6 * MT * NT * KS, GD = G * 5 / 6;  // MFMAs per step; the other work follows the first GD of them
    auto step = [&](int kt, Set &s, const Frag &cur, Frag &nxt) {
        const char *rs = sm[(kt + 1) & 1];
        char *ws = sm[kt & 1];
        const int kl = min(kt + 4, nk - 1);
        static_for<0, G>([&](auto gc) {
            constexpr int g = decltype(gc)::value, u = g / (6 * MT * NT), o = g % (6 * MT * NT), pr = o / (MT * NT);
            constexpr int i = o % (MT * NT) / NT, j = o % NT;
            constexpr int pa = pr == 0 ? 2 : pr == 1 || pr >= 4 ? 0 : 1, pb = pr == 1 ? 2 : pr == 2 || pr == 4 ? 1 : 0;
            v16f &sum = pr == 5 ? acc[i][j] : lo[i][j];
            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur.b[u][pb][j], cur.a[u][pa][i], sum, 0, 0, 0);
            static_for<(g < GD ? g * R / GD : R), (g < GD ? (g + 1) * R / GD : R)>([&](auto c) { read_frag(c, rs, nxt); });
            if constexpr (PW == 0)
                static_for<(g < GD ? g * SEGS / GD : SEGS), (g < GD ? (g + 1) * SEGS / GD : SEGS)>(
                    [&](auto c) { segment(c, s, kt + 2, ws, kl); });
            sched_fence();
        });
        // every wave's LDS reads and writes are done before the stages change roles (the loads stay outstanding)
        wait_vmcnt_barrier<63>();
    };
    Frag f0, f1;
    if constexpr (PW > 0) wait_vmcnt_barrier<63>();
    else prologue();
    static_for<0, R>([&](auto c) { read_frag(c, sm[0], f0); });
    wait_vmcnt_barrier<63>();  // stage 0 is read before step 0 writes it
    for (int kt = 0; kt < nk; kt += 2) {
        step(kt, s0, f0, f1);
        step(kt + 1, s1, f1, f0);
    }

    // the results the parts cannot hold
    if constexpr (PW == 0) store_max();
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; i++) {
        constexpr uint32_t kLossy = ((127u - 109u) << 24) - 1u, kUnder = ((127u - 120u) << 24) - 1u;
        const float ra = __builtin_bit_cast(float, amax[wr + 32 * i + (l & 31)]);
        const bool la = amin[wr + 32 * i + (l & 31)] < kLossy;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            // whether the tile can hold such a result: one is not finite or nonzero below 2^-120; or (bounds over the
            // tile's rows and columns; lane l holds row and column l % 32) small beside a column where a row holds a
            // value below 2^-109, or the other way round; or zero with no product of 2^-120.  Element by element only
            // then: probabilities of a Softmax have such rows all over.
            float top = 0.f;
            uint32_t low = ~0u;
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = acc[i][j][r] + lo[i][j][r];
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const float v0 = acc[i][j][r], v1 = acc[i][j][r + 1];
                top = __builtin_elementwise_maximum(__builtin_elementwise_maximum(fabsf(v0), fabsf(v1)), top);
                low = min(min((__builtin_bit_cast(uint32_t, v0) << 1) - 1u, (__builtin_bit_cast(uint32_t, v1) << 1) - 1u), low);
            }
            const bool lc = bmin[wc + 32 * j + (l & 31)] < kLossy;
            const float c0 = __builtin_bit_cast(float, bmax[wc + 32 * j + (l & 31)]);
            if (!__any(!(top < __builtin_inff()) || low < kUnder)) {
                const bool lossy_row = __any(la), lossy_col = __any(lc);
                if (!lossy_row && !lossy_col && !__any((ra != 0.f && ra < 0x1p-60f) || (c0 != 0.f && c0 < 0x1p-60f))) continue;
                const auto larger = [](float x, float y) { return fmaxf(x, y); };
                const auto smaller = [](float x, float y) { return fminf(x, y); };
                const float rx = wave_reduce_dpp(ra, larger), cx = wave_reduce_dpp(c0, larger);
                const float rn = wave_reduce_dpp(ra != 0.f ? ra : __builtin_inff(), smaller);
                const float cn = wave_reduce_dpp(c0 != 0.f ? c0 : __builtin_inff(), smaller);
                const float lim = fmaxf(lossy_row ? cx : 0.f, lossy_col ? rx : 0.f) * 0x1p-96f;
                bool zero = false;
#pragma unroll
                for (int r = 0; r < 16; r++) zero = zero || acc[i][j][r] == 0.f;
                const bool none = low == ~0u;  // all of this lane's are zero
                if (!__any((!none && __builtin_bit_cast(float, (low + 1u) >> 1) < lim) ||
                           (zero && (lim > 0.f || rn * cn < 0x1p-120f))))
                    continue;
            }
            uint32_t again = 0;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int c = wc + 32 * j + 8 * (r / 4) + 4 * (l / 32) + r % 4;
                const float cb = __builtin_bit_cast(float, bmax[c]), v = fabsf(acc[i][j][r]);
                const bool lossy = v < fmaxf(la ? cb : 0.f, bmin[c] < kLossy ? ra : 0.f) * 0x1p-96f;
                const bool under = v < 0x1p-120f && (v != 0.f || ra * cb < 0x1p-120f);
                again |= (ra != 0.f && cb != 0.f && (lossy || under)) || !(v < __builtin_inff()) ? 1u << r : 0u;
            }
            if (__any(again != 0)) {
                const v16f x = f32_tile<BT>(A + ao, B + bo, M, N, p.lda, p.ldb, row0 + wr + 32 * i, col0 + wc + 32 * j,
                                            kbeg, kbeg + kr, l);
#pragma unroll
                for (int r = 0; r < 16; r++)
                    if (again >> r & 1) acc[i][j][r] = x[r];
            }
        }
    }
    if constexpr (SPLIT)
        mm_store_part<MT, NT>(acc, p.part + ((int64_t)(blockIdx.z - zb * p.split) * p.batch + zb) * M * N, M, N,
                              row0 + wr, col0 + wc, l);
    else if (vc)
        mm_epilogue<MT, NT, true, GELU>(acc, C, p, co, row0 + wr, col0 + wc, l, tab);
    else
        mm_epilogue<MT, NT, false, GELU>(acc, C, p, co, row0 + wr, col0 + wc, l, tab);
}

// 64x64 tiles of a float product: of the whole call, not of a launch's share of a large batch, and of one matrix in a
// grouped launch, which has to give the bits of its single products.  `fold`: of the rows of the whole batch where every
// matrix of it meets one right operand, whether the call could fold them into one product (dense rows) or not (a
// transposed view, a bias row per batch), so that both run on one unit.
static int64_t f32_tiles(const MatMulArgs &p, bool fold) {
    const int64_t cols = ((int64_t)p.n + 63) / 64;
    if (p.split_per_matrix) return ((int64_t)p.m + 63) / 64 * cols;
    int64_t batch = 1;
    for (int d = 0; d < p.nbatch; d++) {
        batch *= p.bdims[d];
        fold = fold && (p.bdims[d] == 1 || p.b_bstr[d] == 0);
    }
    return fold ? (p.m * batch + 63) / 64 * cols : ((int64_t)p.m + 63) / 64 * cols * batch;
}

constexpr int kB3MinK = 256, kB3LoneK = 512, kB3SplitK = 1024, kB3NarrowK = 1024;
// Whether a K range of kr goes to k_matmul_f32_b3: kB3MinK or more, N above 32 (a context product of 32-wide heads is
// bound by its loads: [96,512,512]x[96,512,32] 24 us on the fp32 MFMA, 26 in parts), and strides whose offsets within
// a tile and a step stay below 2^31 bytes (rows of up to 8 MB; longer ones keep the fp32 MFMA).  A range of up to kB3LoneK
// whose 64x64 tiles (f32_tiles, whichever tile b3_tile then takes) find a CU each keeps the fp32 MFMA too: the parts' first
// stage and last check cost 1.2 us more than a block of so few steps gains (six batches of 384^3 11.8 against 10.2 us, 12
// of [512,512]x[512,128] 12.3 / 11.9; past the line [4096,384]x[384,384] 14.9 / 15.9, 12 batches of 384^3 17.4 / 17.0,
// [788,768]x[768,768] 14.7 / 15.1).  So does a K below kB3NarrowK over 64 columns (the context of 64-wide heads: a left
// operand that is read once) unless a CU has two tiles: [96,512,512]x[96,512,64] 35.3 / 32.4, [48,197,512]x[48,512,64]
// 12.7 / 12.0; [192,128,512]x[192,512,64] 18.2 / 20.7, [96,512,1024]x[96,1024,64] 61.5 / 61.3.  Where the direct-load fp32
// kernel does not take the operands (K no multiple of 64, N no multiple of 4 or below 64) the other one is slower, and K
// of 512 and N of 33 to 64 run in parts: [12,512,512]x[12,512,65] 14.1 / 33.9, [48,197,512]x[48,512,40] 12.0 / 18.2.  The
// ranges of a split product, at most one block per CU and mostly of few rows, keep it up to kB3SplitK: there the parts'
// 4-byte loads of B count too (ranges of 512: [60,2560]x[2560,4096] 18.0 us in parts, 16.5; 768: [256,3072]x[3072,768]
// 18.9, 18.3; 1024: [384,3072]x[3072,768] 22.6, 22.5; 1536: [640,3072]x[3072,640] 29.3, 30.1).
static bool f32_b3(const MatMulArgs &p, int kr) {
    const int64_t lim = kMatMulPartsRow;
    if (kr < kB3MinK || p.n <= 32 || p.lda > lim || p.ldb > lim || p.k > (1 << 24)) return false;
    if (kr < p.k) return kr > kB3SplitK;
    const int64_t tiles = f32_tiles(p, true);
    const bool direct = kr % 64 == 0 && p.n % 4 == 0 && p.n >= 64;
    if (direct && p.n == 64 && kr < kB3NarrowK) return tiles > 256 && tiles <= 512;
    return kr >= kB3LoneK + (direct ? 1 : 0) || tiles > 256;
}

// The block tile: the least estimated time.  A block takes `fixed` us (first stage, check, stores) and per step of 16 k
// `lone` us when it has a CU to itself, `full` us per block in a launch of several blocks per CU (r of them at once, else
// one after another): rounds of r blocks, then the rest.  Fitted to [4096, 384..3072] x [.., 384..3072], [788, ..],
// 1024^3 to 2048^3 and 12 batches of 384^3 and 512^3, where the tile it picks is the fastest or within 4%.  128x128 has
// two forms: eight waves of 64x32, one block per CU, and four of 64x64, two of them (255 registers), whose first stage and
// epilogue the other block covers: [4096,768]x[768,3072] 118 against 111 us, [4096,3072]x[3072,768] (192 tiles, a block
// per CU) 118 against 130.
static int b3_tile(const MatMulArgs &p, bool only_general) {
    struct B3Tile {
        int bm, bn, r;
        double fixed, lone, full;
    };
    static const B3Tile cand[] = {{128, 128, 1, 2.9, 0.58, 0.62}, {128, 64, 1, 1.8, 0.35, 0.44},
                                  {64, 64, 3, 1.5, 0.27, 0.25}, {64, 64, 1, 1.0, 0.21, 0.28},
                                  {128, 128, 2, 2.5, 0.62, 0.64}};
    const double steps = (double)((p.k + 15) / 16);
    int best = 0;
    double cost = 0;
    for (int i = 0; i < 5; i++) {
        if (only_general && i != 0 && i != 2) continue;
        const B3Tile &c = cand[i];
        const int64_t tiles = (int64_t)((p.m + c.bm - 1) / c.bm) * ((p.n + c.bn - 1) / c.bn) * p.batch;
        const int64_t per_cu = (tiles + 255) / 256, rounds = per_cu / c.r, rest = per_cu - rounds * c.r;
        const double t = per_cu == 1 ? c.fixed + steps * c.lone
                                     : rounds * (c.fixed + steps * c.r * c.full) +
                                           (rest ? c.fixed + steps * (rest > 1 ? rest * c.full : c.lone) : 0);
        if (i == 0 || t < cost) {
            best = i;
            cost = t;
        }
    }
    return best;
}

template <int BM, int BN, int WM, int WN, int PW, int KS, int WE, bool VEC, bool TAIL, bool BT>
static void b3_launch(const float *a, const float *b, float *c, const MatMulArgs &p, bool vc, hipStream_t s) {
    const dim3 g((p.n + BN - 1) / BN, (p.m + BM - 1) / BM, (unsigned)p.batch), blk((WM * WN + PW) * 64);
    if constexpr (!BT) {
        if (p.gelu) {
            hipLaunchKernelGGL((k_matmul_f32_b3<BM, BN, WM, WN, PW, KS, WE, VEC, TAIL, false, true>), g, blk, 0, s, a, b, c, p, (int)vc);
            return;
        }
    }
    hipLaunchKernelGGL((k_matmul_f32_b3<BM, BN, WM, WN, PW, KS, WE, VEC, TAIL, BT, false>), g, blk, 0, s, a, b, c, p, (int)vc);
}

// vec: f32_vec (the epilogue's 16-byte accesses)
static void launch_f32_b3(const float *a, const float *b, float *c, const MatMulArgs &p, bool vec, hipStream_t s) {
    // 16-byte loads along K: A's rows (and B's columns, by columns) aligned, K a multiple of 4
    bool va = p.k % 4 == 0 && p.lda % 4 == 0 && (uintptr_t)a % 16 == 0 &&
              (!p.bt || (p.ldb % 4 == 0 && (uintptr_t)b % 16 == 0));
    for (int d = 0; d < p.nbatch; d++) va = va && p.a_bstr[d] % 4 == 0 && (!p.bt || p.b_bstr[d] % 4 == 0);
    const bool whole = va && p.k % 64 == 0;  // whole step pairs of every tile
    const int tile = b3_tile(p, p.bt || !whole);
    if (p.bt) {
        if (whole && tile == 0) b3_launch<128, 128, 2, 4, 0, 1, 2, true, false, true>(a, b, c, p, vec, s);
        else if (whole) b3_launch<64, 64, 2, 2, 0, 2, 3, true, false, true>(a, b, c, p, vec, s);
        else b3_launch<64, 64, 2, 2, 0, 2, 2, false, true, true>(a, b, c, p, vec, s);
        return;
    }
    if (!va) {  // unaligned rows: scalar loads
        if (tile == 0) b3_launch<128, 128, 2, 4, 0, 1, 2, false, true, false>(a, b, c, p, vec, s);
        else b3_launch<64, 64, 2, 2, 0, 2, 2, false, true, false>(a, b, c, p, vec, s);
        return;
    }
    if (!whole) {
        if (tile == 0) b3_launch<128, 128, 2, 4, 0, 1, 2, true, true, false>(a, b, c, p, vec, s);
        else b3_launch<64, 64, 2, 2, 0, 2, 2, true, true, false>(a, b, c, p, vec, s);
        return;
    }
    switch (tile) {
    case 0: b3_launch<128, 128, 2, 4, 0, 1, 2, true, false, false>(a, b, c, p, vec, s); break;
    case 4: b3_launch<128, 128, 2, 2, 0, 1, 2, true, false, false>(a, b, c, p, vec, s); break;
    case 1: b3_launch<128, 64, 4, 2, 0, 2, 2, true, false, false>(a, b, c, p, vec, s); break;
    case 2: b3_launch<64, 64, 2, 2, 0, 2, 3, true, false, false>(a, b, c, p, vec, s); break;
    default: b3_launch<64, 64, 2, 2, 8, 2, 3, true, false, false>(a, b, c, p, vec, s); break;
    }
}

// the K ranges of a split product into p.part: 64x64 tiles, at most one per CU
static void launch_f32_parts(const float *a, const float *b, float *c, const MatMulArgs &p, hipStream_t s) {
    const dim3 g((p.n + 63) / 64, (p.m + 63) / 64, (unsigned)(p.batch * p.split));
    if (f32_b3(p, p.k / p.split))
        hipLaunchKernelGGL((k_matmul_f32_b3<64, 64, 2, 2, 8, 2, 3, true, false, false, false, true>), g, dim3(768), 0, s, a, b, c, p, 1);
    else
        hipLaunchKernelGGL((k_matmul_f32_dl<64, 64, 2, 2, 4, 3, 8, false, true>), g, dim3(256), 0, s, a, b, c, p);
}

// ---------------------------------------------------------------------------
// float, split products of few rows (a short query's projections): one launch
// ---------------------------------------------------------------------------
// The K ranges of a split product and their ordered sum in one block, on the VALU: v_mfma_f32_32x32x2f32 is two fused
// multiply-adds per result, the lower lanes' k first (checked bit for bit over 200,000 results of every magnitude), so
// a chain of v_fma_f32 in the fp32 kernels' order gives the partial products' bits without the rows of zeros that the
// MFMA would multiply.  A block takes kSmallR rows and kSmallC columns, a lane one column of one range (four ranges per
// wave): its 64 elements of the right operand are loaded at once, one memory latency for the whole of K; the rows come
// from LDS, each range padded by four floats (the four ranges of a wave read different banks).  The partials then meet
// in LDS and are summed in range order with the epilogue, exactly as k_matmul_split_sum does.
// Bound: launches and memory latency.  5.1 us a product ([8,1536]x[1536,384] and the like) in place of 4.3 for the
// tiles and 3.7 to 5.4 for the sum; a captured encoder of 12 layers of 384, replayed in a row, at 8 tokens 513 -> 400 us,
// at 32 540 -> 442, at 64 585 -> 512.
constexpr int kSmallR = 4, kSmallC = 16, kSmallRanges = 64;

template <bool GELU>
__global__ __launch_bounds__(1024) void k_matmul_small(const float *__restrict__ A, const float *__restrict__ B,
                                                       float *__restrict__ C, MatMulArgs p) {
    extern __shared__ float sh[];  // rows [kSmallR][split * (range + 4)], then partials [split][kSmallR][kSmallC]
    __shared__ ExpTable tab;
    if constexpr (GELU) exp_table_fill(tab);
    constexpr int RL = 64;  // the length of a range
    const int M = p.m, N = p.n, R = p.split, LD = R * (RL + 4);
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int col0 = blockIdx.x * kSmallC, row0 = blockIdx.y * kSmallR;
    int64_t ao = 0, bo = 0, co = 0;
    if (p.nbatch) batch_offsets(p.batch_base + blockIdx.z, p, &ao, &bo, &co);
    // the rows first (they are waited for first): each wave its own four ranges, lane l 16 bytes of range l / 16
    constexpr int RW = 64 / kSmallC;  // ranges per wave
    const int range = min(w * RW + l / kSmallC, R - 1), c = l % kSmallC;
    v4f av[kSmallR];
    const float *Ar = A + ao + range * RL + 4 * c;
#pragma unroll
    for (int r = 0; r < kSmallR; r++) av[r] = *reinterpret_cast<const v4f *>(Ar + (int64_t)min(row0 + r, M - 1) * p.lda);
    sched_fence();
    const float *Bc = B + bo + (int64_t)range * RL * p.ldb + min(col0 + c, N - 1);
    float b[RL];
#pragma unroll
    for (int k = 0; k < RL; k++) b[k] = Bc[(int64_t)k * p.ldb];
    sched_fence();
    // the outputs' bias and residual with them
    const int orow = row0 + (int)threadIdx.x / kSmallC, ocol = col0 + (int)threadIdx.x % kSmallC;
    const bool out = threadIdx.x < kSmallR * kSmallC && orow < M && ocol < N;
    const int64_t bz = p.batch_base + blockIdx.z;
    const float bias = out && p.bias ? p.bias[bz * p.bias_bstr + ocol] : 0.f;
    const float res = out && p.res ? p.res[bz * (int64_t)M * N + (int64_t)orow * N + ocol] : 0.f;
    float *as = sh + range * (RL + 4);
#pragma unroll
    for (int r = 0; r < kSmallR; r++) *reinterpret_cast<v4f *>(as + r * LD + 4 * c) = av[r];
    // a wave reads only the ranges it wrote
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float acc[kSmallR];
#pragma unroll
    for (int r = 0; r < kSmallR; r++) acc[r] = 0.f;
#pragma unroll
    for (int s = 0; s < RL; s += 16)
#pragma unroll
        for (int r = 0; r < kSmallR; r++) {
            v4f a[4];
#pragma unroll
            for (int i = 0; i < 4; i++) a[i] = *reinterpret_cast<const v4f *>(as + r * LD + s + 4 * i);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                acc[r] = __builtin_fmaf(a[j / 4][j % 4], b[s + j], acc[r]);
                acc[r] = __builtin_fmaf(a[2 + j / 4][j % 4], b[s + 8 + j], acc[r]);
            }
        }
    float *part = sh + kSmallR * LD;  // (ranges past the last: the last one's values again)
#pragma unroll
    for (int r = 0; r < kSmallR; r++) part[(range * kSmallR + r) * kSmallC + c] = acc[r];
    __syncthreads();
    if (!out) return;
    constexpr int kOut = kSmallR * kSmallC, kChunk = 8;
    const float *P = part + threadIdx.x;
    float v = P[0];
    for (int g0 = 1; g0 < R; g0 += kChunk) {
        float x[kChunk];
#pragma unroll
        for (int g = 0; g < kChunk; g++) x[g] = P[min(g0 + g, R - 1) * kOut];
#pragma unroll
        for (int g = 0; g < kChunk; g++)
            if (g0 + g < R) v = v + x[g];
    }
    if (p.bias) v = v + bias;
    if (p.res) v = v + res;
    if constexpr (GELU) {
        v = gelu_erf_lx(v, tab);
    }
    C[co + (int64_t)orow * p.ldc + ocol] = v;
}

// Whether a product of `split` ranges goes to k_matmul_small: ranges of 64 (K below 128 times the ranges the chip has
// room for), at most kSmallRanges of them (a block of 16 waves), and at most kSmallM rows: every four rows read the
// right operand again from L2, and above a tile of 64 the ranges of a long K are no longer 64.  Blocks of eight rows
// measured slower up to 64 rows (32 rows: 473 against 430 us for the 12-layer encoder).
constexpr int kSmallM = 64;
static bool f32_small(const void *a, const void *b, const void *c, const MatMulArgs &p, int split) {
    if (split <= 1 || split > kSmallRanges || p.k / split != 64 || p.m > kSmallM || p.bt) return false;
    // a result over an operand: blocks still read what others have written (the two launches read both first)
    int64_t ea = (int64_t)(p.m - 1) * p.lda + p.k, eb = (int64_t)(p.k - 1) * p.ldb + p.n, ec = (int64_t)(p.m - 1) * p.ldc + p.n;
    for (int d = 0; d < p.nbatch; d++) {
        ea += (p.bdims[d] - 1) * p.a_bstr[d];
        eb += (p.bdims[d] - 1) * p.b_bstr[d];
        ec += (p.bdims[d] - 1) * p.c_bstr[d];
    }
    const float *fa = (const float *)a, *fb = (const float *)b, *fc = (const float *)c;
    return !(fc < fa + ea && fa < fc + ec) && !(fc < fb + eb && fb < fc + ec);
}
static void launch_f32_small(const float *a, const float *b, float *c, const MatMulArgs &p, hipStream_t s) {
    const dim3 g((p.n + kSmallC - 1) / kSmallC, (p.m + kSmallR - 1) / kSmallR, (unsigned)p.batch);
    const dim3 blk(64 * ((p.split + 64 / kSmallC - 1) / (64 / kSmallC)));
    const size_t lds = (size_t)(kSmallR * (p.k + 4 * p.split) + p.split * kSmallR * kSmallC) * sizeof(float);
    if (p.gelu) hipLaunchKernelGGL(k_matmul_small<true>, g, blk, lds, s, a, b, c, p);
    else hipLaunchKernelGGL(k_matmul_small<false>, g, blk, lds, s, a, b, c, p);
}

// Split K (p.split ranges, p.part holding the partials): 64x64 tiles, then the ordered sum with the epilogue.
static void launch_f32_split(const float *a, const float *b, float *c, const MatMulArgs &p, hipStream_t s) {
    launch_f32_parts(a, b, c, p, s);
    const int64_t nq = (int64_t)p.m * p.n / 4 * p.batch;
    const dim3 gs((unsigned)((nq + 255) / 256));
    if (p.gelu) hipLaunchKernelGGL(k_matmul_split_sum<true>, gs, dim3(256), 0, s, c, p);
    else hipLaunchKernelGGL(k_matmul_split_sum<false>, gs, dim3(256), 0, s, c, p);
}

template <int BM, int BN, int WM, int WN>
static void launch_f32(const float *a, const float *b, float *c, const MatMulArgs &p, bool vec, hipStream_t s) {
    dim3 g((p.n + BN - 1) / BN, (p.m + BM - 1) / BM, (unsigned)p.batch);
    const dim3 blk(WM * WN * 64);
    if (p.bt) {  // a transposed view of B, without an epilogue
        if (vec) hipLaunchKernelGGL((k_matmul_f32<BM, BN, WM, WN, true, false, true>), g, blk, 0, s, a, b, c, p);
        else hipLaunchKernelGGL((k_matmul_f32<BM, BN, WM, WN, false, false, true>), g, blk, 0, s, a, b, c, p);
        return;
    }
    if (p.gelu) {
        if (vec) hipLaunchKernelGGL((k_matmul_f32<BM, BN, WM, WN, true, true>), g, blk, 0, s, a, b, c, p);
        else hipLaunchKernelGGL((k_matmul_f32<BM, BN, WM, WN, false, true>), g, blk, 0, s, a, b, c, p);
    } else {
        if (vec) hipLaunchKernelGGL((k_matmul_f32<BM, BN, WM, WN, true, false>), g, blk, 0, s, a, b, c, p);
        else hipLaunchKernelGGL((k_matmul_f32<BM, BN, WM, WN, false, false>), g, blk, 0, s, a, b, c, p);
    }
}

// ---------------------------------------------------------------------------
// double: MFMA 16x16x4
// ---------------------------------------------------------------------------
// BM x BN block tile, four waves in a 2 x 2 grid, each (BM / 2) x (BN / 2) = MT x NT MFMA tiles of 16x16.  K steps
// of 16, double-buffered in LDS with k as the outer index (A transposed to [k][m], B as [k][n]), fed from
// registers one step ahead; VEC: 16-byte loads (k, n, the row and batch strides even, the operands 16-byte
// aligned).  Each dot product is summed in K order, four products per MFMA.
constexpr int kDBK = 16, kDPad = 2;

template <int BM, int BN, bool VEC>
__global__ __launch_bounds__(256) void k_matmul_f64(const double *__restrict__ A, const double *__restrict__ B,
                                                    double *__restrict__ C, MatMulArgs p) {
    constexpr int WTM = BM / 2, WTN = BN / 2, MT = WTM / 16, NT = WTN / 16;
    constexpr int AV = BM * kDBK / 2, BV = BN * kDBK / 2;  // 16-byte pairs of A and of B per K step
    static_assert(AV % 256 == 0 && BV % 256 == 0 && MT * 16 == WTM && NT * 16 == WTN, "whole tiles and loads");
    constexpr int LA = AV / 256, LB = BV / 256;
    constexpr int KQ = kDBK / 2, BQ = BN / 2;              // pairs per A row and per B row of a step
    __shared__ double As[2][kDBK][BM + kDPad];
    __shared__ double Bs[2][kDBK][BN + kDPad];
    const int M = p.m, N = p.n, K = p.k;
    const int t = threadIdx.x, l = t & 63, w = t >> 6;
    const int row0 = blockIdx.y * BM, col0 = blockIdx.x * BN;
    int64_t ao, bo, co;
    batch_offsets(p.batch_base + blockIdx.z, p, &ao, &bo, &co);
    const double *Ab = A + ao;
    const double *Bb = B + bo;
    double *Cb = C + co;
    const int64_t lda = p.lda, ldb = p.ldb;
    double2 ra[LA], rb[LB];
    auto load = [&](int k0) {
#pragma unroll
        for (int h = 0; h < LA; h++) {
            const int e = t + 256 * h;
            const int r = row0 + e / KQ, kk = k0 + (e % KQ) * 2;
            if constexpr (VEC) {
                ra[h] = (r < M && kk < K) ? *reinterpret_cast<const double2 *>(Ab + (int64_t)r * lda + kk)
                                          : make_double2(0.0, 0.0);
            } else {
                ra[h].x = (r < M && kk < K) ? Ab[(int64_t)r * lda + kk] : 0.0;
                ra[h].y = (r < M && kk + 1 < K) ? Ab[(int64_t)r * lda + kk + 1] : 0.0;
            }
        }
#pragma unroll
        for (int h = 0; h < LB; h++) {
            const int e = t + 256 * h;
            const int kb = k0 + e / BQ, c = col0 + (e % BQ) * 2;
            if constexpr (VEC) {
                rb[h] = (kb < K && c < N) ? *reinterpret_cast<const double2 *>(Bb + (int64_t)kb * ldb + c)
                                          : make_double2(0.0, 0.0);
            } else {
                rb[h].x = (kb < K && c < N) ? Bb[(int64_t)kb * ldb + c] : 0.0;
                rb[h].y = (kb < K && c + 1 < N) ? Bb[(int64_t)kb * ldb + c + 1] : 0.0;
            }
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int h = 0; h < LA; h++) {
            const int e = t + 256 * h;
            const int r = e / KQ, kk = (e % KQ) * 2;
            As[buf][kk][r] = ra[h].x;
            As[buf][kk + 1][r] = ra[h].y;
        }
#pragma unroll
        for (int h = 0; h < LB; h++) {
            const int e = t + 256 * h;
            *reinterpret_cast<double2 *>(&Bs[buf][e / BQ][(e % BQ) * 2]) = rb[h];
        }
    };
    const int wr = (w >> 1) * WTM, wc = (w & 1) * WTN;
    v4d acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[i][j][r] = 0.0;
    const int nk = (K + kDBK - 1) / kDBK;
    load(0);
    store(0);
    __syncthreads();
    int buf = 0;
    for (int kt = 0; kt < nk; kt++) {
        if (kt + 1 < nk) load((kt + 1) * kDBK);
#pragma unroll
        for (int kk = 0; kk < kDBK; kk += 4) {
            const int kr = kk + l / 16;
            double a[MT], b[NT];
#pragma unroll
            for (int i = 0; i < MT; i++) a[i] = As[buf][kr][wr + 16 * i + (l % 16)];
#pragma unroll
            for (int j = 0; j < NT; j++) b[j] = Bs[buf][kr][wc + 16 * j + (l % 16)];
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < nk) store(buf ^ 1);
        __syncthreads();
        buf ^= 1;
    }
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const int c = col0 + wc + 16 * j + (l % 16);
            if (c >= N) continue;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = row0 + wr + 16 * i + l / 16 + 4 * r;
                if (row < M) Cb[(int64_t)row * p.ldc + c] = acc[i][j][r];
            }
        }
}

template <int BM, int BN>
static void launch_f64(const double *a, const double *b, double *c, const MatMulArgs &p, hipStream_t s) {
    bool vec = p.k % 2 == 0 && p.n % 2 == 0 && p.lda % 2 == 0 && p.ldb % 2 == 0 &&
               (((uintptr_t)a | (uintptr_t)b) % 16 == 0);
    for (int d = 0; d < p.nbatch; d++) vec = vec && p.a_bstr[d] % 2 == 0 && p.b_bstr[d] % 2 == 0;
    const dim3 g((p.n + BN - 1) / BN, (p.m + BM - 1) / BM, (unsigned)p.batch);
    if (vec) hipLaunchKernelGGL((k_matmul_f64<BM, BN, true>), g, dim3(256), 0, s, a, b, c, p);
    else hipLaunchKernelGGL((k_matmul_f64<BM, BN, false>), g, dim3(256), 0, s, a, b, c, p);
}

// ---------------------------------------------------------------------------
// int32: exact wrapping multiply-add (C# unchecked int arithmetic) on the int8 matrix unit
// ---------------------------------------------------------------------------
// Modulo 2^32 an int32 is four signed base-256 digits, x = d0 + 2^8 d1 + 2^16 d2 + 2^24 d3, -128 <= d <= 127: the
// bytes of (x + 0x80808080) ^ 0x80808080.  A product is then the ten digit products of weight below 2^32, those of one
// weight summed in one int32 accumulator by v_mfma_i32_32x32x32_i8: exact below 2^31, i.e. for 2^15 k (up to four
// products of 2^14 each per k), so every kI32Fold the four accumulators are folded into the wrapping result.
//
// k_matmul_i32: 64x64 tile, four waves of 32x32 (four accumulators each), K steps of 64.  Elements go from global memory
// to registers one step ahead, are split (two instructions, then a 4x4 byte transpose) and written to LDS as four digit
// planes, [row][64 k] bytes with rows 80 bytes apart (the 16-byte fragment reads are free of bank conflicts); two
// stages, one barrier per step.  Past M, N and K loads clamp; elements past K are zero.
// Bound: the latency of a step's loads and its splitting (about 1.5 us a step), not the matrix unit: 12 products of
// 512^3 206 us on the VALU (16 TOPS), 36 here (90 TOPS).
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4u __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes at 4-byte alignment: one load
constexpr int kI32Fold = 16384;

// sixteen elements k .. k + 15 of a row of K (clamped to the row)
__device__ __forceinline__ void i32_load_row(const int32_t *row, int k, int K, uint32_t (&x)[16]) {
    if (k + 16 <= K) {
#pragma unroll
        for (int g = 0; g < 16; g += 4) {
            const i32x4u v = *reinterpret_cast<const i32x4u *>(row + k + g);
#pragma unroll
            for (int e = 0; e < 4; e++) x[g + e] = (uint32_t)v[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 16; e++) x[e] = (uint32_t)row[min(k + e, K - 1)];
    }
}
// and of a column, ldb apart
__device__ __forceinline__ void i32_load_col(const int32_t *col, int64_t ldb, int k, int K, uint32_t (&y)[16]) {
#pragma unroll
    for (int e = 0; e < 16; e++) y[e] = (uint32_t)col[(int64_t)min(k + e, K - 1) * ldb];
}
// the digits of sixteen elements (zero from element `left` on), one 16-byte row piece per plane
template <int PLANE>
__device__ __forceinline__ void i32_store_digits(const uint32_t (&v)[16], int left, char *d) {
    i32x4 dig[4];
#pragma unroll
    for (int g = 0; g < 4; g++) {
        uint32_t q[4];
#pragma unroll
        for (int e = 0; e < 4; e++) q[e] = 4 * g + e < left ? (v[4 * g + e] + 0x80808080u) ^ 0x80808080u : 0u;
        const uint32_t a01 = __builtin_amdgcn_perm(q[1], q[0], 0x05010400u);  // bytes 0, 0', 1, 1'
        const uint32_t b01 = __builtin_amdgcn_perm(q[1], q[0], 0x07030602u);  // bytes 2, 2', 3, 3'
        const uint32_t a23 = __builtin_amdgcn_perm(q[3], q[2], 0x05010400u);
        const uint32_t b23 = __builtin_amdgcn_perm(q[3], q[2], 0x07030602u);
        dig[0][g] = (int)__builtin_amdgcn_perm(a23, a01, 0x05040100u);
        dig[1][g] = (int)__builtin_amdgcn_perm(a23, a01, 0x07060302u);
        dig[2][g] = (int)__builtin_amdgcn_perm(b23, b01, 0x05040100u);
        dig[3][g] = (int)__builtin_amdgcn_perm(b23, b01, 0x07060302u);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) *reinterpret_cast<i32x4 *>(d + i * PLANE) = dig[i];
}
// one 32x32 tile over 32 k: the fragments of the four planes of A at fa and of B at fb
template <int PLANE>
__device__ __forceinline__ void i32_mfma10(const char *fa, const char *fb, i32x16 (&acc)[4]) {
    i32x4 a[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        a[i] = *reinterpret_cast<const i32x4 *>(fa + i * PLANE);
        b[i] = *reinterpret_cast<const i32x4 *>(fb + i * PLANE);
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; i + j < 4; j++) acc[i + j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(b[j], a[i], acc[i + j], 0, 0, 0);
}
__device__ __forceinline__ void i32_fold(i32x16 (&acc)[4], uint32_t (&total)[16]) {
#pragma unroll
    for (int r = 0; r < 16; r++) {
        total[r] += (uint32_t)acc[0][r] + ((uint32_t)acc[1][r] << 8) + ((uint32_t)acc[2][r] << 16) + ((uint32_t)acc[3][r] << 24);
        acc[0][r] = acc[1][r] = acc[2][r] = acc[3][r] = 0;
    }
}

__global__ __launch_bounds__(256) void k_matmul_i32(const int32_t *__restrict__ A, const int32_t *__restrict__ B,
                                                    int32_t *__restrict__ C, MatMulArgs p, int vc) {
    constexpr int KB = 64, LD = KB + 16, PLANE = 64 * LD;
    __shared__ __attribute__((aligned(16))) char sm[2][8 * PLANE];  // digit planes of A, then of B
    const int M = p.m, N = p.n, K = p.k;
    const int t = threadIdx.x, l = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int row0 = blockIdx.y * 64, col0 = blockIdx.x * 64;
    int64_t ao, bo, co;
    batch_offsets(p.batch_base + blockIdx.z, p, &ao, &bo, &co);
    // this thread's elements of a step: 16 k of one row of A, 16 k of one column of B
    const int ak = t % 4 * 16, bk = w * 16;
    const int32_t *Ar = A + ao + (int64_t)min(row0 + t / 4, M - 1) * p.lda;
    const int32_t *Bc = B + bo + min(col0 + l, N - 1);
    const int aw = t / 4 * LD + ak, bw = 4 * PLANE + l * LD + bk;
    const int fa = (w / 2 * 32 + l % 32) * LD + l / 32 * 16, fb = 4 * PLANE + (w % 2 * 32 + l % 32) * LD + l / 32 * 16;
    uint32_t x[16], y[16], total[16];
    i32x16 acc[4];
#pragma unroll
    for (int r = 0; r < 16; r++) {
        total[r] = 0;
        acc[0][r] = acc[1][r] = acc[2][r] = acc[3][r] = 0;
    }
    if (K > 0) {
        i32_load_row(Ar, ak, K, x);
        i32_load_col(Bc, p.ldb, bk, K, y);
    }
    for (int k0 = 0; k0 < K; k0 += KB) {
        char *st = sm[k0 / KB & 1];
        i32_store_digits<PLANE>(x, K - k0 - ak, st + aw);
        i32_store_digits<PLANE>(y, K - k0 - bk, st + bw);
        // (one barrier per step: a wave writes this stage again only after the next step's barrier, which every wave
        // reaches with its reads of it done)
        __syncthreads();
        if (k0 + KB < K) {
            i32_load_row(Ar, k0 + KB + ak, K, x);
            i32_load_col(Bc, p.ldb, k0 + KB + bk, K, y);
        }
#pragma unroll
        for (int u = 0; u < KB; u += 32) i32_mfma10<PLANE>(st + fa + u, st + fb + u, acc);
        if (k0 % kI32Fold == kI32Fold - KB) i32_fold(acc, total);
    }
    i32_fold(acc, total);
    const int row = row0 + w / 2 * 32 + l % 32;
    if (row >= M) return;
    int32_t *Cr = C + co + (int64_t)row * p.ldc;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const int col = col0 + w % 2 * 32 + 8 * g + l / 32 * 4;
        if (vc) {
            if (col < N) *reinterpret_cast<i32x4 *>(Cr + col) = i32x4{(int)total[4 * g], (int)total[4 * g + 1], (int)total[4 * g + 2], (int)total[4 * g + 3]};
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (col + e < N) Cr[col + e] = (int32_t)total[4 * g + e];
        }
    }
}

// Few tiles: 32x32 tiles whose K is dealt out to the block's waves in steps of 32, every wave splitting and multiplying
// its own steps from its own planes (no barrier), the waves' sums joined in LDS.
constexpr int kI32Waves = 8, kI32FewLd = 48, kI32FewPlane = 32 * kI32FewLd;  // rows 48 bytes apart: free of conflicts
__global__ __launch_bounds__(kI32Waves * 64) void k_matmul_i32_few(const int32_t *__restrict__ A, const int32_t *__restrict__ B,
                                                                  int32_t *__restrict__ C, MatMulArgs p) {
    constexpr int KB = 32, LD = kI32FewLd, PLANE = kI32FewPlane;
    extern __shared__ __attribute__((aligned(16))) char dyn[];
    const int M = p.m, N = p.n, K = p.k;
    const int t = threadIdx.x, l = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), nw = blockDim.x >> 6;
    const int row0 = blockIdx.y * 32, col0 = blockIdx.x * 32;
    int64_t ao, bo, co;
    batch_offsets(p.batch_base + blockIdx.z, p, &ao, &bo, &co);
    const int ak = l % 2 * 16, bk = l / 32 * 16;
    const int32_t *Ar = A + ao + (int64_t)min(row0 + l / 2, M - 1) * p.lda;
    const int32_t *Bc = B + bo + min(col0 + l % 32, N - 1);
    char *st = dyn + w * 8 * PLANE;
    uint32_t x[16], y[16], total[16];
    i32x16 acc[4];
#pragma unroll
    for (int r = 0; r < 16; r++) {
        total[r] = 0;
        acc[0][r] = acc[1][r] = acc[2][r] = acc[3][r] = 0;
    }
    int k0 = w * KB, n = 0;
    if (k0 < K) {
        i32_load_row(Ar, k0 + ak, K, x);
        i32_load_col(Bc, p.ldb, k0 + bk, K, y);
    }
    auto wave_sync = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    for (; k0 < K; k0 += nw * KB) {
        i32_store_digits<PLANE>(x, K - k0 - ak, st + l / 2 * LD + ak);
        i32_store_digits<PLANE>(y, K - k0 - bk, st + 4 * PLANE + l % 32 * LD + bk);
        wave_sync();
        if (k0 + nw * KB < K) {
            i32_load_row(Ar, k0 + nw * KB + ak, K, x);
            i32_load_col(Bc, p.ldb, k0 + nw * KB + bk, K, y);
        }
        i32_mfma10<PLANE>(st + l % 32 * LD + l / 32 * 16, st + 4 * PLANE + l % 32 * LD + l / 32 * 16, acc);
        wave_sync();
        if (++n % (kI32Fold / KB) == 0) i32_fold(acc, total);
    }
    i32_fold(acc, total);
    // [wave][r][lane], r 65 words apart; then output i of the tile is row i / 32, column i % 32
    uint32_t *sum = (uint32_t *)dyn;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; r++) sum[(w * 16 + r) * 65 + l] = total[r];
    __syncthreads();
    for (int i = t; i < 1024; i += blockDim.x) {
        const int row = i / 32, col = i % 32, s0 = (4 * (col / 8) + col % 4) * 65 + row + col / 4 % 2 * 32;
        uint32_t v = 0;
        for (int g = 0; g < nw; g++) v += sum[g * 16 * 65 + s0];
        if (row0 + row < M && col0 + col < N) C[co + (int64_t)(row0 + row) * p.ldc + col0 + col] = (int32_t)v;
    }
}

// Short K: the multiply-adds on the VALU, an output per thread.
__global__ __launch_bounds__(256) void k_matmul_i32_short(const int32_t *__restrict__ A, const int32_t *__restrict__ B,
                                                          int32_t *__restrict__ C, MatMulArgs p) {
    __shared__ uint32_t As[16][17], Bs[16][17];
    const int M = p.m, N = p.n, K = p.k;
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    const int row = blockIdx.y * 16 + ty, col = blockIdx.x * 16 + tx;
    int64_t ao, bo, co;
    batch_offsets(p.batch_base + blockIdx.z, p, &ao, &bo, &co);
    const int32_t *Ab = A + ao;
    const int32_t *Bb = B + bo;
    uint32_t acc = 0;
    for (int k0 = 0; k0 < K; k0 += 16) {
        As[ty][tx] = (row < M && k0 + tx < K) ? (uint32_t)Ab[(int64_t)row * p.lda + k0 + tx] : 0u;
        Bs[ty][tx] = (k0 + ty < K && col < N) ? (uint32_t)Bb[(int64_t)(k0 + ty) * p.ldb + col] : 0u;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 16; k++) acc += As[ty][k] * Bs[k][tx];
        __syncthreads();
    }
    if (row < M && col < N) C[co + (int64_t)row * p.ldc + col] = (int32_t)acc;
}

// Which kernel (us a call).  K of one step of 16, and K up to kI32ShortK of at most kI32ShortWork multiply-adds: the
// VALU, done before a split pays (12 products of 32^3 4.2 against 6.3 in 32x32 tiles, 64^3 4.2 / 5.0, 12 of 70^3 5.0 /
// 5.6, [768,16]x[16,768] 4.4 / 4.9 in 64x64 tiles; past it 12 of 100^3 6.4 / 5.4, [768,64]x[64,768] 8.1 / 4.7).  Then, of
// at most kI32FewTiles tiles of 64x64 (half the CUs): 32x32 tiles with K over the waves ([1,768]x[768,768] 22.5 on the
// VALU, 21.4 in 64x64 tiles, 7.5; 384^3 16.1 / 12.1 / 5.5; six of 250^3 17.9 / 11.1 / 9.4).  More tiles take the 64x64
// form, which reads the operands half as often (six of 384^3, 216 tiles: 51.5 / 13.5 / 18.8; 12 of 256^3, 192 tiles:
// 31.1 / 10.0 / 12.2; 12 of 512^3: 205 / 36 / 60).
constexpr int kI32FewTiles = 128, kI32ShortK = 96;
constexpr int64_t kI32ShortWork = (int64_t)1 << 23;
static void launch_i32(const int32_t *a, const int32_t *b, int32_t *c, const MatMulArgs &p, hipStream_t s) {
    const int64_t tiles = (((int64_t)p.m + 63) / 64) * (((int64_t)p.n + 63) / 64) * p.batch;
    if (p.k <= 16 || (p.k <= kI32ShortK && (int64_t)p.m * p.n <= kI32ShortWork / p.k / p.batch)) {
        const dim3 g((p.n + 15) / 16, (p.m + 15) / 16, (unsigned)p.batch);
        hipLaunchKernelGGL(k_matmul_i32_short, g, dim3(256), 0, s, a, b, c, p);
        return;
    }
    if (tiles <= kI32FewTiles) {
        const int nw = min(kI32Waves, (p.k + 31) / 32);
        const dim3 g((p.n + 31) / 32, (p.m + 31) / 32, (unsigned)p.batch);
        hipLaunchKernelGGL(k_matmul_i32_few, g, dim3(64 * nw), (size_t)nw * 8 * kI32FewPlane, s, a, b, c, p);
        return;
    }
    // 16-byte stores of C's rows
    bool vc = p.n % 4 == 0 && p.ldc % 4 == 0 && (uintptr_t)c % 16 == 0;
    for (int d = 0; d < p.nbatch; d++) vc = vc && p.c_bstr[d] % 4 == 0;
    const dim3 g((p.n + 63) / 64, (p.m + 63) / 64, (unsigned)p.batch);
    hipLaunchKernelGGL(k_matmul_i32, g, dim3(256), 0, s, a, b, c, p, (int)vc);
}

// ---------------------------------------------------------------------------
// dense copy of a strided view (the broadcast operands of MatMul's rank-1 case)
// ---------------------------------------------------------------------------
struct StridedView {
    int32_t rank;
    int64_t dims[8];
    int64_t strides[8];
};

template <typename T>
__global__ __launch_bounds__(256) void k_strided_copy(const T *__restrict__ x, T *__restrict__ y, int64_t n,
                                                      StridedView v) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        int64_t r = i, off = 0;
        for (int d = v.rank - 1; d >= 0; d--) {
            off += (r % v.dims[d]) * v.strides[d];
            r /= v.dims[d];
        }
        y[i] = x[off];
    }
}

hipError_t launch_strided_copy(int esize, const void *x, void *y, int rank, const int64_t *dims, const int64_t *strides,
                               hipStream_t s) {
    StridedView v;
    v.rank = rank;
    int64_t n = 1;
    for (int d = 0; d < rank; d++) {
        v.dims[d] = dims[d];
        v.strides[d] = strides[d];
        n *= dims[d];
    }
    if (n == 0) return hipSuccess;
    int64_t g = (n + 255) / 256;
    if (g > 65536) g = 65536;
    if (esize == 4)
        hipLaunchKernelGGL(k_strided_copy<uint32_t>, dim3((unsigned)g), dim3(256), 0, s, (const uint32_t *)x, (uint32_t *)y, n, v);
    else if (esize == 8)
        hipLaunchKernelGGL(k_strided_copy<uint64_t>, dim3((unsigned)g), dim3(256), 0, s, (const uint64_t *)x, (uint64_t *)y, n, v);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

// VEC: 16-byte loads of A and B and 16-byte epilogue accesses of C, the residual and the bias
static bool f32_vec(const void *a, const void *b, const void *c, const MatMulArgs &p) {
    bool vec = (p.k % 4 == 0) && (p.n % 4 == 0) &&
               (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c | (uintptr_t)p.res | (uintptr_t)p.bias) % 16 == 0) &&
               p.bias_bstr % 4 == 0 && p.lda % 4 == 0 && p.ldb % 4 == 0 && p.ldc % 4 == 0;
    for (int d = 0; d < p.nbatch; d++)
        vec = vec && (p.a_bstr[d] % 4 == 0) && (p.b_bstr[d] % 4 == 0) && (p.c_bstr[d] % 4 == 0);
    return vec;
}

// K ranges of a float product on the direct-load kernel's terms (16-byte operands, K a multiple of 64): with
// T tiles of 64x64 over the batch as it is launched (f32_tiles), the most ranges, each a whole number
// of passes of 64, that divide K / 64 into equal parts and keep T times the ranges within 256 blocks (one per
// CU); 1 when T alone reaches 128 or K is a single pass.  A product of few tiles otherwise leaves
// most CUs idle while its blocks each walk the whole of K ([8,1536] x [1536,384]: 6 blocks).  With
// split_per_matrix (T counts one matrix's tiles) a batch above kMatMulSplitBatch does not split.
static int f32_split(const MatMulArgs &p, bool vec) {
    if (!vec || p.k % 64 != 0) return 1;
    if (p.split_per_matrix && p.batch > kMatMulSplitBatch) return 1;
    const int64_t tiles = f32_tiles(p, false);
    if (tiles >= 128) return 1;
    const int steps = p.k / 64;
    int best = 1;
    for (int r = 2; r <= steps; r++)
        if (steps % r == 0 && tiles * r <= 256) best = r;
    return best;
}

bool matmul_ln_fusable(int dtype, const void *a, const void *b, const void *c, const MatMulArgs &p) {
    return dtype == kFloat && !p.gelu && !p.bt && p.n % 4 == 0 && p.n >= 256 && p.n <= 4096 &&
           matmul_part_bytes(dtype, a, b, c, p) > 0;
}

hipError_t launch_matmul_ln(const void *a, const void *b, void *y, const MatMulArgs &p0, const float *gamma,
                            const float *beta, float eps, hipStream_t s) {
    if (!matmul_ln_fusable(kFloat, a, b, y, p0) || !p0.part) return hipErrorInvalidValue;
    MatMulArgs p = p0;
    p.split = f32_split(p, f32_vec(a, b, y, p));
    launch_f32_parts((const float *)a, (const float *)b, (float *)y, p, s);
    const dim3 gr((unsigned)(p.batch * p.m));
    float *fy = (float *)y;
    switch ((p.n + 255) / 256) {
#define LX_MM_LN_CASE(NV) \
    case NV: hipLaunchKernelGGL(k_matmul_split_sum_ln<NV>, gr, dim3(64), 0, s, gamma, beta, eps, fy, p); break;
        LX_MM_LN_CASE(1) LX_MM_LN_CASE(2) LX_MM_LN_CASE(3) LX_MM_LN_CASE(4) LX_MM_LN_CASE(5) LX_MM_LN_CASE(6)
        LX_MM_LN_CASE(7) LX_MM_LN_CASE(8) LX_MM_LN_CASE(9) LX_MM_LN_CASE(10) LX_MM_LN_CASE(11) LX_MM_LN_CASE(12)
        LX_MM_LN_CASE(13) LX_MM_LN_CASE(14) LX_MM_LN_CASE(15) LX_MM_LN_CASE(16)
#undef LX_MM_LN_CASE
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

int64_t matmul_part_bytes(int dtype, const void *a, const void *b, const void *c, const MatMulArgs &p) {
    if (dtype != kFloat || p.m == 0 || p.n == 0 || p.batch == 0) return 0;
    const int r = f32_split(p, f32_vec(a, b, c, p));
    return r > 1 && !f32_small(a, b, c, p, r) ? (int64_t)r * p.batch * p.m * p.n * (int64_t)sizeof(float) : 0;
}

hipError_t launch_matmul(int dtype, const void *a, const void *b, void *c, const MatMulArgs &p0, hipStream_t s) {
    if (p0.m == 0 || p0.n == 0 || p0.batch == 0) return hipSuccess;
    // grid z holds at most 65535 batches: larger batch counts take several launches
    if (p0.batch > 65535) {
        for (int64_t b0 = 0; b0 < p0.batch; b0 += 65535) {
            MatMulArgs q = p0;
            q.batch_base = p0.batch_base + b0;
            q.batch = p0.batch - b0 < 65535 ? p0.batch - b0 : 65535;
            hipError_t e = launch_matmul(dtype, a, b, c, q, s);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    const MatMulArgs &p = p0;
    if (dtype == kFloat) {
        const bool vec = f32_vec(a, b, c, p);
        const float *fa = (const float *)a, *fb = (const float *)b;
        float *fc = (float *)c;
        const int split = f32_split(p, vec);
        if (f32_small(a, b, c, p, split)) {
            MatMulArgs q = p;
            q.split = split;
            launch_f32_small(fa, fb, fc, q, s);
            return hipGetLastError();
        }
        if (split > 1) {
            if (!p.part || p.bt) return hipErrorInvalidValue;  // the caller sizes it with matmul_part_bytes
            MatMulArgs q = p;
            q.split = split;
            launch_f32_split(fa, fb, fc, q, s);
            return hipGetLastError();
        }
        if (f32_b3(p, p.k)) {
            launch_f32_b3(fa, fb, fc, p, vec, s);
            return hipGetLastError();
        }
        // What f32_b3 leaves.  Block tile: among the tiles that give each of the 256 CUs two or more blocks (a lone block
        // per CU leaves its barrier and load latencies unhidden: measured 93 against 104 TF/s for
        // [4096,3072]x[3072,768]), the one whose busiest CU has the least work -- ceil(blocks / 256)
        // blocks, each costing its area over the tile's relative efficiency; 64x64 when none does
        struct Tile {
            int bm, bn;
            double eff;
        };
        // (eight-wave 256x128 / 128x256 tiles measured 129.6 against 126.3 TFLOP/s at 4096^3 and far
        // slower wherever they leave fewer than two blocks per CU: not worth a candidate)
        static const Tile cand[] = {{128, 128, 1.0}, {128, 96, 0.93}, {96, 128, 0.93},
                                    {128, 64, 0.85}, {64, 128, 0.85}, {64, 64, 0.65}};
        constexpr int kCand = (int)(sizeof(cand) / sizeof(cand[0]));
        int best = 5;
        double best_cost = 0;
        for (int i = 0; i < kCand; i++) {
            const int64_t blocks =
                (int64_t)((p.m + cand[i].bm - 1) / cand[i].bm) * ((p.n + cand[i].bn - 1) / cand[i].bn) * p.batch;
            if (blocks < 512) continue;
            const double cost = (double)((blocks + 255) / 256) * cand[i].bm * cand[i].bn / cand[i].eff;
            if (best == 5 || cost < best_cost) {
                best = i;
                best_cost = cost;
            }
        }
        // a short K (at most 64, attention scores): the epilogue outweighs the K loop, and 64x64 tiles run
        // faster than the large ones ([16,12,512,64]x[16,12,64,512]: 70 against 66 TFLOP/s)
        if (p.k <= 64) best = 5;
        // The direct-load kernel (K a multiple of 64, 16-byte aligned operands) for every shape but short K
        // (attention scores, K = 64: the register-staged kernel 81 against 78 TFLOP/s); both kernels sum in one
        // order, so the choice never changes a result.  Tile: the least cost, where a tile config that holds r
        // blocks per CU at once (its LDS and its occupancy hint) runs ceil(tiles / (256 r)) rounds, each as long
        // as min(r, tiles per CU) of its tiles, each costing its area over a measured efficiency.  128x128 runs
        // with at most two waves per SIMD (accumulators in AGPRs: 135 TFLOP/s at 4096^3 against 104 with them in
        // VGPRs for three waves), 128x96 with one or two, the smaller tiles with three or more.
        // N of at most 32 (the attention context of 32-wide heads): 128x32 tiles, four waves of 32x32
        // ([8,12,512,512]x[8,12,512,32]: 65 against 43 TFLOP/s for the register-staged kernel's 64x64)
        // (B by columns, p.bt: the register-staged kernel only, never split -- the host checks)
        if (!p.bt && vec && p.k % 64 == 0 && p.k > 64 && p.n <= 32 && p.m >= 64) {
            launch_f32_dl<128, 32, 4, 1, 1, 2>(fa, fb, fc, p, s);
            return hipGetLastError();
        }
        if (!p.bt && vec && p.k % 64 == 0 && p.k > 64 && p.n >= 64 && p.m >= 64) {
            struct DTile {
                int bm, bn, resident;
                double eff;
            };
            static const DTile dcand[] = {{128, 128, 2, 1.0}, {128, 96, 2, 0.9}, {64, 64, 4, 0.97}, {128, 64, 3, 0.95}};
            auto tiles_of = [&](const DTile &c) {
                return (int64_t)((p.m + c.bm - 1) / c.bm) * ((p.n + c.bn - 1) / c.bn) * p.batch;
            };
            int dt = 0;
            double bc = 0;
            for (int i = 0; i < 4; i++) {
                const int64_t tiles = tiles_of(dcand[i]);
                const int64_t rounds = (tiles + 256 * dcand[i].resident - 1) / (256 * dcand[i].resident);
                const int64_t per_cu = std::min<int64_t>(dcand[i].resident, (tiles + 255) / 256);
                const double cost = (double)(rounds * per_cu) * dcand[i].bm * dcand[i].bn / dcand[i].eff;
                if (i == 0 || cost < bc) {
                    dt = i;
                    bc = cost;
                }
            }
            switch (dt) {
            case 0: launch_f32_dl<128, 128, 2, 2, 1, 2>(fa, fb, fc, p, s); break;
            case 1: launch_f32_dl<128, 96, 4, 1, 1, 2>(fa, fb, fc, p, s); break;
            case 2: launch_f32_dl<64, 64, 2, 2, 3, 8>(fa, fb, fc, p, s); break;
            default: launch_f32_dl<128, 64, 2, 2, 3, 8>(fa, fb, fc, p, s); break;
            }
            return hipGetLastError();
        }
        switch (best) {
        case 0: launch_f32<128, 128, 2, 2>(fa, fb, fc, p, vec, s); break;
        case 1: launch_f32<128, 96, 4, 1>(fa, fb, fc, p, vec, s); break;
        case 2: launch_f32<96, 128, 1, 4>(fa, fb, fc, p, vec, s); break;
        case 3: launch_f32<128, 64, 2, 2>(fa, fb, fc, p, vec, s); break;
        case 4: launch_f32<64, 128, 2, 2>(fa, fb, fc, p, vec, s); break;
        default: launch_f32<64, 64, 2, 2>(fa, fb, fc, p, vec, s); break;
        }
    } else if (dtype == kDouble) {
        // the largest of 128x128, 64x64 and 32x32 tiles that gives every CU a block
        const double *da = (const double *)a, *db = (const double *)b;
        double *dc = (double *)c;
        auto tiles = [&](int t) { return (((int64_t)p.m + t - 1) / t) * (((int64_t)p.n + t - 1) / t) * p.batch; };
        if (tiles(128) >= 256) launch_f64<128, 128>(da, db, dc, p, s);
        else if (tiles(64) >= 256) launch_f64<64, 64>(da, db, dc, p, s);
        else launch_f64<32, 32>(da, db, dc, p, s);
    } else if (dtype == kInt32) {
        launch_i32((const int32_t *)a, (const int32_t *)b, (int32_t *)c, p, s);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace lx
