// What an encode does before, between and after its trellis searches, in kernels of its own: in torch these are a hundred and fifty launches over a few
// hundred kilobytes for a fit that knows its inputs, which left the GPU idle for two fifths of it (encode.py holds the same steps in torch, for the CPU).
//
//   nq_enc_cols_k, nq_enc_rows_k   per-channel scales of a weight (encode.prepare)
//   nq_enc_rotate_k    scales out or in, Hadamard-128 on both sides: a weight's targets, also in ring order; an input second moment
//   nq_enc_inverse_k   inverse of a 128 x 128 diagonal block, for the block LDL factors (encode._block_ldl_gpu)
//   nq_enc_targets_k   one column chunk's targets of every level from the weight and what the later chunks feed back, in ring order
//   nq_enc_base_k      the searched base plane of a chunk: the better orientation of each ring, its errors
//   nq_enc_feed_k      a fitted refinement plane of a chunk, its errors
//
// Arithmetic is fp64 throughout, as there; sums are taken in another order, which moves results by about 1e-16 relative.
#include "nq_decode.hpp"
#include "nq_host.hpp"

namespace nq {

constexpr int ENC_UNIT = 2048;

// element (row, col) of a 16 x 128 unit -> its index in ring order (ring g = index / 256)
__device__ __forceinline__ int unit_to_ring(int row, int col)
{
    const int cc = col & 15;
    return (row & 7) * 256 + ((cc >> 1) & 3) * 64 + 2 * (4 * (col >> 4) + (row >> 3) + 2 * (cc >> 3)) + (cc & 1);
}
__device__ __forceinline__ void ring_to_unit_at(int i, int& row, int& col)
{
    const int g = i >> 8, p = i & 255, t4 = p >> 6, pp = (p & 63) >> 1, e = p & 1, t = pp >> 2, r = pp & 3;
    col = 16 * t + 2 * t4 + 8 * (r >> 1) + e; row = g + 8 * (r & 1);
}

__device__ __forceinline__ double enc_scale(double mean)         // a channel's scale; NaN stays NaN
{
    const double v = sqrt(mean);
    return v < 1e-12 ? 1e-12 : v;
}

// grid (K / 16), block 1024 = 64 row lanes x 16 columns: c[k] = max(sqrt(mean of W[:, k]^2), 1e-12), su = fp16(sign * c)
__global__ void __launch_bounds__(1024) nq_enc_cols_k(const float* __restrict__ W, int N, int K, const int64_t* __restrict__ sgn, double* c, _Float16* su)
{
    __shared__ double sh[64][17];
    const int col = threadIdx.x & 15, lane = threadIdx.x >> 4, k = blockIdx.x * 16 + col;
    double s = 0.0;
    for (int n = lane; n < N; n += 64) { const double v = (double)W[(size_t)n * K + k]; s += v * v; }
    sh[lane][col] = s;
    for (int m = 32; m; m >>= 1)
    {
        __syncthreads();
        if (lane < m) sh[lane][col] += sh[lane + m][col];
    }
    if (lane == 0)
    {
        const double v = enc_scale(sh[0][col] / N);
        c[k] = v;
        su[k] = (_Float16)(float)(sgn[k] ? v : -v);
    }
}

// grid (N), block 256: sv[n] = fp16(sign * max(sqrt(mean of (W[n, :] / c)^2), 1e-12))
__global__ void __launch_bounds__(256) nq_enc_rows_k(const float* __restrict__ W, int K, const double* __restrict__ c, const int64_t* __restrict__ sgn, _Float16* sv)
{
    __shared__ double sh[4];
    const int n = blockIdx.x;
    double s = 0.0;
    for (int k = threadIdx.x; k < K; k += 256) { const double v = (double)W[(size_t)n * K + k] / c[k]; s += v * v; }
#pragma unroll
    for (int m = 32; m; m >>= 1) s += __shfl_xor(s, m);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0)
    {
        const double v = enc_scale(((sh[0] + sh[1]) + (sh[2] + sh[3])) / K);
        sv[n] = (_Float16)(float)(sgn[n] ? v : -v);
    }
}

// Hadamard over 128 elements, thread part q = lane & 3 holding elements 32 q + i in v[i]; not scaled
__device__ __forceinline__ void had128_parts(double* v, int q)
{
#pragma unroll
    for (int d = 1; d < 32; d <<= 1)
#pragma unroll
        for (int i = 0; i < 32; ++i)
            if (!(i & d)) { const double a = v[i], b = v[i + d]; v[i] = a + b; v[i + d] = a - b; }
#pragma unroll
    for (int m = 1; m < 4; m <<= 1)
#pragma unroll
        for (int i = 0; i < 32; ++i) { const double o = __shfl_xor(v[i], m); v[i] = (q & m) ? o - v[i] : v[i] + o; }
}

// A 128 x 128 tile of X, rows and columns scaled, times the orthonormal Hadamard on both sides; grid (columns / 128, rows / 128), block 512: four
// threads per row, then, through LDS, per column. WEIGHT: X fp32 divided by su[col] and sv[row] -> fp32 matrix and, if given, rings (T of
// them, units of 16 x 128 by strips) and once more negated; else X fp64 multiplied by su[row] and su[col] -> fp64 matrix.
// The scale is the codebase's fp32 value of 1 / sqrt(128) on each side. Bound by latency: 8 tiles 9 us.
template <bool WEIGHT>
__global__ void __launch_bounds__(512) nq_enc_rotate_k(const void* __restrict__ X, const _Float16* __restrict__ su, const _Float16* __restrict__ sv, int K,
                                                        void* out, float* rings, int64_t negated)
{
    extern __shared__ __align__(16) double enc_tile[];           // [128][129]
    const int line = threadIdx.x >> 2, q = threadIdx.x & 3, c0 = blockIdx.x * 128, r0 = blockIdx.y * 128;
    const double h = (double)(1.0f / 11.313708498984761f), scale = h * h;
    double v[32];
    {
        const size_t at = (size_t)(r0 + line) * K + c0 + 32 * q;
        const double rs = (double)(WEIGHT ? sv : su)[r0 + line];
#pragma unroll
        for (int i = 0; i < 32; ++i)
        {
            const double cs = (double)su[c0 + 32 * q + i];
            if constexpr (WEIGHT) v[i] = (double)((const float*)X)[at + i] / cs / rs;
            else v[i] = ((const double*)X)[at + i] * rs * cs;
        }
    }
    had128_parts(v, q);
#pragma unroll
    for (int i = 0; i < 32; ++i) enc_tile[line * 129 + 32 * q + i] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 32; ++i) v[i] = enc_tile[(32 * q + i) * 129 + line];
    had128_parts(v, q);
#pragma unroll
    for (int i = 0; i < 32; ++i)
    {
        const int row = 32 * q + i;
        const double o = v[i] * scale;
        const size_t at = (size_t)(r0 + row) * K + c0 + line;
        if constexpr (WEIGHT)
        {
            const float f = (float)o;
            ((float*)out)[at] = f;
            if (rings)
            {
                const size_t u = ((size_t)((r0 + row) >> 4) * (K / 128) + blockIdx.x) * ENC_UNIT + unit_to_ring(row & 15, line);
                rings[u] = f;
                if (negated) rings[u + negated] = -f;
            }
        }
        else ((double*)out)[at] = o;
    }
}

int launch_enc_prepare(const float* W, int N, int K, const int64_t* sgn, double* c, void* su, void* sv, float* target, float* rings, int negated, hipStream_t st)
{
    const int shm = 128 * 129 * 8;
    const hipError_t e = hipFuncSetAttribute((const void*)nq_enc_rotate_k<true>, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
    if (e != hipSuccess) return set_error("nq_enc_prepare: LDS %d bytes: %s", shm, hipGetErrorString(e));
    nq_enc_cols_k<<<K / 16, 1024, 0, st>>>(W, N, K, sgn, c, (_Float16*)su);
    nq_enc_rows_k<<<N, 256, 0, st>>>(W, K, c, sgn + K, (_Float16*)sv);
    nq_enc_rotate_k<true><<<dim3(K / 128, N / 128), 512, shm, st>>>(W, (const _Float16*)su, (const _Float16*)sv, K, target, rings, negated ? (int64_t)N * K : 0);
    NQ_LAUNCH_CHECK("nq_enc_prepare");
    return 0;
}

int launch_enc_hessian(const double* H, int K, const void* su, double* out, hipStream_t st)
{
    const int shm = 128 * 129 * 8;
    const hipError_t e = hipFuncSetAttribute((const void*)nq_enc_rotate_k<false>, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
    if (e != hipSuccess) return set_error("nq_enc_hessian: LDS %d bytes: %s", shm, hipGetErrorString(e));
    nq_enc_rotate_k<false><<<dim3(K / 128, K / 128), 512, shm, st>>>(H, (const _Float16*)su, nullptr, K, out, nullptr, 0);
    NQ_LAUNCH_CHECK("nq_enc_hessian");
    return 0;
}

// Inverse of a symmetric positive definite 128 x 128 matrix (rows lda apart) by Gauss-Jordan steps without exchanges, whose pivots are those of
// its LDL^T: one that is not positive sets *bad (if not set yet) to order0 + its number + 1. One workgroup, a 4 x 4 patch per thread in registers; a step's row and
// column pass through LDS. Bound by 128 steps of one barrier each.
__global__ void __launch_bounds__(1024) nq_enc_inverse_k(const double* __restrict__ A, int lda, double* out, int32_t* bad, int order0)
{
    __shared__ double row_s[2][128], col_s[2][128];
    const int ty = threadIdx.x >> 5, tx = threadIdx.x & 31;
    double a[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) a[i][j] = A[(size_t)(4 * ty + i) * lda + 4 * tx + j];
    int failed = 0;
    for (int k4 = 0; k4 < 32; ++k4)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
        {
            const int k = 4 * k4 + kk, b = kk & 1;
            if (ty == k4)
#pragma unroll
                for (int j = 0; j < 4; ++j) row_s[b][4 * tx + j] = a[kk][j];
            if (tx == k4)
#pragma unroll
                for (int i = 0; i < 4; ++i) col_s[b][4 * ty + i] = a[i][kk];
            __syncthreads();
            const double p = row_s[b][k], ip = 1.0 / p;
            if (!failed && !(p > 0.0)) failed = k + 1;
            double r[4], c[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) r[j] = row_s[b][4 * tx + j] * ip;
#pragma unroll
            for (int i = 0; i < 4; ++i) c[i] = col_s[b][4 * ty + i];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    const bool on_row = 4 * ty + i == k, on_col = 4 * tx + j == k;
                    a[i][j] = on_row ? (on_col ? ip : r[j]) : on_col ? -c[i] * ip : a[i][j] - c[i] * r[j];
                }
        }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) out[(4 * ty + i) * 128 + 4 * tx + j] = a[i][j];
    if (threadIdx.x == 0 && failed && *bad == 0) *bad = order0 + failed;
}
int launch_enc_inverse(const double* A, int lda, double* out, int32_t* bad, int order0, hipStream_t st)
{
    nq_enc_inverse_k<<<1, 1024, 0, st>>>(A, lda, out, bad, order0);
    NQ_LAUNCH_CHECK("nq_enc_inverse");
    return 0;
}

// grid (strips), block 256: one column chunk (columns col0 .. + 127) of every strip. T_l = W + fed_l (fed: fp64 [levels][rows][128], null for the first chunk);
// mix: rings of (1 - lam) T_0 + lam T_1 (and negated `negated` floats further on), else rings of T_0 alone. T: fp64 [levels][rows][128], kept for the errors.
__global__ void __launch_bounds__(256) nq_enc_targets_k(const float* __restrict__ W, int K, int col0, const double* __restrict__ fed, int levels, double lam, int mix,
                                                         int N, double* T, float* rings, int64_t negated)
{
    const int s = blockIdx.x;
    for (int i = threadIdx.x; i < ENC_UNIT; i += 256)
    {
        const int row = 16 * s + (i >> 7), col = i & 127;
        const double w = (double)W[(size_t)row * K + col0 + col];
        double t[2] = {w, w};
#pragma unroll
        for (int l = 0; l < 2; ++l)
            if (l < levels)
            {
                const size_t at = ((size_t)l * N + row) * 128 + col;
                if (fed) t[l] = w + fed[at];
                T[at] = t[l];
            }
        const size_t r = (size_t)s * ENC_UNIT + unit_to_ring(row & 15, col);
        auto put = [&](float* p, double v) { p[r] = (float)v; };
        if (mix)
        {
            const float f = (float)((1.0 - lam) * t[0] + lam * t[1]);
            rings[r] = f;
            if (negated) rings[r + negated] = -f;
            put(rings + (negated ? 2 : 1) * (size_t)N * 128, t[1]);
        }
        else put(rings, t[0]);
    }
}
int launch_enc_targets(const float* W, int N, int K, int col0, const double* fed, int levels, double lam, int mix, double* T, float* rings, int negated, hipStream_t st)
{
    nq_enc_targets_k<<<N / 16, 256, 0, st>>>(W, K, col0, fed, levels, lam, mix, N, T, rings, negated ? (int64_t)N * 128 : 0);
    NQ_LAUNCH_CHECK("nq_enc_targets");
    return 0;
}

// grid (strips), block 256 = thread per ring position: the searched base plane of chunk `chunk`. st: the rings' states and, with var, those of the
// negated rings `T` further on; of the two the one with the smaller squared error stays (the first of equals). Values with the ring's sign: errors
// against the weight (err) and against the chunk's own target T0 (eta), fp64 [rows][K] at col0; states and signs by strip, and in their place
// of all units. W null: the choice alone, own and sign.
__global__ void __launch_bounds__(256) nq_enc_base_k(const int64_t* __restrict__ st, int64_t T, int var, const float* __restrict__ rings, const float* __restrict__ lut,
                                                      const float* __restrict__ W, const double* __restrict__ T0, int K, int chunk, int64_t* own, float* sign,
                                                      int64_t* st_all, float* sign_all, double* err, double* eta)
{
    __shared__ double sh[8][4][2];
    const int s = blockIdx.x, p = threadIdx.x, lane = p & 63, warp = p >> 6, C = K / 128;
    int64_t st0[8], st1[8];
#pragma unroll
    for (int g = 0; g < 8; ++g)
    {
        const size_t at = (size_t)s * ENC_UNIT + g * 256 + p;
        st0[g] = st[at]; st1[g] = 0;
        if (!var) continue;
        st1[g] = st[at + T * 256];
        const float x = rings[at], d0 = lut[st0[g] & 0xFFFF] - x, d1 = lut[st1[g] & 0xFFFF] + x;
        double e0 = (double)(d0 * d0), e1 = (double)(d1 * d1);
#pragma unroll
        for (int m = 32; m; m >>= 1) { e0 += __shfl_xor(e0, m); e1 += __shfl_xor(e1, m); }
        if (lane == 0) { sh[g][warp][0] = e0; sh[g][warp][1] = e1; }
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < 8; ++g)
    {
        float sg = 1.f;
        if (var)
        {
            const double e0 = (sh[g][0][0] + sh[g][1][0]) + (sh[g][2][0] + sh[g][3][0]), e1 = (sh[g][0][1] + sh[g][1][1]) + (sh[g][2][1] + sh[g][3][1]);
            if (e1 < e0) { sg = -1.f; st0[g] = st1[g]; }
        }
        const int i = g * 256 + p;
        const size_t unit = (size_t)s * C + chunk;
        own[(size_t)s * ENC_UNIT + i] = st0[g];
        if (p == 0) sign[s * 8 + g] = sg;
        if (!W) continue;                                        // the choice alone
        st_all[unit * ENC_UNIT + i] = st0[g];
        if (p == 0) sign_all[unit * 8 + g] = sg;
        int row, col;
        ring_to_unit_at(i, row, col);
        row += 16 * s;
        const size_t at = (size_t)row * K + chunk * 128 + col;
        const double q = (double)(lut[st0[g] & 0xFFFF] * sg);
        err[at] = (double)W[at] - q;
        eta[at] = T0[(size_t)row * 128 + col] - q;
    }
}
int launch_enc_base(const int64_t* st, int N, int var, const float* rings, const float* lut, const float* W, const double* T0, int K, int chunk, int64_t* own, float* sign,
                    int64_t* st_all, float* sign_all, double* err, double* eta, hipStream_t s)
{
    nq_enc_base_k<<<N / 16, 256, 0, s>>>(st, (int64_t)N / 2, var, rings, lut, W, T0, K, chunk, own, sign, st_all, sign_all, err, eta);
    NQ_LAUNCH_CHECK("nq_enc_base");
    return 0;
}

// grid (strips), block 256: a refinement plane fitted to chunk `chunk` (states, values Q in ring order, block words) to its place among all units, and
// its errors as in nq_enc_base_k
__global__ void __launch_bounds__(256) nq_enc_feed_k(const int64_t* __restrict__ st, const float* __restrict__ Q, const int64_t* __restrict__ Mb, const int64_t* __restrict__ Nw,
                                                      const float* __restrict__ W, const double* __restrict__ T0, int K, int chunk, int64_t* st_all, float* Q_all,
                                                      int64_t* Mb_all, int64_t* N_all, double* err, double* eta)
{
    const int s = blockIdx.x, C = K / 128;
    const size_t unit = (size_t)s * C + chunk;
    for (int i = threadIdx.x; i < ENC_UNIT; i += 256)
    {
        const size_t from = (size_t)s * ENC_UNIT + i;
        const float q = Q[from];
        st_all[unit * ENC_UNIT + i] = st[from];
        Q_all[unit * ENC_UNIT + i] = q;
        int row, col;
        ring_to_unit_at(i, row, col);
        row += 16 * s;
        const size_t at = (size_t)row * K + chunk * 128 + col;
        err[at] = (double)W[at] - (double)q;
        eta[at] = T0[(size_t)row * 128 + col] - (double)q;
    }
    if (threadIdx.x == 0) { Mb_all[unit] = Mb[s]; N_all[unit] = Nw[s]; }
}
int launch_enc_feed(const int64_t* st, const float* Q, const int64_t* Mb, const int64_t* Nw, const float* W, const double* T0, int N, int K, int chunk, int64_t* st_all, float* Q_all,
                    int64_t* Mb_all, int64_t* N_all, double* err, double* eta, hipStream_t s)
{
    nq_enc_feed_k<<<N / 16, 256, 0, s>>>(st, Q, Mb, Nw, W, T0, K, chunk, st_all, Q_all, Mb_all, N_all, err, eta);
    NQ_LAUNCH_CHECK("nq_enc_feed");
    return 0;
}

}  // namespace nq
