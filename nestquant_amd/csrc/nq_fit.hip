// Block-word fit of one refinement stage of the encoder (encode.encode_residual in torch; reference nq_encode.py:186-198,286-316,
// nq_decode.py:158-163): given the frozen base plane and the states of a refinement plane, the step size delta by least squares, the
// twelve block words around it, the cost of the values the decoder really produces with each of them, and the best one.
//
//   nq_fit_residual_k  r = target * sign - base value (fp64), its rms per unit, r / (rms / scale) as the trellis search's targets
//   nq_fit_delta_k     delta per unit and the twelve candidates
//   nq_fit_cost_k      cost of candidate c of unit u: sum of squared errors, or tr(Do E Da E^T) with the unit's metrics
//   nq_fit_pick_k      the first candidate of least cost; its values
//   nq_fit_pack_k      a plane as the decoder reads it, and its values as a matrix
//
// A unit is 16 x 128 weights, held as 8 rings of 256 (ring position order), 2048 values on one workgroup of 256 threads. In torch
// the same is about three hundred launches over a few hundred kilobytes per stage, with a synchronisation at each of the twelve
// masked updates: bound by the host. Here it is four launches bound by latency. Sums are fp64 in another order than torch's, which
// moves delta and the costs by about 1e-16 relative; values, candidates and the choice follow the same formulas.
#include "nq_decode.hpp"
#include "nq_host.hpp"

namespace nq {

constexpr int FIT_CAND = 12, UNIT = 2048;
constexpr double FIT_A = 1774.0 / 262144.0, FIT_K0 = 1024.0 * FIT_A - 2658.0 / 256.0;   // fp16 0x1eee, 1024 A + fp16 0xc931: value of byte sum 0

// index of element i of a unit in ring order (ring i / 256, position i % 256) -> row, column of the 16 x 128 unit
__device__ __forceinline__ void ring_to_unit(int i, int& row, int& col)
{
    const int g = i >> 8, p = i & 255, t4 = p >> 6, pp = (p & 63) >> 1, e = p & 1, t = pp >> 2, r = pp & 3;
    col = 16 * t + 2 * t4 + 8 * (r >> 1) + e; row = g + 8 * (r & 1);
}
__device__ __forceinline__ uint32_t byte_sum(uint32_t st) { return __builtin_amdgcn_sad_u8(st * HASH_MUL, 0u, 0u); }
__device__ __forceinline__ float sign_of(const float* sign, int u, int i) { return sign ? sign[u * 8 + (i >> 8)] : 1.f; }

// sum over the 256 threads of the block, in every thread
__device__ __forceinline__ double block_sum(double v, double* sh)
{
#pragma unroll
    for (int m = 32; m; m >>= 1) v += __shfl_xor(v, m);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

__global__ void __launch_bounds__(256) nq_fit_residual_k(const float* __restrict__ target, const float* __restrict__ sign, const int64_t* __restrict__ st_base,
                                                          const float* __restrict__ lut, double scale, float* __restrict__ out)
{
    __shared__ double sh[4];
    const int u = blockIdx.x, t = threadIdx.x;
    double r[8], s = 0.0;
#pragma unroll
    for (int q = 0; q < 8; ++q)
    {
        const int i = t + 256 * q;
        const size_t at = (size_t)u * UNIT + i;
        r[q] = (double)(target[at] * sign_of(sign, u, i)) - (double)lut[st_base[at] & 0xFFFF];
        s += r[q] * r[q];
    }
    const double rms = fmax(sqrt(block_sum(s, sh) / UNIT), 1e-12), s0 = rms / scale;
#pragma unroll
    for (int q = 0; q < 8; ++q) out[(size_t)u * UNIT + t + 256 * q] = (float)(r[q] / s0);
}

__global__ void __launch_bounds__(256) nq_fit_delta_k(const float* __restrict__ target, const float* __restrict__ sign, const int64_t* __restrict__ st_base,
                                                       const int64_t* __restrict__ st_res, const float* __restrict__ lut, double* delta, int* cand)
{
    __shared__ double sh[4];
    const int u = blockIdx.x, t = threadIdx.x;
    double num = 0.0, den = 0.0;
#pragma unroll
    for (int q = 0; q < 8; ++q)
    {
        const int i = t + 256 * q;
        const size_t at = (size_t)u * UNIT + i;
        const double r = (double)(target[at] * sign_of(sign, u, i)) - (double)lut[st_base[at] & 0xFFFF];
        const double a = FIT_A * (double)byte_sum((uint32_t)st_res[at]) + FIT_K0;
        num += a * r; den += a * a;
    }
    num = block_sum(num, sh); den = block_sum(den, sh);
    const double d = fmax(num / fmax(den, 1e-30), 0.0);
    if (t == 0) delta[u] = d;
    if (t < FIT_CAND)
    {   // Mb - 0 .. 3 below the largest Mb whose N / Mb nears delta, N - 1 .. N + 1; a word out of range is replaced by the first
        const int Mb0 = (int)fmin(fmax(floor(257.0 / (1.0 + d)), 1.0), 255.0);
        const int N0 = (int)fmin(rint(d * Mb0), (double)(257 - Mb0));
        const int Mb = max(Mb0 - t / 3, 1);
        const double Nd = rint(d * Mb) + (double)(t % 3 - 1);
        const bool ok = Nd >= 0.0 && Nd <= 255.0 && Mb + Nd <= 257.0;
        cand[u * FIT_CAND + t] = ok ? (Mb | (int)Nd << 8) : (Mb0 | min(N0, 255) << 8);
    }
}

// value of the fold with block word dw, before the ring's sign (bit-exact the decoder's)
__device__ __forceinline__ float fold_value(uint32_t Sb, uint32_t Sr, int dw, const FoldK& k)
{
    const uint32_t F = (((uint32_t)dw & 0xFFu) * Sb + ((uint32_t)dw >> 8) * Sr + 128u) >> 8;
    const uint32_t h = pk_fma((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(float)(1024u + F)), k.A2, k.C2);
    return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}

// grid (FIT_CAND, U)
__global__ void __launch_bounds__(256) nq_fit_cost_k(const float* __restrict__ target, const float* __restrict__ sign, const int64_t* __restrict__ st_base,
                                                      const int64_t* __restrict__ st_res, const int* __restrict__ cand, const double* __restrict__ Da, int64_t da_step,
                                                      const double* __restrict__ Do, int64_t do_step, double* cost)
{
    __shared__ double sh[4];
    __shared__ double E[16][128];
    const int u = blockIdx.y, t = threadIdx.x, dw = cand[u * FIT_CAND + blockIdx.x];
    const FoldK k = consts_fold((uint32_t)dw, 0u);
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < 8; ++q)
    {
        const int i = t + 256 * q;
        const size_t at = (size_t)u * UNIT + i;
        const float v = fold_value(byte_sum((uint32_t)st_base[at]), byte_sum((uint32_t)st_res[at]), dw, k) * sign_of(sign, u, i);
        const double e = (double)(target[at] - v);
        if (Da) { int row, col; ring_to_unit(i, row, col); E[row][col] = e; }
        else s += e * e;
    }
    if (Da)
    {   // thread: column j, rows 8 half .. + 7 of E Da
        __syncthreads();
        const double* D = Da + (size_t)u * da_step;
        const int j = t & 127, half = t >> 7;
        double acc[8] = {};
        for (int kk = 0; kk < 128; ++kk)
        {
            const double d = D[kk * 128 + j];
#pragma unroll
            for (int q = 0; q < 8; ++q) acc[q] += E[8 * half + q][kk] * d;
        }
        if (!Do)
#pragma unroll
            for (int q = 0; q < 8; ++q) s += acc[q] * E[8 * half + q][j];
        else
        {   // (Do X) * E summed = X * (Do^T E) summed: no exchange of X
            const double* O = Do + (size_t)u * do_step;
#pragma unroll
            for (int q = 0; q < 8; ++q)
            {
                double w = 0.0;
                for (int r = 0; r < 16; ++r) w += O[r * 16 + 8 * half + q] * E[r][j];
                s += acc[q] * w;
            }
        }
    }
    s = block_sum(s, sh);
    if (t == 0) cost[u * FIT_CAND + blockIdx.x] = s;
}

__global__ void __launch_bounds__(256) nq_fit_pick_k(const float* __restrict__ sign, const int64_t* __restrict__ st_base, const int64_t* __restrict__ st_res,
                                                      const int* __restrict__ cand, const double* __restrict__ cost, float* Q, int64_t* Mb, int64_t* N)
{
    const int u = blockIdx.x, t = threadIdx.x;
    int b = 0;
    for (int c = 1; c < FIT_CAND; ++c) if (cost[u * FIT_CAND + c] < cost[u * FIT_CAND + b]) b = c;
    const int dw = cand[u * FIT_CAND + b];
    const FoldK k = consts_fold((uint32_t)dw, 0u);
#pragma unroll
    for (int q = 0; q < 8; ++q)
    {
        const int i = t + 256 * q;
        const size_t at = (size_t)u * UNIT + i;
        Q[at] = fold_value(byte_sum((uint32_t)st_base[at]), byte_sum((uint32_t)st_res[at]), dw, k) * sign_of(sign, u, i);
    }
    if (t == 0) { Mb[u] = dw & 0xFF; N[u] = dw >> 8; }
}

// What a fit hands out for one plane, one unit per workgroup: the states' new bits as lane records, the block words, the ring signs as a
// byte, and the values as a matrix (from the codebook, or given in ring order). In torch some forty launches a plane, and the check of
// the ring, which stops the host, in each: three planes of a 128 x 256 weight took 0.96 ms. A ring is whole if every state's upper bits are the
// next one's lower bits; the first that is not sets *bad, which the host reads once for all planes.
struct PackArgs
{
    const int64_t* st; const float* values; const float* sign; const float* lut; const int64_t* Mb; const int64_t* N;
    int32_t* words; int32_t* dw; uint8_t* var; float* Q; int32_t* bad; int K, C;
};
__global__ void __launch_bounds__(256) nq_fit_pack_k(PackArgs a)
{
    __shared__ uint16_t st[8][256];
    __shared__ float tile[16][129];
    const int u = blockIdx.x, t = threadIdx.x, K = a.K;
    const size_t u0 = (size_t)u * UNIT;
    int whole = 1;
#pragma unroll
    for (int g = 0; g < 8; ++g)
    {
        const int64_t s = a.st[u0 + g * 256 + t];
        whole &= s >= 0 && s < 65536;
        st[g][t] = (uint16_t)s;
    }
    __syncthreads();
    for (int g = 0; g < 8; ++g)
    {
        const uint32_t s = st[g][t];
        whole &= (s >> K) == (st[g][(t + 1) & 255] & (0xFFFFu >> K));
        if (!a.Q) continue;
        int row, col;
        ring_to_unit(g * 256 + t, row, col);
        tile[row][col] = a.values ? a.values[u0 + g * 256 + t] : a.lut[s] * sign_of(a.sign, u, g * 256);
    }
    if (!whole) *a.bad = 1;
    const int per = 32 / K, ring_words = 8 * K;                  // steps of a word, words of a ring (four records of 2 K)
    for (int w = t; w < 8 * ring_words; w += 256)
    {
        const int g = w / ring_words, p0 = (w - g * ring_words) * per;
        uint32_t v = 0;
        for (int j = 0; j < per; ++j) v |= (st[g][p0 + j] & ((1u << K) - 1u)) << (K * j);
        a.words[(size_t)u * 8 * ring_words + w] = (int32_t)v;
    }
    if (t == 0 && a.dw) a.dw[u] = (int32_t)(uint32_t)(a.Mb[u] | a.N[u] << 8);
    if (t == 0 && a.var)
    {
        uint32_t m = 0;
        for (int g = 0; g < 8; ++g) m |= (a.sign[u * 8 + g] < 0.f ? 1u : 0u) << g;
        a.var[u] = (uint8_t)m;
    }
    if (!a.Q) return;
    __syncthreads();
    const size_t cols = (size_t)a.C * 128, at = (size_t)(u / a.C) * 16 * cols + (size_t)(u % a.C) * 128;
    for (int i = t; i < UNIT; i += 256) a.Q[at + (i >> 7) * cols + (i & 127)] = tile[i >> 7][i & 127];
}
int launch_fit_pack(const int64_t* st, int K, const float* values, const float* sign, const float* lut, const int64_t* Mb, const int64_t* N, int U, int C,
                    int32_t* words, int32_t* dw, uint8_t* var, float* Q, int32_t* bad, hipStream_t s)
{
    nq_fit_pack_k<<<U, 256, 0, s>>>(PackArgs{st, values, sign, lut, Mb, N, words, dw, var, Q, bad, K, C});
    NQ_LAUNCH_CHECK("nq_fit_pack");
    return 0;
}

int launch_fit_residual(const float* target, const float* sign, const int64_t* st_base, const float* lut, double scale, int U, float* out, hipStream_t st)
{
    nq_fit_residual_k<<<U, 256, 0, st>>>(target, sign, st_base, lut, scale, out);
    NQ_LAUNCH_CHECK("nq_fit_residual");
    return 0;
}

int launch_fit_words(const float* target, const float* sign, const int64_t* st_base, const int64_t* st_res, const float* lut, int U, const double* Da, int64_t da_step,
                     const double* Do, int64_t do_step, void* ws, float* Q, int64_t* Mb, int64_t* N, double* delta, hipStream_t st)
{
    double* cost = (double*)ws;
    int* cand = (int*)(cost + (size_t)U * FIT_CAND);
    nq_fit_delta_k<<<U, 256, 0, st>>>(target, sign, st_base, st_res, lut, delta, cand);
    nq_fit_cost_k<<<dim3(FIT_CAND, U), 256, 0, st>>>(target, sign, st_base, st_res, cand, Da, da_step, Do, do_step, cost);
    nq_fit_pick_k<<<U, 256, 0, st>>>(sign, st_base, st_res, cand, cost, Q, Mb, N);
    NQ_LAUNCH_CHECK("nq_fit_words");
    return 0;
}

}  // namespace nq
