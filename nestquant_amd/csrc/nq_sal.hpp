// Decode salience export, the part shared by its own launch (nq_sal.hip) and the routing launch of a layer call (nq_moe.hip):
// sal[e] += sum over the picks (t, k) of expert e of (rsf * w[t][k])^2 * |x[t]|^2, a running fp64 sum per expert on the device,
// every touched entry mirrored to host-mapped memory (reference sm120/nqsal.cu:19-78).
//
// One workgroup of NW wavefronts, NW / T of them (at least one) on a token's row, the rows side by side; a row is walked in 16-byte
// steps (eight fp16 / bf16 values, or four fp32 values rounded through fp16), several in flight per lane; the lane sums meet in a
// butterfly and the wavefront sums through LDS, in a fixed order. The picks are then the lanes of wavefront 0: each adds the fp64
// terms of its expert in pick order from LDS (independent reads, no chain of lane exchanges), and the expert's first pick
// updates the accumulator (calls on one layer are stream-ordered, so no atomics). The squared norm is an fp32 sum (about 1e-6
// relative at H = 6144); weights pass through fp16 as the caller's cast would leave them.
#pragma once
#include "nq_tile.hpp"

namespace nq {

struct SalArgs
{
    const void* x; int64_t sx; const void* w; const void* ids;
    int T, H, K, E; int x_dtype, w_dtype, ids_dtype;       // x / w: 0 f16, 1 bf16, 2 f32 (rounded through fp16); ids: 0 i64, 1 i32
    float rsf; double* acc; double* host;
};
struct SalShared { float part[16][8]; double term[64]; int e[64]; };

__device__ __forceinline__ float sal_elem(const void* p, int64_t i, int dt)
{
    if (dt == 0) return (float)((const _Float16*)p)[i];
    if (dt == 1) return bf16_to_f(((const uint16_t*)p)[i]);
    return (float)(_Float16)((const float*)p)[i];
}
// sum of the squares of a lane's share of a row: 16-byte steps thr, thr + nthr, .. of nv, twelve in flight
template <int DT>
__device__ __forceinline__ float sal_row(const uint4* row, int nv, int thr, int nthr)
{
    float s = 0.f;
    for (int i0 = thr; i0 < nv; i0 += 12 * nthr)
    {
        uint4 v[12];
#pragma unroll
        for (int u = 0; u < 12; ++u) v[u] = i0 + u * nthr < nv ? row[i0 + u * nthr] : make_uint4(0u, 0u, 0u, 0u);   // zero bits are 0.0 in all three types
#pragma unroll
        for (int u = 0; u < 12; ++u)
        {
            const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
            for (int q = 0; q < 4; ++q)
            {
                if constexpr (DT == 2) { const float f = (float)(_Float16)__builtin_bit_cast(float, w[q]); s = __builtin_fmaf(f, f, s); }
                else
                {
                    const float lo = DT == 0 ? (float)__builtin_bit_cast(_Float16, (uint16_t)w[q]) : bf16_to_f((uint16_t)w[q]);
                    const float hi = DT == 0 ? (float)__builtin_bit_cast(_Float16, (uint16_t)(w[q] >> 16)) : bf16_to_f((uint16_t)(w[q] >> 16));
                    s = __builtin_fmaf(hi, hi, __builtin_fmaf(lo, lo, s));
                }
            }
        }
    }
    return s;
}

template <int NW>
__device__ __forceinline__ void salience(const SalArgs& a, SalShared* S)
{
    const int tid = threadIdx.x, lane = tid & 63, warp = tid >> 6, n = a.T * a.K;      // n <= 64: one pick per lane of wavefront 0
    int e = -1; float wf = 0.f; double old = 0.0;
    if (warp == 0 && lane < n)
    {   // the pick and the accumulator are requested before the rows, so that nothing is waited for after them
        wf = (float)(_Float16)sal_elem(a.w, lane, a.w_dtype);
        const long long id = id_at(a.ids, a.ids_dtype, lane);
        if (id >= 0 && id < a.E) { e = (int)id; old = a.acc[e]; }
        if (wf == 0.f) e = -1;                                      // weight 0 or an id outside the table: skipped, as the hit counters do
    }
    const int esz = a.x_dtype == 2 ? 4 : 2, per = 16 / esz;
    // as many wavefronts on a row as there are to spare, the rows side by side
    const int per_row = a.T >= NW ? 1 : NW / a.T, sub = warp % per_row, nthr = 64 * per_row, thr = sub * 64 + lane;
    for (int t = warp / per_row; t < a.T; t += NW / per_row)
    {
        const char* row = (const char*)a.x + (int64_t)t * a.sx * esz;
        float s = 0.f;
        int done = 0;
        if (((uintptr_t)row & 15) == 0)
        {
            const int nv = a.H / per;
            const uint4* r16 = (const uint4*)row;
            s = a.x_dtype == 0 ? sal_row<0>(r16, nv, thr, nthr) : a.x_dtype == 1 ? sal_row<1>(r16, nv, thr, nthr) : sal_row<2>(r16, nv, thr, nthr);
            done = nv * per;
        }
        for (int i = done + thr; i < a.H; i += nthr) { const float f = sal_elem(row, i, a.x_dtype); s = __builtin_fmaf(f, f, s); }   // rest, or a row off 16-byte alignment
#pragma unroll
        for (int m = 32; m; m >>= 1) s += __shfl_xor(s, m);
        if (lane == 0) S->part[sub][t] = s;
    }
    __syncthreads();
    if (warp != 0) return;
    double term = 0.0;
    if (e >= 0)
    {
        float norm2 = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) if (w < per_row) norm2 += S->part[w][lane / a.K];
        const double ww = (double)(wf * a.rsf);
        term = ww * ww * (double)norm2;
    }
    S->e[lane] = e; S->term[lane] = term;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    double tot = 0.0; bool first = true;
#pragma unroll 8
    for (int j = 0; j < n; ++j)
    {
        const bool same = S->e[j] == e;
        tot += same ? S->term[j] : 0.0;
        first = first && !(same && j < lane);
    }
    if (e >= 0 && first) { const double v = old + tot; a.acc[e] = v; a.host[e] = v; }
}

}  // namespace nq
