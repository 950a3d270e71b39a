// Decode salience export, the part shared by its own launch (nq_sal.hip) and the routing launch of a layer call (nq_moe.hip):
// sal[e] += sum over the picks (t, k) of expert e of (rsf * w[t][k])^2 * |x[t]|^2, a running fp64 sum per expert on the device,
// every touched entry mirrored to host-mapped memory (reference sm120/nqsal.cu:19-78).
//
// One workgroup of NW wavefronts; its threads walk every token's row together in 16-byte steps (eight fp16 / bf16 values, or four
// fp32 values rounded through fp16), so that a row is two or three loads per thread, all in flight at once; the lane sums meet in a
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
// squares of the values of one 16-byte step, added to s
__device__ __forceinline__ float sal_sq16(uint4 u, int dt, float s)
{
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int q = 0; q < 4; ++q)
    {
        if (dt == 2) { const float f = (float)(_Float16)__builtin_bit_cast(float, w[q]); s = __builtin_fmaf(f, f, s); continue; }
        const float lo = dt == 0 ? (float)__builtin_bit_cast(_Float16, (uint16_t)w[q]) : bf16_to_f((uint16_t)w[q]);
        const float hi = dt == 0 ? (float)__builtin_bit_cast(_Float16, (uint16_t)(w[q] >> 16)) : bf16_to_f((uint16_t)(w[q] >> 16));
        s = __builtin_fmaf(hi, hi, __builtin_fmaf(lo, lo, s));
    }
    return s;
}

template <int NW>
__device__ __forceinline__ void salience(const SalArgs& a, SalShared* S)
{
    const int tid = threadIdx.x, lane = tid & 63, warp = tid >> 6;
    const int esz = a.x_dtype == 2 ? 4 : 2, per = 16 / esz;
    for (int t = 0; t < a.T; ++t)
    {
        const char* row = (const char*)a.x + (int64_t)t * a.sx * esz;
        float s = 0.f;
        int done = 0;
        if (((uintptr_t)row & 15) == 0)
        {
            const int nv = a.H / per;
#pragma unroll 4
            for (int i = tid; i < nv; i += 64 * NW) s = sal_sq16(((const uint4*)row)[i], a.x_dtype, s);
            done = nv * per;
        }
        for (int i = done + tid; i < a.H; i += 64 * NW) { const float f = sal_elem(row, i, a.x_dtype); s = __builtin_fmaf(f, f, s); }   // rest, or a row off 16-byte alignment
#pragma unroll
        for (int m = 32; m; m >>= 1) s += __shfl_xor(s, m);
        if (lane == 0) S->part[warp][t] = s;
    }
    __syncthreads();
    if (warp != 0) return;
    const int n = a.T * a.K;                                        // <= 64: one pick per lane
    int e = -1; double term = 0.0;
    if (lane < n)
    {
        const float wf = (float)(_Float16)sal_elem(a.w, lane, a.w_dtype);
        const long long id = id_at(a.ids, a.ids_dtype, lane);
        if (wf != 0.f && id >= 0 && id < a.E)                       // weight 0 or an id outside the table: skipped, as the hit counters do
        {
            e = (int)id;
            float norm2 = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) norm2 += S->part[w][lane / a.K];
            const double ww = (double)(wf * a.rsf);
            term = ww * ww * (double)norm2;
        }
    }
    S->e[lane] = e; S->term[lane] = term;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (e < 0) return;
    double tot = 0.0; bool first = true;
    for (int j = 0; j < n; ++j)
        if (S->e[j] == e) { tot += S->term[j]; first = first && j >= lane; }
    if (first) { const double v = a.acc[e] + tot; a.acc[e] = v; a.host[e] = v; }
}

}  // namespace nq
