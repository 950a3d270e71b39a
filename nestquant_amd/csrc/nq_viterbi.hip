// Tail-biting trellis search of the encoder (the reference leaves it to CUDA kernels of its own; restated from the algorithm of
// threads/05-exl3-harness/harness.py:297-364): for every ring of L targets the path of least squared error through the 16-bit
// shift-register trellis with K = 1 or 2 new bits per step, in two passes -- pass 1, rolled by half a ring, finds the state that
// enters step 0; pass 2 starts from and ends in it. encode.viterbi_ring is the same search in torch, and the results are equal
// bit for bit: every candidate is (value - target)^2 + cost in fp32 with the torch code's roundings (no contraction), and ties go
// to the smallest predecessor.
//
// One workgroup of 1024 threads per ring. "Edge" = the low 16 - K bits of a state (E of them); the candidates of edge e are its
// 2^K states, each with predecessor edge (q << (16 - 2 K)) | (e >> K), so 2^K neighbouring edges (a group) share their
// predecessors: thread t owns the groups t + 1024 r, keeps the 64 codebook values of their states in registers through a
// pass, reads 2^K costs per group from LDS and writes 2^K. Both directions of that traffic are free of bank conflicts. The
// decisions of a thread in one step (16 edges x 2 bits, or 32 x 1) fill one word, stored to a scratch of 4 KB per step; the way
// back is walked by one lane over blocks of steps brought to LDS, the next block in flight.
// Bound: vector-instruction issue. A step is 65536 candidates of three fp32 operations plus the selection, ~21 instructions per
// four candidates (K = 2) = 340 per wavefront; with sixteen wavefronts per CU, one ring per CU.
#include "nq_host.hpp"

namespace nq {

constexpr int VT = 1024, VIT_LMAX = 1024;

struct VitArgs { const float* w; const float* lut; int64_t* st; uint32_t* back; int T, L, rev; };

// all wavefronts' LDS accesses so far are done; stores to global memory stay in flight (a __syncthreads would wait for them)
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// one step of the search: costs cur -> nxt (K = 1: the same array), decisions -> the returned word
template <int K>
__device__ __forceinline__ uint32_t vit_step(const float (&v)[64 >> (2 * K)][1 << K][1 << K], float wv, const float* cur, float* nxt, int t)
{
    constexpr int Q = 1 << K, R = 64 >> (2 * K), G = 1024 * R;
    float c[R][Q];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int q = 0; q < Q; ++q) c[r][q] = cur[q * G + t + 1024 * r];
    if constexpr (K == 1) lds_barrier();                         // one array: everybody has read before anybody writes
    uint32_t word = 0;
#pragma unroll
    for (int r = 0; r < R; ++r)
    {
        uint32_t m[Q];
#pragma unroll
        for (int j = 0; j < Q; ++j)
        {
            uint32_t x[Q];                                       // costs are >= +0: their bit patterns order as they do
#pragma unroll
            for (int q = 0; q < Q; ++q)
            {
                const float d = v[r][j][q] - wv;
                x[q] = __builtin_bit_cast(uint32_t, d * d + c[r][q]);
            }
            uint32_t i;
            if constexpr (K == 2)
            {
                const uint32_t m01 = x[1] < x[0] ? x[1] : x[0], m23 = x[3] < x[2] ? x[3] : x[2];
                const uint32_t i01 = x[1] < x[0] ? 1u : 0u, i23 = x[3] < x[2] ? 3u : 2u;
                m[j] = m23 < m01 ? m23 : m01; i = m23 < m01 ? i23 : i01;
            }
            else { m[j] = x[1] < x[0] ? x[1] : x[0]; i = x[1] < x[0] ? 1u : 0u; }
            word |= i << (K * (r * Q + j));
        }
        asm volatile("" : "+v"(word));                           // one group at a time: mixing them would not fit the registers
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (K == 2) *(uint4*)(nxt + 4 * (t + 1024 * r)) = make_uint4(m[0], m[1], m[2], m[3]);
        else *(uint2*)(nxt + 2 * (t + 1024 * r)) = make_uint2(m[0], m[1]);
    }
    return word;
}

// walk back over the rows hi .. 0 of the decisions: sl[row] = state at that row. back rows are 4 KB; 16 rows per block, the
// block after next requested while a lane walks. Returns (to thread 0) the edge entering row 0.
template <int K>
__device__ __forceinline__ int vit_trace(const uint32_t* back, int hi, int edge, uint32_t* buf, int* sl, int t)
{
    constexpr int Q = 1 << K, KR = 16 - K, ROWS = 16;
    uint4 nx[ROWS / 4];
    auto request = [&](int top) {                                // rows top - 15 .. top (those >= 0), 16 bytes per thread and load
#pragma unroll
        for (int u = 0; u < ROWS / 4; ++u)
        {
            const int row = top - (4 * u + (t >> 8));
            nx[u] = row >= 0 ? *(const uint4*)(back + (size_t)row * VT + 4 * (t & 255)) : make_uint4(0, 0, 0, 0);
        }
    };
    request(hi);
    for (int top = hi; top >= 0; top -= ROWS)
    {
#pragma unroll
        for (int u = 0; u < ROWS / 4; ++u) *(uint4*)(buf + (4 * u + (t >> 8)) * VT + 4 * (t & 255)) = nx[u];
        if (top >= ROWS) request(top - ROWS);
        lds_barrier();
        if (t == 0)
            for (int s = 0; s < ROWS && top - s >= 0; ++s)
            {
                const int g = edge >> K;
                const uint32_t q = (buf[s * VT + (g & 1023)] >> (K * ((g >> 10) * Q + (edge & (Q - 1))))) & (Q - 1);
                const int st = (int)(q << KR) | edge;
                sl[top - s] = st;
                edge = st >> K;
            }
        lds_barrier();
    }
    return edge;
}

template <int K>
__global__ void __launch_bounds__(VT) nq_viterbi_k(VitArgs a)
{
    constexpr int Q = 1 << K, KR = 16 - K, E = 1 << KR, R = 64 >> (2 * K);
    extern __shared__ __align__(16) float cost[];                // 128 KB: two arrays of E costs (K = 2), or one (K = 1); then the walk's blocks
    __shared__ float wl[VIT_LMAX];
    __shared__ int sl[VIT_LMAX];
    __shared__ unsigned long long red[VT / 64];
    __shared__ int start_sh;
    const int t = threadIdx.x, L = a.L;
    uint32_t* back = a.back + (size_t)blockIdx.x * L * VT;
    for (int ring = blockIdx.x; ring < a.T; ring += gridDim.x)
    {
        for (int i = t; i < L; i += VT) wl[i] = a.w[(size_t)ring * L + (a.rev ? (L - i) % L : i)];
        int start = -1;
#pragma clang loop unroll(disable)
        for (int pass = 0; pass < 2; ++pass)
        {
            asm volatile("" : "+s"(pass));                       // one copy of the loop below
            const int roll = pass == 0 ? L / 2 : 0, keep = pass == 0 && L > 1 ? L - roll : 0;
            for (int e = t; e < E; e += VT) cost[e] = pass == 0 || e == start ? 0.f : __builtin_inff();
            float v[R][Q][Q];                                    // the pass's codebook values: loaded here so that nothing else shares their registers
            uint32_t off = Q * t * 4u;
            asm volatile("" : "+v"(off));
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int q = 0; q < Q; ++q)
                {
                    const char* base = (const char*)(a.lut + (q << KR) + Q * 1024 * r);
#pragma unroll
                    for (int j = 0; j < Q; ++j) v[r][j][q] = *(const float*)(base + off + 4 * j);
                }
            lds_barrier();
            for (int i = 0; i < L; ++i)
            {
                const int ri = i + roll < L ? i + roll : i + roll - L;
                float* cur = K == 2 ? cost + (i & 1) * E : cost;
                float* nxt = K == 2 ? cost + (~i & 1) * E : cost;
                const uint32_t word = vit_step<K>(v, wl[ri], cur, nxt, t);
                if (i >= keep) back[(size_t)ri * VT + t] = word;
                lds_barrier();
            }
            int edge = start;
            if (pass == 0)
            {   // the cheapest edge after the last step, the smallest of equals
                const float* fin = K == 2 ? cost + (L & 1) * E : cost;
                unsigned long long best = ~0ull;
                for (int e = t; e < E; e += VT)
                {
                    const unsigned long long k = ((unsigned long long)__builtin_bit_cast(uint32_t, fin[e]) << 32) | (unsigned)e;
                    best = k < best ? k : best;
                }
#pragma unroll
                for (int m = 32; m; m >>= 1) { const unsigned long long o = __shfl_xor(best, m); best = o < best ? o : best; }
                if ((t & 63) == 0) red[t >> 6] = best;
                lds_barrier();
                best = red[0];
                for (int w = 1; w < VT / 64; ++w) best = red[w] < best ? red[w] : best;
                edge = (int)(best & 0xFFFFFFFFu);
            }
            __syncthreads();                                     // the decisions of all wavefronts are in memory
            edge = vit_trace<K>(back, pass == 0 && L > 1 ? roll - 1 : L - 1, edge, (uint32_t*)cost, sl, t);
            if (pass == 0)
            {
                if (t == 0) start_sh = edge;
                lds_barrier();
                start = start_sh;
            }
        }
        for (int i = t; i < L; i += VT) a.st[(size_t)ring * L + (a.rev ? (L - i) % L : i)] = sl[i];
        lds_barrier();                                           // sl and wl are free again
    }
}

int launch_viterbi(const float* w, int T, int L, int K, const float* lut, int64_t* st, uint32_t* back, int slots, int rev, hipStream_t s)
{
    const VitArgs a{w, lut, st, back, T, L, rev};
    const int shm = 2 * 16384 * 4;
    auto kern = K == 2 ? nq_viterbi_k<2> : nq_viterbi_k<1>;
    const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
    if (e != hipSuccess) return set_error("nq_viterbi: LDS %d bytes: %s", shm, hipGetErrorString(e));
    kern<<<T < slots ? T : slots, VT, shm, s>>>(a);
    NQ_LAUNCH_CHECK("nq_viterbi");
    return 0;
}

}  // namespace nq
