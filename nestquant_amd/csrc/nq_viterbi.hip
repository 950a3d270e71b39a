// Tail-biting trellis search of the encoder (the reference leaves it to CUDA kernels of its own; restated from the algorithm of
// threads/05-exl3-harness/harness.py:297-364): for every ring of L targets the path of least squared error through the 16-bit
// shift-register trellis with K = 1 or 2 new bits per step, in two passes -- pass 1, rolled by half a ring, finds the state that
// enters step 0; pass 2 starts from and ends in it. encode.viterbi_ring is the same search in torch, and the results are equal
// bit for bit: every candidate is (value - target)^2 + cost in fp32 with the torch code's roundings (no contraction), and ties go
// to the smallest predecessor.
//
// One workgroup of 1024 threads per ring, or per pass over it (launch_viterbi). "Edge" = the low 16 - K bits of a state (E of them); the
// candidates of edge e are its 2^K states, each with predecessor edge (q << (16 - 2 K)) | (e >> K), so 2^K neighbouring edges (a
// group) share their predecessors: thread t owns the groups t + 1024 r, keeps the 64 codebook values of their states in registers through
// a pass, reads 2^K costs per group from LDS and writes 2^K. Both directions of that traffic are free of bank conflicts.
// The decisions of a thread in one step (16 edges x 2 bits, or 32 x 1) fill one word, stored to a scratch of 4 KB per step; the way
// back is walked by one lane over blocks of steps brought to LDS, the next block on its way meanwhile.
//
// Bound: instruction issue of sixteen wavefronts in lockstep, and with all CUs at work the clock that the power limit leaves. A step is 65536
// candidates of three fp32 operations plus the selection. ns per four candidates (K = 2), wavefront and SIMD in a loop of nothing else:
// the twelve fp32 operations 12.8; with three minima 14.1 (a three-way one and one of two 15.0); with the decision besides, as comparisons
// whose lane masks are carried into the word, 20.9; as minima of doubles, below, 18.5. At K = 1 the sign of a difference shifted into
// the word (9.3 for two candidates) is ahead of the carried mask (9.6) by more than that inside the kernel, of minima of doubles too.
// Measured, us for 128 / 256 / 512 rings of 256 steps: K = 2 725 / 935 / 1785 (858 / 1019 / 2034 with the carried masks, decisions in steps
// that nobody walks back over, and a walk that waited for each of its blocks), K = 1 932 / 1050 / 1990 (1084 / 1190 / 2300; its
// single array costs a second barrier). 267 vector instructions per wavefront and step at K = 2, one per 3.0 clocks and SIMD over the
// whole launch, 288 and 3.9 at K = 1 (313 and 3.1, 320 and 4.0 with the carried masks). The walks back are about 40 of them. Without any decisions 640 and 758 (K = 2): keeping
// every seventh step's costs instead and finding the decisions anew from them cost more in traffic than that gives.
#include "nq_decode.hpp"
#include "nq_host.hpp"

namespace nq {

constexpr int VT = 1024, VIT_LMAX = 1024;

struct VitArgs { const float* w; const float* lut; int64_t* st; uint32_t* back; int T, L, rev; int from, to; };

// all wavefronts' LDS accesses so far are done; stores to global memory stay in flight (a __syncthreads would wait for them)
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Wavefronts lower their priority as they get on with a step: the arbiter otherwise serves the oldest first, and a step ends with
// the youngest wavefront of every SIMD alone, which cannot issue more than one instruction in six clocks.
__device__ __forceinline__ void step_priority(int quarter)
{
    if (quarter == 0) __builtin_amdgcn_s_setprio(3);
    else if (quarter == 1) __builtin_amdgcn_s_setprio(2);
    else if (quarter == 2) __builtin_amdgcn_s_setprio(1);
    else __builtin_amdgcn_s_setprio(0);
}

template <int K> constexpr int VIT_R = 64 >> (2 * K);           // groups per thread
template <int K> using Values = float[VIT_R<K>][1 << K][1 << K];                         // [group][edge of the group][candidate]

// The least of candidates and which one it was, in one instruction: a cost's bits as the upper half of a double, the candidate's number as the
// lower half. Costs are >= +0 and never NaN (vit_target, vit_value), so doubles order as (cost, number) do, subnormal ones included: the first of the
// least wins.
typedef uint32_t Tagged __attribute__((ext_vector_type(2)));     // number, cost
__device__ __forceinline__ Tagged vit_min(Tagged a, Tagged b)
{
    double d;
    asm("v_min_f64 %0, %1, %2" : "=v"(d) : "v"(__builtin_bit_cast(double, a)), "v"(__builtin_bit_cast(double, b)));
    return __builtin_bit_cast(Tagged, d);
}
// a target that is not a finite number makes all candidates equally dear, infinitely so; a value that is no number is never near
__device__ __forceinline__ float vit_target(float w) { return __builtin_fabsf(w) <= 3.4028234e38f ? w : 3e38f; }
__device__ __forceinline__ float vit_value(float v) { return v == v ? v : __builtin_inff(); }

// one step of the search: costs cur -> nxt (K = 1: the same array); DECIDE: the decisions -> the returned word
template <int K, bool DECIDE>
__device__ __forceinline__ uint32_t vit_step(const Values<K>& v, float wv, const float* cur, float* nxt, Tagged (&x)[1 << K], int t)
{
    constexpr int Q = 1 << K, R = VIT_R<K>, G = 1024 * R;
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
        step_priority(4 * r / R);
        uint32_t m_of[Q];
#pragma unroll
        for (int j = 0; j < Q; ++j)
        {
            auto cand = [&](int q) { const float d = v[r][j][q] - wv; return __builtin_bit_cast(uint32_t, d * d + c[r][q]); };
            uint32_t m;
            if constexpr (K == 2 && DECIDE)
            {
#pragma unroll
                for (int q = 0; q < Q; ++q) x[q].y = cand(q);
                const Tagged b = vit_min(vit_min(x[0], x[1]), vit_min(x[2], x[3]));
                asm("v_lshl_or_b32 %0, %0, 2, %1" : "+v"(word) : "v"(b.x));           // (as an expression it becomes a tree that keeps all numbers alive)
                m = b.y;
            }
            else
            {
                const uint32_t x0 = cand(0), x1 = cand(1);
                m = x1 < x0 ? x1 : x0;
                if constexpr (K == 2)
                {
                    uint32_t n;                                  // (two minima of two: a three-way one issues at half the rate)
                    asm("v_min_u32 %0, %1, %2" : "=v"(n) : "v"(cand(2)), "v"(cand(3)));
                    asm("v_min_u32 %0, %1, %2" : "=v"(m) : "v"(m), "v"(n));
                }
                else if constexpr (DECIDE) asm("v_alignbit_b32 %0, %0, %1, 31" : "+v"(word) : "v"(x1 - x0));     // word << 1 | sign of the difference
            }
            m_of[j] = m;
        }
        __builtin_amdgcn_sched_barrier(0);                       // one group at a time: mixing them would not fit the registers
        if constexpr (K == 2) *(uint4*)(nxt + 4 * (t + 1024 * r)) = make_uint4(m_of[0], m_of[1], m_of[2], m_of[3]);
        else *(uint2*)(nxt + 2 * (t + 1024 * r)) = make_uint2(m_of[0], m_of[1]);
    }
    return word;
}

// walk back over the rows hi .. 0 of the decisions: sl[row] = state at that row. back rows are 4 KB; 16 rows per block, walked by one lane
// while the next block is written to the other half of buf and the one after that is on its way. Returns the edge entering row 0.
template <int K>
__device__ __forceinline__ int vit_trace(const uint32_t* back, int hi, int edge, uint32_t* buf, int* sl, int& edge_sh, int t)
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
    auto place = [&](uint32_t* half) {
#pragma unroll
        for (int u = 0; u < ROWS / 4; ++u) *(uint4*)(half + (4 * u + (t >> 8)) * VT + 4 * (t & 255)) = nx[u];
    };
    request(hi);
    place(buf);
    if (hi >= ROWS) request(hi - ROWS);
    for (int top = hi, b = 0; top >= 0; top -= ROWS, b ^= 1)
    {
        lds_barrier();                                           // block b is there, block b ^ 1 has been walked
        if (top >= ROWS) place(buf + (b ^ 1) * ROWS * VT);
        if (top >= 2 * ROWS) request(top - 2 * ROWS);
        if (t == 0)
            for (int s = 0; s < ROWS && top - s >= 0; ++s)
            {
                const int g = edge >> K;
                const uint32_t q = (buf[(b * ROWS + s) * VT + (g & 1023)] >> (32 - K - K * ((g >> 10) * Q + (edge & (Q - 1))))) & (Q - 1);   // first pushed = highest
                const int st = (int)(q << KR) | edge;
                sl[top - s] = st;
                edge = st >> K;
            }
    }
    if (t == 0) edge_sh = edge;
    lds_barrier();
    return edge_sh;
}

template <int K, bool HALVES>
__global__ void __launch_bounds__(VT) nq_viterbi_k(VitArgs a)
{
    constexpr int Q = 1 << K, KR = 16 - K, E = 1 << KR, R = VIT_R<K>;
    extern __shared__ __align__(16) float cost[];                // 128 KB: two arrays of E costs (K = 2), or one (K = 1); then the walk's blocks
    __shared__ float wl[VIT_LMAX];
    __shared__ int sl[VIT_LMAX];
    __shared__ unsigned long long red[VT / 64];
    __shared__ int edge_sh;
    const int t = threadIdx.x, L = a.L;
    uint32_t* back = a.back + (size_t)blockIdx.x * L * VT;
    for (int u = (HALVES ? a.from : 0) + blockIdx.x; u < (HALVES ? a.to : a.T); u += gridDim.x)
    {   // a whole ring, or one pass over it: pass 1 of ring u, pass 2 of ring u - T, whose first state pass 1 has left in st
        const int first = HALVES && u >= a.T ? 1 : 0, last = HALVES ? first + 1 : 2, ring = HALVES && first ? u - a.T : u;
        for (int i = t; i < L; i += VT) wl[i] = vit_target(a.w[(size_t)ring * L + (a.rev ? (L - i) % L : i)]);
        int start = HALVES && first ? (int)a.st[(size_t)ring * L] : -1;
#pragma clang loop unroll(disable)
        for (int pass = first; pass < last; ++pass)
        {
            if (HALVES) pass = __builtin_amdgcn_readfirstlane(pass);
            asm volatile("" : "+s"(pass));                       // one copy of the loops below
            const int roll = pass == 0 ? L / 2 : 0, keep = pass == 0 && L > 1 ? L - roll : 0;     // nobody walks back over the steps before `keep`
            for (int e = t; e < E; e += VT) cost[e] = pass == 0 || e == start ? 0.f : __builtin_inff();
            Values<K> v;                                         // the pass's codebook values: loaded here so that nothing else shares their registers
            uint32_t off = Q * t * 4u;
            asm volatile("" : "+v"(off));
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int q = 0; q < Q; ++q)
                {
                    const char* base = (const char*)(a.lut + (q << KR) + Q * 1024 * r);
#pragma unroll
                    for (int j = 0; j < Q; ++j) v[r][j][q] = vit_value(*(const float*)(base + off + 4 * j));
                }
            Tagged x[Q];                                         // their numbers stay where they are through all steps
#pragma unroll
            for (int q = 0; q < Q; ++q) { uint32_t num = q; asm volatile("" : "+v"(num)); x[q].x = num; }
            lds_barrier();
            auto steps = [&](auto decide, int from, int to) {
                constexpr bool D = decltype(decide)::value != 0;
                for (int i = from; i < to; ++i)
                {
                    const int ri = i + roll < L ? i + roll : i + roll - L;
                    float* cur = K == 2 ? cost + (i & 1) * E : cost;
                    float* nxt = K == 2 ? cost + (~i & 1) * E : cost;
                    const uint32_t word = vit_step<K, D>(v, wl[ri], cur, nxt, x, t);
                    if (D) back[(size_t)ri * VT + t] = word;
                    lds_barrier();
                }
            };
            steps(CodeTag<0>{}, 0, keep);
            steps(CodeTag<1>{}, keep, L);
            __builtin_amdgcn_s_setprio(0);
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
            start = vit_trace<K>(back, pass == 0 && L > 1 ? roll - 1 : L - 1, edge, (uint32_t*)cost, sl, edge_sh, t);
        }
        if (HALVES && last == 1) { if (t == 0) a.st[(size_t)ring * L] = start; }
        else for (int i = t; i < L; i += VT) a.st[(size_t)ring * L + (a.rev ? (L - i) % L : i)] = sl[i];
        lds_barrier();                                           // sl and wl are free again
    }
}

int launch_viterbi(const float* w, int T, int L, int K, const float* lut, int64_t* st, uint32_t* back, int slots, int rev, hipStream_t s)
{
    const int shm = 2 * 16384 * 4;
    // Where the last round would leave at least half of the workgroups idle, its rings and those of the round before are searched pass by pass, in
    // three launches of at most `slots` passes (all first ones, then all second ones: more than `slots` rings, so the two of a ring are in different
    // launches): three halves of a round in place of two rounds. us for 320 / 384 rings of 256 steps on 256 CUs: K = 2 1480 / 1560 -> 1265 /
    // 1380, K = 1 1874 / 1872 -> 1523 / 1590. The rounds before them are whole rings in one launch, whose workgroups need not wait for the slowest of
    // each round. ms for 2688 / 10304 / 24640 rings, all whole, all passes in launches of their own, and so: K = 2 7.54 / 28.3 / 66.8, 7.45 / 28.7 /
    // 68.4, 7.32 / 28.2 / 66.8; K = 1 9.95 / 37.0 / 87.7, 9.88 / 38.0 / 90.4, 9.60 / 36.7 / 87.5.
    const int rest = T % slots;
    const int whole = T > slots && rest > 0 && 2 * (int64_t)rest <= slots ? T - rest - slots : T;
    auto launch = [&](auto kern, int grid, const VitArgs& A) {
        const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
        if (e != hipSuccess) return set_error("nq_viterbi: LDS %d bytes: %s", shm, hipGetErrorString(e));
        kern<<<grid, VT, shm, s>>>(A);
        NQ_LAUNCH_CHECK("nq_viterbi");
        return 0;
    };
    if (whole > 0)
        if (int rc = launch(K == 2 ? nq_viterbi_k<2, false> : nq_viterbi_k<1, false>, whole < slots ? whole : slots, VitArgs{w, lut, st, back, whole, L, rev, 0, 0})) return rc;
    const int n = T - whole;
    for (int from = 0; from < 2 * n; from += slots)
    {
        const int to = 2 * n - from < slots ? 2 * n : from + slots;
        if (int rc = launch(K == 2 ? nq_viterbi_k<2, true> : nq_viterbi_k<1, true>, to - from, VitArgs{w + (size_t)whole * L, lut, st + (size_t)whole * L, back, n, L, rev, from, to})) return rc;
    }
    return 0;
}

// ---- the second plane of the interleaved two-plane level 4, with the first one frozen (encode.viterbi_ring_given_p3) -------------
// State b: eight bits of plane P4, one new bit per step; the value at step t is lut[spread(a_t) | spread(b) << 1] with P3's eight bits
// a_t. 128 edges: one wavefront per ring, lane l owns edges 2 l and 2 l + 1, which share the predecessors l and 64 + l. Costs pass
// through LDS (256 words per wavefront), decisions are two lane masks per step, kept in LDS for the walk back. The four codebook
// values of a step do not depend on the search and are requested two steps ahead. Bound by the latency of one step's chain (LDS
// round trip, three fp32 operations, one selection), so the rings' number counts, not their length.
constexpr int P4_L = 256, P4_WAVES = 4;
struct VitP4Args { const float* w; const int64_t* a; const float* lut; int64_t* b; int T, L, rev; };

__device__ __forceinline__ uint32_t spread8(uint32_t v)          // bit i -> bit 2 i
{
    v = (v | (v << 4)) & 0x0F0Fu; v = (v | (v << 2)) & 0x3333u;
    return (v | (v << 1)) & 0x5555u;
}
__global__ void __launch_bounds__(64 * P4_WAVES) nq_viterbi_p4_k(VitP4Args A)
{
    __shared__ float cost_s[P4_WAVES][2][128];
    __shared__ unsigned long long back_s[P4_WAVES][P4_L][2];
    __shared__ float w_s[P4_WAVES][P4_L];
    __shared__ unsigned short sa_s[P4_WAVES][P4_L];
    __shared__ unsigned char b_s[P4_WAVES][P4_L];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, L = A.L, ring = blockIdx.x * P4_WAVES + wv;
    if (ring >= A.T) return;                                     // wave-uniform; nothing below crosses wavefronts
    auto sync = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); __builtin_amdgcn_wave_barrier(); };
    for (int i = lane; i < L; i += 64)
    {
        const size_t at = (size_t)ring * L + (A.rev ? (L - i) % L : i);
        w_s[wv][i] = A.w[at]; sa_s[wv][i] = (unsigned short)spread8((uint32_t)A.a[at] & 0xFFu);
    }
    uint32_t sb[2][2];                                           // [edge][choice]
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 2; ++q) sb[j][q] = spread8((uint32_t)((q << 7) | (2 * lane + j))) << 1;
    sync();
    int start = -1;
    for (int pass = 0; pass < 2; ++pass)
    {
        const int roll = pass == 0 ? L / 2 : 0;
        float* c0 = cost_s[wv][0]; float* c1 = cost_s[wv][1];
        c0[2 * lane] = pass == 0 || 2 * lane == start ? 0.f : __builtin_inff();
        c0[2 * lane + 1] = pass == 0 || 2 * lane + 1 == start ? 0.f : __builtin_inff();
        auto row = [&](int i) { return i + roll < L ? i + roll : i + roll - L; };
        float v[3][2][2];
        auto fetch = [&](int i, float (&d)[2][2]) {
            const uint32_t sa = sa_s[wv][row(i < L ? i : L - 1)];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 2; ++q) d[j][q] = A.lut[sa | sb[j][q]];
        };
        fetch(0, v[0]); fetch(1, v[1]);
        for (int i = 0; i < L; ++i)
        {
            sync();
            const int ri = row(i);
            fetch(i + 2, v[2]);
            const float w = w_s[wv][ri], p0 = c0[lane], p1 = c0[64 + lane];
            float m[2]; bool hi[2];
#pragma unroll
            for (int j = 0; j < 2; ++j)
            {
                const float d0 = v[0][j][0] - w, d1 = v[0][j][1] - w;
                const float x0 = d0 * d0 + p0, x1 = d1 * d1 + p1;
                hi[j] = x1 < x0; m[j] = hi[j] ? x1 : x0;
            }
            *(float2*)(c1 + 2 * lane) = make_float2(m[0], m[1]);
            const unsigned long long b0 = __ballot(hi[0]), b1 = __ballot(hi[1]);
            if (lane == 0) { back_s[wv][ri][0] = b0; back_s[wv][ri][1] = b1; }
            float* t = c0; c0 = c1; c1 = t;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 2; ++q) { v[0][j][q] = v[1][j][q]; v[1][j][q] = v[2][j][q]; }
        }
        sync();
        int edge = start;
        if (pass == 0)
        {   // the cheapest edge after the last step, the smallest of equals
            const float e0 = c0[2 * lane], e1 = c0[2 * lane + 1];
            unsigned long long best = ((unsigned long long)__builtin_bit_cast(uint32_t, e1 < e0 ? e1 : e0) << 32) | (unsigned)(2 * lane + (e1 < e0 ? 1 : 0));
#pragma unroll
            for (int k = 32; k; k >>= 1) { const unsigned long long o = __shfl_xor(best, k); best = o < best ? o : best; }
            edge = (int)(best & 0xFFFFFFFFu);
        }
        for (int r = pass == 0 && L > 1 ? roll - 1 : L - 1; r >= 0; --r)          // every lane walks the same way
        {
            const int q = (int)(back_s[wv][r][edge & 1] >> (edge >> 1)) & 1, st = (q << 7) | edge;
            if (lane == 0) b_s[wv][r] = (unsigned char)st;
            edge = st >> 1;
        }
        start = edge;
        sync();
    }
    for (int i = lane; i < L; i += 64) A.b[(size_t)ring * L + (A.rev ? (L - i) % L : i)] = b_s[wv][i];
}

int launch_viterbi_p4(const float* w, const int64_t* a, int T, int L, const float* lut, int64_t* b, int rev, hipStream_t s)
{
    const VitP4Args A{w, a, lut, b, T, L, rev};
    nq_viterbi_p4_k<<<(T + P4_WAVES - 1) / P4_WAVES, 64 * P4_WAVES, 0, s>>>(A);
    NQ_LAUNCH_CHECK("nq_viterbi_p4");
    return 0;
}

}  // namespace nq
