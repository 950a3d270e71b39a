// Prefill path (steps of more tokens than a decode call takes): every routed expert's weights are decoded once per 16..256-row tile of its tokens, inside
// the grouped GEMM itself, not by way of HBM but for experts of many rows (reference: pf_decode to fp16 in HBM + Triton/cuBLAS grouped GEMM,
// sm120/nqmoe.cu:942-1240, sm120/pf_gemm.py:7-34, sm120/moe.py:282-326).
//
//   nq_pf_sort_k  pairs sorted by expert, per-expert counts, hits; the tile list of a step without tall tiles
//   nq_pf_pre_k   per (token, expert) pair, sorted by expert: xg / xu = fp16(Hadamard-128(x * su_g / su_u)), written in
//                 B-operand column order so the GEMM stages them with straight 16-byte copies      (reference nq_pf_pre)
//   nq_pf_gemm_k  C[rows of expert j][N] = A[rows][K] @ W_j[N][K]^T: grid (N / 128, tiles); a tile = (expert, row0, rows
//                 <= 16 TG). Per 128-column chunk the block stages the tile's activations in LDS while each wavefront
//                 decodes two strips of the expert's records into MFMA A operands, then runs TG x 8 MFMAs
//                 (v_mfma_f32_16x16x32_f16, fp32 accumulate) over the staged tokens. Level from the live table row.
//   nq_pf_short_k the same for all tiles of up to 64 rows in one launch
//   nq_pf_wdecode_k, nq_pf_wide_k   weights of experts with many rows decoded once into a scratch, and their tiles
//   nq_pf_mid_k   Hadamard * sv, SwiGLU, * su_d, Hadamard -> h fp16 (B-operand order)               (reference nq_pf_mid)
//   nq_pf_post_k  out[token] += sum over its picks of rw * sv_o (.) Hadamard(y): gathered per token, no atomics  (reference nq_pf_post)
//   nq_pf_hits_k  hits[e] += counts[e]                                                            (reference nq_pf_hits)
#include "nq_pf_tile.hpp"
#include "../../include/nq_moe_hip.h"

namespace nq {

// Is pair row p (of expert e) held by a tile of one of the heights in the bit mask `heights` (bit k = 16 << k)? tiles / cap:
// the lists of nq_pf_plan_k. The remainder tile of expert e sits at index e of the list of its height and starts at its
// first row; the rows before it belong to the expert's full 256-row tiles. Rows of no valid expert count as height 256.
__device__ __forceinline__ bool row_in_heights(const int32_t* __restrict__ tiles, int cap, int heights, int p, int e, int E)
{
    int k = 4;
    if (e >= 0 && e < E)
#pragma unroll
        for (int q = 0; q < 4; ++q)
        {
            const int4 t = ((const int4*)tiles)[(size_t)q * cap + e];
            if (t.x == e && p >= t.y) k = q;
        }
    return (heights >> k) & 1;
}

// grid (row groups, column parts), block 256: wavefront w of column part y rotates segment 4 y + w (512 columns, four chunks; lanes of
// chunks beyond H repeat the last one) of `rows` pair rows, gate and up together, holding the scale vectors while the expert stays the same.
// tiles (optional): work only on the rows of the tile heights in `heights`.
// Bound by memory, 197 MB written and 57 read at 4.0 TB/s with 8024 rows of 6144 columns: 64 us, one vector instruction per 7 clocks
// and SIMD (profiles/grouped_steps.txt). With two columns per lane (about 50 vector instructions per chunk) it took 84. Fetching
// the next row's activations ahead changed nothing.
__global__ void __launch_bounds__(256) nq_pf_pre_k(const void* __restrict__ x, int xdt, const int32_t* __restrict__ pt, const int32_t* __restrict__ pe, int np, int rows,
                                                    const int64_t* __restrict__ table, _Float16* xg, _Float16* xu, float* zg, int E, int H, int I,
                                                    const int32_t* __restrict__ tiles, int cap, int heights)
{
    __shared__ float zsh[4][4];
    const int lane = threadIdx.x & 63, warp = threadIdx.x >> 6, L = wht_place(lane);
    const int chunk = (4 * blockIdx.y + warp) * 4 + (lane >> 4), ng = H / 128;
    const bool mine = chunk < ng;
    const int col = (mine ? chunk : ng - 1) * 128 + 32 * (L >> 2) + 2 * (L & 3);    // this lane's columns: col + {0, 1} + {0, 8} + {0, 16}
    const WhtSigns ws = wht_signs(lane);
    const int p1 = min(np, (int)(blockIdx.x + 1) * rows);
    half2_t sg[4], su[4];
    int held = -1;                                               // the expert whose scales sg and su hold
    for (int p = blockIdx.x * rows; p < p1; ++p)
    {
        const int e = pe[p];
        if (tiles && !row_in_heights(tiles, cap, heights, p, e, E)) continue;     // block-uniform, like every branch on e
        const bool live = e >= 0 && e < E && table[(size_t)e * TBL_W] > 0;
        const size_t xr = live ? (size_t)pt[p] * H : 0;         // first element of the token's row
        // low-rank plane (table words 14, 16): zg[p] = x V_gu^T over the raw activations, for the mid kernel
        const _Float16* lr = live ? (const _Float16*)table[(size_t)e * TBL_W + 14] : nullptr;
        const int rg = lr ? (int)table[(size_t)e * TBL_W + 16] : 0;
        if (zg && rg && blockIdx.y == 0)
        {
            float zz[4] = {0.f, 0.f, 0.f, 0.f};
            for (int k = 2 * threadIdx.x; k < H; k += 512)
            {
                const half2_t xv = act2_at(x, xdt, xr + k);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (r < rg) { const half2_t vv = *(const half2_t*)(lr + (size_t)r * H + k); zz[r] += (float)xv.x * (float)vv.x + (float)xv.y * (float)vv.y; }
            }
            __syncthreads();                                     // the previous row's sums have been read
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
#pragma unroll
                for (int m = 32; m >= 1; m >>= 1) zz[r] += __shfl_xor(zz[r], m);
                if (lane == 0) zsh[warp][r] = zz[r];
            }
            __syncthreads();
            if (threadIdx.x < 4) zg[(size_t)p * 4 + threadIdx.x] = zsh[0][threadIdx.x] + zsh[1][threadIdx.x] + zsh[2][threadIdx.x] + zsh[3][threadIdx.x];
        }
        uint4 bg = make_uint4(0, 0, 0, 0), bu = bg;              // rows of no live expert are zero
        if (live)
        {
            half2_t xv[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) xv[q] = act2_at(x, xdt, xr + col + 8 * q);
            if (e != held)
            {
                const _Float16 *sug = (const _Float16*)table[(size_t)e * TBL_W + 9], *suu = sug + 2 * H + 3 * I;
#pragma unroll
                for (int q = 0; q < 4; ++q) { sg[q] = *(const half2_t*)(sug + col + 8 * q); su[q] = *(const half2_t*)(suu + col + 8 * q); }
                held = e;
            }
            float g[8], u[8];
#pragma unroll
            for (int q = 0; q < 4; ++q)
            {
                const float x0 = (float)xv[q].x, x1 = (float)xv[q].y;
                g[2 * q] = x0 * (float)sg[q].x; g[2 * q + 1] = x1 * (float)sg[q].y;
                u[2 * q] = x0 * (float)su[q].x; u[2 * q + 1] = x1 * (float)su[q].y;
            }
            wht8_bop(g, ws); wht8_bop(u, ws);
            bg = bop_block(g); bu = bop_block(u);
        }
        if (mine)
        {
            const size_t at = (size_t)p * H + chunk * 128 + 8 * L;
            *(uint4*)(xg + at) = bg;
            *(uint4*)(xu + at) = bu;
        }
    }
}

// grid (row groups), block 256: acc_gu [P][2I] fp32 (gate | up) -> h [P][I] fp16 in B-operand order. The wavefronts take the tasks
// (pair row of the group, segment of 512 columns) in turn; lanes of chunks beyond I repeat the last one. With in_had_down = 512
// (table word 18) the four chunks of a segment are combined with the Sylvester H_4 / 2 before the single rounding to fp16.
// tiles (optional): work only on the rows of the tile heights in `heights`, as nq_pf_pre_k
// Bound by memory, 5 bytes per output element and no reuse: 8024 rows of 2 x 2048 sums 66 -> 41 us (4.1 TB/s) with eight columns per
// lane, which halves the vector instructions as there.
constexpr int MID_ROWS = 8;                                      // most rows of a group
__global__ void __launch_bounds__(256) nq_pf_mid_k(const float* __restrict__ acc_gu, const int32_t* __restrict__ pe, int np, int rows,
                                                    const int64_t* __restrict__ table, _Float16* h, const float* zg, float* zd, int E, int H, int I,
                                                    const int32_t* __restrict__ tiles, int cap, int heights)
{
    __shared__ float zsh[MID_ROWS][4][4];
    const int lane = threadIdx.x & 63, warp = threadIdx.x >> 6, L = wht_place(lane);
    const int p0 = blockIdx.x * rows, nr = min(rows, np - p0), ni = I / 128, nseg = (ni + 3) / 4;
    const WhtSigns ws = wht_signs(lane);
    __shared__ int held[MID_ROWS];                               // is the row of the heights?
    if (tiles)
    {   // looked up side by side: one after the other, as the loop comes to them, every row waited for its own
        const bool in = (int)threadIdx.x < nr && row_in_heights(tiles, cap, heights, p0 + threadIdx.x, pe[p0 + threadIdx.x], E);
        if (threadIdx.x < MID_ROWS) held[threadIdx.x] = in;
        if (!__syncthreads_or(in)) return;
    }
    if (zd)
    {
        for (int i = threadIdx.x; i < MID_ROWS * 16; i += 256) (&zsh[0][0][0])[i] = 0.f;
        __syncthreads();
    }
    for (int t = warp; t < nr * nseg; t += 4)                    // e, live, ... are the same for the whole wavefront
    {
        const int row = t / nseg, p = p0 + row, chunk = (t - row * nseg) * 4 + (lane >> 4);
        const int e = pe[p];
        if (tiles && !held[row]) continue;
        const bool mine = chunk < ni, live = e >= 0 && e < E && table[(size_t)e * TBL_W] > 0;
        uint4 b = make_uint4(0, 0, 0, 0);
        if (live)
        {
            const _Float16* signs = (const _Float16*)table[(size_t)e * TBL_W + 9];
            const _Float16 *sv_g = signs + H, *sv_u = sv_g + I, *su_d = sv_u + I;
            const int col = (mine ? chunk : ni - 1) * 128 + 8 * L;
            float g[8], u[8];
            const float* ag = acc_gu + (size_t)p * 2 * I + col;
            *(float4_t*)g = *(const float4_t*)ag; *(float4_t*)(g + 4) = *(const float4_t*)(ag + 4);
            *(float4_t*)u = *(const float4_t*)(ag + I); *(float4_t*)(u + 4) = *(const float4_t*)(ag + I + 4);
            const half8_t svg = *(const half8_t*)(sv_g + col), svu = *(const half8_t*)(sv_u + col), sud = *(const half8_t*)(su_d + col);
            wht8_row(g, ws); wht8_row(u, ws);
#pragma unroll
            for (int i = 0; i < 8; ++i) { g[i] *= (float)svg[i]; u[i] *= (float)svu[i]; }
            // low-rank plane: g / u += zg (U2 [+ U4 at level 4]); zd[p] = sw V_dn^T for the post kernel
            const _Float16* lr = (const _Float16*)table[(size_t)e * TBL_W + 14];
            const int rg = lr && zg ? (int)table[(size_t)e * TBL_W + 16] : 0, rd = lr && zd ? (int)table[(size_t)e * TBL_W + 17] : 0;
            const _Float16* U2g = lr + (size_t)rg * H, *U2u = U2g + (size_t)rg * I, *Vd = U2u + (size_t)rg * I;
            if (rg)
            {
                const _Float16* lr4 = table[(size_t)e * TBL_W] == 4 ? (const _Float16*)table[(size_t)e * TBL_W + 15] : nullptr;
                for (int r = 0; r < rg; ++r)
                {
                    const float z = zg[(size_t)p * 4 + r];
                    half8_t ug = *(const half8_t*)(U2g + (size_t)r * I + col), uu = *(const half8_t*)(U2u + (size_t)r * I + col);
#pragma unroll
                    for (int i = 0; i < 8; ++i) { g[i] += z * (float)ug[i]; u[i] += z * (float)uu[i]; }
                    if (lr4)
                    {
                        ug = *(const half8_t*)(lr4 + (size_t)r * I + col); uu = *(const half8_t*)(lr4 + (size_t)(rg + r) * I + col);
#pragma unroll
                        for (int i = 0; i < 8; ++i) { g[i] += z * (float)ug[i]; u[i] += z * (float)uu[i]; }
                    }
                }
            }
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = g[i] / (1.f + __expf(-g[i])) * u[i];
            for (int r = 0; r < rd; ++r)
            {
                const half8_t vv = *(const half8_t*)(Vd + (size_t)r * I + col);
                float z = 0.f;
#pragma unroll
                for (int i = 0; i < 8; ++i) z += v[i] * (float)vv[i];
                if (!mine) z = 0.f;
#pragma unroll
                for (int m = 32; m >= 1; m >>= 1) z += __shfl_xor(z, m);
                if (lane == 0) zsh[row][warp][r] += z;           // this wavefront's own sums, segment by segment
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] *= (float)sud[i];
            wht8_row(v, ws);
            if (table[(size_t)e * TBL_W + 18] == 512)            // I % 512 == 0: every chunk of the segment is there
            {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                {
                    float o = 0.f;
#pragma unroll
                    for (int q = 0; q < 4; ++q) o += ((__builtin_popcount((lane >> 4) & q) & 1) ? -0.5f : 0.5f) * __shfl(v[i], 16 * q + (lane & 15));
                    v[i] = o;
                }
            }
            b = bop_block_of_row(v, lane);
        }
        if (mine) *(uint4*)(h + (size_t)p * I + chunk * 128 + 8 * L) = b;
    }
    if (!zd) return;
    __syncthreads();
    for (int i = threadIdx.x; i < nr * 4; i += 256)
    {
        const int p = p0 + i / 4, r = i & 3, e = pe[p];
        if (e < 0 || e >= E || table[(size_t)e * TBL_W] <= 0 || !table[(size_t)e * TBL_W + 14] || table[(size_t)e * TBL_W + 17] <= r) continue;
        if (tiles && !held[i / 4]) continue;
        zd[(size_t)p * 4 + r] = zsh[i / 4][0][r] + zsh[i / 4][1][r] + zsh[i / 4][2][r] + zsh[i / 4][3][r];
    }
}

// grid (T, column parts), block 64 or 256: out[t] (+)= sum over the token's picks whose pair row lies in [row_lo, row_lo + nrows) of
// rw * sv_o (.) Hadamard(y[row]); pos[t][k] = row of pair (t, k) in the expert-sorted order; add: on top of what out holds (fp32),
// else out is written whole, zeros included. One block owns a token, so
// the sum needs no atomics and its order is fixed (the reference's pf_post adds with float atomics in arrival order).
__global__ void __launch_bounds__(256) nq_pf_post_k(const float* __restrict__ y, const int32_t* __restrict__ pos, const void* __restrict__ sel, int sdt,
                                                     const void* __restrict__ rw, int wdt, int topk, int row_lo, int nrows,
                                                     const int64_t* __restrict__ table, void* out, int odt, int add, const float* zd, int E, int H, int I)
{
    const int t = blockIdx.x, lane = threadIdx.x & 63, warp = threadIdx.x >> 6;
    // the token's live picks, gathered once: row, weight and sign vector (picks keep their order, so does the sum)
    __shared__ int p_row[64]; __shared__ float p_w[64]; __shared__ const _Float16* p_sv[64]; __shared__ int p_n;
    __shared__ const _Float16* p_u2[64]; __shared__ const _Float16* p_u4[64]; __shared__ int p_rd[64];   // low-rank plane: U2_d, U4_d (level 4) and r_dn
    if (warp == 0)
    {
        bool ok = false; int r = 0, rdn = 0; float w = 0.f; const _Float16* sv = nullptr; const _Float16* u2 = nullptr; const _Float16* u4 = nullptr;
        if (lane < topk)
        {
            r = pos[(size_t)t * topk + lane] - row_lo;
            const long long e = id_at(sel, sdt, (size_t)t * topk + lane);
            w = w_at(rw, wdt, (size_t)t * topk + lane);
            if (r >= 0 && r < nrows && e >= 0 && e < E && w != 0.f && table[(size_t)e * TBL_W] > 0)
            {
                ok = true; sv = (const _Float16*)table[(size_t)e * TBL_W + 9] + H + 3 * I;
                const _Float16* lr = (const _Float16*)table[(size_t)e * TBL_W + 14];
                if (lr && zd)
                {
                    const int rg = (int)table[(size_t)e * TBL_W + 16];
                    rdn = (int)table[(size_t)e * TBL_W + 17];
                    u2 = lr + (size_t)rg * (H + 2 * I) + (size_t)rdn * I;
                    if (table[(size_t)e * TBL_W] == 4) u4 = (const _Float16*)table[(size_t)e * TBL_W + 15] + (size_t)rg * 2 * I;
                }
            }
        }
        const unsigned long long m = __ballot(ok);
        if (ok) { const int i = __popcll(m & ((1ull << lane) - 1ull)); p_row[i] = r; p_w[i] = w; p_sv[i] = sv; p_u2[i] = u2; p_u4[i] = u4; p_rd[i] = rdn; }
        if (lane == 0) p_n = __popcll(m);
    }
    __syncthreads();
    const int np = p_n;
    if (np == 0 && add) return;
    const int nw = blockDim.x >> 6, ng = H / 128, L = wht_place(lane);
    const WhtSigns ws = wht_signs(lane);                         // eight columns per lane: 8024 rows 62 -> 46 us (4.5 TB/s)
    for (int sg = nw * blockIdx.y + warp; 4 * sg < ng; sg += nw * gridDim.y)       // segments of 512 columns, eight per lane; lanes beyond H repeat the last chunk
    {
        const int chunk = 4 * sg + (lane >> 4), col = (chunk < ng ? chunk : ng - 1) * 128 + 8 * L;
        float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int k0 = 0; k0 < np; k0 += 4)                       // four picks at a time, reads first
        {
            float v[4][8]; half8_t sv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                const int k = k0 + u < np ? k0 + u : k0;
                const float* row = y + (size_t)p_row[k] * H + col;
                *(float4_t*)v[u] = *(const float4_t*)row; *(float4_t*)(v[u] + 4) = *(const float4_t*)(row + 4);
                sv[u] = *(const half8_t*)(p_sv[k] + col);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                if (k0 + u >= np) break;
                wht8_row(v[u], ws);
                const float w = p_w[k0 + u];
#pragma unroll
                for (int i = 0; i < 8; ++i) v[u][i] *= (float)sv[u][i];
                for (int r = 0; r < p_rd[k0 + u]; ++r)           // y += (sw V_dn^T) (U2_d [+ U4_d])
                {
                    const float zr = zd[(size_t)p_row[k0 + u] * 4 + r];
                    half8_t ud = *(const half8_t*)(p_u2[k0 + u] + (size_t)r * H + col);
#pragma unroll
                    for (int i = 0; i < 8; ++i) v[u][i] += zr * (float)ud[i];
                    if (p_u4[k0 + u])
                    {
                        ud = *(const half8_t*)(p_u4[k0 + u] + (size_t)r * H + col);
#pragma unroll
                        for (int i = 0; i < 8; ++i) v[u][i] += zr * (float)ud[i];
                    }
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) o[i] += w * v[u][i];
            }
        }
        if (chunk >= ng) continue;
        const size_t at = (size_t)t * H + col;
        if (add)                                                 // fp32 results only
#pragma unroll
            for (int i = 0; i < 8; ++i) o[i] = ((const float*)out)[at + i] + o[i];
        if (odt == DT_OUT_F16) *(uint4*)((_Float16*)out + at) = make_uint4(pack_f16(o[0], o[1]), pack_f16(o[2], o[3]), pack_f16(o[4], o[5]), pack_f16(o[6], o[7]));
        else
#pragma unroll
            for (int i = 0; i < 8; i += 2) res2_store(out, odt, at + i, o[i], o[i + 1]);
    }
}

__global__ void nq_pf_hits_k(const int32_t* counts, int32_t* hits, int E)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < E && counts[e]) __hip_atomic_fetch_add(hits + e, counts[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---- tile lists on the device ------------------------------------------------------------------------------------------
// One workgroup. counts[e] = pairs of expert e over the whole call (pairs sorted by expert, so expert e owns the pair rows
// [sum of counts before e, + counts[e])); the chunk is the pair rows [row_lo, row_lo + nrows). Every expert's rows inside
// the chunk are cut into 256-row tiles; the remainder goes to the list of the smallest compiled height (16 << k) that holds
// it, at index e of list k; the full tiles follow at indices E.. of list 4. tiles: int32 [5][cap][4] = (expert, first row in
// the chunk, rows, 0); entries without a tile get expert -1, which the GEMM skips. Replaces the host loop over the expert
// counts and with it the call's one host synchronisation.
__device__ __forceinline__ void block_scan(int* a, int n)
{   // inclusive prefix sum of a[0..n) in LDS, in place; all threads of the block call it (at most 16 wavefronts), a[] written before a barrier
    __shared__ int part[16];
    const int lane = threadIdx.x & 63, warp = threadIdx.x >> 6, per = (n + (int)blockDim.x - 1) / (int)blockDim.x;
    const int lo = min(n, (int)threadIdx.x * per), hi = min(n, lo + per);
    int s = 0;
    for (int i = lo; i < hi; ++i) s += a[i];
    int v = s;                                                   // sum of this and the wavefront's earlier threads
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) { const int o = __shfl_up(v, m); if (lane >= m) v += o; }
    if (lane == 63) part[warp] = v;
    __syncthreads();
    v -= s;
    for (int w = 0; w < warp; ++w) v += part[w];
    for (int i = lo; i < hi; ++i) a[i] = v += a[i];
    __syncthreads();
}

// hot (may be null): experts with at least hot_min rows in the chunk get a slot 0 .. hot_cap - 1 of the decoded-weight scratch (in
// expert order, as far as the slots reach), written to hot[e] (-1: none) and, plus one, into the fourth word of their tiles in list 4 (a
// remainder of up to 128 rows is decoded inside its GEMM: as dear as a whole unit of nq_pf_wide_k). wide (may be null): those tiles
// once more without gaps from wide + 4 on, their number in wide[0]. dense (may be null, with the live table `rows`): the tiles of
// lists 0 to 2 [E] | of list 3 [E] | of list 4 [cap] once more without gaps, then entries of expert -1: what the GEMMs are launched on, over as many
// tiles as the rows can make. Experts above level 2, whose decode takes twice as long, come first in the two lists of remainders.
__global__ void __launch_bounds__(256) nq_pf_plan_k(const int32_t* __restrict__ counts, int E, int row_lo, int nrows, int32_t* tiles, int cap,
                                                    int32_t* hot, int hot_min, int hot_cap, int32_t* wide, int wide_min, const int64_t* __restrict__ table,
                                                    int32_t* dense, const int64_t* __restrict__ rows)
{
    extern __shared__ int plan_sh[];
    int *incl = plan_sh, *fincl = plan_sh + E, *wincl = plan_sh + 2 * E, *hrank = plan_sh + 3 * E;
    for (int e = threadIdx.x; e < E; e += blockDim.x) incl[e] = counts[e] > 0 ? counts[e] : 0;
    __syncthreads();
    block_scan(incl, E);
    const int row_hi = row_lo + nrows;
    auto rows_of = [&](int e, int& r0) {                         // of expert e in the chunk, the first of them at r0
        const int c = counts[e] > 0 ? counts[e] : 0, start = incl[e] - c;
        const int u = start > row_lo ? start : row_lo, v = start + c < row_hi ? start + c : row_hi;
        r0 = u - row_lo;
        return v > u ? v - u : 0;
    };
    auto is_hot = [&](int e, int n) { return hot != nullptr && n >= hot_min && (table == nullptr || table[(size_t)e * TBL_W] > 2); };
    for (int e = threadIdx.x; e < E; e += blockDim.x)
    {
        int r0;
        const int n = rows_of(e, r0);
        fincl[e] = n / 256;
        hrank[e] = is_hot(e, n);
    }
    __syncthreads();
    block_scan(hrank, E);                                        // inclusive: hot experts up to and including e
    block_scan(fincl, E);                                        // full tiles, likewise
    auto slot1_of = [&](int e, int n) { return is_hot(e, n) && hrank[e] <= hot_cap ? hrank[e] : 0; };        // scratch slot + 1
    if (wide)
    {
        for (int e = threadIdx.x; e < E; e += blockDim.x)
        {
            int r0;
            const int n = rows_of(e, r0);
            wincl[e] = slot1_of(e, n) ? n / 256 + (n % 256 > 128) : 0;
        }
        __syncthreads();
        block_scan(wincl, E);
        if (wincl[E - 1] < wide_min) hot_cap = 0;                // too few to fill the GPU: nobody takes a slot
        if (threadIdx.x == 0) wide[0] = hot_cap ? wincl[E - 1] : 0;
    }
    int4 *T4 = (int4*)tiles, *W4 = (int4*)wide + 1;
    for (int e = threadIdx.x; e < E; e += blockDim.x)
    {
        int r0;
        const int n = rows_of(e, r0), nf = n / 256, rem = n % 256;
        const int k = rem == 0 ? -1 : rem <= 16 ? 0 : rem <= 32 ? 1 : rem <= 64 ? 2 : rem <= 128 ? 3 : 4;
        const int slot1 = slot1_of(e, n);
        if (hot != nullptr) hot[e] = slot1 - 1;
        const int4 last = make_int4(e, r0 + 256 * nf, rem, k == 4 ? slot1 : 0);
#pragma unroll
        for (int q = 0; q < 5; ++q) T4[(size_t)q * cap + e] = q == k ? last : make_int4(-1, 0, 0, 0);
        const int base = E + fincl[e] - nf, wbase = wide && slot1 ? wincl[e] - nf - (k == 4) : 0;
        for (int j = 0; j < nf; ++j)
        {
            const int4 t = make_int4(e, r0 + 256 * j, 256, slot1);
            T4[(size_t)4 * cap + base + j] = t;
            if (wide && slot1) W4[wbase + j] = t;
        }
        if (wide && slot1 && k == 4) W4[wbase + nf] = last;
    }
    const int total = E + fincl[E - 1];
    for (int i = total + threadIdx.x; i < cap; i += blockDim.x) T4[(size_t)4 * cap + i] = make_int4(-1, 0, 0, 0);
    if (!dense) return;
    // the counts per expert in low (above level 2) and high half words (E <= 4096); those of 256 rows in one order
    auto level_class = [&](int e, int n) {
        const int64_t lv = n > 0 ? rows[(size_t)e * TBL_W] : 0;
        return lv > 2 ? 1 : lv > 0 ? 1 << 16 : 0;
    };
    __syncthreads();                                             // the ranks have been read
    for (int e = threadIdx.x; e < E; e += blockDim.x)
    {
        int r0;
        const int n = rows_of(e, r0), rem = n % 256, cls = level_class(e, n);
        hrank[e] = rem > 0 && rem <= SHORT_ROWS ? cls : 0;
        wincl[e] = rem > SHORT_ROWS && rem <= 128 ? cls : 0;
        fincl[e] = cls ? n / 256 + (rem > 128) : 0;
    }
    __syncthreads();
    block_scan(hrank, E);
    block_scan(wincl, E);
    block_scan(fincl, E);
    int4 *D4 = (int4*)dense, *tall = D4 + 2 * E;
    for (int e = threadIdx.x; e < E; e += blockDim.x)
    {
        int r0;
        const int n = rows_of(e, r0), nf = n / 256, rem = n % 256, cls = level_class(e, n);
        const int slot1 = hot ? hot[e] + 1 : 0;
        for (int q = 0; q < 2; ++q)
        {
            const int* rank = q ? wincl : hrank;
            const int above = rank[E - 1] & 0xffff, all = above + (rank[E - 1] >> 16);
            if (cls && rem > q * SHORT_ROWS && rem <= (q + 1) * SHORT_ROWS)
                D4[q * E + (cls == 1 ? (rank[e] & 0xffff) - 1 : above + (rank[e] >> 16) - 1)] = make_int4(e, r0 + 256 * nf, rem, 0);
            if (e >= all) D4[q * E + e] = make_int4(-1, 0, 0, 0);
        }
        if (!cls) continue;
        int at = fincl[e] - nf - (rem > 128);
        for (int j = 0; j < nf; ++j) tall[at++] = make_int4(e, r0 + 256 * j, 256, slot1);
        if (rem > 128) tall[at] = make_int4(e, r0 + 256 * nf, rem, slot1);
    }
    for (int i = fincl[E - 1] + threadIdx.x; i < cap; i += blockDim.x) tall[i] = make_int4(-1, 0, 0, 0);
}

int launch_pf_plan(const int32_t* counts, int E, int row_lo, int nrows, int32_t* tiles, int cap, int32_t* hot, int hot_min, int hot_cap, int32_t* wide, int wide_min, const int64_t* table,
                   int32_t* dense, const int64_t* rows, hipStream_t st)
{
    nq_pf_plan_k<<<1, 256, 4 * E * sizeof(int), st>>>(counts, E, row_lo, nrows, tiles, cap, hot, hot_min, hot_cap, wide, wide_min, table, dense, rows);
    NQ_LAUNCH_CHECK("nq_pf_plan");
    return 0;
}

// ---- decoded-weight scratch of hot experts --------------------------------------------------------------------------------
// An expert with many pair rows is cut into several 256-row tiles, and every tile's workgroups would decode the expert again.
// Such experts are decoded once per call instead, into fp16 scratch laid out as MFMA A operands: for strip pair sp (32 weight rows),
// chunk c, MFMA (mm, rho) one 1 KB block of 64 lanes x 16 bytes. nq_pf_wide_k multiplies them.
// Slot k of the scratch holds gate|up ([2I / 32][H / 128][8] blocks) followed by down ([H / 32][I / 128][8] blocks).
__device__ __forceinline__ size_t wop_base(int slot, int mode, int H, int I)
{   // in 16-byte units
    const size_t gu = (size_t)(2 * I / 32) * (H / 128) * 8 * 64, dn = (size_t)(H / 32) * (I / 128) * 8 * 64;
    return (size_t)slot * (gu + dn) + (mode ? gu : 0);
}

// chunks c0 .. c1 - 1 of one strip pair; dst: the strip pair's blocks
template <bool RES, int CODE>
__device__ __forceinline__ void wdecode_chunks(const Planes& P, const LaneCtx& L, int c0, int c1, u32x4* dst, int lane)
{
    constexpr int NW = RES ? Rec<CODE>::NW : 1;
    u32x4 nb;
    uint32_t nr[NW + 2] = {0}, ndw = 0, nvar = 0;
    auto request = [&](int c) {
        nb = load_base<0>(P, L.rec0 + (uint32_t)c * 32, L.nrec);
        if constexpr (RES) { load_record<CODE>(nr, P.res, L.rec0 + (uint32_t)c * 32, L.nrec); ndw = at_offset<uint32_t>((gp_u8)P.dw, (L.unit0 + c) * 4u); }
        if (P.var) nvar = at_offset<uint8_t>(P.var, L.unit0 + c);
    };
    request(c0);
    for (int c = c0; c < c1; ++c)
    {
        uint32_t wb[6], wr[NW + 2];
        wb[0] = nb.x; wb[1] = nb.y; wb[2] = nb.z; wb[3] = nb.w;
#pragma unroll
        for (int i = 0; i < NW; ++i) wr[i] = nr[i];
        const uint32_t dw = ndw, var = nvar;
        if (c + 1 < c1) request(c + 1);
        ext_base<0>(wb, __shfl(wb[0], L.src));
        const uint32_t sgm = ((var >> L.g) & 1u) * 0x80008000u;
        FoldK k;
        if constexpr (RES) { prepare_record<CODE>(wr); ext_words<Rec<CODE>::BITS, Rec<CODE>::NW>(wr, __shfl(wr[0], L.src)); k = consts_fold(dw, sgm); }
        else k = consts_l2(sgm);
        u32x4* d = dst + (size_t)c * 8 * 64 + lane;
        static_for<4>([&](auto mm) {
            constexpr int MM = decltype(mm)::value;
            d[(MM * 2 + 0) * 64] = __builtin_bit_cast(u32x4, a_operand<RES, CODE, MM, 0>(wb, wr, k));
            d[(MM * 2 + 1) * 64] = __builtin_bit_cast(u32x4, a_operand<RES, CODE, MM, 1>(wb, wr, k));
        });
    }
}

// grid (N / 128, k-slices, slots), block 256: 128 weight rows x WDEC_CHUNKS chunks of the expert with scratch slot slot0 + blockIdx.z, if its row is
// of the common kind (K = 2 base plane, no mask-mode flags; others keep decoding inside the GEMM, whatever hot[] says). Bound by its writes:
// 16 experts' down projections 89 us = 4.5 TB/s (a whole row of chunks per wavefront: 126 us, too few in flight); gate|up beside other launches 3.5 TB/s.
// tiles (may be null): the number of tiles of decoded weights.
constexpr int WDEC_CHUNKS = 8;
__global__ void __launch_bounds__(256) nq_pf_wdecode_k(const int64_t* table, const int32_t* hot, int E, const int32_t* tiles, int mode, u32x4* Wop, int slot0, int H, int I)
{
    const int slot = slot0 + blockIdx.z;
    if (tiles && *tiles == 0) return;                            // no tile of decoded weights
    int e = -1;
    for (int i0 = 0; i0 < E && e < 0; i0 += 64)                  // every wavefront looks for itself
    {
        const int i = i0 + (threadIdx.x & 63);
        const unsigned long long m = __ballot(i < E && hot[i] == slot);
        if (m) e = i0 + __ffsll((long long)m) - 1;
    }
    if (e < 0) return;
    const int64_t* ent = table + (size_t)e * TBL_W;
    const int lv = (int)ent[0];
    if (lv <= 0) return;
    const Planes P = planes_of(ent, mode);
    if (P.bcode != 0 || P.flags != nullptr) return;
    const int lane = threadIdx.x & 63, warp = threadIdx.x >> 6;
    const int N = mode == 0 ? 2 * I : H, K = mode == 0 ? H : I, C = K / 128;
    const int c0 = blockIdx.y * WDEC_CHUNKS, c1 = min(C, c0 + WDEC_CHUNKS);
    const int sp = blockIdx.x * 4 + warp, t4 = lane >> 4, ss = (lane >> 3) & 1, g = lane & 7;
    LaneCtx L;
    L.unit0 = (uint32_t)(2 * sp + ss) * C; L.rec0 = L.unit0 * 32 + 4 * g + t4;
    L.nrec = (size_t)(N / 16) * C * 32;
    L.src = (lane + 16) & 63; L.g = g; L.xs = nullptr; L.xstep = 0;
    L.strip = (uint32_t)(2 * sp + ss); L.nstrips = (size_t)(N / 16); L.chunk0 = 0; L.half0 = (uint32_t)(2 * sp + (lane >> 5)) * C;
    u32x4* dst = Wop + wop_base(slot, mode, H, I) + (size_t)sp * C * 8 * 64;
    if (lv == 2) wdecode_chunks<false, 0>(P, L, c0, c1, dst, lane);
    else dispatch_code(P.code, [&](auto tag) { wdecode_chunks<true, decltype(tag)::value>(P, L, c0, c1, dst, lane); });
}

int launch_pf_wdecode(const int64_t* table, const int32_t* hot, int E, const int32_t* tiles, int mode, void* Wop, int slots, int H, int I, hipStream_t st)
{
    const int N = mode == 0 ? 2 * I : H, C = (mode == 0 ? H : I) / 128;
    for (int s0 = 0; s0 < slots; s0 += 65535)                    // what a grid's third dimension holds
    {
        nq_pf_wdecode_k<<<dim3(N / 128, (C + WDEC_CHUNKS - 1) / WDEC_CHUNKS, std::min(slots - s0, 65535)), 256, 0, st>>>(table, hot, E, tiles, mode, (u32x4*)Wop, s0, H, I);
        NQ_LAUNCH_CHECK("nq_pf_wdecode");
    }
    return 0;
}

// ---- grouped GEMM over decoded weights --------------------------------------------------------------------------------------
struct PfWide
{
    const int64_t* table; const int32_t* tiles; const int32_t* count;      // count: tiles in the list, or null: `ntiles`
    const _Float16* A0; const _Float16* A1; float* C; const u32x4* Wop; int mode, E, H, I, ntiles;
};
constexpr int WIDE_GRID = 512;                                  // workgroups, one per CU at a time; most steps have fewer units than they might
constexpr int WIDE_STAGES = 4, WIDE_GROUP = 4;                   // stages of 32 columns in LDS; tiles that share column blocks at a time
constexpr uint32_t WIDE_HALF = 16384, WIDE_STAGE = 2 * WIDE_HALF; // LDS bytes of a stage: weights, then tokens

__device__ __forceinline__ void to_lds2(const void* base, uint32_t off, uint32_t at)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024" :: "s"(at), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ half8_t from_lds(uint32_t at) { return *(const __attribute__((address_space(3))) half8_t*)(uintptr_t)at; }
// slot of a token row's four 16-byte columns of a stage: q ^ wide_swizzle(row), without bank conflicts for the operand reads
__device__ __forceinline__ int wide_swizzle(int row) { return ((row >> 2) & 1) * 2 ^ ((row >> 3) & 1) * 3; }

__device__ __forceinline__ void wide_unit(const PfWide& a, int unit, int nt, int ncol, int nb, char* smem)
{
    const int grp = unit / (WIDE_GROUP * ncol), in = unit - grp * WIDE_GROUP * ncol, gt = min(WIDE_GROUP, nt - WIDE_GROUP * grp);
    const int bx = in / gt, t = WIDE_GROUP * grp + in % gt;
    const int e = a.tiles[4 * t], row0 = a.tiles[4 * t + 1], nrows = a.tiles[4 * t + 2], slot = a.tiles[4 * t + 3] - 1;
    if (e < 0 || e >= a.E || nrows <= 0 || slot < 0) return;
    const int64_t* ent = a.table + (size_t)e * TBL_W;
    if ((int)ent[0] <= 0) return;
    const Planes P = planes_of(ent, a.mode);
    if (P.bcode != 0 || P.flags != nullptr) return;              // decoded inside nq_pf_gemm_k
    const int N = a.mode == 0 ? 2 * a.I : a.H, K = a.mode == 0 ? a.H : a.I, S = K / 32;
    const bool upper = a.mode == 0 && bx >= nb;                  // the up half has activations of its own
    const int w0 = a.mode == 0 ? (upper ? a.I + 256 * (bx - nb) : 256 * bx) : 256 * bx;
    const int mrows = min(256, (a.mode == 0 ? (upper ? 2 * a.I : a.I) : a.H) - w0);       // 128 or 256
    const int lane = threadIdx.x & 63, warp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t4 = lane >> 4, n = lane & 15;
    const int wm = warp & 1, wn = warp >> 1;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    // wavefront w brings strip pair w (beyond the block: the last one again) and pair rows 32 w .. 32 w + 31 (beyond the tile: its last row again)
    const char* wsrc = (const char*)(a.Wop + wop_base(slot, a.mode, a.H, a.I)) + (size_t)(w0 / 32 + min(warp, mrows / 32 - 1)) * S * 2048;
    const char* tsrc = (const char*)((upper ? a.A1 : a.A0) + (size_t)row0 * K);
    const uint32_t woff = lane * 16;
    uint32_t toff[2];
#pragma unroll
    for (int q = 0; q < 2; ++q)
        toff[q] = (uint32_t)min(32 * warp + 16 * q + (lane >> 2), nrows - 1) * K * 2 + (uint32_t)(((lane & 3) ^ wide_swizzle(lane >> 2)) * 16);
    auto fetch = [&](int s, uint32_t stage) {                    // stages beyond the last repeat it, so that every wait below counts the same loads
        s = s < S ? s : S - 1;
        to_lds2(wsrc + (size_t)s * 2048, woff, stage + warp * 2048);
#pragma unroll
        for (int q = 0; q < 2; ++q) to_lds(tsrc + (size_t)s * 64, toff[q], stage + WIDE_HALF + warp * 2048 + q * 1024);
    };
    float4_t acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    const uint32_t aoff = wm * 8192 + lane * 16, boff = WIDE_HALF + (64 * wn + n) * 64 + ((t4 ^ wide_swizzle(n)) << 4);
#pragma unroll
    for (int s = 0; s < WIDE_STAGES - 1; ++s) fetch(s, lds0 + s * WIDE_STAGE);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"(4 * (WIDE_STAGES - 2)) : "memory");
    if (warp >= 4) asm volatile("s_barrier" ::: "memory");       // half a stage behind from here on; wavefronts 0 .. 3 make up for it at the end
    uint32_t cur = lds0, prev = lds0 + (WIDE_STAGES - 1) * WIDE_STAGE;
    for (int s = 0; s < S; ++s)
    {
        half8_t A[8], B[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) B[j] = from_lds(cur + boff + j * 1024);
#pragma unroll
        for (int i = 0; i < 8; ++i) A[i] = from_lds(cur + aoff + i * 1024);
        fetch(s + WIDE_STAGES - 1, prev);                        // everybody has read stage s - 1
        // this wavefront's share of stage s + 1 has landed, and its operands of stage s are in registers
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(4 * (WIDE_STAGES - 2)) : "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[i], B[j], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        prev = cur;
        cur = cur + WIDE_STAGE == lds0 + WIDE_STAGES * WIDE_STAGE ? lds0 : cur + WIDE_STAGE;
    }
    if (warp < 4) asm volatile("s_barrier" ::: "memory");
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");  // the repeated loads have landed: LDS is free for the next unit, or for somebody else
    if (128 * wm >= mrows) return;
    // lane (t4, n) holds, for pair row 16 j + n, weight rows 32 (i / 2) + 8 (i & 1) + 16 (t4 >> 1) + 4 (t4 & 1) + 0 .. 3
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        const int tok = 64 * wn + 16 * j + n;
        if (tok >= nrows) continue;
        float* c = a.C + (size_t)(row0 + tok) * N + w0 + 128 * wm + 16 * (t4 >> 1) + 4 * (t4 & 1);
#pragma unroll
        for (int i = 0; i < 8; ++i) *(float4_t*)(c + 32 * (i >> 1) + 8 * (i & 1)) = acc[i][j];
    }
}
// The tiles of experts whose weights nq_pf_wdecode_k has laid out. A unit = 256 weight rows x a tile of at most 256 pair rows, one workgroup of
// eight wavefronts, each 128 weight rows x 64 pair rows (128 accumulators). Both operands pass through LDS in stages of 32 columns (one MFMA deep),
// requested three stages ahead. Wavefronts w and w + 4 share a SIMD and work half a stage apart: one multiplies while the other reads its
// operands and requests the next stage, so the matrix pipe always has a wavefront with its operands at hand (without that, all eight reading ahead
// in step: 126 instead of 110 us for 64 units of 6144 columns on an otherwise idle GPU). Products and their order are those of the decode-fused
// tiles, so are the bits. 16 experts of 2048 rows, 6144 x 2048, in a row of steps: gate|up 1.54 ms and down 0.88 = 1070 / 940 TFLOP/s at the 1.4 GHz that the
// power limit leaves; launches apart from one another (profiles/prefill_gemm_counters.txt) 1.39 and 0.83 ms at 1.9 to 2.0 GHz, the matrix pipe busy
// 57 and 49 % of the clocks. A clock 40 % higher gives 10 %, so what bounds it is not the clock alone; the order of products and the number of stages
// or of wavefronts made no difference, 32 x 32 products were 6 % slower (the same bits). 18.9 us per 256 rows, where a decode-fused tile takes
// 29.5 at level 4 and 23 at level 2. Its weights have to be decoded first: 17 us an expert.
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) nq_pf_wide_k(PfWide a)
{
    extern __shared__ __align__(16) char smem[];
    const int nb = (a.I + 255) / 256, ncol = a.mode == 0 ? 2 * nb : (a.H + 255) / 256;
    const int nt = a.count ? *a.count : a.ntiles, units = nt * ncol;
    if (!a.count)
    {   // a list of the caller's, nq_pf_plan's with its gaps: units dealt out one by one, or a few XCDs have all tiles. gate|up of 98 tiles in 385
        // places, 78 of them of decoded weights, 3226 us in runs, 1514 so
        for (int unit = blockIdx.x; unit < units; unit += gridDim.x) wide_unit(a, unit, nt, ncol, nb, smem);
        return;
    }
    // An XCD works through a run of neighbouring units: WIDE_GROUP tiles by one column block after the other
    const int per = (units + 7) / 8, first = (int)(blockIdx.x & 7) * per;
    for (int unit = first + (int)(blockIdx.x >> 3); unit < min(units, first + per); unit += (int)gridDim.x >> 3)
        wide_unit(a, unit, nt, ncol, nb, smem);
}

static int launch_wide(const PfWide& a, int most, hipStream_t st)
{
    const int shm = WIDE_STAGES * WIDE_STAGE, ncol = a.mode == 0 ? 2 * ((a.I + 255) / 256) : (a.H + 255) / 256;
    const hipError_t e = hipFuncSetAttribute((const void*)nq_pf_wide_k, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
    if (e != hipSuccess) return set_error("nq_pf_wide: LDS %d bytes: %s", shm, hipGetErrorString(e));
    nq_pf_wide_k<<<(int)std::min<int64_t>(WIDE_GRID, ((int64_t)most * ncol + 7) / 8 * 8), 512, shm, st>>>(a);
    NQ_LAUNCH_CHECK("nq_pf_wide");
    return 0;
}

// ---- pairs sorted by expert ----------------------------------------------------------------------------------------------
// One launch in place of a library sort, its gathers and the counting scatter. Every workgroup counts all picks in LDS, those before its
// own share of the pairs apart, so that it knows where its pairs of an expert begin without waiting for another workgroup; then it ranks its
// pairs, 512 at a time, one per lane: within a wavefront by the ids' bits, between wavefronts by taking turns at the experts' cursors.
// Rows of an expert are in pair order. Picks outside [0, E) form a last group of rows of no expert (pe = -1), which every later kernel
// passes over. One workgroup more writes the counts, the hits and the tile list of nq_pf_short_k: at most 64 rows per tile, experts above
// level 2 first (their tiles take twice as long, so they start first), unused entries -1.
// Bound by the counting's LDS atomics beyond a few thousand pairs, by latency below. us at 384 / 1608 / 8024 / 32768 pairs of 256 experts: 7.7 / 8.3 / 10.2 / 20.2, where
// eight experts a workgroup, each gathered by one wavefront that looked at every pair, took 10.7 / 11.9 / 21.1 / 89.7.
constexpr int SORT_BLOCK = 512, SORT_WGS = 256;
struct PfSort
{
    const void* sel; const void* rw; int sdt, wdt; int P, topk, E;
    const int64_t* table; int32_t* cnt; int32_t* pe; int32_t* pt; int32_t* pos; int* hits; int32_t* tiles; int cap;
    int per;                                                     // blocks of SORT_BLOCK pairs per workgroup
};
__global__ void __launch_bounds__(1024) nq_pf_sort_k(PfSort a)
{
    extern __shared__ int sort_sh[];
    const int E1 = a.E + 1, tid = threadIdx.x, lane = tid & 63, warp = tid >> 6;
    int *bef = sort_sh, *tot = bef + E1, *ext = tot + E1;       // pairs before this workgroup's, all pairs, scans
    const bool list = blockIdx.x == gridDim.x - 1;               // block-uniform
    const int begin = list ? a.P : min((int64_t)a.P, (int64_t)blockIdx.x * a.per * SORT_BLOCK), end = min((int64_t)a.P, (int64_t)begin + a.per * SORT_BLOCK);
    auto id_of = [&](int i) { const long long e = id_at(a.sel, a.sdt, i); return e >= 0 && e < a.E ? (int)e : a.E; };
    int id = tid < SORT_BLOCK && begin + tid < end ? id_of(begin + tid) : -1;        // requested before the counting
    int lv[4] = {};                                              // levels of experts tid + 1024 k (E <= 4096)
    if (list && a.tiles)
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (tid + 1024 * k < a.E) lv[k] = (int)a.table[(size_t)(tid + 1024 * k) * TBL_W];
    for (int e = tid; e < E1; e += 1024) { bef[e] = 0; tot[e] = 0; ext[e] = 0; }
    __syncthreads();
    for (int64_t i0 = tid; i0 < a.P; i0 += 8 * 1024)
    {
        int e[8]; bool hit[8];                                   // eight in flight before the first is counted
#pragma unroll
        for (int u = 0; u < 8; ++u)
        {
            const int64_t i = i0 + 1024 * u;
            e[u] = i < a.P ? id_of((int)i) : -1;
            hit[u] = list && a.hits && i < a.P && w_at(a.rw, a.wdt, i) != 0.f;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
        {
            if (e[u] >= 0) atomicAdd((i0 + 1024 * u < begin ? bef : tot) + e[u], 1);
            if (hit[u]) atomicAdd(ext + e[u], 1);
        }
    }
    __syncthreads();
    if (list && a.hits)
        for (int e = tid; e < a.E; e += 1024)
            if (ext[e]) __hip_atomic_fetch_add(a.hits + e, ext[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    for (int e = tid; e < E1; e += 1024) ext[e] = tot[e] += bef[e];
    __syncthreads();
    block_scan(ext, E1);
    if (!list)
    {
        for (int e = tid; e < E1; e += 1024) bef[e] += ext[e] - tot[e];              // row of the expert's next pair here
        const int bits = 32 - __builtin_clz(a.E);
        for (int p0 = begin; p0 < end; p0 += SORT_BLOCK)
        {
            if (p0 > begin) id = tid < SORT_BLOCK && p0 + tid < end ? id_of(p0 + tid) : -1;
            unsigned long long same = __ballot(id >= 0);         // the lanes with this lane's id
            for (int b = 0; b < bits; ++b)
            {
                const unsigned long long m = __ballot((id >> b) & 1);
                same &= ((id >> b) & 1) ? m : ~m;
            }
            const int before = __popcll(same & ((1ull << lane) - 1ull));
            int row = 0;
            for (int w = 0; w < SORT_BLOCK / 64; ++w)
            {
                __syncthreads();
                if (w == warp && id >= 0 && before == 0) { row = bef[id]; bef[id] = row + __popcll(same); }
            }
            row = __shfl(row, id >= 0 ? __ffsll((long long)same) - 1 : lane) + before;
            if (id >= 0)
            {
                const int pair = p0 + tid;
                a.pos[pair] = row; a.pt[row] = pair / a.topk; a.pe[row] = id < a.E ? id : -1;
            }
        }
        return;
    }
    for (int e = tid; e < a.E; e += 1024) a.cnt[e] = tot[e];
    if (!a.tiles) return;
    // per class (0: above level 2, 1: level 2) a scan of the tile counts
    int4* T4 = (int4*)a.tiles;
    int* nt = bef;
    int base = 0;
    for (int cls = 0; cls < 2; ++cls)
    {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            const int x = tid + 1024 * k;
            if (x < a.E) nt[x] = lv[k] > 0 && (lv[k] > 2) == (cls == 0) ? (tot[x] + SHORT_ROWS - 1) / SHORT_ROWS : 0;
        }
        __syncthreads();
        block_scan(nt, a.E);
        for (int x = tid; x < a.E; x += 1024)
        {
            const int k = nt[x] - (x ? nt[x - 1] : 0), at = base + nt[x] - k, n = tot[x], start = ext[x] - n;
            for (int q = 0; q < k; ++q)
                T4[at + q] = make_int4(x, start + SHORT_ROWS * q, n - SHORT_ROWS * q < SHORT_ROWS ? n - SHORT_ROWS * q : SHORT_ROWS, 0);
        }
        base += nt[a.E - 1];
    }
    for (int i = base + tid; i < a.cap; i += 1024) T4[i] = make_int4(-1, 0, 0, 0);
}

// pair rows per workgroup of the row kernels: what leaves about two thousand workgroups (eight per CU), at most eight
static int row_group(int np, int parts) { return std::min(MID_ROWS, std::max(1, (int)((int64_t)np * parts / 2048))); }
int launch_pf_pre(const void* x, int xdt, const int32_t* pt, const int32_t* pe, int np, const int64_t* table, void* xg, void* xu, float* zg, int E, int H, int I,
                  const int32_t* tiles, int cap, int heights, hipStream_t st)
{
    if (!np) return 0;
    const int parts = (H / 128 + 15) / 16, rows = row_group(np, parts);
    nq_pf_pre_k<<<dim3((np + rows - 1) / rows, parts), 256, 0, st>>>(x, xdt, pt, pe, np, rows, table, (_Float16*)xg, (_Float16*)xu, zg, E, H, I, tiles, cap, heights);
    NQ_LAUNCH_CHECK("nq_pf_pre");
    return 0;
}
int launch_pf_mid(const float* acc_gu, const int32_t* pe, int np, const int64_t* table, void* h, const float* zg, float* zd, int E, int H, int I,
                  const int32_t* tiles, int cap, int heights, hipStream_t st)
{
    if (!np) return 0;
    const int rows = row_group(np, 1);
    nq_pf_mid_k<<<(np + rows - 1) / rows, 256, 0, st>>>(acc_gu, pe, np, rows, table, (_Float16*)h, zg, zd, E, H, I, tiles, cap, heights);
    NQ_LAUNCH_CHECK("nq_pf_mid");
    return 0;
}
int launch_pf_post(const float* y, const int32_t* pos, const void* sel, int sdt, const void* rw, int wdt, int T, int topk, int row_lo, int nrows,
                   const int64_t* table, void* out, int odt, int add, const float* zd, int E, int H, int I, hipStream_t st)
{
    if (!T || (!nrows && add)) return 0;
    // few tokens: one wavefront per segment of 512 columns, each a workgroup of its own, so that every CU has some
    const int segs = (H / 128 + 3) / 4;
    const dim3 grid = T >= 1024 ? dim3(T, 1) : dim3(T, segs);
    nq_pf_post_k<<<grid, T >= 1024 ? 256 : 64, 0, st>>>(y, pos, sel, sdt, rw, wdt, topk, row_lo, nrows, table, out, odt, add, zd, E, H, I);
    NQ_LAUNCH_CHECK("nq_pf_post");
    return 0;
}
int launch_pf_hits(const int32_t* counts, int32_t* hits, int E, hipStream_t st)
{
    nq_pf_hits_k<<<(E + 255) / 256, 256, 0, st>>>(counts, hits, E);
    NQ_LAUNCH_CHECK("nq_pf_hits");
    return 0;
}

int launch_pf_gemm(const int64_t* table, const int32_t* tiles, int ntiles, int bm, int mode, const void* A0, const void* A1, float* C,
                   int E, int H, int I, int wide, hipStream_t st)
{
    if (!ntiles) return 0;
    if (bm != 16 && bm != 32 && bm != 64 && bm != 128 && bm != 256) return set_error("nq_pf_gemm: tile height %d not in {16, 32, 64, 128, 256}", bm);
    const PfGemm a{table, tiles, (const _Float16*)A0, (const _Float16*)A1, C, mode & 1, E, H, I, (mode & 4) != 0, wide};
    return mode & 2 ? launch_tiles<true>(a, bm, ntiles, st) : launch_tiles<false>(a, bm, ntiles, st);
}

int launch_pf_wide(const int64_t* table, const int32_t* tiles, int ntiles, int mode, const void* A0, const void* A1, float* C, int E, int H, int I, const void* Wop, hipStream_t st)
{
    if (!ntiles) return 0;
    return launch_wide(PfWide{table, tiles, nullptr, (const _Float16*)A0, (const _Float16*)A1, C, (const u32x4*)Wop, mode & 1, E, H, I, ntiles}, ntiles, st);
}

// ---- a whole step --------------------------------------------------------------------------------------------------------
// Bytes of the int32 scratch of a step: cnt [E] | pe [P] | pt [P] | pos [P] | hot [E] | tile lists | tiles of decoded weights | tiles without gaps, each on 16 bytes.
struct PfMeta { int32_t *cnt, *pe, *pt, *pos, *hot, *tiles, *wide, *dense; int cap, scap; size_t bytes; };
static PfMeta pf_meta(void* ws, int P, int R, int E)
{
    PfMeta m;
    size_t off = 0;
    auto take = [&](size_t n) { int32_t* p = (int32_t*)((char*)ws + off); off += (n * 4 + 15) & ~(size_t)15; return p; };
    m.cap = E + R / 256 + 1; m.scap = E + P / SHORT_ROWS + 1;
    m.cnt = take(E); m.pe = take(P); m.pt = take(P); m.pos = take(P); m.hot = take(E);
    m.tiles = take(4 * (size_t)(5 * m.cap > m.scap ? 5 * m.cap : m.scap)); m.wide = take(4 * ((size_t)m.cap + 1)); m.dense = take(4 * (2 * (size_t)E + m.cap));
    m.bytes = off;
    return m;
}

// Which steps take the one-launch plan of short tiles. An expert of n rows is decoded n / 64 times there, n / 256 times by the tall
// tiles, which cost a launch more to list them, two or three for every one of the other plan, and the events of the side streams. us short / tall:
//   few rows per expert (E = 256 of 6144 x 2048, top-8): 200 tokens, level 4, evenly 2387 / 2400, Zipf(1.1) popularity 2196 / 2169; 400 tokens
//   2465 / 2477 and 2579 / 2451; 1000 tokens 2850 / 2865 and 3319 / 2970, of mixed levels 2014 / 2043 and 2313 / 2135. The line is where
//   popular experts begin to take several short tiles, at 8 rows an expert on average: beyond it up to 1.5 % lost evenly, 4 to 10 gained.
//   little work beside what the plan costs (a decode's price goes with H I): up to rows * H * I = 2^32 always (1000 tokens, 16 experts of 512 x 256
//   85 / 115; 50 tokens, 8 of 6144 x 2048 156 / 190), up to 2^34 unless the average expert has more than 96 rows, two tiles (400 tokens, 64 of
//   2048 x 1024 220 / 250; 170 tokens, 16 of 6144 x 2048, Zipf 288 / 308; 32 370 / 385, 455 / 500; but 130 tokens, 8 330 / 232; 3000 tokens, 64 of 1024 x
//   512 209 / 187).
// Without side streams the chains follow one another, and the lines lie at 32 rows an expert and at 2^35: 200 tokens, 64 experts, Zipf 580 / 695, 300
// 698 / 743; 400 tokens, 256 experts 2546 / 2559, 1000 2323 / 2200 and evenly 2011 / 2030; 170 tokens, 16 experts 300 / 433. Beyond them 383 tokens, 16
// experts 729 / 690 and evenly 740 / 466; 683, 64 experts 1364 / 1245 and 1462 / 1040.
static bool pf_is_short(int64_t P, int E, int H, int I, bool fork)
{
    const int64_t work = P * H * I;
    return P <= (fork ? 8 : 32) * (int64_t)E || work <= (int64_t)1 << 32 || (P <= 96 * (int64_t)E && work <= (int64_t)1 << (fork ? 34 : 35));
}

// Which experts take decoded weights: at least WIDE_MIN rows (two and a half tiles), above level 2, if their tiles make WIDE_UNITS units of gate|up
// together (two per CU; the plan counts them). us a step from 512 / 640 / 768 / 1024 rows on (6144 x 2048, top-8, level 4): 4096 tokens, 256
// experts, Zipf 5198 / 5260 / 5300 / 5222; 64 experts, Zipf 4002 / 3890 / 3962 / 3896; 32, evenly 3656 / 3665 / 3666 / 3850; 16, Zipf 3270 / 3275 / 3268 / 3484;
// 2000 tokens, 64 experts, Zipf 2190 / 2210 / 2225 / 2220; 16, evenly 1791 / 1792 / 1793 / 1892: 640 and 768 cannot be told apart. Without decoded
// weights / by this rule, in turn on one box, two routings: 4096 tokens, 256 experts, Zipf 5503 / 5378 and 5433 / 5304; 64 4091 / 3935, 4100 / 4028; 32,
// evenly 3891 / 3698, 3923 / 3739; 16, Zipf 3833 / 3311, 3858 / 3634; 2000 tokens, 16, evenly 1902 / 1788, 1923 / 1800; of 2048 x 2048, 4096 tokens
// 1439 / 1285, 1454 / 1294. Where the sizes allow it but the planner then finds too few tiles, the four launches that do nothing cost up to 25 us, most in
// small steps: 256 experts of mixed levels, Zipf 4286 / 4326; 2000 tokens, 64 experts, Zipf 2211 / 2240; 4096, 16 experts, 2 picks 1085 / 1099. At level 2, where a tile's decode is half as long, 16 experts of 2048 rows lose: 3173 / 3281.
// Fewer units leave CUs idle for the 0.2 ms of one: 1000 tokens, 16 experts, Zipf (a single expert of 993 rows) 1070 / 1173.
// A block of 128 weight rows costs what one of 256 does: 2304 + 4096 rows, 11 % of them padding in gate|up, 1922 / 1961. Scratch: 2 GB at most.
constexpr int WIDE_MIN = 640, WIDE_UNITS = 512;
constexpr int64_t WIDE_BYTES = (int64_t)1 << 31;
static int wide_tiles(int I) { const int ncol = 2 * ((I + 255) / 256); return (WIDE_UNITS + ncol - 1) / ncol; }

int launch_pf_step(const NqPfArgs& a, hipStream_t st)
{
    const int P = a.T * a.topk, R = a.rows < P ? a.rows : P, E = a.E, H = a.H, I = a.I;
    const int variants = a.variants & 3;
    const bool advised = a.variants & 4;
    const PfMeta m = pf_meta(a.meta, P, R, E);
    if (m.bytes > (size_t)a.meta_bytes) return set_error("nq_pf_step: meta needs %zu bytes, has %lld", m.bytes, (long long)a.meta_bytes);
    const bool fork = a.side[0] != nullptr, brief = R == P && !a.wop && pf_is_short(P, E, H, I, fork);
    {
        const int blocks = (int)(((int64_t)P + SORT_BLOCK - 1) / SORT_BLOCK), per = (blocks + SORT_WGS - 1) / SORT_WGS;
        const PfSort s{a.sel, a.rw, a.sel_dtype, a.rw_dtype, P, a.topk, E, a.table, m.cnt, m.pe, m.pt, m.pos, a.hits, brief ? m.tiles : nullptr, m.scap, per};
        const int shm = 3 * (E + 1) * 4;
        if (shm > 48 * 1024)
        {
            const hipError_t e = hipFuncSetAttribute((const void*)nq_pf_sort_k, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
            if (e != hipSuccess) return set_error("nq_pf_sort: LDS %d bytes: %s", shm, hipGetErrorString(e));
        }
        nq_pf_sort_k<<<(per ? (blocks + per - 1) / per : 0) + 1, 1024, shm, st>>>(s);
        NQ_LAUNCH_CHECK("nq_pf_sort");
    }
    float *acc = (float*)a.acc, *y = (float*)a.y;
    if (brief)
    {
        if (int rc = launch_pf_pre(a.x, a.x_dtype, m.pt, m.pe, P, a.table, a.xg, a.xu, a.zg, E, H, I, nullptr, 0, 0, st)) return rc;
        for (int mode = 0; mode < 2; ++mode)
        {
            const PfGemm g{a.table, m.tiles, (const _Float16*)(mode ? a.h : a.xg), (const _Float16*)(mode ? nullptr : a.xu), mode ? y : acc, mode, E, H, I, variants == 1, 0};
            if (variants & 1) if (int rc = launch_tiles<false>(g, SHORT_LIST, m.scap, st)) return rc;
            if (variants & 2) if (int rc = launch_tiles<true>(g, SHORT_LIST, m.scap, st)) return rc;
            if (mode == 0) if (int rc = launch_pf_mid(acc, m.pe, P, a.table, a.h, a.zg, a.zd, E, H, I, nullptr, 0, 0, st)) return rc;
        }
        return launch_pf_post(y, m.pos, a.sel, a.sel_dtype, a.rw, a.rw_dtype, a.T, a.topk, 0, P, a.table, a.out, a.out_dtype, 0, a.zd, E, H, I, st);
    }
    // Tile heights 256 | 128 | up to 64 as three chains: the tallest on the caller's stream, the others on side streams between two
    // events. A GEMM launch ends with the GPU partly idle while its last workgroups drain; the chains fill each other's tails, and
    // the memory-bound kernels of one height run under the GEMMs of another. The tiles of up to 64 rows are one launch over one list.
    // Without side streams the chains follow one another on the caller's. us a step as four chains over five lists with a place for every expert / as
    // now: 1000 tokens, 256 experts, level 4, Zipf 2835 / 2760, evenly 2745 / 2665; 4096 tokens of mixed levels 4195 / 4000; 170 tokens, 8 experts
    // 335 / 261; without side streams 1000 tokens, 16 experts 1353 / 1165, 2000, 64 experts 2793 / 2330. With the tallest on a side stream and
    // the rest on the caller's 170 tokens, 8 experts took 328.
    // The activations are prepared for all rows in one launch (a launch per height, each passing over the others' rows, 315 us in place of 261); so is h where nothing runs beside it.
    constexpr int CHAINS = 3;
    static const int heights[CHAINS] = {16, 8, 7};               // bit k = height 16 << k
    hipStream_t streams[CHAINS] = {st, st, st};
    for (int i = 1; fork && i < CHAINS; ++i) streams[i] = (hipStream_t)a.side[i - 1];
    auto hip_ok = [](hipError_t e) { return e == hipSuccess ? 0 : set_error("nq_pf_step: %s", hipGetErrorString(e)); };
    for (int c = 0; c < P; c += R)
    {
        const int n = P - c < R ? P - c : R;
        const bool wop = a.wop && n >= a.hot_min;
        if (int rc = launch_pf_plan(m.cnt, E, c, n, m.tiles, m.cap, wop ? m.hot : nullptr, a.hot_min, a.wop_slots, wop ? m.wide : nullptr, advised ? wide_tiles(I) : 0, advised ? a.table : nullptr,
                                    m.dense, a.table, st)) return rc;
        const int most = std::min(m.cap, n / 256 + a.wop_slots / 2 + 1);       // tiles of decoded weights: an expert of r rows has (r + 127) / 256
        if (int rc = launch_pf_pre(a.x, a.x_dtype, m.pt + c, m.pe + c, n, a.table, a.xg, a.xu, a.zg, E, H, I, nullptr, 0, 0, st)) return rc;
        if (fork) if (int rc = hip_ok(hipEventRecord((hipEvent_t)a.events[0], st))) return rc;
        for (int i = 1; fork && i < CHAINS; ++i) if (int rc = hip_ok(hipStreamWaitEvent(streams[i], (hipEvent_t)a.events[0], 0))) return rc;
        auto gemms = [&](int mode) {
            const int32_t* lists[CHAINS] = {m.dense + 8 * (size_t)E, m.dense + 4 * (size_t)E, m.dense};
            const int counts[CHAINS] = {std::min(m.cap, n / 129), std::min(E, n / 65), std::min(E, n)};   // the most tiles that n rows make, all inside the list
            for (int i = 0; i < CHAINS; ++i)
            {
                static const int bm[CHAINS] = {256, 128, SHORT_LIST};
                const PfGemm g{a.table, lists[i], (const _Float16*)(mode ? a.h : a.xg), (const _Float16*)(mode ? nullptr : a.xu), mode ? y : acc, mode, E, H, I, variants == 1, wop};
                if (!counts[i]) continue;
                if (variants & 1) if (int rc = launch_tiles<false>(g, bm[i], counts[i], streams[i])) return rc;
                if (variants & 2) if (int rc = launch_tiles<true>(g, bm[i], counts[i], streams[i])) return rc;
            }
            if (wop) if (int rc = launch_pf_wdecode(a.table, m.hot, E, m.wide, mode, a.wop, std::min(a.wop_slots, E), H, I, st)) return rc;
            if (wop)
                if (int rc = launch_wide(PfWide{a.table, m.wide + 4, m.wide, (const _Float16*)(mode ? a.h : a.xg), (const _Float16*)(mode ? nullptr : a.xu), mode ? y : acc, (const u32x4*)a.wop,
                                                mode, E, H, I, 0}, most, st)) return rc;
            return 0;
        };
        auto chains = [&]() {
            if (int rc = gemms(0)) return rc;
            for (int i = 0; i < (fork ? CHAINS : 1); ++i)
                if (int rc = launch_pf_mid(acc, m.pe + c, n, a.table, a.h, a.zg, a.zd, E, H, I, fork ? m.tiles : nullptr, m.cap, heights[i], streams[i])) return rc;
            return gemms(1);
        };
        const int failed = chains();
        for (int i = 1; fork && i < CHAINS; ++i)                 // joined in any case: the caller gives the buffers back in its stream's order
        {
            if (int rc = hip_ok(hipEventRecord((hipEvent_t)a.events[i], streams[i]))) return rc;
            if (int rc = hip_ok(hipStreamWaitEvent(st, (hipEvent_t)a.events[i], 0))) return rc;
        }
        if (failed) return failed;
        if (int rc = launch_pf_post(y, m.pos, a.sel, a.sel_dtype, a.rw, a.rw_dtype, a.T, a.topk, c, n, a.table, a.out, a.out_dtype, c != 0, a.zd, E, H, I, st)) return rc;
    }
    return 0;
}

int pf_wide_slots(int T, int P, int R, int E, int H, int I, bool fork, int* hot_min)
{
    *hot_min = WIDE_MIN;
    const int64_t real = (int64_t)3 * H * I, padded = (int64_t)512 * ((I + 255) / 256) * H + (int64_t)256 * ((H + 255) / 256) * I;
    if (T < WIDE_MIN || R / 256 < wide_tiles(I) || 20 * padded > 21 * real || (R == P && pf_is_short(P, E, H, I, fork))) return 0;
    return (int)std::min<int64_t>(std::min(E, R / WIDE_MIN), WIDE_BYTES / ((int64_t)6 * H * I));
}

int64_t pf_meta_bytes(int P, int R, int E) { return (int64_t)pf_meta(nullptr, P, R, E).bytes; }

}  // namespace nq
