// Tiles of one expert's rows, decoded and multiplied in one kernel: the bodies, kernels and launchers behind nq_prefill.hip. Compiled in parts that build
// side by side: tiles of plain experts (nq_pf_tiles.hip), of experts in mask mode or with a base window code other than 0 (nq_pf_masked.hip), and
// those of more than 128 rows of either kind (nq_pf_tall.hip).
#pragma once
#include "nq_tile.hpp"
#include "nq_host.hpp"

namespace nq {

constexpr int PF_ROW = 256;                    // LDS bytes per staged token and chunk; 16-byte column q of row r sits in slot q ^ (r & 15)
constexpr int SHORT_ROWS = 64;                 // most rows of a tile of nq_pf_short_k

struct PfGemm
{
    const int64_t* table; const int32_t* tiles;   // tiles [ntiles][4]: expert, first row, rows (<= 16 TG), unused
    const _Float16* A0; const _Float16* A1;         // activations in B-operand order: A0 for weight rows < I (or all rows of down), A1 above
    float* C; int mode, E, H, I;
    int solo;                                       // the other kernel variant will not be launched on these tiles: a tile that is its kind comes out NaN
    int wide;                                       // tiles of experts with decoded weights (fourth word > 0) are nq_pf_wide_k's
};

// 64 lanes x 16 bytes from base + off to LDS from `at` on (twice: and the next 1 KB of both). The offset of an instruction counts on both
// sides. Asm, because the compiler would wait for these loads before every LDS read that it cannot tell apart from them.
__device__ __forceinline__ void to_lds(const void* base, uint32_t off, uint32_t at)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(at), "v"(off), "s"(base) : "memory", "m0");
}

// The MFMA phase of one chunk: TG x 8 MFMAs, tokens 16 tg + n as the N dimension (rows of the last group beyond the tile multiply copies of its last
// row, whose results are never stored). Two row groups, or three where one would be left over, are interleaved so that four different
// accumulators or more separate an MFMA from the next one that depends on it, and the operand reads run one step (one mm of such a set) ahead
// of the MFMAs that use them.
template <int TG>
__device__ __forceinline__ void pf_mfmas(const half8_t (*aop)[2], const char* smem, const uint32_t* boff, float4_t (*acc)[2])
{
    constexpr int SETS = TG == 1 ? 1 : TG / 2;                   // of two row groups, the last of three if their number is odd
    half8_t bq[2][3];
    auto members = [](int set) { return TG == 1 ? 1 : set == SETS - 1 ? 2 + TG % 2 : 2; };
    auto bread = [&](int step, half8_t* dst) {
#pragma unroll
        for (int u = 0; u < 3; ++u)
            if (u < members(step / 4)) dst[u] = *(const half8_t*)(smem + boff[step % 4] + (step / 4 * 2 + u) * 16 * PF_ROW);
    };
    bread(0, bq[0]);
#pragma unroll
    for (int q = 0; q < 4 * SETS; ++q)
    {
        if (q + 1 < 4 * SETS) bread(q + 1, bq[(q + 1) % 2]);
        __builtin_amdgcn_sched_barrier(0);
        const int tg = q / 4 * 2, mm = q % 4;
#pragma unroll
        for (int u = 0; u < 3; ++u)
        {
            if (u >= members(q / 4)) break;
            const half8_t b = bq[q % 2][u];
            acc[tg + u][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(aop[mm][0], b, acc[tg + u][0], 0, 0, 0);
            acc[tg + u][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(aop[mm][1], b, acc[tg + u][1], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Token staging shared by the GEMM bodies: wavefront w copies rows 16 u + 4 w + (lane >> 4), u = 0 .. TG - 1, of the tile, one
// 1 KB global -> LDS load per u (64 lanes x 16 bytes land in LDS in lane order, so a load fills 4 rows x 256 bytes). The lane
// picks which 16-byte column of its row it fetches: column (lane & 15) ^ (row & 15) goes to slot lane & 15, and the MFMA reads
// undo the XOR, which spreads the 16 tokens of an operand read over all banks without padding. Rows beyond the tile re-read
// its last row: their products are never stored.
// PART = 0 .. 3 issues a quarter of the loads (all of them in part 0 when there are fewer than four): the decode-fused body
// spreads them over its decode, because the texture path takes 16 clocks per 1 KB load and a wavefront that issues sixteen in
// a row stalls behind its own requests (measured: 1450 clocks per chunk at 256 rows) with the record loads queued after them.
// A load's address is a scalar base (the tile's chunk and row group) and the lane's offset inside the group, one register for all groups; from the
// group that holds the tile's last row on, that group is read again with an offset that stops there. With a lane offset formed per group (a move, an
// addition, a selection, a lane read for the LDS address) the tokens of a chunk were up to 18 of 290 vector instructions at 64 rows.
struct TokenSource { const char* base; uint32_t off, last_off; int last; size_t step; uint32_t lds; };       // last: the row group of the tile's last row
__device__ __forceinline__ TokenSource token_source(const _Float16* A, int K, int row0, int nrows, const char* smem, int warp, int lane)
{
    const int srow = 4 * warp + (lane >> 4), last = (nrows - 1) >> 4;            // srow = row & 15 of every row this lane stages
    const uint32_t scol = (uint32_t)(((lane & 15) ^ srow) * 16);                 // byte offset of the fetched column inside the chunk
    return TokenSource{(const char*)(A + (size_t)row0 * K), (uint32_t)(srow * K * 2) + scol, (uint32_t)(min(srow, nrows - 1 - 16 * last) * K * 2) + scol, last,
                       (size_t)K * 32, (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)smem + (uint32_t)__builtin_amdgcn_readfirstlane(4 * warp * PF_ROW)};
}
template <int TG, int PART>
__device__ __forceinline__ void pf_stage_tokens(const TokenSource& t, int c)
{
    constexpr int U0 = TG >= 4 ? PART * TG / 4 : 0, U1 = TG >= 4 ? (PART + 1) * TG / 4 : (PART == 0 ? TG : 0);
#pragma unroll
    for (int u = U0; u < U1; ++u)
    {
        const bool whole = TG > 1 && u < t.last;                 // block-uniform
        to_lds(t.base + (size_t)c * 256 + (whole ? u : t.last) * t.step, whole ? t.off : t.last_off, t.lds + 16 * u * PF_ROW);
    }
}

// body for one (RES, CODE): all K / 128 chunks of this wave's two strips against the tile's tokens
template <int TG, bool RES, int CODE, bool MASKED, int BK = 0>
__device__ __forceinline__ void pf_chunks(const Planes& P, const LaneCtx& L, int C, const _Float16* A, int K, int row0, int nrows,
                                          char* smem, float4_t (*acc)[2])
{
    constexpr int NW = RES ? Rec<CODE>::NW : 1;
    u32x4 nb = load_base<BK>(P, L.rec0, L.nrec);
    uint32_t nr[NW + 2] = {0}, nvar = 0;
    constexpr bool masked = RES && MASKED;                       // the kernel variant for experts in mask mode
    // an expert without flags that comes through this variant (base code other than 0) reads as "every chunk refined",
    // for which the compact residual indexing is the dense one
    const uint64_t mflags = masked ? (P.flags ? P.flags[L.strip] : (C >= 64 ? ~0ull : (1ull << C) - 1ull)) : 0ull;
    if constexpr (RES && !masked) load_record<CODE>(nr, P.res, L.rec0, L.nrec);
    UnitConsts<RES> consts;                                      // mask mode works a chunk's constants out itself
    if constexpr (!masked) consts.start(unit_words(P, L, 0, C, RES));
    else if (P.var) nvar = at_offset<uint8_t>(P.var, L.unit0);
    const int lane = threadIdx.x & 63, warp = threadIdx.x >> 6, t4 = lane >> 4, n = lane & 15;
    const TokenSource tokens = token_source(A, K, row0, nrows, smem, warp, lane);
    auto stage = [&](auto part, int c) {
        if constexpr (MASKED && TG == 16)                        // two registers too many: formed anew for every part
        {
            int l = lane;
            asm volatile("" : "+v"(l));
            pf_stage_tokens<TG, decltype(part)::value>(token_source(A, K, row0, nrows, smem, warp, l), c);
        }
        else pf_stage_tokens<TG, decltype(part)::value>(tokens, c);
    };
    uint32_t boff[4];                                            // B-operand read offsets of this lane for mm = 0..3
#pragma unroll
    for (int mm = 0; mm < 4; ++mm) boff[mm] = (uint32_t)(n * PF_ROW + (((4 * mm + t4) ^ n) << 4));
    for (int c = 0; c < C; ++c)
    {
        // ---- decode this wave's unit pair of chunk c into A operands; prefetch chunk c + 1; request the tile's tokens for chunk c
        // a quarter at a time between the decode stages (asynchronous: they arrive while the decode runs)
        uint32_t wb[6], wr[NW + 2];
        wb[0] = nb.x; wb[1] = nb.y; wb[2] = nb.z; wb[3] = nb.w;
#pragma unroll
        for (int i = 0; i < NW; ++i) wr[i] = nr[i];
        uint32_t dw = 0u;
        const uint32_t var = nvar;
        bool on = true;                                          // mask mode: is chunk c refined? (the same for the whole workgroup)
        if constexpr (masked)
            {   // residual records are compact over the refined chunks and fetched when needed
                const MaskedUnit m = masked_unit(mflags, L.strip, c, L.nstrips);
                on = __builtin_amdgcn_readfirstlane((int)m.on) != 0;
                if (on) { load_record<CODE>(wr, P.res, m.unit * 32 + (L.rec0 & 31), m.nrec); dw = P.dw[m.unit]; }
            }
        if (c + 1 < C)
        {
            nb = load_base<BK>(P, L.rec0 + (uint32_t)(c + 1) * 32, L.nrec);
            if constexpr (RES && !masked) load_record<CODE>(nr, P.res, L.rec0 + (uint32_t)(c + 1) * 32, L.nrec);
            if (masked && P.var) nvar = at_offset<uint8_t>(P.var, L.unit0 + c + 1);
        }
        if constexpr (!masked) consts.begin(P, L, c, C);
        ext_base<BK>(wb, __shfl(wb[0], L.src));
        const uint32_t sgm = masked ? ((var >> L.g) & 1u) * 0x80008000u : 0u;
        half8_t aop[4][2];
        if (RES && (!masked || on))
        {
            if constexpr (RES)
            {
                prepare_record<CODE>(wr);
                ext_words<Rec<CODE>::BITS, Rec<CODE>::NW>(wr, __shfl(wr[0], L.src));
                if constexpr (masked) consts.k = consts_fold(dw, sgm); else consts.take(P, L, c);
                const FoldK& k = consts.k;
                static_for<4>([&](auto mm) {
                    constexpr int MM = decltype(mm)::value;
                    stage(mm, c);
                    aop[MM][0] = a_operand<RES, CODE, MM, 0, BK>(wb, wr, k);
                    aop[MM][1] = a_operand<RES, CODE, MM, 1, BK>(wb, wr, k);
                });
            }
        }
        else
        {
            if constexpr (masked) consts.k = consts_l2(sgm); else consts.take(P, L, c);
            const FoldK& k = consts.k;
            static_for<4>([&](auto mm) {
                constexpr int MM = decltype(mm)::value;
                stage(mm, c);
                aop[MM][0] = a_operand<false, 0, MM, 0, BK>(wb, wr, k);
                aop[MM][1] = a_operand<false, 0, MM, 1, BK>(wb, wr, k);
            });
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // this wavefront's share of the tile has landed
        __syncthreads();
        __builtin_amdgcn_s_setprio(3);                           // MFMA phase first: see below
        pf_mfmas<TG>(aop, smem, boff, acc);
        __builtin_amdgcn_s_setprio(0);
        __syncthreads();                                         // every wavefront has read chunk c before chunk c + 1 overwrites it
    }
}

// grid (N / 128, ntiles), block 256 (4 wavefronts x 2 strips = 128 weight rows); dynamic LDS = 16 TG * PF_ROW bytes
// two workgroups per CU at every tile height (the tallest would otherwise need one register too many): while one decodes on
// the vector ALUs the other runs its MFMAs
// MASKED = false skips the tiles of experts in mask mode (table flags word set) or with a base window code other than 0,
// MASKED = true takes only those: the rarely used paths keep their extra registers out of the common kernel
// Workgroups go to the eight XCDs in turn, and each XCD has an L2 of its own. Sixteen workgroups of neighbouring column blocks, which
// read the same token rows, are therefore taken from one XCD's share of the grid (what does not fill 128 keeps its place): a
// tile's rows come into two L2s instead of eight: prompt of 1003 tokens 2038 -> 2000 us, step of 201 1361 -> 1347. nq_pf_short_k only: nq_pf_gemm_k
// was timed with it when its lists had unused entries between the tiles, which sixteen workgroups at a time spread less evenly over the
// XCDs (a 4096-token step lost 3 to 7 %; with the 256-row list alone, which had none, 0 to 1), and not since they have no gaps.
struct Block { int x, y; };
__device__ __forceinline__ Block xcd_block()
{
    const uint32_t gx = gridDim.x, n = gx * gridDim.y, id = blockIdx.y * gx + blockIdx.x;
    uint32_t at = id;
    if (id < (n & ~127u)) { const uint32_t j = id >> 3; at = (((j >> 4) << 3) + (id & 7)) * 16 + (j & 15); }
    return Block{(int)(at % gx), (int)(at / gx)};
}
template <int TG, bool MASKED>
__device__ __forceinline__ void pf_tile(const PfGemm& a, int bx, int e, int row0, int nrows, int slot, char* smem)
{
    const int lane = threadIdx.x & 63, warp = threadIdx.x >> 6;
    const int64_t* ent = a.table + (size_t)e * TBL_W;
    const int lv = (int)ent[0];
    if (lv <= 0) return;                                         // rows of a level-0 expert are skipped downstream
    const int N = a.mode == 0 ? 2 * a.I : a.H, K = a.mode == 0 ? a.H : a.I, C = K / 128;
    const int sp = bx * 4 + warp;                        // strip pair of this wavefront
    const _Float16* A = (a.mode == 0 && bx * 128 >= a.I) ? a.A1 : a.A0;
    const int t4 = lane >> 4, ss = (lane >> 3) & 1, g = lane & 7, n = lane & 15;
    const Planes P = planes_of(ent, a.mode);
    if (!MASKED && a.wide && slot >= 0 && P.bcode == 0 && P.flags == nullptr) return;        // block-uniform: nq_pf_wide_k's tile
    if (((P.flags != nullptr && lv == 4) || P.bcode != 0) != MASKED)              // block-uniform: the other variant's tile
    {
        if (a.solo)
        {   // nobody will compute it (the host vouched for rows of one kind only): NaN, not whatever the scratch held
            const float nan = __builtin_nanf("");
            for (int i = threadIdx.x; i < nrows * 32; i += blockDim.x)
                *(float4_t*)(a.C + (size_t)(row0 + i / 32) * N + bx * 128 + 4 * (i % 32)) = float4_t{nan, nan, nan, nan};
        }
        return;
    }
    LaneCtx L;
    L.unit0 = (uint32_t)(2 * sp + ss) * C; L.rec0 = L.unit0 * 32 + 4 * g + t4;
    L.nrec = (size_t)(N / 16) * C * 32;
    L.src = (lane + 16) & 63; L.g = g; L.xs = nullptr; L.xstep = 0;
    L.strip = (uint32_t)(2 * sp + ss); L.nstrips = (size_t)(N / 16); L.chunk0 = 0; L.half0 = (uint32_t)(2 * sp + (lane >> 5)) * C;
    float4_t acc[TG][2];
#pragma unroll
    for (int tg = 0; tg < TG; ++tg) { acc[tg][0] = float4_t{0.f, 0.f, 0.f, 0.f}; acc[tg][1] = float4_t{0.f, 0.f, 0.f, 0.f}; }
    if constexpr (!MASKED)
    {
        if (lv == 2) pf_chunks<TG, false, 0, false>(P, L, C, A, K, row0, nrows, smem, acc);
        else dispatch_code(P.code, [&](auto tag) { pf_chunks<TG, true, decltype(tag)::value, false>(P, L, C, A, K, row0, nrows, smem, acc); });
    }
    else
        dispatch_base(P.bcode, [&](auto bk) {
            constexpr int BK = decltype(bk)::value;
            if (lv == 2) pf_chunks<TG, false, 0, false, BK>(P, L, C, A, K, row0, nrows, smem, acc);
            else dispatch_code(P.code, [&](auto tag) { pf_chunks<TG, true, decltype(tag)::value, true, BK>(P, L, C, A, K, row0, nrows, smem, acc); });
        });
    // lane (t4, n) holds, for token 16 tg + n, weight rows 32 sp + 16 (t4 >> 1) + 4 (t4 & 1) + i (+ 8 for acc[..][1])
    const int wrow = 32 * sp + 16 * (t4 >> 1) + 4 * (t4 & 1);
#pragma unroll
    for (int tg = 0; tg < TG; ++tg)
    {
        const int tok = 16 * tg + n;
        if (tok < nrows)
        {
            float* c = a.C + (size_t)(row0 + tok) * N + wrow;
            *(float4_t*)c = acc[tg][0];
            *(float4_t*)(c + 8) = acc[tg][1];
        }
    }
}

// A launch takes tiles of up to 16 TG rows, and its workgroup runs the body of as many row groups as its tile has: the tallest alone multiplied
// up to half a tile of rows that are not there, and at 128 rows the products already take as long as the decode. A body of its own,
// because a loop that ends early made the compiler copy the accumulators (1068 spilled registers at 256 rows). us a step, TG row groups always / in
// steps of TG / 4 / of one (two above 128 rows) / of one: 4096 tokens over 256 experts of mixed levels, evenly, 4850 / 4500 / 4265 / 4195; 1000 tokens,
// 64 experts, level 4 1435 / 1365 / 1325 / 1295; 2000 tokens, 256 experts 3730 / 3565 / 3490 / 3450; 4096 tokens, Zipf, 5640 / 5520 / 5490 / 5490.
// Masked tiles have one body more at 64 and 128 rows (all of them would double a build of three minutes) and none at 256, where it spilled.
constexpr int pf_step(int TG, bool masked) { return masked ? (TG + 3) / 4 : 1; }
constexpr int pf_lowest(int TG, bool masked) { return TG <= 2 || (masked && TG == 16) ? TG : TG / 2 + pf_step(TG, masked); }
template <int TG, bool MASKED, int LESS>
__device__ __forceinline__ void pf_fit(const PfGemm& a, int e, int row0, int nrows, int slot, char* smem)
{
    if constexpr (LESS < TG)
        if (nrows > 16 * LESS) return pf_fit<TG, MASKED, LESS + pf_step(TG, MASKED)>(a, e, row0, nrows, slot, smem);
    pf_tile<LESS, MASKED>(a, blockIdx.x, e, row0, nrows, slot, smem);
}

template <int TG, bool MASKED>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) nq_pf_gemm_k(PfGemm a)
{
    extern __shared__ __align__(16) char smem[];
    const int32_t* tile = a.tiles + 4 * blockIdx.y;
    const int e = tile[0], row0 = tile[1], nrows = tile[2], slot = tile[3] - 1;
    if (e < 0 || e >= a.E || nrows <= 0) return;
    pf_fit<TG, MASKED, pf_lowest(TG, MASKED)>(a, e, row0, nrows, slot, smem);
}

// Tiles of up to 64 rows of any height in one launch (the plan of nq_pf_sort_k). Steps of a few hundred tokens over many experts
// have nothing taller, so a projection is one launch on the caller's stream instead of three on three; with at most 64 rows a tile
// costs little more than decoding its expert, and the registers of the 64-row body (127) still let four wavefronts share a SIMD. The body of 48 rows
// takes a prompt of 1003 tokens (24 to 47 rows an expert) from 1930 to 1865 us. Bound by
// instruction issue: one vector instruction per 4.0 to 4.2 clocks and SIMD at 200 and 1000 tokens (profiles/grouped_steps.txt).
template <bool MASKED>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MASKED ? 2 : 4))) nq_pf_short_k(PfGemm a)
{
    extern __shared__ __align__(16) char smem[];
    const Block blk = xcd_block();
    const int32_t* tile = a.tiles + 4 * blk.y;
    const int e = tile[0], row0 = tile[1], nrows = tile[2];
    if (e < 0 || e >= a.E || nrows <= 0) return;
    if (nrows <= 16) pf_tile<1, MASKED>(a, blk.x, e, row0, nrows, -1, smem);
    else if (nrows <= 32) pf_tile<2, MASKED>(a, blk.x, e, row0, nrows, -1, smem);
    else if (nrows <= 48) pf_tile<3, MASKED>(a, blk.x, e, row0, nrows, -1, smem);
    else pf_tile<4, MASKED>(a, blk.x, e, row0, nrows, -1, smem);
}

template <int TG, bool MASKED>
int launch_gemm_tg(const PfGemm& a, int ntiles, int N, hipStream_t st)
{
    const int shm = 16 * TG * PF_ROW;
    if (shm > 48 * 1024)
    {
        hipError_t e = hipFuncSetAttribute((const void*)nq_pf_gemm_k<TG, MASKED>, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
        if (e != hipSuccess) return set_error("nq_pf_gemm: LDS %d bytes: %s", shm, hipGetErrorString(e));
    }
    nq_pf_gemm_k<TG, MASKED><<<dim3(N / 128, ntiles), 256, shm, st>>>(a);
    NQ_LAUNCH_CHECK("nq_pf_gemm");
    return 0;
}

// The kernels of one kind: tiles of up to bm rows, or the mixed list of short tiles (bm = SHORT_LIST).
constexpr int SHORT_LIST = 0;
template <bool MASKED>
int launch_tiles(const PfGemm& a, int bm, int ntiles, hipStream_t st)
{
    const int N = a.mode == 0 ? 2 * a.I : a.H;
    switch (bm)
    {
        case 16: return launch_gemm_tg<1, MASKED>(a, ntiles, N, st);
        case 32: return launch_gemm_tg<2, MASKED>(a, ntiles, N, st);
        case 64: return launch_gemm_tg<4, MASKED>(a, ntiles, N, st);
        case 128: return launch_gemm_tg<8, MASKED>(a, ntiles, N, st);
        case 256: return launch_gemm_tg<16, MASKED>(a, ntiles, N, st);
        case SHORT_LIST:
            nq_pf_short_k<MASKED><<<dim3(N / 128, ntiles), 256, SHORT_ROWS * PF_ROW, st>>>(a);
            NQ_LAUNCH_CHECK("nq_pf_short");
            return 0;
    }
    return set_error("nq_pf_gemm: no tiles of %d rows", bm);
}
extern template int launch_gemm_tg<16, false>(const PfGemm&, int, int, hipStream_t);
extern template int launch_gemm_tg<16, true>(const PfGemm&, int, int, hipStream_t);
extern template int launch_tiles<false>(const PfGemm&, int, int, hipStream_t);
extern template int launch_tiles<true>(const PfGemm&, int, int, hipStream_t);

}  // namespace nq
