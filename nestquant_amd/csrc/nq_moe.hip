// Decode-path MoE layer for 1..8 tokens (reference sm120/nqmoe.cu:375-449 route, :493-771 do_item, :858-907 moe_forward,
// :908-929 mailbox). Three launches on one stream (two for calls of few workgroups, see launch_moe), every routing / level / pointer decision read on the device:
//
//   nq_prep_k        routing once per call (picks -> runs of distinct experts, their table rows -> run headers in RouteWs) and
//                 the rotation of the activations of every active pick (x * su -> Hadamard-128 -> fp16, B-operand order).
//   nq_gemv_k<0, *>  gate|up: grid (strip-pair blocks, k-slices, runs). A run = one distinct routed expert + the tokens that
//                 picked it. The block copies those tokens' rotated x into LDS, then every wavefront decodes the records of
//                 two strips chunk by chunk straight into MFMA A operands (v_mfma_f32_16x16x32_f16, tokens as the N
//                 dimension) and writes its k-slice partial sums. In a call of both launches that is all; in a gate|up-only
//                 call (and for rows with a low-rank plane or the 512-wide rotation) the block that arrives last at a
//                 (run, 128-column group) counter finishes the group: Hadamard * sv, SwiGLU, * su_d, Hadamard -> h fp16.
//   nq_gemv_k<1, *>  down: staging forms h from the gate|up partial sums (or reads it), same decode loop; the last block of a
//                 128-row output group (counter over all runs) combines:
//                 out[b] = sum_k rw[b,k] * sv_o (.) Hadamard(sum of partials).
//   A call with a mailbox: one workgroup of an extra plane of blocks of the call's LAST projection launch applies it
//   (table <- stage, device applied <- seq); the NEXT routing launch publishes applied to the host. See mailbox_apply.
//
// Lane mapping of the GEMV (wave64): lane = 16 * t4 + 8 * ss + g decodes the record of lane (4 g + t4) of unit
// (strip0 + ss, chunk); it holds 32 weights of row g and 32 of row g + 8, in columns 16 t + 2 t4 + {0,1,8,9}. An MFMA
// 16x16x32 takes 8 fp16 per lane: lanes with equal (ss, g) and different t4 are the k-groups of one A row, so the decoded
// pairs are A operands as they leave the decoder, with no cross-lane movement. The B operand (tokens) comes from LDS,
// staged in the matching column order. Partial sums instead of float atomics make the layer output bitwise repeatable;
// the arrival counters are zero on entry and are reset by the block that consumes them.
#include "nq_sal.hpp"
#include "nq_host.hpp"
#include <algorithm>
#include <mutex>
#include "../../include/nq_moe_hip.h"

namespace nq {

// Partial sums cross workgroups (and XCDs, whose L2s are not coherent with each other) inside one kernel. They are
// written and read with device-scope relaxed atomics (sc1: write-through / read-through to the device coherence point)
// and ordered by "all my stores are acknowledged (vmcnt 0) -> bump the group's arrival counter". A full device-scope
// fence would also be correct but writes back and invalidates the whole L2 once per workgroup, which costs several times
// the kernel's own run time.
// The compiler waits after every atomic load, which serialises the finisher's reads (one memory round trip per k-slice),
// so the loads are issued as a batch of sc0 sc1 loads and waited for once; the wait names the destination registers so
// that no use can move above it.
__device__ __forceinline__ void st_dev4(float* p, float4_t v)
{
    asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" :: "v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void st_dev2(float* p, float2 v)
{
    asm volatile("global_store_dwordx2 %0, %1, off sc0 sc1" :: "v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ float2 ld_dev2_issue(const float* p)
{
    float2 v;
    asm volatile("global_load_dwordx2 %0, %1, off sc0 sc1" : "=v"(v) : "v"(p) : "memory");
    return v;
}
__device__ __forceinline__ void ld_wait(float2& a, float2& b, float2& c, float2& d)
{
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(a), "+v"(b), "+v"(c), "+v"(d) :: "memory");
}
// A launch's last workgroups run the tail's code cold: straight on, 2 KB of it cost 2300 clk instead of 1030, and each jump over code that
// is not wanted waits for a line from the L2. What few calls need stands out of line.
__device__ __forceinline__ bool rare(bool c) { return __builtin_expect(c, 0); }
// sums over k-slices y of the two floats at p[q] + y * stride, for NR rows q at once: the reads of all rows are in flight
// together, four slices per row at a time (device-coherent reads)
template <int NR>
__device__ __forceinline__ void sum_partials(const float* const* p, size_t stride, int NY, float2* out)
{
#pragma unroll
    for (int q = 0; q < NR; ++q) out[q] = make_float2(0.f, 0.f);
    for (int y = 0; y < NY; y += 4)
    {
        float2 v[NR][4];
#pragma unroll
        for (int q = 0; q < NR; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) v[q][i] = ld_dev2_issue(p[q] + (size_t)(y + i < NY ? y + i : y) * stride);
#pragma unroll
        for (int q = 0; q < NR; ++q) ld_wait(v[q][0], v[q][1], v[q][2], v[q][3]);
#pragma unroll
        for (int q = 0; q < NR; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) if (y + i < NY) { out[q].x += v[q][i].x; out[q].y += v[q][i].y; }
    }
}

__device__ __forceinline__ long long sel_at(const MoeArgs& a, int i) { return id_at(a.sel, a.sel_dtype, i); }
__device__ __forceinline__ float rw_at(const MoeArgs& a, int i) { return w_at(a.rw, a.rw_dtype, i); }
__device__ __forceinline__ half2_t x2_at(const MoeArgs& a, size_t i) { return act2_at(a.x, a.x_dtype, i); }
__device__ __forceinline__ void out2_store(const MoeArgs& a, size_t i, float v0, float v1) { res2_store(a.out, a.out_dtype, i, v0, v1); }

constexpr int MAXTOK = 8;                      // tokens of one run = tokens of one call (the MFMA N dimension holds 16)
// What the projection launches need to know about run r, written once per call by nq_prep_k (one per projection: the plane
// addresses differ). A run = one distinct routed expert + the tokens that picked it.
struct alignas(64) RunHdr
{
    Planes P;                     // this projection of the run's expert
    const _Float16* signs;        // su_g | sv_g | sv_u | su_d | sv_o | su_u
    const _Float16* lr; const _Float16* lr4;      // low-rank plane of the run's expert (lr == nullptr: none)
    int level, ntok;
    int had;                      // width of the Hadamard on the down projection's input: 128 or 512
    int rg, rd;
    int pad;
    unsigned char slot[MAXTOK];   // pick index (token * topk + k) of the run's tokens: their row of MoeArgs::xrot and of the partial sums
    __device__ __forceinline__ int slot_of(int j) const       // by shifts: a run-time index into slot[] would put the header into scratch memory
    {
        unsigned long long v;
        __builtin_memcpy(&v, slot, 8);
        return (int)((v >> (8 * j)) & 0xFFull);
    }
};
struct PickInfo                   // per pick, for the down launch's combine
{
    float w[64];                  // routing weight, 0 for picks that contribute nothing
    const _Float16* signs[64];
    const _Float16* lr[64]; const _Float16* lr4[64]; unsigned char rg[64], rd[64], lv[64];
};
struct RouteWs { int nruns; int ny_gu; int pad[14]; PickInfo picks; RunHdr run[2][64]; };   // ny_gu: k-slices of the gate|up launch that filled part_gu
static_assert(sizeof(RunHdr) == 128, "RunHdr is read as 32 scalar words");
static_assert(sizeof(RouteWs) <= NQ_ROUTE_WS_BYTES, "NQ_ROUTE_WS_BYTES in include/nq_moe_hip.h is too small");

// ---- mailbox rows: 20 int64 read past every cache (a copy engine may have written them while kernels ran), all in flight
// together and waited for once (the compiler would wait after each atomic load: twenty round trips)
__device__ __forceinline__ void ld_sys_row(const int64_t* p, int64_t* f)
{
#pragma unroll
    for (int i = 0; i < TBL_W; ++i) asm volatile("global_load_dwordx2 %0, %1, off offset:%2 sc0 sc1" : "=v"(f[i]) : "v"(p), "n"(8 * i) : "memory");
#pragma unroll
    for (int i = 0; i < TBL_W; i += 4) asm volatile("s_waitcnt vmcnt(0)" : "+v"(f[i]), "+v"(f[i + 1]), "+v"(f[i + 2]), "+v"(f[i + 3]) :: "memory");
}

// ---- routing dedup: picks -> runs (refined experts first, then by first occurrence); slots in pick order ----------------
// One wavefront; lane s owns pick s (S <= 64). A run takes at most one pick per token: a token that names the same expert twice
// opens a second run of that expert, so a run never has more than B tokens. Every lane requests all fields of its own pick's table
// row together, so the leader's fields cost no second round trip. The routing reads the table and nothing else: no kernel writes
// the table while a routing launch runs (the mailbox of a call is applied by its last projection launch, see mailbox_apply), so
// every workgroup of the launch sees the same rows and the rows cannot be torn.
struct PrepRows { int nq; unsigned char pick[64]; const _Float16* signs[64]; };   // LDS: the active picks, in order
__device__ __forceinline__ bool pick_expert(const MoeArgs& a, int lane, int& e)
{
    if (lane >= a.B * a.topk) return false;
    const long long ee = sel_at(a, lane);
    if (ee < 0 || ee >= a.E) return false;
    e = (int)ee;
    return true;
}
// What a workgroup of the rotation needs: the active picks and their sign vectors, no numbering of runs.
__device__ __forceinline__ void list_picks(const MoeArgs& a, int lane, PrepRows* Q)
{
    int e = 0, lv = 0; const _Float16* sg = nullptr;
    bool ok = false;
    if (pick_expert(a, lane, e))
    {
        const int64_t* ent = a.table + (size_t)e * TBL_W;
        lv = (int)ent[0]; sg = (const _Float16*)ent[9];
        ok = rw_at(a, lane) != 0.f && lv > 0;
    }
    const unsigned long long okm = __ballot(ok);
    if (ok)
    {
        const int q = __popcll(okm & ((1ull << lane) - 1ull));
        Q->pick[q] = (unsigned char)lane; Q->signs[q] = sg;
    }
    if (lane == 0) Q->nq = __popcll(okm);
}
// pick `lane`: its expert (-1: none), the fields of the expert's row, the level it runs at, and whether it contributes
struct Pick { int e, level; bool inrange, ok; int64_t f[TBL_W]; };
__device__ __forceinline__ Pick load_pick(const MoeArgs& a, int lane)
{
    Pick p;
    p.e = -1; p.ok = false;
    int lv = 0;
    p.inrange = pick_expert(a, lane, p.e);
#pragma unroll
    for (int i = 0; i < TBL_W; ++i) p.f[i] = 0;
    if (p.inrange)
    {
        const int64_t* ent = a.table + (size_t)p.e * TBL_W;
#pragma unroll
        for (int i = 0; i < TBL_W; ++i) p.f[i] = ent[i];
        lv = (int)p.f[0];
        p.ok = rw_at(a, lane) != 0.f && lv > 0;
    }
    p.level = a.force_level ? a.force_level : lv;
    return p;
}
struct Place { int run, pos, ntok, nruns; };                     // the run this lane's pick goes into (-1: none), its place there, the run's size; the number of runs
__device__ __forceinline__ Place number_runs(const MoeArgs& a, int e, bool ok, int level, int lane)
{
    const int S = a.B * a.topk;
    // Runs of refined experts (level 3, 4: twice the decode work per chunk) are numbered before the level-2 ones, each group
    // by first occurrence: workgroups are dispatched in run order, so the long ones start first and spread over all CUs, and
    // the short ones fill in around them (gate|up 44.0 -> 42.6 us, down 28.4 -> 27.2 us on the benchmark's level mix).
    const unsigned long long okm = __ballot(ok);
    const unsigned long long heavy = __ballot(ok && level > 2);
    const unsigned long long below = (1ull << lane) - 1ull;
    const int tok = lane / a.topk, sh = tok * a.topk;
    const unsigned long long mytok = sh < 64 ? (a.topk >= 64 ? ~0ull : ((1ull << a.topk) - 1ull)) << sh : 0ull;
    Place p{-1, 0, 0, 0};
    unsigned long long eq = 0ull;                                // the active picks of this lane's expert
#pragma unroll 4
    for (int j = 0; j < S; ++j)
    {
        const unsigned long long m = __ballot(ok && e == __builtin_amdgcn_readlane(e, j));
        eq = lane == j ? m : eq;
    }
    if (__ballot(ok && (eq & mytok & below)) == 0ull)
    {   // no token names an expert twice: a run is an expert, and all are numbered at once (one after the other, thirty runs took 5 us)
        const unsigned long long first = __ballot(ok && (eq & below) == 0ull), fh = first & heavy, fl = first & ~heavy;
        const int mine = ((heavy >> lane) & 1ull) ? __popcll(fh & below) : __popcll(fh) + __popcll(fl & below);
        const int run = __shfl(mine, eq ? __ffsll((long long)eq) - 1 : lane);
        if (ok) { p.run = run; p.pos = __popcll(eq & below); p.ntok = __popcll(eq); }
        p.nruns = __popcll(first);
    }
    else
        for (int pass = 0; pass < 2; ++pass)
        {
            unsigned long long rem = pass == 0 ? heavy : okm & ~heavy;
            while (rem)
            {
                const int ev = __builtin_amdgcn_readlane(e, __ffsll((long long)rem) - 1);
                const unsigned long long same = __ballot(((rem >> lane) & 1ull) && e == ev);
                const unsigned long long m = __ballot(((same >> lane) & 1ull) && (same & mytok & below) == 0ull);   // first pick per token
                if ((m >> lane) & 1ull) { p.run = p.nruns; p.pos = __popcll(m & below); p.ntok = __popcll(m); }
                rem &= ~m; ++p.nruns;
            }
        }
    return p;
}
__device__ __forceinline__ void write_header(RunHdr& R, const int64_t (&f)[TBL_W], int mode, int level, int ntok)      // all but the slots
{
    const int o = mode == 0 ? 1 : 5;
    R.P.base = (gp_u4)f[o]; R.P.res = (gp_u8)f[o + 1]; R.P.dw = (gp_u32)f[o + 2]; R.P.flags = (gp_u64)f[o + 3];
    R.P.var = (gp_u8)f[12 + mode]; R.P.code = (int)f[10 + mode]; R.P.bcode = (int)((f[19] >> (8 * mode)) & 0xFF);
    R.signs = (const _Float16*)f[9];
    R.level = level;
    R.had = f[18] == 512 ? 512 : 128;
    R.lr = (const _Float16*)f[14]; R.lr4 = (const _Float16*)f[15]; R.rg = (int)f[16]; R.rd = (int)f[17];
    R.ntok = ntok;
}
__device__ __forceinline__ void route(const MoeArgs& a, RouteWs* W, int lane)
{
    const Pick p = load_pick(a, lane);
    const int64_t (&f)[TBL_W] = p.f;
    const int level = p.level;
    if (a.hits && p.inrange && rw_at(a, lane) != 0.f)
        __hip_atomic_fetch_add(a.hits + p.e, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    const Place at = number_runs(a, p.e, p.ok, level, lane);
    const int my_run = at.run, my_pos = at.pos;
    // the headers, after the numbering: every lane holds its own pick's row, so the first lanes of all runs write their runs'
    // headers side by side (inside the loop above the same stores would be issued once per run, one lane at a time)
    if (my_run >= 0)
    {
        W->run[0][my_run].slot[my_pos] = (unsigned char)lane; W->run[1][my_run].slot[my_pos] = (unsigned char)lane;
        if (my_pos == 0)
        {
#pragma unroll
            for (int mode = 0; mode < 2; ++mode) write_header(W->run[mode][my_run], f, mode, level, at.ntok);
        }
    }
    PickInfo& K = W->picks;
    K.w[lane] = p.ok ? rw_at(a, lane) : 0.f; K.signs[lane] = (const _Float16*)f[9];
    K.lr[lane] = (const _Float16*)f[14]; K.lr4[lane] = (const _Float16*)f[15];
    K.rg[lane] = (unsigned char)f[16]; K.rd[lane] = (unsigned char)f[17]; K.lv[lane] = (unsigned char)level;
    if (lane == 0) W->nruns = at.nruns;
}
// run z of the call and the number of runs, found by one wavefront of the workgroup itself (the gate|up launch of a call without a routing
// launch): the header that route() writes, in LDS
struct OwnRun { RunHdr run; int nruns; };
__device__ __forceinline__ void own_run(const MoeArgs& a, int z, int lane, OwnRun* W)
{
    const Pick p = load_pick(a, lane);
    const Place at = number_runs(a, p.e, p.ok, p.level, lane);
    if (lane == 0) W->nruns = at.nruns;
    if (at.run != z) return;
    W->run.slot[at.pos] = (unsigned char)lane;
    if (at.pos == 0) write_header(W->run, p.f, 0, p.level, at.ntok);
}

// The mailbox of a layer call (reference nq_mailbox, sm120/nqmoe.cu:908-923, a launch of its own there), in two halves that
// keep the reference's rule "once applied_host[e] == seq[e] no later kernel can reference the old row's slot":
//   apply   -- one workgroup of the call's LAST projection launch: for every e with seq[e] != applied[e], table[e] <- stage[e]
//              and the device copy applied[e] <- seq[e]. This is the call's only reading of seq / stage (a single observer),
//              it comes after the call's routing launch has ended (the routing of this call used the old rows, identically in
//              all its workgroups), and neither projection launch reads the table, so a row cannot be torn and no two parts of
//              the call can disagree about a row. Nothing is published to the host here: this call's launches may still be
//              decoding from the slot that the old row names.
//   publish -- the routing launch of the NEXT call (publish_applied): applied_host[e] <- applied[e] for every e. It runs after
//              every launch of the earlier calls has ended (stream order), and from this routing launch on every launch works
//              from rows read after the apply, so a slot released by a published row is no longer referenced by anything.
// A row whose seq lands while call n runs is therefore used from call n + 1 on and published at the head of call n + 1, which is
// when the reference's mailbox launch at the head of call n + 1 would have applied and published it.
__device__ __forceinline__ void mailbox_apply(int64_t* table, const int64_t* stage, const int32_t* seq, int32_t* applied, int E)
{
    for (int e = threadIdx.x; e < E; e += blockDim.x)
    {
        const int32_t ap = applied[e];
        const int32_t sq = __hip_atomic_load(seq + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (sq == ap) continue;                                  // the row is requested only after seq has been seen (the copy
        int64_t row[TBL_W];                                      // stream wrote the row before seq)
        ld_sys_row(stage + (size_t)e * TBL_W, row);
#pragma unroll
        for (int i = 0; i < TBL_W; ++i) table[(size_t)e * TBL_W + i] = row[i];
        applied[e] = sq;                                         // read again only by later launches on this stream
    }
}
// host mirror of the device's applied[]: plain re-publication of every entry (values only ever grow, equal values are harmless)
__device__ __forceinline__ void publish_applied(const int32_t* applied, int32_t* applied_host, int E, int first, int step)
{
    for (int e = first; e < E; e += step)
        __hip_atomic_store(applied_host + e, applied[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ void call_salience(const MoeArgs& a)  // by a workgroup of 256 threads
{
    __shared__ SalShared S;
    const SalArgs sa{a.x, a.H, a.rw, a.sel, a.B, a.H, a.topk, a.E, a.x_dtype, a.rw_dtype, a.sel_dtype, a.sal_rsf, a.sal_acc, a.sal_host};
    salience<4>(sa, &S);
}
// fp16(Hadamard-128(x[token] * su)) of a chunk of 128 columns, eight of them per lane (place L8 of 16), in B-operand order
__device__ __forceinline__ uint4 rotate8(const MoeArgs& a, int token, const _Float16* su, int chunk, int L8, const WhtSigns& ws)
{
    const int col = chunk * 128 + 32 * (L8 >> 2) + 2 * (L8 & 3);
    half2_t xv[4], sv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) { xv[i] = x2_at(a, (size_t)token * a.H + col + 8 * i); sv[i] = *(const half2_t*)(su + col + 8 * i); }
    float v[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) { v[2 * i] = (float)xv[i].x * (float)sv[i].x; v[2 * i + 1] = (float)xv[i].y * (float)sv[i].y; }
    wht8_bop_sums(v, ws);
    return bop_block_scaled(v, ws.scale);
}

// First launch of a layer call, except where the gate|up launch does its work (launch_moe). Workgroup 0 does the routing: run headers for both projection launches, which then read one
// header each instead of repeating the dependent loads sel -> table row in every one of their ~1800 workgroups, the per-pick
// data of the combine, the hits export; with a mailbox in the call its other three wavefronts publish what earlier calls applied
// (publish_applied). Nothing here reads seq or stage and nothing writes the table. With salience in the call workgroup 1 exports
// it (a launch of its own in front of the call cost 9 us at one token, 20 us at four). All others rotate the activations, one
// task per (active pick, gate or up, 128-column chunk): xrot[pick][gate|up][chunk] = fp16(Hadamard-128(x[token] * su)) in the
// MFMA B-operand column order, which the gate|up launch copies into LDS; rows are numbered by pick, so a rotating workgroup
// needs the list of active picks but not the runs.
// Bound by latency: three dependent round trips (sel, table row, sign vector and activations) in either branch; 5.2 us at one
// token, 7.3 us at four with salience (15 us while every workgroup numbered the runs, one after the other, and a single wavefront
// walked all tokens for the salience).
__global__ void __launch_bounds__(256) nq_prep_k(MoeArgs a)
{
    __shared__ PrepRows Q;
    const int lane = threadIdx.x & 63;
    const int extra = a.sal_acc ? 2 : 1;                         // workgroup 0 routes; 1 exports the salience of a call that asks for it
    if (a.sal_acc && blockIdx.x == 1) { call_salience(a); return; }
    if (blockIdx.x == 0)
    {
        if (threadIdx.x < 64) route(a, a.route, lane);
        else if (a.mb_table && a.mb_applied_host) publish_applied(a.mb_applied, a.mb_applied_host, a.E, threadIdx.x - 64, 192);
        return;
    }
    if (threadIdx.x < 64) list_picks(a, lane, &Q);
    __syncthreads();
    const int C = a.H / 128, ntask = Q.nq * 2 * C, nrot = (int)gridDim.x - extra;
    for (int t = ((int)blockIdx.x - extra) * 4 + (threadIdx.x >> 6); t < ntask; t += nrot * 4)
    {
        const int q = t / (2 * C), r = t - q * 2 * C, up = r / C, c = r - up * C, kk = c * 128 + 2 * lane, pick = Q.pick[q];
        const _Float16* su = Q.signs[q] + (up ? 2 * a.H + 3 * a.I : 0);
        const half2_t xv = x2_at(a, (size_t)(pick / a.topk) * a.H + kk), sv = *(const half2_t*)(su + kk);
        float v0 = (float)xv.x * (float)sv.x, v1 = (float)xv.y * (float)sv.y;
        wht128_sums(v0, v1, lane);
        _Float16* dst = a.xrot + ((size_t)pick * 2 + up) * a.H + c * 128;
        dst[bop_index(2 * lane)] = f16_scaled(v0, WHT128_SCALE); dst[bop_index(2 * lane + 1)] = f16_scaled(v1, WHT128_SCALE);
    }
}

// finisher of gate|up for (run z, 128-column group grp): h[slot] = fp16(WHT(silu(g) * u * su_d)), g = WHT(sum_y part_g) * sv_g.
// With a 512-wide Hadamard on the down projection's input (in_had_down, reference sm120/nqmoe.cu:36-40,673-712;
// WHT_512 = H_4 (x) WHT_128 / 2) the group's WHT_128 result goes, in fp32, into the gate columns of k-slice 0 that this
// finisher has just consumed, and the last of the four groups of a 512-column block combines them with the Sylvester H_4
// and rounds to fp16 once.
__device__ __forceinline__ void finish_gu(const MoeArgs& a, const RunHdr& R, float (*zl)[4], int z, int grp, int NY, int warp, int SB, int lane, int& last)
{
    const _Float16 *sv_g = R.signs + a.H, *sv_u = sv_g + a.I, *su_d = sv_u + a.I;
    const int S = a.B * a.topk, col = grp * 128 + 2 * lane;
    const bool wide = R.had == 512;
    // low-rank plane (reference sm120/nqmoe.cu:41-45,611-645): lr = V_gu [rg][H] | U2_g [rg][I] | U2_u [rg][I] | V_dn [rd][I] |
    // U2_d [rd][H], lr4 = U4_g | U4_u | U4_d (level 4 only). z = x V_gu^T over the raw activations, one wavefront per token
    const bool lowrank = R.lr != nullptr;                        // block-uniform
    const int rg = lowrank ? R.rg : 0, rd = lowrank ? R.rd : 0;
    if (rg)
    {
        for (int j = warp; j < R.ntok; j += SB)
        {
            const int tok = R.slot_of(j) / a.topk;
            float zz[4] = {0.f, 0.f, 0.f, 0.f};
            for (int k = 2 * lane; k < a.H; k += 128)
            {
                const half2_t xv = x2_at(a, (size_t)tok * a.H + k);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (r < rg) { const half2_t vv = *(const half2_t*)(R.lr + (size_t)r * a.H + k); zz[r] += (float)xv.x * (float)vv.x + (float)xv.y * (float)vv.y; }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
#pragma unroll
                for (int m = 32; m >= 1; m >>= 1) zz[r] += __shfl_xor(zz[r], m);
                if (lane == 0) zl[j][r] = zz[r];
            }
        }
        __syncthreads();
    }
    const _Float16* U2g = R.lr + (size_t)rg * a.H, *U2u = U2g + (size_t)rg * a.I, *Vd = U2u + (size_t)rg * a.I;
    const _Float16* U4g = R.lr4, *U4u = U4g + (size_t)rg * a.I;
    for (int j = warp; j < R.ntok; j += SB)
    {
        const int s = R.slot_of(j);
        const float* p = a.part_gu + (size_t)s * 2 * a.I + col;
        const half2_t svg = *(const half2_t*)(sv_g + col), svu = *(const half2_t*)(sv_u + col), sud = *(const half2_t*)(su_d + col);
        const float* const rows2[2] = {p, p + a.I};
        float2 pq[2];
        sum_partials<2>(rows2, (size_t)S * 2 * a.I, NY, pq);
        float g0 = pq[0].x, g1 = pq[0].y, u0 = pq[1].x, u1 = pq[1].y;
        wht128(g0, g1, lane); wht128(u0, u1, lane);
        g0 *= (float)svg.x; g1 *= (float)svg.y; u0 *= (float)svu.x; u1 *= (float)svu.y;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (r < rg)
            {
                const float zr = zl[j][r];
                half2_t ug = *(const half2_t*)(U2g + (size_t)r * a.I + col), uu = *(const half2_t*)(U2u + (size_t)r * a.I + col);
                g0 += zr * (float)ug.x; g1 += zr * (float)ug.y; u0 += zr * (float)uu.x; u1 += zr * (float)uu.y;
                if (R.level == 4)
                {
                    ug = *(const half2_t*)(U4g + (size_t)r * a.I + col); uu = *(const half2_t*)(U4u + (size_t)r * a.I + col);
                    g0 += zr * (float)ug.x; g1 += zr * (float)ug.y; u0 += zr * (float)uu.x; u1 += zr * (float)uu.y;
                }
            }
        const float sw0 = g0 / (1.f + __expf(-g0)) * u0, sw1 = g1 / (1.f + __expf(-g1)) * u1;
        if (rd)
        {   // this group's share of z_d = sw V_dn^T, summed over the groups by the down combine
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                float t = 0.f;
                if (r < rd) { const half2_t vv = *(const half2_t*)(Vd + (size_t)r * a.I + col); t = sw0 * (float)vv.x + sw1 * (float)vv.y; }
#pragma unroll
                for (int m = 32; m >= 1; m >>= 1) t += __shfl_xor(t, m);
                if (lane == 0) a.zd[((size_t)s * (a.I / 128) + grp) * 4 + r] = t;
            }
        }
        float v0 = sw0 * (float)sud.x, v1 = sw1 * (float)sud.y;
        wht128(v0, v1, lane);
        // h = fp16 of the fp32 rotation result (two roundings, as the reference's kernel and its torch restatement). Left alone,
        // the compiler merges the rotation's last multiply into the conversion (v_fma_mixlo_f16: one rounding) at some call
        // sites and not at others; this one and the down launch's staging must give the same bits.
        asm volatile("" : "+v"(v0), "+v"(v1));
        if (wide) st_dev2(a.part_gu + (size_t)s * 2 * a.I + col, make_float2(v0, v1));
        else
        {
            half2_t hv; hv.x = (_Float16)v0; hv.y = (_Float16)v1;
            *(half2_t*)(a.h + (size_t)s * a.I + col) = hv;       // read by the next kernel on the stream
        }
    }
    if (!wide) return;                                           // block-uniform
    int* cnt = a.cnt_h + z * (a.I / 128) + grp / 4;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) last = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 3;
    __syncthreads();
    if (!last) return;
    const int c0 = (grp / 4) * 512 + 2 * lane;
    for (int j = warp; j < R.ntok; j += SB)
    {
        const int s = R.slot_of(j);
        float2 w[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) w[q] = ld_dev2_issue(a.part_gu + (size_t)s * 2 * a.I + c0 + q * 128);
        ld_wait(w[0], w[1], w[2], w[3]);
#pragma unroll
        for (int q = 0; q < 4; ++q)
        {
            float h0 = 0.f, h1 = 0.f;
#pragma unroll
            for (int pp = 0; pp < 4; ++pp)
            {
                const float sg = (__builtin_popcount(q & pp) & 1) ? -0.5f : 0.5f;
                h0 += sg * w[pp].x; h1 += sg * w[pp].y;
            }
            half2_t hv; hv.x = (_Float16)h0; hv.y = (_Float16)h1;
            *(half2_t*)(a.h + (size_t)s * a.I + c0 + q * 128) = hv;
        }
    }
    if (threadIdx.x == 0) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What the combine needs to know of the call's picks, lane s holding pick s: one coalesced read of PickInfo for all of them, issued
// under the decode's last partial sums. Read pick by pick inside the combine (weight -> sign vector's address -> its values, then the
// low-rank address) these were four dependent round trips per token on the launch's last workgroup. Layer of H 512, I 256, 4 picks, 2
// tokens: 17.5 -> 16.95 us a call; at 6144 x 2048 the same within 0.3 % (there other workgroups still decode under it).
struct PickLanes
{
    float w; unsigned long long signs; int rd;                   // rd: rank of the low-rank plane's down half, 0 without one
    __device__ __forceinline__ float weight(int s) const { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), s)); }
    __device__ __forceinline__ const _Float16* sign_row(int s) const
    {
        const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)signs, s), hi = __builtin_amdgcn_readlane((int)(signs >> 32), s);
        return (const _Float16*)(((unsigned long long)hi << 32) | lo);
    }
    __device__ __forceinline__ int rank(int s) const { return __builtin_amdgcn_readlane(rd, s); }
};
__device__ __forceinline__ PickLanes pick_lanes(const PickInfo& R, int lane)
{
    PickLanes P;
    P.w = R.w[lane]; P.signs = (unsigned long long)R.signs[lane]; P.rd = R.lr[lane] ? R.rd[lane] : 0;
    return P;
}
// the output scales of picks k and k + SB of the first token for this lane's two columns (nothing for picks that do not contribute)
__device__ __forceinline__ void pick_scales(const MoeArgs& a, const PickLanes& P, int k, int SB, int col, half2_t* sv)
{
#pragma unroll
    for (int q = 0; q < 2; ++q)
    {
        const int kq = k + q * SB;
        sv[q] = half2_t{};
        if (kq < a.topk && P.weight(kq & 63) != 0.f) sv[q] = *(const half2_t*)(P.sign_row(kq & 63) + a.H + 3 * a.I + col);
    }
}
// o += weight of pick s * (its output scales (.) WHT(its partial sums pv) + its low-rank term), for this lane's two columns
__device__ __forceinline__ void add_pick(const MoeArgs& a, const PickInfo& R, const PickLanes& P, int s, float w, float2 pv, half2_t sv, int col, int lane, float& o0, float& o1)
{
    float v0 = pv.x, v1 = pv.y;
    wht128(v0, v1, lane);
    if (w == 0.f) return;
    v0 *= (float)sv.x; v1 *= (float)sv.y;
    const int prd = P.rank(s);
    if (rare(prd))
    {   // y += (sw V_dn^T) (U2_d [+ U4_d]): z_d summed over the I / 128 groups written by the gate|up finishers
        const int prg = R.rg[s];
        const _Float16* U2d = R.lr[s] + (size_t)prg * (a.H + 2 * a.I) + (size_t)prd * a.I;
        const _Float16* U4d = R.lr4[s] + (size_t)prg * 2 * a.I;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (r < prd)
            {
                float zr = 0.f;
                for (int gq = 0; gq < a.I / 128; ++gq) zr += a.zd[((size_t)s * (a.I / 128) + gq) * 4 + r];
                half2_t ud = *(const half2_t*)(U2d + (size_t)r * a.H + col);
                v0 += zr * (float)ud.x; v1 += zr * (float)ud.y;
                if (R.lv[s] == 4) { ud = *(const half2_t*)(U4d + (size_t)r * a.H + col); v0 += zr * (float)ud.x; v1 += zr * (float)ud.y; }
            }
    }
    o0 += w * v0; o1 += w * v1;
}
// out[o], out[o + 1] = the sums of a token's n <= 4 wavefronts (those beyond n are not written: their reads are turned to the last)
__device__ __forceinline__ void sum_waves(const MoeArgs& a, size_t o, const float* red, int n)
{
    float2 v[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) v[w] = *(const float2*)(red + min(w, n - 1) * 128);
    float r0 = 0.f, r1 = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w)
        if (w < n) { r0 += v[w].x; r1 += v[w].y; }
    out2_store(a, o, r0, r1);
}

// combine of the down projection for output rows [grp * 128, +128): out[b] = sum_k rw[b,k] * sv_o[e] (.) WHT(sum_y part_d[slot])
// picks of a token are spread over the block's wavefronts and reduced through LDS. One token: two picks of a wavefront in flight
// (red: SB * 128 floats); `next`: the scales of the first two, requested before the arrival counter.
__device__ __forceinline__ void finish_dn(const MoeArgs& a, const PickInfo& R, const PickLanes& P, half2_t* next, int grp, int NY, int warp, int SB, int lane, float* red)
{
    const int col = grp * 128 + 2 * lane;
    float o0 = 0.f, o1 = 0.f;
    for (int k = warp; k < a.topk; k += 2 * SB)
    {
        float2 pv[2] = {make_float2(0.f, 0.f), make_float2(0.f, 0.f)};
        float w[2] = {0.f, 0.f};
        half2_t sv[2] = {next[0], next[1]};
        const float* rows2[2] = {a.part_d, a.part_d};
#pragma unroll
        for (int q = 0; q < 2; ++q)
        {
            const int s = k + q * SB;
            if (s >= a.topk || P.weight(s & 63) == 0.f) continue;    // what route() saw: no second look at the table
            w[q] = P.weight(s & 63); rows2[q] = a.part_d + (size_t)s * a.H + col;
        }
        if (k + 2 * SB < a.topk) pick_scales(a, P, k + 2 * SB, SB, col, next);
        if (w[0] == 0.f && w[1] == 0.f) continue;
        sum_partials<2>(rows2, (size_t)a.topk * a.H, NY, pv);
#pragma unroll
        for (int q = 0; q < 2; ++q) add_pick(a, R, P, (k + q * SB) & 63, w[q], pv[q], sv[q], col, lane, o0, o1);
    }
    *(float2*)(red + warp * 128 + 2 * lane) = make_float2(o0, o1);
    __syncthreads();
    if (warp == 0) sum_waves(a, col, red + 2 * lane, SB);
}

// Several tokens: all at once (red: B * SB * 128 floats), N picks of a wavefront in flight with their scales, one barrier. Token by token as
// above, with two barriers each, the last workgroup's tail grew with the tokens: us a call, before and now: 512 x 256, 2 tokens 16.9 -> 15.6;
// 1024 x 384, 4 tokens 29.8 -> 28.3; 4736 x 1152, 3 tokens 72.9 -> 70.9; 2048 x 1024, 4 tokens 52.8 -> 51.8, 8 tokens 83.2 -> 80.0; 6144 x 2048
// the same within the noise. For one token the walk over tokens costs more than it gives (30.7 against 30.5 at 2048 x 1024); N = 2 where
// that is all a wavefront has (four reads' worth of dummies cost 1 us at 512 x 256), else 4.
template <int N>
__device__ __forceinline__ void finish_dn_all(const MoeArgs& a, const PickInfo& R, const PickLanes& P, int grp, int NY, int warp, int SB, int lane, float* red)
{
    const int col = grp * 128 + 2 * lane;
    float o0 = 0.f, o1 = 0.f;
    int b = warp < a.topk ? 0 : a.B, k = warp;                   // the wavefront's next pick: of every token the picks warp, warp + SB, ...
    while (b < a.B)
    {
        int tb[N], ts[N];                                        // token (-1: nothing), pick; the sign of ts: the token's last of this wavefront
        bool end[N];
        float w[N];
        half2_t sv[N];
        float2 pv[N];
        const float* rows[N];
        bool any = false;
#pragma unroll
        for (int q = 0; q < N; ++q)
        {
            tb[q] = b; ts[q] = (b * a.topk + k) & 63; end[q] = k + SB >= a.topk;
            w[q] = b < a.B ? P.weight(ts[q]) : 0.f;              // what route() saw: no second look at the table
            sv[q] = half2_t{};
            rows[q] = a.part_d; pv[q] = make_float2(0.f, 0.f);
            if (w[q] != 0.f)
            {
                sv[q] = *(const half2_t*)(P.sign_row(ts[q]) + a.H + 3 * a.I + col);
                rows[q] = a.part_d + (size_t)ts[q] * a.H + col;
                any = true;
            }
            k += SB;
            if (k >= a.topk) { k = warp; ++b; }
        }
        if (any) sum_partials<N>(rows, (size_t)a.B * a.topk * a.H, NY, pv);
#pragma unroll
        for (int q = 0; q < N; ++q)
        {
            if (tb[q] >= a.B) break;
            add_pick(a, R, P, ts[q], w[q], pv[q], sv[q], col, lane, o0, o1);
            if (end[q])
            {
                *(float2*)(red + (tb[q] * SB + warp) * 128 + 2 * lane) = make_float2(o0, o1);
                o0 = o1 = 0.f;
            }
        }
    }
    __syncthreads();
    for (int t = warp; t < a.B; t += SB) sum_waves(a, (size_t)t * a.H + col, red + t * SB * 128 + 2 * lane, min(SB, a.topk));
}

// MODE 0: gate|up (N = 2I, K = H, input x rotated here). MODE 1: down (N = H, K = I, input h).
// grid (N / 32 / SB, C / NC, S); block 64 * SB threads (SB = 1, 2 or 4: a block covers at most one 128-row group);
// dynamic LDS = rows * (NC * 256 + 16) + 256 bytes (>= rows * SB * 512 for the combine), one row per token of the call
// ANYROW = false: the kernel of a layer whose rows are all of the common kind, base window code 0 and no mask-mode flags (the
// host says so, MoeArgs::common_rows). A run whose row is nevertheless of another kind is not decoded as if it were common:
// its plane is not read and its partial sums are NaN, so every token that picked it comes out NaN. ANYROW = true also
// carries the decode loops of the other base codes and of mask mode, which cost ~35 registers that the common kernel does
// not have to pay for. Four wavefronts per SIMD is the measured optimum for the gate|up launch (three: +4 us per layer; five:
// +1.5 us), so the register allocator is told to aim at exactly that. The common down launch gains from five (90 registers): its
// 1536 workgroups then need 1.2 rounds instead of 1.5 (-0.4 us per layer at one token, -2.5 us at four).
// OWN (gate|up of the common rows only): no routing launch comes before, see launch_moe; the last plane of blocks does that launch's other
// work. A kernel of its own: carried along in the other one, unused, it cost 0.5 to 1.5 % of a call. FEW: gemv_chunks', see launch_moe.
template <int MODE, bool ANYROW, bool OWN = false, bool FEW = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MODE == 1 && !ANYROW ? 5 : 4, MODE == 1 && !ANYROW ? 5 : 4)))
nq_gemv_k(MoeArgs a, int NC)
{
    static_assert(!OWN || MODE == 0, "the gate|up launch takes over the routing");
    extern __shared__ __align__(16) char smem[];
    // Exactly four gate|up workgroups per CU: at one token the launch has four for every CU, and with room for a fifth the
    // dispatcher fills some CUs with five and leaves others with three. The body needs 90 registers; naming v100 claims 104.
    if constexpr (MODE == 0 && !ANYROW) asm volatile("" ::: "v100");
    __builtin_amdgcn_s_setprio(3);                               // the head is a chain of latencies (see progress_priority)
    __shared__ float zl[MAXTOK][4];                              // gate|up finisher: x V_gu^T of the run's tokens (low-rank plane)
    __shared__ int last;
    const int lane = threadIdx.x & 63, warp = threadIdx.x >> 6, SB = blockDim.x >> 6;
    int cnt_step = a.cnt_d_step;
    if constexpr (MODE == 1) asm volatile("" : "+s"(cnt_step));  // read with the first arguments, not in the tail
    if (a.mb_apply && blockIdx.z == gridDim.z - 1)
    {   // the extra plane of blocks of the last projection launch of a call with a mailbox: one of them applies it
        if (blockIdx.x == 0 && blockIdx.y == 0) mailbox_apply(a.mb_table, a.mb_stage, a.mb_seq, a.mb_applied, a.E);
        return;
    }
    if constexpr (OWN) if (blockIdx.z == gridDim.z - 1)
    {   // the extra plane of blocks does the routing launch's other work: what the down launch reads, the publication, the salience
        const int id = blockIdx.x + gridDim.x * blockIdx.y;
        if (id == 0)
        {
            if (threadIdx.x < 64) route(a, a.route, lane);
            else if (a.mb_table && a.mb_applied_host) publish_applied(a.mb_applied, a.mb_applied_host, a.E, threadIdx.x - 64, 192);
            if (threadIdx.x == 0) a.route->ny_gu = gridDim.y;
        }
        else if (id == 1 && a.sal_acc) call_salience(a);
        return;
    }
    // the run's header, written by nq_prep_k: block-uniform, read through the scalar cache (constant address space)
    typedef const __attribute__((address_space(4))) RouteWs* cws_t;
    const cws_t W = (cws_t)a.route;
    struct RawHdr { uint32_t w[sizeof(RunHdr) / 4]; } raw;       // requested together with nruns: one round trip, not two
    int nruns, ny_gu = 0;
    if constexpr (OWN)
    {
        __shared__ OwnRun ow;
        if (warp == 0) own_run(a, blockIdx.z, lane, &ow);
        __syncthreads();
        const uint32_t v = ((const uint32_t*)&ow)[lane < (int)sizeof(OwnRun) / 4 ? lane : 0];      // a word per lane, then into scalar registers
#pragma unroll
        for (int i = 0; i < (int)(sizeof(RunHdr) / 4); ++i) raw.w[i] = __builtin_amdgcn_readlane(v, i);
        nruns = __builtin_amdgcn_readlane(v, sizeof(RunHdr) / 4);
    }
    else
    {
        const __attribute__((address_space(4))) uint32_t* src = (const __attribute__((address_space(4))) uint32_t*)&a.route->run[MODE][blockIdx.z];
#pragma unroll
        for (int i = 0; i < (int)(sizeof(RunHdr) / 4); ++i) raw.w[i] = src[i];
        nruns = W->nruns;
        ny_gu = W->ny_gu;                                        // MODE 1: how many k-slices the gate|up launch that filled part_gu wrote
    }
    const int N = MODE == 0 ? 2 * a.I : a.H, K = MODE == 0 ? a.H : a.I, C = K / 128;
    if (MODE == 1 && nruns == 0 && blockIdx.z == 0 && blockIdx.y == 0)
    {   // no active pick at all: nobody will arrive last, so the first plane of blocks writes the zero output
        for (int i = threadIdx.x; i < a.B * SB * 16; i += blockDim.x)
            out2_store(a, (size_t)(i / (SB * 16)) * a.H + blockIdx.x * SB * 32 + 2 * (i % (SB * 16)), 0.f, 0.f);
    }
    if ((int)blockIdx.z >= nruns) return;                        // block-uniform
    const RunHdr R = __builtin_bit_cast(RunHdr, raw);
    const int NY = C / NC;
    if (MODE == 0 && !OWN && threadIdx.x == 0 && blockIdx.x + blockIdx.y + blockIdx.z == 0) a.route->ny_gu = NY;   // for the down launch's fused staging
    const int ntok = R.ntok, chunk0 = blockIdx.y * NC, k0 = chunk0 * 128;
    const int rowstride = NC * 256 + 16;                         // bytes per staged token (+16: spread tokens over banks)
    char* zero = smem + ntok * rowstride;                        // 256 zero bytes after the token rows
    const _Float16* signs = R.signs;

    // ---- lane context; the first base record is requested now so that its latency overlaps the staging below
    const int t4 = lane >> 4, ss = (lane >> 3) & 1, g = lane & 7, n = lane & 15;
    const int strip = 2 * (blockIdx.x * SB + warp) + ss;
    const Planes P = R.P;                                        // block-uniform: the plane addresses stay in scalar registers
    LaneCtx L;
    L.unit0 = (uint32_t)strip * C + chunk0; L.rec0 = L.unit0 * 32 + 4 * g + t4;
    L.nrec = (size_t)(N / 16) * C * 32;
    L.src = a.G == 2 ? lane ^ 16 : (lane + 16) & 63;             // next record of the ring: rings of four lanes, or of two
    L.g = g; L.strip = (uint32_t)strip; L.nstrips = (size_t)(N / 16); L.chunk0 = chunk0;
    L.half0 = (uint32_t)(2 * (blockIdx.x * SB + warp) + (lane >> 5)) * C + chunk0;
    L.xs = (n < ntok ? smem + n * rowstride : zero) + t4 * 16; L.xstep = n < ntok ? 256 : 0;
    // block-uniform: a row the common kernel has no loop for (its plane is not read: the records have another size or order)
    const bool foreign = !ANYROW && (P.bcode != 0 || (P.flags != nullptr && R.level != 2));
    u32x4 nb0 = {0u, 0u, 0u, 0u};
    if constexpr (ANYROW) { if (P.bcode == 1) nb0 = load_base<1>(P, L.rec0, L.nrec); else nb0 = load_base<0>(P, L.rec0, L.nrec); }
    else if (!foreign) nb0 = load_base<0>(P, L.rec0, L.nrec);

    // ---- stage the run's tokens for this k-slice in B-operand order
    if constexpr (MODE == 0)
    {
        const bool up = (int)(blockIdx.x * SB * 32) >= a.I;      // gate rows are rotated with su_g, up rows with su_u
        _Float16* xr = a.xrot + (up ? a.H : 0) + k0;
        if constexpr (OWN)
        {   // (token, chunk) tasks, four per wavefront at a time; the first row block of either kind leaves its rows where nq_prep_k would
            const WhtSigns ws = wht_signs(lane);
            const int L8 = wht_place(lane), tasks = ntok * NC;
            const bool keep = blockIdx.x * SB * 32 == (up ? a.I : 0);
            for (int q0 = 4 * warp; q0 < tasks; q0 += 4 * SB)
            {
                const int q = min(q0 + (lane >> 4), tasks - 1), j = q / NC, c = q - j * NC, pick = R.slot_of(j);       // lanes beyond the last task repeat it
                const uint4 b = rotate8(a, pick / a.topk, signs + (up ? 2 * a.H + 3 * a.I : 0), chunk0 + c, L8, ws);
                *(uint4*)(smem + j * rowstride + c * 256 + 16 * L8) = b;
                if (keep) *(uint4*)(xr + (size_t)pick * 2 * a.H + c * 128 + 8 * L8) = b;
            }
        }
        else for (int i = threadIdx.x; i < ntok * NC * 16; i += blockDim.x)
        {
            // rotated by nq_prep_k, already in B-operand order: 16 bytes per thread and step
            const int j = i / (NC * 16), r = i - j * NC * 16;
            *(u32x4*)(smem + j * rowstride + r * 16) = *(const u32x4*)(xr + (size_t)R.slot_of(j) * 2 * a.H + r * 8);
        }
    }
    else if (a.fuse && R.had != 512 && R.lr == nullptr)
    {
        // The gate|up finisher, done here for this k-slice's columns of the run's tokens: g = WHT(sum of gate partials) * sv_g,
        // u likewise, h = fp16(WHT(silu(g) * u * su_d)), written straight into the B-operand rows (same operations in the same
        // order as finish_gu, so the same bits). Every column block of the run repeats it; in exchange the gate|up launch ends
        // with its last partial sum and h makes no round trip through memory. Runs whose row has a low-rank plane or the
        // 512-wide rotation keep the finisher in the gate|up launch: both launches read the same row, so they agree.
        const _Float16 *sv_g = signs + a.H, *sv_u = sv_g + a.I, *su_d = sv_u + a.I;
        const int Sgu = a.B * a.topk;
        for (int task = warp; task < ntok * NC; task += SB)
        {
            const int j = task / NC, c = task - j * NC, col = k0 + c * 128 + 2 * lane;
            const float* p = a.part_gu + (size_t)R.slot_of(j) * 2 * a.I + col;
            const float* const rows2[2] = {p, p + a.I};
            const half2_t svg = *(const half2_t*)(sv_g + col), svu = *(const half2_t*)(sv_u + col), sud = *(const half2_t*)(su_d + col);
            float2 pq[2];
            sum_partials<2>(rows2, (size_t)Sgu * 2 * a.I, ny_gu, pq);
            float g0 = pq[0].x, g1 = pq[0].y, u0 = pq[1].x, u1 = pq[1].y;
            wht128(g0, g1, lane); wht128(u0, u1, lane);
            g0 *= (float)svg.x; g1 *= (float)svg.y; u0 *= (float)svu.x; u1 *= (float)svu.y;
            const float sw0 = g0 / (1.f + __expf(-g0)) * u0, sw1 = g1 / (1.f + __expf(-g1)) * u1;
            float v0 = sw0 * (float)sud.x, v1 = sw1 * (float)sud.y;
            wht128(v0, v1, lane);
            asm volatile("" : "+v"(v0), "+v"(v1));            // as in finish_gu: the scaled fp32 value is rounded to fp16, in two steps
            _Float16* dst = (_Float16*)(smem + j * rowstride + c * 256);
            dst[bop_index(2 * lane)] = (_Float16)v0; dst[bop_index(2 * lane + 1)] = (_Float16)v1;
            if (blockIdx.x == 0)                                 // h stays inspectable, as the gate|up finisher leaves it
            {
                half2_t hv; hv.x = (_Float16)v0; hv.y = (_Float16)v1;
                *(half2_t*)(a.h + (size_t)R.slot_of(j) * a.I + col) = hv;
            }
        }
    }
    else
    {
        for (int i = threadIdx.x; i < ntok * NC * 64; i += blockDim.x)
        {
            const int j = i / (NC * 64), r = i % (NC * 64), c = r >> 6, p = r & 63;
            const half2_t hv = *(const half2_t*)(a.h + (size_t)R.slot_of(j) * a.I + k0 + c * 128 + 2 * p);
            _Float16* dst = (_Float16*)(smem + j * rowstride + c * 256);
            dst[bop_index(2 * p)] = hv.x; dst[bop_index(2 * p + 1)] = hv.y;
        }
    }
    if (threadIdx.x < 64) ((uint32_t*)zero)[threadIdx.x] = 0u;
    __syncthreads();

    // ---- decode + MFMA over the k-slice
    float4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    if constexpr (ANYROW)
        dispatch_base(P.bcode, [&](auto bk) {
            constexpr int BK = decltype(bk)::value;
            if (R.level == 2) gemv_chunks<false, 0, BK, true, false, FEW>(P, L, NC, acc, nb0);
            else dispatch_code(P.code, [&](auto tag) { gemv_chunks<true, decltype(tag)::value, BK, true, false, FEW>(P, L, NC, acc, nb0); });
        });
    else if (foreign)
    {
        const float nan = __builtin_nanf("");
        acc[0] = float4_t{nan, nan, nan, nan}; acc[1] = acc[0];
    }
    else if (R.level == 2)
    {
        if (a.hoist && P.var == nullptr) gemv_chunks<false, 0, 0, false, true, FEW>(P, L, NC, acc, nb0);   // block-uniform: the caller's option
        else gemv_chunks<false, 0, 0, false, false, FEW>(P, L, NC, acc, nb0);
    }
    else if (a.hoist && P.var == nullptr) dispatch_code(P.code, [&](auto tag) { gemv_chunks<true, decltype(tag)::value, 0, false, true, FEW>(P, L, NC, acc, nb0); });
    else dispatch_code(P.code, [&](auto tag) { gemv_chunks<true, decltype(tag)::value, 0, false, false, FEW>(P, L, NC, acc, nb0); });

    __builtin_amdgcn_s_setprio(3);                               // the tail is a chain of latencies: nothing should wait behind decoders
    PickLanes picks = {};
    if constexpr (MODE == 1) picks = pick_lanes(a.route->picks, lane);

    // ---- k-slice partial sums: lane (t4, n) holds rows 16 (strip0 + t4 / 2) + 4 (t4 & 1) + i (+ 8 for acc[1]) of token n
    if (n < ntok)
    {
        const int S = a.B * a.topk;
        float* part = (MODE == 0 ? a.part_gu : a.part_d) + ((size_t)blockIdx.y * S + R.slot_of(n)) * N;
        const int row = 16 * (2 * (blockIdx.x * SB + warp) + (t4 >> 1)) + 4 * (t4 & 1);
        st_dev4(part + row, acc[0]);
        st_dev4(part + row + 8, acc[1]);
    }

    // fused finisher: the down launch's staging forms h from these partial sums itself (no arrival counter, no finisher here)
    if (MODE == 0 && a.fuse && R.had != 512 && R.lr == nullptr) return;   // block-uniform (a property of the run's row)

    // ---- arrival counter of the 128-row group this block belongs to; the last block to arrive finishes the group
    const int rows0 = blockIdx.x * SB * 32;
    const int grp = MODE == 0 ? (rows0 % a.I) / 128 : rows0 / 128;
    int* cnt = MODE == 0 ? a.cnt_gu + blockIdx.z * (a.I / 128) + grp : a.cnt_d + grp * cnt_step;
    const int expect = (MODE == 0 ? 2 : nruns) * NY * (128 / (SB * 32));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // this wavefront's partial sums are acknowledged
    const int wv = __builtin_amdgcn_readfirstlane(warp);
    half2_t scales[2] = {};
    if constexpr (MODE == 1) if (a.B == 1) pick_scales(a, picks, wv, SB, grp * 128 + 2 * lane, scales);
    __syncthreads();
    if (threadIdx.x == 0)
        last = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == expect - 1;
    __syncthreads();
    if (!last) return;                                           // block-uniform
    if constexpr (MODE == 0) finish_gu(a, R, zl, blockIdx.z, grp, NY, warp, SB, lane, last);
    else if (!rare(a.B != 1)) finish_dn(a, a.route->picks, picks, scales, grp, NY, wv, SB, lane, (float*)smem);
    else if (a.B * a.topk <= 2 * SB) finish_dn_all<2>(a, a.route->picks, picks, grp, NY, wv, SB, lane, (float*)smem);
    else finish_dn_all<4>(a, a.route->picks, picks, grp, NY, wv, SB, lane, (float*)smem);
    if (threadIdx.x == 0) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The stand-alone mailbox (reference nq_mailbox, sm120/nqmoe.cu:914-923): table[e] <- stage[e] where seq[e] != applied[e], then
// applied[e] <- seq[e]; the host mirror gets every entry of applied, changed or not, so that rows applied by the mailbox block
// of an earlier layer call (which publishes nothing itself) are published here too. Safe to publish at once: this launch
// follows every earlier launch on the stream, and every later one reads the table after it.
__global__ void nq_mailbox_k(int64_t* table, const int64_t* stage, const int32_t* seq, int32_t* applied, int32_t* applied_host, int E)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    const int32_t sq = __hip_atomic_load(seq + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    int32_t ap = applied[e];
    if (sq != ap)
    {
#pragma unroll
        for (int i = 0; i < TBL_W; ++i)
            table[(size_t)e * TBL_W + i] = __hip_atomic_load(stage + (size_t)e * TBL_W + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __threadfence();
        applied[e] = ap = sq;
    }
    if (applied_host) __hip_atomic_store(applied_host + e, ap, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Which calls do without the routing launch: both projections in the call, rows of the common kind, and a gate|up launch of at most two
// workgroups on each of 256 CUs. Every one of them then repeats the routing (about 2 us, three dependent reads) and rotates
// its own columns, beside one another, in place of a launch of 3.4 to 4.9 us before them. us a call with / without the routing launch: 256 x 128,
// 1 token 15.0 / 12.8; 512 x 256, 2 tokens 15.6 / 14.3; 2048 x 1024, 3 picks 18.0 / 16.7; 6144 x 2048, 4 picks 41.7 / 40.3. With four on each (1024)
// 2048 x 1024, 8 picks 24.2 / 23.4, but 6144 x 2048, 8 picks 58.0 / 56.2 to 58.9 from one process to the next; beyond that a second round
// pays for it again: 2048 x 1024, 6 picks (1536) 22.9 / 24.6, 896 x 512, 8 tokens (3584) 45.6 / 63.9.
// With a layer and inputs met for the first time, nothing of them in any cache, the heads cost more and the gain is smaller. us of the two
// projection kernels, and of the routing launch before them: 512 x 256, 2 tokens 4.4 + 17.4 / 20.1; repeated 3.4 + 14.0 / 14.2.
constexpr int OWN_ROUTE_WGS = 512;
// Slices of fewer chunks work a unit's constants out where they are needed (gemv_chunks' FEW). us a call of mixed levels in a graph, UnitConsts
// in both projections / in gate|up alone / in down alone / in neither; chunks of a gate|up and a down slice. One chunk, where there is nothing to share:
//   1152 x 640, 8 picks (1, 1) 19.30 / 19.23 / 19.33 / 19.17; 1536 x 768, 8 (1, 1) 21.24 / 21.14 / 21.08 / 20.91; 2176 x 896, 24 (1, 1) 48.47 / 48.13 / 48.20 / 47.95;
//   2048 x 1024, 6 (1, 1) 23.29 / 23.28 / 22.99 / 23.08, 16 (4, 1) 41.19 / 40.56 / 42.35 / 41.79; 6144 x 2048, 2 (3, 1) 33.19 / 33.04 / 33.25 / 33.32.
// Two and more: 3072 x 1536, 16 (8, 3) 47.65 / 48.08 / 48.37 / 48.65; 4096 x 2048, 8 (8, 2) 46.92 / 47.01 / 47.46 / 47.59; 6144 x 2048, 8 (12, 4)
//   60.81 / 61.14 / 61.21 / 61.77, 32 (24, 4) 201.2 / 202.1 / 204.4 / 205.4.
// A lone projection's slices likewise (launch_proj), UnitConsts / without, its weights in no cache: 6144 x 4096, 8 tokens, level 3, three chunks 14.63 / 15.18.
// In slices of one, weights at hand, 2048 x 2048, 8 tokens, level 4 7.38 / 7.22; 1024 x 1024, one 5.97 / 5.79; 512 x 512, 8, level 3 6.28 / 6.08.
constexpr int FEW_CHUNKS = 2;
int launch_moe(const MoeArgs& a, const int* cfg_gu, const int* cfg_dn, int which, hipStream_t st)
{
    const int S = a.B * a.topk;
    const bool reuse = (which & 4) != 0;                          // the routing launch of an earlier call left route_ws / xrot as this call needs them
    const bool defer = (which & 8) != 0;                          // two-call form of the one-call arithmetic: h is formed by the down launch
    which &= 3;
    const bool own = which == 3 && !reuse && a.common_rows == 1 && cfg_gu[1] == 4 && (2 * a.I / 128) * (a.H / 128 / (cfg_gu[0] * cfg_gu[2])) * S <= OWN_ROUTE_WGS;
    if (!reuse && !own)
    {
        const int ntask = S * 2 * (a.H / 128);                   // upper bound: every pick active
        nq_prep_k<<<std::min((ntask + 3) / 4, 1023) + (a.sal_acc ? 2 : 1), 256, 0, st>>>(a);       // one workgroup per four rotation tasks, plus the one that routes
        NQ_LAUNCH_CHECK("moe_forward (routing)");
    }
    // a call with a mailbox and no projection launch: the apply half as a launch of its own (nothing is published here either)
    if (a.mb_table && which == 0) return launch_mailbox(a.mb_table, a.mb_stage, a.mb_seq, a.mb_applied, nullptr, a.E, st);
    const int last_mode = (which & 2) ? 1 : 0;
    for (int mode = 0; mode < 2; ++mode)
    {
        if (!((which >> mode) & 1)) continue;
        const int* cf = mode == 0 ? cfg_gu : cfg_dn;
        const int NC = cf[0] * cf[2], SB = cf[1];
        const int N = mode == 0 ? 2 * a.I : a.H, K = mode == 0 ? a.H : a.I, C = K / 128;
        const int NX = N / 32 / SB, NY = C / NC;
        const int shm = std::max(a.B * (NC * 256 + 16) + 256, (mode == 1 ? a.B : 1) * SB * 512);
        const bool any = a.common_rows != 1;
        MoeArgs b = a;
        b.fuse = which == 3 || defer;                             // both launches belong to this call (or the caller says the other one follows)
        b.mb_apply = a.mb_table != nullptr && mode == last_mode;  // the call's last projection launch carries the mailbox block
        const bool self = own && mode == 0;
        const bool few = own || NC < FEW_CHUNKS;
        auto kern = self ? nq_gemv_k<0, false, true, true>
                  : mode == 0 ? (any ? few ? nq_gemv_k<0, true, false, true> : nq_gemv_k<0, true> : few ? nq_gemv_k<0, false, false, true> : nq_gemv_k<0, false>)
                              : (any ? few ? nq_gemv_k<1, true, false, true> : nq_gemv_k<1, true> : few ? nq_gemv_k<1, false, false, true> : nq_gemv_k<1, false>);
        if (shm > 48 * 1024)
        {
            hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
            if (e != hipSuccess) return set_error("moe_forward: LDS %d bytes: %s", shm, hipGetErrorString(e));
        }
        kern<<<dim3(NX, NY, S + (b.mb_apply || self ? 1 : 0)), 64 * SB, shm, st>>>(b, NC);
        NQ_LAUNCH_CHECK("moe_forward");
    }
    return 0;
}

// ---- nq_moe_forward_static: the same two launches with every workspace carved from one built-in device array --------------
// For callers that cannot allocate (stream capture, serving loops, harnesses that forbid hipMalloc). Each GPU holds its own
// copy of the array at its own address; in host code the array's name is only a handle for hipGetSymbolAddress, which is
// asked once per device, with that device current, and the address it returns is what the kernels are given. Calls on one
// GPU share the array: two calls that overlap on one GPU (different streams) race.
constexpr size_t STATIC_SCRATCH_BYTES = (size_t)NQ_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];
constexpr int MAX_DEVICES = 64;
static unsigned char* g_scratch_ptr[MAX_DEVICES] = {};
static std::mutex g_scratch_mu;

__global__ void nq_clear_k(int* p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

int launch_moe_static(MoeArgs a, const int* cfg_gu, const int* cfg_dn, int which, hipStream_t st)
{
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return set_error("nq_moe_forward_static: current device %d: %s", dev, hipGetErrorString(e));
    unsigned char* base;
    {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        if (!g_scratch_ptr[dev])
        {
            void* ptr = nullptr;
            e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
            if (e != hipSuccess || !ptr) return set_error("nq_moe_forward_static: address of the built-in scratch on device %d: %s", dev, hipGetErrorString(e));
            g_scratch_ptr[dev] = (unsigned char*)ptr;
        }
        base = g_scratch_ptr[dev];
    }
    const size_t S = (size_t)a.B * a.topk, G128 = (size_t)a.I / 128;
    const size_t ny_gu = (size_t)(a.H / 128) / (cfg_gu[0] * cfg_gu[2]), ny_dn = (size_t)(a.I / 128) / (cfg_dn[0] * cfg_dn[2]);
    size_t off = 0;
    auto take = [&](size_t bytes) { const size_t o = off; off += (bytes + 255) & ~(size_t)255; return o; };
    const size_t o_gu = take(ny_gu * S * 2 * a.I * sizeof(float)), o_d = take(ny_dn * S * a.H * sizeof(float));
    const size_t o_h = take(S * a.I * sizeof(_Float16)), o_zd = take(S * G128 * 4 * sizeof(float)), o_route = take(sizeof(RouteWs)), o_xrot = take(S * 2 * a.H * sizeof(_Float16));
    const size_t before = off, wide = (2 * S * G128 + (size_t)a.H / 128 * NQ_CNT_STEP) * sizeof(int);      // the counters as far apart as there is room
    a.cnt_d_step = before + wide <= STATIC_SCRATCH_BYTES ? NQ_CNT_STEP : 1;
    const size_t o_cnt = take((2 * S * G128 + (size_t)a.H / 128 * a.cnt_d_step) * sizeof(int));             // cnt_gu | cnt_h | cnt_d: cleared below
    if (off > STATIC_SCRATCH_BYTES)
        return set_error("nq_moe_forward_static: this call needs %zu bytes of workspace (B=%d topk=%d H=%d I=%d, %zu and %zu k-slices), the built-in "
                         "scratch holds %zu: use coarser k-slices, or nq_moe_forward with workspaces of the caller's", off, a.B, a.topk, a.H, a.I, ny_gu, ny_dn,
                         STATIC_SCRATCH_BYTES);
    a.cnt_gu = (int*)(base + o_cnt); a.cnt_h = a.cnt_gu + S * G128; a.cnt_d = a.cnt_h + S * G128;
    a.part_gu = (float*)(base + o_gu); a.part_d = (float*)(base + o_d); a.h = (_Float16*)(base + o_h); a.zd = (float*)(base + o_zd);
    a.route = (RouteWs*)(base + o_route); a.xrot = (_Float16*)(base + o_xrot);
    // the counters must be zero on entry; a fill kernel, not hipMemsetAsync, so that the call can be recorded into a graph
    const int ncnt = (int)(2 * S * G128 + (size_t)a.H / 128 * a.cnt_d_step);
    nq_clear_k<<<(ncnt + 255) / 256, 256, 0, st>>>(a.cnt_gu, ncnt);
    NQ_LAUNCH_CHECK("nq_moe_forward_static");
    return launch_moe(a, cfg_gu, cfg_dn, which, st);
}

// ---- a lone projection ---------------------------------------------------------------------------------------------------------
// out[B][2I] = W_gu . fp16(Hadamard-128(x * su)) of one expert for B tokens in one launch: what a gate|up launch of one run computes,
// whose routing the host knows. grid (row blocks, k-slices), block 64 * SB; a workgroup reads the table row, rotates its own k-slice of
// the tokens (eight columns per lane, four chunks per wavefront at a time: a tenth of its decode) and decodes as nq_gemv_k does. The
// last workgroup of a 128-row group adds the group's slices in slice order. Common rows only, as nq_gemv_k<0, false>: another kind comes out NaN.
// Bound by latency beside the decode: table row, then records and sign vector, then 5.8 us of decode issue at level 3 (6144 x 4096), then
// acknowledged stores, arrival counter and the slices' sums. Eight tokens, us a call: levels 2 / 3 / 4 10.7 / 13.7 / 13.8, where routing
// launch, gate|up launch and slice sums took 20.4 / 19.0 / 19.0; slices of 2, 3, 6 or 8 chunks 13.5, 13.6, 14.2, 16.9 at level 3.
struct ProjArgs { const void* x; const int64_t* row; float* part; int* cnt; float* out; int x_dtype, B, H, I, G, cnt_step; };
__device__ __forceinline__ float4_t ld_dev4_issue(const float* p)
{
    float4_t v;
    asm volatile("global_load_dwordx4 %0, %1, off sc0 sc1" : "=v"(v) : "v"(p) : "memory");
    return v;
}
template <bool FEW>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) nq_proj_k(ProjArgs a, int NC)
{
    extern __shared__ __align__(16) char smem[];
    __builtin_amdgcn_s_setprio(3);
    __shared__ int last;
    const int lane = threadIdx.x & 63, warp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), SB = blockDim.x >> 6;
    int64_t ent[TBL_W];                                          // block-uniform: through the scalar cache
    const __attribute__((address_space(4))) int64_t* src = (const __attribute__((address_space(4))) int64_t*)a.row;
#pragma unroll
    for (int i = 0; i < TBL_W; ++i) ent[i] = src[i];
    const int N = 2 * a.I, C = a.H / 128, NY = C / NC, chunk0 = blockIdx.y * NC, rowstride = NC * 256 + 16;
    const int t4 = lane >> 4, ss = (lane >> 3) & 1, g = lane & 7, n = lane & 15;
    // the tokens' k-slice, before the row is there: chunk-tasks (token, chunk), four per wavefront at a time
    const int L8 = wht_place(lane), tasks = a.B * NC, col8 = 32 * (L8 >> 2) + 2 * (L8 & 3);
    const int strip = 2 * (blockIdx.x * SB + warp) + ss;
    const int level = (int)ent[0];
    const Planes P = planes_of(ent, 0);
    const bool live = level > 0, foreign = P.bcode != 0 || (P.flags != nullptr && level != 2);
    LaneCtx L;
    L.unit0 = (uint32_t)strip * C + chunk0; L.rec0 = L.unit0 * 32 + 4 * g + t4;
    L.nrec = (size_t)(N / 16) * C * 32;
    L.src = a.G == 2 ? lane ^ 16 : (lane + 16) & 63;
    L.g = g; L.strip = (uint32_t)strip; L.nstrips = (size_t)(N / 16); L.chunk0 = chunk0;
    L.half0 = (uint32_t)(2 * (blockIdx.x * SB + warp) + (lane >> 5)) * C + chunk0;
    char* zero = smem + a.B * rowstride;
    L.xs = (n < a.B ? smem + n * rowstride : zero) + t4 * 16; L.xstep = n < a.B ? 256 : 0;
    u32x4 nb0 = {0u, 0u, 0u, 0u};
    if (live && !foreign) nb0 = load_base<0>(P, L.rec0, L.nrec);
    const WhtSigns ws = wht_signs(lane);
    const _Float16* su = (const _Float16*)ent[9] + ((int)(blockIdx.x * SB * 32) >= a.I ? 2 * a.H + 3 * a.I : 0);
    for (int q0 = 4 * warp; live && q0 < tasks; q0 += 4 * SB)
    {
        const int q = min(q0 + (lane >> 4), tasks - 1), j = q / NC, c = q - j * NC;       // lanes beyond the last task repeat it
        const size_t at = (size_t)j * a.H + (chunk0 + c) * 128 + col8;
        half2_t xv[4], sv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) { xv[i] = act2_at(a.x, a.x_dtype, at + 8 * i); sv[i] = *(const half2_t*)(su + (chunk0 + c) * 128 + col8 + 8 * i); }
        float v[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) { v[2 * i] = (float)xv[i].x * (float)sv[i].x; v[2 * i + 1] = (float)xv[i].y * (float)sv[i].y; }
        wht8_bop_sums(v, ws);
        *(uint4*)(smem + j * rowstride + c * 256 + 16 * L8) = bop_block_scaled(v, ws.scale);      // one rounding, as nq_prep_k: the same bits
    }
    if (threadIdx.x < 64) ((uint32_t*)zero)[threadIdx.x] = 0u;
    __syncthreads();

    float4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    if (foreign) { const float nan = __builtin_nanf(""); acc[0] = float4_t{nan, nan, nan, nan}; acc[1] = acc[0]; }
    else if (level == 2) gemv_chunks<false, 0, 0, false, false, FEW>(P, L, NC, acc, nb0);
    else if (live) dispatch_code(P.code, [&](auto tag) { gemv_chunks<true, decltype(tag)::value, 0, false, false, FEW>(P, L, NC, acc, nb0); });
    __builtin_amdgcn_s_setprio(3);

    const int row = 16 * (2 * (blockIdx.x * SB + warp) + (t4 >> 1)) + 4 * (t4 & 1);
    if (NY == 1)
    {
        if (n < a.B) { float* o = a.out + (size_t)n * N + row; *(float4_t*)o = acc[0]; *(float4_t*)(o + 8) = acc[1]; }
        return;
    }
    if (n < a.B)
    {
        float* part = a.part + ((size_t)blockIdx.y * a.B + n) * N + row;
        st_dev4(part, acc[0]); st_dev4(part + 8, acc[1]);
    }
    // the hand-off of nq_gemv_k: acknowledged stores, then the group's counter; the last to arrive reads the slices device-coherently
    const int grp = blockIdx.x * SB * 32 / 128, expect = NY * (128 / (SB * 32));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) last = __hip_atomic_fetch_add(a.cnt + grp * a.cnt_step, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == expect - 1;
    __syncthreads();
    if (!last) return;
    for (int i = threadIdx.x; i < a.B * 32; i += blockDim.x)     // four rows of one token each
    {
        const size_t at = (size_t)(i >> 5) * N + grp * 128 + 4 * (i & 31);
        float4_t s = {0.f, 0.f, 0.f, 0.f};
        for (int y = 0; y < NY; y += 8)
        {
            float4_t v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = ld_dev4_issue(a.part + (size_t)(y + k < NY ? y + k : y) * a.B * N + at);
#pragma unroll
            for (int k = 0; k < 8; k += 4) asm volatile("s_waitcnt vmcnt(0)" : "+v"(v[k]), "+v"(v[k + 1]), "+v"(v[k + 2]), "+v"(v[k + 3]) :: "memory");
#pragma unroll
            for (int k = 0; k < 8; ++k) if (y + k < NY) s += v[k];
        }
        *(float4_t*)(a.out + at) = s;
    }
    if (threadIdx.x == 0) __hip_atomic_store(a.cnt + grp * a.cnt_step, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
int launch_proj(const void* x, int x_dtype, int B, const int64_t* row, int H, int I, int G, int NC, int SB, float* part, int* cnt, int cnt_step, float* out, hipStream_t st)
{
    const ProjArgs a{x, row, part, cnt, out, x_dtype, B, H, I, G, cnt_step};
    const int shm = B * (NC * 256 + 16) + 256;
    auto kern = NC < FEW_CHUNKS ? nq_proj_k<true> : nq_proj_k<false>;
    if (shm > 48 * 1024)
    {
        const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
        if (e != hipSuccess) return set_error("nq_proj: LDS %d bytes: %s", shm, hipGetErrorString(e));
    }
    kern<<<dim3(2 * I / 32 / SB, H / 128 / NC), 64 * SB, shm, st>>>(a, NC);
    NQ_LAUNCH_CHECK("nq_proj");
    return 0;
}

// out[i] = sum over the ny k-slices of part[y * n + i], in slice order (n a multiple of 4): what is left of a lone projection. Bound by
// the launch: 24 slices of 8 x 4096 (3 MB, just written, so from the last-level cache) take 2.8 us where a library sum over the first
// dimension took 5.4 us and chose its blocks on the host first; a projection of eight tokens 21.4 -> 19.3 us.
__global__ void __launch_bounds__(256) nq_sum_slices_k(const float* __restrict__ part, int ny, int64_t n, float* __restrict__ out)
{
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= n) return;
    float4_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int y = 0; y < ny; ++y) s += *(const float4_t*)(part + y * n + i);
    *(float4_t*)(out + i) = s;
}
int launch_sum_slices(const float* part, int ny, int64_t n, float* out, hipStream_t st)
{
    nq_sum_slices_k<<<(unsigned)((n / 4 + 255) / 256), 256, 0, st>>>(part, ny, n, out);
    NQ_LAUNCH_CHECK("nq_sum_slices");
    return 0;
}

// resident workgroups per CU, registers and spill bytes of a decode kernel for a launch shape
int query_occ(int mode, int any_rows, int sb, int shm, int* out)
{
    auto kern = mode == 0 ? (any_rows ? nq_gemv_k<0, true> : nq_gemv_k<0, false>) : (any_rows ? nq_gemv_k<1, true> : nq_gemv_k<1, false>);
    hipError_t e;
    if (shm > 48 * 1024 && (e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, shm)) != hipSuccess)
        return set_error("nq_occ: LDS %d bytes: %s", shm, hipGetErrorString(e));
    int nb = 0;
    if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, (const void*)kern, 64 * sb, (size_t)shm)) != hipSuccess)
        return set_error("nq_occ: %s", hipGetErrorString(e));
    hipFuncAttributes fa;
    if ((e = hipFuncGetAttributes(&fa, (const void*)kern)) != hipSuccess) return set_error("nq_occ: %s", hipGetErrorString(e));
    out[0] = nb; out[1] = fa.numRegs; out[2] = (int)fa.localSizeBytes;
    return 0;
}

int launch_mailbox(int64_t* table, const int64_t* stage, const int32_t* seq, int32_t* applied, int32_t* applied_host, int E, hipStream_t st)
{
    nq_mailbox_k<<<(E + 127) / 128, 128, 0, st>>>(table, stage, seq, applied, applied_host, E);
    NQ_LAUNCH_CHECK("nq_mailbox");
    return 0;
}

}  // namespace nq
