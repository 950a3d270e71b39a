// Pieces shared by the decode-path GEMV (nq_moe.hip) and the prefill grouped GEMM (nq_prefill.hip): the wavefront
// Hadamard-128, the B-operand column order, and the stream of MFMA A operands decoded from trellis records.
//
// Lane mapping (wave64): lane = 16 * t4 + 8 * ss + g decodes the record of lane (4 g + t4) of unit (strip0 + ss, chunk).
// It holds 32 weights of row g and 32 of row g + 8, in columns 16 t + 2 t4 + {0,1,8,9}. v_mfma_f32_16x16x32_f16 takes 8
// fp16 per lane; lanes with equal (ss, g) and different t4 are the four k-groups of one A row, so the decoded pairs
// (w_j, w_{j+8}) are A operands as they leave the decoder. MFMA (MM, RHO) covers rows g + 8 RHO and the columns of
// t = 2 MM, 2 MM + 1; its B operand (16 tokens) holds the same columns, see bop_index().
#pragma once
#include "nq_decode.hpp"
#include <utility>

namespace nq {

// ---- caller dtypes: the casts a caller would otherwise launch as separate kernels (x.half(), ids.long(), w.half(),
// out.to(x.dtype); reference sm120/serve/nq_vllm.py:522,560,573) happen at the loads and the final store, with the same
// roundings: activations and routing weights pass through fp16, the fp32 result is rounded once to the output type.
constexpr int DT_BF16 = 1, DT_F32 = 2, DT_I32 = 1, DT_OUT_F16 = 1, DT_OUT_BF16 = 2;   // 0 = the default type of each argument (fp16, int64, fp32 out)
__device__ __forceinline__ float bf16_to_f(uint16_t v) { return __builtin_bit_cast(float, (uint32_t)v << 16); }
__device__ __forceinline__ uint16_t f_to_bf16(float f)           // round to nearest even; NaN stays NaN
{
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ long long id_at(const void* sel, int dt, size_t i)
{
    return dt == DT_I32 ? (long long)((const int32_t*)sel)[i] : (long long)((const int64_t*)sel)[i];
}
__device__ __forceinline__ float w_at(const void* rw, int dt, size_t i)   // the weight as fp16 would hold it
{
    if (dt == DT_BF16) return (float)(_Float16)bf16_to_f(((const uint16_t*)rw)[i]);
    if (dt == DT_F32) return (float)(_Float16)((const float*)rw)[i];
    return (float)((const _Float16*)rw)[i];
}
__device__ __forceinline__ half2_t act2_at(const void* x, int dt, size_t i)   // x[i], x[i + 1] (i even) as fp16
{
    if (dt == DT_BF16)
    {
        const uint32_t v = *(const uint32_t*)((const uint16_t*)x + i);
        return half2_t{(_Float16)bf16_to_f((uint16_t)v), (_Float16)bf16_to_f((uint16_t)(v >> 16))};
    }
    if (dt == DT_F32) { const float2 v = *(const float2*)((const float*)x + i); return half2_t{(_Float16)v.x, (_Float16)v.y}; }
    return *(const half2_t*)((const _Float16*)x + i);
}
__device__ __forceinline__ uint4 act8_at(const void* x, int dt, size_t i)     // x[i .. i + 7] (i a multiple of 8) as fp16
{
    if (dt == 0) return *(const uint4*)((const _Float16*)x + i);
    half8_t h;
    if (dt == DT_BF16)
    {
        const uint4 v = *(const uint4*)((const uint16_t*)x + i);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) { h[2 * q] = (_Float16)bf16_to_f((uint16_t)w[q]); h[2 * q + 1] = (_Float16)bf16_to_f((uint16_t)(w[q] >> 16)); }
    }
    else
    {
        const float4 a = *(const float4*)((const float*)x + i), b = *(const float4*)((const float*)x + i + 4);
        const float f[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int q = 0; q < 8; ++q) h[q] = (_Float16)f[q];
    }
    return __builtin_bit_cast(uint4, h);
}
__device__ __forceinline__ void res2_store(void* out, int dt, size_t i, float v0, float v1)   // out[i], out[i + 1] (i even)
{
    if (dt == DT_OUT_F16) { half2_t h; h.x = (_Float16)v0; h.y = (_Float16)v1; *(half2_t*)((_Float16*)out + i) = h; }
    else if (dt == DT_OUT_BF16) *(uint32_t*)((uint16_t*)out + i) = (uint32_t)f_to_bf16(v0) | ((uint32_t)f_to_bf16(v1) << 16);
    else *(float2*)((float*)out + i) = make_float2(v0, v1);
}

// ---- Hadamard-128 on one wavefront: lane holds elements 2 lane, 2 lane + 1 --------------------------------------------
// One in-lane butterfly, then six cross-lane stages: lanes l and l ^ m exchange, the lane with bit m clear keeps a + a',
// the other a' - a (a' = the partner's value), all in fp32 in this order. The exchanges use no LDS: DPP lane selects for
// m = 1, 2, 4, 8 (quad permutes, a half-row mirror, a row rotate), and for m = 16, 32 the row / half swaps of gfx950, which
// leave both partners' values in both lanes. The per-lane sign is a sign-bit flip (or a factor +-1 in an FMA), so every sum
// is the same single rounding as a plain add or subtract. All 64 lanes must be active.
template <int CTRL> __device__ __forceinline__ float dpp_lane(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float flip_sign(float v, uint32_t m) { return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) ^ m); }
// lo / hi = the value of the lane with bit 16 (bit 32) clear / set, in both lanes. The swap exchanges the odd 16-lane rows
// (the upper half) of its first register with the even rows (the lower half) of its second; the two read-write operands
// force two distinct registers that start as the same value. Written as asm because the compiler's builtin for it hands
// back the first register for both results; the compiler therefore does not see the instruction and cannot place the wait
// states it needs after the writes that feed it and before the reads of its results, so they are written out here.
__device__ __forceinline__ void swap_rows16(float v, float& lo, float& hi)
{
    lo = v; hi = v;
    asm volatile("s_nop 3\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 3" : "+v"(lo), "+v"(hi));
}
__device__ __forceinline__ void swap_halves32(float v, float& lo, float& hi)
{
    lo = v; hi = v;
    asm volatile("s_nop 3\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 3" : "+v"(lo), "+v"(hi));
}
constexpr float WHT128_SCALE = 0.08838834764f;                   // 1 / sqrt(128)
__device__ __forceinline__ void wht128_sums(float& a, float& b, int lane)        // still to be multiplied by WHT128_SCALE
{
    const float s = a + b, d = a - b; a = s; b = d;
    const uint32_t l = (uint32_t)lane;
    const uint32_t n1 = (l << 31) & 0x80000000u, n2 = (l << 30) & 0x80000000u, n4 = (l << 29) & 0x80000000u, n8 = (l << 28) & 0x80000000u;
    a = dpp_lane<0xB1>(a) + flip_sign(a, n1); b = dpp_lane<0xB1>(b) + flip_sign(b, n1);                   // quad_perm [1,0,3,2]
    a = dpp_lane<0x4E>(a) + flip_sign(a, n2); b = dpp_lane<0x4E>(b) + flip_sign(b, n2);                   // quad_perm [2,3,0,1]
    a = dpp_lane<0x141>(dpp_lane<0x1B>(a)) + flip_sign(a, n4);                                            // l ^ 3 then l ^ 7 = l ^ 4
    b = dpp_lane<0x141>(dpp_lane<0x1B>(b)) + flip_sign(b, n4);
    a = dpp_lane<0x128>(a) + flip_sign(a, n8); b = dpp_lane<0x128>(b) + flip_sign(b, n8);                 // row_ror 8
    const float s16 = (lane & 16) ? -1.f : 1.f, s32 = (lane & 32) ? -1.f : 1.f;
    float lo, hi;
    swap_rows16(a, lo, hi); a = __builtin_fmaf(hi, s16, lo);
    swap_rows16(b, lo, hi); b = __builtin_fmaf(hi, s16, lo);
    swap_halves32(a, lo, hi); a = __builtin_fmaf(hi, s32, lo);
    swap_halves32(b, lo, hi); b = __builtin_fmaf(hi, s32, lo);
}
__device__ __forceinline__ void wht128(float& a, float& b, int lane)
{
    wht128_sums(a, b, lane);
    a *= WHT128_SCALE; b *= WHT128_SCALE;
}

// ---- Hadamard-128 on sixteen lanes: eight elements per lane, four chunks per wavefront ---------------------------------
// The throughput form for kernels that rotate many rows: three butterflies in the lane, four between lanes of a DPP row, 64 instructions
// for 512 elements (wht128 takes about 50 for 128). A lane's place L = 0..15 in its chunk is chosen so that the four
// lane bits of L are exchanged by the lane masks 1, 2, 7, 8, each one DPP select (wht_place: lane = L0 ^ 2 L1 ^ 7 L2 ^ 8 L3). A lane whose bit is set would
// hold a' - a; it keeps a - a' instead, one multiply-add by +-1 with the exchange inside it, and since a lane's sign is common to all
// it holds and to its partners in the later exchanges, the last multiplication puts it right. The sums and their roundings are
// those of wht128. Which columns a place and its eight elements stand for: wht8_bop, wht8_row.
__device__ __forceinline__ int wht_place(int lane) { return (lane & 4) ? (lane & 15) ^ 3 : lane & 15; }
struct WhtSigns { float s0, s1, s2, s3, scale; };
__device__ __forceinline__ WhtSigns wht_signs(int lane)
{
    const int L = wht_place(lane);
    const float s0 = (L & 1) ? -1.f : 1.f, s1 = (L & 2) ? -1.f : 1.f, s2 = (L & 4) ? -1.f : 1.f, s3 = (L & 8) ? -1.f : 1.f;
    return WhtSigns{s0, s1, s2, s3, WHT128_SCALE * s0 * s1 * s2 * s3};
}
// v[i] = v[i] + s * (v[i] of the partner lane). Asm, because the compiler puts the select into a move of its own; a DPP read needs two
// wait states after the write of its register, which it cannot see, so they are written out.
#define NQ_WHT_LANES(NAME, SELECT) \
__device__ __forceinline__ void NAME(float* v, float s) \
{ \
    asm("s_nop 1\n\t" \
        "v_fmac_f32_dpp %0, %0, %8 " SELECT " row_mask:0xf bank_mask:0xf\n\tv_fmac_f32_dpp %1, %1, %8 " SELECT " row_mask:0xf bank_mask:0xf\n\t" \
        "v_fmac_f32_dpp %2, %2, %8 " SELECT " row_mask:0xf bank_mask:0xf\n\tv_fmac_f32_dpp %3, %3, %8 " SELECT " row_mask:0xf bank_mask:0xf\n\t" \
        "v_fmac_f32_dpp %4, %4, %8 " SELECT " row_mask:0xf bank_mask:0xf\n\tv_fmac_f32_dpp %5, %5, %8 " SELECT " row_mask:0xf bank_mask:0xf\n\t" \
        "v_fmac_f32_dpp %6, %6, %8 " SELECT " row_mask:0xf bank_mask:0xf\n\tv_fmac_f32_dpp %7, %7, %8 " SELECT " row_mask:0xf bank_mask:0xf" \
        : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]) : "v"(s)); \
}
NQ_WHT_LANES(wht_lanes1, "quad_perm:[1,0,3,2]")                  // lane ^ 1
NQ_WHT_LANES(wht_lanes2, "quad_perm:[2,3,0,1]")                  // lane ^ 2
NQ_WHT_LANES(wht_lanes7, "row_half_mirror")                      // lane ^ 7
NQ_WHT_LANES(wht_lanes8, "row_ror:8")                            // lane ^ 8
#undef NQ_WHT_LANES
template <int D> __device__ __forceinline__ void wht_inside(float* v)
{
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if (!(i & D)) { const float a = v[i], b = v[i + D]; v[i] = a + b; v[i + D] = a - b; }
}
// place L = 4 mm + kg of the chunk; v[j + 2 a + 4 b] = column 32 mm + 2 kg + j + 8 a + 16 b
__device__ __forceinline__ void wht8_bop_sums(float* v, const WhtSigns& w)       // still to be multiplied by w.scale
{
    wht_inside<1>(v); wht_lanes1(v, w.s0); wht_lanes2(v, w.s1);        // columns apart by 1, 2, 4
    wht_inside<2>(v); wht_inside<4>(v);                                          // 8, 16
    wht_lanes7(v, w.s2); wht_lanes8(v, w.s3);                        // 32, 64
}
__device__ __forceinline__ void wht8_bop(float* v, const WhtSigns& w)
{
    wht8_bop_sums(v, w);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] *= w.scale;
}
// v[j] = column 8 L + j
__device__ __forceinline__ void wht8_row(float* v, const WhtSigns& w)
{
    wht_inside<1>(v); wht_inside<2>(v); wht_inside<4>(v);
    wht_lanes1(v, w.s0); wht_lanes2(v, w.s1); wht_lanes7(v, w.s2); wht_lanes8(v, w.s3);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] *= w.scale;
}
__device__ __forceinline__ uint32_t pack_f16(float lo, float hi)
{
    half2_t h; h.x = (_Float16)lo; h.y = (_Float16)hi;
    return __builtin_bit_cast(uint32_t, h);
}
// the 16-byte block (mm, kg) of the B-operand order from wht8_bop's arrangement: halfs 2 i + hi = column i's pair (c, c + 16)
__device__ __forceinline__ uint4 bop_block(const float* v)
{
    return make_uint4(pack_f16(v[0], v[4]), pack_f16(v[1], v[5]), pack_f16(v[2], v[6]), pack_f16(v[3], v[7]));
}
// fp16 of scale * v, rounded once. Asm, because the compiler merges a multiplication into a conversion at some call sites and not at
// others, and the rotations of one activation must give the same bits in every launch that makes them.
__device__ __forceinline__ _Float16 f16_scaled(float v, float scale)
{
    uint32_t d;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(d) : "v"(v), "v"(scale));
    return __builtin_bit_cast(_Float16, (uint16_t)d);
}
// the block of scale * v, likewise
__device__ __forceinline__ uint4 bop_block_scaled(const float* v, float scale)
{
    uint32_t d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(d[i]) : "v"(v[i]), "v"(scale));
        asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(d[i]) : "v"(v[i + 4]), "v"(scale));
    }
    return make_uint4(d[0], d[1], d[2], d[3]);
}
// the same from wht8_row's arrangement: two exchanges within the four lanes that hold columns 32 mm .. 32 mm + 31 (places 4 mm + q,
// q = bit 3 of the column + 2 * bit 4): first with the lane 16 columns on, which makes the pairs, then with the one 8 columns on.
template <int CTRL> __device__ __forceinline__ uint32_t dpp_word(uint32_t v) { return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true); }
__device__ __forceinline__ uint4 bop_block_of_row(const float* v, int lane)
{
    const int L = wht_place(lane);
    const bool hi = L & 2, up = L & 1;
    uint32_t d[4];                                               // columns (0, 1), (2, 3), (4, 5), (6, 7)
#pragma unroll
    for (int i = 0; i < 4; ++i) d[i] = pack_f16(v[2 * i], v[2 * i + 1]);
    // kg = 0, 1 go to the lane with column bit 4 clear, kg = 2, 3 to the other
    const uint32_t g0 = dpp_word<0x4E>(hi ? d[0] : d[2]), g1 = dpp_word<0x4E>(hi ? d[1] : d[3]);
    const uint32_t l0 = hi ? g0 : d[0], l1 = hi ? g1 : d[1], h0 = hi ? d[2] : g0, h1 = hi ? d[3] : g1;      // of the lower, of the upper 16 columns
    const uint32_t p0 = __builtin_amdgcn_perm(h0, l0, 0x05040100u), p1 = __builtin_amdgcn_perm(h0, l0, 0x07060302u);   // first kg: pairs of j = 0, 1
    const uint32_t p2 = __builtin_amdgcn_perm(h1, l1, 0x05040100u), p3 = __builtin_amdgcn_perm(h1, l1, 0x07060302u);   // second kg
    // the first kg goes to the lane with column bit 3 clear, the second to the other; its own columns' bit 3 orders the halves
    const uint32_t q0 = dpp_word<0xB1>(up ? p0 : p2), q1 = dpp_word<0xB1>(up ? p1 : p3);
    return up ? make_uint4(q0, q1, p2, p3) : make_uint4(p0, p1, q0, q1);
}

// LDS position (in halfs) of column c of a 128-column chunk in the B-operand order:
// 16-byte block (mm, kg) holds, for i = 0..3, columns 32 mm + 2 kg + 8 (i >> 1) + (i & 1) and that + 16
__device__ __forceinline__ int bop_index(int c)
{
    const int mm = c >> 5, hi = (c >> 4) & 1, kg = (c >> 1) & 3, i = 2 * ((c >> 3) & 1) + (c & 1);
    return (mm * 4 + kg) * 8 + 2 * i + hi;
}

// A operand of MFMA (MM, RHO): rows g + 8 RHO, columns of t = 2 MM and 2 MM + 1
template <bool RES, int CODE, int MM, int RHO, int BK = 0, bool RAW = false>
__device__ __forceinline__ half8_t a_operand(const uint32_t* wb, const uint32_t* wr, const FoldK& k)
{
    constexpr int J = 16 * MM + 2 * RHO;
    uint32_t u[4];
    weight_pairs2<RES, CODE, J + 0, J + 1, BK, RAW>(wb, wr, k, u[0], u[1]);
    weight_pairs2<RES, CODE, J + 4, J + 5, BK, RAW>(wb, wr, k, u[2], u[3]);
    return __builtin_bit_cast(half8_t, *(u32x4*)u);
}

// Wavefront priority by progress through the k-slice. The SIMD's arbiter picks the highest user priority and, among equals,
// the oldest wavefront, so of the co-resident wavefronts (one per workgroup, all with the same amount of work) the oldest
// would finish far ahead of the youngest, and the SIMD would spend the end of the launch with one or two wavefronts, which
// cannot keep the vector ALU busy. Lowering a wavefront's priority as it nears its end lets the others catch up, so that
// they finish together; a wavefront of lower priority still issues whenever the others wait.
// Measured (decode layer, B = 1): gate|up launch 48.2 -> 44.2 us with k-slices of 12 chunks; the down launch gains with
// k-slices of 8 chunks (31.8 -> 29.8 us) and loses with 4, where the steps are too coarse, so short slices keep one priority.
// The thresholds (a half, a quarter, an eighth of the slice left) were the best of six sets tried.
__device__ __forceinline__ void progress_priority(int c, int NC)
{
    if (NC < 8) return;
    const int left = 8 * (NC - c);                               // eighths of chunks left, this chunk included
    if (left > 4 * NC) __builtin_amdgcn_s_setprio(3);
    else if (left > 2 * NC) __builtin_amdgcn_s_setprio(2);
    else if (left > NC) __builtin_amdgcn_s_setprio(1);
    else __builtin_amdgcn_s_setprio(0);
}

struct LaneCtx
{
    uint32_t rec0;        // record index of this lane in chunk 0 of its k-slice: (unit0) * 32 + 4 g + t4
    uint32_t unit0;       // unit index (strip * C + chunk0)
    size_t nrec;          // records of the whole projection (sub-array stride)
    int src;              // lane holding the next record of the ring
    int g;                // ring index (sign-variant bit)
    const char* xs;       // this lane's B-operand base in LDS (bytes), kg folded in
    int xstep;            // bytes per chunk (0 for lanes without a token)
    uint32_t strip; size_t nstrips; int chunk0;   // mask mode: this lane's strip, strips of the projection, first chunk of the k-slice
    uint32_t half0;       // unit index of strip lane / 32 of the wavefront's two, first chunk (UnitConsts)
};

// Block word and sign byte of chunk c + lane % 32 (the last one's beyond it) of strip lane / 32 of the wavefront's two; res: the level has block words
struct UnitWords { uint32_t word, var; };
__device__ __forceinline__ UnitWords unit_words(const Planes& P, const LaneCtx& L, int c, int NC, bool res)
{
    const uint32_t unit = L.half0 + (uint32_t)min(c + (int)(threadIdx.x & 31), NC - 1);
    UnitWords w = {0u, 0u};
    if (res) w.word = at_offset<uint32_t>((gp_u8)P.dw, unit * 4u);
    if (P.var) w.var = at_offset<uint8_t>(P.var, unit);
    return w;
}

// What a chunk's decode needs beside the records, fold constants and ring signs, for 32 chunks of the wavefront's two strips at a time: lane 32 s + i
// reads the block word and sign byte of strip s, chunk c0 + i, and works out its constants; a chunk's come from there by one
// lane permute (two at levels 3 / 4). Worked out by every lane in every chunk they were some 25 of the 600 vector instructions of a refined chunk
// and, with no sign plane, 5 of the 275 of a chunk at level 2, beside one or two loads. A tile of the grouped GEMMs has all chunks of its projection
// (48 of gate|up at 6144 columns), a slice of a decode call at most 24 of gate|up and 4 of down; slices of one: gemv_chunks' FEW. us anew in every chunk /
// as now: 4 tokens of 6144 x 2048 204 / 199, all at level 4 305 / 286, one token 61.1 / 60.5; a lone gate|up projection of 8 tokens at level 3 13.65 / 13.37;
// 48 and 201 tokens, with the scalar token addresses, 1157 / 1136 and 1340 / 1313.
template <bool RES>
struct UnitConsts
{
    uint32_t word, ac, next_word, next_var;       // block word | sign byte << 16; fold_ac of it; as loaded, 32 chunks on
    int from;                                     // 4 * the lane that holds this lane's strip, chunk 0
    FoldK k;
    __device__ __forceinline__ void start(const UnitWords& first)
    {
        word = ac = 0u; next_word = first.word; next_var = first.var;
        from = (int)(threadIdx.x & 8u) << 4;
        k = consts_l2(0u);
    }
    // at chunk c's beginning. gemv_chunks has it ahead of the next chunk's requests: behind them, with a branch in between, the wait for the block words
    // was one for those requests too. In pf_chunks, whose chunks take ten times as long, it is behind them. The reciprocal is divided out (IEEE, the table's bits): its entry would be another latency before a slice's first product.
    __device__ __forceinline__ void begin(const Planes& P, const LaneCtx& L, int c, int NC)
    {
        if ((RES || P.var) && (c & 31) == 0)
        {
            const uint32_t Mb = next_word & 0xFFu;
            if constexpr (RES) ac = fold_ac(next_word, Mb ? 1.0f / (float)Mb : 0.f);
            word = (next_word & 0xFFFFu) | next_var << 16;
            const UnitWords next = unit_words(P, L, c + 32, NC, RES);      // the last chunk's once more, where there are none: no branch
            next_word = next.word; next_var = next.var;
        }
    }
    // the constants of chunk c, in k
    __device__ __forceinline__ void take(const Planes& P, const LaneCtx& L, int c)
    {
        const int lane = from + 4 * (c & 31);
        if constexpr (RES) k = fold_k((uint32_t)__builtin_amdgcn_ds_bpermute(lane, (int)word), (uint32_t)__builtin_amdgcn_ds_bpermute(lane, (int)ac), 0u);
        if (P.var)
        {
            uint32_t sgm = (((uint32_t)__builtin_amdgcn_ds_bpermute(lane, (int)word) >> (16 + L.g)) & 1u) * 0x80008000u;
            asm volatile("" : "+v"(sgm));                        // a branch, not a selection that every chunk pays for
            k.A2 = (RES ? k.A2 : MUL1_A2) ^ sgm; k.C2 = (RES ? k.C2 : MUL1_B2) ^ sgm;
        }
    }
};

// mask mode: chunk by chunk either the folded decode (refined chunks, residual records compact over them) or the level-2
// decode; the choice is the same for every lane of the workgroup. Residual records are fetched when needed (no prefetch).
template <int CODE, int BK>
__device__ __forceinline__ void gemv_chunks_masked(const Planes& P, const LaneCtx& L, int NC, float4_t* acc, u32x4 nb)
{
    constexpr int NW = Rec<CODE>::NW;
    const uint64_t f = P.flags[L.strip];
    uint32_t nvar = P.var ? at_offset<uint8_t>(P.var, L.unit0) : 0u;
    for (int c = 0; c < NC; ++c)
    {
        progress_priority(c, NC);
        uint32_t wb[6], wr[NW + 2] = {0};
        wb[0] = nb.x; wb[1] = nb.y; wb[2] = nb.z; wb[3] = nb.w;
        const uint32_t var = nvar;
        const MaskedUnit m = masked_unit(f, L.strip, L.chunk0 + c, L.nstrips);
        const bool on = __builtin_amdgcn_readfirstlane((int)m.on) != 0;
        uint32_t dw = 0;
        if (on) { load_record<CODE>(wr, P.res, m.unit * 32 + (L.rec0 & 31), m.nrec); dw = P.dw[m.unit]; }
        if (c + 1 < NC)
        {
            nb = load_base<BK>(P, L.rec0 + (uint32_t)(c + 1) * 32, L.nrec);
            if (P.var) nvar = at_offset<uint8_t>(P.var, L.unit0 + c + 1);
        }
        ext_base<BK>(wb, __shfl(wb[0], L.src));
        const uint32_t sgm = ((var >> L.g) & 1u) * 0x80008000u;
        const char* xp = L.xs + c * L.xstep;
        if (on)
        {
            prepare_record<CODE>(wr);
            ext_words<Rec<CODE>::BITS, Rec<CODE>::NW>(wr, __shfl(wr[0], L.src));
            const FoldK k = consts_fold(dw, sgm);
            static_for<4>([&](auto mm) {
                constexpr int MM = decltype(mm)::value;
                const half8_t b = *(const half8_t*)(xp + MM * 64);
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_operand<true, CODE, MM, 0, BK>(wb, wr, k), b, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_operand<true, CODE, MM, 1, BK>(wb, wr, k), b, acc[1], 0, 0, 0);
            });
        }
        else
        {
            const FoldK k = consts_l2(sgm);
            static_for<4>([&](auto mm) {
                constexpr int MM = decltype(mm)::value;
                const half8_t b = *(const half8_t*)(xp + MM * 64);
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_operand<false, 0, MM, 0, BK>(wb, wr, k), b, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_operand<false, 0, MM, 1, BK>(wb, wr, k), b, acc[1], 0, 0, 0);
            });
        }
    }
}

// MASKOK = false leaves the mask-mode loop out (the caller has made sure that P.flags is null)
// RAW (level 2 without a sign plane only: one affine map for the whole plane): the MFMAs multiply the integers 1024 + S, exact in
// fp16, and the value map w = A (1024 + S) + B is applied once to the sums: sum_k w_k x_k = A sum_k (1024 + S_k) x_k + B sum_k x_k,
// with sum_k x_k from one more MFMA per operand against a row of ones. That removes the packed FMA of every weight pair (32 of the
// loop's ~276 vector instructions per chunk) and, with it, the rounding of each weight to fp16: the result is that of the
// UNROUNDED weights, ~2e-4 (relative, l2) from the product with the exact fp16 weights that the other form and the reference
// compute -- inside the layer's 1e-3, outside the 5e-5 that the exact form holds, hence an option the caller has to ask for.
// FEW: every lane works out its own unit's constants chunk by chunk instead. In a slice of one chunk there is nothing for UnitConsts to share, and its
// permutes and its work at the slice's beginning are latency: a layer of 512 x 256, two tokens, 14.1 us / 14.3 with them. Which call takes which: launch_moe.
template <bool RES, int CODE, int BK = 0, bool MASKOK = true, bool RAW = false, bool FEW = false>
__device__ __forceinline__ void gemv_chunks(const Planes& P, const LaneCtx& L, int NC, float4_t* acc, u32x4 nb)
{
    static_assert(!RAW || BK == 0, "the hoisted value map is built for base window code 0");
    float4_t accx = {0.f, 0.f, 0.f, 0.f};
    // RAW at levels 3 / 4: the value map differs from unit to unit, w = A'_u (1024 + F) + C_u, so it is applied chunk by chunk: the
    // chunk's integer products go to accumulators of their own (zero at the chunk's start) and enter the running sums times A'_u;
    // C_u sum_k x_k comes from two more MFMAs per operand whose A operand is C_u in every place (the rows a lane decodes and the
    // rows it supplies to the MFMA are the same, so its own unit's C_u is the right one). The accumulator rows a lane HOLDS belong
    // to the strip (lane >> 5), whose A' it fetches from a lane that decodes that strip.
    const int lane_of_out_strip = (int)((threadIdx.x & 0x37u) | ((threadIdx.x >> 2) & 8u));
    const half8_t ones = {(_Float16)1, (_Float16)1, (_Float16)1, (_Float16)1, (_Float16)1, (_Float16)1, (_Float16)1, (_Float16)1};
    if constexpr (RES && MASKOK)
        if (P.flags) { gemv_chunks_masked<CODE, BK>(P, L, NC, acc, nb); return; }     // block-uniform
    constexpr int NW = RES ? Rec<CODE>::NW : 1;
    uint32_t nr[NW + 2] = {0}, ndw = 0, nvar = 0;
    UnitConsts<RES> consts;
    if constexpr (!FEW) consts.start(unit_words(P, L, 0, NC, RES));              // before the records: they are waited for first
    if constexpr (RES) load_record<CODE>(nr, P.res, L.rec0, L.nrec);
    auto own_words = [&](int c) {                                // FEW
        if constexpr (RES) ndw = at_offset<uint32_t>((gp_u8)P.dw, (L.unit0 + c) * 4u);
        if (P.var) nvar = at_offset<uint8_t>(P.var, L.unit0 + c);
    };
    if constexpr (FEW) own_words(0);
    for (int c = 0; c < NC; ++c)
    {
        progress_priority(c, NC);
        uint32_t wb[6], wr[NW + 2];
        wb[0] = nb.x; wb[1] = nb.y; wb[2] = nb.z; wb[3] = nb.w;
#pragma unroll
        for (int i = 0; i < NW; ++i) wr[i] = nr[i];
        const uint32_t dw = ndw, sgm = ((nvar >> L.g) & 1u) * 0x80008000u;
        if constexpr (!FEW) consts.begin(P, L, c, NC);
        if (c + 1 < NC)                                         // prefetch the next chunk's records
        {
            nb = load_base<BK>(P, L.rec0 + (uint32_t)(c + 1) * 32, L.nrec);
            if constexpr (RES) load_record<CODE>(nr, P.res, L.rec0 + (uint32_t)(c + 1) * 32, L.nrec);
            if constexpr (FEW) own_words(c + 1);
        }
        ext_base<BK>(wb, __shfl(wb[0], L.src));
        if constexpr (RES)
        {
            prepare_record<CODE>(wr);
            ext_words<Rec<CODE>::BITS, Rec<CODE>::NW>(wr, __shfl(wr[0], L.src));
        }
        if constexpr (!FEW) consts.take(P, L, c);
        else consts.k = RES ? consts_fold(dw, sgm) : consts_l2(sgm);
        const FoldK& k = consts.k;
        const char* xp = L.xs + c * L.xstep;
        if constexpr (RAW && RES)
        {
            float4_t c0 = {0.f, 0.f, 0.f, 0.f}, c1 = {0.f, 0.f, 0.f, 0.f};
            const u32x4 cu = {k.C2, k.C2, k.C2, k.C2};
            const half8_t cop = __builtin_bit_cast(half8_t, cu);
            static_for<4>([&](auto mm) {
                constexpr int MM = decltype(mm)::value;
                const half8_t b = *(const half8_t*)(xp + MM * 64);
                c0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_operand<RES, CODE, MM, 0, BK, true>(wb, wr, k), b, c0, 0, 0, 0);
                c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_operand<RES, CODE, MM, 1, BK, true>(wb, wr, k), b, c1, 0, 0, 0);
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(cop, b, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(cop, b, acc[1], 0, 0, 0);
            });
            const float Amine = (float)__builtin_bit_cast(_Float16, (uint16_t)(k.A2 & 0xFFFFu));
            const float Aout = __shfl(Amine, lane_of_out_strip);
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                acc[0][i] = __builtin_fmaf(Aout, c0[i], acc[0][i]);
                acc[1][i] = __builtin_fmaf(Aout, c1[i], acc[1][i]);
            }
        }
        else
            static_for<4>([&](auto mm) {
                constexpr int MM = decltype(mm)::value;
                const half8_t b = *(const half8_t*)(xp + MM * 64);
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_operand<RES, CODE, MM, 0, BK, RAW>(wb, wr, k), b, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_operand<RES, CODE, MM, 1, BK, RAW>(wb, wr, k), b, acc[1], 0, 0, 0);
                if constexpr (RAW) accx = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, b, accx, 0, 0, 0);
            });
    }
    if constexpr (RAW && !RES)
    {   // every row of accx holds the token's sum of x over the k-slice; A and B as the fp32 values of the fp16 constants
        const float A = 0.00676727294921875f /* fp16 0x1eee = 1774 / 2^18 */, B = -10.3828125f /* fp16 0xc931 */;
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            acc[0][i] = __builtin_fmaf(A, acc[0][i], B * accx[i]);
            acc[1][i] = __builtin_fmaf(A, acc[1][i], B * accx[i]);
        }
    }
}


}  // namespace nq
