// Prefill: the grouped expert GEMM over a route table, on the matrix cores, and the SwiGLU quantizer between
// a gate/up pair and its down (crates/gpu/src/gemm/mod.rs:1-50).
//
// The route table is the reference's (crates/gpu/src/gemm/route.rs:1-60,109-125): `cols` lists the slots grouped by
// expert, ascending slot order inside an expert, the refused slots (an id past the stack) at its end; `tiles` holds
// a pair of words a tile, (expert, first index | length << 16), tiles of at most 64 slots; `n_tiles` = {tile count,
// refused count}.
//
// The GEMM's numbers are the decode path's, bit for bit: every (row, slot) value is the one-column row dot of
// bm_device.hpp. The integer sums of each 16-value group come out of the matrix cores exactly, and each enters the f32 accumulator
// of the CPU path's lane that owns it, in the CPU path's order (crates/qdot/src/lib.rs:4363-4447 Q4_K, :4776-4874 Q6_K): eight accumulators a
// value, the min term first, then the groups in increasing k, and the closing sum (t0 + t2) + (t1 + t3).
#include <algorithm>
#include <type_traits>

#include "bm_gemm.hpp"

namespace bmk {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kRouteThreads = 1024;

int gemm_max_tiles(int n_slots, int n_experts) { // crates/gpu/src/gemm/route.rs:55-57
    return n_slots / kGemmBN + (n_experts < n_slots ? n_experts : n_slots);
}

// ------------------------------------------------------------------------------------------------ route

// The slots listed by expert in ascending slot order, bucket n_experts collecting the refused ones at the list's end
// (group_slots_part: as many workgroups as the list has parts, each placing its part; one workgroup on a single compute
// unit took 23 us over 16384 slots, bound by that unit's instruction rate and by lanes queueing on a popular expert's
// counter); one workgroup more places nothing and writes the tiles, an expert's run cut into runs of at most 64. A slot served elsewhere (id 0xffffffff, crates/gpu/src/kquant/sel.rs:22-28) is not
// listed and raises nothing: the list is that many entries shorter, the entries past it hold 0xffffffff, and n_tiles[2]
// counts them.
struct RouteLds {
    GroupLds g;
    u32 off[kGroupBuckets];
};
// With `x`: behind the table's workgroups (route_blocks of them) further ones quantize m rows of k f32 values into `act`,
// the column form picked by q8k (Q8_K: a wave a 256-value block; Q8_2_X4: eight values a thread): the prefill step's two
// first launches, which depend on nothing of each other, as one.
__global__ __launch_bounds__(kRouteThreads) void k_route(const u32 *ids, u32 n_slots, u32 n_experts, u32 *cols,
                                                         u32 *tiles, u32 *n_tiles, u32 route_blocks, const float *x, int m, int k,
                                                         int q8k, uint8_t *act, u32 *fault, u32 layer) {
    if (blockIdx.x >= route_blocks) {
        const u32 qb = blockIdx.x - route_blocks;
        if (q8k) {
            const int b = (int)qb * 16 + (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
            if (b >= m * (k / 256)) return; // whole waves leave
            q8k_wave_block(*reinterpret_cast<const float4 *>(x + (size_t)b * 256 + 4 * lane), act + (size_t)b * BM_Q8K_STRIDE, lane, fault, layer);
        } else {
            const u32 i = qb * kRouteThreads + threadIdx.x, line = (u32)k / 8u;
            if (i >= (u32)m * line) return; // whole quads leave: a block is 32 values, k a multiple of 256
            const int col = (int)(i / line), o = 8 * (int)(i % line);
            const size_t at = (size_t)i * 8;
            const float4 a = *reinterpret_cast<const float4 *>(x + at), b = *reinterpret_cast<const float4 *>(x + at + 4);
            const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
            q82_quad8(v, act + (size_t)col * (k / 256) * BM_Q82_SB_EXT, k / 256, o >> 5, threadIdx.x & 3, fault, layer);
        }
        return;
    }
    __shared__ RouteLds lds;
    GroupLds &g = lds.g;
    const u32 tid = threadIdx.x;
    group_slots_part(g, lds.off, n_slots, n_experts + 1, blockIdx.x, cols, [&](u32 s) {
        const u32 id = ids[s];
        return id < n_experts ? id : id == 0xffffffffu ? kNoBucket : n_experts;
    });
    if (blockIdx.x + 1 != route_blocks) return;
    const u32 listed = g.base[n_experts + 1];
    for (u32 i = listed + tid; i < n_slots; i += kRouteThreads) cols[i] = 0xffffffffu;
    u32 j0 = 0, j1 = 0;
    if (tid < n_experts) {
        j0 = g.base[tid];
        j1 = g.base[tid + 1];
    }
    u32 total;
    u32 t = block_scan_1024((j1 - j0 + kGemmBN - 1) / kGemmBN, g.scan, &total);
    for (u32 j = j0; j < j1; j += kGemmBN, t++) {
        const u32 len = j1 - j < (u32)kGemmBN ? j1 - j : (u32)kGemmBN;
        tiles[2 * t] = tid;
        tiles[2 * t + 1] = j | (len << 16);
    }
    if (tid == 0) {
        const u32 refused = g.base[n_experts + 1] - g.base[n_experts];
        if (refused) bm_raise(fault, layer, kSiteExpertId);
        n_tiles[0] = total;
        n_tiles[1] = refused;
        n_tiles[2] = n_slots - listed;
    }
}

hipError_t route(const Launch &L, const uint32_t *ids, int n_slots, int n_experts, uint32_t *cols, uint32_t *tiles_out,
                 uint32_t *n_tiles, int wtype, const float *x, int m, int k, uint8_t *act) {
    const u32 route_blocks = group_parts((u32)n_slots, (u32)n_experts + 1) + 1;
    u32 quant_blocks = 0;
    const bool q8k = x && bm_takes_q8k(wtype);
    if (x) {
        if (k % 256 != 0 || (reinterpret_cast<uintptr_t>(x) & 15) != 0) return hipErrorInvalidValue;
        quant_blocks = q8k ? (u32)((m * (k / 256) + 15) / 16) : (u32)(((long)m * k + 8 * kRouteThreads - 1) / (8 * kRouteThreads));
    }
    hipLaunchKernelGGL(k_route, dim3(route_blocks + quant_blocks), dim3(kRouteThreads), 0, L.stream, ids, (u32)n_slots, (u32)n_experts,
                       cols, tiles_out, n_tiles, route_blocks, x, m, k, q8k ? 1 : 0, act, L.fault, L.layer);
    return hipGetLastError();
}

// --------------------------------------------------------------------------------------- SwiGLU + quantize

// crates/gpu/src/gemm/swiglu.rs:46-58 in the CPU path's rules: column c of act = Q8_2_X4(swiglu(g, u)) over the k
// values g[c * k ..], u[c * k ..]. One half wave a 32-value block.
// `sel` (optional; crates/gpu/src/gemm/swiglu.rs:96-140 enqueue_swiglu_act_quant_sel): column c belongs to slot c; a slot
// served elsewhere (id 0xffffffff) keeps its column as it stands and raises nothing, any other id at or past n_experts
// raises ExpertId with nothing stored.
__device__ __forceinline__ bool swiglu_column_skipped(const u32 *sel, u32 n_experts, int col, bool first, u32 *fault, u32 layer) {
    if (!sel) return false;
    const u32 id = sel[col];
    if (id < n_experts) return false;
    if (id != 0xffffffffu && first) bm_raise(fault, layer, kSiteExpertId);
    return true;
}

__global__ __launch_bounds__(256) void k_swiglu_quant(const float *g, const float *u, int m, int k, uint8_t *act,
                                                      GateRule rule, const u32 *sel, u32 n_experts, u32 *fault, u32 layer) {
    const u32 bpc = (u32)k / 32u, gblk = blockIdx.x * 8u + (threadIdx.x >> 5);
    if (gblk >= (u32)m * bpc) return;
    const int col = (int)(gblk / bpc), blk = (int)(gblk % bpc), lane32 = threadIdx.x & 31;
    if (swiglu_column_skipped(sel, n_experts, col, blk == 0 && lane32 == 0, fault, layer)) return; // uniform over the half wave
    const size_t at = (size_t)gblk * 32 + lane32;
    bool odd;
    const float v = bm_gate_rule(rule.act, rule.limit, g[at], u[at], odd);
    if (odd) bm_raise(fault, layer, kSiteF32Product);
    Q82Head hd;
    int s16;
    const int code = q82_block(v, &hd, &s16);
    if (hd.bad && lane32 == 0) bm_raise(fault, layer, kSiteQuantColumn);
    q82_store(act + (size_t)col * (k / 256) * BM_Q82_SB_EXT, k / 256, blk, lane32, code, hd, s16);
}

// The same into Q8_K columns, for a down stack that dots against those (IQ2_XXS, ...): a wave a 256-value block, four values a lane.
// (A workgroup a block, a value a thread, spent its time in two barriers and sixteen-step sums: 25.4 -> 11.2 us at 6216 columns of 768 values, 83 -> 31 us at 8192 of 2048.)
__global__ __launch_bounds__(256) void k_swiglu_quant_q8k(const float *g, const float *u, int m, int k, uint8_t *act,
                                                          GateRule rule, const u32 *sel, u32 n_experts, u32 *fault, u32 layer) {
    const u32 bpc = (u32)k / 256u, gblk = blockIdx.x * 4u + (u32)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (gblk >= (u32)m * bpc) return;
    const u32 col = gblk / bpc, blk = gblk % bpc, lane = threadIdx.x & 63;
    if (swiglu_column_skipped(sel, n_experts, (int)col, blk == 0 && lane == 0, fault, layer)) return; // uniform over the wave
    const size_t at = (size_t)gblk * 256 + 4 * lane;
    const float4 g4 = bm_ld4f(g + at), u4 = bm_ld4f(u + at);
    const float gv[4] = {g4.x, g4.y, g4.z, g4.w}, uv[4] = {u4.x, u4.y, u4.z, u4.w};
    float v[4];
    bool any_odd = false;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        bool odd;
        v[i] = bm_gate_rule(rule.act, rule.limit, gv[i], uv[i], odd);
        any_odd |= odd;
    }
    if (any_odd) bm_raise(fault, layer, kSiteF32Product);
    q8k_wave_block(make_float4(v[0], v[1], v[2], v[3]), act + (size_t)gblk * BM_Q8K_STRIDE, (int)lane, fault, layer);
}

// The Q8_2_X4 form with eight values a thread, a block a quad of lanes: two 16-byte loads of each input a thread.
__global__ __launch_bounds__(256) void k_swiglu_quant_wide(const float *g, const float *u, int m, int k, uint8_t *act,
                                                           GateRule rule, const u32 *sel, u32 n_experts, u32 *fault, u32 layer) {
    // (thread numbers fit 32 bits, as a grid's threads do; a division of 64 bits takes some hundred and fifty instructions)
    const u32 i = blockIdx.x * 256u + threadIdx.x, line = (u32)k / 8u;
    if (i >= (u32)m * line) return;
    const int col = (int)(i / line), o = 8 * (int)(i % line);
    const size_t at = (size_t)i * 8;
    if (swiglu_column_skipped(sel, n_experts, col, o == 0, fault, layer)) return; // uniform over a block's quad of lanes
    const float4 g0 = *reinterpret_cast<const float4 *>(g + at), g1 = *reinterpret_cast<const float4 *>(g + at + 4);
    const float4 u0 = *reinterpret_cast<const float4 *>(u + at), u1 = *reinterpret_cast<const float4 *>(u + at + 4);
    const float gv[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
    const float uv[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
    float v[8];
    bool any_odd = false;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        bool odd;
        v[j] = bm_gate_rule(rule.act, rule.limit, gv[j], uv[j], odd);
        any_odd |= odd;
    }
    if (any_odd) bm_raise(fault, layer, kSiteF32Product);
    q82_quad8(v, act + (size_t)col * (k / 256) * BM_Q82_SB_EXT, k / 256, o >> 5, threadIdx.x & 3, fault, layer);
}

hipError_t swiglu_quant(const Launch &L, const float *g, const float *u, int m, int k, uint8_t *act, bool q8k, const uint32_t *sel,
                        uint32_t n_experts) {
    if (!q8k && (((uintptr_t)g | (uintptr_t)u) & 15) == 0) {
        const long threads = (long)m * k / 8;
        hipLaunchKernelGGL(k_swiglu_quant_wide, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, L.stream, g, u, m, k, act,
                           L.rule, sel, n_experts, L.fault, L.layer);
        return hipGetLastError();
    }
    if (q8k) {
        hipLaunchKernelGGL(k_swiglu_quant_q8k, dim3(((unsigned)m * (unsigned)(k / 256) + 3) / 4), dim3(256), 0, L.stream, g, u, m, k, act, L.rule,
                           sel, n_experts, L.fault, L.layer);
        return hipGetLastError();
    }
    const long blocks = (long)m * (k / 32);
    hipLaunchKernelGGL(k_swiglu_quant, dim3((unsigned)((blocks + 7) / 8)), dim3(256), 0, L.stream, g, u, m, k, act,
                       L.rule, sel, n_experts, L.fault, L.layer);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------- GEMM

// (q6 - 32) of four codes a word, as signed bytes: q6 in 0..63.
__device__ __forceinline__ u32 q6_minus_32(u32 q) {
    const u32 t = q ^ 0x20202020u;        // q >= 32: q - 32; q < 32: q + 32
    const u32 m = ~q & 0x20202020u;       // the bytes that went up: they want -64, the two top bits
    return t | (m << 1) | (m << 2);
}

// The exact form's LDS, half a super-block (128 values) at a time, twice: the slab's 64 weight rows and the tile's 64 columns as
// f16 codes, 264 bytes a row (8 x an odd number: sixteen lanes of a wave read sixteen rows at one place, eight bytes each, from
// sixteen different bank pairs), and the f32 factors, a line of 64 rows (or slots) each.
constexpr int kXStride = 2 * 128 + 8;
constexpr int kXCodes = 64 * kXStride; // rows of half 0, rows of half 1, columns of half 0, columns of half 1, the factors
constexpr int kXLine = 80 * 4;         // bytes: the staging's sixteen rows of four lines land on different banks
template <int WT>
struct XLds {
    static constexpr bool kMins = WT != BM_Q6K;
    static constexpr int kScales = kMins ? 4 : 8;           // lines of scale products a half
    static constexpr int kHalf = (kScales + 4) * kXLine;    // a half's factors: the scale products, and four lines of d8
    static constexpr int kMinsAt = 2 * kHalf;               // and a super-block's: eight lines of mins, eight of d8 isum
    static constexpr int kHeadsAt = kMinsAt + (kMins ? 16 * kXLine : 0); // a word a staging thread: the heads of its blocks, or-ed
    static constexpr int kFactors = kHeadsAt + (kMins ? 4 * kXLine : 0);
    static constexpr size_t kBytes = 4 * (size_t)kXCodes + kFactors + sizeof(GemmLds);
};

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef u32 v2u __attribute__((ext_vector_type(2)));
typedef u32 v4u __attribute__((ext_vector_type(4)));

// Two small integers given as f16 bit patterns 1024 + n, less `bias`: exact.
__device__ __forceinline__ u32 h2_less(u32 x, float bias) {
    const _Float16 b = (_Float16)bias;
    return __builtin_bit_cast(u32, __builtin_bit_cast(v2h, x) - (v2h){b, b});
}
// The same of 1024 + 16 n: n - off.
__device__ __forceinline__ u32 h2_16th(u32 x, float off) {
    const _Float16 s = (_Float16)0.0625f, b = (_Float16)(-64.0f - off);
    return __builtin_bit_cast(u32, __builtin_elementwise_fma(__builtin_bit_cast(v2h, x), (v2h){s, s}, (v2h){b, b}));
}

// (x & mask) | bits in one instruction; from the plain expression the compiler makes two or three.
__device__ __forceinline__ u32 and_or(u32 x, u32 mask, u32 bits) {
    u32 r;
    __asm__("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(mask), "v"(bits));
    return r;
}

// One value of a Q4_K or Q5_K row against a column as a plain walk: see k_gemm.
template <int WT>
__device__ __forceinline__ float q45_value(const uint8_t *row, const uint8_t *col, int nb) {
    float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma nounroll
    for (int i = 0; i < nb; i++) {
        const uint8_t *blk = row + (size_t)i * bm_block_bytes<WT>(), *sc = blk + 4, *codes = blk + (WT == BM_Q5K ? 48 : 16);
        const float *pair = reinterpret_cast<const float *>(col + (size_t)nb * BM_Q82_SB_REF + 64 * (size_t)i); // d8, d8 isum of a block
        const float d = bm_half_to_f32((unsigned short)bm_ld2u(blk)), dmin = bm_half_to_f32((unsigned short)bm_ld2u(blk + 2));
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const int m = b < 4 ? sc[b + 4] & 63 : (sc[b + 4] >> 4) | ((sc[b] >> 6) << 4);
            acc[b] = fmaf(pair[2 * b + 1], -(dmin * (float)m), acc[b]);
        }
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const int s = b < 4 ? sc[b] & 63 : (sc[b + 4] & 15) | ((sc[b - 4] >> 6) << 4);
            const float scale = d * (float)s * pair[2 * b];
            const int8_t *a = reinterpret_cast<const int8_t *>(col + (size_t)(2 * i + (b >> 2)) * BM_Q82X4_STRIDE + 16 + 32 * (b & 3));
#pragma unroll
            for (int h = 0; h < 2; h++) {
                int sum = 0;
#pragma nounroll
                for (int n = 16 * h; n < 16 * h + 16; n++) {
                    const int low = (codes[32 * (b >> 1) + n] >> (4 * (b & 1))) & 15;
                    sum += (WT == BM_Q5K ? low | (((blk[16 + n] >> b) & 1) << 4) : low) * a[n];
                }
                acc[4 * h + (b & 3)] = fmaf(scale, (float)sum, acc[4 * h + (b & 3)]);
            }
        }
    }
    return ((acc[0] + acc[4]) + (acc[2] + acc[6])) + ((acc[1] + acc[5]) + (acc[3] + acc[7]));
}

// A workgroup of four waves takes a slab of 64 rows and a tile's 64 slots, a wave 32 x 32 of them. Of a tile of at most 32 slots, which
// is most tiles of a short prompt, a wave takes 32 rows and all the slots but four of the eight accumulators, i.e. every second
// group (Q4_K: group h of a block goes to accumulators 4 h ..), and the two waves of a row group meet in the closing sum: with the
// wide split two waves of such a workgroup had no slots, and the two SIMDs with the others did all the arithmetic (top-8 of 128 experts, Q4_K /
// Q6_K, us a layer: 256 tokens 251 -> 223, 333 tokens 269 -> 241, 1024 tokens 464 -> 433).
// Per (row, slot, 16-value group) the contract is acc[l] = fma(fl(scale d8), sum, acc[l]) over eight accumulators, one fused
// multiply-add that only the vector ALU can do. The rest is on the matrix cores: the group's integer sum comes out of
// v_mfma_f32_32x32x16_f16 as a float (codes of at most eight bits, sums below 2^24: exact, where an int8 product needs a
// conversion a sum), fl(scale d8) over the tile is the outer product v_mfma_f32_32x32x1_2b_f32 (two blocks, or Q6_K's two
// groups, an instruction; a product plus zero is the product's rounding), and a min term fma(d8 isum, min, acc) is the same
// instruction with the accumulators as its addend. (Subnormal factors and products come out as fmaf gives them. The added zero
// is +0, so a product of -0, which takes a scale of -0, comes out as +0; that shows where all eight accumulators of a value are
// zeros, one of them a -0 that a min term has underflowed to: the value's sign. A super-block's d with its sign bit set is
// what it takes, so a workgroup that has staged one, which no quantizer makes, walks its values of zero again by themselves.
// Q6_K, without mins, never has an accumulator of -0.)
// Bound by the vector ALU (the f32 matrix instructions run on it too, 64 cycles each; the f16 ones beside it) as far as two waves a
// SIMD fill it: gate and up of 16384 slots Q4_K take 756 k cycles, of which vector instructions are 62 % (32 multiply-adds a wave and
// 32 x 32 x 32 values, about 30 instructions of staging, addresses) and outer products 14 %; a wave waits a fifth of its time. Down in
// Q6_K: 514 k, 57 % and 10 %, a quarter. The clock is 2.05 GHz under it, what the card's power leaves: a fifth of the vector
// instructions less (the columns as f16 brought to LDS directly) took the same time. The staging of a half (bytes to f16, the factors) is cut
// in eight pieces between the groups of the half before it, each behind the group's matrix instruction, and its codes are asked for seven
// pieces before their use: one barrier a half. 80 KB: two workgroups a CU. 16384 slots of 128 experts, 768 rows of 2048 values
// Q4_K and Q6_K down, a layer: 1459 us with int8 products and the scaling, the conversion and the mins on the vector ALU, 725 with the
// products and scales on the matrix cores, 668 with the waits where they are now and more rows a workgroup.
template <int WT>
__global__ __launch_bounds__(256, 2) void k_gemm(const uint8_t *w, int rpe, int nb, const uint8_t *act, const u32 *cols,
                                                 const u32 *tiles, const u32 *n_tiles, u32 n_units, u32 slot_div,
                                                 u32 n_slots, float *y, u32 slabs, const uint8_t *w_second, float *y_second) {
    using X = XLds<WT>;
    extern __shared__ __align__(16) uint8_t lds[];
    GemmLds *tab = reinterpret_cast<GemmLds *>(lds + 4 * kXCodes + X::kFactors);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const u32 g = tile_of_block(blockIdx.x, n_units);
    // the first of the slabs the workgroup takes one after the other
    int row0 = (int)(take_stack(slab_of_block(blockIdx.x, n_units), n_units, w, y, w_second, y_second) * slabs) * kGemmBM;
    const u32 count = n_tiles[0];
    if (g > count) return;
    if (g == count) { // the refused slots' rows: NaN (crates/gpu/src/gemm/grouped.rs:2283-2287)
        const u32 refused = n_tiles[1];
        const u32 rows = slabs * kGemmBM;
        for (u32 i = tid; i < refused * rows; i += 256) {
            const u32 s = cols[n_slots - n_tiles[2] - refused + i / rows];
            const int r = row0 + (int)(i % rows);
            if (r < rpe) y[(size_t)s * rpe + r] = bm_bits_f32(0x7fc00000u);
        }
        return;
    }
    const u32 e = tiles[2 * g], word = tiles[2 * g + 1];
    const int start = (int)(word & 0xffffu), len = (int)(word >> 16);
    if (tid < kGemmBN) {
        const u32 s = cols[start + (tid < len ? tid : 0)];
        tab->slot[tid] = s;
        tab->col[tid] = s / slot_div;
    }
    __syncthreads();
    constexpr int kBlock = bm_block_bytes<WT>();
    constexpr bool kQ45 = X::kMins;                  // one walk: Q5_K is Q4_K with a fifth bit a code
    constexpr int kCodesAt = WT == BM_Q5K ? 48 : 16; // where a Q4_K / Q5_K block's nibbles start
    const u32 row_bytes = (u32)nb * kBlock, col_bytes = (u32)nb * BM_Q82_SB_EXT;

    // What a thread stages of every half: of row tid / 4 the sixteen code bytes 16 p .. of the half's 64 (p = tid % 4: low
    // nibbles one 16-value group, high nibbles another), of column tid / 4 the codes 16 p .. and 64 + 16 p .., and of both
    // the factors of the half's block p.
    const int wr = tid >> 2, p = tid & 3;
    const uint8_t *we = w + (size_t)e * rpe * row_bytes;
    auto row_at = [&](int first_row) { return (u32)(first_row + wr < rpe ? first_row + wr : rpe - 1) * row_bytes; };
    // (of at most 32 slots: of column tid / 8 the codes 16 (tid % 8) ..; of at most 16: of column tid / 16 the codes 8 (tid % 16) ..)
    const bool narrow = len <= 32, thin = kQ45 && len <= 16;
    const u32 apair = tab->col[wr] * col_bytes + 8 * p + (u32)nb * BM_Q82_SB_REF;
    const u32 acol = thin ? tab->col[tid >> 4] * col_bytes + 16 + 8 * (tid & 15)
                     : narrow ? tab->col[tid >> 3] * col_bytes + 16 + 16 * (tid & 7)
                              : tab->col[wr] * col_bytes + 16 + 16 * p;
    v4u rw, rq = {0, 0, 0, 0}, rh = {0, 0, 0, 0}, ra[2] = {};
    u32 q6d = 0, q6s = 0, q6t = 0; // (Q6_K; words of their own: as parts of a vector they were moved, and waited for, as they came)
    float d8, y0 = 0.0f, y4 = 0.0f;
    auto ld16 = [](const uint8_t *at) {
        v4u v;
        __builtin_memcpy(&v, at, 16);
        return v;
    };
    struct At { // a super-block: of which row, and which
        u32 row; // the row's offset in the expert's rows
        int i;
    };
    auto fetch_row = [&](At at, auto half) __attribute__((always_inline)) {
        constexpr int j = decltype(half)::value;
        const uint8_t *blk = we + (at.row + (u32)at.i * kBlock);
        if constexpr (kQ45) {
            rw = ld16(blk + kCodesAt + 64 * j + 16 * p);
            // Q5_K: value n's fifth bit is bit n / 32 of high byte n % 32 (crates/gguf/src/quant.rs:769-816)
            if constexpr (WT == BM_Q5K) rq = ld16(blk + 16 + 16 * (p & 1));
        } else { // Q6_K: ql bytes 64 j + 16 p .. and the qh bytes that go with them
            rw = ld16(blk + 64 * j + 16 * p);
            rq = ld16(blk + 128 + 32 * j + 16 * (p & 1));
        }
    };
    auto fetch_col = [&](int i, auto half, int q) __attribute__((always_inline)) {
        constexpr int j = decltype(half)::value;
        ra[q] = ld16(act + (acol + (u32)(2 * i + j) * BM_Q82X4_STRIDE) + 64 * q);
    };
    const u32 k1024 = 0x64006400u, m4l = 0x000f000fu, m4h = 0x00f000f0u, m8 = 0x00ff00ffu, mx = WT == BM_Q5K ? 0x00100010u : 0x00300030u,
              my = WT == BM_Q5K ? 0x01000100u : 0x03000300u;
    // (explicit LDS addresses: a base a lane and constants; the reads volatile, so that eight-byte reads stay eight bytes: merged
    // into sixteen they run at half the rate)
    typedef __attribute__((address_space(3))) uint8_t *LdsB;
    typedef __attribute__((address_space(3))) float *LdsF;
    typedef const volatile __attribute__((address_space(3))) v2u *LdsV2;
    typedef const volatile __attribute__((address_space(3))) float *LdsVF;
    const LdsB my_put = (LdsB)lds + wr * kXStride + 32 * p, my_factor = (LdsB)lds + 4 * kXCodes + 4 * wr + kXLine * p;
    const LdsB my_put_few = (LdsB)lds + (tid >> 3) * kXStride + 32 * (tid & 7);
    auto put = [&](LdsB to, int at, u32 a, u32 b) { *(__attribute__((address_space(3))) v2u *)(to + at) = (v2u){a, b}; };
    auto factor = [&](int at, float v) { *(LdsF)(my_factor + at) = v; };
    // Word k of the sixteen code bytes of the row. Four codes a word become f16 in the order 0, 2, 1, 3 (rows and columns alike: a
    // sum's terms may come in any order). Low nibbles: group p of the buffer's first four; high nibbles: of its second four (Q6_K:
    // the values' own order).
    auto stash_word = [&](auto half, int k, u32 x, [[maybe_unused]] u32 high) __attribute__((always_inline)) {
        constexpr int j = decltype(half)::value;
        const u32 x8 = x >> 8;
        u32 l0 = and_or(x, m4l, k1024), l1 = and_or(x8, m4l, k1024), h0 = and_or(x, m4h, k1024), h1 = and_or(x8, m4h, k1024);
        if constexpr (WT == BM_Q5K) { // the fifth bits of blocks 4 j + 2 (p / 2) and the one after
            const u32 t = high >> (4 * j + 2 * (p >> 1));
            l0 = and_or(t << 4, mx, l0);
            l1 = and_or(t >> 4, mx, l1);
            h0 = and_or(t << 7, my, h0);
            h1 = and_or(t >> 1, my, h1);
        }
        if constexpr (WT == BM_Q6K) { // the two high bits of quarters p / 2 and p / 2 + 2
            const u32 t = high >> (2 * (p >> 1)), t4 = t << 4, t8 = t >> 4;
            l0 = and_or(t4, mx, l0);
            l1 = and_or(t8, mx, l1);
            h0 = and_or(t4, my, h0);
            h1 = and_or(t8, my, h1);
        }
        constexpr float kOff = kQ45 ? 0.0f : 32.0f;
        put(my_put, j * kXCodes + 8 * k, h2_less(l0, 1024.0f + kOff), h2_less(l1, 1024.0f + kOff));
        put(my_put, j * kXCodes + 128 + 8 * k, h2_16th(h0, kOff), h2_16th(h1, kOff));
    };
    // Words 2 h and 2 h + 1 of the column's sixteen codes q.
    auto stash_col = [&](auto few, auto half, int q, int h) __attribute__((always_inline)) {
        constexpr int j = decltype(half)::value;
#pragma unroll
        for (int k = 2 * h; k < 2 * h + 2; k++) {
            const u32 u = ra[q][k] ^ 0x80808080u;
            put(decltype(few)::value ? my_put_few : my_put, (2 + j) * kXCodes + 128 * q + 8 * k, h2_less(and_or(u, m8, k1024), 1152.0f),
                h2_less(and_or(u >> 8, m8, k1024), 1152.0f));
        }
    };
    float r4 = 0.0f; // Q4_K, Q5_K: the scale product of block 4 + p, kept for the second half
    auto stash_factors = [&](auto half) __attribute__((always_inline)) {
        constexpr int j = decltype(half)::value;
        if constexpr (kQ45 && j == 0) { // crates/gguf/src/quant.rs:620-628 get_scale_min_k4
            const float d = bm_half_to_f32((unsigned short)(rh.x & 0xffffu)), dmin = bm_half_to_f32((unsigned short)(rh.x >> 16));
            const u32 b0 = (rh.y >> (8 * p)) & 0xffu, b4 = (rh.z >> (8 * p)) & 0xffu, b8 = (rh.w >> (8 * p)) & 0xffu;
            atomicOr((u32 *)(my_factor + X::kHeadsAt), rh.x); // (its own word: an LDS instruction in place of a register that there is not)
            factor(0, d * (float)(b0 & 63u));
            r4 = d * (float)((b8 & 15u) | ((b0 >> 6) << 4));
            factor(X::kMinsAt, -(dmin * (float)(b4 & 63u)));
            factor(X::kMinsAt + 4 * kXLine, -(dmin * (float)((b8 >> 4) | ((b4 >> 6) << 4))));
            factor(X::kMinsAt + 8 * kXLine, y0);
            factor(X::kMinsAt + 12 * kXLine, y4);
        } else if constexpr (kQ45) {
            factor(X::kHalf, r4);
        } else { // groups p and 4 + p of the half
            const float d = bm_half_to_f32((unsigned short)q6d);
            factor(j * X::kHalf, d * (float)(int)(signed char)q6s);
            factor(j * X::kHalf + 4 * kXLine, d * (float)(int)(signed char)q6t);
        }
        factor(j * X::kHalf + X::kScales * kXLine, d8);
    };
    auto fetch_factors = [&](At at, auto half) __attribute__((always_inline)) {
        constexpr int j = decltype(half)::value;
        const uint8_t *blk = we + (at.row + (u32)at.i * kBlock);
        if constexpr (kQ45) {
            if constexpr (j == 0) rh = ld16(blk); // d, dmin, the twelve scale bytes
        } else {
            q6d = bm_ld2u(blk + 208);       // d
            q6s = blk[192 + 8 * j + p];     // the scales of groups p
            q6t = blk[192 + 8 * j + 4 + p]; // and 4 + p
        }
        d8 = *reinterpret_cast<const float *>(act + (apair + 64 * (u32)at.i) + 32 * j); // of block 4 j + p
        if constexpr (kQ45 && j == 0) { // d8 isum of blocks p and 4 + p
            y0 = *reinterpret_cast<const float *>(act + (apair + 64 * (u32)at.i) + 4);
            y4 = *reinterpret_cast<const float *>(act + (apair + 64 * (u32)at.i) + 36);
        }
    };
    // Step st of eight of a half's staging. The codes of the half after it (super-block `next`) are asked for where a register's last
    // word is done with, seven steps before its first use; the half's own factors at step 1, for step 7.
    auto stash = [&](auto few, auto half, int st, At now, At next) __attribute__((always_inline)) {
        constexpr std::integral_constant<int, 1 - decltype(half)::value> after{};
        constexpr int kPieces = decltype(few)::value ? 1 : 2; // of a column's codes
        if (st == 0) fetch_factors(now, half);
        if (st < 4) {
            stash_word(half, st, rw[st], rq[st]);
            if (st == 3) fetch_row(next, after);
        } else if (st < 4 + 2 * kPieces) {
            stash_col(few, half, (st - 4) >> 1, st & 1);
            if (st & 1) fetch_col(next.i, after, (st - 4) >> 1);
        }
        if (st == 7) stash_factors(half);
    };

    // this lane in its wave's 32 x 32 products: operand slot and row lane % 32, eight of a group's sixteen values by lane / 32;
    // result v is slot 8 (v / 4) + 4 (lane / 32) + v % 4 of row lane % 32
    const int l32 = lane & 31, kh = lane >> 5;
    const int wrow0 = 32 * (wv & 1), wslot0 = narrow ? 0 : 32 * (wv >> 1);
    const int gh = wv >> 1; // the half of the accumulators a wave of a narrow tile keeps

    constexpr std::integral_constant<int, 0> kFirst{};
    constexpr std::integral_constant<int, 1> kSecond{};
    const int first_row = row0;
    int left = (rpe - row0 + kGemmBM - 1) / kGemmBM; // slabs to do
    left = left < (int)slabs ? left : (int)slabs;
    auto run = [&](auto few) __attribute__((always_inline)) {
        constexpr bool kFew = decltype(few)::value;
        constexpr int kPairs = kFew ? 2 : 4;
        const int up = kFew ? gh : 0;
        const LdsB my_row = (LdsB)lds + (wrow0 + l32) * kXStride + 16 * kh + 32 * up;
        const LdsB my_col = (LdsB)lds + 2 * kXCodes + ((kFew ? 0 : wslot0) + l32) * kXStride + 16 * kh + 32 * up;
        // the factors of an outer product's two blocks, or of a block's two groups (Q6_K in a wide tile: one d8 for both; in a narrow
        // one two blocks' groups of the wave's half): a half of the lanes each
        const LdsB my_fr = (LdsB)lds + 4 * kXCodes + 4 * (wrow0 + l32), my_fc = (LdsB)lds + 4 * kXCodes + 4 * ((kFew ? 0 : wslot0) + l32);
        const LdsB my_sr = my_fr + (kQ45 || !kFew ? kh : up + 2 * kh) * kXLine;
        const LdsB my_sc = my_fc + (kQ45 || kFew ? kh : 0) * kXLine + X::kScales * kXLine;
        const LdsB my_mr = my_fr + (kh + 4 * up) * kXLine + X::kMinsAt, my_mc = my_fc + (kh + 4 * up) * kXLine + X::kMinsAt + 8 * kXLine;
        v32f acc[kPairs]; // accumulator l (a narrow tile: l + 4 gh): [l / 2], results 16 (l % 2) ..
        // A half's arithmetic, a step a 16-value group, and in the shade of each step's outer product a piece of the staging of the half
        // after it.
        auto arithmetic = [&](auto half, At now, At next) __attribute__((always_inline)) {
            constexpr int j = decltype(half)::value, kSteps = kFew ? 4 : 8;
            const v16f z16 = {};
            const v32f z32 = {};
            v4u a, b;
            v16f sum;
            v32f pd;
            auto rd = [&](int step) { // a step's group of the half's eight
                const int gr = kFew ? 2 * step : step; // (and the wave's half of the groups on top, where the tile is narrow)
                const int at = j * kXCodes + 32 * (kQ45 ? 4 * ((gr >> 1) & 1) + 2 * (gr >> 2) + (gr & 1) : gr), ct = j * kXCodes + 32 * gr;
                const v2u a0 = *(LdsV2)(my_row + at), a1 = *(LdsV2)(my_row + at + 8), b0 = *(LdsV2)(my_col + ct), b1 = *(LdsV2)(my_col + ct + 8);
                a = (v4u){a0.x, a0.y, a1.x, a1.y};
                b = (v4u){b0.x, b0.y, b1.x, b1.y};
            };
            auto product = [&]() {
                sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, b), __builtin_bit_cast(v8h, a), z16, 0, 0, 0);
            };
            // Q4_K, Q5_K: one scale a block; Q6_K: one a group (crates/qdot/src/lib.rs:4403-4440, :4794-4809)
            auto scale = [&](int bk, int gr) {
                const float fc = *(LdsVF)(my_sc + j * X::kHalf + bk * kXLine), fr = *(LdsVF)(my_sr + j * X::kHalf + (kQ45 ? bk : gr) * kXLine);
                pd = __builtin_amdgcn_mfma_f32_32x32x1f32(fc, fr, z32, 0, 0, 0);
            };
            // the min terms come before a super-block's products: accumulator l takes sub-block l's (crates/qdot/src/lib.rs:4389-4394)
            auto min_term = [&](int s) {
                acc[s] = __builtin_amdgcn_mfma_f32_32x32x1f32(*(LdsVF)(my_mc + 2 * s * kXLine), *(LdsVF)(my_mr + 2 * s * kXLine), acc[s], 0, 0, 0);
            };
            rd(0);
            if constexpr (kQ45 && j == 0) {
                min_term(0);
                if constexpr (!kFew) min_term(2);
            }
#pragma unroll
            for (int step = 0; step < kSteps; step++) {
                const int bk = kFew ? step : step >> 1, h = kFew ? 0 : step & 1, l = 4 * h + bk, al = 16 * (l & 1), pb = 16 * (kQ45 || kFew ? bk & 1 : h);
                product();
                if (kFew ? (step & 1) == 0 : (step & (kQ45 ? 3 : 1)) == 0) scale(bk, kFew ? 2 * step : step);
                if constexpr (kQ45 && j == 0) {
                    if (step == (kFew ? 0 : 1)) min_term(1);
                    if (!kFew && step == 3) min_term(kPairs - 1);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (step + 1 < kSteps) rd(step + 1);
#pragma unroll
                for (int st = 8 / kSteps * step; st < 8 / kSteps * (step + 1); st++) stash(few, std::integral_constant<int, 1 - j>{}, st, now, next);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int v = 0; v < 16; v++) acc[l >> 1][al + v] = fmaf(pd[pb + v], sum[v], acc[l >> 1][al + v]);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if constexpr (kQ45) factor(X::kHeadsAt, 0.0f);
        At now = {row_at(row0), 0};
        fetch_row(now, kFirst);
        fetch_col(0, kFirst, 0);
        if constexpr (!kFew) fetch_col(0, kFirst, 1);
        // (the loads in the loop's order, kept by the fences: the loop's first wait counts the loads behind the one it waits for, and
        // where this way into the loop has fewer it waits for all)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int st = 0; st < 8; st++) {
            stash(few, kFirst, st, now, now);
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        // the super-block after `at`, in the next slab behind a slab's last (the very last: itself, staged for no reader)
        auto following = [&](At at) {
            if (at.i + 1 < nb) return At{at.row, at.i + 1};
            return left > 1 ? At{row_at(row0 + kGemmBM), 0} : at;
        };
        // (a half's last readers passed the barrier that ended the half before)
#pragma unroll
        for (int l = 0; l < kPairs; l++)
#pragma unroll
            for (int v = 0; v < 32; v++) acc[l][v] = 0.0f;
        for (; left > 0; left--, row0 += kGemmBM) {
            for (int i = 0; i < nb; i++) {
                const At next = following(now);
                arithmetic(kFirst, now, next);
                __syncthreads();
                arithmetic(kSecond, next, next);
                __syncthreads();
                now = next;
            }
            // the closing sum of the eight lanes (crates/qdot/src/lib.rs:4128 hsum_float_8's order) and the store
            const int row = row0 + wrow0 + l32;
            auto store = [&](int v, float t0, float t1, float t2, float t3) {
                const int n = wslot0 + 8 * (v >> 2) + 4 * kh + (v & 3);
                if (row < rpe && n < len) y[(size_t)tab->slot[n] * rpe + row] = (t0 + t2) + (t1 + t3);
            };
            if constexpr (kFew) {
                // a wave sums eight of a lane's sixteen results and has the other wave's accumulators of them through LDS (the half 1
                // buffers: half 0's hold the next slab's first codes)
                float *const swap = reinterpret_cast<float *>(lds + (wrow0 ? 3 : 1) * kXCodes);
                auto give = [&](auto from) __attribute__((always_inline)) { // accumulators of results `from` .. of the other wave
#pragma unroll
                    for (int l = 0; l < 4; l++)
#pragma unroll
                        for (int v = 0; v < 8; v++) swap[((gh * 4 + l) * 8 + v) * 64 + lane] = acc[l >> 1][16 * (l & 1) + decltype(from)::value + v];
                };
                auto take = [&](auto from) __attribute__((always_inline)) {
#pragma unroll
                    for (int v = 0; v < 8; v++) {
                        float t[4];
#pragma unroll
                        for (int l = 0; l < 4; l++)
                            t[l] = acc[l >> 1][16 * (l & 1) + decltype(from)::value + v] + swap[(((1 - gh) * 4 + l) * 8 + v) * 64 + lane];
                        store(decltype(from)::value + v, t[0], t[1], t[2], t[3]);
                    }
                };
                constexpr std::integral_constant<int, 0> kLow{};
                constexpr std::integral_constant<int, 8> kHigh{};
                if (gh) give(kLow);
                else give(kHigh);
                __syncthreads();
                if (gh) take(kHigh);
                else take(kLow);
                __syncthreads();
            } else {
#pragma unroll
                for (int v = 0; v < 16; v++)
                    store(v, acc[0][v] + acc[kPairs - 2][v], acc[0][16 + v] + acc[kPairs - 2][16 + v], acc[1][v] + acc[kPairs - 1][v],
                          acc[1][16 + v] + acc[kPairs - 1][16 + v]);
            }
#pragma unroll
            for (int l = 0; l < kPairs; l++)
#pragma unroll
                for (int v = 0; v < 32; v++) acc[l][v] = 0.0f;
        }
    };
    // A tile of at most 16 slots: a wave takes 16 rows, all the slots and all the accumulators; products and outer products are the
    // 16 x 16 forms (one of scales four blocks at a time), half the multiply-adds of a 32 x 32 tile's padding. Lane: row (operand: slot, row)
    // lane % 16, four of a group's sixteen values by lane / 16; result r: slot 4 (lane / 16) + r of row lane % 16.
    // So little arithmetic a byte that it is the bytes on their way that bound it: whole super-blocks are asked for two ahead, into a ring
    // of three sets of registers. (Top-8 of 128 experts Q4_K, us a layer: 256 tokens 217 -> 209, 512 tokens 280 -> 275; top-8 of 64 of
    // 7168 x 1536, 300 tokens 890 -> 828. Q6_K, whose bytes come in more and smaller requests, was 2 to 5 % slower this way.)
    [[maybe_unused]] auto run_thin = [&]() __attribute__((always_inline)) {
        const int l16 = lane & 15, kq = lane >> 4;
        const LdsB my_row = (LdsB)lds + (16 * wv + l16) * kXStride + 8 * kq, my_col = (LdsB)lds + 2 * kXCodes + l16 * kXStride + 8 * kq;
        const LdsB my_fr = (LdsB)lds + 4 * kXCodes + 4 * (16 * wv + l16), my_fc = (LdsB)lds + 4 * kXCodes + 4 * l16;
        const LdsB my_sr = my_fr + kq * kXLine, my_sc = my_fc + (X::kScales + kq) * kXLine;
        const LdsB my_mr = my_fr + kq * kXLine + X::kMinsAt, my_mc = my_fc + kq * kXLine + X::kMinsAt + 8 * kXLine;
        // what a thread stages of a column: of column tid / 16 the codes 8 (tid % 16) .., of column tid / 8 % 16 the factors of block tid % 8
        const int wc = (tid >> 3) & 15, wb = tid & 7;
        const u32 col_pair = tab->col[wc] * col_bytes + 8 * wb + (u32)nb * BM_Q82_SB_REF;
        const LdsB put_col = (LdsB)lds + 2 * kXCodes + (tid >> 4) * kXStride + 16 * (tid & 15);
        // (a block of the half that is not being staged goes to a slot that nobody reads)
        const LdsB put_d8[2] = {(LdsB)lds + 4 * kXCodes + (X::kScales + (wb & 3)) * kXLine + 4 * (wc + (wb < 4 ? 0 : 16)),
                                (LdsB)lds + 4 * kXCodes + (X::kScales + (wb & 3)) * kXLine + 4 * (wc + (wb < 4 ? 16 : 0)) + X::kHalf};
        const LdsB put_isum = (LdsB)lds + 4 * kXCodes + X::kMinsAt + (8 + wb) * kXLine + 4 * wc;
        struct Sb { // a super-block's bytes
            v4u w[2], q, head;
            v2u col[2], pair;
        } ring[3];
        auto fetch = [&](Sb &b, At at) __attribute__((always_inline)) {
            const uint8_t *blk = we + (at.row + (u32)at.i * kBlock);
            b.head = ld16(blk);
            b.pair = *reinterpret_cast<const v2u *>(act + (col_pair + 64 * (u32)at.i));
#pragma unroll
            for (int j = 0; j < 2; j++) {
                b.w[j] = ld16(blk + kCodesAt + 64 * j + 16 * p);
                b.col[j] = *reinterpret_cast<const v2u *>(act + (acol + (u32)(2 * at.i + j) * BM_Q82X4_STRIDE));
            }
            b.q = WT == BM_Q5K ? ld16(blk + 16 + 16 * (p & 1)) : (v4u){0, 0, 0, 0};
        };
        auto stage = [&](const Sb &b, auto half) __attribute__((always_inline)) {
            constexpr int j = decltype(half)::value;
#pragma unroll
            for (int k = 0; k < 4; k++) stash_word(half, k, b.w[j][k], b.q[k]);
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const u32 u = b.col[j][k] ^ 0x80808080u;
                put(put_col, j * kXCodes + 8 * k, h2_less(and_or(u, m8, k1024), 1152.0f), h2_less(and_or(u >> 8, m8, k1024), 1152.0f));
            }
            // crates/gguf/src/quant.rs:620-628 get_scale_min_k4
            const float d = bm_half_to_f32((unsigned short)(b.head.x & 0xffffu)), dmin = bm_half_to_f32((unsigned short)(b.head.x >> 16));
            const u32 b0 = (b.head.y >> (8 * p)) & 0xffu, b4 = (b.head.z >> (8 * p)) & 0xffu, b8 = (b.head.w >> (8 * p)) & 0xffu;
            if constexpr (j == 0) {
                atomicOr((u32 *)(my_factor + X::kHeadsAt), b.head.x);
                factor(0, d * (float)(b0 & 63u));
                factor(X::kMinsAt, -(dmin * (float)(b4 & 63u)));
                factor(X::kMinsAt + 4 * kXLine, -(dmin * (float)((b8 >> 4) | ((b4 >> 6) << 4))));
                *(LdsF)put_isum = bm_bits_f32(b.pair.y);
            } else {
                factor(X::kHalf, d * (float)((b8 & 15u) | ((b0 >> 6) << 4)));
            }
            *(LdsF)put_d8[j] = bm_bits_f32(b.pair.x);
        };
        v16f acc[2]; // accumulator 4 h + block: [h], results 4 block ..
        auto arithmetic = [&](auto half, const Sb &staged) __attribute__((always_inline)) {
            constexpr int j = decltype(half)::value;
            const v16f z16 = {};
            const v4f z4 = {};
            v4f sum[8];
            const v16f pd = __builtin_amdgcn_mfma_f32_16x16x1f32(*(LdsVF)(my_sc + j * X::kHalf), *(LdsVF)(my_sr + j * X::kHalf), z16, 0, 0, 0);
            // the min terms come before a super-block's products: accumulator l takes sub-block l's (crates/qdot/src/lib.rs:4389-4394)
            if constexpr (j == 0)
#pragma unroll
                for (int h = 0; h < 2; h++)
                    acc[h] = __builtin_amdgcn_mfma_f32_16x16x1f32(*(LdsVF)(my_mc + 4 * h * kXLine), *(LdsVF)(my_mr + 4 * h * kXLine), acc[h], 0, 0, 0);
#pragma unroll
            for (int gr = 0; gr < 8; gr++) {
                const int at = j * kXCodes + 32 * (4 * ((gr >> 1) & 1) + 2 * (gr >> 2) + (gr & 1)), ct = j * kXCodes + 32 * gr;
                const v2u a = *(LdsV2)(my_row + at), b = *(LdsV2)(my_col + ct);
                sum[gr] = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(v4h, b), __builtin_bit_cast(v4h, a), z4, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            stage(staged, std::integral_constant<int, 1 - j>{});
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int gr = 0; gr < 8; gr++) {
                const int bk = gr >> 1, h = gr & 1;
#pragma unroll
                for (int r = 0; r < 4; r++) acc[h][4 * bk + r] = fmaf(pd[4 * bk + r], sum[gr][r], acc[h][4 * bk + r]);
            }
        };
        factor(X::kHeadsAt, 0.0f);
        int far_left = left, far_row0 = row0; // of the super-block asked for last
        At far = {row_at(row0), 0};
        auto advance = [&]() { // to the super-block after it, in the next slab behind a slab's last (the very last: itself, for no reader)
            if (far.i + 1 < nb) far.i++;
            else if (far_left > 1) far_left--, far_row0 += kGemmBM, far = At{row_at(far_row0), 0};
        };
        fetch(ring[0], far);
        advance();
        __builtin_amdgcn_sched_barrier(0);
        fetch(ring[1], far);
        advance();
        __builtin_amdgcn_sched_barrier(0);
        stage(ring[0], kFirst);
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 16; v++) acc[0][v] = acc[1][v] = 0.0f;
        int todo = left * nb, i = 0;
        auto step = [&](auto at) __attribute__((always_inline)) { // the super-block in the ring's place `at`
            constexpr int c = decltype(at)::value;
            fetch(ring[(c + 2) % 3], far);
            advance();
            __builtin_amdgcn_sched_barrier(0);
            arithmetic(kFirst, ring[c]);
            __syncthreads();
            arithmetic(kSecond, ring[(c + 1) % 3]);
            __syncthreads();
            if (++i < nb) return;
            i = 0;
            // the closing sum of the eight lanes (crates/qdot/src/lib.rs:4128 hsum_float_8's order) and the store
            const int row = row0 + 16 * wv + l16;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int n = 4 * kq + r;
                const float t0 = acc[0][r] + acc[1][r], t1 = acc[0][4 + r] + acc[1][4 + r], t2 = acc[0][8 + r] + acc[1][8 + r], t3 = acc[0][12 + r] + acc[1][12 + r];
                if (row < rpe && n < len) y[(size_t)tab->slot[n] * rpe + row] = (t0 + t2) + (t1 + t3);
            }
#pragma unroll
            for (int v = 0; v < 16; v++) acc[0][v] = acc[1][v] = 0.0f;
            row0 += kGemmBM;
        };
        for (;;) {
            step(std::integral_constant<int, 0>{});
            if (--todo == 0) break;
            step(std::integral_constant<int, 1>{});
            if (--todo == 0) break;
            step(std::integral_constant<int, 2>{});
            if (--todo == 0) break;
        }
    };
    if (thin) {
        if constexpr (kQ45) run_thin();
    } else if (narrow) run(std::true_type{});
    else run(std::false_type{});
    if constexpr (kQ45) {
        u32 heads = 0u;
#pragma unroll
        for (int q = 0; q < 4; q++) heads |= *(const u32 *)(lds + 4 * kXCodes + X::kHeadsAt + 4 * lane + q * kXLine);
        if (__ballot((heads & 0x8000u) != 0u) == 0) return; // (see above)
        // the results this lane stored
        const int end = row0 < rpe ? row0 : rpe, first = narrow && !thin ? 8 * gh : 0, last = thin ? 4 : narrow ? first + 8 : 16;
#pragma nounroll
        for (int row = first_row + (thin ? 16 * wv + (lane & 15) : wrow0 + l32); row < end; row += kGemmBM)
#pragma nounroll
            for (int v = first; v < last; v++) {
                const int n = thin ? 4 * (lane >> 4) + v : wslot0 + 8 * (v >> 2) + 4 * kh + (v & 3);
                if (n >= len) continue;
                float *out = y + (size_t)tab->slot[n] * rpe + row;
                if (*out == 0.0f) *out = q45_value<WT>(we + (size_t)row * row_bytes, act + (size_t)tab->col[n] * col_bytes, nb);
            }
    }
}

typedef int v16i __attribute__((ext_vector_type(16)));

// The tolerance mode (BM_GEMM_FAST). The integer sums are the exact ones, formed by matrix instructions whose K is
// exactly the span one scale covers, so no issued multiply is wasted:
//   Q4_K, Q5_K: a 32-value sub-block of a row against a 32-value block of a column is one v_mfma_i32_32x32x32_i8 over 32
//         rows and 32 slots; the min terms, sum over a super-block's eight sub-blocks of -(dmin m)[row] x (d8 isum)[slot],
//         are a product of two thin matrices and go to v_mfma_f32_32x32x2_f32 (four a super-block), into the same
//         accumulators;
//   Q6_K: a 16-value group, whose scale is its own, is one v_mfma_i32_32x32x16_i8.
// The product of a row's scale and a column's d8 for a whole 32 x 32 tile is an outer product, so it goes to the matrix
// cores too: v_mfma_f32_32x32x8_bf16_1k over K slots that hold the row scale as three bf16 pieces (8 + 8 + 8 bits: the
// f32 exactly) against the column's d8 (a bf16 value as it stands) in the same three slots. Each of the three products
// is exact in f32; their sum is the f32 product to within a rounding. Lanes 32 .. 63 carry K slots 4 .. 7: the row side
// reads a zero there.
// What is left for the vector ALU is two operations a (row, slot, unit): the integer to a float and the multiply-add into
// the one accumulator a value (the CPU path keeps eight and a fixed order: that is the exact mode; this one differs from
// it by f32 rounding only).
// A workgroup of eight waves takes 128 rows and a tile's 64 slots, a wave 32 x 32 of them. LDS holds one super-block: the
// columns' codes, the slab's codes unpacked to a signed byte each, and the scale operands; 72 KB and at most 128 registers,
// so two workgroups, four waves a SIMD, share a CU and fill each other's staging gaps and waits (a wave alone issues a
// vector instruction every five to six cycles, the SIMD takes one every four). The next super-block's global loads are in flight during the
// arithmetic on the present one. Inside a wave a unit's matrix instructions are issued one unit ahead of the vector work
// on their results, and its LDS operands are read two units ahead.
constexpr int kFastRows = 128;
constexpr int kFastThreads = 512;
constexpr int kFastRowLine = kFastRows + 4; // entries a line of the row tables ([unit][row]); entry kFastRows of a line holds zero
constexpr int kFastColLine = kGemmBN + 4;   // entries a line of the column tables ([block][slot])
// a row's or a column's 256 codes, padded so that the operand reads of consecutive rows fall on different banks: the
// reads are 16 bytes a lane for K = 32 and 8 bytes a lane for K = 16
template <int WT>
__host__ __device__ constexpr int fast_code_stride() {
    return WT == BM_Q6K ? 256 + 8 : 256 + 16;
}
template <int WT>
__host__ __device__ constexpr int fast_units() { // scaled units a super-block
    return WT == BM_Q6K ? 16 : 8;
}
template <int WT>
__host__ __device__ constexpr size_t fast_lds_bytes() {
    // codes of both sides; the columns' scale operands ([block][slot], 8 bytes) and d8 * isum; the rows' scale operands
    // ([unit][row], 8 bytes) and mins
    constexpr bool mins = WT != BM_Q6K;
    return sizeof(GemmLds) + (size_t)(kGemmBN + kFastRows) * fast_code_stride<WT>() + 8 * kFastColLine * (8 + (mins ? sizeof(float) : 0)) +
           (size_t)fast_units<WT>() * kFastRowLine * (8 + (mins ? sizeof(float) : 0));
}

__device__ __forceinline__ uint2 scale_operand_row(float v) {
    const u32 hi = bm_f32_bits(v) & 0xffff0000u;
    const float r1 = v - bm_bits_f32(hi);
    const u32 mid = bm_f32_bits(r1) & 0xffff0000u;
    const float r2 = r1 - bm_bits_f32(mid);
    return make_uint2((hi >> 16) | mid, bm_f32_bits(r2) >> 16);
}
__device__ __forceinline__ uint2 scale_operand_col(u32 d8_bits) {
    const u32 h = d8_bits >> 16;
    return make_uint2(h | (h << 16), h);
}
typedef short v4s __attribute__((ext_vector_type(4)));

template <int WT>
__global__ __launch_bounds__(kFastThreads, 2) void k_gemm_fast(const uint8_t *w, int rpe, int nb, const uint8_t *act, const u32 *cols,
                                                      const u32 *tiles, const u32 *n_tiles, u32 n_units, u32 slot_div,
                                                      u32 n_slots, float *y, const uint8_t *w_second, float *y_second) {
    constexpr bool kQ45 = WT == BM_Q4K || WT == BM_Q5K;
    constexpr int kStride = fast_code_stride<WT>(), kUnitsSb = fast_units<WT>(), kBlock = bm_block_bytes<WT>();
    constexpr int kOp = kQ45 ? 16 : 8; // operand bytes a lane
    extern __shared__ __align__(16) uint8_t lds[];
    GemmLds *tab = reinterpret_cast<GemmLds *>(lds);
    uint8_t *a_codes = lds + sizeof(GemmLds);
    uint8_t *w_codes = a_codes + (size_t)kGemmBN * kStride;
    uint2 *d8_t = reinterpret_cast<uint2 *>(w_codes + (size_t)kFastRows * kStride); // [block][slot]
    uint2 *sv_t = d8_t + 8 * kFastColLine;                                           // [unit][row]
    float *my_t = reinterpret_cast<float *>(sv_t + kUnitsSb * kFastRowLine);         // Q4_K, Q5_K only, as is mn_t
    float *mn_t = my_t + 8 * kFastColLine;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const u32 g = tile_of_block(blockIdx.x, n_units);
    const int row0 = (int)take_stack(slab_of_block(blockIdx.x, n_units), n_units, w, y, w_second, y_second) * kFastRows;
    const u32 count = n_tiles[0];
    if (g > count) return;
    if (g == count) { // the refused slots' rows: NaN (crates/gpu/src/gemm/grouped.rs:2283-2287)
        const u32 refused = n_tiles[1];
        for (u32 i = tid; i < refused * kFastRows; i += kFastThreads) {
            const u32 s = cols[n_slots - n_tiles[2] - refused + i / kFastRows];
            const int r = row0 + (int)(i % kFastRows);
            if (r < rpe) y[(size_t)s * rpe + r] = bm_bits_f32(0x7fc00000u);
        }
        return;
    }
    const u32 e = tiles[2 * g], word = tiles[2 * g + 1];
    const int start = (int)(word & 0xffffu), len = (int)(word >> 16);
    if (tid < kGemmBN) {
        const u32 s = cols[start + (tid < len ? tid : 0)];
        tab->slot[tid] = s;
        tab->col[tid] = s / slot_div;
    }
    if (tid < kUnitsSb) sv_t[tid * kFastRowLine + kFastRows] = make_uint2(0u, 0u);
    __syncthreads();
    const u32 row_bytes = (u32)nb * kBlock, col_bytes = (u32)nb * BM_Q82_SB_EXT;
    // what this thread stages of every super-block:
    //   two 16-byte pieces of column codes (column tid / 16 + 32 j, piece tid % 16 of the sixteen: a column's
    //   super-block is two groups of 144 bytes whose first 16 are scales and sums, skipped here),
    //   one (d8, d8 * isum) pair (column tid / 8, block tid % 8),
    //   two 16-byte pieces of weight codes (row tid / 8 + 64 j, piece tid % 8 of the row's eight: eight consecutive lanes
    //   read 128 consecutive bytes),
    //   a quarter of a weight row's scales (row tid / 4)
    const int ac = tid >> 4, ap = tid & 15;
    u32 src_a[2];
#pragma unroll
    for (int j = 0; j < 2; j++) src_a[j] = tab->col[ac + 32 * j] * col_bytes + 16u * (u32)(1 + ap + (ap >> 3));
    const int pcol = tid >> 3, pb = tid & 7;
    const u32 src_p = tab->col[pcol] * col_bytes + (u32)nb * BM_Q82_SB_REF + 8u * (u32)pb;
    const int wr = tid >> 2, wq = tid & 3;
    const uint8_t *we = w + (size_t)e * rpe * row_bytes;
    const u32 src_w = (u32)(row0 + wr < rpe ? row0 + wr : rpe - 1) * row_bytes;
    const int crow = tid >> 3, cc = tid & 7;
    constexpr int kCodesAt = WT == BM_Q5K ? 48 : WT == BM_Q4K ? 16 : 0;
    u32 src_c[2];
#pragma unroll
    for (int j = 0; j < 2; j++)
        src_c[j] = (u32)(row0 + crow + 64 * j < rpe ? row0 + crow + 64 * j : rpe - 1) * row_bytes + kCodesAt + 16u * (u32)cc;
    // the bytes that carry the high bits of piece cc, from the piece's own address: Q5_K's 32 high-bit bytes (value n's
    // fifth bit is bit n / 32 of byte n % 32), Q6_K's qh (piece cc of ql goes with qh piece cc % 2 of its half)
    const int high_at = WT == BM_Q5K ? 16 * (cc & 1) - 32 - 16 * cc : 128 + 32 * (cc >> 2) + 16 * (cc & 1) - 16 * cc;
    uint4 ra0, ra1, rq[2], rh, rx[WT == BM_Q4K ? 1 : 2];
    uint2 rp;
    auto fetch = [&](int i) {
        ra0 = *reinterpret_cast<const uint4 *>(act + (src_a[0] + (u32)i * BM_Q82_SB_REF));
        ra1 = *reinterpret_cast<const uint4 *>(act + (src_a[1] + (u32)i * BM_Q82_SB_REF));
        rp = *reinterpret_cast<const uint2 *>(act + (src_p + (u32)i * 64u));
        const uint8_t *blk = we + (src_w + (u32)i * kBlock);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint8_t *piece = we + (src_c[j] + (u32)i * kBlock);
            if constexpr (kQ45) {
                rq[j] = *reinterpret_cast<const uint4 *>(piece);
                if constexpr (WT == BM_Q5K) rx[j] = *reinterpret_cast<const uint4 *>(piece + high_at);
            } else {
                rq[j] = bm_ld16u(piece);
                rx[j] = bm_ld16u(piece + high_at);
            }
        }
        if constexpr (kQ45) {
            rh = *reinterpret_cast<const uint4 *>(blk); // d, dmin, the twelve scale bytes
        } else { // scales 4 wq .. 4 wq + 3 of the sixteen, and d
            rh.x = bm_ld2u(blk + 192 + 4 * wq) | (bm_ld2u(blk + 194 + 4 * wq) << 16);
            rh.y = bm_ld2u(blk + 208);
        }
    };
    auto put16 = [](uint8_t *dst, u32 a, u32 b, u32 c, u32 d) {
        if constexpr (kOp == 16) {
            *reinterpret_cast<uint4 *>(dst) = make_uint4(a, b, c, d);
        } else { // rows 8 bytes apart modulo 16
            *reinterpret_cast<uint2 *>(dst) = make_uint2(a, b);
            *reinterpret_cast<uint2 *>(dst + 8) = make_uint2(c, d);
        }
    };
    auto stash = [&]() {
        uint8_t *acol = a_codes + ac * kStride + 16 * ap;
        put16(acol, ra0.x, ra0.y, ra0.z, ra0.w);
        put16(acol + 32 * kStride, ra1.x, ra1.y, ra1.z, ra1.w);
        d8_t[pb * kFastColLine + pcol] = scale_operand_col(rp.x);
        if constexpr (kQ45) my_t[pb * kFastColLine + pcol] = bm_bits_f32(rp.y);
        const u32 ml = 0x0f0f0f0fu;
        if constexpr (kQ45) {
            // nibble piece cc of a row: code bytes 16 cc ..: the low nibbles are sub-block 2 p, values 16 (cc % 2) .., the
            // high nibbles sub-block 2 p + 1, the same values, with p = cc / 2
            const int p = cc >> 1, at = 16 * (cc & 1);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                uint8_t *row = w_codes + (crow + 64 * j) * kStride;
                u32 lo[4] = {rq[j].x & ml, rq[j].y & ml, rq[j].z & ml, rq[j].w & ml};
                u32 hi[4] = {(rq[j].x >> 4) & ml, (rq[j].y >> 4) & ml, (rq[j].z >> 4) & ml, (rq[j].w >> 4) & ml};
                if constexpr (WT == BM_Q5K) { // high-bit bytes 16 (cc % 2) ..: bit 2 p for the low nibbles, 2 p + 1 for the high
                    const u32 hw[4] = {rx[j].x, rx[j].y, rx[j].z, rx[j].w};
                    const u32 one = 0x01010101u;
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        lo[k] |= ((hw[k] >> (2 * p)) & one) << 4;
                        hi[k] |= ((hw[k] >> (2 * p + 1)) & one) << 4;
                    }
                }
                put16(row + 64 * p + at, lo[0], lo[1], lo[2], lo[3]);
                put16(row + 64 * p + 32 + at, hi[0], hi[1], hi[2], hi[3]);
            }
            // scale and min of sub-blocks 2 wq and 2 wq + 1 (crates/gguf/src/quant.rs:620-628 get_scale_min_k4): with the
            // twelve bytes as q[0 .. 11], sub-block j < 4 has q[j] & 63 and q[j + 4] & 63; j >= 4 has
            // (q[j + 4] & 15) | (q[j - 4] >> 6) << 4 and (q[j + 4] >> 4) | (q[j] >> 6) << 4
            const float d = bm_half_to_f32(rh.x & 0xffffu), dmin = bm_half_to_f32(rh.x >> 16);
            const bool upper = wq >= 2;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const u32 sh = 8u * (u32)(2 * (wq & 1) + i);
                const u32 qa = (rh.y >> sh) & 0xffu, qb = (rh.z >> sh) & 0xffu, qc = (rh.w >> sh) & 0xffu;
                const u32 scv = upper ? ((qc & 15u) | ((qa >> 6) << 4)) : (qa & 63u);
                const u32 mv = upper ? ((qc >> 4) | ((qb >> 6) << 4)) : (qb & 63u);
                sv_t[(2 * wq + i) * kFastRowLine + wr] = scale_operand_row(d * (float)scv);
                mn_t[(2 * wq + i) * kFastRowLine + wr] = -(dmin * (float)mv);
            }
        } else {
            // ql piece cc of a row (bytes 16 cc ..: half cc / 4, piece c = cc % 4 of it) with qh piece c % 2 of that half: the
            // low nibbles are quarter c / 2 of the half, values 16 (c % 2) .., the high nibbles quarter 2 + c / 2; a quarter's
            // high bits are bits 2 a .. of qh (crates/gguf/src/quant.rs:826-859). Each is one 16-value group: group
            // 8 (cc / 4) + 2 a + c % 2.
            const u32 mh = 0x03030303u;
            const int half = cc >> 2, c = cc & 3;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                uint8_t *row = w_codes + (crow + 64 * j) * kStride;
                const uint4 hq = rx[j];
#pragma unroll
                for (int hn = 0; hn < 2; hn++) {
                    const int a4 = (c >> 1) + 2 * hn, ns = 4 * hn, hs = 2 * a4;
                    put16(row + 128 * half + 32 * a4 + 16 * (c & 1),
                          q6_minus_32(((rq[j].x >> ns) & ml) | (((hq.x >> hs) & mh) << 4)),
                          q6_minus_32(((rq[j].y >> ns) & ml) | (((hq.y >> hs) & mh) << 4)),
                          q6_minus_32(((rq[j].z >> ns) & ml) | (((hq.z >> hs) & mh) << 4)),
                          q6_minus_32(((rq[j].w >> ns) & ml) | (((hq.w >> hs) & mh) << 4)));
                }
            }
            const float d = bm_half_to_f32(rh.y & 0xffffu);
#pragma unroll
            for (int jj = 0; jj < 4; jj++)
                sv_t[(4 * wq + jj) * kFastRowLine + wr] = scale_operand_row(d * (float)(int)(signed char)((rh.x >> (8 * jj)) & 0xffu));
        }
    };
    // this wave's 32 rows (32 rg ..) and 32 slots (32 t ..); this lane in the 32 x 32 product: operand row / slot lane % 32,
    // its share of the unit's values (lane / 32); result v is row 8 (v / 4) + 4 (lane / 32) + v % 4 of slot lane % 32
    const int rg = wv & 3, t = wv >> 2;
    const int l32 = lane & 31, kh = lane >> 5;
    const uint8_t *my_w = w_codes + (32 * rg + l32) * kStride + kOp * kh;
    const uint8_t *my_a = a_codes + (32 * t + l32) * kStride + kOp * kh;
    const uint2 *my_sv = sv_t + (kh ? kFastRows : 32 * rg + l32); // lanes 32 .. 63: the line's zero
    const uint2 *my_d8 = d8_t + 32 * t + l32;
    const bool live = t == 0 || len > 32; // else this wave's slots are all padding
    v16f acc;
#pragma unroll
    for (int v = 0; v < 16; v++) acc[v] = 0.0f;

    // One super-block's products. A step is a unit: its integer sums (one matrix instruction, issued a step ahead), its
    // scale products (another, issued at the end of the step before, behind that step's last use of the one buffer), and on
    // the vector ALU the sums to floats and the multiply-adds.
    auto blocks = [&]() __attribute__((always_inline)) {
        typedef typename std::conditional<kQ45, v4i, long>::type Operand;
        Operand a[2], b[2];
        uint2 sa[2], sb[2];
        v16i sum[2];
        v16f pr;
        auto rd = [&](int u) {
            a[u & 1] = *reinterpret_cast<const Operand *>(my_w + 2 * kOp * u);
            b[u & 1] = *reinterpret_cast<const Operand *>(my_a + 2 * kOp * u);
            sa[u & 1] = my_sv[u * kFastRowLine];
            sb[u & 1] = my_d8[(kQ45 ? u : u >> 1) * kFastColLine];
        };
        auto product = [&](int u) {
            const v16i z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            if constexpr (kQ45) sum[u & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[u & 1], b[u & 1], z, 0, 0, 0);
            else sum[u & 1] = __builtin_amdgcn_mfma_i32_32x32x16_i8(a[u & 1], b[u & 1], z, 0, 0, 0);
        };
        auto scales = [&](int u) {
            const v16f z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            pr = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(__builtin_bit_cast(v4s, sa[u & 1]), __builtin_bit_cast(v4s, sb[u & 1]), z, 0, 0,
                                                         0);
        };
        rd(0);
        rd(1);
        product(0);
        scales(0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kUnitsSb; u++) {
            if (u + 1 < kUnitsSb) product(u + 1);
            __builtin_amdgcn_sched_barrier(0);
            float f[16];
#pragma unroll
            for (int v = 0; v < 16; v++) f[v] = (float)sum[u & 1][v];
#pragma unroll
            for (int v = 0; v < 16; v++) acc[v] = fmaf(pr[v], f[v], acc[v]);
            __builtin_amdgcn_sched_barrier(0);
            if (u + 1 < kUnitsSb) scales(u + 1);
            // the operands two units on, into the buffers of this unit, whose last instructions have been issued
            if (u + 2 < kUnitsSb) rd(u + 2);
        }
        if constexpr (kQ45) {
            // the min terms last, into the same accumulators: a 32 x 8 by 8 x 32 product in f32, two of the eight
            // sub-blocks an instruction; they run on the matrix cores while the workgroup goes through its barrier and the
            // next staging
#pragma unroll
            for (int j = 0; j < 4; j++)
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(mn_t[(2 * j + kh) * kFastRowLine + 32 * rg + l32],
                                                           my_t[(2 * j + kh) * kFastColLine + 32 * t + l32], acc, 0, 0, 0);
        }
    };

    fetch(0);
    for (int i = 0; i < nb; i++) {
        if (i) __syncthreads(); // the readers of the super-block before are done
        stash();
        __syncthreads();
        if (i + 1 < nb) fetch(i + 1);
        if (live) blocks();
    }
    const int n = 32 * t + l32;
    if (n < len) {
        float *out = y + (size_t)tab->slot[n] * rpe + row0 + 32 * rg + 4 * kh;
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) {
            // rows_per_expert is a multiple of 16 and these four rows start at a multiple of 4: all inside or all outside
            if (row0 + 32 * rg + 4 * kh + 8 * q4 < rpe)
                *reinterpret_cast<float4 *>(out + 8 * q4) = make_float4(acc[4 * q4 + 0], acc[4 * q4 + 1], acc[4 * q4 + 2], acc[4 * q4 + 3]);
        }
    }
}

// ------------------------------------------------------------------------------------- IQ2_XXS on Q8_K columns

// The grouped GEMM for IQ2_XXS stacks (crates/gpu/src/gemm/kernels.rs:867 gemm_iq2xxs; the arithmetic is
// crates/gpu/src/gemm/grouped.rs:33-58 with the CPU path's lanes, crates/qdot/src/lib.rs:8677-8724). A super-block of a
// row against a super-block of a Q8_K column is, in the CPU path, eight accumulators: accumulator l first takes
// (dmin dy) (2 s_l + 1) (bsum[2l] + bsum[2l + 1]), then (d dy) sumi[l] with
//     sumi[l] = sum over the eight sub-blocks b of (2 s_b + 1) * sum over i < 4 of u[b][4l + i] a[b][4l + i],
// u = +-grid + 43 the unsigned code byte. sumi[l] is a 32-term integer dot whose weight-side terms (2 s_b + 1) u are at most
// 31 * 86 = 2666: too wide for an int8 operand, so each is split into two signed bytes, 256 h + lo with lo = the low byte
// read as signed and h = (term + 128) >> 8 (0 .. 10), and the dot is two v_mfma_i32_32x32x32_i8 whose sums meet as
// (H << 8) + L, exactly. The LDS copy of a row's (and a column's) super-block is laid out lane-major, [l][b][i], so a matrix
// operand is 16 consecutive bytes. With EXACT the eight accumulators and their order are the CPU path's, bit for bit (the value
// bm_gemv_sel gives); without it (IQ2_XXS, the tolerance mode's small launches: see gemm below) one accumulator takes d dy times the
// super-block's whole sum sum_b (2 s_b + 1) sum_n (u - 43) a, the 43s taken out in integers through two more matrix instructions over
// the column's 32-value sums (split into two bytes the same way).
// A workgroup of four waves takes 64 rows and a tile's 64 slots, a wave 32 x 32 of them.
constexpr int kIqRows = 64;
constexpr int kIqStride = 256 + 16; // bytes a row's or a column's 256 codes take in LDS
constexpr int kIqLine = 64 + 4;     // floats a line of the per-lane tables
template <int WT, bool EXACT = true>
__host__ __device__ constexpr size_t gemm_iq_lds_bytes() {
    return sizeof(GemmLds) + (size_t)tab_bytes<WT>() + (WT == BM_Q3K ? 2 : 3) * (size_t)64 * kIqStride + 2 * 64 * sizeof(float) +
           (EXACT ? 2 * 8 * kIqLine * sizeof(float) : 3 * 64 * 16);
}

// (2 s + 1) u for the four code bytes of `u`, each product split into the signed low byte (lo) and what is left over 256
// (hi): 256 hi + lo is the product.
__device__ __forceinline__ void iq2_planes(u32 u, u32 sc, u32 &hi, u32 &lo) {
    const u32 even = __builtin_amdgcn_perm(0u, u, 0x0c020c00u), odd = __builtin_amdgcn_perm(0u, u, 0x0c030c01u);
    const u32 pe = even * sc, po = odd * sc; // two 16-bit fields each, at most 2666
    lo = __builtin_amdgcn_perm(po, pe, 0x06020400u);
    hi = __builtin_amdgcn_perm(po + 0x00800080u, pe + 0x00800080u, 0x07030501u);
}

typedef unsigned short v2us __attribute__((ext_vector_type(2)));

// Four bytes, each plus `more`, times a signed scale as two pairs of 16-bit products (bytes 0 and 2, bytes 1 and 3), two products an
// instruction: |product| <= 4064, so sixteen bits hold them.
__device__ __forceinline__ void iq_products(u32 bytes, int more, int sc, v2us &even, v2us &odd) {
    const unsigned short s = (unsigned short)sc, m = (unsigned short)(more * sc);
    const v2us scale = {s, s}, add = {m, m};
    even = __builtin_bit_cast(v2us, __builtin_amdgcn_perm(0u, bytes, 0x0c020c00u)) * scale + add;
    odd = __builtin_bit_cast(v2us, __builtin_amdgcn_perm(0u, bytes, 0x0c030c01u)) * scale + add;
}
// The low bytes of four such products, in the bytes' order.
__device__ __forceinline__ u32 iq_low_bytes(v2us even, v2us odd) {
    return __builtin_amdgcn_perm(__builtin_bit_cast(u32, odd), __builtin_bit_cast(u32, even), 0x06020400u);
}

// The same split for a product of four signed bytes with a signed scale: lo the low byte read as signed, hi what is left over 256.
// (Ten instructions. Byte by byte it took some thirty, and the staging was over half of the kernel's vector work: a layer of 777
// tokens, top-8 of 128 experts of 768 x 2048 IQ4_XS, 428 -> 391 us.)
__device__ __forceinline__ void iq_planes_signed(u32 v, int sc, u32 &hi, u32 &lo) {
    v2us even, odd;
    iq_products(v ^ 0x80808080u, -128, sc, even, odd);
    const v2us half = {128, 128};
    lo = iq_low_bytes(even, odd);
    hi = __builtin_amdgcn_perm(__builtin_bit_cast(u32, odd + half), __builtin_bit_cast(u32, even + half), 0x07030501u);
}

// The types that dot against Q8_K columns (crates/gpu/src/gemm/kernels.rs:867 gemm_iq2xxs, :759 gemm_q3k, :1139 gemm_iq3xxs,
// :1248 gemm_iq4xs). What differs between them is how a row's super-block becomes signed code x scale terms (the staging) and
// the f32 step a super-block; the columns, the lane-major operands, the two byte planes and the products are the same.
//   IQ2_XXS, IQ3_XXS: terms (2 s + 1) (offset + u), offset 43 / 64, the offsets folded out through the column's sums first,
//     eight accumulators, d = f16 / 8 and f16 / 4;
//   IQ4_XS: terms scale x level (scale -32 .. 31, the sixteen levels), eight accumulators, one multiply-add a super-block each
//     (crates/qdot/src/lib.rs:11171-11173);
//   Q3_K: terms scale x (u - 4) over the sixteen 16-value groups, -124 .. 128 and so, negated, one signed byte: one plane and one
//     product instead of two (with the products above: the same layer in Q3_K / Q4_K 367 -> 300 us). One integer a super-block and
//     one accumulator, the float step acc + (dcol d) sum with every operation rounded on its own (crates/qdot/src/lib.rs:2223-2245).
// (EXACT only for the three others: the tolerance mode runs them in this order too.)
template <int WT>
struct IqGemm {
    static constexpr bool kFold = WT == BM_IQ2XXS || WT == BM_IQ3XXS;
    static constexpr int kOff = WT == BM_IQ2XXS ? 43 : 64;
    static constexpr int kLanes = WT == BM_Q3K ? 1 : 8;
    static constexpr int kPlanes = WT == BM_Q3K ? 1 : 2; // signed bytes a weight-side term takes
    static constexpr int kBlock = WT == BM_IQ2XXS ? BM_IQ2XXS_BLOCK : WT == BM_IQ3XXS ? BM_IQ3XXS_BLOCK : WT == BM_IQ4XS ? BM_IQ4XS_BLOCK : BM_Q3K_BLOCK;
};

template <int WT, bool EXACT = true>
__global__ __launch_bounds__(256, 2) void k_gemm_iq(const uint8_t *w, int rpe, int nb, const uint8_t *act, const u32 *cols,
                                                    const u32 *tiles, const u32 *n_tiles, u32 n_units, u32 slot_div,
                                                    u32 n_slots, float *y, const uint8_t *w_second, float *y_second) {
    static_assert(EXACT || WT == BM_IQ2XXS, "the one-accumulator form is IQ2_XXS's");
    using G = IqGemm<WT>;
    extern __shared__ __align__(16) uint8_t lds[];
    GemmLds *tab = reinterpret_cast<GemmLds *>(lds);
    [[maybe_unused]] const Iq2Tables tb = stage_tables<WT>(lds + sizeof(GemmLds));
    uint8_t *a_codes = lds + sizeof(GemmLds) + tab_bytes<WT>();
    uint8_t *w_hi = a_codes + 64 * kIqStride;
    uint8_t *w_lo = w_hi + (G::kPlanes - 1) * 64 * kIqStride; // (the one plane where there is one)
    float *dy_t = reinterpret_cast<float *>(w_lo + 64 * kIqStride); // [slot]
    float *d_t = dy_t + 64;                                          // [row]
    float *bs_t = d_t + 64;                                          // EXACT: [l][slot] the 32-value sums, as floats
    float *sc_t = bs_t + 8 * kIqLine;                                // EXACT: [l][row] the scales 2 s + 1, as floats
    uint8_t *x_sc = reinterpret_cast<uint8_t *>(d_t + 64);           // else: [row][16] the scales as bytes, zeros behind
    uint8_t *x_bl = x_sc + 64 * 16;                                  // [slot][16] the sums' low bytes, zeros behind
    uint8_t *x_bh = x_bl + 64 * 16;                                  // [slot][16] what is left of the sums over 256
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const u32 g = tile_of_block(blockIdx.x, n_units);
    const int row0 = (int)take_stack(slab_of_block(blockIdx.x, n_units), n_units, w, y, w_second, y_second) * kIqRows;
    const u32 count = n_tiles[0];
    if (g > count) return;
    if (g == count) { // the refused slots' rows: NaN (crates/gpu/src/gemm/grouped.rs:2283-2287)
        const u32 refused = n_tiles[1];
        for (u32 i = tid; i < refused * kIqRows; i += 256) {
            const u32 s = cols[n_slots - n_tiles[2] - refused + i / kIqRows];
            const int r = row0 + (int)(i % kIqRows);
            if (r < rpe) y[(size_t)s * rpe + r] = bm_bits_f32(0x7fc00000u);
        }
        return;
    }
    const u32 e = tiles[2 * g], word = tiles[2 * g + 1];
    const int start = (int)(word & 0xffffu), len = (int)(word >> 16);
    if (tid < kGemmBN) {
        const u32 s = cols[start + (tid < len ? tid : 0)];
        tab->slot[tid] = s;
        tab->col[tid] = s / slot_div;
    }
    __syncthreads();
    const u32 row_bytes = (u32)nb * G::kBlock, col_bytes = (u32)nb * BM_Q8K_STRIDE;
    // what this thread stages of every super-block:
    //   four 16-byte pieces of column codes (column tid / 16 + 16 j, piece tid % 16 of the sixteen): values 16 (piece % 2) ..
    //   of sub-block piece / 2, i.e. the four-value groups of lanes 4 (piece % 2) .. + 3, one word each;
    //   threads below 64: column tid's scale and its sixteen 16-value sums;
    //   two sub-blocks of a weight row (row tid / 4, sub-blocks 2 (tid % 4) and the one after), the first of the four
    //   also the row's d
    const int ac = tid >> 4, ap = tid & 15;
    u32 src_a[4];
#pragma unroll
    for (int j = 0; j < 4; j++) src_a[j] = tab->col[ac + 16 * j] * col_bytes + 8u + 16u * (u32)ap;
    const u32 src_c = tab->col[tid & 63] * col_bytes;
    const int wr = tid >> 2, wq = tid & 3;
    const uint8_t *we = w + (size_t)e * rpe * row_bytes;
    const u32 src_w = (u32)(row0 + wr < rpe ? row0 + wr : rpe - 1) * row_bytes;
    const int a_dst = ac * kIqStride + 32 * (4 * (ap & 1)) + 4 * (ap >> 1); // word k of a piece: + 32 k

    // A super-block's bytes are asked for one super-block ahead (fetch_rows, fetch_cols: into registers, behind the staging of
    // the present one and before its products) and unpacked into LDS when their turn comes (stage): the loads' way through memory runs
    // under the matrix work instead of in front of it.
    uint4 ra[4];
    uint4 rq = make_uint4(0, 0, 0, 0), rq2 = rq, rq3 = rq, rq4 = rq;
    uint2 rx = make_uint2(0, 0);
    u32 rd = 0, ra2 = 0;
    float cdy = 0.0f;
    uint4 cb0 = make_uint4(0, 0, 0, 0), cb1 = cb0;
    auto fetch_cols = [&](auto few, int i) {
#pragma unroll
        for (int j = 0; j < (decltype(few)::value ? 2 : 4); j++) __builtin_memcpy(&ra[j], act + (src_a[j] + (u32)i * BM_Q8K_STRIDE), 16);
        if (tid < 64) {
            const uint8_t *cs = act + (src_c + (u32)i * BM_Q8K_STRIDE);
            cdy = *reinterpret_cast<const float *>(cs);
            __builtin_memcpy(&cb0, cs + 264, 16);
            __builtin_memcpy(&cb1, cs + 280, 16);
        }
    };
    auto fetch_rows = [&](int i) {
        const uint8_t *blk = we + (src_w + (u32)i * G::kBlock);
        // the row's two sub-blocks 2 wq and 2 wq + 1, as the type lays them out
        if constexpr (WT == BM_IQ2XXS) {
            rq = bm_ld16u(blk + 2 + 16 * wq);
            rd = bm_ld2u(blk);
        } else if constexpr (WT == BM_IQ3XXS) {
            rq = bm_ld16u(blk + 2 + 16 * wq); // the index bytes of the two sub-blocks
            __builtin_memcpy(&rx, blk + 66 + 8 * wq, 8); // their sign/scale words
            rd = bm_ld2u(blk);
        } else if constexpr (WT == BM_IQ4XS) {
            __builtin_memcpy(&rx, blk, 8); // d | scales_h << 16, scales_l
            rq = bm_ld16u(blk + 8 + 32 * wq);
            rq2 = bm_ld16u(blk + 24 + 32 * wq);
            rd = rx.x & 0xffffu;
        } else { // Q3_K: the 32 field bytes of half wq / 2, the 32 high-bit bytes, the scales and d
            rq = bm_ld16u(blk + 32 + 32 * (wq >> 1));
            rq2 = bm_ld16u(blk + 48 + 32 * (wq >> 1));
            rq3 = bm_ld16u(blk);
            rq4 = bm_ld16u(blk + 16);
            const uint4 tail = bm_ld16u(blk + 94); // the twelve scale bytes at 2 .., d at 14
            rx = make_uint2((tail.x >> 16) | (tail.y << 16), (tail.y >> 16) | (tail.z << 16)); // scale words a0, a1
            ra2 = (tail.z >> 16) | (tail.w << 16);                                             // a2: their high bits
            rd = tail.w >> 16;
        }
    };
    auto stage_cols = [&](auto few) {
#pragma unroll
        for (int j = 0; j < (decltype(few)::value ? 2 : 4); j++) {
            uint8_t *dst = a_codes + a_dst + 16 * j * kIqStride;
            *reinterpret_cast<u32 *>(dst) = ra[j].x;
            *reinterpret_cast<u32 *>(dst + 32) = ra[j].y;
            *reinterpret_cast<u32 *>(dst + 64) = ra[j].z;
            *reinterpret_cast<u32 *>(dst + 96) = ra[j].w;
        }
        if (tid < 64) {
            dy_t[tid] = cdy;
            const u32 bw[8] = {cb0.x, cb0.y, cb0.z, cb0.w, cb1.x, cb1.y, cb1.z, cb1.w};
            [[maybe_unused]] u32 bl[2] = {0, 0}, bh[2] = {0, 0};
#pragma unroll
            for (int l = 0; l < 8; l++) { // the two 16-value sums of sub-block l
                const int bs = (int)(short)(bw[l] & 0xffffu) + (int)(short)(bw[l] >> 16);
                if constexpr (EXACT) {
                    if constexpr (G::kFold) bs_t[l * kIqLine + tid] = (float)bs;
                } else { // 256 hi + lo with lo the low byte read as signed
                    bl[l >> 2] |= ((u32)bs & 0xffu) << (8 * (l & 3));
                    bh[l >> 2] |= ((u32)((bs + 128) >> 8) & 0xffu) << (8 * (l & 3));
                }
            }
            if constexpr (!EXACT) {
                *reinterpret_cast<uint4 *>(x_bl + 16 * tid) = make_uint4(bl[0], bl[1], 0u, 0u);
                *reinterpret_cast<uint4 *>(x_bh + 16 * tid) = make_uint4(bh[0], bh[1], 0u, 0u);
            }
        }
    };
    auto stage_rows = [&]() {
        if (wq == 0) {
            const float dh = bm_half_to_f32((unsigned short)rd);
            d_t[wr] = WT == BM_IQ2XXS ? 0.125f * dh : WT == BM_IQ3XXS ? 0.25f * dh : dh;
        }
        [[maybe_unused]] u32 scs[2] = {0, 0};
#pragma unroll
        for (int e2 = 0; e2 < 2; e2++) {
            const int b = 2 * wq + e2;
            // the four values 4 l .. 4 l + 3 of sub-block b, times the scale, as the two byte planes at lane l's place
            auto put = [&](int l, u32 h, u32 lo) {
                const int at = wr * kIqStride + 32 * l + 4 * b;
                *reinterpret_cast<u32 *>(w_hi + at) = h;
                *reinterpret_cast<u32 *>(w_lo + at) = lo;
            };
            if constexpr (WT == BM_IQ2XXS || WT == BM_IQ3XXS) {
                const u32 aux = WT == BM_IQ2XXS ? (e2 ? rq.w : rq.y) : (e2 ? rx.y : rx.x);
                const u32 sc = 2u * (aux >> 28) + 1u;
                if constexpr (EXACT) sc_t[b * kIqLine + wr] = (float)sc;
                else scs[e2] = sc;
#pragma unroll
                for (int q = 0; q < 4; q++) { // values 8 q .. 8 q + 7: lanes 2 q and 2 q + 1
                    u32 c_lo, c_hi;
                    if constexpr (WT == BM_IQ2XXS) {
                        const u32 idx = e2 ? rq.z : rq.x;
                        bm_iq2_codes(tb, (idx >> (8 * q)) & 0xffu, (aux >> (7 * q)) & 127u, c_lo, c_hi);
                    } else { // index bytes 2 q and 2 q + 1 of the sub-block's eight, sign group q
                        const u32 word = e2 ? ((q & 2) ? rq.w : rq.z) : ((q & 2) ? rq.y : rq.x);
                        const u32 pair = word >> (16 * (q & 1));
                        const uint2 g0 = tb.grid3[pair & 0xffu], g1 = tb.grid3[(pair >> 8) & 0xffu];
                        const uint2 sg = tb.signs[(aux >> (7 * q)) & 127u];
                        c_lo = bm_iq_pick(g0.x, g0.y, sg.x);
                        c_hi = bm_iq_pick(g1.x, g1.y, sg.y);
                    }
                    u32 h0, l0, h1, l1;
                    iq2_planes(c_lo, sc, h0, l0);
                    iq2_planes(c_hi, sc, h1, l1);
                    put(2 * q, h0, l0);
                    put(2 * q + 1, h1, l1);
                }
            } else if constexpr (WT == BM_IQ4XS) {
                // crates/gguf/src/quant.rs:1989-1991: nibble b % 2 of scales_l[b / 2] under bits 2b .. of scales_h, less 32
                const u32 sl = (rx.y >> (8 * wq + 4 * e2)) & 15u, sh = (rx.x >> (16 + 4 * wq + 2 * e2)) & 3u;
                const int sc = (int)(sl | (sh << 4)) - 32;
                const uint4 cw = e2 ? rq2 : rq;
                const u32 qw[4] = {cw.x, cw.y, cw.z, cw.w};
#pragma unroll
                for (int l = 0; l < 4; l++) { // low nibbles: values 4 l ..; high nibbles: values 16 + 4 l ..
                    u32 h, lo;
                    iq_planes_signed(bm_iq4_levels<0>(qw[l]), sc, h, lo);
                    put(l, h, lo);
                    iq_planes_signed(bm_iq4_levels<4>(qw[l]), sc, h, lo);
                    put(4 + l, h, lo);
                }
            } else { // Q3_K: sub-block b = 4 j + f is field f of the half's 32 cells; cell p is value p of the sub-block
                const int j = wq >> 1, f = 2 * (wq & 1) + e2;
                // the sixteen six-bit scales (crates/qdot/src/lib.rs:2162-2174): group 8 j + 2 f + odd
                const u32 lo4 = j ? (rx.x >> 4) : rx.x, lo41 = j ? (rx.y >> 4) : rx.y, hi2 = ra2 >> (4 * j);
                const u32 w0 = (lo4 & 0x0f0f0f0fu) | ((hi2 & 0x03030303u) << 4);
                const u32 w1 = (lo41 & 0x0f0f0f0fu) | (((hi2 >> 2) & 0x03030303u) << 4);
                const u32 sword = (f >> 1) ? w1 : w0;
                const u32 qs[8] = {rq.x, rq.y, rq.z, rq.w, rq2.x, rq2.y, rq2.z, rq2.w};
                const u32 hm[8] = {rq3.x, rq3.y, rq3.z, rq3.w, rq4.x, rq4.y, rq4.z, rq4.w};
#pragma unroll
                for (int t = 0; t < 8; t++) { // cells 4 t .. 4 t + 3: lane t
                    const int sc = (int)((sword >> (8 * (2 * (f & 1) + (t >> 2)))) & 0xffu) - 32;
                    const u32 low = (qs[t] >> (2 * f)) & 0x03030303u, high = (hm[t] >> (4 * j + f)) & 0x01010101u;
                    v2us even, odd;
                    iq_products((high << 2) | low, -4, -sc, even, odd);
                    *reinterpret_cast<u32 *>(w_lo + wr * kIqStride + 32 * t + 4 * b) = iq_low_bytes(even, odd);
                }
            }
        }
        if constexpr (!EXACT) { // the row's eight scales as bytes: the thread of sub-blocks 2 wq, 2 wq + 1 writes its two
            *reinterpret_cast<unsigned short *>(x_sc + 16 * wr + 2 * wq) = (unsigned short)(scs[0] | (scs[1] << 8));
            if (wq == 0) *reinterpret_cast<uint2 *>(x_sc + 16 * wr + 8) = make_uint2(0u, 0u);
        }
    };

    // this lane in its wave's 32 x 32 product: operand row / slot lane % 32, terms 16 (lane / 32) .. of the 32; result v
    // is row 8 (v / 4) + 4 (lane / 32) + v % 4 of slot lane % 32
    const int l32 = lane & 31, kh = lane >> 5;
    const int wrow = 32 * (wv & 1);
    const uint8_t *my_h = w_hi + (wrow + l32) * kIqStride + 16 * kh;
    const uint8_t *my_l = w_lo + (wrow + l32) * kIqStride + 16 * kh;
    const v16i z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    constexpr int kAcc = EXACT ? G::kLanes : 1;
    // A tile of at most 32 slots, where there are eight accumulators a value: a wave takes 32 rows, all the slots and four of the
    // accumulators, and the two waves of a row group meet in the closing sum. (With slots for two of the four waves only, the two SIMDs
    // with those did all the arithmetic: top-8 of 128 experts, us a layer, IQ4_XS 200 tokens 232 -> 205, 777 tokens 387 -> 363;
    // 400 tokens of IQ2_XXS, hidden 3072, 402 -> 361.)
    auto run = [&](auto few) __attribute__((always_inline)) {
    constexpr bool kFew = decltype(few)::value;
    constexpr int kMine = kFew ? kAcc / 2 : kAcc;
    const int wslot = kFew ? 0 : 32 * (wv >> 1);
    const int l0 = kFew ? kMine * __builtin_amdgcn_readfirstlane(wv >> 1) : 0; // the wave's first accumulator
    const uint8_t *my_a = a_codes + (wslot + l32) * kIqStride + 16 * kh;
    const bool live = wslot < len; // else none of this wave's slots is real
    v16f acc[kMine];
#pragma unroll
    for (int l = 0; l < kMine; l++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[l][v] = 0.0f;

    // (the columns' bytes too where the registers allow: the exact forms of the types with eight accumulators a value have few
    // to spare - with everything held over they spilled and ran 6 % slower - so there only the rows' bytes, which come from
    // HBM, are asked for ahead, and the columns', which the cache holds, when their turn comes)
    constexpr bool kColsAhead = kMine <= 4;
    fetch_rows(0);
    if constexpr (kColsAhead) fetch_cols(few, 0);
    for (int i = 0; i < nb; i++) {
        if (i) __syncthreads(); // the readers of the super-block before are done
        if constexpr (!kColsAhead) {
            fetch_cols(few, i);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (WT == BM_Q3K) { // (the other way round one in nine of the launches under 60 us takes 3 to 9 % longer)
            stage_cols(few);
            stage_rows();
        } else {
            stage_rows();
            __builtin_amdgcn_sched_barrier(0);
            stage_cols(few);
        }
        if (i + 1 < nb) {
            fetch_rows(i + 1);
            if constexpr (kColsAhead) fetch_cols(few, i + 1);
        }
        __syncthreads();
        if (!kFew && !live) continue;
        const float dy = dy_t[wslot + l32];
        float dd[16];
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) {
            const float4 d4 = *reinterpret_cast<const float4 *>(d_t + wrow + 8 * q4 + 4 * kh);
            dd[4 * q4 + 0] = d4.x;
            dd[4 * q4 + 1] = d4.y;
            dd[4 * q4 + 2] = d4.z;
            dd[4 * q4 + 3] = d4.w;
        }
        if constexpr (G::kLanes == 1) {
            // Q3_K: one integer a super-block, then acc + (dcol d) sum, each operation rounded on its own
            v16i neg = z;
#pragma unroll
            for (int l = 0; l < 8; l++)
                neg = __builtin_amdgcn_mfma_i32_32x32x32_i8(*reinterpret_cast<const v4i *>(my_l + 32 * l),
                                                            *reinterpret_cast<const v4i *>(my_a + 32 * l), neg, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 16; v++)
                acc[0][v] = __fadd_rn(acc[0][v], __fmul_rn(__fmul_rn(dy, dd[v]), (float)-neg[v]));
        } else if constexpr (!EXACT) {
            v16i hs = z, ls = z;
#pragma unroll
            for (int l = 0; l < 8; l++) {
                const v4i b = *reinterpret_cast<const v4i *>(my_a + 32 * l);
                hs = __builtin_amdgcn_mfma_i32_32x32x32_i8(*reinterpret_cast<const v4i *>(my_h + 32 * l), b, hs, 0, 0, 0);
                ls = __builtin_amdgcn_mfma_i32_32x32x32_i8(*reinterpret_cast<const v4i *>(my_l + 32 * l), b, ls, 0, 0, 0);
            }
            // sum_b (2 s_b + 1) (the sub-block's sum of a): the scales against the sums' two bytes, terms 8 .. 31 zero
            const v4i zero4 = {0, 0, 0, 0};
            const v4i xs = kh ? zero4 : *reinterpret_cast<const v4i *>(x_sc + 16 * (wrow + l32));
            const v4i xl = kh ? zero4 : *reinterpret_cast<const v4i *>(x_bl + 16 * (wslot + l32));
            const v4i xh = kh ? zero4 : *reinterpret_cast<const v4i *>(x_bh + 16 * (wslot + l32));
            const v16i ml = __builtin_amdgcn_mfma_i32_32x32x32_i8(xs, xl, z, 0, 0, 0);
            const v16i mh = __builtin_amdgcn_mfma_i32_32x32x32_i8(xs, xh, z, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int total = ((hs[v] << 8) + ls[v]) - 43 * ((mh[v] << 8) + ml[v]);
                acc[0][v] = fmaf(dd[v] * dy, (float)total, acc[0][v]);
            }
        } else {
            if constexpr (G::kFold) {
                // the fold of the offsets first: accumulator l takes sub-block l's scale on its two sums
                // (crates/qdot/src/lib.rs:8691-8694); the product of the two small integers is exact in f32
#pragma unroll
                for (int l = 0; l < kMine; l++) {
                    const float bs = bs_t[(l0 + l) * kIqLine + wslot + l32];
#pragma unroll
                    for (int q4 = 0; q4 < 4; q4++) {
                        const float4 s4 = *reinterpret_cast<const float4 *>(sc_t + (l0 + l) * kIqLine + wrow + 8 * q4 + 4 * kh);
                        const float sv[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            const float dmin = -dd[4 * q4 + k] * (float)G::kOff;
                            acc[l][4 * q4 + k] = fmaf(dmin * dy, sv[k] * bs, acc[l][4 * q4 + k]);
                        }
                    }
                }
            }
#pragma unroll
            for (int l = 0; l < kMine; l++) {
                const int at = 32 * (l0 + l);
                const v4i b = *reinterpret_cast<const v4i *>(my_a + at);
                const v16i hs = __builtin_amdgcn_mfma_i32_32x32x32_i8(*reinterpret_cast<const v4i *>(my_h + at), b, z, 0, 0, 0);
                const v16i ls = __builtin_amdgcn_mfma_i32_32x32x32_i8(*reinterpret_cast<const v4i *>(my_l + at), b, z, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 16; v++) acc[l][v] = fmaf(dd[v] * dy, (float)(hs[v] * 256 + ls[v]), acc[l][v]);
            }
        }
    }
    // the closing sum of the eight lanes (crates/qdot/src/lib.rs:4128 hsum_float_8's order), four rows a store
    const int n = wslot + l32;
    float *const out = y + (size_t)(live ? tab->slot[wslot + l32] : 0) * rpe + row0 + wrow + 4 * kh;
    auto store = [&](int q4, float r0, float r1, float r2, float r3) {
        // rows_per_expert is a multiple of 16 and these four rows start at a multiple of 4: all inside or all outside
        if (live && n < len && row0 + wrow + 4 * kh + 8 * q4 < rpe) *reinterpret_cast<float4 *>(out + 8 * q4) = make_float4(r0, r1, r2, r3);
    };
    if constexpr (kFew) {
        // a wave closes eight of a lane's sixteen results and has the other wave's accumulators of them through LDS
        __syncthreads();
        float *const swap = reinterpret_cast<float *>(a_codes) + 4096 * (wv & 1) + lane;
        const int h = __builtin_amdgcn_readfirstlane(wv >> 1);
        auto close = [&](auto from) __attribute__((always_inline)) {
            constexpr int mine = decltype(from)::value, other = 8 - mine;
#pragma unroll
            for (int l = 0; l < kMine; l++)
#pragma unroll
                for (int v = 0; v < 8; v++) swap[64 * ((h * kMine + l) * 8 + v)] = acc[l][other + v];
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 2; q++) {
                float r[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    float t[kMine];
#pragma unroll
                    for (int l = 0; l < kMine; l++) t[l] = acc[l][mine + 4 * q + k] + swap[64 * (((1 - h) * kMine + l) * 8 + 4 * q + k)];
                    r[k] = (t[0] + t[2]) + (t[1] + t[3]);
                }
                store(mine / 4 + q, r[0], r[1], r[2], r[3]);
            }
        };
        if (h) close(std::integral_constant<int, 8>{});
        else close(std::integral_constant<int, 0>{});
    } else {
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) {
            float r[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int v = 4 * q4 + k;
                if constexpr (kMine == 8) {
                    const float t0 = acc[0][v] + acc[4][v], t1 = acc[1][v] + acc[5][v];
                    const float t2 = acc[2][v] + acc[6][v], t3 = acc[3][v] + acc[7][v];
                    r[k] = (t0 + t2) + (t1 + t3);
                } else {
                    r[k] = acc[0][v];
                }
            }
            store(q4, r[0], r[1], r[2], r[3]);
        }
    }
    };
    if constexpr (kAcc == 8) {
        if (len <= 32) return run(std::true_type{});
    }
    run(std::false_type{});
}

bool gemm_supported(int wtype) {
    return wtype == BM_Q4K || wtype == BM_Q5K || wtype == BM_Q6K || wtype == BM_IQ2XXS || wtype == BM_IQ3XXS || wtype == BM_IQ4XS ||
           wtype == BM_Q3K;
}

hipError_t gemm(const Launch &L, int wtype, const uint8_t *w, int n_experts, int rows_per_expert, int k,
                const uint8_t *act, const uint32_t *cols, const uint32_t *tiles_dev, const uint32_t *n_tiles, int n_slots,
                int slot_div, float *y, int mode, const uint8_t *w_second, float *y_second) {
    const int nb = k / 256;
    const u32 max_tiles = (u32)gemm_max_tiles(n_slots, n_experts) + 1; // one more: the block that fills refused slots
    const u32 stacks = w_second ? 2 : 1;
    auto launch = [&](auto kern, int threads, int slab_rows, size_t lds, auto... more) {
        hipError_t e = allow_lds(kern, lds);
        if (e != hipSuccess) return e;
        const u32 n_units = stacks * (u32)((rows_per_expert + slab_rows - 1) / slab_rows);
        const unsigned grid = ((max_tiles + 7) / 8) * 8 * n_units;
        hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), lds, L.stream, w, rows_per_expert, nb, act, cols, tiles_dev, n_tiles, n_units,
                           (u32)slot_div, (u32)n_slots, y, more..., w_second, y_second);
        return hipGetLastError();
    };
    if (wtype == BM_IQ3XXS) return launch(k_gemm_iq<BM_IQ3XXS>, 256, kIqRows, gemm_iq_lds_bytes<BM_IQ3XXS>());
    if (wtype == BM_IQ4XS) return launch(k_gemm_iq<BM_IQ4XS>, 256, kIqRows, gemm_iq_lds_bytes<BM_IQ4XS>());
    if (wtype == BM_Q3K) return launch(k_gemm_iq<BM_Q3K>, 256, kIqRows, gemm_iq_lds_bytes<BM_Q3K>());
    if (wtype == BM_IQ2XXS) {
        // The tolerance mode: 512-row workgroups that unpack in registers, one a compute unit, or, where those leave the chip's places
        // empty, the int8 form's 64-row workgroups, a sixth as long each. Tiles go to the eight dies in turn, so what counts is the
        // 64-row workgroups of the fullest die's 32 compute units, here in tiles as ids without a favourite would make them; the
        // line lies at three and a half a unit (the int8 form / the other, us, one stack; 64: k 512 8.3 / 15.1, k 2048 23.7 / 35.9,
        // k 7168 73.6 / 117; 96: 14.0 / 18.2, 38.2 / 45.0, 122 / 144; 112: 17.8 / 20.2, 47.3 / 49.1, 148 / 136; 128 with tiles of at
        // most 32 slots: 15.1 / 15.5, 44.7 / 41.6, 143 / 119; 160: 18.7 / 15.7, 57.2 / 42.5, 183 / 118. Of 3958 random launches the rule is 1.2 %
        // behind the better form on average; so are 104 and 128, 80 is 1.8 %).
        const u32 est_tiles = std::max((u32)std::min(n_experts, n_slots), (u32)n_slots / kGemmBN + (u32)n_experts / 2);
        const u32 die_units = (est_tiles + 7) / 8 * stacks * (u32)((rows_per_expert + kIqRows - 1) / kIqRows);
        if (mode != 0 && die_units > 112u)
            return gemm_iq2_fast(L, w, n_experts, rows_per_expert, k, act, cols, tiles_dev, n_tiles, n_slots, slot_div, y, w_second, y_second);
        if (mode != 0) return launch(k_gemm_iq<BM_IQ2XXS, false>, 256, kIqRows, gemm_iq_lds_bytes<BM_IQ2XXS, false>());
        return launch(k_gemm_iq<BM_IQ2XXS>, 256, kIqRows, gemm_iq_lds_bytes<BM_IQ2XXS>());
    }
    if (mode == 2 && gemm_half_supported(wtype)) { // the f16 form of the tolerance mode, where the type has one
        hipError_t e = gemm_half(L, wtype, w, n_experts, rows_per_expert, k, act, cols, tiles_dev, n_tiles, n_slots, slot_div, y);
        if (e == hipSuccess && w_second)
            e = gemm_half(L, wtype, w_second, n_experts, rows_per_expert, k, act, cols, tiles_dev, n_tiles, n_slots, slot_div, y_second);
        return e;
    }
    if (mode == 1 || mode == 2) {
        if (wtype == BM_Q4K) return launch(k_gemm_fast<BM_Q4K>, kFastThreads, kFastRows, fast_lds_bytes<BM_Q4K>());
        if (wtype == BM_Q5K) return launch(k_gemm_fast<BM_Q5K>, kFastThreads, kFastRows, fast_lds_bytes<BM_Q5K>());
        if (wtype == BM_Q6K) return launch(k_gemm_fast<BM_Q6K>, kFastThreads, kFastRows, fast_lds_bytes<BM_Q6K>());
    }
    // A workgroup's start (tile, columns, first bytes: a chain of trips to memory, 4 to 5 us) costs more than a super-block, so where rows
    // are short it takes several slabs, up to about sixteen super-blocks, and no more than leaves some 2400 workgroups: with fewer the
    // tiles, which differ by half in cost, fill the dies unevenly (top-8 of 128 experts, us a layer, one slab / two / four: down of 2048 rows of
    // 768 Q6_K, 333 tokens 247 / 241 / 247, 2048 tokens 706 / 684 / 680, with six 708; gate and up of 768 rows of 2048 Q4_K, 333 tokens
    // 241 / 248 / 282, 2048 tokens 684 / 681 / 697).
    const u32 n_slabs = (u32)((rows_per_expert + kGemmBM - 1) / kGemmBM), slabs_max = std::min(16u / (u32)nb, stacks * max_tiles * n_slabs / 2400u);
    const u32 slabs = slabs_max < 1u ? 1u : slabs_max < n_slabs ? slabs_max : n_slabs;
    const int run = kGemmBM * (int)slabs;
    if (wtype == BM_Q4K) return launch(k_gemm<BM_Q4K>, 256, run, XLds<BM_Q4K>::kBytes, slabs);
    if (wtype == BM_Q5K) return launch(k_gemm<BM_Q5K>, 256, run, XLds<BM_Q5K>::kBytes, slabs);
    if (wtype == BM_Q6K) return launch(k_gemm<BM_Q6K>, 256, run, XLds<BM_Q6K>::kBytes, slabs);
    return hipErrorInvalidValue;
}

} // namespace bmk
