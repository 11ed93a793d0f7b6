// HIP kernels of the quantized MoE expert matmul for gfx950, decode side, and their launch functions: the
// activation quantizers, the dense gemv, the routed expert chain slot by slot (gate . up . SwiGLU, down, combine),
// its fused forms, and the block-sum verification kernel.
#include "bm_kernels.h"

#include <algorithm>
#include <atomic>

#include "bm_stream.hpp"

namespace bmk {

// Timeline of the two decode launches, in measurement builds only (-DBM_TIMELINE: `make timeline` builds
// libbm_moe_hip_timeline.so, which bench.py --timeline loads; the library proper holds none of this). Thread 0 of
// workgroup b of k_gate_up_x leaves the device's constant-rate counter (100 MHz) in row b at marks 0 .. 4 (start, expert
// id known, token quantized, rows dotted, block of h stored); of k_down_combine in row kTimelineRows / 2 + b at marks
// 0 .. 3 (start, columns in LDS, rows dotted, sum stored) and, taken into registers and stored behind the barrier so that no
// store stands among the loads they time, 4 .. 6 (expert id known, the ring's first super-blocks asked for, columns arrived).
// The last launch of each kernel is what the table holds.
#ifdef BM_TIMELINE
__device__ __forceinline__ unsigned bm_block_linear() { return (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x; }
constexpr int kTimelineRows = 4096;
__device__ unsigned long long g_timeline[kTimelineRows * 8];
#define BM_MARK(base, mark)                                                                                            \
    do {                                                                                                               \
        if (threadIdx.x == 0 && (base) + bm_block_linear() < (unsigned)kTimelineRows)                                  \
            g_timeline[((base) + bm_block_linear()) * 8 + (mark)] = wall_clock64();                                           \
    } while (0)
// BM_TICK keeps the counter in a register once `dep` has arrived (no store among the loads it times); BM_TOCK stores it.
#define BM_TICK(var, dep)                                                                                              \
    unsigned long long var;                                                                                            \
    do {                                                                                                               \
        __asm__ volatile("" ::"v"(dep) : "memory");                                                                    \
        var = wall_clock64();                                                                                          \
    } while (0)
#define BM_TOCK(base, mark, var)                                                                                       \
    do {                                                                                                               \
        if (threadIdx.x == 0 && (base) + bm_block_linear() < (unsigned)kTimelineRows)                                  \
            g_timeline[((base) + bm_block_linear()) * 8 + (mark)] = var;                                                      \
    } while (0)
#else
#define BM_MARK(base, mark)                                                                                            \
    do {                                                                                                               \
    } while (0)
#define BM_TICK(var, dep)                                                                                              \
    do {                                                                                                               \
    } while (0)
#define BM_TOCK(base, mark, var)                                                                                       \
    do {                                                                                                               \
    } while (0)
#endif

// ----------------------------------------------------------------------------------------------- fill

__global__ void k_fill_u32(u32 *dst, u32 value, size_t n) {
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = value;
}

hipError_t fill_u32(const Launch &L, uint32_t *dst, uint32_t value, size_t n) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, L.stream, dst, value, n);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------- quantizers

// x: m columns of k values -> Q8_2_X4 columns. One half wave a 32-value block.
__global__ __launch_bounds__(256) void k_quantize_q82x4(const float *x, int m, int k, uint8_t *act, const u32 *live,
                                                        u32 *fault, u32 layer) {
    // (Numbers of blocks and threads fit 32 bits, as a grid's threads do; a division of 64 bits takes some hundred and fifty instructions.)
    const u32 bpc = (u32)k / 32u, gblk = blockIdx.x * 8u + (threadIdx.x >> 5); // blocks a column
    if (gblk >= (u32)m * bpc) return;
    const int col = (int)(gblk / bpc), blk = (int)(gblk % bpc), lane32 = threadIdx.x & 31;
    if (live && (u32)col >= *live) return; // a device-side column count: the columns past it keep what they held
    const float v = x[(size_t)gblk * 32 + lane32];
    Q82Head hd;
    int s16;
    const int code = q82_block(v, &hd, &s16);
    if (hd.bad && lane32 == 0) bm_raise(fault, layer, kSiteQuantColumn);
    q82_store(act + (size_t)col * (k / 256) * BM_Q82_SB_EXT, k / 256, blk, lane32, code, hd, s16);
}

// x: m columns of k values -> Q8_K columns (crates/qdot/src/lib.rs:1787-1809). A wave a 256-value block.
// sel (optional): column c is read by slots c * spc .. c * spc + spc (at most 64); a column none of whose slots names an expert of the stack
// (served elsewhere, or refused) stays as it stands and raises nothing here: its row of x need not hold anything.
__global__ __launch_bounds__(256) void k_quantize_q8k(const float *x, int m, int k, uint8_t *act, const u32 *live,
                                                      const u32 *sel, u32 spc, u32 n_experts, u32 *fault, u32 layer) {
    const u32 bpc = (u32)k / 256u, gblk = blockIdx.x * 4u + (u32)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (gblk >= (u32)m * bpc) return;
    const u32 col = gblk / bpc, lane = threadIdx.x & 63;
    if (live && col >= *live) return;
    const float4 v = bm_ld4f(x + (size_t)gblk * 256 + 4 * lane); // (asked for beside the ids)
    if (sel && __ballot(lane < spc && sel[(size_t)col * spc + (lane < spc ? lane : 0)] < n_experts) == 0) return;
    q8k_wave_block(v, act + (size_t)gblk * BM_Q8K_STRIDE, (int)lane, fault, layer);
}

// The same columns with eight values a thread, a block a quad of lanes (two 16-byte loads a thread, fewer and fatter
// workgroups): the form for many columns at once, where the launch is bound by its traffic and not by its latency.
__global__ __launch_bounds__(256) void k_quantize_q82x4_wide(const float *x, int m, int k, uint8_t *act, const u32 *live,
                                                             u32 *fault, u32 layer) {
    const u32 i = blockIdx.x * 256u + threadIdx.x, line = (u32)k / 8u;
    if (i >= (u32)m * line) return;
    const int col = (int)(i / line), o = 8 * (int)(i % line);
    const size_t at = (size_t)i * 8;
    if (live && (u32)col >= *live) return;
    const float4 a = *reinterpret_cast<const float4 *>(x + at), b = *reinterpret_cast<const float4 *>(x + at + 4);
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    q82_quad8(v, act + (size_t)col * (k / 256) * BM_Q82_SB_EXT, k / 256, o >> 5, threadIdx.x & 3, fault, layer);
}

// Columns from which on the wide form is launched (and only for 16-byte aligned rows).
constexpr long kWideQuantValues = 1 << 18;

hipError_t quantize(const Launch &L, int wtype, const float *x, int m, int k, uint8_t *act, const uint32_t *live,
                    const uint32_t *sel, uint32_t n_experts, int slots_per_col) {
    if (sel && (!bm_takes_q8k(wtype) || slots_per_col < 1 || slots_per_col > 64)) return hipErrorInvalidValue; // the slot-aware form is the Q8_K quantizer's
    if (!bm_takes_q8k(wtype) && (long)m * k >= kWideQuantValues && ((uintptr_t)x & 15) == 0) {
        const long threads = (long)m * k / 8;
        hipLaunchKernelGGL(k_quantize_q82x4_wide, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, L.stream, x, m, k, act,
                           live, L.fault, L.layer);
        return hipGetLastError();
    }
    if (bm_takes_q8k(wtype)) {
        hipLaunchKernelGGL(k_quantize_q8k, dim3(((unsigned)m * (unsigned)(k / 256) + 3) / 4), dim3(256), 0, L.stream, x, m, k, act,
                           live, sel, (u32)slots_per_col, n_experts, L.fault, L.layer);
    } else {
        const long blocks = (long)m * (k / 32);
        hipLaunchKernelGGL(k_quantize_q82x4, dim3((unsigned)((blocks + 7) / 8)), dim3(256), 0, L.stream, x, m, k, act,
                           live, L.fault, L.layer);
    }
    return hipGetLastError();
}

// Fills the two tables of `m` device Q8_2_X4 columns from their reference bytes (after an upload of those bytes).
__global__ __launch_bounds__(256) void k_q82_tables(uint8_t *act, int m, int nb) {
    const long g = (long)blockIdx.x * 256 + threadIdx.x; // one 16-value group a thread
    if (g >= (long)m * nb * 16) return;
    const int col = (int)(g / (nb * 16)), g16 = (int)(g % (nb * 16)), blk = g16 >> 1, half = g16 & 1;
    uint8_t *c = act + (size_t)col * nb * BM_Q82_SB_EXT;
    const uint8_t *group = c + (size_t)(blk >> 2) * BM_Q82X4_STRIDE;
    const signed char *codes = reinterpret_cast<const signed char *>(group + 16 + 32 * (blk & 3) + 16 * half);
    int s = 0;
    for (int n = 0; n < 16; n++) s += codes[n];
    *reinterpret_cast<int *>(c + (size_t)nb * (BM_Q82_SB_REF + 64) + 4 * g16) = s;
    if (half == 0) {
        const float d8 = bm_bf16_to_f32(*reinterpret_cast<const unsigned short *>(group + 2 * (blk & 3)));
        const int isum = *reinterpret_cast<const short *>(group + 8 + 2 * (blk & 3));
        *reinterpret_cast<float2 *>(c + (size_t)nb * BM_Q82_SB_REF + 8 * blk) = make_float2(d8, __fmul_rn(d8, (float)isum));
    }
}

hipError_t q82_tables(const Launch &L, uint8_t *act, int m, int k) {
    const int nb = k / 256;
    const long n = (long)m * nb * 16;
    hipLaunchKernelGGL(k_q82_tables, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, L.stream, act, m, nb);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------ gemv

// y[row * m_total + col0 + c] = row . column (col0 + c), c < m <= M. A quad a row, 64 rows a workgroup. M = 1 is the
// one-column form of the row dot, which reads a super-block's activation operands a super-block ahead.
// T: the workgroup's threads, T / 4 rows: 256, or 64 for a matrix of so few rows that workgroups of 64 rows would leave most of
// the card idle (768 rows are 12 of them, on 12 of 256 compute units, each streaming its 64 rows through one address unit).
template <int WT, int U, int NB, int M, int T = 256>
__global__ __launch_bounds__(T) void k_gemv(const uint8_t *w, long rows, int nb, const uint8_t *act, int m_total,
                                            int col0, int m, float *y) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, q = tid & 3;
    const long row = (long)blockIdx.x * (T / 4) + (tid >> 2);
    const bool active = row < rows;
    const int n = NB > 0 ? NB : nb;
    const size_t row_bytes = (size_t)n * bm_block_bytes<WT>();
    const int col_bytes = bm_act_col_bytes<WT>(n);
    const uint8_t *wrow = w + (size_t)(active ? row : 0) * row_bytes;
    // the columns' first bytes are asked for in front of the rows (vector loads come back in the order they were asked for:
    // behind the rows' requests the columns would wait for those as well); what a thread's few loads do not cover comes after
    Stage<(T == 64 ? 3 : 2), T, !bm_takes_q8k(WT)> st;
    st.load(act + (size_t)col0 * col_bytes, m * col_bytes);
    Blk<WT> b[U];
    preload<WT, U>(b, wrow, n, q);
    const Iq2Tables tb = stage_tables<WT>(lds, T);
    uint8_t *cols = lds + tab_bytes<WT>();
    st.store(cols, act + (size_t)col0 * col_bytes, m * col_bytes);
    __syncthreads();
    float out[M];
    row_dot<WT, U, NB, M>(b, wrow, cols, col_bytes, m, n, q, tb, out, NoTap{});
    if (q == 0 && active) {
#pragma unroll
        for (int c = 0; c < M; c++)
            if (c < m) y[(size_t)row * m_total + col0 + c] = out[c];
    }
}

// The same product of m > 1 columns where 64 rows a workgroup leave most of the card idle: a wave takes 16 rows and C of the
// columns. What bounds it is a wave's own instruction stream (some 150 instructions a super-block and column, five to six cycles each
// while a SIMD has one wave), so the columns go side by side instead of one after the other; a workgroup's waves, `rgs` row
// groups of `cgs` column groups each, share the staged columns and, through the vector cache, the rows' lines. inv: 256 / cgs rounded
// up, T: the workgroup's threads, at most 512 of one column a wave (with a bound of 1024 Q5_K spilled three registers:
// 2000 rows of 2048, 4 columns 4.8 us, 4.5 without). (Where a column group is not whole, its last columns are skipped.)
template <int WT, int U, int NB, int C>
__global__ __launch_bounds__(C == 1 ? 512 : 1024) void k_gemv_cols(const uint8_t *w, long rows, int nb, const uint8_t *act, int m_total, int col0, int m,
                                                    float *y, int cgs, int rgs, int inv, int T) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, q = tid & 3, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = (wv * inv) >> 8, cg = wv - rg * cgs; // (wv below 16, cgs at most 8: the quotient wv / cgs)
    const int n = NB > 0 ? NB : nb;
    const long row = ((long)blockIdx.x * rgs + rg) * 16 + ((tid & 63) >> 2);
    const bool active = row < rows;
    const size_t row_bytes = (size_t)n * bm_block_bytes<WT>();
    const int col_bytes = bm_act_col_bytes<WT>(n), bytes = m * col_bytes;
    const uint8_t *wrow = w + (size_t)(active ? row : 0) * row_bytes;
    const uint8_t *src = act + (size_t)col0 * col_bytes;
    Stage<2, 256, !bm_takes_q8k(WT)> st; // the columns' first bytes in front of the rows, as k_gemv
    st.load(src, bytes, T);
    Blk<WT> b[U];
    preload<WT, U>(b, wrow, n, q);
    const Iq2Tables tb = stage_tables<WT>(lds, T);
    uint8_t *cols = lds + tab_bytes<WT>();
    st.store(cols, src, bytes, T);
    __syncthreads();
    const int c0 = cg * C, mc = m - c0 < C ? m - c0 : C;
    float out[C];
    row_dot<WT, U, NB, C>(b, wrow, cols + (size_t)c0 * col_bytes, col_bytes, mc, n, q, tb, out, NoTap{});
    if (q == 0 && active) {
#pragma unroll
        for (int c = 0; c < C; c++)
            if (c < mc) y[(size_t)row * m_total + col0 + c0 + c] = out[c];
    }
}

// --------------------------------------------------------------------------- the order of a decode launch

// The workgroups of a launch go to the chip's eight dies in turn, each with an L2 of its own. Where slots share experts the decode
// launches give row block b of every slot (or token) to die b % 8 and, on a die, go through all the slots before the next block: the rows of
// an expert that two slots have are read from memory by the one and found in the L2 by the other, at about the same time. Such a grid's
// first dimension is eight, or eight times something, and its last counts the blocks in eights. With few slots (or more blocks than a
// last dimension holds) the plain order: a slot's blocks one after the other, which are neighbours in memory. So too where the last eight
// blocks are not whole: a token's workgroups without a block leave their dies idle, and even with the dies changing places from token to token
// some compute units get a workgroup more than the others, so that they may be two in a hundred, or eight of a launch that fills the card
// more than once (1024 workgroups of 256 threads; random down launches of 64 slots or more, by dies over plain: none empty 0.98, below two in a
// hundred 0.97, up to eight 0.985, but of the smaller launches one in ten then takes 1.08 to 1.2 times as long, beyond thirty 1.07; IQ4_XS of
// 304 rows, 1536 values, top-3, 34 tokens 12.0 / 22.2 us). (us a layer, plain / by
// dies: top-8 of 128 experts Q4_K / Q6_K 16 tokens 75 / 74.5, 20 tokens 89 / 87.7, Q5_K 21 tokens 100.5 / 98.5, IQ2_XXS of
// 1792, 16 tokens 84.5 / 82.5; Q6_K 6 tokens 56.7 / 57.4, Q5_K of 3072, top-6, 3 tokens 46.6 / 47.1.)
constexpr unsigned kDies = 8, kMaxGridZ = 65535;
constexpr int kMaxGridTokens = 65535; // what the grid's second dimension holds
static inline unsigned eighths(unsigned blocks) { return (blocks + kDies - 1) / kDies; }
static inline bool plain_order(int64_t slots, int tokens, unsigned blocks, int threads = 256) {
    const unsigned none = kDies * eighths(blocks) - blocks;
    return slots < 64 || eighths(blocks) > kMaxGridZ || (int64_t)none * ((int64_t)blocks * tokens * threads >= 1024 * 256 ? 12 : 50) > blocks;
}

// --------------------------------------------------------------------------------- gate . up . SwiGLU

// One workgroup = 32 consecutive rows of one slot; eight lanes a row: a quad on the gate row, a quad on the up row.
// With act_h the 32 values are quantized to one q8_2 block of the slot's down activation in the same launch.
struct GateUpColLate { // the end of k_gate_up's arguments (see bm_kernarg_at)
    float *h;
    uint8_t *act_h;
    GateRule rule;
    u32 *fault;
    u32 layer;
};
struct GateUpColArgs { // k_gate_up's argument block
    const uint8_t *wg, *wu;
    u32 n_experts;
    int nb;
    const uint8_t *act;
    const u32 *sel;
    int rpe, spc_word;
    u32 n_slots;
    GateUpColLate late;
};
static_assert(offsetof(GateUpColArgs, late) == 56, "fourteen words in front of the late arguments");
constexpr unsigned kGateUpGridY = 32768; // slots along the grid's second dimension; the third counts the rest

// The grid: (blocks of 32 rows, slots, slots / kGateUpGridY): no division stands before the workgroup's first request.
// spc_word: slots_per_col, and above bit 24 one more than its log2 where it is a power of two.
template <int WT, int U, int NB, int T = 256, bool WIDE = false>
__global__ __launch_bounds__(T) void k_gate_up(const uint8_t *wg, const uint8_t *wu, u32 n_experts, int nb,
                                                 const uint8_t *act, const u32 *sel, int rpe, int spc_word, u32 n_slots,
                                                 GateUpColLate) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, q = tid & 3, which = (tid >> 2) & 1;
    const int slot = (int)(blockIdx.z * kGateUpGridY + blockIdx.y), rb = (int)blockIdx.x;
    if ((u32)slot >= n_slots) return;
    const int r0 = rb * (T / 8);
    const int r = r0 + (tid >> 3);
    const bool active = r < rpe;
    const u32 id = sel[slot];
    const int n = NB > 0 ? NB : nb;
    const int nb_h = rpe / 256;
    const int col_bytes = bm_act_col_bytes<WT>(n);
    const int spc_shift = (spc_word >> 24) - 1;
    const int token = spc_shift >= 0 ? slot >> spc_shift : slot / (spc_word & 0xffffff);
    const uint8_t *act_col = act + (size_t)token * col_bytes;
    Stage<2, T, !bm_takes_q8k(WT)> st;
    st.load(act_col, col_bytes);
    if (id >= n_experts) { // uniform over the workgroup: no weight is read (crates/gpu/src/kquant/sel.rs:22-28)
        if (id == 0xffffffffu) return; // a slot served elsewhere: nothing written, nothing raised (sel.rs:153-161)
        const GateUpColLate late = bm_kernarg_at<GateUpColLate>(offsetof(GateUpColArgs, late));
        float *const h = bm_global(late.h);
        uint8_t *const act_h = bm_global(late.act_h);
        if (tid == 0) bm_raise(bm_global(late.fault), late.layer, kSiteExpertId);
        if (h && active && (tid & 7) == 0) h[(size_t)slot * rpe + r] = bm_bits_f32(0x7fc00000u);
        if (act_h && tid < T / 8 && r0 + tid < rpe) q82_store(act_h + (size_t)slot * nb_h * BM_Q82_SB_EXT, nb_h, (r0 + tid) >> 5, tid & 31, 0, Q82Head{0x7fc0u, 0, true}, 0);
        return;
    }
    const size_t row_bytes = (size_t)n * bm_block_bytes<WT>();
    const uint8_t *wrow = (which ? wu : wg) + ((size_t)id * rpe + (active ? r : 0)) * row_bytes;
    Blk<WT> b[U];
    // (behind the wait for the id; nothing reads them before the column stands in LDS)
    const GateUpColLate late = bm_kernarg_at<GateUpColLate>(offsetof(GateUpColArgs, late));
    preload<WT, U>(b, wrow, n, q);
    const Iq2Tables tb = stage_tables_as<WT, WIDE, T>(lds);
    uint8_t *col = lds + tab_bytes<WT, WIDE>();
    st.store(col, act_col, col_bytes);
    __syncthreads();
    float *const h = bm_global(late.h);
    uint8_t *const act_h = bm_global(late.act_h);
    u32 *const fault = bm_global(late.fault);
    const u32 layer = late.layer;
    uint8_t *hcol = act_h ? act_h + (size_t)slot * nb_h * BM_Q82_SB_EXT : nullptr;
    float v[1];
    row_dot<WT, U, NB, 1, WIDE>(b, wrow, col, col_bytes, 1, n, q, tb, v, NoTap{});
    const float hv = swiglu_of_pair(v[0], which, late.rule, fault, layer);
    if (h && active && (tid & 7) == 0) h[(size_t)slot * rpe + r] = hv;
    if (act_h) { // rpe is a multiple of 256 here, so every row of the block is live
        float *hbuf = reinterpret_cast<float *>(col + col_bytes);
        if ((tid & 7) == 0) hbuf[tid >> 3] = hv;
        __syncthreads();
        if (tid < T / 8 && r0 + tid < rpe) quantize_h_block(hbuf + (tid & ~31), hcol, nb_h, (r0 + tid) >> 5, tid & 31, fault, layer);
    }
}

// ------------------------------------------------------------------------------------- down: gemv_sel

// Slot s: rows of expert sel[s] against column s. A quad a row, 64 rows a workgroup.
template <int WT, int U, int NB>
__global__ __launch_bounds__(256) void k_gemv_sel(const uint8_t *w, u32 n_experts, int nb, const uint8_t *act,
                                                  const u32 *sel, int rpe, float *y, u32 *fault, u32 layer) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, q = tid & 3;
    const int blocks_per_slot = (rpe + 63) / 64;
    const int slot = blockIdx.x / blocks_per_slot, rb = blockIdx.x % blocks_per_slot;
    const int r = rb * 64 + (tid >> 2);
    const bool active = r < rpe;
    const u32 id = sel[slot];
    const int n = NB > 0 ? NB : nb;
    const int col_bytes = bm_act_col_bytes<WT>(n);
    const uint8_t *act_col = act + (size_t)slot * col_bytes;
    Stage<1, 256, !bm_takes_q8k(WT)> st;
    st.load(act_col, col_bytes);
    if (id >= n_experts) { // the slot's rows stay untouched; a host slot is skipped silently
        if (tid == 0 && rb == 0 && id != 0xffffffffu) bm_raise(fault, layer, kSiteExpertId);
        return;
    }
    const size_t row_bytes = (size_t)n * bm_block_bytes<WT>();
    const uint8_t *wrow = w + ((size_t)id * rpe + (active ? r : 0)) * row_bytes;
    Blk<WT> b[U];
    preload<WT, U>(b, wrow, n, q);
    const Iq2Tables tb = stage_tables<WT>(lds);
    uint8_t *col = lds + tab_bytes<WT>();
    st.store(col, act_col, col_bytes);
    __syncthreads();
    float v[1];
    row_dot<WT, U, NB, 1>(b, wrow, col, col_bytes, 1, n, q, tb, v, NoTap{});
    if (q == 0 && active) y[(size_t)slot * rpe + r] = v[0];
}

// --------------------------------------------------------------------------------------------- combine

// crates/gpu/src/arch/qwen3moe/experts.rs:293-318 with crates/gpu/src/elem.rs:658-697: one thread a value.
// With a shared expert's rows: (sum + shexp) + resid, grouped as the reference groups its two adds
// (crates/gpu/src/moe_fused.rs:129-170 moe_combine).
// `sel` (optional): a slot whose id is at or past n_experts adds nothing, as in the fused down + combine launch.
// Bound by latency (a few tokens), then by memory: 4096 tokens x 8 slots x 2048 values read at 5.6 TB/s. So a batch of N slots, then the rest by
// halves: the ids, the weights and behind them the rows are asked for together, where a walk from slot to slot waits for an id and a row N
// times over; the rows that join the sum at its end are asked for first. Thread numbers are of 32 bits, as a grid's threads
// are (a division of 64 bits takes some hundred and fifty instructions). us a launch, 8 slots x 2048 values: 64 tokens 7.3 -> 4.8, 333 tokens
// 8.0 -> 6.0.
template <int N, int W>
__device__ __forceinline__ void combine_slots(const float *down, const float *w, const u32 *sel, u32 n_experts, size_t slot, int n, int rows, u32 d,
                                              float (&acc)[W]) {
    if constexpr (N > 0) {
        for (; n >= N; n -= N, slot += N) {
            u32 id[N];
            float we[N], v[N][W];
#pragma unroll
            for (int e = 0; e < N; e++) {
                id[e] = sel ? sel[slot + e] : 0u;
                we[e] = w[slot + e];
            }
#pragma unroll
            for (int e = 0; e < N; e++)
                if (!sel || id[e] < n_experts) __builtin_memcpy(v[e], __builtin_assume_aligned(down + (slot + e) * rows + d, 4 * W), 4 * W);
#pragma unroll
            for (int e = 0; e < N; e++)
                if (!sel || id[e] < n_experts) {
#pragma unroll
                    for (int k = 0; k < W; k++) acc[k] = fmaf(we[e], v[e][k], acc[k]);
                }
            if (N < 8) return combine_slots<N / 2, W>(down, w, sel, n_experts, slot + N, n - N, rows, d, acc);
        }
        combine_slots<N / 2, W>(down, w, sel, n_experts, slot, n, rows, d, acc);
    }
}
template <int W>
__device__ __forceinline__ void combine_at(const float *down, const float *w, const float *shexp, const float *resid, int rows, int n_slots, int m,
                                           float *y, const u32 *sel, u32 n_experts) {
    const u32 i = blockIdx.x * 256u + threadIdx.x, line = (u32)rows / W; // (the launcher's 256 threads: blockDim.x is a load from memory)
    const u32 t = i / line, d = W * (i % line);
    if (t >= (u32)m) return;
    const size_t at = (size_t)i * W;
    float acc[W], shared[W], before[W];
    if (shexp) __builtin_memcpy(shared, __builtin_assume_aligned(shexp + at, 4 * W), 4 * W);
    if (resid) __builtin_memcpy(before, __builtin_assume_aligned(resid + at, 4 * W), 4 * W);
#pragma unroll
    for (int k = 0; k < W; k++) acc[k] = 0.0f;
    combine_slots<8, W>(down, w, sel, n_experts, (size_t)t * n_slots, n_slots, rows, d, acc);
#pragma unroll
    for (int k = 0; k < W; k++) {
        if (shexp) acc[k] = __fadd_rn(acc[k], shared[k]);
        if (resid) acc[k] = __fadd_rn(acc[k], before[k]);
    }
    __builtin_memcpy(__builtin_assume_aligned(y + at, 4 * W), acc, 4 * W);
}
__global__ __launch_bounds__(256) void k_combine(const float *down, const float *w, const float *shexp, const float *resid,
                                                 int rows, int n_slots, int m, float *y, const u32 *sel, u32 n_experts) {
    combine_at<1>(down, w, shexp, resid, rows, n_slots, m, y, sel, n_experts);
}
__global__ __launch_bounds__(256) void k_combine4(const float *down, const float *w, const float *shexp, const float *resid,
                                                  int rows, int n_slots, int m, float *y, const u32 *sel, u32 n_experts) {
    combine_at<4>(down, w, shexp, resid, rows, n_slots, m, y, sel, n_experts);
}

hipError_t combine_tokens(const Launch &L, const float *down, const float *w, const float *shexp, const float *resid,
                          int rows, int n_slots, int m, float *y, const uint32_t *sel, uint32_t n_experts) {
    const long n = (long)rows * m;
    const uintptr_t align = (uintptr_t)down | (uintptr_t)shexp | (uintptr_t)resid | (uintptr_t)y;
    if (n >= (1 << 18) && rows % 4 == 0 && (align & 15) == 0) {
        hipLaunchKernelGGL(k_combine4, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, L.stream, down, w, shexp, resid, rows,
                           n_slots, m, y, sel, n_experts);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_combine, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, L.stream, down, w, shexp, resid, rows,
                       n_slots, m, y, sel, n_experts);
    return hipGetLastError();
}

struct DownLate { // the end of k_down_combine's arguments
    float *y;
    u32 *fault;
    u32 layer;
};
struct DownArgs { // k_down_combine's argument block
    const uint8_t *w;
    u32 n_experts;
    int nb;
    const uint8_t *act;
    const u32 *sel;
    const float *wts, *resid;
    int spt_word, rpe;
    DownLate late;
};
struct GateUpLate { // the end of k_gate_up_x's arguments
    uint8_t *act_x, *act_h;
    float *h;
    GateRule rule;
    u32 *fault;
    u32 layer;
};
struct GateUpArgs { // k_gate_up_x's argument block
    const float *x;
    const uint8_t *wg, *wu;
    u32 n_experts;
    int nba, nh;
    const u32 *sel;
    int spt;
    GateUpLate late;
};
static_assert(offsetof(DownArgs, late) == 56 && offsetof(GateUpArgs, late) == 56, "fourteen words in front of the late arguments");

// --------------------------------------------------------------------------- down + combine in one launch

// A row's closing sum over its token's slots in slot order, acc = fma(w_s, v_s, acc) for the live slots, then the
// residual (crates/gpu/src/arch/qwen3moe/experts.rs:293-318). v, w and ids lie in LDS. With eight slots every operand is
// read before the first multiply-add (six 16-byte reads in flight at once); a loop that reads as it goes pays an LDS
// round trip a slot, 0.4 us at the end of the launch.
__device__ __forceinline__ float slot_sum(const float *v, const float *w, const u32 *ids, int spt, u32 n_experts,
                                          float resid_v, bool with_resid) {
    float acc = 0.0f;
    if (spt == 8) {
        const float4 v0 = *reinterpret_cast<const float4 *>(v), v1 = *reinterpret_cast<const float4 *>(v + 4);
        const float4 w0 = *reinterpret_cast<const float4 *>(w), w1 = *reinterpret_cast<const float4 *>(w + 4);
        const uint4 i0 = *reinterpret_cast<const uint4 *>(ids), i1 = *reinterpret_cast<const uint4 *>(ids + 4);
        acc = i0.x < n_experts ? fmaf(w0.x, v0.x, acc) : acc;
        acc = i0.y < n_experts ? fmaf(w0.y, v0.y, acc) : acc;
        acc = i0.z < n_experts ? fmaf(w0.z, v0.z, acc) : acc;
        acc = i0.w < n_experts ? fmaf(w0.w, v0.w, acc) : acc;
        acc = i1.x < n_experts ? fmaf(w1.x, v1.x, acc) : acc;
        acc = i1.y < n_experts ? fmaf(w1.y, v1.y, acc) : acc;
        acc = i1.z < n_experts ? fmaf(w1.z, v1.z, acc) : acc;
        acc = i1.w < n_experts ? fmaf(w1.w, v1.w, acc) : acc;
    } else {
        for (int s = 0; s < spt; s++)
            if (ids[s] < n_experts) acc = fmaf(w[s], v[s], acc);
    }
    return with_resid ? __fadd_rn(acc, resid_v) : acc;
}

// Bytes between two slots' Q8_K columns in LDS beside the columns themselves. The IQ types with tables read a column 64 bytes a lane of the quad (four
// lanes' eight bytes in every step), the quads of a wave as many columns as there are slots: columns an odd multiple of eight bytes apart fall on
// banks of their own, columns of eight super-blocks, a multiple of 64 bytes, all on the same ones. (k_down_combine of IQ2_XXS without / with it, us: 2816
// rows of 2048, 8 slots, 5 tokens 31.1 / 20.7; 7168 rows of 2048, 12 slots, 5 tokens 114 / 87; k_down_combine_hq of such rows 0.98 times its time, without it up to
// 1.18 times what it took before a lane held whole sub-blocks.) Up to 32 slots: the entries answer for 4096 bytes of LDS beside the columns.
__host__ __device__ constexpr int slot_col_pad(int wt, int nb, int spt) { return (wt == BM_IQ2XXS || wt == BM_IQ3XXS) && nb % 2 == 0 && spt <= 32 ? 8 : 0; }

// The shared body of the down + combine workgroup: token t, output rows rb * D .. + D with D = 64 / spt, a quad for
// every (row, slot).
template <int WT, int U, int NB, bool EIGHT = false>
__device__ __forceinline__ void down_combine_body(uint8_t *lds, const uint8_t *w, u32 n_experts, int nb,
                                                  const uint8_t *act, const u32 *sel, const float *wts,
                                                  const float *resid, int spt, int rpe, int t, int rb, int spt_shift = -1) {
    const int tid = threadIdx.x, q = tid & 3, quad = tid >> 2;
    BM_MARK(2048, 0);
    if constexpr (EIGHT) spt = 8, spt_shift = 3; // what the launcher has checked: constants from here on
    // (spt_shift: log2 of a power-of-two spt, else -1: the divisions by a count only known at run time are some eighty
    // instructions at the head of a workgroup whose first request waits for them)
    const int D = spt_shift >= 0 ? 64 >> spt_shift : 64 / spt;
    const int e = spt_shift >= 0 ? quad & (spt - 1) : quad % spt, dl = spt_shift >= 0 ? quad >> spt_shift : quad / spt;
    const int r = rb * D + dl;
    const int slot = t * spt + e;
    // eight slots a token: the token's ids through the scalar cache (one request a wave, a shorter way than a vector load's);
    // the lane picks its own out of the eight registers further down, behind the vector requests that do not wait for it
    constexpr bool eight = EIGHT; // (a variant of its own: a run-time choice leaves the id's register waiting for either way's load)
    u32 i8[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    u32 id = 0;
    if constexpr (eight) {
        const u32 *s8 = sel + (size_t)t * 8;
#pragma unroll
        for (int k = 0; k < 8; k++) i8[k] = s8[k];
    } else {
        id = sel[slot];
    }
    // the token's ids and weights for the closing sum, requested now and parked in LDS
    const int si = tid < spt ? tid : 0;
    const u32 my_sel = sel[t * spt + si];
    const float my_w = wts[t * spt + si];
    // the residual value of the row this thread closes, asked for now: at the end it would be a memory round trip
    const float resid_v = resid && tid < D && rb * D + tid < rpe ? resid[(size_t)t * rpe + rb * D + tid] : 0.0f;
    const int n = NB > 0 ? NB : nb;
    const size_t row_bytes = (size_t)n * bm_block_bytes<WT>();
    const int col_bytes = bm_act_col_bytes<WT>(n), pad = slot_col_pad(WT, n, spt), col_stride = col_bytes + pad;
    const uint8_t *act_cols = act + (size_t)t * spt * col_bytes;
    // the token's columns are asked for before anything waits for the expert id: they arrive with it
    StageWords<5> st;
    st.load(act_cols, spt * col_bytes);
    if constexpr (eight) {
        __builtin_amdgcn_sched_barrier(0);
        const u32 a = (e & 1) ? i8[1] : i8[0], b2 = (e & 1) ? i8[3] : i8[2], c = (e & 1) ? i8[5] : i8[4], d = (e & 1) ? i8[7] : i8[6];
        const u32 ab = (e & 2) ? b2 : a, cd = (e & 2) ? d : c;
        id = (e & 4) ? cd : ab;
    }
    const bool live = id < n_experts;
    const bool active = dl < D && r < rpe && live;
    const uint8_t *wrow = w + ((size_t)(live ? id : 0) * rpe + (active ? r : 0)) * row_bytes;
    const Iq2Tables tb = stage_tables<WT>(lds);
    uint8_t *cols = lds + tab_bytes<WT>();
    float *part = reinterpret_cast<float *>(cols + (size_t)spt * col_stride); // [D][spt]
    float *s_w = part + D * spt;                                              // [spt]
    u32 *s_sel = reinterpret_cast<u32 *>(s_w + spt);                          // [spt]
    Blk<WT> b[U];
    BM_TICK(t_id, id);
    // behind the wait for the ids, and nothing reads them before the barrier: their way through memory runs under the columns'
    __builtin_amdgcn_sched_barrier(0);
    const DownLate late = bm_kernarg_at<DownLate>(offsetof(DownArgs, late));
    preload<WT, U>(b, wrow, n, q);
    BM_TICK(t_asked, tid);
    BM_TICK(t_cols, st.v[4].x);
    if constexpr (slot_col_pad(WT, 2, 1) != 0) st.store_apart(cols, act_cols, spt * col_bytes, col_bytes, pad);
    else st.store(cols, act_cols, spt * col_bytes);
    if (tid < spt) {
        s_w[tid] = my_w;
        s_sel[tid] = my_sel;
    }
    __syncthreads();
    float *y = bm_global(late.y);
    if (!live && id != 0xffffffffu && rb == 0 && dl == 0 && q == 0) bm_raise(bm_global(late.fault), late.layer, kSiteExpertId);
    BM_MARK(2048, 1);
    BM_TOCK(2048, 4, t_id);
    BM_TOCK(2048, 5, t_asked);
    BM_TOCK(2048, 6, t_cols);
    float v[1];
    row_dot<WT, U, NB, 1>(b, wrow, cols + (size_t)e * col_stride, col_stride, 1, n, q, tb, v, NoTap{});
    BM_MARK(2048, 2);
    if (q == 0 && dl < D) part[dl * spt + e] = v[0];
    __syncthreads();
    if (tid < D && rb * D + tid < rpe) y[(size_t)t * rpe + rb * D + tid] = slot_sum(part + tid * spt, s_w, s_sel, spt, n_experts, resid_v, resid != nullptr);
    BM_MARK(2048, 3);
}

constexpr int kDownRowMajor = 1 << 30;
template <int WT, int U, int NB, bool EIGHT>
__global__ __launch_bounds__(256) void k_down_combine(const uint8_t *w, u32 n_experts, int nb, const uint8_t *act,
                                                      const u32 *sel, const float *wts, const float *resid, int spt_word,
                                                      int rpe, DownLate) {
    extern __shared__ __align__(16) uint8_t lds[];
    // the grid: (dies, tokens, row blocks of a token in eights). spt_word: the slot count, and above bit 16 one more than its log2
    // where it is a power of two - one word, so that both stand among the first fourteen argument words, which are in registers when
    // the wave starts (an argument behind them is a load from memory in front of the workgroup's first request); bit 30: row blocks in
    // the first dimension
    const int rb = (int)(spt_word & kDownRowMajor ? blockIdx.x : blockIdx.z * kDies + blockIdx.x);
    const int spt = spt_word & 0xffff, shift = ((spt_word >> 16) & 0xff) - 1;
    if (rb * (EIGHT ? 8 : shift >= 0 ? 64 >> shift : 64 / spt) >= rpe) return; // (the last eight of blocks need not be whole)
    down_combine_body<WT, U, NB, EIGHT>(lds, w, n_experts, nb, act, sel, wts, resid, spt, rpe, (int)blockIdx.y, rb, shift);
}

// k_down_combine for a Q6_K stack of NB super-blocks a row with the row's super-blocks dealt to the waves (BM_DOWN_SPLIT, the
// measured alternative: 5.6 us against the ring's 5.2 at the headline shape): a workgroup of 256 NB threads, the same 64
// (row, slot) pairs as k_down_combine's, wave w super-block w % NB of quads 16 (w / NB) .. + 16. Under the ring one wave a SIMD
// runs its loads, its wait and its arithmetic one after the other; here every super-block of every row is asked for at once by
// a wave of its own and NB waves a SIMD overlap. What it shows: the launch is bound by how fast a compute unit's address unit
// takes the quads' scattered 16-byte requests, not by waves to overlap - the twelve waves' requests queue for it, the first
// barrier (every wave's requests issued) comes 2.3 us after the start against 1.9, and the shorter arithmetic behind it (0.95
// us against 1.4) does not win that back. The numbers are the same:
// a wave leaves the operands of its super-block's multiply-adds (the f32 scale product and the integer sum as a float, two
// halves by two accumulators a lane) in LDS, and the wave of the last super-block runs the chain in the CPU path's order,
// super-block by super-block, then closes the quad as bm_quad_finish does.
template <int NB>
__global__ __launch_bounds__(256 * NB) void k_down_combine_q6k_split(const uint8_t *w, u32 n_experts, const uint8_t *act,
                                                                     const u32 *sel, const float *wts, const float *resid,
                                                                     int spt, int rpe, float *y, u32 *fault, u32 layer) {
    extern __shared__ __align__(16) uint8_t lds[];
    constexpr int WT = BM_Q6K;
    const int tid = threadIdx.x, q = tid & 3, wave = tid >> 6;
    BM_MARK(2048, 0);
    const int i = wave % NB, quad = 16 * (wave / NB) + ((tid & 63) >> 2);
    const int D = 64 / spt;
    const int blocks_per_token = (rpe + D - 1) / D;
    const int t = blockIdx.x / blocks_per_token, rb = blockIdx.x % blocks_per_token;
    const int e = quad % spt, dl = quad / spt;
    const int r = rb * D + dl;
    const u32 id = sel[t * spt + e];
    const int si = tid < spt ? tid : 0;
    const u32 my_sel = sel[t * spt + si];
    const float my_w = wts[t * spt + si];
    const bool live = id < n_experts;
    const bool active = dl < D && r < rpe && live;
    const float resid_v = resid && tid < D && rb * D + tid < rpe ? resid[(size_t)t * rpe + rb * D + tid] : 0.0f;
    constexpr size_t row_bytes = (size_t)NB * BM_Q6K_BLOCK;
    constexpr int col_bytes = bm_act_col_bytes<WT>(NB);
    const uint8_t *act_cols = act + (size_t)t * spt * col_bytes;
    StageWords<2, 256 * NB> st; // 16 bytes a thread of 768: the eight columns of 1248 bytes
    st.load(act_cols, spt * col_bytes);
    if (!live && id != 0xffffffffu && rb == 0 && dl == 0 && q == 0 && i == 0) bm_raise(fault, layer, kSiteExpertId);
    const uint8_t *wrow = w + ((size_t)(live ? id : 0) * rpe + (active ? r : 0)) * row_bytes;
    uint8_t *cols = lds;
    float *terms = reinterpret_cast<float *>(cols + (size_t)spt * col_bytes); // [64 quads][NB - 1][4 lanes][8]
    float *part = terms + 64 * (NB - 1) * 32;                                  // [D][spt]
    float *s_w = part + D * spt;                                               // [spt]
    u32 *s_sel = reinterpret_cast<u32 *>(s_w + spt);                           // [spt]
    BM_TICK(t_id, id);
    const Blk<WT> b = bm_load_blk<WT>(wrow, i, q);
    BM_TICK(t_asked, tid);
    st.store(cols, act_cols, spt * col_bytes);
    if (tid < spt) {
        s_w[tid] = my_w;
        s_sel[tid] = my_sel;
    }
    __syncthreads();
    BM_MARK(2048, 1);
    BM_TOCK(2048, 4, t_id);
    BM_TOCK(2048, 5, t_asked);
    const int c = q & 1, h = q >> 1;
    const Act<WT> a = bm_act_q6k(bm_act_view<WT>(cols + (size_t)e * col_bytes, NB), i, c, h);
    float p[4], s[4]; // (half 0: accumulator 0, accumulator 1), (half 1: ...)
    bm_q6k_terms(b, a, c, h, p, s);
    BM_TICK(t_terms, p[3]);
    float *mine = terms + ((size_t)(quad * (NB - 1) + i) * 4 + q) * 8;
    if (i < NB - 1) {
        *reinterpret_cast<float4 *>(mine) = make_float4(p[0], s[0], p[1], s[1]);
        *reinterpret_cast<float4 *>(mine + 4) = make_float4(p[2], s[2], p[3], s[3]);
    }
    __syncthreads();
    BM_MARK(2048, 2);
    BM_TOCK(2048, 6, t_terms);
    if (i == NB - 1) {
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int u = 0; u < NB - 1; u++) {
            const float *o = terms + ((size_t)(quad * (NB - 1) + u) * 4 + q) * 8;
            const float4 lo = *reinterpret_cast<const float4 *>(o), hi = *reinterpret_cast<const float4 *>(o + 4);
            a0 = fmaf(lo.x, lo.y, a0), a1 = fmaf(lo.z, lo.w, a1);
            a0 = fmaf(hi.x, hi.y, a0), a1 = fmaf(hi.z, hi.w, a1);
        }
        a0 = fmaf(p[0], s[0], a0), a1 = fmaf(p[1], s[1], a1);
        a0 = fmaf(p[2], s[2], a0), a1 = fmaf(p[3], s[3], a1);
        const float v = bm_quad_finish<WT>(a0, a1);
        if (q == 0 && dl < D) part[dl * spt + e] = v;
    }
    __syncthreads();
    if (tid < D && rb * D + tid < rpe) y[(size_t)t * rpe + rb * D + tid] = slot_sum(part + tid * spt, s_w, s_sel, spt, n_experts, resid_v, resid != nullptr);
    BM_MARK(2048, 3);
}

// The gate . up . SwiGLU workgroup of the fused step: as k_gate_up's, except that it quantizes its token's f32 row
// itself (into LDS; no quantizer launch, no activation column in memory) and always writes its q8_2 block of the
// slot's down activation.
template <int WA, int UA, int NBA>
__device__ __forceinline__ void gate_up_x_body(uint8_t *lds, const float *x, const uint8_t *wg, const uint8_t *wu,
                                               u32 n_experts, int na, int nh, const u32 *sel, int spt, int slot, int rb, int t) {
    const int tid = threadIdx.x, q = tid & 3, which = (tid >> 2) & 1;
    BM_MARK(0, 0);
    const int hidden = na * 256, ff = nh * 256;
    const int r = rb * 32 + (tid >> 3);
    const u32 id = sel[slot];
    const int col_bytes = bm_act_col_bytes<WA>(na);
    uint8_t *col = lds;
    // the token's row: eight consecutive values a lane, 2048 a pass. Asked for before anything reads an argument that is
    // not in a register when the wave starts (the first thirteen words are): scalar loads come back in any order, so the
    // first wait for one of them is a wait for the expert id as well, and the row's loads would stand behind it
    constexpr int kPasses = NBA > 0 ? (NBA * 256 + 2047) / 2048 : 1;
    float xv[kPasses][8];
#pragma unroll
    for (int p = 0; p < kPasses; p++) {
        int o = p * 2048 + tid * 8;
        o = o < hidden ? o : hidden - 8;
        const float4 lo = *reinterpret_cast<const float4 *>(x + (size_t)t * hidden + o);
        const float4 hi = *reinterpret_cast<const float4 *>(x + (size_t)t * hidden + o + 4);
        xv[p][0] = lo.x, xv[p][1] = lo.y, xv[p][2] = lo.z, xv[p][3] = lo.w;
        xv[p][4] = hi.x, xv[p][5] = hi.y, xv[p][6] = hi.z, xv[p][7] = hi.w;
    }
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (id >= n_experts) { // uniform over the workgroup
        if (id == 0xffffffffu) return; // a slot served elsewhere: nothing written, nothing raised
        const GateUpLate late = bm_kernarg_at<GateUpLate>(offsetof(GateUpArgs, late));
        if (tid == 0) bm_raise(bm_global(late.fault), late.layer, kSiteExpertId);
        if (late.h && (tid & 7) == 0) bm_global(late.h)[(size_t)slot * ff + r] = bm_bits_f32(0x7fc00000u);
        if (late.act_h && tid < 32)
            q82_store(bm_global(late.act_h) + (size_t)slot * nh * BM_Q82_SB_EXT, nh, rb, tid, 0, Q82Head{0x7fc0u, 0, true}, 0);
        return;
    }
    BM_MARK(0, 1);
    const size_t row_bytes = (size_t)na * bm_block_bytes<WA>();
    const uint8_t *wrow = (which ? wu : wg) + ((size_t)id * ff + r) * row_bytes;
    Blk<WA> b[UA];
    // behind the wait for the id, and nothing reads them before the token's column stands in LDS: their way through memory runs
    // under the quantizer's work
    const GateUpLate late = bm_kernarg_at<GateUpLate>(offsetof(GateUpArgs, late));
    preload<WA, UA>(b, wrow, na, q);
    bool bad = false;
#pragma unroll
    for (int p = 0; p < kPasses; p++) {
        const int o = p * 2048 + tid * 8;
        if (o < hidden) bad |= q82_quad8<false>(xv[p], col, na, o >> 5, tid & 3, nullptr, 0);
    }
    if constexpr (NBA == 0) { // longer rows: the passes past the first, straight from memory
        for (int o = 2048 + tid * 8; o < hidden; o += 2048) {
            float v8[8];
            for (int k = 0; k < 8; k++) v8[k] = x[(size_t)t * hidden + o + k];
            bad |= q82_quad8<false>(v8, col, na, o >> 5, tid & 3, nullptr, 0);
        }
    }
    __syncthreads();
    uint8_t *const act_x = bm_global(late.act_x), *const act_h = bm_global(late.act_h);
    float *const h = bm_global(late.h);
    const GateRule rule = late.rule;
    u32 *const fault = bm_global(late.fault);
    const u32 layer = late.layer;
    uint8_t *hcol = act_h ? act_h + (size_t)slot * nh * BM_Q82_SB_EXT : nullptr; // none: the down stack takes Q8_K columns
    if (bad && (tid & 3) == 0) bm_raise(fault, layer, kSiteQuantColumn);
    if (act_x && rb == 0 && slot % spt == 0) stage_bytes(act_x + (size_t)t * col_bytes, col, col_bytes);
    BM_MARK(0, 2);
    float v[1];
    row_dot<WA, UA, NBA, 1>(b, wrow, col, col_bytes, 1, na, q, Iq2Tables{}, v, NoTap{});
    BM_MARK(0, 3);
    const float hv = swiglu_of_pair(v[0], which, rule, fault, layer);
    if (h && (tid & 7) == 0) h[(size_t)slot * ff + r] = hv;
    if (!hcol) return;
    float *hbuf = reinterpret_cast<float *>(col + col_bytes);
    if ((tid & 7) == 0) hbuf[tid >> 3] = hv;
    __syncthreads();
    if (tid < 32) quantize_h_block(hbuf, hcol, nh, rb, tid, fault, layer);
    BM_MARK(0, 4);
}

constexpr int kGateRowMajor = 1 << 30;
// The first half of the fused step as a launch of its own: x -> quantized h, slot by slot.
template <int WA, int UA, int NBA>
__global__ __launch_bounds__(256) void k_gate_up_x(const float *x, const uint8_t *wg, const uint8_t *wu, u32 n_experts,
                                                   int nba, int nh, const u32 *sel, int spt, GateUpLate) {
    extern __shared__ __align__(16) uint8_t lds[];
    // the grid: (dies x slots of a token, tokens, blocks of 32 rows in eights; a slot has 8 nh blocks): no division stands before the
    // workgroup's first request (and no read of the grid's size, which comes from the dispatch packet in memory: spt is an argument, in
    // a register at the start). Bit 30 of spt: (blocks, slots of a token, tokens) instead
    const int slots = spt & ~kGateRowMajor;
    const bool row_major = (spt & kGateRowMajor) != 0;
    const int t = (int)(row_major ? blockIdx.z : blockIdx.y), e = (int)(row_major ? blockIdx.y : blockIdx.x / kDies);
    const int rb = (int)(row_major ? blockIdx.x : blockIdx.z * kDies + blockIdx.x % kDies);
    gate_up_x_body<WA, UA, NBA>(lds, x, wg, wu, n_experts, NBA > 0 ? NBA : nba, nh, sel, slots, t * slots + e, rb, t);
}

// ------------------------------------------------------------- the fused step for the types that take Q8_K columns

// `cols` columns of nb blocks each, f32 rows at x (column c at x + c * nb * 256), into LDS at `dst` by the workgroup's
// waves, block by block. In two steps, as Q82Cols below: a wave's first kAhead blocks are requested in front of the weight rows (memory
// answers in order: asked for behind them, the quantizer began when the rows were there), and encoded while those are on their way. (us a
// launch: 5 tokens x 8 slots of 768 values, IQ4_XS down rows 16.0 -> 13.8.)
// T: the workgroup's thread count.
template <int T>
struct Q8kCols {
    static constexpr int kWaves = T / 64, kAhead = T == 256 ? 6 : T == 512 ? 3 : 2;
    float4 x4[kAhead];
    __device__ __forceinline__ static int wave() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }
    __device__ __forceinline__ static float4 block(const float *x, int b) {
        return *reinterpret_cast<const float4 *>(x + (size_t)b * 256 + 4 * (threadIdx.x & 63));
    }
    __device__ __forceinline__ void load(const float *x, int cols, int nb) {
#pragma unroll
        for (int u = 0; u < kAhead; u++)
            if (wave() + u * kWaves < cols * nb) x4[u] = block(x, wave() + u * kWaves);
        __asm__ volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    }
    // `live` (a column's number): a column whose slot is not live is not encoded (its rows may hold anything)
    // (ONE column: no division by a run-time length)
    template <bool ONE, class Live>
    __device__ __forceinline__ void encode(const float *x, uint8_t *dst, int cols, int nb, int col_stride, u32 *fault, u32 layer, Live live) const {
        const int lane = threadIdx.x & 63;
        auto store = [&](int b, float4 v) __attribute__((always_inline)) {
            const int c = ONE ? 0 : b / nb;
            if (live(c)) q8k_wave_block(v, dst + (size_t)c * col_stride + (size_t)(b - c * nb) * BM_Q8K_STRIDE, lane, fault, layer);
        };
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            const int b = wave() + u * kWaves;
            if (b < cols * nb) store(b, x4[u]);
        }
        for (int b0 = wave() + kAhead * kWaves; b0 < cols * nb; b0 += kAhead * kWaves) { // the rest, as many on their way at a time
            float4 more[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; u++)
                if (b0 + u * kWaves < cols * nb) more[u] = block(x, b0 + u * kWaves);
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                if (b0 + u * kWaves < cols * nb) store(b0 + u * kWaves, more[u]);
            }
        }
    }
};

// `cols` columns of nb super-blocks each, f32 rows at x (column c at x + c * nb * 256), into LDS at `dst` as Q8_2_X4
// columns with their tables: a 32-value block is four consecutive lanes of eight values. In two steps, for a workgroup
// that has something else to request in between: the f32 values of the
// first R tasks a thread are requested at once (memory answers in order, so they are back before anything asked for
// after them), and encoded into LDS later, when those other requests are on their way; tasks past the first R a thread
// go through the plain loop afterwards.
// T: the workgroup's thread count, a constant here: the built-in is read from memory, and a read after the weight
// requests would wait for all of them.
template <int R, int T>
struct Q82Cols {
    float4 lo[R], hi[R];
    u32 id[R]; // the expert of a task's column: a column whose slot is not live is not encoded (its rows may hold anything)
    __device__ __forceinline__ void load(const float *x, int total, int per_col, const u32 *ids) {
#pragma unroll
        for (int u = 0; u < R; u++) {
            int task = (int)threadIdx.x + u * T;
            task = task < total ? task : total - 1; // a read that stays inside the token's rows; the value is not used
            const float *p = x + (size_t)task * 8;
            lo[u] = *reinterpret_cast<const float4 *>(p);
            hi[u] = *reinterpret_cast<const float4 *>(p + 4);
            id[u] = ids[task / per_col];
        }
        __asm__ volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ void encode(const float *x, uint8_t *dst, int cols, int nb, const u32 *ids, u32 n_experts,
                                           u32 *fault, u32 layer) const {
        const int per_col = nb * 32, total = cols * per_col, col_bytes = nb * BM_Q82_SB_EXT;
#pragma unroll
        for (int u = 0; u < R; u++) {
            const int task = (int)threadIdx.x + u * T;
            if (task < total && id[u] < n_experts) { // whole quads: the tasks of a block are four neighbours
                const int c = task / per_col, at = task % per_col;
                const float v8[8] = {lo[u].x, lo[u].y, lo[u].z, lo[u].w, hi[u].x, hi[u].y, hi[u].z, hi[u].w};
                q82_quad8(v8, dst + (size_t)c * col_bytes, nb, at >> 2, task & 3, fault, layer);
            }
        }
        for (int task = (int)threadIdx.x + R * T; task < total; task += T) {
            const int c = task / per_col, at = task % per_col;
            if (ids[c] >= n_experts) continue;
            const float *p = x + (size_t)task * 8;
            const float4 l4 = *reinterpret_cast<const float4 *>(p), h4 = *reinterpret_cast<const float4 *>(p + 4);
            const float v8[8] = {l4.x, l4.y, l4.z, l4.w, h4.x, h4.y, h4.z, h4.w};
            q82_quad8(v8, dst + (size_t)c * col_bytes, nb, at >> 2, task & 3, fault, layer);
        }
    }
};

// k_gate_up_x for gate / up stacks that dot against Q8_K columns (Q3_K, IQ2_XXS, IQ3_XXS, IQ4_XS): the token's row is
// quantized by every workgroup into LDS, h is written as f32 rows, and where the down stack takes Q8_2_X4 columns
// (act_h given) the workgroup's 32 values also become their block of the slot's column.
template <int WA, int UA, int NBA, int T = 256, bool WIDE = false>
__global__ __launch_bounds__(T) void k_gate_up_xq(const float *x, const uint8_t *wg, const uint8_t *wu, u32 n_experts,
                                                    int nba, int nh, const u32 *sel, int spt_word, uint8_t *act_x,
                                                    uint8_t *act_h, float *h, GateRule rule, u32 *fault, u32 layer) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, q = tid & 3, which = (tid >> 2) & 1;
    // the grid as k_gate_up_x's
    const bool row_major = (spt_word & kGateRowMajor) != 0;
    const int spt = spt_word & ~kGateRowMajor;
    const int t = (int)(row_major ? blockIdx.z : blockIdx.y), slot = t * spt + (int)(row_major ? blockIdx.y : blockIdx.x / kDies);
    const int rb = (int)(row_major ? blockIdx.x : blockIdx.z * kDies + blockIdx.x % kDies);
    const int na = NBA > 0 ? NBA : nba;
    const int hidden = na * 256, ff = nh * 256;
    const int r0 = rb * (T / 8), r = r0 + (tid >> 3);
    if (T > 256 && r0 >= ff) return; // (by dies, the last eight blocks need not be whole)
    Q8kCols<T> xrow;
    xrow.load(x + (size_t)t * hidden, 1, na);
    const u32 id = sel[slot];
    uint8_t *hcol = act_h ? act_h + (size_t)slot * nh * BM_Q82_SB_EXT : nullptr;
    if (id >= n_experts) { // uniform over the workgroup
        if (id == 0xffffffffu) return; // a slot served elsewhere: nothing written, nothing raised
        if (tid == 0) bm_raise(fault, layer, kSiteExpertId);
        if (h && (tid & 7) == 0) h[(size_t)slot * ff + r] = bm_bits_f32(0x7fc00000u);
        if (hcol && tid < T / 8) q82_store(hcol, nh, (r0 + tid) >> 5, tid & 31, 0, Q82Head{0x7fc0u, 0, true}, 0);
        return;
    }
    const size_t row_bytes = (size_t)na * bm_block_bytes<WA>();
    const uint8_t *wrow = (which ? wu : wg) + ((size_t)id * ff + r) * row_bytes;
    Blk<WA> b[UA];
    preload<WA, UA>(b, wrow, na, q);
    const Iq2Tables tb = stage_tables_as<WA, WIDE, T>(lds);
    uint8_t *col = lds + tab_bytes<WA, WIDE>();
    const int col_bytes = bm_act_col_bytes<WA>(na);
    xrow.template encode<true>(x + (size_t)t * hidden, col, 1, na, 0, fault, layer, [](int) { return true; });
    __syncthreads();
    if (act_x && rb == 0 && slot % spt == 0) stage_bytes<T>(act_x + (size_t)t * col_bytes, col, col_bytes);
    float v[1];
    row_dot<WA, UA, NBA, 1, WIDE>(b, wrow, col, col_bytes, 1, na, q, tb, v, NoTap{});
    const float hv = swiglu_of_pair(v[0], which, rule, fault, layer);
    if (h && (tid & 7) == 0) h[(size_t)slot * ff + r] = hv;
    if (hcol) {
        float *hbuf = reinterpret_cast<float *>(col + col_bytes);
        if ((tid & 7) == 0) hbuf[tid >> 3] = hv;
        __syncthreads();
        if (tid < T / 8) quantize_h_block(hbuf + (tid & ~31), hcol, nh, (r0 + tid) >> 5, tid & 31, fault, layer);
    }
}

// (Workgroups of 64 or 128 threads, as k_gemv takes for a matrix of few rows, measure slower here: 4.35 and 3.89 us against
// 3.55 at 768 x 2048 - a wave then quantizes four or two times as much of the column before its first product.)
// k_gemv with the activation quantizer folded in: grid row c is column c, an f32 row of k values that every workgroup
// quantizes into LDS for itself (the form its weight type dots against), so a matrix-vector product from f32 is one
// launch and no column passes through memory. With act_out the first workgroup of a column leaves its bytes there.
template <int WT, int U, int NB>
__global__ __launch_bounds__(256) void k_gemv_x(const float *x, const uint8_t *w, long rows, int nb, int m, uint8_t *act_out,
                                                float *y, u32 *fault, u32 layer) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, q = tid & 3, c = blockIdx.y;
    const long row = (long)blockIdx.x * 64 + (tid >> 2);
    const bool active = row < rows;
    const int n = NB > 0 ? NB : nb;
    const int k = n * 256;
    const size_t row_bytes = (size_t)n * bm_block_bytes<WT>();
    const int col_bytes = bm_act_col_bytes<WT>(n);
    const uint8_t *wrow = w + (size_t)(active ? row : 0) * row_bytes;
    const float *xc = x + (size_t)c * k;
    // the column's first values (2048, or 6144) are asked for in front of the rows: vector loads come back in the order they were asked
    // for, and behind the rows' requests the quantizer would wait for those as well
    float4 x_lo = make_float4(0, 0, 0, 0), x_hi = x_lo;
    [[maybe_unused]] Q8kCols<256> xcol;
    if constexpr (bm_takes_q8k(WT)) {
        xcol.load(xc, 1, n);
    } else {
        const int o = tid * 8 < k ? tid * 8 : k - 8;
        x_lo = *reinterpret_cast<const float4 *>(xc + o), x_hi = *reinterpret_cast<const float4 *>(xc + o + 4);
        __asm__ volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    }
    Blk<WT> b[U];
    preload<WT, U>(b, wrow, n, q);
    const Iq2Tables tb = stage_tables<WT>(lds);
    uint8_t *col = lds + tab_bytes<WT>();
    if constexpr (bm_takes_q8k(WT)) {
        xcol.template encode<true>(xc, col, 1, n, 0, fault, layer, [](int) { return true; });
    } else { // a q8_2 block is four lanes of eight values; 2048 values a pass
        if (tid * 8 < k) {
            const float v8[8] = {x_lo.x, x_lo.y, x_lo.z, x_lo.w, x_hi.x, x_hi.y, x_hi.z, x_hi.w};
            q82_quad8(v8, col, n, tid >> 2, tid & 3, fault, layer);
        }
        for (int o = 2048 + tid * 8; o < k; o += 2048) {
            const float4 lo = *reinterpret_cast<const float4 *>(xc + o), hi = *reinterpret_cast<const float4 *>(xc + o + 4);
            float v8[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            q82_quad8(v8, col, n, o >> 5, tid & 3, fault, layer);
        }
    }
    __syncthreads();
    if (act_out && blockIdx.x == 0) stage_bytes(act_out + (size_t)c * col_bytes, col, col_bytes);
    float v[1];
    row_dot<WT, U, NB, 1>(b, wrow, col, col_bytes, 1, n, q, tb, v, NoTap{});
    if (q == 0 && active) y[(size_t)row * m + c] = v[0];
}

// k_down_combine for down stacks that dot against Q8_K columns: the token's slot rows of h (f32) are quantized by
// every workgroup into LDS; the first workgroup of a token also leaves the columns in act_h.
template <int WT, int U, int NB, int T, bool WIDE = false>
__global__ __launch_bounds__(T) void k_down_combine_hq(const uint8_t *w, u32 n_experts, int nb, const float *h,
                                                       uint8_t *act_h, const u32 *sel, const float *wts,
                                                         const float *resid, int spt_word, int rpe, float *y, u32 *fault,
                                                         u32 layer) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, q = tid & 3, quad = tid >> 2;
    // the grid and spt_word as k_down_combine's
    const int rb = (int)(spt_word & kDownRowMajor ? blockIdx.x : blockIdx.z * kDies + blockIdx.x), t = (int)blockIdx.y;
    const int spt = spt_word & 0xffff, shift = ((spt_word >> 16) & 0xff) - 1;
    const int D = shift >= 0 ? (T / 4) >> shift : T / 4 / spt;
    if (rb * D >= rpe) return;
    const int e = shift >= 0 ? quad & (spt - 1) : quad % spt, dl = shift >= 0 ? quad >> shift : quad / spt;
    const int r = rb * D + dl;
    const int n = NB > 0 ? NB : nb;
    const u32 id = sel[t * spt + e];
    const int si = (tid & 63) < spt ? tid & 63 : 0; // (every wave has the token's ids, slot l's in lane l: at most 64 slots)
    const u32 my_sel = sel[t * spt + si];
    // the token's f32 rows of h are asked for before anything that waits for the expert id, so they arrive with it and are
    // encoded while the weight rows are on their way
    typename std::conditional<bm_takes_q8k(WT), Q8kCols<T>, Q82Cols<4, T>>::type hrows;
    if constexpr (bm_takes_q8k(WT)) hrows.load(h + (size_t)t * spt * n * 256, spt, n);
    else hrows.load(h + (size_t)t * spt * n * 256, spt * n * 32, n * 32, sel + t * spt);
    const float my_w = wts[t * spt + si];
    const bool live = id < n_experts;
    const bool active = dl < D && r < rpe && live;
    const float resid_v = resid && tid < D && rb * D + tid < rpe ? resid[(size_t)t * rpe + rb * D + tid] : 0.0f;
    if (!live && id != 0xffffffffu && rb == 0 && dl == 0 && q == 0) bm_raise(fault, layer, kSiteExpertId);
    const size_t row_bytes = (size_t)n * bm_block_bytes<WT>();
    const int col_bytes = bm_act_col_bytes<WT>(n), col_stride = col_bytes + slot_col_pad(WT, n, spt);
    const uint8_t *wrow = w + ((size_t)(live ? id : 0) * rpe + (active ? r : 0)) * row_bytes;
    Blk<WT> b[U];
    preload<WT, U>(b, wrow, n, q);
    const Iq2Tables tb = stage_tables_as<WT, WIDE, T>(lds);
    uint8_t *cols = lds + tab_bytes<WT, WIDE>();
    float *part = reinterpret_cast<float *>(cols + (size_t)spt * col_stride); // [D][spt]
    float *s_w = part + D * spt;                                              // [spt]
    u32 *s_sel = reinterpret_cast<u32 *>(s_w + spt);                          // [spt]
    if constexpr (bm_takes_q8k(WT))
        hrows.template encode<false>(h + (size_t)t * spt * n * 256, cols, spt, n, col_stride, fault, layer,
                     [&](int c) { return (u32)__builtin_amdgcn_readlane((int)my_sel, __builtin_amdgcn_readfirstlane(c)) < n_experts; });
    else hrows.encode(h + (size_t)t * spt * n * 256, cols, spt, n, sel + t * spt, n_experts, fault, layer);
    if (tid < spt) {
        s_w[tid] = my_w;
        s_sel[tid] = my_sel;
    }
    __syncthreads();
    if (act_h && rb == 0) // the live slots' columns; the others keep what they held
        for (int c = 0; c < spt; c++)
            if (s_sel[c] < n_experts) stage_bytes<T>(act_h + ((size_t)t * spt + c) * col_bytes, cols + (size_t)c * col_stride, col_bytes);
    float v[1];
    row_dot<WT, U, NB, 1, WIDE>(b, wrow, cols + (size_t)e * col_stride, col_stride, 1, n, q, tb, v, NoTap{});
    if (q == 0 && dl < D) part[dl * spt + e] = v[0];
    __syncthreads();
    if (tid < D && rb * D + tid < rpe) y[(size_t)t * rpe + rb * D + tid] = slot_sum(part + tid * spt, s_w, s_sel, spt, n_experts, resid_v, resid != nullptr);
}

// ------------------------------------------------------------------------------------------ verification

struct StoreTap {
    static constexpr bool kActive = true;
    int *out; // 16 words a super-block, zeroed before the quad runs
    __device__ __forceinline__ void q4k(int i, int s, int, int v) const { atomicAdd(&out[16 * i + s], v); }
    __device__ __forceinline__ void q4k_isum(int i, int s, int v) const { out[16 * i + 8 + s] = v; }
    __device__ __forceinline__ void q6k(int i, int g, int v) const { out[16 * i + g] = v; }
    __device__ __forceinline__ void iq2(int i, int b, int q, int v) const {
        atomicAdd(&out[16 * i + b], v);
        (void)q;
    }
    __device__ __forceinline__ void iq4_sub(int i, int b, int v) const { out[16 * i + b] = v; }
    __device__ __forceinline__ void iq4_lane(int i, int l, int v) const { out[16 * i + 8 + l] = v; }
};

template <int WT, int U, int NB>
__global__ __launch_bounds__(64) void k_block_sums(const uint8_t *wrow, int nb, const uint8_t *act_col, int *out) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, q = tid & 3;
    const int n = NB > 0 ? NB : nb;
    const int col_bytes = bm_act_col_bytes<WT>(n);
    for (int i = tid; i < 16 * n; i += 64) out[i] = 0;
    const Iq2Tables tb = stage_tables<WT>(lds, 64);
    uint8_t *col = lds + tab_bytes<WT>();
    stage_bytes<64>(col, act_col, col_bytes);
    __threadfence();
    __syncthreads();
    if (tid >= 4) return;
    Blk<WT> b[U];
    preload<WT, U>(b, wrow, n, q);
    float v[1];
    row_dot<WT, U, NB, 1>(b, wrow, col, col_bytes, 1, n, q, tb, v, StoreTap{out});
    if constexpr (WT == BM_IQ2XXS || WT == BM_IQ3XXS) {
        // the eight scales 2s + 1 of each super-block, as the dot reads them
        if (q == 0)
            for (int i = 0; i < n; i++)
                for (int s = 0; s < 8; s++) {
                    u32 aux;
                    if constexpr (WT == BM_IQ2XXS)
                        __builtin_memcpy(&aux, wrow + (size_t)i * BM_IQ2XXS_BLOCK + 6 + 8 * s, 4);
                    else
                        __builtin_memcpy(&aux, wrow + (size_t)i * BM_IQ3XXS_BLOCK + 66 + 4 * s, 4);
                    out[16 * i + 8 + s] = 2 * (int)(aux >> 28) + 1;
                }
    }
}

// ---------------------------------------------------------------------------------------- launch helpers

constexpr unsigned kCardUnits = 256; // compute units of the card these kernels are written for

int act_col_bytes(int wtype, int k) {
    const int nb = k / 256;
    return bm_takes_q8k(wtype) ? nb * BM_Q8K_STRIDE : nb * BM_Q82_SB_EXT;
}

int gemv_max_cols(int wtype, int k) {
    int m = (kMaxLds - tab_bytes_rt(wtype)) / act_col_bytes(wtype, k);
    return m > 8 ? 8 : m;
}

// From how many super-blocks a row on the columns of a matrix of 513 to 1024 groups of 16 rows (`far`: of more than 768) are dealt to
// waves. There k_gemv, a wave a group and all columns, has up to a wave a SIMD and its time no longer grows with the rows, while the
// other form's does: it loses where its start counts (short rows), where half of a wave's last column pair is idle (odd counts, three
// above all) and for the types whose unpacking is dear beside a column's dot. It gains most where k_gemv has no ring (`ringless`: an odd count
// past three). Past 1024 groups k_gemv: dealt columns take 1.08 (Q4_K) to 1.38 times (Q6_K) its time on average there, though up to 24000 rows those
// of rows without a ring would still gain (four columns 0.77 to 0.9). us, k_gemv / columns dealt: 16384 rows, 8 columns, Q6_K k 512 5.7 / 7.6, k 768 7.0 / 9.3, k 2304
// 20.1 / 17.1, IQ3_XXS k 2048 16.9 / 18.1, Q4_K k 2048 13.6 / 11.2; 12288 rows, 8 columns, Q6_K k 512 5.7 / 6.5, k 2048 14.4 / 13.2; 16384
// rows, 5 columns, Q5_K k 512 4.7 / 5.2, k 2048 11.5 / 10.7; of Q6_K's rows the longer ones lose most past 768 groups: 14657 rows of 4096, 8
// columns 29.2 / 35.3, 4 columns of 4608 21.3 / 24.4. (10193 calls from 600 to 17000 rows, seven types, 256 to 5120 values, 2 to 8 columns.)
static int gemv_cols_from(int wtype, int m, bool far, bool ringless) {
    constexpr int kNever = 1 << 30;
    const bool q8k = bm_takes_q8k(wtype), odd = m % 2 != 0;
    if (m == 2) return 1;
    if (wtype == BM_Q6K && (ringless ? far && m == 7 : far || odd)) return kNever;
    if (ringless) return odd && (m == 3 ? q8k : far && wtype != BM_Q3K && wtype != BM_Q4K && wtype != BM_Q5K) ? 9 : 1;
    if (m == 3) {
        if (q8k) return kNever;
        far = true;
    }
    if (wtype == BM_Q6K) return m == 4 ? 3 : 8;
    if (!far) return m == 8 || (m == 4 && q8k) ? 2 : 3;
    if (wtype == BM_Q3K || wtype == BM_Q4K) return odd ? 8 : 3;
    if (wtype == BM_Q5K) return 8;
    if (wtype == BM_IQ3XXS) return odd ? kNever : 16;
    return odd ? 16 : 8;
}

hipError_t gemv(const Launch &L, int wtype, const uint8_t *w, int64_t rows, int k, const uint8_t *act, int m_total,
                int col0, int m, float *y) {
    const int nb = k / 256;
    const size_t lds = tab_bytes_rt(wtype) + (size_t)m * act_col_bytes(wtype, k);
    if (m == 1) {
        const bool few = (rows + 63) / 64 < (int64_t)kCardUnits; // a matrix whose 64-row blocks do not fill the card
#define CALL_BODY                                                                                                      \
    auto kern = few ? k_gemv<WT, U, NB, 1, 64> : k_gemv<WT, U, NB, 1>;                                                 \
    hipError_t e = allow_lds(kern, lds);                                                                               \
    if (e != hipSuccess) return e;                                                                                     \
    const int T = few ? 64 : 256, per = T / 4;                                                                         \
    hipLaunchKernelGGL(kern, dim3((unsigned)((rows + per - 1) / per)), dim3(T), lds, L.stream, w, (long)rows, nb, act, \
                       m_total, col0, m, y);
        BM_DISPATCH(wtype, nb)
#undef CALL_BODY
        return hipGetLastError();
    }
    // Several columns of a matrix whose rows do not fill the card: the columns are dealt to waves as well, one a wave up to about a wave a
    // SIMD, two (which unpack a row once for both) beyond; row groups share a workgroup, and the columns it stages, where there
    // are more of them than compute units. us, one launch, k_gemv / one column a wave / two: Q6_K 7168 x 2048, 2 columns
    // 7.5 / 5.5 / 6.4, 4 columns 9.4 / 8.6 / 6.9, 8 columns 13.5 / 15 / 9.5; Q4_K 768 x 2048, 4 columns 7.3 / 3.9 / 5.6; Q5_K
    // 2048 x 7168, 8 columns 36 / 19 / 20. (Q6_K goes over to two a little sooner: 3000 rows of 512, 7 columns
    // 5.2 / 4.6 / 3.8. Rows of an odd number of super-blocks, where two columns a wave have no ring: two columns go one a wave all the way, IQ3_XXS
    // 12288 x 2304 10.8 / 10.2 / 12.2. Else two a wave past 512 groups, but for three super-blocks.)
    const int64_t groups = (rows + 15) / 16;
    const bool ringless = nb % 2 != 0 && nb > 3;
    if (groups <= 512 || (groups <= 1024 && nb >= gemv_cols_from(wtype, m, groups > 768, ringless))) {
        const bool one = ringless ? m == 2 || groups * m <= 1280
                         : wtype == BM_Q6K ? groups * (m + m % 2) <= 1024 : groups * m <= 1280 && (groups <= 512 || nb == 3);
        const int per = one ? 1 : 2, cgs = (m + per - 1) / per;
        const int rgs = (int)std::max<int64_t>(1, std::min<int64_t>((groups + kCardUnits - 1) / kCardUnits, (one ? 8 : 16) / cgs));
        const int T = 64 * rgs * cgs;
#define BM_COLS_LAUNCH(C)                                                                                              \
    auto kern = k_gemv_cols<WT, U, NB, C>;                                                                             \
    hipError_t e = allow_lds(kern, lds);                                                                               \
    if (e != hipSuccess) return e;                                                                                     \
    hipLaunchKernelGGL(kern, dim3((unsigned)((groups + rgs - 1) / rgs)), dim3(T), lds, L.stream, w, (long)rows, nb,    \
                       act, m_total, col0, m, y, cgs, rgs, (256 + cgs - 1) / cgs, T);
#define CALL_BODY BM_COLS_LAUNCH(1)
        if (per == 1) {
            BM_DISPATCH(wtype, nb)
            return hipGetLastError();
        }
#undef CALL_BODY
#define CALL_BODY BM_COLS_LAUNCH(2)
        BM_DISPATCH_COLS(wtype, nb)
#undef CALL_BODY
#undef BM_COLS_LAUNCH
        return hipGetLastError();
    }
#define CALL_BODY                                                                                                      \
    auto kern = k_gemv<WT, U, NB, 8>;                                                                                  \
    hipError_t e = allow_lds(kern, lds);                                                                               \
    if (e != hipSuccess) return e;                                                                                     \
    hipLaunchKernelGGL(kern, dim3((unsigned)((rows + 63) / 64)), dim3(256), lds, L.stream, w, (long)rows, nb, act,     \
                       m_total, col0, m, y);
    BM_DISPATCH_COLS(wtype, nb)
#undef CALL_BODY
    return hipGetLastError();
}

size_t gemv_x_lds(int wtype, int k) { return tab_bytes_rt(wtype) + (size_t)act_col_bytes(wtype, k); }

hipError_t gemv_x(const Launch &L, int wtype, const uint8_t *w, int64_t rows, int k, const float *x, int m, uint8_t *act_out,
                  float *y) {
    const int nb = k / 256;
    const size_t lds = gemv_x_lds(wtype, k);
#define CALL_BODY                                                                                                      \
    auto kern = k_gemv_x<WT, U, NB>;                                                                                   \
    hipError_t e = allow_lds(kern, lds);                                                                               \
    if (e != hipSuccess) return e;                                                                                     \
    hipLaunchKernelGGL(kern, dim3((unsigned)((rows + 63) / 64), (unsigned)m), dim3(256), lds, L.stream, x, w,          \
                       (long)rows, nb, m, act_out, y, L.fault, L.layer);
    BM_DISPATCH(wtype, nb)
#undef CALL_BODY
    return hipGetLastError();
}

// Whether a launch of one-column row dots takes the IQ tables in copies: `lds` bytes with them, `threads` a workgroup. Not where they leave a
// compute unit fewer than sixteen waves, and not for rows of one super-block, which end before the larger tables are laid out (gate . up 1.2 times
// the plain tables' launch, down 1.01 on average and up to 1.3).
static bool copies_fit(int wtype, int nb, size_t lds, int threads) {
    return (wtype == BM_IQ2XXS || wtype == BM_IQ3XXS) && nb >= 2 && (size_t)kMaxLds / lds * (size_t)threads >= 16 * 64;
}
#define BM_WITH_TABLES(PLAIN, WIDE)                                                                                    \
    {                                                                                                                  \
        if constexpr (WT == BM_IQ2XXS || WT == BM_IQ3XXS)                                                              \
            if (wide) return launch(WIDE);                                                                             \
        return launch(PLAIN);                                                                                          \
    }
// A gate . up launch of `blocks` workgroups of 32 row pairs as one of workgroups of 64 that hold the tables in copies: where the blocks make an even
// number of rounds over the compute units, so that two of the smaller workgroups would share a unit to the end (an odd round makes a larger
// workgroup's unit work twice as long as the others': 1.02 to 1.06 times the plain tables' launch at three, five and seven rounds, 0.85 to 0.98 at two,
// four, six and eight). Beyond eight rounds, where rounds no longer stand out, by the rows: from 13 super-blocks of IQ2_XXS (0.98 to 1.02, shorter ones 1.05
// to 1.13), from 7 of IQ3_XXS (0.86 to 1.02). 1200 random launches of 1 to 28
// super-blocks: the rule is 0.3 % behind the better side, 0.92 of the plain time where it takes the copies.
static bool gate_up_in_copies(int wtype, int k, int64_t blocks) {
    const int64_t rounds = (blocks + kCardUnits - 1) / kCardUnits;
    const int nb = k / 256;
    if (rounds <= 8 ? rounds % 2 != 0 : nb < (wtype == BM_IQ2XXS ? 13 : 7)) return false;
    return copies_fit(wtype, nb, tab_bytes_rt(wtype, true) + (size_t)act_col_bytes(wtype, k) + 64 * sizeof(float), 512);
}

hipError_t gate_up(const Launch &L, int wtype, const uint8_t *wg, const uint8_t *wu, int n_experts, int k,
                   const uint8_t *act, const uint32_t *sel, int n_slots, int rows_per_expert, int slots_per_col,
                   float *h, uint8_t *act_h) {
    const int nb = k / 256, rpe = rows_per_expert;
    if (n_slots <= 0 || slots_per_col <= 0) return hipErrorInvalidValue;
    if (slots_per_col > 0xffffff) { // (more slots a column than there are slots: column 0 either way)
        if (n_slots > 0xffffff) return hipErrorInvalidValue;
        slots_per_col = 0xffffff;
    }
    const unsigned grid_y = (unsigned)n_slots < kGateUpGridY ? (unsigned)n_slots : kGateUpGridY;
    const unsigned grid_z = ((unsigned)n_slots + kGateUpGridY - 1) / kGateUpGridY;
    const int spc_shift = (slots_per_col & (slots_per_col - 1)) == 0 ? __builtin_ctz((unsigned)slots_per_col) : -1;
    const bool wide = gate_up_in_copies(wtype, k, (int64_t)n_slots * ((rpe + 31) / 32));
    const int T = wide ? 512 : 256;
    const size_t bytes = tab_bytes_rt(wtype, wide) + (size_t)act_col_bytes(wtype, k) + T / 8 * sizeof(float);
    auto launch = [&](auto kern) {
        hipError_t e = allow_lds(kern, bytes);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kern, dim3((unsigned)((rpe + T / 8 - 1) / (T / 8)), grid_y, grid_z), dim3(T), bytes, L.stream, wg, wu, (u32)n_experts, nb,
                           act, sel, rpe, slots_per_col | ((spc_shift + 1) << 24), (u32)n_slots, GateUpColLate{h, act_h, L.rule, L.fault, L.layer});
        return hipGetLastError();
    };
#define CALL_BODY BM_WITH_TABLES((k_gate_up<WT, U, NB>), (k_gate_up<WT, U, NB, 512, true>))
    BM_DISPATCH(wtype, nb)
#undef CALL_BODY
    return hipErrorInvalidValue;
}

hipError_t gemv_sel(const Launch &L, int wtype, const uint8_t *w, int n_experts, int k, const uint8_t *act,
                    const uint32_t *sel, int n_slots, int rows_per_expert, float *y) {
    const int nb = k / 256, rpe = rows_per_expert;
    const size_t lds = tab_bytes_rt(wtype) + (size_t)act_col_bytes(wtype, k);
    const unsigned grid = (unsigned)n_slots * (unsigned)((rpe + 63) / 64);
#define CALL_BODY                                                                                                      \
    auto kern = k_gemv_sel<WT, U, NB>;                                                                                 \
    hipError_t e = allow_lds(kern, lds);                                                                               \
    if (e != hipSuccess) return e;                                                                                     \
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), lds, L.stream, w, (u32)n_experts, nb, act, sel, rpe, y, L.fault,   \
                       L.layer);
    BM_DISPATCH(wtype, nb)
#undef CALL_BODY
    return hipGetLastError();
}

size_t down_combine_lds(int wtype, int k, int spt) {
    const int D = 64 / spt;
    return tab_bytes_rt(wtype) + (size_t)spt * (act_col_bytes(wtype, k) + slot_col_pad(wtype, k / 256, spt)) + ((size_t)D * spt + 2 * (size_t)spt) * sizeof(float);
}

hipError_t down_combine(const Launch &L, int wtype, const uint8_t *w, int n_experts, int k, const uint8_t *act,
                        const uint32_t *sel, const float *wts, const float *resid, int slots_per_token, int m,
                        int rows_per_expert, float *y) {
    const int nb = k / 256, rpe = rows_per_expert, spt = slots_per_token;
    if (m > kMaxGridTokens) {
        const size_t slots = (size_t)kMaxGridTokens * spt, rows = (size_t)kMaxGridTokens * rpe;
        const hipError_t e = down_combine(L, wtype, w, n_experts, k, act, sel, wts, resid, spt, kMaxGridTokens, rpe, y);
        if (e != hipSuccess) return e;
        return down_combine(L, wtype, w, n_experts, k, act + slots * act_col_bytes(wtype, k), sel + slots, wts + slots,
                            resid ? resid + rows : nullptr, spt, m - kMaxGridTokens, rpe, y + rows);
    }
    const int D = 64 / spt;
    const int spt_shift = (spt & (spt - 1)) == 0 ? __builtin_ctz((unsigned)spt) : -1;
    const size_t lds = down_combine_lds(wtype, k, spt);
    const unsigned blocks = (unsigned)((rpe + D - 1) / D), grid = (unsigned)m * blocks;
    const bool row_major = plain_order((int64_t)m * spt, m, blocks);
    if (L.down_form == 1 && wtype == BM_Q6K && nb == 3 && 64 % spt == 0) { // BM_DOWN_SPLIT where it is built: the super-blocks of a row dealt to the waves
        constexpr int NB = 3;
        const size_t lds_split = (size_t)spt * bm_act_col_bytes<BM_Q6K>(NB) + (64 * (NB - 1) * 32 + D * spt + 2 * spt) * sizeof(float);
        hipLaunchKernelGGL(k_down_combine_q6k_split<NB>, dim3(grid), dim3(256 * NB), lds_split, L.stream, w, (u32)n_experts, act, sel, wts,
                           resid, spt, rpe, y, L.fault, L.layer);
        return hipGetLastError();
    }
#define BM_DOWN_LAUNCH(EIGHT)                                                                                          \
    {                                                                                                                  \
        auto kern = k_down_combine<WT, U, NB, EIGHT>;                                                                  \
        hipError_t e = allow_lds(kern, lds);                                                                           \
        if (e != hipSuccess) return e;                                                                                 \
        hipLaunchKernelGGL(kern, row_major ? dim3(blocks, (unsigned)m) : dim3(kDies, (unsigned)m, eighths(blocks)), dim3(256), lds, L.stream,   \
                           w, (u32)n_experts, nb, act, sel, wts, resid,                                                \
                           spt | ((spt_shift + 1) << 16) | (row_major ? kDownRowMajor : 0), rpe, DownLate{y, L.fault, L.layer});       \
    }
    // (eight slots a token: the form that takes the token's ids through the scalar cache)
#define CALL_BODY                                                                                                      \
    if (spt == 8) BM_DOWN_LAUNCH(true) else BM_DOWN_LAUNCH(false)
    BM_DISPATCH(wtype, nb)
#undef CALL_BODY
#undef BM_DOWN_LAUNCH
    return hipGetLastError();
}

static bool tab_known(int t) {
    return t == BM_Q3K || t == BM_Q4K || t == BM_Q5K || t == BM_Q6K || t == BM_IQ2XXS || t == BM_IQ3XXS || t == BM_IQ4XS;
}

// every type this library has a row dot for goes on either side of the fused step
bool moe_decode_supported(int gate_type, int down_type) { return tab_known(gate_type) && tab_known(down_type); }

hipError_t gate_up_x(const Launch &L, int gate_type, const float *x, const uint8_t *wg, const uint8_t *wu,
                     int n_experts, int hidden, int ff, const uint32_t *sel, int slots_per_token, int m,
                     uint8_t *act_x, uint8_t *act_h, float *h) {
    const int nba = hidden / 256, nbb = ff / 256, spt = slots_per_token;
    const size_t lds_a = (size_t)act_col_bytes(gate_type, hidden) + 32 * sizeof(float);
    const bool row_major = plain_order((int64_t)m * spt, m, kDies * (unsigned)nbb);
    const dim3 grid_a = row_major ? dim3((unsigned)(ff / 32), (unsigned)spt, (unsigned)m) : dim3(kDies * (unsigned)spt, (unsigned)m, (unsigned)nbb);
#define BM_GUX(WA, UA, NA)                                                                                             \
    {                                                                                                                  \
        auto kern = k_gate_up_x<WA, UA, NA>;                                                                           \
        hipError_t e = allow_lds(kern, lds_a);                                                                         \
        if (e != hipSuccess) return e;                                                                                 \
        hipLaunchKernelGGL(kern, grid_a, dim3(256), lds_a, L.stream, x, wg, wu, (u32)n_experts, nba, nbb, sel,         \
                           spt | (row_major ? kGateRowMajor : 0), GateUpLate{act_x, act_h, h, L.rule, L.fault, L.layer});              \
    }
    if (gate_type == BM_Q4K) {
        if (nba == 8) BM_GUX(BM_Q4K, kRingQ4K, 8)
        else BM_GUX(BM_Q4K, kRing, 0)
    } else if (gate_type == BM_Q5K) {
        if (nba == 8) BM_GUX(BM_Q5K, kRingQ5K, 8)
        else BM_GUX(BM_Q5K, 1, 0)
    } else if (gate_type == BM_Q6K) {
        BM_GUX(BM_Q6K, kRing, 0)
    } else if (bm_takes_q8k(gate_type)) {
        const int nb = nba;
        const int wtype = gate_type;
        const bool wide = gate_up_in_copies(wtype, hidden, (int64_t)m * spt * (ff / 32));
        const int T = wide ? 512 : 256;
        const size_t bytes = tab_bytes_rt(wtype, wide) + (size_t)act_col_bytes(gate_type, hidden) + T / 8 * sizeof(float);
        const unsigned blocks = (unsigned)(ff / (T / 8));
        const bool row_major = plain_order((int64_t)m * spt, m, blocks, T);
        auto launch = [&](auto kern) {
            hipError_t e = allow_lds(kern, bytes);
            if (e != hipSuccess) return e;
            const dim3 grid = row_major ? dim3(blocks, (unsigned)spt, (unsigned)m) : dim3(kDies * (unsigned)spt, (unsigned)m, eighths(blocks));
            hipLaunchKernelGGL(kern, grid, dim3(T), bytes, L.stream, x, wg, wu, (u32)n_experts, nba, nbb, sel,
                               spt | (row_major ? kGateRowMajor : 0), act_x, act_h, h, L.rule, L.fault, L.layer);
            return hipGetLastError();
        };
#define CALL_BODY BM_WITH_TABLES((k_gate_up_xq<WT, U, NB>), (k_gate_up_xq<WT, U, NB, 512, true>))
        BM_DISPATCH(gate_type, nb)
#undef CALL_BODY
    } else {
        return hipErrorInvalidValue;
    }
#undef BM_GUX
    return hipGetLastError();
}

// How many threads a workgroup of down + combine takes where it quantizes the token's slot rows of h itself: `blocks` blocks of 256 values,
// some 25 instructions a wave and block beside a row dot's 50 a lane and super-block; a larger workgroup shares that between more rows.
// 256 threads where the blocks are at most eight, or at most twenty and the launch is a single small round. Else 512, or 1024, of which a
// compute unit holds one (84 to 102 registers a lane): a round of 256 takes 9.3 us where half a round's work takes 5.1 with 512, so 1024 where
// its last round is more than half full or there are more than five. 256 again, which end most evenly, where that is not so, the blocks are at
// most 24 and what 512 have behind a round or two of 512 is less than a quarter of one. (us with 256 / 512 / 1024 threads, top-8 of 768
// values, IQ4_XS, 2048 rows: 1 token 7.7 / 7.3 / 9.0, 2 tokens 10.2 / 8.1 / 9.6, 3 tokens 12.2 / 11.2 / 10.1, 4 tokens 14.8 / 12.0 / 10.8, 6
// tokens 20.2 / 17.0 / 18.3, 7 tokens 22.4 / 20.4 / 18.9, 10 tokens 29.3 / 25.5 / 26.8, 16 tokens 47.6 / 40.1 / 37.0; IQ2_XXS, 1536
// values, 5120 rows, one token 19.4 / 17.6 / 16.0, top-2, 880 rows, 7 tokens 9.1 / 9.9 / 13.3, top-7 of 512, 1824 rows, 11 tokens 18.8 /
// 20.7 / 20.9. Of 3800 random calls of the four types, 2 to 8 super-blocks a row, 256 to 7200 rows, top-1 to 12, 1 to 40 tokens, the rule is
// 1.4 % behind the best of the three, 256 threads for all 11 %.)
static int down_threads(int spt, int m, int rpe, int blocks) {
    auto units = [&](int T) {
        const int D = T / 4 / spt;
        return (int64_t)m * ((rpe + D - 1) / D);
    };
    constexpr int64_t kCard = kCardUnits;
    if (blocks <= 8 || (blocks <= 20 && units(256) <= kCard)) return 256;
    const int64_t of_1024 = units(1024), rounds = (of_1024 + kCard - 1) / kCard, of_512 = units(512), last = of_512 % (2 * kCard);
    if ((of_1024 + kCard / 2 - 1) / (kCard / 2) == 2 * rounds || rounds > 5) return 1024;
    return blocks <= 24 && of_512 > 2 * kCard && of_512 < 6 * kCard && last > 0 && last < kCard / 2 ? 256 : 512;
}

// Down + combine from the f32 rows of h, for a down stack that takes Q8_K columns; act_h (optional) receives them.
hipError_t down_combine_hq(const Launch &L, int wtype, const uint8_t *w, int n_experts, int k, const float *h,
                           uint8_t *act_h, const uint32_t *sel, const float *wts, const float *resid,
                           int slots_per_token, int m, int rows_per_expert, float *y) {
    const int nb = k / 256, rpe = rows_per_expert, spt = slots_per_token;
    if (m > kMaxGridTokens) {
        const size_t slots = (size_t)kMaxGridTokens * spt, rows = (size_t)kMaxGridTokens * rpe;
        const hipError_t e = down_combine_hq(L, wtype, w, n_experts, k, h, act_h, sel, wts, resid, spt, kMaxGridTokens, rpe, y);
        if (e != hipSuccess) return e;
        return down_combine_hq(L, wtype, w, n_experts, k, h + slots * k, act_h ? act_h + slots * act_col_bytes(wtype, k) : nullptr, sel + slots,
                               wts + slots, resid ? resid + rows : nullptr, spt, m - kMaxGridTokens, rpe, y + rows);
    }
    const int spt_shift = (spt & (spt - 1)) == 0 ? __builtin_ctz((unsigned)spt) : -1;
    const int T = bm_takes_q8k(wtype) ? down_threads(spt, m, rpe, spt * nb) : 256; // (Q8_2_X4 columns are encoded from registers, four tasks a thread of 256)
    const int D = T / 4 / spt;
    const size_t lds = down_combine_lds(wtype, k, spt) + (size_t)(D - 64 / spt) * spt * sizeof(float);
    const unsigned blocks = (unsigned)((rpe + D - 1) / D);
    const bool row_major = plain_order((int64_t)m * spt, m, blocks, T);
    // (from 512 threads on: of 256 a compute unit holds too few beside the copies; 980 random launches of two super-blocks and more 0.98, by rows 0.96 to
    // 1.0, at worst 1.12, two super-blocks of IQ2_XXS)
    const bool wide = copies_fit(wtype, nb, lds + (size_t)(tab_bytes_rt(wtype, true) - tab_bytes_rt(wtype)), T);
    const size_t bytes = lds + (size_t)(tab_bytes_rt(wtype, wide) - tab_bytes_rt(wtype));
    auto launch = [&](auto kern) {
        hipError_t e = allow_lds(kern, bytes);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kern, row_major ? dim3(blocks, (unsigned)m) : dim3(kDies, (unsigned)m, eighths(blocks)), dim3((unsigned)T), bytes,
                           L.stream, w, (u32)n_experts, nb, h, act_h, sel, wts, resid,
                           spt | ((spt_shift + 1) << 16) | (row_major ? kDownRowMajor : 0), rpe, y, L.fault, L.layer);
        return hipGetLastError();
    };
#define CALL_BODY                                                                                                      \
    if constexpr (bm_takes_q8k(WT)) {                                                                                  \
        if (T == 1024) BM_WITH_TABLES((k_down_combine_hq<WT, U, NB, 1024>), (k_down_combine_hq<WT, U, NB, 1024, true>)) \
        if (T == 512) BM_WITH_TABLES((k_down_combine_hq<WT, U, NB, 512>), (k_down_combine_hq<WT, U, NB, 512, true>)) \
    }                                                                                                                  \
    return launch(k_down_combine_hq<WT, U, NB, 256>)
    BM_DISPATCH(wtype, nb)
#undef CALL_BODY
    return hipErrorInvalidValue;
}

hipError_t moe_decode(const Launch &L, int gate_type, int down_type, const float *x, const uint8_t *wg, const uint8_t *wu,
                      const uint8_t *wd, int n_experts, int hidden, int ff, const uint32_t *sel, const float *wts,
                      const float *resid, int slots_per_token, int m, uint8_t *act_x, uint8_t *act_h, float *h, float *y) {
    const int spt = slots_per_token;
    if (!moe_decode_supported(gate_type, down_type)) return hipErrorInvalidValue;
    // a down stack on Q8_K columns cannot get them from the gate . up launch (a column's block spans eight of
    // its workgroups): that launch leaves h as f32 rows and the down launch quantizes them itself
    // (for a down stack on Q8_2_X4 columns the same split measures slower, 12.2 us a token against 11.3 at the
    // Qwen3 shape: the gate . up launch loses its quantizer epilogue, 0.5 us, but every down workgroup then encodes
    // the token's 6144 values, 700 instructions a wave that do not hide behind its weight stream)
    const bool hq = bm_takes_q8k(down_type);
    hipError_t e = gate_up_x(L, gate_type, x, wg, wu, n_experts, hidden, ff, sel, spt, m, act_x, hq ? nullptr : act_h, h);
    if (e != hipSuccess) return e;
    if (hq) return down_combine_hq(L, down_type, wd, n_experts, ff, h, act_h, sel, wts, resid, spt, m, hidden, y);
    return down_combine(L, down_type, wd, n_experts, ff, act_h, sel, wts, resid, spt, m, hidden, y);
}

// --------------------------------------------------------------- the fused step on scratch the library holds

// What bm_moe_decode takes from its caller as act_h (and h, for a down stack on Q8_K columns), held here instead: one
// array a device for as long as the process lives, so the entry that uses it calls no allocator. Room for
// kStaticValues values of h (slots x ff): their activation columns in the wider of the two column forms first, their
// f32 rows after them.
constexpr size_t kStaticColBytes = kStaticValues / 256 * BM_Q82_SB_EXT; // Q8_K columns (296 a super-block) fit too
constexpr size_t kStaticBytes = kStaticColBytes + kStaticValues * sizeof(float);
static __device__ __align__(256) uint8_t scratch[kStaticBytes];

// The array's address on each device. Host code may not hand the symbol itself to a kernel (on the host it names a
// stand-in, not device memory): the address is asked for once a device, with that device current, and every launch
// takes it from here.
constexpr int kStaticMaxDevices = 64;
static std::atomic<uint8_t *> g_scratch_at[kStaticMaxDevices]; // contexts may be made from several threads at once

hipError_t static_scratch_init(int device) {
    if (device < 0 || device >= kStaticMaxDevices) return hipErrorInvalidDevice;
    if (g_scratch_at[device].load(std::memory_order_acquire)) return hipSuccess;
    void *at = nullptr;
    const hipError_t e = hipGetSymbolAddress(&at, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!at) return hipErrorInvalidSymbol;
    g_scratch_at[device].store(static_cast<uint8_t *>(at), std::memory_order_release); // every thread finds the same address
    return hipSuccess;
}

hipError_t moe_decode_static(const Launch &L, int device, int gate_type, int down_type, const float *x, const uint8_t *wg,
                             const uint8_t *wu, const uint8_t *wd, int n_experts, int hidden, int ff, const uint32_t *sel,
                             const float *wts, const float *resid, int slots_per_token, int m, float *y) {
    uint8_t *base = device < 0 || device >= kStaticMaxDevices ? nullptr : g_scratch_at[device].load(std::memory_order_acquire);
    if (!base) return hipErrorNotInitialized;
    if ((size_t)m * (size_t)slots_per_token * (size_t)ff > kStaticValues) return hipErrorInvalidValue;
    uint8_t *act_h = base;
    // the f32 rows of h are only read by a down stack on Q8_K columns: no other call writes them
    float *h = bm_takes_q8k(down_type) ? reinterpret_cast<float *>(base + kStaticColBytes) : nullptr;
    // every live slot's column (or f32 rows) is written whole by the first launch before the second reads it, and a
    // slot that is not live is never read into a sum: nothing here has to start at zero
    return moe_decode(L, gate_type, down_type, x, wg, wu, wd, n_experts, hidden, ff, sel, wts, resid,
                      slots_per_token, m, nullptr, act_h, h, y);
}

hipError_t block_sums(const Launch &L, int wtype, const uint8_t *wrow, int k, const uint8_t *col, int32_t *out) {
    const int nb = k / 256;
    const size_t lds = tab_bytes_rt(wtype) + (size_t)act_col_bytes(wtype, k);
#define CALL_BODY                                                                                                      \
    auto kern = k_block_sums<WT, U, NB>;                                                                               \
    hipError_t e = allow_lds(kern, lds);                                                                               \
    if (e != hipSuccess) return e;                                                                                     \
    hipLaunchKernelGGL(kern, dim3(1), dim3(64), lds, L.stream, wrow, nb, col, out);
    BM_DISPATCH(wtype, nb)
#undef CALL_BODY
    return hipGetLastError();
}

} // namespace bmk

#ifdef BM_TIMELINE
// The table above, copied to the host: dst holds kTimelineRows * 8 words. Measurement builds only; not part of the C ABI.
extern "C" int bm_timeline_read(unsigned long long *dst) {
    return (int)hipMemcpyFromSymbol(dst, HIP_SYMBOL(bmk::g_timeline), sizeof(unsigned long long) * bmk::kTimelineRows * 8);
}
#endif
