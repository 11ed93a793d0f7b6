// The softmax router over given logits (crates/gpu/src/route_softmax.rs:1203 softmax_router_route, the routing body
// :177 route_warp): a token's probabilities, its top `used` experts by probability and their weights, renormalised
// to sum to one when the model's rule says so.
//
// Numbers, op for op (crates/model/src/moe.rs:246-279, crates/gpu/src/route_softmax.rs:38-51): the max of the logits
// (exact, any order); exp(logit - max) in f32; the sum of the exps in f64; each probability the f32 divide by the sum
// rounded to f32; the top `used` by descending probability, ties toward the smaller id; the chosen probabilities
// summed in f64 in slot order, rounded once, each weight the f32 divide of its probability by it.
// exp: the CPU path's is the host library's expf, correctly rounded in all but rare cases; here exp in f64 rounded to
// f32, which is the correctly rounded value in all but rare cases too. The f64 sums are taken lane by lane and then
// over the lanes (the order the reference's launch takes them in); they differ from a serial sum below 2^-50 of the
// sum, which its rounding to f32 hides except on an exact tie of that rounding.
//
// A token with a logit that is not finite has no defined routing: it raises Router on the fault word, gets NaN
// probabilities and weights, and keeps its ids as they stand (crates/gpu/src/route_softmax.rs:53-62).
#include <type_traits>

#include "bm_stream.hpp"

namespace bmk {

// Timeline of the router launch, in measurement builds only (-DBM_TIMELINE, the library bench.py --timeline loads): thread 0 of
// workgroup b keeps the device's constant-rate counter (100 MHz) in registers at six points of router_logits_body and stores
// them at its end in row b: start, the token's row arrived, normed, rows and token in LDS (behind the barrier), dots done,
// the routing done (the workgroup that routes: start, maximum known, exponentials summed, probabilities formed, logits held, routed,
// places found by the second wave).
#ifdef BM_TIMELINE
constexpr int kRouterTimelineRows = 1024;
__device__ unsigned long long g_router_timeline[kRouterTimelineRows * 8];
#define BM_RTICK(var, dep)                                                                                             \
    do {                                                                                                               \
        __asm__ volatile("" ::"v"(dep) : "memory");                                                                    \
        var = wall_clock64();                                                                                          \
    } while (0)
#define BM_RTOCK(mark, var)                                                                                            \
    do {                                                                                                               \
        if (threadIdx.x == 0 && blockIdx.x < (unsigned)kRouterTimelineRows) g_router_timeline[blockIdx.x * 8 + (mark)] = var; \
    } while (0)
#else
#define BM_RTICK(var, dep)                                                                                             \
    do {                                                                                                               \
    } while (0)
#define BM_RTOCK(mark, var)                                                                                            \
    do {                                                                                                               \
    } while (0)
#endif


typedef float v4f __attribute__((ext_vector_type(4)));

constexpr u32 kSiteRouter = 5; // crates/device/src/fault.rs:84-86

// Sum / maximum over the wave, every lane ending with it: pairs, quads, eights and sixteens by data-parallel-primitive moves, the
// two sixteens of a half and the two halves by row swaps (a few cycles each, where the LDS crossbar is a hundred). The sum's
// association: ((pairs) quads) ... halves.
struct Pair32 {
    u32 a, b;
};
// a: the lower row of sixteen of every half, in both its rows; b: the upper one (wave halves: the lower half, the upper half).
__device__ __forceinline__ Pair32 rows_of_half(u32 v) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return {r[0], r[1]};
}
__device__ __forceinline__ Pair32 halves(u32 v) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return {r[0], r[1]};
}
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    return __hiloint2double((int)bm_dpp<CTRL>((u32)__double2hiint(v)), (int)bm_dpp<CTRL>((u32)__double2loint(v)));
}
__device__ __forceinline__ double wave_sum_f64(double v) {
    v += dpp_f64<kDppXor1>(v);
    v += dpp_f64<kDppXor2>(v);
    v += dpp_f64<kDppHalfMirror>(v);
    v += dpp_f64<kDppMirror>(v);
    const Pair32 h = rows_of_half((u32)__double2hiint(v)), l = rows_of_half((u32)__double2loint(v));
    v = __hiloint2double((int)h.a, (int)l.a) + __hiloint2double((int)h.b, (int)l.b);
    const Pair32 hh = halves((u32)__double2hiint(v)), ll = halves((u32)__double2loint(v));
    return __hiloint2double((int)hh.a, (int)ll.a) + __hiloint2double((int)hh.b, (int)ll.b);
}
__device__ __forceinline__ float wave_max_f32(float v) {
    v = fmaxf(v, bm_dppf<kDppXor1>(v));
    v = fmaxf(v, bm_dppf<kDppXor2>(v));
    v = fmaxf(v, bm_dppf<kDppHalfMirror>(v));
    v = fmaxf(v, bm_dppf<kDppMirror>(v));
    const Pair32 r = rows_of_half(bm_f32_bits(v));
    v = fmaxf(bm_bits_f32(r.a), bm_bits_f32(r.b));
    const Pair32 h = halves(bm_f32_bits(v));
    return fmaxf(bm_bits_f32(h.a), bm_bits_f32(h.b));
}

// Token t's routing; lane L of a wave owns experts L + 64 j, j < PER. `v`: this lane's logits, expert lane + 64 j in v[j] (-inf past
// n_exp).
template <int PER>
__device__ __forceinline__ bool logits_finite(const float (&v)[PER], u32 n_exp) {
    bool odd = false;
#pragma unroll
    for (int j = 0; j < PER; j++) odd |= (threadIdx.x & 63) + 64 * j < n_exp && !(fabsf(v[j]) <= 3.402823466e38f);
    return __ballot(odd) == 0;
}
// A token with a logit that is not finite.
__device__ __forceinline__ void route_refuse(u32 t, u32 n_exp, u32 used, float *probs, float *weights, u32 *fault, u32 layer) {
    const u32 lane = threadIdx.x & 63;
    const float nan = bm_bits_f32(0x7fc00000u);
    if (probs)
        for (u32 e = lane; e < n_exp; e += 64) probs[(size_t)t * n_exp + e] = nan;
    if (lane < used) weights[(size_t)t * used + lane] = nan;
    if (lane == 0) bm_raise(fault, layer, kSiteRouter);
}
// The probabilities of finite logits, zero past n_exp.
template <int PER>
__device__ __forceinline__ void route_probs_wave(const float (&v)[PER], u32 n_exp, float (&p)[PER]) {
    const u32 lane = threadIdx.x & 63;
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < PER; j++) mx = fmaxf(mx, v[j]);
    mx = wave_max_f32(mx);
    [[maybe_unused]] unsigned long long tl_a = 0, tl_b = 0, tl_c = 0;
    BM_RTICK(tl_a, mx);
    double sum = 0.0;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        p[j] = lane + 64 * j < n_exp ? (float)exp((double)(v[j] - mx)) : 0.0f;
        sum += (double)p[j];
    }
    sum = wave_sum_f64(sum);
    BM_RTICK(tl_b, sum);
    const float inv = (float)sum;
#pragma unroll
    for (int j = 0; j < PER; j++) p[j] = p[j] / inv;
    BM_RTICK(tl_c, p[0]);
    BM_RTOCK(1, tl_a);
    BM_RTOCK(2, tl_b);
    BM_RTOCK(3, tl_c);
}
template <int PER>
__device__ __forceinline__ void store_probs(const float (&p)[PER], u32 t, u32 n_exp, float *probs) {
    if (!probs) return;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const u32 e = (threadIdx.x & 63) + 64 * j;
        if (e < n_exp) probs[(size_t)t * n_exp + e] = p[j];
    }
}

// The picks by the wave alone, where counting (below) has met a tie: `used` rounds of a wave argmax under (probability descending, id ascending): the
// largest probability left (its bits order as its value: not negative) as one unsigned maximum over the wave, then the
// smallest id that holds it: expert lane + 64 j, so the first j with a holder and that ballot's lowest lane. The winning
// lane marks its entry.
template <int PER>
__device__ __forceinline__ void route_pick_rounds(const float (&p)[PER], u32 t, u32 n_exp, u32 used, u32 renorm, u32 *ids,
                                                  float *weights) {
    const u32 lane = threadIdx.x & 63;
    u32 taken = 0;
    double chosen = 0.0;
    float mine = 0.0f;
    for (u32 s = 0; s < used; s++) {
        u32 best = 0;
        bool any = false;
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const bool open = lane + 64 * j < n_exp && !((taken >> j) & 1u);
            const u32 bits = bm_f32_bits(p[j]);
            best = open && bits > best ? bits : best;
            any |= open;
        }
        const u32 half = bm_max32(best);
        const u32 m0 = (u32)__builtin_amdgcn_readlane((int)half, 0), m1 = (u32)__builtin_amdgcn_readlane((int)half, 32);
        const u32 top = m0 > m1 ? m0 : m1;
        u32 bi = 0xffffffffu; // none left
        if (__ballot(any) != 0) {
#pragma unroll
            for (int j = PER - 1; j >= 0; j--) {
                const bool open = lane + 64 * j < n_exp && !((taken >> j) & 1u);
                const unsigned long long holders = __ballot(open && bm_f32_bits(p[j]) == top);
                if (holders) bi = (u32)(64 * j + __builtin_ctzll(holders)); // uniform; the smallest j wins: it comes last
            }
        }
        const float bv = bi != 0xffffffffu ? bm_bits_f32(top) : 0.0f;
        if ((bi & 63u) == lane && bi != 0xffffffffu) taken |= 1u << (bi >> 6);
        if (lane == 0) ids[(size_t)t * used + s] = bi;
        chosen += (double)bv;
        if (lane == s) mine = bv;
    }
    if (lane < used) weights[(size_t)t * used + lane] = renorm ? mine / (float)chosen : mine;
}

// A token's places (0 .. used, the last one past the picks) and probabilities in LDS.
constexpr u32 kNoExpert = 0xffffffffu;
template <int PER>
struct PickLds {
    __align__(16) float value[64]; // the entries that may be among the first, in any order
    u32 id[64];
    u32 at[kRouteMaxPicks + 1];
    float p[64 * PER];
};
// (between LDS stores and loads of one wave's lanes, which the LDS takes in order: for the compiler)
__device__ __forceinline__ void lds_of_wave() { __asm__ volatile("" ::: "memory"); }

// In front of places_by_counting, by its wave.
template <int PER>
__device__ __forceinline__ void places_clear(PickLds<PER> &L) {
    const u32 lane = threadIdx.x & 63;
    L.value[lane] = -INFINITY;
    if (lane <= (u32)kRouteMaxPicks) L.at[lane] = kNoExpert;
    lds_of_wave();
}

// The places of the first `used` + 1 entries in descending order of v, by one wave: at[r] = e for the entry e that r others are
// larger than. Entries of equal value have the same count: they take the same place and leave the next one as it was, so a
// caller finds out, and picks by rounds; so it does where more than 64 entries pass the bound (equal ones, or large ones crowded into few groups).
// Not every entry is compared with every other (128 of them: a quarter of it a wave, over LDS, took 0.9 us, and the rounds are a
// chain of eighty dependent instructions each): an entry below `used` + 1 others' maxima cannot be among the first, so the maxima of
// sixteen groups of lanes (of 32 for sixteen picks and more, of the 64 lanes for more still) give a bound that about as many entries pass as are
// wanted; those go to LDS, a lane each, and are compared with one another. A group costs a step of the count: of sixteen picks of 128 experts 4.2 us
// a k_route_softmax with 64 groups, 3.8 with 32. (Counts of 32 and 64 are one loop: as code of its own, which fewer picks jump over, the count of 32 made
// eight picks' k_route_softmax 5.0 -> 5.1 us and k_norm_route of 4 tokens x 256 experts x 7168 values 11.6 -> 12.4 where other launches stand between:
// instructions come from memory in order.) With no more than half again as many groups as picks too many entries pass (31 of 32 groups: the
// list overflows, 256 experts 5.3 -> 13.7 us; 24 of 32 past 256 experts 8.3 -> 17.6).
template <int PER>
__device__ __forceinline__ void places_by_counting(const float (&v)[PER], u32 n_exp, u32 used, PickLds<PER> &L) {
    const u32 lane = threadIdx.x & 63;
    float top = -INFINITY; // the lane's largest, then its group's
#pragma unroll
    for (int j = 0; j < PER; j++) top = fmaxf(top, lane + 64 * j < n_exp ? v[j] : -INFINITY);
    u32 above = 0; // groups with a larger maximum
    auto count_group = [&](u32 g) { above += bm_bits_f32((u32)__builtin_amdgcn_readlane((int)bm_f32_bits(top), (int)g)) > top ? 1u : 0u; };
    if (used < 16) {
        top = fmaxf(top, bm_dppf<kDppXor1>(top));
        top = fmaxf(top, bm_dppf<kDppXor2>(top));
#pragma unroll
        for (u32 g = 0; g < 64; g += 4) count_group(g);
    } else {
        const u32 lanes = used < (PER <= 4 ? 24u : 20u) ? 2 : 1;
        const float pair = fmaxf(top, bm_dppf<kDppXor1>(top));
        if (lanes == 2) top = pair;
        for (u32 g0 = 0; g0 < 64; g0 += 16 * lanes)
#pragma unroll
            for (u32 g = 0; g < 16; g++) count_group(g0 + g * lanes);
    }
    // the maximum with `used` above it: no entry below it is wanted (none, where maxima are equal or fewer: then every entry may be)
    const unsigned long long bound_at = __ballot(above == used);
    const float bound = bound_at ? bm_bits_f32((u32)__builtin_amdgcn_readlane((int)bm_f32_bits(top), __builtin_ctzll(bound_at))) : -INFINITY;
    u32 n = 0;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const bool in = lane + 64 * j < n_exp && v[j] >= bound;
        const unsigned long long who = __ballot(in);
        const u32 to = n + __builtin_amdgcn_mbcnt_hi((u32)(who >> 32), __builtin_amdgcn_mbcnt_lo((u32)who, 0));
        if (in && to < 64) L.value[to] = v[j], L.id[to] = lane + 64 * j;
        n += (u32)__builtin_popcountll(who);
    }
    if (n > 64) return;
    lds_of_wave();
    const float mine = L.value[lane];
    const u32 id = L.id[lane];
    u32 ahead = 0;
    for (u32 c = 0; c < n; c += 16) { // (the list ends in -inf)
        float4 o[4];
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = *reinterpret_cast<const float4 *>(&L.value[c + 4 * k]);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            ahead += o[k].x > mine ? 1u : 0u;
            ahead += o[k].y > mine ? 1u : 0u;
            ahead += o[k].z > mine ? 1u : 0u;
            ahead += o[k].w > mine ? 1u : 0u;
        }
    }
    if (lane < n && ahead <= used) L.at[ahead] = id;
    lds_of_wave();
}

// The picks of a token whose places and probabilities are in LDS, by one wave: false, with nothing stored, where two of the
// probabilities that decide are equal (two places' entries, or entries that share a place). Weights from the chosen
// probabilities added in pick order, as the rounds do.
template <int PER>
__device__ __forceinline__ bool picks_from_places(const PickLds<PER> &L, u32 t, u32 n_exp, u32 used, u32 renorm, u32 *ids, float *weights) {
    const u32 lane = threadIdx.x & 63, s = lane < used ? lane : used - 1;
    const u32 id = L.at[s], id_next = L.at[s + 1];
    const bool have_next = s + 1 < n_exp;
    const float p = L.p[id < n_exp ? id : 0], p_next = have_next ? L.p[id_next < n_exp ? id_next : 0] : -1.0f;
    if (__ballot(id == kNoExpert || (have_next && id_next == kNoExpert) || !(p > p_next)) != 0) return false;
    const float term = lane < used ? p : 0.0f;
    double chosen = 0.0;
    for (u32 i = 0; i < used; i += 8)
#pragma unroll
        for (u32 k = 0; k < 8; k++) chosen += (double)bm_bits_f32((u32)__builtin_amdgcn_readlane((int)bm_f32_bits(term), (int)(i + k)));
    if (lane < used) {
        ids[(size_t)t * used + lane] = id;
        weights[(size_t)t * used + lane] = renorm ? p / (float)chosen : p;
    }
    return true;
}

// A barrier that waits for the wave's LDS traffic only: the routing workgroup's waves meet over LDS while stores to memory are
// still on their way, and a barrier that waited for those to be acknowledged cost the routing 1 us.
__device__ __forceinline__ void lds_barrier() { __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// One wave a token. One or two picks (one, past 256 experts) go by the rounds: counting takes as long whatever their number (us a launch by rounds / by
// counting, 64 tokens and fewer: one pick of 128 experts 2.8 / 3.3, of 256 3.2 / 3.7; two 2.9 / 3.2, 3.6 / 3.7; two of 590 7.1 / 6.6). One copy of the
// rounds serves them and the ties.
template <int PER>
__global__ __launch_bounds__(256) void k_route_softmax(const float *logits, u32 n_tok, u32 n_exp, u32 used, u32 renorm,
                                                       float *probs, u32 *ids, float *weights, u32 *fault, u32 layer) {
    __shared__ PickLds<PER> s_pick[4];
    const u32 wave = (u32)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), t = blockIdx.x * 4 + wave;
    if (t >= n_tok) return; // whole waves leave
    PickLds<PER> &L = s_pick[wave];
    float v[PER], p[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const u32 e = (threadIdx.x & 63) + 64 * j;
        v[j] = e < n_exp ? logits[(size_t)t * n_exp + e] : -INFINITY;
    }
    if (!logits_finite<PER>(v, n_exp)) return route_refuse(t, n_exp, used, probs, weights, fault, layer);
    places_clear(L);
    route_probs_wave<PER>(v, n_exp, p);
    store_probs<PER>(p, t, n_exp, probs);
    if (used > (PER <= 4 ? 2u : 1u)) {
#pragma unroll
        for (int j = 0; j < PER; j++) L.p[(threadIdx.x & 63) + 64 * j] = p[j];
        places_by_counting<PER>(p, n_exp, used, L);
        if (picks_from_places(L, t, n_exp, used, renorm, ids, weights)) return;
    }
    route_pick_rounds<PER>(p, t, n_exp, used, renorm, ids, weights);
}

hipError_t route_softmax(const Launch &L, const float *logits, int n_tok, int n_exp, int used, int renorm, float *probs,
                         uint32_t *ids, float *weights) {
    const dim3 grid((unsigned)((n_tok + 3) / 4)), block(256);
    if (n_exp <= 128)
        hipLaunchKernelGGL(k_route_softmax<2>, grid, block, 0, L.stream, logits, (u32)n_tok, (u32)n_exp, (u32)used, (u32)renorm,
                           probs, ids, weights, L.fault, L.layer);
    else if (n_exp <= 256)
        hipLaunchKernelGGL(k_route_softmax<4>, grid, block, 0, L.stream, logits, (u32)n_tok, (u32)n_exp, (u32)used, (u32)renorm,
                           probs, ids, weights, L.fault, L.layer);
    else
        hipLaunchKernelGGL(k_route_softmax<16>, grid, block, 0, L.stream, logits, (u32)n_tok, (u32)n_exp, (u32)used,
                           (u32)renorm, probs, ids, weights, L.fault, L.layer);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------- the norm and the router's logits

// The FFN norm and the router's f32 logits of m tokens (crates/gpu/src/route_softmax.rs:1667-1674 enqueue_norm_fused does
// norm, quantizer and routing in one launch; here the norm and the logits are this launch, the routing
// k_route_softmax's, and the quantizer is folded into the expert launches). Numbers, op for op: the norm
// (crates/model/src/ops.rs:350-368) sums the f32 squares in f64 - lane by lane and then over the lanes; any order gives
// the same f32 mean except on an exact tie of that rounding, as the reference notes of its own two orders - narrows the
// mean to f32, takes scale = 1 / sqrt(mean + eps) and writes (scale * gain) * x; a logit is the f32 row dot of
// crates/qdot/src/lib.rs:11349-11386: eight lane accumulators (a product, then fused multiply-adds in increasing k) and
// (l0 + l4 + l2 + l6) + (l1 + l5 + l3 + l7).
//
// A workgroup takes T tokens and R router rows: the tokens' rows are normed into LDS by all 256 threads, then a wave takes a row.
//
// A row dot is eight chains of hidden / 8 fused multiply-adds, serial by the order's definition: a chain's steps cost 6 cycles each
// when their operands stand in registers, and what they cost more than that is the operands' way there (eight lanes a row,
// reading four steps at a time from LDS: 11 cycles a step, and the rows had to be laid out accumulator-major for it). So a row is
// spread over the whole wave: lane 8 l + s holds the 32 operands of accumulator l in super-block s of eight (256 values, 32 steps),
// read by one instruction a step for all the lanes - the router's row from memory, eight lanes of which are 32 consecutive bytes,
// the token's from LDS, whose super-blocks stand eight floats more than their length apart so that a wave's 64 words fall on 64
// banks. Then the chains run super-block by super-block: every lane does its 32 steps, only the lanes of the chains' present place
// with a meaning, and a move to the next lane hands the accumulators on.
constexpr int kRouterSb = 256 + 8; // floats from one super-block of a token's row in LDS to the next
__host__ __device__ constexpr int router_line(int hidden) { return (hidden + 255) / 256 * kRouterSb; }
// Super-blocks of a router row that a wave has in LDS at a time (n4: see norm_rows): of short rows no more than they have, which lets the more
// workgroups stand on a compute unit (eight of them throughout: rows of 304 to 760 values took up to 1.39 times as long as with eight lanes a row).
__host__ __device__ constexpr int router_lines(int n4, int hidden) {
    const int sbs = (hidden + 255) / 256;
    return n4 == 1 ? 4 : n4 == -2 && sbs < 8 ? sbs : 8;
}

// (k_norm_route's arguments: what the head of a logits workgroup needs stands in the first fourteen words, which are in registers when a
// wave starts - m_word is the token count, bit 31 set where the quantized column is asked for - and the rest travels as one
// struct behind them that a workgroup reads when it gets there: see bm_kernarg_at.)
struct NormRouteLate {
    u32 used, renorm;
    float *probs;
    u32 *ids;
    float *weights;
    u32 *hand;
    uint8_t *act_x;
    int q8k;
    u32 layer;
    u32 *fault;
    u32 max_polls, unused;
};
struct NormRouteArgs { // k_norm_route's argument block
    const float *router, *x, *gain;
    float eps;
    int n_exp, hidden;
    u32 m_word;
    float *normed_out, *logits;
    NormRouteLate late;
};
static_assert(offsetof(NormRouteArgs, late) == 56, "fourteen words in front of the late arguments");

// The norm of T rows (of tokens t0 .., the last token's where there are fewer: its numbers again) into LDS, row after row of
// router_line(hidden) floats, without a barrier behind it; and to normed_out where that is wanted. Without a gain the rows as they are. N4: 16-byte
// pieces of a row a thread holds in registers (rows of whole super-blocks and up to 1024 N4 values; -2, -4: as many, and any rows of so many values);
// 0: rows of any length, through LDS. `behind_requests` is
// called when the rows have been asked for, `behind_sums` when their squares are summed.
template <int T, int N4, class F, class G>
__device__ __forceinline__ void norm_rows(float *xs, double (*s_part)[4], const float *x, const float *gain, float eps, int hidden, float *normed_out,
                                          int t0, int m, F behind_requests, G behind_sums) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n4 = hidden / 4, line = router_line(hidden);
    auto in_lds = [&](int tt, int i) { return reinterpret_cast<float4 *>(xs + tt * line + 4 * i + 8 * (i >> 6)); };
    auto row = [&](int tt) { return (size_t)(t0 + tt < m ? t0 + tt : m - 1) * hidden; };
    auto squares = [](double &sum, const float4 v) {
        sum += (double)__fmul_rn(v.x, v.x);
        sum += (double)__fmul_rn(v.y, v.y);
        sum += (double)__fmul_rn(v.z, v.z);
        sum += (double)__fmul_rn(v.w, v.w);
    };
    auto normed = [](float scale, const float4 g, const float4 v) {
        return make_float4(__fmul_rn(__fmul_rn(scale, g.x), v.x), __fmul_rn(__fmul_rn(scale, g.y), v.y), __fmul_rn(__fmul_rn(scale, g.z), v.z),
                           __fmul_rn(__fmul_rn(scale, g.w), v.w));
    };
    auto put = [&](int tt, int i, const float4 v) {
        *in_lds(tt, i) = v;
        if (normed_out && t0 + tt < m) reinterpret_cast<float4 *>(normed_out + row(tt))[i] = v;
    };
    constexpr bool kInRegs = N4 != 0, kRagged = N4 <= 0;
    constexpr int kRegs = N4 > 0 ? N4 : N4 < 0 ? -N4 : 1;
    [[maybe_unused]] float4 xv[T][kRegs], gv[kRegs];
    [[maybe_unused]] unsigned long long tl_row = 0, tl_norm = 0;
    double sum[T];
#pragma unroll
    for (int tt = 0; tt < T; tt++) sum[tt] = 0.0;
    if constexpr (kInRegs) {
#pragma unroll
        for (int tt = 0; tt < T; tt++)
#pragma unroll
            for (int j = 0; j < kRegs; j++)
                if (tid + 256 * j < n4) xv[tt][j] = reinterpret_cast<const float4 *>(x + row(tt))[tid + 256 * j];
        if (gain)
#pragma unroll
            for (int j = 0; j < kRegs; j++)
                if (tid + 256 * j < n4) gv[j] = reinterpret_cast<const float4 *>(gain)[tid + 256 * j];
        behind_requests();
        if (gain)
#pragma unroll
            for (int tt = 0; tt < T; tt++)
#pragma unroll
                for (int j = 0; j < kRegs; j++)
                    if (tid + 256 * j < n4) squares(sum[tt], xv[tt][j]);
    } else {
        behind_requests();
        for (int tt = 0; tt < T; tt++)
            for (int i = tid; i < n4; i += 256) {
                const float4 v = reinterpret_cast<const float4 *>(x + row(tt))[i];
                if (gain) {
                    *in_lds(tt, i) = v;
                    squares(sum[tt], v);
                } else {
                    put(tt, i, v);
                }
            }
    }
    if constexpr (kRagged) // the steps past a row's end, to a whole super-block: -0, which times +0 leaves a chain as it is
        for (int tt = 0; tt < T; tt++)
            for (int k = hidden + tid; k < (hidden + 255) / 256 * 256; k += 256) xs[tt * line + k + 8 * (k >> 8)] = -0.0f;
    BM_RTICK(tl_row, sum[0]);
    BM_RTOCK(1, tl_row);
    if (!gain) {
        behind_sums();
        if constexpr (kInRegs)
#pragma unroll
            for (int tt = 0; tt < T; tt++)
#pragma unroll
                for (int j = 0; j < kRegs; j++)
                    if (tid + 256 * j < n4) put(tt, tid + 256 * j, xv[tt][j]);
        return;
    }
#pragma unroll
    for (int tt = 0; tt < T; tt++) {
        sum[tt] = wave_sum_f64(sum[tt]);
        if (lane == 0) s_part[tt][wave] = sum[tt];
    }
    lds_barrier();
    double part[T][4];
#pragma unroll
    for (int tt = 0; tt < T; tt++)
#pragma unroll
        for (int k = 0; k < 4; k++) part[tt][k] = s_part[tt][k];
    behind_sums();
    float scale[T];
#pragma unroll
    for (int tt = 0; tt < T; tt++) {
        const double total = (part[tt][0] + part[tt][1]) + (part[tt][2] + part[tt][3]);
        const float mean = (float)(total / (double)hidden);
        scale[tt] = __fdiv_rn(1.0f, bm_sqrt_rn(__fadd_rn(mean, eps)));
    }
    BM_RTICK(tl_norm, scale[0]);
    BM_RTOCK(2, tl_norm);
    if constexpr (kInRegs) {
#pragma unroll
        for (int tt = 0; tt < T; tt++)
#pragma unroll
            for (int j = 0; j < kRegs; j++)
                if (tid + 256 * j < n4) put(tt, tid + 256 * j, normed(scale[tt], gv[j], xv[tt][j]));
    } else {
        for (int tt = 0; tt < T; tt++)
            for (int i = tid; i < n4; i += 256) // (a thread's own pieces)
                put(tt, i, normed(scale[tt], reinterpret_cast<const float4 *>(gain)[i], *in_lds(tt, i)));
    }
}

// The logits of tokens t0 .. t0 + T - 1 against router rows e0 .. e0 + R - 1. A wave takes one row and all the
// tokens, whose chains run side by side. N4: see norm_rows. Rows of one pass (up to eight super-blocks) hold one set of operands: registers a
// lane 74 (up to 1024 values), 100 (2048), 168 (4096, two sets), 186, of two tokens 99, 116, 234; ragged ones up to six more.
template <int R, int T, int N4, bool COH>
__device__ __forceinline__ void router_logits_body(uint8_t *lds, const float *router, const float *x, const float *gain, float eps, int n_exp,
                                                   int hidden, int m, float *normed_out, float *logits, int t0, int e0) {
    static_assert((R == 1 && T == 1) || R == 4, "a wave takes one row, and all the tokens");
    float *const xs = reinterpret_cast<float *>(lds);
    __shared__ double s_part[T][4];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    [[maybe_unused]] unsigned long long tl_start = 0, tl_lds = 0, tl_dots = 0;
    BM_RTICK(tl_start, tid);
    BM_RTOCK(0, tl_start);
    const int r = wave; // the wave's row
    const bool has_dot = wave < R;
    const int acc_l = lane >> 3, sb_l = lane & 7, line = router_line(hidden), sbs = (hidden + 255) / 256;
    constexpr bool kRagged = N4 <= 0, kOnePass = N4 == 1 || N4 == 2 || N4 == -2; // (rows of up to 1024, 2048 values)
    const int passes = kOnePass ? 1 : (sbs + 7) / 8;
    constexpr int kLines = N4 == 1 ? 4 : 8;
    constexpr bool kFewer = N4 == -2;
    const int lines = router_lines(N4, hidden);
    const float *const wrow = router + (size_t)(e0 + r < n_exp ? e0 + r : n_exp - 1) * hidden;
    struct Row { // a lane's operands of a pass
        float w[32], x[T][32];
    };
    // The router's row comes in whole lines, a super-block an instruction, and goes through the wave's own eight super-blocks of LDS:
    // asked for straight into the lanes that use it, 32 bytes here and there, it kept the address unit busy for 33 cycles an instruction.
    float4 *const ws = reinterpret_cast<float4 *>(xs + T * line + wave * (lines * kRouterSb));
    v4f raw[kLines];
    auto ask = [&](int q) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kLines; i++) {
            if (kFewer && i >= lines) break;
            const int sb = 8 * q + i < sbs ? 8 * q + i : sbs - 1, at = 256 * sb + 4 * lane; // (past the row's end: its last, for no reader)
            if constexpr (!kRagged) {
                raw[i] = *reinterpret_cast<const v4f *>(wrow + at);
            } else {
                const bool in = at < hidden;
                raw[i] = *reinterpret_cast<const v4f *>(wrow + (in ? at : hidden - 4));
                if (!in) raw[i] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
    };
    auto park = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kLines; i++)
            if (!kFewer || i < lines) *reinterpret_cast<v4f *>(ws + (kRouterSb / 4) * i + lane) = raw[i];
        lds_of_wave();
    };
    auto read_row = [&](Row &o) __attribute__((always_inline)) {
        const float *const from = reinterpret_cast<const float *>(ws) + kRouterSb * (sb_l < lines ? sb_l : lines - 1) + acc_l;
#pragma unroll
        for (int j = 0; j < 32; j++) o.w[j] = from[8 * j];
        lds_of_wave();
    };
    auto read_token = [&](Row &o, int q) __attribute__((always_inline)) {
        const int sb = 8 * q + sb_l < sbs ? 8 * q + sb_l : sbs - 1;
        const float *const from = xs + kRouterSb * sb + acc_l;
#pragma unroll
        for (int tt = 0; tt < T; tt++)
#pragma unroll
            for (int j = 0; j < 32; j++) o.x[tt][j] = from[tt * line + 8 * j];
    };
    Row a, b;
    norm_rows<T, N4>(xs, s_part, x, gain, eps, hidden, e0 == 0 ? normed_out : nullptr, t0, m, [&]() __attribute__((always_inline)) {
        if (has_dot) ask(0);
    }, [&]() __attribute__((always_inline)) {
        if (!has_dot) return;
        park();
        if (passes > 1) ask(1);
        read_row(a);
    });
    lds_barrier();
    BM_RTICK(tl_lds, tid);
    BM_RTOCK(3, tl_lds);
    if (!has_dot) return;
    // (k_norm_route's hand-over words: an argument behind the preloaded ones, read here, where its way through memory runs under
    // the dots)
    [[maybe_unused]] u32 *hand = nullptr;
    if constexpr (COH) hand = bm_global(bm_kernarg_at<u32 *>(offsetof(NormRouteArgs, late) + offsetof(NormRouteLate, hand)));
    float acc[T];
#pragma unroll
    for (int tt = 0; tt < T; tt++) acc[tt] = -0.0f; // (a first product keeps its own sign of zero, as the product that starts the chain does)
    auto steps = [&](const Row &o) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 32; j++)
#pragma unroll
            for (int tt = 0; tt < T; tt++) acc[tt] = fmaf(o.x[tt][j], o.w[j], acc[tt]);
    };
    auto pass = [&](const Row &o, int q, auto behind_first) __attribute__((always_inline)) {
        if (q > 0)
#pragma unroll
            for (int tt = 0; tt < T; tt++) acc[tt] = bm_dppf<kDppShl7>(acc[tt]); // from the eighth super-block's lanes to the first's
        steps(o);
        behind_first();
        const int here = sbs - 8 * q < 8 ? sbs - 8 * q : 8;
#pragma nounroll
        for (int sb = 1; sb < here; sb++) {
#pragma unroll
            for (int tt = 0; tt < T; tt++) acc[tt] = bm_dppf<kDppShr1>(acc[tt]);
            steps(o);
        }
    };
    read_token(a, 0);
    // two sets of operands: a pass's are read, and the bytes of the one after it asked for, while the pass before runs
    auto prepare = [&](Row &o, int q) __attribute__((always_inline)) {
        park();
        if (q + 1 < passes) ask(q + 1);
        read_row(o);
        read_token(o, q);
    };
    // (behind the pass's first super-block: the counter of LDS reads on their way ends at fifteen, and a wait for the pass's own in
    // front of its first step would be one for the next pass's)
    for (int q = 0;; q += 2) {
        pass(a, q, [&]() __attribute__((always_inline)) {
            if (q + 1 < passes) prepare(b, q + 1);
        });
        if (q + 1 >= passes) break;
        pass(b, q + 1, [&]() __attribute__((always_inline)) {
            if (q + 2 < passes) prepare(a, q + 2);
        });
        if (q + 2 >= passes) break;
    }
    // s_l = acc_l + acc_{l+4}, then (s0 + s2) + (s1 + s3): accumulators 4 apart stand a half of the wave apart, 2 apart a row of
    // sixteen, neighbours eight lanes
    const int last = (sbs - 1) & 7; // the lanes of the last super-block hold the sums
#pragma unroll
    for (int tt = 0; tt < T; tt++) {
        const Pair32 h = halves(bm_f32_bits(acc[tt]));
        const float s = __fadd_rn(bm_bits_f32(h.a), bm_bits_f32(h.b));
        const Pair32 q = rows_of_half(bm_f32_bits(s));
        const float pair = __fadd_rn(bm_bits_f32(q.a), bm_bits_f32(q.b));
        const float out = __fadd_rn(pair, bm_dppf<kDppShl8>(pair));
        BM_RTICK(tl_dots, out);
        const int t = t0 + tt;
        if (lane == last && e0 + r < n_exp && t < m) {
            // k_norm_route's hand-over: the logit as a device-scope store of its own, into a word that held the armed pattern
            if constexpr (COH) __hip_atomic_store(hand + (size_t)t * n_exp + e0 + r, bm_f32_bits(out), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            logits[(size_t)t * n_exp + e0 + r] = out;
        }
    }
    BM_RTOCK(4, tl_dots);
}

template <int R, int T, int N4>
__global__ __launch_bounds__(256) void k_router_logits(const float *router, const float *x, const float *gain, float eps, int n_exp, int hidden, int m,
                                                       float *normed_out, float *logits) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int row_blocks = (n_exp + R - 1) / R;
    router_logits_body<R, T, N4, false>(lds, router, x, gain, eps, n_exp, hidden, m, normed_out, logits, (int)(blockIdx.x / row_blocks) * T,
                                        (int)(blockIdx.x % row_blocks) * R);
}

// A normed row as norm_rows leaves it in LDS into column t of act_x.
__device__ __forceinline__ void quant_normed_row(const float *xs, int hidden, int t, uint8_t *act_x, int q8k, u32 *fault, u32 layer) {
    const int nb = hidden / 256, tid = threadIdx.x;
    if (q8k) {
        uint8_t *col = act_x + (size_t)t * nb * BM_Q8K_STRIDE;
        for (int b = tid >> 6; b < nb; b += 4) // a wave a 256-value block, four consecutive values a lane
            q8k_wave_block(*reinterpret_cast<const float4 *>(xs + kRouterSb * b + 4 * (tid & 63)), col + (size_t)b * BM_Q8K_STRIDE, tid & 63, fault, layer);
    } else {
        uint8_t *col = act_x + (size_t)t * nb * BM_Q82_SB_EXT;
        for (int k = 8 * tid; k < hidden; k += 2048) { // a quad of lanes a 32-value block, eight consecutive values a lane
            const float4 *at = reinterpret_cast<const float4 *>(xs + k + 8 * (k >> 8));
            const float4 lo = at[0], hi = at[1];
            const float v8[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            q82_quad8(v8, col, nb, k >> 5, tid & 3, fault, layer);
        }
    }
}

// Norm, logits and routing in one launch (crates/gpu/src/route_softmax.rs:1667-1674 enqueue_norm_fused; the quantizer of
// that launch is an option here, see below). The workgroups are k_router_logits's, and behind them in the grid one more a
// token, which routes it with k_route_softmax's numbers. The hand-over is one trip through memory: `hand` holds a
// word a (token, expert) that is armed between launches - kRouteArmed, a signalling NaN pattern, which no arithmetic
// leaves behind (an operation on it gives the quiet form) - each logit is stored over its word with a device-scope store as
// soon as it is formed, and the routing waves read their words with device-scope loads until none is armed, so they have the
// logits the moment the last one lands: no acknowledgement is waited for, no count is kept, nothing is read back (a count
// raised behind acknowledged stores by the last workgroup to finish, which then read the logits back, took 2.3 us longer). Two polls are on
// their way at once (5.5 us a token against 5.7 with one, 5.75 with four). Two waves have the logits: the first forms the probabilities
// while the second finds the places - by the logits, whose order the probabilities have but where two of them round to the same
// value, which picks_from_places sees - and the first picks. It arms the words again before it ends, so a graph replay
// needs no memset. A routing workgroup comes after every workgroup it waits for in the grid, so those are dispatched
// whatever else the card runs; the wait is bounded all the same (max_polls polls, kRoutePolls = 2^24 or some ten seconds unless the caller says otherwise - an XCD busy with another stream's work may hold some of them back for
// a while - then BM_SITE_ROUTER and NaN weights), and
// every wave ends. Launches over the same `hand` must not overlap.
// With act_x (the reference launch's quantizer, route_softmax.rs:1679): one more workgroup a token, between the two kinds in
// the grid, norms the token's row the same way and leaves it as the token's quantized column (q8k: a Q8_K column, else a
// Q8_2_X4 one with its tables), the bytes bm_quantize makes of normed_out. The routing waits for none of it.
// Latency: 1 token x 128 experts x 2048 values 7.9 -> 5.5 us a launch (us after its start: row arrived 0.6, normed 1.2, in LDS 1.4, dots done
// 2.3 - 2.4, logits held 3.5, routed 4.6; before: 0.9, 1.25, 1.9, 3.5 - 4.0, 5.0, 7.1), 16 tokens 11.0 -> 7.7, 4 tokens x 256 x 7168 22.1 -> 10.9.
template <int R, int T, int N4, int PER>
__global__ __launch_bounds__(256) void k_norm_route(const float *router, const float *x, const float *gain, float eps, int n_exp,
                                                    int hidden, u32 m_word, float *normed_out, float *logits, NormRouteLate) {
    extern __shared__ __align__(16) uint8_t lds[];
    const u32 row_blocks = (u32)((n_exp + R - 1) / R);
    const u32 m = m_word & 0x7fffffffu;
    const u32 n_logit_blocks = (m + T - 1) / T * row_blocks, n_quant_blocks = (m_word >> 31) ? m : 0u;
    if (blockIdx.x >= n_logit_blocks + n_quant_blocks) { // a routing workgroup: two waves of it
        const u32 wave = (u32)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        if (wave > 1) return;
        __shared__ PickLds<PER> pick;
        const u32 t = blockIdx.x - n_logit_blocks - n_quant_blocks, lane = threadIdx.x & 63;
        const NormRouteLate late = bm_kernarg_at<NormRouteLate>(offsetof(NormRouteArgs, late));
        const u32 used = late.used, renorm = late.renorm, layer = late.layer, max_polls = late.max_polls;
        float *const probs = bm_global(late.probs), *const weights = bm_global(late.weights);
        u32 *const ids = bm_global(late.ids), *const hand = bm_global(late.hand), *const fault = bm_global(late.fault);
        u32 *const mine = hand + (size_t)t * n_exp;
        if (wave == 1) places_clear(pick);
        [[maybe_unused]] unsigned long long tl_start = 0, tl_seen = 0, tl_places = 0, tl_routed = 0;
        BM_RTICK(tl_start, lane);
        // (several polls on their way at once, spread over the time one takes: the logits are seen that much sooner after they are there)
        constexpr int kPolls = 2;
        u32 w[kPolls][PER];
        auto poll = [&](u32(&o)[PER]) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < PER; j++) {
                const u32 e = lane + 64 * j;
                o[j] = e < (u32)n_exp ? __hip_atomic_load(mine + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
            }
        };
        u32 got[PER];
        bool waiting = true;
#pragma unroll
        for (int k = 0; k < kPolls; k++) {
            poll(w[k]);
            __builtin_amdgcn_s_sleep(4);
        }
        for (u32 spin = 0; waiting; spin += kPolls) {
#pragma unroll
            for (int k = 0; k < kPolls; k++) {
                bool armed = false;
#pragma unroll
                for (int j = 0; j < PER; j++) {
                    got[j] = w[k][j];
                    armed |= got[j] == kRouteArmed;
                }
                waiting = __ballot(armed) != 0 && spin + k + 1 < max_polls;
                if (!waiting) break;
                poll(w[k]);
            }
        }
        BM_RTICK(tl_seen, got[0]);
        float v[PER], p[PER];
#pragma unroll
        for (int j = 0; j < PER; j++) // (a word still armed after the last poll: the NaN it is, which is refused as any is)
            v[j] = lane + 64 * j < (u32)n_exp ? bm_bits_f32(got[j]) : -INFINITY;
        const bool finite = logits_finite<PER>(v, (u32)n_exp);
        if (wave == 1) {
            if (finite) places_by_counting<PER>(v, (u32)n_exp, used, pick);
            BM_RTICK(tl_places, lane);
        } else {
            route_probs_wave<PER>(v, (u32)n_exp, p);
#pragma unroll
            for (int j = 0; j < PER; j++) pick.p[lane + 64 * j] = p[j];
        }
        lds_barrier();
#ifdef BM_TIMELINE
        if (wave == 1 && lane == 0 && blockIdx.x < (unsigned)kRouterTimelineRows) g_router_timeline[blockIdx.x * 8 + 6] = tl_places;
#endif
        if (wave == 1) return;
        // (both waves have their logits: the words are armed again)
#pragma unroll
        for (int j = 0; j < PER; j++)
            if (lane + 64 * j < (u32)n_exp) __hip_atomic_store(mine + lane + 64 * j, kRouteArmed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (!finite) return route_refuse(t, (u32)n_exp, used, probs, weights, fault, layer);
        if (!picks_from_places(pick, t, (u32)n_exp, used, renorm, ids, weights))
            route_pick_rounds<PER>(p, t, (u32)n_exp, used, renorm, ids, weights);
        store_probs<PER>(p, t, (u32)n_exp, probs);
        BM_RTICK(tl_routed, threadIdx.x);
        BM_RTOCK(0, tl_start);
        BM_RTOCK(4, tl_seen);
        BM_RTOCK(5, tl_routed);
        return;
    }
    if (blockIdx.x >= n_logit_blocks) { // a quantizer workgroup
        const int tq = (int)(blockIdx.x - n_logit_blocks);
        __shared__ double s_part[1][4];
        norm_rows<1, N4>(reinterpret_cast<float *>(lds), s_part, x, gain, eps, hidden, nullptr, tq, (int)m, []() {}, []() {});
        lds_barrier();
        const NormRouteLate late = bm_kernarg_at<NormRouteLate>(offsetof(NormRouteArgs, late));
        uint8_t *const act_x = bm_global(late.act_x);
        u32 *const fault = bm_global(late.fault);
        const u32 layer = late.layer;
        const int q8k = late.q8k;
        quant_normed_row(reinterpret_cast<const float *>(lds), hidden, tq, act_x, q8k, fault, layer);
        return;
    }
    router_logits_body<R, T, N4, true>(lds, router, x, gain, eps, n_exp, hidden, (int)m, normed_out, logits, (int)(blockIdx.x / row_blocks) * T,
                                       (int)(blockIdx.x % row_blocks) * R);
}

// ---- many tokens

// The norm of many tokens' rows, a workgroup a token: into normed_out and, with act_x, into the token's quantized column.
template <int N4>
__global__ __launch_bounds__(256) void k_norm_rows(const float *x, const float *gain, float eps, int hidden, float *normed_out, uint8_t *act_x,
                                                   int q8k, u32 *fault, u32 layer) {
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ double s_part[1][4];
    const int t = (int)blockIdx.x;
    norm_rows<1, N4>(reinterpret_cast<float *>(lds), s_part, x, gain, eps, hidden, normed_out, t, t + 1, []() {}, []() {});
    if (!act_x) return;
    lds_barrier();
    quant_normed_row(reinterpret_cast<const float *>(lds), hidden, t, act_x, q8k, fault, layer);
}

// The logits of many tokens' normed rows: tiles of tokens x experts on the matrix cores. v_mfma_f32_16x16x4_f32 runs four steps of
// a 16 x 16 tile's multiply-add chains in increasing k, each with one rounding - fmaf's bits, subnormal values and signed zeros
// included (checked over millions of values) - so accumulator l of a row dot is a chain of these instructions over its places,
// and the logits are k_router_logits's bit for bit. Lane (row = lane % 16, s = lane / 16) of the instruction for accumulator l
// holds value 8 (4 i + s) + l of its row, so over the eight accumulators a lane's operands are eight consecutive values. The chain
// starts at -0 (a first product then keeps its own sign of zero, as the product that starts the CPU path's chain does), and
// the places past a row's end hold -0 x 0.
// A workgroup is four waves:
//   SPLIT = 1: 16 tokens x 64 experts, a tile and its eight accumulators a wave;
//   SPLIT = 4: the waves share one 16 x 16 tile, two accumulators each, which meet in LDS: a chain is then a quarter of the matrix
//     instructions, the form for batches whose tiles would leave most of the card idle (it brings twice the bytes a value to LDS).
// Both sides go through LDS in chunks of KC values a row, pieces of 16 bytes swizzled by the row's number so that sixteen rows at
// one place fall on sixteen different bank groups. Three chunks: while chunk i is multiplied, chunk i + 1 is there already (so
// operands are read a step ahead of their use, over the chunks' ends too), and chunk i + 2 goes in over chunk i - 1. The loads
// (five chunks ahead), LDS stores and LDS reads stand one by one between the matrix instructions, in whose shadow they issue.
// Without RAGGED the loop has no branch: a branch round an LDS store (for the padding of a last chunk) cost 55 ns a store, as
// much as four matrix instructions, so rows that are whole groups of four chunks have a form of their own.
// No unit is full (2048 tokens: one wave a SIMD, matrix cores busy 40 % of the cycles, LDS 23 %, vector ALU 12 %, waiting 23 %; 4096:
// 52, 31, 15, 19 %): a wave's chain of matrix instructions, 256 cycles a step of 32 values, is stretched by the LDS accesses that stand
// between them (26 KB a step and workgroup). Two tiles of experts a wave, which halve the reads of a matrix instruction, were no faster
// (39.1 against 39.8 us at 4096 tokens: half the workgroups). Measured, with the norm's launch, against workgroups of a token each: 4096 tokens x 128 experts x 2048 values
// 827 -> 40 us, 2048 tokens 416 -> 25, 333 tokens 71 -> 13.7, 64 tokens 16.7 -> 11.1; 1024 tokens x 256 experts x 7168 values
// 2867 -> 64 us. Workgroups of a token or two read the router's rows once a token or two.
template <int SPLIT, int KC, bool RAGGED>
__global__ __launch_bounds__(256) void k_router_tiles(const float *router, const float *x, int m, int n_exp, int hidden, float *logits) {
    constexpr int kTok = 16, kExp = SPLIT == 1 ? 64 : 16, kAcc = 8 / SPLIT, kRows = kTok + kExp;
    constexpr int kLine = KC / 4;                 // 16-byte pieces of a row's chunk
    constexpr int kLoads = kRows * kLine / 256;   // pieces a thread brings in a chunk, of rows 256 / kLine apart,
    constexpr int kTokLoads = kTok * kLine / 256; // the first of them pieces of tokens' rows
    constexpr int kSteps = KC / 32, kSlots = kSteps * kAcc, kRing = 4;
    static_assert(SPLIT == 1 || SPLIT == 4, "four waves: a tile each, or two accumulators of one tile each");
    static_assert(kTok * kLine % 256 == 0 && kExp * kLine % 256 == 0 && KC % 64 == 0 && 256 % kLine == 0, "whole pieces a thread");
    static_assert(2 * kLoads <= kSlots, "a slot of the chain for every load and every LDS store");
    static_assert(kSteps % 2 == 0, "the two sets of operands alternate over whole chunks");
    constexpr int kChunk = kRows * kLine;
    extern __shared__ __align__(16) uint8_t lds[];
    float4 *const s_buf = reinterpret_cast<float4 *>(lds); // three chunks: [kRows][kLine]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int exp_groups = (n_exp + kExp - 1) / kExp;
    const int t0 = (int)(blockIdx.x / exp_groups) * kTok, e0 = (int)(blockIdx.x % exp_groups) * kExp;
    const int chunks = (hidden + KC - 1) / KC, n4 = hidden / 4;
    // what this thread brings of every chunk: piece `col` of rows row0, row0 + 256 / kLine, ..., tokens first
    const int col = tid % kLine, row0 = tid / kLine;
    const uint8_t *const x0 = reinterpret_cast<const uint8_t *>(x + (size_t)t0 * hidden);
    const uint8_t *const w0 = reinterpret_cast<const uint8_t *>(router + (size_t)e0 * hidden);
    u32 src[kLoads];
    int dst[kLoads];
#pragma unroll
    for (int j = 0; j < kLoads; j++) {
        const int r = row0 + 256 / kLine * j;
        const int in_tile = j < kTokLoads ? (t0 + r < m ? r : m - 1 - t0) : (e0 + r - kTok < n_exp ? r - kTok : n_exp - 1 - e0);
        src[j] = (u32)in_tile * (u32)hidden * 4u + 16u * (u32)col;
        dst[j] = r * kLine + (col ^ (r & 15));
    }
    // (places past a row's end, in the last chunk and behind it: the row's last piece, which park replaces)
    const int past = col - (n4 - 1 - (chunks - 1) * kLine);
    const u32 tail = past > 0 ? 16u * (u32)past : 0u;
    float4 ring[kRing][kLoads];
    auto fetch = [&](int i, int j, float4(&v)[kLoads]) {
        const int c = i < chunks ? i : chunks - 1;
        const u32 back = RAGGED && i >= chunks - 1 ? tail : 0u;
        v[j] = *reinterpret_cast<const float4 *>((j < kTokLoads ? x0 : w0) + (size_t)c * (KC * 4) + (src[j] - back));
    };
    auto park = [&](int i, int j, int buf, const float4(&v)[kLoads]) { // a piece into LDS
        float4 w = v[j];
        if (RAGGED && (i >= chunks || (i == chunks - 1 && past > 0))) {
            const float pad = j < kTokLoads ? -0.0f : 0.0f;
            w = make_float4(pad, pad, pad, pad);
        }
        s_buf[buf + dst[j]] = w;
    };
#pragma unroll
    for (int u = 0; u < kRing; u++)
#pragma unroll
        for (int j = 0; j < kLoads; j++) fetch(u, j, ring[u]);
    const int l16 = lane & 15, ks = lane >> 4;
    const int wexp = SPLIT == 1 ? 16 * wave : 0; // this wave's experts of the workgroup's
    const int l0 = SPLIT == 1 ? 0 : kAcc * wave; // this wave's first accumulator
    v4f acc[kAcc];
#pragma unroll
    for (int l = 0; l < kAcc; l++) acc[l] = v4f{-0.0f, -0.0f, -0.0f, -0.0f};
    struct Step { // a lane's operands of 32 values: kAcc consecutive ones of its token's row and of its expert's row
        float a[kAcc], b[kAcc];
    };
    // piece `part` of a step's operands, of kParts: values 8 (4 s + ks) + l0 .. of the lane's token row (first) and of its expert's
    constexpr int kRowParts = kAcc == 2 ? 1 : 2, kParts = 2 * kRowParts;
    static_assert(kParts <= kAcc, "a slot of the chain for every LDS read");
    auto rd = [&](int buf, int s, int part, Step &st) {
        const bool exp = part >= kRowParts;
        const int j = part % kRowParts, r = exp ? kTok + wexp + l16 : l16;
        float(&v)[kAcc] = exp ? st.b : st.a;
        const float4 *row = s_buf + buf + r * kLine;
        const int p = 8 * s + 2 * ks;
        if constexpr (kAcc == 2) {
            const float2 q = *reinterpret_cast<const float2 *>(reinterpret_cast<const float *>(row + ((p + (wave >> 1)) ^ (r & 15))) + 2 * (wave & 1));
            v[0] = q.x, v[1] = q.y;
        } else {
            const float4 q = row[(p + j) ^ (r & 15)];
            v[4 * j] = q.x, v[4 * j + 1] = q.y, v[4 * j + 2] = q.z, v[4 * j + 3] = q.w;
        }
    };
    int now = 0, next = kChunk, over = 2 * kChunk; // the buffers of chunks i, i + 1, i + 2
#pragma unroll
    for (int j = 0; j < kLoads; j++) park(0, j, now, ring[0]);
#pragma unroll
    for (int j = 0; j < kLoads; j++) fetch(kRing, j, ring[0]);
#pragma unroll
    for (int j = 0; j < kLoads; j++) park(1, j, next, ring[1]);
    lds_barrier();
    Step st[2];
#pragma unroll
    for (int r = 0; r < kParts; r++) rd(now, 0, r, st[0]);
    for (int i = 0; i < chunks; i += kRing) {
#pragma unroll
        for (int u = 0; u < kRing; u++) {
#pragma unroll
            for (int s = 0; s < kSteps; s++) {
#pragma unroll
                for (int l = 0; l < kAcc; l++) {
                    __builtin_amdgcn_sched_barrier(0);
                    acc[l] = __builtin_amdgcn_mfma_f32_16x16x4f32(st[s & 1].a[l], st[s & 1].b[l], acc[l], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (l < kParts) rd(s + 1 < kSteps ? now : next, (s + 1) % kSteps, l, st[(s + 1) & 1]);
                    const int slot = s * kAcc + l;
                    if (slot < kLoads) fetch(i + u + 1 + kRing, slot, ring[(u + 1) % kRing]);
                    if (slot >= kSlots - kLoads) park(i + u + 2, slot - (kSlots - kLoads), over, ring[(u + 2) % kRing]);
                }
            }
            lds_barrier();
            const int done = now;
            now = next, next = over, over = done;
        }
    }
    // s_l = acc_l + acc_{l+4}, then (s_0 + s_2) + (s_1 + s_3); result v of a tile is token 4 ks + v against expert l16
    if constexpr (SPLIT == 1) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const float s0 = __fadd_rn(acc[0][v], acc[4][v]), s1 = __fadd_rn(acc[1][v], acc[5][v]);
            const float s2 = __fadd_rn(acc[2][v], acc[6][v]), s3 = __fadd_rn(acc[3][v], acc[7][v]);
            const int t = t0 + 4 * ks + v, ex = e0 + wexp + l16;
            if (t < m && ex < n_exp) logits[(size_t)t * n_exp + ex] = __fadd_rn(__fadd_rn(s0, s2), __fadd_rn(s1, s3));
        }
    } else {
        __shared__ float s_acc[8][16][17];
#pragma unroll
        for (int l = 0; l < kAcc; l++)
#pragma unroll
            for (int v = 0; v < 4; v++) s_acc[l0 + l][4 * ks + v][l16] = acc[l][v];
        __syncthreads();
        const int r = tid >> 4, c = tid & 15;
        float s[4];
#pragma unroll
        for (int l = 0; l < 4; l++) s[l] = __fadd_rn(s_acc[l][r][c], s_acc[l + 4][r][c]);
        if (t0 + r < m && e0 + c < n_exp) logits[(size_t)(t0 + r) * n_exp + e0 + c] = __fadd_rn(__fadd_rn(s[0], s[2]), __fadd_rn(s[1], s[3]));
    }
}

// LDS of a workgroup of so many tokens, whose dots take so many waves.
static constexpr size_t router_lds_bytes(int tokens, int waves, int hidden, int n4) {
    return ((size_t)tokens * router_line(hidden) + (size_t)waves * router_lines(n4, hidden) * kRouterSb) * sizeof(float);
}

// The longest rows the router takes are the entries' contract (kRouteMaxHidden); every form's LDS holds them beside its arrays of fixed size.
static_assert(router_lds_bytes(1, 4, kRouteMaxHidden, 0) + sizeof(PickLds<16>) + 1024 <= (size_t)kMaxLds, "four rows a workgroup, rows of any length");
static_assert(router_lds_bytes(2, 4, 4096, 4) + sizeof(PickLds<16>) + 1024 <= (size_t)kMaxLds, "four rows and two tokens, rows of up to 4096 values");
bool router_logits_fits(int hidden) { return hidden <= kRouteMaxHidden; }

// Router rows and tokens a workgroup takes. A row and a token each while that leaves no more workgroups than stand on the card at once: a
// launch of few workgroups is a wave's chain behind the norm of its token's row, and nothing is shorter than one of each (rows of up to 1024
// values are so short that sharing the norm soon pays). Then four rows a token, a wave each, and from three workgroups a compute unit on two tokens
// a workgroup, which ask for a row's bytes once: where that needs fewer rounds over the card. A compute unit holds two workgroups of 4 x 2 and three of
// 4 x 1 of rows of 2304 to 4096 values (so 4 x 2 between one round of the one and of the other), two of either where such rows are ragged,
// as many as have work of the short whole rows (always 4 x 1).
// (us a launch, 1 x 1 / 4 x 1 / 4 x 2, 128 experts: 2048 values 1 token 5.5 / 6.2 / 7.4, 8 tokens 7.0 / 6.4 / 7.8; 4096 values 4 tokens 7.7 / 8.5 / 10.4, 8 tokens
// 11.9 / 8.8 / 10.7; 7168 values 4 tokens 9.9 / 10.3 / 13.5. 3300 random launches of 8 to 8192 values, by such fours: 1300 to 2048 values 900 fours
// 1.15 / 1.0 and 1.04 / 1.0 times the better of 4 x 1 and 4 x 2, 768 1.0 / 1.07; 4096 values 640 1.0 / 1.04, 900 1.12 / 1.0, 1300 1.0 / 1.04; up to 1024 values
// 1.0 / 1.05 at 1300, ragged 1.07 / 1.0.)
enum RouterForm { kForm1x1, kForm4x1, kForm4x2 };
static long router_fours(int m, int n_exp) { return (long)m * ((n_exp + 3) / 4); }
static RouterForm router_form(int m, int n_exp, int hidden) {
    const bool ragged = hidden % 256 != 0;
    const long fours = router_fours(m, n_exp);
    if ((long)m * n_exp <= (hidden <= 1024 ? 256 : hidden <= 4096 && !ragged ? 640 : 512)) return kForm1x1;
    if (hidden <= 1024) return ragged && fours > 1024 ? kForm4x2 : kForm4x1;
    if (hidden <= 2048) return fours > 768 ? kForm4x2 : kForm4x1;
    if (hidden <= 4096) return (ragged ? fours > 512 : fours > 768 && fours <= 1024) ? kForm4x2 : kForm4x1;
    return kForm4x1;
}

// Calls f with the form's rows and tokens and the pieces of a row a thread holds as constants.
// (The order is the kernels' order in the library: the forms of whole rows together, in front. k_norm_route of 4 tokens x 256 experts x 7168 values among
// a layer's other launches, us: 12.2 behind the ragged forms' kernels, 11.4 in front of them.)
template <class F>
static hipError_t with_form(RouterForm form, int hidden, F f) {
    using std::integral_constant;
    constexpr integral_constant<int, 1> one{};
    constexpr integral_constant<int, 2> two{};
    constexpr integral_constant<int, 4> four{};
    auto tokens = [&](auto n4) { return form == kForm1x1 ? f(one, one, n4) : form == kForm4x1 ? f(four, one, n4) : f(four, two, n4); };
    if (hidden % 256 == 0) {
        if (hidden <= 1024) return tokens(one);
        if (hidden <= 2048) return tokens(two);
        if (hidden <= 4096) return tokens(four);
        if (hidden <= 8192) return tokens(integral_constant<int, 8>{});
    }
    if (hidden <= 2048) return tokens(integral_constant<int, -2>{});
    if (hidden <= 4096) return tokens(integral_constant<int, -4>{});
    return tokens(integral_constant<int, 0>{});
}

// Whether the norm and the logits go as two launches, rows and then tiles: by workgroups of four rows, from the later the shorter the rows, whose
// workgroups are the cheaper (and the more of them stand on a compute unit), and whose tiles are mostly their launch. (one launch / the tiles' two,
// with the routing's as well where it is asked for, as times the better: up to 1024 values 2500 of them 1.0 / 1.13 to 1.18, 3500 1.08 / 1.03; 1280 to 2048
// values 1800 1.01 / 1.14, 2200 1.09 / 1.04, ragged 2500 1.0 / 1.1, 3500 1.09 / 1.0; 2304 to 4096 values 1400 1.0 / 1.2, 1800 1.09 / 1.07, ragged 1800 1.0 / 1.09,
// 2500 1.13 / 1.0; longer 1200 1.0 / 1.2, 1400 1.07 / 1.06.) The tiles read normed rows from memory: a caller that wants none of them stays with the workgroups that norm their own.
static bool router_tiled(int m, int n_exp, int hidden, const float *gain, const float *normed_out) {
    const bool ragged = hidden % 256 != 0;
    const int from = hidden <= 1024 ? 3072 : hidden <= 2048 ? (ragged ? 3072 : 2048) : hidden <= 4096 ? (ragged ? 2048 : 1536) : 1280;
    return router_fours(m, n_exp) > from && (!gain || normed_out);
}

static hipError_t router_tiles(const Launch &L, const float *router, const float *x, const float *gain, float eps, int m, int n_exp,
                               int hidden, float *normed_out, float *logits, uint8_t *act_x = nullptr, bool q8k = false) {
    if (normed_out || act_x) {
        const size_t lds = router_lds_bytes(1, 0, hidden, 0);
        auto kern = hidden % 256 != 0 || hidden > 8192 ? k_norm_rows<0> : hidden > 2048 ? k_norm_rows<8> : k_norm_rows<2>;
        hipError_t e = allow_lds(kern, lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kern, dim3((unsigned)m), dim3(256), lds, L.stream, x, gain, eps, hidden, normed_out, act_x, q8k ? 1 : 0, L.fault,
                           L.layer);
    }
    auto launch = [&](auto kern, unsigned grid, unsigned rows, unsigned kc) {
        const size_t lds = 3 * (size_t)rows * kc * sizeof(float);
        hipError_t e = allow_lds(kern, lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kern, dim3(grid), dim3(256), lds, L.stream, router, normed_out ? normed_out : x, m, n_exp, hidden, logits);
        return hipGetLastError();
    };
    const unsigned t16 = (unsigned)((m + 15) / 16), e16 = (unsigned)((n_exp + 15) / 16), e64 = (e16 + 3) / 4;
    // up to two split workgroups a compute unit (777 tokens x 128 experts: split 19.9, a tile a wave 24.0 us; 2048 tokens: 33.9 and 24.9)
    if ((long)t16 * e16 <= 512)
        return hidden % 512 ? launch(k_router_tiles<4, 128, true>, t16 * e16, 32, 128) : launch(k_router_tiles<4, 128, false>, t16 * e16, 32, 128);
    return hidden % 256 ? launch(k_router_tiles<1, 64, true>, t16 * e64, 80, 64) : launch(k_router_tiles<1, 64, false>, t16 * e64, 80, 64);
}

hipError_t router_logits(const Launch &L, const float *router, const float *x, const float *gain, float eps, int m, int n_exp,
                         int hidden, float *normed_out, float *logits) {
    if (router_tiled(m, n_exp, hidden, gain, normed_out)) return router_tiles(L, router, x, gain, eps, m, n_exp, hidden, normed_out, logits);
    if (!router_logits_fits(hidden)) return hipErrorInvalidValue;
    return with_form(router_form(m, n_exp, hidden), hidden, [&](auto r, auto t, auto n4) {
        auto kern = k_router_logits<decltype(r)::value, decltype(t)::value, decltype(n4)::value>;
        const size_t lds = router_lds_bytes(t, r, hidden, n4);
        hipError_t e = allow_lds(kern, lds);
        if (e != hipSuccess) return e;
        const unsigned grid = (unsigned)((m + t - 1) / t) * (unsigned)((n_exp + r - 1) / r);
        hipLaunchKernelGGL(kern, dim3(grid), dim3(256), lds, L.stream, router, x, gain, eps, n_exp, hidden, m, normed_out, logits);
        return hipGetLastError();
    });
}

hipError_t norm_route(const Launch &L, const float *router, const float *x, const float *gain, float eps, int m, int n_exp,
                      int hidden, float *normed_out, float *logits, int used, int renorm, float *probs, uint32_t *ids,
                      float *weights, uint32_t *hand, uint8_t *act_x, bool q8k, uint32_t max_polls) {
    if (!router_logits_fits(hidden)) return hipErrorInvalidValue;
    if (act_x && hidden % 256 != 0) return hipErrorInvalidValue;
    if (router_tiled(m, n_exp, hidden, gain, normed_out)) {
        const hipError_t e = router_tiles(L, router, x, gain, eps, m, n_exp, hidden, normed_out, logits, act_x, q8k);
        return e != hipSuccess ? e : route_softmax(L, logits, m, n_exp, used, renorm, probs, ids, weights);
    }
    return with_form(router_form(m, n_exp, hidden), hidden, [&](auto r, auto t, auto n4) {
        constexpr int R = decltype(r)::value, T = decltype(t)::value, N4 = decltype(n4)::value;
        auto kern = n_exp <= 128 ? k_norm_route<R, T, N4, 2> : n_exp <= 256 ? k_norm_route<R, T, N4, 4> : k_norm_route<R, T, N4, 16>;
        const size_t lds = router_lds_bytes(T, R, hidden, N4);
        hipError_t e = allow_lds(kern, lds);
        if (e != hipSuccess) return e;
        const unsigned grid = (unsigned)((m + T - 1) / T) * (unsigned)((n_exp + R - 1) / R) + (act_x ? (unsigned)m : 0u) + (unsigned)m;
        hipLaunchKernelGGL(kern, dim3(grid), dim3(256), lds, L.stream, router, x, gain, eps, n_exp, hidden,
                           (u32)m | (act_x ? 0x80000000u : 0u), normed_out, logits,
                           NormRouteLate{(u32)used, (u32)renorm, probs, ids, weights, hand, act_x, q8k ? 1 : 0, L.layer, L.fault, max_polls, 0u});
        return hipGetLastError();
    });
}

} // namespace bmk

#ifdef BM_TIMELINE
// The router's table, copied to the host: dst holds 1024 * 8 words. Measurement builds only; not part of the C ABI.
extern "C" int bm_router_timeline_read(unsigned long long *dst) {
    return (int)hipMemcpyFromSymbol(dst, HIP_SYMBOL(bmk::g_router_timeline), sizeof(unsigned long long) * bmk::kRouterTimelineRows * 8);
}
#endif
