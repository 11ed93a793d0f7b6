// Prefill, tolerance mode (BM_GEMM_FAST): the grouped expert GEMM of IQ2_XXS stacks on the f16 matrix cores. (Launches too small
// for its workgroups go to k_gemm_iq's int8 form: the line is in gemm, bm_prefill.hip.)
//
// A row against a Q8_K column is, a super-block, (d / 8) dy times sum over the 256 values of ((2 s + 1) g) a: g = +-8, 25 or 43 the
// grid's value, 2 s + 1 the sub-block's scale, a the column's code. The term (2 s + 1) g is an integer of at most 1333 and exact in
// f16, so is a, so one v_mfma_f32_32x32x16_f16 does what takes two int8 products on split bytes, and the sum stays in its f32
// accumulators for the whole super-block: one multiply-add a (row, slot, super-block) is all that is left of the scaling.
//
// The sum is the exact integer, rounded once where it becomes the multiply-add's operand, as an int32 sum would be. An f32 accumulator
// holds it exactly while every partial sum is at most 2^24, which sum |a| <= 2^24 / 1333 over the column's block guarantees: the
// staging adds the |a| up beside its conversions, and a super-block with a column past that (about one in 2 x 10^5 blocks of normal
// values, every block whose values have one magnitude) is summed again by `wide_block`, which closes into integers every
// 64 terms (64 x 1333 x 128 < 2^24). The guard is some twenty of 750 vector instructions a super-block: 2 to 5 % of the kernel, 2.3 %
// of the layer below (2.28 -> 2.33 ms).
//
// Bound by the vector ALU, which makes the terms, 16 instructions for eight values a lane, with LDS (the grid, the columns) and the
// weights' scattered lines close behind: an expert has about as many slots as one tile, so every weight is unpacked about once
// and used for one 32- or 64-slot product. So:
//   * a wave takes 64 rows and all slots of the tile: no weight is unpacked twice, none goes through LDS, a column operand serves two
//     row groups;
//   * a lane owns a row (lane % 32) and sixteen bytes (lane / 32) of each 32 of a super-block in the file, so that two lanes next to
//     each other ask for 32 contiguous bytes of a row;
//   * a grid entry is two eight-byte halves of f16 values, in sixteen copies that start on sixteen different bank pairs: the lookups
//     of a wave, 64 different entries, never collide (a single copy collides about three deep). An entry's address is one byte
//     permute of the index and the lane's copy;
//   * signs are shifted out of the seven-bit field and its parity straight into the f16 sign bits;
//   * the terms of a 16-value step are made between the matrix instructions of the step before, and a super-block's bytes are asked for
//     a whole super-block ahead, one request every second step (one a step: 1 to 2 % slower; a wave's request covers 32 rows, and
//     eight waves asking at once fill the address unit's queue);
//   * a row group's lookups go out as soon as its last terms are made, half a step earlier than both groups' at the step's end. That, the
//     order of the requests and three vector instructions less a lookup (the LDS base, a multiplication by 2^14 + 1 and its wait state):
//     600 tokens of 64 experts 265 -> 255 us a layer, 192 tokens of 7168 values 497 -> 472, 1024 tokens of the large layer 2.34 -> 2.29 ms;
//   * tiles of at most 32 slots leave the second slot group out; a gate and an up are one launch, whose last round of workgroups
//     is then half as much of the whole.
// 133 KB of LDS, one workgroup of eight waves a CU. 8192 slots of 256 experts, gate and up of 2048 rows of 7168 values:
// 2 x 1266 -> 1232 us; down of 7168 rows of 2048: 1266 -> 693 us, against int8 products on split bytes through LDS. The weights alone
// take 376 and 188 us from memory. Counters of the pair: vector ALU 62 % of the cycles, matrix cores 29 %, LDS 41 % (a third of that
// bank conflicts), the address units 58 % (a lane's sixteen bytes lie at odd multiples of two), a wave waits a third of its time, at the
// super-block's barrier and for LDS: two waves a SIMD, no unit full. Sixteen waves of 32 rows instead, four a SIMD, were 3 to 15 % slower
// (twice the column reads), a table of spread signs in LDS no faster. (These times are without the guard above.)
#include "bm_gemm.hpp"

namespace bmk {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef u32 v2u __attribute__((ext_vector_type(2)));
typedef u32 v4u __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) uint8_t *LdsB;
// volatile: eight-byte reads stay eight bytes (merged into sixteen they run at half the rate)
typedef const volatile __attribute__((address_space(3))) v2u *LdsV2;

constexpr int kIqThreads = 512, kIqWgRows = 512; // eight waves of 64 rows
constexpr int kGridBytes = 256 * 256;            // an entry: sixteen copies of the first half, sixteen of the second
constexpr int kIqColStride = 2 * 256 + 8;        // a column's 256 codes as f16: 8 x an odd number
constexpr int kIqCols = 64 * kIqColStride;
struct IqLds {
    uint8_t grid[kGridBytes];
    uint8_t cols[2][kIqCols];
    float dy[2][64];
    u32 mag[2][4][64]; // sum |a| of a column's block, in as many parts as thread quads stage it
    GemmLds tab;
};
constexpr u32 kIqMagMax = (1u << 24) / (31u * 43u);

// (x & mask) | bits in one instruction; from the plain expression the compiler makes two.
__device__ __forceinline__ u32 iq_and_or(u32 x, u32 mask, u32 bits) {
    u32 r;
    __asm__("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(mask), "v"(bits));
    return r;
}
// x | x << 14. (Left to the compiler it becomes a multiplication and a wait state behind it.)
__device__ __forceinline__ u32 iq_twice14(u32 x) {
    u32 r;
    __asm__("v_lshl_or_b32 %0, %1, 14, %1" : "=v"(r) : "v"(x));
    return r;
}
// Bits 0 and 16 of x into the sign bits of a pair of f16 values that have none: a product modulo 2^16 and a sum.
__device__ __forceinline__ u32 iq_low_bit_sign(u32 x, u32 pair) {
    u32 r;
    __asm__("v_pk_mad_u16 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(0x80008000u), "v"(pair));
    return r;
}
__device__ __forceinline__ u32 iq_f16_pair(float a, float b) {
    return __builtin_bit_cast(u32, (v2h){(_Float16)a, (_Float16)b});
}

// One row slab after another of a tile, NCT groups of 32 slots of it.
template <int NCT>
__device__ __forceinline__ void iq2_tile(uint8_t *lds, const uint8_t *we, const uint8_t *act, int rpe, int nb, int row0, int slabs, int len, float *y) {
    IqLds *L = reinterpret_cast<IqLds *>(lds);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const u32 row_bytes = (u32)nb * BM_IQ2XXS_BLOCK, col_bytes = (u32)nb * BM_Q8K_STRIDE;
    // What a thread stages of a super-block: one or two runs of sixteen codes of one column.
    const int sc = NCT == 2 ? (tid >> 2) & 63 : (tid >> 2) & 31, sq = (tid & 3) + 4 * (NCT == 2 ? tid >> 8 : tid >> 7);
    const u32 src = L->tab.col[sc] * col_bytes + 8u + 16u * (u32)sq;
    const LdsB my_put = (LdsB)lds + kGridBytes + sc * kIqColStride + 32 * sq;
    constexpr int kMagParts = 4 / NCT;
    u32 mag; // sum |a| of what this thread stages
    constexpr int kPieces = NCT; // of sixteen codes: NCT 2: pieces sq and sq + 8 of the sixteen, NCT 1: piece sq
    v4u ra[kPieces];
    float cdy = 0.0f;
    auto fetch_cols = [&](int i) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < kPieces; q++) __builtin_memcpy(&ra[q], act + (src + (u32)i * BM_Q8K_STRIDE) + 128 * q, 16);
        cdy = *reinterpret_cast<const float *>(act + (src + (u32)i * BM_Q8K_STRIDE) - 8); // (the block's scale where sq is 0, else unused)
    };
    const u32 k1024 = 0x64006400u, m8 = 0x00ff00ffu, msign = 0x80008000u;
    auto less_1152 = [](u32 x) {
        const _Float16 b = (_Float16)1152.0f;
        return __builtin_bit_cast(u32, __builtin_bit_cast(v2h, x) - (v2h){b, b});
    };
    auto stash_word = [&](int at, int k) __attribute__((always_inline)) { // of 4 kPieces; `at`: the buffer
        const u32 u = ra[k >> 2][k & 3] ^ 0x80808080u;
        mag = __builtin_amdgcn_sad_u8(u, 0x80808080u, k ? mag : 0u);
        *(__attribute__((address_space(3))) v2u *)(my_put + at + 256 * (k >> 2) + 8 * (k & 3)) =
            (v2u){less_1152(iq_and_or(u, m8, k1024)), less_1152(iq_and_or(u >> 8, m8, k1024))};
    };

    auto mag_quad = [&]() __attribute__((always_inline)) { // over the quad of lanes, 64 or 128 codes of one column
        mag += (u32)__builtin_amdgcn_mov_dpp((int)mag, 0xb1, 0xf, 0xf, true); // lane ^ 1
        mag += (u32)__builtin_amdgcn_mov_dpp((int)mag, 0x4e, 0xf, 0xf, true); // lane ^ 2
    };
    auto stash_ends = [&](int buf) __attribute__((always_inline)) { // the sum, and the column's scale
        if ((sq & 3) == 0) {
            L->mag[buf][sq >> 2][sc] = mag;
            if (sq == 0) L->dy[buf][sc] = cdy;
        }
    };

    const int l32 = lane & 31, kh = lane >> 5;
    const u32 my_copy = 8u * (u32)(lane & 15);
    const LdsB my_col = (LdsB)lds + kGridBytes + l32 * kIqColStride + 128 * kh;
    v16f acc[2][NCT], sum[2][NCT]; // [row group][slot group]; result v: slot 8 (v / 4) + 4 kh + v % 4, row l32
    v4u raw[2][2], ahead[2][2]; // [row group][q]: sub-blocks 4 q + 2 kh and the next: index word, sign/scale word, twice; the next block's
    u32 rd;                     // the next block's d of row group kh
    u32 wofs[2], dofs; // where this lane's requests for rows start
    v2u gr[2][2];   // [row group][half]: a grid entry
    v4u term[2][2]; // [step % 2][row group]
    v4u colv[NCT];  // [slot group]
    u32 scale[2];   // [row group] (2 s + 1) twice, f16
    // Two lanes next to each other ask for one row's 32 bytes (they share a line; lanes 32 apart would look it up twice), and the
    // pieces are dealt to the lanes that own them through the LDS crossbar.
    auto fetch_raw = [&](int i, int n) __attribute__((always_inline)) { // request n of five
        const u32 at = (u32)i * BM_IQ2XXS_BLOCK;
        if (n < 4) __builtin_memcpy(&ahead[n & 1][n >> 1], we + (wofs[n & 1] + at) + 2 + 32 * (n >> 1), 16);
        else rd = bm_ld2u(we + (dofs + at));
    };
    const int owner = 4 * (2 * l32 + kh);
    auto deal = [&](int q) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int k = 0; k < 4; k++) raw[r][q][k] = (u32)__builtin_amdgcn_ds_bpermute(owner, (int)ahead[r][q][k]);
    };
    float d[2]; // the row's d / 8
    auto take_d = [&]() __attribute__((always_inline)) {
        const float mine = 0.125f * bm_half_to_f32((unsigned short)rd), other = __shfl_xor(mine, 32);
        d[0] = kh ? other : mine;
        d[1] = kh ? mine : other;
    };
    // The eight values that byte j of an index word stands for: the grid's magnitudes, and with signs and scale from the other word.
    auto grid_of = [&](u32 index, int j, v2u(&half)[2]) __attribute__((always_inline)) {
        const u32 at = __builtin_amdgcn_perm(index, my_copy, 0x0c0c0000u | ((4u + (u32)j) << 8));
        // (the grid is where LDS starts: with the array's own address, a zero that only the linker fills in, each lookup would add it)
        half[0] = *(LdsV2)(uintptr_t)at;
        half[1] = *(LdsV2)(uintptr_t)(at + 128u);
    };
    auto scale_of = [&](u32 aux) __attribute__((always_inline)) { // 1024 + 2 s + 1 less 1024
        const u32 x = (2u * (aux >> 28)) | 0x6401u, b = x | (x << 16);
        const _Float16 k = (_Float16)1024.0f;
        return __builtin_bit_cast(u32, __builtin_bit_cast(v2h, b) - (v2h){k, k});
    };
    auto terms_of = [&](u32 aux, int j, const v2u(&half)[2], u32 scale_pair) __attribute__((always_inline)) {
        const u32 v = (aux >> (7 * j)) & 127u;
        const u32 v8 = v | ((u32)__builtin_popcount(v) << 7); // bit 7: the parity
        const u32 s = iq_twice14(v8); // bits 0, 1, 4, 5 and sixteen on: the signs of values 0, 1, 4, 5 and 2, 3, 6, 7
        const u32 m[4] = {iq_low_bit_sign(s, half[0].x), iq_and_or(s << 14, msign, half[0].y), iq_and_or(s << 11, msign, half[1].x),
                          iq_and_or(s << 10, msign, half[1].y)};
        v4u out;
#pragma unroll
        for (int k = 0; k < 4; k++) out[k] = __builtin_bit_cast(u32, __builtin_bit_cast(v2h, m[k]) * __builtin_bit_cast(v2h, scale_pair));
        return out;
    };
    // step t of sixteen: eight values of index byte t % 4 of the lane's sub-block t / 4
    auto lookup = [&](int t, int r) __attribute__((always_inline)) { grid_of(raw[r][t >> 3][2 * ((t >> 2) & 1)], t & 3, gr[r]); };
    auto make = [&](int t, int r) __attribute__((always_inline)) {
        const u32 aux = raw[r][t >> 3][2 * ((t >> 2) & 1) + 1];
        if ((t & 3) == 0) scale[r] = scale_of(aux);
        term[t & 1][r] = terms_of(aux, t & 3, gr[r], scale[r]);
    };
    auto read_col = [&](int at, int t, int c) __attribute__((always_inline)) {
        const LdsB p = my_col + at + 32 * kIqColStride * c + 256 * (t >> 3) + 16 * (t & 7);
        const v2u a = *(LdsV2)p, b = *(LdsV2)(p + 8);
        colv[c] = (v4u){a.x, a.y, b.x, b.y};
    };

    // A super-block's rows asked for and made ready, none of it in the shade of products: a slab's first one, and around a wide one.
    auto rows_of = [&](int i) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < 5; n++) fetch_raw(i, n);
        deal(0);
        deal(1);
        lookup(0, 0);
        lookup(0, 1);
        make(0, 0);
        make(0, 1);
        lookup(1, 0);
        lookup(1, 1);
    };
    // the super-block's scaled sums into the accumulators of slot group c
    auto scale_sums = [&](int buf, int c) __attribute__((always_inline)) {
        const float *dy = L->dy[buf];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const v4f y4 = *reinterpret_cast<const v4f *>(dy + 32 * c + 8 * q + 4 * kh);
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int r = 0; r < 2; r++) acc[r][c][4 * q + k] = fmaf(d[r] * y4[k], sum[r][c][4 * q + k], acc[r][c][4 * q + k]);
        }
    };
    u32 mag_all; // sum |a| of a column of the super-block at hand
    auto read_mag = [&](int buf) __attribute__((always_inline)) {
        const int col = NCT == 2 ? lane : l32;
        mag_all = L->mag[buf][0][col];
#pragma unroll
        for (int p = 1; p < kMagParts; p++) mag_all += L->mag[buf][p][col];
    };
    // The sums of such a super-block, closed into integers every 64 terms. (A loop that stays one: unrolled, what its passes have in
    // common was kept in registers that the products behind it do not leave.)
    auto wide_block = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < NCT; c++)
#pragma unroll
            for (int r = 0; r < 2; r++) {
                v16i whole = {};
#pragma nounroll
                for (int n = 0; n < 4; n++) {
                    const v4u words = n < 2 ? raw[r][0] : raw[r][1];
                    const u32 index = n & 1 ? words.z : words.x, aux = n & 1 ? words.w : words.y, by = scale_of(aux);
                    const LdsB col = my_col + buf * kIqCols + 32 * kIqColStride * c + 256 * (n >> 1) + 64 * (n & 1);
                    v16f part = {};
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        v2u half[2];
                        grid_of(index, j, half);
                        const v2u a0 = *(LdsV2)(col + 16 * j), a1 = *(LdsV2)(col + 16 * j + 8);
                        const v4u a = {a0.x, a0.y, a1.x, a1.y}, b = terms_of(aux, j, half, by);
                        part = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), part, 0, 0, 0);
                    }
#pragma unroll
                    for (int v = 0; v < 16; v++) whole[v] += (int)part[v];
                }
#pragma unroll
                for (int v = 0; v < 16; v++) sum[r][c][v] = (float)whole[v];
                __builtin_amdgcn_sched_barrier(0);
            }
    };

    for (int left = (int)slabs; left > 0 && row0 < rpe; left--, row0 += kIqWgRows) {
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int row = row0 + 64 * wv + 32 * r + l32;
            const int asked = row0 + 64 * wv + 32 * r + (lane >> 1);
            wofs[r] = (u32)(asked < rpe ? asked : rpe - 1) * row_bytes + 16u * (u32)(lane & 1);
            if (r == kh) dofs = (u32)(row < rpe ? row : rpe - 1) * row_bytes;
#pragma unroll
            for (int c = 0; c < NCT; c++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[r][c][v] = 0.0f;
        }
        fetch_cols(0);
        rows_of(0);
#pragma unroll
        for (int k = 0; k < 4 * kPieces; k++) stash_word(0, k);
        mag_quad();
        stash_ends(0);
        __syncthreads();
        for (int i = 0; i < nb; i++) {
            const int next = i + 1 < nb ? i + 1 : i, now_at = (i & 1) * kIqCols, next_at = kIqCols - now_at; // the last one's staging has no reader
            const v16f z = {};
            read_col(now_at, 0, 0);
            if (NCT == 2) read_col(now_at, 0, NCT - 1);
            fetch_cols(next); // before the rows' bytes: loads come back in order, and these are waited for first
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 16; t++) {
                // the matrix instructions of step t; between them the terms of step t + 1 and what is read for the steps behind
                auto product = [&](int r, int c) __attribute__((always_inline)) {
                    sum[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, colv[c]), __builtin_bit_cast(v8h, term[t & 1][r]),
                                                                      t ? sum[r][c] : z, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                };
                product(0, 0);
                make((t + 1) & 15, 0);
                lookup((t + 2) & 15, 0);
                __builtin_amdgcn_sched_barrier(0);
                product(1, 0);
                if (t < 15) read_col(now_at, t + 1, 0);
                if (t % 2 == 0 && t < 8) fetch_raw(next, t / 2); // (a run of them fills the address unit's queue and stops the wave)
                if (t == 8) {
                    take_d();
                    fetch_raw(next, 4);
                }
                if (t >= 16 - 4 * kPieces) stash_word(next_at, t - (16 - 4 * kPieces));
                __builtin_amdgcn_sched_barrier(0);
                if (NCT == 2) product(0, NCT - 1);
                make((t + 1) & 15, 1);
                lookup((t + 2) & 15, 1);
                __builtin_amdgcn_sched_barrier(0);
                if (NCT == 2) product(1, NCT - 1);
                if (NCT == 2 && t < 15) read_col(now_at, t + 1, NCT - 1);
                // (a half's words are done with when step 6, or 14, has made the last terms of them)
                if (t == 12) deal(0);
                if (t == 15) deal(1);
                if (t == 14) read_mag(i & 1);
                if (t == 15) {
                    mag_quad();
                    stash_ends((i + 1) & 1);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (__ballot(mag_all > kIqMagMax)) { // a column whose sums may have passed 2^24: the same answer in every wave
                rows_of(i);
                wide_block(i & 1);
                rows_of(next);
            }
#pragma unroll
            for (int c = 0; c < NCT; c++) scale_sums(i & 1, c);
            __syncthreads();
        }
#pragma unroll
        for (int c = 0; c < NCT; c++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int n = 32 * c + 8 * (v >> 2) + 4 * kh + (v & 3);
                if (n < len) {
                    const int row = row0 + 64 * wv + l32;
                    float *out = y + (size_t)L->tab.slot[n] * rpe;
                    if (row < rpe) out[row] = acc[0][c][v];
                    if (row + 32 < rpe) out[row + 32] = acc[1][c][v];
                }
            }
    }
}

__global__ __launch_bounds__(kIqThreads, 1) void k_gemm_iq2_fast(const uint8_t *w, int rpe, int nb, const uint8_t *act, const u32 *cols,
                                                                 const u32 *tiles, const u32 *n_tiles, u32 n_units, u32 slot_div,
                                                                 u32 n_slots, float *y, u32 slabs, const uint8_t *w_second, float *y_second) {
    extern __shared__ __align__(16) uint8_t lds[];
    IqLds *L = reinterpret_cast<IqLds *>(lds);
    const int tid = threadIdx.x;
    const u32 g = tile_of_block(blockIdx.x, n_units);
    const int row0 = (int)(take_stack(slab_of_block(blockIdx.x, n_units), n_units, w, y, w_second, y_second) * slabs) * kIqWgRows;
    const u32 count = n_tiles[0];
    if (g > count) return;
    if (g == count) { // the refused slots' rows: NaN (crates/gpu/src/gemm/grouped.rs:2283-2287)
        const u32 refused = n_tiles[1], rows = slabs * kIqWgRows;
        for (u32 i = tid; i < refused * rows; i += kIqThreads) {
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
        L->tab.slot[tid] = s;
        L->tab.col[tid] = s / slot_div;
    }
    // the grid: magnitudes in the order 0, 2, 1, 3 of each four, as the columns' codes below
    for (int i = tid; i < 256 * 32; i += kIqThreads) {
        const int entry = i >> 5, half = (i >> 4) & 1, copy = i & 15;
        const u32 m = (u32)(BM_IQ2XXS_GRID[entry] >> (32 * half));
        const v2u v = {iq_f16_pair((float)(m & 0xffu), (float)((m >> 16) & 0xffu)), iq_f16_pair((float)((m >> 8) & 0xffu), (float)(m >> 24))};
        *reinterpret_cast<v2u *>(L->grid + 256 * entry + 128 * half + 8 * copy) = v;
    }
    __syncthreads();
    const uint8_t *we = w + (size_t)e * rpe * ((u32)nb * BM_IQ2XXS_BLOCK);
    if (len > 32) iq2_tile<2>(lds, we, act, rpe, nb, row0, (int)slabs, len, y);
    else iq2_tile<1>(lds, we, act, rpe, nb, row0, (int)slabs, len, y);
}

hipError_t gemm_iq2_fast(const Launch &L, const uint8_t *w, int n_experts, int rows_per_expert, int k, const uint8_t *act,
                         const uint32_t *cols, const uint32_t *tiles_dev, const uint32_t *n_tiles, int n_slots, int slot_div, float *y,
                         const uint8_t *w_second, float *y_second) {
    const u32 max_tiles = (u32)gemm_max_tiles(n_slots, n_experts) + 1; // one more: the block that fills refused slots
    const u32 n_slabs = (u32)((rows_per_expert + kIqWgRows - 1) / kIqWgRows), stacks = w_second ? 2 : 1;
    hipError_t e = allow_lds(k_gemm_iq2_fast, sizeof(IqLds));
    if (e != hipSuccess) return e;
    // (a workgroup builds the grid's copies once, a microsecond or two: several slabs each where that leaves eight rounds of 256)
    const u32 slabs_max = stacks * max_tiles * n_slabs / 2048u, slabs = slabs_max < 1u ? 1u : slabs_max < n_slabs ? slabs_max : n_slabs;
    const u32 n_units = stacks * ((n_slabs + slabs - 1) / slabs);
    hipLaunchKernelGGL(k_gemm_iq2_fast, dim3(((max_tiles + 7) / 8) * 8 * n_units), dim3(kIqThreads), sizeof(IqLds), L.stream, w, rows_per_expert,
                       k / 256, act, cols, tiles_dev, n_tiles, n_units, (u32)slot_div, (u32)n_slots, y, slabs, w_second, y_second);
    return hipGetLastError();
}

} // namespace bmk
