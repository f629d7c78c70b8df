// Rows times a packed weight of a superblock type or of a type with blocks of 32: y[M, N] = x[M, K] * W[N, K]^T on
// v_mfma_f32_32x32x16_f16, for f32 rows (ten of them up to a prompt) and bf16 rows.  The
// reference composition is dequantize_tensor -> f32 sgemm (crates/axonml-quant/src/dequantize.rs:34-54,
// crates/axonml-core/src/backends/cpu.rs:566-598).
//
// Time of a call with f32 rows, before (groups of eight vectors, or two-stage operands in LDS) and now, us:
//   rows                  10          16          32          64
//   Q4_K 28672 x 4096     41.4 35.7   42.0 36.2   83.7 44.4   61.7 47 to 54
//   Q4_K 4096 x 4096      21.9 15.7   21.9 17.2   39.9 20.8   33.0 22.7
//   Q4_K 4096 x 14336     as before (see axq_dev_rows_gemm_pays)   63.5 36.8   64.0 37.7
//   Q4_0 4096 x 11008, 21 rows: 41.9 26.8; Q4_0 4096 x 4096, 10 and 39 rows: 21.7 14.4, 54.7 21.2; Q8_0 11008 x 4096, 64 rows: 43.1 34.9;
//   bf16 rows, Q8_0 4096 x 4096, 16: 26.0 14.5; Q4_0 11008 x 4096, 128: 48.4 36.5; Q4_K 14336 x 4096, 2048: 325 to 328 265 to 290
// What bounds it: at few rows the fixed parts (pre-pass, reduction and the launches around them: 14 us of the 4096 x 4096 calls) and
// the LDS reads of x, which every wave makes for its 32 columns (0.35 us per step with one tile of x, 0.6 with two); at many the matrix
// pipe beside the vector instructions that make operands.  2048 bf16 rows x 14336 take 254 to 285 us in the kernel as the clock goes (273 in the
// first passes, 256 behind hundreds of others), 845 to 945 TFLOP/s: a product keeps its SIMD's issue for about half of its 33 cycles, four vector
// instructions fit beside it, and there are five; a tile's way in and out, 5 and 13 us a round (all workgroups write at once); and
// the card's power: the same products alone, without operands, copies and results, take 208 us, 167 if every x is zero.
//
// Numerics.  A bf16 row goes in as f16 under a power-of-two row scale that puts its largest element right below f16's limit: exact
// down to 2^-31 of that element, and what is smaller to within 2^-39 of it.  An f32 row goes in as two f16 rows, leading eleven
// bits and remainder, whose results are added (22 bits, and 2^-39 of the row's largest), from 40 rows on; fewer rows, which the
// small-batch GEMV with its 28 bits below the largest of every 32 is the alternative for, as three limbs.  The first is a multiple of
// 2^-8 of the power of two above its block's largest, so that its sums over a block are exact and have few bits (with eight or nine
// bits below that power in place of seven Q4_0 at K = 4096 has an error of 5.9 and 6.7 instead of 5.0); the second and the third, f16
// themselves and 2^9 times as large as they count, hold the next 22 bits of what is left of each element: 32 bits below the
// block's largest, 22 bits of the element where that is less, down to 2^-48 of the row's largest.  A weight goes in without rounding:
//   Q4_K, Q5_K   w = d (sc (q - C)) + (C d sc - dmin m), C = 8 or 16: sc (q - C) is an integer below 2^10, exact in f16, and is
//                the operand; sums of them are in units of d, or 8 d to be exact.  A step's sum starts from zero and joins the total, or, where
//                registers are short (rows_wide_kernel), the accumulators of a column hold the running sum and change their
//                unit at a superblock boundary (one multiply per register and 256 k).  The offset, one number per sub-block of
//                32, joins in the same unit as an f16 pair, against the sub-block's sum of x as an f16 pair: two products more
//                per superblock.  Where dmin is so large beside d that the pair would leave f16's range, the unit is d times a
//                power of two and the operands are divided by it (exact).
//   Q6_K         w = d sc (q - 32): sc (q - 32) has 13 bits and goes in as two exact operands, sc times the multiple of eight
//                and sc times the rest, two products per weight.
//   blocks of 32 w = d (q - C) + (m + C d): q - C is the operand, a block's sum starts from zero and joins its superblock's times d; the
//                offsets of eight blocks, as an f16 pair under a common power of two, meet the blocks' sums of x.  C is the middle
//                code, or, with a minimum, the code nearest to a weight of zero (see Block32::centre).
// Centred codes because sums over uncentred ones cancel for rows with a mean.  Accumulation is f32 throughout.  rows_gemm_kernel: products of a step (limbs, blocks;
// else of two) from zero, steps into a superblock's sum, superblocks into the total.  rows_apart_kernel: two steps from zero, into the total of one of two halves.
// Large tiles have registers for the total only, which a block's sum (rows_blocks_kernel) or every product (rows_wide_kernel) joins.
// Root mean square error against 64 bits over that of the result, normal x, K = 1024 / 4096 / 14336, in 1e-8, before and now:
//   rows       up to 39                       40 and more, f32                     f32, large tiles (before the same but for Q5_1)
//   Q4_0       7.2 8.6 10.3   5.0 5.0 5.5     8.5 10.6 15.5   7.9 8.3 9.5          11.5 21.0 38.3
//   Q5_1       9.4 10.5 12.9  6.4 6.3 6.8     9.1 11.2 16.4   8.1 8.5 9.6          12.4 22.4 40.7   12.1 22.2 40.7
//   Q4_K       9.4 10.5 12.8  7.4 7.3 7.5     13.0 17.7 31.4  10.8 11.0 11.7       16.4 31.4 58.6
//   Q6_K       8.9 10.0 12.4  5.3 5.2 5.5     15.8 21.6 38.8  12.0 12.1 12.7       20.6 40.8 76.7
// (64 f32 rows times 14336 x 4096 in rows_apart_kernel, Q4_K and Q6_K: 11.9 and 12.9, as in rows_gemm_kernel.)
// (K in parts, whose sums gemm_reduce_kernel adds together with what their additions round off: without that Q4_0, K = 4096 has 8.4 in
// place of the 6.7 of nine bits, and 9.7 in place of 8.3.  Limbs in one accumulator: Q4_0 8.6 11.7 16.5; the matrix pipe cuts sums off where it adds small products to large ones.)
//
// Shape (rows_gemm_kernel).  A workgroup of eight waves; a wave computes 32 MI x 32 outputs.  Four waves lie side by side along N; the other
// factor of two is rows (WM = 2: 64 MI rows) or K (WM = 1: each four waves take half of the workgroup's superblocks, and the
// two sums meet in LDS).  What the design turns on:
//   - weights never pass through LDS as operands.  Their packed codes come into LDS as they are (global_load_lds, two K steps
//     at a time, up to three such units ahead), a lane reads the 16 bytes it multiplies with and makes the B operand in registers:
//     eleven vector instructions per eight Q4 codes ((w & 0x00F000F0) | 0x5400 is the f16 pair 64 + q, one packed multiply-add
//     makes sc (q - 8) of it).  An operand written to LDS and read back costs four times the bytes, and binds conversion to
//     the barrier.
//   - x lies in memory in operand order (rows_prep_kernel): a wave's fragment is one kilobyte, lane after lane, so the copy
//     into LDS is linear and the fragment reads are free of conflicts.
//   - one barrier per K step of 64, in front of the step's last products: the next step's first fragments are requested
//     behind it and arrive while those products run.
#include <hip/hip_fp16.h>

#include <type_traits>

#include "axq_internal.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void gbl_void;

constexpr int LB = 7; // bits of the first limb below its block's largest power of two

struct RowsArgs {
    const uint8_t *codes, *meta, *qh;
    uint32_t codes_pitch, meta_pitch, qh_pitch;
    const _Float16 *xa;    // x in operand order: [tile of 32 rows][step of 64 k][t = 0..3][lane][8]
    const _Float16 *xs;    // its sub-block sums: [tile][superblock][leading halves, remainders][lane][8]: sub-blocks 4 (lane / 32) .., twice
    const float *rowscale; // [m]
    float *y, *ypart;      // ypart: [splits][rows][part_pitch] unscaled sums (NULL: one workgroup covers all of K)
    int m, n, k;           // m rows of xa; with `pair` rows 2t and 2t + 1 are the parts of row t, and y has m / 2 rows
    int sb_per_split, pair;
    const float *bias, *resid;
    int swiglu;            // y [rows][n / 2] takes silu(gate) * up: columns alternate, four gates and their four ups
};

__device__ inline float h2f(uint32_t bits) { return (float)__builtin_bit_cast(_Float16, (unsigned short)bits); }
__device__ inline half2v halfs(uint32_t v) { return __builtin_bit_cast(half2v, v); }
__device__ inline uint32_t bits(half2v v) { return __builtin_bit_cast(uint32_t, v); }
__device__ inline half2v pk2(float v) { return __builtin_bit_cast(half2v, __builtin_amdgcn_cvt_pkrtz(v, v)); } // exact for what is put in
__device__ inline half8 octet(const uint32_t (&o)[4]) { return __builtin_bit_cast(half8, u32x4{o[0], o[1], o[2], o[3]}); }

template <int N>
__device__ inline void wait_loads_and_lds() { // s_waitcnt vmcnt(N) lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(((N >> 4) << 14) | (7 << 4) | (N & 15));
    asm volatile("" ::: "memory");
}
__device__ inline void barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// A lane of an operand of step j (0..3) of a superblock, product t (0..3): elements 64 j + 32 (t / 2) + 16 (lane / 32) + 8 (t % 2)
// + {0, 2, 1, 3, 4, 6, 5, 7}: the order in which masks take code pairs out of a dword.
//
// A block type says
//   PAIRS    32-byte pieces of a row's codes per unit of two steps; piece_src: the first byte of one, in row 0
//   SIDE16, SIDE4   16-byte and 4-byte pieces of a row's superblock besides codes (scales, fifth bits); side_src
//   Side, Raw       what a lane reads of them, and of the codes per step, from LDS
//   make     the operand(s) of product t; PRODUCTS operands per weight; MIN: there is an offset term
template <bool Q5>
struct SuperQ45 {
    static constexpr int PAIRS = 2, PRODUCTS = 1, SIDE16 = Q5 ? 3 : 1, SIDE4 = 0;
    static constexpr bool MIN = true, BLOCKS = false;
    static constexpr float CENTRE = Q5 ? 16.0f : 8.0f;
    struct Side { u32x4 h, b; };
    struct Raw { u32x4 q; };
    // piece p: the 16-byte halves p of two neighbouring pairs of sub-blocks (see q4k_code_offset)
    __device__ static const uint8_t *piece_src(const RowsArgs &a, int unit, int p) {
        const int pair = 2 * unit, slice = pair >> 6, left = (a.k >> 6) - (slice << 6), P = left < 64 ? left : 64;
        return a.codes + (size_t)slice * 2048 + (size_t)(p * 16 * P + (pair & 63) * 16);
    }
    __device__ static uint32_t piece_pitch(const RowsArgs &a, int) { return a.codes_pitch; }
    __device__ static const uint8_t *side_src(const RowsArgs &a, int sb, int c) { // the header, then the two halves of the fifth bits
        return c == 0 ? a.meta + (size_t)sb * 16 : a.qh + (size_t)sb * 32 + (c - 1) * 16;
    }
    __device__ static uint32_t side_pitch(const RowsArgs &a, int c) { return c == 0 ? a.meta_pitch : a.qh_pitch; }
    template <int N>
    __device__ static void read_side(const uint8_t *stage, int row, int hh, int, Side &s) {
        s.h = *reinterpret_cast<const u32x4 *>(stage + row * 16);
        if constexpr (Q5) s.b = *reinterpret_cast<const u32x4 *>(stage + (1 + hh) * N * 16 + row * 16);
    }
    // u, the accumulators' unit for a superblock, inv = 1 / u and shrink = d / u: u = d 2^p, p = 3 unless dmin / d >= 64 (p <= 24:
    // operands stay multiples of f16's smallest number, see `excess`); dmin where d = 0; 0 for a superblock of zeros.  Not d itself:
    // the sums of x come times 1 / 64, and 64 times an offset has to stay within f16
    __device__ static void unit_of(const Side &s, float &u, float &inv, float &shrink) {
        const float d = h2f(s.h[0] & 0xFFFFu), dm = h2f(s.h[0] >> 16);
        auto expo = [](float v) { return (int)((__builtin_bit_cast(uint32_t, v) >> 23) & 0xFF); };
        int p = expo(dm) - expo(d) - 2;
        p = p < 3 ? 3 : (p > 24 ? 24 : p);
        u = d == 0.f ? dm : d * __builtin_bit_cast(float, (uint32_t)(127 + p) << 23);
        shrink = d == 0.f ? 0.f : __builtin_bit_cast(float, (uint32_t)(127 - p) << 23);
        inv = 1.0f / (u == 0.f ? 1.0f : u);
    }
    // How many powers of two dmin / d lies beyond what p takes up: up to 13 more (f16's largest over its smallest number), 0 for
    // anything that comes of values.  The offsets are divided by 2^excess and join accumulators that are divided by it meanwhile.
    __device__ static int excess(const Side &s) {
        const float d = h2f(s.h[0] & 0xFFFFu), dm = h2f(s.h[0] >> 16);
        auto expo = [](float v) { return (int)((__builtin_bit_cast(uint32_t, v) >> 23) & 0xFF); };
        const int r = expo(dm) - expo(d) - 2 - 24;
        return d == 0.f || r < 0 ? 0 : r;
    }
    // four of the offsets of a superblock, sub-blocks 4 hh .. 4 hh + 3, in units of u 2^excess and times 64 (their sums of x come
    // times 1 / 64), |.| <= 8 (16 * 63 + 64 * 63): leading halves, then remainders
    __device__ static half8 offsets(const Side &s, int hh, float inv) { // inv = 1 / (u 2^excess)
        // C d sc - dmin m: both products exact (11 x 6 bits), so that their difference loses nothing where they nearly cancel
        const float dc = CENTRE * h2f(s.h[0] & 0xFFFFu), dm = -h2f(s.h[0] >> 16), to_unit = 64.0f * inv;
        const uint32_t sc = hh ? (s.h[3] & 0x0F0F0F0Fu) | ((s.h[1] >> 2) & 0x30303030u) : s.h[1] & 0x3F3F3F3Fu;
        const uint32_t mn = hh ? ((s.h[3] >> 4) & 0x0F0F0F0Fu) | ((s.h[2] >> 2) & 0x30303030u) : s.h[2] & 0x3F3F3F3Fu;
        uint32_t o[4];
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const float c0 = fmaf((float)((sc >> (16 * p)) & 0xFF), dc, (float)((mn >> (16 * p)) & 0xFF) * dm) * to_unit;
            const float c1 = fmaf((float)((sc >> (16 * p + 8)) & 0xFF), dc, (float)((mn >> (16 * p + 8)) & 0xFF) * dm) * to_unit;
            const half2v h = __builtin_bit_cast(half2v, __builtin_amdgcn_cvt_pkrtz(c0, c1)); // the leading eleven bits
            o[p] = bits(h);
            o[2 + p] = bits(half2v{(_Float16)(c0 - (float)h[0]), (_Float16)(c1 - (float)h[1])});
        }
        return octet(o);
    }
    __device__ static void read_raw(const uint8_t *tile, int col, int hh, int j, Raw &r) {
        r.q = *reinterpret_cast<const u32x4 *>(tile + hh * 1024 + ((col * 2) + ((j & 1) ^ ((col >> 3) & 1))) * 16);
    }
    // per superblock: sub-block scales times shrink, two to a dword (2p low, 2p + 1 high), and -(64 + C) times them; both exact
    // (72 * 63 = 8 * 567, 80 * 63 = 16 * 315)
    struct Scales { half2v sc[4], off[4]; };
    __device__ static void scales(const Side &s, float shrink, int, Scales &o) {
        const uint32_t lo = s.h[1] & 0x3F3F3F3Fu, hi = (s.h[3] & 0x0F0F0F0Fu) | ((s.h[1] >> 2) & 0x30303030u); // sub-blocks 0..3, 4..7
        const half2v k = {(_Float16)-1024.0f, (_Float16)-1024.0f}, f = pk2(shrink);
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const uint32_t pair = __builtin_amdgcn_perm(0x64646464u, p < 2 ? lo : hi, (p & 1) ? 0x04030402u : 0x04010400u); // 1024 + scale
            o.sc[p] = (halfs(pair) + k) * f;
            o.off[p] = o.sc[p] * (_Float16)(-(64.0f + CENTRE));
        }
    }
    __device__ static void make(const Raw &r, const Side &s, const Scales &c, uint32_t mask, int j, int t, int, half8 (&o)[1]) {
        const half2v sc = (t >> 1) ? __builtin_shufflevector(c.sc[j], c.sc[j], 1, 1) : __builtin_shufflevector(c.sc[j], c.sc[j], 0, 0);
        const half2v off = (t >> 1) ? __builtin_shufflevector(c.off[j], c.off[j], 1, 1) : __builtin_shufflevector(c.off[j], c.off[j], 0, 0);
        uint32_t w[4];
#pragma unroll
        for (int d = 0; d < 2; d++) {
            const uint32_t q = r.q[2 * (t & 1) + d];
            // a code at bits 4..7 (4..8) of a half with 0x5400 is the f16 number 64 + q
            uint32_t e = (((t >> 1) ? q : q << 4) & mask) | 0x54005400u, f = (((t >> 1) ? q >> 8 : q >> 4) & mask) | 0x54005400u;
            if constexpr (Q5) {
                const uint32_t b = s.b[2 * (t & 1) + d] >> (2 * j + (t >> 1)); // bit 0 of every byte
                e |= (b & 0x00010001u) << 8;
                f |= b & 0x01000100u;
            }
            w[2 * d] = bits(__builtin_elementwise_fma(halfs(e), sc, off));
            w[2 * d + 1] = bits(__builtin_elementwise_fma(halfs(f), sc, off));
        }
        o[0] = octet(w);
    }
    template <int PR>
    __device__ static void make_part(const Raw &r, const Side &s, const Scales &c, uint32_t mask, int j, int t, half8 &o) {
        half8 all[1];
        make(r, s, c, mask, j, t, 0, all);
        o = all[0];
    }
};

struct SuperQ6 {
    static constexpr int PAIRS = 3, PRODUCTS = 2, SIDE16 = 1, SIDE4 = 1;
    static constexpr bool MIN = false, BLOCKS = false;
    struct Side { u32x4 sc; uint32_t d; };
    struct Raw { u32x4 ql[2], qh; };
    // a unit is half a superblock, 128 elements: pieces 0 and 1 its 64 bytes of low nibbles, piece 2 its 32 bytes of bit pairs
    __device__ static const uint8_t *piece_src(const RowsArgs &a, int unit, int p) {
        return p < 2 ? a.codes + (size_t)unit * 64 + p * 32 : a.qh + (size_t)unit * 32;
    }
    __device__ static uint32_t piece_pitch(const RowsArgs &a, int p) { return p < 2 ? a.codes_pitch : a.qh_pitch; }
    __device__ static const uint8_t *side_src(const RowsArgs &a, int sb, int c) { // the scales; the d of this superblock and its neighbour
        return c == 0 ? a.meta + (size_t)sb * 16 : a.meta + (size_t)(a.k >> 8) * 16 + (size_t)(sb & ~1) * 2;
    }
    __device__ static uint32_t side_pitch(const RowsArgs &a, int) { return a.meta_pitch; }
    template <int N>
    __device__ static void read_side(const uint8_t *stage, int row, int, int sb, Side &s) {
        s.sc = *reinterpret_cast<const u32x4 *>(stage + row * 16);
        s.d = (*reinterpret_cast<const uint32_t *>(stage + N * 16 + row * 4) >> (16 * (sb & 1))) & 0xFFFFu;
    }
    __device__ static void unit_of(const Side &s, float &u, float &inv, float &shrink) {
        u = h2f(s.d);
        inv = 1.0f / (u == 0.f ? 1.0f : u);
        shrink = u == 0.f ? 0.f : 1.0f;
    }
    __device__ static void read_raw(const uint8_t *tile, int col, int hh, int, Raw &r) {
        const uint8_t *at = tile + (col * 2 + (hh ^ ((col >> 3) & 1))) * 16;
        r.ql[0] = *reinterpret_cast<const u32x4 *>(at);
        r.ql[1] = *reinterpret_cast<const u32x4 *>(at + 1024);
        r.qh = *reinterpret_cast<const u32x4 *>(at + 2048);
    }
    // this lane's scales, dword j = step j: sub-blocks 4 j + hh (low half) and 4 j + 2 + hh, as f16
    struct Scales { half2v sc[4]; };
    __device__ static void scales(const Side &s, float shrink, int hh, Scales &o) {
        const half2v f = pk2(shrink);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t b = hh ? s.sc[j] >> 8 : s.sc[j];
            o.sc[j] = half2v{(_Float16)(short)(int8_t)(b & 0xFF), (_Float16)(short)(int8_t)((b >> 16) & 0xFF)} * f;
        }
    }
    // element byte l of the unit: nibble j % 2 of ql[t / 2], bits 2 (2 (j % 2) + t / 2) of qh
    __device__ static void make(const Raw &r, const Side &, const Scales &c, uint32_t, int j, int t, int, half8 (&o)[2]) {
        const half2v f = (t >> 1) ? __builtin_shufflevector(c.sc[j], c.sc[j], 1, 1) : __builtin_shufflevector(c.sc[j], c.sc[j], 0, 0);
        const half2v c1 = {(_Float16)-1056.0f, (_Float16)-1056.0f}, c0 = {(_Float16)-1024.0f, (_Float16)-1024.0f};
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int d = 0; d < 2; d++) {
            const int at = 2 * (t & 1) + d;
            const uint32_t u = ((r.ql[t >> 1][at] >> (4 * (j & 1))) & 0x0F0F0F0Fu) | (((r.qh[at] >> (2 * (2 * (j & 1) + (t >> 1)))) & 0x03030303u) << 4);
            const uint32_t v = u >> 8;
            hi[2 * d] = bits((halfs((u & 0x00380038u) | 0x64006400u) + c1) * f);
            hi[2 * d + 1] = bits((halfs((v & 0x00380038u) | 0x64006400u) + c1) * f);
            lo[2 * d] = bits((halfs((u & 0x00070007u) | 0x64006400u) + c0) * f);
            lo[2 * d + 1] = bits((halfs((v & 0x00070007u) | 0x64006400u) + c0) * f);
        }
        o[0] = octet(hi);
        o[1] = octet(lo);
    }
    template <int PR>
    __device__ static void make_part(const Raw &r, const Side &s, const Scales &c, uint32_t mask, int j, int t, half8 &o) {
        half8 both[2];
        make(r, s, c, mask, j, t, 0, both);
        o = both[PR];
    }
};

// Blocks of 32 with an f16 scale d each (and a minimum m): the operand is the centred code, an integer; a block's sum starts from
// zero and joins the total times d; m + C d meets the block's sum of x, eight blocks at a time.  With a minimum the centre is the
// code that lies nearest to zero: the middle for weights around zero, the lowest one for a block of one value, whose d says nothing
// about its weights (the quantisers write 1) and would come back 8 or 16 times in both sums.
template <int BITS, bool WITH_MIN>
struct Block32 {
    static constexpr int PAIRS = BITS == 8 ? 4 : 2, PRODUCTS = 1, REC = WITH_MIN ? 2 : 1, SIDE16 = REC + (BITS == 5 ? 2 : 0), SIDE4 = 0;
    static constexpr bool MIN = WITH_MIN, BLOCKS = true;
    static constexpr float CENTRE = BITS == 8 ? 128.0f : BITS == 5 ? 16.0f : 8.0f;
    struct Side { u32x4 r[REC], b[BITS == 5 ? 2 : 1]; };
    struct Raw { u32x4 q[2]; }; // of the step's two blocks; Q4: the lane's half, in the first two dwords
    struct Scales {};
    __device__ static float centre(uint32_t record) {
        const float zero = -h2f(record >> 16) * __builtin_amdgcn_rcpf(h2f(record & 0xFFFFu)); // where the weight is zero; not a number: code 0
        return rintf(fminf(fmaxf(zero, 0.f), BITS == 5 ? 31.0f : 15.0f));
    }
    __device__ static const uint8_t *piece_src(const RowsArgs &a, int unit, int p) { return a.codes + (size_t)unit * (PAIRS * 32) + p * 32; }
    __device__ static uint32_t piece_pitch(const RowsArgs &a, int) { return a.codes_pitch; }
    __device__ static const uint8_t *side_src(const RowsArgs &a, int sb, int c) { // the records, then the fifth bits
        return c < REC ? a.meta + (size_t)sb * (16 * REC) + c * 16 : a.qh + (size_t)sb * 32 + (c - REC) * 16;
    }
    __device__ static uint32_t side_pitch(const RowsArgs &a, int c) { return c < REC ? a.meta_pitch : a.qh_pitch; }
    template <int N>
    __device__ static void read_side(const uint8_t *stage, int row, int, int, Side &s) {
#pragma unroll
        for (int c = 0; c < REC; c++) s.r[c] = *reinterpret_cast<const u32x4 *>(stage + c * N * 16 + row * 16);
        if constexpr (BITS == 5)
#pragma unroll
            for (int c = 0; c < 2; c++) s.b[c] = *reinterpret_cast<const u32x4 *>(stage + (REC + c) * N * 16 + row * 16);
    }
    __device__ static uint32_t record(const Side &s, int b) { // d of block b of the superblock, and m above it
        return WITH_MIN ? s.r[b >> 2][b & 3] : (s.r[0][b >> 1] >> (16 * (b & 1))) & 0xFFFFu;
    }
    __device__ static float scale(const Side &s, int b) { return h2f(record(s, b) & 0xFFFFu); }
    // Q4, Q5: piece = the step's parity, its halves the step's blocks; Q8: a piece is a block
    __device__ static void read_raw(const uint8_t *tile, int col, int hh, int j, Raw &r) {
        const int x = (col >> 3) & 1;
#pragma unroll
        for (int b = 0; b < 2; b++) {
            if constexpr (BITS == 8) {
                r.q[b] = *reinterpret_cast<const u32x4 *>(tile + (2 * (j & 1) + b) * 1024 + (col * 2 + (hh ^ x)) * 16);
            } else if constexpr (BITS == 5) {
                r.q[b] = *reinterpret_cast<const u32x4 *>(tile + (j & 1) * 1024 + (col * 2 + (b ^ x)) * 16);
            } else {
                typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                const u32x2 v = *reinterpret_cast<const u32x2 *>(tile + (j & 1) * 1024 + (col * 2 + (b ^ x)) * 16 + hh * 8);
                r.q[b][0] = v[0];
                r.q[b][1] = v[1];
            }
        }
    }
    __device__ static void make(const Raw &r, const Side &s, const Scales &, uint32_t mask, int j, int t, int hh, half8 (&o)[1]) {
        const int b = t >> 1, at = t & 1;
        uint32_t w[4];
        if constexpr (BITS == 8) { // signed bytes as unsigned ones + 128; 0x6400 | u is 1024 + u
            const half2v c = {(_Float16)-1152.0f, (_Float16)-1152.0f};
#pragma unroll
            for (int d = 0; d < 2; d++) {
                const uint32_t v = r.q[b][2 * at + d] ^ 0x80808080u;
                w[2 * d] = bits(halfs((v & 0x00FF00FFu) | 0x64006400u) + c);
                w[2 * d + 1] = bits(halfs(((v >> 8) & 0x00FF00FFu) | 0x64006400u) + c);
            }
        } else { // a code at bits 4..7 (4..8) of a half with 0x5400 is 64 + q
            const half2v c = pk2(-64.0f - (WITH_MIN ? centre(record(s, 2 * j + b)) : CENTRE));
            uint32_t e[4];
            if constexpr (BITS == 4) { // byte i = elements 2 i (low), 2 i + 1: dword 2 hh + at is the operand's eight
                const uint32_t p = __builtin_amdgcn_perm(0u, r.q[b][at], 0x03010200u); // bytes 0, 2, 1, 3
                e[0] = p << 4; e[1] = p; e[2] = p >> 4; e[3] = p >> 8;
            } else { // byte i = elements i (low), i + 16: lanes of the upper half take the high nibbles
#pragma unroll
                for (int d = 0; d < 2; d++) {
                    const uint32_t v = r.q[b][2 * at + d] << (4 - 4 * hh);
                    e[2 * d] = v;
                    e[2 * d + 1] = v >> 8;
                }
            }
#pragma unroll
            for (int i = 0; i < 4; i++) e[i] = (e[i] & mask) | 0x54005400u;
            if constexpr (BITS == 5) {
                // bits b0..b3 times (2^8 + 2^22): b0 lands on bit 8 and b2 on bit 24 (of the pair 0, 2), nothing else does
                const uint32_t f = s.b[j >> 1][2 * (j & 1) + b] >> (16 * hh + 8 * at);
                e[0] |= ((f & 0xFu) * 0x00400100u) & 0x01000100u;
                e[1] |= (((f >> 1) & 0x7u) * 0x00400100u) & 0x01000100u;
                e[2] |= (((f >> 4) & 0xFu) * 0x00400100u) & 0x01000100u;
                e[3] |= (((f >> 5) & 0x7u) * 0x00400100u) & 0x01000100u;
            }
#pragma unroll
            for (int i = 0; i < 4; i++) w[i] = bits(halfs(e[i]) + c);
        }
        o[0] = octet(w);
    }
    // m + C d of blocks 4 hh .. 4 hh + 3 as f16 pairs, leading halves and then remainders, times a power of two that keeps the
    // superblock's largest within f16: |.| <= max(|m|, |d|) < 2^(e + 1), e the largest exponent of its d and m.  `f`: what undoes it, and the
    // 1 / 64 of the sums of x.
    __device__ static half8 offsets(const Side &s, int hh, float &f) {
        uint32_t most = 0x0400u; // f16 bits; smallest normal number
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const uint32_t r = record(s, b), d = r & 0x7FFFu, m = (r >> 16) & 0x7FFFu;
            most = d > most ? d : most;
            most = m > most ? m : most;
        }
        const int e = (int)(most >> 10) - 15;
        const float up = __builtin_bit_cast(float, (uint32_t)(127 + 13 - e) << 23);
        f = __builtin_bit_cast(float, (uint32_t)(127 - 13 + e + 6) << 23);
        uint32_t o[4];
#pragma unroll
        for (int p = 0; p < 2; p++) {
            float c[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t r = hh ? record(s, 4 + 2 * p + i) : record(s, 2 * p + i);
                c[i] = fmaf(centre(r), h2f(r & 0xFFFFu), h2f(r >> 16)) * up;
            }
            const half2v h = __builtin_bit_cast(half2v, __builtin_amdgcn_cvt_pkrtz(c[0], c[1]));
            o[p] = bits(h);
            o[2 + p] = bits(half2v{(_Float16)(c[0] - (float)h[0]), (_Float16)(c[1] - (float)h[1])});
        }
        return octet(o);
    }
};

// Stages in LDS: NA K steps of x, NW units of codes, the sides and the sums of x of two superblocks.  Half of a group's waves
// copy x, the other half codes and sides: a wave's waits are in order of its requests, and x, which comes from L2 shortly before
// it is used, would otherwise wait for codes that were requested from memory for later.
// AT > 1: x as three limbs (see rows_prep_kernel).  2: up to 16 rows, in two tiles [first | second] and [0 | third] whose products meet in
// one accumulator tile; 3: 32 rows in three tiles, the second and the third meet; 4: up to 40 rows, 32 of them in three tiles and the
// limbs of the other eight in a fourth, two tiles to each of the groups along M (37 rows as two times 32, six tiles, and so, us: Q6_K
// 28672 x 4096 104 84, Q4_K 66 55, Q4_K 4096 x 14336 45 41; f16 pairs, with ten bits less, 81, 51 and 37).
template <class T, int MI, int WM, int AT>
struct RowsTile {
    static constexpr int KG = 2 / WM, GW = 4 * WM, CW = GW / 2;     // groups along K, waves of one, waves that copy x (and codes)
    static constexpr int M = AT == 2 ? 16 : AT == 3 ? 32 : AT == 4 ? 40 : 32 * MI * WM, N = 128; // rows, columns
    static constexpr int XT = AT == 2 || AT == 3 ? AT : MI;         // tiles of x of a wave
    static constexpr int acc_of(int l) { return AT == 3 ? (l > 0 ? 1 : 0) : AT == 2 ? 0 : l; } // accumulator tile of a tile of x
    static constexpr bool first_of(int l) { return l == XT - 1 || acc_of(l) != acc_of(l + 1); }
    static constexpr int HB = T::PAIRS * 32;                        // code bytes of a row and unit
    static constexpr int ABYTES = WM * XT * 4096, WBYTES = N * HB, SBYTES = T::MIN ? WM * XT * 2048 : 0; // of a group's stage
    static constexpr int DBYTES = N * (16 * T::SIDE16 + 4 * T::SIDE4);
    static constexpr int NA = 3;
    static constexpr int FIT = (160 * 1024 - KG * (NA * ABYTES + 2 * SBYTES + 2 * DBYTES)) / (KG * WBYTES), NW = FIT > 4 ? 4 : FIT;
    static constexpr int MAIL = KG == 2 ? 8 * MI * 8 * 64 * 4 : 0; // the groups' exchange, which reuses the stages
    static constexpr int STAGES = KG * (NA * ABYTES + NW * WBYTES + 2 * SBYTES + 2 * DBYTES), LDS = STAGES > MAIL ? STAGES : MAIL;
    // a copying wave's requests: x of a step, sums of a superblock; codes of a unit, sides of a superblock (small ones some of them twice)
    static constexpr int XL = 2 * XT, SL = T::MIN ? XT : 0, WT = 4 / CW, WL = WT * T::PAIRS;
    static constexpr int D16 = (2 * T::SIDE16 + CW - 1) / CW, D4 = (2 * T::SIDE4 + CW - 1) / CW;
    static constexpr int FIRST = 7 > 2 * NW - 1 ? 7 : 2 * NW - 1;
    static_assert(AT == 1 || (AT == 4 ? MI == 2 && WM == 2 : MI == AT - 1 && WM == 1), "limbs");
    static_assert(NW >= 2 && WT * CW == 4 && NA <= FIRST, "stages");
    // Behind barrier b: x of step b + NA and, where b % 4 = 1, the sums of superblock (b + 3) / 4; codes of unit (b + 1) / 2 + NW - 1
    // where b is odd and the sides of superblock (b + 7) / 4 where b % 4 = 1.  In front of barrier g everything that is read
    // behind it must have come (x and codes of step g + 1, at a superblock's end sums and sides of the next): how many of the wave's
    // requests may still be under way then.
    static constexpr int allowed_x(int g) {
        int total = 0, need = 0;
        g += 64;
        for (int b = g - 60; b < g; b++) {
            total += XL;
            if (b + NA == g + 1) need = total;
            if (b % 4 == 1) {
                total += SL;
                if (SL && g % 4 == 3 && b == g - 2 && total > need) need = total;
            }
        }
        return total - need > 63 ? 63 : total - need;
    }
    static constexpr int allowed_w(int g) {
        int total = 0, need = 0;
        g += 64;
        for (int b = g - 60; b < g; b++) {
            if (b & 1) {
                total += WL;
                if ((g & 1) && b == g - 2 * (NW - 1)) need = total;
            }
            if (b % 4 == 1) {
                total += D16 + D4;
                if (g % 4 == 3 && b == g - 6 && total > need) need = total;
            }
        }
        return (g & 1) == 0 || total - need > 63 ? 63 : total - need;
    }
};

// A result on its way out: row gm of the operands, column gn; v2: of row gm + 1, where rows are pairs.
__device__ inline void store_result(const RowsArgs &a, int gm, int gn, float v, float v2) {
    if (gm >= a.m || gn >= a.n) return;
    const size_t row = (size_t)(a.pair ? gm >> 1 : gm), rows = (size_t)(a.pair ? a.m >> 1 : a.m);
    if (a.pair) v += v2;
    if (a.ypart) {
        a.ypart[((size_t)blockIdx.y * rows + row) * axq_part_pitch(a.n) + gn] = v;
    } else {
        float out = v * a.rowscale[gm];
        if (a.bias) out += a.bias[gn];
        if (a.resid) out += a.resid[row * a.n + gn];
        a.y[row * a.n + gn] = out;
    }
}

template <class T, int MI, int WM, int AT>
__global__ void __launch_bounds__(512, 2) rows_gemm_kernel(RowsArgs a) {
    using Tile = RowsTile<T, MI, WM, AT>;
    constexpr int KG = Tile::KG, HB = Tile::HB, ABYTES = Tile::ABYTES, WBYTES = Tile::WBYTES, SBYTES = Tile::SBYTES, DBYTES = Tile::DBYTES, NA = Tile::NA, NW = Tile::NW, XT = Tile::XT;
    extern __shared__ uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave / Tile::GW, wi = wave % Tile::GW, wm = WM == 2 ? wi >> 2 : 0, wn = wave & 3;
    const int nt = (a.n + Tile::N - 1) / Tile::N, wgs = (int)gridDim.x;
    int tile = blockIdx.x;
    if (wgs % 8 == 0) tile = (tile & 7) * (wgs >> 3) + (tile >> 3); // workgroups of one XCD share x tiles
    const int mt0 = (tile / nt) * (WM * XT), n0 = (tile % nt) * Tile::N;
    const int nsb_row = a.k >> 8, steps_row = a.k >> 6;
    const int lo = (int)blockIdx.y * a.sb_per_split, hi = lo + a.sb_per_split < nsb_row ? lo + a.sb_per_split : nsb_row;
    // superblocks of this group: `loops` is what every wave of the workgroup walks through, `mine` what this group multiplies
    const int loops = (hi - lo + KG - 1) / KG, sb0 = lo + kg * loops;
    const int mine = hi - sb0 < loops ? (hi - sb0 > 0 ? hi - sb0 : 0) : loops;
    uint8_t *abase = lds + kg * NA * ABYTES, *wbase = lds + KG * NA * ABYTES + kg * NW * WBYTES;
    uint8_t *sbase = lds + KG * (NA * ABYTES + NW * WBYTES) + kg * 2 * SBYTES, *dbase = sbase + (KG - kg) * 2 * SBYTES + kg * 2 * DBYTES;
    const bool x_wave = wi < Tile::CW; // copies x, the others codes and sides
    const int cw = x_wave ? wi : wi - Tile::CW;

    // ---- copies into LDS (past the end of the row: its last step, unit or superblock again, which nobody looks at)
    auto copy = [&](const void *src, uint8_t *dst) { __builtin_amdgcn_global_load_lds((gbl_void *)src, (lds_void *)dst, 16, 0, 0); };
    auto in_order = [] { asm volatile("" ::: "memory"); }; // the waits in front of the barriers count on the order of the requests
    auto copy_x = [&](int g, int at) { // x of step g of the group into the stage at byte `at`
        int step = sb0 * 4 + g;
        step = step < steps_row ? step : steps_row - 1;
#pragma unroll
        for (int q = 0; q < Tile::XL; q++) {
            const int kb = cw * Tile::XL + q, mt = kb >> 2, t = kb & 3;
            copy(a.xa + ((size_t)(mt0 + mt) * steps_row + step) * 2048 + t * 512 + lane * 8, abase + at + kb * 1024);
        }
        in_order();
    };
    auto copy_sums = [&](int sb) {
        const int at = sb0 + sb < nsb_row ? sb0 + sb : nsb_row - 1;
#pragma unroll
        for (int q = 0; q < Tile::SL; q++) {
            const int kb = cw * Tile::SL + q;
            copy(a.xs + ((size_t)(mt0 + (kb >> 1)) * nsb_row + at) * 1024 + (kb & 1) * 512 + lane * 8, sbase + (sb & 1) * SBYTES + kb * 1024);
        }
        in_order();
    };
    // codes: lane -> (row of 32, 16-byte half of its piece): the halves of rows 8..15 and 24..31 change places, so that sixteen
    // lanes that read the same half of consecutive rows touch all banks
    const int cr = lane >> 1, cs = (lane & 1) ^ ((cr >> 3) & 1);
    auto row_of = [&](int r) { return (uint32_t)(n0 + r < a.n ? r : a.n - 1 - n0); }; // row r of the tile; past the end the last one
    auto copy_codes = [&](int u, int at) { // codes of unit u of the group
        int unit = sb0 * 2 + u;
        unit = unit < 2 * nsb_row ? unit : 2 * nsb_row - 1;
#pragma unroll
        for (int q = 0; q < Tile::WT; q++) {
            const int ct = cw * Tile::WT + q; // column tile of 32 rows
            const uint32_t row = row_of(ct * 32 + cr);
#pragma unroll
            for (int p = 0; p < T::PAIRS; p++)
                copy(T::piece_src(a, unit, p) + (size_t)n0 * T::piece_pitch(a, p) + (row * T::piece_pitch(a, p) + cs * 16),
                     wbase + at + ct * 32 * HB + p * 1024);
        }
        in_order();
    };
    auto copy_sides = [&](int sb) { // 64 rows of a piece at a time
        const int at = sb0 + sb < nsb_row ? sb0 + sb : nsb_row - 1;
        uint8_t *dst = dbase + (sb & 1) * DBYTES;
#pragma unroll
        for (int q = 0; q < Tile::D16; q++) {
            const int ii = (cw + q * Tile::CW) % (2 * T::SIDE16), c = ii / 2, r0 = ii % 2 * 64;
            copy(T::side_src(a, at, c) + (size_t)n0 * T::side_pitch(a, c) + row_of(r0 + lane) * T::side_pitch(a, c), dst + c * Tile::N * 16 + r0 * 16);
        }
#pragma unroll
        for (int q = 0; q < Tile::D4; q++) {
            const int r0 = (cw + q * Tile::CW) % 2 * 64;
            __builtin_amdgcn_global_load_lds((gbl_void *)(T::side_src(a, at, T::SIDE16) + (size_t)n0 * T::side_pitch(a, T::SIDE16) +
                                                          row_of(r0 + lane) * T::side_pitch(a, T::SIDE16)),
                                             (lds_void *)(dst + T::SIDE16 * Tile::N * 16 + r0 * 4), 4, 0, 0);
        }
        in_order();
    };

    // ---- products
    float unit, inv;
    typename T::Side side, next_side;
    typename T::Scales scales;
    uint32_t mask; // in a vector register: an instruction takes one scalar operand, and (w & mask) | base has its base there
    asm("v_mov_b32 %0, 0x00f000f0" : "=v"(mask));
    auto read_sides = [&](int sb) { T::template read_side<Tile::N>(dbase + (sb & 1) * DBYTES, wn * 32 + li, hh, sb0 + sb, next_side); };
    const uint8_t *my_x = abase + wm * XT * 4096 + lane * 16, *my_codes = wbase + wn * 32 * HB;
    int a_rd = 0, w_rd = 0; // stage of the step, of the unit that is read next
    auto read_x = [&](int t, half8 (&f)[XT]) {
#pragma unroll
        for (int i = 0; i < XT; i++) f[i] = *reinterpret_cast<const half8 *>(my_x + a_rd + i * 4096 + t * 1024);
    };
    // behind the barrier of step 4 sb + J: the stages of that step have been read by everybody, and what the next one reads is there
    auto meet = [&](int sb, auto step) {
        constexpr int J = decltype(step)::value;
        if (x_wave) {
            wait_loads_and_lds<Tile::allowed_x(J)>();
            barrier();
            copy_x(4 * sb + J + NA, a_rd);
            if (J == 1 && T::MIN) copy_sums(sb + 1);
        } else {
            wait_loads_and_lds<Tile::allowed_w(J)>();
            barrier();
            if (J & 1) copy_codes(2 * sb + (J >> 1) + NW, w_rd);
            if (J == 1) copy_sides(sb + 2);
        }
        a_rd = a_rd == (NA - 1) * ABYTES ? 0 : a_rd + ABYTES;
        if (J & 1) w_rd = w_rd == (NW - 1) * WBYTES ? 0 : w_rd + WBYTES;
    };
    auto add_offsets = [&](int sb, float16v (&to)[MI]) {
        if constexpr (T::MIN && !T::BLOCKS) {
            const int over = T::excess(side);
            const bool any_over = __builtin_amdgcn_ballot_w64(over > 0) != 0; // a column's lanes all have its factor; exact, being a power of two
            auto times_pow2 = [&](int e) {
                const float f = __builtin_bit_cast(float, (uint32_t)(127 + e) << 23);
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int q = 0; q < 16; q++) to[i][q] *= f;
            };
            if (any_over) times_pow2(-over);
            const half8 o = T::offsets(side, hh, inv * __builtin_bit_cast(float, (uint32_t)(127 - over) << 23));
#pragma unroll
            for (int i = 0; i < XT; i++) {
                const uint8_t *x = sbase + (sb & 1) * SBYTES + (wm * XT + i) * 2048 + lane * 16;
                to[Tile::acc_of(i)] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8 *>(x), o, to[Tile::acc_of(i)], 0, 0, 0);
                to[Tile::acc_of(i)] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8 *>(x + 1024), o, to[Tile::acc_of(i)], 0, 0, 0);
            }
            if (any_over) times_pow2(over);
        }
    };
    using S0 = std::integral_constant<int, 0>; using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, 2>; using S3 = std::integral_constant<int, 3>;
#pragma unroll
    for (int b = -Tile::FIRST; b < 0; b++) { // the requests in front of the first step, in the order of the later ones
        if (x_wave) {
            if (b + NA >= 0) copy_x(b + NA, (b + NA) * ABYTES);
            if (b == -3 && T::MIN) copy_sums(0);
        } else {
            if ((b & 1) && (b + 1) / 2 + NW - 1 >= 0) copy_codes((b + 1) / 2 + NW - 1, ((b + 1) / 2 + NW - 1) * WBYTES);
            if (b == -7 || b == -3) copy_sides((b + 7) / 4);
        }
    }
    if (x_wave) wait_loads_and_lds<Tile::allowed_x(3)>();
    else wait_loads_and_lds<Tile::allowed_w(3)>();
    barrier();
    read_sides(0);
    // meet, request the next step's fragments, work on this step's
    constexpr int AHEAD = T::BLOCKS ? 1 : 2; // blocks: the next step's fragments take the place of the products' that are done
    half8 af[AHEAD][4][XT];
    typename T::Raw raw[2];
    // a step's products (a block's, with blocks) start from zero, their sums meet in the superblock's, and that joins the total:
    // few of the additions that round are of the total's size
    const float16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float16v part[MI], sum[MI], total[MI];
#pragma unroll
    for (int i = 0; i < MI; i++) total[i] = sum[i] = zero;
    auto each = [&](auto fn) {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int q = 0; q < 16; q++) fn(i, q);
    };
    auto read_step = [&](int j4, bool first = false) {
        T::read_raw(my_codes + w_rd, li, hh, j4, raw[j4 & 1]);
        if (!T::BLOCKS || first)
#pragma unroll
            for (int t = 0; t < 4; t++) read_x(t, af[j4 % AHEAD][t]);
        asm volatile("" ::: "memory"); // requested here, not where they are used
    };
    auto products = [&](auto at, auto t0, auto t1, auto fresh) { // t0 .. t1 - 1 of a step, from zero where `fresh`
        constexpr int J = decltype(at)::value, T0 = decltype(t0)::value, T1 = decltype(t1)::value;
        half8 bf[T1 - T0][T::PRODUCTS];
        auto mul = [&](int t, int l) {
#pragma unroll
            for (int pr = 0; pr < T::PRODUCTS; pr++)
                part[Tile::acc_of(l)] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                    af[J % AHEAD][t][l], bf[t - T0][pr], decltype(fresh)::value && Tile::first_of(l) && t == T0 && pr == 0 ? zero : part[Tile::acc_of(l)], 0, 0, 0);
        };
        if constexpr (XT == MI) { // every tile of x has an accumulator of its own
#pragma unroll
            for (int t = T0; t < T1; t++) {
                T::make(raw[J & 1], side, scales, mask, J, t, hh, bf[t - T0]);
#pragma unroll
                for (int l = XT - 1; l >= 0; l--) mul(t, l);
            }
        } else {
#pragma unroll
            for (int t = T0; t < T1; t++) T::make(raw[J & 1], side, scales, mask, J, t, hh, bf[t - T0]);
#pragma unroll
            for (int l = XT - 1; l >= 0; l--) // the third limbs first
#pragma unroll
                for (int t = T0; t < T1; t++) mul(t, l);
        }
    };
    using S4 = std::integral_constant<int, 4>;
    auto step = [&](int sb, auto at) {
        constexpr int J = decltype(at)::value;
        // the last step's sums are in `sum` here: left to itself the compiler keeps the blocks' sums of a superblock apart
#pragma unroll
        for (int i = 0; i < MI; i++) {
            if (J == 0) asm volatile("" : "+v"(total[i]));
            else asm volatile("" : "+v"(sum[i]));
        }
        meet(sb, at);
        read_step((J + 1) & 3);
        if (J == 3) read_sides(sb + 1); // looked at behind the next barrier
        if (J == 0) {
            side = next_side;
            if constexpr (!T::BLOCKS) {
                float shrink;
                T::unit_of(side, unit, inv, shrink);
                T::scales(side, shrink, hh, scales);
            }
        }
        if constexpr (T::BLOCKS) {
            auto block = [&](auto half) {
                constexpr int B = decltype(half)::value;
                const float d = T::scale(side, 2 * J + B);
                products(at, std::integral_constant<int, 2 * B>{}, std::integral_constant<int, 2 * B + 2>{}, std::true_type{});
                asm volatile("" ::: "memory");
                read_x(2 * B, af[0][2 * B]);
                read_x(2 * B + 1, af[0][2 * B + 1]);
                asm volatile("" ::: "memory");
                each([&](int i, int q) { sum[i][q] = J == 0 && B == 0 ? part[i][q] * d : fmaf(part[i][q], d, sum[i][q]); });
            };
            block(S0{});
            block(S1{});
            if constexpr (T::MIN && J == 1) { // the superblock's offsets
                float f;
                const half8 o = T::offsets(side, hh, f);
#pragma unroll
                for (int i = XT - 1; i >= 0; i--) {
                    constexpr auto acc_of = Tile::acc_of;
                    const uint8_t *x = sbase + (sb & 1) * SBYTES + (wm * XT + i) * 2048 + lane * 16;
                    part[acc_of(i)] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8 *>(x), o, Tile::first_of(i) ? zero : part[acc_of(i)], 0, 0, 0);
                    part[acc_of(i)] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8 *>(x + 1024), o, part[acc_of(i)], 0, 0, 0);
                }
                each([&](int i, int q) { sum[i][q] = fmaf(part[i][q], f, sum[i][q]); });
            }
            if (J == 3) each([&](int i, int q) { total[i][q] += sum[i][q]; });
        } else {
            // f32 pairs and bf16 rows: two steps to a sum, half the additions (Q4_K 28672 x 4096, 64 f32 rows 56.4 -> 53.9 us)
            constexpr int RUN = AT == 1 ? 2 : 1;
            products(at, S0{}, S4{}, std::integral_constant<bool, J % RUN == 0>{});
            if constexpr (T::MIN && J == 1) add_offsets(sb, part);
            if (J == RUN - 1) each([&](int i, int q) { sum[i][q] = part[i][q]; });
            else if (J % RUN == RUN - 1) each([&](int i, int q) { sum[i][q] += part[i][q]; });
            if (J == 3) each([&](int i, int q) { total[i][q] = fmaf(sum[i][q], unit, total[i][q]); });
        }
    };
    read_step(0, true);
    for (int sb = 0; sb < mine; sb++) {
        step(sb, S0{}); step(sb, S1{}); step(sb, S2{}); step(sb, S3{});
    }
    for (int sb = mine; sb < loops; sb++) { // the other group has one more
        meet(sb, S0{}); meet(sb, S1{}); meet(sb, S2{}); meet(sb, S3{});
    }
    wait_loads_and_lds<0>(); // nothing of this workgroup may still be on its way into LDS

    // ---- results.  D layout: lane -> column li; register r -> row 8 (r / 4) + 4 (lane / 32) + r % 4
    // the first limbs' results and the others', which come times 2^(LB + 2); the others of sixteen rows lie sixteen rows below
    constexpr float BELOW = 1.0f / (1 << (LB + 2));
    if constexpr (AT == 4) { // the third limbs of 32 rows come from the other group; the eight rows' limbs lie eight rows below each other
        barrier();
        float *mail = reinterpret_cast<float *>(lds) + wn * (16 * 64) + lane;
        static_assert(4 * 16 * 64 * 4 <= Tile::LDS, "mail");
        if (wm == 1)
#pragma unroll
            for (int r = 0; r < 16; r++) mail[r * 64] = total[0][r];
        __syncthreads();
        if (wm == 1) {
#pragma unroll
            for (int r = 0; r < 4; r++) total[0][r] = fmaf(total[1][r + 4] + total[1][r + 8], BELOW, total[1][r]);
        } else {
#pragma unroll
            for (int r = 0; r < 16; r++) total[0][r] = fmaf(total[1][r] + mail[r * 64], BELOW, total[0][r]);
        }
    } else if constexpr (AT > 1)
#pragma unroll
        for (int r = 0; r < (AT == 2 ? 8 : 16); r++) total[0][r] = fmaf(AT == 2 ? total[0][r + 8 & 15] : total[MI - 1][r], BELOW, total[0][r]);
    constexpr int MR = AT > 1 ? 1 : MI;
    auto store = [&](int i, int r, float v, float v2) {
        store_result(a, (AT > 1 ? mt0 / AT + wm : mt0 + wm * MI + i) * 32 + 8 * (r >> 2) + 4 * hh + (r & 3), n0 + wn * 32 + li, v, v2);
    };
    const int step_r = a.pair ? 2 : 1;
    if constexpr (KG == 2) { // a group finishes half of the registers and hands the other half over
        barrier();
        float *mail = reinterpret_cast<float *>(lds) + (kg * 4 + wn) * (MR * 8 * 64) + lane;
#pragma unroll
        for (int i = 0; i < MR; i++)
#pragma unroll
            for (int r = 0; r < 8; r++) {
                float lower = total[i][r], upper = total[i][r + 8];
                asm("" : "+v"(lower), "+v"(upper)); // a choice between two registers, not of a register's number
                mail[(i * 8 + r) * 64] = kg ? lower : upper;
            }
        __syncthreads();
        const float *got = reinterpret_cast<const float *>(lds) + ((1 - kg) * 4 + wn) * (MR * 8 * 64) + lane;
#pragma unroll
        for (int i = 0; i < MR; i++) {
            float v[8];
#pragma unroll
            for (int r = 0; r < 8; r++) {
                float lower = total[i][r], upper = total[i][r + 8];
                asm("" : "+v"(lower), "+v"(upper));
                v[r] = (kg ? upper : lower) + got[(i * 8 + r) * 64];
            }
#pragma unroll
            for (int r = 0; r < 8; r++)
                if (r % step_r == 0) store(i, kg * 8 + r, v[r], v[r | 1]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < MR; i++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (r % step_r == 0 && (AT != 4 || r < 4 || wm == 0)) store(i, r, total[i][r], total[i][r | 1]);
    }
}

// Results on their way out, 32 rows at a time through a patch of LDS of the wave's own, from which a lane takes four neighbouring columns
// of a row: straight from the accumulators they are a store of four bytes each, with its own place and options to work out (2048 rows, Q4_K
// 8192 x 512, 256 x 256 outputs, which is mostly that: 50 us; so: 40).  D layout: lane -> column; register r -> row 8 (r / 4) + 4 (lane / 32) + r % 4.
template <int MI, int NJ>
__device__ inline void write_rows(const RowsArgs &a, const float16v (&acc)[MI][NJ], float *patch, int gm0, int n0, int lane) {
    typedef float float4v __attribute__((ext_vector_type(4)));
    typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
    constexpr int PITCH = NJ * 32 + 4, QUADS = NJ * 8, AT_ONCE = 64 / QUADS;
    const int li = lane & 31, hh = lane >> 5, quad = lane % QUADS, col = n0 + quad * 4, rows = a.pair ? a.m >> 1 : a.m;
    const int pitch = a.ypart ? axq_part_pitch(a.n) : a.n;
    float *out = a.ypart ? a.ypart + (size_t)blockIdx.y * rows * pitch : a.y;
    const bool whole = col + 3 < pitch; // four columns of y, whose rows lie where they lie: any n takes 16-byte accesses
    // silu(gate) * up: half the columns (n is a multiple of eight there), and the pre-pass behind them reads half as much.  512 tokens at the 7B shape
    // 19.06 -> 18.39 ms, four steps of 64 sequences 21.66 -> 20.84; the same bits.
    constexpr int GROUPS = QUADS / 2, ROWS_AT_ONCE = 64 / GROUPS;
    float4v bias = {0.f, 0.f, 0.f, 0.f};
    if (a.bias && !a.ypart)
#pragma unroll
        for (int e = 0; e < 4; e++) bias[e] = col + e < a.n ? a.bias[col + e] : 0.f;
#pragma unroll
    for (int i = 0; i < MI; i++) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the last rows have been read
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) patch[(8 * (r >> 2) + 4 * hh + (r & 3)) * PITCH + j * 32 + li] = acc[i][j][r];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (a.swiglu) {
            const int group = lane % GROUPS;
            for (int r = lane / GROUPS; r < (a.pair ? 16 : 32); r += ROWS_AT_ONCE) {
                const int row = (a.pair ? (gm0 + i * 32) >> 1 : gm0 + i * 32) + r;
                if (row >= rows || n0 + group * 8 >= a.n) continue;
                const float *from = patch + (a.pair ? 2 * r : r) * PITCH + group * 8;
                float4v g = *reinterpret_cast<const float4v *>(from), u = *reinterpret_cast<const float4v *>(from + 4);
                if (a.pair) {
                    g += *reinterpret_cast<const float4v *>(from + PITCH);
                    u += *reinterpret_cast<const float4v *>(from + PITCH + 4);
                }
                const float scale = a.rowscale[a.pair ? 2 * row : row];
                float4v v;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float gate = g[e] * scale;
                    v[e] = (gate * (1.0f / (1.0f + expf(-gate)))) * (u[e] * scale); // as rows_prep_kernel
                }
                *reinterpret_cast<float4u *>(a.y + (size_t)row * (a.n >> 1) + ((n0 + group * 8) >> 1)) = v;
            }
            continue;
        }
        for (int r = lane / QUADS; r < (a.pair ? 16 : 32); r += AT_ONCE) {
            const int row = (a.pair ? (gm0 + i * 32) >> 1 : gm0 + i * 32) + r;
            if (row >= rows || col >= a.n) continue;
            const float *from = patch + (a.pair ? 2 * r : r) * PITCH + quad * 4;
            float4v v = *reinterpret_cast<const float4v *>(from);
            if (a.pair) v += *reinterpret_cast<const float4v *>(from + PITCH);
            const size_t at = (size_t)row * pitch + col;
            if (!a.ypart) {
                v = v * a.rowscale[a.pair ? 2 * row : row];
                if (a.bias) v += bias;
                if (a.resid) {
                    if (whole) v += *reinterpret_cast<const float4u *>(a.resid + at);
                    else
                        for (int e = 0; e < 4; e++)
                            if (col + e < a.n) v[e] += a.resid[at + e];
                }
            }
            if (whole) *reinterpret_cast<float4u *>(out + at) = v;
            else
                for (int e = 0; e < 4; e++)
                    if (col + e < a.n) out[at + e] = v[e];
        }
    }
}

// 256 x 256 outputs of a superblock type, 128 x 64 per wave, with the two waves of a SIMD taking turns: while one multiplies, the
// other reads x and codes from LDS, makes its next operands of them and requests what comes into LDS after them.  Waves 0 .. 3 (rows 0 ..
// 127) and 4 .. 7 are half a round apart, with a barrier behind every turn.  A turn is sixteen products (half a K step of 64, twice as many
// for Q6_K), and so are a superblock's offsets against its sums of x, which lie in the ring of x like half a step.
// The first half's waves copy x, the second half's codes and sides, piece by piece between their products, in a loop of its own for each half: a request
// keeps its wave for 40 to 50 cycles, beside which the matrix pipe works on, where requests in the fetch kept the whole workgroup, and a branch between
// products for what only one half copies costs more than the copy.  Cycles of a turn (fetch, products, all; Q4_K, stamped): 993 588 1988 with
// requests in the fetch, 869 for the products with the branches, 657 692 1657 so.  Half of a turn's x is read between the products as well.
// 2048 bf16 rows x 14336 x 4096, whole call, requests in the fetch and so, us: Q4_K 302 to 313 276 to 286, Q5_K 338 308, Q6_K 477 440; 512 f32 rows,
// Q4_K 28672 x 4096 287 265.
template <class T>
struct WideTile {
    static constexpr int HB = T::PAIRS * 32, XBYTES = 16384, WBYTES = 256 * HB, DBYTES = 256 * (16 * T::SIDE16 + 4 * T::SIDE4);
    static constexpr int TURNS = T::MIN ? 9 : 8, OFFSETS = T::MIN ? 4 : -1; // of a superblock; the one of its offsets
    static constexpr int NW = 3, FIT = (160 * 1024 - 2 * DBYTES - NW * WBYTES) / XBYTES, NX = FIT > 6 ? 6 : FIT;
    static constexpr int LDS = NX * XBYTES + NW * WBYTES + 2 * DBYTES;
    // a copying wave's requests: half a step of x; codes of a unit, sides of a superblock
    static constexpr int XL = 4, WL = 2 * T::PAIRS, D16 = T::SIDE16, D4 = T::SIDE4, D = D16 + D4;
    static_assert(NX >= 4 && NW == 3 && XL <= 4 && WL <= 8 && D <= 8, "stages, and eight places between products");
};

template <class T>
__global__ void __launch_bounds__(512, 2) rows_wide_kernel(RowsArgs a) {
    using Tile = WideTile<T>;
    constexpr int MI = 4, NJ = 2, NX = Tile::NX, NW = Tile::NW, XBYTES = Tile::XBYTES, WBYTES = Tile::WBYTES, DBYTES = Tile::DBYTES, HB = Tile::HB, TURNS = Tile::TURNS;
    extern __shared__ uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = wave >> 2, wn = wave & 3;
    const int nt = (a.n + 255) / 256, total = (int)gridDim.x;
    int tile = blockIdx.x;
    if (total % 8 == 0) tile = (tile & 7) * (total >> 3) + (tile >> 3); // workgroups of one XCD share x tiles
    const int mt0 = (tile / nt) * 8, n0 = (tile % nt) * 256;
    const int nsb_row = a.k >> 8;
    const int sb0 = (int)blockIdx.y * a.sb_per_split, mine = sb0 + a.sb_per_split < nsb_row ? a.sb_per_split : nsb_row - sb0;
    uint8_t *xbase = lds, *wbase = lds + NX * XBYTES, *dbase = wbase + NW * WBYTES;

    // ---- copies into LDS (past the end of the row: its last superblock or unit again, which nobody looks at)
    auto copy = [&](const void *base, uint32_t off, uint8_t *dst) { // a wave's place in scalar registers, a lane's in 32 bits: registers are short
        asm volatile("" : "+v"(off)); // extended where it is used
        __builtin_amdgcn_global_load_lds((gbl_void *)(reinterpret_cast<const uint8_t *>(base) + off), (lds_void *)dst, 16, 0, 0);
    };
    const uint32_t lane16 = lane * 16;
    auto in_order = [] { asm volatile("" ::: "memory"); }; // the waits in front of the barriers count on the order of the requests
    auto copy_x = [&](int sb, int h, int at, int piece) { // of turn h of superblock sb of this workgroup into the place at byte `at`
        const int g = sb0 + sb < nsb_row ? sb0 + sb : nsb_row - 1, hs = T::MIN && h > Tile::OFFSETS ? h - 1 : h, q = piece >> 1, t = piece & 1;
        const size_t mt = (size_t)(mt0 + wn * 2 + q);
        copy(h == Tile::OFFSETS ? a.xs + ((mt * nsb_row + g) * 1024 + t * 512) : a.xa + ((mt * nsb_row + g) * 8192 + hs * 1024 + t * 512), lane16,
             xbase + at + (wn * 2 + q) * 2048 + t * 1024);
        in_order();
    };
    const int cr = lane >> 1, cs = (lane & 1) ^ ((cr >> 3) & 1); // see rows_gemm_kernel
    auto row_of = [&](int r) { return (uint32_t)(n0 + r < a.n ? r : a.n - 1 - n0); };
    auto copy_codes = [&](int u, int at, int piece) {
        int unit = sb0 * 2 + u;
        unit = unit < 2 * nsb_row ? unit : 2 * nsb_row - 1;
        const int ct = wn * 2 + piece / T::PAIRS, p = piece % T::PAIRS; // column tile of 32 rows
        const uint32_t row = row_of(ct * 32 + cr);
        copy(T::piece_src(a, unit, p) + (size_t)n0 * T::piece_pitch(a, p), row * T::piece_pitch(a, p) + cs * 16, wbase + at + ct * 32 * HB + p * 1024);
        in_order();
    };
    auto copy_sides = [&](int sb, int c) { // 64 rows of piece c
        const int at = sb0 + sb < nsb_row ? sb0 + sb : nsb_row - 1, r0 = wn * 64;
        uint8_t *dst = dbase + (sb & 1) * DBYTES;
        const uint8_t *src = T::side_src(a, at, c) + (size_t)n0 * T::side_pitch(a, c);
        uint32_t off = row_of(r0 + lane) * T::side_pitch(a, c);
        asm volatile("" : "+v"(off));
        if (c < T::SIDE16) copy(src, off, dst + c * 256 * 16 + r0 * 16);
        else __builtin_amdgcn_global_load_lds((gbl_void *)(src + off), (lds_void *)(dst + T::SIDE16 * 256 * 16 + r0 * 4), 4, 0, 0);
        in_order();
    };
    auto all = [](int n, auto fn) {
#pragma unroll
        for (int p = 0; p < n; p++) fn(p);
    };
    auto turn_over = [] {
        __builtin_amdgcn_sched_barrier(0);
        barrier();
        __builtin_amdgcn_sched_barrier(0);
    };

    float16v acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
    float unit[NJ] = {1.0f, 1.0f}, ratio[NJ], inv[NJ];
    typename T::Side side[NJ];
    typename T::Scales scales[NJ];
    uint32_t mask; // in a vector register: an instruction takes one scalar operand, and (w & mask) | base has its base there
    asm("v_mov_b32 %0, 0x00f000f0" : "=v"(mask));
    auto read_sides = [&](int sb, typename T::Side (&s)[NJ]) {
#pragma unroll
        for (int j = 0; j < NJ; j++) T::template read_side<256>(dbase + (sb & 1) * DBYTES, (wn * NJ + j) * 32 + li, hh, sb0 + sb, s[j]);
    };
    auto new_side = [&] { // what the superblock in `side` asks for; the accumulators change their unit with its first products
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            float u, shrink;
            T::unit_of(side[j], u, inv[j], shrink);
            T::scales(side[j], shrink, hh, scales[j]);
            ratio[j] = u == 0.f ? 1.0f : unit[j] / u;
            unit[j] = u == 0.f ? unit[j] : u;
        }
    };
    const uint8_t *my_x = xbase + half * (MI * 2048) + lane * 16, *my_codes = wbase + wn * NJ * 32 * HB;
    int x_at = 0, w_at = 0; // of the turn's x, of the unit of codes that is read next
    typename T::Raw raw[NJ];
    auto read_codes = [&](int j4) {
#pragma unroll
        for (int j = 0; j < NJ; j++) T::read_raw(my_codes + w_at + j * 32 * HB, li, hh, j4, raw[j]);
        if (j4 & 1) w_at = w_at == (NW - 1) * WBYTES ? 0 : w_at + WBYTES; // its last step
    };

    // ---- the requests in front of the first turn, in the order of the later ones
    if (half == 0) {
#pragma unroll
        for (int g = 0; g < NX - 1; g++) all(Tile::XL, [&](int p) { copy_x(0, g, g * XBYTES, p); });
        wait_loads_and_lds<(NX - 2) * Tile::XL>();
    } else {
        all(Tile::D, [&](int p) { copy_sides(0, p); });
        all(Tile::WL, [&](int p) { copy_codes(0, 0, p); });
        all(Tile::D, [&](int p) { copy_sides(1, p); });
        all(Tile::WL, [&](int p) { copy_codes(1, WBYTES, p); });
        all(Tile::WL, [&](int p) { copy_codes(2, 2 * WBYTES, p); });
        wait_loads_and_lds<Tile::D + 2 * Tile::WL>();
    }
    static_assert(NX - 1 <= TURNS, "turns");
    barrier();
    if (half) turn_over(); // the second half is a turn behind
    read_codes(0);
    read_sides(0, side);
    int w_to = 0; // where the next unit of codes goes: the place of the one that has been read
    auto turn = [&](int sb, auto which, auto copier) __attribute__((always_inline)) {
        constexpr int HALF = decltype(copier)::value;
        constexpr int h = decltype(which)::value, hs = T::MIN && h > Tile::OFFSETS ? h - 1 : h, J = hs >> 1, P = hs & 1;
        constexpr bool OFFS = h == Tile::OFFSETS;
        // Operands are made in the fetch, while x is on its way.  LATE: of its products t = 1 between the ones before, in the place of what those are done
        // with: two operands per weight leave no registers for the others (Q6_K, 2048 x 14336 x 4096: 453 us with thirteen of them spilt, 442 so; with
        // one operand per weight it is the longer way: Q4_K 292 and 303).
        constexpr bool LATE = T::PRODUCTS == 2;
        half8 xf[MI], wf[LATE ? 1 : 2][NJ][T::PRODUCTS];
        auto operand = [&](int t, int j, int pr) -> half8 & { return wf[LATE ? 0 : t][j][pr]; };
        auto make = [&](auto tt, int j, auto part) {
            constexpr int t = decltype(tt)::value, pr = decltype(part)::value;
            T::template make_part<pr>(raw[j], side[j], scales[j], mask, J, 2 * P + t, operand(t, j, pr));
            asm volatile("" : "+v"(operand(t, j, pr)));
        };
        using C0 = std::integral_constant<int, 0>; using C1 = std::integral_constant<int, 1>;
        auto read_x = [&](int t, int i) { xf[i] = *reinterpret_cast<const half8 *>(my_x + x_at + i * 2048 + t * 1024); };
        int over[NJ] = {0, 0};
        // ---- fetch
#pragma unroll
        for (int i = 0; i < MI; i++) read_x(0, i);
        in_order();
        if constexpr (h == 0) new_side();
        if constexpr (OFFS) {
            if constexpr (T::MIN)
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                over[j] = T::excess(side[j]);
                wf[0][j][0] = T::offsets(side[j], hh, inv[j] * __builtin_bit_cast(float, (uint32_t)(127 - over[j]) << 23));
                asm volatile("" : "+v"(wf[0][j][0]));
            }
        } else {
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                make(C0{}, j, C0{});
                if constexpr (LATE) make(C0{}, j, C1{});
                else make(C1{}, j, C0{});
            }
        }
        if constexpr (!LATE && !OFFS && P == 1) read_codes((J + 1) & 3);
        if constexpr (h == TURNS - 1) read_sides(sb + 1, side);
        // what the next turns read first, sides included; here, since the first half reads it in the next phase
        if (HALF && (h == 2 || h == TURNS - 2)) wait_loads_and_lds<Tile::D + Tile::WL>();
        else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        turn_over();
        // ---- multiply
        __builtin_amdgcn_s_setprio(1);
        auto times_pow2 = [&](int j, int e) { // a column's lanes all have its factor; exact, being a power of two
            if (__builtin_amdgcn_ballot_w64(over[j] > 0) == 0) return;
            const float f = __builtin_bit_cast(float, (uint32_t)(127 + e * over[j]) << 23);
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int q = 0; q < 16; q++) acc[i][j][q] *= f;
        };
        if constexpr (OFFS)
            for (int j = 0; j < NJ; j++) times_pow2(j, -1);
        // what this wave copies in this turn
        auto between = [&](int slot) {
            constexpr int ahead = h + NX - 1;
            __builtin_amdgcn_sched_barrier(0);
            if (HALF == 0) {
                if (slot % 2 == 0) copy_x(ahead >= TURNS ? sb + 1 : sb, ahead >= TURNS ? ahead - TURNS : ahead, x_at == 0 ? (NX - 1) * XBYTES : x_at - XBYTES, slot / 2);
            } else {
                if (h == 0 && slot < Tile::D) copy_sides(sb + 2, slot);
                if ((h == 2 || h == TURNS - 2) && slot < Tile::WL) copy_codes(2 * sb + (h == 2 ? 0 : 1) + NW, w_to, slot);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int pr = 0; pr < T::PRODUCTS; pr++)
#pragma unroll
                for (int i = 0; i < MI; i++) {
                    if constexpr (h == 0)
                        if (t == 0 && pr == 0)
#pragma unroll
                            for (int j = 0; j < NJ; j++)
#pragma unroll
                                for (int q = 0; q < 16; q++) acc[i][j][q] *= ratio[j];
                    if constexpr (LATE) {
                        if (t == 0 && pr == 1 && i % 2 == 0) make(C1{}, i / 2, C0{});
                        if (t == 1 && pr == 0 && i % 2 == 0) make(C1{}, i / 2, C1{});
                    }
#pragma unroll
                    for (int j = 0; j < NJ; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[i], operand(OFFS ? 0 : t, j, pr), acc[i][j], 0, 0, 0);
                    if constexpr (h == 0)
                        if (t == 0 && pr == 0) // a tile changes its unit right in front of its first product
#pragma unroll
                            for (int j = 0; j < NJ; j++) {
                                __builtin_amdgcn_sched_group_barrier(2, 16, 0);
                                __builtin_amdgcn_sched_group_barrier(8, 1, 0);
                            }
                    if (pr == 0) between(t * MI + i);
                    if (t == 0 && pr == T::PRODUCTS - 1) read_x(1, i); // in the place of what the products are done with: sixteen registers fewer, and the fetch reads half as much
                }
        if constexpr (LATE && P == 1) read_codes((J + 1) & 3);
        if constexpr (OFFS)
            for (int j = 0; j < NJ; j++) times_pow2(j, 1);
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        if (HALF == 0) wait_loads_and_lds<(NX - 2) * Tile::XL>(); // the next turn's x
        else if (h == 2 || h == TURNS - 2) w_to = w_to == (NW - 1) * WBYTES ? 0 : w_to + WBYTES;
        turn_over();
        x_at = x_at == (NX - 1) * XBYTES ? 0 : x_at + XBYTES;
    };
    // a loop for each half: what a half copies is no branch between the products, which would cost more than the copy
    auto run = [&](auto copier) __attribute__((always_inline)) {
        for (int sb = 0; sb < mine; sb++) {
            turn(sb, std::integral_constant<int, 0>{}, copier); turn(sb, std::integral_constant<int, 1>{}, copier); turn(sb, std::integral_constant<int, 2>{}, copier);
            turn(sb, std::integral_constant<int, 3>{}, copier); turn(sb, std::integral_constant<int, 4>{}, copier); turn(sb, std::integral_constant<int, 5>{}, copier);
            turn(sb, std::integral_constant<int, 6>{}, copier); turn(sb, std::integral_constant<int, 7>{}, copier);
            if constexpr (TURNS == 9) turn(sb, std::integral_constant<int, 8>{}, copier);
        }
    };
    if (half == 0) run(std::integral_constant<int, 0>{});
    else run(std::integral_constant<int, 1>{});
    if (!half) barrier();
    wait_loads_and_lds<0>(); // nothing of this workgroup may still be on its way into LDS

    barrier();
    constexpr int PATCH = 32 * (NJ * 32 + 4);
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int q = 0; q < 16; q++) acc[i][j][q] *= unit[j];
    write_rows<MI, NJ>(a, acc, reinterpret_cast<float *>(lds) + wave * PATCH, (mt0 + half * MI) * 32, n0 + wn * 64, lane);
}

// 256 x 128 outputs of a type with blocks of 32, 128 x 32 per wave, with the waves taking turns as above: a turn is a block's eight products,
// which start from zero and join the total times the block's d in the next fetch, beside the other half's products.  What bounds it is
// that work, 64 multiply-adds per eight products, and the making of operands.  Copies go between the products (see rows_wide_kernel; in the fetch 2048 bf16
// rows x 14336 x 4096 take, and so, us: Q4_0 402 331, Q5_0 425 365, Q8_0 402 354, Q5_1 464 414).
template <class T>
struct BlocksTile {
    static constexpr int HB = T::PAIRS * 32, XBYTES = 16384, WBYTES = 128 * HB, DBYTES = 128 * 16 * T::SIDE16;
    static constexpr int TURNS = T::MIN ? 9 : 8, OFFSETS = T::MIN ? 4 : -1; // of a superblock; the one of its offsets
    static constexpr int NW = 3, FIT = (160 * 1024 - 2 * DBYTES - NW * WBYTES) / XBYTES, NX = FIT > 6 ? 6 : FIT;
    static constexpr int LDS = NX * XBYTES + NW * WBYTES + 2 * DBYTES;
    // a copying wave's requests: half a step of x; codes of a unit, sides of a superblock
    static constexpr int XL = 4, WL = T::PAIRS, D = T::SIDE16;
    static_assert(NX >= 4 && NW == 3 && XL <= 4 && WL <= 8 && D <= 8, "stages, and eight places between products");
};

template <class T>
__global__ void __launch_bounds__(512, 2) rows_blocks_kernel(RowsArgs a) {
    using Tile = BlocksTile<T>;
    constexpr int MI = 4, NX = Tile::NX, NW = Tile::NW, XBYTES = Tile::XBYTES, WBYTES = Tile::WBYTES, DBYTES = Tile::DBYTES, HB = Tile::HB, TURNS = Tile::TURNS;
    extern __shared__ uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = wave >> 2, wn = wave & 3;
    const int nt = (a.n + 127) / 128, total = (int)gridDim.x;
    int tile = blockIdx.x;
    if (total % 8 == 0) tile = (tile & 7) * (total >> 3) + (tile >> 3); // workgroups of one XCD share x tiles
    const int mt0 = (tile / nt) * 8, n0 = (tile % nt) * 128;
    const int nsb_row = a.k >> 8;
    const int sb0 = (int)blockIdx.y * a.sb_per_split, mine = sb0 + a.sb_per_split < nsb_row ? a.sb_per_split : nsb_row - sb0;
    uint8_t *xbase = lds, *wbase = lds + NX * XBYTES, *dbase = wbase + NW * WBYTES;

    // ---- copies into LDS (past the end of the row: its last superblock or unit again, which nobody looks at)
    auto copy = [&](const void *base, uint32_t off, uint8_t *dst) { // a wave's place in scalar registers, a lane's in 32 bits: registers are short
        asm volatile("" : "+v"(off)); // extended where it is used
        __builtin_amdgcn_global_load_lds((gbl_void *)(reinterpret_cast<const uint8_t *>(base) + off), (lds_void *)dst, 16, 0, 0);
    };
    const uint32_t lane16 = lane * 16;
    auto in_order = [] { asm volatile("" ::: "memory"); }; // the waits in front of the barriers count on the order of the requests
    auto copy_x = [&](int sb, int h, int at, int piece) { // of turn h of superblock sb of this workgroup into the place at byte `at`
        const int g = sb0 + sb < nsb_row ? sb0 + sb : nsb_row - 1, hs = T::MIN && h > Tile::OFFSETS ? h - 1 : h, q = piece >> 1, t = piece & 1;
        const size_t mt = (size_t)(mt0 + wn * 2 + q);
        copy(h == Tile::OFFSETS ? a.xs + ((mt * nsb_row + g) * 1024 + t * 512) : a.xa + ((mt * nsb_row + g) * 8192 + hs * 1024 + t * 512), lane16,
             xbase + at + (wn * 2 + q) * 2048 + t * 1024);
        in_order();
    };
    const int cr = lane >> 1, cs = (lane & 1) ^ ((cr >> 3) & 1); // see rows_gemm_kernel
    auto row_of = [&](int r) { return (uint32_t)(n0 + r < a.n ? r : a.n - 1 - n0); };
    auto copy_codes = [&](int u, int at, int p) {
        int unit = sb0 * 2 + u;
        unit = unit < 2 * nsb_row ? unit : 2 * nsb_row - 1;
        const uint32_t row = row_of(wn * 32 + cr);
        copy(T::piece_src(a, unit, p) + (size_t)n0 * T::piece_pitch(a, p), row * T::piece_pitch(a, p) + cs * 16, wbase + at + wn * 32 * HB + p * 1024);
        in_order();
    };
    auto copy_sides = [&](int sb, int c) { // 64 rows of piece c, twice
        const int at = sb0 + sb < nsb_row ? sb0 + sb : nsb_row - 1, r0 = (wn & 1) * 64;
        copy(T::side_src(a, at, c) + (size_t)n0 * T::side_pitch(a, c), row_of(r0 + lane) * T::side_pitch(a, c), dbase + (sb & 1) * DBYTES + c * 128 * 16 + r0 * 16);
        in_order();
    };
    auto all = [](int n, auto fn) {
#pragma unroll
        for (int p = 0; p < n; p++) fn(p);
    };
    auto turn_over = [] {
        __builtin_amdgcn_sched_barrier(0);
        barrier();
        __builtin_amdgcn_sched_barrier(0);
    };

    float16v part[MI], sums[MI][1];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) sums[i][0][r] = part[i][r] = 0.f;
    float d = 0.f; // what the products of the last turn count
    typename T::Side side;
    uint32_t mask; // in a vector register: an instruction takes one scalar operand, and (w & mask) | base has its base there
    asm("v_mov_b32 %0, 0x00f000f0" : "=v"(mask));
    auto fold = [&] {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int q = 0; q < 16; q++) sums[i][0][q] = fmaf(part[i][q], d, sums[i][0][q]);
#pragma unroll
        for (int i = 0; i < MI; i++) asm volatile("" : "+v"(sums[i][0])); // here, while x is on its way, not behind the wait
    };
    auto read_sides = [&](int sb) { T::template read_side<128>(dbase + (sb & 1) * DBYTES, wn * 32 + li, hh, sb0 + sb, side); };
    const uint8_t *my_x = xbase + half * (MI * 2048) + lane * 16, *my_codes = wbase + wn * 32 * HB;
    int x_at = 0, w_at = 0; // of the turn's x, of the unit of codes that is read next
    typename T::Raw raw;
    auto read_codes = [&](int j4) {
        T::read_raw(my_codes + w_at, li, hh, j4, raw);
        if (j4 & 1) w_at = w_at == (NW - 1) * WBYTES ? 0 : w_at + WBYTES; // its last step
    };

    // ---- the requests in front of the first turn, in the order of the later ones
    if (half == 0) {
#pragma unroll
        for (int g = 0; g < NX - 1; g++) all(Tile::XL, [&](int p) { copy_x(0, g, g * XBYTES, p); });
        wait_loads_and_lds<(NX - 2) * Tile::XL>();
    } else {
        all(Tile::D, [&](int p) { copy_sides(0, p); });
        all(Tile::WL, [&](int p) { copy_codes(0, 0, p); });
        all(Tile::D, [&](int p) { copy_sides(1, p); });
        all(Tile::WL, [&](int p) { copy_codes(1, WBYTES, p); });
        all(Tile::WL, [&](int p) { copy_codes(2, 2 * WBYTES, p); });
        wait_loads_and_lds<Tile::D + 2 * Tile::WL>();
    }
    static_assert(NX - 1 <= TURNS, "turns");
    barrier();
    if (half) turn_over(); // the second half is a turn behind
    int w_to = 0; // where the next unit of codes goes: the place of the one that has been read
    auto turn = [&](int sb, auto which, auto copier) __attribute__((always_inline)) {
        constexpr int HALF = decltype(copier)::value;
        constexpr int h = decltype(which)::value, hs = T::MIN && h > Tile::OFFSETS ? h - 1 : h, J = hs >> 1, P = hs & 1;
        constexpr bool OFFS = h == Tile::OFFSETS;
        half8 xf[2][MI];
        // ---- fetch
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int i = 0; i < MI; i++) xf[t][i] = *reinterpret_cast<const half8 *>(my_x + x_at + i * 2048 + t * 1024);
        if (h == 0) read_sides(sb);
        if (!OFFS && P == 0) read_codes(J);
        in_order();
        if (h != 0 || sb > 0) fold();
        if (HALF && (h == 3 || h == TURNS - 1)) wait_loads_and_lds<Tile::D + Tile::WL>(); // what the next turns read first, sides included
        else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        turn_over();
        // ---- multiply
        __builtin_amdgcn_s_setprio(1);
        const float16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        half8 wf[1];
        if constexpr (OFFS) {
            if constexpr (T::MIN) wf[0] = T::offsets(side, hh, d);
        } else {
            d = T::scale(side, hs);
        }
        auto between = [&](int slot) { // copies, piece by piece between the products (see rows_wide_kernel)
            constexpr int ahead = h + NX - 1;
            __builtin_amdgcn_sched_barrier(0);
            if (HALF == 0) {
                if (slot % 2 == 0) copy_x(ahead >= TURNS ? sb + 1 : sb, ahead >= TURNS ? ahead - TURNS : ahead, x_at == 0 ? (NX - 1) * XBYTES : x_at - XBYTES, slot / 2);
            } else {
                if (h == 1 && slot < Tile::D) copy_sides(sb + 2, slot);
                if ((h == 3 || h == TURNS - 1) && slot < Tile::WL) copy_codes(2 * sb + (h == 3 ? 0 : 1) + NW, w_to, slot);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int t = 0; t < 2; t++) {
            if constexpr (!OFFS) T::make(raw, side, typename T::Scales(), mask, J, 2 * P + t, hh, wf);
#pragma unroll
            for (int i = 0; i < MI; i++) {
                part[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[t][i], wf[0], t == 0 ? zero : part[i], 0, 0, 0);
                between(t * MI + i);
            }
        }
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        if (HALF == 0) wait_loads_and_lds<(NX - 2) * Tile::XL>(); // the next turn's x
        else if (h == 3 || h == TURNS - 1) w_to = w_to == (NW - 1) * WBYTES ? 0 : w_to + WBYTES;
        turn_over();
        x_at = x_at == (NX - 1) * XBYTES ? 0 : x_at + XBYTES;
    };
    // a loop for each half: what a half copies is no branch between the products, which would cost more than the copy
    auto run = [&](auto copier) __attribute__((always_inline)) {
        for (int sb = 0; sb < mine; sb++) {
            turn(sb, std::integral_constant<int, 0>{}, copier); turn(sb, std::integral_constant<int, 1>{}, copier); turn(sb, std::integral_constant<int, 2>{}, copier);
            turn(sb, std::integral_constant<int, 3>{}, copier); turn(sb, std::integral_constant<int, 4>{}, copier); turn(sb, std::integral_constant<int, 5>{}, copier);
            turn(sb, std::integral_constant<int, 6>{}, copier); turn(sb, std::integral_constant<int, 7>{}, copier);
            if constexpr (TURNS == 9) turn(sb, std::integral_constant<int, 8>{}, copier);
        }
    };
    if (half == 0) run(std::integral_constant<int, 0>{});
    else run(std::integral_constant<int, 1>{});
    fold();
    if (!half) barrier();
    wait_loads_and_lds<0>(); // nothing of this workgroup may still be on its way into LDS

    barrier();
    write_rows<MI, 1>(a, sums, reinterpret_cast<float *>(lds) + wave * (32 * 36), (mt0 + half * MI) * 32, n0 + wn * 32, lane);
}

// 128 x 128 outputs of a superblock type with the waves taking turns as above; the halves of the workgroup have every other half of its
// superblocks, each with stages of its own, and their sums meet in LDS.  A wave computes 128 x 32, so that an operand is made for four
// products (64 x 32 per wave and halves that share K make it for two, and that work is what the kernel waited for: 64 f32 rows, Q4_K
// 28672 x 4096, 55.8 us).  A turn is a K step of 64, sixteen products.  Copies go between the products (see rows_wide_kernel), and so do the reads of x and
// the making of operands for a turn's second half, so that fetch and products take as long: cycles of a turn, stamped, 1290 881 2616 with all of them in
// the fetch but the operands, 844 855 2105 so; that call 53 to 59 us, 47 to 53 so.  Sums of two steps start from
// zero and join the total times the superblock's unit: as many additions of the total's size as superblocks, since each half has half of them.
template <class T>
struct ApartTile {
    static constexpr int HB = T::PAIRS * 32, XBYTES = 16384, WBYTES = 128 * HB, SBYTES = T::MIN ? 8192 : 0, DBYTES = 128 * (16 * T::SIDE16 + 4 * T::SIDE4);
    static constexpr int NX = 3, NW = 2, GROUP = NX * XBYTES + NW * WBYTES + SBYTES + DBYTES, LDS = 2 * GROUP;
    // a copying wave's requests: x of a step; codes of a unit, sums and sides of a superblock
    static constexpr int XL = 8, WL = 2 * T::PAIRS, SL = T::MIN ? 4 : 0, D = T::SIDE16 + T::SIDE4;
    static_assert(LDS <= 160 * 1024 && LDS >= 8 * 32 * 64 * 4 && XL <= 8 && WL <= 16 && SL <= 16 && D <= 16, "stages, and sixteen places between products");
};

template <class T>
__global__ void __launch_bounds__(512, 2) rows_apart_kernel(RowsArgs a) {
    using Tile = ApartTile<T>;
    constexpr int MI = 4, XBYTES = Tile::XBYTES, WBYTES = Tile::WBYTES, HB = Tile::HB, NX = Tile::NX;
    extern __shared__ uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = wave >> 2, wn = wave & 3;
    const int nt = (a.n + 127) / 128, total_tiles = (int)gridDim.x;
    int tile = blockIdx.x;
    if (total_tiles % 8 == 0) tile = (tile & 7) * (total_tiles >> 3) + (tile >> 3); // workgroups of one XCD share x tiles
    const int mt0 = (tile / nt) * MI, n0 = (tile % nt) * 128;
    const int nsb_row = a.k >> 8, steps_row = a.k >> 6;
    const int lo = (int)blockIdx.y * a.sb_per_split, hi = lo + a.sb_per_split < nsb_row ? lo + a.sb_per_split : nsb_row;
    const int loops = (hi - lo + 1) / 2, sb0 = lo + half * loops; // the second half may have one less, and walks through it without its products
    const int mine = hi - sb0 < loops ? hi - sb0 : loops;
    uint8_t *xbase = lds + half * Tile::GROUP, *wbase = xbase + NX * XBYTES, *sbase = wbase + Tile::NW * WBYTES, *dbase = sbase + Tile::SBYTES;
    const bool x_wave = wn < 2; // copies x, the others codes, sums and sides
    const int cw = wn & 1;

    // ---- copies into LDS (past the end of the row: its last step, unit or superblock again, which nobody looks at)
    auto copy = [&](const void *base, uint32_t off, uint8_t *dst) { // a wave's place in scalar registers, a lane's in 32 bits: registers are short
        asm volatile("" : "+v"(off)); // extended where it is used
        __builtin_amdgcn_global_load_lds((gbl_void *)(reinterpret_cast<const uint8_t *>(base) + off), (lds_void *)dst, 16, 0, 0);
    };
    const uint32_t lane16 = lane * 16;
    auto in_order = [] { asm volatile("" ::: "memory"); }; // the waits in front of the barriers count on the order of the requests
    auto copy_x = [&](int g, int at, int piece) {
        int step = sb0 * 4 + g;
        step = step < steps_row ? step : steps_row - 1;
        const int q = piece >> 2, t = piece & 3;
        copy(a.xa + ((size_t)(mt0 + cw * 2 + q) * steps_row + step) * 2048 + t * 512, lane16, xbase + at + (cw * 2 + q) * 4096 + t * 1024);
        in_order();
    };
    auto copy_sums = [&](int sb, int piece) {
        const int at = sb0 + sb < nsb_row ? sb0 + sb : nsb_row - 1;
        const int q = piece >> 1, t = piece & 1;
        if constexpr (T::MIN) copy(a.xs + ((size_t)(mt0 + cw * 2 + q) * nsb_row + at) * 1024 + t * 512, lane16, sbase + (cw * 2 + q) * 2048 + t * 1024);
        in_order();
    };
    const int cr = lane >> 1, cs = (lane & 1) ^ ((cr >> 3) & 1); // see rows_gemm_kernel
    auto row_of = [&](int r) { return (uint32_t)(n0 + r < a.n ? r : a.n - 1 - n0); };
    auto copy_codes = [&](int u, int at, int piece) {
        int unit = sb0 * 2 + u;
        unit = unit < 2 * nsb_row ? unit : 2 * nsb_row - 1;
        const int ct = cw * 2 + piece / T::PAIRS, p = piece % T::PAIRS; // column tile of 32 rows
        const uint32_t row = row_of(ct * 32 + cr);
        copy(T::piece_src(a, unit, p) + (size_t)n0 * T::piece_pitch(a, p), row * T::piece_pitch(a, p) + cs * 16, wbase + at + ct * 32 * HB + p * 1024);
        in_order();
    };
    auto copy_sides = [&](int sb, int c) { // 64 rows of piece c
        const int at = sb0 + sb < nsb_row ? sb0 + sb : nsb_row - 1, r0 = cw * 64;
        const uint8_t *src = T::side_src(a, at, c) + (size_t)n0 * T::side_pitch(a, c);
        uint32_t off = row_of(r0 + lane) * T::side_pitch(a, c);
        asm volatile("" : "+v"(off));
        if (c < T::SIDE16) copy(src, off, dbase + c * 128 * 16 + r0 * 16);
        else __builtin_amdgcn_global_load_lds((gbl_void *)(src + off), (lds_void *)(dbase + T::SIDE16 * 128 * 16 + r0 * 4), 4, 0, 0);
        in_order();
    };
    auto all = [](int n, auto fn) {
#pragma unroll
        for (int p = 0; p < n; p++) fn(p);
    };
    auto turn_over = [] {
        __builtin_amdgcn_sched_barrier(0);
        barrier();
        __builtin_amdgcn_sched_barrier(0);
    };

    float16v part[MI], total[MI][1];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) total[i][0][r] = part[i][r] = 0.f;
    float unit = 0.f, inv = 0.f, shrink;
    typename T::Side side, next_side;
    typename T::Scales scales;
    uint32_t mask; // in a vector register: an instruction takes one scalar operand, and (w & mask) | base has its base there
    asm("v_mov_b32 %0, 0x00f000f0" : "=v"(mask));
    const uint8_t *my_x = xbase + lane * 16, *my_codes = wbase + wn * 32 * HB;
    auto fold = [&] { // the sums of two steps join the total
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int q = 0; q < 16; q++) total[i][0][q] = fmaf(part[i][q], unit, total[i][0][q]);
    };
    // ---- the requests in front of the first turn, in the order of the later ones
    if (x_wave) {
        all(Tile::XL, [&](int p) { copy_x(0, 0, p); });
        all(Tile::XL, [&](int p) { copy_x(1, XBYTES, p); });
        wait_loads_and_lds<Tile::XL>();
    } else {
        all(Tile::D, [&](int p) { copy_sides(0, p); });
        all(Tile::WL, [&](int p) { copy_codes(0, 0, p); });
        all(Tile::SL, [&](int p) { copy_sums(0, p); });
        all(Tile::WL, [&](int p) { copy_codes(1, WBYTES, p); });
        wait_loads_and_lds<Tile::SL + Tile::WL>();
    }
    barrier();
    T::template read_side<128>(dbase, wn * 32 + li, hh, sb0, next_side);
    if (half) turn_over(); // the second half is a turn behind
    int x_at = 0;
    auto turn = [&](int sb, auto which, auto copier) __attribute__((always_inline)) {
        constexpr bool COPIES_X = decltype(copier)::value;
        constexpr int J = decltype(which)::value;
        const bool live = sb < mine;
        // x and operands of the products t = 0 and 1; those of 2 and 3 take their place when they are done with
        half8 xf[2][MI], wf[2][T::PRODUCTS];
        auto read_x = [&](int t, int i) { xf[t & 1][i] = *reinterpret_cast<const half8 *>(my_x + x_at + i * 4096 + t * 1024); };
        typename T::Raw raw;
        half8 offs;
        int over = 0;
        // ---- fetch
        T::read_raw(my_codes + (J >> 1) * WBYTES, li, hh, J, raw);
        in_order();
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int i = 0; i < MI; i++) read_x(t, i);
        in_order();
        if (J == 0) {
            if (sb > 0) fold(); // of the superblock before
            side = next_side;
            T::unit_of(side, unit, inv, shrink);
            T::scales(side, shrink, hh, scales);
        }
        if (J == 2 && live) fold();
        if constexpr (J == 1)
            if constexpr (T::MIN) {
                over = T::excess(side);
                offs = T::offsets(side, hh, inv * __builtin_bit_cast(float, (uint32_t)(127 - over) << 23));
                asm volatile("" : "+v"(offs));
            }
        if (J == 3) T::template read_side<128>(dbase, wn * 32 + li, hh, sb0 + sb + 1, next_side);
#pragma unroll
        for (int i = 0; i < MI; i++) asm volatile("" : "+v"(total[i][0])); // added here, while x is on its way, not behind the wait
        auto make = [&](int t) {
            T::make(raw, side, scales, mask, J, t, hh, wf[t & 1]);
#pragma unroll
            for (int pr = 0; pr < T::PRODUCTS; pr++) asm volatile("" : "+v"(wf[t & 1][pr]));
        };
        make(0);
        make(1);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        turn_over();
        // ---- multiply
        auto between = [&](int slot) { // copies, piece by piece between the products (see rows_wide_kernel)
            __builtin_amdgcn_sched_barrier(0);
            if (COPIES_X) {
                if (slot % 2 == 0) copy_x(4 * sb + J + 2, x_at == 0 ? (NX - 1) * XBYTES : x_at - XBYTES, slot / 2); // the place of the step that everybody has read
            } else {
                if (J == 0 && slot < Tile::D) copy_sides(sb + 1, slot);
                if (J == 2 && slot < Tile::SL) copy_sums(sb + 1, slot);
                if ((J & 1) && slot < Tile::WL) copy_codes(2 * sb + (J >> 1) + 2, (J >> 1) * WBYTES, slot);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        __builtin_amdgcn_s_setprio(1);
        const float16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int pr = 0; pr < T::PRODUCTS; pr++)
#pragma unroll
                for (int i = 0; i < MI; i++) {
                    if (pr == 0 && i == 1 && (t == 1 || t == 2)) make(t + 1);
                    part[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[t & 1][i], wf[t & 1][pr], J % 2 == 0 && t == 0 && pr == 0 ? zero : part[i], 0, 0, 0);
                    if (pr == 0) between(t * MI + i);
                    if (t < 2 && pr == T::PRODUCTS - 1) read_x(t + 2, i);
                }
        if constexpr (T::MIN && J == 1) {
            auto times_pow2 = [&](int e) { // a column's lanes all have its factor; exact, being a power of two
                if (__builtin_amdgcn_ballot_w64(over > 0) == 0) return;
                const float f = __builtin_bit_cast(float, (uint32_t)(127 + e * over) << 23);
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int q = 0; q < 16; q++) part[i][q] *= f;
            };
            times_pow2(-1);
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int i = 0; i < MI; i++)
                    part[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8 *>(sbase + i * 2048 + t * 1024 + lane * 16), offs, part[i], 0, 0, 0);
            times_pow2(1);
        }
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        if (COPIES_X) wait_loads_and_lds<Tile::XL>(); // what the next turns read
        else if (J == 0 || J == 1) wait_loads_and_lds<Tile::WL + Tile::D>();
        else wait_loads_and_lds<Tile::WL + Tile::SL>();
        turn_over();
        x_at = x_at == (NX - 1) * XBYTES ? 0 : x_at + XBYTES;
    };
    auto run = [&](auto copier) __attribute__((always_inline)) { // a loop for each kind of wave, see rows_wide_kernel
        for (int sb = 0; sb < loops; sb++) {
            turn(sb, std::integral_constant<int, 0>{}, copier); turn(sb, std::integral_constant<int, 1>{}, copier);
            turn(sb, std::integral_constant<int, 2>{}, copier); turn(sb, std::integral_constant<int, 3>{}, copier);
        }
    };
    if (x_wave) run(std::true_type{});
    else run(std::false_type{});
    if (mine == loops) fold(); // else the last one was not this half's
    if (!half) barrier();
    wait_loads_and_lds<0>(); // nothing of this workgroup may still be on its way into LDS
    barrier();
    // ---- each half finishes two of the four row tiles and hands the sums of the others over
    float *mail = reinterpret_cast<float *>(lds) + (half * 4 + wn) * 2048 + lane;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) mail[(i * 16 + r) * 64] = half ? total[i][0][r] : total[i + 2][0][r];
    __syncthreads();
    const float *got = reinterpret_cast<const float *>(lds) + ((1 - half) * 4 + wn) * 2048 + lane;
    float16v out[2][1];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) out[i][0][r] = (half ? total[i + 2][0][r] : total[i][0][r]) + got[(i * 16 + r) * 64];
    __syncthreads(); // the patches lie where the mail was
    write_rows<2, 1>(a, out, reinterpret_cast<float *>(lds) + wave * (32 * 36), (mt0 + half * 2) * 32, n0 + wn * 32, lane);
}

// Rows of x in operand order (see RowsArgs::xa, xs) under a power-of-two scale per row.  IN: 0 f32 rows, RMS-normalised where
// norm_w is given ((x * inv_rms) * norm_w, RMSNorm::forward, llm/src/llama.rs:158-187); 1 f32 rows of 2 k gate/up values, four
// and four, which become silu(gate) * up; 2 bf16 rows.  f32 rows become two rows each.  A workgroup per row, a thread per
// eight elements; the row stays in registers (NC times 4096 elements) or, NC = 0, is read once per pass.  Few rows: NC workgroups
// per row, which all look for its largest element and write 4096 elements each (see launch_prep).  3: as 0, of rows that are still sums of
// parts of K, which are added up, in gemm_reduce_kernel's order, and written as well.
// Eight neighbouring rows' pieces fill a line of 128 bytes of the operand (four rows', where rows become two), so they go to one XCD, whose L2
// puts the line together: workgroups go round the XCDs, and the number of a row is that of its workgroup with the middle digits exchanged
// (as many workgroups as make whole 64 rows).  2048 bf16 rows of 4096: 18.5 us with row = workgroup, 11.5 so; SwiGLU, 511 rows of 14336: 26.4, 22.5; whole
// calls: 2048 x 14336 x 4096 291.5 285.3, 509 x 4096 x 4096 54.5 52.7, 33 f32 rows x 4096 x 14336 36.9 35.1.
struct PartSums {
    const float *part, *scale; // [splits][rows][k]; scale of row t at [t * mul]
    int splits, mul;
    const float *resid;        // [rows][k] or NULL
    float *y;
};
struct NoSums {};
__device__ inline void add_parts(const PartSums &ps, size_t row, int rows, int k, int c, float (&e)[8]) {
    typedef float float4v __attribute__((ext_vector_type(4)));
    const size_t stride = (size_t)rows * k / 4;
    const float4v *from = reinterpret_cast<const float4v *>(ps.part + row * k) + 2 * c;
    float lost[8];
    float4v v[8][2];
#pragma unroll
    for (int s = 0; s < 8; s++)
        if (s < ps.splits) {
            v[s][0] = from[s * stride];
            v[s][1] = from[s * stride + 1];
        }
    const float scale = ps.scale[row * ps.mul];
    float4v res[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    if (ps.resid) {
        res[0] = (reinterpret_cast<const float4v *>(ps.resid + row * k) + 2 * c)[0];
        res[1] = (reinterpret_cast<const float4v *>(ps.resid + row * k) + 2 * c)[1];
    }
#pragma unroll
    for (int q = 0; q < 8; q++) {
        e[q] = v[0][q >> 2][q & 3];
        lost[q] = 0.f;
    }
    auto add = [&](int q, float x) {
        const float sum = e[q] + x, part = sum - e[q];
        lost[q] += (e[q] - (sum - part)) + (x - part);
        e[q] = sum;
    };
#pragma unroll
    for (int s = 1; s < 8; s++)
        if (s < ps.splits)
#pragma unroll
            for (int q = 0; q < 8; q++) add(q, v[s][q >> 2][q & 3]);
    for (int s = 8; s < ps.splits; s++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float4v x = from[s * stride + h];
#pragma unroll
            for (int q = 0; q < 4; q++) add(4 * h + q, x[q]);
        }
    float4v out[2];
#pragma unroll
    for (int q = 0; q < 8; q++) {
        e[q] = (lost[q] == lost[q] ? e[q] + lost[q] : e[q]) * scale; // not a number beside an infinite sum
        if (ps.resid) e[q] += res[q >> 2][q & 3];
        out[q >> 2][q & 3] = e[q];
    }
    float4v *to = reinterpret_cast<float4v *>(ps.y + row * k) + 2 * c;
    to[0] = out[0];
    to[1] = out[1];
}
template <int IN, int NC, bool LIMBS>
__global__ void __launch_bounds__(512) rows_prep_kernel(const void *x, const float *norm_w, float eps, int rows, int k, int kp, _Float16 *xa, _Float16 *xs,
                                                        float *rowscale, std::conditional_t<IN == 3, PartSums, NoSums> sums) {
    constexpr int HELD = NC > 0 ? NC : 1;
    __shared__ float red[8];
    const int row = (int)((blockIdx.x & ~63u) | (blockIdx.x & 7) << 3 | (blockIdx.x >> 3 & 7)), tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, chunks = k >> 3, all = kp >> 3; // of eight elements: the row's, the operand's (zeros behind the row)
    if (row >= rows) return;
    float v[HELD][8];
    auto load = [&](int c, float (&e)[8]) {
        if constexpr (IN == 3) {
            add_parts(sums, row, rows, k, c, e);
        } else if (IN == 2) {
            const u32x4 r = reinterpret_cast<const u32x4 *>(reinterpret_cast<const uint16_t *>(x) + (size_t)row * k)[c];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                e[2 * i] = __builtin_bit_cast(float, r[i] << 16);
                e[2 * i + 1] = __builtin_bit_cast(float, r[i] & 0xFFFF0000u);
            }
        } else if (IN == 1) {
            const float4 *p = reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(x) + (size_t)row * 2 * k) + 4 * (size_t)c;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const float4 g = p[2 * i], u = p[2 * i + 1];
                e[4 * i] = (g.x * (1.0f / (1.0f + expf(-g.x)))) * u.x;
                e[4 * i + 1] = (g.y * (1.0f / (1.0f + expf(-g.y)))) * u.y;
                e[4 * i + 2] = (g.z * (1.0f / (1.0f + expf(-g.z)))) * u.z;
                e[4 * i + 3] = (g.w * (1.0f / (1.0f + expf(-g.w)))) * u.w;
            }
        } else {
            const float4 *p = reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(x) + (size_t)row * k) + 2 * (size_t)c;
            const float4 l = p[0], h = p[1];
            e[0] = l.x; e[1] = l.y; e[2] = l.z; e[3] = l.w; e[4] = h.x; e[5] = h.y; e[6] = h.z; e[7] = h.w;
        }
    };
    // all threads go through `all` in steps of 512; `fn(e, c, i)`: e the elements of chunk c, the i-th of this thread
    auto each = [&](bool first, auto fn) {
        if constexpr (NC > 0) {
#pragma unroll
            for (int i = 0; i < NC; i++) {
                const int c = i * 512 + tid;
                if (first) {
                    if (c < chunks) load(c, v[i]);
                    else
#pragma unroll
                        for (int q = 0; q < 8; q++) v[i][q] = 0.f;
                }
                fn(v[i], c);
            }
        } else {
            for (int c = tid; c < (all + 511) / 512 * 512; c += 512) {
                float e[8];
                if (c < chunks) load(c, e);
                else
#pragma unroll
                    for (int q = 0; q < 8; q++) e[q] = 0.f;
                fn(e, c);
            }
        }
    };
    float inv = 1.0f;
    const bool norm = (IN == 0 || IN == 3) && norm_w;
    bool first = true;
    if (norm) {
        float ss = 0.f;
        each(true, [&](float (&e)[8], int) {
#pragma unroll
            for (int q = 0; q < 8; q++) ss = fmaf(e[q], e[q], ss);
        });
        first = false;
#pragma unroll
        for (int s = 32; s >= 1; s >>= 1) ss += __shfl_xor(ss, s);
        if (lane == 0) red[wave] = ss;
        __syncthreads();
        ss = ((red[0] + red[1]) + (red[2] + red[3])) + ((red[4] + red[5]) + (red[6] + red[7]));
        __syncthreads();
        inv = 1.0f / sqrtf(ss / (float)k + eps);
    }
    auto normed = [&](float (&e)[8], int c) {
        if (!norm || c >= chunks) return;
        const float4 l = reinterpret_cast<const float4 *>(norm_w)[2 * c], h = reinterpret_cast<const float4 *>(norm_w)[2 * c + 1];
        e[0] = (e[0] * inv) * l.x; e[1] = (e[1] * inv) * l.y; e[2] = (e[2] * inv) * l.z; e[3] = (e[3] * inv) * l.w;
        e[4] = (e[4] * inv) * h.x; e[5] = (e[5] * inv) * h.y; e[6] = (e[6] * inv) * h.z; e[7] = (e[7] * inv) * h.w;
    };
    uint32_t top = 0; // largest |v| as an integer: a NaN ranks above everything and is not dropped
    each(first, [&](float (&e)[8], int c) {
        normed(e, c); // the registers hold normed values from here on
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const uint32_t b = __builtin_bit_cast(uint32_t, e[q]) & 0x7FFFFFFFu;
            top = b > top ? b : top;
        }
    });
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) {
        const uint32_t o = (uint32_t)__shfl_xor((int)top, s);
        top = o > top ? o : top;
    }
    if (lane == 0) red[wave] = __builtin_bit_cast(float, top);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t o = __builtin_bit_cast(uint32_t, red[i]);
        top = o > top ? o : top;
    }
    // top in [2^e, 2^(e+1)) -> multiply by 2^(14 - e), the most that f16 holds: what the smallest elements lose is what lies below
    // 2^-39 of the row's largest; a sum of 32 stays below 2^20; inf/nan rows are passed through unscaled
    int eb = (int)(top >> 23);
    if (eb == 0 || eb == 0xFF) eb = 127 + 14;
    int sb = 127 + 14 - (eb - 127);
    sb = sb < 1 ? 1 : (sb > 254 ? 254 : sb);
    const float f = __builtin_bit_cast(float, (uint32_t)sb << 23);
    constexpr int PARTS = LIMBS ? 3 : IN == 2 ? 1 : 2;
    const int r0 = row * PARTS, steps = kp >> 6, nsb = kp >> 8;
    auto slot = [&](int part) { // of the operand's rows: pairs are neighbours; limbs see RowsTile, part 3 = the zeros
        if (!LIMBS) return r0 + part;
        return rows <= 16 ? (part < 2 ? part : 5 - part) * 16 + row : row < 32 ? part * 32 + row : 96 + part * 8 + (row & 7);
    };
    each(false, [&](float (&e)[8], int c) {
        if (NC > 1 && gridDim.y > 1 && (unsigned)(c >> 9) != blockIdx.y) return; // another workgroup's
        if (NC == 0) normed(e, c);
        _Float16 p[PARTS][8];
        float sum[PARTS];
#pragma unroll
        for (int part = 0; part < PARTS; part++) sum[part] = 0.f;
        // limbs: the first is a multiple of 2^(g - LB), at most 2^(LB + 1) of it, 2^g the magnitude of the block's largest (a block of 32
        // is four threads'); the second and the third, times 2^(LB + 2), are what that leaves
        float grid = 0.f, ungrid = 0.f;
        if (LIMBS) {
            uint32_t most = 0;
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const uint32_t b = __builtin_bit_cast(uint32_t, e[q] * f) & 0x7FFFFFFFu;
                most = b > most ? b : most;
            }
#pragma unroll
            for (int m = 1; m <= 2; m <<= 1) {
                const uint32_t o = (uint32_t)__shfl_xor((int)most, m);
                most = o > most ? o : most;
            }
            int g = (int)(most >> 23) - 127;
            g = g < LB - 24 ? LB - 24 : g > 14 ? 14 : g; // f16's smallest number is 2^-24
            grid = __builtin_bit_cast(float, (uint32_t)(127 + g - LB) << 23);
            ungrid = __builtin_bit_cast(float, (uint32_t)(127 - g + LB) << 23);
        }
#pragma unroll
        for (int q = 0; q < 8; q++) {
            float s = e[q] * f;
#pragma unroll
            for (int part = 0; part < PARTS; part++) {
                p[part][q] = LIMBS && part == 0 ? (_Float16)(rintf(s * ungrid) * grid) : (_Float16)s;
                sum[part] += (float)p[part][q];
                s -= (float)p[part][q];
                if (LIMBS && part == 0) s *= (float)(1 << (LB + 2));
            }
        }
        float carry = 0.f; // what a limb's pair of sums does not hold goes to the next limb's
        // chunk c: step c / 8, product t, half of the lanes (see the order of elements above)
        const int at = c & 7, t = (at >> 2) * 2 + (at & 1), h = (at >> 1) & 1;
#pragma unroll
        for (int part = 0; part < PARTS + (LIMBS ? 1 : 0); part++) {
            if (part == PARTS && rows > 16) break;
            const int at_row = slot(part), lrow = at_row & 31;
            _Float16 *xt = xa + (size_t)(at_row >> 5) * steps * 2048, *st = xs + (size_t)(at_row >> 5) * nsb * 1024;
            const _Float16 *s = p[part < PARTS ? part : 0];
            const half8 out = part < PARTS ? half8{s[0], s[2], s[1], s[3], s[4], s[6], s[5], s[7]} : half8{0, 0, 0, 0, 0, 0, 0, 0};
            if (c < all)
                *reinterpret_cast<half8 *>(xt + ((size_t)(c >> 3) * 4 + t) * 512 + (h * 32 + lrow) * 8) = out;
            // the sum of 32 elements: four threads; times 1 / 64 it stays within f16's range
            float g = part < PARTS ? sum[part] : 0.f;
            g += __shfl_xor(g, 1);
            g += __shfl_xor(g, 2);
            if ((tid & 3) == 0 && c < all) {
                g = part < PARTS ? fmaf(g, 1.0f / 64.0f, carry) : 0.f;
                const _Float16 ghi = (_Float16)g, glo = (_Float16)(g - (float)ghi);
                if (LIMBS) carry = (g - (float)ghi - (float)glo) * (part == 0 ? (float)(1 << (LB + 2)) : 1.0f);
                const int sub = (c >> 2) & 7;
                _Float16 *d = st + (size_t)(c >> 5) * 1024 + ((sub >> 2) * 32 + lrow) * 8 + (sub & 3);
                d[0] = ghi; d[4] = ghi;
                d[512] = glo; d[516] = glo;
            }
        }
    });
    if ((NC <= 1 || blockIdx.y == 0) && tid < (LIMBS ? 1 : PARTS)) rowscale[(LIMBS ? row : r0) + tid] = 1.0f / f;
}

template <class T, int MI, int WM, int AT>
int launch_tile(axq_ctx *ctx, const RowsArgs &a, int splits) {
    using Tile = RowsTile<T, MI, WM, AT>;
    static std::atomic<uint64_t> lds_allowed{0};
    if (int rc = axq_allow_lds(ctx, reinterpret_cast<const void *>(rows_gemm_kernel<T, MI, WM, AT>), lds_allowed, Tile::LDS)) return rc;
    const unsigned tiles = (unsigned)(((a.n + Tile::N - 1) / Tile::N) * ((a.m + Tile::M - 1) / Tile::M));
    rows_gemm_kernel<T, MI, WM, AT><<<dim3(tiles, (unsigned)splits), 512, Tile::LDS, ctx->stream>>>(a);
    AXQ_LAUNCH_CHECK(ctx, "rows_gemm_kernel");
    return AXQ_OK;
}

template <class T>
int launch_wide(axq_ctx *ctx, const RowsArgs &a, int splits) {
    static std::atomic<uint64_t> lds_allowed{0};
    if (int rc = axq_allow_lds(ctx, reinterpret_cast<const void *>(rows_wide_kernel<T>), lds_allowed, WideTile<T>::LDS)) return rc;
    const unsigned tiles = (unsigned)(((a.n + 255) / 256) * ((a.m + 255) / 256));
    rows_wide_kernel<T><<<dim3(tiles, (unsigned)splits), 512, WideTile<T>::LDS, ctx->stream>>>(a);
    AXQ_LAUNCH_CHECK(ctx, "rows_wide_kernel");
    return AXQ_OK;
}

template <class T>
int launch_blocks(axq_ctx *ctx, const RowsArgs &a, int splits) {
    static std::atomic<uint64_t> lds_allowed{0};
    if (int rc = axq_allow_lds(ctx, reinterpret_cast<const void *>(rows_blocks_kernel<T>), lds_allowed, BlocksTile<T>::LDS)) return rc;
    const unsigned tiles = (unsigned)(((a.n + 127) / 128) * ((a.m + 255) / 256));
    rows_blocks_kernel<T><<<dim3(tiles, (unsigned)splits), 512, BlocksTile<T>::LDS, ctx->stream>>>(a);
    AXQ_LAUNCH_CHECK(ctx, "rows_blocks_kernel");
    return AXQ_OK;
}

template <class T>
int launch_apart(axq_ctx *ctx, const RowsArgs &a, int splits) {
    static std::atomic<uint64_t> lds_allowed{0};
    if (int rc = axq_allow_lds(ctx, reinterpret_cast<const void *>(rows_apart_kernel<T>), lds_allowed, ApartTile<T>::LDS)) return rc;
    const unsigned tiles = (unsigned)(((a.n + 127) / 128) * ((a.m + 127) / 128));
    rows_apart_kernel<T><<<dim3(tiles, (unsigned)splits), 512, ApartTile<T>::LDS, ctx->stream>>>(a);
    AXQ_LAUNCH_CHECK(ctx, "rows_apart_kernel");
    return AXQ_OK;
}

// Up to 64 rows of more than 4096 elements a workgroup for every 4096 of each: as many as there are rows leave most of the chip idle, and what a
// row costs most is its conversion (21 rows of 11008, limbs: 8.6 us with one, 6.5 so; 64 rows of 14336, SwiGLU: 9.7, 8.1).
template <int IN, bool LIMBS>
void launch_prep(hipStream_t st, const void *x, const float *norm_w, float eps, int rows, int k, int kp, _Float16 *xa, _Float16 *xs, float *rs) {
    const unsigned grid = (unsigned)(rows + 63) / 64 * 64;
    const int parts = rows <= 64 ? (kp + 4095) / 4096 : 1;
    if (kp <= 4096) rows_prep_kernel<IN, 1, LIMBS><<<grid, 512, 0, st>>>(x, norm_w, eps, rows, k, kp, xa, xs, rs, {});
    else if (kp <= 8192) rows_prep_kernel<IN, 2, LIMBS><<<dim3(grid, parts), 512, 0, st>>>(x, norm_w, eps, rows, k, kp, xa, xs, rs, {});
    else if (IN == 1 || kp <= 16384) rows_prep_kernel<IN, 4, LIMBS><<<dim3(grid, parts), 512, 0, st>>>(x, norm_w, eps, rows, k, kp, xa, xs, rs, {}); // SwiGLU rows are no longer
    else if constexpr (IN != 1) rows_prep_kernel<IN, 0, LIMBS><<<grid, 512, 0, st>>>(x, norm_w, eps, rows, k, kp, xa, xs, rs, {});
}

// How many tiles of 128 x 128 outputs a call of m rows of operands has, where 256 x 256 are the alternative.
int64_t square_tiles(int64_t m, int64_t n) { return m <= 128 ? 0 : (m + 127) / 128 * ((n + 127) / 128); }

// Superblock types: 256 x 256 outputs per workgroup, which make an operand once for twice the rows, where tiles of 128 x 128 are
// more than one to two compute units, or where K in parts of at least four superblocks (shorter ones are mostly the start and the
// partial sums) gives the large tiles a workgroup per compute unit.  Else 128 x 128.  Time with large and small tiles, us:
//   f32 rows   Q4_K 4096 x 4096, 128: 36.8 27.3 (16 large tiles and eight parts are half the chip); 256: 43.0 39.5
//              Q4_K 1024 x 4096, 128: 34.4 21.3;  Q5_K 4096 x 4096, 128: 38.8 29.4;  Q6_K 4096 x 14336, 128: 102 83
//              Q4_K 4096 x 14336, 256 (128 small tiles, 32 large ones in eight parts): 93 105;  Q5_K 6144 x 4096, 160 (144): 54 61
//   bf16 rows  Q4_K 4096 x 4096, 256: 43.0 29.0; 512 (128 small ones): 52 42;  1024 x 4096, 1024: 47 34.5;  4096 x 14336, 700 (192): 141 173
bool wide_tiles(const axq_ctx *ctx, int64_t m, int64_t n, int64_t k) {
    const int64_t cus = ctx->prop.multiProcessorCount, parts = k >> 10;
    return m > 128 && (square_tiles(m, n) > cus / 2 || (m + 255) / 256 * ((n + 255) / 256) * (parts < 8 ? parts : 8) >= cus);
}

// How a call goes to the workgroups.
struct RowsPlan {
    bool limbs, wide, apart;     // kinds of tile: see launch_rows
    int parts, m, bm;            // rows of the operand per row of x, all of them, and of a tile
    long tiles;
    int splits, sb_per_split;    // of K
};

RowsPlan rows_plan(const axq_ctx *ctx, const axq_weight *w, int in, int rows, bool whole_k = false) {
    RowsPlan p;
    p.limbs = in != AXQ_ROWS_BF16 && rows < AXQ_ROWS_PAIRS_MIN;
    p.parts = in == AXQ_ROWS_BF16 || p.limbs ? 1 : 2;
    p.m = rows * p.parts;
    const bool super = w->type == AXQ_Q4_K || w->type == AXQ_Q5_K || w->type == AXQ_Q6_K;
    const int n = (int)w->n_rows, nsb = (int)(w->kp >> 8);
    // Blocks of 32 take large tiles where the small ones are more than one to a compute unit: their sums of a superblock, which keep additions
    // of the total's size few, fit the registers of 128 x 128 outputs only (Q4_0, K = 4096: an error of 0.83 10^-7 there, 2.0 in large tiles).
    // bf16 rows, us in the former kernel of that range, with operands in LDS, and now: 2048 x 14336 x 4096 Q4_0 414 331, Q5_0 482 365,
    // Q5_1 557 414, Q8_0 447 354.
    p.wide = !p.limbs && (super ? wide_tiles(ctx, p.m, n, w->kp) : square_tiles(p.m, n) > ctx->prop.multiProcessorCount);
    const int groups = p.m <= (p.limbs ? 32 : 64) ? 2 : 1; // of waves along K
    p.bm = p.limbs ? (rows <= 32 ? 32 : 40) : p.m <= 32 ? 32 : p.m <= 64 ? 64 : p.wide ? 256 : 128;
    const int bn = p.wide && super ? 256 : 128;
    p.tiles = (long)((n + bn - 1) / bn) * ((p.m + p.bm - 1) / p.bm);
    // K is split over as many workgroups as leave every group of waves a superblock, up to one workgroup per compute unit: into sixteen
    // parts at most for 17 to 39 rows (eight and sixteen, 1024 x 14336: Q6_K, 39 rows 55.5 42.4 us; Q4_K, 17 rows 33.9 29.6, with
    // thirty-two 30.4), else eight (2048 x 8192, ten rows: Q4_0 19.6 us, sixteen 20.4; Q4_K 20.8, 21.6)
    static_assert(AXQ_ROWS_PAIRS_MIN <= 40, "limbs of at most 40 rows");
    const int most = p.limbs && rows > 16 ? 16 : 8;
    int splits = (int)(ctx->prop.multiProcessorCount / p.tiles);
    if (splits > nsb / groups) splits = nsb / groups;
    if (splits > most) splits = most;
    if (splits < 2 || whole_k) splits = 1;
    p.sb_per_split = (nsb + splits - 1) / splits;
    p.splits = (nsb + p.sb_per_split - 1) / p.sb_per_split;
    // 128 x 128 outputs whose halves have K of their own, from two superblocks per workgroup on (a last part may have one: its second half then only
    // keeps step).  f32 rows, us so and with shared K: 64 rows, Q4_K 28672 x 4096
    // (sixteen per workgroup) 52.5 62.7, Q5_K and Q6_K 14336 x 4096 (eight) 36.5 43.7 and 44.0 52.0, 4096 x 14336 (seven) Q4_K 36.5 36.8, Q5_K
    // 41.3 43.8, Q6_K 48.6 50.8, 6144 x 4096 (four) Q4_K 24.3 26.4, Q6_K 27.9 31.1, Q4_K 4096 x 4096 (two) 21.5 23.1; 100 bf16 rows, Q4_K 4096 x
    // 14336 36.1 37.0.  Error against 64 bits, 64 rows, three seeds, 1e-8: Q4_K 6144 x 4096 11.29 11.34 11.30 and 11.26 11.32 11.30, 4096 x 14336
    // 11.75 11.76 11.74 and 11.71 11.72 11.70, Q6_K 6144 x 4096 12.31 12.33 12.33 and 12.31 12.34 12.33: the same additions in another order.
    p.apart = super && !p.limbs && !p.wide && p.m > 64 && p.sb_per_split >= 2;
    return p;
}

// The tile of a call.  Limbs: up to 16 and 32 rows the two halves of the waves on two parts of K, since a workgroup's time is then its
// number of steps; more, which are fewer than 40, see RowsTile.  Others: up to 32 and 64 rows of operands the same with one and two row tiles
// per wave; above two times two row tiles, or halves on K of their own, or large tiles (see rows_plan for both).
template <class T>
int launch_rows(axq_ctx *ctx, const RowsArgs &a, const RowsPlan &p) {
    if (p.limbs) {
        if (a.m > 32) return launch_tile<T, 2, 2, 4>(ctx, a, p.splits);
        if (a.m > 16) return launch_tile<T, 2, 1, 3>(ctx, a, p.splits);
        return launch_tile<T, 1, 1, 2>(ctx, a, p.splits);
    }
    if constexpr (!T::BLOCKS) {
        if (p.wide) return launch_wide<T>(ctx, a, p.splits);
        if (p.apart) return launch_apart<T>(ctx, a, p.splits);
    }
    if constexpr (T::BLOCKS)
        if (p.wide) return launch_blocks<T>(ctx, a, p.splits);
    if (a.m > 64) return launch_tile<T, 2, 2, 1>(ctx, a, p.splits);
    if (a.m > 32) return launch_tile<T, 2, 1, 1>(ctx, a, p.splits);
    return launch_tile<T, 1, 1, 1>(ctx, a, p.splits);
}

} // namespace

// Packed types at any number of rows, whole superblocks in the planes; K a multiple of 64, which every GEMM asks for, whatever its planes hold.
bool axq_dev_rows_gemm_covers(const axq_weight *w, int rows) {
    if (w->kp % 256 != 0 || w->k % 64 != 0 || w->kp > INT32_MAX || w->n_rows > INT32_MAX || rows < 1) return false;
    switch (w->type) {
    case AXQ_Q4_K: case AXQ_Q5_K: case AXQ_Q6_K: case AXQ_Q4_0: case AXQ_Q4_1: case AXQ_Q5_0: case AXQ_Q5_1: case AXQ_Q8_0: return true;
    default: return false;
    }
}

// Whether axq_gemv_f32 takes this kernel for `rows` f32 rows, of which the small-batch GEMV would make groups of eight.  From 17 on,
// where those are three passes over the weights or more, always: 1.03 (1024 x 14336) to 2.8 times as fast.  10 to 16 rows are two
// passes, beside which the pre-pass, a workgroup per row, and the reduction weigh more the longer K is and the fewer weight rows there
// are.  Speed over two passes with 10 and 16 rows:
//              Q8_0        Q6_K        Q4_0        Q5_1        Q4_K        Q5_K
//   4096x14336 1.20 1.18   1.06 1.05   1.05 1.02   1.00 0.98   0.98 0.97   0.93 0.91
//   1024x14336 0.85 0.78   0.84 0.80   0.87 0.82   0.78 0.73   0.83 0.78   0.77 0.73
//   4096x8192  1.22 1.17   1.12 1.09   1.12 1.06   1.07 1.02   1.05 1.01   1.04 0.99
//   2048x8192  1.09 1.02   0.95 0.93   1.18 1.12   0.96 0.90   1.10 1.04   1.00 0.95
//   4096x4096  1.38 1.30   1.22 1.16   1.50 1.41   1.26 1.17   1.35 1.29   1.27 1.20
//   6144x4096  1.08 1.04   1.09 1.05   1.06 1.00   1.01 0.97   1.02 0.97   0.96 0.92   (three quarters of the compute units)
//   9216x4096  1.34 1.32   1.28 1.27   1.21 1.14   1.16 1.13   1.14 1.11   1.15 1.12
bool axq_dev_rows_gemm_pays(const axq_ctx *ctx, const axq_weight *w, int rows) {
    if (rows < AXQ_ROWS_GEMM_MIN || !axq_dev_rows_gemm_covers(w, rows)) return false;
    if (rows > 16) return true;
    const bool slow_gemv = w->type == AXQ_Q8_0 || w->type == AXQ_Q6_K || w->type == AXQ_Q4_0;
    if (w->k > 8192) return slow_gemv && w->n_rows >= 4096;
    if (w->k > 4096) return w->n_rows >= 4096 || (w->n_rows >= 2048 && (w->type == AXQ_Q8_0 || w->type == AXQ_Q4_0 || w->type == AXQ_Q4_K));
    const RowsPlan p = rows_plan(ctx, w, AXQ_ROWS_F32, rows);
    return slow_gemv || w->n_rows <= 4096 || p.tiles * p.splits * 5 >= ctx->prop.multiProcessorCount * 4;
}

// The kernels whose results leave row by row do, where a workgroup has all of K.
bool axq_dev_rows_gemm_makes_swiglu(const axq_ctx *ctx, const axq_weight *w, int rows) {
    if (!axq_dev_rows_gemm_covers(w, rows) || w->n_rows % 8 != 0) return false;
    const RowsPlan p = rows_plan(ctx, w, AXQ_ROWS_F32, rows);
    return p.splits == 1 && (p.wide || p.apart);
}

// Scratch: x in operand order | its sub-block sums | row scales | partial sums of a split K | the next call's first three.  Operands that a
// call before has left for this one lie behind that call's; partial sums then lie in front of them if they fit there.
struct RowsRoom {
    size_t xa, xs, rs, part;
    size_t operands() const { return xa + xs + rs; }
    size_t part_at(size_t at) const { return at && part <= at ? 0 : at + operands(); }
    size_t end(size_t at) const { // of a call whose operands lie at `at`
        const size_t p = part_at(at) + part, o = at + operands();
        return axq_align_up(p > o ? p : o, 256);
    }
};
static RowsRoom rows_room(const RowsPlan &p, int rows, const axq_weight *w) {
    RowsRoom r;
    const size_t mtiles = p.limbs ? (rows <= 16 ? 2 : rows <= 32 ? 3 : 4) : (size_t)(p.m + p.bm - 1) / p.bm * (p.bm / 32);
    r.xa = mtiles * 32 * (size_t)w->kp * 2;
    r.xs = mtiles * (size_t)(w->kp >> 8) * 2048;
    r.rs = axq_align_up((size_t)p.m * 4, 256);
    r.part = p.splits > 1 ? (size_t)p.splits * rows * (size_t)axq_part_pitch((int)w->n_rows) * 4 : 0;
    return r;
}

template <bool LIMBS>
static void launch_prep_sums(hipStream_t st, const PartSums &ps, const float *norm_w, float eps, int rows, int k, _Float16 *xa, _Float16 *xs, float *rs) {
    const unsigned grid = (unsigned)(rows + 63) / 64 * 64;
    if (k <= 4096) rows_prep_kernel<3, 1, LIMBS><<<grid, 512, 0, st>>>(nullptr, norm_w, eps, rows, k, k, xa, xs, rs, ps);
    else if (k <= 8192) rows_prep_kernel<3, 2, LIMBS><<<grid, 512, 0, st>>>(nullptr, norm_w, eps, rows, k, k, xa, xs, rs, ps);
    else rows_prep_kernel<3, 4, LIMBS><<<grid, 512, 0, st>>>(nullptr, norm_w, eps, rows, k, k, xa, xs, rs, ps);
}

// `chain`: the weight that takes y as f32 rows next, RMS-normalised where chain->norm_w is given.  Where K is split, its operands are made with the
// reduction, in one pass over the sums (64 rows of 4096, eight parts: 10.2 us in two launches, 6.8 in one), and chain->ready_at says where: the
// next call, of that weight and as many rows and with nothing in between, takes them.
int axq_dev_rows_gemm(axq_ctx *ctx, const axq_weight *w, const void *x, int in, int rows, const float *norm_w, float eps, const float *bias,
                      const float *resid, float *y, axq_rows_chain *chain) {
    const size_t at = chain && chain->ready_for == w ? chain->ready_at : 0;
    RowsPlan p = rows_plan(ctx, w, in, rows);
    RowsRoom room = rows_room(p, rows, w);
    if (w->n_rows % 4 != 0 && p.splits > 1 && axq_gemm_reserve(ctx, room.end(at)) != AXQ_OK) { // no room for parts of K: whole, as such calls always can
        (void)hipGetLastError();
        p = rows_plan(ctx, w, in, rows, true);
        room = rows_room(p, rows, w);
    }
    const bool limbs = p.limbs;
    const int m = p.m, n = (int)w->n_rows, k = (int)w->k, kp = (int)w->kp, splits = p.splits;
    const bool ready = at != 0;
    const axq_weight *next = chain ? chain->next : nullptr;
    if (chain) {
        chain->ready_for = nullptr;
        chain->sums = {};
    }
    size_t next_at = 0;
    RowsPlan np;
    RowsRoom nroom = {};
    if (next && splits > 1 && !bias && next->k == n && next->kp == n && next->k <= 16384 && axq_dev_rows_gemm_covers(next, rows)) {
        np = rows_plan(ctx, next, AXQ_ROWS_F32, rows);
        nroom = rows_room(np, rows, next);
        next_at = room.end(at);
        const size_t next_end = nroom.end(next_at);
        if (ready ? ctx->gemm_scratch_bytes < next_end : axq_gemm_reserve(ctx, next_end) != AXQ_OK) { // (this call's operands lie there)
            (void)hipGetLastError();
            next_at = 0; // no room: two launches need less
        }
    }
    if (int rc = axq_gemm_reserve(ctx, room.end(at))) return rc;
    RowsArgs a;
    a.sb_per_split = p.sb_per_split;
    uint8_t *base = reinterpret_cast<uint8_t *>(ctx->gemm_scratch);
    auto operands = [&](size_t from, const RowsRoom &r, _Float16 *&xa, _Float16 *&xs, float *&rs) {
        xa = reinterpret_cast<_Float16 *>(base + from);
        xs = reinterpret_cast<_Float16 *>(base + from + r.xa);
        rs = reinterpret_cast<float *>(base + from + r.xa + r.xs);
    };
    _Float16 *xa, *xs;
    float *rs;
    operands(at, room, xa, xs, rs);
    if (!ready) switch (in) {
    case AXQ_ROWS_BF16: launch_prep<2, false>(ctx->stream, x, nullptr, 0.f, rows, k, kp, xa, xs, rs); break;
    case AXQ_ROWS_SWIGLU:
        if (limbs) launch_prep<1, true>(ctx->stream, x, nullptr, 0.f, rows, k, kp, xa, xs, rs);
        else launch_prep<1, false>(ctx->stream, x, nullptr, 0.f, rows, k, kp, xa, xs, rs);
        break;
    default:
        if (limbs) launch_prep<0, true>(ctx->stream, x, norm_w, eps, rows, k, kp, xa, xs, rs);
        else launch_prep<0, false>(ctx->stream, x, norm_w, eps, rows, k, kp, xa, xs, rs);
        break;
    }
    a.codes = w->codes; a.meta = w->meta; a.qh = w->qh;
    a.codes_pitch = (uint32_t)w->codes_pitch; a.meta_pitch = (uint32_t)w->meta_pitch; a.qh_pitch = (uint32_t)w->qh_pitch;
    a.xa = xa; a.xs = xs; a.rowscale = rs; a.y = y;
    a.ypart = splits > 1 ? reinterpret_cast<float *>(base + room.part_at(at)) : nullptr;
    a.m = m; a.n = n; a.k = kp; a.pair = p.parts == 2; a.bias = bias; a.resid = resid;
    a.swiglu = chain && chain->swiglu;
    if (a.swiglu && (splits != 1 || !(p.wide || p.apart) || bias || resid || n % 8 != 0))
        return axq_fail(ctx, AXQ_ERR_INVALID_ARGUMENT, "axq_dev_rows_gemm: no SwiGLU of these results");
    int rc;
    switch (w->type) {
    case AXQ_Q4_K: rc = launch_rows<SuperQ45<false>>(ctx, a, p); break;
    case AXQ_Q5_K: rc = launch_rows<SuperQ45<true>>(ctx, a, p); break;
    case AXQ_Q6_K: rc = launch_rows<SuperQ6>(ctx, a, p); break;
    case AXQ_Q4_0: rc = launch_rows<Block32<4, false>>(ctx, a, p); break;
    case AXQ_Q4_1: rc = launch_rows<Block32<4, true>>(ctx, a, p); break;
    case AXQ_Q5_0: rc = launch_rows<Block32<5, false>>(ctx, a, p); break;
    case AXQ_Q5_1: rc = launch_rows<Block32<5, true>>(ctx, a, p); break;
    default: rc = launch_rows<Block32<8, false>>(ctx, a, p); break;
    }
    if (rc || splits == 1) return rc;
    if (chain && chain->leave_sums && !bias && !resid) {
        chain->sums.part = a.ypart;
        chain->sums.scale = rs;
        chain->sums.splits = splits;
        chain->sums.row_mul = p.parts;
        chain->sums.pitch = axq_part_pitch(n);
        chain->sums.stride = (size_t)rows * axq_part_pitch(n);
        return AXQ_OK;
    }
    if (next_at) {
        const PartSums ps = {a.ypart, rs, splits, p.parts, resid, y};
        _Float16 *nxa, *nxs;
        float *nrs;
        operands(next_at, nroom, nxa, nxs, nrs);
        if (np.limbs) launch_prep_sums<true>(ctx->stream, ps, chain->norm_w, eps, rows, n, nxa, nxs, nrs);
        else launch_prep_sums<false>(ctx->stream, ps, chain->norm_w, eps, rows, n, nxa, nxs, nrs);
        AXQ_LAUNCH_CHECK(ctx, "rows_prep_kernel");
        chain->ready_for = next;
        chain->ready_at = next_at;
        return AXQ_OK;
    }
    return axq_gemm_reduce(ctx, a.ypart, rs, rows, n, splits, 1.0f, p.parts, bias, resid, y);
}
