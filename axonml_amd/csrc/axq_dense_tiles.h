// Products of rows and weights of 16 bits on the matrix pipe: the tiles, for bfloat16 products of several weights and of experts (axq_dense.hip) and for
// products of one 16-bit weight (axq_dense16.hip), each of which has its instances in a code object of its own: a program loads what it uses.
#pragma once
#include "axq_dense.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4))); // at any float's address
typedef const __attribute__((address_space(1))) void gbl_void;
typedef __attribute__((address_space(3))) void lds_void;

// ---------------------------------------------------------------------------------------------------------------------
// GEMM on bf16 rows: tiles of BM x BN, K in steps of 64, operands straight from memory into LDS (16 bytes per lane,
// two stages).  Row r of a tile is 128 bytes of LDS whose 16-byte pieces are exchanged by (r / 2) & 7 (the loads take the
// permuted source address, the destination being fixed): sixteen lanes that read the same piece of consecutive rows touch all
// 64 banks (exchanged by r & 7, rows r and r + 8 share theirs and every operand read takes twice as long).
// The product is taken as D[row of x][row of W]: a lane's accumulators are one output column.
// The barrier of a step stands in front of its last quarter of products: behind it the step after next is requested into the
// stage that has just been read, and the next step's first operands, which arrive while those products run.
// Tiles: 128 x 128 with four waves, two workgroups to a compute unit; smaller ones, with eight waves of which four take every other
// step (KG = 2) where there is no second workgroup.  256 x 256, and 128 x 128 without a second workgroup: dense_turns_kernel (2047 x 2048,
// K = 2048: 37.8 us in this one with KG = 2, 33.2 there).
struct GemmArgs {
    axq_parts parts;
    int m, k, ldx, mt, tiles;
    int wk;       // x holds k / wk addends one behind the other, which all meet the weight's wk columns
    int split_k;  // K of a workgroup: blockIdx.y's part of it, whose results lie m rows behind the last part's
    axq_groups g; // grouped form
};
// column of the weight that column kt (in steps) of x meets, kw steps of them
__device__ inline int weight_step(int kt, int kw) { return kt - (kt >= 2 * kw ? 2 * kw : kt >= kw ? kw : 0); }

template <bool HALF>
__device__ inline f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
    if constexpr (HALF) return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// A product's result on its way out (act_done: the activation has been applied)
__device__ inline void finish(const axq_part &p, float cap, int m, int n, float v, bool act_done = false) {
    if (p.unscale) v *= p.unscale[m];
    if (p.bias) v += p.bias[n];
    if (!act_done) v = axq_act(p.act, v, cap);
    if (p.scale) v *= p.scale[m];
    const size_t i = (size_t)m * p.ldy + n;
    if (p.resid) v += p.resid[i];
    if (p.out16) reinterpret_cast<uint16_t *>(p.y)[i] = axq_to_bf16(v);
    else reinterpret_cast<float *>(p.y)[i] = v;
}

// ... and, once a thread's results are written, the mean over the layers at one of them
__device__ inline void finish_mean(const axq_part &p, int m, int n) {
    const size_t i = (size_t)m * p.ldy + n;
    p.avg.out[i] = axq_average(p.avg, i, reinterpret_cast<const float *>(p.y)[i]);
}

__device__ inline int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// Tiles in an order that gives each XCD (workgroups go round them) a contiguous run; a run walks the row tiles of a
// column tile first, so that a weight tile is read by one XCD's L2.
__device__ inline int xcd_tile(int tiles) {
    const int b = blockIdx.x, per = tiles >> 3, rest = tiles & 7, x = b & 7;
    return x * per + (x < rest ? x : rest) + (b >> 3);
}

// The tile of a workgroup: column tile `ct`, rows m0 .. m1 - 1, and which weight; false: there is none.  A grouped product's runs walk the
// column tiles first, over as many row tiles as there are: a run is a few weights, each read by one XCD with the rows that go
// through it, where a column tile of every weight would bring all rows to every XCD.
template <bool GROUPED>
__device__ inline bool find_tile(const GemmArgs &a, int bm, int bn, int &ct, int &m0, int &m1, size_t &woff) {
    if (GROUPED) {
        const int cts = (a.parts.p[0].n + bn - 1) / bn, tiles = a.g.tiles[0] * cts;
        if ((int)blockIdx.x >= tiles) return false;
        const int tile = xcd_tile(tiles);
        const int32_t *e = a.g.tiles + 4 + 4 * (tile / cts);
        ct = tile % cts;
        woff = (size_t)e[0] * a.g.stride;
        m0 = e[1];
        m1 = e[2];
    } else {
        const int tile = xcd_tile(a.tiles);
        ct = tile / a.mt;
        m0 = (tile - ct * a.mt) * bm;
        m1 = a.m;
    }
    return true;
}

// A wave's results on their way out, 32 rows at a time through a patch of LDS of its own: a lane then has four neighbouring columns
// of a row (16-byte loads and stores), and bias, activation, residual and mean are a short loop.  (Straight from the accumulators,
// an element at a time with every option asked for each, this was most of the kernel at K = 2048: 100 of 144 us at 2047 x 8192.)
template <int MT, int NT, bool GROUPED>
__device__ inline void write_tile(const axq_part &p, float cap, const f32x16 (&acc)[MT][NT], float *patch, int m_base, int m1, int n_base, int lane) {
    constexpr int P = NT * 32 + 8; // row pitch: rows four apart lie half the banks apart
    const int li = lane & 31;
    const bool glu = NT == 2 && p.act == AXQ_ACT_GLU_GELU; // the wave's two column tiles are a group of gates and its ups
    const int cols = glu ? p.n / 2 : p.n, n_first = glu ? n_base / 2 : n_base, quads = glu ? 8 : NT * 8, rows_at_once = 64 / quads;
    const int row_l = lane / quads, quad = lane % quads, n = n_first + quad * 4;
    // four columns at once: bf16 results where they are aligned, f32 ones anywhere
    const bool vec = p.out16 ? ((p.ldy | cols) & 3) == 0 && (reinterpret_cast<uintptr_t>(p.y) & 7) == 0 : n + 4 <= cols;
    auto load4 = [&](const float *q) -> f32x4 {
        if (n + 4 <= cols) return *reinterpret_cast<const f32x4_any *>(q);
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        for (int e = 0; e < 4; e++)
            if (n + e < cols) v[e] = q[e];
        return v;
    };
    const f32x4 bias = p.bias && n < cols ? load4(p.bias + n) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < MT; i++) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the last rows have been read
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) patch[acc_row(r, lane) * P + j * 32 + li] = acc[i][j][r];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (p.act != AXQ_ACT_NONE) { // in place, in a loop of its own: sixteen elements' code in each of the loops below is too much of it
#pragma clang loop unroll(disable)
            for (int r = row_l; r < 32; r += rows_at_once) {
                f32x4 *at = reinterpret_cast<f32x4 *>(patch + r * P + quad * 4);
                f32x4 v = *at;
                if (glu) {
                    const f32x4 up = at[8];
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = axq_gelu_tanh(v[e]) * up[e];
                } else {
                    v += bias;
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = axq_act(p.act, v[e], cap);
                }
                *at = v;
            }
        }
#pragma clang loop unroll(disable)
        for (int r0 = 0; r0 < 32; r0 += 4 * rows_at_once) { // four rows of a lane at a time: their loads are under way together
            f32x4 v[4], o[4];
            bool ok[4];
            size_t at[4];
            int m[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int r = r0 + q * rows_at_once + row_l;
                m[q] = m_base + i * 32 + r;
                ok[q] = m[q] < m1 && n < cols;
                at[q] = (size_t)m[q] * p.ldy + n;
                if (p.resid && ok[q]) o[q] = load4(p.resid + at[q]);
                v[q] = *reinterpret_cast<const f32x4 *>(patch + r * P + quad * 4);
                if (p.unscale && ok[q]) v[q] *= p.unscale[m[q]];
                if (glu || p.act == AXQ_ACT_NONE) v[q] += bias;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                if (!ok[q]) continue;
                if (p.scale) v[q] *= p.scale[m[q]];
                if (p.resid) v[q] += o[q];
                if (vec && p.out16) {
                    *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(p.y) + at[q]) =
                        make_uint2(axq_to_bf16(v[q][0]) | (uint32_t)axq_to_bf16(v[q][1]) << 16, axq_to_bf16(v[q][2]) | (uint32_t)axq_to_bf16(v[q][3]) << 16);
                } else if (vec) {
                    *reinterpret_cast<f32x4_any *>(reinterpret_cast<float *>(p.y) + at[q]) = v[q];
                } else {
                    for (int e = 0; e < 4; e++)
                        if (n + e < cols) {
                            if (p.out16) reinterpret_cast<uint16_t *>(p.y)[at[q] + e] = axq_to_bf16(v[q][e]);
                            else reinterpret_cast<float *>(p.y)[at[q] + e] = v[q][e];
                        }
                }
            }
            if (!GROUPED && p.avg.out) { // the mean over the layers (axq_average's sum)
                f32x4 s[4];
#pragma unroll
                for (int q = 0; q < 4; q++) s[q] = f32x4{0.f, 0.f, 0.f, 0.f};
                for (int j = 0; j < p.avg.n; j++) {
                    const float w = p.avg.w[j];
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        if (ok[q]) o[q] = load4(p.avg.past + j * p.avg.stride + at[q]);
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        for (int e = 0; e < 4; e++) s[q][e] = fmaf(w, o[q][e], s[q][e]);
                }
                const float w = p.avg.w[p.avg.n];
#pragma unroll
                for (int q = 0; q < 4; q++)
                    for (int e = 0; e < 4; e++)
                        if (ok[q] && n + e < cols) p.avg.out[at[q] + e] = fmaf(w, v[q][e], s[q][e]);
            }
        }
    }
}

constexpr int gemm_patch(int mt, int nt, int kg) {
    const int rows = 32 * (nt * 32 + 8), mail = kg == 2 ? mt * nt * 16 * 64 : 0; // write_tile's rows; the other group's sums
    return rows > mail ? rows : mail;
}

// FOLD: a step's products start from zero and join the total by an addition that rounds, where the matrix pipe cuts its sums off: error of 300 bf16 rows times
// 4100 x 4096 39.6 10^-8 without, 15.4 with it (through the two planes, K in parts, 21.9).
template <int BM, int BN, int WM, int WN, int KG, bool GROUPED, bool HALF, bool FOLD>
__global__ void __launch_bounds__(64 * WM * WN * KG, 2) dense_gemm_kernel(GemmArgs a) {
    constexpr int MT = BM / 32 / WM, NT = BN / 32 / WN; // 32 x 32 tiles of a wave
    constexpr int GW = WM * WN;                         // waves of a group along K
    constexpr int AL = BM / 8 / GW, BL = BN / 8 / GW;   // 16-byte loads per thread and step
    constexpr int STEP = (BM + BN) * 64;                // elements of a step's tile
    constexpr int PATCH = gemm_patch(MT, NT, KG);       // floats of LDS that a wave's results pass through
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[]; // [stage][group][STEP]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kg = wave / GW, gw = wave % GW, wm = gw / WN, wn = gw % WN;
    int ct, m0, m1, pi = 0;
    size_t woff = 0;
    if (!find_tile<GROUPED>(a, BM, BN, ct, m0, m1, woff)) return;
    while (!GROUPED && pi + 1 < a.parts.n_parts && ct >= a.parts.p[pi + 1].blk0) pi++;
    const axq_part &p = a.parts.p[pi];
    const int n0 = (ct - p.blk0) * BN;
    const uint16_t *x = reinterpret_cast<const uint16_t *>(p.x);

    const uint16_t *ga[AL], *gb[BL];
#pragma unroll
    for (int i = 0; i < AL; i++) {
        const int idx = (i * GW + gw) * 64 + lane, r = idx >> 3, c = (idx & 7) ^ ((r >> 1) & 7);
        int row = m0 + r < m1 ? m0 + r : m1 - 1;
        if (GROUPED && a.g.src) row = a.g.src[row];
        ga[i] = x + (size_t)row * a.ldx + c * 8;
    }
#pragma unroll
    for (int i = 0; i < BL; i++) {
        const int idx = (i * GW + gw) * 64 + lane, r = idx >> 3, c = (idx & 7) ^ ((r >> 1) & 7);
        const int row = n0 + r < p.n ? n0 + r : p.n - 1;
        gb[i] = p.w + woff + (size_t)row * p.ldw + c * 8;
    }
    const int kt0 = GROUPED ? 0 : (int)blockIdx.y * (a.split_k >> 6), left = (a.k >> 6) - kt0;
    const int kts = GROUPED || left < (a.split_k >> 6) ? left : a.split_k >> 6, its = (kts + KG - 1) / KG;
    auto fetch = [&](int it) { // this group's step of iteration `it` (past the end the last one again, which nobody multiplies)
        int kt = it * KG + kg;
        kt = kt0 + (kt < kts ? kt : kts - 1);
        const int wt = GROUPED ? kt : weight_step(kt, a.wk >> 6);
        uint16_t *la = lds + ((it & 1) * KG + kg) * STEP, *lb = la + BM * 64;
#pragma unroll
        for (int i = 0; i < AL; i++)
            __builtin_amdgcn_global_load_lds((gbl_void *)(ga[i] + (size_t)kt * 64), (lds_void *)(la + (i * GW + gw) * 512), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < BL; i++)
            __builtin_amdgcn_global_load_lds((gbl_void *)(gb[i] + (size_t)wt * 64), (lds_void *)(lb + (i * GW + gw) * 512), 16, 0, 0);
        asm volatile("" ::: "memory");
    };
    f32x16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    const int li = lane & 31, lh = lane >> 5, sw = (li >> 1) & 7; // tiles of a wave start at multiples of 32 rows
    const uint16_t *la = lds + kg * STEP + (wm * (BM / WM) + li) * 64, *lb = lds + kg * STEP + (BM + wn * (BN / WN) + li) * 64;
    u32x4 fa[2][MT], fb[2][NT];
    auto read = [&](int it, int ks, int b) {
        const int at = (it & 1) * KG * STEP + (((ks * 2 + lh) ^ sw) << 3);
#pragma unroll
        for (int i = 0; i < MT; i++) fa[b][i] = *reinterpret_cast<const u32x4 *>(la + at + i * 32 * 64);
#pragma unroll
        for (int j = 0; j < NT; j++) fb[b][j] = *reinterpret_cast<const u32x4 *>(lb + at + j * 32 * 64);
    };
    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    f32x16 part[FOLD ? MT : 1][FOLD ? NT : 1];
    auto meet = [&] { // what this wave has requested is in LDS and what it has read has arrived; then everybody's
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    fetch(0);
    meet();
    if (its > 1) fetch(1);
    read(0, 0, 0);
    for (int it = 0; it < its; it++) {
        const bool live = KG == 1 || it * KG + kg < kts;
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            if (ks < 3) {
                read(it, ks + 1, (ks + 1) & 1);
            } else if (it + 1 < its) {
                meet();
                if (it + 2 < its) fetch(it + 2);
                read(it + 1, 0, 0);
            }
            if (live)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < NT; j++) {
                        if constexpr (FOLD) part[i][j] = mma<HALF>(fa[ks & 1][i], fb[ks & 1][j], ks ? part[i][j] : zero);
                        else acc[i][j] = mma<HALF>(fa[ks & 1][i], fb[ks & 1][j], acc[i][j]);
                    }
        }
        if constexpr (FOLD)
            if (live)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < NT; j++) acc[i][j] += part[i][j];
    }
    if constexpr (KG == 2) { // the second group's sums join the first one's, which finishes
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        float *mail = reinterpret_cast<float *>(lds) + gw * PATCH + lane;
        if (kg == 1)
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) mail[((i * NT + j) * 16 + r) * 64] = acc[i][j][r];
        __syncthreads();
        if (kg == 1) return;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] += mail[((i * NT + j) * 16 + r) * 64];
    }
    else {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the stages have been read: they take the results' patches
        __builtin_amdgcn_s_barrier();
    }
    float *patch = reinterpret_cast<float *>(lds) + gw * PATCH; // a wave's own: it has read its mail
    const int below = GROUPED ? 0 : (int)blockIdx.y * a.m;
    write_tile<MT, NT, GROUPED>(p, a.parts.cap, acc, patch, below + m0 + wm * (BM / WM), below + m1, n0 + wn * (BN / WN), lane);
}

// The same product with the two waves of a SIMD taking turns: while one multiplies, and between its products requests what comes into LDS
// after them (a request keeps its wave for 40 to 50 cycles, the matrix pipe works on; among the reads, before and so, us: BF16 2048 bf16 rows x
// 14336 x 4096 250 240, 2047 x 2048 x 2048 30.5 27.6, 2047 x 8192 x 2048 75 74, F16 1278 x 7520 x 1856 65 61.6), the other reads the operands of
// its next products from LDS.  Waves 0 .. 3 are one half of the workgroup and 4 .. 7 the other, half a
// round apart, with a barrier behind every turn: a turn is sixteen products (0.26 us of the matrix pipe), the other half's reads hide
// behind it whole, and no wave has its reads, their latency and its products in one line.
// LDS is a ring of five units of 32 KB, filled four ahead: every request has two and a half turns of each half (1.3 us) on its way.
//   SPLIT = false: 256 x 256 outputs, a unit is 32 of K, which both halves (128 x 64 per wave) read.
//   SPLIT = true: 128 x 128 outputs, a unit is 64 of K; the halves take every other one, and their sums meet in LDS.
// A row of a unit is 64 or 128 bytes whose 16-byte pieces are exchanged so that sixteen consecutive rows' reads touch all banks.
// FOLD (SPLIT only): as in dense_gemm_kernel; a turn's sum joins the total in the next fetch, beside the other half's products.
template <bool SPLIT, bool HALF, bool FOLD>
__global__ void __launch_bounds__(512, 2) dense_turns_kernel(GemmArgs a) {
    constexpr int BM = SPLIT ? 128 : 256, WM = 2, WN = SPLIT ? 2 : 4, MT = BM / 32 / WM, NT = 2;
    constexpr int KU = SPLIT ? 64 : 32, KS = KU / 16, PIECES = KU / 8, ROWS = 64 / PIECES; // rows of a load of a wave
    constexpr int LW = SPLIT ? 4 : 8, L = BM / ROWS / LW;                                  // waves that load a unit, their loads per operand
    constexpr int UNIT = 16384, RING = 5;                                                  // elements: x, then W
    constexpr int PATCH = gemm_patch(MT, NT, SPLIT ? 2 : 1);
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = wave >> 2, gw = SPLIT ? wave & 3 : wave, wm = gw / WN, wn = gw % WN;
    const int tile = xcd_tile(a.tiles), ct = tile / a.mt;
    const int m0 = (tile - ct * a.mt) * BM, m1 = a.m;
    int pi = 0;
    while (pi + 1 < a.parts.n_parts && ct >= a.parts.p[pi + 1].blk0) pi++;
    const axq_part &p = a.parts.p[pi];
    const int n0 = (ct - p.blk0) * BM;
    const uint16_t *x = reinterpret_cast<const uint16_t *>(p.x);
    auto exchanged = [](int row) { return SPLIT ? (row >> 1) & 7 : (row >> 2) & 3; };

    const uint16_t *ga[L], *gb[L];
#pragma unroll
    for (int i = 0; i < L; i++) {
        const int r = (i * LW + gw) * ROWS + lane / PIECES, c = (lane % PIECES) ^ exchanged(r);
        int row = m0 + r < m1 ? m0 + r : m1 - 1;
        ga[i] = x + (size_t)row * a.ldx + c * 8;
        row = n0 + r < p.n ? n0 + r : p.n - 1;
        gb[i] = p.w + (size_t)row * p.ldw + c * 8;
    }
    const int units = a.k / KU, its = SPLIT ? (units + 1) / 2 : units;
    auto request = [&](int u, int at, int piece) { // of unit u (past the end the last one again, which nobody multiplies) to element `at` of LDS
        u = u < units ? u : units - 1;
        const int wu = weight_step(u, a.wk / KU), i = piece % L;
        uint16_t *to = lds + at + gw * 512 + i * LW * 512;
        if (piece < L) __builtin_amdgcn_global_load_lds((gbl_void *)(ga[i] + (size_t)u * KU), (lds_void *)to, 16, 0, 0);
        else __builtin_amdgcn_global_load_lds((gbl_void *)(gb[i] + (size_t)wu * KU), (lds_void *)(to + UNIT / 2), 16, 0, 0);
        asm volatile("" ::: "memory");
    };
    auto fetch = [&](int u, int at) {
#pragma unroll
        for (int q = 0; q < 2 * L; q++) request(u, at, q);
    };
    auto barrier = [] {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    f32x16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    const int li = lane & 31, lh = lane >> 5, sw = exchanged(li); // tiles of a wave start at multiples of 32 rows
    const uint16_t *la = lds + (wm * (BM / WM) + li) * KU, *lb = lds + UNIT / 2 + (wn * 64 + li) * KU;
    // first units, and the wait for the first of them
    if (SPLIT) {
        fetch(half, half * UNIT);
        fetch(half + 2, (half + 2) * UNIT);
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    } else {
#pragma unroll
        for (int u = 0; u < 4; u++) fetch(u, u * UNIT);
        asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
    }
    barrier();
    if (half) barrier(); // the second half is a turn behind
    int at = SPLIT ? half * UNIT : 0; // of the unit that is read next
    static_assert(SPLIT || !FOLD, "no registers for a second sum");
    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    f32x16 part[FOLD ? MT : 1][FOLD ? NT : 1];
    auto fold = [&] {
        if constexpr (FOLD)
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    acc[i][j] += part[i][j];
                    asm volatile("" : "+v"(acc[i][j])); // here, not behind the wait
                }
    };
    for (int it = 0; it < its; it++) {
        const int u = SPLIT ? 2 * it + half : it;
        u32x4 fa[KS][MT], fb[KS][NT];
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c = at + (((ks * 2 + lh) ^ sw) << 3);
#pragma unroll
            for (int j = 0; j < NT; j++) fb[ks][j] = *reinterpret_cast<const u32x4 *>(lb + c + j * 32 * KU);
#pragma unroll
            for (int i = 0; i < MT; i++) fa[ks][i] = *reinterpret_cast<const u32x4 *>(la + c + i * 32 * KU);
        }
        asm volatile("" ::: "memory");
        if (it > 0) fold();
        // what the next turns read has come behind the barriers: of a shared unit both halves' requests in front of the first half's turn
        if (SPLIT) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
        barrier();
        if (!SPLIT || u < units) {
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
#pragma unroll
                for (int i = 0; i < MT; i++) {
#pragma unroll
                    for (int j = 0; j < NT; j++) {
                        if constexpr (FOLD) part[i][j] = mma<HALF>(fa[ks][i], fb[ks][j], ks ? part[i][j] : zero);
                        else acc[i][j] = mma<HALF>(fa[ks][i], fb[ks][j], acc[i][j]);
                    }
                    // unit u + 4 takes the place of unit u - 1, which both halves have read; a piece of it behind every pair of products, or every other
                    __builtin_amdgcn_sched_barrier(0);
                    const int slot = ks * MT + i, every = KS * MT / (2 * L);
                    if (slot % every == 0) request(u + 4, at == 0 ? (RING - 1) * UNIT : at - UNIT, slot / every);
                    __builtin_amdgcn_sched_barrier(0);
                }
            __builtin_amdgcn_s_setprio(0);
        }
        if (SPLIT) {
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        }
        barrier();
        const int next = at + (SPLIT ? 2 : 1) * UNIT;
        at = next >= RING * UNIT ? next - RING * UNIT : next;
    }
    if (2 * (its - 1) + half < units) fold(); // else the last turn had no products, and the one before has been added
    if (!half) barrier();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // nothing is on its way into LDS any more
    barrier();
    if constexpr (SPLIT) { // the second half's sums join the first one's, which finishes
        float *mail = reinterpret_cast<float *>(lds) + gw * PATCH + lane;
        if (half)
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) mail[((i * NT + j) * 16 + r) * 64] = acc[i][j][r];
        __syncthreads();
        if (half) return;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] += mail[((i * NT + j) * 16 + r) * 64];
    }
    float *patch = reinterpret_cast<float *>(lds) + gw * PATCH; // a wave's own: it has read its mail
    write_tile<MT, NT, false>(p, a.parts.cap, acc, patch, m0 + wm * (BM / WM), m1, n0 + wn * 64, lane);
}

template <int BM, int BN, int WM, int WN, int KG, bool GROUPED, bool HALF = false, bool FOLD = false>
int launch_gemm(axq_ctx *ctx, const GemmArgs &a, int splits = 1) {
    static std::atomic<uint64_t> lds_allowed{0};
    constexpr size_t stages = (size_t)2 * KG * (BM + BN) * 64 * 2, out = (size_t)WM * WN * gemm_patch(BM / 32 / WM, BN / 32 / WN, KG) * 4, lds = stages > out ? stages : out;
    if (lds > 48 * 1024)
        if (int rc = axq_allow_lds(ctx, reinterpret_cast<const void *>(dense_gemm_kernel<BM, BN, WM, WN, KG, GROUPED, HALF, FOLD>), lds_allowed, lds)) return rc;
    dense_gemm_kernel<BM, BN, WM, WN, KG, GROUPED, HALF, FOLD><<<dim3(a.tiles, splits), 64 * WM * WN * KG, lds, ctx->stream>>>(a);
    AXQ_LAUNCH_CHECK(ctx, "dense_gemm_kernel");
    return AXQ_OK;
}

template <bool SPLIT, bool HALF = false, bool FOLD = false>
int launch_turns(axq_ctx *ctx, const GemmArgs &a) {
    static std::atomic<uint64_t> lds_allowed{0};
    constexpr size_t lds = 160 * 1024;
    if (int rc = axq_allow_lds(ctx, reinterpret_cast<const void *>(dense_turns_kernel<SPLIT, HALF, FOLD>), lds_allowed, lds)) return rc;
    dense_turns_kernel<SPLIT, HALF, FOLD><<<a.tiles, 512, lds, ctx->stream>>>(a);
    AXQ_LAUNCH_CHECK(ctx, "dense_turns_kernel");
    return AXQ_OK;
}

int count_tiles(GemmArgs &a, int bm, int bn) {
    int ct = 0;
    for (int i = 0; i < a.parts.n_parts; i++) {
        a.parts.p[i].blk0 = ct;
        ct += (a.parts.p[i].n + bn - 1) / bn;
    }
    a.parts.n_blocks = ct;
    a.mt = (a.m + bm - 1) / bm;
    return a.tiles = ct * a.mt;
}

} // namespace
