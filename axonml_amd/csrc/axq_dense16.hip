// Products with one f16 or bfloat16 weight as it is: the GEMM of bf16 rows and of f32 rows' addends, and a few f32 rows in 32-bit products.
#include <type_traits>

#include "axq_dense_tiles.h"

namespace {

// Few f32 rows, every weight read once: products of 32 bits on the matrix pipe (16 x 16 x 4).  Eight waves share 16 NT columns of 16 MT rows and take
// blocks of 32 of K in turn; lane (c, g) has the eight elements from 8 g on of a block, of weight row c and of rows c and c + 16 of x:
// product e of a block takes element e of every lane.  CHAIN products are added up by the matrix pipe, which cuts sums off instead of rounding them, the others by the
// vector unit (error, 10^-8, 6 rows of 1024: 12.6 with eight, 10.3 with four, 8.7 with one; one vector at a time it was 8.5 with f16 and 9.8 with bf16 weights).  The waves' sums meet in LDS.  blockIdx.y: a part of K, whose sums go to
// `part` (rows axq_part_pitch(n) apart).
template <bool HALF, int MT, int NT, int CHAIN>
__global__ void __launch_bounds__(512) dense_few_kernel(const uint16_t *w, int ldw, const float *x, int rows, int k, int n, int split_blocks, const float *bias, float *y, float *part) {
    constexpr int AHEAD = MT + NT == 2 ? 4 : MT + NT == 3 ? 3 : 2; // blocks under way
    extern __shared__ __attribute__((aligned(16))) float few_sums[];
    float (*sums)[MT * NT][64][4] = reinterpret_cast<float (*)[MT * NT][64][4]>(few_sums);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * (16 * NT), from = blockIdx.y * split_blocks, left = (k >> 5) - from;
    const int blocks = left < split_blocks ? left : split_blocks, mine = (blocks - wave + 7) >> 3;
    const float *px[MT];
    const uint16_t *pw[NT];
#pragma unroll
    for (int t = 0; t < MT; t++) px[t] = x + (size_t)(c + 16 * t < rows ? c + 16 * t : rows - 1) * k + (from + wave) * 32 + g * 8;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int row = n0 + t * 16 + c < n ? n0 + t * 16 + c : n - 1;
        pw[t] = w + (size_t)row * ldw + (from + wave) * 32 + g * 8;
    }
    f32x4 xa[AHEAD][MT][2], acc[MT][NT];
    u32x4 wa[AHEAD][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto request = [&](int b, int slot) {
        const size_t at = (size_t)(b < mine ? b : mine - 1) * 256;
#pragma unroll
        for (int t = 0; t < NT; t++) wa[slot][t] = *reinterpret_cast<const u32x4 *>(pw[t] + at);
#pragma unroll
        for (int t = 0; t < MT; t++) {
            xa[slot][t][0] = *reinterpret_cast<const f32x4 *>(px[t] + at);
            xa[slot][t][1] = *reinterpret_cast<const f32x4 *>(px[t] + at + 4);
        }
    };
    if (mine > 0) {
#pragma unroll
        for (int s = 0; s < AHEAD; s++) request(s, s);
        for (int b0 = 0; b0 < mine; b0 += AHEAD) {
#pragma unroll
            for (int s = 0; s < AHEAD; s++) {
                if (b0 + s < mine) {
                    constexpr int PARTS = 8 / CHAIN;
                    f32x4 part[MT][NT][PARTS];
#pragma unroll
                    for (int e = 0; e < 8; e++)
#pragma unroll
                        for (int t = 0; t < NT; t++) {
                            const uint32_t two = wa[s][t][e >> 1];
                            const float v = HALF ? (float)__builtin_bit_cast(_Float16, (unsigned short)(e & 1 ? two >> 16 : two & 0xFFFFu))
                                                 : (e & 1 ? axq_bf16_hi(two) : axq_bf16_lo(two));
#pragma unroll
                            for (int i = 0; i < MT; i++)
                                part[i][t][e % PARTS] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[s][i][e >> 2][e & 3], v, e < PARTS ? f32x4{0.f, 0.f, 0.f, 0.f} : part[i][t][e % PARTS], 0, 0, 0);
                        }
#pragma unroll
                    for (int i = 0; i < MT; i++)
#pragma unroll
                        for (int t = 0; t < NT; t++) {
#pragma unroll
                            for (int d = 1; d < PARTS; d <<= 1)
#pragma unroll
                                for (int q = 0; q < PARTS; q += 2 * d) part[i][t][q] += part[i][t][q + d];
                            acc[i][t] += part[i][t][0];
                        }
                }
                request(b0 + s + AHEAD, s);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int t = 0; t < NT; t++) *reinterpret_cast<f32x4 *>(&sums[wave][i * NT + t][lane][0]) = acc[i][t];
    __syncthreads();
    for (int i = tid; i < MT * NT * 256; i += 512) { // neighbouring threads: neighbouring columns of a row
        const int t = i >> 8, col = i & 15, row = i >> 4 & 15, at = n0 + t % NT * 16 + col, m = t / NT * 16 + row;
        float v[8];
#pragma unroll
        for (int s = 0; s < 8; s++) v[s] = sums[s][t][(row >> 2) * 16 + col][row & 3];
        const float sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        if (m >= rows || at >= n) continue;
        if (part) part[((size_t)blockIdx.y * rows + m) * axq_part_pitch(n) + at] = sum;
        else y[(size_t)m * n + at] = bias ? sum + bias[at] : sum;
    }
}

} // namespace

// Up to 16 rows always, up to 32 where the product with the rows' addends (axq_dense16_gemm) does not read its weight more cheaply.  us, vector by
// vector or through the two planes, with addends, and so:
//   2 to 16 rows   BF16 900 x 13312, 6: 62.0 - 12.5; 7184 x 3264, 7: 66.9 - 14.4; F16 720 x 832, 6: 16.4 - 4.7; 28000 x 4096, 16: 87.8 74.0 53.7
//   24 rows        F16 1024 x 11008: 39.3 19.9 17.3; 4096 x 2048: 16.8 14.1 12.0; 4096 x 4096: 22.3 17.2 20.6; 20000 x 4096: 88.4 67.7 79.6
//                  BF16 4096 x 11008: 39.0 49.8 36.4; 15901 x 4608, 30 rows: 95.4 68.5 54.5
bool axq_dense_few_pays(const axq_weight *w, const float *x, int rows) {
    if ((w->type != AXQ_BF16 && w->type != AXQ_F16) || w->k % 64 != 0 || w->k > INT32_MAX || w->n_rows > INT32_MAX || (reinterpret_cast<uintptr_t>(x) & 15) != 0) return false;
    return rows <= 16 || (rows <= 32 && (w->type == AXQ_BF16 || w->n_rows * w->k <= 12 << 20));
}

namespace {
template <bool HALF>
int launch_few(axq_ctx *ctx, const axq_weight *w, const float *x, int rows, const float *bias, float *y) {
    const uint16_t *codes = reinterpret_cast<const uint16_t *>(w->codes);
    const int ldw = (int)(w->codes_pitch / 2), n = (int)w->n_rows, k = (int)w->k, cus = ctx->prop.multiProcessorCount, blocks = k >> 5;
    // columns of a workgroup: more of them where there are workgroups enough, which read x as often as there are workgroups (us with 16, 32 and 64: 2 rows,
    // 28000 x 4096 51.0 56.7 70.5; 7 rows, 7184 x 3264 19.0 14.4 26.6; 16 rows, 28000 x 4096 89.0 72.3 53.7, 3776 x 2304 10.2 10.7 17.9; 24 rows, 4096 x
    // 4096 20.6 - 27.1, 4096 x 11008 46.2 - 37.4)
    const int nt = rows <= 4 || n < 16 * cus ? 1 : rows <= 8 ? 2 : rows <= 16 ? (n >= 64 * cus ? 4 : 2) : n >= 32 * cus || k >= 8192 ? 4 : 1;
    const int tiles = (n + 16 * nt - 1) / (16 * nt);
    int splits = cus / tiles;
    splits = splits > 8 ? 8 : splits;
    if (splits > blocks / 64) splits = blocks / 64;
    float *part = nullptr;
    if (splits > 1) { // parts of K where the GEMM's scratch may be used and has the room
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(ctx->stream, &status) != hipSuccess || status != hipStreamCaptureStatusNone ||
            axq_gemm_reserve(ctx, (size_t)splits * rows * axq_part_pitch(n) * 4) != AXQ_OK) {
            (void)hipGetLastError();
            splits = 1;
        } else {
            part = static_cast<float *>(ctx->gemm_scratch);
        }
    }
    const int each = splits > 1 ? (blocks + splits - 1) / splits : blocks;
    if (splits > 1) splits = (blocks + each - 1) / each;
    const dim3 grid(tiles, splits > 1 ? splits : 1);
    auto go = [&](auto mt, auto nc, auto ch) -> int {
        constexpr int MT = decltype(mt)::value, NT = decltype(nc)::value, CHAIN = decltype(ch)::value;
        static std::atomic<uint64_t> lds_allowed{0};
        constexpr size_t lds = (size_t)8 * MT * NT * 1024;
        if (lds > 48 * 1024)
            if (int rc = axq_allow_lds(ctx, reinterpret_cast<const void *>(dense_few_kernel<HALF, MT, NT, CHAIN>), lds_allowed, lds)) return rc;
        dense_few_kernel<HALF, MT, NT, CHAIN><<<grid, 512, lds, ctx->stream>>>(codes, ldw, x, rows, k, n, each, bias, y, part);
        return AXQ_OK;
    };
    using I1 = std::integral_constant<int, 1>; using I2 = std::integral_constant<int, 2>; using I4 = std::integral_constant<int, 4>;
    if (int rc = rows > 16 ? (nt == 4 ? go(I2{}, I4{}, I4{}) : go(I2{}, I1{}, I4{})) : rows > 8 ? (nt == 4 ? go(I1{}, I4{}, I4{}) : nt == 2 ? go(I1{}, I2{}, I4{}) : go(I1{}, I1{}, I4{}))
                           : nt == 2 ? go(I1{}, I2{}, I1{}) : go(I1{}, I1{}, I1{})) return rc;
    AXQ_LAUNCH_CHECK(ctx, "dense_few_kernel");
    return part ? axq_gemm_reduce(ctx, part, nullptr, rows, n, splits, 1.0f, 1, bias, nullptr, y) : AXQ_OK;
}
} // namespace

int axq_dense_few(axq_ctx *ctx, const axq_weight *w, const float *x, int rows, const float *bias, float *y) {
    return w->type == AXQ_F16 ? launch_few<true>(ctx, w, x, rows, bias, y) : launch_few<false>(ctx, w, x, rows, bias, y);
}

namespace {
// Tiles of a product with one 16-bit weight: as axq_dense_gemm, and 64 x 64 in parts of K of at least eight steps for two workgroups to a compute
// unit (one: F16 3674 x 4096, 187 rows 28.2 us, two 23.6; 336 x 4096, 1664 rows 33.3, 27.4; four: 25.9, 31.9).
enum { DENSE16_TURNS, DENSE16_SQUARE, DENSE16_SQUARE_TURNS, DENSE16_SMALL };
int dense16_tile(int cus, int n, int m, int k, int &splits) {
    const int wide = (m + 255) / 256 * ((n + 255) / 256), square = (m + 127) / 128 * ((n + 127) / 128), small = (m + 63) / 64 * ((n + 63) / 64);
    splits = 1;
    if (m > 128 && k >= 1536 && 3 * ((wide + cus - 1) / cus) < 2 * ((square + 2 * cus - 1) / (2 * cus))) return DENSE16_TURNS;
    if (m > 64 && square > cus) return DENSE16_SQUARE;
    if (m > 64 && square > cus / 2) return DENSE16_SQUARE_TURNS;
    if (small <= cus) {
        splits = 2 * cus / small;
        splits = splits < k / 512 ? splits : k / 512;
        splits = splits > 16 ? 16 : splits < 1 ? 1 : splits;
    }
    return DENSE16_SMALL;
}
template <bool HALF>
int dense16(axq_ctx *ctx, GemmArgs &g, const axq_dense16 &a, bool whole_k) {
    const int cus = ctx->prop.multiProcessorCount;
    int splits;
    switch (dense16_tile(cus, a.n, a.m, g.k, splits)) {
    case DENSE16_TURNS: count_tiles(g, 256, 256); return launch_turns<false, HALF>(ctx, g);
    case DENSE16_SQUARE: count_tiles(g, 128, 128); return launch_gemm<128, 128, 2, 2, 1, false, HALF, true>(ctx, g);
    case DENSE16_SQUARE_TURNS: count_tiles(g, 128, 128); return launch_turns<true, HALF, true>(ctx, g);
    default: break;
    }
    const int tiles = count_tiles(g, 64, 64);
    if (tiles > cus) return launch_gemm<64, 64, 2, 2, 1, false, HALF, true>(ctx, g);
    if (whole_k || splits == 1) return launch_gemm<64, 64, 2, 2, 2, false, HALF, true>(ctx, g);
    g.split_k = ((g.k >> 6) + splits - 1) / splits * 64;
    splits = (g.k + g.split_k - 1) / g.split_k;
    axq_part &p = g.parts.p[0];
    p.unscale = p.bias = p.resid = nullptr;
    p.y = a.part;
    p.ldy = axq_part_pitch(a.n);
    if (int rc = launch_gemm<64, 64, 2, 2, 2, false, HALF, true>(ctx, g, splits)) return rc;
    return axq_gemm_reduce(ctx, a.part, a.unscale, a.m, a.n, splits, 1.0f, 1, a.bias, a.resid, a.y);
}
} // namespace

size_t axq_dense16_room(axq_ctx *ctx, int n, int m, int k) {
    int splits;
    dense16_tile(ctx->prop.multiProcessorCount, n, m, k, splits);
    return splits > 1 ? (size_t)splits * m * axq_part_pitch(n) : 0;
}

int axq_dense16_gemm(axq_ctx *ctx, const axq_dense16 &a, bool whole_k) {
    GemmArgs g;
    g.parts = {};
    g.parts.n_parts = 1;
    axq_part &p = g.parts.p[0];
    p.w = reinterpret_cast<const uint16_t *>(a.w);
    p.ldw = a.ldw; p.n = a.n; p.x = a.x; p.y = a.y; p.ldy = a.n; p.unscale = a.unscale; p.bias = a.bias; p.resid = a.resid;
    g.m = a.m;
    g.wk = a.k;
    g.k = g.ldx = g.split_k = a.k * a.parts;
    return a.half ? dense16<true>(ctx, g, a, whole_k) : dense16<false>(ctx, g, a, whole_k);
}
