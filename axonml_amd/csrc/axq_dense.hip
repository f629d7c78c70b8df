// Products with bfloat16 weights: the GEMV of a decode step (input transforms, activations and residual adds ride in
// it) and the GEMM of many rows (bf16 rows on the matrix pipe, or f32 rows in true 32-bit), both over several weights
// per launch; and the row operations of a prompt around them.
#include <type_traits>

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

__device__ inline float tanh_norm(float x, float alpha, float w, float b) { return tanhf(alpha * x) * w + b; }

// ---------------------------------------------------------------------------------------------------------------------
// GEMV.  A workgroup (eight waves) stages f(x) in LDS once per distinct input and walks a contiguous range of row blocks
// (8 R rows, R per wave); a lane's step is 16 bytes (8 weights) of each of its R rows, U steps make an item.  The next
// item's weights are requested before the current one is worked on, the first one's before x is staged.  x lies in LDS
// as two planes, elements 8c .. 8c + 3 and 8c + 4 .. 8c + 7 of every chunk c, so that both 16-byte reads of a wave are
// free of bank conflicts.
// ---------------------------------------------------------------------------------------------------------------------
constexpr int GT = 512, GW = GT / 64; // threads and waves of a workgroup
struct GemvArgs {
    axq_parts parts;
    axq_in in;
    int steps; // of 512 elements
};

// Of a step of AXQ_IN_SEGMENTS: its weight's columns, their row pitch and 16-byte chunks; its inputs, their number and factor.
struct Step { const uint16_t *w; int ldw, c8; const float *x; float f; int k, glu; };

// Four inputs from e on, zeros past the end
__device__ inline f32x4 load_quad(const float *x, int e, int k) {
    if (e + 4 <= k) return *reinterpret_cast<const f32x4_any *>(x + e);
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    for (int i = 0; i < 4; i++)
        if (e + i < k) v[i] = x[e + i];
    return v;
}
__device__ inline f32x4 load_step(const Step &t, int e) {
    f32x4 v;
    if (t.glu) { // both halves are padded to whole groups
        const float *z = t.x + (e / AXQ_GLU_GROUP) * 2 * AXQ_GLU_GROUP + e % AXQ_GLU_GROUP;
        v = load_quad(z, 0, t.k - e) * load_quad(z + AXQ_GLU_GROUP, 0, t.k - e);
    } else {
        v = load_quad(t.x, e, t.k);
    }
    return v * t.f;
}

template <int MODE>
__device__ void stage_x(const GemvArgs &a, const axq_part &p, const Step *table, float *xs, float *scratch) {
    const axq_in &in = a.in;
    const float *mu = p.mu;
    const int k = in.k, tid = threadIdx.x, xl = a.steps * 512, half = xl >> 1, quads = xl >> 2;
    auto slot = [half](int e) { return ((e >> 3) << 2) + (e & 3) + ((e & 4) ? half : 0); };
    auto quad = [half, xs](int q) -> f32x4 & { return *reinterpret_cast<f32x4 *>(xs + ((q >> 1) << 2) + ((q & 1) ? half : 0)); };
    if (MODE == AXQ_IN_SEGMENTS) { // four loads under way per thread
        for (int q0 = tid; q0 < quads; q0 += 4 * GT) {
            f32x4 v[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int q = q0 + i * GT;
                if (q < quads) v[i] = load_step(table[q >> 7], (q & 127) << 2);
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (q0 + i * GT < quads) quad(q0 + i * GT) = v[i];
        }
    } else if (MODE == AXQ_IN_LAYER_NORM) {
        constexpr int NW = 2; // the first quads' weights are requested with the inputs
        f32x4 w[NW];
        float sum = 0.f, ss = 0.f;
#pragma unroll
        for (int i = 0; i < NW; i++)
            if (tid + i * GT < quads) w[i] = load_quad(p.nw, (tid + i * GT) << 2, k);
        for (int q = tid; q < quads; q += GT) {
            const f32x4 v = load_quad(in.x, q << 2, k);
            quad(q) = v;
            sum += (v[0] + v[1]) + (v[2] + v[3]);
        }
        const float mean = axq_block_sum(sum, scratch) / (float)k;
        for (int q = tid; q < quads; q += GT) {
            const f32x4 v = quad(q);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float d = (q << 2) + i < k ? v[i] - mean : 0.f;
                ss = fmaf(d, d, ss);
            }
        }
        const float inv = 1.0f / sqrtf(axq_block_sum(ss, scratch) / (float)k + in.eps);
#pragma unroll
        for (int i = 0; i < NW; i++)
            if (tid + i * GT < quads) quad(tid + i * GT) = (quad(tid + i * GT) - mean) * inv * w[i]; // zeros past the end
        for (int q = tid + NW * GT; q < quads; q += GT) quad(q) = (quad(q) - mean) * inv * load_quad(p.nw, q << 2, k);
    } else
    if (MODE == AXQ_IN_RMS_GATE) {
        float ss = 0.f;
        for (int e = tid; e < k; e += GT) {
            const float v = in.x[e];
            xs[slot(e)] = v;
            ss = fmaf(v, v, ss);
        }
        ss = axq_block_sum(ss, scratch);
        const float inv = 1.0f / sqrtf(ss / (float)k + in.eps);
        for (int e = tid; e < xl; e += GT) xs[slot(e)] = e < k ? xs[slot(e)] * inv * in.nw[e] * in.gate[e] : 0.f;
    } else if (MODE == AXQ_IN_POLY_NORM) {
        float s1 = 0.f, s2 = 0.f, s3 = 0.f;
        for (int e = tid; e < k; e += GT) {
            const float z = in.x[e], z2 = z * z, z3 = z2 * z;
            xs[slot(e)] = z;
            s1 += z2; s2 = fmaf(z2, z2, s2); s3 = fmaf(z3, z3, s3);
        }
        s1 = axq_block_sum(s1, scratch);
        s2 = axq_block_sum(s2, scratch);
        s3 = axq_block_sum(s3, scratch);
        const float c1 = in.coef[0] / sqrtf(s1 / (float)k + in.eps), c2 = in.coef[1] / sqrtf(s2 / (float)k + in.eps);
        const float c3 = in.coef[2] / sqrtf(s3 / (float)k + in.eps), c0 = in.coef[3];
        for (int e = tid; e < xl; e += GT) {
            const float z = e < k ? xs[slot(e)] : 0.f;
            xs[slot(e)] = e < k ? fmaf(fmaf(fmaf(c3, z, c2), z, c1), z, c0) : 0.f;
        }
    } else {
        const float alpha = MODE == AXQ_IN_PLAIN ? 0.f : in.alpha[0];
        const bool first = MODE == AXQ_IN_TANH_NORM_MIX && in.pos[0] == 0;
        for (int e = tid; e < xl; e += GT) {
            float v = 0.f;
            if (e < k) {
                v = in.x[e];
                if (MODE != AXQ_IN_PLAIN) v = tanh_norm(v, alpha, in.nw[e], in.nb[e]);
                if (MODE == AXQ_IN_TANH_NORM_MIX && mu) {
                    const float p = first ? 0.f : in.prev[e];
                    v = fmaf(p - v, mu[e], v);
                }
            }
            xs[slot(e)] = v;
        }
    }
    __syncthreads();
}

template <int MODE, int R>
__global__ void __launch_bounds__(GT, 4) dense_gemv_kernel(GemvArgs a) {
    extern __shared__ __attribute__((aligned(16))) float xs[];
    __shared__ float scratch[16];
    constexpr bool SEG = MODE == AXQ_IN_SEGMENTS;
    __shared__ Step table[SEG ? AXQ_DENSE_MAX_K / 512 : 1];
    constexpr int U = 8 / R;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nb = a.parts.n_blocks, b0 = (int)((long long)nb * blockIdx.x / gridDim.x), b1 = (int)((long long)nb * (blockIdx.x + 1) / gridDim.x);
    const int half = a.steps * 256, k8 = (a.in.k + 7) >> 3;
    auto part_of_block = [&](int b) {
        int pi = 0;
        while (pi + 1 < a.parts.n_parts && b >= a.parts.p[pi + 1].blk0) pi++;
        return pi;
    };
    if (SEG) {
        for (int t = tid; t < a.steps; t += GT) {
            int si = 0;
            while (si + 1 < a.in.n_seg && t >= a.in.seg[si + 1].step0) si++;
            const axq_seg &g = a.in.seg[si];
            const int i = (t - g.step0) / g.steps, s = (t - g.step0) - i * g.steps;
            table[t].w = g.w + (size_t)(g.sel ? g.sel[i] : i) * g.stride + (size_t)s * 512;
            table[t].ldw = g.ldw;
            table[t].c8 = ((g.k + 7) >> 3) - s * 64;
            table[t].x = g.x + (size_t)i * g.ldx + (size_t)s * (g.glu ? 1024 : 512);
            table[t].f = g.scale ? g.scale[i] : 1.0f;
            table[t].k = g.k - s * 512;
            table[t].glu = g.glu;
        }
        __syncthreads();
    }
    // chunks past a row's end: a valid chunk against zeros; rows past the end: the last row, dropped
    auto request = [&](int b, int s0, u32x4 (&q)[U][R]) {
        const axq_part &p = a.parts.p[part_of_block(b)];
        const int row0 = ((b - p.blk0) * GW + wave) * R;
#pragma unroll
        for (int r = 0; r < R; r++) {
            int row = row0 + r < p.n ? row0 + r : p.n - 1;
            if (SEG) {
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const Step &t = table[s0 + u < a.steps ? s0 + u : a.steps - 1];
                    const int c = lane < t.c8 ? lane : t.c8 - 1;
                    q[u][r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(t.w + (size_t)row * t.ldw + (size_t)c * 8));
                }
                continue;
            }
            if (MODE == AXQ_IN_LAYER_NORM && p.sel) {
                const int i = row / p.sel_rows;
                row += (p.sel[i] - i) * p.sel_rows;
            }
            const uint16_t *w = p.w + (size_t)row * p.ldw;
#pragma unroll
            for (int u = 0; u < U; u++) {
                int c = (s0 + u) * 64 + lane;
                c = c < k8 ? c : k8 - 1;
                q[u][r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(w + (size_t)c * 8));
            }
        }
    };
    u32x4 qa[U][R], qb[U][R];
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 0.f;
    int staged = -1;
    // one item: the products of block b from step s0 on, and at the row's end the results
    auto work = [&](int b, int s0, const u32x4 (&q)[U][R]) {
        const int pi = part_of_block(b);
        const axq_part &p = a.parts.p[pi];
        if (staged < 0 || (MODE == AXQ_IN_TANH_NORM_MIX && staged != pi) ||
            (MODE == AXQ_IN_LAYER_NORM && a.parts.p[staged].nw != p.nw)) { // the same for all waves
            if (staged >= 0) __syncthreads();
            stage_x<MODE>(a, p, table, xs, scratch);
            staged = pi;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (s0 + u < a.steps) {
                const int c = (s0 + u) * 64 + lane;
                const float4 xa = *reinterpret_cast<const float4 *>(xs + c * 4), xb = *reinterpret_cast<const float4 *>(xs + half + c * 4);
#pragma unroll
                for (int r = 0; r < R; r++) {
                    float t = acc[r];
                    t = fmaf(axq_bf16_lo(q[u][r][0]), xa.x, t); t = fmaf(axq_bf16_hi(q[u][r][0]), xa.y, t);
                    t = fmaf(axq_bf16_lo(q[u][r][1]), xa.z, t); t = fmaf(axq_bf16_hi(q[u][r][1]), xa.w, t);
                    t = fmaf(axq_bf16_lo(q[u][r][2]), xb.x, t); t = fmaf(axq_bf16_hi(q[u][r][2]), xb.y, t);
                    t = fmaf(axq_bf16_lo(q[u][r][3]), xb.z, t); t = fmaf(axq_bf16_hi(q[u][r][3]), xb.w, t);
                    acc[r] = t;
                }
            }
        }
        if (s0 + U >= a.steps) {
#pragma unroll
            for (int r = 0; r < R; r++) acc[r] = axq_wave_sum(acc[r]);
            float v = acc[0];
#pragma unroll
            for (int r = 1; r < R; r++) v = lane == r ? acc[r] : v;
            const int row = ((b - p.blk0) * GW + wave) * R + lane;
            if (lane < R && row < p.n) {
                if (p.bias) v += p.bias[row];
                v = p.act == AXQ_ACT_GLU_GELU ? ((row & AXQ_GLU_GROUP) ? v : axq_gelu_tanh(v)) : axq_act(p.act, v, a.parts.cap);
                if (p.resid) v += p.resid[row];
                reinterpret_cast<float *>(p.y)[row] = v;
                if (p.avg.out) p.avg.out[row] = axq_average(p.avg, row, v);
            }
#pragma unroll
            for (int r = 0; r < R; r++) acc[r] = 0.f;
        }
    };
    auto advance = [&](int &b, int &s0) {
        s0 += U;
        if (s0 >= a.steps) { s0 = 0; b++; }
    };
    int b = b0, s0 = 0;
    if (b >= b1) return;
    request(b, s0, qa);
    while (true) {
        int nb1 = b, ns1 = s0;
        advance(nb1, ns1);
        if (nb1 < b1) request(nb1, ns1, qb);
        work(b, s0, qa);
        if (nb1 >= b1) break;
        b = nb1; s0 = ns1;
        advance(b, s0);
        if (b < b1) request(b, s0, qa);
        work(nb1, ns1, qb);
        if (b >= b1) break;
    }
}

template <int MODE, int R>
int launch_gemv(axq_ctx *ctx, GemvArgs &a) {
    int nb = 0;
    for (int i = 0; i < a.parts.n_parts; i++) {
        a.parts.p[i].blk0 = nb;
        nb += (a.parts.p[i].n + GW * R - 1) / (GW * R);
    }
    a.parts.n_blocks = nb;
    const size_t lds = (size_t)a.steps * 512 * sizeof(float);
    const int most = (lds > 76 * 1024 ? 1 : 2) * ctx->prop.multiProcessorCount; // as many as are there at once
    static std::atomic<uint64_t> lds_allowed{0};
    int rc;
    if (lds > 48 * 1024 &&
        (rc = axq_allow_lds(ctx, reinterpret_cast<const void *>(&dense_gemv_kernel<MODE, R>), lds_allowed, (size_t)AXQ_DENSE_MAX_K * 4)))
        return rc;
    dense_gemv_kernel<MODE, R><<<nb < most ? nb : most, GT, lds, ctx->stream>>>(a);
    AXQ_LAUNCH_CHECK(ctx, "dense_gemv_kernel");
    return AXQ_OK;
}

template <int MODE>
int launch_gemv_mode(axq_ctx *ctx, GemvArgs &a) {
    long long rows = 0;
    for (int i = 0; i < a.parts.n_parts; i++) rows += a.parts.p[i].n;
    if (rows >= 8192) return launch_gemv<MODE, 2>(ctx, a);
    return launch_gemv<MODE, 1>(ctx, a);
}

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

// The same product with the two waves of a SIMD taking turns: while one multiplies, the other fetches the operands of its next
// products from LDS and requests what comes into LDS after them.  Waves 0 .. 3 are one half of the workgroup and 4 .. 7 the other, half a
// round apart, with a barrier behind every turn: a turn is sixteen products (0.26 us of the matrix pipe), the other half's reads hide
// behind it whole, and no wave has its reads, their latency and its products in one line.
// LDS is a ring of five units of 32 KB, filled four ahead: every request has three turns of each half (1.5 us) on its way.
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
    auto fetch = [&](int u, int at) { // unit u (past the end the last one again, which nobody multiplies) to element `at` of LDS
        u = u < units ? u : units - 1;
        const int wu = weight_step(u, a.wk / KU);
        uint16_t *to = lds + at + gw * 512;
#pragma unroll
        for (int i = 0; i < L; i++) __builtin_amdgcn_global_load_lds((gbl_void *)(ga[i] + (size_t)u * KU), (lds_void *)(to + i * LW * 512), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < L; i++) __builtin_amdgcn_global_load_lds((gbl_void *)(gb[i] + (size_t)wu * KU), (lds_void *)(to + UNIT / 2 + i * LW * 512), 16, 0, 0);
        asm volatile("" ::: "memory");
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
        // unit u + 4 takes the place of unit u - 1, which both halves have read; what the next turns read has come behind the barriers:
        // of a shared unit both halves' requests in front of the first half's turn
        fetch(u + 4, at == 0 ? (RING - 1) * UNIT : at - UNIT);
        if (it > 0) fold();
        if (SPLIT) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(12) lgkmcnt(0)" ::: "memory");
        barrier();
        if (!SPLIT || u < units) {
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < NT; j++) {
                        if constexpr (FOLD) part[i][j] = mma<HALF>(fa[ks][i], fb[ks][j], ks ? part[i][j] : zero);
                        else acc[i][j] = mma<HALF>(fa[ks][i], fb[ks][j], acc[i][j]);
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

// GEMM on f32 rows in true 32-bit: 64 x 64 tiles, 4 x 4 results per thread, K in steps of 16.
template <bool GROUPED>
__global__ void __launch_bounds__(256) dense_gemm_f32_kernel(GemmArgs a) {
    __shared__ __attribute__((aligned(16))) float as[16][68], bs[16][68];
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    int ct, m0, m1, pi = 0;
    size_t woff = 0;
    if (!find_tile<GROUPED>(a, 64, 64, ct, m0, m1, woff)) return;
    while (!GROUPED && pi + 1 < a.parts.n_parts && ct >= a.parts.p[pi + 1].blk0) pi++;
    const axq_part &p = a.parts.p[pi];
    const int n0 = (ct - p.blk0) * 64;
    const float *x = reinterpret_cast<const float *>(p.x);
    const int lr = tid >> 2, lc = (tid & 3) * 4; // this thread's four elements of a step: row lr, columns lc ..
    int row = m0 + lr < m1 ? m0 + lr : m1 - 1;
    if (GROUPED && a.g.src) row = a.g.src[row];
    const float *ga = x + (size_t)row * a.ldx + lc;
    const uint16_t *gb = p.w + woff + (size_t)(n0 + lr < p.n ? n0 + lr : p.n - 1) * p.ldw + lc;
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = 0.f;
    for (int k = 0; k < a.k; k += 16) {
        const float4 va = *reinterpret_cast<const float4 *>(ga + k);
        const uint2 vb = *reinterpret_cast<const uint2 *>(gb + k);
        __syncthreads();
        as[lc][lr] = va.x; as[lc + 1][lr] = va.y; as[lc + 2][lr] = va.z; as[lc + 3][lr] = va.w;
        bs[lc][lr] = axq_bf16_lo(vb.x); bs[lc + 1][lr] = axq_bf16_hi(vb.x); bs[lc + 2][lr] = axq_bf16_lo(vb.y); bs[lc + 3][lr] = axq_bf16_hi(vb.y);
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 16; kk++) {
            const float4 fa = *reinterpret_cast<const float4 *>(&as[kk][ty * 4]), fb = *reinterpret_cast<const float4 *>(&bs[kk][tx * 4]);
            const float av[4] = {fa.x, fa.y, fa.z, fa.w}, bv[4] = {fb.x, fb.y, fb.z, fb.w};
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = fmaf(av[i], bv[j], acc[i][j]);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int m = m0 + ty * 4 + i, n = n0 + tx * 4 + j;
            if (m < m1 && n < p.n) {
                const bool glu = p.act == AXQ_ACT_GLU_GELU;
                finish(p, a.parts.cap, m, n, glu && !(n & AXQ_GLU_GROUP) ? axq_gelu_tanh(acc[i][j]) : acc[i][j], glu);
                if (!GROUPED && p.avg.out) finish_mean(p, m, n);
            }
        }
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

// ---------------------------------------------------------------------------------------------------------------------
// Row operations of a prompt, one workgroup per row.
// ---------------------------------------------------------------------------------------------------------------------
__device__ inline void put(const axq_rows_out &o, size_t row, int e, float v) {
    if (o.f32) reinterpret_cast<float *>(o.x)[row * o.ldx + e] = v;
    else reinterpret_cast<uint16_t *>(o.x)[row * o.ldx + e] = axq_to_bf16(v);
}

__device__ inline void put_quad(const axq_rows_out &o, size_t row, int e, f32x4 v) { // e and rows: multiples of 4
    if (o.f32) *reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(o.x) + row * o.ldx + e) = v;
    else
        *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(o.x) + row * o.ldx + e) =
            make_uint2(axq_to_bf16(v[0]) | (uint32_t)axq_to_bf16(v[1]) << 16, axq_to_bf16(v[2]) | (uint32_t)axq_to_bf16(v[3]) << 16);
}

__global__ void __launch_bounds__(256) embed_pos_kernel(const uint16_t *emb16, const float *emb32, const float *pos_table, const int32_t *tok,
                                                        const int32_t *pos, int pos0, int width, float *h) {
    const int e = blockIdx.x * 256 + threadIdx.x, t = blockIdx.y;
    if (e >= width) return;
    const int p = pos ? pos[0] + t : pos0 + t;
    const size_t i = (size_t)tok[t] * width + e;
    const float v = emb32 ? emb32[i] : (float)__builtin_bit_cast(_Float16, emb16[i]);
    h[(size_t)t * width + e] = pos_table ? v + pos_table[(size_t)p * width + e] : v;
}

struct MixPtrs { const float *mu[AXQ_MAX_PARTS]; };

// These kernels are their rows' bytes, so they go 16 bytes of f32 and 8 of bf16 a lane at a time.  2047 rows, us, an element and four at a time: tanh norm
// of 2048 columns 16.4 and 12.3; poly norm of 7168, kept in registers between its sums and its results, 34.5 and 20.6; root mean square and gate of 2048
// columns 11.6 and 7.5, in groups of 64 18.7 and 7.5.
__global__ void __launch_bounds__(256) rows_tanh_norm_kernel(axq_in in, int m, int first, int n_mix, MixPtrs mix, axq_rows_out out) {
    const int t = blockIdx.x, k = in.k;
    const float alpha = in.alpha[0];
    const float *h = in.x + (size_t)(in.rows ? in.rows[t] : t) * k;
    for (int e = threadIdx.x * 4; e < out.ldx; e += 1024) { // past the end everything is zero
        const f32x4 nw = load_quad(in.nw, e, k), nb = load_quad(in.nb, e, k), x = load_quad(h, e, k);
        f32x4 n, p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; i++) n[i] = e + i < k ? tanh_norm(x[i], alpha, nw[i], nb[i]) : 0.f;
        if (n_mix == 0) {
            put_quad(out, t, e, n);
            continue;
        }
        if (t > 0) {
            const f32x4 y = load_quad(h - k, e, k);
#pragma unroll
            for (int i = 0; i < 4; i++) p[i] = e + i < k ? tanh_norm(y[i], alpha, nw[i], nb[i]) : 0.f;
        } else if (!first) {
            p = load_quad(in.prev, e, k);
        }
        for (int j = 0; j < n_mix; j++) {
            const f32x4 mu = load_quad(mix.mu[j], e, k);
            f32x4 v;
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = fmaf(p[i] - n[i], mu[i], n[i]);
            put_quad(out, (size_t)j * m + t, e, v);
        }
    }
}

__global__ void __launch_bounds__(256) store_prev_kernel(axq_in in, int m, float *prev) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e < in.k) prev[e] = tanh_norm(in.x[(size_t)(m - 1) * in.k + e], in.alpha[0], in.nw[e], in.nb[e]);
}

// one workgroup per row and group (the last group's workgroup zeroes the tail)
__global__ void __launch_bounds__(256) rows_rms_gate_kernel(axq_in in, int group, axq_rows_out out) {
    __shared__ float scratch[16];
    const int t = blockIdx.x, e0 = blockIdx.y * group;
    const float *x = in.x + (size_t)t * in.k, *g = in.gate + (size_t)t * in.k;
    float ss = 0.f;
    for (int e = e0 + threadIdx.x; e < e0 + group; e += blockDim.x) ss = fmaf(x[e], x[e], ss);
    ss = axq_block_sum(ss, scratch);
    const float inv = 1.0f / sqrtf(ss / (float)group + in.eps);
    for (int e = e0 + threadIdx.x; e < e0 + group; e += blockDim.x) put(out, t, e, x[e] * inv * in.nw[e] * g[e]);
    if (blockIdx.y == gridDim.y - 1)
        for (int e = in.k + threadIdx.x; e < out.ldx; e += blockDim.x) put(out, t, e, 0.f);
}

// The same for groups of 4, 8, .. 256 (a group in as many neighbouring lanes as it has quads) or, GROUP = 0, one group that is the row: one workgroup
// per row, which keeps up to 4096 elements of it.
template <bool WHOLE>
__global__ void __launch_bounds__(256) rows_rms_gate_quads_kernel(axq_in in, int group, axq_rows_out out) {
    __shared__ float scratch[16];
    constexpr int NR = 4;
    const int t = blockIdx.x, k = in.k, tid = threadIdx.x;
    const float *x = in.x + (size_t)t * k, *g = in.gate + (size_t)t * k;
    auto dot = [](f32x4 v) { return fmaf(v[0], v[0], v[1] * v[1]) + fmaf(v[2], v[2], v[3] * v[3]); };
    auto write = [&](int e, f32x4 v, float inv) {
        const f32x4 w = load_quad(in.nw, e, k), y = load_quad(g, e, k);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = e + i < k ? v[i] * inv * w[i] * y[i] : 0.f;
        put_quad(out, t, e, v);
    };
    if constexpr (WHOLE) {
        f32x4 r[NR];
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < NR; i++) {
            r[i] = load_quad(x, (tid + i * 256) * 4, k);
            ss += dot(r[i]);
        }
        for (int e = (NR * 256 + tid) * 4; e < k; e += 1024) ss += dot(load_quad(x, e, k));
        const float inv = 1.0f / sqrtf(axq_block_sum(ss, scratch) / (float)k + in.eps);
#pragma unroll
        for (int i = 0; i < NR; i++)
            if ((tid + i * 256) * 4 < out.ldx) write((tid + i * 256) * 4, r[i], inv);
        for (int e = (NR * 256 + tid) * 4; e < out.ldx; e += 1024) write(e, load_quad(x, e, k), inv);
    } else {
        for (int e0 = 0; e0 < out.ldx; e0 += 1024) { // all lanes of a group together
            const int e = e0 + tid * 4;
            const f32x4 v = load_quad(x, e, k);
            float ss = dot(v);
            for (int s = 1; s < group / 4; s <<= 1) ss += __shfl_xor(ss, s);
            if (e < out.ldx) write(e, v, 1.0f / sqrtf(ss / (float)group + in.eps));
        }
    }
}

__global__ void __launch_bounds__(256) rows_poly_norm_kernel(axq_in in, axq_rows_out out) {
    __shared__ float scratch[3][4];
    constexpr int NR = 8; // quads of a row that a thread keeps; wider rows are read again
    const int t = blockIdx.x, k = in.k, tid = threadIdx.x;
    const float *x = in.x + (size_t)t * k;
    float s[3] = {0.f, 0.f, 0.f};
    f32x4 r[NR];
    auto add = [&](f32x4 v) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float z = v[i], z2 = z * z, z3 = z2 * z;
            s[0] += z2; s[1] = fmaf(z2, z2, s[1]); s[2] = fmaf(z3, z3, s[2]);
        }
    };
#pragma unroll
    for (int i = 0; i < NR; i++) r[i] = load_quad(x, (tid + i * 256) * 4, k);
#pragma unroll
    for (int i = 0; i < NR; i++) add(r[i]);
    for (int e = (NR * 256 + tid) * 4; e < k; e += 1024) add(load_quad(x, e, k));
#pragma unroll
    for (int i = 0; i < 3; i++) {
        s[i] = axq_wave_sum(s[i]);
        if ((tid & 63) == 0) scratch[i][tid >> 6] = s[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 3; i++) s[i] = (scratch[i][0] + scratch[i][1]) + (scratch[i][2] + scratch[i][3]);
    const float c1 = in.coef[0] / sqrtf(s[0] / (float)k + in.eps), c2 = in.coef[1] / sqrtf(s[1] / (float)k + in.eps);
    const float c3 = in.coef[2] / sqrtf(s[2] / (float)k + in.eps), c0 = in.coef[3];
    auto write = [&](int e, f32x4 v) {
        if (e >= out.ldx) return;
        f32x4 y;
#pragma unroll
        for (int i = 0; i < 4; i++) y[i] = e + i < k ? fmaf(fmaf(fmaf(c3, v[i], c2), v[i], c1), v[i], c0) : 0.f;
        put_quad(out, t, e, y);
    };
#pragma unroll
    for (int i = 0; i < NR; i++) write((tid + i * 256) * 4, r[i]);
    for (int e = (NR * 256 + tid) * 4; e < out.ldx; e += 1024) write(e, load_quad(x, e, k));
}

__global__ void __launch_bounds__(256) rows_layer_norm_kernel(axq_in in, const float *nw1, axq_rows_out out1, const float *nw2, axq_rows_out out2) {
    __shared__ float scratch[16];
    constexpr int NR = 4; // quads of a row that a thread keeps; wider rows are read again
    const int t = blockIdx.x, k = in.k, tid = threadIdx.x, quads = out1.ldx >> 2;
    const float *x = in.x + (size_t)(in.rows ? in.rows[t] : t) * k;
    f32x4 r[NR];
    float sum = 0.f, ss = 0.f;
#pragma unroll
    for (int i = 0; i < NR; i++) {
        r[i] = tid + i * 256 < quads ? load_quad(x, (tid + i * 256) << 2, k) : f32x4{0.f, 0.f, 0.f, 0.f};
        sum += (r[i][0] + r[i][1]) + (r[i][2] + r[i][3]);
    }
    for (int e = NR * 1024 + tid; e < k; e += 256) sum += x[e];
    const float mean = axq_block_sum(sum, scratch) / (float)k;
#pragma unroll
    for (int i = 0; i < NR; i++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const float d = ((tid + i * 256) << 2) + c < k ? r[i][c] - mean : 0.f;
            ss = fmaf(d, d, ss);
        }
    for (int e = NR * 1024 + tid; e < k; e += 256) {
        const float d = x[e] - mean;
        ss = fmaf(d, d, ss);
    }
    const float inv = 1.0f / sqrtf(axq_block_sum(ss, scratch) / (float)k + in.eps);
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const int q = tid + i * 256;
        if (q >= quads) break;
        const f32x4 n = (r[i] - mean) * inv; // past the end the weights are zeros
        put_quad(out1, t, q << 2, n * load_quad(nw1, q << 2, k));
        if (nw2) put_quad(out2, t, q << 2, n * load_quad(nw2, q << 2, k));
    }
    for (int e = NR * 1024 + tid; e < out1.ldx; e += 256) {
        const float n = e < k ? (x[e] - mean) * inv : 0.f;
        put(out1, t, e, e < k ? n * nw1[e] : 0.f);
        if (nw2) put(out2, t, e, e < k ? n * nw2[e] : 0.f);
    }
}

__global__ void __launch_bounds__(256) rows_glu_kernel(const float *z, int ldz, int k, axq_rows_out out) {
    const float *row = z + (size_t)blockIdx.x * ldz;
    static_assert(AXQ_GLU_GROUP % 4 == 0, "a quad lies in one group");
    for (int e = threadIdx.x * 4; e < out.ldx; e += 1024) {
        const float *g = row + (e / AXQ_GLU_GROUP) * 2 * AXQ_GLU_GROUP + e % AXQ_GLU_GROUP - e; // g[e]
        put_quad(out, blockIdx.x, e, load_quad(g, e, k) * load_quad(g + AXQ_GLU_GROUP, e, k));
    }
}

__global__ void __launch_bounds__(64) rows_zero_tail_kernel(int k, axq_rows_out out) {
    for (int e = k + threadIdx.x; e < out.ldx; e += 64) put(out, blockIdx.x, e, 0.f);
}

} // namespace

int axq_dense_gemv(axq_ctx *ctx, int mode, const axq_in &in, axq_parts &parts) {
    if ((mode != AXQ_IN_SEGMENTS && (in.k < 1 || in.k > AXQ_DENSE_MAX_K)) || parts.n_parts < 1 || parts.n_parts > AXQ_MAX_PARTS)
        return axq_fail(ctx, AXQ_ERR_SHAPE_MISMATCH, "Shape mismatch: a decode product takes 1 to %d inputs and 1 to %d weights, got %d and %d",
                        AXQ_DENSE_MAX_K, AXQ_MAX_PARTS, in.k, parts.n_parts);
    GemvArgs a;
    a.parts = parts;
    a.in = in;
    a.steps = (in.k + 511) / 512;
    if (mode == AXQ_IN_SEGMENTS) {
        a.steps = 0;
        int items = 0;
        for (int i = 0; i < in.n_seg; i++) {
            axq_seg &g = a.in.seg[i];
            if (g.k < 1 || g.count < 1) return axq_fail(ctx, AXQ_ERR_SHAPE_MISMATCH, "Shape mismatch: segment %d of %d x %d elements", i, g.count, g.k);
            g.step0 = a.steps;
            g.steps = (g.k + 511) / 512;
            a.steps += g.count * g.steps;
            items += g.count;
        }
        if (in.n_seg < 1 || in.n_seg > AXQ_MAX_SEGS || items > AXQ_MAX_SEG_ITEMS || a.steps > AXQ_DENSE_MAX_K / 512 || parts.n_parts != 1)
            return axq_fail(ctx, AXQ_ERR_SHAPE_MISMATCH, "Shape mismatch: a decode product over %d steps of 512 (at most %d)", a.steps, AXQ_DENSE_MAX_K / 512);
    }
    switch (mode) {
    case AXQ_IN_PLAIN: return launch_gemv_mode<AXQ_IN_PLAIN>(ctx, a);
    case AXQ_IN_TANH_NORM: return launch_gemv_mode<AXQ_IN_TANH_NORM>(ctx, a);
    case AXQ_IN_TANH_NORM_MIX: return launch_gemv_mode<AXQ_IN_TANH_NORM_MIX>(ctx, a);
    case AXQ_IN_RMS_GATE: return launch_gemv_mode<AXQ_IN_RMS_GATE>(ctx, a);
    case AXQ_IN_POLY_NORM: return launch_gemv_mode<AXQ_IN_POLY_NORM>(ctx, a);
    case AXQ_IN_LAYER_NORM: return launch_gemv_mode<AXQ_IN_LAYER_NORM>(ctx, a);
    case AXQ_IN_SEGMENTS: return launch_gemv_mode<AXQ_IN_SEGMENTS>(ctx, a);
    default: return axq_fail(ctx, AXQ_ERR_INVALID_ARGUMENT, "axq_dense_gemv: unknown input mode %d", mode);
    }
}

int axq_dev_dense_gemv(axq_ctx *ctx, const axq_weight *w, const float *x, const float *bias, float *y) {
    axq_in in;
    in.x = x;
    in.k = (int)w->k;
    axq_parts parts = {};
    parts.n_parts = 1;
    parts.p[0].w = reinterpret_cast<const uint16_t *>(w->codes);
    parts.p[0].ldw = (int)(w->codes_pitch / 2);
    parts.p[0].n = (int)w->n_rows;
    parts.p[0].bias = bias;
    parts.p[0].y = y;
    return axq_dense_gemv(ctx, AXQ_IN_PLAIN, in, parts);
}

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

int axq_dense_gemm(axq_ctx *ctx, axq_parts &parts, int m, int k, int ldx, bool f32) {
    GemmArgs a;
    a.parts = parts;
    a.m = m;
    a.k = a.wk = a.split_k = (k + 63) / 64 * 64;
    a.ldx = ldx;
    if (m < 1 || k < 1 || ldx % 64 != 0 || ldx < a.k || parts.n_parts < 1 || parts.n_parts > AXQ_MAX_PARTS)
        return axq_fail(ctx, AXQ_ERR_SHAPE_MISMATCH, "Shape mismatch: %d rows of %d elements (%d apart), %d weights", m, k, ldx, parts.n_parts);
    for (int i = 0; i < parts.n_parts; i++)
        if (parts.p[i].ldw < a.k || parts.p[i].n < 1)
            return axq_fail(ctx, AXQ_ERR_SHAPE_MISMATCH, "Shape mismatch: weight %d has rows of %d elements, %d wanted", i, parts.p[i].ldw, a.k);
    bool glu = false;
    for (int i = 0; i < parts.n_parts; i++) glu |= parts.p[i].act == AXQ_ACT_GLU_GELU;
    if (f32) {
        count_tiles(a, 64, 64);
        dense_gemm_f32_kernel<false><<<a.tiles, 256, 0, ctx->stream>>>(a);
        AXQ_LAUNCH_CHECK(ctx, "dense_gemm_f32_kernel");
        return AXQ_OK;
    }
    // Cost of a launch in units of a 128 x 128 tile that has a compute unit to itself: two 128 x 128 workgroups share one, a 256 x 256
    // tile is four at 1.35 times the rate (2047 rows, K = 2048, 8192 columns: 98 against 130 us).  The 256 x 256 tiles get the widest weights, as many as is cheapest, the others a launch of their own: a few
    // columns more than whole rounds of the chip (a narrow projection beside wide ones) would cost a round of large tiles.  Not at short K,
    // where a large tile is mostly its start and its way out (prompts, us, with large tiles, then with all waves in step, and without: K = 1024, Gemosun,
    // 1200 and 2048 tokens 1100 1075, 1352 1334, Lakulix, 2048 1043 1038; K = 2048, Lakulix, 1200 and 2048 tokens 1400 1410, 1691 1748,
    // Gemosun, 2048 2377 2417).
    const int cus = ctx->prop.multiProcessorCount;
    auto square_cost = [&](int tiles) { return 2.0f * (float)((tiles + 2 * cus - 1) / (2 * cus)); };
    if (m > 128 && a.k >= 1536) {
        int order[AXQ_MAX_PARTS], n = parts.n_parts;
        for (int i = 0; i < n; i++) {
            int at = i;
            for (; at > 0 && parts.p[order[at - 1]].n < parts.p[i].n; at--) order[at] = order[at - 1];
            order[at] = i;
        }
        const int mt2 = (m + 255) / 256, mt1 = (m + 127) / 128;
        int square = 0, wide = 0, cut = 0;
        for (int i = 0; i < n; i++) square += mt1 * ((parts.p[i].n + 127) / 128);
        float best = square_cost(square);
        for (int i = 0, left = square; i < n; i++) {
            wide += mt2 * ((parts.p[order[i]].n + 255) / 256);
            left -= mt1 * ((parts.p[order[i]].n + 127) / 128);
            const float cost = 3.0f * (float)((wide + cus - 1) / cus) + (left ? 0.2f + square_cost(left) * (left > cus ? 1.0f : 0.5f) : 0.f);
            if (cost < best) {
                best = cost;
                cut = i + 1;
            }
        }
        if (cut > 0) {
            axq_parts rest = parts;
            a.parts.n_parts = rest.n_parts = 0;
            for (int i = 0; i < n; i++)
                if (i < cut) a.parts.p[a.parts.n_parts++] = parts.p[order[i]];
                else rest.p[rest.n_parts++] = parts.p[order[i]];
            count_tiles(a, 256, 256);
            if (int rc = launch_turns<false>(ctx, a)) return rc;
            if (!rest.n_parts) return AXQ_OK;
            a.parts = rest;
        }
    }
    if (m > 64) {
        const int square = count_tiles(a, 128, 128);
        if (square > cus) return launch_gemm<128, 128, 2, 2, 1, false>(ctx, a);
        if (square > cus / 2) return launch_turns<true>(ctx, a);
    }
    if (glu)
        return count_tiles(a, 64, 128) > cus ? launch_gemm<64, 128, 2, 2, 1, false>(ctx, a) : launch_gemm<64, 128, 2, 2, 2, false>(ctx, a);
    return count_tiles(a, 64, 64) > cus ? launch_gemm<64, 64, 2, 2, 1, false>(ctx, a) : launch_gemm<64, 64, 2, 2, 2, false>(ctx, a);
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

int axq_dense_gemm_rows_per_tile(int rows, int groups, bool f32) { return !f32 && rows >= 96 * groups ? 128 : 64; }

int axq_dense_gemm_grouped(axq_ctx *ctx, axq_part &part, const axq_groups &g, int k, int ldx, bool f32) {
    GemmArgs a;
    a.parts = {};
    a.parts.p[0] = part;
    a.parts.n_parts = 1;
    a.m = 0;
    a.k = a.wk = a.split_k = (k + 63) / 64 * 64;
    a.ldx = ldx;
    a.g = g;
    if (k < 1 || ldx % 64 != 0 || ldx < a.k || part.ldw < a.k || part.n < 1 || g.max_tiles < 1 || (g.bm != 64 && g.bm != 128))
        return axq_fail(ctx, AXQ_ERR_SHAPE_MISMATCH, "Shape mismatch: grouped rows of %d elements (%d apart) against rows of %d", k, ldx, part.ldw);
    const int bn = f32 ? 64 : (g.bm == 128 ? 128 : 64);
    a.mt = g.max_tiles;
    a.tiles = (part.n + bn - 1) / bn * a.mt;
    if (!f32) return g.bm == 128 ? launch_gemm<128, 128, 2, 2, 1, true>(ctx, a) : launch_gemm<64, 64, 2, 2, 1, true>(ctx, a);
    dense_gemm_f32_kernel<true><<<a.tiles, 256, 0, ctx->stream>>>(a);
    AXQ_LAUNCH_CHECK(ctx, "grouped dense_gemm_f32_kernel");
    return AXQ_OK;
}

int axq_rows_embed(axq_ctx *ctx, const uint16_t *emb16, const float *emb32, const float *pos_table, const int32_t *tok, const int32_t *pos,
                   int pos0, int m, int width, float *h) {
    embed_pos_kernel<<<dim3((width + 255) / 256, m), 256, 0, ctx->stream>>>(emb16, emb32, pos_table, tok, pos, pos0, width, h);
    AXQ_LAUNCH_CHECK(ctx, "embed_pos_kernel");
    return AXQ_OK;
}

int axq_rows_tanh_norm(axq_ctx *ctx, const axq_in &in, int m, bool first, int n_mix, const float *const *mu, axq_rows_out out) {
    MixPtrs mix = {};
    for (int i = 0; i < n_mix; i++) mix.mu[i] = mu[i];
    rows_tanh_norm_kernel<<<m, 256, 0, ctx->stream>>>(in, m, first ? 1 : 0, n_mix, mix, out);
    AXQ_LAUNCH_CHECK(ctx, "rows_tanh_norm_kernel");
    return AXQ_OK;
}

int axq_store_prev(axq_ctx *ctx, const axq_in &in, int m, float *prev) {
    store_prev_kernel<<<(in.k + 255) / 256, 256, 0, ctx->stream>>>(in, m, prev);
    AXQ_LAUNCH_CHECK(ctx, "store_prev_kernel");
    return AXQ_OK;
}

int axq_rows_rms_gate(axq_ctx *ctx, const axq_in &in, int m, int group, axq_rows_out out) {
    if (group <= 256 && group >= 4 && (group & (group - 1)) == 0) rows_rms_gate_quads_kernel<false><<<m, 256, 0, ctx->stream>>>(in, group, out);
    else if (group == in.k) rows_rms_gate_quads_kernel<true><<<m, 256, 0, ctx->stream>>>(in, group, out);
    else rows_rms_gate_kernel<<<dim3(m, in.k / group), group <= 128 ? 64 : 256, 0, ctx->stream>>>(in, group, out);
    AXQ_LAUNCH_CHECK(ctx, "rows_rms_gate_kernel");
    return AXQ_OK;
}

int axq_rows_poly_norm(axq_ctx *ctx, const axq_in &in, int m, axq_rows_out out) {
    rows_poly_norm_kernel<<<m, 256, 0, ctx->stream>>>(in, out);
    AXQ_LAUNCH_CHECK(ctx, "rows_poly_norm_kernel");
    return AXQ_OK;
}

int axq_rows_layer_norm(axq_ctx *ctx, const axq_in &in, int m, const float *nw1, axq_rows_out out1, const float *nw2, axq_rows_out out2) {
    if (out1.ldx % 4) return axq_fail(ctx, AXQ_ERR_SHAPE_MISMATCH, "Shape mismatch: layer norms of rows %d apart", out1.ldx);
    if (nw2 && out2.ldx != out1.ldx) return axq_fail(ctx, AXQ_ERR_SHAPE_MISMATCH, "Shape mismatch: layer norms of rows %d and %d apart", out1.ldx, out2.ldx);
    rows_layer_norm_kernel<<<m, 256, 0, ctx->stream>>>(in, nw1, out1, nw2, out2);
    AXQ_LAUNCH_CHECK(ctx, "rows_layer_norm_kernel");
    return AXQ_OK;
}

int axq_rows_glu(axq_ctx *ctx, const float *z, int ldz, int k, int m, axq_rows_out out) {
    rows_glu_kernel<<<m, 256, 0, ctx->stream>>>(z, ldz, k, out);
    AXQ_LAUNCH_CHECK(ctx, "rows_glu_kernel");
    return AXQ_OK;
}

int axq_rows_zero_tail(axq_ctx *ctx, int m, int k, axq_rows_out out) {
    if (k == out.ldx) return AXQ_OK;
    rows_zero_tail_kernel<<<m, 64, 0, ctx->stream>>>(k, out);
    AXQ_LAUNCH_CHECK(ctx, "rows_zero_tail_kernel");
    return AXQ_OK;
}
