// Prefill-path quantized matmul: y[M, N] = x[M, K] (bf16) * W[N, K]^T, f32 accumulate and output.  Superblock types
// (Q4_K, Q5_K, Q6_K) have a kernel of their own (axq_gemm_rows.hip).
//
// The reference composition is dequantize_tensor -> f32 sgemm (crates/axonml-quant/src/dequantize.rs:34-54,
// crates/axonml-core/src/backends/cpu.rs:566-598).  Here the packed weights are read once per M tile,
// dequantised in registers into LDS tiles and multiplied on the matrix pipe (v_mfma_f32_32x32x16_f16).
//
// Numerics: results must agree with the f32 reference to 1e-3 per element even where the output is
// small, which plain f16 weights (11 bits) do not give.  So
//   - a dequantised weight w (f32, rounded exactly as the reference rounds it) is split into two f16
//     values w = wh + wl (22 bits), and both halves are multiplied: two MFMAs per tile and K step;
//   - x comes in bf16 (8 significant bits) and is converted to f16 exactly: a small pre-pass scales
//     every row by a power of two so that its largest magnitude sits below 2^15, which keeps every
//     element that matters inside f16's normal range; the row scale is undone on the output.
// Accumulation is f32 inside the MFMA, in K order.
//
// Tiling: a workgroup computes BM x 128 outputs (BM = 128 or 256); K advances 64 at a time through two LDS
// stages, each holding the x tile and the two weight tiles.  Half of the waves multiply, the other half
// feed (see gemm_kernel).
#include <hip/hip_fp16.h>

#include <stdlib.h>

#include <type_traits>

#include "axq_internal.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4))); // a 16-byte register quad (arrays of HIP's uint4 struct end up in scratch)

constexpr int BN = 128;  // output columns (weight rows) per workgroup
constexpr int BK = 64;   // K per stage
constexpr int LDK = 72;  // LDS row length in halfs (64 + 8 padding against bank conflicts)

struct GemmArgs {
    const uint8_t *codes, *meta, *qh;
    size_t codes_pitch, meta_pitch, qh_pitch;
    const _Float16 *xh;    // [M, K] row-scaled f16
    const float *rowscale; // [M]
    float *y;              // [M, N]
    float *ypart;          // split K: [splits, M, N] unscaled partial sums (NULL when one workgroup covers all of K)
    int m, n, k;
    int steps_per_split;   // K steps per workgroup (grid.y of them cover K)
    // pair mode (f32 activations): rows 2t and 2t + 1 of xh are the two f16 parts of activation row t, and their results
    // are added into output row t (+ bias[n] + resid[t, n]); y, ypart and resid then have m / 2 rows
    int pair;
    const float *bias, *resid;
    int wm;                // 1: 128-row tiles, 2: 256-row tiles
    // gemm_blk32_kernel only: the rows' block sums as f16 pairs, per superblock [hi | hi | lo | zeros]
    const _Float16 *xs3;
    int xs3_pitch;         // halfs per xs3 row
};

__device__ inline float h2f(uint32_t bits) { return __half2float(__ushort_as_half((unsigned short)bits)); }
template <int B>
__device__ inline float ubyte(uint32_t v) { // byte B of v as a float, one instruction
    float r;
    if (B == 0) asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(r) : "v"(v));
    else if (B == 1) asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(r) : "v"(v));
    else if (B == 2) asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(r) : "v"(v));
    else asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// Weights go through the matrix pipe as WSCALE * w = wh + wl with wh, wl in f16: the power-of-two factor
// keeps the low part of ordinary weights (|w| > 5e-4) out of f16's subnormal range; the epilogue divides
// it out again.  A trait names its factor WS, and says PRESCALED when its convert step applies it already.
constexpr float WSCALE = 256.0f;

// ---------------------------------------------------------------------------
// Dequantisation units.  A unit is 16 weights of one weight row inside the current 64-wide K step:
// two runs of 8 consecutive k (k0.., k1..).  unit index u4 = 0..3 per row.  Each trait reproduces the
// element formula of crates/axonml-quant/src/dequantize.rs (Q8_0 :89-92, Q4_0 :116-121, Q4_1 :145-151)
// or of the GGUF spec (Q5_0, Q5_1), rounding as the f32 reference does (multiply, then add).
// ---------------------------------------------------------------------------
template <bool WITH_MIN>
struct GQ4x { // reference nibble order: byte i = elements 2i (low), 2i+1 (high)
    static constexpr bool PRESCALED = true;
    static constexpr float WS = WSCALE;
    struct Raw { uint2 q; uint32_t m; };
    __device__ static void load16(const GemmArgs &a, size_t row, int kstep, int u4, Raw &r) {
        const int blk = kstep * 2 + (u4 >> 1), part = u4 & 1;
        r.q = *reinterpret_cast<const uint2 *>(a.codes + row * a.codes_pitch + (size_t)blk * 16 + part * 8);
        const uint8_t *mp = a.meta + row * a.meta_pitch;
        r.m = WITH_MIN ? *reinterpret_cast<const uint32_t *>(mp + (size_t)blk * 4)
                       : (uint32_t) * reinterpret_cast<const uint16_t *>(mp + (size_t)blk * 2);
    }
    __device__ static void cvt16(const Raw &r, int, int u4, float (&w)[16], int &k0, int &k1) {
        const int part = u4 & 1;
        // (nib - 8) * d = nib * d - 8 d exactly; with a minimum one rounding (fma) where the f32 reference has two: far
        // below what f16 pairs resolve.  Four codes per mask, one conversion per code straight from its byte.
        const float scale = WSCALE * h2f(r.m & 0xFFFF), mn = WITH_MIN ? WSCALE * h2f(r.m >> 16) : -8.0f * scale;
        const uint32_t qq[2] = {r.q.x, r.q.y};
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t lo = qq[j] & 0x0F0F0F0Fu, hi = (qq[j] >> 4) & 0x0F0F0F0Fu;
            w[8 * j + 0] = fmaf(ubyte<0>(lo), scale, mn); w[8 * j + 1] = fmaf(ubyte<0>(hi), scale, mn);
            w[8 * j + 2] = fmaf(ubyte<1>(lo), scale, mn); w[8 * j + 3] = fmaf(ubyte<1>(hi), scale, mn);
            w[8 * j + 4] = fmaf(ubyte<2>(lo), scale, mn); w[8 * j + 5] = fmaf(ubyte<2>(hi), scale, mn);
            w[8 * j + 6] = fmaf(ubyte<3>(lo), scale, mn); w[8 * j + 7] = fmaf(ubyte<3>(hi), scale, mn);
        }
        k0 = (u4 >> 1) * 32 + part * 16;
        k1 = k0 + 8;
    }
};

template <bool WITH_MIN>
struct GQ5x { // byte j = elements j (low nibble) and j + 16 (high); qh bit e = bit 4 of element e
    static constexpr bool PRESCALED = true;
    static constexpr float WS = WSCALE;
    struct Raw { uint2 q; uint32_t qh, m; };
    __device__ static void load16(const GemmArgs &a, size_t row, int kstep, int u4, Raw &r) {
        const int blk = kstep * 2 + (u4 >> 1), part = u4 & 1;
        r.q = *reinterpret_cast<const uint2 *>(a.codes + row * a.codes_pitch + (size_t)blk * 16 + part * 8);
        r.qh = *reinterpret_cast<const uint32_t *>(a.qh + row * a.qh_pitch + (size_t)blk * 4);
        const uint8_t *mp = a.meta + row * a.meta_pitch;
        r.m = WITH_MIN ? *reinterpret_cast<const uint32_t *>(mp + (size_t)blk * 4)
                       : (uint32_t) * reinterpret_cast<const uint16_t *>(mp + (size_t)blk * 2);
    }
    __device__ static void cvt16(const Raw &r, int, int u4, float (&w)[16], int &k0, int &k1) {
        const int part = u4 & 1;
        const uint32_t qh = r.qh;
        // (u - 16) * d = u * d - 16 d exactly; with a minimum one rounding (fma) where the f32 reference has two.
        const float d = WSCALE * h2f(r.m & 0xFFFF), mn = WITH_MIN ? WSCALE * h2f(r.m >> 16) : -16.0f * d;
        const uint32_t qq[2] = {r.q.x, r.q.y};
        // four bits of qh -> bit 4 of four bytes: the copies of the multiplication lie 7 bits apart and do not meet
        auto fifth = [](uint32_t four) { return ((four * 0x00204081u) & 0x01010101u) << 4; };
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int e = part * 8 + 4 * j;
            const uint32_t lo = (qq[j] & 0x0F0F0F0Fu) | fifth((qh >> e) & 0xFu);
            const uint32_t hi = ((qq[j] >> 4) & 0x0F0F0F0Fu) | fifth((qh >> (e + 16)) & 0xFu);
            w[4 * j + 0] = fmaf(ubyte<0>(lo), d, mn); w[4 * j + 1] = fmaf(ubyte<1>(lo), d, mn);
            w[4 * j + 2] = fmaf(ubyte<2>(lo), d, mn); w[4 * j + 3] = fmaf(ubyte<3>(lo), d, mn);
            w[8 + 4 * j + 0] = fmaf(ubyte<0>(hi), d, mn); w[8 + 4 * j + 1] = fmaf(ubyte<1>(hi), d, mn);
            w[8 + 4 * j + 2] = fmaf(ubyte<2>(hi), d, mn); w[8 + 4 * j + 3] = fmaf(ubyte<3>(hi), d, mn);
        }
        k0 = (u4 >> 1) * 32 + part * 8;
        k1 = k0 + 16;
    }
};

struct GQ80 {
    static constexpr bool PRESCALED = true;
    static constexpr float WS = WSCALE;
    struct Raw { uint4 q; uint32_t m; };
    __device__ static void load16(const GemmArgs &a, size_t row, int kstep, int u4, Raw &r) {
        const int blk = kstep * 2 + (u4 >> 1), part = u4 & 1;
        r.q = *reinterpret_cast<const uint4 *>(a.codes + row * a.codes_pitch + (size_t)blk * 32 + part * 16);
        r.m = *reinterpret_cast<const uint16_t *>(a.meta + row * a.meta_pitch + (size_t)blk * 2);
    }
    __device__ static void cvt16(const Raw &r, int, int u4, float (&w)[16], int &k0, int &k1) {
        const int part = u4 & 1;
        // q * d = (q + 128) * d - 128 d exactly: the codes as unsigned bytes, one conversion each
        const float scale = WSCALE * h2f(r.m), off = -128.0f * scale;
        const uint32_t qq[4] = {r.q.x ^ 0x80808080u, r.q.y ^ 0x80808080u, r.q.z ^ 0x80808080u, r.q.w ^ 0x80808080u};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            w[4 * j + 0] = fmaf(ubyte<0>(qq[j]), scale, off); w[4 * j + 1] = fmaf(ubyte<1>(qq[j]), scale, off);
            w[4 * j + 2] = fmaf(ubyte<2>(qq[j]), scale, off); w[4 * j + 3] = fmaf(ubyte<3>(qq[j]), scale, off);
        }
        k0 = (u4 >> 1) * 32 + part * 16;
        k1 = k0 + 8;
    }
};

struct GF16 {
    static constexpr bool PRESCALED = false;
    static constexpr float WS = 1.0f; // plain weights may be large: no headroom to give away
    struct Raw { uint4 v0, v1; };
    __device__ static void load16(const GemmArgs &a, size_t row, int kstep, int u4, Raw &r) {
        const uint4 *p = reinterpret_cast<const uint4 *>(a.codes + row * a.codes_pitch + ((size_t)kstep * 64 + u4 * 16) * 2);
        r.v0 = p[0];
        r.v1 = p[1];
    }
    __device__ static void cvt16(const Raw &r, int, int u4, float (&w)[16], int &k0, int &k1) {
        const uint4 v0 = r.v0, v1 = r.v1;
        const uint32_t qq[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            w[2 * i] = h2f(qq[i] & 0xFFFF);
            w[2 * i + 1] = h2f(qq[i] >> 16);
        }
        k0 = u4 * 16;
        k1 = k0 + 8;
    }
};

struct GBF16 { // rows are padded to a multiple of 64 elements
    static constexpr bool PRESCALED = false;
    static constexpr float WS = 1.0f;
    struct Raw { uint4 v0, v1; };
    __device__ static void load16(const GemmArgs &a, size_t row, int kstep, int u4, Raw &r) {
        const uint4 *p = reinterpret_cast<const uint4 *>(a.codes + row * a.codes_pitch + ((size_t)kstep * 64 + u4 * 16) * 2);
        r.v0 = p[0];
        r.v1 = p[1];
    }
    __device__ static void cvt16(const Raw &r, int, int u4, float (&w)[16], int &k0, int &k1) {
        const uint4 v0 = r.v0, v1 = r.v1;
        const uint32_t qq[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            w[2 * i] = __builtin_bit_cast(float, qq[i] << 16);
            w[2 * i + 1] = __builtin_bit_cast(float, qq[i] & 0xFFFF0000u);
        }
        k0 = u4 * 16;
        k1 = k0 + 8;
    }
};

struct GF32 {
    static constexpr bool PRESCALED = false;
    static constexpr float WS = 1.0f; // plain weights may be large: no headroom to give away
    struct Raw { float4 v[4]; };
    __device__ static void load16(const GemmArgs &a, size_t row, int kstep, int u4, Raw &r) {
        const float4 *p = reinterpret_cast<const float4 *>(a.codes + row * a.codes_pitch + ((size_t)kstep * 64 + u4 * 16) * 4);
#pragma unroll
        for (int i = 0; i < 4; i++) r.v[i] = p[i];
    }
    __device__ static void cvt16(const Raw &r, int, int u4, float (&w)[16], int &k0, int &k1) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float4 v = r.v[i];
            w[4 * i] = v.x; w[4 * i + 1] = v.y; w[4 * i + 2] = v.z; w[4 * i + 3] = v.w;
        }
        k0 = u4 * 16;
        k1 = k0 + 8;
    }
};

// Eight values times `scale` -> eight f16 high parts and eight f16 remainders, as
// two 16-byte vectors.  The high part is the value with its mantissa cut to f16's eleven bits, a mask, exact in
// f16; the remainder is exact in f32 and keeps its own top eleven bits.
__device__ inline void split8_f16(const float *w, float scale, uint4 &hi, uint4 &lo) {
    uint32_t h[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float a = w[2 * i] * scale, b = w[2 * i + 1] * scale; // scale 1 folds away
        const float ah = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, a) & 0xFFFFE000u);
        const float bh = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, b) & 0xFFFFE000u);
        h[i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(ah, bh));
        l[i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a - ah, b - bh));
    }
    hi = make_uint4(h[0], h[1], h[2], h[3]);
    lo = make_uint4(l[0], l[1], l[2], l[3]);
}

// A workgroup barrier that orders LDS traffic only: __syncthreads() also waits for every global load in flight, which
// would pull the prefetched operands of later steps in front of every barrier.
__device__ inline void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0); // nothing moves across: what follows may count on the waits in front of the barrier
}

// WM = 1 or 2: the workgroup computes (128 * WM) x 128 outputs with eight waves of two kinds.
//   - four "multiplier" waves each own a (64 * WM) x 64 block (2 WM x 2 MFMA tiles) and do nothing but read the
//     current LDS stage and issue MFMAs;
//   - four "feeder" waves fetch the x tile and the packed weights of the step after next, convert the
//     next step's weights (dequantise, split into two f16) and write the other LDS stage.
// Waves are dealt to the four SIMDs in turn, so every SIMD holds one wave of each kind and its vector ALU converts
// while its matrix pipe multiplies; one barrier per K step hands the stages over.
template <class T, int WM>
__global__ void __launch_bounds__(512) gemm_kernel(GemmArgs a) {
    constexpr int BM = 128 * WM, NTF = 256;      // rows of x per tile; feeder threads
    constexpr int MI = 2 * WM;                   // MFMA tiles of a multiplier wave along M
    constexpr int XV = BM * 8 / NTF;             // 16-byte x vectors per feeder thread and K step (4 or 8)
    constexpr int UNITS = BN * 4 / NTF;          // 16-weight units per feeder thread and K step (= 2)
    constexpr int STAGE = (BM + 2 * BN) * LDK;   // halfs per LDS stage
    extern __shared__ _Float16 lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool feeder = tid >= NTF;
    // Workgroups of one XCD (those with equal id modulo 8) take consecutive tiles, N fastest: the x tile is
    // the big operand of a step (BM x 64 halfs against 128 x 64 packed weights), so the workgroups that share
    // an x tile should share an L2.
    const int nt = (a.n + BN - 1) / BN, total = (int)gridDim.x;
    int tile = blockIdx.x;
    if (total % 8 == 0) tile = (tile & 7) * (total >> 3) + (tile >> 3);
    const int m0 = (tile / nt) * BM, n0 = (tile % nt) * BN;
    // split K: workgroup (x, y) covers K steps [kbeg, kbeg + ksteps)
    const int kbeg = (int)blockIdx.y * a.steps_per_split;
    const int ksteps = a.k / BK - kbeg < a.steps_per_split ? a.k / BK - kbeg : a.steps_per_split;

    if (feeder) {
        const int ft = tid - NTF;
        u32x4 xa[XV];
        typename T::Raw raw[UNITS];
        // row addresses do not change from step to step
        const _Float16 *xrow[XV];
        size_t wrow[UNITS];
#pragma unroll
        for (int i = 0; i < XV; i++) {
            int v = ft + i * NTF;
            int gm = m0 + (v >> 3);
            gm = gm < a.m ? gm : a.m - 1;
            xrow[i] = a.xh + (size_t)gm * a.k + (v & 7) * 8;
        }
#pragma unroll
        for (int u = 0; u < UNITS; u++) {
            int gn = n0 + ((ft + u * NTF) >> 2);
            wrow[u] = (size_t)(gn < a.n ? gn : a.n - 1);
        }
        auto fetch = [&](int ks) { // clamped: past the last step the feeders re-read it and nobody looks
            ks = ks < ksteps ? ks : ksteps - 1;
#pragma unroll
            for (int i = 0; i < XV; i++) xa[i] = *reinterpret_cast<const u32x4 *>(xrow[i] + (size_t)(kbeg + ks) * BK);
#pragma unroll
            for (int u = 0; u < UNITS; u++) T::load16(a, wrow[u], kbeg + ks, (ft + u * NTF) & 3, raw[u]);
        };
        fetch(0);
        for (int ks = 0; ks <= ksteps; ks++) {
            // registers hold step ks: convert it into stage ks & 1, with step ks + 1 already requested
            _Float16 *As = lds + (ks & 1) * STAGE, *Bh = As + BM * LDK, *Bl = Bh + BN * LDK;
            const int kcur = ks < ksteps ? ks : ksteps - 1;
            u32x4 xs[XV];
            float w[UNITS][16];
            int k0[UNITS], k1[UNITS];
#pragma unroll
            for (int i = 0; i < XV; i++) xs[i] = xa[i];
#pragma unroll
            for (int u = 0; u < UNITS; u++) T::cvt16(raw[u], kbeg + kcur, (ft + u * NTF) & 3, w[u], k0[u], k1[u]);
            fetch(ks + 1);
            if (ks < ksteps) {
#pragma unroll
                for (int i = 0; i < XV; i++) {
                    int v = ft + i * NTF;
                    int row = v >> 3, c = v & 7;
                    *reinterpret_cast<u32x4 *>(As + row * LDK + c * 8) = xs[i];
                }
#pragma unroll
                for (int u = 0; u < UNITS; u++) {
                    int row = (ft + u * NTF) >> 2;
                    uint4 h0, l0, h1, l1;
                    split8_f16(w[u], T::PRESCALED ? 1.0f : T::WS, h0, l0);
                    split8_f16(w[u] + 8, T::PRESCALED ? 1.0f : T::WS, h1, l1);
                    *reinterpret_cast<uint4 *>(Bh + row * LDK + k0[u]) = h0;
                    *reinterpret_cast<uint4 *>(Bh + row * LDK + k1[u]) = h1;
                    *reinterpret_cast<uint4 *>(Bl + row * LDK + k0[u]) = l0;
                    *reinterpret_cast<uint4 *>(Bl + row * LDK + k1[u]) = l1;
                }
            }
            lds_barrier(); // barrier ks: stage ks & 1 is complete, stage (ks + 1) & 1 has been read; the loads of step
                           // ks + 1 stay in flight across it
        }
        return;
    }

    const int wm = (wave >> 1) * (32 * MI), wn = (wave & 1) * 64; // this wave's block inside the tile
    const int li = lane & 31, lk = (lane >> 5) * 8;
    float16v acc[MI][2];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
    __syncthreads(); // barrier 0
    for (int ks = 0; ks < ksteps; ks++) {
        const _Float16 *As = lds + (ks & 1) * STAGE, *Bh = As + BM * LDK, *Bl = Bh + BN * LDK;
        // fragments of sub-step kk + 1 are read from LDS while the sixteen MFMAs of sub-step kk run
        half8 af[2][MI], bh[2][2], bl[2][2];
        auto read_frags = [&](int kk, int slot) {
#pragma unroll
            for (int i = 0; i < MI; i++) af[slot][i] = *reinterpret_cast<const half8 *>(As + (wm + i * 32 + li) * LDK + kk + lk);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                bh[slot][j] = *reinterpret_cast<const half8 *>(Bh + (wn + j * 32 + li) * LDK + kk + lk);
                bl[slot][j] = *reinterpret_cast<const half8 *>(Bl + (wn + j * 32 + li) * LDK + kk + lk);
            }
        };
        read_frags(0, 0);
#pragma unroll
        for (int t = 0; t < BK / 16; t++) {
            if (t + 1 < BK / 16) read_frags((t + 1) * 16, (t + 1) & 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[t & 1][i], bl[t & 1][j], acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[t & 1][i], bh[t & 1][j], acc[i][j], 0, 0, 0);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads(); // barrier ks + 1
    }
    // D layout: lane -> column li; register r -> row 8 * (r / 4) + 4 * (lane / 32) + r % 4
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int gn = n0 + wn + j * 32 + li;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int gm = m0 + wm + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (gm < a.m && gn < a.n) {
                    if (!a.pair) {
                        if (a.ypart) a.ypart[((size_t)blockIdx.y * a.m + gm) * a.n + gn] = acc[i][j][r];
                        else a.y[(size_t)gm * a.n + gn] = acc[i][j][r] * (a.rowscale[gm] * (1.0f / T::WS));
                    } else if ((r & 1) == 0) { // gm is even: this register and the next hold the two parts of row gm / 2
                        const size_t t = (size_t)(gm >> 1);
                        const float v = acc[i][j][r] + acc[i][j][r + 1];
                        if (a.ypart) {
                            a.ypart[((size_t)blockIdx.y * (a.m >> 1) + t) * a.n + gn] = v;
                        } else {
                            float out = v * (a.rowscale[gm] * (1.0f / T::WS));
                            if (a.bias) out += a.bias[gn];
                            if (a.resid) out += a.resid[t * a.n + gn];
                            a.y[t * a.n + gn] = out;
                        }
                    }
                }
            }
        }
}

typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void gbl_void;

// s_waitcnt vmcnt(N) lgkmcnt(0) (gfx9 encoding: vmcnt in bits 3:0 and 15:14, expcnt 6:4 left at 7, lgkmcnt 11:8)
template <int N>
__device__ inline void wait_vm_and_lds() {
    __builtin_amdgcn_s_waitcnt(((N >> 4) << 14) | (7 << 4) | (N & 15));
}

// ---------------------------------------------------------------------------
// Q4_0 / Q4_1 / Q5_0 / Q5_1 / Q8_0 (blocks of 32): one MFMA per product, the block's scale applied by the vector ALU.
//
// w = d * (q - c) (Q4_0: c = 8, Q5_0: 16, Q8_0: the code is a signed byte) or d * q + m (Q4_1, Q5_1) with f16 d (and
// m) per block of 32.  The B operand is the centred code q - c itself, an integer that f16 holds exactly: the two
// MFMAs of a block (32 k) start from zero, so their result is the block's sum of (q - c) * x, exact in f32 to within
// the accumulation, and every lane then adds it, times the d of its column and block, into its accumulators (a lane of
// the 32 x 32 MFMA output owns one column): sixteen v_fma per tile and block where gemm_kernel pays a second MFMA per
// product and about ten vector-ALU instructions per weight for the dequantisation and the high/low split.  Converting
// costs two instructions per pair of weights: the code pairs come out of the packed nibbles two at a time with one mask
// each (Q4: after one byte permutation, its neighbours share a byte; Q8_0: bytes 0, 2 and 1, 3 of a dword), Q5's fifth
// bits out of qh four at a time with one multiplication, 0x6400 | q is the f16 number 1024 + q, and one packed
// subtraction of 1024 + c centres it.  x is stored with elements 1 and 2 of every four exchanged, which is
// the order the masks produce.
// The types with a minimum go in as d * (q - c) + (m + c d): the first sum is then as well conditioned as the weights
// themselves (with q as it is, two sums three times the size of the result would cancel in f32).  The second,
// sum_b (m + c d)[n, b] * (sum of x over block b), goes through the matrix pipe too, two MFMAs per tile and
// superblock of 256 k: A = the eight block sums of the row as f16 pairs (hi for k 0..7, lo for k 8..15, written by the
// x pre-pass, times 1 / 64), B = the column's eight offsets m + c d as f16 pairs
// (the leading halves twice, then the remainders against the sums' leading halves); the sum is added times 256 and
// the main term's scales are d * 256 / 64 to match.
//
// 256 x 128 outputs per workgroup of eight waves (64 x 64 each), all of K: the calls that come here have more than half as many of
// them as the chip has compute units (see axq_dev_rows_gemm_covers).  x tiles straight from memory into three LDS stages, two weight
// stages, one barrier per K step that waits for LDS only, explicit counts of the loads issued since.  A thread converts half a block
// (16 weights of one row) per step.  The scale records of the tile's columns lie in LDS too, a superblock of them at a time.
// ---------------------------------------------------------------------------
constexpr int PBM = 256, PBN = 128;        // rows of x and output columns (weight rows) per workgroup
constexpr float XSUM_SCALE = 1.0f / 64.0f; // the x pre-pass stores the block sums times this

template <int BITS, bool WITH_MIN>
__global__ void __launch_bounds__(512) gemm_blk32_kernel(GemmArgs a) {
    constexpr int BM = PBM, NW = 8, AROWS = BM / NW, XL = AROWS / 8;
    constexpr int MI = BM / 128;                           // MFMA tiles of a wave along M: the waves lie 4 x 2, (32 MI) x 64 each
    constexpr int ASTAGE = BM * 64, BSTAGE = PBN * 64, BOFF = 3 * ASTAGE; // halfs
    constexpr int F = BITS == 5 ? 2 : 1;   // loads of a weight request: codes (and fifth bits)
    constexpr int CENTER = BITS == 5 ? 16 : BITS == 4 ? 8 : 128; // the codes go in centred (Q5_0's, Q4_0's and Q8_0's own form)
    constexpr int ML = 1;                  // per superblock: this wave's kilobyte of scale records
    constexpr float OFF = 1024.0f + CENTER; // 0x6400 | q is 1024 + q
    constexpr float ASCALE = WSCALE * XSUM_SCALE; // the accumulators hold the result times this
    extern __shared__ _Float16 lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nt = (a.n + PBN - 1) / PBN, total = (int)gridDim.x;
    int tile = blockIdx.x;
    if (total % 8 == 0) tile = (tile & 7) * (total >> 3) + (tile >> 3); // workgroups of one XCD share x tiles
    const int m0 = (tile / nt) * BM, n0 = (tile % nt) * PBN;
    const int T = a.k / BK; // steps of 64 k: a multiple of 4 (whole superblocks)

    // ---- x tiles (rows of the scratch buffer are allocated up to a multiple of BM: no clamp)
    const uint8_t *xbase = reinterpret_cast<const uint8_t *>(a.xh + (size_t)m0 * a.k);
    const uint32_t xrow_l = (uint32_t)(wave * AROWS + (lane >> 3)), xchunk_l = (uint32_t)((lane & 7) ^ (lane >> 4));
    const uint32_t xoff = (xrow_l * (uint32_t)a.k + xchunk_l * 8) * 2;
    const size_t x8rows = (size_t)8 * a.k * 2;
    auto load_x = [&](int step, int stage) {
        step = step < T ? step : T - 1;
        const uint8_t *g = xbase + (size_t)step * (BK * 2);
        _Float16 *dst = lds + stage * ASTAGE + wave * AROWS * 64;
#pragma unroll
        for (int i = 0; i < XL; i++)
            __builtin_amdgcn_global_load_lds((gbl_void *)(g + i * x8rows + ((i & 1) ? xoff ^ 64u : xoff)), (lds_void *)(dst + i * 8 * 64), 16, 0, 0);
        asm volatile("" ::: "memory"); // what is requested after this stays after it: the waits in front of the barriers count on the order
    };

    // ---- weights: this thread's half block (16 weights) of every step
    const int wrow = tid & 127, bis = tid >> 8, half = (tid >> 7) & 1; // row of the tile; which of the step's two blocks; which half of it
    const int crow = n0 + wrow < a.n ? n0 + wrow : a.n - 1;
    const uint8_t *cp = a.codes + (size_t)crow * a.codes_pitch, *qp = BITS == 5 ? a.qh + (size_t)crow * a.qh_pitch : nullptr;
    struct Raw { u32x4 q; uint32_t qh; };
    // the thread's block of a step: 16 bytes of nibbles (Q5: both halves fetch all of them, they interleave), or its own
    // 16 of the block's 32 bytes (Q8_0)
    auto fetch = [&](int step, Raw &r) {
        step = step < T ? step : T - 1;
        const size_t blk = (size_t)step * 2 + bis;
        r.q = *reinterpret_cast<const u32x4 *>(BITS == 8 ? cp + blk * 32 + half * 16 : cp + blk * 16);
        if (BITS == 5) r.qh = *reinterpret_cast<const uint32_t *>(qp + blk * 4);
        asm volatile("" ::: "memory");
    };
    const int b_wr = wrow * 64; // the thread's row in a weight plane; chunk ch of it lies at (ch ^ ((wrow / 2) & 7)) * 8
    const int b_sw = (wrow >> 1) & 7;
    // chunk c = 2 half + cc (cc = 0, 1: elements 8 c .. 8 c + 7) of the block in `r` -> weight stage `stage`, as pairs of
    // codes in the two halves of a dword, in the order [e0, e2, e1, e3, e4, e6, e5, e7]
    auto convert = [&](const Raw &r, int cc, int stage) {
        const int c = 2 * half + cc;
        uint32_t pr[4];
        if (BITS == 5) { // GGUF: byte j = elements j (low nibble) and j + 16 (high); qh bit e = bit 4 of element e
            const uint32_t d0 = cc ? r.q[2] : r.q[0], d1 = cc ? r.q[3] : r.q[1];
            const int sh = half * 4;
            pr[0] = (d0 >> sh) & 0x000F000Fu; pr[1] = (d0 >> (sh + 8)) & 0x000F000Fu;
            pr[2] = (d1 >> sh) & 0x000F000Fu; pr[3] = (d1 >> (sh + 8)) & 0x000F000Fu;
            // bits b0..b3 of `four` times (2^4 + 2^18): b0 lands on bit 4 and b2 on bit 20 (of the pair e, e + 2), nothing else does
            const uint32_t eight = (r.qh >> (8 * c)) & 0xFFu;
            pr[0] |= ((eight & 0xFu) * 0x40010u) & 0x00100010u;
            pr[1] |= (((eight >> 1) & 0x7u) * 0x40010u) & 0x00100010u;
            pr[2] |= ((eight >> 4) * 0x40010u) & 0x00100010u;
            pr[3] |= ((eight >> 5) * 0x40010u) & 0x00100010u;
        } else if (BITS == 4) { // reference nibble order: byte i = elements 2 i (low), 2 i + 1 (high): dword c is the chunk
            const uint32_t w = half ? (cc ? r.q[3] : r.q[2]) : (cc ? r.q[1] : r.q[0]);
            const uint32_t p4 = __builtin_amdgcn_perm(w, w, 0x03010200u); // bytes 0, 2, 1, 3: a half dword = two neighbours
            pr[0] = p4 & 0x000F000Fu; pr[1] = (p4 >> 4) & 0x000F000Fu;
            pr[2] = (p4 >> 8) & 0x000F000Fu; pr[3] = (p4 >> 12) & 0x000F000Fu;
        } else { // signed bytes in element order, as unsigned ones (+ 128)
            const uint32_t x0 = (cc ? r.q[2] : r.q[0]) ^ 0x80808080u, x1 = (cc ? r.q[3] : r.q[1]) ^ 0x80808080u;
            pr[0] = x0 & 0x00FF00FFu; pr[1] = (x0 >> 8) & 0x00FF00FFu;
            pr[2] = x1 & 0x00FF00FFu; pr[3] = (x1 >> 8) & 0x00FF00FFu;
        }
        const half2v off2 = {(_Float16)OFF, (_Float16)OFF};
        uint32_t oh[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t bits = pr[i] | 0x64006400u;
            const half2v qf = __builtin_bit_cast(half2v, bits) - off2; // exact: integers below 2048
            oh[i] = __builtin_bit_cast(uint32_t, qf);
        }
        _Float16 *bs = lds + BOFF + stage * BSTAGE + b_wr + (((4 * bis + c) ^ b_sw) * 8);
        *reinterpret_cast<u32x4 *>(bs) = u32x4{oh[0], oh[1], oh[2], oh[3]};
    };

    // ---- multiplier side
    const int wm = (wave >> 1) * (32 * MI), wn = (wave & 1) * 64;
    const int li = lane & 31, hh = lane >> 5;
    const int sw = ((hh ^ (li >> 1)) & 7) * 8;
    const int a_rd = (wm + li) * 64 + sw, b_rd = BOFF + (wn + li) * 64 + sw;
    float16v acc[MI][2];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
    // The scale records of the tile's 128 columns, eight blocks of a superblock each ((d, m) pairs for Q5_1: 32 bytes;
    // d alone for Q5_0: 16 bytes), lie in LDS behind the weight stages, two superblocks of them: every wave brings in a
    // kilobyte of the next superblock's at the first step of a superblock (the same kilobyte twice or four times over:
    // one request per wave keeps the waves' counts of loads equal).
    constexpr int RV = WITH_MIN ? 2 : 1;      // 16-byte vectors per column and superblock
    constexpr int RECB = PBN * 16 * RV;       // bytes of one superblock's records
    uint8_t *rec_lds = reinterpret_cast<uint8_t *>(lds + BOFF + 2 * BSTAGE);
    const int nsb = T >> 2;
    const int rc0 = WITH_MIN ? (wave & 3) * 32 : (wave & 1) * 64; // first column of this wave's kilobyte
    int rcol = n0 + rc0 + (WITH_MIN ? lane >> 1 : lane);
    rcol = rcol < a.n ? rcol : a.n - 1;
    const uint8_t *rsrc = a.meta + (size_t)rcol * a.meta_pitch + (WITH_MIN ? (lane & 1) * 16 : 0);
    auto fetch_records = [&](int sb) {
        sb = sb < nsb ? sb : nsb - 1;
        __builtin_amdgcn_global_load_lds((gbl_void *)(rsrc + (size_t)sb * (16 * RV)), (lds_void *)(rec_lds + (sb & 1) * RECB + rc0 * 16 * RV), 16, 0, 0);
        asm volatile("" ::: "memory");
    };
    u32x4 mx[MI];
    const uint8_t *x3p = reinterpret_cast<const uint8_t *>(a.xs3 + (size_t)(m0 + wm + li) * a.xs3_pitch + hh * 16);
    auto fetch_sums = [&](int sb) {
#pragma unroll
        for (int i = 0; i < MI; i++) mx[i] = *reinterpret_cast<const u32x4 *>(x3p + ((size_t)i * 32 * a.xs3_pitch + (size_t)sb * 32) * 2);
    };
    // d of block bq (0..7) of superblock sb, column j of this lane, times WSCALE
    const uint8_t *rlane = rec_lds + (wn + li) * 16 * RV;
    auto scale_of = [&](int sb, int j, int bq) {
        const uint16_t w = *reinterpret_cast<const uint16_t *>(rlane + (sb & 1) * RECB + j * 32 * 16 * RV + bq * (WITH_MIN ? 4 : 2));
        return ASCALE * h2f(w);
    };
    // One block of 32 k = two sub-steps t0 = 2 hb, t0 + 1 of the step: its sum over k, then times the block's d into the
    // accumulators.  bq: the block's number in the superblock.
    auto multiply_block = [&](int as, int par, int hb, int sb, int bq) {
        const float16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        const int t0 = 2 * hb, t1 = 2 * hb + 1;
        const float df[2] = {scale_of(sb, 0, bq), scale_of(sb, 1, bq)};
        half8 b0[2], b1[2]; // the block's weight fragments serve both row tiles
#pragma unroll
        for (int j = 0; j < 2; j++) {
            b0[j] = *reinterpret_cast<const half8 *>(lds + par * BSTAGE + (b_rd ^ (t0 * 16)) + j * 32 * 64);
            b1[j] = *reinterpret_cast<const half8 *>(lds + par * BSTAGE + (b_rd ^ (t1 * 16)) + j * 32 * 64);
        }
#pragma unroll
        for (int i = 0; i < MI; i++) { // one row tile's two sums at a time: registers
            const half8 a0 = *reinterpret_cast<const half8 *>(lds + as + (a_rd ^ (t0 * 16)) + i * 32 * 64);
            const half8 a1 = *reinterpret_cast<const half8 *>(lds + as + (a_rd ^ (t1 * 16)) + i * 32 * 64);
            float16v S[2];
#pragma unroll
            for (int j = 0; j < 2; j++) S[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, b0[j], zero, 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 2; j++) S[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, b1[j], S[j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] = fmaf(S[j][r], df[j], acc[i][j][r]);
        }
    };
    auto multiply_min = [&](int sb) {
        // B = the blocks' offsets m + CENTER d (the weight of the middle code), each worked out in f32 (exact to its last
        // bit) and cut into two f16, vh + vl: the first product takes [vh | vh] against the sums' [hi | lo], the second
        // [vl | 0].  Kept apart (m against the sums, then CENTER d against the sums, added afterwards) the two halves of the
        // offset are each as large as a block's range times sum x and cancel in f32: 1.1e-3 at the strict floor of the
        // parity test for rows with a mean; together they are the block's middle, small for weights around zero.  An
        // offset beyond f16's range (weights past 65504) saturates.
        half8 bh[2], bl[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            uint32_t oh[4], ol[4];
#pragma unroll
            for (int q = 0; q < 4; q++) { // blocks 2 q, 2 q + 1: (d, m) records
                // (read as a plain vector: a read through HIP's uint2 made the compiler wait for every load in flight)
                typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                const u32x2 r2 = *reinterpret_cast<const u32x2 *>(rlane + (sb & 1) * RECB + j * 32 * 16 * RV + q * 8);
                const float v0 = fmaf((float)CENTER, h2f(r2[0] & 0xFFFFu), h2f(r2[0] >> 16));
                const float v1 = fmaf((float)CENTER, h2f(r2[1] & 0xFFFFu), h2f(r2[1] >> 16));
                const auto vh = __builtin_amdgcn_cvt_pkrtz(v0, v1);
                oh[q] = __builtin_bit_cast(uint32_t, vh);
                const uint32_t low = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(v0 - (float)vh[0], v1 - (float)vh[1]));
                ol[q] = hh ? 0u : low; // the sums' low halves meet vh only
            }
            bh[j] = __builtin_bit_cast(half8, u32x4{oh[0], oh[1], oh[2], oh[3]});
            bl[j] = __builtin_bit_cast(half8, u32x4{ol[0], ol[1], ol[2], ol[3]});
        }
        // the block sums are stored times XSUM_SCALE: with the factor below the accumulators receive the term times
        // WSCALE * XSUM_SCALE, which is what the main term scales its sums to (scale_of)
        // (added by the vector ALU like the main term: accumulators that the matrix pipe also wrote would be kept twice)
        const float16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < MI; i++) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                float16v S = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, mx[i]), bh[j], zero, 0, 0, 0);
                S = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, mx[i]), bl[j], S, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] = fmaf(S[r], WSCALE, acc[i][j][r]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    // Steps g = 0 .. T - 1 in groups of four (a superblock).  Step g multiplies x stage g % 3 with weight stage g & 1,
    // brings the x tile of step g + 2 into its stage, converts the weights of step g + 1 into the other weight stage
    // and requests those of step g + 3; the first step of a group also requests the scale records of the next
    // superblock, the third this one's block sums.  Every wave issues the same loads in the same order, so that the
    // wait in front of a barrier (for the x tile of step g + 1, requested a step ago) can leave the younger requests in
    // flight.
    Raw buf[4]; // the blocks of steps g .. g + 3, at g % 4 ..
    load_x(0, 0);
    load_x(1, 1);
    fetch(0, buf[0]);
    fetch(1, buf[1]);
    fetch(2, buf[2]);
    fetch_records(0);
    convert(buf[0], 0, 0);
    convert(buf[0], 1, 0);
    wait_vm_and_lds<0>();
    lds_barrier();
    int g3 = 0;
    for (int sb = 0; sb < nsb; sb++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int g = 4 * sb + i;
            const int as = g3 * ASTAGE, xs = (g3 == 0 ? 2 : g3 - 1);
            // the order of the requests: the weight blocks first, so that the wait at the end of the next step, which
            // lets that step's x tile and what follows it stay out, covers them
            if (WITH_MIN && i == 2) { // this superblock's block sums, for the end of the next step: ahead of the step's other
                fetch_sums(sb);       // requests, so that the wait at its end covers them
                asm volatile("" ::: "memory");
            }
            fetch(g + 3, buf[(i + 3) & 3]);
            load_x(g + 2, xs);
            if (i == 0) fetch_records(sb + 1);
            // (past the last step the conversion writes a stage that nobody reads)
#pragma unroll
            for (int hb = 0; hb < 2; hb++) {
                multiply_block(as, i & 1, hb, sb, 2 * i + hb);
                convert(buf[(i + 1) & 3], hb, (i + 1) & 1);
            }
            if (WITH_MIN && i == 3) multiply_min(sb);
            // younger than the x tile of step g + 1 (requested a step ago): what followed it in that step, and this step's
            if (i == 0) wait_vm_and_lds<F + XL + ML>();
            else if (i == 1) wait_vm_and_lds<ML + F + XL>();
            else wait_vm_and_lds<F + XL>();
            lds_barrier();
            g3 = g3 == 2 ? 0 : g3 + 1;
        }
    }
    wait_vm_and_lds<0>(); // nothing of this workgroup may still be on its way into LDS when it ends
    // D layout: lane -> column li; register r -> row 8 * (r / 4) + 4 * (lane / 32) + r % 4
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int gn = n0 + wn + j * 32 + li;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int gm = m0 + wm + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (gm < a.m && gn < a.n) {
                    if (!a.pair) a.y[(size_t)gm * a.n + gn] = acc[i][j][r] * (a.rowscale[gm] * (1.0f / ASCALE));
                }
            }
#pragma unroll
            for (int r = 0; r < 16; r += 2) { // pair mode: an even row and the next hold the two parts of activation row gm / 2
                const int gm = m0 + wm + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (a.pair && gm < a.m && gn < a.n) {
                    const size_t t = (size_t)(gm >> 1);
                    const float v = acc[i][j][r] + acc[i][j][r + 1];
                    float out = v * (a.rowscale[gm] * (1.0f / ASCALE));
                    if (a.bias) out += a.bias[gn];
                    if (a.resid) out += a.resid[t * a.n + gn];
                    a.y[t * a.n + gn] = out;
                }
            }
        }
}

// What gemm_blk32_kernel wants from the x pre-pass besides the scaled f16 rows: elements 1 and 2 of every group of four
// exchanged, and the sums of every 32 consecutive (scaled, f16) elements as f16 pairs hi + lo: 32 halfs per superblock,
// [hi of its 8 sub-blocks | the same | lo | zeros] (NULL xs3: plain rows for the other kernels).
struct XSums {
    _Float16 *xs3;
    int pitch; // halfs per row: 32 per superblock and 32 or 64 zeros, see xs3_pitch
};
// one or two superblocks of zeros end a row
__host__ __device__ inline int xs3_pitch(int64_t k) { return (int)(((k >> 8) + 2) & ~(int64_t)1) * 32; }

// The sum `s` of the caller's four elements, added over the eight threads of a 32-element group; the first of them
// stores the pair.  g = index of the group along the row.
__device__ inline void store_group_sum(float s, int g, int n_groups, _Float16 *row3, const XSums &xs) {
    s += __shfl_xor(s, 1);
    s += __shfl_xor(s, 2);
    s += __shfl_xor(s, 4);
    if ((threadIdx.x & 7) == 0 && g < n_groups) {
        s *= XSUM_SCALE; // 32 elements below 2^15 each: the sum must not leave f16's range
        const _Float16 hi = (_Float16)s, lo = (_Float16)(s - (float)hi);
        _Float16 *base = row3 + (size_t)(g >> 3) * 32 + (g & 7);
        base[0] = hi;
        base[8] = hi;
        base[16] = lo;
        base[24] = (_Float16)0.f;
    }
}

// bf16 rows -> f16 rows scaled by a power of two (largest magnitude below 2^15), and the scale to undo it.
__global__ void __launch_bounds__(256) gemm_prep_x_kernel(const uint16_t *x, int m, int k, _Float16 *xh, float *rowscale, XSums xs) {
    __shared__ float red[4];
    const int row = blockIdx.x;
    const uint16_t *xr = x + (size_t)row * k;
    uint32_t amax_bits = 0;
    for (int i = threadIdx.x; i < k; i += blockDim.x) {
        uint32_t b = (uint32_t)(xr[i] & 0x7FFF);
        amax_bits = b > amax_bits ? b : amax_bits;
    }
    float amax = __builtin_bit_cast(float, amax_bits << 16);
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) amax = fmaxf(amax, __shfl_xor(amax, s));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
    _Float16 *row3 = xs.xs3 ? xs.xs3 + (size_t)row * xs.pitch : nullptr;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    // amax in [2^e, 2^(e+1)) -> multiply by 2^(14 - e); inf/nan rows are passed through unscaled
    int eb = (int)((__builtin_bit_cast(uint32_t, amax) >> 23) & 0xFF);
    if (eb == 0 || eb == 0xFF) eb = 127 + 14;
    int sb = 127 + 14 - (eb - 127);
    sb = sb < 1 ? 1 : (sb > 254 ? 254 : sb);
    const float f = __builtin_bit_cast(float, (uint32_t)sb << 23);
    typedef _Float16 half4 __attribute__((ext_vector_type(4)));
    for (int i4 = threadIdx.x; i4 < (k >> 2); i4 += blockDim.x) { // k is a multiple of 64: whole groups of eight threads
        const uint2 raw = reinterpret_cast<const uint2 *>(xr)[i4];
        const _Float16 h0 = (_Float16)(__builtin_bit_cast(float, raw.x << 16) * f), h1 = (_Float16)(__builtin_bit_cast(float, raw.x & 0xFFFF0000u) * f);
        const _Float16 h2 = (_Float16)(__builtin_bit_cast(float, raw.y << 16) * f), h3 = (_Float16)(__builtin_bit_cast(float, raw.y & 0xFFFF0000u) * f);
        if (row3) {
            reinterpret_cast<half4 *>(xh + (size_t)row * k)[i4] = half4{h0, h2, h1, h3};
            store_group_sum(((float)h0 + (float)h1) + ((float)h2 + (float)h3), i4 >> 3, k >> 5, row3, xs);
        } else {
            reinterpret_cast<half4 *>(xh + (size_t)row * k)[i4] = half4{h0, h1, h2, h3};
        }
    }
    if (row3 && (int)threadIdx.x < xs.pitch - (k >> 8) * 32) row3[(size_t)(k >> 8) * 32 + threadIdx.x] = (_Float16)0.f; // the zeros that end a row
    if (threadIdx.x == 0) rowscale[row] = 1.0f / f;
}

// y = (sum over the splits, in order) * rowscale / ws (+ bias + resid): four outputs per thread.  `rows` output rows;
// row_mul = 2 in pair mode (output row t was scaled as activation rows 2t, 2t + 1).  Latency bounds it: all parts are requested at
// once, S of them, or, S = 0, seven at a time behind the first (one after the other the two-sums made BF16 weights 2048 x 4096 times
// 100 rows, eight parts, 0.45 us slower than plain additions, 30.5 for 30.1 us; 28.9 so).
template <int S>
__global__ void __launch_bounds__(256) gemm_reduce_kernel(const float *ypart, const float *rowscale, int rows, int n, int parts,
                                                          float inv_ws, int row_mul, const float *bias, const float *resid, float *y) {
    const int splits = S > 0 ? S : parts;
    const size_t i4 = (size_t)blockIdx.x * blockDim.x + threadIdx.x, total4 = (size_t)rows * n / 4;
    if (i4 >= total4) return;
    const float4 first = reinterpret_cast<const float4 *>(ypart)[i4];
    float acc[4] = {first.x, first.y, first.z, first.w}, lost[4] = {0.f, 0.f, 0.f, 0.f}; // the sum, and what its additions rounded off (two-sum)
    constexpr int AHEAD = S > 0 ? S - 1 : 7;
    for (int s0 = 1; s0 < splits; s0 += AHEAD) {
        float4 v4[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; i++)
            if (s0 + i < splits) v4[i] = reinterpret_cast<const float4 *>(ypart + (size_t)(s0 + i) * rows * n)[i4];
#pragma unroll
        for (int i = 0; i < AHEAD; i++) {
            if (s0 + i >= splits) break;
            const float v[4] = {v4[i].x, v4[i].y, v4[i].z, v4[i].w};
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float sum = acc[c] + v[c], part = sum - acc[c];
                lost[c] += (acc[c] - (sum - part)) + (v[c] - part);
                acc[c] = sum;
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 4; c++) acc[c] = lost[c] == lost[c] ? acc[c] + lost[c] : acc[c]; // not a number beside an infinite sum
    const size_t row = (i4 * 4) / (size_t)n, col = (i4 * 4) % (size_t)n; // n is a multiple of 4: the four share a row
    const float f = rowscale[row * row_mul] * inv_ws;
    float4 out = make_float4(acc[0] * f, acc[1] * f, acc[2] * f, acc[3] * f);
    if (bias) {
        out.x += bias[col]; out.y += bias[col + 1]; out.z += bias[col + 2]; out.w += bias[col + 3];
    }
    if (resid) {
        const float4 r = reinterpret_cast<const float4 *>(resid)[i4];
        out.x += r.x; out.y += r.y; out.z += r.z; out.w += r.w;
    }
    reinterpret_cast<float4 *>(y)[i4] = out;
}

template <class T>
int launch_gemm(axq_ctx *ctx, GemmArgs a, int splits) {
    static std::atomic<uint64_t> lds_allowed[2]; // per kernel: a bit per device
    const int wm = a.wm, bm = 128 * wm;
    const unsigned tiles = (unsigned)(((a.n + BN - 1) / BN) * ((a.m + bm - 1) / bm));
    const dim3 grid(tiles, (unsigned)splits);
    const size_t lds = (size_t)2 * (bm + 2 * BN) * LDK * sizeof(_Float16); // two stages
    {
        int rc;
        if ((rc = axq_allow_lds(ctx, reinterpret_cast<const void *>(gemm_kernel<T, 2>), lds_allowed[1], 2 * (256 + 2 * BN) * LDK * 2))) return rc;
        if ((rc = axq_allow_lds(ctx, reinterpret_cast<const void *>(gemm_kernel<T, 1>), lds_allowed[0], 2 * (128 + 2 * BN) * LDK * 2))) return rc;
    }
    if (wm == 2) gemm_kernel<T, 2><<<grid, 512, lds, ctx->stream>>>(a);
    else gemm_kernel<T, 1><<<grid, 512, lds, ctx->stream>>>(a);
    AXQ_LAUNCH_CHECK(ctx, "gemm_kernel");
    if (splits == 1) return AXQ_OK;
    return axq_gemm_reduce(ctx, a.ypart, a.rowscale, a.pair ? a.m / 2 : a.m, a.n, splits, 1.0f / T::WS, a.pair ? 2 : 1, a.bias, a.resid, a.y);
}

// f32 rows, optionally RMS-normalised on the way ((x * inv_rms) * norm_w, RMSNorm::forward, llm/src/llama.rs:158-187),
// -> two f16 rows each under one power-of-two scale: row 2t holds the leading 11 bits of every element, row 2t + 1
// what those leave, so that their GEMM results add up to the f32 product (the GEMM's epilogue adds them: pair mode).
// SWIGLU: x holds rows of 2 k gate/up values, four gate values followed by the four up values of the same indices (the row
// order of the fused gate/up weight), and the row that is split is silu(gate) * up (k a multiple of 4, at most 16384).
template <bool SWIGLU>
__global__ void __launch_bounds__(256) gemm_prep_x_f32_kernel(const float *x, const float *norm_w, float eps, int m, int k,
                                                              _Float16 *xh, float *rowscale, XSums xs) {
    // the row stays in registers between the passes: 16 bytes per thread and step, up to 16 steps (k <= 16384);
    // longer rows (or k not a multiple of 4) take the plain loops below
    constexpr int STEPS = 16;
    __shared__ float red[4];
    const int row = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float *xr = x + (size_t)row * (SWIGLU ? 2 * k : k);
    const bool in_regs = SWIGLU || ((k & 3) == 0 && k <= STEPS * 256 * 4);
    float4 v[STEPS];
    if (in_regs) {
#pragma unroll
        for (int c = 0; c < STEPS; c++) {
            const int i4 = c * 256 + threadIdx.x;
            if (SWIGLU) {
                v[c] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (i4 * 4 < k) {
                    const float4 g = reinterpret_cast<const float4 *>(xr)[2 * i4], u = reinterpret_cast<const float4 *>(xr)[2 * i4 + 1];
                    v[c].x = (g.x * (1.0f / (1.0f + expf(-g.x)))) * u.x;
                    v[c].y = (g.y * (1.0f / (1.0f + expf(-g.y)))) * u.y;
                    v[c].z = (g.z * (1.0f / (1.0f + expf(-g.z)))) * u.z;
                    v[c].w = (g.w * (1.0f / (1.0f + expf(-g.w)))) * u.w;
                }
            } else {
                v[c] = i4 * 4 < k ? reinterpret_cast<const float4 *>(xr)[i4] : make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
    }
    float inv = 1.0f;
    if (norm_w) {
        float ss = 0.f;
        if (in_regs) {
#pragma unroll
            for (int c = 0; c < STEPS; c++) {
                ss = fmaf(v[c].x, v[c].x, ss); ss = fmaf(v[c].y, v[c].y, ss); ss = fmaf(v[c].z, v[c].z, ss); ss = fmaf(v[c].w, v[c].w, ss);
            }
        } else {
            for (int i = threadIdx.x; i < k; i += blockDim.x) ss = fmaf(xr[i], xr[i], ss);
        }
#pragma unroll
        for (int s = 32; s >= 1; s >>= 1) ss += __shfl_xor(ss, s);
        if (lane == 0) red[wave] = ss;
        __syncthreads();
        ss = (red[0] + red[1]) + (red[2] + red[3]);
        __syncthreads();
        inv = 1.0f / sqrtf(ss / (float)k + eps);
        if (in_regs) {
#pragma unroll
            for (int c = 0; c < STEPS; c++) {
                const int i4 = c * 256 + threadIdx.x;
                if (i4 * 4 < k) {
                    const float4 w = reinterpret_cast<const float4 *>(norm_w)[i4];
                    v[c] = make_float4((v[c].x * inv) * w.x, (v[c].y * inv) * w.y, (v[c].z * inv) * w.z, (v[c].w * inv) * w.w);
                }
            }
        }
    }
    uint32_t amax_bits = 0; // of |v| as integers: a NaN ranks above everything and is not dropped
    auto note = [&](float f) {
        const uint32_t b = __builtin_bit_cast(uint32_t, f) & 0x7FFFFFFFu;
        amax_bits = b > amax_bits ? b : amax_bits;
    };
    if (in_regs) {
#pragma unroll
        for (int c = 0; c < STEPS; c++) { note(v[c].x); note(v[c].y); note(v[c].z); note(v[c].w); }
    } else {
        for (int i = threadIdx.x; i < k; i += blockDim.x) note(norm_w ? (xr[i] * inv) * norm_w[i] : xr[i]);
    }
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) {
        const uint32_t o = (uint32_t)__shfl_xor((int)amax_bits, s);
        amax_bits = o > amax_bits ? o : amax_bits;
    }
    if (lane == 0) red[wave] = __builtin_bit_cast(float, amax_bits);
    __syncthreads();
    uint32_t ab = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t o = __builtin_bit_cast(uint32_t, red[i]);
        ab = o > ab ? o : ab;
    }
    // amax in [2^e, 2^(e+1)) -> multiply by 2^(14 - e); inf/nan rows are passed through unscaled
    int eb = (int)((ab >> 23) & 0xFF);
    if (eb == 0 || eb == 0xFF) eb = 127 + 14;
    int sb = 127 + 14 - (eb - 127);
    sb = sb < 1 ? 1 : (sb > 254 ? 254 : sb);
    const float f = __builtin_bit_cast(float, (uint32_t)sb << 23);
    _Float16 *hi_row = xh + (size_t)(2 * row) * k, *lo_row = hi_row + k;
    // gemm_blk32_kernel's extras (callers ask for them only when the row fits the registers and k is a multiple of 64)
    _Float16 *hi3 = xs.xs3 ? xs.xs3 + (size_t)(2 * row) * xs.pitch : nullptr, *lo3 = hi3 ? hi3 + xs.pitch : nullptr;
    if (in_regs) {
#pragma unroll
        for (int c = 0; c < STEPS; c++) {
            const int i4 = c * 256 + threadIdx.x;
            if (c * 256 * 4 < k) { // uniform per step; with the extras k is a multiple of 32 and whole groups of eight threads are in
                const bool live = i4 * 4 < k;
                const float e[4] = {v[c].x * f, v[c].y * f, v[c].z * f, v[c].w * f};
                _Float16 h[4], l[4];
#pragma unroll
                for (int j = 0; j < 4; j++) { h[j] = (_Float16)e[j]; l[j] = (_Float16)(e[j] - (float)h[j]); }
                typedef _Float16 half4 __attribute__((ext_vector_type(4)));
                if (hi3) {
                    if (live) {
                        reinterpret_cast<half4 *>(hi_row)[i4] = half4{h[0], h[2], h[1], h[3]};
                        reinterpret_cast<half4 *>(lo_row)[i4] = half4{l[0], l[2], l[1], l[3]};
                    }
                    store_group_sum(((float)h[0] + (float)h[1]) + ((float)h[2] + (float)h[3]), live ? i4 >> 3 : k, k >> 5, hi3, xs);
                    store_group_sum(((float)l[0] + (float)l[1]) + ((float)l[2] + (float)l[3]), live ? i4 >> 3 : k, k >> 5, lo3, xs);
                } else if (live) {
                    reinterpret_cast<half4 *>(hi_row)[i4] = half4{h[0], h[1], h[2], h[3]};
                    reinterpret_cast<half4 *>(lo_row)[i4] = half4{l[0], l[1], l[2], l[3]};
                }
            }
        }
    } else {
        for (int i = threadIdx.x; i < k; i += blockDim.x) {
            const float e = (norm_w ? (xr[i] * inv) * norm_w[i] : xr[i]) * f;
            const _Float16 hi = (_Float16)e;
            hi_row[i] = hi;
            lo_row[i] = (_Float16)(e - (float)hi);
        }
    }
    if (hi3 && (int)threadIdx.x < xs.pitch - (k >> 8) * 32) { // the zeros that end a row
        hi3[(size_t)(k >> 8) * 32 + threadIdx.x] = (_Float16)0.f;
        lo3[(size_t)(k >> 8) * 32 + threadIdx.x] = (_Float16)0.f;
    }
    if (threadIdx.x == 0) {
        rowscale[2 * row] = 1.0f / f;
        rowscale[2 * row + 1] = 1.0f / f;
    }
}

} // namespace

// The context's GEMM scratch, grown to `need` bytes (work that still uses the old one is waited for first).
int axq_gemm_reserve(axq_ctx *ctx, size_t need) {
    if (ctx->gemm_scratch_bytes >= need) return AXQ_OK;
    const char *most = getenv("AXQ_GEMM_SCRATCH_MAX"); // development knob: as if the card had no room for more bytes than this
    if (most && need > strtoull(most, nullptr, 10))
        return axq_fail(ctx, AXQ_ERR_ALLOCATION_FAILED, "GEMM scratch of %zu bytes: beyond AXQ_GEMM_SCRATCH_MAX", need);
    AXQ_HIP(ctx, hipStreamSynchronize(ctx->stream), AXQ_ERR_DRIVER);
    if (ctx->gemm_scratch) (void)hipFree(ctx->gemm_scratch);
    ctx->gemm_scratch = nullptr;
    ctx->gemm_scratch_bytes = 0;
    AXQ_HIP(ctx, hipMalloc(&ctx->gemm_scratch, need), AXQ_ERR_ALLOCATION_FAILED);
    ctx->gemm_scratch_bytes = need;
    return AXQ_OK;
}

// y from the partial sums of a split K, on the context's stream (see gemm_reduce_kernel).
int axq_gemm_reduce(axq_ctx *ctx, const float *ypart, const float *rowscale, int rows, int n, int splits, float inv_ws, int row_mul,
                    const float *bias, const float *resid, float *y) {
    const size_t total4 = (size_t)rows * n / 4;
    decltype(&gemm_reduce_kernel<0>) kernel;
    switch (splits) {
    case 2: kernel = gemm_reduce_kernel<2>; break;
    case 3: kernel = gemm_reduce_kernel<3>; break;
    case 4: kernel = gemm_reduce_kernel<4>; break;
    case 5: kernel = gemm_reduce_kernel<5>; break;
    case 6: kernel = gemm_reduce_kernel<6>; break;
    case 7: kernel = gemm_reduce_kernel<7>; break;
    case 8: kernel = gemm_reduce_kernel<8>; break;
    default: kernel = gemm_reduce_kernel<0>; break;
    }
    kernel<<<(unsigned)((total4 + 255) / 256), 256, 0, ctx->stream>>>(ypart, rowscale, rows, n, splits, inv_ws, row_mul, bias, resid, y);
    AXQ_LAUNCH_CHECK(ctx, "gemm_reduce_kernel");
    return AXQ_OK;
}

namespace {

struct GemmPlan {
    int splits, steps_per_split, wm;
    bool q5;      // the one-MFMA kernel of the types with blocks of 32 (gemm_blk32_kernel)
    size_t xh_bytes, rs_bytes, part_bytes, xs3_bytes;
};

// Whether gemm_blk32_kernel takes this call.
bool q5_route(const axq_weight *w, bool in_regs_only) {
    static const bool off = getenv("AXQ_GEMM_BLK32") && getenv("AXQ_GEMM_BLK32")[0] == '0'; // development knob
    const bool type_ok = w->type == AXQ_Q4_0 || w->type == AXQ_Q4_1 || w->type == AXQ_Q5_0 || w->type == AXQ_Q5_1 || w->type == AXQ_Q8_0;
    return !off && type_ok && w->k % 256 == 0 && w->meta_pitch % 16 == 0 && (!in_regs_only || w->k <= 16 * 256 * 4);
}

// Split K when the output tiles alone leave most compute units idle (short prompts): the splits' partial sums go
// through scratch and are added in order by a second kernel.  Scratch (kept in the context, grown on demand):
// f16 activations [m, k] | row scales [m] | partial sums of a split K | block sums (gemm_blk32_kernel) | `extra` bytes for the caller.
int plan_gemm(axq_ctx *ctx, const axq_weight *w, int m, bool f32_rows, size_t extra, GemmPlan *p) {
    if (w->k % BK != 0)
        return axq_fail(ctx, AXQ_ERR_INVALID_BLOCK_SIZE, "Invalid block size: the prefill GEMM needs k %% 64 == 0, got %lld",
                        (long long)w->k);
    if (w->n_rows > INT32_MAX || w->k > INT32_MAX)
        return axq_fail(ctx, AXQ_ERR_SHAPE_MISMATCH, "Shape mismatch: weight dimensions exceed 2^31");
    static const int bm_knob = getenv("AXQ_GEMM_BM") ? atoi(getenv("AXQ_GEMM_BM")) : 0; // development knob: 128 or 256 for every shape of the two-plane kernel
    p->q5 = q5_route(w, f32_rows);
    const int bm = p->q5 ? PBM : bm_knob ? bm_knob : (m > 128 ? 256 : 128);
    p->wm = bm / 128;
    const long tiles = (long)((w->n_rows + BN - 1) / BN) * ((m + bm - 1) / bm);
    const int ksteps = (int)(w->k / BK), cus = ctx->prop.multiProcessorCount;
    int splits = (int)(cus / tiles);
    splits = splits > 8 ? 8 : splits;
    if (splits > ksteps / 4) splits = ksteps / 4;
    if (p->q5 || splits < 2 || w->n_rows % 4 != 0) splits = 1;
    p->steps_per_split = (ksteps + splits - 1) / splits;
    p->splits = (ksteps + p->steps_per_split - 1) / p->steps_per_split;
    // gemm_blk32_kernel reads whole row tiles without a clamp: its x buffers have rows up to a multiple of the tile
    const size_t mpad = p->q5 ? (size_t)(m + bm - 1) / bm * bm : (size_t)m;
    p->xh_bytes = axq_align_up(mpad * (size_t)w->k * 2, 256);
    p->rs_bytes = axq_align_up((size_t)m * 4, 256);
    p->part_bytes = axq_align_up(p->splits > 1 ? (size_t)p->splits * m * (size_t)w->n_rows * 4 : 0, 256);
    p->xs3_bytes = axq_align_up(p->q5 ? mpad * (size_t)xs3_pitch(w->k) * 2 : 0, 256);
    return axq_gemm_reserve(ctx, p->xh_bytes + p->rs_bytes + p->part_bytes + p->xs3_bytes + extra);
}

// What the x pre-pass has to write besides the rows (nothing for the two-plane kernel).
XSums plan_sums(axq_ctx *ctx, const axq_weight *w, const GemmPlan &p) {
    XSums xs = {nullptr, 0};
    if (p.q5) {
        xs.xs3 = reinterpret_cast<_Float16 *>(reinterpret_cast<uint8_t *>(ctx->gemm_scratch) + p.xh_bytes + p.rs_bytes + p.part_bytes);
        xs.pitch = xs3_pitch(w->k);
    }
    return xs;
}

template <int BITS, bool WITH_MIN>
int launch_blk32(axq_ctx *ctx, const GemmArgs &a) {
    static std::atomic<uint64_t> lds_allowed{0};
    constexpr size_t lds = (size_t)(3 * PBM * 64 + 2 * PBN * 64) * sizeof(_Float16) + 2 * PBN * 32; // three x stages, two weight stages, scale records
    if (int rc = axq_allow_lds(ctx, reinterpret_cast<const void *>(gemm_blk32_kernel<BITS, WITH_MIN>), lds_allowed, lds)) return rc;
    const unsigned tiles = (unsigned)(((a.n + PBN - 1) / PBN) * ((a.m + PBM - 1) / PBM));
    gemm_blk32_kernel<BITS, WITH_MIN><<<tiles, 512, lds, ctx->stream>>>(a);
    AXQ_LAUNCH_CHECK(ctx, "gemm_blk32_kernel");
    return AXQ_OK;
}

int launch_gemm_q5(axq_ctx *ctx, const GemmArgs &a, int type) {
    switch (type) {
    case AXQ_Q4_0: return launch_blk32<4, false>(ctx, a);
    case AXQ_Q4_1: return launch_blk32<4, true>(ctx, a);
    case AXQ_Q5_0: return launch_blk32<5, false>(ctx, a);
    case AXQ_Q5_1: return launch_blk32<5, true>(ctx, a);
    default: return launch_blk32<8, false>(ctx, a);
    }
}

// The GEMM proper over activations that already sit in scratch as scaled f16 rows.
int run_gemm(axq_ctx *ctx, const axq_weight *w, int m, const GemmPlan &p, float *y, bool pair = false, const float *bias = nullptr,
             const float *resid = nullptr) {
    uint8_t *base = reinterpret_cast<uint8_t *>(ctx->gemm_scratch);
    GemmArgs a;
    a.codes = w->codes; a.meta = w->meta; a.qh = w->qh;
    a.codes_pitch = w->codes_pitch; a.meta_pitch = w->meta_pitch; a.qh_pitch = w->qh_pitch;
    a.xh = reinterpret_cast<_Float16 *>(base); a.rowscale = reinterpret_cast<float *>(base + p.xh_bytes); a.y = y;
    a.ypart = p.splits > 1 ? reinterpret_cast<float *>(base + p.xh_bytes + p.rs_bytes) : nullptr;
    a.m = m; a.n = (int)w->n_rows; a.k = (int)w->k;
    a.steps_per_split = p.steps_per_split;
    a.pair = pair ? 1 : 0; a.bias = bias; a.resid = resid; a.wm = p.wm;
    const XSums xs = plan_sums(ctx, w, p);
    a.xs3 = xs.xs3; a.xs3_pitch = xs.pitch;
    if (p.q5) return launch_gemm_q5(ctx, a, w->type);
    switch (w->type) {
    case AXQ_Q4_0: return launch_gemm<GQ4x<false>>(ctx, a, p.splits);
    case AXQ_Q4_1: return launch_gemm<GQ4x<true>>(ctx, a, p.splits);
    case AXQ_Q5_0: return launch_gemm<GQ5x<false>>(ctx, a, p.splits);
    case AXQ_Q5_1: return launch_gemm<GQ5x<true>>(ctx, a, p.splits);
    case AXQ_Q8_0: return launch_gemm<GQ80>(ctx, a, p.splits);
    case AXQ_F16: return launch_gemm<GF16>(ctx, a, p.splits);
    case AXQ_F32: return launch_gemm<GF32>(ctx, a, p.splits);
    case AXQ_BF16: return launch_gemm<GBF16>(ctx, a, p.splits);
    default: return axq_fail(ctx, AXQ_ERR_INVALID_QUANT_TYPE, "Invalid quantization type: %d", w->type);
    }
}

} // namespace

int axq_dev_gemm_bf16(axq_ctx *ctx, const axq_weight *w, const uint16_t *x, int m, float *y) {
    if (axq_dev_rows_gemm_covers(ctx, w, m, true)) return axq_dev_rows_gemm(ctx, w, x, AXQ_ROWS_BF16, m, nullptr, 0.f, nullptr, nullptr, y);
    GemmPlan p;
    int rc;
    if ((rc = plan_gemm(ctx, w, m, false, 0, &p))) return rc;
    uint8_t *base = reinterpret_cast<uint8_t *>(ctx->gemm_scratch);
    gemm_prep_x_kernel<<<m, 256, 0, ctx->stream>>>(x, m, (int)w->k, reinterpret_cast<_Float16 *>(base),
                                                   reinterpret_cast<float *>(base + p.xh_bytes), plan_sums(ctx, w, p));
    return run_gemm(ctx, w, m, p, y);
}

bool axq_dev_gemm_f32_covers(const axq_weight *w, int m) {
    return w->k % BK == 0 && m >= 1 && m <= AXQ_GEMM_F32_MAX_ROWS && w->n_rows <= INT32_MAX && w->k <= INT32_MAX;
}

// y[m, n] = f(x)[m, k] W^T (+ bias[n]) (+ resid[m, n], which may be y) with f32 activations: each row goes through the
// matrix pipe as two adjacent f16 rows (2m rows in all), and the GEMM's epilogue adds the two results.  f = RMSNorm with weight norm_w
// when that is given.
int axq_dev_gemm_f32(axq_ctx *ctx, const axq_weight *w, const float *x, int m, const float *norm_w, float eps, const float *bias,
                     const float *resid, float *y) {
    return axq_dev_gemm_f32_ex(ctx, w, x, false, m, norm_w, eps, bias, resid, y);
}

// The same with f = SwiGLU when `swiglu`: x holds m rows of 2 k interleaved gate/up values (see the pre-pass).
bool axq_dev_gemm_f32_takes_swiglu(const axq_weight *w) { return w->k % 4 == 0 && w->k <= 16 * 256 * 4; }

int axq_dev_gemm_f32_ex(axq_ctx *ctx, const axq_weight *w, const float *x, bool swiglu, int m, const float *norm_w, float eps,
                        const float *bias, const float *resid, float *y) {
    GemmPlan p;
    int rc;
    if (swiglu && (norm_w || !axq_dev_gemm_f32_takes_swiglu(w)))
        return axq_fail(ctx, AXQ_ERR_INVALID_ARGUMENT, "axq_dev_gemm_f32_ex: SwiGLU rows need k %% 4 == 0, k <= 16384 and no norm");
    if (axq_dev_rows_gemm_covers(ctx, w, m, false))
        return axq_dev_rows_gemm(ctx, w, x, swiglu ? AXQ_ROWS_SWIGLU : AXQ_ROWS_F32, m, norm_w, eps, bias, resid, y);
    if ((rc = plan_gemm(ctx, w, 2 * m, true, 0, &p))) return rc;
    uint8_t *base = reinterpret_cast<uint8_t *>(ctx->gemm_scratch);
    _Float16 *xh = reinterpret_cast<_Float16 *>(base);
    float *rowscale = reinterpret_cast<float *>(base + p.xh_bytes);
    if (swiglu) gemm_prep_x_f32_kernel<true><<<m, 256, 0, ctx->stream>>>(x, nullptr, eps, m, (int)w->k, xh, rowscale, plan_sums(ctx, w, p));
    else gemm_prep_x_f32_kernel<false><<<m, 256, 0, ctx->stream>>>(x, norm_w, eps, m, (int)w->k, xh, rowscale, plan_sums(ctx, w, p));
    return run_gemm(ctx, w, 2 * m, p, y, true, bias, resid);
}
