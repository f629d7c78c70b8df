// Prefill-path quantized matmul: y[M, N] = x[M, K] (bf16) * W[N, K]^T, f32 accumulate and output, of plain f32 weights, some of f16 and bf16 ones
// and of blocks whose rows are no whole superblocks: packed types with K a multiple of 256 have kernels of their own (axq_gemm_rows.hip).
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

#include "axq_dense.h"
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
                        if (a.ypart) a.ypart[((size_t)blockIdx.y * a.m + gm) * axq_part_pitch(a.n) + gn] = acc[i][j][r];
                        else a.y[(size_t)gm * a.n + gn] = acc[i][j][r] * (a.rowscale[gm] * (1.0f / T::WS));
                    } else if ((r & 1) == 0) { // gm is even: this register and the next hold the two parts of row gm / 2
                        const size_t t = (size_t)(gm >> 1);
                        const float v = acc[i][j][r] + acc[i][j][r + 1];
                        if (a.ypart) {
                            a.ypart[((size_t)blockIdx.y * (a.m >> 1) + t) * axq_part_pitch(a.n) + gn] = v;
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

// bf16 rows -> f16 rows scaled by a power of two (largest magnitude below 2^15), and the scale to undo it.
__global__ void __launch_bounds__(256) gemm_prep_x_kernel(const uint16_t *x, int m, int k, _Float16 *xh, float *rowscale) {
    __shared__ float red[4];
    const int row = blockIdx.x;
    const uint16_t *xr = x + (size_t)row * k;
    uint32_t amax_bits = 0;
    for (int i4 = threadIdx.x; i4 < (k >> 2); i4 += blockDim.x) { // k is a multiple of 64
        const uint2 raw = reinterpret_cast<const uint2 *>(xr)[i4];
        const uint32_t b[4] = {raw.x & 0x7FFFu, raw.x >> 16 & 0x7FFFu, raw.y & 0x7FFFu, raw.y >> 16 & 0x7FFFu};
#pragma unroll
        for (int j = 0; j < 4; j++) amax_bits = b[j] > amax_bits ? b[j] : amax_bits;
    }
    float amax = __builtin_bit_cast(float, amax_bits << 16);
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) amax = fmaxf(amax, __shfl_xor(amax, s));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    // amax in [2^e, 2^(e+1)) -> multiply by 2^(14 - e); inf/nan rows are passed through unscaled
    int eb = (int)((__builtin_bit_cast(uint32_t, amax) >> 23) & 0xFF);
    if (eb == 0 || eb == 0xFF) eb = 127 + 14;
    int sb = 127 + 14 - (eb - 127);
    sb = sb < 1 ? 1 : (sb > 254 ? 254 : sb);
    const float f = __builtin_bit_cast(float, (uint32_t)sb << 23);
    typedef _Float16 half4 __attribute__((ext_vector_type(4)));
    for (int i4 = threadIdx.x; i4 < (k >> 2); i4 += blockDim.x) {
        const uint2 raw = reinterpret_cast<const uint2 *>(xr)[i4];
        const _Float16 h0 = (_Float16)(__builtin_bit_cast(float, raw.x << 16) * f), h1 = (_Float16)(__builtin_bit_cast(float, raw.x & 0xFFFF0000u) * f);
        const _Float16 h2 = (_Float16)(__builtin_bit_cast(float, raw.y << 16) * f), h3 = (_Float16)(__builtin_bit_cast(float, raw.y & 0xFFFF0000u) * f);
        reinterpret_cast<half4 *>(xh + (size_t)row * k)[i4] = half4{h0, h1, h2, h3};
    }
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
    const size_t i4 = (size_t)blockIdx.x * blockDim.x + threadIdx.x, quads = (size_t)axq_part_pitch(n) / 4, total4 = (size_t)rows * quads;
    if (i4 >= total4) return;
    const float4 first = reinterpret_cast<const float4 *>(ypart)[i4];
    float acc[4] = {first.x, first.y, first.z, first.w}, lost[4] = {0.f, 0.f, 0.f, 0.f}; // the sum, and what its additions rounded off (two-sum)
    constexpr int AHEAD = S > 0 ? S - 1 : 7;
    for (int s0 = 1; s0 < splits; s0 += AHEAD) {
        float4 v4[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; i++)
            if (s0 + i < splits) v4[i] = reinterpret_cast<const float4 *>(ypart)[(size_t)(s0 + i) * total4 + i4];
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
    typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
    const size_t row = i4 / quads, col = i4 % quads * 4, at = row * n + col;
    const float f = rowscale ? rowscale[row * row_mul] * inv_ws : inv_ws;
    if (col + 4 <= (size_t)n) {
        float4u out = {acc[0] * f, acc[1] * f, acc[2] * f, acc[3] * f};
        if (bias) out += *reinterpret_cast<const float4u *>(bias + col);
        if (resid) out += *reinterpret_cast<const float4u *>(resid + at);
        *reinterpret_cast<float4u *>(y + at) = out;
    } else {
        for (int c = 0; c < n % 4; c++) y[at + c] = (acc[c] * f + (bias ? bias[col + c] : 0.f)) + (resid ? resid[at + c] : 0.f);
    }
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
// FORM: the two f16 rows, or the addends of a row one behind the other, smallest first, so that few additions are of the total's size: two f16
// ones, or three bf16 ones (all 24 bits, and no scale).
enum { PREP_TWO_ROWS, PREP_TWO_F16, PREP_THREE_BF16 };
template <int FORM>
__device__ inline void put_addends(const float (&e)[4], _Float16 *to, int i4, int k) { // four elements from 4 i4 on of a row; `to`: its addends
    typedef _Float16 half4 __attribute__((ext_vector_type(4)));
    if constexpr (FORM == PREP_THREE_BF16) {
        uint32_t p[3][4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uint32_t b = __builtin_bit_cast(uint32_t, e[j]);
            const bool finite = (b & 0x7F800000u) != 0x7F800000u;
            if ((b & 0x7FFFFFFFu) > 0x7F800000u) b |= 0x00400000u; // what says that it is not a number may lie in the lower half
            const float hi = __builtin_bit_cast(float, b & 0xFFFF0000u), r = finite ? e[j] - hi : 0.f;
            const float mid = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, r) & 0xFFFF0000u);
            p[2][j] = b >> 16;
            p[1][j] = __builtin_bit_cast(uint32_t, mid) >> 16;
            p[0][j] = __builtin_bit_cast(uint32_t, r - mid) >> 16;
        }
#pragma unroll
        for (int a = 0; a < 3; a++) reinterpret_cast<uint2 *>(to + (size_t)a * k)[i4] = make_uint2(p[a][0] | p[a][1] << 16, p[a][2] | p[a][3] << 16);
    } else {
        _Float16 h[4], l[4];
#pragma unroll
        for (int j = 0; j < 4; j++) { h[j] = (_Float16)e[j]; l[j] = (_Float16)(e[j] - (float)h[j]); }
        constexpr bool FIRST = FORM == PREP_TWO_ROWS; // the leading bits' place
        reinterpret_cast<half4 *>(to + (FIRST ? 0 : k))[i4] = half4{h[0], h[1], h[2], h[3]};
        reinterpret_cast<half4 *>(to + (FIRST ? k : 0))[i4] = half4{l[0], l[1], l[2], l[3]};
    }
}
template <bool SWIGLU, int FORM>
__global__ void __launch_bounds__(256) gemm_prep_x_f32_kernel(const float *x, const float *norm_w, float eps, int m, int k,
                                                              _Float16 *xh, float *rowscale) {
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
    const float f = FORM == PREP_THREE_BF16 ? 1.0f : __builtin_bit_cast(float, (uint32_t)sb << 23);
    _Float16 *to = xh + (size_t)(FORM == PREP_THREE_BF16 ? 3 : 2) * row * k;
    if (in_regs) {
#pragma unroll
        for (int c = 0; c < STEPS; c++) {
            const int i4 = c * 256 + threadIdx.x;
            if (i4 * 4 < k) {
                const float e[4] = {v[c].x * f, v[c].y * f, v[c].z * f, v[c].w * f};
                put_addends<FORM>(e, to, i4, k);
            }
        }
    } else {
        for (int i4 = threadIdx.x; i4 * 4 < k; i4 += blockDim.x) { // k is a multiple of 64
            float e[4];
#pragma unroll
            for (int j = 0; j < 4; j++) e[j] = (norm_w ? (xr[4 * i4 + j] * inv) * norm_w[4 * i4 + j] : xr[4 * i4 + j]) * f;
            put_addends<FORM>(e, to, i4, k);
        }
    }
    if (FORM != PREP_THREE_BF16 && threadIdx.x == 0) {
        const int mul = FORM == PREP_TWO_ROWS ? 2 : 1;
        rowscale[mul * row] = 1.0f / f;
        if (mul == 2) rowscale[2 * row + 1] = 1.0f / f;
    }
}

} // namespace

// The context's GEMM scratch, grown to `need` bytes (work that still uses the old one is waited for first; not while the stream is captured, which the
// wait would spoil for good: the stream took no launch any more).
int axq_gemm_reserve(axq_ctx *ctx, size_t need) {
    if (ctx->gemm_scratch_bytes >= need) return AXQ_OK;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ctx->stream, &status) != hipSuccess || status != hipStreamCaptureStatusNone)
        return axq_fail(ctx, AXQ_ERR_ALLOCATION_FAILED, "GEMM scratch of %zu bytes: cannot grow while the stream is captured", need);
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
    const size_t total4 = (size_t)rows * (axq_part_pitch(n) / 4);
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
    size_t xh_bytes, rs_bytes, part_bytes;
};

// Split K when the output tiles alone leave most compute units idle (short prompts): the splits' partial sums go
// through scratch and are added in order by a second kernel.  Scratch (kept in the context, grown on demand):
// f16 activations [m, k] | row scales [m] | partial sums of a split K.
int plan_gemm(axq_ctx *ctx, const axq_weight *w, int m, GemmPlan *p) {
    if (w->k % BK != 0)
        return axq_fail(ctx, AXQ_ERR_INVALID_BLOCK_SIZE, "Invalid block size: the prefill GEMM needs k %% 64 == 0, got %lld",
                        (long long)w->k);
    if (w->n_rows > INT32_MAX || w->k > INT32_MAX)
        return axq_fail(ctx, AXQ_ERR_SHAPE_MISMATCH, "Shape mismatch: weight dimensions exceed 2^31");
    static const int bm_knob = getenv("AXQ_GEMM_BM") ? atoi(getenv("AXQ_GEMM_BM")) : 0; // development knob: 128 or 256 for every shape of the two-plane kernel
    const int bm = bm_knob ? bm_knob : (m > 128 ? 256 : 128);
    p->wm = bm / 128;
    const long tiles = (long)((w->n_rows + BN - 1) / BN) * ((m + bm - 1) / bm);
    const int ksteps = (int)(w->k / BK), cus = ctx->prop.multiProcessorCount;
    int splits = (int)(cus / tiles);
    splits = splits > 8 ? 8 : splits;
    if (splits > ksteps / 4) splits = ksteps / 4;
    if (splits < 2) splits = 1;
    p->steps_per_split = (ksteps + splits - 1) / splits;
    p->splits = (ksteps + p->steps_per_split - 1) / p->steps_per_split;
    p->xh_bytes = axq_align_up((size_t)m * (size_t)w->k * 2, 256);
    p->rs_bytes = axq_align_up((size_t)m * 4, 256);
    p->part_bytes = axq_align_up(p->splits > 1 ? (size_t)p->splits * m * (size_t)axq_part_pitch((int)w->n_rows) * 4 : 0, 256);
    const int rc = axq_gemm_reserve(ctx, p->xh_bytes + p->rs_bytes + p->part_bytes);
    if (rc == AXQ_OK || p->splits == 1 || w->n_rows % 4 == 0) return rc;
    (void)hipGetLastError(); // no room for parts of K: whole, as calls of so many columns always can
    p->splits = 1;
    p->steps_per_split = ksteps;
    p->part_bytes = 0;
    return axq_gemm_reserve(ctx, p->xh_bytes + p->rs_bytes);
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

namespace {

// 16-bit weights: rows of the weight's own type, no conversion and one product per weight and addend of x.  us, through the two planes and so:
//   bf16 rows   BF16 3394 x 4096, 42: 87.7 11.7; 471 x 4096, 1536: 152 22.4; 14336 x 3328, 2048: 473 179
//               F16 3674 x 4096, 187: 41.9 23.6; 14336 x 1280, 1672: 241 106; 7520 x 1856, 1278: 157 60
//   f32 rows    F16 4096 x 4096, 64: 24.4 19.4; 20000 x 4096, 64: 90.8 69.7; 20000 x 11008, 64: 220 279
//               BF16 1024 x 11008, 64: 40.1 28.1; 8192 x 2048, 64: 23.3 22.8; 4096 x 11008, 64: 41.1 55.7
// Few f32 rows against much of a weight stay with the planes: each addend reads the weight again.
bool covers16(const axq_weight *w, int m, bool f32) {
    if ((w->type != AXQ_BF16 && w->type != AXQ_F16) || w->k % BK != 0 || w->n_rows > INT32_MAX || w->k > INT32_MAX / 4) return false;
    return !f32 || m > 128 || w->n_rows * w->k <= (w->type == AXQ_F16 ? 128 << 20 : 17 << 20);
}

// Scratch: rows (`addends` times the caller's; 0: none) | row scales | partial sums of a split K.  Without room for the last, K whole.
struct Room16 { _Float16 *x; float *scale, *part; };
int room16(axq_ctx *ctx, const axq_weight *w, int m, int addends, Room16 *r) {
    const size_t xb = axq_align_up((size_t)m * (size_t)w->k * 2 * addends, 256), sb = addends ? axq_align_up((size_t)m * 4, 256) : 0;
    const size_t pb = axq_dense16_room(ctx, (int)w->n_rows, m, (int)w->k * (addends ? addends : 1)) * 4;
    int rc = axq_gemm_reserve(ctx, xb + sb + pb);
    const bool whole = rc != AXQ_OK && pb;
    if (whole) {
        (void)hipGetLastError();
        rc = axq_gemm_reserve(ctx, xb + sb);
    }
    uint8_t *base = reinterpret_cast<uint8_t *>(ctx->gemm_scratch);
    *r = {reinterpret_cast<_Float16 *>(base), reinterpret_cast<float *>(base + xb), whole || !pb ? nullptr : reinterpret_cast<float *>(base + xb + sb)};
    return rc;
}
axq_dense16 dense16_of(const axq_weight *w, int m, int addends, const void *x, float *y, const Room16 &r) {
    axq_dense16 d = {};
    d.w = w->codes; d.ldw = (int)(w->codes_pitch / 2); d.n = (int)w->n_rows; d.k = (int)w->k; d.m = m; d.parts = addends; d.half = w->type == AXQ_F16;
    d.x = x; d.y = y; d.part = r.part;
    return d;
}

} // namespace

int axq_dev_gemm_bf16(axq_ctx *ctx, const axq_weight *w, const uint16_t *x, int m, float *y) {
    if (covers16(w, m, false)) {
        const bool own_rows = w->type == AXQ_F16 || (reinterpret_cast<uintptr_t>(x) & 15) != 0; // the product takes 16 bytes at a time
        Room16 r;
        if (int rc = room16(ctx, w, m, own_rows, &r)) return rc;
        axq_dense16 d = dense16_of(w, m, 1, own_rows ? static_cast<const void *>(r.x) : x, y, r);
        if (d.half) {
            gemm_prep_x_kernel<<<m, 256, 0, ctx->stream>>>(x, m, (int)w->k, r.x, r.scale);
            d.unscale = r.scale;
        } else if (own_rows) {
            AXQ_HIP(ctx, hipMemcpyAsync(r.x, x, (size_t)m * (size_t)w->k * 2, hipMemcpyDeviceToDevice, ctx->stream), AXQ_ERR_COPY_FAILED);
        }
        return axq_dense16_gemm(ctx, d, !r.part);
    }
    if (axq_dev_rows_gemm_covers(w, m)) return axq_dev_rows_gemm(ctx, w, x, AXQ_ROWS_BF16, m, nullptr, 0.f, nullptr, nullptr, y);
    GemmPlan p;
    int rc;
    if ((rc = plan_gemm(ctx, w, m, &p))) return rc;
    uint8_t *base = reinterpret_cast<uint8_t *>(ctx->gemm_scratch);
    gemm_prep_x_kernel<<<m, 256, 0, ctx->stream>>>(x, m, (int)w->k, reinterpret_cast<_Float16 *>(base),
                                                   reinterpret_cast<float *>(base + p.xh_bytes));
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
                        const float *bias, const float *resid, float *y, axq_rows_chain *chain) {
    GemmPlan p;
    int rc;
    if (swiglu && (norm_w || !axq_dev_gemm_f32_takes_swiglu(w)))
        return axq_fail(ctx, AXQ_ERR_INVALID_ARGUMENT, "axq_dev_gemm_f32_ex: SwiGLU rows need k %% 4 == 0, k <= 16384 and no norm");
    if (axq_dev_rows_gemm_covers(w, m))
        return axq_dev_rows_gemm(ctx, w, x, swiglu ? AXQ_ROWS_SWIGLU : AXQ_ROWS_F32, m, norm_w, eps, bias, resid, y, chain);
    if (chain) {
        chain->ready_for = nullptr;
        chain->sums = {};
    }
    if (covers16(w, m, true)) {
        const bool half = w->type == AXQ_F16;
        Room16 r;
        if ((rc = room16(ctx, w, m, half ? 2 : 3, &r))) return rc;
        if (half && swiglu) gemm_prep_x_f32_kernel<true, PREP_TWO_F16><<<m, 256, 0, ctx->stream>>>(x, nullptr, eps, m, (int)w->k, r.x, r.scale);
        else if (half) gemm_prep_x_f32_kernel<false, PREP_TWO_F16><<<m, 256, 0, ctx->stream>>>(x, norm_w, eps, m, (int)w->k, r.x, r.scale);
        else if (swiglu) gemm_prep_x_f32_kernel<true, PREP_THREE_BF16><<<m, 256, 0, ctx->stream>>>(x, nullptr, eps, m, (int)w->k, r.x, r.scale);
        else gemm_prep_x_f32_kernel<false, PREP_THREE_BF16><<<m, 256, 0, ctx->stream>>>(x, norm_w, eps, m, (int)w->k, r.x, r.scale);
        axq_dense16 d = dense16_of(w, m, half ? 2 : 3, r.x, y, r);
        d.unscale = half ? r.scale : nullptr;
        d.bias = bias;
        d.resid = resid;
        return axq_dense16_gemm(ctx, d, !r.part);
    }
    if ((rc = plan_gemm(ctx, w, 2 * m, &p))) return rc;
    uint8_t *base = reinterpret_cast<uint8_t *>(ctx->gemm_scratch);
    _Float16 *xh = reinterpret_cast<_Float16 *>(base);
    float *rowscale = reinterpret_cast<float *>(base + p.xh_bytes);
    if (swiglu) gemm_prep_x_f32_kernel<true, PREP_TWO_ROWS><<<m, 256, 0, ctx->stream>>>(x, nullptr, eps, m, (int)w->k, xh, rowscale);
    else gemm_prep_x_f32_kernel<false, PREP_TWO_ROWS><<<m, 256, 0, ctx->stream>>>(x, norm_w, eps, m, (int)w->k, xh, rowscale);
    return run_gemm(ctx, w, 2 * m, p, y, true, bias, resid);
}
