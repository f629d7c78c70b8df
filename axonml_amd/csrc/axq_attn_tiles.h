// What the attention kernels of described layers share: the layout of their f16 caches and of matrix-pipe tiles.
//
// Cache in f16: keys [kv_head][position][DP] (head size padded with zeros to 64, 128 or 256), values transposed,
// [kv_head][DVP][position] with positions 4..7 and 8..11 of every 16 exchanged (value_slot), so that both operands of a
// matrix-pipe tile are 16 contiguous bytes per lane.  In f32: keys and values row-major, products on the vector ALU.
#pragma once
#include <hip/hip_fp16.h>

#include "axq_dense.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef const __attribute__((address_space(1))) void gbl_void;
typedef __attribute__((address_space(3))) void lds_void;

constexpr int CHUNK = 64;          // positions per workgroup of a decode step
constexpr float PSCALE = 32768.0f; // weights enter the second product as f16 times this: (0, 1] stays normal down to 2^-29

inline int pad_dim(int d) { return d <= 64 ? 64 : (d <= 128 ? 128 : 256); }
inline int pad_cap(int cap) { return (cap + 63) / 64 * 64; }

__device__ inline _Float16 to_half(float f) { return (_Float16)fminf(fmaxf(f, -65504.f), 65504.f); }

// Where position p of a value row lies: bits 2 and 3 exchanged.
__device__ inline int value_slot(int p) { return (p & ~12) | ((p & 4) << 1) | ((p & 8) >> 1); }

// Row of a 32 x 32 accumulator's register r.
__device__ inline int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// Values of a prompt's rows into the transposed f16 cache through LDS: tiles of 32 positions and 32 elements of a kv head, position by position first, of 256
// threads each, so that both sides are runs of 64 bytes or more.
__host__ __device__ inline int value_tiles(int m, int vdim, int kv_heads) { return (m + 31) / 32 * ((vdim + 31) / 32) * kv_heads; }
__device__ inline void append_values(int i, const float *v, int ldv, int vdim, int m, int pos0, void *vc, int dvp, int capp) {
    __shared__ float tile[32][33];
    const int mt = (m + 31) / 32, vt = (vdim + 31) / 32;
    const int t0 = i % mt * 32, e0 = i / mt % vt * 32, h = i / (mt * vt), x = threadIdx.x & 31, y = threadIdx.x >> 5;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int j = y + r * 8;
        tile[j][x] = (t0 + j < m && e0 + x < vdim) ? v[(size_t)(t0 + j) * ldv + (size_t)h * vdim + e0 + x] : 0.f;
    }
    __syncthreads();
    _Float16 *o = reinterpret_cast<_Float16 *>(vc) + (size_t)h * dvp * capp;
    for (int j = y; j < 32; j += 8)
        if (e0 + j < vdim && t0 + x < m) o[(size_t)(e0 + j) * capp + value_slot(pos0 + t0 + x)] = to_half(tile[x][j]);
}

// Queries and keys of a prompt's rows on their way to f16, and the values, in one launch: the first workgroups take a tile of values each, the others four
// heads, a wave each, of four rows, whose elements are requested together (a workgroup for every row, and the values in a launch behind it, us: 16 heads of 128 on 4, 2000
// rows, rotated, 10.9 and 6.2, 20 heads normed by workgroups of a wave 15.0 and 6.5).
constexpr int PREP_ROWS = 4, PREP_CHUNKS = 4; // rows of a wave; 64 elements each of a head
inline int prep_groups(int heads) { return (heads + 3) / 4; }
inline unsigned prep_grid(int m, int heads, int values) { return (unsigned)(values + (m + PREP_ROWS - 1) / PREP_ROWS * prep_groups(heads)); }
// this wave's head and first row
__device__ inline void prep_place(int values, int heads, int &h, int &t0) {
    const int b = (int)blockIdx.x - values, groups = (heads + 3) / 4;
    h = b % groups * 4 + (threadIdx.x >> 6);
    t0 = b / groups * PREP_ROWS;
}
// x: the rows' heads, `ld` apart, zeros beyond their ends
__device__ inline void prep_load(const float *x, int ld, int dim, int t0, int m, float (&v)[PREP_ROWS][PREP_CHUNKS]) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int r = 0; r < PREP_ROWS; r++)
#pragma unroll
        for (int i = 0; i < PREP_CHUNKS; i++) {
            v[r][i] = 0.f;
            if (i * 64 < dim && t0 + r < m && i * 64 + lane < dim) v[r][i] = x[(size_t)(t0 + r) * ld + i * 64 + lane];
        }
}

} // namespace
