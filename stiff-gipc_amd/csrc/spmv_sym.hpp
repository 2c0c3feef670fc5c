// Device side of the symmetric block-3x3 SpMV over the upper BCOO.
//
// Reference: S/linear_system/utils/spmv.cu:8-133 (upper BCOO, head-segmented
// warp row sums plus FP64 atomics for the transposed half).  Here a group of
// G lanes owns one block row j and sums, in a fixed order, the transposed
// references A(i,j)^T x_i (i < j) and then the row's own upper blocks
// A(j,k) x_k, both listed in one per-row entry array: no atomics,
// deterministic.  y = a A x + b y, the residuals and the FP64 batched solves
// read the values in place from the converted BCOO (9 doubles per block,
// column-major); the single-system PCG, and mixed batched solves, read a copy of
// both triangles in entry order (FullCopy below).
#pragma once
#include "context.hpp"

namespace sgipc {

// Rows are handled in chunks of (256 / G) rows.  The chunks are cut into 8
// contiguous ranges, one per XCD (consecutive workgroups are dispatched
// round-robin over the 8 XCDs), so the blocks a row references through the
// transpose -- blocks of nearby rows -- are usually still in that XCD's L2.
struct ChunkWalk {
    int first, step, end;
};
__device__ inline ChunkWalk xcd_chunks(int nchunks) {
    ChunkWalk w;
    int g = gridDim.x;
    if (g % 8 != 0) {
        w.first = blockIdx.x; w.step = g; w.end = nchunks;
        return w;
    }
    int per = g / 8, x = blockIdx.x % 8, loc = blockIdx.x / 8;
    int span = (nchunks + 7) / 8;
    w.first = x * span + loc;
    w.step = per;
    w.end = min((x + 1) * span, nchunks);
    return w;
}

// Block k of the value array, column-major a[p + 3q] = A(p, q), transposed
// in registers when tr.  FP64: the BCOO itself (72 B per block, 8-byte
// aligned), read as four 16-byte and one 8-byte load.  FP32: the padded copy
// (48 B per block, columns in float4 lanes 0-2), three aligned 16-byte loads.
typedef double double2_a8 __attribute__((ext_vector_type(2), aligned(8)));
constexpr int kF32BlockStride = 12;  // floats per block in the FP32 copy

template <typename TV>
__device__ inline void load_block(const TV* __restrict__ vals, int k, bool tr, TV a[9]);

template <>
__device__ inline void load_block<double>(const double* __restrict__ vals, int k, bool tr, double a[9]) {
    const double* A = vals + 9 * (size_t)k;
    const double2_a8* A2 = reinterpret_cast<const double2_a8*>(A);
    double2_a8 u0 = A2[0], u1 = A2[1], u2 = A2[2], u3 = A2[3];
    a[0] = u0.x; a[1] = u0.y; a[2] = u1.x; a[3] = u1.y; a[4] = u2.x; a[5] = u2.y; a[6] = u3.x; a[7] = u3.y;
    a[8] = A[8];
    if (tr) {  // a[p + 3q] <-> a[q + 3p]
        double t;
        t = a[1]; a[1] = a[3]; a[3] = t;
        t = a[2]; a[2] = a[6]; a[6] = t;
        t = a[5]; a[5] = a[7]; a[7] = t;
    }
}

template <>
__device__ inline void load_block<float>(const float* __restrict__ vals, int k, bool tr, float a[9]) {
    const float4* A4 = reinterpret_cast<const float4*>(vals + kF32BlockStride * (size_t)k);
    float4 c0 = A4[0], c1 = A4[1], c2 = A4[2];
    a[0] = c0.x; a[1] = c0.y; a[2] = c0.z; a[3] = c1.x; a[4] = c1.y; a[5] = c1.z; a[6] = c2.x; a[7] = c2.y;
    a[8] = c2.z;
    if (tr) {
        float t;
        t = a[1]; a[1] = a[3]; a[3] = t;
        t = a[2]; a[2] = a[6]; a[6] = t;
        t = a[5]; a[5] = a[7]; a[7] = t;
    }
}

// one block-times-vector term: block k (transposed when tr) times x_j
template <typename TV, typename XF>
__device__ inline void block_term(const TV* __restrict__ vals, int k, int j, bool tr, const XF& xv, TV& s0, TV& s1,
                                  TV& s2) {
    TV a[9];
    load_block<TV>(vals, k, tr, a);
    TV x0 = (TV)xv(3 * (size_t)j), x1 = (TV)xv(3 * (size_t)j + 1), x2 = (TV)xv(3 * (size_t)j + 2);
    s0 += a[0] * x0 + a[3] * x1 + a[6] * x2;
    s1 += a[1] * x0 + a[4] * x1 + a[7] * x2;
    s2 += a[2] * x0 + a[5] * x1 + a[8] * x2;
}

// Partial row sums of this lane (before the group reduction).  Row `row`
// owns entries ent[eptr[row] .. eptr[row+1]) = {upper block index, column}:
// first its transposed references (column < row), then its own upper
// blocks.  Lane `sub` takes entries sub, sub+G, ...  xv(i) returns entry i
// of the vector being multiplied.
template <int G, typename TV, typename XF>
__device__ inline void sym_row_lane(int row, int sub, const int* __restrict__ eptr, const int2* __restrict__ ent,
                                    const TV* __restrict__ vals, const XF& xv, TV& s0, TV& s1, TV& s2) {
    const int e0 = eptr[row] + sub, end = eptr[row + 1];
    int e = e0;
    // two entries in flight per lane for 4-byte values; 8-byte values would
    // cost occupancy (registers) for no gain
    if (sizeof(TV) == 4 && e + G < end) {
        int2 q0 = ent[e], q1 = ent[e + G];
        TV a[9], b[9];
        load_block<TV>(vals, q0.x, q0.y < row, a);
        load_block<TV>(vals, q1.x, q1.y < row, b);
        TV x0 = (TV)xv(3 * (size_t)q0.y), x1 = (TV)xv(3 * (size_t)q0.y + 1), x2 = (TV)xv(3 * (size_t)q0.y + 2);
        TV y0 = (TV)xv(3 * (size_t)q1.y), y1 = (TV)xv(3 * (size_t)q1.y + 1), y2 = (TV)xv(3 * (size_t)q1.y + 2);
        s0 += a[0] * x0 + a[3] * x1 + a[6] * x2;
        s1 += a[1] * x0 + a[4] * x1 + a[7] * x2;
        s2 += a[2] * x0 + a[5] * x1 + a[8] * x2;
        s0 += b[0] * y0 + b[3] * y1 + b[6] * y2;
        s1 += b[1] * y0 + b[4] * y1 + b[7] * y2;
        s2 += b[2] * y0 + b[5] * y1 + b[8] * y2;
        e += 2 * G;
    }
    for (; e < end; e += G) {
        int2 q = ent[e];
        block_term<TV>(vals, q.x, q.y, q.y < row, xv, s0, s1, s2);
    }
}

// Copy of both triangles in entry order: entry e of ent as its 3x3 block,
// transposed where it is a transposed reference, with its column.  Entries lie
// in groups of 64, the pieces of a group one after the other (64 pieces of 16
// bytes each, ..., the last element and the column), so that 64 lanes reading
// 64 consecutive entries read contiguous memory with every load: 40 bytes an
// entry in FP32, 76 in FP64.
typedef float f3_a4 __attribute__((ext_vector_type(3), aligned(4)));
typedef double d2_a8 __attribute__((ext_vector_type(2), aligned(8)));

template <typename T>
struct FullCopy;
template <>
struct FullCopy<float> {
    static constexpr int kGroup = 640;  // floats per group of 64 entries
    __device__ static inline void load(const float* __restrict__ vf, int e, float a[9], int& col) {
        const float* g = vf + (size_t)(e >> 6) * kGroup;
        const int l = e & 63;
        const float4 u = reinterpret_cast<const float4*>(g)[l], v = reinterpret_cast<const float4*>(g + 256)[l];
        const int2 w = reinterpret_cast<const int2*>(g + 512)[l];
        a[0] = u.x; a[1] = u.y; a[2] = u.z; a[3] = u.w; a[4] = v.x; a[5] = v.y; a[6] = v.z; a[7] = v.w;
        a[8] = __int_as_float(w.x);
        col = w.y;
    }
    __device__ static inline void store(float* __restrict__ vf, int e, const float a[9], int col) {
        float* g = vf + (size_t)(e >> 6) * kGroup;
        const int l = e & 63;
        reinterpret_cast<float4*>(g)[l] = make_float4(a[0], a[1], a[2], a[3]);
        reinterpret_cast<float4*>(g + 256)[l] = make_float4(a[4], a[5], a[6], a[7]);
        reinterpret_cast<int2*>(g + 512)[l] = make_int2(__float_as_int(a[8]), col);
    }
};
template <>
struct FullCopy<double> {
    static constexpr int kGroup = 608;  // doubles per group of 64 entries
    __device__ static inline void load(const double* __restrict__ vf, int e, double a[9], int& col) {
        const double* g = vf + (size_t)(e >> 6) * kGroup;
        const int l = e & 63;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const double2 u = reinterpret_cast<const double2*>(g + 128 * k)[l];
            a[2 * k] = u.x;
            a[2 * k + 1] = u.y;
        }
        a[8] = g[512 + l];
        col = reinterpret_cast<const int*>(g + 576)[l];
    }
    __device__ static inline void store(double* __restrict__ vf, int e, const double a[9], int col) {
        double* g = vf + (size_t)(e >> 6) * kGroup;
        const int l = e & 63;
#pragma unroll
        for (int k = 0; k < 4; ++k) reinterpret_cast<double2*>(g + 128 * k)[l] = make_double2(a[2 * k], a[2 * k + 1]);
        g[512 + l] = a[8];
        reinterpret_cast<int*>(g + 576)[l] = col;
    }
};
// the three components of block row c of a vector
__device__ inline void load_x3(const float* __restrict__ z, int c, float x[3]) {
    const f3_a4 v = *reinterpret_cast<const f3_a4*>(z + 3 * (size_t)c);
    x[0] = v.x; x[1] = v.y; x[2] = v.z;
}
__device__ inline void load_x3(const double* __restrict__ z, int c, double x[3]) {
    const d2_a8 v = *reinterpret_cast<const d2_a8*>(z + 3 * (size_t)c);
    x[0] = v.x; x[1] = v.y; x[2] = z[3 * (size_t)c + 2];
}

template <int G, typename TV>
__device__ inline void group_sum3(TV& s0, TV& s1, TV& s2) {
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) {
        s0 += __shfl_xor(s0, off, G);
        s1 += __shfl_xor(s1, off, G);
        s2 += __shfl_xor(s2, off, G);
    }
}

}  // namespace sgipc
