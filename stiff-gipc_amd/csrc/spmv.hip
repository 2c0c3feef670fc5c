// Symmetric block-3x3 SpMV  y = a A x + b y  on the upper BCOO resident in
// the triplet view, with the transposed-reference structure built here.
//
// Reference: S/linear_system/utils/spmv.cu:8-133.  The transposed half is
// gathered per row from a list of references to upper blocks instead of
// scattered with atomics, so each row is written once and the sum order is
// fixed.
#include "spmv_sym.hpp"

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/iterator/counting_iterator.hpp>

namespace sgipc {
namespace {

template <int G, typename TV, typename TX, typename TY>
__global__ void __launch_bounds__(256) k_spmv_sym(int nb, const int* __restrict__ eptr, const int2* __restrict__ ent,
                                                  const TV* __restrict__ vals, double a, const TX* __restrict__ x,
                                                  double b, TY* __restrict__ y) {
    constexpr int RPB = 256 / G;
    const int nchunks = (nb + RPB - 1) / RPB;
    ChunkWalk w = xcd_chunks(nchunks);
    for (int ch = w.first; ch < w.end; ch += w.step) {
        int row = ch * RPB + threadIdx.x / G, sub = threadIdx.x % G;
        TV s0 = 0, s1 = 0, s2 = 0;
        auto xv = [x](size_t i) { return x[i]; };
        if (row < nb) sym_row_lane<G, TV>(row, sub, eptr, ent, vals, xv, s0, s1, s2);
        group_sum3<G, TV>(s0, s1, s2);
        if (sub == 0 && row < nb) {
            size_t o = 3 * (size_t)row;
            if (b == 0.0) {
                y[o] = (TY)(a * s0); y[o + 1] = (TY)(a * s1); y[o + 2] = (TY)(a * s2);
            } else {
                y[o] = (TY)(a * s0 + b * (double)y[o]);
                y[o + 1] = (TY)(a * s1 + b * (double)y[o + 1]);
                y[o + 2] = (TY)(a * s2 + b * (double)y[o + 2]);
            }
        }
    }
}

// lower-reference counts per row: block (i, j), i < j, is referenced by row j
__global__ void k_low_count(int K, const int* __restrict__ r, const int* __restrict__ c, int* __restrict__ cnt) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= K) return;
    if (r[k] != c[k]) atomicAdd(cnt + c[k], 1);
}

// sort key of upper block k for the lower references: its column, or nb
// (after every column) for a diagonal block, which has none
__global__ void k_low_keys(int K, const int* __restrict__ r, const int* __restrict__ c, int nb,
                           unsigned* __restrict__ key) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= K) return;
    key[k] = r[k] == c[k] ? (unsigned)nb : (unsigned)c[k];
}

// references in (column, block index) order: block ids from the stable sort
__global__ void k_low_fill(int K, const int* __restrict__ nlow, const int* __restrict__ kk, const int* __restrict__ r,
                           int2* __restrict__ lref) {
    int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= K || q >= *nlow) return;
    const int k = kk[q];
    lref[q] = make_int2(k, r[k]);
}

// per-row entry list: transposed references, then the row's upper blocks
__global__ void k_entries(int nb, const int* __restrict__ lptr, const int2* __restrict__ lref,
                          const int* __restrict__ ustart, const int* __restrict__ ucol, int* __restrict__ eptr,
                          int2* __restrict__ ent) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j > nb) return;
    int base = lptr[j] + ustart[j];
    eptr[j] = base;
    if (j == nb) return;
    int nl = lptr[j + 1] - lptr[j];
    for (int e = 0; e < nl; ++e) ent[base + e] = lref[lptr[j] + e];
    for (int k = ustart[j]; k < ustart[j + 1]; ++k) ent[base + nl + (k - ustart[j])] = make_int2(k, ucol[k]);
}

// FP32 copy of the BCOO values, 12 floats per block: column q in lanes
// 4q .. 4q+2, lane 4q+3 zero
__global__ void k_to_f32(long long K, const double* __restrict__ s, float* __restrict__ d) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < K * kF32BlockStride;
         i += (long long)gridDim.x * blockDim.x) {
        const long long k = i / kF32BlockStride;
        const int e = (int)(i % kF32BlockStride), q = e >> 2, p = e & 3;
        d[i] = (p < 3) ? (float)s[9 * k + p + 3 * q] : 0.0f;
    }
}

// copy of both triangles in entry order (FullCopy): one thread per entry, so
// the stores are contiguous.  Entry (k, c) is block k transposed where c is
// the block's row and not its column.  Workgroups take entries in per-XCD
// ranges: the blocks that nearby rows share, once upright and once
// transposed, meet in one L2.
template <typename T>
__global__ void __launch_bounds__(256) k_full_copy(int nb, const int* __restrict__ eptr, const int2* __restrict__ ent,
                                                   const int* __restrict__ cols, const double* __restrict__ vals,
                                                   T* __restrict__ vf) {
    const int n = eptr[nb];
    const ChunkWalk w = xcd_chunks((n + 255) / 256);
    for (int ch = w.first; ch < w.end; ch += w.step) {
        const int e = ch * 256 + (int)threadIdx.x;
        if (e >= n) continue;
        const int2 q = ent[e];
        double a[9];
        load_block<double>(vals, q.x, cols[q.x] != q.y, a);
        T t[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) t[k] = (T)a[k];
        FullCopy<T>::store(vf, e, t, q.y);
    }
}

}  // namespace

// Build the transposed-reference structure for the BCOO now resident in the
// triplet view (rows/cols/vals [0, K)); uniq_start holds the row starts.
void bsr_build(Ctx& c) {
    if (!c.have_bcoo) throw state_error("bsr_build: convert first");
    hipStream_t s = c.stream;
    int nb = c.nb, K = c.K;
    SymBcoo& S = c.bsr;
    int* cnt = c.row_count.reserve((size_t)nb + 1);
    int* lptr = S.lptr.reserve((size_t)nb + 2);
    int* dint = c.dev_int.reserve(8);
    fill<int>(cnt, 0, nb, s);
    if (K > 0) {
        hipLaunchKernelGGL(k_low_count, dim3(div_up(K, 256)), dim3(256), 0, s, K, c.t_rows, c.t_cols, cnt);
        SGIPC_LAUNCH_CHECK();
    }
    exclusive_scan(c, cnt, lptr, nb, dint + 4, s);
    // the count of lower references (dint[4]) stays on the device: every
    // off-diagonal block has one, so K bounds it and sizes the buffers
    S.nb = nb;
    S.K = K;
    int2* lref = S.lref.reserve((size_t)K + 1);
    if (K > 0) {
        // the lower references of row j are the off-diagonal blocks of column
        // j, in block order (= row order): one stable radix sort by column
        int bc = 1;
        while ((1ll << bc) <= (long long)nb) ++bc;
        unsigned* key = S.lkey.reserve((size_t)K + 1);
        unsigned* key2 = S.lkey2.reserve((size_t)K + 1);
        int* kk = S.lidx.reserve((size_t)K + 1);
        hipLaunchKernelGGL(k_low_keys, dim3(div_up(K, 256)), dim3(256), 0, s, K, c.t_rows, c.t_cols, nb, key);
        SGIPC_LAUNCH_CHECK();
        if (c.sort_impl == SORT_OWN) {
            radix_sort_pairs(c, key, key2, nullptr, 0, kk, K, bc, s);
        } else {  // rocPRIM as the cross-check
            rocprim::counting_iterator<int> ids(0);
            size_t bytes = 0;
            SGIPC_HIP(rocprim::radix_sort_pairs(nullptr, bytes, key, key2, ids, kk, (size_t)K, 0, bc, s));
            char* tmp = S.ltmp.reserve(bytes + 1);
            SGIPC_HIP(rocprim::radix_sort_pairs((void*)tmp, bytes, key, key2, ids, kk, (size_t)K, 0, bc, s));
        }
        hipLaunchKernelGGL(k_low_fill, dim3(div_up(K, 256)), dim3(256), 0, s, K, (const int*)(dint + 4),
                           (const int*)kk, c.t_rows, lref);
        SGIPC_LAUNCH_CHECK();
    }
    int* eptr = S.eptr.reserve((size_t)nb + 2);
    int2* ent = S.ent.reserve(2 * (size_t)K + 1);
    hipLaunchKernelGGL(k_entries, dim3(div_up(nb + 1, 256)), dim3(256), 0, s, nb, (const int*)lptr,
                       (const int2*)lref, (const int*)c.uniq_start.p, (const int*)c.t_cols, eptr, ent);
    SGIPC_LAUNCH_CHECK();
    S.valf_ok = false;
    S.full32_ok = false;
    c.have_bsr = true;
}

// values of a copy: 2K bounds the entries (lower references + upper blocks; how
// many blocks lie on the diagonal only the device knows); whole groups of 64
template <typename T>
static size_t full_size(const SymBcoo& S) {
    return ((2 * (size_t)S.K + 63) / 64 + 1) * FullCopy<T>::kGroup;
}
template <typename T>
static void full_copy(Ctx& c, T* vf) {
    const SymBcoo& S = c.bsr;
    if (S.nb > 0 && S.K > 0) {
        const int blocks = 8 * std::max(1, std::min((int)div_up(2LL * S.K, 8 * 256), 1024));
        hipLaunchKernelGGL(k_full_copy<T>, dim3(blocks), dim3(256), 0, c.stream, S.nb, (const int*)S.eptr.p,
                           (const int2*)S.ent.p, (const int*)c.t_cols, (const double*)c.t_vals, vf);
        SGIPC_LAUNCH_CHECK();
    }
}
// Kept until the next convert: the mixed solves' refinement takes its residuals
// from the converted values themselves.
const float* bsr_full(Ctx& c, float) {
    if (!c.have_bsr) bsr_build(c);
    SymBcoo& S = c.bsr;
    float* vf = S.full32.reserve(full_size<float>(S));
    if (!S.full32_ok) full_copy(c, vf);
    S.full32_ok = true;
    return vf;
}
// Made anew by every solve: the values are the caller's, who may have written to
// them since (nothing else of an FP64 solve would notice).  Null where the upper
// blocks in place are the better choice, or where it does not fit (152 bytes per
// upper block).
const double* bsr_full(Ctx& c, double) {
    if (!fp64_on_copy(c)) return nullptr;
    if (!c.have_bsr) bsr_build(c);
    double* vf = c.bsr.full64.try_reserve(full_size<double>(c.bsr));
    if (vf) full_copy(c, vf);
    return vf;
}

// FP32 copy of the BCOO values for the mixed-precision solve
const float* bsr_values_f32(Ctx& c) {
    if (!c.have_bsr) bsr_build(c);
    SymBcoo& S = c.bsr;
    float* vf = S.valf.reserve((size_t)kF32BlockStride * S.K + 4);
    if (!S.valf_ok && S.K > 0) {
        long long n = (long long)kF32BlockStride * S.K;
        int g = (int)std::min<long long>(div_up(n, 256), 8192);
        hipLaunchKernelGGL(k_to_f32, dim3(g), dim3(256), 0, c.stream, (long long)S.K, (const double*)c.t_vals, vf);
        SGIPC_LAUNCH_CHECK();
    }
    S.valf_ok = true;
    return vf;
}

void spmv64(Ctx& c, double a, const double* x, double b, double* y) {
    if (!c.have_bsr) bsr_build(c);
    const SymBcoo& S = c.bsr;
    constexpr int G = 8;
    int nchunks = div_up((long long)S.nb, 256 / G);
    int blocks = std::max(8, (int)div_up(nchunks, 8) * 8);
    hipLaunchKernelGGL((k_spmv_sym<G, double, double, double>), dim3(blocks), dim3(256), 0, c.stream, S.nb, S.eptr.p,
                       S.ent.p, (const double*)c.t_vals, a, x, b, y);
    SGIPC_LAUNCH_CHECK();
}

}  // namespace sgipc
