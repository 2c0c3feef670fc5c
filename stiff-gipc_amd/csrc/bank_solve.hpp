// MAS bank inverses in memory, and the bank solve by one wavefront.
//
// 32-vertex banks (96 rows): the upper triangle packed by rows.
//
// 16-vertex banks (48 rows): by cyclic diagonals.  Diagonal d holds
// c_d[i] = A(i, (i + d) mod 48), d = 0 .. 23 for every i and d = 24 for i < 24:
// with A symmetric, each entry once (1176, as a packed triangle has).  Lane i
// of a wavefront keeps its c_d in registers, read as 16-byte pieces (4 FP32, 2
// FP64 or 8 FP16 diagonals of one lane side by side, lanes next to each
// other), and row i of A r is
//   sum_d c_d[i] r[(i + d) mod 48] + sum_{d > 0} c_d[i - d] r[(i - d) mod 48]:
// the first sum reads r from LDS at a fixed offset per diagonal, the second
// comes from lane i - d.  Every LDS access is of consecutive words and its
// offset a constant, and the matrix is not staged there.  Counted at 10,359
// banks: no bank conflicts in FP64; 14 % of the LDS cycles in FP32, which
// fetches the second sum's terms by lane (ds_bpermute).  (From a packed triangle
// in LDS a row's elements lie at strides that change with the lane: 48 reads,
// each with its address, 2.4 us of latency per FP64 bank.)
#pragma once
#include "common.hpp"
#include <type_traits>

namespace sgipc {

// place of element (r, c), r <= c, of a D x D inverse stored in type S
template <int D, typename S>
__host__ __device__ inline int inv_index(int r, int c) {
    if constexpr (D == 48) {
        constexpr int V = 16 / (int)sizeof(S);
        const int d0 = c - r, d = d0 > 24 ? 48 - d0 : d0, i = d0 > 24 ? c : r;
        return d == 24 ? 24 * 48 + i : (d / V) * (48 * V) + i * V + d % V;
    } else {
        return r * (2 * D - r + 1) / 2 + (c - r);
    }
}

typedef float v4f __attribute__((ext_vector_type(4)));  // (float4 arrays in a struct end up in scratch memory)

// One 48 x 48 bank solve by one wavefront (T: arithmetic, S: storage): load()
// and load_r() issue every load and wait for none; solve() gives row `lane` of
// inv r (lane < 48).  lds: kBankLds values of this wavefront's own.
// S = half: inv = D S D with D = diag(sqrt(inv_ii)) (FP32, one per bank row)
// and S (unit diagonal, |S_ij| <= 1 for an SPD inverse) in FP16, 2352 + 192
// bytes a bank; z_i = d_i sum_j S_ij (d_j r_j), FP32 arithmetic.
constexpr int kBankLds = 192;
template <typename T, typename S>
struct BankSolve {
    static constexpr int D = 48, NP = D * (D + 1) / 2, V = 16 / (int)sizeof(S), NG = 24 / V;
    static constexpr bool H = sizeof(S) == 2;
    v4f q[NG];
    S last;
    T rv;
    float di;
    __device__ __forceinline__ void load(const void* __restrict__ inv, const float* __restrict__ dsc, int b, int lane) {
        const char* base = static_cast<const char*>(inv) + (size_t)b * (NP * sizeof(S));
        const int i = min(lane, D - 1);
#pragma unroll
        for (int g = 0; g < NG; ++g) q[g] = reinterpret_cast<const v4f*>(base)[g * D + i];
        last = reinterpret_cast<const S*>(base)[24 * D + min(lane, 23)];
        di = H ? dsc[(size_t)b * D + i] : 1.f;
    }
    __device__ __forceinline__ void load_r(const T* __restrict__ R, int b, int lane) {
        rv = R[(size_t)b * D + min(lane, D - 1)];
    }
    template <int K>
    __device__ __forceinline__ T elem() const {
        typedef S piece __attribute__((ext_vector_type(V)));
        return (T)__builtin_bit_cast(piece, q[K / V])[K % V];
    }
    // diagonal K: row `lane` gets c x[lane + K], row lane + K gets c r.  The
    // latter is added in LDS by FP64 atomics (consecutive words, in diagonal
    // order); FP32 ones run at a fraction of their rate (70 us instead of
    // 11 us for 10,359 banks), so FP32 fetches it from lane - K (from: its
    // byte address, mod 48) and adds it to acc2.
    __device__ __forceinline__ void term_of(T c, int K, T& acc, T& acc2, T* x, T* y, unsigned& from) const {
        acc += c * x[K];
        if (K == 0) return;
        if constexpr (sizeof(T) == 8) {
            (void)__hip_atomic_fetch_add(y + K, c * rv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        } else {
            from = min(from - 4u, from + 4u * (D - 1));
            acc2 += __int_as_float(__builtin_amdgcn_ds_bpermute((int)from, __float_as_int(c * rv)));
        }
    }
    template <int... K>
    __device__ __forceinline__ void terms(T& acc, T& acc2, T* x, T* y, unsigned& from,
                                          std::integer_sequence<int, K...>) const {
        (term_of(elem<K>(), K, acc, acc2, x, y, from), ...);
    }
    __device__ __forceinline__ static void wave_sync() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    __device__ __forceinline__ T solve(T* lds, int lane) {
        T *x = lds + lane, *y = lds + 2 * D + lane, acc = 0, acc2 = 0;
        if constexpr (H) rv *= di;
        if (lane < D) {
            x[0] = x[D] = rv;
            if constexpr (sizeof(T) == 8) y[0] = y[D] = (T)0;
        }
        wave_sync();
        if (lane < D) {
            unsigned from = 4u * (unsigned)lane;
            terms(acc, acc2, x, y, from, std::make_integer_sequence<int, 24>{});
            term_of(lane < 24 ? (T)last : (T)0, 24, acc, acc2, x, y, from);
        }
        if constexpr (sizeof(T) == 8) {
            wave_sync();
            if (lane < D) acc2 = y[0] + y[D];
        }
        acc += acc2;
        wave_sync();  // every lane's reads are done before the area is used again
        if constexpr (H) acc *= di;
        return acc;
    }
};

}  // namespace sgipc
