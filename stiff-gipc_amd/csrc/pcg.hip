// Preconditioned conjugate gradients on the converted block system.
//
// Reference: S/linear_system/solver/pcg_solver.cu:158-267 (PCGSolver::pcg),
// dot products :8-150 (two-stage warp reduction + blocking cudaMemcpy per
// dot), vector updates :105-122; config pcg_solver.h:6-16.
//
// Here every scalar (rz, alpha, beta, the stop decision) lives in device
// memory: each producer of a dot product writes one partial per workgroup
// and every consumer workgroup sums the partials itself in a fixed order
// (deterministic, no atomics, no host round trip).  The iteration counter
// and the stop flag are device words too, so an iteration pair is a fixed
// launch sequence that is captured once into a HIP graph and replayed; the
// host only polls the stop flag every few iterations.  The iteration count
// and the iterate are those of the reference loop (stop test on the stale
// rz after the x/r update).
#include "spmv_sym.hpp"
#include "pcg_dev.hpp"
#include <atomic>
#include <chrono>
#include <thread>
#include <cmath>

namespace sgipc {
namespace {

constexpr int kThreads = 1024;    // workgroup size of the PCG kernels (16 waves)
constexpr int kRedBlocks = 1024;  // producers of dot partials use at most this many workgroups
constexpr int kCollectThreads = 256;  // MAS collect: one block row per thread, workgroups for every CU

// partial dot products of a.b, one per block (FP64 accumulation)
template <typename VA, typename VB>
__global__ void __launch_bounds__(kThreads) k_dot_part(long long N, const VA* __restrict__ a, const VB* __restrict__ b,
                                                       double* __restrict__ part, const int* __restrict__ ctrl) {
    if (ctrl && ctrl[C_STOP]) return;
    __shared__ double sh[kThreads / 64];
    double v = 0.0;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (long long)gridDim.x * blockDim.x)
        v += (double)a[i] * (double)b[i];
    write_partial(v, part, sh);
}

// scalar = sum of partials into sc[idx] (one block)
__global__ void __launch_bounds__(kThreads) k_store_sum(const double* __restrict__ part, int np, double* __restrict__ sc,
                                                        int idx) {
    __shared__ double sh[kThreads / 64];
    double s = sum_partials(part, np, sh);
    if (threadIdx.x == 0) sc[idx] = s;
}

// Direction update fused with the SpMV.  With beta = rz_(k-1) / rz_(k-2)
// (0 at k = 1): p_k = z + beta p_(k-1) and, by linearity,
// A p_k = A z + beta A p_(k-1), so the kernel gathers only z (symmetric
// SpMV over the upper BCOO + transposed references), forms p and Ap row by
// row in place, and writes per-workgroup partials of p.Ap.  First kernel of
// an iteration: enforces the iteration budget (iteration k runs while
// k < max_iter).
template <int G, typename MV, typename V>
__global__ void __launch_bounds__(kThreads) k_spmv_pap(int nb, const int* __restrict__ eptr, const int2* __restrict__ ent,
                                                       const MV* __restrict__ val, const V* __restrict__ z,
                                                       V* __restrict__ p, V* __restrict__ Ap,
                                                       const double* __restrict__ rz_last,
                                                       const double* __restrict__ rz_prev, int np_rz,
                                                       double* __restrict__ part, int* __restrict__ ctrl) {
    if (ctrl[C_STOP]) return;
    const int iter = ctrl[C_ITER];
    if (iter >= ctrl[C_MAXIT]) {
        if (blockIdx.x == 0 && threadIdx.x == 0) { ctrl[C_NOCONV] = 1; ctrl[C_STOP] = ctrl[C_MAXIT]; }
        return;
    }
    __shared__ double sh[2 * (kThreads / 64)];
    const bool first = iter == 1;
    double be = 0.0;
    if (!first) {
        double rn, ro;
        sum_partials2(rz_last, np_rz, rz_prev, np_rz, sh, rn, ro);
        be = rn / ro;
    }
    auto zv = [z](size_t i) { return z[i]; };
    constexpr int RPB = kThreads / G;
    const int nchunks = (nb + RPB - 1) / RPB;
    ChunkWalk w = xcd_chunks(nchunks);
    double contrib = 0.0;
    for (int ch = w.first; ch < w.end; ch += w.step) {
        int row = ch * RPB + threadIdx.x / G, sub = threadIdx.x % G;
        MV s0 = 0, s1 = 0, s2 = 0;
        if (row < nb) sym_row_lane<G, MV>(row, sub, eptr, ent, val, zv, s0, s1, s2);
        group_sum3<G, MV>(s0, s1, s2);  // every lane of the group holds the row sums
        if (sub < 3 && row < nb) {        // lane q forms component q
            const size_t o = 3 * (size_t)row + sub;
            const V aw = (V)(sub == 0 ? s0 : (sub == 1 ? s1 : s2));
            V pq, aq;
            if (first) {
                pq = z[o];
                aq = aw;
            } else {
                pq = (V)((double)z[o] + be * (double)p[o]);
                aq = (V)((double)aw + be * (double)Ap[o]);
            }
            p[o] = pq;
            Ap[o] = aq;
            contrib += (double)pq * (double)aq;
        }
    }
    write_partial(contrib, part, sh);
}

// alpha = rz / p.Ap ; x += alpha p ; r -= alpha Ap ; partials of r.r ; then
// the iteration counter advances (read again only by the next iteration's
// kernels and the stop tests, which report ctrl[C_ITER] - 1).
template <typename V>
__global__ void __launch_bounds__(kThreads) k_update_xr(long long N, double* __restrict__ x, V* __restrict__ r,
                                                        const V* __restrict__ p, const V* __restrict__ Ap,
                                                        const double* __restrict__ part_pap, int np_pap,
                                                        const double* __restrict__ part_rz, int np_rz,
                                                        double* __restrict__ part_rr, int* __restrict__ ctrl) {
    if (ctrl[C_STOP]) return;
    __shared__ double sh[2 * (kThreads / 64)];
    double rz, pap;
    sum_partials2(part_rz, np_rz, part_pap, np_pap, sh, rz, pap);
    double al = rz / pap;
    double v = 0.0;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (long long)gridDim.x * blockDim.x) {
        x[i] += al * (double)p[i];
        V ri = (V)((double)r[i] - al * (double)Ap[i]);
        r[i] = ri;
        v += (double)ri * (double)ri;
    }
    write_partial(v, part_rr, sh);
    if (blockIdx.x == 0 && threadIdx.x == 0) ctrl[C_ITER] += 1;
}

// Stop test, then z = sum_l Z_l[node_l(v)] on the MAS range, the 12x12
// block-Jacobi of the affine bodies on block rows < abd_rows (when abd_inv is
// set), identity elsewhere, and partials of r.z; one thread per block row.
// Bound by dependent round trips (two workgroups per CU at 137 k rows), so
// nothing waits that need not: the node ids, the stop test's partials and the
// residual are loaded before the stop word is looked at, and the two
// workgroup sums (stop test and r.z) share one barrier.  At 137 k block rows
// 7.6 -> 6.0 us per launch in FP32, 8.5 -> 7.0 us in FP64; 5.0 -> 4.3 us at 525.
template <typename V, typename T>
__global__ void __launch_bounds__(kCollectThreads) k_collect_dot(int nb, const V* __restrict__ r, V* __restrict__ z,
                                                          int sub_off, int n_mas, int L, const int* __restrict__ node_of,
                                                          const T* __restrict__ Z, const double* __restrict__ abd_inv,
                                                          int abd_rows, double* __restrict__ part_rz,
                                                          const double* __restrict__ part_rz_prev, int np_rz,
                                                          const double* __restrict__ part_rr, int np_rr,
                                                          double* __restrict__ sc, int* __restrict__ ctrl, int rule,
                                                          volatile int* hp, volatile double* hq) {
    __shared__ double sh[2 * (kCollectThreads / 64)];
    // node ids of a row's first kLevelBatch levels, and its residual
    int id[kLevelBatch];
    V rv[3];
    auto fetch = [&](int row) {
        const int vt = row - sub_off;
        const bool in = row < nb && vt >= 0 && vt < n_mas;
#pragma unroll
        for (int k = 0; k < kLevelBatch; ++k) id[k] = in && k < L ? node_of[(size_t)k * n_mas + vt] : 0;
        if (row < nb) load_x3(r, row, rv);
    };
    int row = blockIdx.x * kCollectThreads + threadIdx.x;
    const int stopped = ctrl[C_STOP];
    Share<4, kCollectThreads> test;  // the stop test's partials (rule < 0: none)
    test.take(rule == 0 ? part_rz_prev : part_rr, rule == 0 ? np_rz : rule > 0 ? np_rr : 0);
    fetch(row);
    if (stopped) {
        if (hp && blockIdx.x == 0 && threadIdx.x == 0) publish_progress(ctrl, sc, hp, hq);
        return;
    }
    double v = 0.0;
    for (; row < nb; row += gridDim.x * kCollectThreads) {
        const V r0 = rv[0], r1 = rv[1], r2 = rv[2];
        V z0, z1, z2;
        const int vt = row - sub_off;
        if (vt >= 0 && vt < n_mas) {
            // levels eight at a time: all Z values are loaded before the sums
            // (kept in level order)
            T s0 = 0, s1 = 0, s2 = 0;
            for (int l0 = 0; l0 < L; l0 += kLevelBatch) {
                if (l0) {
#pragma unroll
                    for (int k = 0; k < kLevelBatch; ++k) id[k] = l0 + k < L ? node_of[(size_t)(l0 + k) * n_mas + vt] : 0;
                }
                T q[kLevelBatch][3];
#pragma unroll
                for (int k = 0; k < kLevelBatch; ++k)
                    if (l0 + k < L) load_x3(Z, id[k], q[k]);
#pragma unroll
                for (int k = 0; k < kLevelBatch; ++k)
                    if (l0 + k < L) { s0 += q[k][0]; s1 += q[k][1]; s2 += q[k][2]; }
            }
            z0 = (V)s0; z1 = (V)s1; z2 = (V)s2;
        } else if (row < abd_rows) {
            const int b = row >> 2, k = row & 3;
            const double* P = abd_inv + 144 * (size_t)b + 36 * k;  // rows 3k .. 3k+2 of the body inverse
            const V* rb = r + 12 * (size_t)b;
            double s0 = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll 2  // a full unroll's 36 loads in flight would set the whole kernel's register budget
            for (int j = 0; j < 12; ++j) {
                const double rj = (double)rb[j];
                s0 += P[j] * rj; s1 += P[12 + j] * rj; s2 += P[24 + j] * rj;
            }
            z0 = (V)s0; z1 = (V)s1; z2 = (V)s2;
        } else {
            z0 = r0; z1 = r1; z2 = r2;
        }
        const size_t o = 3 * (size_t)row;
        z[o] = z0; z[o + 1] = z1; z[o + 2] = z2;
        v += (double)r0 * (double)z0 + (double)r1 * (double)z1 + (double)r2 * (double)z2;
        fetch(row + gridDim.x * kCollectThreads);
    }
    constexpr int NW = kCollectThreads / 64;
    wave_sums_put(test.sum(), sh);
    wave_sums_put(v, sh + NW);
    __syncthreads();
    const bool stop = stop_test_sum(rule, wave_sums_total<NW>(sh), sc, ctrl);
    if (threadIdx.x != 0) return;
    // the thread that ran the test's writes publishes its outcome
    if (hp && blockIdx.x == 0) publish_progress(ctrl, sc, hp, hq);
    if (!stop) part_rz[blockIdx.x] = wave_sums_total<NW>(sh + NW);
}

// Stop test, then z = D^-1 r (block Jacobi) or z = r, and partials of r.z
template <typename V>
__global__ void __launch_bounds__(kThreads) k_simple_precond_dot(long long N, const V* __restrict__ r, V* __restrict__ z,
                                                                 const double* __restrict__ Dinv, double* __restrict__ part_rz,
                                                                 const double* __restrict__ part_rz_prev, int np_rz,
                                                                 const double* __restrict__ part_rr, int np_rr,
                                                                 double* __restrict__ sc, int* __restrict__ ctrl,
                                                                 int rule) {
    if (ctrl[C_STOP]) return;
    __shared__ double sh[kThreads / 64];
    double v = 0.0;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (long long)gridDim.x * blockDim.x) {
        V zi;
        if (Dinv) {
            long long b = i / 3;
            int p = (int)(i % 3);
            const double* D = Dinv + 9 * (size_t)b;
            zi = (V)(D[p] * (double)r[3 * b] + D[p + 3] * (double)r[3 * b + 1] + D[p + 6] * (double)r[3 * b + 2]);
        } else {
            zi = r[i];
        }
        z[i] = zi;
        v += (double)r[i] * (double)zi;
    }
    if (stop_test(rule, part_rz_prev, np_rz, part_rr, np_rr, sc, ctrl, sh)) return;
    write_partial(v, part_rz, sh);
}

// The same over the copy of both triangles (FullCopy): a workgroup takes a
// chunk of R consecutive block rows and reads their entries as one contiguous
// run, one entry per thread and load, whatever the rows' lengths; the products
// A_e z_e (three per entry) go to LDS, and every row component is then summed
// from there by g lanes (g a power of two that fills the workgroup: 1 for the
// largest chunks, whose lanes keep four running sums).
// Rows of this matrix have 7 or 19 entries (and more at contacts), so lanes
// per row leave half the lanes idle or take a third round; here every lane
// has an entry, the loads are contiguous, and the row pointers, the previous
// dots and the row's own z, p and Ap are in flight before them.
// Measured per launch against 8 lanes per row: at 137 k block rows FP32
// (70 MB) 20.3 -> 17.7 us, FP64 (134 MB; the upper BCOO has 68 MB, but a
// scattered 72-byte gather per transposed block) 37.3 -> 28.6 us, where a plain
// read of as many bytes takes about 12 and 21 us; at 525 block rows 8.9 ->
// 4.9 us.  Counted there: 81 MB and 155 MB past L2, 30 % and 24 % of the L2
// requests hit (the gathers of z), 14 and 11 wavefronts per CU on average over
// a launch, 8 % of the LDS cycles are bank conflicts.  Several entries in flight
// per thread were slower (more registers, fewer wavefronts): 21.3 and 22.6 us
// for two and four against 19.8 us.
constexpr int kFT = 256;          // threads
constexpr int kFRows = 72;        // block rows per chunk, at most (three components each, of 256 threads)
constexpr int kFRowsBodies = 24;  // the same with affine bodies
constexpr int kFBatch = 1024;     // entries per LDS batch
constexpr int kFChunks = 4096;    // workgroups (p.Ap partials), at most

template <typename V>
__global__ void __launch_bounds__(kFT) k_spmv_pap_full(int nb, int R, int nchunks, int g, const int* __restrict__ eptr,
                                                       const V* __restrict__ vf, const V* __restrict__ z,
                                                       V* __restrict__ p, V* __restrict__ Ap,
                                                       const double* __restrict__ rz_last,
                                                       const double* __restrict__ rz_prev, int np_rz,
                                                       double* __restrict__ part, int* __restrict__ ctrl) {
    __shared__ V prod[3 * kFBatch];
    __shared__ int er[kFRows + 1];
    __shared__ double sh[3 * kFT / 64];
    const int t = threadIdx.x, wv = t >> 6;
    const ChunkWalk w = xcd_chunks(nchunks);
    const int task = t / g, sub = t & (g - 1);  // this thread's row component of the chunk
    const int row = task / 3;
    // loads that depend on nothing: the first chunk's row pointers, the dots
    const int stopped = ctrl[C_STOP], iter = ctrl[C_ITER], maxit = ctrl[C_MAXIT];
    Share<4, kFT> rn, ro;
    rn.take(rz_last, np_rz);
    ro.take(rz_prev, np_rz);
    int ev = 0;
    if (w.first < w.end && t <= R) ev = eptr[min(w.first * R + t, nb)];
    if (stopped) return;
    if (iter >= maxit) {
        if (blockIdx.x == 0 && t == 0) { ctrl[C_NOCONV] = 1; ctrl[C_STOP] = maxit; }
        return;
    }
    const bool first = iter == 1;
    // the waves' sums meet at the first chunk's barrier
    wave_sums_put(rn.sum(), sh);
    wave_sums_put(ro.sum(), sh + kFT / 64);
    double be = 0.0, contrib = 0.0;
    for (int ch = w.first; ch < w.end; ch += w.step) {
        const int r0 = ch * R, nr = min(R, nb - r0);
        if (ch != w.first) {
            if (t <= R) ev = eptr[min(r0 + t, nb)];
            __syncthreads();  // every read of the previous chunk's er is done
        }
        if (t <= R) er[t] = ev;
        const bool mine = row < nr;
        const size_t o = 3 * (size_t)r0 + task;
        V zo = 0, po = 0, ao = 0;
        if (mine && sub == 0) {
            zo = z[o];
            if (!first) {
                po = p[o];
                ao = Ap[o];
            }
        }
        __syncthreads();
        if (!first && ch == w.first) be = wave_sums_total<kFT / 64>(sh) / wave_sums_total<kFT / 64>(sh + kFT / 64);
        const int e0 = er[0], e1 = er[nr];
        const int lo = mine ? er[row] : 0, hi = mine ? er[row + 1] : 0;
        V s0 = 0, s1 = 0, s2 = 0, s3 = 0;
        // batches start at a whole group of 64 entries; rows without triplets
        // can leave a chunk with no entry (e0 == e1), where there is none to clamp to
        for (int b0 = e0 < e1 ? e0 & ~63 : e1; b0 < e1; b0 += kFBatch) {
            // (an index outside the chunk's run is clamped to it; a wavefront
            // past the run does nothing)
#pragma unroll
            for (int j = 0; j < kFBatch / kFT; ++j) {
                if (b0 + j * kFT + 64 * wv >= e1) continue;
                V a[9], x[3];
                int c;
                FullCopy<V>::load(vf, max(e0, min(b0 + j * kFT + t, e1 - 1)), a, c);
                load_x3(z, c, x);
                V* pr = prod + 3 * (j * kFT + t);
                pr[0] = a[0] * x[0] + a[3] * x[1] + a[6] * x[2];
                pr[1] = a[1] * x[0] + a[4] * x[1] + a[7] * x[2];
                pr[2] = a[2] * x[0] + a[5] * x[1] + a[8] * x[2];
            }
            __syncthreads();
            if (mine) {
                const int last = min(hi, b0 + kFBatch), st = 3 * g;
                int e = lo + sub;
                if (e < b0) e += (b0 - e + g - 1) / g * g;
                const V* q = prod + 3 * (e - b0) + (task - 3 * row);
                for (; e + 3 * g < last; e += 4 * g, q += 4 * st) {  // four running sums
                    s0 += q[0];
                    s1 += q[st];
                    s2 += q[2 * st];
                    s3 += q[3 * st];
                }
                if (e < last) s0 += q[0];
                if (e + g < last) s1 += q[st];
                if (e + 2 * g < last) s2 += q[2 * st];
            }
            __syncthreads();
        }
        V aw = (s0 + s1) + (s2 + s3);
        for (int off = g >> 1; off > 0; off >>= 1) aw += __shfl_xor(aw, off, 64);
        if (mine && sub == 0) {
            V pq, aq;
            if (first) {
                pq = zo;
                aq = aw;
            } else {
                pq = (V)((double)zo + be * (double)po);
                aq = (V)((double)aw + be * (double)ao);
            }
            p[o] = pq;
            Ap[o] = aq;
            contrib += (double)pq * (double)aq;
        }
    }
    wave_sums_put(contrib, sh + 2 * kFT / 64);
    __syncthreads();
    if (t == 0) part[blockIdx.x] = wave_sums_total<kFT / 64>(sh + 2 * kFT / 64);
}

template <typename TD, typename TS>
__global__ void k_copy_cast(long long N, TD* __restrict__ dst, const TS* __restrict__ src) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (long long)gridDim.x * blockDim.x)
        dst[i] = (TD)src[i];
}

__global__ void k_axpy(long long N, double* __restrict__ y, double a, const double* __restrict__ x) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (long long)gridDim.x * blockDim.x)
        y[i] += a * x[i];
}


__global__ void k_ctrl_init(int* ctrl, int maxit) {
    ctrl[C_STOP] = 0;
    ctrl[C_ITER] = 1;
    ctrl[C_MAXIT] = maxit;
    ctrl[C_NOCONV] = 0;
    ctrl[C_PUB] = 0;
}

// Last kernel of a captured group of iterations: copies the stop and
// iteration words and the progress ratio to pinned host memory, then (after
// a system-scope fence) the publication count the host waits on.
__global__ void k_publish(int* __restrict__ ctrl, const double* __restrict__ sc, volatile int* hp,
                          volatile double* hq) {
    publish_progress(ctrl, sc, hp, hq);
}

__global__ void k_set_scalar(double* sc, int idx, double v) { sc[idx] = v; }

// rz0 = sum of the r.z partials; a zero rz0 (zero right-hand side) stops the
// loop before its first iteration, so x stays 0 (the reference would divide
// 0/0), with no host round trip: the caller reads rz0 with the final words.
__global__ void __launch_bounds__(kThreads) k_store_rz0(const double* __restrict__ part, int np,
                                                        double* __restrict__ sc, int* __restrict__ ctrl) {
    __shared__ double sh[kThreads / 64];
    const double s = sum_partials(part, np, sh);
    if (threadIdx.x == 0) {
        sc[S_RZ0] = s;
        if (s == 0.0) ctrl[C_STOP] = 1;
    }
}

__global__ void k_diag_inv(int K, const int* __restrict__ rows, const int* __restrict__ cols,
                           const double* __restrict__ vals, double* __restrict__ Dinv) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= K || rows[k] != cols[k]) return;
    const double* M = vals + 9 * (size_t)k;  // column-major
    double a = M[0], b = M[3], c = M[6], d = M[1], e = M[4], f = M[7], g = M[2], h = M[5], i = M[8];
    double A = e * i - f * h, Bq = -(d * i - f * g), C = d * h - e * g;
    double id = 1.0 / (a * A + b * Bq + c * C);
    double* R = Dinv + 9 * (size_t)rows[k];
    R[0] = A * id; R[3] = -(b * i - c * h) * id; R[6] = (b * f - c * e) * id;
    R[1] = Bq * id; R[4] = (a * i - c * g) * id; R[7] = -(a * f - c * d) * id;
    R[2] = C * id; R[5] = -(a * h - b * g) * id; R[8] = (a * e - b * d) * id;
}

// the affine-body block-Jacobi applies on the body rows below the MAS range
const double* abd_inv(const Ctx& c) {
    return (c.abd.inv_ready && c.sub_offset >= 4 * c.abd.nb) ? (const double*)c.abd.inv.p : nullptr;
}
int abd_rows(const Ctx& c) { return abd_inv(c) ? 4 * c.abd.nb : 0; }

int grid_for(long long N) {
    int g = div_up(N, kThreads);
    return g < 1 ? 1 : (g > kRedBlocks ? kRedBlocks : g);
}

// ---- the PCG engine --------------------------------------------------------
// Vectors of type V (double or float), matrix values MV, MAS data T.
template <typename V, typename MV, typename T>
struct Engine {
    Ctx& c;
    long long N;
    int gN, gS;
    V *r, *z, *p, *Ap;
    double* x;
    double *part_rz[2], *part_pap, *part_rr, *part_bb;
    double* sc;
    int* ctrl;
    const MV* val;
    bool mas;
    T *R, *Z;
    const double* Dinv;
    int rule;
    int maxit = 0;
    double tol_now = 0.0;  // tolerance of the current run (progress prediction)
    int gU = 1;  // workgroups (and r.r partials) of the x/r update
    int nRZ = 1; // r.z partials written by the preconditioner apply
    bool fused = false;  // MAS apply as one launch

    int G = 8;  // lanes per block row in the SpMV (4, 8 or 16)
    double rz0_h = 0.0;  // rz0 of the last run, read with its final words
    // copy of both triangles in entry order (null: the upper BCOO) and its
    // SpMV's chunks of rF block rows, nF of them, g lanes per row component
    const V* vfull = nullptr;
    int rF = 1, nF = 1, gF = 1;
    // Rows per chunk: at least 8, so that small systems spread over many
    // workgroups (one entry per thread), and more once there are 1920 chunks, 7.5
    // workgroups per CU (8 fit by registers in FP32, 6 in FP64), up to 72.  Per
    // launch, FP64 / FP32, the rule's own number first:
    //   1,331 rows:   8: 4.6 / 4.8 us, 4: 5.3 / 5.4, 32: 5.2 / 5.4, 72: 6.9 / 6.5
    //   19,683 rows: 11: 8.6 / 7.1, 16: 7.0 / 6.7, 32: 6.7 / 6.6, 72: 7.5 / 7.1
    //   43,904 rows: 23: 13.4 / 7.8, 32: 10.7 / 7.4, 48: 10.5 / 7.0, 72: 10.5 / 7.3
    //   137,842 rows: 72: 26.1 / 15.6, 42: 29.0 / 17.9, 54: 26.0 / 17.1, 64: 26.2 / 18.6, 85: 28.4 / 16.2
    //   265,302 rows: 72: 48.0 / 26.7, 48: 48.9 / 25.6, 64: 49.5 / 27.9, 85: 50.7 / 27.3
    // so it is within 4 % of the best at both ends, and up to 28 % off it in
    // FP64 between 20 k and 44 k rows, where larger chunks do better.  (Solves
    // without a preconditioner: the matrix stays in the Infinity Cache.)
    // The rows of affine bodies come first and have hundreds of entries (about 250
    // for 64 bodies in columns), and a chunk's entries pass through one workgroup a
    // batch at a time, its rows summed by g lanes: 72 such rows took longer than all
    // the others.  With bodies a chunk has at most 24 rows.  An iteration of FP64
    // / mixed, with 8, 16, 24, 32 and 72 rows: 214,477 rows, 64 bodies 135 / 76, 118
    // / 68, 114 / 65, 120 / 70 and 161 / 98 us; 106,117 rows 62 / 49, 55 / 43, 53 /
    // 45, 54 / 43 and 69 / 56; 360,637 rows 207 / 140, 181 / 119, 175 / 119, 190 /
    // 129 and 272 / 201.
    void use_full(const V* vf) {
        vfull = vf;
        rF = std::max(8, std::min(c.abd.nb > 0 ? kFRowsBodies : kFRows, (int)div_up(c.nb, 1920)));
        nF = (int)div_up(c.nb, rF);
        gF = 1;
        while (gF < 64 && 2 * gF * 3 * rF <= kFT) gF *= 2;
        gS = std::min(kFChunks, std::max(8, (int)div_up(nF, 8) * 8));
    }
    // pinned progress words published by the MAS collect kernel (set while
    // the last iteration of a captured group is enqueued)
    volatile int* pub_h = nullptr;
    volatile double* pub_q = nullptr;
    static constexpr bool kFp32Mas = sizeof(T) == 4;

    // z = M^-1 r fused with the r.z partials (nRZ workgroups) and the stop test
    void precond_dot(double* rz_out, const double* rz_prev, int rule_now) {
        hipStream_t s = c.stream;
        if (mas) {
            if (fused) mas_solve_with_top(c, kFp32Mas, ctrl);
            else mas_bank_solve(c, kFp32Mas, ctrl);
            hipLaunchKernelGGL((k_collect_dot<V, T>), dim3(nRZ), dim3(kCollectThreads), 0, s, c.nb, r, z, c.sub_offset,
                               c.mas.n, c.mas.L, c.mas.node_of.p, (const T*)Z, abd_inv(c), abd_rows(c), rz_out,
                               rz_prev, nRZ, part_rr, gU, sc, ctrl, rule_now, pub_h, pub_q);
            SGIPC_LAUNCH_CHECK();
        } else {
            hipLaunchKernelGGL((k_simple_precond_dot<V>), dim3(gN), dim3(kThreads), 0, s, N, r, z, Dinv, rz_out,
                               rz_prev, nRZ, part_rr, gU, sc, ctrl, rule_now);
            SGIPC_LAUNCH_CHECK();
        }
    }

    // kernels of iteration k with parity par = k & 1
    void enqueue_iteration(int par) {
        hipStream_t s = c.stream;
        const SymBcoo& S = c.bsr;
        double* rz_last = part_rz[par ^ 1];  // rz_(k-1)
        double* rz_this = part_rz[par];      // holds rz_(k-2); receives rz_k
        prof_begin(c, PROF_SPMV);
        auto launch = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(gS), dim3(kThreads), 0, s, S.nb, S.eptr.p, S.ent.p, val, (const V*)z, p, Ap,
                               (const double*)rz_last, (const double*)rz_this, nRZ, part_pap, ctrl);
        };
        if (vfull) {
            hipLaunchKernelGGL((k_spmv_pap_full<V>), dim3(gS), dim3(kFT), 0, s, S.nb, rF, nF, gF, S.eptr.p, vfull,
                               (const V*)z, p, Ap, (const double*)rz_last, (const double*)rz_this, nRZ, part_pap, ctrl);
        } else if (G == 4) launch(k_spmv_pap<4, MV, V>);
        else if (G == 16) launch(k_spmv_pap<16, MV, V>);
        else launch(k_spmv_pap<8, MV, V>);
        SGIPC_LAUNCH_CHECK();
        prof_end(c, PROF_SPMV);
        if (mas) {
            mas_update_restrict(c, x, r, p, Ap, part_pap, gS, rz_last, nRZ, part_rr, ctrl, kFp32Mas, !fused);
        } else {
            hipLaunchKernelGGL((k_update_xr<V>), dim3(gN), dim3(kThreads), 0, s, N, x, r, (const V*)p, (const V*)Ap,
                               (const double*)part_pap, gS, (const double*)rz_last, nRZ, part_rr, ctrl);
            SGIPC_LAUNCH_CHECK();
        }
        precond_dot(rz_this, rz_last, rule);
    }

    // r holds the right-hand side, x the initial guess is zero.  rz0 stays on
    // the device (run() reads it with its final words into rz0_h; 0 means a
    // zero right-hand side, for which the loop stops at once).
    void init(double tol, int max_iter) {
        hipStream_t s = c.stream;
        maxit = max_iter;
        tol_now = tol;
        if (mas) {
            int g1, gx;
            mas_update_layout(c, g1, gx);
            gU = g1 + gx;
        } else {
            gU = gN;
        }
        fused = mas && mas_fused(c);
        // r.z partials: one per workgroup of the collect (256-thread
        // workgroups, so a system of ~100 k block rows spreads over every CU)
        // or of the simple preconditioner apply
        nRZ = mas ? std::max(1, std::min(div_up(c.nb, kCollectThreads), kRedBlocks)) : gN;
        hipLaunchKernelGGL(k_ctrl_init, dim3(1), dim3(1), 0, s, ctrl, max_iter);
        SGIPC_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_set_scalar, dim3(1), dim3(1), 0, s, sc, (int)S_TOL, tol);
        SGIPC_LAUNCH_CHECK();
        fill<double>(x, 0.0, N, s);
        hipLaunchKernelGGL((k_dot_part<V, V>), dim3(gN), dim3(kThreads), 0, s, N, r, r, part_bb, (const int*)nullptr);
        SGIPC_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_store_sum, dim3(1), dim3(kThreads), 0, s, part_bb, gN, sc, (int)S_BB);
        SGIPC_LAUNCH_CHECK();
        if (mas) mas_restrict(c, r, 3LL * c.sub_offset, kFp32Mas, ctrl, !fused);
        precond_dot(part_rz[0], part_rz[1], -1);
        hipLaunchKernelGGL(k_store_rz0, dim3(1), dim3(kThreads), 0, s, part_rz[0], nRZ, sc, ctrl);
        SGIPC_LAUNCH_CHECK();
    }

    size_t graph_key() const {
        GraphKey key;
        auto mix = [&](size_t v) { key.mix(v); };
        const SymBcoo& S = c.bsr;
        mix((size_t)N); mix((size_t)gN); mix((size_t)gS); mix((size_t)G); mix((size_t)rF); mix((size_t)nF); mix((size_t)gF); mix((size_t)gU); mix((size_t)S.nb); mix((size_t)S.K);
        mix((size_t)S.eptr.p); mix((size_t)S.ent.p); mix((size_t)val); mix((size_t)r); mix((size_t)z); mix((size_t)p);
        mix((size_t)Ap); mix((size_t)x); mix((size_t)part_rz[0]); mix((size_t)sc);
        mix((size_t)ctrl); mix((size_t)mas); mix((size_t)R); mix((size_t)Z); mix((size_t)Dinv); mix((size_t)rule);
        mix((size_t)c.sub_offset); mix((size_t)c.nb); mix((size_t)c.stream);
        mix((size_t)abd_inv(c)); mix((size_t)abd_rows(c)); mix((size_t)vfull);
        mix((size_t)fused); mix((size_t)nRZ);
        if (mas) key.mix(c.mas);
        return key.h;
    }

    static constexpr int kBigGroup = 8;  // iterations in the long captured group (even: parities repeat)

    // Capture n (even) iterations into a graph; with pinned polling the
    // group's last collect kernel (or k_publish) publishes the progress.
    hipGraphExec_t capture_group(int n, bool pinned, PinnedPoll& pp) {
        hipStream_t s = c.stream;
        hipGraph_t g = nullptr;
        SGIPC_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        try {
            for (int i = 0; i < n; ++i) {
                if (i == n - 1 && pinned && mas) {  // the group's last collect kernel publishes
                    pub_h = pp.d;
                    pub_q = reinterpret_cast<volatile double*>(pp.d + 8);
                }
                enqueue_iteration((i + 1) & 1);
            }
            pub_h = nullptr;
            pub_q = nullptr;
            if (pinned && !mas) {
                hipLaunchKernelGGL(k_publish, dim3(1), dim3(1), 0, s, ctrl, (const double*)sc, pp.d,
                                   reinterpret_cast<double*>(pp.d + 8));
                SGIPC_LAUNCH_CHECK();
            }
        } catch (...) {
            pub_h = nullptr;
            pub_q = nullptr;
            hipGraph_t dead = nullptr;
            (void)hipStreamEndCapture(s, &dead);
            if (dead) (void)hipGraphDestroy(dead);
            throw;
        }
        SGIPC_HIP(hipStreamEndCapture(s, &g));
        hipGraphExec_t exec = nullptr;
        hipError_t e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        SGIPC_HIP(e);
        return exec;
    }

    // Run iterations until the device stop flag is set; returns the
    // reference iteration count and whether it converged.
    int run(PcgGraph& gcache, int check_every, bool& converged) {
        hipStream_t s = c.stream;
        if (maxit <= 1) {  // no iteration fits the budget
            SGIPC_HIP(hipMemcpyAsync(&rz0_h, sc + S_RZ0, sizeof(double), hipMemcpyDeviceToHost, s));
            SGIPC_HIP(hipStreamSynchronize(s));
            converged = false;
            return maxit;
        }
        // profiling records events per kernel, which a captured graph cannot
        const bool use_graph = !c.prof.on;
        int pairs_per_check = std::max(1, check_every / 2);
        PinnedPoll& pp = c.pcg.poll;
        if (use_graph && !pp.h && !pp.failed) {
            void* hptr = nullptr;
            if (hipHostMalloc(&hptr, 64, hipHostMallocMapped | hipHostMallocCoherent) == hipSuccess) {
                void* dptr = nullptr;
                if (hipHostGetDevicePointer(&dptr, hptr, 0) == hipSuccess) {
                    pp.h = static_cast<int*>(hptr);
                    pp.d = static_cast<int*>(dptr);
                } else {
                    (void)hipHostFree(hptr);
                    pp.failed = true;
                }
            } else {
                pp.failed = true;
            }
            (void)hipGetLastError();
        }
        const bool pinned = use_graph && pp.h;
        if (use_graph) {
            size_t key = graph_key();
            if (!gcache.exec || gcache.key != key) {
                if (gcache.exec) { (void)hipGraphExecDestroy(gcache.exec); gcache.exec = nullptr; }
                if (gcache.exec_big) { (void)hipGraphExecDestroy(gcache.exec_big); gcache.exec_big = nullptr; }
                gcache.exec = capture_group(2, pinned, pp);
                if (pinned) gcache.exec_big = capture_group(kBigGroup, pinned, pp);
                gcache.key = key;
            }
        }
        int hc[C_NUM] = {0};
        if (pinned) {
            // Keep two groups of iterations queued ahead of the device and
            // follow its published progress in pinned memory: the device never
            // waits for the host, and at most two groups run past the stop
            // (their kernels read their first data and store nothing).  Groups are kBigGroup
            // iterations long (one graph launch and one publication per
            // group) while the convergence rate seen in the publications
            // predicts more than that many iterations to go, two iterations
            // near the stop, so few iterations run past it.
            volatile int* hp = pp.h;
            volatile double* hq = reinterpret_cast<volatile double*>(pp.h + 8);
            hp[0] = 0; hp[1] = 0; hp[2] = 0;
            std::atomic_thread_fence(std::memory_order_seq_cst);
            constexpr int kAhead = 2;
            int launched = 0, last_done = -1;
            long long launched_iters = 0;
            int k_prev = -1;
            double q_prev = 0.0, stop_pred = -1.0;  // predicted stopping iteration (< 0: none yet)
            auto last_change = std::chrono::steady_clock::now();
            for (;;) {
                const int done = hp[2];
                std::atomic_thread_fence(std::memory_order_acquire);
                if (done > 0 && hp[0] != 0) break;  // stopped (converged or budget)
                if (done != last_done && done > 0) {  // a new publication: update the prediction
                    const int k = hp[1] - 1;
                    const double q = hq[0];
                    if (k_prev >= 0 && k > k_prev && q > 0.0 && q_prev > q && tol_now > 0.0) {
                        const double rate = std::log(q / q_prev) / (double)(k - k_prev);  // < 0
                        stop_pred = (double)k + std::log(tol_now / q) / rate;
                    }
                    k_prev = k;
                    q_prev = q;
                }
                if (launched_iters < (long long)maxit + 2 && launched - done < kAhead) {
                    const bool big = gcache.exec_big &&
                                     (stop_pred < 0.0 || stop_pred - (double)launched_iters > kBigGroup + 2);
                    SGIPC_HIP(hipGraphLaunch(big ? gcache.exec_big : gcache.exec, s));
                    launched_iters += big ? kBigGroup : 2;
                    ++launched;
                    if (done != last_done) {
                        last_done = done;
                        last_change = std::chrono::steady_clock::now();
                    }
                    continue;
                }
                if (done >= launched) break;        // all launched groups ran, none stopped: budget used up
                if (done != last_done) {
                    last_done = done;
                    last_change = std::chrono::steady_clock::now();
                } else if (std::chrono::steady_clock::now() - last_change > std::chrono::seconds(2)) {
                    // no progress for 2 s: let the stream report its state
                    const hipError_t q = hipStreamQuery(s);
                    if (q != hipSuccess && q != hipErrorNotReady) SGIPC_HIP(q);
                    if (q == hipSuccess) break;     // idle: read the words below
                    last_change = std::chrono::steady_clock::now();
                }
#if defined(__x86_64__)
                __builtin_ia32_pause();
#else
                std::this_thread::yield();
#endif
            }
            SGIPC_HIP(hipMemcpyAsync(hc, ctrl, sizeof(int) * C_NUM, hipMemcpyDeviceToHost, s));
            SGIPC_HIP(hipMemcpyAsync(&rz0_h, sc + S_RZ0, sizeof(double), hipMemcpyDeviceToHost, s));
            SGIPC_HIP(hipStreamSynchronize(s));
        } else if (use_graph) {
            // Poll the stop word; after two polls the next one is placed where
            // the measured convergence rate predicts the stop (at most twice
            // the nominal interval ahead), so few polls are needed and few
            // iterations run past the stop.
            int npairs = pairs_per_check, k_prev = 0;
            double q_prev = 0.0, q = 0.0;
            for (;;) {
                for (int j = 0; j < npairs; ++j) SGIPC_HIP(hipGraphLaunch(gcache.exec, s));
                SGIPC_HIP(hipMemcpyAsync(hc, ctrl, sizeof(int) * C_NUM, hipMemcpyDeviceToHost, s));
                SGIPC_HIP(hipMemcpyAsync(&q, sc + S_PROG, sizeof(double), hipMemcpyDeviceToHost, s));
                SGIPC_HIP(hipMemcpyAsync(&rz0_h, sc + S_RZ0, sizeof(double), hipMemcpyDeviceToHost, s));
                SGIPC_HIP(hipStreamSynchronize(s));
                if (hc[C_STOP]) break;
                const int k = hc[C_ITER] - 1;  // iterations done; q is the ratio after iteration k
                npairs = pairs_per_check;
                if (k_prev > 0 && k > k_prev && q > 0.0 && q_prev > q && tol_now > 0.0) {
                    const double rate = std::log(q / q_prev) / (double)(k - k_prev);  // < 0
                    const double need = std::log(tol_now / q) / rate;                  // iterations left
                    npairs = std::max(1, std::min(2 * pairs_per_check, (int)std::ceil(need / 2.0)));
                }
                k_prev = k;
                q_prev = q;
            }
        } else {
            // timed (eager) mode: same batching; the event records of launches
            // after the stop (no work done) are dropped afterwards
            const size_t base_spmv = c.prof.pend[PROF_SPMV].size();
            const size_t base_mas = c.prof.pend[PROF_MAS_SOLVE].size();
            for (;;) {
                for (int q = 0; q < pairs_per_check; ++q) {
                    enqueue_iteration(1);
                    enqueue_iteration(0);
                }
                SGIPC_HIP(hipMemcpyAsync(hc, ctrl, sizeof(int) * C_NUM, hipMemcpyDeviceToHost, s));
                SGIPC_HIP(hipMemcpyAsync(&rz0_h, sc + S_RZ0, sizeof(double), hipMemcpyDeviceToHost, s));
                SGIPC_HIP(hipStreamSynchronize(s));
                if (hc[C_STOP]) break;
            }
            const size_t useful = (size_t)(hc[C_NOCONV] ? hc[C_STOP] - 1 : hc[C_STOP]);
            prof_drop_tail(c, PROF_SPMV, base_spmv + useful);
            if (mas) prof_drop_tail(c, PROF_MAS_SOLVE, base_mas + useful);
        }
        converged = hc[C_NOCONV] == 0;
        return hc[C_STOP];
    }
};

}  // namespace

void diag_build(Ctx& c) {
    if (!c.have_bcoo) throw state_error("diag preconditioner: convert first");
    double* D = c.pcg.Dinv.reserve(9 * (size_t)c.nb + 1);
    fill<double>(D, 0.0, 9LL * c.nb, c.stream);
    if (c.K > 0) {
        hipLaunchKernelGGL(k_diag_inv, dim3(div_up(c.K, 256)), dim3(256), 0, c.stream, c.K, c.t_rows, c.t_cols, c.t_vals, D);
        SGIPC_LAUNCH_CHECK();
    }
}

// z = M^-1 r with the configured preconditioner (standalone, outside PCG)
void precond_apply(Ctx& c, const double* r, double* z) {
    long long N = 3LL * c.nb;
    hipStream_t s = c.stream;
    if (c.precond_kind == 2 || c.precond_kind == 3) {
        long long off = 3LL * c.sub_offset, len = 3LL * c.mas.n;
        if (off > 0 || off + len < N) {
            hipLaunchKernelGGL((k_copy_cast<double, double>), dim3(grid_for(N)), dim3(kThreads), 0, s, N, z, r);
            SGIPC_LAUNCH_CHECK();
        }
        if (c.precond_kind == 2) mas_apply64(c, r + off, z + off);
        else mas_apply32(c, r + off, z + off);
        if (abd_inv(c)) abd_precond_apply(c, r, z);
        return;
    }
    double* part = c.pcg.partials.reserve(5 * kPart);
    int* ctrl = c.pcg.ctrl.reserve(C_NUM + 8);
    fill<int>(ctrl, 0, C_NUM, s);
    hipLaunchKernelGGL((k_simple_precond_dot<double>), dim3(grid_for(N)), dim3(kThreads), 0, s, N, r, z,
                       c.precond_kind == 1 ? (const double*)c.pcg.Dinv.p : (const double*)nullptr, part, part, 1, part,
                       1, (double*)nullptr, ctrl, -1);
    SGIPC_LAUNCH_CHECK();
}

// ||v||^2 into the device scalar sc[idx] (no host read)
static void device_norm2_to(Ctx& c, const double* v, long long N, double* part, double* sc, int idx) {
    hipStream_t s = c.stream;
    int g = grid_for(N);
    hipLaunchKernelGGL((k_dot_part<double, double>), dim3(g), dim3(kThreads), 0, s, N, v, v, part, (const int*)nullptr);
    SGIPC_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_store_sum, dim3(1), dim3(kThreads), 0, s, part, g, sc, idx);
    SGIPC_LAUNCH_CHECK();
}
// device scalars sc[i0] and sc[i1] to the host in one synchronisation
static void read_scalars(Ctx& c, const double* sc, int i0, int i1, double& a, double& b) {
    const int lo = std::min(i0, i1), hi = std::max(i0, i1);
    double h[16];
    SGIPC_HIP(hipMemcpyAsync(h, sc + lo, sizeof(double) * (hi - lo + 1), hipMemcpyDeviceToHost, c.stream));
    SGIPC_HIP(hipStreamSynchronize(c.stream));
    a = h[i0 - lo];
    b = h[i1 - lo];
}

void pcg_solve(Ctx& c, const double* b, double* x, const SolveOpts& o, SolveStats& st) {
    if (!c.have_bcoo) throw state_error("solve: convert first");
    if (!c.have_bsr) bsr_build(c);
    hipStream_t s = c.stream;
    const long long N = 3LL * c.nb;
    PcgWork& w = c.pcg;
    const bool mas = (c.precond_kind == 2 || c.precond_kind == 3);
    if (mas && !c.mas.ready) throw state_error("solve: MAS preconditioner not built");
    if (c.precond_kind == 1 && !w.Dinv.p) throw state_error("solve: block-Jacobi preconditioner not built");
    double* parts = w.partials.reserve(5 * kPart + kFChunks);
    double* sc = w.scal.reserve(S_NUM + 8);
    int* ctrl = w.ctrl.reserve(C_NUM + 8);
    const int max_iter = o.max_iter > 0 ? o.max_iter : (int)(o.max_iter_ratio * (double)N);
    const int gN = grid_for(N);
    // SpMV on the upper BCOO: chunks of kThreads / G block rows, a multiple of 8 workgroups (one range per XCD)
    const int G = c.spmv_group;
    const int nchunks = (int)div_up((long long)c.nb, kThreads / G);
    const int gS = std::min(kPart, std::max(8, (int)div_up(nchunks, 8) * 8));
    st.refinements = 0;
    if (o.precision == 0) {
        auto run64 = [&](auto tag) {
            using T = decltype(tag);
            const bool fp32mas = sizeof(T) == 4;
            Engine<double, double, T> E{c, N, gN, gS,
                                        w.r.reserve(N + 1), w.z.reserve(N + 1), w.p.reserve(N + 1),
                                        w.Ap.reserve(N + 1),
                                        x, {parts, parts + kPart}, parts + 5 * kPart, parts + 2 * kPart,
                                        parts + 3 * kPart, sc, ctrl, (const double*)c.t_vals, mas,
                                        mas ? (T*)(fp32mas ? (void*)c.mas.R32.p : (void*)c.mas.R64.p) : nullptr,
                                        mas ? (T*)(fp32mas ? (void*)c.mas.Z32.p : (void*)c.mas.Z64.p) : nullptr,
                                        c.precond_kind == 1 ? w.Dinv.p : nullptr, o.stop_rule};
            E.G = G;
            w.xw.reserve(N + 1);  // the true residual's, before the copy takes what is left
            if (const double* vf = bsr_full(c, double{})) E.use_full(vf);
            hipLaunchKernelGGL((k_copy_cast<double, double>), dim3(gN), dim3(kThreads), 0, s, N, E.r, b);
            SGIPC_LAUNCH_CHECK();
            E.init(o.tol, max_iter);
            bool conv = false;
            const int it = E.run(fp32mas ? w.graph32 : w.graph64, o.check_every, conv);
            st.rz0 = E.rz0_h;
            if (st.rz0 == 0.0) {
                // zero right-hand side: the loop stopped at once and x = 0 is
                // exact (the reference would divide 0/0)
                st.iterations = 0;
                st.converged = 1;
            } else {
                st.iterations = it;
                st.converged = conv ? 1 : 0;
            }
        };
        if (c.precond_kind == 3) run64(float{});
        else run64(double{});
    } else {
        // mixed precision: FP32 SpMV / MAS / Krylov vectors with FP64 dots,
        // outer iterative refinement on the FP64 true residual
        if (!mas && c.precond_kind != 0 && c.precond_kind != 1) throw arg_error("solve: unsupported preconditioner");
        float* rf = w.rf.reserve(N + 1);
        double* r64 = w.r64b.reserve(N + 1);
        double* d64 = w.d64.reserve(N + 1);
        Engine<float, float, float> E{c, N, gN, gS,
                                      rf, w.zf.reserve(N + 1), w.pf.reserve(N + 1),
                                      w.Apf.reserve(N + 1),
                                      d64, {parts, parts + kPart}, parts + 5 * kPart, parts + 2 * kPart,
                                      parts + 3 * kPart, sc, ctrl,
                                      c.spmv_full32 ? nullptr : bsr_values_f32(c),  // the full copy replaces it
                                      mas,
                                      mas ? c.mas.R32.p : nullptr, mas ? c.mas.Z32.p : nullptr,
                                      c.precond_kind == 1 ? w.Dinv.p : nullptr, 1};
        E.G = G;
        if (c.spmv_full32) E.use_full(bsr_full(c, float{}));
        fill<double>(x, 0.0, N, s);
        hipLaunchKernelGGL((k_copy_cast<double, double>), dim3(gN), dim3(kThreads), 0, s, N, r64, b);
        SGIPC_LAUNCH_CHECK();
        double* part_o = parts + 4 * kPart;
        // ||b||^2 stays on the device until the first true residual is read
        // with it (the first inner tolerance needs only ||r|| = ||b||)
        constexpr int S_B2 = S_NUM + 1;
        device_norm2_to(c, b, N, part_o, sc, S_B2);
        int total = 0;
        bool conv = false, have = false;  // have: rr, bb read from the device
        double bb = 0.0, rr = 0.0, bn = 0.0, rn = 0.0;  // rr: ||b - A x||^2 of the current x
        st.rz0 = 0.0;
        for (int outer = 0; outer < 50 && total < max_iter; ++outer) {
            if (have && (rn <= o.tol * bn || bn == 0.0)) { conv = true; break; }
            double eta = have ? std::max(0.9 * o.tol * bn / rn, o.inner_tol) : std::max(0.9 * o.tol, o.inner_tol);
            hipLaunchKernelGGL((k_copy_cast<float, double>), dim3(gN), dim3(kThreads), 0, s, N, rf, r64);
            SGIPC_LAUNCH_CHECK();
            E.init(eta, max_iter - total);
            bool c2 = false;
            int it = E.run(w.graph_mixed, o.check_every, c2);
            if (outer == 0) st.rz0 = E.rz0_h;
            if (E.rz0_h == 0.0) { conv = true; break; }  // the residual is zero: x is exact
            total += it;
            hipLaunchKernelGGL(k_axpy, dim3(gN), dim3(kThreads), 0, s, N, x, 1.0, (const double*)d64);
            SGIPC_LAUNCH_CHECK();
            // FP64 true residual r = b - A x
            hipLaunchKernelGGL((k_copy_cast<double, double>), dim3(gN), dim3(kThreads), 0, s, N, r64, b);
            SGIPC_LAUNCH_CHECK();
            spmv64(c, -1.0, x, 1.0, r64);
            device_norm2_to(c, r64, N, part_o, sc, S_NUM);
            read_scalars(c, sc, S_NUM, S_B2, rr, bb);
            have = true;
            rn = std::sqrt(rr);
            bn = std::sqrt(bb);
            st.refinements = outer + 1;
        }
        if (!have) {  // no residual computed (zero right-hand side or no budget): x = 0, r = b
            read_scalars(c, sc, S_B2, S_B2, bb, bb);
            rr = bb;
            rn = bn = std::sqrt(bb);
        }
        if (rn <= o.tol * bn) conv = true;
        st.iterations = total;
        st.converged = conv ? 1 : 0;
        // the refinement loop's last FP64 true residual is that of the final x
        st.rel_residual = bb > 0.0 ? std::sqrt(rr / bb) : std::sqrt(rr);
        return;
    }
    // true residual ||b - A x|| / ||b||, FP64
    double* tmp = w.xw.reserve(N + 1);
    hipLaunchKernelGGL((k_copy_cast<double, double>), dim3(gN), dim3(kThreads), 0, s, N, tmp, b);
    SGIPC_LAUNCH_CHECK();
    spmv64(c, -1.0, x, 1.0, tmp);
    // ||b||^2 is the init's S_BB (r held b); one read for both
    device_norm2_to(c, tmp, N, parts + 4 * kPart, sc, S_NUM);
    double rr = 0.0, bb = 0.0;
    read_scalars(c, sc, S_NUM, S_BB, rr, bb);
    st.rel_residual = bb > 0.0 ? std::sqrt(rr / bb) : std::sqrt(rr);
}

}  // namespace sgipc
