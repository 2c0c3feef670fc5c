// Batched PCG: many independent scenes concatenated into one converted
// system (scene s owns block rows [row_start[s], row_start[s+1]); no block
// couples two scenes), each scene running its own preconditioned conjugate
// gradients -- its own rz, alpha, beta and stop decision -- in the same
// kernel launches.  The MAS preconditioner is built once over the union: its
// banks aggregate connected nodes only, so it is block-diagonal per scene
// and each scene sees exactly its own preconditioner.
//
// Layout: block rows are cut into chunks that never straddle a scene (1024/G
// rows for the SpMV with G lanes per row); one workgroup per chunk writes one
// partial per dot product, and every wavefront that needs a scene's sum adds
// its partials in chunk order (deterministic, no FP atomics; the same value
// everywhere), so no launch only sums -- except where scenes have hundreds of
// chunks (kFoldWork).  A stopped scene's rows are left
// untouched by every later kernel.  The iteration sequence
//   SpMV (Ap, p.Ap) -> alpha; x, r update (r.r) -> MAS restrict + bank solve
//   -> collect (z, r.z) -> stop test, beta; p update
// is captured once into a HIP graph (several iterations per graph) and
// replayed until every scene has stopped.
//
// Per scene the arithmetic is the reference loop (PCGSolver::pcg,
// S/linear_system/solver/pcg_solver.cu:174-267): x0 = 0, stop rule 0 on the
// pre-update |rz| <= tol rz0, or rule 1 on ||r|| <= tol ||b||, iteration
// count as the reference's.  The reference has no batched solver.
#include "spmv_sym.hpp"
#include "pcg_dev.hpp"
#include <cmath>

namespace sgipc {
namespace {

constexpr int kBT = 256;       // threads of the row-wise batched kernels
constexpr int kScalT = 1024;   // the start-up scalars: one wave per scene, 16 scenes per workgroup

enum BPhase { B_INIT_BB = 0, B_INIT_RZ, B_SEGSUM };

__device__ inline double wave_sum_partials(const double* __restrict__ part, int lo, int hi) {
    const int lane = threadIdx.x & 63;
    double v = 0.0;
    for (int i = lo + lane; i < hi; i += 64) v += part[i];
    return __shfl(wave_sum(v), 0, 64);  // (the tree ends in the first lane)
}

// The same sum in the same order, sixteen partials of a lane in flight: for the
// one wavefront that sums a scene's partials for all of its chunks
__device__ inline double wave_sum_partials_ahead(const double* __restrict__ part, int lo, int hi) {
    constexpr int U = 16;
    const int lane = threadIdx.x & 63;
    double v = 0.0;
    for (int i = lo + lane; i < hi; i += 64 * U) {
        double q[U];
#pragma unroll
        for (int k = 0; k < U; ++k) q[k] = part[min(i + 64 * k, hi - 1)];
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (i + 64 * k < hi) v += q[k];
    }
    return __shfl(wave_sum(v), 0, 64);
}

// Sums of every scene's partials, one wavefront a scene (BEngine::fold)
__global__ void __launch_bounds__(64) k_bfold(const int* __restrict__ scene_chunk, const int* __restrict__ sstop,
                                              const double* __restrict__ pa, double* __restrict__ fa,
                                              const double* __restrict__ pb, double* __restrict__ fb,
                                              const int* __restrict__ ctrl) {
    const int s = blockIdx.x;
    if (ctrl[C_STOP] || sstop[s]) return;
    const int lo = scene_chunk[s], hi = scene_chunk[s + 1];
    const double a = wave_sum_partials_ahead(pa, lo, hi), b = pb ? wave_sum_partials_ahead(pb, lo, hi) : 0.0;
    if (threadIdx.x == 0) {
        fa[s] = a;
        if (pb) fb[s] = b;
    }
}

// Ap = A p on the chunk's rows, partial p.Ap per chunk
template <int G, typename MV, typename V>
__global__ void __launch_bounds__(1024) k_bspmv(const BatchChunk* __restrict__ chunk,
                                                const int* __restrict__ eptr, const int2* __restrict__ ent,
                                                const MV* __restrict__ val, const V* __restrict__ p,
                                                V* __restrict__ Ap, const int* __restrict__ sstop,
                                                double* __restrict__ part, const int* __restrict__ ctrl) {
    __shared__ double sh[1024 / 64];
    const BatchChunk c = chunk[blockIdx.x];
    if (ctrl[C_STOP] || sstop[c.scene]) return;
    const int r1 = c.r1;
    const int row = c.r0 + threadIdx.x / G, sub = threadIdx.x % G;
    auto pv = [p](size_t i) { return p[i]; };
    MV s0 = 0, s1 = 0, s2 = 0;
    if (row < r1) sym_row_lane<G, MV>(row, sub, eptr, ent, val, pv, s0, s1, s2);
    group_sum3<G, MV>(s0, s1, s2);
    double contrib = 0.0;
    if (sub < 3 && row < r1) {
        const size_t o = 3 * (size_t)row + sub;
        const V a = (V)(sub == 0 ? s0 : (sub == 1 ? s1 : s2));
        Ap[o] = a;
        contrib = (double)p[o] * (double)a;
    }
    write_partial(contrib, part, sh);
}

// The same over the row-contiguous FP32 copy of both triangles (mixed
// solves): the G lanes of a row stream consecutive entries; same entry
// order and products as k_bspmv, so the same sums.
template <int G>
__global__ void __launch_bounds__(1024) k_bspmv_full(const BatchChunk* __restrict__ chunk,
                                                     const int* __restrict__ eptr,
                                                     const float* __restrict__ vf,
                                                     const float* __restrict__ p, float* __restrict__ Ap,
                                                     const int* __restrict__ sstop, double* __restrict__ part,
                                                     const int* __restrict__ ctrl) {
    __shared__ double sh[1024 / 64];
    const BatchChunk c = chunk[blockIdx.x];
    if (ctrl[C_STOP] || sstop[c.scene]) return;
    const int r1 = c.r1;
    const int row = c.r0 + threadIdx.x / G, sub = threadIdx.x % G;
    float s0 = 0, s1 = 0, s2 = 0;
    if (row < r1) {
        const int end = eptr[row + 1];
        int e = eptr[row] + sub;
        auto madd = [&](const float a[9], const float x[3]) {
            s0 += a[0] * x[0] + a[3] * x[1] + a[6] * x[2];
            s1 += a[1] * x[0] + a[4] * x[1] + a[7] * x[2];
            s2 += a[2] * x[0] + a[5] * x[1] + a[8] * x[2];
        };
        float a[9], b[9], xa[3], xb[3];
        int ca, cb;
        for (; e + G < end; e += 2 * G) {  // two entries in flight
            FullCopy<float>::load(vf, e, a, ca);
            FullCopy<float>::load(vf, e + G, b, cb);
            load_x3(p, ca, xa);
            load_x3(p, cb, xb);
            madd(a, xa);
            madd(b, xb);
        }
        if (e < end) {
            FullCopy<float>::load(vf, e, a, ca);
            load_x3(p, ca, xa);
            madd(a, xa);
        }
    }
    group_sum3<G, float>(s0, s1, s2);
    double contrib = 0.0;
    if (sub < 3 && row < r1) {
        const size_t o = 3 * (size_t)row + sub;
        const float a = sub == 0 ? s0 : (sub == 1 ? s1 : s2);
        Ap[o] = a;
        contrib = (double)p[o] * (double)a;
    }
    write_partial(contrib, part, sh);
}

// x += alpha_s p ; r -= alpha_s Ap ; partial r.r per chunk.  Every wavefront
// sums its scene's partials of r.z and p.Ap for alpha; the scene's first chunk
// keeps the old r.z for k_bpupdate.  Bound by dependent round trips, like the
// two kernels below: the vectors are in flight while the partials are summed.
// (Where the scenes have too many chunks for that, fold_* hold the sums.)
// With alpha here and the stop test and beta in k_bpupdate, an iteration of 48
// scenes has six launches instead of eight: 49.4 -> 40.5 us.
template <typename V, bool FOLD>
__global__ void __launch_bounds__(kBT) k_bupdate(const BatchChunk* __restrict__ chunk, double* __restrict__ x,
                                                 V* __restrict__ r, const V* __restrict__ p, const V* __restrict__ Ap,
                                                 const double* __restrict__ part_rz,
                                                 const double* __restrict__ part_pap,
                                                 const double* __restrict__ fold_rz,
                                                 const double* __restrict__ fold_pap, double* __restrict__ rz,
                                                 const int* __restrict__ sstop, double* __restrict__ part,
                                                 int* __restrict__ ctrl) {
    __shared__ double sh[kBT / 64];
    const BatchChunk c = chunk[blockIdx.x];
    const int stopped = ctrl[C_STOP], ended = sstop[c.scene];
    const double rzv = FOLD ? fold_rz[c.scene] : wave_sum_partials(part_rz, c.c0, c.c1);
    const double pap = FOLD ? fold_pap[c.scene] : wave_sum_partials(part_pap, c.c0, c.c1);
    constexpr int U = 2;
    const long long i1 = 3LL * c.r1;
    long long i = 3LL * c.r0 + threadIdx.x;
    double xv[U];
    V rv[U], pv[U], av[U];
    auto take = [&]() {
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const long long j = min(i + k * kBT, i1 - 1);
            xv[k] = x[j];
            rv[k] = r[j];
            pv[k] = p[j];
            av[k] = Ap[j];
        }
    };
    take();
    if (stopped) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) ctrl[C_ITER] += 1;
    if (ended) return;
    const double al = rzv / pap;
    double v = 0.0;
    for (;;) {
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const long long j = i + k * kBT;
            if (j >= i1) break;
            x[j] = xv[k] + al * (double)pv[k];
            const V ri = (V)((double)rv[k] - al * (double)av[k]);
            r[j] = ri;
            v += (double)ri * (double)ri;
        }
        i += U * kBT;
        if (i - threadIdx.x >= i1) break;
        take();
    }
    write_partial(v, part, sh);
    if ((int)blockIdx.x == c.c0 && threadIdx.x == 0) rz[c.scene] = rzv;
}

// z = sum_l Z_l[node_l(v)] (MAS over all rows), partial r.z per chunk; every
// level's node, then every level's values, are loaded before any is used
template <typename V, typename T>
__global__ void __launch_bounds__(kBT) k_bcollect(const BatchChunk* __restrict__ chunk, const V* __restrict__ r,
                                                  V* __restrict__ z, int n, int L, const int* __restrict__ node_of,
                                                  const T* __restrict__ Z, const int* __restrict__ sstop,
                                                  double* __restrict__ part, const int* __restrict__ ctrl) {
    __shared__ double sh[kBT / 64];
    constexpr int kL = 6;  // levels, at most
    const BatchChunk c = chunk[blockIdx.x];
    if (ctrl[C_STOP] || sstop[c.scene]) return;
    double v = 0.0;
    for (int row = c.r0 + threadIdx.x; row < c.r1; row += kBT) {
        int g[kL];
#pragma unroll
        for (int l = 0; l < kL; ++l) g[l] = node_of[(size_t)min(l, L - 1) * n + row];
        const size_t o = 3 * (size_t)row;
        const V r0 = r[o], r1 = r[o + 1], r2 = r[o + 2];
        T q[kL][3];
#pragma unroll
        for (int l = 0; l < kL; ++l)
#pragma unroll
            for (int e = 0; e < 3; ++e) q[l][e] = Z[3 * (size_t)g[l] + e];
        T s0 = 0, s1 = 0, s2 = 0;
#pragma unroll
        for (int l = 0; l < kL; ++l)
            if (l < L) {
                s0 += q[l][0];
                s1 += q[l][1];
                s2 += q[l][2];
            }
        const V z0 = (V)s0, z1 = (V)s1, z2 = (V)s2;
        z[o] = z0; z[o + 1] = z1; z[o + 2] = z2;
        v += (double)r0 * (double)z0 + (double)r1 * (double)z1 + (double)r2 * (double)z2;
    }
    write_partial(v, part, sh);
}

struct BScal {
    double *bb, *rz, *rz0, *tol, *out;
    int *stop, *iters, *noconv;
};

constexpr int kCActive = C_NUM;      // scenes that have not stopped (after the shared C_* words)
constexpr int kCTicket = C_NUM + 1;  // workgroups of the start-up scalars done

// Stop test of the scene, then p = z + beta_s p.  Every wavefront takes the
// same decision from the same sums; the scene's first chunk writes it, and the
// last scene to stop sets the stop word.  (A chunk that starts later and sees
// its scene stopped would have left p alone as well.)
template <typename V, bool FOLD>
__global__ void __launch_bounds__(kBT) k_bpupdate(const BatchChunk* __restrict__ chunk, const V* __restrict__ z,
                                                  V* __restrict__ p, const double* __restrict__ part_rr,
                                                  const double* __restrict__ part_rz,
                                                  const double* __restrict__ fold_rr,
                                                  const double* __restrict__ fold_rz, BScal q, int rule,
                                                  int* __restrict__ ctrl) {
    const BatchChunk c = chunk[blockIdx.x];
    const int s = c.scene;
    const int stopped = ctrl[C_STOP], ended = q.stop[s], k = ctrl[C_ITER] - 1, maxit = ctrl[C_MAXIT];
    const double rr = FOLD ? fold_rr[s] : wave_sum_partials(part_rr, c.c0, c.c1);
    const double rzn = FOLD ? fold_rz[s] : wave_sum_partials(part_rz, c.c0, c.c1);
    const double rz = q.rz[s], tol = q.tol[s], ref = rule == 0 ? q.rz0[s] : q.bb[s];
    constexpr int U = 2;
    const long long i1 = 3LL * c.r1;
    long long i = 3LL * c.r0 + threadIdx.x;
    V zv[U], pv[U];
    auto take = [&]() {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long long j = min(i + u * kBT, i1 - 1);
            zv[u] = z[j];
            pv[u] = p[j];
        }
    };
    take();
    if (stopped || ended) return;
    const bool met = rule == 0 ? fabs(rz) <= tol * ref : sqrt(rr) <= tol * sqrt(ref);
    if (met || k + 1 >= maxit) {
        if ((int)blockIdx.x == c.c0 && threadIdx.x == 0) {
            q.iters[s] = met ? k : maxit;
            if (!met) q.noconv[s] = 1;
            q.stop[s] = 1;
            if (atomicSub(ctrl + kCActive, 1) == 1) ctrl[C_STOP] = 1;
        }
        return;
    }
    const double be = rzn / rz;
    for (;;) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long long j = i + u * kBT;
            if (j < i1) p[j] = (V)((double)zv[u] + be * (double)pv[u]);
        }
        i += U * kBT;
        if (i - threadIdx.x >= i1) break;
        take();
    }
}

// partials of a.b per chunk (all scenes)
template <typename VA, typename VB>
__global__ void __launch_bounds__(kBT) k_bdot(const BatchChunk* __restrict__ chunk, const VA* __restrict__ a,
                                              const VB* __restrict__ b, double* __restrict__ part) {
    __shared__ double sh[kBT / 64];
    const BatchChunk c = chunk[blockIdx.x];
    const long long i1 = 3LL * c.r1;
    double v = 0.0;
    for (long long i = 3LL * c.r0 + threadIdx.x; i < i1; i += kBT) v += (double)a[i] * (double)b[i];
    write_partial(v, part, sh);
}

// Per-scene sums outside the iterations: one wave per scene, 16 scenes per
// workgroup.  INIT_RZ counts the scenes that have work; the last workgroup to
// finish sets the stop word.
__global__ void __launch_bounds__(kScalT) k_bscalars(int phase, int S, const int* __restrict__ scene_chunk,
                                                     const double* __restrict__ pa, BScal q, int* __restrict__ ctrl) {
    __shared__ int act[kScalT / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int s = blockIdx.x * (kScalT / 64) + w;
    int active = 0;
    if (s < S) {
        const double v = wave_sum_partials(pa, scene_chunk[s], scene_chunk[s + 1]);
        if (lane == 0) {
            if (phase == B_SEGSUM) q.out[s] = v;
            if (phase == B_INIT_BB) q.bb[s] = v;
            if (phase == B_INIT_RZ) {
                q.rz[s] = v;
                q.rz0[s] = v;
                q.iters[s] = 0;
                q.noconv[s] = 0;
                if (v == 0.0 || q.bb[s] == 0.0) q.stop[s] = 1;  // zero right-hand side: x = 0 is exact
                if (!q.stop[s] && ctrl[C_MAXIT] <= 1) {        // no iteration fits the budget
                    q.stop[s] = 1;
                    q.iters[s] = ctrl[C_MAXIT];
                    q.noconv[s] = 1;
                }
                if (!q.stop[s]) active = 1;
            }
        }
    }
    if (phase != B_INIT_RZ) return;
    if (lane == 0) act[w] = active;
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
        for (int i = 0; i < kScalT / 64; ++i) tot += act[i];
        if (tot) atomicAdd(ctrl + kCActive, tot);
        __threadfence();
        if (atomicAdd(ctrl + kCTicket, 1) == (int)gridDim.x - 1) {  // last workgroup
            __threadfence();
            ctrl[kCTicket] = 0;
            ctrl[C_ITER] = 1;
            ctrl[C_STOP] = atomicAdd(ctrl + kCActive, 0) == 0 ? 1 : 0;
            ctrl[C_NOCONV] = 0;
        }
    }
}

__global__ void k_bctrl_init(int* ctrl, int maxit) {
    ctrl[C_STOP] = 0;
    ctrl[C_ITER] = 1;
    ctrl[C_MAXIT] = maxit;
    ctrl[C_NOCONV] = 0;
    ctrl[kCActive] = 0;
    ctrl[kCTicket] = 0;
}

template <typename TD, typename TS>
__global__ void k_bcast(long long N, TD* __restrict__ dst, const TS* __restrict__ src) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (long long)gridDim.x * blockDim.x)
        dst[i] = (TD)src[i];
}

__global__ void k_baxpy(long long N, double* __restrict__ y, const double* __restrict__ x) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (long long)gridDim.x * blockDim.x)
        y[i] += x[i];
}

// counts blocks whose row and column lie in different scenes
__global__ void k_coupling(int K, const int* __restrict__ rows, const int* __restrict__ cols,
                           const int* __restrict__ rs, int S, int* __restrict__ bad) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= K) return;
    auto scene_of = [&](int v) {
        int lo = 0, hi = S;  // largest s with rs[s] <= v
        while (hi - lo > 1) {
            int mid = (lo + hi) >> 1;
            if (rs[mid] <= v) lo = mid; else hi = mid;
        }
        return lo;
    };
    if (scene_of(rows[k]) != scene_of(cols[k])) atomicAdd(bad, 1);
}

int flat_grid(long long N) {
    long long g = div_up(N, 256);
    return (int)(g < 1 ? 1 : (g > 4096 ? 4096 : g));
}

template <typename V, typename MV, typename T>
struct BEngine {
    Ctx& c;
    BatchWork& w;
    long long N;
    int S, nch, G;
    V *r, *z, *p, *Ap;
    double* x;
    const MV* val;
    bool fp32mas;
    int rule;
    const float* vfull = nullptr;  // mixed: row-contiguous FP32 copy of both triangles (else the upper BCOO)

    // Per-scene sums by launches of their own instead of by every wavefront that
    // needs one (build_chunks decides; the same bits)
    double *fold_rz() { return w.fold_on ? w.fold.p : nullptr; }
    double *fold_pap() { return w.fold_on ? w.fold.p + S : nullptr; }
    double *fold_rr() { return w.fold_on ? w.fold.p + 2 * (size_t)S : nullptr; }
    void fold(const double* pa, double* fa, const double* pb, double* fb) {
        if (!w.fold_on) return;
        hipLaunchKernelGGL(k_bfold, dim3(S), dim3(64), 0, c.stream, (const int*)w.scene_chunk.p, (const int*)w.stop.p,
                           pa, fa, pb, fb, (const int*)w.ctrl.p);
        SGIPC_LAUNCH_CHECK();
    }

    BScal scal() {
        return BScal{w.bb.p, w.rz.p, w.rz0.p, w.tol.p, w.segout.p, w.stop.p, w.iters.p, w.noconv.p};
    }
    T* Rm() { return fp32mas ? (T*)(void*)c.mas.R32.p : (T*)(void*)c.mas.R64.p; }
    T* Zm() { return fp32mas ? (T*)(void*)c.mas.Z32.p : (T*)(void*)c.mas.Z64.p; }

    void scalars(int phase, const double* pa) {
        hipLaunchKernelGGL(k_bscalars, dim3(div_up(S, kScalT / 64)), dim3(kScalT), 0, c.stream, phase, S,
                           (const int*)w.scene_chunk.p, pa, scal(), w.ctrl.p);
        SGIPC_LAUNCH_CHECK();
    }

    void precond() {
        // z = M^-1 r over the union, then r.z partials per chunk
        const SceneSkip skip{w.bank_scene.p, w.stop.p};
        const bool fused = mas_fused(c);  // top-level restriction inside the bank-solve launch
        mas_restrict(c, r, 0, fp32mas, w.ctrl.p, !fused, skip);
        if (fused) mas_solve_with_top(c, fp32mas, w.ctrl.p, skip);
        else mas_bank_solve(c, fp32mas, w.ctrl.p, skip);
        hipLaunchKernelGGL((k_bcollect<V, T>), dim3(nch), dim3(kBT), 0, c.stream,
                           (const BatchChunk*)w.chunk.p, (const V*)r, z, c.mas.n, c.mas.L, (const int*)c.mas.node_of.p,
                           (const T*)Zm(), (const int*)w.stop.p, w.part_rz.p, (const int*)w.ctrl.p);
        SGIPC_LAUNCH_CHECK();
    }

    void iteration() {
        hipStream_t s = c.stream;
        const SymBcoo& B = c.bsr;
        auto launch = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(nch), dim3(1024), 0, s, (const BatchChunk*)w.chunk.p,
                               (const int*)B.eptr.p, (const int2*)B.ent.p, val,
                               (const V*)p, Ap, (const int*)w.stop.p, w.part_pap.p, (const int*)w.ctrl.p);
        };
        if constexpr (sizeof(MV) == 4 && sizeof(V) == 4) {
            if (vfull) {
                auto launchf = [&](auto kern) {
                    hipLaunchKernelGGL(kern, dim3(nch), dim3(1024), 0, s,
                                       (const BatchChunk*)w.chunk.p, (const int*)B.eptr.p, vfull,
                                       (const float*)p, (float*)Ap, (const int*)w.stop.p, w.part_pap.p,
                                       (const int*)w.ctrl.p);
                };
                if (G == 4) launchf(k_bspmv_full<4>);
                else if (G == 16) launchf(k_bspmv_full<16>);
                else launchf(k_bspmv_full<8>);
            }
        }
        if (!vfull) {
            if (G == 4) launch(k_bspmv<4, MV, V>);
            else if (G == 16) launch(k_bspmv<16, MV, V>);
            else launch(k_bspmv<8, MV, V>);
        }
        SGIPC_LAUNCH_CHECK();
        fold(w.part_pap.p, fold_pap(), nullptr, nullptr);
        auto update = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(nch), dim3(kBT), 0, s, (const BatchChunk*)w.chunk.p, x, r, (const V*)p,
                               (const V*)Ap, (const double*)w.part_rz.p, (const double*)w.part_pap.p,
                               (const double*)fold_rz(), (const double*)fold_pap(), w.rz.p, (const int*)w.stop.p,
                               w.part_rr.p, w.ctrl.p);
        };
        if (w.fold_on) update(k_bupdate<V, true>);
        else update(k_bupdate<V, false>);
        SGIPC_LAUNCH_CHECK();
        precond();
        fold(w.part_rr.p, fold_rr(), w.part_rz.p, fold_rz());
        auto direction = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(nch), dim3(kBT), 0, s, (const BatchChunk*)w.chunk.p, (const V*)z, p,
                               (const double*)w.part_rr.p, (const double*)w.part_rz.p, (const double*)fold_rr(),
                               (const double*)fold_rz(), scal(), rule, w.ctrl.p);
        };
        if (w.fold_on) direction(k_bpupdate<V, true>);
        else direction(k_bpupdate<V, false>);
        SGIPC_LAUNCH_CHECK();
    }

    // r = rhs (already in r), x = 0; per-scene tolerances and initial stop
    // flags are in w.tol / w.stop.  Computes bb, z, rz, rz0, p.
    void init(int maxit) {
        hipStream_t s = c.stream;
        hipLaunchKernelGGL(k_bctrl_init, dim3(1), dim3(1), 0, s, w.ctrl.p, maxit);
        SGIPC_LAUNCH_CHECK();
        fill<double>(x, 0.0, N, s);
        hipLaunchKernelGGL((k_bdot<V, V>), dim3(nch), dim3(kBT), 0, s, (const BatchChunk*)w.chunk.p,
                           (const V*)r, (const V*)r, w.part_rr.p);
        SGIPC_LAUNCH_CHECK();
        scalars(B_INIT_BB, w.part_rr.p);
        precond();
        scalars(B_INIT_RZ, w.part_rz.p);
        fold(w.part_rz.p, fold_rz(), nullptr, nullptr);
        hipLaunchKernelGGL((k_bcast<V, V>), dim3(flat_grid(N)), dim3(256), 0, s, N, p, (const V*)z);
        SGIPC_LAUNCH_CHECK();
    }

    size_t key(int per_graph) const {
        GraphKey k;
        auto mix = [&](size_t v) { k.mix(v); };
        const SymBcoo& B = c.bsr;
        mix((size_t)N); mix((size_t)S); mix((size_t)nch); mix((size_t)G); mix((size_t)per_graph);
        mix((size_t)rule); mix((size_t)r); mix((size_t)z); mix((size_t)p); mix((size_t)Ap); mix((size_t)x);
        mix((size_t)val); mix((size_t)fp32mas); mix((size_t)B.eptr.p); mix((size_t)B.ent.p); mix((size_t)B.nb);
        mix((size_t)vfull); mix((size_t)mas_fused(c));
        for (const void* q : {(const void*)w.chunk.p, (const void*)w.scene_chunk.p,
                              (const void*)w.part_pap.p, (const void*)w.part_rr.p, (const void*)w.part_rz.p,
                              (const void*)w.bb.p, (const void*)w.rz.p, (const void*)w.rz0.p, (const void*)w.tol.p, (const void*)w.segout.p,
                              (const void*)w.stop.p, (const void*)w.iters.p, (const void*)w.noconv.p,
                              (const void*)w.ctrl.p, (const void*)w.bank_scene.p,
                              (const void*)(w.fold_on ? w.fold.p : nullptr)})
            mix((size_t)q);
        mix((size_t)c.stream);
        k.mix(c.mas);
        return k.h;
    }

    void run(PcgGraph& gc, int per_graph) {
        hipStream_t s = c.stream;
        int hc[C_NUM] = {0};
        SGIPC_HIP(hipMemcpyAsync(hc, w.ctrl.p, sizeof(int) * C_NUM, hipMemcpyDeviceToHost, s));
        SGIPC_HIP(hipStreamSynchronize(s));
        if (hc[C_STOP]) return;
        size_t k = key(per_graph);
        if (!gc.exec || gc.key != k) {
            if (gc.exec) { (void)hipGraphExecDestroy(gc.exec); gc.exec = nullptr; }
            hipGraph_t g = nullptr;
            SGIPC_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
            try {
                for (int i = 0; i < per_graph; ++i) iteration();
            } catch (...) {
                hipGraph_t dead = nullptr;
                (void)hipStreamEndCapture(s, &dead);
                if (dead) (void)hipGraphDestroy(dead);
                throw;
            }
            SGIPC_HIP(hipStreamEndCapture(s, &g));
            hipError_t e = hipGraphInstantiate(&gc.exec, g, nullptr, nullptr, 0);
            (void)hipGraphDestroy(g);
            SGIPC_HIP(e);
            gc.key = k;
        }
        for (;;) {
            SGIPC_HIP(hipGraphLaunch(gc.exec, s));
            SGIPC_HIP(hipMemcpyAsync(hc, w.ctrl.p, sizeof(int) * C_NUM, hipMemcpyDeviceToHost, s));
            SGIPC_HIP(hipStreamSynchronize(s));
            if (hc[C_STOP]) break;
        }
    }
};

// per-scene sums of a chunk-partial array, to the host
void seg_to_host(Ctx& c, BatchWork& w, int S, const double* part, std::vector<double>& out) {
    hipLaunchKernelGGL(k_bscalars, dim3(div_up(S, kScalT / 64)), dim3(kScalT), 0, c.stream, (int)B_SEGSUM, S,
                       (const int*)w.scene_chunk.p, part,
                       BScal{w.bb.p, w.rz.p, w.rz0.p, w.tol.p, w.segout.p, w.stop.p, w.iters.p, w.noconv.p},
                       w.ctrl.p);
    SGIPC_LAUNCH_CHECK();
    out.resize(S);
    SGIPC_HIP(hipMemcpyAsync(out.data(), w.segout.p, sizeof(double) * S, hipMemcpyDeviceToHost, c.stream));
    SGIPC_HIP(hipStreamSynchronize(c.stream));
}

// Every wavefront of a scene sums the scene's partials itself, which saves two
// launches an iteration and costs reads in proportion to the square of the
// scene's chunks: with more than kFoldWork of those squares over all scenes the
// sums get their launches.  Sixty FP64 iterations, by every wavefront / by
// launches: 48 scenes of 18 k squares 4.36 / 4.62 ms; one scene of 112 k 3.37 /
// 3.28; 16 scenes of 233 k 14.8 / 15.0; one scene of 269 k 5.88 / 5.62, of 387 k
// 4.28 / 3.94, of 1.08 M 5.86 / 5.19, of 34.7 M (753,571 rows) 37.6 / 21.1; 256
// scenes of 1.05 M 41.7 / 41.1.
constexpr long long kFoldWork = 250000;

// chunk table: scenes cut into chunks of at most `rows` block rows
void build_chunks(Ctx& c, BatchWork& w, const std::vector<int>& rs, int rows) {
    const int S = (int)rs.size() - 1;
    std::vector<BatchChunk> chunk;
    std::vector<int> schunk(S + 1, 0);
    long long squares = 0;
    for (int s = 0; s < S; ++s) {
        const int c0 = (int)chunk.size(), c1 = c0 + (rs[s + 1] - rs[s] + rows - 1) / rows;
        schunk[s] = c0;
        squares += (long long)(c1 - c0) * (c1 - c0);
        for (int r0 = rs[s]; r0 < rs[s + 1]; r0 += rows)
            chunk.push_back(BatchChunk{r0, std::min(r0 + rows, rs[s + 1]), s, c0, c1});
    }
    const int nch = (int)chunk.size();
    schunk[S] = nch;
    w.nch = nch;
    w.fold_on = squares > kFoldWork;
    if (w.fold_on) w.fold.reserve(3 * (size_t)S);
    w.chunk.reserve(nch + 1);
    w.scene_chunk.reserve(S + 1);
    if (nch) SGIPC_HIP(hipMemcpy(w.chunk.p, chunk.data(), sizeof(BatchChunk) * nch, hipMemcpyHostToDevice));
    SGIPC_HIP(hipMemcpy(w.scene_chunk.p, schunk.data(), sizeof(int) * (S + 1), hipMemcpyHostToDevice));
    for (DBuf<double>* b : {&w.part_pap, &w.part_rr, &w.part_rz}) b->reserve(nch + 1);
}

}  // namespace

void batch_check_coupling(Ctx& c, const std::vector<int>& rs) {
    BatchWork& w = c.batch;
    const int S = (int)rs.size() - 1;
    int* d_rs = w.rstart.reserve((size_t)S + 1);
    int* bad = w.bad.reserve(1);
    SGIPC_HIP(hipMemcpyAsync(d_rs, rs.data(), sizeof(int) * (S + 1), hipMemcpyHostToDevice, c.stream));
    fill<int>(bad, 0, 1, c.stream);
    if (c.K > 0) {
        hipLaunchKernelGGL(k_coupling, dim3(div_up(c.K, 256)), dim3(256), 0, c.stream, c.K, (const int*)c.t_rows,
                           (const int*)c.t_cols, (const int*)d_rs, S, bad);
        SGIPC_LAUNCH_CHECK();
    }
    int h = 0;
    SGIPC_HIP(hipMemcpyAsync(&h, bad, sizeof(int), hipMemcpyDeviceToHost, c.stream));
    SGIPC_HIP(hipStreamSynchronize(c.stream));
    if (h) throw arg_error("solve_batched: " + std::to_string(h) + " matrix blocks couple two scenes");
}

void pcg_solve_batched(Ctx& c, int S, const int* h_row_start, const double* b, double* x, const SolveOpts& o,
                       SolveStats* st) {
    if (!c.have_bcoo) throw state_error("solve_batched: convert first");
    const bool mas = (c.precond_kind == 2 || c.precond_kind == 3);
    if (!mas || !c.mas.ready) throw state_error("solve_batched: needs a built MAS preconditioner");
    if (c.sub_offset != 0 || c.mas.n != c.nb)
        throw state_error("solve_batched: the MAS preconditioner must cover every block row");
    if (S <= 0) throw arg_error("solve_batched: no scenes");
    if (o.stop_rule != 0 && o.stop_rule != 1) throw arg_error("solve_batched: stop rule must be 0 or 1");
    std::vector<int> rs(h_row_start, h_row_start + S + 1);
    if (rs[0] != 0 || rs[S] != c.nb) throw arg_error("solve_batched: row_start must run from 0 to the block rows");
    for (int s = 0; s < S; ++s)
        if (rs[s + 1] < rs[s]) throw arg_error("solve_batched: row_start must be non-decreasing");
    if (!c.have_bsr) bsr_build(c);
    if (c.batch_persistent && c.mas.bank == 16) {
        batch_check_coupling(c, rs);
        pcg_solve_batched_persistent(c, S, rs, b, x, o, st);
        return;
    }
    hipStream_t s = c.stream;
    BatchWork& w = c.batch;
    const int G = c.spmv_group;
    build_chunks(c, w, rs, 1024 / G);
    batch_check_coupling(c, rs);
    batch_scene_maps(c, S, w.rstart.p, nullptr, nullptr);  // banks of stopped scenes are skipped
    for (DBuf<double>* q : {&w.bb, &w.rz, &w.rz0, &w.tol, &w.segout}) q->reserve(S + 1);
    for (DBuf<int>* q : {&w.stop, &w.iters, &w.noconv}) q->reserve(S + 1);
    w.ctrl.reserve(C_NUM + 8);
    const long long N = 3LL * c.nb;
    const int max_iter = o.max_iter > 0 ? o.max_iter : (int)(o.max_iter_ratio * (double)N);
    const int per_graph = std::max(1, c.batch_iters_per_graph);
    std::vector<int> hit(S), hnc(S), hstop(S, 0);
    std::vector<double> htol(S, o.tol);
    PcgWork& pw = c.pcg;
    for (int i = 0; i < S; ++i) st[i] = SolveStats{};
    if (o.precision == 0) {
        auto run64 = [&](auto tag) {
            using T = decltype(tag);
            BEngine<double, double, T> E{c, w, N, S, w.nch, G, pw.r.reserve(N + 1), pw.z.reserve(N + 1),
                                         pw.p.reserve(N + 1), pw.Ap.reserve(N + 1), x, (const double*)c.t_vals,
                                         sizeof(T) == 4, o.stop_rule};
            hipLaunchKernelGGL((k_bcast<double, double>), dim3(flat_grid(N)), dim3(256), 0, s, N, E.r, b);
            SGIPC_LAUNCH_CHECK();
            SGIPC_HIP(hipMemcpyAsync(w.tol.p, htol.data(), sizeof(double) * S, hipMemcpyHostToDevice, s));
            SGIPC_HIP(hipMemcpyAsync(w.stop.p, hstop.data(), sizeof(int) * S, hipMemcpyHostToDevice, s));
            E.init(max_iter);
            E.run(sizeof(T) == 4 ? w.graph32 : w.graph64, per_graph);
        };
        if (c.precond_kind == 3) run64(float{});
        else run64(double{});
        SGIPC_HIP(hipMemcpyAsync(hit.data(), w.iters.p, sizeof(int) * S, hipMemcpyDeviceToHost, s));
        SGIPC_HIP(hipMemcpyAsync(hnc.data(), w.noconv.p, sizeof(int) * S, hipMemcpyDeviceToHost, s));
        SGIPC_HIP(hipStreamSynchronize(s));
        for (int i = 0; i < S; ++i) {
            st[i].iterations = hit[i];
            st[i].converged = hnc[i] ? 0 : 1;
        }
    } else {
        // FP32 inner solves (FP32 values, FP32 MAS, FP64 dots) with FP64
        // outer refinement on each scene's true residual
        if (c.precond_kind != 3 && c.precond_kind != 2) throw arg_error("solve_batched: unsupported preconditioner");
        if (!c.mas.inv32.p) throw state_error("solve_batched: mixed precision needs the FP32 MAS inverses");
        float* rf = pw.rf.reserve(N + 1);
        double* r64 = pw.r64b.reserve(N + 1);
        double* d64 = pw.d64.reserve(N + 1);
        // the SpMV reads the row-contiguous FP32 copy of both triangles, or
        // (SGIPC_SPMV_FULL32=0) the FP32 copy of the upper BCOO; only one is built
        const float* vfull = c.spmv_full32 ? bsr_full(c, float{}) : nullptr;
        BEngine<float, float, float> E{c, w, N, S, w.nch, G, rf, pw.zf.reserve(N + 1), pw.pf.reserve(N + 1),
                                      pw.Apf.reserve(N + 1), d64, vfull ? nullptr : bsr_values_f32(c), true, 1};
        E.vfull = vfull;
        fill<double>(x, 0.0, N, s);
        hipLaunchKernelGGL((k_bcast<double, double>), dim3(flat_grid(N)), dim3(256), 0, s, N, r64, b);
        SGIPC_LAUNCH_CHECK();
        std::vector<double> bb, rr;
        hipLaunchKernelGGL((k_bdot<double, double>), dim3(w.nch), dim3(kBT), 0, s, (const BatchChunk*)w.chunk.p, b, b,
                           w.part_rr.p);
        SGIPC_LAUNCH_CHECK();
        seg_to_host(c, w, S, w.part_rr.p, bb);
        rr = bb;
        std::vector<int> total(S, 0), done(S, 0), nc(S, 0);
        for (int outer = 0; outer < 50; ++outer) {
            int left = 0;
            for (int i = 0; i < S; ++i) {
                const double bn = std::sqrt(bb[i]), rn = std::sqrt(rr[i]);
                if (!done[i] && (rn <= o.tol * bn || bn == 0.0)) done[i] = 1;
                if (!done[i] && total[i] >= max_iter) { done[i] = 1; nc[i] = 1; }
                hstop[i] = done[i];
                htol[i] = done[i] ? 0.0 : std::max(0.9 * o.tol * bn / rn, o.inner_tol);
                left += done[i] ? 0 : 1;
            }
            if (!left) break;
            int budget = 0;
            for (int i = 0; i < S; ++i)
                if (!done[i]) budget = std::max(budget, max_iter - total[i]);
            hipLaunchKernelGGL((k_bcast<float, double>), dim3(flat_grid(N)), dim3(256), 0, s, N, rf,
                               (const double*)r64);
            SGIPC_LAUNCH_CHECK();
            SGIPC_HIP(hipMemcpyAsync(w.tol.p, htol.data(), sizeof(double) * S, hipMemcpyHostToDevice, s));
            SGIPC_HIP(hipMemcpyAsync(w.stop.p, hstop.data(), sizeof(int) * S, hipMemcpyHostToDevice, s));
            E.init(budget);
            E.run(w.graph_mixed, per_graph);
            SGIPC_HIP(hipMemcpyAsync(hit.data(), w.iters.p, sizeof(int) * S, hipMemcpyDeviceToHost, s));
            SGIPC_HIP(hipStreamSynchronize(s));
            for (int i = 0; i < S; ++i)
                if (!done[i]) {
                    total[i] += hit[i];
                    st[i].refinements = outer + 1;
                }
            hipLaunchKernelGGL(k_baxpy, dim3(flat_grid(N)), dim3(256), 0, s, N, x, (const double*)d64);
            SGIPC_LAUNCH_CHECK();
            hipLaunchKernelGGL((k_bcast<double, double>), dim3(flat_grid(N)), dim3(256), 0, s, N, r64, b);
            SGIPC_LAUNCH_CHECK();
            spmv64(c, -1.0, x, 1.0, r64);
            hipLaunchKernelGGL((k_bdot<double, double>), dim3(w.nch), dim3(kBT), 0, s, (const BatchChunk*)w.chunk.p,
                               (const double*)r64, (const double*)r64, w.part_rr.p);
            SGIPC_LAUNCH_CHECK();
            seg_to_host(c, w, S, w.part_rr.p, rr);
        }
        for (int i = 0; i < S; ++i) {
            const double bn = std::sqrt(bb[i]);
            st[i].iterations = total[i];
            st[i].converged = (!nc[i] && (std::sqrt(rr[i]) <= o.tol * bn || bn == 0.0)) ? 1 : 0;
        }
    }
    // per-scene FP64 true residuals
    double* tmp = pw.xw.reserve(N + 1);
    hipLaunchKernelGGL((k_bcast<double, double>), dim3(flat_grid(N)), dim3(256), 0, s, N, tmp, b);
    SGIPC_LAUNCH_CHECK();
    spmv64(c, -1.0, x, 1.0, tmp);
    std::vector<double> rr, bb;
    hipLaunchKernelGGL((k_bdot<double, double>), dim3(w.nch), dim3(kBT), 0, s, (const BatchChunk*)w.chunk.p,
                       (const double*)tmp, (const double*)tmp, w.part_rr.p);
    SGIPC_LAUNCH_CHECK();
    seg_to_host(c, w, S, w.part_rr.p, rr);
    hipLaunchKernelGGL((k_bdot<double, double>), dim3(w.nch), dim3(kBT), 0, s, (const BatchChunk*)w.chunk.p, b, b,
                       w.part_rr.p);
    SGIPC_LAUNCH_CHECK();
    seg_to_host(c, w, S, w.part_rr.p, bb);
    for (int i = 0; i < S; ++i) st[i].rel_residual = bb[i] > 0.0 ? std::sqrt(rr[i] / bb[i]) : std::sqrt(rr[i]);
}

}  // namespace sgipc

namespace sgipc {

// Schedule autotuner: times a fixed number of PCG iterations (unreachable
// tolerance) for each candidate schedule on the current system and keeps the
// fastest.  Candidates: lanes per block row in the SpMV (4, 8, 16; where the
// SpMV has them: the batched solvers and the upper BCOO's) and, for the batched
// solver, iterations captured per graph launch (2, 4, 8) of the
// launch sequence, and (16-vertex banks) the persistent form with 512 or
// 1024 threads per workgroup.  For the batched solver the fixed-iteration
// trial only shortlists: the fastest launch sequence and the fastest
// persistent form of each workgroup size are then timed on a whole solve to
// a 1e-6 true relative residual, where scenes stop at their own iteration
// counts (which can rank the persistent forms the other way round), and the
// fastest of those is kept.  Returns the chosen (group, iterations per
// graph); the chosen batched form stays in the context.
void autotune(Ctx& c, const double* b, int S, const int* h_row_start, int precision, int& group, int& per_graph) {
    if (!c.have_bcoo) throw state_error("autotune: convert first");
    const long long N = 3LL * c.nb;
    double* x = c.tune_x.reserve(N + 1);
    SolveOpts o;
    o.precision = precision;
    o.stop_rule = 1;
    o.tol = 0.0;            // never met: every candidate runs the same iteration count
    o.max_iter = 48;
    o.inner_tol = 0.0;
    o.check_every = 48;
    struct Cand {
        int group, per_graph, persistent, threads;
    };
    std::vector<Cand> cands;
    // a single system's SpMV over the copy of both triangles has no lanes per
    // row: one candidate, the group as it was set (its solve refuses what any
    // solve refuses)
    const bool by_entries = S == 0 && (precision == 0 ? fp64_on_copy(c) : c.spmv_full32 != 0);
    for (int g : {4, 8, 16}) {
        if (S > 0)
            for (int pg : {2, 4, 8}) cands.push_back({g, pg, 0, c.batch_threads});
        else if (!by_entries || g == c.spmv_group)
            cands.push_back({g, c.batch_iters_per_graph, 0, c.batch_threads});
    }
    if (S > 0 && c.mas.ready && c.mas.bank == 16)
        for (int g : {4, 8, 16})
            for (int th : {512, 1024}) cands.push_back({g, c.batch_iters_per_graph, 1, th});
    const Cand save{c.spmv_group, c.batch_iters_per_graph, c.batch_persistent, c.batch_threads};
    auto apply = [&](const Cand& k) {
        c.spmv_group = k.group;
        c.batch_iters_per_graph = k.per_graph;
        c.batch_persistent = k.persistent;
        c.batch_threads = k.threads;
    };
    double best = 1e300;
    Cand pick = save;
    int best_pg = save.per_graph;  // iterations per graph of the fastest launch-sequence candidate
    double best_seq = 1e300;
    // shortlist for the whole-solve round: fastest sequence, fastest
    // persistent form with 512 and with 1024 threads
    Cand short_c[3] = {save, save, save};
    double short_ms[3] = {1e300, 1e300, 1e300};
    std::vector<SolveStats> st(S > 0 ? S : 1);
    hipEvent_t e0, e1;
    SGIPC_HIP(hipEventCreate(&e0));
    SGIPC_HIP(hipEventCreate(&e1));
    auto time_solve = [&](const SolveOpts& so) {
        float ms = 0.f;
        for (int rep = 0; rep < 2; ++rep) {  // first run builds the graphs
            SGIPC_HIP(hipEventRecord(e0, c.stream));
            if (S > 0) pcg_solve_batched(c, S, h_row_start, b, x, so, st.data());
            else pcg_solve(c, b, x, so, st[0]);
            SGIPC_HIP(hipEventRecord(e1, c.stream));
            SGIPC_HIP(hipEventSynchronize(e1));
            SGIPC_HIP(hipEventElapsedTime(&ms, e0, e1));
        }
        return (double)ms;
    };
    try {
        for (const Cand& k : cands) {
            apply(k);
            const double ms = time_solve(o);
            if (ms < best) { best = ms; pick = k; }
            if (!k.persistent && ms < best_seq) { best_seq = ms; best_pg = k.per_graph; }
            const int slot = !k.persistent ? 0 : (k.threads == 512 ? 1 : 2);
            if (ms < short_ms[slot]) { short_ms[slot] = ms; short_c[slot] = k; }
        }
        if (S > 0 && short_ms[1] < 1e300) {
            SolveOpts full;
            full.precision = precision;
            full.stop_rule = 1;
            full.tol = 1e-6;
            full.inner_tol = c.inner_tol;
            double best_full = 1e300;
            for (int i = 0; i < 3; ++i) {
                if (short_ms[i] >= 1e300) continue;
                apply(short_c[i]);
                const double ms = time_solve(full);
                if (ms < best_full) { best_full = ms; pick = short_c[i]; }
            }
        }
    } catch (...) {
        apply(save);
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        throw;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (pick.persistent) pick.per_graph = best_pg;
    apply(pick);
    group = pick.group;
    per_graph = pick.per_graph;
}

}  // namespace sgipc
