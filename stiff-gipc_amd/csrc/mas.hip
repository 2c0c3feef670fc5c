// Multilevel additive Schwarz (MAS) preconditioner: aggregation tables,
// Galerkin bank matrices, Gauss-Jordan bank inverses and the apply
//   z = sum_l R_l^T D_l^{-1} R_l r.
//
// Reference: S/MASPreconditioner.cu -- ReorderRealtime :1772-1813 and its
// kernels (:63-627), _buildCollisionConnection_new :1132-1540,
// PrepareHessian_bcoo :1816-2062, __inverse6_P96x96 :630-726,
// preconditioning :2221-2262 (__buildMultiLevelR_optimized_new :729-847,
// _schwarzLocalXSym6 :957-1027, __collectFinalZ_new :850-879),
// computeNumLevels :1724-1743; bank map S/gl_main.cu:1066-1093.
//
// Table semantics are identical to the reference (integer, bit-exact); the
// reference's warp-synchronous 16-lane-bank tricks become explicit LDS stages
// with block barriers (a bank is a quarter of a wave64).  The restriction is
// a deterministic per-bank component sum (no FP atomics); the apply is a dense
// product with the symmetric inverse, a wavefront per 16-vertex bank (from
// registers, bank_solve.hpp) or a workgroup per 32-vertex one.
#include "context.hpp"
#include <rocprim/device/device_radix_sort.hpp>
#include <utility>
#include "pcg_dev.hpp"
#include "bank_solve.hpp"
#include <algorithm>

namespace sgipc {
namespace {

constexpr int kTB = 256;  // threads per block for bank-parallel kernels

__device__ inline unsigned ltmask(int lane) { return lane >= 32 ? 0xffffffffu : ((1u << lane) - 1u); }
__device__ inline int lowbit(unsigned m) { return __ffs(m) - 1; }

// closure of lane's mask over the original masks of its bank (BFS on bits)
__device__ inline unsigned closure(unsigned own, int lane, const unsigned* bank_masks) {
    unsigned conn = own, visited = 1u << lane;
    for (int it = 0; it < 32; ++it) {
        unsigned todo = visited ^ conn;
        if (!todo) break;
        int nv = lowbit(todo);
        visited |= 1u << nv;
        conn |= bank_masks[nv];
    }
    return conn;
}

// ---- level 0 ---------------------------------------------------------------
constexpr int kNbrBatch = 8;  // neighbour-list gathers in flight per thread

__global__ void k_l0_masks(int M, int B, const int* __restrict__ part_map, const int* __restrict__ real_map,
                           const unsigned* __restrict__ nstart, const unsigned* __restrict__ nnum,
                           const unsigned* __restrict__ nlist, unsigned* __restrict__ fine_mask) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= M) return;
    int v = part_map[s];
    if (v < 0) return;
    int bank = s / B, lane = s % B;
    unsigned msk = 1u << lane, st = nstart[v], nn = nnum[v];
    // neighbours eight at a time: their ids, then their slots, are loaded
    // before any is used, so the gathers overlap (the OR is order-free)
    for (unsigned i0 = 0; i0 < nn; i0 += kNbrBatch) {
        int ids[kNbrBatch], su[kNbrBatch];
#pragma unroll
        for (int k = 0; k < kNbrBatch; ++k) ids[k] = (i0 + k < nn) ? (int)nlist[st + i0 + k] : -1;
#pragma unroll
        for (int k = 0; k < kNbrBatch; ++k) su[k] = ids[k] >= 0 ? real_map[ids[k]] : -1;
#pragma unroll
        for (int k = 0; k < kNbrBatch; ++k)
            if (ids[k] >= 0 && su[k] / B == bank) msk |= 1u << (su[k] % B);
    }
    fine_mask[v] = msk;
}

// contact-pair connectivity (decode of the int4 sign encoding)
__device__ inline int decode_pair(int4 q, int node_offset, int* v) {
    int x = q.x, y = q.y, z = q.z, w = q.w, cnt;
    if (x >= 0) {
        if (w < 0) w = -w - 1;
        v[0] = x; v[1] = y; v[2] = z; v[3] = w; cnt = 4;
    } else {
        x = -x - 1;
        if (z < 0) {
            if (y < 0) { y = -y - 1; z = -z - 1; w = -w - 1; v[0] = x; v[1] = y; v[2] = z; v[3] = w; cnt = 4; }
            else { v[0] = x; v[1] = y; v[2] = -1; v[3] = -1; cnt = 2; }
        } else if (w < 0) {
            if (y < 0) { y = -y - 1; w = -w - 1; v[0] = x; v[1] = y; v[2] = z; v[3] = w; cnt = 4; }
            else { v[0] = x; v[1] = y; v[2] = z; v[3] = -1; cnt = 3; }
        } else { v[0] = x; v[1] = y; v[2] = z; v[3] = w; cnt = 4; }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (i < cnt) ? v[i] - node_offset : -1;
    return cnt;
}

// Masks ORed into global words by one workgroup: the words [base, base +
// kOrWin) meet in LDS first, and each that gets a bit costs the workgroup one
// read and at most one atomic.  Device-scope atomics of the eight XCDs meet in
// memory, some 40 ns each on one line: with one a wavefront the levels of a few
// nodes took up to 90 us at 137 k vertices.
constexpr int kOrT = 512;
constexpr int kOrWin = 1024;
struct OrWindow {
    unsigned* w;  // kOrWin words of LDS
    int base;
    __device__ void clear() const {
        for (int i = threadIdx.x; i < kOrWin; i += kOrT) w[i] = 0u;
        __syncthreads();
    }
    __device__ void add(unsigned* dst, int node, unsigned m) const {
        const unsigned k = (unsigned)(node - base);
        if (k < (unsigned)kOrWin) atomicOr(w + k, m);
        else atomicOr(dst + node, m);
    }
    __device__ void flush(unsigned* dst) const {
        __syncthreads();
        for (int i = threadIdx.x; i < kOrWin; i += kOrT) {
            const unsigned m = w[i];
            if (!m) continue;
            const unsigned cur = __hip_atomic_load(dst + base + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((cur | m) != cur) atomicOr(dst + base + i, m);
        }
    }
};

// level < 0: ids are slots and dst is indexed by vertex; else ids are the
// level-local coarse ids from coarse_space row (level-1), dst indexed by id.
// Coarse levels funnel many pairs onto few nodes: levels of up to kOrWin nodes
// go through the window.  9.9 us a level at 137 k vertices with leader rounds of
// a read and an atomic each, now 4.4.
__global__ void __launch_bounds__(kOrT) k_collision(int np, const int4* __restrict__ pairs, int node_offset, int n,
                                                    int B, int level, const int* __restrict__ ls,
                                                    const int* __restrict__ real_map,
                                                    const int* __restrict__ coarse_space, unsigned* __restrict__ dst) {
    __shared__ unsigned win[kOrWin];
    const bool few = level >= 0 && ls[2 * level] <= kOrWin;
    const OrWindow W{win, 0};
    if (few) W.clear();
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    int v[4] = {-1, -1, -1, -1}, cp[4];
    int cnt = (p < np) ? decode_pair(pairs[p], node_offset, v) : 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (i >= cnt || v[i] < 0 || v[i] >= n) cp[i] = -1;
        else cp[i] = (level < 0) ? real_map[v[i]] : coarse_space[(size_t)(level - 1) * n + v[i]];
    }
    const int lb = __ffs(B) - 1;
    unsigned msk[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = i + 1; j < 4; ++j) {
            if (cp[i] < 0 || cp[j] < 0 || cp[i] == cp[j]) continue;
            if ((cp[i] >> lb) == (cp[j] >> lb)) {
                msk[i] |= 1u << (cp[j] & (B - 1));
                msk[j] |= 1u << (cp[i] & (B - 1));
            }
        }
    if (few) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (msk[i]) W.add(dst, cp[i], msk[i]);
        W.flush(dst);
        return;
    }
    unsigned cur[4];  // the four words are read together; an OR that adds no bit is left out
#pragma unroll
    for (int i = 0; i < 4; ++i)
        cur[i] = msk[i] ? __hip_atomic_load(dst + (level < 0 ? v[i] : cp[i]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                        : 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if ((cur[i] | msk[i]) != cur[i]) atomicOr(dst + (level < 0 ? v[i] : cp[i]), msk[i]);
}

// closure inside each level-0 bank, component count per bank
__global__ void __launch_bounds__(kTB) k_l0_closure(int M, int B, const int* __restrict__ part_map,
                                                     unsigned* __restrict__ fine_mask, int* __restrict__ prefix0) {
    __shared__ unsigned sm[kTB];
    __shared__ unsigned sc[kTB];
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    int lane = threadIdx.x % B, bbase = threadIdx.x - lane;
    int v = (s < M) ? part_map[s] : -1;
    sm[threadIdx.x] = (v >= 0) ? fine_mask[v] : 0u;
    __syncthreads();
    unsigned cl = 0u;
    if (v >= 0) {
        cl = closure(sm[threadIdx.x], lane, sm + bbase);
        fine_mask[v] = cl;
    }
    sc[threadIdx.x] = (v >= 0 && (cl & ltmask(lane)) == 0u) ? 1u : 0u;
    __syncthreads();
    if (lane == 0 && s < M) {
        int cnt = 0;
        for (int l = 0; l < B; ++l) cnt += (int)sc[bbase + l];
        prefix0[s / B] = cnt;
    }
}

// sizes of the next level: ls[2*(level+1)] = total comps, ls[2*(level+1)+1] =
// begin_level + pad(count_level) (Mpad after level 0)
__device__ inline void set_level_size(int* __restrict__ ls, int level, int total, int B, int first_begin) {
    ls[2 * (level + 1)] = total;
    ls[2 * (level + 1) + 1] = level == 0 ? first_begin : ls[2 * level + 1] + (ls[2 * level] + B - 1) / B * B;
}

__global__ void __launch_bounds__(kTB) k_level1(int M, int Mpad, int n, int B, const int* __restrict__ part_map,
                                                 const unsigned* __restrict__ fine_mask,
                                                 const int* __restrict__ psum0, int* __restrict__ coarse_space,
                                                 int* __restrict__ going_next, SlotNode* __restrict__ slot_node,
                                                 const int* __restrict__ total, int* __restrict__ ls) {
    __shared__ unsigned sel[kTB];
    if (blockIdx.x == 0 && threadIdx.x == 0) set_level_size(ls, 0, *total, B, Mpad);
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    int lane = threadIdx.x % B, bbase = threadIdx.x - lane;
    int v = (s < M) ? part_map[s] : -1;
    unsigned fm = (v >= 0) ? fine_mask[v] : 0u;
    sel[threadIdx.x] = (v >= 0 && (fm & ltmask(lane)) == 0u) ? (1u << lane) : 0u;
    __syncthreads();
    if (v < 0) {
        if (s < M) slot_node[s] = SlotNode{-1, -1, 0u, 0u};
        return;
    }
    unsigned elected = 0u;
    for (int l = 0; l < B; ++l) elected |= sel[bbase + l];
    int el = lowbit(fm);
    int pre = __popc(elected & ltmask(el)) + psum0[s / B];
    coarse_space[v] = pre;
    going_next[v] = pre + Mpad;
    slot_node[s] = SlotNode{v, pre, fm, 0u};
}

// coarse connectivity at `level` (nodes are level-local ids in coarse_space
// row level-1).  Vertices are numbered in bank order, so a workgroup's nodes
// are few and close together: their masks meet in an LDS window (OrWindow)
// that begins a little before its first vertex's node.  A vertex whose
// neighbours are all in its own node has nothing to add on any level above:
// `outer` marks the others, and the levels after the first look at those only.
// Per level at 137 k vertices: 20 us with an atomic a wavefront or vertex and
// all vertices looked at, now 10 (workgroups of 1024 the same; at 44 k vertices,
// 43 workgroups then, 10.9 against 7.7).
__global__ void __launch_bounds__(kOrT) k_lx_masks(int n, int B, int level, const int* __restrict__ ls,
                                                   const unsigned* __restrict__ nstart,
                                                   const unsigned* __restrict__ nnum,
                                                   const unsigned* __restrict__ nlist,
                                                   const int* __restrict__ coarse_space,
                                                   unsigned* __restrict__ next_mask,
                                                   unsigned char* __restrict__ outer) {
    __shared__ unsigned win[kOrWin];
    const int v0 = blockIdx.x * kOrT, v = v0 + threadIdx.x;
    const bool live = v < n && (level == 1 || outer[v]);
    if (!__syncthreads_or(live)) return;
    const int* cs = coarse_space + (size_t)(level - 1) * n;
    const OrWindow W{win, ls[2 * level] <= kOrWin ? 0 : max(0, cs[v0] - 64)};
    W.clear();
    if (live) {
        const int ci = cs[v], lb = __ffs(B) - 1, bank = ci >> lb;
        const unsigned st = nstart[v], nn = nnum[v];
        unsigned msk = 0u;
        bool out = false;
        for (unsigned i0 = 0; i0 < nn; i0 += kNbrBatch) {  // as in k_l0_masks
            int ids[kNbrBatch], cu[kNbrBatch];
#pragma unroll
            for (int k = 0; k < kNbrBatch; ++k) ids[k] = (i0 + k < nn) ? (int)nlist[st + i0 + k] : v;
#pragma unroll
            for (int k = 0; k < kNbrBatch; ++k) ids[k] = ids[k] < 0 ? v : ids[k];  // (padding)
#pragma unroll
            for (int k = 0; k < kNbrBatch; ++k) cu[k] = cs[ids[k]];
#pragma unroll
            for (int k = 0; k < kNbrBatch; ++k)
                if (cu[k] != ci) {
                    out = true;
                    if ((cu[k] >> lb) == bank) msk |= 1u << (cu[k] & (B - 1));
                }
        }
        if (level == 1 || !out) outer[v] = out ? 1 : 0;
        if (msk) W.add(next_mask, ci, msk);
    }
    W.flush(next_mask);
}

__global__ void __launch_bounds__(kTB) k_lx_closure(int nmax, int B, int level, const int* __restrict__ ls,
                                                     unsigned* __restrict__ next_mask, int* __restrict__ next_prefix,
                                                     unsigned* __restrict__ comp_mask) {
    __shared__ unsigned sm[kTB];
    __shared__ unsigned sc[kTB];
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    int lane = threadIdx.x % B, bbase = threadIdx.x - lane;
    int number = ls[2 * level + 0];
    bool valid = c < number;
    sm[threadIdx.x] = valid ? ((1u << lane) | next_mask[c]) : 0u;
    __syncthreads();
    unsigned cl = 0u;
    if (valid) cl = closure(sm[threadIdx.x], lane, sm + bbase);
    sc[threadIdx.x] = (valid && (cl & ltmask(lane)) == 0u) ? 1u : 0u;
    __syncthreads();
    if (valid) {
        next_mask[c] = cl;
        comp_mask[(size_t)ls[2 * level + 1] + c] = cl;  // component lanes of global node beg + c
    }
    if (lane == 0 && c < nmax) {
        int cnt = 0;
        for (int l = 0; l < B; ++l) cnt += (int)sc[bbase + l];
        next_prefix[c / B] = cnt;
    }
}

__global__ void __launch_bounds__(kTB) k_lx_renumber(int B, int level, int* ls, const int* __restrict__ total,
                                                      unsigned* __restrict__ next_mask,
                                                      const int* __restrict__ next_psum, int* __restrict__ going_next,
                                                      size_t going_cap) {
    __shared__ unsigned sel[kTB];
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    int lane = threadIdx.x % B, bbase = threadIdx.x - lane;
    int number = ls[2 * level + 0], begin = ls[2 * level + 1];
    int pad = (number + B - 1) / B * B;
    if (c == 0) set_level_size(ls, level, *total, B, 0);  // (this level's words are read only)
    bool valid = c < number;
    unsigned cm = valid ? next_mask[c] : 0u;
    sel[threadIdx.x] = (valid && (cm & ltmask(lane)) == 0u) ? (1u << lane) : 0u;
    __syncthreads();
    if (!valid) return;
    unsigned elected = 0u;
    for (int l = 0; l < B; ++l) elected |= sel[bbase + l];
    int pre = __popc(elected & ltmask(lowbit(cm))) + next_psum[c / B];
    next_mask[c] = (unsigned)pre;  // every lane of the block read its mask before the barrier
    size_t g = (size_t)begin + c;
    if (g < going_cap) going_next[g] = pre + begin + pad;
}

// node of every vertex at the next level; clears the masks of that level
// (`clear`: the buffer the level before this one used)
__global__ void k_next_table(int n, int level, int* __restrict__ coarse_space, const unsigned* __restrict__ next_mask,
                             unsigned* __restrict__ clear, int nclear) {
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v < nclear) clear[v] = 0u;
    if (v >= n) return;
    int nx = coarse_space[(size_t)(level - 1) * n + v];
    coarse_space[(size_t)level * n + v] = (int)next_mask[nx];
}

__global__ void k_aggregate(int n, int L, const int* __restrict__ real_map, const int* __restrict__ going_next,
                            int* __restrict__ coarse_table, int* __restrict__ node_of) {
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    int cur = v;
    node_of[v] = real_map[v];
    for (int l = 0; l < L - 1; ++l) {
        int nx = going_next[cur];
        coarse_table[6 * (size_t)v + l] = nx;
        node_of[(size_t)(l + 1) * n + v] = nx;
        cur = nx;
    }
    for (int l = L - 1; l < 6; ++l) coarse_table[6 * (size_t)v + l] = 0;
}

// ---- Galerkin projection ----------------------------------------------------
__device__ inline int pack_index(int B, int r, int c) { return B * r - r * (r + 1) / 2 + c; }  // r <= c

// Projection of one BCOO block H = A(r, c) (r <= c, column-major) onto the
// level-l bank entry of its node pair: the packed index and the 3x3 block
// (H + H^T on a coarse diagonal, H^T below the bank diagonal).
__device__ inline int project_block(int B, int li, int lj, bool same_vertex, const double* H, double* blk) {
    if (li == lj) {
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int q = 0; q < 3; ++q) blk[p + 3 * q] = same_vertex ? H[p + 3 * q] : H[p + 3 * q] + H[q + 3 * p];
        return pack_index(B, li, li);
    }
    if (li < lj) {
#pragma unroll
        for (int e = 0; e < 9; ++e) blk[e] = H[e];
        return pack_index(B, li, lj);
    }
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int q = 0; q < 3; ++q) blk[p + 3 * q] = H[q + 3 * p];
    return pack_index(B, lj, li);
}

// Galerkin projection for 16-vertex banks when vertex ids follow slot order:
// workgroup b owns the vertices whose level-1 node lies in level-1 bank b,
// i.e. the contiguous BCOO rows [vlo_b, vhi_b).  Level 0 targets are unique
// (read and added to without atomics; they were zeroed before).  Level-1 and level-2 targets accumulate in one-bank LDS
// windows (the first owned vertex's banks, which hold nearly every target)
// flushed once; the top levels (>= top_lvl, at most kProjTopBanksMax banks)
// accumulate in LDS and are written as per-workgroup partials, summed
// afterwards in a fixed order (k_project_top_reduce).  Other levels and
// window misses use global FP64 atomics.
// A block whose two vertices share the first owned vertex's level-2 node
// (most blocks: that node usually covers every owned vertex) adds the same
// 3x3 block, H + H^T (H on the diagonal), to that node's diagonal block on
// every level from 2 up, since nodes nest; such blocks are summed in
// registers and once over the workgroup instead of with LDS atomics that
// all lanes of a wavefront would aim at the same nine words.
constexpr int kProjWin1 = 1, kProjWin2 = 1;  // LDS window banks of levels 1 and 2
constexpr int kProjWinBanks = kProjWin1 + kProjWin2;
constexpr int kProjWinLevels = 2;
constexpr int kProjBank16 = 136 * 9;  // doubles per packed 16-vertex bank
constexpr int kProjTopBanks = 6;      // with the windows: 78 KB of LDS, two workgroups per CU
constexpr int kProjTopBanksMax = 12;  // larger top levels: 137 KB, one workgroup per CU
template <int TOPB>
__global__ void __launch_bounds__(512) k_project_banked(
    const int* __restrict__ ustart, const int* __restrict__ rows, const int* __restrict__ cols,
    const double* __restrict__ vals, int off, int n, int L, const int* __restrict__ node_of,
    const int* __restrict__ vlo, const int* __restrict__ vhi, int nbanks, double* __restrict__ bank_upper,
    int win_levels, int top_lvl, int top_lo, int top_nb, double* __restrict__ top_scratch) {
    constexpr int B = 16, NB = kProjBank16;
    __shared__ double win[kProjWinBanks * NB];  // level 1, then level 2
    __shared__ double top[TOPB * NB];
    __shared__ double red[9][512 / 64];
    __shared__ int wbase[kProjWinLevels];
    const int b = blockIdx.x, t = threadIdx.x;
    for (int i = t; i < kProjWinBanks * NB; i += blockDim.x) win[i] = 0.0;
    for (int i = t; i < top_nb * NB; i += blockDim.x) top[i] = 0.0;
    const int v0 = vlo[b], v1 = vhi[b];
    if (t < kProjWinLevels) wbase[t] = (v0 < v1 && t + 1 < L) ? node_of[(size_t)(t + 1) * n + v0] / B : -1;
    const int dom2 = (v0 < v1 && L > 2) ? node_of[2 * (size_t)n + v0] : -1;
    // LDS (or global) address of packed entry pidx of bank `bank` at level l >= 1
    auto target = [&](int l, int bank, int pidx) -> double* {
        if (l >= top_lvl) return top + (size_t)(bank - top_lo) * NB + 9 * pidx;
        if (l <= win_levels) {
            const int w = bank - wbase[l - 1];
            if (l == 1 && w == 0) return win + 9 * pidx;
            if (l == 2 && w >= 0 && w < kProjWin2) return win + (size_t)(kProjWin1 + w) * NB + 9 * pidx;
        }
        return bank_upper + (size_t)bank * NB + 9 * pidx;
    };
    double acc[9];
#pragma unroll
    for (int e = 0; e < 9; ++e) acc[e] = 0.0;
    __syncthreads();
    if (v0 < v1) {
        const int k0 = ustart[v0 + off], k1 = ustart[v1 + off];
        for (int k = k0 + t; k < k1; k += blockDim.x) {
            const int r = rows[k] - off, c = cols[k] - off;
            if (c < 0 || c >= n) continue;
            double H[9];
#pragma unroll
            for (int e = 0; e < 9; ++e) H[e] = vals[9 * (size_t)k + e];
            const bool dom = dom2 >= 0 && node_of[2 * (size_t)n + r] == dom2 && node_of[2 * (size_t)n + c] == dom2;
            const int lend = dom ? 2 : L;  // levels >= 2 of a dominant block: summed below
            for (int l = 0; l < lend; ++l) {
                const int I = node_of[(size_t)l * n + r], J = node_of[(size_t)l * n + c];
                if (I / B != J / B) continue;
                const int bank = I / B;
                double blk[9];
                const int pidx = project_block(B, I % B, J % B, r == c, H, blk);
                if (l == 0) {
                    double* dst = bank_upper + (size_t)bank * NB + 9 * pidx;  // unique per BCOO block
#pragma unroll
                    for (int e = 0; e < 9; ++e) dst[e] += blk[e];
                    continue;
                }
                double* dst = target(l, bank, pidx);
#pragma unroll
                for (int e = 0; e < 9; ++e)
                    if (blk[e] != 0.0) atomicAdd(dst + e, blk[e]);
            }
            if (dom) {
#pragma unroll
                for (int p = 0; p < 3; ++p)
#pragma unroll
                    for (int q = 0; q < 3; ++q) acc[p + 3 * q] += (r == c) ? H[p + 3 * q] : H[p + 3 * q] + H[q + 3 * p];
            }
        }
    }
    // the dominant blocks' sum, over the workgroup, onto the diagonal block
    // of the first owned vertex's node on every level from 2 up
#pragma unroll
    for (int e = 0; e < 9; ++e) {
        const double s = wave_sum(acc[e]);
        if ((t & 63) == 0) red[e][t >> 6] = s;
    }
    __syncthreads();
    if (t == 0 && dom2 >= 0) {
        double s[9];
#pragma unroll
        for (int e = 0; e < 9; ++e) {
            s[e] = 0.0;
            for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s[e] += red[e][w];
        }
        for (int l = 2; l < L; ++l) {
            const int I = node_of[(size_t)l * n + v0];
            double* dst = target(l, I / B, pack_index(B, I % B, I % B));
#pragma unroll
            for (int e = 0; e < 9; ++e)
                if (s[e] != 0.0) atomicAdd(dst + e, s[e]);
        }
    }
    __syncthreads();
    for (int q = t; q < kProjWinBanks * NB; q += blockDim.x) {
        const double v = win[q];
        const int w = q / NB, e = q % NB;
        const int lw = w < kProjWin1 ? 0 : 1;
        if (lw >= win_levels) continue;
        const int bank = wbase[lw] + (w < kProjWin1 ? w : w - kProjWin1);
        if (v != 0.0 && bank >= 0 && bank < nbanks) atomicAdd(bank_upper + (size_t)bank * NB + e, v);
    }
    double* out = top_scratch + (size_t)b * top_nb * NB;
    for (int q = t; q < top_nb * NB; q += blockDim.x) out[q] = top[q];
}

// Deterministic projection (opt-in): every BCOO block writes its level-0
// target directly and, for each coarse level where its node pair shares a
// bank, one (entry, block) record; a stable radix sort by entry groups the
// records in block order, and a fixed-order segmented sum (tiles of
// kProjTile records, see below) adds each group.  Same result on every run,
// for any bank size or numbering.
__global__ void k_proj_records(int K, const int* __restrict__ rows, const int* __restrict__ cols,
                               const double* __restrict__ vals, int off, int n, int B, int L,
                               const int* __restrict__ node_of, double* __restrict__ bank_upper, unsigned sentinel,
                               unsigned* __restrict__ key, unsigned* __restrict__ rec) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= K) return;
    const int npack = B * (B + 1) / 2;
    const int r = rows[k] - off, c = cols[k] - off;
    const bool in = r >= 0 && c >= 0 && r < n && c < n;
    for (int l = 1; l < L; ++l) {
        unsigned kk = sentinel;
        if (in) {
            const int I = node_of[(size_t)l * n + r], J = node_of[(size_t)l * n + c];
            if (I / B == J / B) {
                const int li = I % B, lj = J % B;
                kk = (unsigned)(I / B) * (unsigned)npack + (unsigned)(li <= lj ? pack_index(B, li, lj) : pack_index(B, lj, li));
            }
        }
        key[(size_t)k * (L - 1) + (l - 1)] = kk;
        rec[(size_t)k * (L - 1) + (l - 1)] = (unsigned)k * 8u + (unsigned)l;
    }
    if (!in) return;
    const int I = node_of[r], J = node_of[c];
    if (I / B != J / B) return;
    double H[9], blk[9];
#pragma unroll
    for (int e = 0; e < 9; ++e) H[e] = vals[9 * (size_t)k + e];
    const int pidx = project_block(B, I % B, J % B, r == c, H, blk);
    double* dst = bank_upper + ((size_t)(I / B) * npack + pidx) * 9;  // level 0: unique per BCOO block
#pragma unroll
    for (int e = 0; e < 9; ++e) dst[e] += blk[e];
}

// Fixed-order segmented sum of the sorted records: a workgroup takes a tile of
// kProjTile of them, puts their 3x3 contributions in LDS and adds every (entry,
// tile) piece in record order, nine lanes (one component each) a piece.  A
// piece that is a whole entry goes to its bank; one that begins in this tile
// and goes on, or continues one of the tile before, goes to `part` and is added
// in tile order by k_proj_carry.  Bound by the gather of the blocks (72 bytes
// a record).  Contributions through memory with one thread a piece took 97 +
// 710 + 64 us for 48 scenes (710 serial in pieces of up to 256), now 50 + 12; 64 to
// 10 us for the one of 20 x 4 x 4 cells.
constexpr int kProjTile = 256;
__global__ void __launch_bounds__(kProjTile) k_proj_tiles(long long m, const unsigned* __restrict__ key,
                                                          const unsigned* __restrict__ rec,
                                                          const int* __restrict__ rows, const int* __restrict__ cols,
                                                          const double* __restrict__ vals, int off, int n, int B,
                                                          const int* __restrict__ node_of, unsigned sentinel,
                                                          double* __restrict__ bank_upper, double* __restrict__ part) {
    __shared__ double v[kProjTile][9];
    __shared__ unsigned keys[kProjTile];
    __shared__ int head[kProjTile + 1];
    __shared__ int waves[kProjTile / 64];
    __shared__ int carried;  // the first piece continues one of the tile before
    const int t = threadIdx.x;
    const long long base = (long long)blockIdx.x * kProjTile, i = base + t;
    const unsigned kk = i < m ? key[i] : sentinel;
    const unsigned before = (i > 0 && i < m) ? key[i - 1] : sentinel;
    const unsigned after = base + kProjTile < m ? key[base + kProjTile] : sentinel;
    const bool valid = kk != sentinel;
    keys[t] = kk;
    if (valid) {
        const unsigned q = rec[i];
        const int k = (int)(q >> 3), l = (int)(q & 7u);
        const int r = rows[k] - off, c = cols[k] - off;
        double H[9], blk[9];
#pragma unroll
        for (int e = 0; e < 9; ++e) H[e] = vals[9 * (size_t)k + e];
        const int I = node_of[(size_t)l * n + r], J = node_of[(size_t)l * n + c];
        (void)project_block(B, I % B, J % B, r == c, H, blk);
#pragma unroll
        for (int e = 0; e < 9; ++e) v[t][e] = blk[e];
    }
    const bool first = valid && (t == 0 || before != kk);
    const unsigned long long heads = __ballot(first);
    if ((t & 63) == 0) waves[t >> 6] = __popcll(heads);
    const int nvalid = __syncthreads_count(valid);
    int at = __popcll(heads & ((1ull << (t & 63)) - 1ull)), np = 0;
#pragma unroll
    for (int w = 0; w < kProjTile / 64; ++w) {
        if (w < (t >> 6)) at += waves[w];
        np += waves[w];
    }
    if (first) head[at] = t;
    if (t == 0) {
        head[np] = nvalid;  // the sentinels sort last
        carried = valid && before == kk;
    }
    __syncthreads();
    for (int w = t; w < 9 * np; w += kProjTile) {
        const int p = w / 9, e = w - 9 * p, h = head[p], end = head[p + 1];
        double acc = v[h][e];
#pragma unroll 8
        for (int j = h + 1; j < end; ++j) acc += v[j][e];
        if (p == 0 && carried)
            part[((size_t)blockIdx.x * 2) * 9 + e] = acc;
        else if (end == kProjTile && after == keys[h])
            part[((size_t)blockIdx.x * 2 + 1) * 9 + e] = acc;
        else
            bank_upper[(size_t)keys[h] * 9 + e] = acc;
    }
}

// entries that run over several tiles: the piece of their first tile, then the
// following ones in tile order (16 lanes a tile, eight pieces in flight)
__global__ void k_proj_carry(long long m, int ntiles, const unsigned* __restrict__ key, unsigned sentinel,
                             const double* __restrict__ part, double* __restrict__ bank_upper) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x, tile = g >> 4, e = g & 15;
    if (tile + 1 >= ntiles || e >= 9) return;
    const long long base = (long long)tile * kProjTile;
    const unsigned kk = key[base + kProjTile - 1];
    if (kk == sentinel || key[base + kProjTile] != kk) return;
    if (tile > 0 && key[base] == kk && key[base - 1] == kk) return;  // began in an earlier tile
    double acc = part[((size_t)tile * 2 + 1) * 9 + e];
    constexpr int U = 8;
    for (int t0 = tile + 1; t0 < ntiles; t0 += U) {
        unsigned k[U];
        double p[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int q = min(t0 + u, ntiles - 1);
            k[u] = key[(long long)q * kProjTile];
            p[u] = part[((size_t)q * 2) * 9 + e];
        }
        bool on = true;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            on = on && t0 + u < ntiles && k[u] == kk;
            if (on) acc += p[u];
        }
        if (!on) break;
    }
    bank_upper[(size_t)kk * 9 + e] = acc;
}

// top-level bank entries = sum of the per-workgroup partials, fixed order
// (four interleaved partial sums per entry, combined in order).  Each sum reads
// 16 partials ahead of its adds: at 605 workgroups 42 us without, now 9.
__global__ void __launch_bounds__(256) k_project_top_reduce(const double* __restrict__ scratch, int nwg, int len,
                                                            double* __restrict__ dst) {
    __shared__ double part[4][64];
    const int e = blockIdx.x * 64 + (threadIdx.x & 63), q = threadIdx.x >> 6;
    constexpr int U = 16;
    double s = 0.0;
    if (e < len)
        for (int w = q; w < nwg; w += 4 * U) {
            double v[U];
#pragma unroll
            for (int k = 0; k < U; ++k) v[k] = scratch[(size_t)min(w + 4 * k, nwg - 1) * len + e];
#pragma unroll
            for (int k = 0; k < U; ++k)
                if (w + 4 * k < nwg) s += v[k];
        }
    part[q][threadIdx.x & 63] = s;
    __syncthreads();
    if (q == 0 && e < len) dst[e] = ((part[0][threadIdx.x] + part[1][threadIdx.x]) + part[2][threadIdx.x]) +
                                    part[3][threadIdx.x];
}

// ---- bank inverse: unpivoted in-place Gauss-Jordan in LDS -------------------
template <int B>
__global__ void __launch_bounds__(B == 16 ? 64 : 128) k_bank_inverse(int nbanks, const double* __restrict__ bank_upper,
                                                                      double* __restrict__ inv64,
                                                                      float* __restrict__ inv32) {
    constexpr int D = 3 * B;
    constexpr int npack = B * (B + 1) / 2;
    __shared__ double S[D][D + 1];
    __shared__ double colm[D];
    __shared__ double rt_s;
    int b = blockIdx.x;
    int i = threadIdx.x;  // column owned by this thread
    const double* src = bank_upper + (size_t)b * npack * 9;
    if (i < D) {
        int ci = i / 3, qi = i % 3;
        for (int j = 0; j < D; ++j) {
            int rj = j / 3, pj = j % 3;
            double v;
            if (ci >= rj) v = src[(size_t)pack_index(B, rj, ci) * 9 + pj + 3 * qi];   // block (rj,ci) elem (pj,qi)
            else v = src[(size_t)pack_index(B, ci, rj) * 9 + qi + 3 * pj];            // transpose of block (ci,rj)
            if (i == j && v == 0.0) v = 1.0;
            S[j][i] = v;
        }
    }
    __syncthreads();
    for (int j = 0; j < D; ++j) {
        if (i == 0) rt_s = S[j][j];
        if (i < D) colm[i] = S[i][j];
        __syncthreads();
        double rt = rt_s;
        if (i < D) S[i][j] = (i == j) ? 1.0 : 0.0;
        __syncthreads();
        if (i < D) {
            double pj = S[j][i] / rt;
            S[j][i] = pj;
            for (int k = 0; k < D; ++k)
                if (k != j) S[k][i] += -colm[k] * pj;
        }
        __syncthreads();
    }
    // symmetric result: keep the upper triangle, packed by rows
    if (i < D) {
        constexpr int NP = D * (D + 1) / 2;
        double* o64 = inv64 + (size_t)b * NP;
        float* o32 = inv32 + (size_t)b * NP;
        for (int r = 0; r <= i; ++r) {
            o64[inv_index<D, double>(r, i)] = S[r][i];
            o32[inv_index<D, float>(r, i)] = (float)S[r][i];
        }
    }
}

// Same elimination for 16-vertex banks (D = 48) with the matrix held in
// registers: thread i owns column i; at step j the owner of column j
// publishes it (double-buffered LDS, one barrier per step) and every thread
// updates its own column.  Steps are instantiated per compile-time j so every
// register index is static.  Arithmetic and order equal k_bank_inverse's.
template <int J, int D>
__device__ __forceinline__ void gj_step(double (&S)[D], double (*colm)[D], int i) {
    double* cm = colm[J & 1];
    if (i == J) {
#pragma unroll
        for (int k = 0; k < D; ++k) cm[k] = S[k];
    }
    __syncthreads();
    const double rt = cm[J];
    if (i == J) {
#pragma unroll
        for (int k = 0; k < D; ++k) S[k] = (k == J) ? 1.0 : 0.0;
    }
    const double pv = S[J] / rt;
    S[J] = pv;
#pragma unroll
    for (int k = 0; k < D; ++k)
        if (k != J) S[k] += -cm[k] * pv;
}

template <int D, int... J>
__device__ __forceinline__ void gj_all(double (&S)[D], double (*colm)[D], int i, std::integer_sequence<int, J...>) {
    (gj_step<J, D>(S, colm, i), ...);
}

// value v of lane `lane` (a compile-time constant) in every lane, through
// scalar registers
template <int LANE>
__device__ __forceinline__ double lane_value(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u & 0xffffffffu), LANE);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), LANE);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// The same step with the pivot column broadcast lane to lane (no LDS, no
// barrier).  Each entry k of the owner's column is read before the owner
// overwrites it in the same iteration; the owner starts from the unit
// vector e_J, as in gj_step, so the arithmetic is identical.
// (The owner's base is its entry times 0.0 -- one multiply instead of a
// 64-bit select; the same value up to the sign of a zero.)
template <int J, int D, int K>
__device__ __forceinline__ void gj_rl_entry(double (&S)[D], double pv, double keep) {
    if constexpr (K != J) {
        const double c = lane_value<J>(S[K]);
        const double base = S[K] * keep;
        S[K] = base + -c * pv;
    }
}
template <int J, int D, int... K>
__device__ __forceinline__ void gj_rl_step(double (&S)[D], int i, std::integer_sequence<int, K...>) {
    const bool own = i == J;
    const double keep = own ? 0.0 : 1.0;
    const double rt = lane_value<J>(S[J]);
    const double pv = (own ? 1.0 : S[J]) / rt;
    (gj_rl_entry<J, D, K>(S, pv, keep), ...);
    S[J] = pv;
}
template <int D, int... J>
__device__ __forceinline__ void gj_rl_all(double (&S)[D], int i, std::integer_sequence<int, J...>) {
    (gj_rl_step<J, D>(S, i, std::make_integer_sequence<int, D>{}), ...);
}

constexpr bool kBankInverseReadlane = true;  // pivot column by lane broadcast (false: through LDS)
__global__ void __launch_bounds__(64) k_bank_inverse_reg48(int nbanks, const double* __restrict__ bank_upper,
                                                           double* __restrict__ inv64, float* __restrict__ inv32) {
    constexpr int B = 16, D = 48, npack = B * (B + 1) / 2, NP = D * (D + 1) / 2;
    __shared__ double colm[2][D];
    const int b = blockIdx.x, i = threadIdx.x;
    const bool act = i < D;
    const double* src = bank_upper + (size_t)b * npack * 9;
    double S[D];
    const int ci = i / 3, qi = i % 3;
#pragma unroll
    for (int j = 0; j < D; ++j) {
        const int rj = j / 3, pj = j % 3;
        double v = 0.0;
        if (act) {
            v = (ci >= rj) ? src[(size_t)pack_index(B, rj, ci) * 9 + pj + 3 * qi]
                           : src[(size_t)pack_index(B, ci, rj) * 9 + qi + 3 * pj];
            if (i == j && v == 0.0) v = 1.0;
        }
        S[j] = v;
    }
    if (kBankInverseReadlane) {
        (void)colm;
        gj_rl_all<D>(S, i, std::make_integer_sequence<int, D>{});
    } else {
        gj_all<D>(S, colm, i, std::make_integer_sequence<int, D>{});
    }
    if (act) {
        double* o64 = inv64 + (size_t)b * NP;
        float* o32 = inv32 + (size_t)b * NP;
#pragma unroll
        for (int r = 0; r < D; ++r)
            if (r <= i) {
                o64[inv_index<D, double>(r, i)] = S[r];
                o32[inv_index<D, float>(r, i)] = (float)S[r];
            }
    }
}

// Half-storage form of the packed 48 x 48 inverses for the fused FP32 bank
// solves: D = sqrt of the inverse's diagonal (1 where it is not positive),
// S = D^-1 inv D^-1 rounded to FP16 (unit diagonal; |S_ij| <= 1 for an SPD
// inverse, clamped to the FP16 range otherwise).  One wavefront per bank,
// FP64 arithmetic from the FP64 inverses when they were built.
template <typename S>
__global__ void __launch_bounds__(64) k_pack_inv_half(int nbanks, const S* __restrict__ inv,
                                                      unsigned short* __restrict__ h, float* __restrict__ dsc) {
    constexpr int D = 48, NP = D * (D + 1) / 2;
    __shared__ double d[D];
    const int b = blockIdx.x, i = threadIdx.x;
    if (b >= nbanks) return;
    const S* src = inv + (size_t)b * NP;
    if (i < D) {
        const double a = (double)src[inv_index<D, S>(i, i)];
        const double di = a > 0.0 ? sqrt(a) : 1.0;
        d[i] = di;
        dsc[(size_t)b * D + i] = (float)di;
    }
    __syncthreads();
    unsigned short* dst = h + (size_t)b * NP;
    for (int r = 0; r < D; ++r) {
        const int c = r + i;
        if (c < D) {
            const float v = (float)((double)src[inv_index<D, S>(r, c)] / (d[r] * d[c]));
            const _Float16 hv = (_Float16)fminf(fmaxf(v, -65504.f), 65504.f);
            dst[inv_index<D, _Float16>(r, c)] = __builtin_bit_cast(unsigned short, hv);
        }
    }
}

// ---- apply -----------------------------------------------------------------
// address-space-qualified pointers for the direct global -> LDS load builtin
typedef __attribute__((address_space(1))) const void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

// z_bank = A^-1 r_bank for every bank of every level, 32-vertex banks: the
// packed inverse is staged through LDS (the bytes of this kernel are almost
// all inverse bytes), then lane i forms row i, summing over columns in order.
template <typename T>
__global__ void __launch_bounds__(128) k_bank_solve32(const T* __restrict__ inv, const T* __restrict__ R,
                                                      T* __restrict__ Z, const int* __restrict__ ctrl,
                                                      SceneSkip skip) {
    if (ctrl && ctrl[0]) return;
    if (skip.stopped(blockIdx.x)) return;
    constexpr int D = 96, NT = 128;
    constexpr int NP = D * (D + 1) / 2;
    constexpr int NV = NP * (int)sizeof(T) / 16;
    static_assert(NP * sizeof(T) % 16 == 0, "packed bank must be a whole number of 16-byte vectors");
    using V4 = typename std::conditional<sizeof(T) == 8, double2, float4>::type;
    constexpr int PER = (NV + NT - 1) / NT;
    __shared__ V4 As[PER * NT];  // padded to whole 1 KB wave chunks
    __shared__ T rs[D];
    const int b = blockIdx.x, i = threadIdx.x;
    const V4* src = reinterpret_cast<const V4*>(inv + (size_t)b * NP);
    // Direct global -> LDS loads (16 B per lane, one 1 KB chunk per wave and
    // instruction), all in flight together; lanes past the bank re-read its
    // last vector into the padding.
    const int wv = __builtin_amdgcn_readfirstlane(i / 64), lane = i % 64;
    T rv = R[(size_t)b * D + min(i, D - 1)];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int q0 = k * NT + wv * 64;
        __builtin_amdgcn_global_load_lds((gptr_t)(src + min(q0 + lane, NV - 1)), (lptr_t)(As + q0), 16, 0, 0);
    }
    __builtin_amdgcn_s_waitcnt(0);
    if (i < D) rs[i] = rv;
    __syncthreads();
    if (i >= D) return;
    const T* A = reinterpret_cast<const T*>(As);
    // Row i of the symmetric bank from the packed upper triangle: element
    // (j, i) for j <= i, then (i, j); the packed index advances by D - 1 - j
    // while j < i and by 1 after.
    T acc = 0;
    int idx = i;  // (0, i)
#pragma unroll 8
    for (int j = 0; j < D; ++j) {
        acc += A[idx] * rs[j];
        idx += (j < i) ? (D - 1 - j) : 1;
    }
    Z[(size_t)b * D + i] = acc;
}

// 16-vertex banks: one wavefront per bank
constexpr int kBankWaves = 4;
template <typename T>
__global__ void __launch_bounds__(64 * kBankWaves) k_bank_solve16(int nbanks, const T* __restrict__ inv,
                                                                  const T* __restrict__ R, T* __restrict__ Z,
                                                                  const int* __restrict__ ctrl, SceneSkip skip) {
    if (ctrl && ctrl[0]) return;
    __shared__ T lds[kBankWaves][kBankLds];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, b = blockIdx.x * kBankWaves + wv;
    if (b >= nbanks || skip.stopped(b)) return;
    BankSolve<T, T> B;
    B.load_r(R, b, lane);
    B.load(inv, nullptr, b, lane);
    const T z = B.solve(lds[wv], lane);
    if (lane < 48) Z[(size_t)b * 48 + lane] = z;
}

template <typename T>
__global__ void k_collect(int n, int L, const int* __restrict__ node_of, const T* __restrict__ Z,
                          double* __restrict__ z) {
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    T s0 = 0, s1 = 0, s2 = 0;
    for (int l = 0; l < L; ++l) {
        size_t g = (size_t)node_of[(size_t)l * n + v];
        s0 += Z[3 * g]; s1 += Z[3 * g + 1]; s2 += Z[3 * g + 2];
    }
    z[3 * (size_t)v] = (double)s0; z[3 * (size_t)v + 1] = (double)s1; z[3 * (size_t)v + 2] = (double)s2;
}

// Component sum of one bank-aligned group of nodes held in LDS (one node
// per thread).  `mask` holds the bank lanes of this node's component (its
// closure, self included); only the lowest lane of the component sums, in
// ascending lane order (U lanes' values are read at once; a lane outside the
// component adds nothing).  Returns true for that lane, with the sums.
template <typename T, int U = 16>
__device__ inline bool component_sum(unsigned mask, const T* a0, const T* a1, const T* a2, int B, T& s0, T& s1,
                                     T& s2) {
    const int t = threadIdx.x, lane = t & (B - 1), bbase = t - lane;
    if (mask & ltmask(lane)) return false;
    s0 = 0; s1 = 0; s2 = 0;
    for (int h = 0; h < B; h += U) {
        T q[U][3];
#pragma unroll
        for (int l = 0; l < U; ++l) {
            q[l][0] = a0[bbase + h + l];
            q[l][1] = a1[bbase + h + l];
            q[l][2] = a2[bbase + h + l];
        }
#pragma unroll
        for (int l = 0; l < U; ++l)
            if ((mask >> (h + l)) & 1u) { s0 += q[l][0]; s1 += q[l][1]; s2 += q[l][2]; }
    }
    return true;
}

// level-0 slots -> level-1 sums of the nodes of level-1 bank b, then
// level 1 -> 2 inside that bank.  `load(v)` reads what a vertex's level-0
// value needs and `value(v, ...)` gives it (and does what else the owner of v
// does).  A vertex is owned by exactly one workgroup: the one whose level-1
// bank holds the vertex's level-1 node.  Only the owner reads or writes the
// vertex's data, so a level-0 bank whose coarse nodes straddle two level-1
// banks is split between their workgroups with no slot touched twice (a
// component's lanes all share one level-1 node).  slot_node: vertex, level-1
// node and component lanes of every level-0 slot; comp_mask: component lanes
// of each coarse node.
// The loads of level-1 bank b that do not depend on the residual: its level-0
// slot range, the first slot chunk's entries and the level 1 -> 2 mapping of
// its nodes.  Issued before a kernel's partial-sum reduction, their latency
// overlaps it.
struct BankIdx {
    int lo, hi, q;
    SlotNode sn;
    unsigned mask2;
    bool valid;
};
__device__ inline BankIdx bank_index(int b, int B, int L, int cnt1, int beg1, const SlotNode* __restrict__ slot_node,
                                     const int* __restrict__ going_next, const unsigned* __restrict__ comp_mask,
                                     const int* __restrict__ l1lo, const int* __restrict__ l1hi) {
    const int t = threadIdx.x;
    BankIdx x;
    const int loc2 = b * B + t;
    x.lo = l1lo[b] * B;
    x.hi = l1hi[b] * B;
    x.valid = L >= 3 && t < B && loc2 < cnt1;
    x.q = -1;
    x.mask2 = 0u;
    if (x.valid) {
        x.q = going_next[(size_t)beg1 + loc2];
        x.mask2 = comp_mask[(size_t)beg1 + loc2];
    }
    const int sl = x.lo + t;
    x.sn = (sl < x.hi) ? slot_node[sl] : SlotNode{-1, -1, 0u, 0u};
    return x;
}

// this workgroup's (bank b's) own slot among those read
__device__ inline bool owned(const SlotNode& s, int b, int B) { return s.v >= 0 && (s.node & ~(B - 1)) == b * B; }

template <typename T, typename FL, typename FV>
__device__ inline void restrict_bank(int b, int B, int L, int beg1, const SlotNode* __restrict__ slot_node,
                                     const BankIdx& pre, T* __restrict__ R, T (*sv)[kTB], T (*l1v)[32], bool loaded,
                                     FL load, FV value) {
    const int t = threadIdx.x;
    const bool valid = pre.valid;
    const int lo = pre.lo, hi = pre.hi;
    for (int c0 = lo; c0 < hi; c0 += kTB) {
        const int sl = c0 + t;
        SlotNode sn = pre.sn;
        if (c0 != lo) sn = (sl < hi) ? slot_node[sl] : SlotNode{-1, -1, 0u, 0u};
        const bool own = owned(sn, b, B);
        T v0 = 0, v1 = 0, v2 = 0;
        if (own) {
            if (c0 != lo || !loaded) load(sn.v);
            value(sn.v, v0, v1, v2);
            R[3 * (size_t)sl] = v0; R[3 * (size_t)sl + 1] = v1; R[3 * (size_t)sl + 2] = v2;
        }
        sv[0][t] = v0; sv[1][t] = v1; sv[2][t] = v2;
        __syncthreads();
        T s0, s1, s2;
        if (own && component_sum<T>(sn.mask, sv[0], sv[1], sv[2], B, s0, s1, s2)) {
            size_t g = (size_t)beg1 + sn.node;
            R[3 * g] = s0; R[3 * g + 1] = s1; R[3 * g + 2] = s2;
            l1v[0][sn.node - b * B] = s0; l1v[1][sn.node - b * B] = s1; l1v[2][sn.node - b * B] = s2;
        }
        __syncthreads();
    }
    if (L < 3) return;
    // level 1 -> 2: nodes past the bank's last are in no component's mask
    T s0, s1, s2;
    if (valid && component_sum<T>(pre.mask2, l1v[0], l1v[1], l1v[2], B, s0, s1, s2)) {
        R[3 * (size_t)pre.q] = s0; R[3 * (size_t)pre.q + 1] = s1; R[3 * (size_t)pre.q + 2] = s2;
    }
}

// Multilevel restriction R_l = sum of children, levels 0 to 2 in one launch.
// Workgroup b owns level-1 bank b: it goes through the level-0 slots of every
// level-0 bank holding one of its children (slot_node), takes the residual r of
// those whose level-1 node lies in b (they alone are read, and written to R_0,
// here), forms its level-1 sums, and from them the level-2 nodes (whose children always
// lie in one level-1 bank).  Sum orders are those of the level-by-level
// component sums, so results do not depend on the schedule.
template <typename V, typename T>
__global__ void __launch_bounds__(kTB) k_restrict_all(const V* __restrict__ r, long long sub3, int B, int L,
                                                       const int* __restrict__ ls,
                                                       const SlotNode* __restrict__ slot_node,
                                                       const int* __restrict__ going_next,
                                                       const unsigned* __restrict__ comp_mask,
                                                       const int* __restrict__ l1lo, const int* __restrict__ l1hi,
                                                       T* __restrict__ R,
                                                       const int* __restrict__ ctrl, SceneSkip skip) {
    const BankIdx pre = bank_index(blockIdx.x, B, L, ls[2], ls[3], slot_node, going_next, comp_mask, l1lo, l1hi);
    if (ctrl && ctrl[0]) return;
    if (skip.bank_scene && skip.stopped(ls[3] / B + (int)blockIdx.x)) return;
    __shared__ T sv[3][kTB];
    __shared__ T l1v[3][32];
    V q0 = 0, q1 = 0, q2 = 0;
    auto load = [&](int v) {
        const V* rv = r + sub3 + 3 * (size_t)v;
        q0 = rv[0]; q1 = rv[1]; q2 = rv[2];
    };
    auto value = [&](int, T& v0, T& v1, T& v2) { v0 = (T)q0; v1 = (T)q1; v2 = (T)q2; };
    restrict_bank<T>(blockIdx.x, B, L, ls[3], slot_node, pre, R, sv, l1v, false, load, value);
}

// One PCG step fused with the restriction of its new residual:
// alpha = rz / p.Ap, x += alpha p, r -= alpha Ap, partials of r.r, and
// R_0..R_2 of the new r.  Workgroups [0, g1) walk the level-1 banks: each
// recomputes r for every vertex of its banks (identical arithmetic wherever
// a level-0 bank straddles two level-1 banks) and stores x, r and R_0 only
// for the banks it owns; workgroups [g1, grid) update the dofs outside the
// preconditioned range.  The iteration counter advances at the end.
// Bound by dependent round trips (606 workgroups at 137 k rows): the slot
// entries, the vectors of the first slots and both sets of dot partials are in
// flight before the stop word is looked at, one barrier joins both sums, and
// a component's lanes are summed from reads issued together.  At 137 k block
// rows 12.3 -> 8.4 us per launch in FP32, 14.4 -> 11.3 us in FP64; 7.5 -> 6.7 us
// at 525.
template <typename V, typename T>
__global__ void __launch_bounds__(kTB) k_update_restrict(
    long long N, double* __restrict__ x, V* __restrict__ r, const V* __restrict__ p, const V* __restrict__ Ap,
    const double* __restrict__ part_pap, int np_pap, const double* __restrict__ part_rz, int np_rz,
    double* __restrict__ part_rr, int* __restrict__ ctrl, int sub_off, int n_mas, int B, int L,
    const int* __restrict__ ls, const SlotNode* __restrict__ slot_node, const int* __restrict__ going_next,
    const unsigned* __restrict__ comp_mask, const int* __restrict__ l1lo,
    const int* __restrict__ l1hi, int nb1, int g1, T* __restrict__ R) {
    constexpr int NW = kTB / 64;
    __shared__ double sh[3 * NW];
    __shared__ T sv[3][kTB];
    __shared__ T l1v[3][32];
    const bool banked = (int)blockIdx.x < g1 && (int)blockIdx.x < nb1;
    const int stopped = ctrl[C_STOP], cnt1 = ls[2], beg1 = ls[3];
    Share<4, kTB> rz_share;
    Share<8, kTB> pap_share;
    rz_share.take(part_rz, np_rz);
    pap_share.take(part_pap, np_pap);
    // this workgroup's first bank: its indices, then its vertices' vectors
    BankIdx pre{0, 0, -1, SlotNode{-1, -1, 0u, 0u}, 0u, false};
    if (banked) pre = bank_index(blockIdx.x, B, L, cnt1, beg1, slot_node, going_next, comp_mask, l1lo, l1hi);
    V rv[3], av[3], pv[3];
    double xv[3];
    // only the vertex's owner reads and updates r in place (see restrict_bank)
    auto load = [&](int v) {
        const size_t o = 3 * ((size_t)sub_off + v);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            rv[k] = r[o + k];
            av[k] = Ap[o + k];
            pv[k] = p[o + k];
            xv[k] = x[o + k];
        }
    };
    if (owned(pre.sn, blockIdx.x, B)) load(pre.sn.v);
    if (stopped) return;
    wave_sums_put(rz_share.sum(), sh);
    wave_sums_put(pap_share.sum(), sh + NW);
    __syncthreads();
    const double al = wave_sums_total<NW>(sh) / wave_sums_total<NW>(sh + NW);
    double acc = 0.0;
    if ((int)blockIdx.x < g1) {
        auto value = [&](int v, T& v0, T& v1, T& v2) {
            const size_t o = 3 * ((size_t)sub_off + v);
            V rn[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                rn[k] = (V)((double)rv[k] - al * (double)av[k]);
                x[o + k] = xv[k] + al * (double)pv[k];
                r[o + k] = rn[k];
                acc += (double)rn[k] * (double)rn[k];
            }
            v0 = (T)rn[0]; v1 = (T)rn[1]; v2 = (T)rn[2];
        };
        for (int b = blockIdx.x; b < nb1; b += g1) {
            const bool at_first = b == (int)blockIdx.x;
            if (!at_first) {
                __syncthreads();  // the previous bank's level-1 sums have been read
                pre = bank_index(b, B, L, cnt1, beg1, slot_node, going_next, comp_mask, l1lo, l1hi);
            }
            restrict_bank<T>(b, B, L, beg1, slot_node, pre, R, sv, l1v, at_first, load, value);
        }
    } else {
        const long long m0 = 3LL * sub_off, m1 = 3LL * ((long long)sub_off + n_mas), nout = N - (m1 - m0);
        for (long long q = (long long)(blockIdx.x - g1) * kTB + threadIdx.x; q < nout;
             q += (long long)(gridDim.x - g1) * kTB) {
            long long i = q < m0 ? q : q + (m1 - m0);
            x[i] += al * (double)p[i];
            V ri = (V)((double)r[i] - al * (double)Ap[i]);
            r[i] = ri;
            acc += (double)ri * (double)ri;
        }
    }
    wave_sums_put(acc, sh + 2 * NW);
    __syncthreads();
    if (threadIdx.x == 0) {
        part_rr[blockIdx.x] = wave_sums_total<NW>(sh + 2 * NW);
        if (blockIdx.x == 0) ctrl[C_ITER] += 1;
    }
}

// Levels 2 -> 3 -> ... -> L-1 (few nodes): one workgroup, level by level.
// A level's sums stay in LDS as the next level's input when that level has
// at most kTop nodes; otherwise they are read back from R (written by this
// workgroup before a barrier).
constexpr int kTop = 1024;
template <typename T>
__global__ void __launch_bounds__(kTop) k_restrict_top(int B, int L, const int* __restrict__ ls,
                                                        const int* __restrict__ going_next,
                                                        const unsigned* __restrict__ comp_mask, T* __restrict__ R,
                                                        const int* __restrict__ ctrl) {
    if (ctrl && ctrl[0]) return;
    __shared__ T sv[3][kTop];
    __shared__ T nx[3][kTop];
    const int t = threadIdx.x;
    bool in_lds = false;  // this level's values are in nx
    for (int l = 2; l + 1 < L; ++l) {
        const int cnt = ls[2 * l], beg = ls[2 * l + 1], cntn = ls[2 * l + 2], begn = ls[2 * l + 3];
        const bool next_fits = cntn <= kTop;
        for (int c0 = 0; c0 < cnt; c0 += kTop) {
            int cc = c0 + t;
            bool valid = cc < cnt;
            size_t g = (size_t)beg + cc;
            int pp = valid ? going_next[g] : -1;
            unsigned mask = valid ? comp_mask[g] : 0u;
            T v0 = 0, v1 = 0, v2 = 0;
            if (valid) {
                if (in_lds) { v0 = nx[0][cc]; v1 = nx[1][cc]; v2 = nx[2][cc]; }
                else { v0 = R[3 * g]; v1 = R[3 * g + 1]; v2 = R[3 * g + 2]; }
            }
            __syncthreads();  // nx fully read before this pass overwrites it
            sv[0][t] = v0; sv[1][t] = v1; sv[2][t] = v2;
            __syncthreads();
            T s0, s1, s2;
            if (valid && component_sum<T>(mask, sv[0], sv[1], sv[2], B, s0, s1, s2)) {
                size_t q = (size_t)pp;
                R[3 * q] = s0; R[3 * q + 1] = s1; R[3 * q + 2] = s2;
                if (next_fits) { int j = (int)(q - begn); nx[0][j] = s0; nx[1][j] = s1; nx[2][j] = s2; }
            }
            __syncthreads();
        }
        in_lds = next_fits;
    }
}

// ---- top-level restriction overlapped with the bank solves (16-vertex banks) -
// k_mas_solve_top replaces k_restrict_top + k_bank_solve in a PCG iteration
// (the x/r update before it restricts levels 0..2; k_collect_dot follows):
// workgroup 0 restricts levels 2 -> L-1 (the sums of k_restrict_top) and
// then solves the banks of levels >= 3 on its own results; the other
// workgroups solve every bank of levels 0..2, whose restriction is complete
// at launch, at the same time.  No workgroup waits for another.
constexpr int kCW = 8;               // wavefronts per workgroup
constexpr int kCT = 64 * kCW;

// NB banks per wavefront of the other workgroups (levels 0 .. 2).  Bound by the
// inverses' bytes: 10,359 banks, 49 MB FP32 / 97 MB FP64, 13.2 -> 9.7 us and
// 20.0 -> 17.2 us per launch against staging packed triangles in LDS (a plain
// read of as many bytes takes about 8 and 15 us).
template <typename T, bool H, int NB>
__global__ void __launch_bounds__(kCT) k_mas_solve_top(int L, const int* __restrict__ ls,
                                                     const int* __restrict__ going_next,
                                                     const unsigned* __restrict__ comp_mask, int top_bank0,
                                                     int nbanks, const void* __restrict__ inv,
                                                     const float* __restrict__ dsc, T* __restrict__ R,
                                                     T* __restrict__ Z, const int* __restrict__ ctrl, SceneSkip skip) {
    static_assert(!H || sizeof(T) == 4, "half-storage inverses serve FP32 applies");
    using Solve = BankSolve<T, typename std::conditional<H, _Float16, T>::type>;
    constexpr int D = 48;
    static_assert(6 * kCT >= kCW * kBankLds, "one area for the restriction and the bank solves");
    __shared__ T lds[6 * kCT];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    T* mine = lds + kBankLds * wv;
    const int stopped = ctrl[C_STOP];
    if (blockIdx.x == 0) {
        // this wavefront's first top bank, loaded while the levels are restricted
        Solve B;
        const int b0 = top_bank0 + wv;
        B.load(inv, dsc, min(b0, nbanks - 1), lane);
        if (stopped) return;
        // levels 2 -> L-1, one level at a time (the sums of k_restrict_top)
        T(*sv)[kCT] = reinterpret_cast<T(*)[kCT]>(lds);
        T(*nx)[kCT] = reinterpret_cast<T(*)[kCT]>(lds + 3 * kCT);
        const int t = threadIdx.x;
        bool in_lds = false;
        for (int l = 2; l + 1 < L; ++l) {
            const int cnt = ls[2 * l], beg = ls[2 * l + 1], cntn = ls[2 * l + 2], begn = ls[2 * l + 3];
            const bool next_fits = cntn <= kCT;
            for (int c0 = 0; c0 < cnt; c0 += kCT) {
                const int cc = c0 + t;
                const bool valid = cc < cnt;
                const size_t g = (size_t)beg + cc;
                const int pp = valid ? going_next[g] : -1;
                const unsigned mask = valid ? comp_mask[g] : 0u;
                T v0 = 0, v1 = 0, v2 = 0;
                if (valid) {
                    if (in_lds) { v0 = nx[0][cc]; v1 = nx[1][cc]; v2 = nx[2][cc]; }
                    else { v0 = R[3 * g]; v1 = R[3 * g + 1]; v2 = R[3 * g + 2]; }
                }
                __syncthreads();
                sv[0][t] = v0; sv[1][t] = v1; sv[2][t] = v2;
                __syncthreads();
                T s0, s1, s2;
                if (valid && component_sum<T, 4>(mask, sv[0], sv[1], sv[2], 16, s0, s1, s2)) {
                    const size_t q = (size_t)pp;
                    R[3 * q] = s0; R[3 * q + 1] = s1; R[3 * q + 2] = s2;
                    if (next_fits) { const int j = (int)(q - begn); nx[0][j] = s0; nx[1][j] = s1; nx[2][j] = s2; }
                }
                __syncthreads();
            }
            in_lds = next_fits;
        }
        // the top banks, on this workgroup's restriction (R written above;
        // the barrier orders this workgroup's global writes and reads)
        __threadfence_block();
        __syncthreads();
        if (b0 < nbanks && !skip.stopped(b0)) {
            B.load_r(R, b0, lane);
            const T zb = B.solve(mine, lane);
            if (lane < D) Z[(size_t)b0 * D + lane] = zb;
        }
        for (int b = b0 + kCW; b < nbanks; b += kCW) {
            if (skip.stopped(b)) continue;
            Solve C;
            C.load(inv, dsc, b, lane);
            C.load_r(R, b, lane);
            const T zb = C.solve(mine, lane);
            if (lane < D) Z[(size_t)b * D + lane] = zb;
        }
        return;
    }
    Solve B[NB];
    bool on[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) {
        const int b = ((blockIdx.x - 1) * NB + k) * kCW + wv;
        on[k] = b < top_bank0 && !skip.stopped(b);
        if (on[k]) {
            B[k].load_r(R, b, lane);
            B[k].load(inv, dsc, b, lane);
        }
    }
    if (stopped) return;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
        if (!on[k]) continue;
        const int b = ((blockIdx.x - 1) * NB + k) * kCW + wv;
        const T zb = B[k].solve(mine, lane);
        if (lane < D) Z[(size_t)b * D + lane] = zb;
    }
}

// level-0 bank range of each level-1 bank (children of its nodes), and the
// vertices [vlo, vhi) of the level-0 banks whose first node it holds (vertex
// ids in slot order); a lane per slot, one of each bank writes
__global__ void __launch_bounds__(kTB) k_l1_ranges(int M, int B, const int* __restrict__ prefix0,
                                                   const int* __restrict__ psum0, const int* __restrict__ part_map,
                                                   int* __restrict__ lo, int* __restrict__ hi, int* __restrict__ vlo,
                                                   int* __restrict__ vhi) {
    const int s = blockIdx.x * kTB + threadIdx.x, cb = s / B;
    const bool in = s < M;  // (M is a multiple of B)
    const int v = in ? part_map[s] : -1, first = in ? psum0[cb] : 0, cnt = in ? prefix0[cb] : 0;
    int mn = v >= 0 ? v : 0x7fffffff, mx = v;
    for (int off = B / 2; off > 0; off >>= 1) {
        mn = min(mn, __shfl_xor(mn, off));
        mx = max(mx, __shfl_xor(mx, off));
    }
    if (s % B != 0 || cnt <= 0) return;
    const int f = first / B, e = (first + cnt - 1) / B;
    for (int b = f; b <= e; ++b) {
        atomicMin(lo + b, cb);
        atomicMax(hi + b, cb + 1);
    }
    if (mx >= 0) {
        atomicMin(vlo + f, mn);
        atomicMax(vhi + f, mx + 1);
    }
}

// ---- the whole numbering in one workgroup -----------------------------------
// Systems of up to kSmallN vertices, kSmallM slots, kSmallList neighbours and
// kSmallPairs contact pairs: every table of the hierarchy in one launch, with
// the integers of the level-by-level kernels above.  Those take seven or eight
// launches a level, 2 to 5 us each however small the level; here the neighbour
// lists (16-bit), the masks and the vertices' nodes of the current level live
// in LDS, a phase ends with a barrier, and only the tables go to memory.
// Latency-bound: 20 us at 125 vertices and 59 us at 1331, where the launches
// it replaces (about 40) took 90 and 150 us of a step.  A whole build, this
// launch against those: 76 and 140 us at 125 vertices, 94 and 152 at 512, 120 and
// 164 at 1000, 128 and 167 at 1331, 161 and 175 at 1728, 172 and 188 at 2000.
// Above 2048 vertices (two per thread) one CU is too few: 369 us against 170 at
// 5488 vertices, with the lists read from memory because they no longer fit LDS.
constexpr int kSmallT = 1024;
constexpr int kSmallN = 2048;
constexpr int kSmallM = 4096;
constexpr int kSmallPairs = 4096;
constexpr int kSmallList = 40960;       // 80 KB of the 112 KB of LDS in use
constexpr int kSmallV = kSmallN / kSmallT;
static_assert(kSmallM / 16 <= kSmallT, "one scan step holds the banks of a level");

struct SmallTables {
    int M, Mpad, n, B, L, node_offset, npairs, nb1_cap, nlist_len;
    const int *part_map, *real_map;
    const unsigned *nstart, *nnum, *nlist;
    const int4* pairs;
    int *ls, *going_next, *coarse_space, *coarse_table, *node_of, *prefix0, *psum0, *l1lo, *l1hi, *own_lo, *own_hi;
    unsigned *fine_mask, *comp_mask;
    SlotNode* slot_node;
    size_t going_cap;
};

// exclusive scan of cnt entries (at most kSmallT) of v in LDS, in place; returns the total
__device__ inline int small_scan(int* v, int cnt, int* sh) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int mine = t < cnt ? v[t] : 0;
    int incl = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int u = __shfl_up(incl, off, 64);
        if (lane >= off) incl += u;
    }
    if (lane == 63) sh[w] = incl;
    __syncthreads();
    int before = 0, total = 0;
    for (int q = 0; q < kSmallT / 64; ++q) {
        if (q < w) before += sh[q];
        total += sh[q];
    }
    if (t < cnt) v[t] = before + incl - mine;
    __syncthreads();
    return total;
}

__global__ void __launch_bounds__(kSmallT) k_small_tables(SmallTables A) {
    __shared__ unsigned fm[kSmallN];    // level-0 masks by vertex
    __shared__ unsigned nm[kSmallN];    // this level's masks, then next ids, by node
    __shared__ int cs[kSmallN];         // the vertices' slots, then their nodes at this level
    __shared__ unsigned short nl[kSmallList];
    __shared__ unsigned sm[kSmallT];
    __shared__ int pre[kSmallT];        // components per bank, then their scan
    __shared__ int sh[kSmallT / 64];
    const int t = threadIdx.x, n = A.n, M = A.M, B = A.B, L = A.L;
    const int lb = __ffs(B) - 1;  // ids are divided by shifts
    const int lane = t & (B - 1), bbase = t - lane;
    for (size_t i = t; i < A.going_cap; i += kSmallT) A.going_next[i] = 0;
    for (int i = t; i < 2 * (L + 2); i += kSmallT) A.ls[i] = 0;
    for (int i = t; i <= A.nb1_cap; i += kSmallT) {
        A.l1lo[i] = M >> lb;
        A.l1hi[i] = 0;
        A.own_lo[i] = 0x7fffffff;
        A.own_hi[i] = 0;
    }
    unsigned nst[kSmallV], nnn[kSmallV];  // neighbour ranges of this thread's vertices
#pragma unroll
    for (int j = 0; j < kSmallV; ++j) {
        const int v = t + j * kSmallT;
        nst[j] = v < n ? A.nstart[v] : 0u;
        nnn[j] = v < n ? A.nnum[v] : 0u;
        if (v < n) cs[v] = A.real_map[v];
    }
    for (int i = t; i < A.nlist_len; i += kSmallT) nl[i] = (unsigned short)A.nlist[i];
    __syncthreads();  // the lists are whole; none of the cleared tables is written before
    // the vertex's own bit and its neighbours' in the same bank
    auto bank_mask = [&](int v, unsigned st, unsigned nn) {
        const int c = cs[v], bank = c >> lb;
        unsigned msk = 1u << (c & (B - 1));
        for (unsigned i = 0; i < nn; ++i) {
            const int cu = cs[nl[st + i]];
            if ((cu >> lb) == bank) msk |= 1u << (cu & (B - 1));
        }
        return msk;
    };
#pragma unroll
    for (int j = 0; j < kSmallV; ++j) {
        const int v = t + j * kSmallT;
        if (v < n) fm[v] = bank_mask(v, nst[j], nnn[j]);
    }
    __syncthreads();
    // contact pairs: every two nodes of a pair that share a bank are connected
    auto collide = [&](bool level0, unsigned* dst) {
        for (int p = t; p < A.npairs; p += kSmallT) {
            int v[4], cp[4];
            const int cnt = decode_pair(A.pairs[p], A.node_offset, v);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                cp[i] = (i >= cnt || v[i] < 0 || v[i] >= n) ? -1 : cs[v[i]];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                unsigned msk = 0u;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (j != i && cp[i] >= 0 && cp[j] >= 0 && cp[i] != cp[j] && (cp[i] >> lb) == (cp[j] >> lb))
                        msk |= 1u << (cp[j] & (B - 1));
                if (msk) atomicOr(dst + (level0 ? v[i] : cp[i]), msk);
            }
        }
        __syncthreads();
    };
    collide(true, fm);
    // closure in every bank and its component count; fm is read and written
    // by the vertex's own thread only
    const int nb0 = M >> lb;
    for (int s0 = 0; s0 < M; s0 += kSmallT) {
        const int s = s0 + t, v = s < M ? A.part_map[s] : -1;
        sm[t] = v >= 0 ? fm[v] : 0u;
        __syncthreads();
        unsigned cl = 0u;
        if (v >= 0) {
            cl = closure(sm[t], lane, sm + bbase);
            fm[v] = cl;
            A.fine_mask[v] = cl;
        }
        const unsigned long long lead = __ballot(v >= 0 && (cl & ltmask(lane)) == 0u);
        if (lane == 0 && s < M) {
            const int c = __popcll((lead >> (t & 63)) & ((1ull << B) - 1ull));
            pre[s >> lb] = c;
            A.prefix0[s >> lb] = c;
        }
        __syncthreads();
    }
    int total = small_scan(pre, nb0, sh);
    // level-1 nodes
    int begin = A.Mpad, number = total;
    for (int s0 = 0; s0 < M; s0 += kSmallT) {
        const int s = s0 + t, v = s < M ? A.part_map[s] : -1;
        const unsigned f = v >= 0 ? fm[v] : 0u;
        const unsigned long long lead = __ballot(v >= 0 && (f & ltmask(lane)) == 0u);
        if (v >= 0) {
            const unsigned elected = (unsigned)((lead >> ((t & 63) - lane)) & ((1ull << B) - 1ull));
            const int id = __popc(elected & ltmask(lowbit(f))) + pre[s >> lb];
            cs[v] = id;
            A.coarse_space[v] = id;
            A.going_next[v] = id + A.Mpad;
            A.slot_node[s] = SlotNode{v, id, f, 0u};
            A.node_of[v] = A.real_map[v];
            A.node_of[(size_t)n + v] = begin + id;  // (L >= 2 always)
            A.coarse_table[6 * (size_t)v] = begin + id;
            for (int l = L - 1; l < 6; ++l) A.coarse_table[6 * (size_t)v + l] = 0;
            // vertices owned by the level-1 bank of the level-0 bank's first node
            const int f1 = pre[s >> lb] >> lb;
            atomicMin(A.own_lo + f1, v);
            atomicMax(A.own_hi + f1, v + 1);
        } else if (s < M) {
            A.slot_node[s] = SlotNode{-1, -1, 0u, 0u};
        }
        if (lane == 0 && s < M) {
            const int first = pre[s >> lb], last = ((s >> lb) + 1 < nb0 ? pre[(s >> lb) + 1] : total) - 1;
            A.psum0[s >> lb] = first;
            for (int b = first >> lb; first <= last && b <= last >> lb; ++b) {
                atomicMin(A.l1lo + b, s >> lb);
                atomicMax(A.l1hi + b, (s >> lb) + 1);
            }
        }
    }
    if (t == 0) {
        A.psum0[nb0] = total;
        A.ls[2] = total;
        A.ls[3] = A.Mpad;
    }
    for (int level = 1; level < L; ++level) {
        __syncthreads();
        for (int c = t; c < number; c += kSmallT) nm[c] = 0u;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kSmallV; ++j) {
            const int v = t + j * kSmallT;
            if (v < n) atomicOr(nm + cs[v], bank_mask(v, nst[j], nnn[j]));
        }
        __syncthreads();
        collide(false, nm);
        const int nbk = (number + B - 1) >> lb, pad = nbk * B;
        for (int c0 = 0; c0 < number; c0 += kSmallT) {
            const int c = c0 + t;
            const bool valid = c < number;
            sm[t] = valid ? ((1u << lane) | nm[c]) : 0u;
            __syncthreads();
            unsigned cl = 0u;
            if (valid) {
                cl = closure(sm[t], lane, sm + bbase);
                nm[c] = cl;
                A.comp_mask[(size_t)begin + c] = cl;
            }
            const unsigned long long lead = __ballot(valid && (cl & ltmask(lane)) == 0u);
            if (lane == 0 && valid) pre[c >> lb] = __popcll((lead >> (t & 63)) & ((1ull << B) - 1ull));
            __syncthreads();
        }
        total = small_scan(pre, nbk, sh);
        for (int c0 = 0; c0 < number; c0 += kSmallT) {
            const int c = c0 + t;
            const bool valid = c < number;
            const unsigned cm = valid ? nm[c] : 0u;
            const unsigned long long lead = __ballot(valid && (cm & ltmask(lane)) == 0u);
            if (valid) {
                const unsigned elected = (unsigned)((lead >> ((t & 63) - lane)) & ((1ull << B) - 1ull));
                const int id = __popc(elected & ltmask(lowbit(cm))) + pre[c >> lb];
                nm[c] = (unsigned)id;
                if ((size_t)begin + c < A.going_cap) A.going_next[(size_t)begin + c] = id + begin + pad;
            }
        }
        __syncthreads();
        begin += pad;
        for (int v = t; v < n; v += kSmallT) {
            const int id = (int)nm[cs[v]];
            cs[v] = id;
            A.coarse_space[(size_t)level * n + v] = id;
            if (level + 1 < L) {
                A.node_of[(size_t)(level + 1) * n + v] = begin + id;
                A.coarse_table[6 * (size_t)v + level] = begin + id;
            }
        }
        number = total;
        if (t == 0) {
            A.ls[2 * (level + 1)] = total;
            A.ls[2 * (level + 1) + 1] = begin;
        }
    }
}

int num_levels(int nn, int B) {
    int nLevel = 1;
    int levelSz = (nn + B - 1) / B * B;
    while (levelSz > B) {
        levelSz /= B;
        nLevel++;
        levelSz = (levelSz + B - 1) / B * B;
    }
    nLevel = nLevel + 1;
    return nLevel > 6 ? 6 : nLevel;
}

template <typename V, typename T>
void mas_restrict_t(Ctx& c, const V* r, long long sub3, T* R, const int* ctrl, bool top = true,
                    SceneSkip skip = SceneSkip{}) {
    MasState& m = c.mas;
    if (m.nb1 <= 0) return;
    hipLaunchKernelGGL((k_restrict_all<V, T>), dim3(m.nb1), dim3(kTB), 0, c.stream, r, sub3, m.bank, m.L,
                       (const int*)m.level_size.p, (const SlotNode*)m.slot_node.p, (const int*)m.going_next.p,
                       (const unsigned*)m.comp_mask.p, (const int*)m.l1lo.p, (const int*)m.l1hi.p, R, ctrl, skip);
    SGIPC_LAUNCH_CHECK();
    if (top && m.L >= 4) {
        hipLaunchKernelGGL((k_restrict_top<T>), dim3(1), dim3(kTop), 0, c.stream, m.bank, m.L,
                           (const int*)m.level_size.p, (const int*)m.going_next.p, (const unsigned*)m.comp_mask.p, R, ctrl);
        SGIPC_LAUNCH_CHECK();
    }
}

template <typename T>
void mas_solve_t(Ctx& c, const T* inv, const T* R, T* Z, const int* ctrl, SceneSkip skip = SceneSkip{}) {
    MasState& m = c.mas;
    prof_begin(c, PROF_MAS_SOLVE);
    if (m.bank == 16)
        hipLaunchKernelGGL(k_bank_solve16<T>, dim3(div_up(m.nbanks, kBankWaves)), dim3(64 * kBankWaves), 0, c.stream,
                           m.nbanks, inv, R, Z, ctrl, skip);
    else
        hipLaunchKernelGGL(k_bank_solve32<T>, dim3(m.nbanks), dim3(128), 0, c.stream, inv, R, Z, ctrl, skip);
    SGIPC_LAUNCH_CHECK();
    prof_end(c, PROF_MAS_SOLVE);
}

template <typename T>
void mas_apply_t(Ctx& c, const double* r, double* z, T* R, T* Z, const T* inv) {
    MasState& m = c.mas;
    hipStream_t s = c.stream;
    if (m.n <= 0) return;
    mas_restrict_t<double, T>(c, r, 0, R, nullptr);
    mas_solve_t<T>(c, inv, R, Z, nullptr);
    hipLaunchKernelGGL(k_collect<T>, dim3(div_up(m.n, 256)), dim3(256), 0, s, m.n, m.L, m.node_of.p, Z, z);
    SGIPC_LAUNCH_CHECK();
}

}  // namespace

void mas_set_topology(Ctx& c, int n, int node_offset, const unsigned* nstart, const unsigned* nnum,
                      const unsigned* nlist, int nlist_len, const int* part_map, int M, const int* real_map,
                      int bank) {
    if (bank != 16 && bank != 32) throw arg_error("MAS bank size must be 16 or 32");
    if (n < 0 || M < 0 || M % bank != 0) throw arg_error("MAS map size must be a multiple of the bank size");
    if (nlist_len < 0) throw arg_error("negative neighbour list length");
    // validate the maps and neighbour indices on the host
    for (int v = 0; v < n; ++v) {
        int sl = real_map[v];
        if (sl < 0 || sl >= M || part_map[sl] != v) throw arg_error("MAS real_map/part_map inconsistent");
        if ((long long)nstart[v] + nnum[v] > nlist_len) throw arg_error("MAS neighbour CSR out of range");
    }
    bool padded = false;  // ids with the top bit set are no neighbours
    for (int i = 0; i < nlist_len; ++i) {
        if ((int)nlist[i] >= n) throw arg_error("MAS neighbour index out of range");
        padded = padded || (int)nlist[i] < 0;
    }
    for (int s2 = 0; s2 < M; ++s2)
        if (part_map[s2] >= n) throw arg_error("MAS part_map entry out of range");
    MasState& m = c.mas;
    m.ready = false;
    m.bank = bank;
    m.n = n;
    m.slot_ordered = true;  // vertex ids increase with their bank slot
    for (int v = 1; v < n; ++v)
        if (real_map[v] <= real_map[v - 1]) { m.slot_ordered = false; break; }
    m.node_offset = node_offset;
    m.M = M;
    m.nlist_len = nlist_len;
    m.nlist_padded = padded;
    m.L = num_levels(std::max(M, n), bank);
    int Mpad = (M + bank - 1) / bank * bank;
    m.going_cap = (size_t)Mpad + (size_t)m.L * ((size_t)n + bank) + bank;
    m.part_map.reserve((size_t)M + 1);
    m.real_map.reserve((size_t)n + 1);
    m.nstart.reserve((size_t)n + 1);
    m.nnum.reserve((size_t)n + 1);
    m.nlist.reserve((size_t)nlist_len + 1);
    if (M) SGIPC_HIP(hipMemcpy(m.part_map.p, part_map, sizeof(int) * M, hipMemcpyHostToDevice));
    if (n) {
        SGIPC_HIP(hipMemcpy(m.real_map.p, real_map, sizeof(int) * n, hipMemcpyHostToDevice));
        SGIPC_HIP(hipMemcpy(m.nstart.p, nstart, sizeof(unsigned) * n, hipMemcpyHostToDevice));
        SGIPC_HIP(hipMemcpy(m.nnum.p, nnum, sizeof(unsigned) * n, hipMemcpyHostToDevice));
    }
    if (nlist_len) SGIPC_HIP(hipMemcpy(m.nlist.p, nlist, sizeof(unsigned) * nlist_len, hipMemcpyHostToDevice));
    m.fine_mask.reserve((size_t)n + 1);
    m.slot_node.reserve((size_t)M + 1);
    m.next_mask.reserve(2 * ((size_t)n + bank));
    m.outer.reserve((size_t)n + 1);
    size_t nbk = (size_t)std::max(M, n) / bank + 2;
    m.prefix0.reserve(nbk);
    m.psum0.reserve(nbk + 1);
    m.next_prefix.reserve(nbk);
    m.next_psum.reserve(nbk + 1);
    m.level_size.reserve(2 * ((size_t)m.L + 2));
    m.coarse_space.reserve((size_t)m.L * n + 1);
    m.going_next.reserve(m.going_cap);
    m.comp_mask.reserve(m.going_cap);
    m.coarse_table.reserve(6 * (size_t)n + 1);
    m.node_of.reserve((size_t)m.L * n + 1);
    m.level_size_h.assign(2 * ((size_t)m.L + 2), 0);
}

void mas_build(Ctx& c, int sub_offset, int sub_nb, const int* pairs, int npairs) {
    MasState& m = c.mas;
    if (!c.have_bcoo) throw state_error("MAS build: convert the system first");
    if (m.M == 0 && m.n == 0) throw state_error("MAS build: topology not set");
    hipStream_t s = c.stream;
    const int n = m.n, M = m.M, B = m.bank, L = m.L;
    const int Mpad = (M + B - 1) / B * B;
    if (sub_nb != n) throw arg_error("MAS build: subsystem block count differs from the MAS topology");
    m.ready = false;
    int* ls = m.level_size.p;
    const int nb1_cap = div_up(n, B);
    int* l1lo = m.l1lo.reserve((size_t)nb1_cap + 2);
    int* l1hi = m.l1hi.reserve((size_t)nb1_cap + 2);
    int* vlo = m.own_lo.reserve((size_t)nb1_cap + 2);
    int* vhi = m.own_hi.reserve((size_t)nb1_cap + 2);
    // (its 16-bit lists have no room for padding)
    const bool small = n > 0 && n <= kSmallN && M <= kSmallM && m.nlist_len <= kSmallList && !m.nlist_padded &&
                       npairs <= kSmallPairs;
    if (small) {
        hipLaunchKernelGGL(k_small_tables, dim3(1), dim3(kSmallT), 0, s,
                           (SmallTables{M, Mpad, n, B, L, m.node_offset, npairs, nb1_cap, m.nlist_len, m.part_map.p, m.real_map.p,
                                        m.nstart.p, m.nnum.p, m.nlist.p, (const int4*)pairs, ls, m.going_next.p,
                                        m.coarse_space.p, m.coarse_table.p, m.node_of.p, m.prefix0.p, m.psum0.p, l1lo,
                                        l1hi, vlo, vhi, m.fine_mask.p, m.comp_mask.p, m.slot_node.p, m.going_cap}));
        SGIPC_LAUNCH_CHECK();
    } else {
        // the masks of a level: two buffers, the next level's cleared while this one's is read
        const size_t mask_len = (size_t)n + B;
        FillRanges f;
        f.add(ls, 0u, 2LL * (L + 2)).add(m.going_next.p, 0u, (long long)m.going_cap);
        fill_ranges(f.add(m.next_mask.p, 0u, (long long)mask_len), s);
        // level 0
        hipLaunchKernelGGL(k_l0_masks, dim3(div_up(M, 256)), dim3(256), 0, s, M, B, m.part_map.p, m.real_map.p, m.nstart.p,
                           m.nnum.p, m.nlist.p, m.fine_mask.p);
        SGIPC_LAUNCH_CHECK();
        if (npairs > 0) {
            hipLaunchKernelGGL(k_collision, dim3(div_up(npairs, kOrT)), dim3(kOrT), 0, s, npairs, (const int4*)pairs,
                               m.node_offset, n, B, -1, ls, m.real_map.p, m.coarse_space.p, m.fine_mask.p);
            SGIPC_LAUNCH_CHECK();
        }
        hipLaunchKernelGGL(k_l0_closure, dim3(div_up(M, kTB)), dim3(kTB), 0, s, M, B, m.part_map.p, m.fine_mask.p,
                           m.prefix0.p);
        SGIPC_LAUNCH_CHECK();
        int* tot = c.dev_int.reserve(8);
        exclusive_scan(c, m.prefix0.p, m.psum0.p, M / B, tot + 6, s);
        hipLaunchKernelGGL(k_level1, dim3(div_up(M, kTB)), dim3(kTB), 0, s, M, Mpad, n, B, m.part_map.p, m.fine_mask.p,
                           m.psum0.p, m.coarse_space.p, m.going_next.p, m.slot_node.p, (const int*)(tot + 6), ls);
        SGIPC_LAUNCH_CHECK();
        const int nmax = n;  // level-local node count never exceeds n
        for (int level = 1; level < L; ++level) {
            unsigned* next = m.next_mask.p + (level & 1 ? 0 : mask_len);
            unsigned* other = m.next_mask.p + (level & 1 ? mask_len : 0);
            hipLaunchKernelGGL(k_lx_masks, dim3(div_up(n, kOrT)), dim3(kOrT), 0, s, n, B, level, ls, m.nstart.p, m.nnum.p,
                               m.nlist.p, m.coarse_space.p, next, m.outer.p);
            SGIPC_LAUNCH_CHECK();
            if (npairs > 0) {
                hipLaunchKernelGGL(k_collision, dim3(div_up(npairs, kOrT)), dim3(kOrT), 0, s, npairs, (const int4*)pairs,
                                   m.node_offset, n, B, level, ls, m.real_map.p, m.coarse_space.p, next);
                SGIPC_LAUNCH_CHECK();
            }
            int nbk = div_up(nmax, B);
            hipLaunchKernelGGL(k_lx_closure, dim3(div_up((long long)nbk * B, kTB)), dim3(kTB), 0, s, nbk * B, B, level, ls,
                               next, m.next_prefix.p, m.comp_mask.p);
            SGIPC_LAUNCH_CHECK();
            exclusive_scan(c, m.next_prefix.p, m.next_psum.p, nbk, tot + 6, s);
            hipLaunchKernelGGL(k_lx_renumber, dim3(div_up((long long)nbk * B, kTB)), dim3(kTB), 0, s, B, level, ls,
                               (const int*)(tot + 6), next, m.next_psum.p, m.going_next.p, m.going_cap);
            SGIPC_LAUNCH_CHECK();
            hipLaunchKernelGGL(k_next_table, dim3(div_up((long long)mask_len, 256)), dim3(256), 0, s, n, level,
                               m.coarse_space.p, (const unsigned*)next, other, (int)mask_len);
            SGIPC_LAUNCH_CHECK();
        }
        hipLaunchKernelGGL(k_aggregate, dim3(div_up(n, 256)), dim3(256), 0, s, n, L, m.real_map.p, m.going_next.p,
                           m.coarse_table.p, m.node_of.p);
        SGIPC_LAUNCH_CHECK();
    }
    SGIPC_HIP(hipMemcpyAsync(m.level_size_h.data(), ls, sizeof(int) * 2 * (L + 1), hipMemcpyDeviceToHost, s));
    SGIPC_HIP(hipStreamSynchronize(s));
    m.total = m.level_size_h[2 * L + 1];
    if (m.total <= 0 || m.total % B) throw state_error("MAS build: inconsistent cluster count");
    m.nbanks = m.total / B;
    const int npack = B * (B + 1) / 2;
    const int D = 3 * B;
    m.bank_upper.reserve((size_t)m.nbanks * npack * 9);
    m.inv64.reserve((size_t)m.nbanks * (D * (D + 1) / 2));
    m.inv32.reserve((size_t)m.nbanks * (D * (D + 1) / 2));
    // apply work vectors: allocated here so their addresses are stable for
    // captured PCG graphs; padding entries stay zero (never written)
    m.R64.reserve(3 * (size_t)m.total + 3);
    m.Z64.reserve(3 * (size_t)m.total + 3);
    m.R32.reserve(3 * (size_t)m.total + 3);
    m.Z32.reserve(3 * (size_t)m.total + 3);
    m.nb1 = div_up(m.level_size_h[2], B);
    {
        // bank matrices and residuals to zero; level-0 bank ranges and owned
        // vertices of the level-1 banks
        FillRanges f;
        f.add(m.bank_upper.p, 0u, (long long)m.nbanks * npack * 9).add(m.R64.p, 0u, 3LL * m.total + 3);
        f.add(m.R32.p, 0u, 3LL * m.total + 3);
        const int nb0 = M / B;
        if (small) {
            fill_ranges(f, s);
        } else {
            FillRanges g;
            g.add(l1lo, (unsigned)nb0, m.nb1 + 1).add(l1hi, 0u, m.nb1 + 1).add(vlo, 0x7fffffffu, m.nb1 + 1);
            g.add(vhi, 0u, m.nb1 + 1);
            fill_ranges(f, s);
            fill_ranges(g, s);
            if (nb0 > 0) {
                hipLaunchKernelGGL(k_l1_ranges, dim3(div_up(M, kTB)), dim3(kTB), 0, s, M, B, m.prefix0.p, m.psum0.p,
                                   m.part_map.p, l1lo, l1hi, vlo, vhi);
                SGIPC_LAUNCH_CHECK();
            }
        }
    }
    // The banked projection (16-vertex banks, vertex ids in slot order) sums
    // coarse levels in LDS with few atomics; every other case -- and the
    // deterministic mode -- uses the ordered projection, which sorts
    // (entry, block) records and sums each entry in a fixed order: no atomic
    // contention where many fine blocks land on few coarse entries
    // (32-vertex banks: 23 ms with global FP64 atomics at 137 k vertices).
    const bool banked = (B == 16) && m.slot_ordered && m.nb1 > 0 && L >= 2;
    if (c.K > 0 && (c.deterministic || !banked)) {
        if ((long long)c.K >= (1LL << 29)) throw capacity_error("MAS build: too many blocks for the ordered projection");
        const unsigned sentinel = (unsigned)((long long)m.nbanks * npack);
        int bits = 1;
        while (bits < 32 && (1ULL << bits) <= (unsigned long long)sentinel) ++bits;
        const long long mrec = (long long)c.K * std::max(L - 1, 0);
        if (L > 1) {
            unsigned* key = m.proj_key.reserve(2 * (size_t)mrec);
            unsigned* rec = m.proj_rec.reserve(2 * (size_t)mrec);
            hipLaunchKernelGGL(k_proj_records, dim3(div_up(c.K, 256)), dim3(256), 0, s, c.K, (const int*)c.t_rows,
                               (const int*)c.t_cols, (const double*)c.t_vals, sub_offset, n, B, L,
                               (const int*)m.node_of.p, m.bank_upper.p, sentinel, key, rec);
            SGIPC_LAUNCH_CHECK();
            if (c.sort_impl == SORT_OWN) {
                radix_sort_pairs(c, key, key + mrec, (const int*)rec, 0, (int*)(rec + mrec), mrec, bits, s);
            } else {  // rocPRIM as the cross-check
                size_t bytes = 0;
                SGIPC_HIP(rocprim::radix_sort_pairs(nullptr, bytes, key, key + mrec, rec, rec + mrec, (size_t)mrec, 0,
                                                    bits, s));
                void* tmp = m.proj_sort_tmp.reserve(bytes + 1);
                SGIPC_HIP(rocprim::radix_sort_pairs(tmp, bytes, key, key + mrec, rec, rec + mrec, (size_t)mrec, 0,
                                                    bits, s));
            }
            const int ntiles = div_up(mrec, kProjTile);
            double* part = m.proj_part.reserve(18 * (size_t)ntiles);
            const unsigned* skey = key + mrec;
            hipLaunchKernelGGL(k_proj_tiles, dim3(ntiles), dim3(kProjTile), 0, s, mrec, skey,
                               (const unsigned*)(rec + mrec), (const int*)c.t_rows, (const int*)c.t_cols,
                               (const double*)c.t_vals, sub_offset, n, B, (const int*)m.node_of.p, sentinel,
                               m.bank_upper.p, part);
            SGIPC_LAUNCH_CHECK();
            hipLaunchKernelGGL(k_proj_carry, dim3(div_up(16LL * ntiles, 256)), dim3(256), 0, s, mrec, ntiles, skey,
                               sentinel, (const double*)part, m.bank_upper.p);
            SGIPC_LAUNCH_CHECK();
        } else {
            hipLaunchKernelGGL(k_proj_records, dim3(div_up(c.K, 256)), dim3(256), 0, s, c.K, (const int*)c.t_rows,
                               (const int*)c.t_cols, (const double*)c.t_vals, sub_offset, n, B, L,
                               (const int*)m.node_of.p, m.bank_upper.p, sentinel, (unsigned*)nullptr,
                               (unsigned*)nullptr);
            SGIPC_LAUNCH_CHECK();
        }
    } else if (c.K > 0 && banked) {
        // top levels: the highest levels whose banks fit kProjTopBanksMax
        // (the kernel with kProjTopBanks of them, when they fit, runs two
        // workgroups per CU; a level left out goes to global atomics)
        int top_lvl = L, top_lo = m.nbanks, top_nb = 0;
        for (int l = L - 1; l >= 1; --l) {
            int beg = m.level_size_h[2 * l + 1] / B;
            int end = m.level_size_h[2 * (l + 1) + 1] / B;
            if (top_nb + (end - beg) > kProjTopBanksMax) break;
            top_nb += end - beg;
            top_lo = beg;
            top_lvl = l;
        }
        const int win_levels = std::min(kProjWinLevels, top_lvl - 1);
        const int top_len = top_nb * kProjBank16;
        double* scratch = m.proj_scratch.reserve((size_t)m.nb1 * (top_len > 0 ? top_len : 1));
        auto launch = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(m.nb1), dim3(512), 0, s, (const int*)c.uniq_start.p, (const int*)c.t_rows,
                               (const int*)c.t_cols, (const double*)c.t_vals, sub_offset, n, L,
                               (const int*)m.node_of.p, (const int*)vlo, (const int*)vhi, m.nbanks, m.bank_upper.p,
                               win_levels, top_lvl, top_lo, top_nb, scratch);
        };
        if (top_nb <= kProjTopBanks) launch(k_project_banked<kProjTopBanks>);
        else launch(k_project_banked<kProjTopBanksMax>);
        SGIPC_LAUNCH_CHECK();
        if (top_len > 0) {
            hipLaunchKernelGGL(k_project_top_reduce, dim3(div_up(top_len, 64)), dim3(256), 0, s,
                               (const double*)scratch, m.nb1, top_len, m.bank_upper.p + (size_t)top_lo * kProjBank16);
            SGIPC_LAUNCH_CHECK();
        }
    }
    // the FP32-with-refinement inverses serve FP32 applies only
    int inv_mode = c.bank_inverse;
    if (inv_mode == BANK_INV_MFMA32_REFINED && c.precond_kind != 3) inv_mode = BANK_INV_MFMA64;
    m.inv64_ok = inv_mode != BANK_INV_MFMA32_REFINED;
    // half storage for the fused FP32 bank solves (16-vertex banks only):
    // written by the FP64 MFMA inversion itself, else packed afterwards
    m.inv16_ok = false;
    const bool half = c.bank_store == BANK_STORE_F16 && B == 16 && m.nbanks > 0;
    if (half) {
        m.inv16.reserve((size_t)m.nbanks * (D * (D + 1) / 2) + 8);  // 2352 bytes a bank: 16-byte aligned banks
        m.inv16_d.reserve((size_t)m.nbanks * D);
    }
    const bool half_fused = half && inv_mode == BANK_INV_MFMA64;
    if (inv_mode != BANK_INV_VALU64) {
        bank_inverse_mfma(c, B, m.nbanks, m.bank_upper.p, m.inv64.p, m.inv32.p, inv_mode,
                          half_fused ? m.inv16.p : nullptr, half_fused ? m.inv16_d.p : nullptr);
    } else {
        if (B == 16)
            hipLaunchKernelGGL(k_bank_inverse_reg48, dim3(m.nbanks), dim3(64), 0, s, m.nbanks, m.bank_upper.p,
                               m.inv64.p, m.inv32.p);
        else
            hipLaunchKernelGGL(k_bank_inverse<32>, dim3(m.nbanks), dim3(128), 0, s, m.nbanks, m.bank_upper.p,
                               m.inv64.p, m.inv32.p);
        SGIPC_LAUNCH_CHECK();
    }
    if (half && !half_fused) {
        if (m.inv64_ok)
            hipLaunchKernelGGL(k_pack_inv_half<double>, dim3(m.nbanks), dim3(64), 0, s, m.nbanks,
                               (const double*)m.inv64.p, m.inv16.p, m.inv16_d.p);
        else
            hipLaunchKernelGGL(k_pack_inv_half<float>, dim3(m.nbanks), dim3(64), 0, s, m.nbanks,
                               (const float*)m.inv32.p, m.inv16.p, m.inv16_d.p);
        SGIPC_LAUNCH_CHECK();
    }
    m.inv16_ok = half;
    m.ready = true;
}

void mas_apply64(Ctx& c, const double* r, double* z) {
    if (!c.mas.ready) throw state_error("MAS apply: build first");
    if (!c.mas.inv64_ok) throw state_error("MAS apply: only FP32 inverses were built");
    mas_apply_t<double>(c, r, z, c.mas.R64.p, c.mas.Z64.p, c.mas.inv64.p);
}
void mas_apply32(Ctx& c, const double* r, double* z) {
    if (!c.mas.ready) throw state_error("MAS apply: build first");
    mas_apply_t<float>(c, r, z, c.mas.R32.p, c.mas.Z32.p, c.mas.inv32.p);
}
void mas_restrict(Ctx& c, const double* r, long long sub3, bool fp32, const int* ctrl, bool top, SceneSkip skip) {
    if (fp32) mas_restrict_t<double, float>(c, r, sub3, c.mas.R32.p, ctrl, top, skip);
    else mas_restrict_t<double, double>(c, r, sub3, c.mas.R64.p, ctrl, top, skip);
}
void mas_restrict(Ctx& c, const float* r, long long sub3, bool fp32, const int* ctrl, bool top, SceneSkip skip) {
    if (!fp32) throw state_error("MAS: FP32 residual needs the FP32 preconditioner data");
    mas_restrict_t<float, float>(c, r, sub3, c.mas.R32.p, ctrl, top, skip);
}


// workgroups of the fused update: level-1 banks (grid-stride) plus a few for
// the dofs outside the preconditioned range; one r.r partial each
void mas_update_layout(const Ctx& c, int& g1, int& gx) {
    const MasState& m = c.mas;
    long long nout = 3LL * c.nb - 3LL * m.n;
    gx = nout > 0 ? (int)std::min<long long>(64, div_up(nout, kTB)) : 0;
    g1 = std::max(1, std::min(m.nb1, kPart - gx));
}

template <typename V>
static void update_restrict_t(Ctx& c, double* x, V* r, const V* p, const V* Ap, const double* part_pap, int np_pap,
                              const double* part_rz, int np_rz, double* part_rr, int* ctrl, bool fp32, bool top) {
    MasState& m = c.mas;
    int g1, gx;
    mas_update_layout(c, g1, gx);
    const long long N = 3LL * c.nb;
    if (fp32) {
        hipLaunchKernelGGL((k_update_restrict<V, float>), dim3(g1 + gx), dim3(kTB), 0, c.stream, N, x, r, p, Ap,
                           part_pap, np_pap, part_rz, np_rz, part_rr, ctrl, c.sub_offset, m.n, m.bank, m.L,
                           (const int*)m.level_size.p, (const SlotNode*)m.slot_node.p, (const int*)m.going_next.p,
                           (const unsigned*)m.comp_mask.p, (const int*)m.l1lo.p, (const int*)m.l1hi.p, m.nb1, g1, m.R32.p);
    } else {
        if (sizeof(V) != 8) throw state_error("MAS: FP32 residual needs the FP32 preconditioner data");
        hipLaunchKernelGGL((k_update_restrict<V, double>), dim3(g1 + gx), dim3(kTB), 0, c.stream, N, x, r, p, Ap,
                           part_pap, np_pap, part_rz, np_rz, part_rr, ctrl, c.sub_offset, m.n, m.bank, m.L,
                           (const int*)m.level_size.p, (const SlotNode*)m.slot_node.p, (const int*)m.going_next.p,
                           (const unsigned*)m.comp_mask.p, (const int*)m.l1lo.p, (const int*)m.l1hi.p, m.nb1, g1, m.R64.p);
    }
    SGIPC_LAUNCH_CHECK();
    if (m.L >= 4 && top) {
        if (fp32)
            hipLaunchKernelGGL((k_restrict_top<float>), dim3(1), dim3(kTop), 0, c.stream, m.bank, m.L,
                               (const int*)m.level_size.p, (const int*)m.going_next.p, (const unsigned*)m.comp_mask.p,
                               m.R32.p, (const int*)ctrl);
        else
            hipLaunchKernelGGL((k_restrict_top<double>), dim3(1), dim3(kTop), 0, c.stream, m.bank, m.L,
                               (const int*)m.level_size.p, (const int*)m.going_next.p, (const unsigned*)m.comp_mask.p,
                               m.R64.p, (const int*)ctrl);
        SGIPC_LAUNCH_CHECK();
    }
}

void mas_update_restrict(Ctx& c, double* x, double* r, const double* p, const double* Ap, const double* part_pap,
                         int np_pap, const double* part_rz, int np_rz, double* part_rr, int* ctrl, bool fp32,
                         bool top) {
    update_restrict_t<double>(c, x, r, p, Ap, part_pap, np_pap, part_rz, np_rz, part_rr, ctrl, fp32, top);
}
void mas_update_restrict(Ctx& c, double* x, float* r, const float* p, const float* Ap, const double* part_pap,
                         int np_pap, const double* part_rz, int np_rz, double* part_rr, int* ctrl, bool fp32,
                         bool top) {
    update_restrict_t<float>(c, x, r, p, Ap, part_pap, np_pap, part_rz, np_rz, part_rr, ctrl, fp32, top);
}

template <typename T, bool H>
static void solve_top_t(Ctx& c, const void* inv, const float* dsc, T* R, T* Z, const int* ctrl, SceneSkip skip) {
    MasState& m = c.mas;
    const int top_bank0 = mas_top_bank0(m);
    prof_begin(c, PROF_MAS_SOLVE);
    auto launch = [&](auto kern, int nb) {
        hipLaunchKernelGGL(kern, dim3(1 + div_up(top_bank0, kCW * nb)), dim3(kCT), 0, c.stream, m.L,
                           (const int*)m.level_size.p, (const int*)m.going_next.p, (const unsigned*)m.comp_mask.p,
                           top_bank0, m.nbanks, inv, dsc, R, Z, ctrl, skip);
    };
    // Two banks per wavefront once one each would not be resident at once
    // (256 CUs x 32 wavefronts): 10,359 FP32 banks 10.2 -> 9.7 us.  FP64 banks
    // hold 24 more registers and gain nothing (17.2, 17.4 us); few banks lose
    // the second one's latency.
    if (sizeof(T) == 4 && top_bank0 > 8192) launch(k_mas_solve_top<T, H, sizeof(T) == 4 ? 2 : 1>, 2);
    else launch(k_mas_solve_top<T, H, 1>, 1);
    SGIPC_LAUNCH_CHECK();
    prof_end(c, PROF_MAS_SOLVE);
}

bool mas_fused(const Ctx& c) { return c.mas_fused && c.mas.bank == 16 && c.mas.ready; }

void mas_solve_with_top(Ctx& c, bool fp32, const int* ctrl, SceneSkip skip) {
    MasState& m = c.mas;
    if (fp32 && m.inv16_ok) solve_top_t<float, true>(c, m.inv16.p, m.inv16_d.p, m.R32.p, m.Z32.p, ctrl, skip);
    else if (fp32) solve_top_t<float, false>(c, m.inv32.p, nullptr, m.R32.p, m.Z32.p, ctrl, skip);
    else {
        if (!m.inv64_ok) throw state_error("MAS: only FP32 inverses were built");
        solve_top_t<double, false>(c, m.inv64.p, nullptr, m.R64.p, m.Z64.p, ctrl, skip);
    }
}

void mas_bank_solve(Ctx& c, bool fp32, const int* ctrl, SceneSkip skip) {
    if (fp32) mas_solve_t<float>(c, c.mas.inv32.p, c.mas.R32.p, c.mas.Z32.p, ctrl, skip);
    else {
        if (!c.mas.inv64_ok) throw state_error("MAS: only FP32 inverses were built");
        mas_solve_t<double>(c, c.mas.inv64.p, c.mas.R64.p, c.mas.Z64.p, ctrl, skip);
    }
}

}  // namespace sgipc
