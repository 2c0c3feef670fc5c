// Contact-pair broad phase: a linear BVH over the surface triangles and one
// over the surface edges, queried per surface vertex (point-triangle) and
// per edge (edge-edge) for boxes within sqrt(dhat) of each other.  The
// output is the candidate quadruples that the narrow phase
// (sgipc_classify_contacts) classifies and encodes.  With a search
// direction the boxes are swept from x to x - alpha dir (the reference's
// _calcLeafBvs_ccd / _selfQuery_vf_ccd / _selfQuery_ee_ccd, mlbvh.cu
// :1172-1204, :1408-1507, :1634-1760): the candidates of the CCD step bound.
//
// Reference: S/mlbvh.cu -- leaf boxes _calcLeafBvs (:1147-1170), scene box
// _reduct_max_box (:1062-1145), Morton keys _calcMChash (:1206-1225, 10 bits
// per axis of the box centre in the scene box, original index in the low
// 32 bits), Karras internal nodes _calcInternalNodes with determine_range /
// find_split (:126-227, :1247-1267), internal boxes _calcInternalAABB
// (:1269-1296), self queries _selfQuery_vf (:1306-1406) and _selfQuery_ee
// (:1509-1632) with the reference's filters (point not in the face, edges
// sharing no vertex and obj > self, not all four vertices of btype >= 2,
// different bodies or body id -1) and box test `overlap` (:33-42).
//
// Both trees are built and queried by the same launches: their leaves are
// sorted together (one tree bit above the 30-bit codes), and every kernel's
// first workgroups take the triangles, the rest the edges.
//
// Differences: the reference appends pairs with an atomic counter while it
// traverses; here each query counts its hits (and keeps the first kHits of
// them), an exclusive scan places them, and a second launch writes them, so
// the candidate order is (query index, traversal order) -- deterministic.
// The reference climbs the tree with per-node arrival counters to merge the
// boxes; a node of a Karras tree covers a contiguous range of the sorted
// leaves, so here its box is a range query on a segment tree of leaf boxes:
// no atomics, no release / acquire between XCDs per tree level.
#include "context.hpp"
#include <rocprim/device/device_radix_sort.hpp>

namespace sgipc {
namespace {

constexpr unsigned kLeaf = 0x80000000u;   // child code: kLeaf | primitive, else internal node
constexpr int kStack = 64;
constexpr int kQT = 64;                   // queries per workgroup (one wavefront)
constexpr int kHits = 32;                 // hits per query kept by the counting pass
constexpr int kPend = 32;                 // leaves a query collects before testing them
constexpr int kPartBoxes = 256;           // partial scene boxes per tree, at most
constexpr unsigned kCodeMask = (1u << 30) - 1u;

struct Box {
    double lx, ly, lz, ux, uy, uz;
};

__device__ inline Box empty_box() { return Box{1e32, 1e32, 1e32, -1e32, -1e32, -1e32}; }
__device__ inline void grow(Box& b, const double* __restrict__ x, unsigned v) {
    double px = x[3 * (size_t)v], py = x[3 * (size_t)v + 1], pz = x[3 * (size_t)v + 2];
    b.lx = fmin(b.lx, px); b.ly = fmin(b.ly, py); b.lz = fmin(b.lz, pz);
    b.ux = fmax(b.ux, px); b.uy = fmax(b.uy, py); b.uz = fmax(b.uz, pz);
}
// the vertex at x and, when swept, at x - alpha dir
__device__ inline void grow_swept(Box& b, const double* __restrict__ x, const double* __restrict__ dir, double alpha,
                                  unsigned v) {
    grow(b, x, v);
    if (dir) {
        double px = x[3 * (size_t)v] - alpha * dir[3 * (size_t)v];
        double py = x[3 * (size_t)v + 1] - alpha * dir[3 * (size_t)v + 1];
        double pz = x[3 * (size_t)v + 2] - alpha * dir[3 * (size_t)v + 2];
        b.lx = fmin(b.lx, px); b.ly = fmin(b.ly, py); b.lz = fmin(b.lz, pz);
        b.ux = fmax(b.ux, px); b.uy = fmax(b.uy, py); b.uz = fmax(b.uz, pz);
    }
}
__device__ inline Box merge(const Box& a, const Box& b) {
    return Box{fmin(a.lx, b.lx), fmin(a.ly, b.ly), fmin(a.lz, b.lz), fmax(a.ux, b.ux), fmax(a.uy, b.uy),
               fmax(a.uz, b.uz)};
}
// boxes closer than gap on every axis (the reference's overlap with gapL)
__device__ inline bool near(const Box& a, const Box& b, double gap) {
    if (b.lx - a.ux >= gap || a.lx - b.ux >= gap) return false;
    if (b.ly - a.uy >= gap || a.ly - b.uy >= gap) return false;
    if (b.lz - a.uz >= gap || a.lz - b.uz >= gap) return false;
    return true;
}


// FP32 boxes rounded outward, for the internal nodes: a query box widened by
// the gap and rounded outward too never misses a node that the FP64 test
// would visit, and the leaves are tested in FP64, so the hits and their
// order are those of FP64 boxes throughout.  They halve a node (both
// children's boxes and codes in one 64-byte line: one load per visit).
struct FBox {
    float lx, ly, lz, ux, uy, uz;
    unsigned top;  // largest primitive id inside + 1
};
__device__ inline float round_down(double d) {
    const float f = (float)d;
    return (double)f > d ? nextafterf(f, -INFINITY) : f;
}
__device__ inline float round_up(double d) {
    const float f = (float)d;
    return (double)f < d ? nextafterf(f, INFINITY) : f;
}
__device__ inline FBox empty_fbox() {
    return FBox{INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY, 0u};
}
__device__ inline FBox outward(const Box& b, unsigned e) {
    return FBox{round_down(b.lx), round_down(b.ly), round_down(b.lz),
                round_up(b.ux),   round_up(b.uy),   round_up(b.uz),   e + 1u};
}
// the query box widened by gap, one more step outward for the rounding of the sums
__device__ inline FBox query_box(const Box& b, double gap) {
    return FBox{nextafterf(round_down(b.lx - gap), -INFINITY), nextafterf(round_down(b.ly - gap), -INFINITY),
                nextafterf(round_down(b.lz - gap), -INFINITY), nextafterf(round_up(b.ux + gap), INFINITY),
                nextafterf(round_up(b.uy + gap), INFINITY),   nextafterf(round_up(b.uz + gap), INFINITY), 0u};
}
__device__ inline FBox merge(const FBox& a, const FBox& b) {
    return FBox{fminf(a.lx, b.lx), fminf(a.ly, b.ly), fminf(a.lz, b.lz), fmaxf(a.ux, b.ux), fmaxf(a.uy, b.uy),
                fmaxf(a.uz, b.uz), max(a.top, b.top)};
}
__device__ inline bool apart(const FBox& q, float lx, float ly, float lz, float ux, float uy, float uz) {
    return lx > q.ux || ux < q.lx || ly > q.uy || uy < q.ly || lz > q.uz || uz < q.lz;
}

struct alignas(64) QNode {
    float4 a, b, c;       // left box (lx ly lz ux | uy uz), right box (lx ly | lz ux uy uz)
    unsigned left, right; // child codes
    unsigned ltop, rtop;  // largest primitive id below each child + 1
};

// one tree's part of the shared arrays: m primitives from position base
struct Tree {
    int m, base;
    const unsigned* prim;  // K vertex ids per primitive
    int K;
};
struct Trees {
    Tree t[2];   // triangles, edges
    int nb0;     // workgroups of tree 0 in this launch
    __device__ const Tree& mine(int& block) const {
        block = (int)blockIdx.x;
        if (block < nb0) return t[0];
        block -= nb0;
        return t[1];
    }
};

template <int NW>
__device__ inline Box block_box(Box b, Box* sh) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        b.lx = fmin(b.lx, __shfl_xor(b.lx, off)); b.ly = fmin(b.ly, __shfl_xor(b.ly, off));
        b.lz = fmin(b.lz, __shfl_xor(b.lz, off)); b.ux = fmax(b.ux, __shfl_xor(b.ux, off));
        b.uy = fmax(b.uy, __shfl_xor(b.uy, off)); b.uz = fmax(b.uz, __shfl_xor(b.uz, off));
    }
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = b;
    __syncthreads();
    b = sh[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) b = merge(b, sh[w]);
    return b;
}

// leaf boxes (FP64, in primitive order) and one partial scene box per workgroup
__global__ void __launch_bounds__(256) k_leaf_boxes(Trees T, int stride0, int stride1, const double* __restrict__ x,
                                                    const double* __restrict__ dir, double alpha,
                                                    Box* __restrict__ leaf, Box* __restrict__ part) {
    __shared__ Box sh[4];
    int blk;
    const Tree& t = T.mine(blk);
    const bool tri = &t == &T.t[0];
    const int stride = 256 * (tri ? stride0 : stride1);
    Box all = empty_box();
    for (int i = blk * 256 + (int)threadIdx.x; i < t.m; i += stride) {
        Box b = empty_box();
        for (int k = 0; k < t.K; ++k) grow_swept(b, x, dir, alpha, t.prim[t.K * (size_t)i + k]);
        leaf[t.base + (size_t)i] = b;
        all = merge(all, b);
    }
    all = block_box<4>(all, sh);
    if (threadIdx.x == 0) part[(tri ? 0 : kPartBoxes) + blk] = all;
}

__device__ inline unsigned spread10(unsigned v) {
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}
__device__ inline unsigned cell10(double t) {
    t = fmin(fmax(t * 1024.0, 0.0), 1023.0);
    return (unsigned)t;
}

// 30-bit Morton code of every leaf box's centre in its tree's scene box
// (merged here from the partials), the tree bit above it
__global__ void __launch_bounds__(256) k_morton(Trees T, int np0, int np1, const Box* __restrict__ leaf,
                                                const Box* __restrict__ part, unsigned* __restrict__ code,
                                                unsigned* __restrict__ idx) {
    __shared__ Box sh[4];
    int blk;
    const Tree& t = T.mine(blk);
    const bool tri = &t == &T.t[0];
    const int np = tri ? np0 : np1;
    const Box S = block_box<4>((int)threadIdx.x < np ? part[(tri ? 0 : kPartBoxes) + threadIdx.x] : empty_box(), sh);
    const int i = blk * 256 + (int)threadIdx.x;
    if (i >= t.m) return;
    const Box b = leaf[t.base + (size_t)i];
    // a flat scene axis maps every centre to cell 0 on it
    double sx = S.ux - S.lx, sy = S.uy - S.ly, sz = S.uz - S.lz;
    double cx = 0.5 * (b.lx + b.ux) - S.lx, cy = 0.5 * (b.ly + b.uy) - S.ly, cz = 0.5 * (b.lz + b.uz) - S.lz;
    unsigned xx = spread10(sx > 0.0 ? cell10(cx / sx) : 0u);
    unsigned yy = spread10(sy > 0.0 ? cell10(cy / sy) : 0u);
    unsigned zz = spread10(sz > 0.0 ? cell10(cz / sz) : 0u);
    code[t.base + (size_t)i] = ((xx << 2) + (yy << 1) + zz) | (tri ? 0u : kCodeMask + 1u);
    idx[t.base + (size_t)i] = (unsigned)i;
}

// Segment tree over a tree's sorted leaf boxes: level k holds the merged
// boxes of aligned runs of 2^k leaves, ceil(m / 2^k) of them; a tree's
// levels lie one after the other from 2 * base + 64 * tree.
__device__ inline size_t seg_base(const Tree& t, bool tri) { return 2 * (size_t)t.base + (tri ? 0 : 64); }
__device__ inline int seg_count(int m, int k) { return (int)(((long long)m + (1ll << k) - 1) >> k); }

// sorted leaves: keys, level 0 of the segment tree, and its levels 1 to 8 (a
// workgroup's 256 leaves are one run of level 8)
__global__ void __launch_bounds__(256) k_leaves(Trees T, const unsigned* __restrict__ sidx,
                                                const unsigned* __restrict__ scode, const Box* __restrict__ leaf,
                                                FBox* __restrict__ seg, unsigned long long* __restrict__ key) {
    __shared__ FBox sh[256];
    int blk;
    const Tree& t = T.mine(blk);
    const bool tri = &t == &T.t[0];
    const int tid = (int)threadIdx.x, i = blk * 256 + tid;
    FBox b = empty_fbox();
    FBox* lv = seg + seg_base(t, tri);
    if (i < t.m) {
        const unsigned e = sidx[t.base + (size_t)i];
        key[t.base + (size_t)i] = ((unsigned long long)(scode[t.base + (size_t)i] & kCodeMask) << 32) | e;
        b = outward(leaf[t.base + (size_t)e], e);
        lv[i] = b;
    }
    sh[tid] = b;
#pragma unroll
    for (int k = 1; k <= 8; ++k) {
        lv += seg_count(t.m, k - 1);
        __syncthreads();
        if (tid < (256 >> k)) b = merge(sh[2 * tid], sh[2 * tid + 1]);
        __syncthreads();
        if (tid < (256 >> k)) {
            sh[tid] = b;
            const int q = blk * (256 >> k) + tid;
            if (q < seg_count(t.m, k)) lv[q] = b;
        }
    }
}

// levels 9 and up, one workgroup per tree
__global__ void __launch_bounds__(1024) k_seg_top(Trees T, FBox* __restrict__ seg) {
    int blk;
    const Tree& t = T.mine(blk);
    const FBox* lo = seg + seg_base(t, &t == &T.t[0]);
    for (int k = 0; k < 8; ++k) lo += seg_count(t.m, k);
    for (int k = 9; seg_count(t.m, k - 1) > 1; ++k) {
        const int below = seg_count(t.m, k - 1), n = seg_count(t.m, k);
        FBox* hi = const_cast<FBox*>(lo) + below;
        for (int q = (int)threadIdx.x; q < n; q += 1024)
            hi[q] = 2 * q + 1 < below ? merge(lo[2 * q], lo[2 * q + 1]) : lo[2 * q];
        __syncthreads();  // this workgroup's stores are read by its next level
        lo = hi;
    }
}

// merged boxes of the sorted leaves lo .. mid and mid + 1 .. hi (a node's two
// children), their loads of one level in flight together
__device__ inline void child_boxes(const FBox* __restrict__ lv, int m, int lo, int mid, int hi, FBox& L, FBox& R) {
    L = R = empty_fbox();
    int l0 = lo, r0 = mid + 1, l1 = mid + 1, r1 = hi + 1;
    for (int k = 0; l0 < r0 || l1 < r1; ++k) {
        FBox a = empty_fbox(), b = a, c = a, d = a;
        if (l0 < r0) {
            if (l0 & 1) a = lv[l0++];
            if (r0 & 1) b = lv[--r0];
        }
        if (l1 < r1) {
            if (l1 & 1) c = lv[l1++];
            if (r1 & 1) d = lv[--r1];
        }
        lv += seg_count(m, k);
        L = merge(L, merge(a, b));
        R = merge(R, merge(c, d));
        l0 >>= 1;
        r0 >>= 1;
        l1 >>= 1;
        r1 >>= 1;
    }
}

__device__ inline int prefix(const unsigned long long* __restrict__ key, int m, int i, int j) {
    if (j < 0 || j >= m) return -1;
    return __clzll(key[i] ^ key[j]);
}

// Karras (2012) radix-tree construction over the unique sorted keys: internal
// node i covers the leaves lo .. hi split after gamma; its two children's
// boxes come from the segment tree
__global__ void __launch_bounds__(256) k_internal(Trees T, const unsigned long long* __restrict__ keys,
                                                  const unsigned* __restrict__ sidx, const FBox* __restrict__ seg,
                                                  QNode* __restrict__ nodes) {
    int blk;
    const Tree& tr = T.mine(blk);
    const int m = tr.m, i = blk * 256 + (int)threadIdx.x;
    if (i >= m - 1) return;
    const unsigned long long* key = keys + tr.base;
    const int d = (prefix(key, m, i, i + 1) - prefix(key, m, i, i - 1)) > 0 ? 1 : -1;
    const int dmin = prefix(key, m, i, i - d);
    int lmax = 2;
    while (prefix(key, m, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t > 0; t >>= 1)
        if (prefix(key, m, i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = prefix(key, m, i, j);
    int s = 0, t = l;
    do {
        t = (t + 1) >> 1;
        if (prefix(key, m, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    const int gamma = i + s * d + min(d, 0);
    const int lo = min(i, j), hi = max(i, j);
    const FBox* lv = seg + seg_base(tr, &tr == &T.t[0]);
    FBox L, R;
    child_boxes(lv, m, lo, gamma, hi, L, R);
    QNode n;
    n.a = make_float4(L.lx, L.ly, L.lz, L.ux);
    n.b = make_float4(L.uy, L.uz, R.lx, R.ly);
    n.c = make_float4(R.lz, R.ux, R.uy, R.uz);
    n.left = lo == gamma ? (kLeaf | sidx[tr.base + (size_t)gamma]) : (unsigned)gamma;
    n.right = hi == gamma + 1 ? (kLeaf | sidx[tr.base + (size_t)gamma + 1]) : (unsigned)(gamma + 1);
    n.ltop = L.top;
    n.rtop = R.top;
    nodes[tr.base + (size_t)i] = n;
}

// visit every leaf whose FP32 box is near the query and whose primitive id is
// at least q.top, depth first: a leaf child at once, of two internal children
// the right one first.  stk: this lane's column of the wavefront's LDS stack.
template <typename F>
__device__ inline bool traverse(const QNode* __restrict__ nodes, int m, unsigned only, const FBox& q, unsigned* stk,
                                F&& on_leaf) {
    if (m == 1) {
        on_leaf(only);
        return true;
    }
    int sp = 0;
    unsigned cur = 0;
    for (;;) {
        const QNode n = nodes[cur];
        const bool hl = n.ltop > q.top && !apart(q, n.a.x, n.a.y, n.a.z, n.a.w, n.b.x, n.b.y);
        const bool hr = n.rtop > q.top && !apart(q, n.b.z, n.b.w, n.c.x, n.c.y, n.c.z, n.c.w);
        unsigned next = kLeaf;  // none
        if (hl) {
            if (n.left & kLeaf) on_leaf(n.left & ~kLeaf);
            else next = n.left;
        }
        if (hr) {
            if (n.right & kLeaf) {
                on_leaf(n.right & ~kLeaf);
            } else {
                if (next != kLeaf) {
                    if (sp >= kStack) return false;
                    stk[kQT * sp++] = next;
                }
                next = n.right;
            }
        }
        if (next == kLeaf) {
            if (sp == 0) return true;
            next = stk[kQT * --sp];
        }
        cur = next;
    }
}

__device__ inline bool all_static(const int* __restrict__ bt, unsigned a, unsigned b, unsigned c, unsigned d) {
    return bt && bt[a] >= 2 && bt[b] >= 2 && bt[c] >= 2 && bt[d] >= 2;
}
__device__ inline bool other_body(const int* __restrict__ body, unsigned a, unsigned b) {
    return !body || body[a] == -1 || body[a] != body[b];
}

struct Query {
    int nsv, nbv;                // point queries and their workgroups (before the edges' ones)
    const unsigned* sv;
    const double *x, *dir;
    double alpha, gap;
    const Box* leaf;
    const QNode* nodes;
    const unsigned* sidx;        // sorted primitive ids
    const int *bt, *body;
    int* cnt;                    // hits per query: points, then edges
    const int* off;              // their exclusive scan (pass 1)
    unsigned* hits;              // kHits per query slot, slot fastest
    int4 *pt_out, *ee_out;       // pass 1: null when the list does not fit
    int pt_cap, ee_cap;
    int* err;
};

// Workgroups are dispatched round-robin over the 8 XCDs: the place of the
// q-th of n in an order that gives every XCD a contiguous range.
__device__ inline int xcd_order(int q, int n) {
    const int x = q & 7, per = n >> 3, rem = n & 7;
    return x * per + min(x, rem) + (q >> 3);
}

// Pass 0 counts the hits of every query and keeps the first kHits; pass 1
// writes them at the scanned offsets and traverses again only for a query
// with more.  The edge queries run in sorted (Morton) order, so the lanes of
// a wavefront walk nearby parts of the tree; counts and output are by edge.
// The walk is a chain of dependent loads with few wavefronts per SIMD to hide
// it, so it does nothing but walk: leaves are collected (kPend per lane) and
// their exact tests, whose loads are independent, run together (16 per lane:
// slower than testing at once, as lanes flush apart; 32: most flush once).
// An edge query skips subtrees without an id above its own, and every XCD
// takes a contiguous range of the queries, so that a node is read into its L2
// once and not once per XCD.  76,804 queries of two 40^3 boxes: 216 us with
// the tests in the walk and workgroups in launch order, 150 us so (1201
// wavefronts, 1.8 per CU on average over the launch; 79 % of the L2 requests
// hit).
template <int PASS>
__global__ void __launch_bounds__(kQT) k_query(Trees T, Query Q) {
    __shared__ unsigned stack[kStack * kQT];
    __shared__ unsigned pend[kPend * kQT];
    unsigned *stk = stack + threadIdx.x, *pnd = pend + threadIdx.x;
    const bool vf = (int)blockIdx.x < Q.nbv;
    const Tree& t = vf ? T.t[0] : T.t[1];
    const unsigned* prim = t.prim;
    const int blk = vf ? xcd_order((int)blockIdx.x, Q.nbv) : Q.nbv + xcd_order((int)blockIdx.x - Q.nbv, (int)gridDim.x - Q.nbv);
    const size_t slot = (size_t)blk * kQT + threadIdx.x, nslots = (size_t)gridDim.x * kQT;
    int i = (int)slot - (vf ? 0 : Q.nbv * kQT);
    if (i >= (vf ? Q.nsv : t.m)) return;
    if (!vf) i = (int)Q.sidx[t.base + (size_t)i];
    int4* out = vf ? Q.pt_out : Q.ee_out;
    if (PASS && !out) return;
    const int cap = vf ? Q.pt_cap : Q.ee_cap, qi = vf ? i : Q.nsv + i;
    // the query's vertices: the point, or the edge's ends
    const unsigned a0 = vf ? Q.sv[i] : prim[2 * (size_t)i], a1 = vf ? a0 : prim[2 * (size_t)i + 1];
    auto emit = [&](int pos, unsigned e) {
        if (pos >= cap) return;
        if (vf) out[pos] = make_int4((int)a0, (int)prim[3 * (size_t)e], (int)prim[3 * (size_t)e + 1], (int)prim[3 * (size_t)e + 2]);
        else out[pos] = make_int4((int)a0, (int)a1, (int)prim[2 * (size_t)e], (int)prim[2 * (size_t)e + 1]);
    };
    int base = 0, total = 0;
    if (PASS) {
        base = Q.off[qi] - (vf ? 0 : Q.off[Q.nsv]);
        total = Q.cnt[qi];
        for (int k = 0; k < min(total, kHits); ++k) emit(base + k, Q.hits[(size_t)k * nslots + slot]);
        if (total <= kHits) return;
    }
    Box q = empty_box();
    if (vf) grow_swept(q, Q.x, Q.dir, Q.alpha, a0);
    else q = Q.leaf[t.base + (size_t)i];  // edge i's own box (leaf boxes are kept in edge order)
    FBox fq = query_box(q, Q.gap);
    fq.top = vf ? 0u : (unsigned)i + 1u;
    int k = 0, np = 0;
    // exact tests of the collected leaves, in order, four at a time
    auto flush = [&]() {
        for (int p0 = 0; p0 < np; p0 += 4) {
            unsigned e[4], b[4][3];
            Box eb[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                e[j] = pnd[kQT * min(p0 + j, np - 1)];
                eb[j] = Q.leaf[t.base + (size_t)e[j]];
                const unsigned* pr = prim + t.K * (size_t)e[j];
                b[j][0] = pr[0];
                b[j][1] = pr[1];
                b[j][2] = vf ? pr[2] : pr[1];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (p0 + j >= np || !near(q, eb[j], Q.gap)) continue;
                const unsigned u = b[j][0], v = b[j][1], w = b[j][2];
                if (a0 == u || a0 == v || a0 == w || a1 == u || a1 == v) continue;
                if (!other_body(Q.body, a0, u) || all_static(Q.bt, a0, vf ? u : a1, vf ? v : u, vf ? w : v)) continue;
                if (!PASS) {
                    if (k < kHits) Q.hits[(size_t)k * nslots + slot] = e[j];
                } else if (k >= kHits) {
                    emit(base + k, e[j]);
                }
                ++k;
            }
        }
        np = 0;
    };
    const bool ok = traverse(Q.nodes + t.base, t.m, t.m == 1 ? Q.sidx[t.base] : 0u, fq, stk, [&](unsigned e) {
        pnd[kQT * np++] = e;
        if (np == kPend) flush();
    });
    flush();
    if (!ok) atomicOr(Q.err, 1);
    if (!PASS) Q.cnt[qi] = k;
}

}  // namespace

void broad_phase(Ctx& c, int nsv, const unsigned* sv, int nf, const unsigned* faces, int ne, const unsigned* edges,
                 const double* x, const int* btype, const int* body, double dhat, int* pt_out, int pt_cap, int& n_pt,
                 int* ee_out, int ee_cap, int& n_ee, const double* dir, double alpha) {
    if (!(dhat > 0.0)) throw arg_error("broad_phase: dhat must be positive");
    hipStream_t s = c.stream;
    Lbvh& B = c.lbvh;
    n_pt = n_ee = 0;
    const bool pt = nsv > 0 && nf > 0, ee = ne > 1;
    if (!pt) nsv = 0;
    const int mt = pt ? nf : 0, me = ee ? ne : 0, M = mt + me;
    if (M == 0) return;
    Trees T{{Tree{mt, 0, faces, 3}, Tree{me, mt, edges, 2}}, 0};
    auto blocks = [&](int per) {  // workgroups of `per` leaves, triangles first
        T.nb0 = (int)div_up(mt, per);
        return dim3((unsigned)(T.nb0 + (int)div_up(me, per)));
    };
    int* err = B.err.reserve(1);
    fill<int>(err, 0, 1, s);
    Box* leaf = (Box*)B.leaf.reserve((size_t)M * sizeof(Box));
    Box* part = (Box*)B.part.reserve(2 * kPartBoxes * sizeof(Box));
    unsigned* code = B.code.reserve(2 * (size_t)M);
    unsigned* idx = B.idx.reserve(2 * (size_t)M);
    unsigned long long* key = B.key.reserve((size_t)M);
    FBox* seg = (FBox*)B.seg.reserve((2 * (size_t)M + 128) * sizeof(FBox));
    QNode* nodes = (QNode*)B.nodes.reserve((size_t)M * sizeof(QNode));
    const int np0 = std::min(kPartBoxes, (int)div_up(mt, 256)), np1 = std::min(kPartBoxes, (int)div_up(me, 256));
    T.nb0 = np0;
    hipLaunchKernelGGL(k_leaf_boxes, dim3(np0 + np1), dim3(256), 0, s, T, np0, np1, x, dir, alpha, leaf, part);
    SGIPC_LAUNCH_CHECK();
    const dim3 g256 = blocks(256);
    hipLaunchKernelGGL(k_morton, g256, dim3(256), 0, s, T, np0, np1, (const Box*)leaf, (const Box*)part, code, idx);
    SGIPC_LAUNCH_CHECK();
    if (c.sort_impl == SORT_OWN) {
        radix_sort_pairs(c, code, code + M, (const int*)idx, 0, (int*)(idx + M), M, 31, s);
    } else {  // rocPRIM as the cross-check
        size_t bytes = 0;
        SGIPC_HIP(rocprim::radix_sort_pairs(nullptr, bytes, code, code + M, idx, idx + M, (unsigned)M, 0, 31, s));
        void* tmp = B.sort_tmp.reserve(bytes + 1);
        SGIPC_HIP(rocprim::radix_sort_pairs(tmp, bytes, code, code + M, idx, idx + M, (unsigned)M, 0, 31, s));
    }
    const unsigned* sidx = idx + M;
    hipLaunchKernelGGL(k_leaves, g256, dim3(256), 0, s, T, sidx, (const unsigned*)(code + M), (const Box*)leaf, seg,
                       key);
    SGIPC_LAUNCH_CHECK();
    if (std::max(mt, me) > 256) {
        T.nb0 = mt > 0 ? 1 : 0;
        hipLaunchKernelGGL(k_seg_top, dim3(T.nb0 + (me > 0 ? 1 : 0)), dim3(1024), 0, s, T, seg);
        SGIPC_LAUNCH_CHECK();
    }
    (void)blocks(256);
    hipLaunchKernelGGL(k_internal, g256, dim3(256), 0, s, T, (const unsigned long long*)key, sidx, (const FBox*)seg,
                       nodes);
    SGIPC_LAUNCH_CHECK();
    const int nq = nsv + me, nbv = (int)div_up(nsv, kQT), nbq = nbv + (int)div_up(me, kQT);
    int* cnt = B.cnt.reserve((size_t)nq + 1);
    int* off = B.off.reserve((size_t)nq + 1);
    Query Q{nsv, nbv, sv, x, dir, alpha, sqrt(dhat), leaf, nodes, sidx, btype, body, cnt, off,
            B.hits.reserve((size_t)kHits * nbq * kQT), nullptr, nullptr, pt_cap, ee_cap, err};
    hipLaunchKernelGGL(k_query<0>, dim3(nbq), dim3(kQT), 0, s, T, Q);
    SGIPC_LAUNCH_CHECK();
    exclusive_scan(c, cnt, off, nq, nullptr, s);
    int h[3] = {0, 0, 0};  // point-triangle hits, all hits, traversal error
    SGIPC_HIP(hipMemcpyAsync(&h[0], off + nsv, sizeof(int), hipMemcpyDeviceToHost, s));
    SGIPC_HIP(hipMemcpyAsync(&h[1], off + nq, sizeof(int), hipMemcpyDeviceToHost, s));
    SGIPC_HIP(hipMemcpyAsync(&h[2], err, sizeof(int), hipMemcpyDeviceToHost, s));
    SGIPC_HIP(hipStreamSynchronize(s));
    if (h[2]) throw state_error("broad_phase: BVH traversal stack exceeded");
    n_pt = h[0];
    n_ee = h[1] - h[0];
    Q.pt_out = n_pt > 0 && n_pt <= pt_cap ? (int4*)pt_out : nullptr;
    Q.ee_out = n_ee > 0 && n_ee <= ee_cap ? (int4*)ee_out : nullptr;
    if (Q.pt_out || Q.ee_out) {
        hipLaunchKernelGGL(k_query<1>, dim3(nbq), dim3(kQT), 0, s, T, Q);
        SGIPC_LAUNCH_CHECK();
        SGIPC_HIP(hipStreamSynchronize(s));
    }
}

}  // namespace sgipc
