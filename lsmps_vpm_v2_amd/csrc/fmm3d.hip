// fmm3d.hip -- the 3-D vector treecodes of the reference on gfx950, FP64:
// the default 3-D path (VELOCITY_3D_TYPE 1, src/FMM/fast3DFMM.cpp with the
// fmm3D.cpp helpers) and the second one (VELOCITY_3D_TYPE 2,
// fmm3D::calcVelocity over the 3-D TreeCell, fmm3D.cpp:585-700, 1064-1205;
// treeCell.cpp:1043-1243), which shares the walk and the moments and differs
// in the octree (root box, cell index rule, leaf rule) and in summing every
// particle of a near leaf, inactive ones included.  Type 1 below unless said.
//
// Reference semantics kept exactly:
//   * octree (FMMCell::generateTree, fast3DFMM.cpp:485-745): root box = the
//     particles' box together with the domain centre, side = the longest
//     extent times (1 + expTree / 100), centre = the box midpoint; a particle
//     goes to octant (x > xc) + 2 (y > yc) + 4 (z > zc) of its cell; a child's
//     centre is the parent's plus (size / 2) (bit - 1/2); a particle settles
//     at the first level where its cell holds fewer than critNum particles;
//     a cell is active when a particle of its subtree is active.  The keys
//     below replay these comparisons and additions per particle, so every
//     cell, centre and size is the reference's, bit for bit.
//   * moments: the 10 order-2 Cartesian moments of each vorticity component
//     about the cell centre, d = centre - particle, over active particles
//     (P2M_calc, fmm3D.cpp:84-112).  The reference forms them at the leaves
//     and shifts them upward (M2M_calc :114-145); the order-2 shift is exact,
//     so here each cell shifts its leaves' moments directly (equal up to
//     rounding, one launch instead of one per level).
//   * evaluation (evaluateFMM, fast3DFMM.cpp:318-484): every particle is a
//     target; the traversal starts at the children of the level-1 cells (a
//     level-1 leaf's sources are never summed); an inactive cell is skipped
//     with its subtree; a cell is far when |r|^2 > (2 size)^2 (the same
//     rounded comparison) and then adds its M2P term (M2P_mul_calc,
//     fmm3D.cpp:147-210); a near non-leaf cell is opened; a near leaf adds
//     the direct Biot-Savart sum over its active sources, the target itself
//     excluded.
//
// Mapping: cells are emitted in depth-first pre-order with a skip pointer
// (the next cell after the subtree); every non-leaf cell also has a row of its
// active children, so a wavefront can test many cells at once.  One wavefront
// takes kGrp consecutive sorted targets (wave-uniform coordinates) and puts
// the tree in its lanes: a lane tests one cell against every target, holds one
// far cell's coefficients or one near source, and keeps the kGrp partial
// velocities, which are summed over the lanes once at the end.
//
// This file is compiled without FMA contraction: cell centres and the
// opening test round as the reference's; the arithmetic of the sums opts
// back in (contract(fast) blocks).
#include <cmath>

#include "fmm3d.hpp"
#include "prim.hpp"

namespace vpm {
namespace {

constexpr int kHalf = kFmm3Depth / 2;  // levels per key word
constexpr unsigned kF3NonFinite = 1u, kF3Deeper = 2u, kF3Depth = 4u, kF3Degenerate = 8u,
                   kF3OddStrength = 16u;  // a strength beyond kF3MaxStrength, or not finite
// Up to here a strength times a distance is finite, whatever the target: a pair or
// term of it can be masked by a factor of zero.
constexpr double kF3MaxStrength = 1e150;
constexpr int kMomStride = 32;

struct __align__(16) Par3 {
    double x, y, z, ax, ay, az, act, pad;
};

// meta: level (bits 0-7), leaf (bit 8), active (bit 9); [begin, end): the
// cell's particles in tree order, [abegin, aend): its active ones in the
// compacted source array
struct __align__(16) Cell3 {
    double cx, cy, cz, rc2;
    uint32_t begin, end, skip, meta;
    uint32_t abegin, aend, pad0, pad1;
};

// An active source in tree order: position, tree index (for the self test),
// strength.
struct __align__(16) Src3 {
    double x, y, z, idx, ax, ay, az, pad;
};

__device__ __forceinline__ uint64_t pfx(uint64_t k, int L) { return k >> (3 * (kFmm3Depth - L)); }

// -------------------------------------------------------------------------
// bounding box and root
// -------------------------------------------------------------------------
__device__ __forceinline__ double dmin(double a, double b) { return b < a ? b : a; }
__device__ __forceinline__ double dmax(double a, double b) { return b > a ? b : a; }

__global__ void __launch_bounds__(256)
    k3_bbox(const double *__restrict__ x, const double *__restrict__ y,
            const double *__restrict__ z, int n, double *__restrict__ part) {
    __shared__ double sm[4][7];
    double mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
    double bad = 0.0;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n;
         i += (long long)gridDim.x * 256) {
        const double p[3] = {x[i], y[i], z[i]};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (!isfinite(p[d])) {
                bad = 1.0;
                continue;
            }
            mn[d] = dmin(mn[d], p[d]);
            mx[d] = dmax(mx[d], p[d]);
        }
    }
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            mn[d] = dmin(mn[d], __shfl_xor(mn[d], m, kWave));
            mx[d] = dmax(mx[d], __shfl_xor(mx[d], m, kWave));
        }
        bad = dmax(bad, __shfl_xor(bad, m, kWave));
    }
    const int w = threadIdx.x / kWave;
    if ((threadIdx.x & (kWave - 1)) == 0) {
        for (int d = 0; d < 3; ++d) {
            sm[w][d] = mn[d];
            sm[w][3 + d] = mx[d];
        }
        sm[w][6] = bad;
    }
    __syncthreads();
    if (threadIdx.x < 7) {
        double r = sm[0][threadIdx.x];
        for (int q = 1; q < 4; ++q) {
            const double o = sm[q][threadIdx.x];
            r = (threadIdx.x < 3) ? dmin(r, o) : dmax(r, o);
        }
        part[(size_t)blockIdx.x * 8 + threadIdx.x] = r;
    }
}

// The root.  Type 1, FMMCell::generateTree (fast3DFMM.cpp:507-531): the
// box starts at the domain centre, side = max extent * (1 + expTree / 100),
// centre = the box midpoint.  Type 2, TreeCell::initializeTree
// (treeCell.cpp:1066-1091): the box of the particles alone, side = the
// longest extent * (1 + expTree / 100), pivot (lower corner) = (max + min -
// side) / 2.  Also clears the header's counters.
__global__ void __launch_bounds__(256)
    k3_root(const double *__restrict__ part, int nb, double c0, double c1, double c2,
            double exp_tree, int type, Fmm3Hdr *__restrict__ h) {
    __shared__ double sm[4][7];
    const bool t2 = type == 2;
    double mn[3] = {c0, c1, c2}, mx[3] = {c0, c1, c2}, bad = 0.0;
    if (t2)
        for (int d = 0; d < 3; ++d) {
            mn[d] = INFINITY;
            mx[d] = -INFINITY;
        }
    for (int b = threadIdx.x; b < nb; b += 256) {
        for (int d = 0; d < 3; ++d) {
            mn[d] = dmin(mn[d], part[(size_t)b * 8 + d]);
            mx[d] = dmax(mx[d], part[(size_t)b * 8 + 3 + d]);
        }
        bad = dmax(bad, part[(size_t)b * 8 + 6]);
    }
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            mn[d] = dmin(mn[d], __shfl_xor(mn[d], m, kWave));
            mx[d] = dmax(mx[d], __shfl_xor(mx[d], m, kWave));
        }
        bad = dmax(bad, __shfl_xor(bad, m, kWave));
    }
    const int w = threadIdx.x / kWave;
    if ((threadIdx.x & (kWave - 1)) == 0) {
        for (int d = 0; d < 3; ++d) {
            sm[w][d] = mn[d];
            sm[w][3 + d] = mx[d];
        }
        sm[w][6] = bad;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < 4; ++q) {
            for (int d = 0; d < 3; ++d) {
                sm[0][d] = dmin(sm[0][d], sm[q][d]);
                sm[0][3 + d] = dmax(sm[0][3 + d], sm[q][3 + d]);
            }
            sm[0][6] = dmax(sm[0][6], sm[q][6]);
        }
        double root = 0.0;
        unsigned f = sm[0][6] != 0.0 ? kF3NonFinite : 0u;
        if (!t2) {
            for (int d = 0; d < 3; ++d) {
                const double len = sm[0][3 + d] - sm[0][d];
                root = (len < root) ? root : len;  // std::max(len, root)
                h->root_c[d] = 0.5 * (sm[0][3 + d] + sm[0][d]);
                h->pivot[d] = 0.0;
            }
            root *= (1 + (exp_tree / 100));
        } else {
            for (int d = 0; d < 3; ++d) {
                const double side = fabs(sm[0][3 + d] - sm[0][d]);
                if (side > root) root = side;
            }
            root *= 1.0 + (exp_tree / 100.0);
            for (int d = 0; d < 3; ++d) {
                h->pivot[d] = (sm[0][3 + d] + sm[0][d] - root) / 2.0;
                h->root_c[d] = h->pivot[d] + (0.5 * root);  // the root cell's centre
            }
            if (!(root > 0.0)) f |= kF3Degenerate;
        }
        h->root_len = root;
        h->flags = f;
        h->min_settle = 0;
        h->depth = 0;
        h->n_leaves = 0;
        h->pairs = 0;
        h->m2p = 0;
        h->wave_pairs = 0;
        h->wave_m2p = 0;
    }
}

// -------------------------------------------------------------------------
// keys, sort, gather
// -------------------------------------------------------------------------
// The particle's octant path, level by level from the root (the octant from
// the parent centre, then the child centre from the parent's).  hi holds
// levels 1..10, lo levels 11..20; sk receives the word the first sort pass
// orders (hi for a 10-level sort, lo for the first of a 20-level one).
//
// Type 2 (TreeCell): the level-L index is (int)((x - pivot) / (side / 2^L))
// (coord2index, treeCell.cpp:290-298).  side / 2^L is exact and scaling by a
// power of two commutes with rounding, so that index is the top L bits of
// t = (x - pivot) / side taken to 20 binary places: one division per axis,
// and every level's index nests in the next.
__global__ void __launch_bounds__(256)
    k3_keys(const double *__restrict__ x, const double *__restrict__ y,
            const double *__restrict__ z, int n, const Fmm3Hdr *__restrict__ h,
            uint32_t *__restrict__ khi, uint32_t *__restrict__ klo, uint32_t *__restrict__ sk,
            uint32_t *__restrict__ sv, int deep, int type) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const double px = x[i], py = y[i], pz = z[i];
    uint32_t hi = 0, lo = 0;
    if (type == 2) {
        const double R = h->root_len;
        uint32_t id[3];
        const double p[3] = {px, py, pz};
        for (int d = 0; d < 3; ++d) {
            const double t = (p[d] - h->pivot[d]) / R;
            const double sc = t * (double)(1u << kFmm3Depth);
            id[d] = sc >= 0.0 && sc < (double)(1u << kFmm3Depth) ? (uint32_t)sc : 0u;
        }
        for (int L = 1; L <= kFmm3Depth; ++L) {
            const int sh = kFmm3Depth - L;
            const uint32_t o = ((id[0] >> sh) & 1u) | (((id[1] >> sh) & 1u) << 1) |
                               (((id[2] >> sh) & 1u) << 2);
            if (L <= kHalf)
                hi = (hi << 3) | o;
            else
                lo = (lo << 3) | o;
        }
    } else {
        double cx = h->root_c[0], cy = h->root_c[1], cz = h->root_c[2], sz = h->root_len;
        for (int L = 1; L <= kFmm3Depth; ++L) {
            const uint32_t o = (px > cx ? 1u : 0u) | (py > cy ? 2u : 0u) | (pz > cz ? 4u : 0u);
            if (L <= kHalf)
                hi = (hi << 3) | o;
            else
                lo = (lo << 3) | o;
            const double cl = sz / 2.0;
            cx = cx + cl * ((double)(o & 1u) - 0.5);
            cy = cy + cl * ((double)((o >> 1) & 1u) - 0.5);
            cz = cz + cl * ((double)((o >> 2) & 1u) - 0.5);
            sz = cl;
        }
    }
    khi[i] = hi;
    klo[i] = lo;
    sk[i] = deep ? lo : hi;
    sv[i] = (uint32_t)i;
}

// Second pass of a 20-level sort: the high words in the order of the first.
__global__ void __launch_bounds__(256)
    k3_regather(const uint32_t *__restrict__ perm, const uint32_t *__restrict__ khi, int n,
                uint32_t *__restrict__ sk, uint32_t *__restrict__ sv) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= n) return;
    const uint32_t i = perm[j];
    sk[j] = khi[i];
    sv[j] = i;
}

// Sorted particle records, 60-bit keys, active flags.  The vortex strength
// is formed as velocity_fmm_3d_fast does (velocity_calc.cpp:2429-2431):
// omega * s^3 / (4 pi); without sizes (s null) (wx, wy, wz) are the
// strengths.
__global__ void __launch_bounds__(256)
    k3_gather(const uint32_t *__restrict__ perm, const uint32_t *__restrict__ khi,
              const uint32_t *__restrict__ klo, const double *__restrict__ x,
              const double *__restrict__ y, const double *__restrict__ z,
              const double *__restrict__ s, const double *__restrict__ wx,
              const double *__restrict__ wy, const double *__restrict__ wz,
              const uint8_t *__restrict__ active, int n, Par3 *__restrict__ P,
              uint64_t *__restrict__ key, uint8_t *__restrict__ act8, Fmm3Hdr *__restrict__ h) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= n) return;
    const uint32_t i = perm[j];
    key[j] = ((uint64_t)khi[i] << 30) | (uint64_t)klo[i];
    const bool a = active[i] != 0;
    Par3 r;
    r.x = x[i];
    r.y = y[i];
    r.z = z[i];
    if (s) {
        const double s3 = pow(s[i], 3.0);
        const double k4pi = 4 * M_PI;
        r.ax = wx[i] * s3 / k4pi;
        r.ay = wy[i] * s3 / k4pi;
        r.az = wz[i] * s3 / k4pi;
    } else {  // the strengths themselves (calcVelocityFast's alpha)
        r.ax = wx[i];
        r.ay = wy[i];
        r.az = wz[i];
    }
    r.act = a ? 1.0 : 0.0;
    r.pad = 0.0;
    auto tame = [](double a) { return fabs(a) <= kF3MaxStrength; };
    const uint64_t odd = __ballot(!(tame(r.ax) && tame(r.ay) && tame(r.az)));
    if (odd && (threadIdx.x & (kWave - 1)) == (uint32_t)(__ffsll((unsigned long long)odd) - 1))
        atomicOr(&h->flags, kF3OddStrength);
    P[j] = r;
    act8[j] = a ? 1 : 0;
}

// -------------------------------------------------------------------------
// leaf levels and cell emission
// -------------------------------------------------------------------------
__device__ __forceinline__ int common_levels(uint64_t a, uint64_t b, int D) {
    const uint64_t d = a ^ b;
    const int m = d ? (kFmm3Depth - 1) - (63 - __clzll((long long)d)) / 3 : D;
    return min(m, D);
}

// Per-block depth, leaf count and shallowest leaf level (k3_settle_stats
// combines them); the rare unsettled flag is the only atomic.
__device__ __forceinline__ void settle_block_stats(bool valid, int st, int mp, bool unsettled,
                                                   int D, uint4 *__restrict__ bstat,
                                                   Fmm3Hdr *__restrict__ h) {
    __shared__ uint32_t s_d[4], s_l[4], s_m[4];
    int dmax_ = st, dmin_ = valid && st > 0 ? st : 255;
    for (int m = 1; m < kWave; m <<= 1) {
        dmax_ = max(dmax_, __shfl_xor(dmax_, m, kWave));
        dmin_ = min(dmin_, __shfl_xor(dmin_, m, kWave));
    }
    const uint64_t leaves = __ballot(valid && st > mp);
    const bool any_unsettled = __ballot(unsettled) != 0;
    if ((threadIdx.x & (kWave - 1)) == 0) {
        s_d[threadIdx.x / kWave] = (uint32_t)dmax_;
        s_l[threadIdx.x / kWave] = (uint32_t)__popcll(leaves);
        s_m[threadIdx.x / kWave] = (uint32_t)dmin_;
        if (any_unsettled) atomicOr(&h->flags, D < kFmm3Depth ? kF3Deeper : kF3Depth);
    }
    __syncthreads();
    if (threadIdx.x == 0)
        bstat[blockIdx.x] = make_uint4(max(max(s_d[0], s_d[1]), max(s_d[2], s_d[3])),
                                       s_l[0] + s_l[1] + s_l[2] + s_l[3],
                                       min(min(s_m[0], s_m[1]), min(s_m[2], s_m[3])), 0u);
}

// lcpw[j] (j <= n - crit): levels shared by the ends of the window of crit
// sorted particles starting at j.  The cell of particle i at level L holds
// crit particles or more exactly when some window containing i has
// lcpw >= L (the keys are sorted, so a window's ends bound it).
__global__ void __launch_bounds__(256)
    k3_lcpw(const uint64_t *__restrict__ key, int n, int D, int crit,
            uint8_t *__restrict__ lcpw) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j > n - crit) return;
    lcpw[j] = (uint8_t)common_levels(key[j], key[j + crit - 1], D);
}

// settle[i]: the first level whose cell around particle i holds fewer than
// crit particles (1 + the largest lcpw of the windows containing i);
// mprev[i]: levels shared with particle i - 1; starts[i]: the cells particle
// i opens in pre-order (levels mprev + 1 .. settle).
__global__ void __launch_bounds__(256)
    k3_settle(const uint64_t *__restrict__ key, const uint8_t *__restrict__ lcpw, int n, int D,
              int crit, uint8_t *__restrict__ settle, uint8_t *__restrict__ mprev,
              uint32_t *__restrict__ starts, uint4 *__restrict__ bstat,
              Fmm3Hdr *__restrict__ h) {
    extern __shared__ uint8_t s_w[];
    const int i0 = blockIdx.x * 256;
    const int i = i0 + threadIdx.x;
    // windows j in [i0 - crit + 1, i0 + 255] clipped to [0, n - crit]
    const int j_lo = max(0, i0 - crit + 1), j_hi = min(i0 + 255, n - crit);
    for (int j = j_lo + (int)threadIdx.x; j <= j_hi; j += 256) s_w[j - j_lo] = lcpw[j];
    __syncthreads();
    int st = 0, mp = 0;
    bool unsettled = false;
    if (i < n) {
        int mx = 0;
        const int a = max(j_lo, i - crit + 1), b = min(i, j_hi);
        for (int j = a; j <= b; ++j) mx = max(mx, (int)s_w[j - j_lo]);
        unsettled = mx >= D;
        st = unsettled ? 0 : mx + 1;
        if (i > 0) mp = common_levels(key[i - 1], key[i], D);
        settle[i] = (uint8_t)st;
        mprev[i] = (uint8_t)mp;
        starts[i] = st > mp ? (uint32_t)(st - mp) : 0u;
    }
    settle_block_stats(i < n, st, mp, unsettled, D, bstat, h);
}

// Type 2 (TreeCell): the first level whose cell around particle i holds at
// most max_par particles and max_src active ones (the cell's range from two
// binary searches inside the parent's range; its active count from the
// active scan A).
__global__ void __launch_bounds__(256)
    k3_settle_t2(const uint64_t *__restrict__ key, const uint32_t *__restrict__ A, int n, int D,
                 int max_par, int max_src, uint8_t *__restrict__ settle,
                 uint8_t *__restrict__ mprev, uint32_t *__restrict__ starts,
                 uint4 *__restrict__ bstat, Fmm3Hdr *__restrict__ h) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    int st = 0, mp = 0;
    bool unsettled = false;
    if (i < n) {
        const uint64_t ki = key[i];
        int lo = 0, hi = n;
        for (int L = 1; L <= D; ++L) {
            const uint64_t p = pfx(ki, L);
            int a = lo, b = i;
            while (a < b) {
                const int m = (a + b) >> 1;
                if (pfx(key[m], L) < p) a = m + 1;
                else b = m;
            }
            int e0 = i + 1, e1 = hi;
            while (e0 < e1) {
                const int m = (e0 + e1) >> 1;
                if (pfx(key[m], L) > p) e1 = m;
                else e0 = m + 1;
            }
            if (e0 - a <= max_par && (int)(A[e0] - A[a]) <= max_src) {
                st = L;
                break;
            }
            lo = a;
            hi = e0;
        }
        if (i > 0) mp = common_levels(key[i - 1], ki, D);
        unsettled = st == 0;
        settle[i] = (uint8_t)st;
        mprev[i] = (uint8_t)mp;
        starts[i] = st > mp ? (uint32_t)(st - mp) : 0u;
    }
    settle_block_stats(i < n, st, mp, unsettled, D, bstat, h);
}

__global__ void __launch_bounds__(1024)
    k3_settle_stats(const uint4 *__restrict__ bstat, int nb, Fmm3Hdr *__restrict__ h) {
    __shared__ uint32_t sd[16], sl[16], sm[16];
    uint32_t d = 0, l = 0, mn = 255;
    for (int q = threadIdx.x; q < nb; q += 1024) {
        d = max(d, bstat[q].x);
        l += bstat[q].y;
        mn = min(mn, bstat[q].z);
    }
    for (int m = 1; m < kWave; m <<= 1) {
        d = max(d, (uint32_t)__shfl_xor((int)d, m, kWave));
        l += (uint32_t)__shfl_xor((int)l, m, kWave);
        mn = min(mn, (uint32_t)__shfl_xor((int)mn, m, kWave));
    }
    if ((threadIdx.x & (kWave - 1)) == 0) {
        sd[threadIdx.x / kWave] = d;
        sl[threadIdx.x / kWave] = l;
        sm[threadIdx.x / kWave] = mn;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t td = 0, tl = 0, tm = 255;
        for (int q = 0; q < 16; ++q) {
            td = max(td, sd[q]);
            tl += sl[q];
            tm = min(tm, sm[q]);
        }
        h->depth = td;
        h->n_leaves = tl;
        h->min_settle = tm;
    }
}

// Cells of particle i (levels mprev + 1 .. settle) at pre-order positions
// pos[i] ...: centre, (support size)^2, particle range, skip pointer (the
// first cell of the first particle past the range), level, leaf, active (an
// active particle in the range).  The centre is replayed from the root
// (type 1: parent + (size / 2)(bit - 1/2)) or formed from the level's index
// (type 2: pivot + (0.5 + index) size, Cell::Cell, treeCell.hpp:68).  The
// direct-sum sources of a cell are its active particles (type 1) or all of
// them (type 2, fmm3D.cpp:1172-1186 reads no active mark).
__global__ void __launch_bounds__(256)
    k3_emit(const uint64_t *__restrict__ key, const uint8_t *__restrict__ settle,
            const uint8_t *__restrict__ mprev, const uint32_t *__restrict__ pos,
            const uint32_t *__restrict__ A, int n, uint32_t ncell,
            const Fmm3Hdr *__restrict__ h, double support, int type,
            Cell3 *__restrict__ cells) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int st = settle[i], mp = mprev[i];
    if (st <= mp) return;
    const bool t2 = type == 2;
    const uint64_t ki = key[i];
    double cx = h->root_c[0], cy = h->root_c[1], cz = h->root_c[2], sz = h->root_len;
    uint32_t ix = 0, iy = 0, iz = 0;
    uint32_t p = pos[i];
    int hi = n;
    for (int L = 1; L <= st; ++L) {
        const uint32_t o = (uint32_t)(pfx(ki, L) & 7u);
        const double cl = sz / 2.0;
        if (t2) {
            ix = 2u * ix + (o & 1u);
            iy = 2u * iy + ((o >> 1) & 1u);
            iz = 2u * iz + ((o >> 2) & 1u);
            cx = h->pivot[0] + ((0.5 + (double)ix) * cl);
            cy = h->pivot[1] + ((0.5 + (double)iy) * cl);
            cz = h->pivot[2] + ((0.5 + (double)iz) * cl);
        } else {
            cx = cx + cl * ((double)(o & 1u) - 0.5);
            cy = cy + cl * ((double)((o >> 1) & 1u) - 0.5);
            cz = cz + cl * ((double)((o >> 2) & 1u) - 0.5);
        }
        sz = cl;
        if (L <= mp) continue;
        const uint64_t pf = pfx(ki, L);
        int e0 = i + 1, e1 = hi;
        while (e0 < e1) {
            const int m = (e0 + e1) >> 1;
            if (pfx(key[m], L) > pf) e1 = m;
            else e0 = m + 1;
        }
        hi = e0;
        Cell3 c;
        c.cx = cx;
        c.cy = cy;
        c.cz = cz;
        const double rck = sz * support;  // R_check (fast3DFMM.cpp:376)
        c.rc2 = rck * rck;
        c.begin = (uint32_t)i;
        c.end = (uint32_t)e0;
        c.skip = e0 < n ? pos[e0] : ncell;
        c.abegin = t2 ? (uint32_t)i : A[i];
        c.aend = t2 ? (uint32_t)e0 : A[e0];
        c.pad0 = c.pad1 = 0u;
        const bool act = A[e0] > A[i];
        c.meta = (uint32_t)L | (L == st ? 0x100u : 0u) | (act ? 0x200u : 0u);
        if (p < ncell) cells[p] = c;
        ++p;
    }
}

// The direct-sum sources in tree order: the active particles (A: exclusive
// scan of the flags) or, with all, every particle; pad holds the active
// flag (P2M reads active particles only).
__global__ void __launch_bounds__(256)
    k3_compact(const Par3 *__restrict__ P, const uint32_t *__restrict__ A, int n, int all,
               Src3 *__restrict__ S) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= n || (!all && A[j + 1] == A[j])) return;
    const Par3 q = P[j];
    Src3 r;
    r.x = q.x;
    r.y = q.y;
    r.z = q.z;
    r.idx = (double)j;
    r.ax = q.ax;
    r.ay = q.ay;
    r.az = q.az;
    r.pad = q.act;
    S[all ? (uint32_t)j : A[j]] = r;
}

// -------------------------------------------------------------------------
// moments
// -------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) v += __shfl_xor(v, m, kWave);
    return v;
}

// A far cell's term as the evaluation uses it.  With phi = 1 / r the M2P
// multipliers of M2P_mul_calc are -(derivatives of phi), and phi is harmonic:
// phi_xx + phi_yy + phi_zz = 0 and likewise for its derivatives.  So the six
// second-order multipliers of each velocity component need only the seven
// mixed third derivatives T_xxy, T_xxz, T_xyy, T_yyz, T_xzz, T_yzz, T_xyz, and
// the cross product of the 30 moments with the 30 multipliers (60 FMAs)
// becomes 42 FMAs with 27 combinations of the moments, formed once per cell.
// f[0..2] order 0, f[3..11] order 1, f[12..26] order 2, f[27..29] the centre;
// m: component-major moments (x: m[0..9], y: m[10..19], z: m[20..29]).
constexpr int kFarStride = 32;
__device__ __forceinline__ void far_row(const double *m, double cx, double cy, double cz,
                                        double *f) {
    const double *X = m, *Y = m + 10, *Z = m + 20;
    f[0] = X[0];
    f[1] = Y[0];
    f[2] = Z[0];
    f[3] = X[2];
    f[4] = X[3];
    f[5] = Y[1];
    f[6] = Y[3];
    f[7] = Z[1];
    f[8] = Z[2];
    f[9] = Y[2] - Z[3];
    f[10] = Z[3] - X[1];
    f[11] = X[1] - Y[2];
    f[12] = Y[4] - Y[6];
    f[13] = Y[5] - Y[6] - Z[8];
    f[14] = Y[7] - Z[9];
    f[15] = Y[8] - Z[6] + Z[5];
    f[16] = Y[9];
    f[17] = Z[5] - Z[4];
    f[18] = Z[7];
    f[19] = Z[6] - Z[4] - X[9];
    f[20] = Z[8] - X[7];
    f[21] = Z[9] - X[4] + X[6];
    f[22] = X[6] - X[5];
    f[23] = X[8];
    f[24] = X[4] - X[5] - Y[7];
    f[25] = X[7] + Y[4] - Y[5];
    f[26] = X[9] - Y[8];
    f[27] = cx;
    f[28] = cy;
    f[29] = cz;
}

// One thread per cell.  A leaf of level >= 2 (the level-1 cells are never
// tested): P2M of its active particles, as moments (for the shifts of its
// ancestors) and as its far row.  A non-leaf: the row of its active children
// (-1 beyond the last); thread ncell writes the root's row, the non-leaf
// level-1 cells, which the walk opens untested.
constexpr int kKids = 8;
__global__ void __launch_bounds__(256)
    k3_p2m(const Cell3 *__restrict__ cells, int ncell, const Src3 *__restrict__ S,
           double *__restrict__ mom, double *__restrict__ far, int *__restrict__ kids) {
#pragma clang fp contract(fast)
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c > ncell) return;
    const bool root = c == ncell;
    Cell3 C;
    if (!root) C = cells[c];
    if (root || !(C.meta & 0x100u)) {
        int4 *row = reinterpret_cast<int4 *>(kids + (size_t)c * kKids);
        int k[kKids], m = 0;
#pragma unroll
        for (int q = 0; q < kKids; ++q) k[q] = -1;
        int d = root ? 0 : c + 1;
        const int end = root ? ncell : (int)C.skip;
#pragma unroll
        for (int q = 0; q < kKids; ++q) {  // at most eight children
            if (d >= end) break;
            const uint32_t meta = cells[d].meta, skip = cells[d].skip;
            const bool keep = root ? !(meta & 0x100u) : (meta & 0x200u) != 0;
#pragma unroll
            for (int z = 0; z < kKids; ++z)
                if (keep && z == m) k[z] = d;
            m += keep ? 1 : 0;
            d = (int)skip;
        }
        row[0] = make_int4(k[0], k[1], k[2], k[3]);
        row[1] = make_int4(k[4], k[5], k[6], k[7]);
        return;
    }
    const int L = (int)(C.meta & 0xffu);
    if (L < 2 || (C.meta & 0x300u) != 0x300u) return;
    double m[30];
#pragma unroll
    for (int k = 0; k < 30; ++k) m[k] = 0.0;
    for (uint32_t j = C.abegin; j < C.aend; ++j) {
        const Src3 q = S[j];
        if (q.pad == 0.0) continue;
        const double dx = C.cx - q.x, dy = C.cy - q.y, dz = C.cz - q.z;
        const double t[10] = {1.0,          dx,           dy,           dz,      dx * dx * 0.5,
                              dy * dy * 0.5, dz * dz * 0.5, dx * dy,      dy * dz, dx * dz};
        const double a[3] = {q.ax, q.ay, q.az};
#pragma unroll
        for (int cc = 0; cc < 3; ++cc)
#pragma unroll
            for (int k = 0; k < 10; ++k) m[cc * 10 + k] += a[cc] * t[k];
    }
    double *o = mom + (size_t)c * kMomStride;
#pragma unroll
    for (int k = 0; k < 30; k += 2) *reinterpret_cast<double2 *>(o + k) = make_double2(m[k], m[k + 1]);
    double f[30];
    far_row(m, C.cx, C.cy, C.cz, f);
    o = far + (size_t)c * kFarStride;
#pragma unroll
    for (int k = 0; k < 30; k += 2) *reinterpret_cast<double2 *>(o + k) = make_double2(f[k], f[k + 1]);
}

// One wavefront per non-leaf cell of level >= 2: its leaves' moments shifted
// to its centre (the order-2 shift of M2M_calc, applied from each leaf).
__global__ void __launch_bounds__(256)
    k3_m2m(const Cell3 *__restrict__ cells, int ncell, const double *__restrict__ mom,
           double *__restrict__ far) {
#pragma clang fp contract(fast)
    const int lane = threadIdx.x & (kWave - 1);
    const int c = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + threadIdx.x / kWave));
    if (c >= ncell) return;
    const Cell3 C = cells[c];
    const int L = (int)(C.meta & 0xffu);
    if (L < 2 || (C.meta & 0x300u) != 0x200u) return;
    double m[30];
#pragma unroll
    for (int k = 0; k < 30; ++k) m[k] = 0.0;
    for (uint32_t d = (uint32_t)c + 1 + lane; d < C.skip; d += kWave) {
        const Cell3 D = cells[d];
        if ((D.meta & 0x300u) != 0x300u) continue;
        const double dx = C.cx - D.cx, dy = C.cy - D.cy, dz = C.cz - D.cz;
        const double *mc = mom + (size_t)d * kMomStride;
#pragma unroll
        for (int cc = 0; cc < 3; ++cc) {
            const double *q = mc + cc * 10;
            double *o = m + cc * 10;
            const double q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3];
            o[0] += q0;
            o[1] += q1 + q0 * dx;
            o[2] += q2 + q0 * dy;
            o[3] += q3 + q0 * dz;
            o[4] += q[4] + q0 * dx * dx * 0.5 + q1 * dx;
            o[5] += q[5] + q0 * dy * dy * 0.5 + q2 * dy;
            o[6] += q[6] + q0 * dz * dz * 0.5 + q3 * dz;
            o[7] += q[7] + q0 * dx * dy + q1 * dy + q2 * dx;
            o[8] += q[8] + q0 * dy * dz + q2 * dz + q3 * dy;
            o[9] += q[9] + q0 * dx * dz + q1 * dz + q3 * dx;
        }
    }
#pragma unroll
    for (int k = 0; k < 30; ++k) m[k] = wave_sum(m[k]);
    double f[30];
    far_row(m, C.cx, C.cy, C.cz, f);
    if (lane < 30) {
        double v = f[0];
#pragma unroll
        for (int k = 1; k < 30; ++k) v = lane == k ? f[k] : v;
        far[(size_t)c * kFarStride + lane] = v;
    }
}

// -------------------------------------------------------------------------
// evaluation
// -------------------------------------------------------------------------
// Lanes of one wavefront read what other lanes of it wrote to LDS.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// |r|^2 as the reference rounds it (no contraction: the opening test must
// take the same side).
__device__ __forceinline__ double r2_exact(double dx, double dy, double dz) {
    return dx * dx + dy * dy + dz * dz;
}

// 1 / sqrt(x) for finite x > 0: the hardware estimate y0 refined by the
// binomial series (1 - t)^(-1/2) = 1 + t/2 + 3 t^2/8 + ..., t = 1 - x y0^2.
__device__ __forceinline__ double rsqrt_pos(double x) {
#pragma clang fp contract(fast)
    const double y0 = __builtin_amdgcn_rsq(x);
    const double t = fma(-x * y0, y0, 1.0);
    return fma(y0 * t, fma(t, 0.375, 0.5), y0);
}

// x where bit t of m is set, else +0 (whatever x): a bit mask, not a select,
// which the compiler would turn into a branch around what forms x.
__device__ __forceinline__ double masked(double x, uint32_t m, int t) {
    const uint32_t k = (uint32_t)((int32_t)(m << (31 - t)) >> 31);
    return __hiloint2double((int)((uint32_t)__double2hiint(x) & k),
                            (int)((uint32_t)__double2loint(x) & k));
}

// The far-cell term (far_row) at a target displaced by (dx, dy, dz) from the
// centre, added to the velocity where bit t of m is set: about 90 instructions.
__device__ __forceinline__ void far_term(const double (&f)[27], double dx, double dy, double dz,
                                         uint32_t m, int t, double &vu, double &vv,
                                         double &vw) {
#pragma clang fp contract(fast)
    const double ir = masked(rsqrt_pos(dx * dx + dy * dy + dz * dz), m, t);
    const double i2 = ir * ir, i3 = i2 * ir, a = (3.0 * i2) * i3, c = 5.0 * i2;
    const double gx = dx * i3, gy = dy * i3, gz = dz * i3;
    const double ax = a * dx, ay = a * dy, az = a * dz;
    const double uxy = ax * dy, uxz = ax * dz, uyz = ay * dz;
    const double pxx = ax * dx, pyy = ay * dy, pzz = az * dz;
    const double sx = i3 - pxx, sy = i3 - pyy, sz = i3 - pzz;
    const double qx = fma(c, pxx, -a), qy = fma(c, pyy, -a), qz = fma(c, pzz, -a);
    const double txxy = qx * dy, txxz = qx * dz, txyy = qy * dx, tyyz = qy * dz, txzz = qz * dx,
                 tyzz = qz * dy, txyz = c * uxy * dz;
    vu = fma(f[1], gz, vu);
    vu = fma(-f[2], gy, vu);
    vu = fma(f[6], sz, vu);
    vu = fma(-f[8], sy, vu);
    vu = fma(-f[5], uxz, vu);
    vu = fma(-f[9], uyz, vu);
    vu = fma(f[7], uxy, vu);
    vu = fma(f[12], txxz, vu);
    vu = fma(f[13], tyyz, vu);
    vu = fma(f[14], txyz, vu);
    vu = fma(f[15], tyzz, vu);
    vu = fma(f[16], txzz, vu);
    vu = fma(f[17], txxy, vu);
    vu = fma(-f[18], txyy, vu);
    vv = fma(f[2], gx, vv);
    vv = fma(-f[0], gz, vv);
    vv = fma(f[7], sx, vv);
    vv = fma(-f[4], sz, vv);
    vv = fma(-f[10], uxz, vv);
    vv = fma(-f[8], uxy, vv);
    vv = fma(f[3], uyz, vv);
    vv = fma(f[17], txyy, vv);
    vv = fma(f[19], txzz, vv);
    vv = fma(f[18], txxy, vv);
    vv = fma(f[20], txyz, vv);
    vv = fma(f[21], txxz, vv);
    vv = fma(f[22], tyyz, vv);
    vv = fma(-f[23], tyzz, vv);
    vw = fma(f[0], gy, vw);
    vw = fma(-f[1], gx, vw);
    vw = fma(f[3], sy, vw);
    vw = fma(-f[5], sx, vw);
    vw = fma(-f[11], uxy, vw);
    vw = fma(-f[4], uyz, vw);
    vw = fma(f[6], uxz, vw);
    vw = fma(f[24], txxy, vw);
    vw = fma(f[22], tyzz, vw);
    vw = fma(f[25], txyy, vw);
    vw = fma(f[12], txzz, vw);
    vw = fma(f[23], tyyz, vw);
    vw = fma(f[26], txyz, vw);
    vw = fma(-f[16], txxz, vw);
}

// Workgroups are dispatched to the 8 XCDs in turn (workgroup b to XCD
// b mod 8); this order hands each XCD one contiguous run of the targets, so
// the cells and sources around them stay in that XCD's L2 (7.22 -> 6.82 ms
// for the 780k-particle vortex ring).  A tail of fewer than 8 per XCD keeps
// the plain order.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_block(int b, int nb) {
    const int per = nb / kXcds;
    if (b >= per * kXcds) return b;
    return (b % kXcds) * per + b / kXcds;
}

// The evaluation: one wavefront per kGrp consecutive sorted targets.
//
// The walk keeps a stack of opened cells, each with the mask of the targets
// that opened it; a step pops up to 8 of them and gives each lane one child to
// test against every target of the mask.  Far cells and near leaves go to
// queues in LDS (with their target masks); 64 queued far cells, or the sources
// of 64 queued leaves, are then evaluated with a cell or a source per lane and
// the targets in turn.  A lane's far cell or source is loaded once for kGrp
// terms (the cells' rows through LDS: coalesced 256-byte rows in, a row per
// lane out), and every wavefront step is 64 terms, of which the mask keeps
// those whose target takes this cell.
//
// The kernel is bound by vector-ALU issue in FP64 (0.83 of the cycles), so what
// counts is the share of a step's 64 lane slots that hold a wanted term.  One
// lane per target, one cell or source at a time for 64 targets, used 0.53
// (far) and 0.30 (near) of them: the far cells and near leaves of 64
// consecutive targets are 1.9 and 3.3 times those of one.  With 8 targets it
// is 0.74 and 0.58, and the far term takes 93 instructions instead of 150
// (far_row): 5.91 -> 3.6 ms on the 780k-particle vortex ring, 0.92 -> 0.22 ms
// at 60k, where 64 targets per wavefront also left most of the chip idle.
// kGrp 8 holds the 24 partial velocities, a cell's 27 coefficients and the
// term's temporaries in 168 registers (3 wavefronts per SIMD); one wavefront
// per workgroup lets LDS hold as many (2 and 4 per workgroup: 1 % and 7 %
// slower at 780k).
//
// The stack holds at most 64 cells of a level: a step pops from the deepest
// level down, so whatever stays is no deeper than what was popped, and the
// entries of a level all come from one step.
constexpr int kGrp = 8;
constexpr int kEvalWaves = 1;
constexpr int kFarRow = 18;     // LDS stride of a staged half row, in doubles (conflict-free)
constexpr int kQueue = 128;     // far cells / near leaves queued (64 evaluated at a time)
constexpr int kTakeMax = 16;    // sources a lane emits per round from its leaf
constexpr int kSrcQueue = kWave * kTakeMax + kWave;

struct EvalLds {
    union {
        double row[kWave * kFarRow];
        struct {
            uint32_t idx[kSrcQueue];
            uint8_t m[kSrcQueue];
        } s;
    };
    uint32_t fq[kQueue];
    uint32_t nb[kQueue], ne[kQueue];
    uint32_t left[kWave];  // sources carried to the next leaf batch
    uint8_t fm[kQueue], nm[kQueue], leftm[kWave];
};

typedef double v2d __attribute__((ext_vector_type(2)));

struct Acc3 {
    double u[kGrp], v[kGrp], w[kGrp];
};

// The far cells fq[base .. base + cnt) (cnt <= 64).  A masked term is multiplied by
// zero; with STRICT (near_terms) it is left out, whatever the cell's coefficients.
template <bool STRICT>
__device__ __forceinline__ void eval_far(EvalLds &l, int base, int cnt, int lane,
                                         const double *__restrict__ far, const double (&xt)[kGrp],
                                         const double (&yt)[kGrp], const double (&zt)[kGrp],
                                         Acc3 &acc) {
    const uint32_t m = lane < cnt ? (uint32_t)l.fm[base + lane] : 0u;
    // rows of 32 doubles: 8 lanes load half a row (every load in flight before
    // the first is stored), and the halves pass through LDS in turn
    v2d ta[8], tb[8], fa[8], fb[7];
#pragma unroll
    for (int it = 0; it < 8; ++it) {
        const size_t c = l.fq[base + min(it * 8 + (lane >> 3), cnt - 1)];
        const v2d *row = reinterpret_cast<const v2d *>(far + c * kFarStride) + (lane & 7);
        ta[it] = row[0];
        tb[it] = row[8];
    }
    v2d *in = reinterpret_cast<v2d *>(&l.row[(lane >> 3) * kFarRow]) + (lane & 7);
    const v2d *out = reinterpret_cast<const v2d *>(&l.row[lane * kFarRow]);
#pragma unroll
    for (int it = 0; it < 8; ++it) in[it * 4 * kFarRow] = ta[it];
    wave_sync();
#pragma unroll
    for (int k = 0; k < 8; ++k) fa[k] = out[k];
    wave_sync();
#pragma unroll
    for (int it = 0; it < 8; ++it) in[it * 4 * kFarRow] = tb[it];
    wave_sync();
#pragma unroll
    for (int k = 0; k < 7; ++k) fb[k] = out[k];
    wave_sync();
    const double fc[27] = {fa[0].x, fa[0].y, fa[1].x, fa[1].y, fa[2].x, fa[2].y, fa[3].x,
                           fa[3].y, fa[4].x, fa[4].y, fa[5].x, fa[5].y, fa[6].x, fa[6].y,
                           fa[7].x, fa[7].y, fb[0].x, fb[0].y, fb[1].x, fb[1].y, fb[2].x,
                           fb[2].y, fb[3].x, fb[3].y, fb[4].x, fb[4].y, fb[5].x};
    const double cx = fb[5].y, cy = fb[6].x, cz = fb[6].y;
#pragma unroll
    for (int t = 0; t < kGrp; ++t) {
        if (STRICT) {
            double u = 0.0, v = 0.0, w = 0.0;
            far_term(fc, xt[t] - cx, yt[t] - cy, zt[t] - cz, m, t, u, v, w);
            acc.u[t] += masked(u, m, t);
            acc.v[t] += masked(v, m, t);
            acc.w[t] += masked(w, m, t);
        } else {
            far_term(fc, xt[t] - cx, yt[t] - cy, zt[t] - cz, m, t, acc.u[t], acc.v[t], acc.w[t]);
        }
        __builtin_amdgcn_sched_barrier(0);  // one target's temporaries at a time
    }
}

// The pairs of the lane's source q with the targets of m.  A masked pair is
// multiplied by zero; with STRICT its strength is masked too (k3_eval).
template <bool STRICT>
__device__ __forceinline__ void near_terms(const Src3 &q, uint32_t m, const double (&xt)[kGrp],
                                           const double (&yt)[kGrp], const double (&zt)[kGrp],
                                           Acc3 &acc) {
#pragma clang fp contract(fast)
#pragma unroll
    for (int t = 0; t < kGrp; ++t) {
        const double ex = xt[t] - q.x, ey = yt[t] - q.y, ez = zt[t] - q.z;
        const double ir = masked(rsqrt_pos(ex * ex + ey * ey + ez * ez), m, t);
        const double i3 = ir * ir * ir;
        const double ax = STRICT ? masked(q.ax, m, t) : q.ax, ay = STRICT ? masked(q.ay, m, t) : q.ay,
                     az = STRICT ? masked(q.az, m, t) : q.az;
        acc.u[t] += (ay * ez - az * ey) * i3;
        acc.v[t] += (az * ex - ax * ez) * i3;
        acc.w[t] += (ax * ey - ay * ex) * i3;
        if (t & 1) __builtin_amdgcn_sched_barrier(0);
    }
}

// The sources s.idx[base .. base + cnt) (cnt <= 64); i0: the first target's
// tree index (a target is not its own source).
template <bool STRICT>
__device__ __forceinline__ void eval_near(EvalLds &l, int base, int cnt, int lane, int i0,
                                          const Src3 *__restrict__ S, const double (&xt)[kGrp],
                                          const double (&yt)[kGrp], const double (&zt)[kGrp],
                                          Acc3 &acc) {
#pragma clang fp contract(fast)
    uint32_t m = lane < cnt ? (uint32_t)l.s.m[base + lane] : 0u;
    const Src3 q = S[l.s.idx[base + min(lane, cnt - 1)]];
    const double self = q.idx - (double)i0;
    if (self >= 0.0 && self < (double)kGrp) m &= ~(1u << (int)self);
    near_terms<STRICT>(q, m, xt, yt, zt, acc);
}

// The sources of the leaves [nb, ne)[base .. base + cnt): each lane lists its
// leaf's sources, kTakeMax a round, at the offsets of a wave scan; whole
// batches of 64 are evaluated, the rest is carried in left / leftm (with last,
// evaluated too).
template <bool STRICT>
__device__ __forceinline__ void eval_leaves(EvalLds &l, int base, int cnt, int lane, int i0,
                                            const Src3 *__restrict__ S,
                                            const double (&xt)[kGrp], const double (&yt)[kGrp],
                                            const double (&zt)[kGrp], Acc3 &acc, bool last,
                                            int &nleft, uint32_t &wpair) {
    uint32_t b = 0, rem = 0;
    uint8_t m = 0;
    if (lane < cnt) {
        b = l.nb[base + lane];
        rem = l.ne[base + lane] - b;
        m = l.nm[base + lane];
    }
    bool more;
    do {
        const uint32_t take = min(rem, (uint32_t)kTakeMax);
        uint32_t inc = take, most = take;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const uint32_t y = __shfl_up(inc, o, kWave);
            if (lane >= o) inc += y;
            most = max(most, (uint32_t)__shfl_xor((int)most, o, kWave));
        }
        int total = __builtin_amdgcn_readlane((int)inc, kWave - 1) + nleft;
        most = (uint32_t)__builtin_amdgcn_readfirstlane((int)most);
        const uint32_t pos = (uint32_t)nleft + inc - take;
        if (lane < nleft) {
            l.s.idx[lane] = l.left[lane];
            l.s.m[lane] = l.leftm[lane];
        }
        for (uint32_t k = 0; k < most; ++k)
            if (k < take) {
                l.s.idx[pos + k] = b + k;
                l.s.m[pos + k] = m;
            }
        b += take;
        rem -= take;
        wave_sync();
        more = __ballot(rem > 0) != 0;
        while (total >= kWave || (last && !more && total > 0)) {
            const int nb = min(total, kWave);
            total -= nb;
            eval_near<STRICT>(l, total, nb, lane, i0, S, xt, yt, zt, acc);
            wpair += kGrp;
        }
        if (lane < total) {
            l.left[lane] = l.s.idx[lane];
            l.leftm[lane] = l.s.m[lane];
        }
        nleft = total;
        wave_sync();
    } while (more);
}

// STRICT for fields with a strength that is not finite, or whose product with a
// distance may not be: such a source may reach only the targets that take it
// (inactive particles of type 2 are summed by near targets alone).
template <bool STRICT>
__global__ void __launch_bounds__(kEvalWaves *kWave) __attribute__((amdgpu_waves_per_eu(3, 3)))
    k3_eval(const Cell3 *__restrict__ cells, int ncell, const int *__restrict__ kids,
            const double *__restrict__ far, const Par3 *__restrict__ P,
            const Src3 *__restrict__ S, const uint32_t *__restrict__ perm, int n, int stk_cap,
            double u_inf, double v_inf, double w_inf, double *__restrict__ u,
            double *__restrict__ v, double *__restrict__ w, int src_all,
            unsigned long long *__restrict__ wstat) {
    __shared__ EvalLds lds[kEvalWaves];
    extern __shared__ uint32_t stk_mem[];  // per wavefront: stk_cap cells, then stk_cap masks
    const int lane = threadIdx.x & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int blk = xcd_block((int)blockIdx.x, (int)gridDim.x);
    const int wave = __builtin_amdgcn_readfirstlane(blk * kEvalWaves + wv);
    const int i0 = wave * kGrp;
    if (i0 >= n) return;
    EvalLds &l = lds[wv];
    uint32_t *stk = stk_mem + (size_t)wv * (stk_cap + stk_cap / 4);
    uint8_t *stkm = reinterpret_cast<uint8_t *>(stk + stk_cap);
    const int nt = min(kGrp, n - i0);
    const uint32_t all = (1u << nt) - 1u;
    double xt[kGrp], yt[kGrp], zt[kGrp];
    uint32_t act = 0;  // targets that are sources too
#pragma unroll
    for (int t = 0; t < kGrp; ++t) {
        const Par3 &q = P[i0 + min(t, nt - 1)];
        xt[t] = q.x;
        yt[t] = q.y;
        zt[t] = q.z;
        act |= (src_all || q.act != 0.0) ? 1u << t : 0u;
    }
    Acc3 acc;
#pragma unroll
    for (int t = 0; t < kGrp; ++t) acc.u[t] = acc.v[t] = acc.w[t] = 0.0;
    uint32_t npair = 0, nfar = 0;
    uint32_t wfar = 0, wpair = 0;  // wavefront steps (uniform)
    const uint64_t below = lane ? ~0ull >> (kWave - lane) : 0ull;
    // the non-leaf level-1 cells are opened untested
    int sp, nf = 0, nn = 0, nleft = 0;
    {
        const int c = lane < kKids ? kids[(size_t)ncell * kKids + lane] : -1;
        const uint64_t b = __ballot(c >= 0);
        if (c >= 0) {
            stk[__popcll(b & below)] = (uint32_t)c;
            stkm[__popcll(b & below)] = (uint8_t)all;
        }
        sp = __popcll(b);
        wave_sync();
    }
    for (bool done = false; !done;) {
        if (sp > 0) {
            const int np = min(sp, kWave / kKids);
            sp -= np;
            int c = -1;
            uint32_t pm = 0;
            if ((lane >> 3) < np) {
                pm = stkm[sp + (lane >> 3)];
                c = kids[(size_t)stk[sp + (lane >> 3)] * kKids + (lane & 7)];
            }
            const bool live = c >= 0;
            Cell3 C{};
            if (live) C = cells[c];
            uint32_t fb = 0;
#pragma unroll
            for (int t = 0; t < kGrp; ++t)
                fb |= r2_exact(xt[t] - C.cx, yt[t] - C.cy, zt[t] - C.cz) > C.rc2 ? 1u << t : 0u;
            const uint32_t fm = live ? fb & pm : 0u, nm = live ? ~fb & pm : 0u;
            const bool leaf = (C.meta & 0x100u) != 0;
            const uint64_t bf = __ballot(fm != 0), bl = __ballot(nm != 0 && leaf),
                           bo = __ballot(nm != 0 && !leaf);
            wave_sync();  // the popped entries have been read
            if (fm) {
                const int p = nf + __popcll(bf & below);
                l.fq[p] = (uint32_t)c;
                l.fm[p] = (uint8_t)fm;
                nfar += __popc(fm);
            }
            if (nm && leaf) {
                const int p = nn + __popcll(bl & below);
                l.nb[p] = C.abegin;
                l.ne[p] = C.aend;
                l.nm[p] = (uint8_t)nm;
                // targets in this leaf that are sources: their own pair is left out
                const int lo = max((int)C.begin - i0, 0), hi = min((int)C.end - i0, kGrp);
                const uint32_t own = hi > lo ? ((1u << hi) - 1u) & ~((1u << lo) - 1u) : 0u;
                npair += (uint32_t)__popc(nm) * (C.aend - C.abegin) - (uint32_t)__popc(nm & own & act);
            }
            if (nm && !leaf) {
                const int p = sp + __popcll(bo & below);
                stk[p] = (uint32_t)c;
                stkm[p] = (uint8_t)nm;
            }
            nf += __popcll(bf);
            nn += __popcll(bl);
            sp += __popcll(bo);
            wave_sync();
        }
        done = sp == 0;
        if (nf >= kWave || (done && nf > 0)) {
            const int cnt = min(nf, kWave);
            nf -= cnt;
            eval_far<STRICT>(l, nf, cnt, lane, far, xt, yt, zt, acc);
            wfar += kGrp;
        }
        done = done && nf == 0;
        if (nn >= kWave || (done && nn + nleft > 0)) {
            const int cnt = min(nn, kWave);
            nn -= cnt;
            eval_leaves<STRICT>(l, nn, cnt, lane, i0, S, xt, yt, zt, acc, done && nn == 0, nleft,
                                wpair);
        }
        done = done && nn == 0;
    }
    // sums over the lanes: three halving exchanges leave one target per lane
    // (bit k of its index = bit 5 - k of the lane), then the remaining bits
    static_assert(kGrp == 8, "three halving exchanges");
    double r[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        double a[kGrp];
#pragma unroll
        for (int t = 0; t < kGrp; ++t) a[t] = q == 0 ? acc.u[t] : q == 1 ? acc.v[t] : acc.w[t];
#pragma unroll
        for (int h = kGrp / 2, x = kWave / 2; h >= 1; h /= 2, x /= 2) {
            const bool up = (lane & x) != 0;
#pragma unroll
            for (int t = 0; t < h; ++t) {
                const double keep = up ? a[t + h] : a[t], send = up ? a[t] : a[t + h];
                a[t] = keep + __shfl_xor(send, x, kWave);
            }
        }
        r[q] = a[0];
#pragma unroll
        for (int x = kWave / (2 * kGrp); x >= 1; x /= 2) r[q] += __shfl_xor(r[q], x, kWave);
    }
    const int t = lane / kGrp;
    if (lane % kGrp == 0 && t < nt) {
        const uint32_t o = perm[i0 + t];
        u[o] = r[0] + u_inf;
        v[o] = r[1] + v_inf;
        w[o] = r[2] + w_inf;
    }
    // work counts per wavefront (summed by k3_eval_stats; same-address
    // atomics from every wavefront would serialise)
    unsigned long long sn = npair, sf = nfar;
    for (int m = 1; m < kWave; m <<= 1) {
        sn += __shfl_xor(sn, m, kWave);
        sf += __shfl_xor(sf, m, kWave);
    }
    if (lane == 0) {
        ulonglong4 q;
        q.x = sn;
        q.y = sf;
        q.z = wpair;
        q.w = wfar;
        reinterpret_cast<ulonglong4 *>(wstat)[wave] = q;
    }
}

// Sum of the per-wavefront work counts into the header (cleared with the root):
// kStatRows3 records a workgroup, every load under way at once, then one addition
// per count.  It stands in front of the solve's last synchronisation: one workgroup
// reading all 97k records of the 780k-particle ring in turn took 37 us, this 5.
constexpr int kStatBlock3 = 256, kStatRows3 = 4 * kStatBlock3;

__global__ void __launch_bounds__(kStatBlock3)
    k3_eval_stats(const unsigned long long *__restrict__ wstat, int nw,
                  Fmm3Hdr *__restrict__ h) {
    __shared__ unsigned long long sm[kStatBlock3 / kWave][4];
    unsigned long long a[4] = {0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < kStatRows3 / kStatBlock3; ++t) {
        const int q = blockIdx.x * kStatRows3 + t * kStatBlock3 + (int)threadIdx.x;
        const ulonglong4 r = reinterpret_cast<const ulonglong4 *>(wstat)[min(q, nw - 1)];
        a[0] += q < nw ? r.x : 0;
        a[1] += q < nw ? r.y : 0;
        a[2] += q < nw ? r.z : 0;
        a[3] += q < nw ? r.w : 0;
    }
    for (int m = 1; m < kWave; m <<= 1)
        for (int k = 0; k < 4; ++k) a[k] += __shfl_xor(a[k], m, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0)
        for (int k = 0; k < 4; ++k) sm[threadIdx.x / kWave][k] = a[k];
    __syncthreads();
    if (threadIdx.x < 4) {
        unsigned long long t = 0;
        for (int q = 0; q < kStatBlock3 / kWave; ++q) t += sm[q][threadIdx.x];
        atomicAdd(&h->pairs + threadIdx.x, t);  // pairs, m2p, wave_pairs, wave_m2p
    }
}

}  // namespace

Ctx3::~Ctx3() {
    if (hdr_h) (void)hipHostFree(hdr_h);
}

void fmm3d_velocity(Ctx3 &c, hipStream_t s, int n, const double *x, const double *y,
                    const double *z, const double *sz, const double *wx, const double *wy,
                    const double *wz, const uint8_t *active, const Fmm3Params &p, double *u,
                    double *v, double *w, hipEvent_t *ev) {
    if (n < 1) throw Error(kBadArg, "n must be >= 1");
    if (!x || !y || !z || !wx || !wy || !wz || !active || !u || !v || !w)
        throw Error(kBadArg, "null pointer");
    if (p.type != 1 && p.type != 2) throw Error(kBadArg, "type must be 1 or 2");
    const bool t2 = p.type == 2;
    if (!t2 && (p.crit_num < 1 || p.crit_num > 4096))
        throw Error(kBadArg, "crit_num must be in [1, 4096]");
    if (t2 && (p.max_par < 0 || p.max_par > 4096 || p.max_src < 0 || p.max_src > 4096))
        throw Error(kBadArg, "max_par and max_src must be in [0, 4096]");
    if (p.max_depth < 1 || p.max_depth > kFmm3Depth)
        throw Error(kBadArg, "max_depth must be in [1, 20]");
    if (!(p.exp_tree >= 0.0) || !std::isfinite(p.exp_tree)) throw Error(kBadArg, "exp_tree must be >= 0");
    // with no expansion the type-2 box's upper face holds a particle whose
    // index is out of range (the reference's index2ID throws there)
    if (t2 && !(p.exp_tree > 0.0)) throw Error(kBadArg, "exp_tree must be > 0 for type 2");
    if (!(p.support > 0.0) || !std::isfinite(p.support)) throw Error(kBadArg, "support must be > 0");
    for (double q : {p.center[0], p.center[1], p.center[2], p.u_inf, p.v_inf, p.w_inf})
        if (!std::isfinite(q)) throw Error(kBadArg, "centre and free stream must be finite");
    if (!c.hdr_h) VPM_HIP(hipHostMalloc(&c.hdr_h, sizeof(Fmm3Hdr), hipHostMallocDefault));
    c.hdr_d = c.hdr_buf.as<Fmm3Hdr>(1);
    Fmm3Hdr *hd = c.hdr_d;
    c.last = p;

    const int nb = div_up(n, 256);
    const int nbb = std::min(1024, div_up(n, 256 * 8));
    double *part = c.bbox.as<double>(8 * (size_t)nbb);
    if (ev) VPM_HIP(hipEventRecord(ev[0], s));
    k3_bbox<<<nbb, 256, 0, s>>>(x, y, z, n, part);
    VPM_LAUNCH_CHECK();

    uint32_t *khi = c.khi.as<uint32_t>(n), *klo = c.klo.as<uint32_t>(n);
    uint32_t *ka = c.key_a.as<uint32_t>(n), *kb = c.key_b.as<uint32_t>(n);
    uint32_t *va = c.val_a.as<uint32_t>(n), *vb = c.val_b.as<uint32_t>(n);
    const size_t tmp_words = std::max(radix_tmp_words(n), scan_tmp_words((long long)n + 1)) + 64;
    uint32_t *tmp = c.tmp.as<uint32_t>(tmp_words);
    Par3 *P = c.par.as<Par3>(n);
    uint64_t *key = c.key64.as<uint64_t>(n);
    uint8_t *act8 = c.act8.as<uint8_t>(n);
    uint32_t *A = c.act_scan.as<uint32_t>((size_t)n + 1);
    uint8_t *settle = c.settle.as<uint8_t>(n), *mprev = c.mprev.as<uint8_t>(n);
    uint32_t *starts = c.starts.as<uint32_t>(n), *pos = c.pos.as<uint32_t>((size_t)n + 1);

    // The sort resolves 10 levels when the tree is that shallow, else 20; the
    // choice is a function of the tree alone (a build sorted the other way is
    // repeated), so the order inside a leaf, and every rounding after it,
    // depends on the input only.
    int D = c.levels_guess;
    for (int attempt = 0;; ++attempt) {
        const int deep = D > kHalf;
        // (the root kernel also clears the header's flags and counters)
        k3_root<<<1, 256, 0, s>>>(part, nbb, p.center[0], p.center[1], p.center[2], p.exp_tree,
                                  p.type, hd);
        k3_keys<<<nb, 256, 0, s>>>(x, y, z, n, hd, khi, klo, ka, va, deep, p.type);
        const bool alt = radix_sort_pairs(ka, va, kb, vb, n, 0, 3 * kHalf, tmp, s);
        uint32_t *perm = alt ? vb : va;
        if (deep) {
            uint32_t *k2 = alt ? ka : kb, *v2 = alt ? va : vb;
            uint32_t *k3 = alt ? kb : ka, *v3 = alt ? vb : va;
            k3_regather<<<nb, 256, 0, s>>>(perm, khi, n, k2, v2);
            const bool alt2 = radix_sort_pairs(k2, v2, k3, v3, n, 0, 3 * kHalf, tmp, s);
            perm = alt2 ? v3 : v2;
        }
        c.perm = perm;
        k3_gather<<<nb, 256, 0, s>>>(perm, khi, klo, x, y, z, sz, wx, wy, wz, active, n, P, key,
                                     act8, hd);
        scan_exclusive_u8(act8, A, n, &hd->n_active, true, tmp, s);
        uint4 *bstat = c.bstat.as<uint4>(nb);
        if (t2) {
            k3_settle_t2<<<nb, 256, 0, s>>>(key, A, n, D, p.max_par, p.max_src, settle, mprev,
                                            starts, bstat, hd);
        } else {
            uint8_t *lcpw = c.lcpw.as<uint8_t>(n);
            if (n >= p.crit_num)
                k3_lcpw<<<div_up(n - p.crit_num + 1, 256), 256, 0, s>>>(key, n, D, p.crit_num,
                                                                        lcpw);
            k3_settle<<<nb, 256, (size_t)(256 + p.crit_num), s>>>(
                key, lcpw, n, D, p.crit_num, settle, mprev, starts, bstat, hd);
        }
        k3_settle_stats<<<1, 1024, 0, s>>>(bstat, nb, hd);
        scan_exclusive_u32(starts, pos, n, &hd->n_cells, true, tmp, s);
        VPM_LAUNCH_CHECK();
        VPM_HIP(hipMemcpyAsync(c.hdr_h, hd, sizeof(Fmm3Hdr), hipMemcpyDeviceToHost, s));
        VPM_HIP(hipStreamSynchronize(s));
        const Fmm3Hdr &hh = *c.hdr_h;
        if (hh.flags & kF3NonFinite) throw Error(kNonFinite, "non-finite particle coordinate");
        if (hh.flags & kF3Degenerate)
            throw Error(kDegenerate, "every particle at one point (the type-2 root has no size)");
        if (hh.flags & kF3Depth)
            throw Error(kDepth, "octree deeper than 20 levels (too many coincident particles?)");
        const int want = ((hh.flags & kF3Deeper) || (int)hh.depth > kHalf) ? kFmm3Depth : kHalf;
        if (want != D && attempt == 0) {
            D = want;
            c.levels_guess = want;
            continue;
        }
        if (want != D) throw Error(kInternal, "3-D sort depth did not settle");
        break;
    }
    const Fmm3Hdr hh = *c.hdr_h;
    if ((int)hh.depth > p.max_depth) throw Error(kDepth, "octree deeper than max_depth");
    // type 2 asks every level-1 cell for its children (fmm3D.cpp:1150-1152);
    // get_childID throws for a leaf (treeCell.cpp:384-388), so a level-1 leaf
    // beside deeper cells has no result in the reference
    if (t2 && hh.depth >= 2 && hh.min_settle == 1)
        throw Error(kLevel1Leaf, "type 2: a level-1 cell is a leaf while the tree goes deeper "
                                 "(the reference's get_childID throws there)");
    const uint32_t ncell = hh.n_cells;
    Fmm3Info &fi = c.info;
    fi.n = n;
    fi.n_active = (int)hh.n_active;
    fi.n_cells = (int)ncell;
    fi.n_leaves = (int)hh.n_leaves;
    fi.depth = (int)hh.depth;
    for (int d = 0; d < 3; ++d) fi.root_c[d] = hh.root_c[d];
    fi.root_len = hh.root_len;
    fi.sorted_levels = D;

    Cell3 *cells = c.cells.as<Cell3>(ncell);
    double *mom = c.mom.as<double>((size_t)ncell * kMomStride);
    double *far = c.far.as<double>((size_t)ncell * kFarStride);
    int *kids = c.kids.as<int>(((size_t)ncell + 1) * kKids);
    Src3 *S = c.src.as<Src3>((size_t)std::max(1u, t2 ? (uint32_t)n : hh.n_active));
    k3_emit<<<nb, 256, 0, s>>>(key, settle, mprev, pos, A, n, ncell, hd, p.support, p.type,
                               cells);
    k3_compact<<<nb, 256, 0, s>>>(P, A, n, t2 ? 1 : 0, S);
    if (ev) VPM_HIP(hipEventRecord(ev[1], s));
    k3_p2m<<<div_up((long long)ncell + 1, 256), 256, 0, s>>>(cells, (int)ncell, S, mom, far, kids);
    if (ncell > 0) k3_m2m<<<div_up(ncell, 4), 256, 0, s>>>(cells, (int)ncell, mom, far);
    if (ev) VPM_HIP(hipEventRecord(ev[2], s));
    const int waves = div_up(n, kGrp);
    unsigned long long *wstat = c.wstat.as<unsigned long long>(4 * (size_t)waves);
    // the walk's stack holds at most 64 cells per non-leaf level
    const int stk_cap = kWave * std::max(1, (int)hh.depth);
    ((hh.flags & kF3OddStrength) ? k3_eval<true> : k3_eval<false>)<<<
        div_up(waves, kEvalWaves), kEvalWaves * kWave, kEvalWaves * 5 * (size_t)stk_cap, s>>>(
        cells, (int)ncell, kids, far, P, S, c.perm, n, stk_cap, p.u_inf, p.v_inf, p.w_inf, u, v, w,
        t2 ? 1 : 0, wstat);
    if (ev) VPM_HIP(hipEventRecord(ev[3], s));
    k3_eval_stats<<<div_up(waves, kStatRows3), kStatBlock3, 0, s>>>(wstat, waves, hd);
    VPM_LAUNCH_CHECK();
    VPM_HIP(hipMemcpyAsync(c.hdr_h, hd, sizeof(Fmm3Hdr), hipMemcpyDeviceToHost, s));
    VPM_HIP(hipStreamSynchronize(s));
    fi.pairs = c.hdr_h->pairs;
    fi.m2p = c.hdr_h->m2p;
    fi.wave_pairs = c.hdr_h->wave_pairs;
    fi.wave_m2p = c.hdr_h->wave_m2p;
    fi.ms_tree = fi.ms_moments = fi.ms_eval = -1.0;
    if (ev) {
        float a = 0.f, b = 0.f, e = 0.f;
        VPM_HIP(hipEventElapsedTime(&a, ev[0], ev[1]));
        VPM_HIP(hipEventElapsedTime(&b, ev[1], ev[2]));
        VPM_HIP(hipEventElapsedTime(&e, ev[2], ev[3]));
        fi.ms_tree = a;
        fi.ms_moments = b;
        fi.ms_eval = e;
    }
}

void fmm3d_cells(Ctx3 &c, hipStream_t s, int32_t *level, int64_t *key, int32_t *count,
                 uint8_t *leaf, uint8_t *active, double *centre3, double *size) {
    const int nc = c.info.n_cells, n = c.info.n;
    if (n == 0) throw Error(kBadArg, "no 3-D solve has run on this handle");
    std::vector<Cell3> cl((size_t)nc);
    std::vector<uint64_t> k((size_t)n);
    if (nc)
        VPM_HIP(hipMemcpyAsync(cl.data(), c.cells.p, sizeof(Cell3) * nc, hipMemcpyDeviceToHost, s));
    VPM_HIP(hipMemcpyAsync(k.data(), c.key64.p, sizeof(uint64_t) * n, hipMemcpyDeviceToHost, s));
    VPM_HIP(hipStreamSynchronize(s));
    for (int j = 0; j < nc; ++j) {
        const Cell3 &q = cl[(size_t)j];
        const int L = (int)(q.meta & 0xffu);
        if (level) level[j] = L;
        if (key) key[j] = (int64_t)(k[q.begin] >> (3 * (kFmm3Depth - L)));
        if (count) count[j] = (int32_t)(q.end - q.begin);
        if (leaf) leaf[j] = (q.meta >> 8) & 1u;
        if (active) active[j] = (q.meta >> 9) & 1u;
        if (centre3) {
            centre3[3 * j] = q.cx;
            centre3[3 * j + 1] = q.cy;
            centre3[3 * j + 2] = q.cz;
        }
        if (size) size[j] = std::ldexp(c.info.root_len, -L);
    }
}

void fmm3d_perm(Ctx3 &c, hipStream_t s, int32_t *perm) {
    if (c.info.n == 0 || !c.perm) throw Error(kBadArg, "no 3-D solve has run on this handle");
    VPM_HIP(hipMemcpyAsync(perm, c.perm, sizeof(uint32_t) * c.info.n, hipMemcpyDeviceToHost, s));
    VPM_HIP(hipStreamSynchronize(s));
}

}  // namespace vpm
