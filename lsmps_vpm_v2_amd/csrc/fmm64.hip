// fmm64.hip -- plain FP64 FMM stages on gfx950.
//
// Expansion conventions follow fmm2D (reference src/FMM/fmm2D.cpp):
//   multipole a_p = sum q (z - zc)^p                 (P2M, :237-284)
//   M2M  a_p += a'_0 d^p + sum_k C(p-1,k-1)(p/k) a'_k d^(p-k),  d = zc' - zc   (:361-376)
//   M2L  b_p -= a_0/p d^-p + sum_k C(p+k-1,k-1)(-1)^k/k a_k d^-(p+k), d = zs - zt (:465-481)
//   L2L  b'_p += sum_{k>=p} C(k,p) b_k d^(k-p),  d = zc' - zc      (:637-643)
//   M2P  F = sum a_p (z - zc)^-(p+1)                  (list 3, :1052-1062)
//   L2P  F = sum_{p>=1} p b_p (z - zc)^(p-1)          (:1083-1093)
//   Ex += Re F, Ey -= Im F; P2P Ex += q dx/r^2, Ey += q dy/r^2 (:164-173).
// b_0 is never formed: L2L feeds b_p only from b_k with k >= p and L2P starts
// at p = 1, so b_0 cannot reach the field.
//
// The per-order coefficient tables (M2L including the reference's int32
// binomials in parity mode) are built on the host (api.cpp) and read from
// global memory.  Thread mappings, orders up to 16: 16 lanes per leaf (P2M), a
// workgroup per subtree of three levels (M2M, L2L), the matrix cores (list-2 M2L;
// the potential and list 4 a wavefront per cell), one or four wavefronts per leaf
// (evaluation, any order).  Above order 16 the translations take one thread per
// (cell, order): Horner in the translation distance, no per-thread arrays.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <vector>

#include "ctx.hpp"

namespace vpm {
namespace {

constexpr unsigned kLeaf = 1u, kActive = 2u;

struct cd {
    double x, y;
};
__device__ __forceinline__ cd cmul(cd a, cd b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
__device__ __forceinline__ cd cadd(cd a, cd b) { return {a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ cd csub(cd a, cd b) { return {a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ cd cscale(cd a, double s) { return {a.x * s, a.y * s}; }
__device__ __forceinline__ cd cinv(cd a) {
    const double r = 1.0 / (a.x * a.x + a.y * a.y);
    return {a.x * r, -a.y * r};
}
__device__ __forceinline__ cd cpowi(cd z, int p) {
    cd r = {1.0, 0.0};
    while (p > 0) {
        if (p & 1) r = cmul(r, z);
        z = cmul(z, z);
        p >>= 1;
    }
    return r;
}
__device__ __forceinline__ cd ld(const double2 *a, size_t i) {
    double2 v = a[i];
    return {v.x, v.y};
}
__device__ __forceinline__ void st(double2 *a, size_t i, cd v) { a[i] = make_double2(v.x, v.y); }

__device__ __forceinline__ double shfl_xor_d(double v, int m) {
    return __shfl_xor(v, m, kWave);
}

// Lanes of one wavefront read what other lanes of it wrote to LDS.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// P2M (fmm2D.cpp:237-284, with the sign and 1/p folded into the translation
// tables): four leaves per wavefront, 16 lanes each.  A leaf's lanes take 16
// of its particles at a time, and lane i stages q z^b (b = 0..3) and z^(4a)
// (a = 0..3) of its particle, z from the leaf's centre (zero for a particle without
// strength or inactive, whatever its powers would be); lane r then adds its own order p = 4a + b as
// one complex product per particle, four FMAs from two LDS reads, with no
// cross-lane reduction.  Orders beyond 15 take further chunks of 16.  (Forming
// z^p afresh per particle and order took about 40 operations: 37 -> 13 us at
// 780k particles, order 10; 21 -> 5 us at 2,000.)
// Block 0 also clears the rows no later stage writes: the root's multipole,
// and the local expansions of levels 0 and 1 (nz rows of bk, stride bs).
constexpr int kP2m64Waves = 4;
constexpr int kP2mLanes = 16;                    // lanes per leaf
constexpr int kP2mLeaves = kWave / kP2mLanes;    // leaves per wavefront

__global__ void __launch_bounds__(kWave *kP2m64Waves)
    k_p2m64(const uint32_t *leaf_idx, int nl, int P, const uint8_t *c_flags,
            const uint32_t *c_begin, const uint32_t *c_end, const double *c_cx,
            const double *c_cy, const double *xs, const double *ys, const double *qs,
            const uint8_t *as, double2 *ak, double2 *bk, int nz, int bs) {
    // row b of leaf g from b 68 + g 17: the 16 rows a wavefront reads at a time
    // lie on different banks
    constexpr int kB = 68, kG = kP2mLanes + 1;
    __shared__ double2 lo[kP2m64Waves][4 * kB], hi[kP2m64Waves][4 * kB];
    const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    const int g = lane / kP2mLanes, r = lane % kP2mLanes;
    const long long t = ((long long)blockIdx.x * kP2m64Waves + w) * kP2mLeaves + g;
    const int P1 = P + 1;
    if (blockIdx.x == 0) {
        for (int k = threadIdx.x; k < P1; k += blockDim.x) ak[k] = make_double2(0.0, 0.0);
        for (int k = threadIdx.x; k < nz * bs; k += blockDim.x) bk[k] = make_double2(0.0, 0.0);
    }
    const bool has = t < nl;
    const int j = has ? (int)leaf_idx[t] : 0;
    const bool act = has && (c_flags[j] & kActive) != 0;
    const uint32_t b = has ? c_begin[j] : 0u, cnt = has ? c_end[j] - b : 0u;
    const double cx = has ? c_cx[j] : 0.0, cy = has ? c_cy[j] : 0.0;
    // rounds of 16 particles: the largest of the wavefront's leaves (uniform)
    uint32_t mx = cnt;
    for (int m = kP2mLanes; m < kWave; m <<= 1) mx = max(mx, (uint32_t)__shfl_xor((int)mx, m, kWave));
    mx = (uint32_t)__builtin_amdgcn_readfirstlane((int)mx);
    for (int k0 = 0; k0 < P1; k0 += kP2mLanes) {
        const int p = k0 + r;
        cd acc = {0.0, 0.0};
        for (uint32_t base = 0; base < mx; base += kP2mLanes) {
            const bool in = act && base + (uint32_t)r < cnt;
            const uint32_t i = in ? b + base + (uint32_t)r : 0u;
            const uint8_t ai = as[i];  // (the four loads in one round)
            const double xi = xs[i], yi = ys[i], qi = qs[i];
            const bool src = in && ai != 0 && qi != 0.0;
            const cd z = {src ? xi - cx : 0.0, src ? yi - cy : 0.0};
            const double q = src ? qi : 0.0;
            const cd z2 = cmul(z, z), z4 = cmul(z2, z2), z8 = cmul(z4, z4);
            cd f = {q, 0.0};
            if (k0 > 0) f = cscale(cpowi(z, k0), q);
            const cd f1 = cmul(f, z), f2 = cmul(f, z2);
            const int me = g * kG + r;
            st(lo[w], me, f);
            st(lo[w], kB + me, f1);
            st(lo[w], 2 * kB + me, f2);
            st(lo[w], 3 * kB + me, cmul(f1, z2));
            st(hi[w], me, cd{1.0, 0.0});
            st(hi[w], kB + me, z4);
            st(hi[w], 2 * kB + me, z8);
            st(hi[w], 3 * kB + me, cmul(z8, z4));
            wave_sync();
            const double2 *fl = lo[w] + (r & 3) * kB + g * kG, *fh = hi[w] + (r >> 2) * kB + g * kG;
#pragma unroll 4
            for (int u = 0; u < kP2mLanes; ++u) {
                const double2 x = fl[u], y = fh[u];
                acc.x += x.x * y.x - x.y * y.y;
                acc.y += x.x * y.y + x.y * y.x;
            }
            wave_sync();
        }
        if (has && p < P1) st(ak, (size_t)j * P1 + p, acc);
    }
}

// M2M for the non-leaf cells of one level: thread per (parent, p),
//   a_p(parent) = sum_children sum_{k=0..p} c_pk a_k(child) d^(p-k),
// d = z_child - z_parent, c_p0 = 1 (fmm2D.cpp:309-379).
__global__ void __launch_bounds__(256)
    k_m2m64(int j0, int j1, int P, const double *tab, const uint8_t *c_flags, const double *c_cx,
            const double *c_cy, const int *c_child, double2 *ak) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int P1 = P + 1;
    if (idx >= (long long)(j1 - j0) * P1) return;
    const int j = j0 + (int)(idx / P1), p = (int)(idx % P1);
    if (c_flags[j] & kLeaf) return;
    const double cx = c_cx[j], cy = c_cy[j];
    cd acc = {0.0, 0.0};
    for (int q = 0; q < 4; ++q) {
        const int ch = c_child[4 * j + q];
        if (ch < 0) continue;
        const cd d = {c_cx[ch] - cx, c_cy[ch] - cy};
        const size_t b = (size_t)ch * P1;
        // Horner from k = 0, which carries the power d^p
        cd sacc = ld(ak, b);
        for (int k = 1; k <= p; ++k) sacc = cadd(cmul(sacc, d), cscale(ld(ak, b + k), tab[p * P1 + k]));
        acc = cadd(acc, sacc);
    }
    st(ak, (size_t)j * P1 + p, acc);
}

// M2M and L2L in spans of three levels (orders P <= 16): one workgroup per cell
// of a span's top level walks that cell's subtree through the span, 16 lanes
// per cell and 16 cells at a time.  A subtree of three levels holds at most 4 +
// 16 + 64 cells however the tree is shaped, so the workgroups stay balanced,
// and a pass over ten levels is three launches instead of seven or nine, each
// of which cost 5 to 9 us whatever it held.  What bounds a launch is its chain
// of dependent loads (about 0.8 us each): the child slots of the three levels,
// then every row and centre of the subtree at once, into LDS, where the levels
// follow each other.
constexpr int kTrP1 = 17;      // orders up to 16
constexpr int kSpan = 3;
constexpr int kSpanBlock = 256;
constexpr int kSpanLanes = 16;                          // lanes per cell
constexpr int kSpanCells = kSpanBlock / kSpanLanes;     // cells at a time

// The subtree of a cell, n <= 3 levels deep: the cells of each level are
// consecutive (the children of consecutive cells, in level-major Morton
// order).  Slot of cell i of level l: span_base(l) + i (0; 1..4; 5..20); link
// (slot, q) = 4 slot + q stands for child q of a slot.
struct SpanTree {
    int child[4 * 21];           // cell index per link, -1: none
    int up[4 + 16 + 64];         // link of cell i of level l at span_up(l) + i
    int lo[kSpan + 1], hi[kSpan + 1];
};
__device__ __forceinline__ int span_base(int l) { return l == 0 ? 0 : l == 1 ? 1 : 5; }
__device__ __forceinline__ int span_up(int l) { return l == 1 ? 0 : l == 2 ? 4 : 20; }

// Fills t (every thread calls it; the first wavefront walks).
__device__ __forceinline__ void span_walk(SpanTree &t, int j, int n, const int *c_child) {
    if (threadIdx.x >= kWave && threadIdx.x < kWave + 4 * 21) t.child[threadIdx.x - kWave] = -1;
    __syncthreads();
    if (threadIdx.x < kWave) {
        const int i = (int)threadIdx.x;
        int a = j, b = j + 1;
        if (i == 0) {
            t.lo[0] = a;
            t.hi[0] = b;
        }
        for (int l = 1; l <= n; ++l) {
            const int c = i < 4 * (b - a) ? c_child[4 * a + i] : -1;  // at most 16 cells
            if (c >= 0) t.child[4 * span_base(l - 1) + i] = c;
            int mn = c >= 0 ? c : 0x7fffffff, mx = c >= 0 ? c + 1 : 0;
#pragma unroll
            for (int m = 1; m < kWave; m <<= 1) {
                mn = min(mn, __shfl_xor(mn, m, kWave));
                mx = max(mx, __shfl_xor(mx, m, kWave));
            }
            a = mx > 0 ? mn : 0;
            b = mx;
            if (c >= 0) t.up[span_up(l) + c - a] = 4 * span_base(l - 1) + i;
            if (i == 0) {
                t.lo[l] = a;
                t.hi[l] = b;
            }
        }
    }
    __syncthreads();
}
__device__ __forceinline__ bool span_leaf(const SpanTree &t, int slot) {
    const int *c = t.child + 4 * slot;
    return (c[0] & c[1] & c[2] & c[3]) < 0;  // every slot -1
}

// M2M for the cells of the `levels` levels from each level-L0 cell (j0 + block)
// down, from the multipoles of the level below them (formed before) and of the
// leaves: lane p of a cell runs k_m2m64's Horner sums over the children's rows
// and its result is both stored and left as its parent's operand.
__global__ void __launch_bounds__(kSpanBlock)
    k_m2m64_span(int j0, int levels, int P, const double *tab, const double *c_cx,
                 const double *c_cy, const int *c_child, double2 *ak) {
    __shared__ SpanTree t;
    __shared__ double s_tab[kTrP1 * kTrP1];
    __shared__ double2 op[4 * 21][kTrP1];  // a child's row per link
    __shared__ double2 ctr[1 + 4 * 21];    // centres: the top cell's, then per link
    const int P1 = P + 1, g = threadIdx.x / kSpanLanes, r = threadIdx.x % kSpanLanes;
    const int top = j0 + (int)blockIdx.x;
    for (int u = threadIdx.x; u < P1 * P1; u += blockDim.x) s_tab[u] = tab[u];
    span_walk(t, top, levels, c_child);
    const int links = 4 * (levels == 1 ? 1 : levels == 2 ? 5 : 21);
    for (int e = threadIdx.x; e < links * P1; e += blockDim.x) {
        const int k = e / P1, ch = t.child[k], s = k >> 2;
        const int l = s == 0 ? 0 : s < 5 ? 1 : 2;
        if (ch >= 0 && (l + 1 == levels || span_leaf(t, span_base(l + 1) + ch - t.lo[l + 1])))
            op[k][e - k * P1] = ak[(size_t)ch * P1 + (e - k * P1)];
    }
    for (int k = threadIdx.x; k <= links; k += blockDim.x) {
        const int ch = k == 0 ? top : t.child[k - 1];
        if (ch >= 0) ctr[k] = make_double2(c_cx[ch], c_cy[ch]);
    }
    __syncthreads();
    for (int l = levels - 1; l >= 0; --l) {
        const int j = t.lo[l] + g, slot = span_base(l) + g;
        if (j < t.hi[l] && !span_leaf(t, slot)) {
            const int up = l == 0 ? -1 : t.up[span_up(l) + g];
            const double2 c0 = ctr[up + 1];
            const double2 (*a)[kTrP1] = op + 4 * slot;
            cd d[4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                d[q] = {ctr[4 * slot + q + 1].x - c0.x, ctr[4 * slot + q + 1].y - c0.y};
            for (int p = r; p < P1; p += kSpanLanes) {
                // the four children's sums side by side, every order's lane
                // over all k (its own end by a select)
                cd sacc[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) sacc[q] = ld(a[q], 0);
#pragma unroll 2
                for (int k = 1; k <= P; ++k) {
                    const double tk = s_tab[p * P1 + k];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const cd n = cadd(cmul(sacc[q], d[q]), cscale(ld(a[q], k), tk));
                        sacc[q] = {k <= p ? n.x : sacc[q].x, k <= p ? n.y : sacc[q].y};
                    }
                }
                cd acc = {0.0, 0.0};
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (t.child[4 * slot + q] >= 0) acc = cadd(acc, sacc[q]);
                st(ak, (size_t)j * P1 + p, acc);
                if (l > 0) st(op[up], p, acc);
            }
        }
        __syncthreads();  // the next level up reads these rows
    }
}

// Principal complex logarithm, as std::log: log|z| + i arg z.
__device__ __forceinline__ cd clog(cd z) { return {log(hypot(z.x, z.y)), atan2(z.y, z.x)}; }

// M2L for every cell of level >= 2 from lists 2 and 4 (fmm2D.cpp:409-556):
// thread per (cell, order).  tab[p][k] holds the coefficient of a_k w^(p+k),
// w = 1/(zs - zt), so b_p = w^p sum_k tab[p][k] a_k w^k (Horner in w).  With
// POT the order-0 row of the potential is formed too (fmm2D.cpp:463-467,
// 504-508): b_0 = a_0 log(z_t - z_s) - sum_{k>=1} a_k (-1)^k / k w^k, and by
// P2L b_0 += q log(z_t - z_i) (:540).  Orders above 16.
template <bool POT>
__global__ void __launch_bounds__(256)
    k_m2l64(int j0, int nc, int P, int list4_mode, const double *tab, const int *l2,
            const uint8_t *n2, const int *l4, const uint8_t *n4, const double *c_cx,
            const double *c_cy, const uint32_t *c_begin, const uint32_t *c_end, const double *xs,
            const double *ys, const double *qs, const uint8_t *as, const double2 *ak, double2 *bk) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int P1 = P + 1, NP = POT ? P1 : P;  // orders formed: 0..P (potential) or 1..P
    if (idx >= (long long)(nc - j0) * NP) return;
    const int j = j0 + (int)(idx / NP), p = (POT ? 0 : 1) + (int)(idx % NP);
    const double cx = c_cx[j], cy = c_cy[j];
    const double *row = tab + (size_t)p * P1;
    cd acc = {0.0, 0.0};
    const int m2 = n2[j], m4 = n4[j];
    for (int u = 0; u < m2 + (list4_mode == 1 ? m4 : 0); ++u) {
        const int sidx = u < m2 ? l2[27 * j + u] : l4[8 * j + (u - m2)];
        const cd w = cinv(cd{c_cx[sidx] - cx, c_cy[sidx] - cy});
        const size_t b = (size_t)sidx * P1;
        if (POT && p == 0) {
            cd sw = {0.0, 0.0};
            for (int k = P; k >= 1; --k)
                sw = cmul(cadd(sw, cscale(ld(ak, b + k), ((k & 1) ? 1.0 : -1.0) / k)), w);
            acc = cadd(acc, cadd(sw, cmul(ld(ak, b), clog(cd{cx - c_cx[sidx], cy - c_cy[sidx]}))));
            continue;
        }
        cd s = cscale(ld(ak, b + P), row[P]);
        for (int k = P - 1; k >= 0; --k) s = cadd(cmul(s, w), cscale(ld(ak, b + k), row[k]));
        acc = cadd(acc, cmul(s, cpowi(w, p)));
    }
    if (list4_mode == 2) {
        // P2L from the active particles of each list-4 leaf (fmm2D.cpp:526-553)
        const double inv_p = p > 0 ? 1.0 / (double)p : 0.0;
        for (int u = 0; u < m4; ++u) {
            const int sidx = l4[8 * j + u];
            for (uint32_t i = c_begin[sidx]; i < c_end[sidx]; ++i) {
                if (!as[i]) continue;
                if (POT && p == 0) {
                    acc = cadd(acc, cscale(clog(cd{cx - xs[i], cy - ys[i]}), qs[i]));
                    continue;
                }
                const cd w = cinv(cd{xs[i] - cx, ys[i] - cy});
                acc = cadd(acc, cscale(cpowi(w, p), -qs[i] * inv_p));
            }
        }
    }
    st(bk, (size_t)j * P1 + p, acc);
}

// M2L by one wavefront per target cell, for orders P <= 16 (the same sums as
// k_m2l64).  The wave stages its M2L sources' coefficients a_k and
// w = 1/(zs - zt) in LDS once; lane l = g NP + i (NP orders per cell) forms order
// p = i (+1 for the field) over the sources u = g, g + G, ... (G = 64 / NP
// groups), and the groups' partial sums are added in group order.  Every lane
// works, and a source's coefficients are read from HBM / L2 once per target
// instead of once per (target, order).
// POT, the potential: lists 2 and 4 (orders 0 .. P).  The field (orders 1 .. P)
// takes list 4 alone, skips a cell without one and adds its sum to b_p, which the
// matrix-core list-2 kernel has written.  List 4 by M2L (list4_mode 1) or P2L (2),
// whose particles the groups split the same way.
constexpr int kM2lwWaves = 4;
constexpr int kM2lwSrc = 27 + 8;  // list 2 <= 27, list 4 <= 8
constexpr int kM2lwP1 = kTrP1;    // orders up to 16

template <bool POT>
__global__ void __launch_bounds__(kWave *kM2lwWaves)
    k_m2l64w(int j0, int nc, int P, int list4_mode, const double *tab, const int *l2,
             const uint8_t *n2, const int *l4, const uint8_t *n4, const double *c_cx,
             const double *c_cy, const uint32_t *c_begin, const uint32_t *c_end,
             const double *xs, const double *ys, const double *qs, const uint8_t *as,
             const double2 *ak, double2 *bk) {
    // sources staged per wavefront: lists 2 and 4, or list 4 alone (a
    // smaller LDS footprint, so more wavefronts reside)
    constexpr int NS = POT ? kM2lwSrc : 8;
    __shared__ double2 sak[kM2lwWaves][NS * kM2lwP1];
    __shared__ double2 sw[kM2lwWaves][NS], slg[kM2lwWaves][NS];
    __shared__ double2 red[kM2lwWaves][kWave];
    const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    const int j = j0 + blockIdx.x * kM2lwWaves + w;
    if (j >= nc) return;  // uniform over the wavefront
    const int P1 = P + 1, NP = POT ? P1 : P, G = kWave / NP;
    const int g = lane / NP, i = lane % NP, p = (POT ? 0 : 1) + i;
    const double cx = c_cx[j], cy = c_cy[j];
    const int m2 = POT ? n2[j] : 0, m4 = n4[j];
    if (!POT && m4 == 0) return;  // uniform over the wavefront
    const int ns = m2 + (list4_mode == 1 ? m4 : 0);
    // staging: w and (potential) log(z_t - z_s) per source, then the a_k rows
    if (lane < ns) {
        const int sidx = lane < m2 ? l2[27 * j + lane] : l4[8 * j + (lane - m2)];
        const cd wv = cinv(cd{c_cx[sidx] - cx, c_cy[sidx] - cy});
        sw[w][lane] = make_double2(wv.x, wv.y);
        if (POT) {
            const cd lg = clog(cd{cx - c_cx[sidx], cy - c_cy[sidx]});
            slg[w][lane] = make_double2(lg.x, lg.y);
        }
    }
    for (int r = lane; r < ns * P1; r += kWave) {
        const int u = r / P1, k = r % P1;
        const int sidx = u < m2 ? l2[27 * j + u] : l4[8 * j + (u - m2)];
        sak[w][u * kM2lwP1 + k] = ak[(size_t)sidx * P1 + k];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    cd acc = {0.0, 0.0};
    if (g < G) {
        const double *row = tab + (size_t)p * P1;
        for (int u = g; u < ns; u += G) {
            const double2 w2 = sw[w][u];
            const cd wv = {w2.x, w2.y};
            const double2 *a = &sak[w][u * kM2lwP1];
            if (POT && p == 0) {
                cd sm = {0.0, 0.0};
                for (int k = P; k >= 1; --k)
                    sm = cmul(cadd(sm, cscale(ld(a, k), ((k & 1) ? 1.0 : -1.0) / k)), wv);
                const double2 lg = slg[w][u];
                acc = cadd(acc, cadd(sm, cmul(ld(a, 0), cd{lg.x, lg.y})));
                continue;
            }
            cd sm = cscale(ld(a, P), row[P]);
            for (int k = P - 1; k >= 0; --k) sm = cadd(cmul(sm, wv), cscale(ld(a, k), row[k]));
            acc = cadd(acc, cmul(sm, cpowi(wv, p)));
        }
        if (list4_mode == 2) {
            // P2L (fmm2D.cpp:526-553): the list-4 leaves' active particles,
            // taken in turn by the groups
            const double inv_p = p > 0 ? 1.0 / (double)p : 0.0;
            int q = 0;
            for (int u = 0; u < m4; ++u) {
                const int sidx = l4[8 * j + u];
                for (uint32_t pi = c_begin[sidx]; pi < c_end[sidx]; ++pi, ++q) {
                    if (q % G != g || !as[pi]) continue;
                    if (POT && p == 0) {
                        acc = cadd(acc, cscale(clog(cd{cx - xs[pi], cy - ys[pi]}), qs[pi]));
                        continue;
                    }
                    const cd wv = cinv(cd{xs[pi] - cx, ys[pi] - cy});
                    acc = cadd(acc, cscale(cpowi(wv, p), -qs[pi] * inv_p));
                }
            }
        }
    }
    red[w][lane] = make_double2(acc.x, acc.y);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane < NP) {
        cd sum = {0.0, 0.0};
        for (int gg = 0; gg < G; ++gg) sum = cadd(sum, ld(red[w], gg * NP + lane));
        const size_t o = (size_t)j * P1 + (POT ? 0 : 1) + lane;
        st(bk, o, POT ? sum : cadd(ld(bk, o), sum));
    }
}

// M2L of the FP64 path on the matrix cores (orders P <= 16, field and velocity;
// the potential keeps k_m2l64w) and of the type-1 path (T1, ND = P <= 16).
// With len the level's cell side and delta = (zs - zt) / len (|dx|, |dy| <= 3,
// not both <= 1: 40 offsets), the list-2 sum
//   b_p = sum_k tab[p][k] a_k (zs - zt)^-(p+k)
// is, in the scaled coefficients a^_k = a_k len^-k and b^_p = b_p len^p,
//   b^ = sum over offsets of M_delta a^,  M_delta[p][k] = tab[p][k] delta^-(p+k),
// a realified 2P x 2(P+1) matrix per offset (fmm64_mfma_table), the A operand;
// the B operand is a source cell's a^.  Type 1 has a_0..a_{P-1} and Cauchy
// coefficients b_0..b_P: b_l = sum_k tab[l][k] a_k (zs - zt)^-(l+1+k), 2(P+1) x
// 2P.  The offset is exact here, where the reference forms zs - zt from rounded
// centres.  A stored centre is off its grid position by up to 2^-53 |coordinate|
// per rounding, which over the cell side is eps, and b by about that much: 1e-12
// for a field 100 of its own sizes from the origin, level 7.  Type 1, whose
// other stages use the stored centres, moves the sources' expansions to the grid
// and the targets' back to their own centres, to first order in eps: 1e-15 of the
// oracle (without it 6e-13 at 50 sizes from the origin, 4e-10 at 5e4, 2e-12 at
// level 16).  Trees with a larger eps (t1_on_grid) go to k_m2l_t1.
//
// A workgroup takes 96 consecutive cells of one level and sorts them into the
// four classes of a cell's place in its parent: list 2 lies within the
// parent's neighbours, so a class has 27 of the 40 offsets, and 32 targets of
// one class (16 above order 12) take an offset's matrix together.  Two
// wavefronts share a class (every other offset each, summed through LDS).
// What bound 16 unsorted targets at a time (120 us on the 780k flat plate, the
// matrix cores busy a quarter of it) was the L1: 1 GB of matrices from L2, and
// a lane's 8 or 16 bytes of a source row at a time, 64 accesses a load, up to 27
// times per row.  The source rows of the workgroup, about 200, are found with a
// hash table and staged in LDS once, scaled; a matrix is read once per 32
// targets, the next one's loads under way while this one's products run, and a
// half of the 32 without a source at the offset takes no products: 81 us, now
// bound by the products (14 offsets a wavefront; the matrix cores are busy on 0.33
// of the cycles) and, a quarter, by the lists' and rows' dependent loads.  Type 1
// at 200k: one thread per order and cell 121 us, 37 us.  (96 cells and not 128:
// where some children are missing a class would exceed its 32 targets and need a
// second round.)
//
// NQ = 1: a workgroup takes one of the four classes, all its wavefronts the
// class's offsets.  A tree of a few workgroups' cells leaves the chip idle
// while each of them runs its 14 offsets in turn (18 of 28 us): the 2000
// particle solve takes 226 us with four classes per workgroup and 218 with one,
// 54k vortices 371 and 364; the lists are read four times, which a larger tree
// pays for: 780k 543 and 593, type 1 at 200k 422 and 435.
//
// Rows beyond a multiple of 16 go four at a time to v_mfma_f64_4x4x4f64 if they
// are at most 8 (a quarter of the cycles each): its A operand holds row l % 4
// and column l / 16 of a step, its B operand is laid out as the 16x16x4 one
// (target l % 16, step row l / 16) and its result is row l / 16 of target
// l % 16.  The 16x16x4 result is row 4 v + l / 16 of target l % 16.
constexpr int kM2lCells = 96;   // cells per workgroup
constexpr int kM2lWaves = 8;
constexpr int kM2lBlock = kWave * kM2lWaves;
constexpr int kM2lSlots = 36;   // 6 x 6 source places around the parent's neighbourhood
constexpr int kM2lHash = 1024;  // hash table of the workgroup's sources
constexpr int kM2lProbes = 16;
constexpr int kM2lRowBytes = 56 * 1024;  // LDS of the staged rows
typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t compact1by1(uint32_t v) {
    v &= 0x55555555u;
    v = (v | (v >> 1)) & 0x33333333u;
    v = (v | (v >> 2)) & 0x0F0F0F0Fu;
    v = (v | (v >> 4)) & 0x00FF00FFu;
    v = (v | (v >> 8)) & 0x0000FFFFu;
    return v;
}

// Type 1: what the k-th scaled coefficient of a source gains when its expansion
// is moved from the cell's own centre to the grid's, residual eps sides away:
// k eps a^_{k-1} (the next term is of order eps^2, below 1e-20 of a^).
__device__ __forceinline__ cd on_grid(v2d eps, v2d prev, double sc, int k) {
    return cscale(cmul(cd{eps.x, eps.y}, cd{prev.x * sc, prev.y * sc}), (double)k);
}

// Row 2 l, 2 l + 1 of a cell's scaled result: the parts of b + 2 l.
__device__ __forceinline__ void store_row(double *b, int row, double v, const double *sc) {
    b[row] = v * sc[row / 2 + 1];
}

// The workgroups of each level: level L (2 .. maxL) has blocks first[L] ..
// first[L + 1] - 1 and cells cell0[L] .. cell0[L + 1] - 1.
struct M2lLevels {
    int first[kMaxDepth + 2], cell0[kMaxDepth + 2];
    int maxL;
};

// Sizes of an order's matrices (host and device).
template <int P, bool T1>
struct M2lShape {
    static constexpr int RW = T1 ? 2 * P + 2 : 2 * P;        // rows
    static constexpr int K = T1 ? 2 * P : 2 * P + 2;         // columns
    static constexpr int KP = (K + 7) / 8, KS = 2 * KP;      // steps of 4 columns, in pairs
    static constexpr int R16 = RW / 16, REM = RW % 16;
    static constexpr int T16 = REM > 8 ? R16 + 1 : R16;      // 16-row tiles
    static constexpr int T4 = REM > 8 ? 0 : (REM + 3) / 4;   // 4-row tiles after them
    static constexpr int NS = T16 + T4;
    static constexpr int ACC = 4 * T16 + T4;                 // accumulators per lane and target set
    // sets of 16 targets per wavefront: two up to order 12, where they need the 128
    // registers and up to 72 bytes of scratch beside them (orders 8 to 12); a solve
    // of a 200k plate takes 322, 335 and 350 us at orders 8, 10 and 12 and, with one
    // set, 361 and 434 at 13 and 16
    static constexpr int U = P <= 12 ? 2 : 1;
    static constexpr bool AHEAD = KS * NS <= 12;             // and the next matrix too
};

template <int P, bool T1, int NQ>
__global__ void __launch_bounds__(kM2lBlock) __attribute__((amdgpu_waves_per_eu(4, 4)))
    k_m2l64_mfma(const DevHdr *hdr, M2lLevels lv, const uint32_t *c_key, const int *l2,
                 const uint8_t *n2, const double *R, const double2 *cres, const double2 *ak,
                 double2 *bk) {
    using Sh = M2lShape<P, T1>;
    constexpr int K = Sh::K, KP = Sh::KP, KS = Sh::KS, NS = Sh::NS, T16 = Sh::T16, T4 = Sh::T4;
    constexpr int P1 = P + 1, U = Sh::U;
    constexpr int kShare = kM2lWaves / NQ;          // wavefronts per class
    constexpr int AS = T1 ? P : P1;                 // coefficients per cell of ak
    constexpr int kFit = kM2lRowBytes / (16 * AS);  // rows that fit (a row has a hash slot)
    constexpr int kRows = kFit < kM2lHash ? kFit : kM2lHash;
    __shared__ union {
        double2 row[kRows][AS];
        double red[NQ][kShare - 1][U * Sh::ACC][kWave];
    } s;
    // source per target and place: a staged row, -1: none, below: cell -2 - v
    __shared__ int src[kM2lCells][kM2lSlots];
    __shared__ int ht[kM2lHash];            // source cells by hash, -1: free
    __shared__ uint16_t hid[kM2lHash];      // their rows
    __shared__ int rowcell[kRows];
    __shared__ uint8_t memb[4][kM2lCells];  // the classes' members
    __shared__ int n_memb[2][4], n_rows;
    __shared__ double s_sc[P1 + 1];         // len^-k
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lane = tid & (kWave - 1);
    const int blk = (int)blockIdx.x / (4 / NQ), only = NQ == 1 ? (int)blockIdx.x % 4 : 0;
    int L = 2;
    while (L < lv.maxL && blk >= lv.first[L + 1]) ++L;
    const int j0 = lv.cell0[L] + kM2lCells * (blk - lv.first[L]);
    const int cnt = min(kM2lCells, lv.cell0[L + 1] - j0);
    // list entries of the workgroup's cells, 27 places per cell
    constexpr int kPer = (27 * kM2lCells + kM2lBlock - 1) / kM2lBlock;
    int ent[kPer], slot[kPer];
    uint32_t kt[kPer], ks[kPer];  // keys of the target and the source
    {
        // (every load of a round in flight together: clamped, then selected)
        int len[kPer];
#pragma unroll
        for (int v = 0; v < kPer; ++v) {
            const int e = min(tid + v * kM2lBlock, 27 * cnt - 1), c = e / 27;
            len[v] = (int)n2[j0 + c];
            kt[v] = c_key[j0 + c];
            ent[v] = l2[27 * (size_t)j0 + e];
        }
#pragma unroll
        for (int v = 0; v < kPer; ++v) {
            const int e = tid + v * kM2lBlock;
            if (e >= 27 * cnt || e % 27 >= len[v] || (NQ == 1 && (int)(kt[v] & 3u) != only))
                ent[v] = -1;
        }
#pragma unroll
        for (int v = 0; v < kPer; ++v) ks[v] = c_key[max(ent[v], 0)];
    }
    if (tid <= P1) {
        const double inv = ldexp(1.0 / hdr->root_len, L);
        double sc = 1.0;
        for (int k = 0; k < tid; ++k) sc *= inv;
        s_sc[tid] = sc;
    }
    for (int t = tid; t < kM2lCells * kM2lSlots; t += kM2lBlock) (&src[0][0])[t] = -1;
    for (int t = tid; t < kM2lHash; t += kM2lBlock) ht[t] = -1;
    if (tid == 0) n_rows = 0;
    // the classes' members, in cell order (two wavefronts hold a cell a lane)
    const int cls = tid < cnt ? (int)(c_key[j0 + tid] & 3u) : -1;
    uint64_t same = 0;
    if (w < 2) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint64_t m = __ballot(cls == q);
            if (cls == q) same = m;
            if (lane == 0) n_memb[w][q] = __popcll(m);
        }
    }
    __syncthreads();
    if (cls >= 0) {
        const int r = __popcll(same & (lane ? ~0ull >> (kWave - lane) : 0ull)) +
                      (w == 1 ? n_memb[0][cls] : 0);
        memb[cls][r] = (uint8_t)tid;
    }
    // the distinct sources: hash slot of every entry (none after kM2lProbes
    // probes: read from global memory below), then a row per used slot
#pragma unroll
    for (int v = 0; v < kPer; ++v) {
        slot[v] = -1;
        if (ent[v] < 0) continue;
        uint32_t h = ((uint32_t)ent[v] * 2654435761u) >> 22;
#pragma unroll 1
        for (int t = 0; t < kM2lProbes; ++t, h = (h + 1) & (kM2lHash - 1)) {
            const int old = atomicCAS(&ht[h], -1, ent[v]);
            if (old == -1 || old == ent[v]) {
                slot[v] = (int)h;
                break;
            }
        }
    }
    __syncthreads();
    for (int t = tid; t < kM2lHash; t += kM2lBlock) {
        const bool used = ht[t] >= 0;
        const uint64_t m = __ballot(used);
        int base = 0;
        if (lane == 0) base = atomicAdd(&n_rows, __popcll(m));
        base = __builtin_amdgcn_readfirstlane(base);
        const int id = base + __popcll(m & (lane ? ~0ull >> (kWave - lane) : 0ull));
        hid[t] = (uint16_t)id;
        if (used && id < kRows) rowcell[id] = ht[t];
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < kPer; ++v) {
        if (ent[v] < 0) continue;
        const int c = (tid + v * kM2lBlock) / 27;
        // place of a source: (dx + 2 + qx) + 6 (dy + 2 + qy), with (qx, qy) the
        // target's place in its parent
        const int jx = (int)compact1by1(kt[v]), jy = (int)compact1by1(kt[v] >> 1);
        const int px = (int)compact1by1(ks[v]) - jx + 2 + (jx & 1);
        const int py = (int)compact1by1(ks[v] >> 1) - jy + 2 + (jy & 1);
        const int id = slot[v] >= 0 ? (int)hid[slot[v]] : kRows;
        src[c][px + 6 * py] = id < kRows ? id : -2 - ent[v];
    }
    const int nrow = min(n_rows, kRows);
    const int q = NQ == 1 ? only : w & 3, part = w / NQ;  // class, share
    const int qx = q & 1, qy = q >> 1;
    const int nm = n_memb[0][q] + n_memb[1][q];
    const int n = lane % 16, kq = lane / 16;
    double *bo = reinterpret_cast<double *>(bk);
    // (uniform over the workgroup: the classes' longest member list; more than
    // one round only in ragged trees)
    int most = 0;
    for (int k = 0; k < 4; ++k)
        if (NQ == 4 || k == only) most = max(most, n_memb[0][k] + n_memb[1][k]);
    for (int rd = 0; 16 * U * rd < most; ++rd) {
        __syncthreads();  // (the sums of the round before share the rows' space)
        for (int e0 = tid; e0 < nrow * AS; e0 += 4 * kM2lBlock) {
            v2d v[4], pv[T1 ? 4 : 1], eps[T1 ? 4 : 1];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int e = min(e0 + t * kM2lBlock, nrow * AS - 1), r = e / AS, k = e - r * AS;
                const v2d *row = reinterpret_cast<const v2d *>(ak) + (size_t)rowcell[r] * AS;
                v[t] = row[k];
                if (T1) {
                    pv[t] = row[max(k - 1, 0)];
                    eps[t] = reinterpret_cast<const v2d *>(cres)[rowcell[r]];
                }
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int e = min(e0 + t * kM2lBlock, nrow * AS - 1), r = e / AS, k = e - r * AS;
                cd a = {v[t].x * s_sc[k], v[t].y * s_sc[k]};
                if (T1 && k > 0) a = cadd(a, on_grid(eps[T1 ? t : 0], pv[T1 ? t : 0], s_sc[k - 1], k));
                st(s.row[r], k, a);
            }
        }
        __syncthreads();
        v4d acc[U][T16 > 0 ? T16 : 1];
        double acc4[U][T4 > 0 ? T4 : 1];
        int mt[U], cs[U];  // the lane's targets, and their sources at the place
        bool use[U];       // whether any lane has one
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int t = 0; t < T16; ++t) acc[u][t] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int t = 0; t < T4; ++t) acc4[u][t] = 0.0;
            const int r = 16 * (U * rd + u) + n;
            mt[u] = r < nm ? memb[q][r] : -1;
        }
        // the next place of this wavefront that a target of the round uses
        int place = -1, turn = 0;
        auto next = [&]() {
#pragma unroll 1
            for (++place; place < kM2lSlots; ++place) {
                const int dx = place % 6 - 2 - qx, dy = place / 6 - 2 - qy;
                if (dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1) continue;
                if (turn++ % kShare != part) continue;
                bool any = false;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    cs[u] = mt[u] >= 0 ? src[mt[u]][place] : -1;
                    use[u] = __ballot(cs[u] != -1) != 0;
                    any |= use[u];
                }
                if (any) return;
            }
        };
        // the matrix of the place (index of its offset among the 40, dy major)
        auto matrix = [&](double (&A)[KS * NS]) {
            const int dx = place % 6 - 2 - qx, dy = place / 6 - 2 - qy;
            const int oc = (dx + 3) + 7 * (dy + 3) -
                           (dy < -1 ? 0 : dy > 1 ? 9 : 3 * (dy + 1) + (dx > 1 ? 3 : 0));
            const double *Ro = R + (size_t)oc * KS * NS * kWave + lane;
#pragma unroll
            for (int t = 0; t < KS * NS; ++t) A[t] = Ro[t * kWave];
        };
        double A[KS * NS], nA[Sh::AHEAD ? KS * NS : 1];
        next();
        if (Sh::AHEAD && place < kM2lSlots) matrix(A);
        while (place < kM2lSlots) {
            if (!Sh::AHEAD) matrix(A);
            int cu[U];
            bool on[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                cu[u] = cs[u];
                on[u] = use[u];
            }
            next();
            if constexpr (Sh::AHEAD)
                if (place < kM2lSlots) matrix(nA);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (U > 1 && !on[u]) continue;
                // the lane's columns 8 m + 2 kq and + 1 are a_k's parts, k = 4 m + kq
                v2d b[KP];
#pragma unroll
                for (int m = 0; m < KP; ++m) {
                    b[m] = v2d{0.0, 0.0};
                    if (cu[u] >= 0 && 4 * m + kq < K / 2)
                        b[m] = *reinterpret_cast<const v2d *>(&s.row[cu[u]][4 * m + kq]);
                }
                if (__ballot(cu[u] < -1))  // rows beyond the staged ones
#pragma unroll
                    for (int m = 0; m < KP; ++m)
                        if (cu[u] < -1 && 4 * m + kq < K / 2) {
                            const int k = 4 * m + kq, sc = -2 - cu[u];
                            const v2d *row = reinterpret_cast<const v2d *>(ak) + (size_t)sc * AS;
                            cd a = {row[k].x * s_sc[k], row[k].y * s_sc[k]};
                            if (T1 && k > 0)
                                a = cadd(a, on_grid(reinterpret_cast<const v2d *>(cres)[sc],
                                                    row[k - 1], s_sc[k - 1], k));
                            b[m] = v2d{a.x, a.y};
                        }
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const double x = b[ks / 2][ks & 1];
#pragma unroll
                    for (int t = 0; t < T16; ++t)
                        acc[u][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[ks * NS + t], x,
                                                                         acc[u][t], 0, 0, 0);
#pragma unroll
                    for (int t = 0; t < T4; ++t)
                        acc4[u][t] = __builtin_amdgcn_mfma_f64_4x4x4f64(A[ks * NS + T16 + t], x,
                                                                        acc4[u][t], 0, 0, 0);
                }
            }
            if constexpr (Sh::AHEAD)
#pragma unroll
                for (int t = 0; t < KS * NS; ++t) A[t] = nA[t];
        }
        // sum of the class's wavefronts, and the store by the first of them
        __syncthreads();
        if (part > 0) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
#pragma unroll
                for (int t = 0; t < T16; ++t)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        s.red[NQ == 1 ? 0 : q][part - 1][u * Sh::ACC + 4 * t + v][lane] = acc[u][t][v];
#pragma unroll
                for (int t = 0; t < T4; ++t)
                    s.red[NQ == 1 ? 0 : q][part - 1][u * Sh::ACC + 4 * T16 + t][lane] = acc4[u][t];
            }
        }
        __syncthreads();
        if (part == 0) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int mc = mt[u];
                double(*red)[kWave] = &s.red[NQ == 1 ? 0 : q][0][u * Sh::ACC];
                // sum i, row 4 i + kq: stored, or (type 1) left in LDS
                auto put = [&](double v, int i) {
#pragma unroll
                    for (int o = 0; o < kShare - 1; ++o)
                        v += s.red[NQ == 1 ? 0 : q][o][u * Sh::ACC + i][lane];
                    if constexpr (T1) red[i][lane] = v;
                    else if (mc >= 0 && 4 * i + kq < Sh::RW)
                        store_row(bo + (size_t)(j0 + mc) * P1 * 2 + 2, 4 * i + kq, v, s_sc);
                };
#pragma unroll
                for (int t = 0; t < T16; ++t)
#pragma unroll
                    for (int v = 0; v < 4; ++v) put(acc[u][t][v], 4 * t + v);
#pragma unroll
                for (int t = 0; t < T4; ++t) put(acc4[u][t], 4 * T16 + t);
                if constexpr (T1) {
                    // from the grid's centre to the target's: b_l + (l + 1) eps
                    // b_{l+1}, whose parts are two rows on
                    wave_sync();
                    const double2 e = mc >= 0 ? cres[j0 + mc] : make_double2(0.0, 0.0);
#pragma unroll 1
                    for (int i = 0; 4 * i < Sh::RW; ++i) {
                        const int row = 4 * i + kq, nxt = row + 2;
                        double v = red[i][lane];
                        if (nxt < Sh::RW)
                            v += (double)(row / 2 + 1) *
                                 (e.x * red[nxt / 4][16 * (nxt & 3) + n] +
                                  (row & 1 ? e.y : -e.y) * red[nxt / 4][16 * ((nxt & 3) ^ 1) + n]);
                        if (mc >= 0 && row < Sh::RW)
                            store_row(bo + (size_t)(j0 + mc) * P1 * 2, row, v, s_sc);
                    }
                }
                if (!T1 && kq == 0 && mc >= 0)  // b_0 is not formed
                    bk[(size_t)(j0 + mc) * P1] = make_double2(0.0, 0.0);
            }
        }
    }
}

// L2L for the cells of one level (>= 3): each child adds its parent's shifted
// local expansion.  tab[p][k] = C(k, p).  Orders 1..P, and 0 for the
// potential (fmm2D.cpp:637-643 runs p from 0).
template <bool POT>
__global__ void __launch_bounds__(256)
    k_l2l64(int j0, int j1, int P, const double *tab, const int *c_parent, const double *c_cx,
            const double *c_cy, double2 *bk) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int P1 = P + 1, NP = POT ? P1 : P;
    if (idx >= (long long)(j1 - j0) * NP) return;
    const int j = j0 + (int)(idx / NP), p = (POT ? 0 : 1) + (int)(idx % NP);
    const int par = c_parent[j];
    const cd d = {c_cx[j] - c_cx[par], c_cy[j] - c_cy[par]};
    const size_t b = (size_t)par * P1;
    const double *row = tab + (size_t)p * P1;
    cd s = cscale(ld(bk, b + P), row[P]);
    for (int k = P - 1; k >= p; --k) s = cadd(cmul(s, d), cscale(ld(bk, b + k), row[k]));
    const size_t o = (size_t)j * P1 + p;
    st(bk, o, cadd(ld(bk, o), s));
}

// L2L for the cells up to `levels` below each level-L0 cell (j0 + block), whose
// own expansion is complete (k_m2m64_span's walk, downward): a cell's parent's
// row is read from LDS, lane p of the cell forms its order's sum, and the row
// stays in LDS for the next level.
enum L2lKind { kL2lField, kL2lPot, kL2lT1 };

// Type-1 L2L (biotsavart_fmm_2d.cpp:283-312), order l of a child displaced by d
// from its parent (local coefficients b, orders 0..ND):
//   sum_{k = l..ND} coef[l][k] d^expo[l][k] b_k,
// with the table of the shift as the reference runs it (or the exact one).
// Along a row the exponent rises by one per term except at most once, where
// it is formed afresh.
__device__ __forceinline__ cd l2l_t1_sum(int l, int ND, const double *coef, const int *expo, cd d,
                                         const double2 *b) {
    const int NL = ND + 1;
    cd s = {0.0, 0.0}, pw = {1.0, 0.0};
    int e_prev = 0;
    for (int k = l; k <= ND; ++k) {
        const int e = expo[l * NL + k];
        if (e == e_prev + 1) pw = cmul(pw, d);
        else if (e != e_prev) pw = cpowi(d, e);
        e_prev = e;
        s = cadd(s, cscale(cmul(pw, ld(b, k)), coef[l * NL + k]));
    }
    return s;
}

template <int KIND>
__global__ void __launch_bounds__(kSpanBlock)
    k_l2l64_span(int j0, int levels, int P, const double *tab, const int *expo,
                 const int *c_child, const double *c_cx, const double *c_cy, double2 *bk) {
    __shared__ SpanTree t;
    __shared__ double s_tab[kTrP1 * kTrP1];
    __shared__ int s_exp[KIND == kL2lT1 ? kTrP1 * kTrP1 : 1];
    __shared__ double2 row[1 + 4 * 21][kTrP1];  // the top cell's, then per link
    __shared__ double2 ctr[1 + 4 * 21];
    __shared__ double2 pw[KIND == kL2lT1 ? kSpanCells : 1][kTrP1];  // powers of d
    const int P1 = P + 1, g = threadIdx.x / kSpanLanes, r = threadIdx.x % kSpanLanes;
    const int top = j0 + (int)blockIdx.x;
    for (int u = threadIdx.x; u < P1 * P1; u += blockDim.x) {
        s_tab[u] = tab[u];
        if (KIND == kL2lT1) s_exp[u] = expo[u];
    }
    span_walk(t, top, levels, c_child);
    const int links = 4 * (levels == 1 ? 1 : levels == 2 ? 5 : 21);
    for (int e = threadIdx.x; e < (links + 1) * P1; e += blockDim.x) {
        const int k = e / P1, j = k == 0 ? top : t.child[k - 1];
        if (j >= 0) row[k][e - k * P1] = bk[(size_t)j * P1 + (e - k * P1)];
    }
    for (int k = threadIdx.x; k <= links; k += blockDim.x) {
        const int j = k == 0 ? top : t.child[k - 1];
        if (j >= 0) ctr[k] = make_double2(c_cx[j], c_cy[j]);
    }
    __syncthreads();
    for (int l = 1; l <= levels; ++l) {
        for (int i = g; i < t.hi[l] - t.lo[l]; i += kSpanCells) {
            const int link = t.up[span_up(l) + i], slot = link >> 2;
            // the parent's own link, or the top cell
            const int par = slot == 0 ? 0 : t.up[span_up(l - 1) + slot - span_base(l - 1)] + 1;
            const double2 *b = row[par];
            const cd d = {ctr[link + 1].x - ctr[par].x, ctr[link + 1].y - ctr[par].y};
            if (KIND == kL2lT1) {
                for (int p = r; p < P1; p += kSpanLanes) st(pw[g], p, cpowi(d, p));
                wave_sync();
            }
            for (int p = r; p < P1; p += kSpanLanes) {
                cd v = ld(row[link + 1], p);
                if (KIND == kL2lT1) {
                    // l2l_t1_sum with the powers at hand
                    cd s = {0.0, 0.0};
#pragma unroll 4
                    for (int k = 0; k < P1; ++k) {
                        const cd n = cscale(cmul(ld(pw[g], s_exp[p * P1 + k]), ld(b, k)),
                                            s_tab[p * P1 + k]);
                        s = {k >= p ? s.x + n.x : s.x, k >= p ? s.y + n.y : s.y};
                    }
                    v = cadd(v, s);
                } else if (KIND == kL2lPot || p > 0) {
                    const double *tr = s_tab + p * P1;
                    cd s = cscale(ld(b, P), tr[P]);
#pragma unroll 4
                    for (int k = P - 1; k >= (KIND == kL2lPot ? 0 : 1); --k) {
                        const cd n = cadd(cmul(s, d), cscale(ld(b, k), tr[k]));
                        s = {k >= p ? n.x : s.x, k >= p ? n.y : s.y};
                    }
                    v = cadd(v, s);
                }
                if (KIND != kL2lField || p > 0) st(bk, (size_t)(t.lo[l] + i) * P1 + p, v);
                st(row[link + 1], p, v);
            }
            if (KIND == kL2lT1) wave_sync();
        }
        __syncthreads();  // the next level down reads these rows
    }
}

// 1/x to full double precision: the hardware estimate y (error under 2^-22)
// corrected by y (e + e^2), e = 1 - x y, which leaves e^3.
__device__ __forceinline__ double rcp64(double x) {
    const double y = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, y, 1.0);
    return fma(y, fma(e, e, e), y);
}

// a / b as the division rounds it, for a and b well inside the range: a rcp64(b)
// corrected by its remainder (without it a quarter of the quotients are off in the
// last place; the two FMAs do not show in a solve, 417 us with and 423 without at
// 200k, Gaussian).
__device__ __forceinline__ double div64(double a, double b) {
    const double y = rcp64(b), q = a * y;
    return fma(fma(-b, q, a), y, q);
}

// Regularization factor of a near-field pair, 2 pi q of regul_func_2d
// (regularization_function_2d.cpp:11-37) at rho^2 = r^2 / sij^2, in the
// reference's form: 1 high-order algebraic, 2 Gaussian, 3 super-Gaussian.
template <int ICUT>
__device__ __forceinline__ double regul64(double rho2) {
    if (ICUT == 1) return (rho2 * (rho2 + 2.0)) / ((rho2 + 1.0) * (rho2 + 1.0));
    const double qt = -0.5 * rho2;
    if (ICUT == 2) return 1.0 - exp(qt);
    return 1.0 - (1.0 - qt) * exp(qt);
}

// Evaluation: W wavefronts per leaf (1, or 4 when the leaves alone would leave
// most of the chip idle).  Lanes split into G groups of 64 / G; a lane owns two
// targets, a group all of the leaf's (G by leaf size), and the groups and
// wavefronts split the sources and list-3 cells and are reduced at the end.
//
// The kernel is bound by vector-ALU issue where leaves abound (0.76 of the
// cycles on the 780k flat plate, half of them outside the pair loop, whose
// leaves hold 16 targets) and by the latency of one leaf's chain where they
// do not.  Two targets per lane halve the LDS reads per pair (24 B a source,
// no index: only the leaf's own particles need the self test); the list-1
// cells' ranges are read 64 at a time, so a leaf waits for three dependent
// loads, not for three per cell.  780k flat plate 162 -> 115 us; 2,000
// particles 55 -> 13 us; 100k clusters with the Gaussian kernel 146 -> 88 us.
//
// MODE 0: the singular P2P of fmm2D (fmm2D.cpp:164-173); a pair at r = 0
// raises DUPLICATE_POINTS.  1..3: the type-1 near field of direct_sum
// (subroutine_all_fmm_2d.cpp:594-627): each pair term times regul64 at
// sij^2 = (si^2 + sj^2) / 4 (ss: the sorted sizes); pairs at r = 0 add nothing.
// kPot: the potential (fmm2D::calcPotential, fmm2D.cpp:681-896): P2P
// q log(r^2) / 2 (potDirSum, :77-122), M2P Re[a_0 log(z - zc) -
// sum_p a_p (z - zc)^-p / p] (:817-834), L2P Re[b_0 + sum_p b_p (z - z0)^p]
// (:854-866); a pair at r = 0 raises DUPLICATE_POINTS (log 0).
// T1: the type-1 FMM (biotsavart_fmm_2d.cpp:321-419): pairs at r = 0 add
// nothing whatever the kernel; the multipoles hold orders 0..P-1 (stride P)
// and the local expansions orders 0..P (stride P + 1) in the Cauchy form
// F = sum_l b_l (z - z0)^l.
constexpr int kEvalWaves = 4;
constexpr int kStage64 = 128;   // sources staged per wavefront per round
constexpr int kPot = 4;
constexpr int kEvalP1 = 41;     // coefficients of a leaf's local expansion (orders up to 40)

struct Eval64Args {
    const uint32_t *leaf_idx;
    int nl, P;
    const uint8_t *c_flags;
    const uint32_t *c_begin, *c_end;
    const double *c_cx, *c_cy;
    const uint32_t *off1;
    const int *l1;
    const uint32_t *off3;
    const int *l3;
    const double *xs, *ys, *qs, *ss;
    const uint32_t *perm;
    const double2 *ak, *bk;
    int velocity, mask;
    double u_inf, v_inf;
    double *out_a, *out_b;
    const DevHdr *hdr;
    unsigned *flags;
};

// LDS of one wavefront: staged sources (the list-3 rows and the partial sums
// pass through the same space), the list-1 cells' offsets, the leaf's local
// coefficients.
template <int MODE>
struct Eval64Lds {
    double2 xy[kStage64];
    double q[kStage64];
    double s2[MODE >= 1 && MODE <= 3 ? kStage64 : 1];
    uint32_t off[kWave], beg[kWave];
    double2 b[kEvalP1];
};

// One pair's contribution to a target at (xi, yi): the field in (ex, ey), or
// the potential in ex.  skip: the target itself (own leaf only); tame: every
// size of the round is well inside the range of div64 (a size of zero, say, is
// not: the division's limits then hold).
template <int MODE, bool T1, bool OWN>
__device__ __forceinline__ void pair64(double xi, double yi, double si2, double2 s, double q,
                                       double sj2, bool skip, bool tame, double &ex,
                                       double &ey) {
    const double dx = xi - s.x, dy = yi - s.y;
    const double r2 = dx * dx + dy * dy;
    if (MODE == kPot) {
        const double t = q * log(r2) / 2.0;
        ex += OWN && skip ? 0.0 : t;
        return;
    }
    double qr = q * rcp64(r2);
    if (MODE == 0) {
        if (T1) qr = r2 > 0.0 ? qr : 0.0;
        else if (OWN) qr = skip ? 0.0 : qr;
    } else {
        const double sij2 = 0.25 * (si2 + sj2);
        const double rho2 = tame ? div64(r2, sij2) : r2 / sij2;
        // the factor is 1 to the last bit beyond rho^2 = 90 (1 - (1 + h) e^-h,
        // h = 45); a wavefront with no closer pair skips the exponential
        if (MODE == 1 || __ballot(!(rho2 > 90.0 && rho2 < 1e300))) qr *= regul64<MODE>(rho2);
        qr = r2 > 0.0 ? qr : 0.0;
    }
    ex += qr * dx;
    ey += qr * dy;
}

// The staged sources g, g + G, ... (nu of them per group, padded) against the
// lane's two targets; r0: the sorted index of stage slot 0 (own leaf).
template <int MODE, bool T1, bool OWN, int G>
__device__ __forceinline__ void pairs64g(const Eval64Lds<MODE> &l, int g, int nu,
                                         const double (&xi)[2], const double (&yi)[2],
                                         const double (&si2)[2], uint32_t r0, uint32_t i0,
                                         uint32_t i1, bool tame, double (&ex)[2],
                                         double (&ey)[2]) {
    constexpr int kUnroll = MODE == 0 ? 2 : 1;
#pragma unroll kUnroll
    for (int u = 0; u < nu; ++u) {
        const int r = g + u * G;
        const double2 s = l.xy[r];
        const double q = l.q[r], sj2 = MODE >= 1 && MODE <= 3 ? l.s2[r] : 0.0;
        const uint32_t src = r0 + (uint32_t)r;
        pair64<MODE, T1, OWN>(xi[0], yi[0], si2[0], s, q, sj2, OWN && src == i0, tame, ex[0],
                              ey[0]);
        pair64<MODE, T1, OWN>(xi[1], yi[1], si2[1], s, q, sj2, OWN && src == i1, tame, ex[1],
                              ey[1]);
    }
}

// The same with the group count G a compile-time constant (LDS offsets and
// unrolling), chosen per call.
template <int MODE, bool T1, bool OWN>
__device__ __forceinline__ void pairs64(const Eval64Lds<MODE> &l, int G, int g, int nu,
                                        const double (&xi)[2], const double (&yi)[2],
                                        const double (&si2)[2], uint32_t r0, uint32_t i0,
                                        uint32_t i1, bool tame, double (&ex)[2],
                                        double (&ey)[2]) {
    switch (G) {
        case 16: pairs64g<MODE, T1, OWN, 16>(l, g, nu, xi, yi, si2, r0, i0, i1, tame, ex, ey); break;
        case 8: pairs64g<MODE, T1, OWN, 8>(l, g, nu, xi, yi, si2, r0, i0, i1, tame, ex, ey); break;
        case 4: pairs64g<MODE, T1, OWN, 4>(l, g, nu, xi, yi, si2, r0, i0, i1, tame, ex, ey); break;
        case 2: pairs64g<MODE, T1, OWN, 2>(l, g, nu, xi, yi, si2, r0, i0, i1, tame, ex, ey); break;
        default: pairs64g<MODE, T1, OWN, 1>(l, g, nu, xi, yi, si2, r0, i0, i1, tame, ex, ey); break;
    }
}

// Returns whether a sum of this lane's targets is not finite.
template <int MODE, bool T1, int W>
__device__ __forceinline__ bool eval64_leaf(const Eval64Args &A, int t, int j, int wi, int lane,
                                            int G, Eval64Lds<MODE> *lds) {
    const int LG = kWave / G;   // lanes of a group
    constexpr bool kSized = MODE >= 1 && MODE <= 3;
    Eval64Lds<MODE> &l = lds[wi];
    const int tl = lane & (LG - 1), g = lane / LG;
    const int P = A.P, P1 = P + 1;
    const uint32_t b = (uint32_t)__builtin_amdgcn_readfirstlane((int)A.c_begin[j]);
    const uint32_t e = (uint32_t)__builtin_amdgcn_readfirstlane((int)A.c_end[j]);
    const bool own = (A.c_flags[j] & kActive) != 0;  // the leaf is in its own list 1
    const double lcx = A.c_cx[j], lcy = A.c_cy[j];
    const uint32_t a1 = A.off1[t], z1 = A.off1[t + 1], a3 = A.off3[t], z3 = A.off3[t + 1];
    // padding source: zero strength, outside the root box, of a size at which any
    // target's factor is finite (a zero size would leave 0 NaN)
    const double padx = lcx + 4.0 * A.hdr->root_len;
    const double pads2 = A.hdr->root_len * A.hdr->root_len;
    if (wi == 0)
        for (int k = lane; k < P1; k += kWave) l.b[k] = A.bk[(size_t)j * P1 + k];
    bool odd = false;
    for (uint32_t tb = b; tb < e; tb += 2 * LG) {
        const uint32_t i0 = tb + tl, i1 = i0 + LG;
        const bool valid[2] = {i0 < e, i1 < e};
        const uint32_t ic[2] = {valid[0] ? i0 : b, valid[1] ? i1 : b};
        double xi[2], yi[2], si2[2] = {0.0, 0.0}, ex[2] = {0.0, 0.0}, ey[2] = {0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            xi[k] = A.xs[ic[k]];
            yi[k] = A.ys[ic[k]];
            if (kSized) si2[k] = A.ss[ic[k]] * A.ss[ic[k]];
        }
        auto wild = [](double v) { return !(v > 1e-280 && v < 1e280); };
        const bool tame_t = !kSized || __ballot(wild(si2[0]) || wild(si2[1])) == 0;
        const bool two = tb + LG < e;  // (uniform) some lane has a second target
        // P2P from the leaf's own particles, the wavefronts taking a share each
        if ((A.mask & 1) && own) {
            const uint32_t n = e - b, per = (n + W - 1) / W;
            const uint32_t lo = min(n, wi * per), hi = min(n, lo + per);
            for (uint32_t base = lo; base < hi; base += kStage64) {
                const int fill = (int)min<uint32_t>(kStage64, hi - base);
                const int nu = (fill + G - 1) / G;
                bool odd_s = false;
                for (int r = lane; r < nu * G; r += kWave) {
                    const uint32_t src = b + base + min(r, fill - 1);
                    l.xy[r] = r < fill ? make_double2(A.xs[src], A.ys[src])
                                       : make_double2(padx, lcy);
                    l.q[r] = r < fill ? A.qs[src] : 0.0;
                    if (kSized) {
                        const double s2 = r < fill ? A.ss[src] * A.ss[src] : pads2;
                        l.s2[r] = s2;
                        odd_s |= r < fill && wild(s2);
                    }
                }
                const bool tame = tame_t && (!kSized || __ballot(odd_s) == 0);
                wave_sync();
                pairs64<MODE, T1, true>(l, G, g, nu, xi, yi, si2, b + base, ic[0],
                                           two ? ic[1] : ic[0], tame, ex, ey);
                wave_sync();
            }
        }
        // P2P from the other list-1 cells, 64 cells at a time: lane k fetches
        // cell k's range, a wave scan gives its offset in the concatenated
        // source list, of which each wavefront stages a share
        for (uint32_t c0 = a1; (A.mask & 1) && c0 < z1; c0 += kWave) {
            const int ncell = (int)min<uint32_t>(kWave, z1 - c0);
            uint32_t cnt = 0, beg = 0;
            if (lane < ncell) {
                const int sc = A.l1[c0 + lane];
                if (sc != j) {  // the own leaf was done above
                    beg = A.c_begin[sc];
                    cnt = A.c_end[sc] - beg;
                }
            }
            uint32_t inc = cnt;
            for (int o = 1; o < kWave; o <<= 1) {
                const uint32_t y = __shfl_up(inc, o, kWave);
                if (lane >= o) inc += y;
            }
            const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)inc, kWave - 1);
            l.off[lane] = inc - cnt;
            l.beg[lane] = beg;
            wave_sync();
            const uint32_t per = (n + W - 1) / W, lo = min(n, wi * per), hi = min(n, lo + per);
            for (uint32_t base = lo; base < hi; base += kStage64) {
                const int fill = (int)min<uint32_t>(kStage64, hi - base);
                const int nu = (fill + G - 1) / G;
                bool odd_s = false;
                for (int r = lane; r < nu * G; r += kWave) {
                    const uint32_t gi = base + (uint32_t)min(r, fill - 1);
                    // last cell whose offset is <= gi (empty cells share the
                    // offset of the next one and are never the last)
                    int cl = 0, ch = ncell - 1;
                    while (cl < ch) {
                        const int mid = (cl + ch + 1) >> 1;
                        if (l.off[mid] <= gi) cl = mid;
                        else ch = mid - 1;
                    }
                    const uint32_t src = l.beg[cl] + (gi - l.off[cl]);
                    l.xy[r] = r < fill ? make_double2(A.xs[src], A.ys[src])
                                       : make_double2(padx, lcy);
                    l.q[r] = r < fill ? A.qs[src] : 0.0;
                    if (kSized) {
                        const double s2 = r < fill ? A.ss[src] * A.ss[src] : pads2;
                        l.s2[r] = s2;
                        odd_s |= r < fill && wild(s2);
                    }
                }
                const bool tame = tame_t && (!kSized || __ballot(odd_s) == 0);
                wave_sync();
                pairs64<MODE, T1, false>(l, G, g, nu, xi, yi, si2, 0u, 0u, 0u, tame, ex, ey);
                wave_sync();
            }
        }
        if ((MODE == 0 && !T1) || MODE == kPot)
#pragma unroll
            for (int k = 0; k < 2; ++k) odd |= valid[k] && !isfinite(ex[k] + ey[k]);
        // M2P over list 3: this wavefront's cells a3 + wi, a3 + wi + W, ...,
        // their coefficients staged as many at a time as fit
        const int PM = T1 ? P - 1 : P;  // highest multipole order
        const int per3 = min(kWave, kStage64 / (PM + 1));
        for (uint32_t v0 = a3 + wi; (A.mask & 2) && v0 < z3; v0 += W * per3) {
            const int nc = min(per3, (int)((z3 - v0 + W - 1) / W));
            double2 *zc = reinterpret_cast<double2 *>(l.q);
            for (int r = lane; r < nc * (PM + 1); r += kWave)
                l.xy[r] = A.ak[(size_t)A.l3[v0 + W * (r / (PM + 1))] * (PM + 1) + r % (PM + 1)];
            for (int r = lane; r < nc; r += kWave) {
                const int sc = A.l3[v0 + W * r];
                zc[r] = make_double2(A.c_cx[sc], A.c_cy[sc]);
            }
            wave_sync();
            for (int c = g; c < nc; c += G) {
                const double2 z0 = zc[c];
                const double2 *a = &l.xy[c * (PM + 1)];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const cd zr = {xi[k] - z0.x, yi[k] - z0.y};
                    const cd wv = cinv(zr);
                    if (MODE == kPot) {
                        // sum_{p>=1} a_p w^p / p by Horner, then a_0 log(z - zc) minus it
                        cd f = {0.0, 0.0};
                        for (int p = PM; p >= 1; --p)
                            f = cmul(cadd(f, cscale(ld(a, p), 1.0 / p)), wv);
                        ex[k] += cmul(ld(a, 0), clog(zr)).x - f.x;
                    } else {
                        cd f = ld(a, PM);
                        for (int p = PM - 1; p >= 0; --p) f = cadd(cmul(f, wv), ld(a, p));
                        f = cmul(f, wv);
                        ex[k] += f.x;
                        ey[k] -= f.y;
                    }
                }
            }
            wave_sync();
        }
        for (int m = LG; m < kWave; m <<= 1)
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                ex[k] += shfl_xor_d(ex[k], m);
                if (MODE != kPot) ey[k] += shfl_xor_d(ey[k], m);
            }
        if (W > 1) {
            // the wavefronts' sums, added in wavefront order (two rows of 64)
            __syncthreads();
            if (g == 0) {
                l.xy[tl] = make_double2(ex[0], ey[0]);
                l.xy[kWave + tl] = make_double2(ex[1], ey[1]);
            }
            __syncthreads();
            if (wi == 0)
#pragma unroll
                for (int k = 0; k < 2; ++k)
                    for (int u = 1; u < W; ++u) {
                        const double2 o = lds[u].xy[k * kWave + tl];
                        ex[k] += o.x;
                        ey[k] += o.y;
                    }
            __syncthreads();
        } else {
            wave_sync();  // (the local coefficients)
        }
        // every group holds the sums: groups 0 and 1 finish the lanes' first
        // and second targets (the only group both in turn when G is 1)
        if (wi == 0) {
            for (int pass = 0; pass < (G == 1 ? 2 : 1); ++pass) {
                const bool second = G == 1 ? pass == 1 : g == 1;
                if (g > 1 || !(second ? valid[1] : valid[0])) continue;
                double fx = second ? ex[1] : ex[0], fy = second ? ey[1] : ey[0];
                if (A.mask & 4) {  // L2P
                    const cd z = {(second ? xi[1] : xi[0]) - lcx, (second ? yi[1] : yi[0]) - lcy};
                    cd f;
                    if (T1 || MODE == kPot) {
                        f = ld(l.b, P);
                        for (int p = P - 1; p >= 0; --p) f = cadd(cmul(f, z), ld(l.b, p));
                    } else {
                        f = cscale(ld(l.b, P), (double)P);
                        for (int p = P - 1; p >= 1; --p)
                            f = cadd(cmul(f, z), cscale(ld(l.b, p), (double)p));
                    }
                    fx += f.x;
                    fy -= f.y;
                }
                const uint32_t o = A.perm[second ? ic[1] : ic[0]];
                if (MODE == kPot) {
                    A.out_a[o] = fx;
                } else if (A.velocity) {
                    A.out_a[o] = fy + A.u_inf;
                    A.out_b[o] = -fx + A.v_inf;
                } else {
                    A.out_a[o] = fx;
                    A.out_b[o] = fy;
                }
            }
        }
    }
    return odd;
}

// The singular kernel is held to 80 registers (6 wavefronts per SIMD; 5 equal,
// 8 spills, 1 % slower); the others keep what they need.
template <int MODE, bool T1, int W>
__global__ void __launch_bounds__(kWave *kEvalWaves)
    __attribute__((amdgpu_waves_per_eu(MODE == 0 ? 6 : 4, 8))) k_eval64(Eval64Args A) {
    __shared__ Eval64Lds<MODE> lds[kEvalWaves];
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const int lane = threadIdx.x & (kWave - 1);
    const int t = W == 1 ? (int)blockIdx.x * kEvalWaves + w : (int)blockIdx.x;
    if (t >= A.nl) return;  // (W > 1: uniform over the workgroup)
    const int j = __builtin_amdgcn_readfirstlane((int)A.leaf_idx[t]);
    const int nt = (int)(A.c_end[j] - A.c_begin[j]);
    Eval64Lds<MODE> *l = W == 1 ? lds + w : lds;
    const int wi = W == 1 ? 0 : w;
    const int G = nt <= 8 ? 16 : nt <= 16 ? 8 : nt <= 32 ? 4 : nt <= 64 ? 2 : 1;
    const bool odd = eval64_leaf<MODE, T1, W>(A, t, j, wi, lane, G, l);
    if ((MODE == 0 && !T1) || MODE == kPot)
        // a pair at r = 0 leaves a sum that is not finite; so does a strength
        // that is not, so the positions decide
        if (__ballot(odd)) {
            bool dup = false;
            const uint32_t b = A.c_begin[j], e = A.c_end[j];
            for (uint32_t i = b + lane; i < e; i += kWave)
                for (uint32_t u = A.off1[t]; u < A.off1[t + 1]; ++u) {
                    const int c = A.l1[u];
                    for (uint32_t r = A.c_begin[c]; r < A.c_end[c]; ++r) {
                        const double dx = A.xs[i] - A.xs[r], dy = A.ys[i] - A.ys[r];
                        dup |= r != i && dx * dx + dy * dy == 0.0;
                    }
                }
            if (dup) atomicOr(A.flags, kFlagDuplicate);
        }
}

// Leaves up to which a leaf is shared by four wavefronts: the chip holds 6,144
// wavefronts at 6 per SIMD, and below about that many leaves the longest
// leaf's chain is what the launch waits for (about 5,000 leaves of 100k
// clusters, Gaussian kernel: 426 us a solve with one wavefront per leaf, 397
// with four; about 13,000 of a 200k plate: 531 and 570).
constexpr int kSplitLeaves = 8192;

template <int MODE, bool T1>
void eval64_launch(const Eval64Args &A, hipStream_t s) {
    if (A.nl <= kSplitLeaves)
        k_eval64<MODE, T1, 4><<<A.nl, kWave * kEvalWaves, 0, s>>>(A);
    else
        k_eval64<MODE, T1, 1><<<div_up(A.nl, kEvalWaves), kWave * kEvalWaves, 0, s>>>(A);
}

// Type-1 M2L and P2L (biotsavart_fmm_2d.cpp:199-271) for every cell of level
// >= 1, thread per (cell, order l = 0..ND), with multipoles a_0..a_{ND-1}
// (stride ND) of strengths q = -g / (2 pi):
//   b_l = sum_{list 2} w^(l+1) sum_j tab[l][j] a_j w^j,   w = 1 / (zs - zt),
//         tab[l][j] = (-1)^(j+1) C(l + j, j)              (Horner in w)
//       - sum_{list 4} sum_i q_i w_i^(l+1),               w_i = 1 / (z_i - zt)
// (the reference's list 4 is always P2L from the leaf's particles).  Cells of
// level 1 have no lists (their locals are zero, as in the reference).
// m2l_t1_sum: order l from one source's multipoles a, d = zs - zt.
__device__ __forceinline__ cd m2l_t1_sum(int l, int ND, const double *row, const double2 *a,
                                         cd d) {
    const cd w = cinv(d);
    cd sm = cscale(ld(a, ND - 1), row[ND - 1]);
    for (int k = ND - 2; k >= 0; --k) sm = cadd(cmul(sm, w), cscale(ld(a, k), row[k]));
    return cmul(sm, cpowi(w, l + 1));
}

__global__ void __launch_bounds__(256)
    k_m2l_t1(int j0, int nc, int ND, const double *tab, const uint8_t *c_level, const int *l2,
             const uint8_t *n2, const int *l4, const uint8_t *n4, const double *c_cx,
             const double *c_cy, const uint32_t *c_begin, const uint32_t *c_end, const double *xs,
             const double *ys, const double *qs, const double2 *ak, double2 *bk) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int NL = ND + 1;
    if (idx >= (long long)(nc - j0) * NL) return;
    const int j = j0 + (int)(idx / NL), l = (int)(idx % NL);
    cd acc = {0.0, 0.0};
    if (c_level[j] >= 2) {
        const double cx = c_cx[j], cy = c_cy[j];
        const double *row = tab + (size_t)l * ND;
        const int m2 = n2[j], m4 = n4[j];
        for (int u = 0; u < m2; ++u) {
            const int sidx = l2[27 * j + u];
            acc = cadd(acc, m2l_t1_sum(l, ND, row, ak + (size_t)sidx * ND,
                                       cd{c_cx[sidx] - cx, c_cy[sidx] - cy}));
        }
        for (int u = 0; u < m4; ++u) {
            const int sidx = l4[8 * j + u];
            for (uint32_t i = c_begin[sidx]; i < c_end[sidx]; ++i) {
                const cd w = cinv(cd{xs[i] - cx, ys[i] - cy});
                acc = csub(acc, cscale(cpowi(w, l + 1), qs[i]));
            }
        }
    }
    st(bk, (size_t)j * NL + l, acc);
}

// Type-1 P2L from list 4 (k_m2l_t1's second sum) added to the list-2 sum of the
// matrix cores, and with it the list-2 sources beside their target (t1_beside),
// which are not among the 40 offsets of k_m2l64_mfma: the list build flags a
// tree that has any (their pairs are a whole row of boxes; without them the
// velocity there is of no use).  One wavefront per target cell, skipped by a
// cell without either; lane l forms order l % NL over the particles and sources
// of its group, the groups added in order.
constexpr int kP2lT1Waves = 4;

__global__ void __launch_bounds__(kWave *kP2lT1Waves)
    k_p2l_t1(int j0, int nc, int ND, const DevHdr *hdr, const double *tab, const uint8_t *c_level,
             const int *l2, const uint8_t *n2, const int *l4, const uint8_t *n4,
             const double *c_cx, const double *c_cy, const uint32_t *c_begin,
             const uint32_t *c_end, const double *xs, const double *ys, const double *qs,
             const double2 *ak, double2 *bk) {
    __shared__ double2 red[kP2lT1Waves][kWave];
    const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    const int j = j0 + blockIdx.x * kP2lT1Waves + w;
    if (j >= nc) return;
    const int m4 = n4[j];
    const double cx = c_cx[j], cy = c_cy[j];
    int s2 = -1;
    uint64_t beside = 0;
    if (hdr->flags & kFlagT1Beside) {
        if (lane < (int)n2[j]) s2 = l2[27 * (size_t)j + lane];
        const double side = ldexp(hdr->root_len, -(int)c_level[j]);
        beside = __ballot(s2 >= 0 && t1_beside(c_cx[max(s2, 0)] - cx, c_cy[max(s2, 0)] - cy, side));
    }
    if (m4 == 0 && beside == 0) return;  // uniform over the wavefront
    const int NL = ND + 1, G = kWave / NL, g = lane / NL, l = lane % NL;
    cd acc = {0.0, 0.0};
    for (int q = 0; beside; beside &= beside - 1, ++q) {
        const int sc = __shfl(s2, __ffsll((unsigned long long)beside) - 1, kWave);
        if (q % G == g)
            acc = cadd(acc, m2l_t1_sum(l, ND, tab + (size_t)l * ND, ak + (size_t)sc * ND,
                                       cd{c_cx[sc] - cx, c_cy[sc] - cy}));
    }
    if (g < G)
        for (int u = 0; u < m4; ++u) {
            const int sc = l4[8 * j + u];
            for (uint32_t i = c_begin[sc] + g; i < c_end[sc]; i += G) {
                const cd wv = cinv(cd{xs[i] - cx, ys[i] - cy});
                acc = csub(acc, cscale(cpowi(wv, l + 1), qs[i]));
            }
        }
    st(red[w], lane, acc);
    wave_sync();
    if (lane < NL) {
        cd sum = ld(bk, (size_t)j * NL + lane);
        for (int gg = 0; gg < G; ++gg) sum = cadd(sum, ld(red[w], gg * NL + lane));
        st(bk, (size_t)j * NL + lane, sum);
    }
}

// Type-1 L2L for the cells of one level (>= 3; level-1 locals are zero), thread
// per (cell, l): orders ND above 16.
__global__ void __launch_bounds__(256)
    k_l2l_t1(int j0, int j1, int ND, const double *coef, const int *expo, const int *c_parent,
             const double *c_cx, const double *c_cy, double2 *bk) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int NL = ND + 1;
    if (idx >= (long long)(j1 - j0) * NL) return;
    const int j = j0 + (int)(idx / NL), l = (int)(idx % NL);
    const int par = c_parent[j];
    const cd d = {c_cx[j] - c_cx[par], c_cy[j] - c_cy[par]};
    const size_t o = (size_t)j * NL + l;
    st(bk, o, cadd(ld(bk, o), l2l_t1_sum(l, ND, coef, expo, d, bk + (size_t)par * NL)));
}

// FP64 direct sum with LDS source tiles (accuracy reference only).
__global__ void __launch_bounds__(256)
    k_direct64(int n, const double *x, const double *y, const double *q, const uint8_t *mask,
               int nt, const int *tidx, double *ex, double *ey) {
    __shared__ double sx[256], sy[256], sq[256];
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    int i = t < nt ? (tidx ? tidx[t] : t) : -1;
    if (i >= n) i = -1;
    const bool valid = i >= 0;
    const double xi = valid ? x[i] : 0.0, yi = valid ? y[i] : 0.0;
    double ax = 0.0, ay = 0.0;
    for (int base = 0; base < n; base += 256) {
        const int jj = base + threadIdx.x;
        if (jj < n) {
            sx[threadIdx.x] = x[jj];
            sy[threadIdx.x] = y[jj];
            sq[threadIdx.x] = (mask && !mask[jj]) ? 0.0 : q[jj];
        }
        __syncthreads();
        const int m = min(256, n - base);
        for (int k = 0; k < m; ++k) {
            const int src = base + k;
            if (src == i) continue;
            const double dx = xi - sx[k], dy = yi - sy[k];
            const double qr = sq[k] / (dx * dx + dy * dy);
            ax += qr * dx;
            ay += qr * dy;
        }
        __syncthreads();
    }
    if (t < nt) {  // an out-of-range target index yields NaN
        ex[t] = valid ? ax : __builtin_nan("");
        ey[t] = valid ? ay : __builtin_nan("");
    }
}

}  // namespace

static Eval64Args eval64_args(const Ctx &c, int P, bool velocity, double u_inf, double v_inf,
                              int mask, double *out_a, double *out_b) {
    Eval64Args A{};
    A.leaf_idx = (const uint32_t *)c.leaf_idx.p;
    A.nl = c.info.n_leaves;
    A.P = P;
    A.c_flags = (const uint8_t *)c.c_flags.p;
    A.c_begin = (const uint32_t *)c.c_begin.p;
    A.c_end = (const uint32_t *)c.c_end.p;
    A.c_cx = (const double *)c.c_cx.p;
    A.c_cy = (const double *)c.c_cy.p;
    A.off1 = (const uint32_t *)c.off1.p;
    A.l1 = (const int *)c.l1.p;
    A.off3 = (const uint32_t *)c.off3.p;
    A.l3 = (const int *)c.l3.p;
    A.xs = (const double *)c.xs.p;
    A.ys = (const double *)c.ys.p;
    A.qs = (const double *)c.qs.p;
    A.ss = (const double *)c.ss.p;
    A.perm = c.perm_sorted;
    A.ak = (const double2 *)c.ak.p;
    A.bk = (const double2 *)c.bk.p;
    A.velocity = velocity ? 1 : 0;
    A.mask = mask;
    A.u_inf = u_inf;
    A.v_inf = v_inf;
    A.out_a = out_a;
    A.out_b = out_b;
    A.hdr = c.hdr_d;
    A.flags = &c.hdr_d->flags;
    return A;
}

// List-2 M2L of every cell of level >= 2 on the matrix cores, order P <= 16.
template <bool T1>
static void m2l64_run(const Ctx &c, int P, const double *R, const double2 *ak, double2 *bk,
                      hipStream_t s) {
    const TreeInfo &ti = c.info;
    M2lLevels lv{};
    lv.maxL = ti.max_level;
    int blocks = 0;
    for (int L = 2; L <= ti.max_level; ++L) {
        lv.first[L] = blocks;
        lv.cell0[L] = (int)ti.lev_off[L];
        blocks += div_up((long long)(ti.lev_off[L + 1] - ti.lev_off[L]), kM2lCells);
    }
    if (blocks == 0) return;
    lv.first[ti.max_level + 1] = blocks;
    lv.cell0[ti.max_level + 1] = (int)ti.lev_off[ti.max_level + 1];
    const uint32_t *c_key = (const uint32_t *)c.c_key.p;
    const int *l2 = (const int *)c.l2.p;
    const uint8_t *n2 = (const uint8_t *)c.n2.p;
    const double2 *cres = (const double2 *)c.c_res.p;  // (type 1)
    // One class per workgroup while four times the workgroups still fit the
    // chip's 256 CUs at once (k_m2l64_mfma's comment has both sides).  From there
    // to 255 workgroups some CUs have none: 177 of 256 at 780k.
    constexpr int split = 64;
    switch (P) {
#define M2L64_CASE(PP)                                                                          \
    case PP:                                                                                    \
        if (blocks <= split)                                                                    \
            k_m2l64_mfma<PP, T1, 1><<<4 * blocks, kM2lBlock, 0, s>>>(c.hdr_d, lv, c_key, l2,    \
                                                                    n2, R, cres, ak, bk);   \
        else                                                                                    \
            k_m2l64_mfma<PP, T1, 4><<<blocks, kM2lBlock, 0, s>>>(c.hdr_d, lv, c_key, l2, n2, R, \
                                                                 cres, ak, bk);             \
        break;
        M2L64_CASE(1) M2L64_CASE(2) M2L64_CASE(3) M2L64_CASE(4) M2L64_CASE(5) M2L64_CASE(6)
        M2L64_CASE(7) M2L64_CASE(8) M2L64_CASE(9) M2L64_CASE(10) M2L64_CASE(11)
        M2L64_CASE(12) M2L64_CASE(13) M2L64_CASE(14) M2L64_CASE(15) M2L64_CASE(16)
#undef M2L64_CASE
        default: break;
    }
}

// M2M from the leaves' multipoles up to level 1.
static void m2m64_run(const TreeInfo &ti, int P, const double *tab, const uint8_t *c_flags,
                      const double *c_cx, const double *c_cy, const int *c_child, double2 *ak,
                      hipStream_t s) {
    if (P < kTrP1) {
        for (int S = ti.max_level; S > 1; S -= kSpan) {
            const int L0 = std::max(1, S - kSpan);
            k_m2m64_span<<<(int)(ti.lev_off[L0 + 1] - ti.lev_off[L0]), kSpanBlock, 0, s>>>(
                (int)ti.lev_off[L0], S - L0, P, tab, c_cx, c_cy, c_child, ak);
        }
        return;
    }
    for (int L = ti.max_level - 1; L >= 1; --L) {
        const int j0 = (int)ti.lev_off[L], j1 = (int)ti.lev_off[L + 1];
        k_m2m64<<<div_up((long long)(j1 - j0) * (P + 1), 256), 256, 0, s>>>(
            j0, j1, P, tab, c_flags, c_cx, c_cy, c_child, ak);
    }
}

void fmm64_run(Ctx &c, int P, int list4_mode, int stage_mask, double *out_a, double *out_b,
               bool velocity, double u_inf, double v_inf, const FmmMarks &mk, bool potential) {
    hipStream_t s = c.stream;
    const TreeInfo &ti = c.info;
    const int nc = ti.n_cells, nl = ti.n_leaves, P1 = P + 1;
    double2 *ak = c.ak.as<double2>((size_t)nc * P1), *bk = c.bk.as<double2>((size_t)nc * P1);
    // every row a later stage reads is written by the stage that forms it, the
    // exceptions by P2M; above order 16 order 0 of the local rows is not
    if (P >= kTrP1) VPM_HIP(hipMemsetAsync(bk, 0, sizeof(double2) * (size_t)nc * P1, s));
    const uint8_t *c_flags = (const uint8_t *)c.c_flags.p;
    const uint32_t *c_begin = (const uint32_t *)c.c_begin.p, *c_end = (const uint32_t *)c.c_end.p;
    const double *c_cx = (const double *)c.c_cx.p, *c_cy = (const double *)c.c_cy.p;
    const int *c_child = (const int *)c.c_child.p, *c_parent = (const int *)c.c_parent.p;
    const double *xs = (const double *)c.xs.p, *ys = (const double *)c.ys.p,
                 *qs = (const double *)c.qs.p;
    const uint8_t *as = (const uint8_t *)c.acts.p;
    const uint32_t *leaf_idx = (const uint32_t *)c.leaf_idx.p;
    const double *t_m2l = (const double *)c.tab_m2l.p, *t_m2m = (const double *)c.tab_m2m.p,
                 *t_l2l = (const double *)c.tab_l2l.p;

    k_p2m64<<<div_up(nl, kP2m64Waves * kP2mLeaves), kWave * kP2m64Waves, 0, s>>>(
        leaf_idx, nl, P, c_flags, c_begin, c_end, c_cx, c_cy, xs, ys, qs, as, ak, bk,
        (int)ti.lev_off[2], P1);
    m2m64_run(ti, P, t_m2m, c_flags, c_cx, c_cy, c_child, ak, s);
    mk.mark(3, s);
    // M2L: every cell of level >= 2
    const int j2 = (int)ti.lev_off[2];
    const int NP = potential ? P1 : P;  // orders formed per cell
    if (nc > j2 && P < kTrP1) {
        const int *l2 = (const int *)c.l2.p, *l4 = (const int *)c.l4.p;
        const uint8_t *n2 = (const uint8_t *)c.n2.p, *n4 = (const uint8_t *)c.n4.p;
        if (!potential) {
            // list 2 on the matrix cores, then list 4 added by the wavefront kernel
            if (c.tab_r64_p != P) throw Error(kInternal, "M2L matrices of another order");
            m2l64_run<false>(c, P, (const double *)c.tab_r64.p, ak, bk, s);
        }
        (potential ? k_m2l64w<true> : k_m2l64w<false>)<<<div_up(nc - j2, kM2lwWaves),
                                                         kWave * kM2lwWaves, 0, s>>>(
            j2, nc, P, list4_mode, t_m2l, l2, n2, l4, n4, c_cx, c_cy, c_begin, c_end, xs, ys, qs,
            as, ak, bk);
    }
    if (nc > j2 && P >= kTrP1)
        (potential ? k_m2l64<true> : k_m2l64<false>)<<<
            div_up((long long)(nc - j2) * NP, 256), 256, 0, s>>>(
            j2, nc, P, list4_mode, t_m2l, (const int *)c.l2.p, (const uint8_t *)c.n2.p,
            (const int *)c.l4.p, (const uint8_t *)c.n4.p, c_cx, c_cy, c_begin, c_end, xs, ys, qs,
            as, ak, bk);
    mk.mark(4, s);
    // L2L: children at levels 3 .. maxL (parents 2 .. maxL-1, fmm2D.cpp:587)
    if (P < kTrP1) {
        for (int L = 2; L < ti.max_level; L += kSpan)
            (potential ? k_l2l64_span<kL2lPot> : k_l2l64_span<kL2lField>)<<<
                (int)(ti.lev_off[L + 1] - ti.lev_off[L]), kSpanBlock, 0, s>>>(
                (int)ti.lev_off[L], std::min(kSpan, ti.max_level - L), P, t_l2l, nullptr, c_child,
                c_cx, c_cy, bk);
    } else {
        for (int L = 3; L <= ti.max_level; ++L) {
            const int j0 = (int)ti.lev_off[L], j1 = (int)ti.lev_off[L + 1];
            (potential ? k_l2l64<true> : k_l2l64<false>)<<<div_up((long long)(j1 - j0) * NP, 256),
                                                            256, 0, s>>>(j0, j1, P, t_l2l, c_parent,
                                                                         c_cx, c_cy, bk);
        }
    }
    mk.mark(5, s);
    const Eval64Args ea = eval64_args(c, P, velocity, u_inf, v_inf, stage_mask, out_a, out_b);
    switch (potential ? kPot : c.icut) {
        case 1: eval64_launch<1, false>(ea, s); break;
        case 2: eval64_launch<2, false>(ea, s); break;
        case 3: eval64_launch<3, false>(ea, s); break;
        case kPot: eval64_launch<kPot, false>(ea, s); break;
        default: eval64_launch<0, false>(ea, s); break;
    }
    mk.mark(6, s);
    VPM_LAUNCH_CHECK();
}

// Whether the list-2 M2L of a type-1 tree may use the grid's offsets: up to order
// 16, and while eps, the stored centres' distance from the grid in cell sides, is
// small enough (each of max_level + 1 roundings adds up to 2^-53 of the largest
// coordinate).  The first-order correction (k_m2l64_mfma) leaves eps times the
// truncation error, which falls by about 2.5 per order: a velocity difference from
// the stored-centre form of 2e-13 at order 2 and eps 1e-11, 2e-14 at order 4,
// rounding alone from order 8 on.  The limits keep it at 1e-14 of the velocity;
// near the origin order 10 then takes trees of up to 12 or 13 levels.  (A box of side
// 1e-30 has no list 2 under the box tests' tolerance, and k_m2l_t1 forms no power.)
static bool t1_on_grid(const TreeInfo &ti, int ND) {
    if (ND >= kTrP1) return false;
    double far = 0.0;
    for (int d = 0; d < 2; ++d)
        far = std::max({far, std::fabs(ti.pivot[d]), std::fabs(ti.pivot[d] + ti.root_len)});
    const double side = std::ldexp(ti.root_len, -ti.max_level);
    // the scaled coefficients' powers of a side of any level stay inside the range
    const double range = 290.0 / (ND + 1);
    if (!(std::fabs(std::log10(side)) < range && std::fabs(std::log10(ti.root_len)) < range))
        return false;
    const double limit = std::min(1e-11, 1e-14 * std::pow(2.5, ND));
    return (ti.max_level + 1) * 0x1p-53 * far <= limit * side;
}

void fmm_t1_run(Ctx &c, int ND, double *u, double *v, double u_inf, double v_inf,
                const FmmMarks &mk) {
    hipStream_t s = c.stream;
    const TreeInfo &ti = c.info;
    const int nc = ti.n_cells, nl = ti.n_leaves, NL = ND + 1, PM = ND - 1;
    double2 *ak = c.ak.as<double2>((size_t)nc * ND), *bk = c.bk.as<double2>((size_t)nc * NL);
    const uint8_t *c_flags = (const uint8_t *)c.c_flags.p, *c_level = (const uint8_t *)c.c_level.p;
    const uint32_t *c_begin = (const uint32_t *)c.c_begin.p, *c_end = (const uint32_t *)c.c_end.p;
    const double *c_cx = (const double *)c.c_cx.p, *c_cy = (const double *)c.c_cy.p;
    const int *c_child = (const int *)c.c_child.p, *c_parent = (const int *)c.c_parent.p;
    const double *xs = (const double *)c.xs.p, *ys = (const double *)c.ys.p,
                 *qs = (const double *)c.qs.p;
    const uint8_t *as = (const uint8_t *)c.acts.p;
    const uint32_t *leaf_idx = (const uint32_t *)c.leaf_idx.p;

    // upward: P2M and M2M at order PM = ND - 1 (biotsavart_fmm_2d.cpp:123-188;
    // the exact shift C(p, k), the reference's bico values to rounding)
    k_p2m64<<<div_up(nl, kP2m64Waves * kP2mLeaves), kWave * kP2m64Waves, 0, s>>>(
        leaf_idx, nl, PM, c_flags, c_begin, c_end, c_cx, c_cy, xs, ys, qs, as, ak, bk,
        (int)ti.lev_off[2], NL);
    m2m64_run(ti, PM, (const double *)c.t1_m2m.p, c_flags, c_cx, c_cy, c_child, ak, s);
    mk.mark(3, s);
    // M2L and P2L: every cell of level >= 1 (all of bk written); on the grid
    // list 2 on the matrix cores, then P2L added, and level 1 cleared by P2M
    const int j1 = (int)ti.lev_off[1], j2 = (int)ti.lev_off[2];
    const double *t_m2l = (const double *)c.t1_m2l.p;
    const int *l2 = (const int *)c.l2.p, *l4 = (const int *)c.l4.p;
    const uint8_t *n2 = (const uint8_t *)c.n2.p, *n4 = (const uint8_t *)c.n4.p;
    if (t1_on_grid(ti, ND)) {
        m2l64_run<true>(c, ND, (const double *)c.t1_r64.p, ak, bk, s);
        if (nc > j2)
            k_p2l_t1<<<div_up(nc - j2, kP2lT1Waves), kWave * kP2lT1Waves, 0, s>>>(
                j2, nc, ND, c.hdr_d, t_m2l, c_level, l2, n2, l4, n4, c_cx, c_cy, c_begin, c_end,
                xs, ys, qs, ak, bk);
    } else if (nc > j1) {
        k_m2l_t1<<<div_up((long long)(nc - j1) * NL, 256), 256, 0, s>>>(
            j1, nc, ND, t_m2l, c_level, l2, n2, l4, n4, c_cx, c_cy, c_begin, c_end, xs, ys, qs, ak,
            bk);
    }
    mk.mark(4, s);
    const double *coef = (const double *)c.t1_l2l_c.p;
    const int *expo = (const int *)c.t1_l2l_e.p;
    if (ND < kTrP1) {
        for (int L = 2; L < ti.max_level; L += kSpan)
            k_l2l64_span<kL2lT1><<<(int)(ti.lev_off[L + 1] - ti.lev_off[L]), kSpanBlock, 0, s>>>(
                (int)ti.lev_off[L], std::min(kSpan, ti.max_level - L), ND, coef, expo, c_child,
                c_cx, c_cy, bk);
    } else {
        for (int L = 3; L <= ti.max_level; ++L) {
            const int j0 = (int)ti.lev_off[L], jz = (int)ti.lev_off[L + 1];
            k_l2l_t1<<<div_up((long long)(jz - j0) * NL, 256), 256, 0, s>>>(j0, jz, ND, coef, expo,
                                                                          c_parent, c_cx, c_cy, bk);
        }
    }
    mk.mark(5, s);
    const Eval64Args ea = eval64_args(c, ND, true, u_inf, v_inf, 7, u, v);
    switch (c.icut) {
        case 1: eval64_launch<1, true>(ea, s); break;
        case 2: eval64_launch<2, true>(ea, s); break;
        case 3: eval64_launch<3, true>(ea, s); break;
        default: eval64_launch<0, true>(ea, s); break;
    }
    mk.mark(6, s);
    VPM_LAUNCH_CHECK();
}

// Partial sums of |(a, b) - (ja, jb)|^2 and |(ja - a0, jb - b0)|^2 per block.
__global__ void __launch_bounds__(256)
    k_diff_norms(int n, const double *a, const double *b, const double *ja, const double *jb,
                 double a0, double b0, double *part) {
    double num = 0.0, den = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const double da = a[i] - ja[i], db = b[i] - jb[i];
        const double ra = ja[i] - a0, rb = jb[i] - b0;
        num += da * da + db * db;
        den += ra * ra + rb * rb;
    }
    for (int m = 1; m < kWave; m <<= 1) {
        num += __shfl_xor(num, m, kWave);
        den += __shfl_xor(den, m, kWave);
    }
    __shared__ double sn[4], sd[4];
    const int w = threadIdx.x / kWave;
    if ((threadIdx.x & (kWave - 1)) == 0) {
        sn[w] = num;
        sd[w] = den;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = sn[0] + sn[1] + sn[2] + sn[3];
        part[2 * blockIdx.x + 1] = sd[0] + sd[1] + sd[2] + sd[3];
    }
}

// Relative L2 difference of (a, b) against the judge (ja, jb), whose
// reference level (a0, b0) is removed from the norm (the free stream of a
// velocity): sqrt(sum |d|^2 / sum |j - (a0, b0)|^2).  Synchronises the stream.
double rel_diff64(int n, const double *a, const double *b, const double *ja, const double *jb,
                  double a0, double b0, double *part_dev, hipStream_t s) {
    constexpr int kBlocks = 512;
    k_diff_norms<<<kBlocks, 256, 0, s>>>(n, a, b, ja, jb, a0, b0, part_dev);
    VPM_LAUNCH_CHECK();
    std::vector<double> h(2 * kBlocks);
    VPM_HIP(hipMemcpyAsync(h.data(), part_dev, h.size() * sizeof(double), hipMemcpyDeviceToHost,
                           s));
    VPM_HIP(hipStreamSynchronize(s));
    double num = 0.0, den = 0.0;
    for (int k = 0; k < kBlocks; ++k) {
        num += h[2 * k];
        den += h[2 * k + 1];
    }
    return den > 0.0 ? std::sqrt(num / den) : (num > 0.0 ? INFINITY : 0.0);
}

__global__ void __launch_bounds__(256)
    k_fill_pair(double *a, double *b, int n, double va, double vb) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        a[i] = va;
        b[i] = vb;
    }
}

void fill_pair(double *a, double *b, int n, double va, double vb, hipStream_t s) {
    k_fill_pair<<<div_up(n, 256), 256, 0, s>>>(a, b, n, va, vb);
    VPM_LAUNCH_CHECK();
}

void direct64(int n, const double *x, const double *y, const double *q, const uint8_t *src_mask,
              int nt, const int *tidx, double *ex, double *ey, hipStream_t s) {
    k_direct64<<<div_up(nt, 256), 256, 0, s>>>(n, x, y, q, src_mask, nt, tidx, ex, ey);
    VPM_LAUNCH_CHECK();
}

// An entry of the list-2 M2L matrices a thread (R in k_m2l64_mfma's order: 40
// offsets, KS steps, NS tiles, lane): tab[p][k] delta^-(p+k) as a 2 x 2 real
// block.  (On the host the matrices and their upload cost 0.1 ms of a handle's
// first solve.)
__global__ void __launch_bounds__(256)
    k_mfma_table(bool T1, int TS, int RW, int K, int KS, int T16, int NS, const double *tab,
                 double *R) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= 40 * KS * NS * kWave) return;
    const int lane = e % kWave, t = e / kWave % NS, ks = e / (kWave * NS) % KS;
    // the offsets in order, dy major: 14 of dy < -1, 4 each (dx = -3, -2, 2, 3) of
    // dy = -1, 0, 1, 14 of dy > 1
    const int o = e / (kWave * NS * KS), i = o - 14;
    const bool mid = i >= 0 && i < 12;
    const int dy = mid ? i / 4 - 1 : o < 14 ? o / 7 - 3 : (o - 26) / 7 + 2;
    const int dx = mid ? (i % 4 < 2 ? i % 4 - 3 : i % 4) : o < 14 ? o % 7 - 3 : (o - 26) % 7 - 3;
    const int col = 8 * (ks / 2) + 2 * (lane / 16) + (ks & 1);
    const int row = t < T16 ? 16 * t + lane % 16 : 16 * T16 + 4 * (t - T16) + lane % 4;
    double v = 0.0;
    if (row < RW && col < K) {
        const int l = row / 2, k = col / 2;
        // output order l + 1 (type 1: order l, whose power is l + 1 too)
        const double c = tab[(size_t)(T1 ? l : l + 1) * TS + k];
        const double r2 = (double)(dx * dx + dy * dy);
        const cd w = {dx / r2, -dy / r2};  // 1 / delta
        cd pw = w;
        for (int i = 1; i < l + 1 + k; ++i) pw = cmul(pw, w);
        // ((Re, -Im), (Im, Re))
        v = (row & 1) == (col & 1) ? c * pw.x : (row & 1) ? c * pw.y : -(c * pw.y);
    }
    R[e] = v;
}

template <int P, bool T1>
static void mfma_table(const double *tab, DBuf &buf, hipStream_t s) {
    using Sh = M2lShape<P, T1>;
    constexpr int total = 40 * Sh::KS * Sh::NS * kWave;
    double *R = (double *)buf.get(total * sizeof(double));
    k_mfma_table<<<div_up(total, 256), 256, 0, s>>>(T1, T1 ? P : P + 1, Sh::RW, Sh::K, Sh::KS,
                                                    Sh::T16, Sh::NS, tab, R);
    VPM_LAUNCH_CHECK();
}

void fmm64_mfma_table(int P, bool type1, const double *tab, DBuf &R, hipStream_t s) {
    switch (P) {
#define M2L64_CASE(PP)                                                                      \
    case PP:                                                                                \
        type1 ? mfma_table<PP, true>(tab, R, s) : mfma_table<PP, false>(tab, R, s);         \
        break;
        M2L64_CASE(1) M2L64_CASE(2) M2L64_CASE(3) M2L64_CASE(4) M2L64_CASE(5) M2L64_CASE(6)
        M2L64_CASE(7) M2L64_CASE(8) M2L64_CASE(9) M2L64_CASE(10) M2L64_CASE(11)
        M2L64_CASE(12) M2L64_CASE(13) M2L64_CASE(14) M2L64_CASE(15) M2L64_CASE(16)
#undef M2L64_CASE
        default: break;
    }
}

}  // namespace vpm
