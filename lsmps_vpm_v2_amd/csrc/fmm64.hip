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
// global memory.  Thread mappings: one thread per (cell, order) for the
// translations (Horner in the translation distance, no per-thread arrays),
// one wavefront per leaf for the evaluation.
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
// (a = 0..3) of its particle, z from the leaf's centre, zero strength for
// inactive particles and leaves; lane r then adds its own order p = 4a + b as
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
            const bool src = in && ai != 0;
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
// P2L b_0 += q log(z_t - z_i) (:540).  With PT > 0 (orders P <= PT) a
// source's coefficients are loaded into registers at once before the Horner
// sweep, rather than one dependent load per step.
template <bool POT, int PT>
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
        cd s;
        if constexpr (PT > 0) {
            cd a[PT + 1];
#pragma unroll
            for (int k = 0; k <= PT; ++k) a[k] = k <= P ? ld(ak, b + k) : cd{0.0, 0.0};
            s = cscale(a[PT], PT <= P ? row[PT] : 0.0);
#pragma unroll
            for (int k = PT - 1; k >= 0; --k)
                if (k <= P) s = cadd(cmul(s, w), cscale(a[k], row[k]));
        } else {
            s = cscale(ld(ak, b + P), row[P]);
            for (int k = P - 1; k >= 0; --k) s = cadd(cmul(s, w), cscale(ld(ak, b + k), row[k]));
        }
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
// w = 1/(zs - zt) in LDS once (the list-2 entries, then the list-4 ones
// with list4_mode 1); lane l = g NP + i (NP = P orders, P + 1 for the
// potential) forms order p = i (+1 without the potential) over the sources
// u = g, g + G, ... (G = 64 / NP groups), and the groups' partial sums are
// added in group order.  Every lane works, and a source's coefficients are
// read from HBM / L2 once per target instead of once per (target, order).
// P2L (list4_mode 2) splits the list-4 particles over the groups the same way.
// With L4ONLY the wave takes list 4 alone (M2L or P2L by list4_mode), skips a
// cell without one and adds its sum to b_p, which the matrix-core list-2
// kernel has written.
constexpr int kM2lwWaves = 4;
constexpr int kM2lwSrc = 27 + 8;  // list 2 <= 27, list 4 <= 8
constexpr int kM2lwP1 = 17;       // orders up to 16

template <bool POT, bool L4ONLY>
__global__ void __launch_bounds__(kWave *kM2lwWaves)
    k_m2l64w(int j0, int nc, int P, int list4_mode, const double *tab, const int *l2,
             const uint8_t *n2, const int *l4, const uint8_t *n4, const double *c_cx,
             const double *c_cy, const uint32_t *c_begin, const uint32_t *c_end,
             const double *xs, const double *ys, const double *qs, const uint8_t *as,
             const double2 *ak, double2 *bk) {
    // sources staged per wavefront: lists 2 and 4, or list 4 alone (a
    // smaller LDS footprint, so more wavefronts reside)
    constexpr int NS = L4ONLY ? 8 : kM2lwSrc;
    __shared__ double2 sak[kM2lwWaves][NS * kM2lwP1];
    __shared__ double2 sw[kM2lwWaves][NS], slg[kM2lwWaves][NS];
    __shared__ double2 red[kM2lwWaves][kWave];
    const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    const int j = j0 + blockIdx.x * kM2lwWaves + w;
    if (j >= nc) return;  // uniform over the wavefront
    const int P1 = P + 1, NP = POT ? P1 : P, G = kWave / NP;
    const int g = lane / NP, i = lane % NP, p = (POT ? 0 : 1) + i;
    const double cx = c_cx[j], cy = c_cy[j];
    const int m2 = L4ONLY ? 0 : n2[j], m4 = n4[j];
    if (L4ONLY && m4 == 0) return;  // uniform over the wavefront
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
        st(bk, o, L4ONLY ? cadd(ld(bk, o), sum) : sum);
    }
}

// List-2 M2L of the FP64 path on the matrix cores (orders P <= 16, field and
// velocity; the potential keeps k_m2l64w).  A workgroup takes a tile of 16
// consecutive cells of one level; the tiles of levels 2.. follow each other
// in the grid.  With len the level's cell side and delta = (zs - zt) / len
// (|dx|, |dy| <= 3, not both <= 1: 40 offsets), the list-2 sum
//   b_p = sum_k tab[p][k] a_k (zs - zt)^-(p+k)
// is, in the scaled coefficients a^_k = a_k len^-k and b^_p = b_p len^p,
//   b^ = sum over offsets of M_delta a^,  M_delta[p][k] = tab[p][k] delta^-(p+k),
// a realified 2P x 2(P+1) matrix per offset (fmm64_mfma_table), the A operand
// of v_mfma_f64_16x16x4f64; the B operand is a source cell's a^ along
// K = 2(P+1).  Lane l: target column n = l % 16, k-quarter kq = l / 16;
// wavefront w takes the offsets w, w + kM2l64Waves, ... that a target of the
// tile uses, and the wavefronts' accumulators are summed through LDS.  The
// output rows follow the f64 instruction's layout D[4v + l / 16][l % 16].
// The offset is exact here, where the reference forms zs - zt from rounded
// centres: the two agree to the rounding of the centres (about 1e-16 of the
// root box over the cell side).  List 4 is added afterwards by k_m2l64w in
// its list-4 mode.
constexpr int kM2l64Waves = 4;
typedef double v4d __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t compact1by1(uint32_t v) {
    v &= 0x55555555u;
    v = (v | (v >> 1)) & 0x33333333u;
    v = (v | (v >> 2)) & 0x0F0F0F0Fu;
    v = (v | (v >> 4)) & 0x00FF00FFu;
    v = (v | (v >> 8)) & 0x0000FFFFu;
    return v;
}

// Eight resident wavefronts per SIMD (the register budget that allows them:
// 64 per lane, accumulators included): the kernel waits on its gathers, and
// 8 instead of 5 resident wavefronts cut it from 170 to 146 us at 780k (p 10).
template <int P>
__global__ void __launch_bounds__(kWave *kM2l64Waves) __attribute__((amdgpu_waves_per_eu(8, 8)))
    k_m2l64_mfma(const DevHdr *hdr, int maxL, const uint32_t *c_key, const int *l2,
                 const uint8_t *n2, const double *R, const double2 *ak, double2 *bk) {
    constexpr int P1 = P + 1, K = 2 * P1, KS = (K + 3) / 4, MT = (2 * P + 15) / 16;
    __shared__ int smap[16][49];
    __shared__ double red[kM2l64Waves][MT * 4][kWave];
    __shared__ double s_sc[P1];
    __shared__ int s_tile[3];
    const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    if (threadIdx.x == 0) {
        // this block's tile: level L, first cell, cells (up to 16)
        int b = (int)blockIdx.x, L = 2, j0 = -1, cnt = 0;
        for (; L <= maxL; ++L) {
            const int c0 = (int)hdr->lev_off[L], cn = (int)hdr->lev_off[L + 1] - c0;
            const int nt = (cn + 15) / 16;
            if (b < nt) {
                j0 = c0 + 16 * b;
                cnt = min(16, cn - 16 * b);
                break;
            }
            b -= nt;
        }
        s_tile[0] = L;
        s_tile[1] = j0;
        s_tile[2] = cnt;
    }
    for (int t = threadIdx.x; t < 16 * 49; t += blockDim.x) smap[t / 49][t % 49] = -1;
    __syncthreads();
    const int L = s_tile[0], j0 = s_tile[1], cnt = s_tile[2];
    if (j0 < 0) return;  // (uniform over the block)
    if (threadIdx.x < P1) {
        // len^-k, k = 0..P
        const double inv = ldexp(1.0 / hdr->root_len, L);
        double sc = 1.0;
        for (int k = 0; k < (int)threadIdx.x; ++k) sc *= inv;
        s_sc[threadIdx.x] = sc;
    }
    {
        // source map of the tile: slot (dx+3) + 7 (dy+3) -> source cell or -1
        const int tn = threadIdx.x % 16, tu = threadIdx.x / 16;
        const int tj = j0 + tn;
        if (tn < cnt) {
            const uint32_t kj = c_key[tj];
            const int jx = (int)compact1by1(kj), jy = (int)compact1by1(kj >> 1);
            const int m2 = n2[tj];
            for (int u = tu; u < m2; u += (int)blockDim.x / 16) {
                const int sidx = l2[27 * tj + u];
                const uint32_t ks = c_key[sidx];
                const int dx = (int)compact1by1(ks) - jx, dy = (int)compact1by1(ks >> 1) - jy;
                smap[tn][(dx + 3) + 7 * (dy + 3)] = sidx;
            }
        }
    }
    __syncthreads();
    const int n = lane % 16, kq = lane / 16;
    const double *a1 = reinterpret_cast<const double *>(ak);
    // orders 9 and 10: rows 16.. (at most 4) on v_mfma_f64_4x4x4f64, whose
    // A operand holds row 16 + l % 4, column l / 16 of a 4-step, whose B
    // operand is laid out as the 16x16x4 one (target l % 16, step row l / 16)
    // and whose result is row 16 + l / 16 of target l % 16
    constexpr bool LEFT = 2 * P > 16 && 2 * P <= 20;
    v4d acc[MT];
    double acc4 = 0.0;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = v4d{0.0, 0.0, 0.0, 0.0};
    int o = 0;
    for (int slot = 0; slot < 49; ++slot) {
        const int dx = slot % 7 - 3, dy = slot / 7 - 3;
        if (dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1) continue;
        const int oc = o++;
        if (oc % kM2l64Waves != w) continue;
        const int sidx = smap[n][slot];
        if (__ballot(sidx >= 0) == 0) continue;  // no target of the tile uses this offset
        double b[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int col = ks * 4 + kq;  // 2k (Re a_k) or 2k + 1 (Im a_k)
            b[ks] = (sidx >= 0 && col < K) ? a1[(size_t)sidx * K + col] * s_sc[col >> 1] : 0.0;
        }
        const double *Ro = R + (size_t)oc * KS * MT * kWave + lane;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
            for (int mt = 0; mt < (LEFT ? 1 : MT); ++mt)
                acc[mt] = __builtin_amdgcn_mfma_f64_16x16x4f64(Ro[(ks * MT + mt) * kWave], b[ks],
                                                               acc[mt], 0, 0, 0);
            if (LEFT)
                acc4 = __builtin_amdgcn_mfma_f64_4x4x4f64(Ro[(ks * MT + 1) * kWave], b[ks], acc4,
                                                          0, 0, 0);
        }
    }
#pragma unroll
    for (int mt = 0; mt < (LEFT ? 1 : MT); ++mt)
#pragma unroll
        for (int v = 0; v < 4; ++v) red[w][mt * 4 + v][lane] = acc[mt][v];
    if (LEFT) red[w][4][lane] = acc4;
    __syncthreads();
    if (w != 0) return;
    if (lane < cnt) bk[(size_t)(j0 + lane) * P1] = make_double2(0.0, 0.0);  // b_0 is not formed
    double *bo = reinterpret_cast<double *>(bk);
    if (LEFT) {
        double sum = 0.0;
#pragma unroll
        for (int u = 0; u < kM2l64Waves; ++u) sum += red[u][4][lane];
        const int row = 16 + kq;
        if (n < cnt && row < 2 * P) {
            const int p = row / 2 + 1;
            bo[((size_t)(j0 + n) * P1 + p) * 2 + (row & 1)] = sum * s_sc[p];
        }
    }
#pragma unroll
    for (int mt = 0; mt < (LEFT ? 1 : MT); ++mt) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            double sum = 0.0;
#pragma unroll
            for (int u = 0; u < kM2l64Waves; ++u) sum += red[u][mt * 4 + v][lane];
            const int row = mt * 16 + 4 * v + kq;  // Re b^_1, Im b^_1, Re b^_2, ...
            if (n < cnt && row < 2 * P) {
                const int p = row / 2 + 1;
                bo[((size_t)(j0 + n) * P1 + p) * 2 + (row & 1)] = sum * s_sc[p];
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
// The kernel is bound by vector-ALU issue where leaves abound (0.74 of the
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
// size of the round is well inside the range of rcp64 (a size of zero, say, is
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
        const double rho2 = tame ? r2 * rcp64(sij2) : r2 / sij2;
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
    // padding source: zero strength, outside the root box
    const double padx = lcx + 4.0 * A.hdr->root_len;
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
                        const double s2 = A.ss[src] * A.ss[src];
                        l.s2[r] = s2;
                        odd_s |= wild(s2);
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
                        const double s2 = A.ss[src] * A.ss[src];
                        l.s2[r] = s2;
                        odd_s |= wild(s2);
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
            const cd w = cinv(cd{c_cx[sidx] - cx, c_cy[sidx] - cy});
            const size_t b = (size_t)sidx * ND;
            cd sm = cscale(ld(ak, b + ND - 1), row[ND - 1]);
            for (int k = ND - 2; k >= 0; --k) sm = cadd(cmul(sm, w), cscale(ld(ak, b + k), row[k]));
            acc = cadd(acc, cmul(sm, cpowi(w, l + 1)));
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

// Type-1 L2L for the cells of one level (>= 3; level-1 locals are zero), thread
// per (cell, l): orders ND above 15.
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
    const double *t_r64 = (const double *)c.tab_r64.p;
    if (nc > j2 && P >= 1 && P < kM2lwP1 && !potential && t_r64 && c.tab_r64_p == P) {
        // list 2 on the matrix cores, then list 4 added by the wavefront kernel
        int ntiles = 0;
        for (int L = 2; L <= ti.max_level; ++L)
            ntiles += (int)div_up((long long)(ti.lev_off[L + 1] - ti.lev_off[L]), 16LL);
        const uint32_t *c_key = (const uint32_t *)c.c_key.p;
        const int *l2 = (const int *)c.l2.p;
        const uint8_t *n2 = (const uint8_t *)c.n2.p;
        switch (P) {
#define M2L64_CASE(PP)                                                                          \
    case PP:                                                                                    \
        k_m2l64_mfma<PP><<<ntiles, kWave * kM2l64Waves, 0, s>>>(c.hdr_d, ti.max_level, c_key, l2, \
                                                              n2, t_r64, ak, bk);               \
        break;
            M2L64_CASE(1) M2L64_CASE(2) M2L64_CASE(3) M2L64_CASE(4) M2L64_CASE(5) M2L64_CASE(6)
            M2L64_CASE(7) M2L64_CASE(8) M2L64_CASE(9) M2L64_CASE(10) M2L64_CASE(11)
            M2L64_CASE(12) M2L64_CASE(13) M2L64_CASE(14) M2L64_CASE(15) M2L64_CASE(16)
#undef M2L64_CASE
            default: break;
        }
        k_m2l64w<false, true><<<div_up(nc - j2, kM2lwWaves), kWave * kM2lwWaves, 0, s>>>(
            j2, nc, P, list4_mode, t_m2l, l2, n2, (const int *)c.l4.p,
            (const uint8_t *)c.n4.p, c_cx, c_cy, c_begin, c_end, xs, ys, qs, as, ak, bk);
    } else if (nc > j2 && P < kM2lwP1)
        (potential ? k_m2l64w<true, false> : k_m2l64w<false, false>)<<<
            div_up(nc - j2, kM2lwWaves), kWave * kM2lwWaves, 0, s>>>(
            j2, nc, P, list4_mode, t_m2l, (const int *)c.l2.p, (const uint8_t *)c.n2.p,
            (const int *)c.l4.p, (const uint8_t *)c.n4.p, c_cx, c_cy, c_begin, c_end, xs, ys, qs,
            as, ak, bk);
    else if (nc > j2)
        (potential ? k_m2l64<true, 0> : k_m2l64<false, 0>)<<<
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
    // (the root's local row is not read: the tree's leaves are of level >= 1)
    k_p2m64<<<div_up(nl, kP2m64Waves * kP2mLeaves), kWave * kP2m64Waves, 0, s>>>(
        leaf_idx, nl, PM, c_flags, c_begin, c_end, c_cx, c_cy, xs, ys, qs, as, ak, bk, 1, NL);
    m2m64_run(ti, PM, (const double *)c.t1_m2m.p, c_flags, c_cx, c_cy, c_child, ak, s);
    mk.mark(3, s);
    // M2L and P2L: every cell of level >= 1 (all of bk written)
    const int j1 = (int)ti.lev_off[1];
    if (nc > j1)
        k_m2l_t1<<<div_up((long long)(nc - j1) * NL, 256), 256, 0, s>>>(
            j1, nc, ND, (const double *)c.t1_m2l.p, c_level, (const int *)c.l2.p,
            (const uint8_t *)c.n2.p, (const int *)c.l4.p, (const uint8_t *)c.n4.p, c_cx, c_cy,
            c_begin, c_end, xs, ys, qs, ak, bk);
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

// Realified list-2 M2L matrices of order P for k_m2l64_mfma, one per offset
// delta = (dx, dy) (source minus target centre over the cell side; |dx|,
// |dy| <= 3, not both <= 1; slot order, dy major): row 2(p-1) (Re b^_p) and
// 2(p-1)+1 (Im), p = 1..P; column 2k (Re a^_k) and 2k+1 (Im), k = 0..P;
// entry M[p][k] = tab[p][k] delta^-(p+k), tab being the path's M2L table
// (tab[p][0] = -1/p, tab[p][k] = -C(p+k-1, k-1) (-1)^k / k with its
// binomials).  Stored in the A-operand lane order of v_mfma_f64_16x16x4f64:
// R[((o KS + ks) MT + mt) 64 + l] = M[16 mt + l % 16][4 ks + l / 16].
void fmm64_mfma_table(int P, const double *tab, std::vector<double> &R) {
    const int P1 = P + 1, K = 2 * P1, KS = (K + 3) / 4, MT = (2 * P + 15) / 16;
    const bool left = 2 * P > 16 && 2 * P <= 20;  // rows 16.. for the 4x4x4 instruction
    R.assign((size_t)40 * KS * MT * kWave, 0.0);
    std::vector<double> pwr(2 * P + 2), pwi(2 * P + 2);
    int o = 0;
    for (int dy = -3; dy <= 3; ++dy) {
        for (int dx = -3; dx <= 3; ++dx) {
            if (std::abs(dx) <= 1 && std::abs(dy) <= 1) continue;
            const double r2 = (double)(dx * dx + dy * dy);
            const double wr = dx / r2, wi = -dy / r2;  // 1 / delta
            pwr[0] = 1.0;
            pwi[0] = 0.0;
            for (int t = 1; t <= 2 * P + 1; ++t) {
                pwr[t] = pwr[t - 1] * wr - pwi[t - 1] * wi;
                pwi[t] = pwr[t - 1] * wi + pwi[t - 1] * wr;
            }
            for (int p = 1; p <= P; ++p) {
                for (int k = 0; k <= P; ++k) {
                    const double T = tab[(size_t)p * P1 + k];
                    const double Mr = T * pwr[p + k], Mi = T * pwi[p + k];
                    const int r0 = 2 * (p - 1), c0 = 2 * k;
                    const double val[2][2] = {{Mr, -Mi}, {Mi, Mr}};
                    for (int a = 0; a < 2; ++a) {
                        for (int bq = 0; bq < 2; ++bq) {
                            const int row = r0 + a, col = c0 + bq;
                            const int mt = row / 16, ks = col / 4;
                            const size_t base = (((size_t)o * KS + ks) * MT + mt) * kWave;
                            if (left && row >= 16) {
                                // v_mfma_f64_4x4x4f64 A operand: row 16 + l % 4,
                                // step column l / 16, the same for the four blocks
                                for (int q = 0; q < 4; ++q)
                                    R[base + (row - 16) + 4 * q + 16 * (col % 4)] = val[a][bq];
                            } else {
                                const int lane = (row % 16) + 16 * (col % 4);
                                R[base + lane] = val[a][bq];
                            }
                        }
                    }
                }
            }
            ++o;
        }
    }
}

}  // namespace vpm
