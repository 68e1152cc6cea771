// kem_tree.hip -- hierarchical far field: multipole expansions of runs of elements.
//
// A field evaluation at many points spends its time on pairs far apart.  Elements lie in
// compact runs of KEM_TREE_LEAF, KEM_TREE_FAN of which make the next level's run (kem::build_tree).  Each call
// expands the charge of every run about its centre (k_tree_p2m for the lowest level, k_tree_m2m upwards), finds how far
// from it the charge lies (k_tree_reach),
// and each wavefront walks the tree for its 64 points: a run far enough from all of them is one expansion,
// of the order that its distance asks for, and the rest of the elements go pair by pair through the
// same rules as the flat far passes (k_field_far, k_field_far32c).  Expansions are FP64 in both precisions.
//
// With d = (P - c) / a about a run of radius a, centre c, and (x + i y)^m = C_m + i S_m:
//   phi = sum_m [C_m F_m + S_m G_m] / a,   F_m = sum_l A_lm L_l^m,   G_m = sum_l B_lm L_l^m,
// where L_l^m = (l-m)! P_l^m / sin^m / d^(l+m+1) and A - the real and B - the imaginary part of
// (2 - delta_m0) sum_q q conj(R_l^m), R_l^m = d^l P_l^m e^(i m phi) / (l+m)! (no Condon-Shortley phase).
// These normalisations make the gradient a shift of the order: d/dz lowers L_l^m to -L_(l+1)^m, and twice
// the derivative of L_l^m in d^2 at fixed z is -L_(l+1)^(m+1), so the field takes the same A and B against
// L of the next order, six multiply-adds and a four-operation recurrence per (l, m).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "kem_device.hpp"
#include "kem_kernels.h"

namespace kem {

using dev::F4;

namespace {

// Coefficients of one run as (A, B): line m = 0 .. P + 1 holds l = m - 1 .. P + 4, zero outside m <= l <= P, so that
// sums in steps of four may run past the last order.
constexpr int kPad = 6;
__host__ __device__ constexpr int line_start(int P, int m) { return m * (P + kPad) - m * (m - 1) / 2; }
__host__ __device__ constexpr int entry(int P, int l, int m) { return line_start(P, m) + l - m + 1; }
__host__ __device__ constexpr int entries(int P) { return line_start(P, P + 2); }
__host__ __device__ constexpr int tri_index(int l, int m) { return l * (l + 1) / 2 + m; }

// The order stored, and the tolerance that chooses the order summed.  With T_l = sum_q |q| (r_q / a)^l over a run's
// charges (r_q from its centre), the terms of order l are at most T_l (a / d)^l of the potential and (l + 1) T_l (a / d)^l
// of the field, tight for a single charge.  By convexity T_l <= rho^l T_0 up to order L for rho^L = T_L / T_0, so order
// p serves a run at distance d from the sphere around a range of points when, with q = rho a / d,
//   sum_{l > p} (l + 1) q^l (1 - q)^2 = ((p + 2) - (p + 1) q) q^(p+1) <= tol,
// the field's omitted part against the field of the charge rho a from the centre on the points' side (L past the order
// stored and a / d < widest bound what rho does not).  Each call finds rho a of each run (k_tree_reach): at the rim it
// is a, for the elements of a surface 0.8 to 0.9 of it.
// The tolerances keep every point's field as good as the pairs' own rules do it, whatever the charges: one
// charged element at the rim of a run of any level (of 16 to 4,096 elements: 20,000-triangle coax, 100,000-triangle bore, a
// cube, rectangles and wires), points in clumps beyond it, worst / root mean square error of the field: FP64 3.3e-14 / 2.8e-15
// both here and in the flat passes, mixed 4.0e-7 / 1.0e-7 in both (with (a / d)^(p+1) <= 8e-14 and 7e-7, the bound of the
// potential, 8.5e-13 and 4.5e-6).
// The orders (at 2^-21.25 and 2^-45.2): a million points over 20,000 triangles, mixed, 19.5 ms at 20, 19.1 at 22, 19.0 at
// 24, where 400,000 over 100,000 take 8.5, 8.7 and 8.7; 100,000 points over 20,000, FP64, 14.2 ms at 26, 13.5 at 28, 12.9 at 30.
template <bool MIXED>
struct Orders {
    static constexpr int P = MIXED ? 21 : 30;
    static constexpr float log2_tol = MIXED ? -21.7f : -47.2f;
    static constexpr float widest = 0.6f;
    static constexpr int H = (P + 2) / 2;  // L / 2
};

// ------------------------------------------------------------------ expansions
constexpr int kP2MBlock = 256;
constexpr int kP2MElems = 16;  // elements whose nodes are staged at a time

// coefficient v (A or B of an entry) of the stored layout: its order (l, m), false outside m <= l <= P
template <int P>
__device__ __forceinline__ bool order_of(int v, int& l, int& m)
{
    const int q = v >> 1;
    m = 0;
    while (line_start(P, m + 1) <= q) m++;
    l = q - line_start(P, m) + m - 1;
    return l >= m && l <= P;
}

// one quadrature node (position about the run's centre, charge) into line m's sums, scaled as um = (2m-1)!! says
template <int P>
__device__ __forceinline__ void follow(const double4& node, int m, double um, double (&A)[P + 1], double (&B)[P + 1])
{
    const double x = node.x, y = node.y, z = node.z;
    const double d2 = x * x + y * y + z * z;
    // (x + i y)^m by its binary digits
    double C = node.w, S = 0., bx = x, by = y;
#pragma unroll
    for (int bit = 1; bit < 32; bit <<= 1) {
        if (m & bit) {
            const double c = C * bx - S * by;
            S = C * by + S * bx;
            C = c;
        }
        const double c = bx * bx - by * by;
        by = 2. * bx * by;
        bx = c;
    }
    double u0 = 0., u1 = um, f = 2 * m + 1, gd = 0.;  // f = 2l + 1, gd = l^2 - m^2
#pragma unroll
    for (int i = 0; i <= P; i++) {
        if (m + i <= P) {
            A[i] = __builtin_fma(C, u1, A[i]);
            B[i] = __builtin_fma(S, u1, B[i]);
            const double u2 = __builtin_fma(f * z, u1, -(gd * d2) * u0);
            u0 = u1;
            u1 = u2;
            gd += f;
            f += 2.;
        }
    }
}
// from those sums to the stored coefficients of order (l, m)
__device__ __forceinline__ double unscale_divisor(int l, int m)
{
    double f = m ? 0.5 : 1.;  // 2 for the pair of orders m and -m
    for (int k = 2; k <= l + m; k++) f *= k;
    for (int k = 2; k <= l - m; k++) f *= k;
    return f;
}

// Expansion of each run of the lowest stored level: one block per run.  The quadrature nodes (33 per surface
// element, 16 per wire) of 16 elements at a time are staged in LDS, as positions about the centre and charges; half a
// wavefront follows one node, lane m its line m, with the sums in registers; the halves are added by a shuffle and
// the wavefronts in order through LDS.  (Each lane loading its own node waits on three dependent loads per node:
// 438 us for 2,500 runs of 8 at order 18.)
template <int P>
__global__ __launch_bounds__(kP2MBlock) void k_tree_p2m(const double* __restrict__ geom,
                                                        const double* __restrict__ nodes,
                                                        const int32_t* __restrict__ order,
                                                        const double* __restrict__ sigma,
                                                        const double* __restrict__ tnode, int64_t nelem, int run,
                                                        double* __restrict__ mom)
{
    static_assert(P < 32, "a line per lane of half a wavefront");
    constexpr int kNodes = 33, kWaves = kP2MBlock / 64, T = tri_index(P, P) + 1;
    __shared__ double4 pt[kP2MElems * kNodes];
    __shared__ double red[kWaves][T][2];
    const int64_t node = blockIdx.x;
    const double* t = tnode + node * KEM_TREE_STRIDE;
    const double cx = t[0], cy = t[1], cz = t[2], ia = t[5];
    const int64_t e0 = node * run;
    const int ne = (int)(nelem - e0 < run ? nelem - e0 : run);
    const int half = threadIdx.x >> 5, m = threadIdx.x & 31, wave = threadIdx.x >> 6;
    double A[P + 1], B[P + 1];
#pragma unroll
    for (int i = 0; i <= P; i++) A[i] = B[i] = 0.;
    // lines scaled to (l-m)! (l+m)! R_l^m / (x + i y)^m, from (2m)! / (2^m m!) = (2m-1)!! on
    double um = 1.;
    for (int i = 1; i <= m; i++) um *= 2 * i - 1;
    for (int s0 = 0; s0 < ne; s0 += kP2MElems) {
        const int nq = min(ne - s0, kP2MElems) * kNodes;
        __syncthreads();
        for (int q = threadIdx.x; q < nq; q += kP2MBlock) {
            const int e = q / kNodes, k = q - e * kNodes;
            const int64_t j = order[e0 + s0 + e];
            const double* g = geom + j * KG_STRIDE;
            const bool wire = (int)g[KG_TYPE] == KEM_LINESEGMENT;
            const double* nd = nodes + j * KEM_NODE_STRIDE + 4 * (wire ? KEM_L16 + (k & 15) : KEM_N33 + k);
            const double w = wire && k >= 16 ? 0. : nd[3] * g[KG_PREF] * sigma[j];
            pt[q] = double4{(nd[0] - cx) * ia, (nd[1] - cy) * ia, (nd[2] - cz) * ia, w};
        }
        __syncthreads();
        for (int q = half; q < nq; q += kP2MBlock / 32) follow<P>(pt[q], m, um, A, B);
    }
#pragma unroll
    for (int i = 0; i <= P; i++) {
        const double a = A[i] + __shfl_xor(A[i], 32, 64), b = B[i] + __shfl_xor(B[i], 32, 64);
        if ((threadIdx.x & 32) == 0 && m + i <= P) {
            red[wave][tri_index(m + i, m)][0] = a;
            red[wave][tri_index(m + i, m)][1] = b;
        }
    }
    __syncthreads();
    double* o = mom + node * (2 * entries(P));
    for (int v = threadIdx.x; v < 2 * entries(P); v += kP2MBlock) {
        int l, mm;
        double s = 0.;
        if (order_of<P>(v, l, mm)) {
            const int at = tri_index(l, mm);
            for (int k = 0; k < kWaves; k++) s += red[k][at][v & 1];
            s /= unscale_divisor(l, mm);
        }
        o[v] = s;
    }
}

// The same for several charge-density sets: one block per run expands each of its elements at unit charge density once
// (half a wavefront per element, its nodes as above) and leaves the coefficients in LDS; the sets' expansions are sums
// of them, a thread per coefficient (64 sets of 20,000 triangles 0.56 ms, and 2.8 ms the levels above).
template <int P>
__global__ __launch_bounds__(kP2MBlock) void k_tree_p2m_sets(const double* __restrict__ geom,
                                                             const double* __restrict__ nodes,
                                                             const int32_t* __restrict__ order,
                                                             const double* __restrict__ sigma, int64_t nsets,
                                                             const double* __restrict__ tnode, int64_t nelem, int run,
                                                             double* __restrict__ mom, int64_t mom_set)
{
    static_assert(P < 32, "a line per lane of half a wavefront");
    constexpr int kNodes = 33, kElems = 8, T = tri_index(P, P) + 1, kSets = 32;
    __shared__ double4 pt[kElems * kNodes];
    __shared__ double unit[kElems][2 * T];
    __shared__ double sg[kSets][kElems];
    const int64_t node = blockIdx.x;
    const double* t = tnode + node * KEM_TREE_STRIDE;
    const double cx = t[0], cy = t[1], cz = t[2], ia = t[5];
    const int64_t e0 = node * run;
    const int ne = (int)(nelem - e0 < run ? nelem - e0 : run);
    const int half = threadIdx.x >> 5, m = threadIdx.x & 31;
    double um = 1.;
    for (int i = 1; i <= m; i++) um *= 2 * i - 1;
    for (int s0 = 0; s0 < ne; s0 += kElems) {
        const int nq = min(ne - s0, kElems) * kNodes;
        __syncthreads();
        for (int q = threadIdx.x; q < kElems * kNodes; q += kP2MBlock) {
            pt[q] = double4{0., 0., 0., 0.};
            if (q >= nq) continue;
            const int e = q / kNodes, k = q - e * kNodes;
            const int64_t j = order[e0 + s0 + e];
            const double* g = geom + j * KG_STRIDE;
            const bool wire = (int)g[KG_TYPE] == KEM_LINESEGMENT;
            const double* nd = nodes + j * KEM_NODE_STRIDE + 4 * (wire ? KEM_L16 + (k & 15) : KEM_N33 + k);
            const double w = wire && k >= 16 ? 0. : nd[3] * g[KG_PREF];
            pt[q] = double4{(nd[0] - cx) * ia, (nd[1] - cy) * ia, (nd[2] - cz) * ia, w};
        }
        __syncthreads();
        {
            double A[P + 1], B[P + 1];
#pragma unroll
            for (int i = 0; i <= P; i++) A[i] = B[i] = 0.;
            for (int q = half * kNodes; q < (half + 1) * kNodes; q++) follow<P>(pt[q], m, um, A, B);
#pragma unroll
            for (int i = 0; i <= P; i++)
                if (m + i <= P) {
                    const int at = tri_index(m + i, m);
                    unit[half][2 * at] = A[i];
                    unit[half][2 * at + 1] = B[i];
                }
        }
        for (int64_t c0 = 0; c0 < nsets; c0 += kSets) {
            const int nc = (int)(nsets - c0 < kSets ? nsets - c0 : kSets);
            __syncthreads();
            {
                const int e = threadIdx.x & (kElems - 1), c = threadIdx.x / kElems;
                static_assert(kP2MBlock == kElems * kSets, "a charge density per thread");
                sg[c][e] = s0 + e < ne && c < nc ? sigma[(c0 + c) * nelem + order[e0 + s0 + e]] : 0.;
            }
            __syncthreads();
            for (int v = threadIdx.x; v < 2 * entries(P); v += kP2MBlock) {
                int l, mm;
                double u[kElems];
                const bool have = order_of<P>(v, l, mm);
                const int at = have ? 2 * tri_index(l, mm) + (v & 1) : 0;
#pragma unroll
                for (int e = 0; e < kElems; e++) u[e] = have ? unit[e][at] : 0.;
                if (have) {
                    const double f = unscale_divisor(l, mm);
#pragma unroll
                    for (int e = 0; e < kElems; e++) u[e] /= f;
                }
                double* o = mom + c0 * mom_set + node * (2 * entries(P)) + v;
                for (int c = 0; c < nc; c++) {
                    double s = s0 ? o[c * mom_set] : 0.;
#pragma unroll
                    for (int e = 0; e < kElems; e++) s = __builtin_fma(u[e], sg[c][e], s);
                    o[c * mom_set] = s;
                }
            }
        }
    }
}

// Expansions of one level's runs from those of the level below: one block per run (and set, blockIdx.y).  Two groups of 512 threads
// translate a child each at a time by the addition theorem of the R_l^m (exact up to order P), a thread per (l, m).
// Both factors lie in LDS with their negative orders written out, so the sum over (k, j) is two 16-byte
// reads and four multiply-adds a term.
constexpr int kM2MGroup = 512;
template <int P>
__global__ __launch_bounds__(2 * kM2MGroup) void k_tree_m2m(const double* __restrict__ tchild,
                                                            const double* __restrict__ tparent, int64_t nchild,
                                                            const double* __restrict__ mchild,
                                                            double* __restrict__ mparent, int64_t mom_set)
{
    mchild += blockIdx.y * mom_set;
    mparent += blockIdx.y * mom_set;
    constexpr int T = tri_index(P, P) + 1, N = (P + 1) * (P + 1);  // (l, m) at l^2 + l + m
    static_assert(T <= kM2MGroup, "a thread per order");
    __shared__ double2 R[2][N], Q[2][N];
    __shared__ double2 sum[2][T];
    const int64_t node = blockIdx.x;
    const int grp = threadIdx.x / kM2MGroup, t = threadIdx.x - grp * kM2MGroup;
    int l = 0;
    while (tri_index(l + 1, 0) <= t) l++;
    const int m = t - tri_index(l, 0);
    const double* tp = tparent + node * KEM_TREE_STRIDE;
    double re = 0., im = 0.;
    for (int c = grp; c < KEM_TREE_FAN; c += 2) {
        const int64_t child = node * KEM_TREE_FAN + c;
        const bool have = child < nchild;
        __syncthreads();
        if (have) {
            const double* tc = tchild + child * KEM_TREE_STRIDE;
            const double ia = tp[5], ratio = tc[3] * ia;
            const double sg = (m & 1) ? -1. : 1.;  // R_l^(-m) = (-1)^m conj(R_l^m), and so the sums of them
            if (t < T) {
                const double2 v = reinterpret_cast<const double2*>(mchild)[child * entries(P) + entry(P, l, m)];
                double s = m ? 0.5 : 1.;
                for (int k = 0; k < l; k++) s *= ratio;
                Q[grp][l * l + l - m] = double2{sg * s * v.x, -sg * s * v.y};
                Q[grp][l * l + l + m] = double2{s * v.x, s * v.y};
            }
            if (t <= P) {  // line t of the shift's R
                const double x = (tc[0] - tp[0]) * ia, y = (tc[1] - tp[1]) * ia, z = (tc[2] - tp[2]) * ia;
                const double d2 = x * x + y * y + z * z;
                const double sl = (t & 1) ? -1. : 1.;
                double C = 1., S = 0., um = 1.;
                for (int i = 1; i <= t; i++) {
                    const double c1 = C * x - S * y;
                    S = C * y + S * x;
                    C = c1;
                    um *= dev::quot_acc(0.5, (double)i);
                }
                double u0 = 0., u1 = um;
                for (int h = t; h <= P; h++) {
                    R[grp][h * h + h - t] = double2{sl * C * u1, -sl * S * u1};
                    R[grp][h * h + h + t] = double2{C * u1, S * u1};
                    const double u2 = dev::quot_acc((2 * h + 1) * z * u1 - d2 * u0, (double)((h + 1 - t) * (h + 1 + t)));
                    u0 = u1;
                    u1 = u2;
                }
            }
        }
        __syncthreads();
        if (have && t < T)
            for (int k = 0; k <= l; k++) {
                const int h = l - k;
                const int j0 = max(-k, m - h), j1 = min(k, m + h);
                const double2* q = &Q[grp][k * k + k + j0];
                const double2* r = &R[grp][h * h + h + m - j0];
#pragma unroll 2
                for (int j = j0; j <= j1; j++, q++, r--) {
                    re += r->x * q->x - r->y * q->y;
                    im += r->x * q->y + r->y * q->x;
                }
            }
    }
    if (t < T) sum[grp][t] = double2{re, im};
    __syncthreads();
    double* o = mparent + node * (2 * entries(P));
    for (int v = threadIdx.x; v < 2 * entries(P); v += 2 * kM2MGroup) {
        int lo, mo;
        double s = 0.;
        if (order_of<P>(v, lo, mo)) {
            const int at = tri_index(lo, mo);
            s = (v & 1) ? sum[0][at].y + sum[1][at].y : sum[0][at].x + sum[1][at].x;
            if (mo) s += s;
        }
        o[v] = s;
    }
}

// rho a of each run from the lowest stored level up, and of each set (blockIdx.y); L = 2 H.  The mean of r^L over an element
// is at most that over its corners, since it is convex.  Bound by the elements' records, read once per level: 14 us
// for 20,000 triangles, 70 us for 100,000.
template <int H>
__global__ __launch_bounds__(kP2MBlock) void k_tree_reach(const double* __restrict__ geom,
                                                          const int32_t* __restrict__ order,
                                                          const double* __restrict__ sigma,
                                                          const double* __restrict__ tnode, TreeLevels T, int64_t nelem,
                                                          float* __restrict__ reach, int64_t reach_set)
{
    __shared__ double red[kP2MBlock / 64][2];
    const int64_t base = T.first[T.low], node = base + blockIdx.x;
    int lev = T.low;
    int64_t run = T.run;
    while (node >= (int64_t)T.first[lev] + T.count[lev]) {
        lev++;
        run *= KEM_TREE_FAN;
    }
    const int64_t e0 = (node - T.first[lev]) * run, e1 = e0 + run < nelem ? e0 + run : nelem;
    const double* t = tnode + node * KEM_TREE_STRIDE;
    const double* sg = sigma + blockIdx.y * nelem;
    const double cx = t[0], cy = t[1], cz = t[2], ia2 = t[5] * t[5];
    double all = 0., far = 0.;
    for (int64_t e = e0 + threadIdx.x; e < e1; e += kP2MBlock) {
        const int64_t j = order[e];
        const double* g = geom + j * KG_STRIDE;
        const int type = (int)g[KG_TYPE], nv = type == KEM_TRIANGLE ? 3 : type == KEM_RECTANGLE ? 4 : 2;
        double corners = 0.;
        for (int v = 0; v < nv; v++) {
            const double dx = g[KG_V + 3 * v] - cx, dy = g[KG_V + 3 * v + 1] - cy, dz = g[KG_V + 3 * v + 2] - cz;
            double f = 1., b = (dx * dx + dy * dy + dz * dz) * ia2;
#pragma unroll
            for (int k = H; k; k >>= 1) {
                if (k & 1) f *= b;
                b *= b;
            }
            corners += f;
        }
        const double w = fabs(g[KG_PREF] * sg[j]);
        all += w;
        far += w * corners / nv;
    }
    for (int o = 32; o > 0; o >>= 1) {
        all += __shfl_xor(all, o, 64);
        far += __shfl_xor(far, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6][0] = all;
        red[threadIdx.x >> 6][1] = far;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int k = 1; k < kP2MBlock / 64; k++) {
        all += red[k][0];
        far += red[k][1];
    }
    // rounded up, and no less than a mean whose power is still a 32-bit number; charges that are not finite: the radius
    const float rho = all == 0. ? 0.f : exp2f(log2f((float)(far / all)) * (0.5f / H)) * 1.0001f;
    reach[blockIdx.y * reach_set + blockIdx.x] = (float)t[3] * 1.0001f * (rho < 1.f ? fmaxf(rho, 0.0625f) : 1.f);
}

// ------------------------------------------------------------------ evaluation
typedef double Pair __attribute__((ext_vector_type(2)));

// phi and -grad phi of one expansion, stored to order P and summed to order p <= P or one above, at NP points
// (x, y, z) = (P - c) / a of a lane.  The coefficients co lie in LDS and every lane reads the same ones, 16 bytes at a
// time; two points per lane halve those reads per point, which would otherwise bound the sum (16 cycles of LDS per
// step and wavefront, times 4 SIMDs, against 40 of the vector ALU).  One loop for all orders: unrolled per order, the
// compiler keeps whole lines in registers.
template <int P, int NP>
__device__ __forceinline__ void m2p(const Pair* co, int p, const double (&x)[NP], const double (&y)[NP],
                                    const double (&z)[NP], F4 (&out)[NP])
{
    double rho[NP], zh[NP], lm[NP], C[NP], S[NP], Cp[NP], Sp[NP], w[NP], tx[NP], ty[NP];
#pragma unroll
    for (int n = 0; n < NP; n++) {
        const double ir = dev::rsqrt_acc(x[n] * x[n] + y[n] * y[n] + z[n] * z[n]);
        rho[n] = ir * ir;
        zh[n] = z[n] * rho[n];
        lm[n] = ir;  // L_m^m = (2m-1)!! / d^(2m+1)
        C[n] = 1.;
        S[n] = Cp[n] = Sp[n] = w[n] = tx[n] = ty[n] = 0.;
        out[n] = F4{0., 0., 0., 0.};
    }
    double fm = 0.;
    const Pair* own = co + 1;   // (l, m) from l = m on
    const Pair* below = own;    // (l - 1, m - 1); any finite values for m = 0, where Cp = Sp = 0
#pragma unroll 1
    for (int m = 0; m <= p + 1; m++) {
        double F[NP], G[NP], Zc[NP], Zs[NP], Tc[NP], Ts[NP], l0[NP], l1[NP];
#pragma unroll
        for (int n = 0; n < NP; n++) {
            F[n] = G[n] = Zc[n] = Zs[n] = Tc[n] = Ts[n] = l0[n] = 0.;
            l1[n] = lm[n];
        }
        double f = __builtin_fma(2., fm, 1.), gd = 0.;  // 2l + 1, l^2 - m^2
        Pair v = {0., 0.};
        const Pair *o = own, *t = below;
        auto step = [&](const Pair& vo, const Pair& vt) {
#pragma unroll
            for (int n = 0; n < NP; n++) {
                Zc[n] = __builtin_fma(v.x, l1[n], Zc[n]);
                Zs[n] = __builtin_fma(v.y, l1[n], Zs[n]);
                F[n] = __builtin_fma(vo.x, l1[n], F[n]);
                G[n] = __builtin_fma(vo.y, l1[n], G[n]);
                Tc[n] = __builtin_fma(vt.x, l1[n], Tc[n]);
                Ts[n] = __builtin_fma(vt.y, l1[n], Ts[n]);
                // L_(l+1) = ((2l+1) z L_l - (l^2-m^2) L_(l-1)) / d^2
                const double l2 = __builtin_fma(-(gd * l0[n]), rho[n], (f * l1[n]) * zh[n]);
                l0[n] = l1[n];
                l1[n] = l2;
            }
            v = vo;
            gd += f;
            f += 2.;
        };
#pragma unroll 1
        for (int left = p + 2 - m; left > 0; left -= 2) {
            const Pair o0 = o[0], o1 = o[1], t0 = t[0], t1 = t[1];
            step(o0, t0);
            step(o1, t1);
            o += 2;
            t += 2;
        }
#pragma unroll
        for (int n = 0; n < NP; n++) {
            out[n].p = __builtin_fma(C[n], F[n], __builtin_fma(S[n], G[n], out[n].p));
            out[n].z = __builtin_fma(C[n], Zc[n], __builtin_fma(S[n], Zs[n], out[n].z));
            w[n] = __builtin_fma(Cp[n], Tc[n], __builtin_fma(Sp[n], Ts[n], w[n]));
            const double mc = fm * Cp[n], ms = fm * Sp[n];
            tx[n] = __builtin_fma(mc, F[n], __builtin_fma(ms, G[n], tx[n]));
            ty[n] = __builtin_fma(mc, G[n], __builtin_fma(-ms, F[n], ty[n]));
            lm[n] = (__builtin_fma(2., fm, 1.) * lm[n]) * rho[n];
            Cp[n] = C[n];
            Sp[n] = S[n];
            C[n] = Cp[n] * x[n] - Sp[n] * y[n];
            S[n] = Cp[n] * y[n] + Sp[n] * x[n];
        }
        fm += 1.;
        below = m == 0 ? own : below + (P + kPad - m + 1);
        own += P + kPad - m;
    }
#pragma unroll
    for (int n = 0; n < NP; n++) {
        out[n].x = __builtin_fma(x[n], w[n], -tx[n]);
        out[n].y = __builtin_fma(y[n], w[n], -ty[n]);
    }
}

// the sums of one point: Kahan-compensated in FP64 passes, plain FP64 in mixed ones, as in the flat passes
template <bool MIXED>
struct Sums {
    double s0 = 0., s1 = 0., s2 = 0., s3 = 0.;
    double c0 = 0., c1 = 0., c2 = 0., c3 = 0.;
    __device__ __forceinline__ void add(const F4& v, double f, double fp)
    {
        if (MIXED) {
            s0 += v.x * f;
            s1 += v.y * f;
            s2 += v.z * f;
            s3 += v.p * fp;
        } else {
            dev::kahan_add(v.x, f, s0, c0);
            dev::kahan_add(v.y, f, s1, c1);
            dev::kahan_add(v.z, f, s2, c2);
            dev::kahan_add(v.p, fp, s3, c3);
        }
    }
};

// Ranges of a group's points that share a walk.  Usually the whole group; where the curve leaves the points' region and
// comes back, or leaps over a gap, the group is halved until its halves are alike (one not under 0.4 of the whole's
// radius) or hold kRangePoints, so that a few stray points do not blow up the sphere of all.  Record per
// range: centre, radius, first and end point in the group; an empty range ends the list.  SETS: the points lie in curve
// order within their charge-density sets, a range ends where the set changes, and its record holds the set too.
constexpr int kRangePoints = 16;
template <int NP, bool SETS>
struct Ranges {
    static constexpr int N = SETS ? 64 * NP : 64 * NP / kRangePoints;
    double v[N][SETS ? 7 : 6];
};
template <int NP, bool SETS>
__global__ __launch_bounds__(64) void k_tree_ranges(const double* __restrict__ px, const double* __restrict__ py,
                                                    const double* __restrict__ pz,
                                                    const int32_t* __restrict__ pset, int64_t npts,
                                                    Ranges<NP, SETS>* __restrict__ out)
{
    const int lane = threadIdx.x;
    const int64_t grp = blockIdx.x;
    double x[NP], y[NP], z[NP];
#pragma unroll
    for (int n = 0; n < NP; n++) {
        int64_t i = (grp * NP + n) * 64 + lane;
        if (i >= npts) i = npts - 1;
        x[n] = px[i];
        y[n] = py[i];
        z[n] = pz[i];
    }
    // A point with a coordinate that is not a number gives values that are not, whatever is summed, and is left out of
    // the spheres; an infinite coordinate, or a distance past the largest number, makes a range's radius infinite, so
    // that nothing is taken for it and its elements go pair by pair, as in the flat passes.
    bool some[NP];
#pragma unroll
    for (int n = 0; n < NP; n++) some[n] = x[n] == x[n] && y[n] == y[n] && z[n] == z[n];
    double c[3];
    auto sphere = [&](int a, int b) {
        double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        auto in = [&](int n) { return n * 64 + lane >= a && n * 64 + lane < b && some[n]; };
#pragma unroll
        for (int n = 0; n < NP; n++)
            if (in(n)) {
                lo[0] = fmin(lo[0], x[n]), lo[1] = fmin(lo[1], y[n]), lo[2] = fmin(lo[2], z[n]);
                hi[0] = fmax(hi[0], x[n]), hi[1] = fmax(hi[1], y[n]), hi[2] = fmax(hi[2], z[n]);
            }
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const double least = dev::wave_min(lo[k]), most = dev::wave_max(hi[k]);
            c[k] = least <= most ? 0.5 * (least + most) : 0.;  // no point but such: anything
        }
        double far = 0.;
#pragma unroll
        for (int n = 0; n < NP; n++)
            if (in(n)) {
                const double dx = x[n] - c[0], dy = y[n] - c[1], dz = z[n] - c[2];
                const double d2 = dx * dx + dy * dy + dz * dz;
                far = d2 == d2 ? fmax(far, d2) : INFINITY;
            }
        return dev::uniform(sqrt(dev::wave_max(far)));
    };
    int a = 0, len = 64 * NP, k = 0;
    Ranges<NP, SETS>* o = out + grp;
    auto set_of = [&](int at) {
        const int64_t i = grp * NP * 64 + at;
        return pset[i < npts ? i : npts - 1];
    };
    while (a < 64 * NP) {
        const int b = a + len;
        if (SETS && set_of(a) != set_of(b - 1)) {
            len /= 2;
            continue;
        }
        if (len > kRangePoints) {
            const double r1 = sphere(a, a + len / 2), r2 = sphere(a + len / 2, b);
            const double r = sphere(a, b);
            if (fmin(r1, r2) < 0.4 * r) {
                len /= 2;
                continue;
            }
        }
        const double r = sphere(a, b) * (1. + 1e-9) + 1e-12;  // padded against rounding
        if (lane == 0) {
            for (int q = 0; q < 3; q++) o->v[k][q] = c[q];
            o->v[k][3] = r;
            o->v[k][4] = a;
            o->v[k][5] = b;
            if constexpr (SETS) o->v[k][6] = set_of(a);
        }
        k++;
        a = b;
        len = a ? a & -a : len;
    }
    if (lane == 0 && k < Ranges<NP, SETS>::N) o->v[k][5] = 0.;
}

template <bool TRIANGLES>
__device__ __forceinline__ F4 near_pair(const double* __restrict__ g, double x, double y, double z)
{
    if (TRIANGLES) return dev::closed_form<3, true, true>(g, x, y, z);
    return dev::element_near<true>(g, (int)g[KG_TYPE], x, y, z);
}

constexpr int kTreeNeighbours = 8;
constexpr int kTreeWaves = 4;

// A wavefront's stack: 16 popped runs push at most 64, so each level adds at most 48 to the 64 of the first.
constexpr int kTreeStack = 64 + 48 * (KEM_TREE_LEVELS + 1);

// slices blocks of kTreeWaves wavefronts per group of 64 NP points (in curve order), each wavefront taking every
// nsplit-th item of the walk, nsplit = kTreeWaves slices.  A step of the walk tests up to 64 runs at once, a lane
// each (all of the top level, then the children of 16 opened runs): a run whose distance from the sphere around
// the points exceeds its near reach and serves an order is evaluated, others are opened, and at the lowest level
// their elements are evaluated pair by pair, near pairs by the closed forms (which the walk finds without a pass
// of their own).  The walk is the same for all of them, and the sums of a block's wavefronts are added in order
// through LDS.  A run's coefficients pass through LDS too; the other wavefronts of the SIMD cover the wait for
// them.  Three wavefronts per SIMD are asked for: a few registers spill, and the million mixed points over 20,000
// triangles take 18.8 ms instead of 22.2 at two, 100,000 in FP64 13.4 instead of 14.5.  Half expansions, half pairs close
// by.  The vector ALU issues in 84 % of the cycles for the million, which binds it; in 60 to 70 % in FP64, for 64 sets and
// for 400,000 points over 100,000 triangles, where chains of dependent FP64 operations and the loads of the coefficients
// are not covered by three wavefronts.
template <bool MIXED, int NP, bool TRIANGLES, bool SETS>
__global__ __launch_bounds__(64 * kTreeWaves) __attribute__((amdgpu_waves_per_eu(3))) void k_field_tree(
    const double* __restrict__ geom, const double* __restrict__ nodes, const float* __restrict__ nodes32,
    const float* __restrict__ far6, const double* __restrict__ far6_cl, const int32_t* __restrict__ order,
    const double* __restrict__ sigma, const double* __restrict__ tnode, const double* __restrict__ mom,
    const float* __restrict__ reach, TreeLevels T, int64_t nelem, const double* __restrict__ px,
    const double* __restrict__ py, const double* __restrict__ pz, const Ranges<NP, SETS>* __restrict__ ranges,
    int64_t npts, int64_t ngroups, int slices, double* __restrict__ out, int64_t comp_stride, int64_t mom_set,
    int64_t reach_set)
{
    using O = Orders<MIXED>;
    constexpr int E = entries(O::P);
    __shared__ int stacks[kTreeWaves][kTreeStack];
    __shared__ Pair cos[kTreeWaves][E];
    static_assert(sizeof(cos) >= (kTreeWaves - 1) * 4 * NP * 64 * sizeof(double), "the wavefronts' sums fit");
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int* st = stacks[wv];
    Pair* co = cos[wv];
    // consecutive blocks go to the 8 XCDs in turn: each XCD takes kTreeNeighbours groups of points at a time, whose
    // wavefronts read the same runs (a contiguous eighth of the points per XCD leaves the XCDs unequal work)
    const int64_t each = (int64_t)kTreeNeighbours * slices, turn8 = blockIdx.x >> 3;
    const int64_t task = (turn8 / each * 8 + (blockIdx.x & 7)) * each + turn8 % each;
    const int64_t grp = task / slices;
    const int slice = (int)(task - grp * slices);
    const int nsplit = slices * kTreeWaves, split = slice * kTreeWaves + wv;
    if (grp >= ngroups) return;
    double x[NP], y[NP], z[NP];
#pragma unroll
    for (int n = 0; n < NP; n++) {
        int64_t i = (grp * NP + n) * 64 + lane;
        if (i >= npts) i = npts - 1;
        x[n] = px[i];
        y[n] = py[i];
        z[n] = pz[i];
    }
    Sums<MIXED> sum[NP];
    int turn = 0;
    for (int range = 0; range < Ranges<NP, SETS>::N; range++) {
        const double* rg = ranges[grp].v[range];
        const int ra = (int)rg[4], rb = (int)rg[5];
        if (rb == 0) break;
        const double wx = rg[0], wy = rg[1], wz = rg[2], wr = rg[3];
        const double* sg = sigma;
        const double* ms = mom;
        const float* rs = reach - T.first[T.low];
        if constexpr (SETS) {
            const int64_t set = (int64_t)rg[6];
            sg += set * nelem;
            ms += set * mom_set;
            rs += set * reach_set;
        }
        bool in[NP];  // the lane's points that belong to the range
#pragma unroll
        for (int n = 0; n < NP; n++) in[n] = n * 64 + lane >= ra && n * 64 + lane < rb;
        int sp = 0;
        bool top = true;
        for (;;) {
            int lev, idx;
            bool have;
            if (top) {
                top = false;
                lev = T.levels - 1;
                idx = lane;
                have = lane < T.count[T.levels - 1];
            } else {
                if (sp == 0) break;
                const int k = sp < 16 ? sp : 16;
                sp -= k;
                have = (lane >> 2) < k;
                const int e = st[sp + (have ? lane >> 2 : 0)];
                lev = (e >> KEM_TREE_INDEX_BITS) - 1;
                idx = (e & ((1 << KEM_TREE_INDEX_BITS) - 1)) * KEM_TREE_FAN + (lane & 3);
                have = have && idx < T.count[lev];
            }
            const int at = have ? T.first[lev] + idx : T.first[T.low];  // a lane without a run reads the first one
            const double* t = tnode + (int64_t)at * KEM_TREE_STRIDE;
            const double dx = t[0] - wx, dy = t[1] - wy, dz = t[2] - wz;
            const double d = sqrt(dx * dx + dy * dy + dz * dz) * (1. - 1e-9) - wr;
            // the smallest order whose omitted terms stay below the tolerance (Orders), by fixed-point steps: the
            // factor before the power changes slowly with the order, and two steps leave 0.01 of one
            const float id = 1.f / (float)d, q = rs[at] * id, lg = __log2f(q);
            float need = O::log2_tol / lg - 1.f;
#pragma unroll
            for (int k = 0; k < 2; k++) need = (O::log2_tol - __log2f(need + 2.f - (need + 1.f) * q)) / lg - 1.f;
            const int ord = lg < -1.f && (float)t[3] * id < O::widest ? (int)ceilf(need) : O::P + 1;
            const bool take = have && d > t[4] && ord <= O::P;
            const bool open = have && !take && lev > T.low;
            const bool pairs = have && !take && lev == T.low;
            __builtin_amdgcn_wave_barrier();
            const unsigned long long om = __builtin_amdgcn_ballot_w64(open);
            if (open) st[sp + __builtin_popcountll(om & ((1ull << lane) - 1))] = (lev << KEM_TREE_INDEX_BITS) | idx;
            sp += __builtin_popcountll(om);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            unsigned long long items = __builtin_amdgcn_ballot_w64(take);
            // the lane of the next item that is this wavefront's, or -1
            auto next = [&]() {
                while (items) {
                    const int b = __builtin_ctzll(items);
                    items &= items - 1;
                    const bool mine = turn == split;
                    turn = turn + 1 == nsplit ? 0 : turn + 1;
                    if (mine) return b;
                }
                return -1;
            };
            int b;
            while ((b = next()) >= 0) {
                const int node = __builtin_amdgcn_readlane(at, b);
                const int p = max(1, __builtin_amdgcn_readlane(ord, b));
                const double* u = tnode + (int64_t)node * KEM_TREE_STRIDE;
                const Pair* src = reinterpret_cast<const Pair*>(ms) + (int64_t)(node - T.first[T.low]) * E;
                __builtin_amdgcn_wave_barrier();
                for (int k = lane; k < line_start(O::P, p + 2); k += 64) co[k] = src[k];
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                const double ia = u[5];
                double rx[NP], ry[NP], rz[NP];
#pragma unroll
                for (int n = 0; n < NP; n++) {
                    rx[n] = (x[n] - u[0]) * ia;
                    ry[n] = (y[n] - u[1]) * ia;
                    rz[n] = (z[n] - u[2]) * ia;
                }
                F4 v[NP];
                m2p<O::P, NP>(co, p, rx, ry, rz, v);
#pragma unroll
                for (int n = 0; n < NP; n++)
                    if (in[n]) sum[n].add(v[n], ia * ia, ia);
            }
            items = __builtin_amdgcn_ballot_w64(pairs);
            while ((b = next()) >= 0) {
                const int64_t k0 = (int64_t)__builtin_amdgcn_readlane(idx, b) * T.run;
                const int64_t k1 = k0 + T.run < nelem ? k0 + T.run : nelem;
                for (int64_t k = k0; k < k1; k++) {
                    const int64_t j = order[k];
                    const double* g = geom + j * KG_STRIDE;
                    if (!MIXED) {
                        const double sj = sg[j];
#pragma unroll
                        for (int n = 0; n < NP; n++) {
                            const double r2 = dev::dist2(g, x[n], y[n], z[n]);
                            if (!in[n]) continue;
                            F4 v;
                            if (dev::is_near2(g, r2, 0))
                                v = near_pair<TRIANGLES>(g, x[n], y[n], z[n]);
                            else
                                v = dev::element_far(g, nodes + j * KEM_NODE_STRIDE, (int)g[KG_TYPE], r2, x[n], y[n], z[n]);
                            sum[n].add(v, sj, sj);
                        }
                        continue;
                    }
                    const dev::v16f* rv = reinterpret_cast<const dev::v16f*>(far6 + k * KEM_FAR6_STRIDE);
                    const dev::v16f A = rv[0], B = rv[1];
                    const double cx = dev::f2d(B[8], B[9]), cy = dev::f2d(B[10], B[11]), cz = dev::f2d(B[12], B[13]);
                    const double sj = sg[j], wj = g[KG_PREF] * sj;
                    const double ux = wx - cx, uy = wy - cy, uz = wz - cz;
                    const double te = dev::f2d(B[14], B[15]) + wr;
                    const bool six = ux * ux + uy * uy + uz * uz > te * te;
                    // P - cluster centre in FP32; the far records hold the nodes so
                    const double* cl = far6_cl + KEM_FAR_CL_STRIDE * (k / KEM_CLUSTER);
#pragma unroll
                    for (int n = 0; n < NP; n++) {
                        if (!in[n]) continue;
                        float s0, s1, s2, s3;
                        if (six) {
                            const float ex = (float)(x[n] - cl[0]), ey = (float)(y[n] - cl[1]), ez = (float)(z[n] - cl[2]);
                            s0 = s1 = s2 = s3 = 0.f;
                            dev::node32(ex - A[0], ey - A[1], ez - A[2], dev::kW6a, s0, s1, s2, s3);
                            dev::node32(ex - A[4], ey - A[5], ez - A[6], dev::kW6a, s0, s1, s2, s3);
                            dev::node32(ex - A[8], ey - A[9], ez - A[10], dev::kW6a, s0, s1, s2, s3);
                            dev::node32(ex - A[12], ey - A[13], ez - A[14], dev::kW6b, s0, s1, s2, s3);
                            dev::node32(ex - B[0], ey - B[1], ez - B[2], dev::kW6b, s0, s1, s2, s3);
                            dev::node32(ex - B[4], ey - B[5], ez - B[6], dev::kW6b, s0, s1, s2, s3);
                        } else {
                            const double r2 = dev::dist2(g, x[n], y[n], z[n]);
                            if (dev::is_near2(g, r2, 0)) {
                                sum[n].add(near_pair<TRIANGLES>(g, x[n], y[n], z[n]), sj, sj);
                                continue;
                            }
                            const float ex = (float)(x[n] - g[KG_CX]), ey = (float)(y[n] - g[KG_CY]),
                                        ez = (float)(z[n] - g[KG_CZ]);
                            dev::element_far32_wave(g, nodes32 + j * KEM_NODE32_STRIDE, (int)g[KG_TYPE], r2, ex, ey, ez,
                                                    s0, s1, s2, s3);
                        }
                        sum[n].add(F4{(double)s0, (double)s1, (double)s2, (double)s3}, wj, wj);
                    }
                }
            }
        }
    }
    // the wavefronts' sums in order, through the LDS of the coefficients
    double* part = reinterpret_cast<double*>(cos);
    __syncthreads();
    if (wv > 0) {
#pragma unroll
        for (int n = 0; n < NP; n++) {
            double* q = part + ((wv - 1) * NP + n) * 256 + lane;
            q[0] = sum[n].s0;
            q[64] = sum[n].s1;
            q[128] = sum[n].s2;
            q[192] = sum[n].s3;
        }
    }
    __syncthreads();
    if (wv > 0) return;
#pragma unroll
    for (int n = 0; n < NP; n++) {
        for (int k = 0; k < kTreeWaves - 1; k++) {
            const double* q = part + (k * NP + n) * 256 + lane;
            sum[n].add(F4{q[0], q[64], q[128], q[192]}, 1., 1.);
        }
        const int64_t i = (grp * NP + n) * 64 + lane;
        if (i >= npts) continue;
        double* o = out + (int64_t)slice * npts + i;
        o[0] = sum[n].s0;
        o[comp_stride] = sum[n].s1;
        o[2 * comp_stride] = sum[n].s2;
        o[3 * comp_stride] = sum[n].s3;
    }
}

template <bool MIXED>
hipError_t tree_passes(hipStream_t st, const FieldMesh& m, const TreePlan& p, const double* sigma, const int32_t* pset,
                       const double* px, const double* py, const double* pz, int64_t npts, double* mom, double* ranges,
                       double* out, bool moments)
{
    constexpr int P = Orders<MIXED>::P;
    const TreeLevels& T = p.levels;
    const int64_t stride = 2 * entries(P);
    const int64_t base = T.first[T.low], mom_set = p.moments / p.sets;
    const int64_t runs = T.first[T.levels - 1] + T.count[T.levels - 1] - base;
    float* reach = reinterpret_cast<float*>(mom + p.moments);
    if (moments) {
        const double* low = m.tree + base * KEM_TREE_STRIDE;
        k_tree_reach<Orders<MIXED>::H><<<dim3((unsigned)runs, (unsigned)p.sets), kP2MBlock, 0, st>>>(
            m.geom, m.order, sigma, m.tree, T, m.n, reach, runs);
        if (pset)
            k_tree_p2m_sets<P><<<(unsigned)T.count[T.low], kP2MBlock, 0, st>>>(m.geom, m.nodes, m.order, sigma, p.sets,
                                                                              low, m.n, T.run, mom, mom_set);
        else
            k_tree_p2m<P><<<(unsigned)T.count[T.low], kP2MBlock, 0, st>>>(m.geom, m.nodes, m.order, sigma, low, m.n,
                                                                         T.run, mom);
        for (int k = T.low + 1; k < T.levels; k++)
            k_tree_m2m<P><<<dim3((unsigned)T.count[k], (unsigned)p.sets), 2 * kM2MGroup, 0, st>>>(
                m.tree + (int64_t)T.first[k - 1] * KEM_TREE_STRIDE, m.tree + (int64_t)T.first[k] * KEM_TREE_STRIDE,
                T.count[k - 1], mom + (T.first[k - 1] - base) * stride, mom + (T.first[k] - base) * stride, mom_set);
    }
    const int64_t groups = (npts + 64 * p.per_lane - 1) / (64 * p.per_lane);
    const int64_t unit = 8 * (int64_t)kTreeNeighbours * p.slices;
    const unsigned grid = (unsigned)((groups * p.slices + unit - 1) / unit * unit);
    auto launch = [&](auto np, auto sets) {
        constexpr int NP = decltype(np)::value;
        constexpr bool SETS = decltype(sets)::value;
        auto* rg = reinterpret_cast<Ranges<NP, SETS>*>(ranges);
        k_tree_ranges<NP, SETS><<<(unsigned)groups, 64, 0, st>>>(px, py, pz, pset, npts, rg);
        auto run = [&](auto triangles) {
            k_field_tree<MIXED, NP, decltype(triangles)::value, SETS><<<grid, 64 * kTreeWaves, 0, st>>>(
                m.geom, m.nodes, m.nodes32, m.far6, m.far6_cl, m.order, sigma, m.tree, mom, reach, T, m.n, px, py, pz, rg,
                npts, groups, p.slices, out, p.slices * npts, mom_set, runs);
        };
        if (m.triangles)
            run(std::true_type());
        else
            run(std::false_type());
    };
    if (pset)
        launch(std::integral_constant<int, 1>(), std::true_type());
    else if (p.per_lane == 2)
        launch(std::integral_constant<int, 2>(), std::false_type());
    else
        launch(std::integral_constant<int, 1>(), std::false_type());
    return hipGetLastError();
}

}  // namespace

// The hierarchical pass serves planar elements and wires under the numeric policy
// (in mixed precision without an FP64 band), at 4,096 points or more, which the caller has put in curve order.
// Below these sizes the flat pass is the faster one: its cost grows with elements times points, while here the
// expansions take 0.1 to 0.4 ms and a group's walk its elements close by.  Points in the gap of a closed surface (coax,
// bore) have many of those, points around a body few, so the line lies between the sizes where either gains.  Measured,
// us flat / hierarchical:
//   FP64   coax  5,000 x  8,192  1,468 / 1,673   10,000 x  8,192  2,953 / 2,471   20,000 x  4,096  3,291 / 3,977
//          coax  2,500 x 16,384  1,382 / 1,359    5,000 x 16,384  2,500 / 2,059   20,000 x 65,536 35,181 / 12,680
//          coax  1,000 x 131,072 3,249 / 3,400    1,600 x 32,768  1,543 / 1,764    1,600 x 131,072 5,077 / 4,942
//          cube  1,728 x 30,000  1,420 / 842      1,728 x 131,072 5,820 / 1,923
//   mixed  coax  5,000 x 20,000  1,042 / 1,243    5,000 x 65,536  2,159 / 2,272    5,000 x 131,072 4,017 / 3,360
//          coax  2,500 x 131,072 2,254 / 2,808    3,100 x 131,072 2,547 / 3,018   20,000 x 65,536  6,453 / 3,737
//          bore  5,000 x 131,072 3,781 / 4,677   10,000 x 33,000  2,706 / 2,055   30,000 x 33,000  5,425 / 2,781
//          cube  3,072 x 33,000    571 / 441      3,072 x 131,072 1,875 / 897
//          rectangles and wires  3,200 x 33,000  778 / 637   x 131,072  2,567 / 1,615
constexpr int64_t kTreeMinPoints = 4096;
inline bool tree_pays(bool mixed, double n, double m)
{
    if (mixed) return n >= 3000. && n * m >= 1e8;
    return n >= 1536. && (m >= 8192. ? n * m >= 5e7 : n * m >= 1.5e8);
}
// Points of several sets are visited set by set, so the groups are less compact the fewer points a set has, and each set
// has its expansions: the pass serves them from a product of elements and points per set on.  Measured on the coax, us
// flat / hierarchical (elements x points x sets, product per set):
//   FP64   6,000 x 80,000 x 16  3.0e7  13,101 / 11,503   x 32  1.5e7  13,110 / 13,104
//          20,000 x 80,000 x 64  2.5e7  41,728 / 39,288   20,000 x 300,000 x 64  9.4e7  148,520 / 75,234
//   mixed  20,000 x 80,000 x 8  2.0e8  7,903 / 6,352   x 16  1.0e8  7,835 / 8,596
//          20,000 x 160,000 x 16  2.0e8  13,728 / 11,543   x 32  1.0e8  14,448 / 15,346
//          12,000 x 80,000 x 4  2.4e8  5,072 / 4,422   x 8  1.2e8  5,038 / 5,081
//          6,000 x 160,000 x 4  2.4e8  5,061 / 4,989   x 8  1.2e8  5,100 / 5,895
//          and with 300,000 points, where the sides meet lower:
//          20,000 x 32  1.9e8  25,841 / 19,989   x 64  9.4e7  36,158 / 26,060   12,000 x 32  1.1e8  17,160 / 15,845
//          x 64  5.6e7  22,557 / 20,036   6,000 x 8  2.2e8  9,468 / 8,402   x 16  1.1e8  9,449 / 9,644
// (the flat pass's own times rise with elements x sets: its weights, 6 and 10 MB for 64 sets of 12,000 and 20,000
// elements, no longer fit an XCD's 4 MB of L2).
constexpr int64_t kTreeMaxSets = 65535;
inline bool sets_pay(bool mixed, double n, double m, double nsets)
{
    const double each = n * m / nsets;
    return mixed ? each >= (m >= 262144. && n >= 6000. ? 9e7 : 1.9e8) : each >= 3.5e7;
}
// wavefronts in all: kTreeWaves times p.slices of them per group of points.  Many more than the chip holds at once, since
// groups differ in their work, a few by 10 times (400,000 points over 100,000 triangles: 15.5 ms at 8 per group,
// 11.3 at 16, 9.3 at 32, 8.8 at the 40 that this gives, 8.4 at 64; a million points over 20,000: 21.0 at 8, 18.8 at the 16
// that this gives, 19.2 at 32, 21.3 at 64).
constexpr int64_t kTreeWavefronts = 131072;
constexpr int kTreeMaxSlices = 16;
// From this many points on, two per lane; below, groups of 64 points are the more compact ones (20,000-triangle coax,
// mixed: 16,384 points 2.41 ms with two, 1.98 with one; 65,536 points 4.27 and 3.72; 131,072 points 4.90 and 5.00).
constexpr int64_t kTreePairPoints = 65537;
// Expansions of calls that the no-allocation entry point may serve (up to 65,536 points) fit its scratch beside
// the points' ordering, partial sums and the group members' charge densities; other calls' are bounded by 4 GiB.  Runs of
// the lowest level grow until they do: from 33,000 elements on in FP64, 58,000 in mixed precision.  The entry points that
// allocate keep to the same sizes at these points, as their results are the same bit for bit.
constexpr int64_t kTreeSmallPoints = 65536;
constexpr int64_t kTreeSmallDoubles = (int64_t)7 << 19, kTreeSmallPartials = (int64_t)3 << 19;
constexpr int64_t kTreeLargeDoubles = (int64_t)512 << 20;
// partial sums of one chunk of points
constexpr int64_t kTreePartialDoubles = (int64_t)128 << 20;

TreePlan plan_tree(int policy, const FieldMesh& m, bool mixed, double fp64_ratio, bool multi, int64_t nsets,
                   int64_t npts)
{
    TreePlan p;
    if (policy != 0 || m.axisym || !m.tree || !m.order || !m.clusters) return p;
    if (mixed && (fp64_ratio != 0. || !m.nodes32 || !m.far6 || !m.far6_cl)) return p;
    if (npts < kTreeMinPoints || !tree_pays(mixed, (double)m.n, (double)npts) || npts > INT32_MAX ||
        m.n > ((int64_t)1 << KEM_TREE_INDEX_BITS))
        return p;
    if (multi && (nsets > kTreeMaxSets || !sets_pay(mixed, (double)m.n, (double)npts, (double)nsets))) return p;
    p.sets = multi ? nsets : 1;
    TreeLevels& T = p.levels;
    tree_levels(m.n, T);
    const int P = mixed ? Orders<true>::P : Orders<false>::P;
    const int64_t limit = !multi && npts <= kTreeSmallPoints ? kTreeSmallDoubles - m.n : kTreeLargeDoubles;
    const int64_t total = T.first[T.levels - 1] + T.count[T.levels - 1];
    for (T.low = 0; T.low < T.levels; T.low++) {
        p.moments = p.sets * (total - T.first[T.low]) * 2 * entries(P);
        if (p.moments <= limit) break;
    }
    if (T.low >= T.levels) return TreePlan();
    p.reach = (p.sets * (total - T.first[T.low]) + 1) / 2;
    T.run = KEM_TREE_LEAF;
    for (int k = 0; k < T.low; k++) T.run *= KEM_TREE_FAN;
    p.per_lane = !multi && npts >= kTreePairPoints ? 2 : 1;
    const int64_t groups = (npts + 64 * p.per_lane - 1) / (64 * p.per_lane);
    int64_t slices =
        std::min<int64_t>(kTreeMaxSlices, std::max<int64_t>(1, kTreeWavefronts / (kTreeWaves * groups)));
    if (!multi && npts <= kTreeSmallPoints) slices = std::min(slices, kTreeSmallPartials / (4 * npts));
    p.slices = (int)slices;
    const int64_t unit = 64 * p.per_lane;
    p.chunk = std::min(npts, kTreePartialDoubles / (4 * slices) / unit * unit);
    p.partials = 4 * slices * p.chunk;
    p.ranges = (p.chunk + unit - 1) / unit * (multi ? sizeof(Ranges<1, true>) : p.per_lane == 2 ? sizeof(Ranges<2, false>) : sizeof(Ranges<1, false>)) /
               sizeof(double);
    p.use = true;
    return p;
}

hipError_t launch_tree(hipStream_t st, const FieldMesh& m, const TreePlan& p, bool mixed, const double* sigma,
                       const int32_t* pset, const double* px, const double* py, const double* pz, int64_t npts,
                       double* mom, double* ranges, double* out, bool moments)
{
    if (npts <= 0) return hipSuccess;
    return mixed ? tree_passes<true>(st, m, p, sigma, pset, px, py, pz, npts, mom, ranges, out, moments)
                 : tree_passes<false>(st, m, p, sigma, pset, px, py, pz, npts, mom, ranges, out, moments);
}

}  // namespace kem
