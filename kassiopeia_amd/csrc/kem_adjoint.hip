// kem_adjoint.hip -- derivatives of the BEM path with respect to the triangle vertices (no
// reference counterpart: KEMField has no adjoint).
//
// Two vector-Jacobian products, both under the numeric integrator policy with the quadrature
// regime of every pair frozen at the one the forward pass used:
//   field term   d/dV of  sum_k g_k phi(P_k) = sum_k g_k sum_j G(P_k; T_j) sigma_j  (and d/dsigma)
//   matrix term  d/dV of  sum_ij w_i A_ij u_j  with A_ij = G(c_i; T_j), c_i the centroid of T_i
// G(P; T) is the potential of triangle T carrying unit charge density.  For a cubature pair
// (numeric rule with nodes Q_q = sum_m beta_qm v_m, weights w_q, prefactor K * area):
//   dG/dv_m = K (d area/dv_m) S + K area sum_q w_q beta_qm (P - Q_q)/R_q^3,  S = sum_q w_q / R_q
//   dG/dP   = -K area sum_q w_q (P - Q_q)/R_q^3
// with d area/dv_0 = n x (v_2 - v_1)/2 and cyclic.  A closed-form (near) pair is differentiated
// by forward-mode dual numbers through the closed-form potential
//   G = K (sum_e t_e ln((R_b + l_b)/(R_a + l_a)) + h Omega)
// (t_e: distance of P's projection to edge e, l: positions of the edge ends along it, h:
// height over the plane, Omega: Van Oosterom-Strackee solid angle).  Near pairs run in kernels
// of their own, so the register footprint of the dual numbers stays out of the far kernels.
//
// Layouts: one lane per source element j (its vertices and accumulators in registers), the
// points / targets wave-uniform.  Element gradients are per element and vertex corner:
// dvert[j*9 + 3*m + c] = d/d(v_m)_c, v_0 = P0, v_1 = P0 + A N1, v_2 = P0 + B N2 of its record.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "kem_device.hpp"
#include "kem_kernels.h"

namespace kem {
namespace {

constexpr int kBlock = 256;
constexpr int kChunk = 64;  // targets per LDS reduction round

inline unsigned nblocks(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

// ------------------------------------------------------------------ dual numbers
template <int N>
struct Dual {
    double v;
    double d[N];
};

template <int N>
__device__ __forceinline__ Dual<N> cst(double a)
{
    Dual<N> r;
    r.v = a;
    for (int k = 0; k < N; k++) r.d[k] = 0.;
    return r;
}
template <int N>
__device__ __forceinline__ Dual<N> operator+(const Dual<N>& a, const Dual<N>& b)
{
    Dual<N> r;
    r.v = a.v + b.v;
    for (int k = 0; k < N; k++) r.d[k] = a.d[k] + b.d[k];
    return r;
}
template <int N>
__device__ __forceinline__ Dual<N> operator-(const Dual<N>& a, const Dual<N>& b)
{
    Dual<N> r;
    r.v = a.v - b.v;
    for (int k = 0; k < N; k++) r.d[k] = a.d[k] - b.d[k];
    return r;
}
template <int N>
__device__ __forceinline__ Dual<N> operator*(const Dual<N>& a, const Dual<N>& b)
{
    Dual<N> r;
    r.v = a.v * b.v;
    for (int k = 0; k < N; k++) r.d[k] = a.d[k] * b.v + a.v * b.d[k];
    return r;
}
template <int N>
__device__ __forceinline__ Dual<N> operator*(double s, const Dual<N>& a)
{
    Dual<N> r;
    r.v = s * a.v;
    for (int k = 0; k < N; k++) r.d[k] = s * a.d[k];
    return r;
}
template <int N>
__device__ __forceinline__ Dual<N> operator/(const Dual<N>& a, const Dual<N>& b)
{
    Dual<N> r;
    const double ib = 1. / b.v;
    r.v = a.v * ib;
    for (int k = 0; k < N; k++) r.d[k] = (a.d[k] - r.v * b.d[k]) * ib;
    return r;
}
template <int N>
__device__ __forceinline__ Dual<N> dsqrt(const Dual<N>& a)
{
    Dual<N> r;
    r.v = sqrt(a.v);
    const double f = 0.5 / r.v;
    for (int k = 0; k < N; k++) r.d[k] = f * a.d[k];
    return r;
}
template <int N>
__device__ __forceinline__ Dual<N> dlog(const Dual<N>& a)
{
    Dual<N> r;
    r.v = log(a.v);
    const double f = 1. / a.v;
    for (int k = 0; k < N; k++) r.d[k] = f * a.d[k];
    return r;
}
template <int N>
__device__ __forceinline__ Dual<N> datan2(const Dual<N>& y, const Dual<N>& x)
{
    Dual<N> r;
    r.v = atan2(y.v, x.v);
    const double f = 1. / (x.v * x.v + y.v * y.v);
    for (int k = 0; k < N; k++) r.d[k] = (x.v * y.d[k] - y.v * x.d[k]) * f;
    return r;
}

template <class S>
__device__ __forceinline__ S dot3(const S* a, const S* b)
{
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}
template <class S>
__device__ __forceinline__ void cross3(const S* a, const S* b, S* c)
{
    c[0] = a[1] * b[2] - a[2] * b[1];
    c[1] = a[2] * b[0] - a[0] * b[2];
    c[2] = a[0] * b[1] - a[1] * b[0];
}

// Closed-form potential of triangle V (unit charge density) at P.  The edge terms keep their
// t-derivative when P's projection lies on an edge line (t_e = 0, log finite); only a point on
// the line beyond an edge end, where the logarithm diverges, drops the (vanishing) term.
template <int N>
__device__ Dual<N> tri_potential_cf(const Dual<N>* P, const Dual<N> (*V)[3])
{
    Dual<N> e1[3], e2[3], nr[3], n[3], r[3][3], R[3];
    for (int k = 0; k < 3; k++) {
        e1[k] = V[1][k] - V[0][k];
        e2[k] = V[2][k] - V[0][k];
    }
    cross3(e1, e2, nr);
    const Dual<N> nn = dsqrt(dot3(nr, nr));
    for (int k = 0; k < 3; k++) n[k] = nr[k] / nn;
    for (int m = 0; m < 3; m++) {
        for (int k = 0; k < 3; k++) r[m][k] = V[m][k] - P[k];
        R[m] = dsqrt(dot3(r[m], r[m]));
    }
    const Dual<N> h = cst<N>(0.) - dot3(n, r[0]);
    Dual<N> sum = cst<N>(0.);
    for (int e = 0; e < 3; e++) {
        const int a = e, b = (e + 1) % 3;
        Dual<N> ed[3], u[3], mv[3];
        for (int k = 0; k < 3; k++) ed[k] = V[b][k] - V[a][k];
        const Dual<N> L = dsqrt(dot3(ed, ed));
        for (int k = 0; k < 3; k++) u[k] = ed[k] / L;
        cross3(u, n, mv);
        const Dual<N> t = dot3(mv, r[a]);
        const Dual<N> la = dot3(u, r[a]), lb = dot3(u, r[b]);
        // R + l without cancellation: for l < 0, R + l = rho^2 / (R - l) with rho^2 = t^2 + h^2
        // the squared distance of P from the edge line
        const Dual<N> rho2 = t * t + h * h;
        const Dual<N> fa = la.v >= 0. ? R[a] + la : rho2 / (R[a] - la);
        const Dual<N> fb = lb.v >= 0. ? R[b] + lb : rho2 / (R[b] - lb);
        // P on the edge line beyond an end: the term and its limit vanish (t = 0)
        if (!(fa.v > 1e-300) || !(fb.v > 1e-300)) continue;
        sum = sum + t * dlog(fb / fa);
    }
    Dual<N> c12[3];
    cross3(r[1], r[2], c12);
    const Dual<N> trip = dot3(r[0], c12);
    const Dual<N> den = R[0] * R[1] * R[2] + dot3(r[0], r[1]) * R[2] + dot3(r[0], r[2]) * R[1] +
                        dot3(r[1], r[2]) * R[0];
    const Dual<N> om = 2. * datan2(trip, den);
    return dev::kK * (sum + h * om);
}

// ------------------------------------------------------------------ per-element lane state
struct Elem {
    double v[3][3];   // vertices
    double da[3][3];  // K d(area)/dv_m
    double pref;      // K area
    double sig;       // charge density
    bool tri;
};

__device__ __forceinline__ void load_elem(const double* __restrict__ g, double sig, Elem& E)
{
    E.tri = (int)g[KG_TYPE] == KEM_TRIANGLE;
    for (int m = 0; m < 3; m++)
        for (int c = 0; c < 3; c++) E.v[m][c] = g[KG_V + 3 * m + c];
    const double n[3] = {g[KG_NX], g[KG_NY], g[KG_NZ]};
    for (int m = 0; m < 3; m++) {
        // n x (v_{m+2} - v_{m+1}) / 2: the opposite edge, cyclic
        const int p = (m + 1) % 3, q = (m + 2) % 3;
        const double ed[3] = {E.v[q][0] - E.v[p][0], E.v[q][1] - E.v[p][1], E.v[q][2] - E.v[p][2]};
        double c[3];
        cross3(n, ed, c);
        for (int k = 0; k < 3; k++) E.da[m][k] = 0.5 * dev::kK * c[k];
    }
    E.pref = g[KG_PREF];
    E.sig = sig;
}

// cubature derivatives of one far pair: value G, dG/dv (9), dG/dP (3)
__device__ __forceinline__ void far_derivs(const Elem& E, const double* __restrict__ rule, int slot0, int nq,
                                           double px, double py, double pz, double& G, double* dv, double* dP)
{
    double S = 0., F[3][3] = {{0., 0., 0.}, {0., 0., 0.}, {0., 0., 0.}};
    for (int q = 0; q < nq; q++) {
        const double* t = rule + 4 * (slot0 + q);
        const double b0 = t[0], b1 = t[1], b2 = t[2], w = t[3];
        const double qx = b0 * E.v[0][0] + b1 * E.v[1][0] + b2 * E.v[2][0];
        const double qy = b0 * E.v[0][1] + b1 * E.v[1][1] + b2 * E.v[2][1];
        const double qz = b0 * E.v[0][2] + b1 * E.v[1][2] + b2 * E.v[2][2];
        const double rx = px - qx, ry = py - qy, rz = pz - qz;
        const double ir = dev::rsqrt_acc(rx * rx + ry * ry + rz * rz);
        S += w * ir;
        const double t3 = w * ir * ir * ir;
        const double bb[3] = {b0, b1, b2};
        for (int m = 0; m < 3; m++) {
            const double s = t3 * bb[m];
            F[m][0] += s * rx;
            F[m][1] += s * ry;
            F[m][2] += s * rz;
        }
    }
    G = E.pref * S;
    for (int m = 0; m < 3; m++)
        for (int c = 0; c < 3; c++) dv[3 * m + c] = E.da[m][c] * S + E.pref * F[m][c];
    for (int c = 0; c < 3; c++) dP[c] = -E.pref * (F[0][c] + F[1][c] + F[2][c]);
}

// regime of a triangle pair as the forward assembly / pair evaluation chooses it (element_eval)
__device__ __forceinline__ int tri_regime(const double* __restrict__ g, double px, double py, double pz)
{
    const double dr = dev::distance_ratio(g, px, py, pz);
    if (dr > dev::kTriCub12) return 7;
    if (dr > dev::kTriCub33) return 12;
    if (dr > dev::kTriRWG) return 33;
    return 0;
}

// regime of a triangle pair as the forward field pass chooses it (squared thresholds)
__device__ __forceinline__ int tri_regime_field(const double* __restrict__ g, double px, double py, double pz)
{
    const double r2 = dev::dist2(g, px, py, pz);
    if (!(r2 > g[KG_NEAR2])) return 0;
    if (r2 > g[KG_REF7_2]) return 7;
    if (r2 > g[KG_REF12_2]) return 12;
    return 33;
}

__device__ __forceinline__ int rule_slot(int nq) { return nq == 7 ? KEM_N7 : nq == 12 ? KEM_N12 : KEM_N33; }

__device__ __forceinline__ double wave_sum(double v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// ------------------------------------------------------------------ field term
// Far pairs of the field term: partV[s][j][10] = (sum_k g_k G_kj, sum_k g_k sigma_j dG_kj/dv) over the points of
// split s.  Lane = element; the four wavefronts of a block share 64 elements and take chunk <= 64 points of the split at
// a time.  The sums over points are linear in the nodes' own sums A_q = sum_k g_k / R_kq and B_q = sum_k g_k r_kq /
// R_kq^3, so a wavefront runs over the points inside and over the nodes outside: a pair costs 22 operations a
// node, and the node's position and the nine derivatives are formed once per 64 points.  Bound by FP64 issue: 1.24 ms
// for 5,000 elements and 10,000 points, 2.36 ms with the nodes inside (36 operations a node and each lane its own
// rule).  All lanes take the rule with the most nodes that any of them needs for a point, as in the assembly; the
// points are put in LDS by rule.  Near pairs are left out, and near[group * splits + s] says whether there were any,
// so that k_vjp_field_near passes over the others (32 us where there are few, 230 us with its own test of each pair).
constexpr int kVjpWaves = 4;
__global__ __launch_bounds__(64 * kVjpWaves) void k_vjp_field_far(const double* __restrict__ geom,
                                                                  const double* __restrict__ sigma,
                                                                  const double* __restrict__ rule, int64_t n,
                                                                  const double* __restrict__ pts,
                                                                  const double* __restrict__ gk, int64_t npts,
                                                                  int64_t per_split, int chunk,
                                                                  double* __restrict__ partV,
                                                                  int* __restrict__ near)
{
    __shared__ double4 lp[kVjpWaves][64];
    __shared__ int lk[kVjpWaves][64];
    __shared__ double part[kVjpWaves - 1][10][64];
    __shared__ int s_near[kVjpWaves];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int64_t j = (int64_t)blockIdx.x * 64 + lane;
    const bool live = j < n;
    if (!live) j = n - 1;
    const double* g = geom + j * KG_STRIDE;
    Elem E;
    load_elem(g, sigma[j], E);
    const double cx = g[KG_CX], cy = g[KG_CY], cz = g[KG_CZ];
    const double near2 = g[KG_NEAR2], ref7 = g[KG_REF7_2], ref12 = g[KG_REF12_2];
    const bool act = live && E.tri;
    const int64_t k0 = (int64_t)blockIdx.y * per_split;
    const int64_t k1 = std::min<int64_t>(npts, k0 + per_split);
    double4* P = lp[wv];
    int* K = lk[wv];
    double S = 0., F[3][3] = {{0., 0., 0.}, {0., 0., 0.}, {0., 0., 0.}};
    bool any_near = false;
    for (int64_t c0 = k0 + chunk * wv; c0 < k1; c0 += chunk * kVjpWaves) {
        const int cnt = (int)std::min<int64_t>(chunk, k1 - c0);
        const int64_t kl = c0 + std::min(lane, cnt - 1);
        const double4 mine{pts[3 * kl], pts[3 * kl + 1], pts[3 * kl + 2], gk[kl]};
        // the rule that the wavefront takes for each point (lane k keeps point k's), and the lane's near pairs
        int code = 0;
        unsigned long long mask = 0;
        for (int k = 0; k < cnt; k++) {
            auto lane_of = [k](double v) {
                return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), k),
                                        __builtin_amdgcn_readlane(__double2loint(v), k));
            };
            // dist2's operations, so the same pairs are near as in the forward pass
            const double dx = cx - lane_of(mine.x), dy = cy - lane_of(mine.y), dz = cz - lane_of(mine.z);
            const double r2 = __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
            const bool isnear = !(r2 > near2), far = act && !isnear;
            if (isnear) mask |= 1ull << k;
            const int c = __builtin_amdgcn_ballot_w64(far && !(r2 > ref12)) != 0  ? 3
                          : __builtin_amdgcn_ballot_w64(far && !(r2 > ref7)) != 0 ? 2
                          : __builtin_amdgcn_ballot_w64(far) != 0                 ? 1
                                                                                  : 0;
            if (lane == k) code = c;
        }
        const bool some = __builtin_amdgcn_ballot_w64(act && mask != 0) != 0;
        any_near = any_near || some;
        __builtin_amdgcn_wave_barrier();
        int at = 0;
        int start[4];
#pragma unroll
        for (int c = 1; c <= 3; c++) {
            const unsigned long long m = __builtin_amdgcn_ballot_w64(code == c);
            start[c - 1] = at;
            if (code == c) {
                const int to = at + __builtin_popcountll(m & ((1ull << lane) - 1));
                P[to] = mine;
                K[to] = lane;
            }
            at += __builtin_popcountll(m);
        }
        start[3] = at;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll 1
        for (int c = 0; c < 3; c++) {
            const int i0 = c == 0 ? start[0] : c == 1 ? start[1] : start[2];
            const int i1 = c == 0 ? start[1] : c == 1 ? start[2] : start[3];
            if (i0 == i1) continue;
            const int nq = c == 0 ? 7 : c == 1 ? 12 : 33;
            const double* t = rule + 4 * rule_slot(nq);
            // two nodes at a time share the points' reads; the last of an odd rule runs beside itself with weight 0
#pragma unroll 1
            for (int q = 0; q < nq; q += 2) {
                double bq[2][3], w[2], x[2], y[2], z[2], A[2], Bx[2], By[2], Bz[2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const double* r = t + 4 * std::min(q + h, nq - 1);
                    for (int m = 0; m < 3; m++) bq[h][m] = r[m];
                    w[h] = q + h < nq ? r[3] : 0.;
                    x[h] = bq[h][0] * E.v[0][0] + bq[h][1] * E.v[1][0] + bq[h][2] * E.v[2][0];
                    y[h] = bq[h][0] * E.v[0][1] + bq[h][1] * E.v[1][1] + bq[h][2] * E.v[2][1];
                    z[h] = bq[h][0] * E.v[0][2] + bq[h][1] * E.v[1][2] + bq[h][2] * E.v[2][2];
                    A[h] = Bx[h] = By[h] = Bz[h] = 0.;
                }
                for (int i = i0; i < i1; i++) {
                    const double4 p = P[i];
                    const bool skip = some && ((mask >> K[i]) & 1);
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const double rx = p.x - x[h], ry = p.y - y[h], rz = p.z - z[h];
                        double ir = dev::rsqrt_acc(rx * rx + ry * ry + rz * rz);
                        if (skip) ir = 0.;
                        const double a = p.w * ir;
                        const double f = a * ir * ir;
                        A[h] += a;
                        Bx[h] = __builtin_fma(f, rx, Bx[h]);
                        By[h] = __builtin_fma(f, ry, By[h]);
                        Bz[h] = __builtin_fma(f, rz, Bz[h]);
                    }
                }
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    S = __builtin_fma(w[h], A[h], S);
                    for (int m = 0; m < 3; m++) {
                        const double wb = w[h] * bq[h][m];
                        F[m][0] = __builtin_fma(wb, Bx[h], F[m][0]);
                        F[m][1] = __builtin_fma(wb, By[h], F[m][1]);
                        F[m][2] = __builtin_fma(wb, Bz[h], F[m][2]);
                    }
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    // the wavefronts' sums in order
    if (lane == 0) s_near[wv] = any_near;
    if (wv > 0) {
        part[wv - 1][0][lane] = S;
        for (int c = 0; c < 9; c++) part[wv - 1][1 + c][lane] = F[c / 3][c % 3];
    }
    __syncthreads();
    if (wv > 0) return;
    for (int k = 0; k < kVjpWaves - 1; k++) {
        S += part[k][0][lane];
        for (int c = 0; c < 9; c++) F[c / 3][c % 3] += part[k][1 + c][lane];
    }
    if (lane == 0) near[(int64_t)blockIdx.x * gridDim.y + blockIdx.y] = s_near[0] | s_near[1] | s_near[2] | s_near[3];
    if (!live) return;
    double* out = partV + ((int64_t)blockIdx.y * n + j) * 10;
    out[0] = act ? E.pref * S : 0.;
    for (int m = 0; m < 3; m++)
        for (int c = 0; c < 3; c++)
            out[1 + 3 * m + c] = act ? E.sig * (E.da[m][c] * S + E.pref * F[m][c]) : 0.;
}

// Near pairs of the field term, added to k_vjp_field_far's sums where it saw any.  Each wavefront takes a quarter of the
// split's points for the block's 64 elements: one closed-form derivative is thousands of operations, so a block's
// time is that of its longest run of them.
__global__ __launch_bounds__(64 * kVjpWaves) void k_vjp_field_near(const double* __restrict__ geom,
                                                                   const double* __restrict__ sigma, int64_t n,
                                                                   const double* __restrict__ pts,
                                                                   const double* __restrict__ gk, int64_t npts,
                                                                   int64_t per_split, double* __restrict__ partV,
                                                                   const int* __restrict__ near)
{
    if (!near[(int64_t)blockIdx.x * gridDim.y + blockIdx.y]) return;
    __shared__ double part[kVjpWaves - 1][10][64];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int64_t j = (int64_t)blockIdx.x * 64 + lane;
    const bool live = j < n;
    if (!live) j = n - 1;
    const double* g = geom + j * KG_STRIDE;
    Elem E;
    load_elem(g, sigma[j], E);
    const int64_t quarter = (per_split + kVjpWaves - 1) / kVjpWaves;
    const int64_t end = std::min<int64_t>(npts, (blockIdx.y + 1) * per_split);
    const int64_t k0 = std::min<int64_t>(end, blockIdx.y * per_split + wv * quarter);
    const int64_t k1 = std::min<int64_t>(end, k0 + quarter);
    double acc[10];
    for (int c = 0; c < 10; c++) acc[c] = 0.;
    for (int64_t k = k0; k < k1; k++) {
        const double px = pts[3 * k], py = pts[3 * k + 1], pz = pts[3 * k + 2], wk = gk[k];
        if (!live || !E.tri || tri_regime_field(g, px, py, pz) != 0) continue;
        Dual<9> V[3][3], P[3];
        for (int m = 0; m < 3; m++)
            for (int c = 0; c < 3; c++) {
                V[m][c] = cst<9>(E.v[m][c]);
                V[m][c].d[3 * m + c] = 1.;
            }
        P[0] = cst<9>(px);
        P[1] = cst<9>(py);
        P[2] = cst<9>(pz);
        const Dual<9> G = tri_potential_cf<9>(P, V);
        acc[0] += wk * G.v;
        const double ws = wk * E.sig;
        for (int c = 0; c < 9; c++) acc[1 + c] += ws * G.d[c];
    }
    if (wv > 0)
        for (int c = 0; c < 10; c++) part[wv - 1][c][lane] = acc[c];
    __syncthreads();
    if (wv > 0 || !live || !E.tri) return;
    double* out = partV + ((int64_t)blockIdx.y * n + j) * 10;
    for (int c = 0; c < 10; c++) {
        double v = out[c] + acc[c];
        for (int k = 0; k < kVjpWaves - 1; k++) v += part[k][c][lane];
        out[c] = v;
    }
}

// ------------------------------------------------------------------ matrix term
// lanes: sources j; targets i of split blockIdx.y, wave-uniform.  Weight w_ij = lw_i * u_j.
// partV[s][j][1..9] += sum_i w_ij dA_ij/dv_j;  partP[bx][i][3] (+)= sum_{j in block} w_ij dA_ij/dc_i
template <bool NEAR>
__global__ __launch_bounds__(kBlock) void k_vjp_matrix(const double* __restrict__ geom,
                                                       const double* __restrict__ targets,
                                                       const double* __restrict__ rule, int64_t n,
                                                       const double* __restrict__ lw, const double* __restrict__ u,
                                                       int64_t per_split, double* __restrict__ partV,
                                                       double* __restrict__ partP)
{
    __shared__ double sh[kBlock / 64][kChunk][3];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t jr = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const bool live = jr < n;
    const int64_t j = live ? jr : n - 1;
    const double* g = geom + j * KG_STRIDE;
    Elem E;
    load_elem(g, live ? u[j] : 0., E);
    const bool act = live && E.tri;
    const int64_t i0 = (int64_t)blockIdx.y * per_split;
    const int64_t i1 = std::min<int64_t>(n, i0 + per_split);
    double acc[9];
    double* outV = partV + ((int64_t)blockIdx.y * n + j) * 10;
    for (int c = 0; c < 9; c++) acc[c] = (NEAR && live) ? outV[1 + c] : 0.;
    for (int64_t ib = i0; ib < i1; ib += kChunk) {
        const int cnt = (int)std::min<int64_t>(kChunk, i1 - ib);
        for (int ii = 0; ii < cnt; ii++) {
            const int64_t i = ib + ii;
            const double* t = targets + i * KT_STRIDE;
            const double px = t[KT_CX], py = t[KT_CY], pz = t[KT_CZ];
            const double w = lw[i] * E.sig;
            double gp[3] = {0., 0., 0.};
            const int reg = act ? tri_regime(g, px, py, pz) : -1;
            if (NEAR) {
                if (reg == 0) {
                    Dual<12> V[3][3], P[3];
                    for (int m = 0; m < 3; m++)
                        for (int c = 0; c < 3; c++) {
                            V[m][c] = cst<12>(E.v[m][c]);
                            V[m][c].d[3 * m + c] = 1.;
                        }
                    const double pc[3] = {px, py, pz};
                    for (int c = 0; c < 3; c++) {
                        P[c] = cst<12>(pc[c]);
                        P[c].d[9 + c] = 1.;
                    }
                    const Dual<12> G = tri_potential_cf<12>(P, V);
                    for (int c = 0; c < 9; c++) acc[c] += w * G.d[c];
                    for (int c = 0; c < 3; c++) gp[c] = w * G.d[9 + c];
                }
            } else if (reg > 0) {
                double G, dv[9], dP[3];
                far_derivs(E, rule, rule_slot(reg), reg, px, py, pz, G, dv, dP);
                for (int c = 0; c < 9; c++) acc[c] += w * dv[c];
                for (int c = 0; c < 3; c++) gp[c] = w * dP[c];
            }
            for (int c = 0; c < 3; c++) {
                const double s = wave_sum(gp[c]);
                if (lane == 0) sh[wave][ii][c] = s;
            }
        }
        __syncthreads();
        for (int e = threadIdx.x; e < cnt * 3; e += kBlock) {
            const int ii = e / 3, c = e % 3;
            const double s = ((sh[0][ii][c] + sh[1][ii][c]) + sh[2][ii][c]) + sh[3][ii][c];
            double* dst = partP + ((int64_t)blockIdx.x * n + ib + ii) * 3 + c;
            *dst = NEAR ? *dst + s : s;
        }
        __syncthreads();
    }
    if (live)
        for (int c = 0; c < 9; c++) outV[1 + c] = acc[c];
}

// dsig[j] = sum_s partV[s][j][0];  dvert[j*9 + c] = sum_s partV[s][j][1 + c]
__global__ __launch_bounds__(kBlock) void k_vjp_reduce_v(const double* __restrict__ partV, int nsplit, int64_t n,
                                                         double* __restrict__ dsig, double* __restrict__ dvert)
{
    // blockIdx.y = component; the loads of eight splits in flight
    const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const int c = blockIdx.y;
    if (j >= n || (c == 0 && !dsig)) return;
    const double* p = partV + j * 10 + c;
    double s = 0.;
    int k = 0;
    for (; k + 8 <= nsplit; k += 8) {
        double v[8];
#pragma unroll
        for (int q = 0; q < 8; q++) v[q] = p[(int64_t)(k + q) * n * 10];
#pragma unroll
        for (int q = 0; q < 8; q++) s += v[q];
    }
    for (; k < nsplit; k++) s += p[(int64_t)k * n * 10];
    if (c == 0)
        dsig[j] = s;
    else
        dvert[j * 9 + c - 1] = s;
}

// dvert[i*9 + 3m + c] += (sum_bx partP[bx][i][c]) / 3 for each corner m (c_i = mean of the vertices)
__global__ __launch_bounds__(kBlock) void k_vjp_reduce_p(const double* __restrict__ partP, int nbx, int64_t n,
                                                         double* __restrict__ dvert)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    double s[3] = {0., 0., 0.};
    for (int b = 0; b < nbx; b++)
        for (int c = 0; c < 3; c++) s[c] += partP[((int64_t)b * n + i) * 3 + c];
    for (int m = 0; m < 3; m++)
        for (int c = 0; c < 3; c++) dvert[i * 9 + 3 * m + c] += s[c] * (1. / 3.);
}

int vjp_splits(int64_t nbx, int64_t work)
{
    int64_t s = (2048 + nbx - 1) / std::max<int64_t>(nbx, 1);
    s = std::min<int64_t>(s, std::max<int64_t>(1, work / 16));
    return (int)std::max<int64_t>(1, std::min<int64_t>(s, 256));
}

}  // namespace

size_t vjp_workspace_doubles(int64_t n, int64_t npts)
{
    const int64_t nbx = (n + kBlock - 1) / kBlock;
    const int sf = vjp_splits(nbx, npts), sm = vjp_splits(nbx, n);
    // partial sums of the splits, the matrix term's sums per target, the field term's near flags
    return (size_t)std::max<int64_t>(sf, sm) * n * 10 + (size_t)nbx * n * 3 + (size_t)((n + 63) / 64) * 128;
}

hipError_t launch_field_vjp(hipStream_t st, const double* geom, const double* sigma, const double* rule, int64_t n,
                            const double* pts, const double* gk, int64_t npts, double* dsig, double* dvert,
                            double* ws, size_t ws_doubles)
{
    if (n <= 0) return hipSuccess;
    if (ws_doubles < vjp_workspace_doubles(n, npts)) return hipErrorInvalidValue;
    const int64_t nbx = nblocks(n), sf = vjp_splits(nbx, npts);
    // Chunks of 64 points a wavefront where that gives kVjpBlocks blocks, down to 4 points below (a node's own work is
    // about that of two pairs): the closed forms and small calls need the blocks.  Splits within the workspace's.
    // Calls, us, with a thread per element and 16 to 100 points / so: rings 200 elements x 5,000 points 790 / 591,
    // coax 5,000 x 20,000 9,069 / 7,290, cube 700 x 10 215 / 186.  Rounds of 256 points a block throughout were
    // 2.6 times slower than the former on a call of a few hundred elements.
    constexpr int64_t kVjpBlocks = 2048;
    const int64_t groups = (n + 63) / 64;
    int64_t chunk = std::clamp<int64_t>(npts * groups / (kVjpWaves * kVjpBlocks), 4, 64);
    int64_t per = std::max<int64_t>(kVjpWaves * chunk, (npts + sf - 1) / sf);
    chunk = std::min<int64_t>(64, (per + kVjpWaves - 1) / kVjpWaves);
    per = (per + kVjpWaves * chunk - 1) / (kVjpWaves * chunk) * (kVjpWaves * chunk);
    const int ns = (int)std::max<int64_t>(1, (npts + per - 1) / per);
    int* near = reinterpret_cast<int*>(ws + (size_t)sf * n * 10);
    const dim3 grid((unsigned)groups, (unsigned)ns);
    k_vjp_field_far<<<grid, 64 * kVjpWaves, 0, st>>>(geom, sigma, rule, n, pts, gk, npts, per, (int)chunk, ws, near);
    k_vjp_field_near<<<grid, 64 * kVjpWaves, 0, st>>>(geom, sigma, n, pts, gk, npts, per, ws, near);
    k_vjp_reduce_v<<<dim3((unsigned)nbx, 10), kBlock, 0, st>>>(ws, ns, n, dsig, dvert);
    return hipGetLastError();
}

hipError_t launch_matrix_vjp(hipStream_t st, const double* geom, const double* targets, const double* rule,
                             int64_t n, const double* lw, const double* u, double* dvert, double* ws,
                             size_t ws_doubles)
{
    if (n <= 0) return hipSuccess;
    if (ws_doubles < vjp_workspace_doubles(n, 0)) return hipErrorInvalidValue;
    const int64_t nbx = nblocks(n);
    const int s = vjp_splits(nbx, n);
    const int64_t per = (n + s - 1) / s;
    const int ns = (int)((n + per - 1) / per);
    double* partV = ws;
    double* partP = ws + (size_t)s * n * 10;
    dim3 grid((unsigned)nbx, (unsigned)ns);
    k_vjp_matrix<false><<<grid, kBlock, 0, st>>>(geom, targets, rule, n, lw, u, per, partV, partP);
    k_vjp_matrix<true><<<grid, kBlock, 0, st>>>(geom, targets, rule, n, lw, u, per, partV, partP);
    k_vjp_reduce_v<<<dim3((unsigned)nbx, 10), kBlock, 0, st>>>(partV, ns, n, nullptr, dvert);
    k_vjp_reduce_p<<<(unsigned)nbx, kBlock, 0, st>>>(partP, (int)nbx, n, dvert);
    return hipGetLastError();
}

}  // namespace kem
