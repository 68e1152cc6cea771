// kem_sort.hip -- spatial ordering of field points for the field kernels (gfx950).
//
// A wavefront evaluates one element against 64 points at a time and executes every
// quadrature branch that any of its lanes needs.  Points in the caller's order are spatially
// random, so a wavefront typically runs both the 12- and the 33-point loops (and the closed
// form) for one element.  Sorting the points along a Hilbert curve of the cube around them makes the
// 64 points of a wavefront neighbours, so they almost always share one regime, and close to each other, so
// the hierarchical pass accepts more expansions for them.  (A Morton curve's jumps left groups of points up to
// 8 times the usual size, whose wavefronts ran 20 times longer than the others.)
// The results are gathered back to the caller's order.  In its last digits a point's value depends on the
// ordering, and so on the call's other points: which pairs of a wavefront share a rule, and which runs of elements are
// taken as expansions, follows from the points visited with it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <hipcub/hipcub.hpp>

#include <cstdint>

#include "kem_kernels.h"

namespace kem {

namespace {

constexpr int kBlock = 256;
constexpr int kBoxParts = 256;

// per-block min/max of the three coordinates: part[b*6 + {0,1,2}] = min, [3,4,5] = max
__global__ __launch_bounds__(kBlock) void k_bbox_part(const double* __restrict__ x, const double* __restrict__ y,
                                                      const double* __restrict__ z, int64_t n, double* __restrict__ part)
{
    __shared__ double sh[6][kBlock];
    double mn[3] = {1e300, 1e300, 1e300}, mx[3] = {-1e300, -1e300, -1e300};
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const double v[3] = {x[i], y[i], z[i]};
        for (int k = 0; k < 3; k++) {
            mn[k] = fmin(mn[k], v[k]);
            mx[k] = fmax(mx[k], v[k]);
        }
    }
    for (int k = 0; k < 3; k++) {
        sh[k][threadIdx.x] = mn[k];
        sh[3 + k][threadIdx.x] = mx[k];
    }
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            for (int k = 0; k < 3; k++) {
                sh[k][threadIdx.x] = fmin(sh[k][threadIdx.x], sh[k][threadIdx.x + s]);
                sh[3 + k][threadIdx.x] = fmax(sh[3 + k][threadIdx.x], sh[3 + k][threadIdx.x + s]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 6) part[blockIdx.x * 6 + threadIdx.x] = sh[threadIdx.x][0];
}

// spread the low 21 bits of a so that bit k lands at bit 3k
__device__ __forceinline__ uint64_t spread3(uint64_t a)
{
    uint64_t v = a & 0x1fffffull;
    v = (v | (v << 32)) & 0x1f00000000ffffull;
    v = (v | (v << 16)) & 0x1f0000ff0000ffull;
    v = (v | (v << 8)) & 0x100f00f00f00f00full;
    v = (v | (v << 4)) & 0x10c30c30c30c30c3ull;
    v = (v | (v << 2)) & 0x1249249249249249ull;
    return v;
}

// Hilbert key (bits per axis) of each point in the cube over the box spanned by the block
// partials: as many bits as the key holds, up to 21, since a stray point far from the others (a lost particle) widens the
// cube: at 1e5 times their extent it leaves them 21 cells per axis, and at 16 bits one, with
// which 200,000 points in a random order over 20,000 triangles took 61.5 ms instead of 7.0 (mixed).  J. Skilling, "Programming the Hilbert curve" (2004), axes to transposed index.  pset (nullable): the set
// above the curve's bits, for the hierarchical pass.  The flat passes' points of several charge-density sets sort
// together: their kernels read the sets element-major, so a wavefront may mix sets.
constexpr int kCurveBits = 21;
inline int curve_bits(int set_bits) { return std::min(kCurveBits, (64 - set_bits) / 3); }
__global__ __launch_bounds__(kBlock) void k_curve(const double* __restrict__ x, const double* __restrict__ y,
                                                  const double* __restrict__ z, int64_t n,
                                                  const int32_t* __restrict__ pset, int bits,
                                                  const double* __restrict__ part, int nparts,
                                                  uint64_t* __restrict__ key, int32_t* __restrict__ idx)
{
    // the box from the partials: thread t < nparts brings one of them
    __shared__ double sh[6][kBoxParts];
    for (int k = 0; k < 3; k++) {
        const bool have = (int)threadIdx.x < nparts;
        sh[k][threadIdx.x] = have ? part[threadIdx.x * 6 + k] : 1e300;
        sh[3 + k][threadIdx.x] = have ? part[threadIdx.x * 6 + 3 + k] : -1e300;
    }
    __syncthreads();
    for (int s = kBoxParts / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            for (int k = 0; k < 3; k++) {
                sh[k][threadIdx.x] = fmin(sh[k][threadIdx.x], sh[k][threadIdx.x + s]);
                sh[3 + k][threadIdx.x] = fmax(sh[3 + k][threadIdx.x], sh[3 + k][threadIdx.x + s]);
            }
        __syncthreads();
    }
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const double v[3] = {x[i], y[i], z[i]};
    double span = 0.;
    for (int k = 0; k < 3; k++) span = fmax(span, sh[3 + k][0] - sh[k][0]);
    const double most = (1 << bits) - 1;
    uint32_t a[3];
    for (int k = 0; k < 3; k++) {
        double q = span > 0. ? (v[k] - sh[k][0]) / span * most : 0.;
        q = q > 0. ? (q > most ? most : q) : 0.;
        a[k] = (uint32_t)q;
    }
    for (uint32_t q = 1u << (bits - 1); q > 1; q >>= 1) {
        const uint32_t p = q - 1;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            if (a[k] & q) {
                a[0] ^= p;
            } else {
                const uint32_t t = (a[0] ^ a[k]) & p;
                a[0] ^= t;
                a[k] ^= t;
            }
        }
    }
    a[1] ^= a[0];
    a[2] ^= a[1];
    uint32_t t = 0;
    for (uint32_t q = 1u << (bits - 1); q > 1; q >>= 1)
        if (a[2] & q) t ^= q - 1;
    const uint64_t set = pset ? (uint64_t)(uint32_t)pset[i] << (3 * bits) : 0;
    key[i] = set | spread3(a[2] ^ t) | spread3(a[1] ^ t) << 1 | spread3(a[0] ^ t) << 2;
    idx[i] = (int32_t)i;
}

__global__ __launch_bounds__(kBlock) void k_gather3(const int32_t* __restrict__ idx, const double* __restrict__ x,
                                                    const double* __restrict__ y, const double* __restrict__ z,
                                                    const int32_t* __restrict__ pset, int64_t n,
                                                    double* __restrict__ sx, double* __restrict__ sy,
                                                    double* __restrict__ sz, int32_t* __restrict__ sset)
{
    const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (k >= n) return;
    const int32_t i = idx[k];
    sx[k] = x[i];
    sy[k] = y[i];
    sz[k] = z[i];
    if (pset) sset[k] = pset[i];
}

__global__ __launch_bounds__(kBlock) void k_scatter4(const int32_t* __restrict__ idx, const double* __restrict__ s0,
                                                     const double* __restrict__ s1, const double* __restrict__ s2,
                                                     const double* __restrict__ s3, int64_t n, double* __restrict__ d0,
                                                     double* __restrict__ d1, double* __restrict__ d2,
                                                     double* __restrict__ d3)
{
    const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (k >= n) return;
    const int32_t i = idx[k];
    if (d0) d0[i] = s0[k];
    if (d1) d1[i] = s1[k];
    if (d2) d2[i] = s2[k];
    if (d3) d3[i] = s3[k];
}

inline unsigned nblocks(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

inline size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

size_t cub_temp_bytes(int64_t n)
{
    size_t bytes = 0;
    (void)hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const uint64_t*)nullptr, (uint64_t*)nullptr,
                                             (const int32_t*)nullptr, (int32_t*)nullptr, (int)n, 0, 64);
    return bytes;
}

}  // namespace

size_t sort_workspace_bytes(int64_t n)
{
    return align256(8 * n) * 2 + align256(4 * n) * 3 + align256(8 * n) * 7 + align256(8 * 6 * kBoxParts) +
           align256(cub_temp_bytes(n));
}

hipError_t launch_field_sorted(hipStream_t st, int policy, const FieldMesh& m, bool mixed, double fp64_ratio,
                               const double* sigma, const int32_t* pset, int64_t nsets, const double* px,
                               const double* py, const double* pz, int64_t npts, double* phi, double* ex, double* ey,
                               double* ez, void* sort_ws, size_t sort_ws_bytes, double* ws, int64_t ws_doubles,
                               int64_t range_elems, hipEvent_t far_begin, hipEvent_t far_end,
                               const SideStream* side)
{
    if (npts <= 0) return hipSuccess;
    if (npts > INT32_MAX || sort_ws_bytes < sort_workspace_bytes(npts)) return hipErrorInvalidValue;
    if (!phi || !ex || !ey || !ez) return hipErrorInvalidValue;
    char* p = (char*)sort_ws;
    auto take = [&](size_t bytes) {
        char* r = p;
        p += align256(bytes);
        return r;
    };
    uint64_t* k0 = (uint64_t*)take(8 * npts);
    uint64_t* k1 = (uint64_t*)take(8 * npts);
    int32_t* i0 = (int32_t*)take(4 * npts);
    int32_t* i1 = (int32_t*)take(4 * npts);
    int32_t* ss = (int32_t*)take(4 * npts);
    double* sx = (double*)take(8 * npts);
    double* sy = (double*)take(8 * npts);
    double* sz = (double*)take(8 * npts);
    double* o[4];
    for (int c = 0; c < 4; c++) o[c] = (double*)take(8 * npts);
    double* box = (double*)take(8 * 6 * kBoxParts);
    size_t tb = cub_temp_bytes(npts);
    void* tmp = take(tb);

    int nb = (int)((npts + kBlock - 1) / kBlock);
    if (nb > kBoxParts) nb = kBoxParts;
    k_bbox_part<<<nb, kBlock, 0, st>>>(px, py, pz, npts, box);
    // the hierarchical pass takes the points set by set (as launch_field decides)
    int set_bits = 0;
    const TreePlan tp = plan_tree(policy, m, mixed, fp64_ratio, pset != nullptr, nsets, npts);
    const bool by_set = pset && tp.use && tp.doubles() <= ws_doubles;
    if (by_set)
        for (int64_t v = nsets - 1; v > 0; v >>= 1) set_bits++;
    const int bits = curve_bits(set_bits);
    k_curve<<<nblocks(npts), kBlock, 0, st>>>(px, py, pz, npts, by_set ? pset : nullptr, bits, box, nb, k0, i0);
    hipError_t e = hipcub::DeviceRadixSort::SortPairs(tmp, tb, k0, k1, i0, i1, (int)npts, 0, 3 * bits + set_bits, st);
    if (e != hipSuccess) return e;
    k_gather3<<<nblocks(npts), kBlock, 0, st>>>(i1, px, py, pz, pset, npts, sx, sy, sz, ss);
    e = launch_field(st, policy, m, mixed, fp64_ratio, sigma, pset ? ss : nullptr, nsets, sx, sy, sz, npts, o[0], o[1],
                     o[2], o[3], ws, ws_doubles, range_elems, far_begin, far_end, side);
    if (e != hipSuccess) return e;
    k_scatter4<<<nblocks(npts), kBlock, 0, st>>>(i1, o[0], o[1], o[2], o[3], npts, phi, ex, ey, ez);
    return hipGetLastError();
}

hipError_t launch_census_paths_sorted(hipStream_t st, const FieldMesh& m, const double* px, const double* py,
                                      const double* pz, int64_t npts, void* sort_ws, size_t sort_ws_bytes,
                                      unsigned long long* counts)
{
    if (npts <= 0) return hipSuccess;
    if (npts > INT32_MAX || sort_ws_bytes < sort_workspace_bytes(npts)) return hipErrorInvalidValue;
    // the same carving and ordering as launch_field_sorted
    char* p = (char*)sort_ws;
    auto take = [&](size_t bytes) {
        char* r = p;
        p += align256(bytes);
        return r;
    };
    uint64_t* k0 = (uint64_t*)take(8 * npts);
    uint64_t* k1 = (uint64_t*)take(8 * npts);
    int32_t* i0 = (int32_t*)take(4 * npts);
    int32_t* i1 = (int32_t*)take(4 * npts);
    int32_t* ss = (int32_t*)take(4 * npts);
    double* sx = (double*)take(8 * npts);
    double* sy = (double*)take(8 * npts);
    double* sz = (double*)take(8 * npts);
    for (int c = 0; c < 4; c++) (void)take(8 * npts);
    double* box = (double*)take(8 * 6 * kBoxParts);
    size_t tb = cub_temp_bytes(npts);
    void* tmp = take(tb);

    int nb = (int)((npts + kBlock - 1) / kBlock);
    if (nb > kBoxParts) nb = kBoxParts;
    k_bbox_part<<<nb, kBlock, 0, st>>>(px, py, pz, npts, box);
    k_curve<<<nblocks(npts), kBlock, 0, st>>>(px, py, pz, npts, nullptr, kCurveBits, box, nb, k0, i0);
    hipError_t e = hipcub::DeviceRadixSort::SortPairs(tmp, tb, k0, k1, i0, i1, (int)npts, 0, 3 * kCurveBits, st);
    if (e != hipSuccess) return e;
    k_gather3<<<nblocks(npts), kBlock, 0, st>>>(i1, px, py, pz, nullptr, npts, sx, sy, sz, ss);
    return launch_census_paths(st, m, sx, sy, sz, npts, counts);
}

}  // namespace kem
