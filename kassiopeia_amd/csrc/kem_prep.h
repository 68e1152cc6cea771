// kem_prep.h -- host-side element preparation and physical constants.
#ifndef KEM_PREP_H
#define KEM_PREP_H

#include "kem_layout.h"

#include <algorithm>
#include <cstdint>
#include <thread>
#include <vector>

namespace kem {

// f(begin, end) over [0, n) in contiguous parts on up to 8 threads, at least grain elements each; the caller's thread takes
// the first part, and the parts of threads that cannot be started.
template <typename F>
void in_parts(int64_t n, int64_t grain, F f)
{
    const int64_t most = std::min<int64_t>(8, std::max(1u, std::thread::hardware_concurrency()));
    const int64_t parts = std::max<int64_t>(1, std::min(most, n / grain));
    const int64_t each = (n + parts - 1) / parts;
    std::vector<std::thread> started;
    started.reserve((size_t)parts);
    int64_t k = 1;
    try {
        for (; k < parts; k++) started.emplace_back(f, std::min(n, k * each), std::min(n, (k + 1) * each));
    } catch (...) {
    }
    f((int64_t)0, std::min(n, each));
    for (; k < parts; k++) f(std::min(n, k * each), std::min(n, (k + 1) * each));
    for (std::thread& t : started) t.join();
}

// Kommon/Base/Utility/KConst_2021.h:37 (pi), :139-146 (eps0); KEMField/Source/Core/src/KEMConstants.cc:9-12
constexpr double kPi = 3.141592653589793238462643383279502884;
constexpr double kEps0 = 8.8541878128E-12;
constexpr double kOneOverFourPiEps0 = 1. / (4. * kPi * kEps0);

// Expand one KEMField shape record into the device record g[KG_STRIDE] and the node table
// nodes[KEM_NODE_STRIDE].  Returns 0, or -1 for a degenerate / non-finite element.
int prep_element(int type, const double* shape_data, double* g, double* nodes);

// Barycentric coordinates and weights of the triangle rules in node-slot order (7-, 12-,
// 33-point at KEM_N7 / KEM_N12 / KEM_N33): t[4*slot .. 4*slot+3] = (a, b, c, w), the node
// being a*P0 + b*P1 + c*P2 (GaussPoints_Tri7P/12P/33P, KElectrostaticCubatureTriangleIntegrator.cc:34-270).
void triangle_rule_table(double* t);

// FP32 node table for the mixed-precision far field: node positions relative to the
// element's dispatch centre (KG_CX..KG_CZ of g) and weights, KEM_NODE32_STRIDE floats (the
// 52 slots of the FP64 table plus a 6-point triangle rule at KEM_N6).
void prep_nodes32(const double* g, const double* nodes, float* nodes32);

// Collocation target record t[KT_STRIDE]: the shape's Centroid(), unit normal, boundary type
// and Neumann flux.
void prep_target(int type, const double* shape_data, int bc, double flux, double* t);

// Element clusters for the near pass: order[n] lists the elements so that aligned runs of
// KEM_TREE_LEAF * KEM_TREE_FAN^k of them are compact (divided by medians of the dispatch centres); clusters[4 * ceil(n / KEM_CLUSTER)] holds, per run of KEM_CLUSTER
// consecutive entries of order, the centre of their bounding box and a radius R such that
// every point within the near distance of a member lies within R of the centre.
void build_clusters(int64_t n, const double* g, int32_t* order, double* clusters);

// Far records of the mixed far field in cluster order (layout: KEM_FAR6_*, KEM_FAR3_* and
// KEM_FAR_CL_STRIDE in kem_layout.h): far6[KEM_FAR6_STRIDE * n] floats from the FP32 node table
// nodes32 and the element records g, far3[KEM_FAR3_STRIDE * n] floats from the vertices in g,
// far_cl[KEM_FAR_CL_STRIDE * ceil(n / KEM_CLUSTER)] doubles with the clusters' centres taken from
// clusters.
void build_far6(int64_t n, const double* g, const float* nodes32, const int32_t* order, const double* clusters,
                float* far6, float* far3, double* far_cl);

// Levels of the tree over n elements (KEM_TREE_* in kem_layout.h): count[k] runs at first[k].. of the node
// array.  low / run: the lowest level that an evaluation expands, and its elements per run.
struct TreeLevels {
    int levels = 0;
    int low = 0;
    int run = KEM_TREE_LEAF;
    int32_t count[KEM_TREE_LEVELS] = {}, first[KEM_TREE_LEVELS] = {};
};
void tree_levels(int64_t n, TreeLevels& t);
// Node records of all levels, KEM_TREE_STRIDE doubles each, over elements in the order given (planar elements
// and wires).
void build_tree(int64_t n, const double* g, const int32_t* order, const TreeLevels& t, double* tree);

}  // namespace kem

#endif
