// Signed distance at the octree vertices (right-hand side of the fit).
//
// Replaces ThinShells::cpSDFOfTreeNodes (reference ThinShells.cpp:481-509).
// The reference calls igl::signed_distance with the fast winding number sign,
// which is third-party code absent here.  Both this file and the CPU oracle
// use the same definition:
//   - |b| is the exact Euclidean distance to the nearest triangle (closest
//     point on a triangle, Ericson, Real-Time Collision Detection 5.1.5),
//     in binary64.
//   - The sign is negative where the generalised winding number exceeds 1/2.
//     The winding number is the sum of triangle solid angles over 4 pi (Van
//     Oosterom and Strackee 1983), each solid angle in binary32 after a
//     binary64 subtraction of the query point.
//
// Triangle tree.  Triangles are sorted by the Morton code of their centroid
// and cut into buckets of kBucket; an implicit binary tree sits over the
// buckets (node k of level h covers sorted triangles [k*8*2^h, (k+1)*8*2^h)),
// with a binary32 box per node rounded outward, so it holds every vertex
// exactly.  Levels are built one launch each, without atomics.
//   - Distance: a walk, level by level and for packets of neighbouring points
//     (see "packets" below), that skips a node whose box is farther than a
//     binary64 distance known so far, at first to a triangle at the query's
//     own Morton position.  A skipped node holds no triangle whose
//     distance could equal or beat the best, so the minimum and the lowest
//     index among equal minima are those of the full search.
//   - Winding number, exactly (generalised winding numbers, Jacobson,
//     Kavan and Sorkine-Hornung 2013, section 3.2): for a node with triangle
//     set S and a query p outside the node's box, close S with the fan C of
//     its boundary edges around the box centre; S + C is a closed chain
//     inside the convex box, so its winding number at p is 0 and
//     w_S(p) = -w_C(p).  The boundary of S is the signed sum of its half
//     edges (a -> b counts +1 for the min -> max direction, -1 otherwise),
//     which is exact for open, non-manifold or inconsistently oriented
//     meshes too.  A node's fan is stored only when it has at most as many
//     edges as the node has triangles; otherwise the walk descends.
//   - Winding number of a closed mesh, by a ray: when every undirected edge
//     has exactly two half edges of opposite directions, the mesh is an
//     oriented closed surface, and its winding number at p is the signed
//     number of crossings of any ray from p (self-intersecting and nested
//     surfaces included).  Each point takes the axis direction (+-x, +-y,
//     +-z) that leaves the mesh's box soonest; the ray is tested against
//     the triangles whose boxes it meets: p is inside the projection of a
//     triangle across the ray when its three edge orientations agree, and
//     the crossing lies ahead of p when the orientation of the tetrahedron
//     (a, b, c, p) has the sign of the triangle's normal along the ray.  Each
//     orientation is a binary64 determinant whose sign is taken only when it
//     exceeds the rounding bound of its terms (the static filters of
//     Shewchuk, Adaptive Precision Floating-Point Arithmetic and Fast Robust
//     Geometric Predicates, 1997); a point with any undecided orientation
//     (on or within rounding of an edge line or a triangle plane) takes the
//     fan walk above.
//   - With a short boundary, by the ray and the angles of the boundary's half
//     edges (k_rim), under the same conditions.

#include <algorithm>
#include <cmath>
#include <vector>

#include "internal.hpp"

namespace its {
namespace {
constexpr int kT = 256;
constexpr int kBucket = 8;
// query walks treat nodes of this level (at most 64 triangles) as leaves
constexpr int kLeafLevel = 3;
static_assert((kBucket << kLeafLevel) == 64, "one triangle per lane in a leaf");
constexpr int kMaxLevels = 32;

// ------------------------------------------------------------ geometry ----
__device__ inline double d3dot(const double* a, const double* b) { return a[0] * b[0] + (a[1] * b[1] + a[2] * b[2]); }

__device__ double point_tri_dist2(const double p[3], const double a[3], const double b[3], const double c[3]) {
    double ab[3], ac[3], ap[3], q[3];
    for (int i = 0; i < 3; ++i) { ab[i] = b[i] - a[i]; ac[i] = c[i] - a[i]; ap[i] = p[i] - a[i]; }
    double d1 = d3dot(ab, ap), d2 = d3dot(ac, ap);
    if (d1 <= 0.0 && d2 <= 0.0) {
        for (int i = 0; i < 3; ++i) q[i] = a[i];
    } else {
        double bp[3];
        for (int i = 0; i < 3; ++i) bp[i] = p[i] - b[i];
        double d3 = d3dot(ab, bp), d4 = d3dot(ac, bp);
        double cp[3];
        for (int i = 0; i < 3; ++i) cp[i] = p[i] - c[i];
        double d5 = d3dot(ab, cp), d6 = d3dot(ac, cp);
        double vc = d1 * d4 - d3 * d2, vb = d5 * d2 - d1 * d6, va = d3 * d6 - d5 * d4;
        if (d3 >= 0.0 && d4 <= d3) {
            for (int i = 0; i < 3; ++i) q[i] = b[i];
        } else if (vc <= 0.0 && d1 >= 0.0 && d3 <= 0.0) {
            double v = d1 / (d1 - d3);
            for (int i = 0; i < 3; ++i) q[i] = a[i] + v * ab[i];
        } else if (d6 >= 0.0 && d5 <= d6) {
            for (int i = 0; i < 3; ++i) q[i] = c[i];
        } else if (vb <= 0.0 && d2 >= 0.0 && d6 <= 0.0) {
            double w = d2 / (d2 - d6);
            for (int i = 0; i < 3; ++i) q[i] = a[i] + w * ac[i];
        } else if (va <= 0.0 && (d4 - d3) >= 0.0 && (d5 - d6) >= 0.0) {
            double w = (d4 - d3) / ((d4 - d3) + (d5 - d6));
            for (int i = 0; i < 3; ++i) q[i] = b[i] + w * (c[i] - b[i]);
        } else {
            double denom = 1.0 / (va + vb + vc);
            double v = vb * denom, w = vc * denom;
            for (int i = 0; i < 3; ++i) q[i] = a[i] + ab[i] * v + ac[i] * w;
        }
    }
    double d[3] = {p[0] - q[0], p[1] - q[1], p[2] - q[2]};
    return d3dot(d, d);
}

// atan2 for the solid-angle sums: octant reduction to a = min/max in
// [0, 1] and atan(a) = a P(a^2), P of degree 7 fitted here by weighted least
// squares on Chebyshev nodes (Lawson iterations toward the minimax error).
// Absolute error below 3.2e-7 over all quadrants in binary32, signed zeros
// and the +-pi cut as atan2.
__device__ inline float atan2_fit(float y, float x) {
#pragma clang fp contract(fast)
    const float ax = fabsf(x), ay = fabsf(y);
    const float mx = fmaxf(ax, ay), mn = fminf(ax, ay);
    const float a = mx > 1e-30f ? mn * __builtin_amdgcn_rcpf(mx) : 0.f;
    const float q = a * a;
    float r = -0.004054564982652664f;
    r = r * q + 0.021862955763936043f;
    r = r * q - 0.055912334471940994f;
    r = r * q + 0.0964219868183136f;
    r = r * q - 0.1390863060951233f;
    r = r * q + 0.19946566224098206f;
    r = r * q - 0.33329859375953674f;
    r = r * q + 0.9999993443489075f;
    r = r * a;
    if (ay > ax) r = 1.5707963267948966f - r;
    if (x < 0.f) r = 3.141592653589793f - r;
    return copysignf(r, y);
}

// solid angle of triangle ABC seen from p (signed by orientation): binary64
// differences, the rest in binary32 with fused multiply-adds
__device__ inline float solid_angle(const double p[3], const double* A, const double* B, const double* C) {
#pragma clang fp contract(fast)
    float a[3], b[3], c[3];
    for (int i = 0; i < 3; ++i) {
        a[i] = (float)(A[i] - p[i]);
        b[i] = (float)(B[i] - p[i]);
        c[i] = (float)(C[i] - p[i]);
    }
    float la = __builtin_amdgcn_sqrtf(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]);
    float lb = __builtin_amdgcn_sqrtf(b[0] * b[0] + b[1] * b[1] + b[2] * b[2]);
    float lc = __builtin_amdgcn_sqrtf(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
    float det = a[0] * (b[1] * c[2] - b[2] * c[1]) + a[1] * (b[2] * c[0] - b[0] * c[2]) + a[2] * (b[0] * c[1] - b[1] * c[0]);
    float ab = a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
    float bc = b[0] * c[0] + b[1] * c[1] + b[2] * c[2];
    float ca = c[0] * a[0] + c[1] * a[1] + c[2] * a[2];
    float den = la * lb * lc + ab * lc + bc * la + ca * lb;
    return 2.0f * atan2_fit(det, den);
}

// apex of a node's fan: the centre of its binary32 box, in binary64
__host__ __device__ inline double fan_apex(float lo, float hi) { return 0.5 * ((double)lo + (double)hi); }

// solid angle of the fan triangle (apex, a, b) seen from p, from the
// binary32 vectors z = apex - p (|z| = lz), u = a - p, v = b - p: the same
// formula as solid_angle with its first vertex fixed
__device__ inline float fan_angle(const float z[3], float lz, const float u[3], const float v[3]) {
#pragma clang fp contract(fast)
    const float lu = __builtin_amdgcn_sqrtf(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
    const float lv = __builtin_amdgcn_sqrtf(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    const float det = z[0] * (u[1] * v[2] - u[2] * v[1]) + z[1] * (u[2] * v[0] - u[0] * v[2]) +
                      z[2] * (u[0] * v[1] - u[1] * v[0]);
    const float zu = z[0] * u[0] + z[1] * u[1] + z[2] * u[2];
    const float uv = u[0] * v[0] + u[1] * v[1] + u[2] * v[2];
    const float vz = v[0] * z[0] + v[1] * z[1] + v[2] * z[2];
    const float den = lz * lu * lv + zu * lv + uv * lz + vz * lu;
    return 2.0f * atan2_fit(det, den);
}

// binary32 neighbours of a binary64 value, rounded down / up
__device__ inline float f_down(double x) {
    float f = (float)x;
    return ((double)f > x) ? nextafterf(f, -INFINITY) : f;
}
__device__ inline float f_up(double x) {
    float f = (float)x;
    return ((double)f < x) ? nextafterf(f, INFINITY) : f;
}

// Bounding sphere of a triangle in binary32: centre = vertex mean, radius =
// largest centre-vertex distance, both widened by a margin that covers the
// binary32 rounding of every quantity derived from them.
__device__ inline float bound_margin(float scale) { return 1e-5f * scale + 1e-30f; }

__device__ inline float4 tri_sphere(const double* T) {
    double c[3];
    for (int a = 0; a < 3; ++a) c[a] = (T[a] + T[3 + a] + T[6 + a]) / 3.0;
    double r2 = 0, cm = 0;
    for (int v = 0; v < 3; ++v) {
        double d2 = 0;
        for (int a = 0; a < 3; ++a) {
            const double d = T[3 * v + a] - c[a];
            d2 += d * d;
        }
        r2 = fmax(r2, d2);
    }
    for (int a = 0; a < 3; ++a) cm = fmax(cm, fabs(c[a]));
    const double r = sqrt(r2);
    return make_float4((float)c[0], (float)c[1], (float)c[2], (float)(r * (1.0 + 1e-6) + 1e-6 * (cm + r)));
}

// unit normal of a triangle, binary64 rounded once; zero for a degenerate one
__device__ inline float4 tri_unit_normal(const double* T) {
    const double u[3] = {T[3] - T[0], T[4] - T[1], T[5] - T[2]}, v[3] = {T[6] - T[0], T[7] - T[1], T[8] - T[2]};
    const double x = u[1] * v[2] - u[2] * v[1], y = u[2] * v[0] - u[0] * v[2], z = u[0] * v[1] - u[1] * v[0];
    const double l2 = x * x + y * y + z * z;
    // a sliver's normal is mostly rounding: no bound is taken from it
    const double m = fmax(u[0] * u[0] + u[1] * u[1] + u[2] * u[2], v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    if (!(l2 > 1e-12 * m * m)) return make_float4(0.f, 0.f, 0.f, 0.f);
    const double l = sqrt(l2);
    return make_float4((float)(x / l), (float)(y / l), (float)(z / l), 0.f);
}

// ---------------------------------------------------------------- tree ----
struct Shape {
    int32_t T;                  // triangles
    int32_t H;                  // root level; level 0 holds the buckets
    int32_t count[kMaxLevels];  // nodes per level
    int32_t off[kMaxLevels];    // first node of each level
};

__host__ __device__ inline int64_t node_first(int h, int64_t k) { return k * ((int64_t)kBucket << h); }
__host__ __device__ inline int64_t node_last(const Shape& s, int h, int64_t k) {
    return std::min<int64_t>(s.T, (k + 1) * ((int64_t)kBucket << h));
}

// next node in depth-first order after the subtree at (h, k); false at the end
__device__ inline bool tree_next(const Shape& s, int& h, int& k) {
    while (h < s.H) {
        if (!(k & 1) && k + 1 < s.count[h]) {
            ++k;
            return true;
        }
        k >>= 1;
        ++h;
    }
    return false;
}

struct Quant {
    double lo[3], scale[3];
};

__device__ inline uint32_t quant_code(const Quant& q, const double x[3]) {
    uint32_t u[3];
    for (int a = 0; a < 3; ++a) {
        double v = (x[a] - q.lo[a]) * q.scale[a];
        v = fmin(fmax(v, 0.0), 1023.0);
        u[a] = (uint32_t)v;
    }
    return morton3(u[0], u[1], u[2]);
}

struct TreeView {
    Shape s;
    const Quant* q;
    const double* tris;      // 9 per sorted triangle
    const float4* sph;       // bounding sphere per sorted triangle
    const float4* nrm;       // unit normal per sorted triangle (zero: none)
    const int32_t* tid;      // original index per sorted triangle
    const uint32_t* code;    // centroid Morton code per sorted triangle (ascending)
    const float4* node;      // 2 per node: box lo.xyz + first fan edge (int bits in w),
                             // box hi.xyz + fan edge count (int bits in w; -1: no fan)
    const float* fan;        // 6 per fan edge: a - centre, b - centre (centre of its node's box)
    const uint32_t* cell_lb; // per cell_bits-bit code prefix C: first sorted triangle with code >= C's range
    int cell_bits;
};

// -------------------------------------------------------------- build -----
__global__ void k_centroid_box(const double* V, const int32_t* F, int64_t nF, double* part) {
    __shared__ double sh[6][kT];
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < nF; t += (int64_t)gridDim.x * blockDim.x) {
        const double* a = V + 3 * (int64_t)F[3 * t];
        const double* b = V + 3 * (int64_t)F[3 * t + 1];
        const double* c = V + 3 * (int64_t)F[3 * t + 2];
        for (int x = 0; x < 3; ++x) {
            const double m = (a[x] + b[x] + c[x]) / 3.0;
            lo[x] = fmin(lo[x], m);
            hi[x] = fmax(hi[x], m);
        }
    }
    for (int x = 0; x < 3; ++x) { sh[x][threadIdx.x] = lo[x]; sh[3 + x][threadIdx.x] = hi[x]; }
    __syncthreads();
    for (int o = kT / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o)
            for (int x = 0; x < 3; ++x) {
                sh[x][threadIdx.x] = fmin(sh[x][threadIdx.x], sh[x][threadIdx.x + o]);
                sh[3 + x][threadIdx.x] = fmax(sh[3 + x][threadIdx.x], sh[3 + x][threadIdx.x + o]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 6) part[6 * blockIdx.x + threadIdx.x] = sh[threadIdx.x][0];
}

// Morton quantisation over the boxes of k_centroid_box; one workgroup of kT
__global__ __launch_bounds__(kT) void k_quant(const double* part, int nb, Quant* q) {
    __shared__ double sh[6][kT];
    for (int x = 0; x < 3; ++x) {
        double lo = INFINITY, hi = -INFINITY;
        for (int b = threadIdx.x; b < nb; b += kT) {
            lo = fmin(lo, part[6 * b + x]);
            hi = fmax(hi, part[6 * b + 3 + x]);
        }
        sh[x][threadIdx.x] = lo;
        sh[3 + x][threadIdx.x] = hi;
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    for (int x = 0; x < 3; ++x) {
        double lo = INFINITY, hi = -INFINITY;
        for (int k = threadIdx.x; k < kT; k += 64) {
            lo = fmin(lo, sh[x][k]);
            hi = fmax(hi, sh[3 + x][k]);
        }
        for (int o = 32; o > 0; o >>= 1) {
            lo = fmin(lo, __shfl_xor(lo, o));
            hi = fmax(hi, __shfl_xor(hi, o));
        }
        if (threadIdx.x == 0) {
            q->lo[x] = lo;
            q->scale[x] = (hi > lo) ? 1024.0 / (hi - lo) : 0.0;
        }
    }
}

// centroid code of every triangle, with its index as the sort's value
__global__ void k_tri_keys(const double* V, const int32_t* F, int64_t nF, const Quant* q, uint32_t* code,
                           uint32_t* idx) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nF) return;
    const double* a = V + 3 * (int64_t)F[3 * t];
    const double* b = V + 3 * (int64_t)F[3 * t + 1];
    const double* c = V + 3 * (int64_t)F[3 * t + 2];
    double m[3];
    for (int x = 0; x < 3; ++x) m[x] = (a[x] + b[x] + c[x]) / 3.0;
    code[t] = quant_code(*q, m);
    idx[t] = (uint32_t)t;
}

__global__ void k_tri_gather(const uint32_t* idx, int64_t nF, const double* V, const int32_t* F, double* tris,
                             float4* sph, float4* nrm, int32_t* tid, int32_t* pos) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nF) return;
    const int64_t t = (int64_t)idx[i];
    double T[9];
    for (int c = 0; c < 3; ++c)
        for (int a = 0; a < 3; ++a) T[3 * c + a] = V[3 * (int64_t)F[3 * t + c] + a];
    for (int j = 0; j < 9; ++j) tris[9 * i + j] = T[j];
    sph[i] = tri_sphere(T);
    nrm[i] = tri_unit_normal(T);
    tid[i] = (int32_t)t;
    pos[t] = (int32_t)i;
}

__global__ void k_bucket_box(const double* tris, Shape s, float4* node) {
    int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= s.count[0]) return;
    double l[3] = {INFINITY, INFINITY, INFINITY}, u[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int64_t i = node_first(0, k); i < node_last(s, 0, k); ++i)
        for (int v = 0; v < 3; ++v)
            for (int a = 0; a < 3; ++a) {
                l[a] = fmin(l[a], tris[9 * i + 3 * v + a]);
                u[a] = fmax(u[a], tris[9 * i + 3 * v + a]);
            }
    node[2 * (s.off[0] + k)] = make_float4(f_down(l[0]), f_down(l[1]), f_down(l[2]), 0.f);
    node[2 * (s.off[0] + k) + 1] = make_float4(f_up(u[0]), f_up(u[1]), f_up(u[2]), 0.f);
}

__global__ void k_level_box(Shape s, int h, float4* node) {
    int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= s.count[h]) return;
    const int64_t c0 = s.off[h - 1] + 2 * k;
    float4 l = node[2 * c0], u = node[2 * c0 + 1];
    if (2 * k + 1 < s.count[h - 1]) {
        const float4 l1 = node[2 * c0 + 2], u1 = node[2 * c0 + 3];
        l = make_float4(fminf(l.x, l1.x), fminf(l.y, l1.y), fminf(l.z, l1.z), 0.f);
        u = make_float4(fmaxf(u.x, u1.x), fmaxf(u.y, u1.y), fmaxf(u.z, u1.z), 0.f);
    }
    node[2 * (s.off[h] + k)] = l;
    node[2 * (s.off[h] + k) + 1] = u;
}

// Half edges keyed by their undirected edge (min << vb | max); the value is
// the sorted position of the triangle times 2, plus 1 for a max -> min edge.
// Degenerate edges (a == b) close nothing and get the key that sorts last.
__global__ void k_half_edges(const int32_t* F, int64_t nF, const int32_t* pos, int vb, uint64_t none, uint64_t* keys,
                             uint32_t* vals) {
    int64_t h = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= 3 * nF) return;
    const int64_t t = h / 3;
    const int e = (int)(h - 3 * t);
    const uint32_t a = (uint32_t)F[3 * t + e], b = (uint32_t)F[3 * t + (e + 1) % 3];
    keys[h] = (a == b) ? none : (((uint64_t)std::min(a, b) << vb) | std::max(a, b));
    vals[h] = 2u * (uint32_t)pos[t] + (a > b ? 1u : 0u);
}

// Walks the boundary contributions of one undirected edge (the run of equal
// keys starting at head i): for every level h >= 1 and every node holding
// some of its half edges, coef = signed count of those half edges.  Calls
// sink(node, h, k, coef) for coef != 0.  Above the level where one node
// holds all half edges, coef stays at their total; the walk stops there when
// the total is 0 (an interior edge).
template <class Sink>
__device__ void edge_walk(const uint64_t* keys, const uint32_t* vals, int64_t i, int64_t M, const Shape& s, Sink&& sink) {
    int64_t end = i + 1;
    while (end < M && keys[end] == keys[i]) ++end;
    static_assert((kBucket & (kBucket - 1)) == 0, "node spans are powers of two");
    const int bucket_shift = __builtin_ctz(kBucket);
    for (int h = 1; h <= s.H; ++h) {
        // node of level h holding sorted triangle t: t / (kBucket << h)
        const int shift = bucket_shift + h;
        const uint32_t k0 = (vals[i] >> 1) >> shift;
        bool same = true;
        int tot = 0;
        for (int64_t j = i; j < end; ++j) {
            const uint32_t v = vals[j];
            if (((v >> 1) >> shift) != k0) same = false;
            tot += (v & 1u) ? -1 : 1;
        }
        if (same) {
            if (tot == 0) return;
            sink(s.off[h] + (int64_t)k0, h, (int64_t)k0, tot);
            continue;
        }
        for (int64_t j = i; j < end; ++j) {
            const uint32_t kj = (vals[j] >> 1) >> shift;
            bool seen = false;
            for (int64_t jj = i; jj < j && !seen; ++jj) seen = (((vals[jj] >> 1) >> shift) == kj);
            if (seen) continue;
            int coef = 0;
            for (int64_t jj = j; jj < end; ++jj)
                if (((vals[jj] >> 1) >> shift) == kj) coef += (vals[jj] & 1u) ? -1 : 1;
            if (coef) sink(s.off[h] + (int64_t)kj, h, (int64_t)kj, coef);
        }
    }
}

__device__ inline bool edge_head(const uint64_t* keys, int64_t i, uint64_t none) {
    return keys[i] != none && (i == 0 || keys[i] != keys[i - 1]);
}

// A boundary half edge, from a to b, that no opposite one cancels.
struct RimEdge {
    double a[3], b[3];
};
// Longest boundary that the ray and the rim (k_rim) take: see signed_distance.
constexpr int kRimMost = 4096;

// The undirected edges' half edges, counted: open[0] = 1 unless every edge has
// exactly two half edges of opposite directions (a degenerate edge also opens
// the mesh); open[1] = the number of half edges left when opposite ones have
// cancelled, at least if above kRimMost, and rim = these half edges if not, in
// any order.  Called by whole wavefronts: key, number and sum (min -> max less
// max -> min) of an edge per lane, 0 half edges for none.
__device__ inline void boundary_edge(uint64_t key, uint32_t number, int sum, int vb, const double* V, int* open,
                                     RimEdge* rim) {
    if (number != 0 && (number != 2 || sum != 0)) open[0] = 1;
    // places on the list: one atomic per wavefront, none once it is too long
    const int lane = threadIdx.x & 63, copies = min(abs(sum), kRimMost + 1);
    const int upto = wave_incl_scan(copies), total = __shfl(upto, 63);
    if (total == 0) return;
    int first = 0;
    if (lane == 63) {
        first = __hip_atomic_load(open + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (first <= kRimMost) first = atomicAdd(open + 1, total);
    }
    first = __shfl(first, 63) + upto - copies;
    if (copies == 0 || first + copies > kRimMost) return;
    const int64_t lo = (int64_t)(key >> vb), hi = (int64_t)(key & ((1ull << vb) - 1ull));
    const double* a = V + 3 * (sum > 0 ? lo : hi);
    const double* b = V + 3 * (sum > 0 ? hi : lo);
    for (int c = 0; c < copies; ++c)
        for (int x = 0; x < 3; ++x) {
            rim[first + c].a[x] = a[x];
            rim[first + c].b[x] = b[x];
        }
}

// Edges by a hash table: whether a mesh is closed needs no order.  A sort of
// the half edges, which only the fans need, took 12 to 15 launches (60,000 half
// edges: 47 us; the table 14, and 57 at 600,000, bound by the atomics).  A slot
// holds key + 1 (0: empty), and in one word the number of half edges and,
// above it, their sum.  Linear probing; the table has at least 1.5 slots a
// half edge, so an empty slot ends every probe.
struct EdgeSlot {
    unsigned long long key, stat;
};
__global__ void k_edge_insert(const int32_t* F, int64_t nF, int vb, EdgeSlot* slots, int bits, int* open) {
    const int64_t h = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= 3 * nF) return;
    const int64_t t = h / 3;
    const int e = (int)(h - 3 * t);
    const uint32_t a = (uint32_t)F[3 * t + e], b = (uint32_t)F[3 * t + (e + 1) % 3];
    if (a == b) {
        open[0] = 1;
        return;
    }
    const unsigned long long key = (((unsigned long long)std::min(a, b) << vb) | std::max(a, b)) + 1ull;
    const unsigned long long mask = (1ull << bits) - 1ull;
    unsigned long long at = (key * 0x9E3779B97F4A7C15ull) >> (64 - bits);
    for (;; at = (at + 1ull) & mask) {
        unsigned long long k = __hip_atomic_load(&slots[at].key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (k == 0ull) {
            k = atomicCAS(&slots[at].key, 0ull, key);
            if (k == 0ull) k = key;
        }
        if (k == key) break;
    }
    atomicAdd(&slots[at].stat, (a > b ? 0xFFFFFFFF00000001ull : 0x0000000100000001ull));
}
__global__ void k_edge_check(const EdgeSlot* slots, int64_t n, int vb, const double* V, int* open, RimEdge* rim) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    EdgeSlot s{0ull, 0ull};
    if (i < n) s = slots[i];
    boundary_edge(s.key - 1ull, (uint32_t)s.stat, (int)(uint32_t)(s.stat >> 32), vb, V, open, rim);
}

// the same from the sorted half edges
__global__ void k_closed_check(const uint64_t* keys, const uint32_t* vals, int64_t M, uint64_t none, int vb,
                               const double* V, int* open, RimEdge* rim) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t number = 0;
    int sum = 0;
    if (i < M && keys[i] == none) open[0] = 1;
    if (i < M && edge_head(keys, i, none))
        for (int64_t j = i; j < M && keys[j] == keys[i]; ++j, ++number) sum += (vals[j] & 1u) ? -1 : 1;
    boundary_edge(i < M ? keys[i] : 0ull, number, sum, vb, V, open, rim);
}

__global__ void k_fan_node_count(const uint64_t* keys, const uint32_t* vals, int64_t M, Shape s, uint64_t none,
                                 uint32_t* node_cnt) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= M || !edge_head(keys, i, none)) return;
    edge_walk(keys, vals, i, M, s, [&](int64_t node, int, int64_t, int coef) {
        atomicAdd(&node_cnt[node], (uint32_t)abs(coef));
    });
}

// keep[node] != 0: the winding walk uses the node's fan for points outside
// its box (chosen by fan_choice on the host)
__device__ inline bool fan_kept(const uint8_t* keep, int64_t node) { return keep[node] != 0; }

__global__ void k_fan_edge_count(const uint64_t* keys, const uint32_t* vals, int64_t M, Shape s, uint64_t none,
                                 const uint8_t* keep, uint32_t* cnt) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= M) return;
    uint32_t c = 0;
    if (edge_head(keys, i, none))
        edge_walk(keys, vals, i, M, s, [&](int64_t node, int, int64_t, int coef) {
            if (fan_kept(keep, node)) c += (uint32_t)abs(coef);
        });
    cnt[i] = c;
}

__global__ void k_fan_emit(const uint64_t* keys, const uint32_t* vals, int64_t M, Shape s, uint64_t none, int vb,
                           const uint8_t* keep, const uint32_t* off, uint32_t* fan_node, uint64_t* fan_edge) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= M || !edge_head(keys, i, none)) return;
    const uint64_t lo = keys[i] >> vb, hi = keys[i] & ((1ull << vb) - 1);
    uint32_t o = off[i];
    edge_walk(keys, vals, i, M, s, [&](int64_t node, int, int64_t, int coef) {
        if (!fan_kept(keep, node)) return;
        const uint64_t e = coef > 0 ? ((lo << 32) | hi) : ((hi << 32) | lo);
        for (int r = 0; r < abs(coef); ++r) {
            fan_node[o] = (uint32_t)node;
            fan_edge[o] = e;
            ++o;
        }
    });
}

__global__ void k_fan_table(int64_t nodes, const uint32_t* node_cnt, const uint8_t* keep, const uint32_t* fan_off,
                            float4* node) {
    int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= nodes) return;
    const bool kept = fan_kept(keep, n);
    node[2 * n].w = __int_as_float((int)fan_off[n]);
    node[2 * n + 1].w = __int_as_float(kept ? (int)node_cnt[n] : -1);
}

// fan edge ends relative to the centre of their node's box (the fan apex),
// rounded once to binary32
__global__ void k_fan_coords(const uint64_t* fan_edge, const uint32_t* fan_node, int64_t E, const double* V,
                             const float4* node, float* fan) {
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    const uint64_t ab = fan_edge[e];
    const int64_t a = (int64_t)(ab >> 32), b = (int64_t)(ab & 0xffffffffull);
    const int64_t n = fan_node[e];
    const double c[3] = {fan_apex(node[2 * n].x, node[2 * n + 1].x), fan_apex(node[2 * n].y, node[2 * n + 1].y),
                         fan_apex(node[2 * n].z, node[2 * n + 1].z)};
    for (int x = 0; x < 3; ++x) {
        fan[6 * e + x] = (float)(V[3 * a + x] - c[x]);
        fan[6 * e + 3 + x] = (float)(V[3 * b + x] - c[x]);
    }
}

// kept fan edges per node (0 for dropped fans and buckets), for the scan
__global__ void k_fan_kept_count(int64_t nodes, const uint32_t* node_cnt, const uint8_t* keep, uint32_t* kept) {
    int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= nodes) return;
    kept[n] = fan_kept(keep, n) ? node_cnt[n] : 0u;
}

// Which nodes keep their fan, bottom-up with a cost per point outside the
// node: a visit is one node read; a fan adds ceil(edges / 64) rounds of
// solid angles, a leaf one round of its triangles, and descending the costs
// of the children.  A node keeps its fan when that is no dearer than
// descending.  Either way the winding number is exact; only the work varies.
// Nodes below the leaf level are never visited and keep nothing.
std::vector<uint8_t> fan_choice(const Shape& s, int leaf, const std::vector<uint32_t>& node_cnt) {
    std::vector<uint8_t> keep(node_cnt.size(), 0);
    std::vector<double> cost(node_cnt.size(), 0.0);
    for (int h = leaf; h <= s.H; ++h)
        for (int64_t k = 0; k < s.count[h]; ++k) {
            const int64_t n = s.off[h] + k;
            if (h == leaf) {
                cost[n] = 2.0;
                continue;
            }
            const int64_t c0 = s.off[h - 1] + 2 * k;
            const double down = 1.0 + cost[c0] + (2 * k + 1 < s.count[h - 1] ? cost[c0 + 1] : 0.0);
            const double fan = 1.0 + std::ceil(node_cnt[n] / 64.0);
            keep[n] = fan <= down;
            cost[n] = std::min(fan, down);
        }
    return keep;
}

int bits_for(uint64_t maxval) {
    int b = 1;
    while (b < 64 && (maxval >> b) != 0) ++b;
    return b;
}

// ---------------------------------------------------------- radix sort ----
// Stable LSD radix sort on the low `bits` bits of the keys, 8-bit digits,
// three launches per digit:
//   - k_rs_hist: the digit histogram of each tile of ROUNDS * 256 keys (LDS
//     atomics), stored digit-major, hist[d * tiles + tile];
//   - k_rs_offsets: one workgroup per digit scans that digit's row of tile
//     counts (exclusive) and stores the row total;
//   - k_rs_scatter: each tile starts every digit at the sum of the smaller
//     digits' totals plus its row offset, then, in ROUNDS rounds of 256 keys
//     in input order, ranks every key among the keys of its digit before it (a
//     mask of the wavefront's lanes with the same digit from 8 ballots, and
//     per-wave counts in LDS) and writes key and value there.
// Keys with equal digits keep their input order within a tile, and tiles
// follow one another in the offsets, so every pass is stable and equal keys
// end in their input order, which the triangle order and the fan edge order
// rely on.
constexpr int kRsThreads = 256, kRsBins = 256;
static_assert(kRsThreads == kRsBins, "one histogram bin per thread");

template <int ROUNDS, class K>
__global__ __launch_bounds__(kRsThreads) void k_rs_hist(const K* keys, int64_t n, int shift, uint32_t* hist,
                                                       int64_t tiles) {
    __shared__ uint32_t h[kRsBins];
    h[threadIdx.x] = 0u;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * (ROUNDS * kRsThreads);
    for (int j = 0; j < ROUNDS; ++j) {
        const int64_t i = base + (int64_t)j * kRsThreads + threadIdx.x;
        if (i < n) atomicAdd(&h[(uint32_t)(keys[i] >> shift) & (kRsBins - 1)], 1u);
    }
    __syncthreads();
    hist[(int64_t)threadIdx.x * tiles + blockIdx.x] = h[threadIdx.x];
}

// exclusive scan of 256 values of a 256-thread block (valid in every thread)
__device__ inline uint32_t block_excl_scan256(uint32_t v, uint32_t* sh) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t incl = wave_incl_scan(v);
    if (lane == 63) sh[w] = incl;
    __syncthreads();
    uint32_t before = 0;
    for (int q = 0; q < w; ++q) before += sh[q];
    __syncthreads();
    return before + incl - v;
}

// row d = blockIdx.x of the digit-major tile counts -> exclusive offsets
// within the digit; the row total to tot[d]
__global__ __launch_bounds__(kRsThreads) void k_rs_offsets(uint32_t* hist, int64_t tiles, uint32_t* tot) {
    __shared__ uint32_t sh[kRsThreads / 64 + 1];
    uint32_t* row = hist + (int64_t)blockIdx.x * tiles;
    uint32_t carry = 0;
    for (int64_t b0 = 0; b0 < tiles; b0 += kRsThreads) {
        const int64_t b = b0 + threadIdx.x;
        const uint32_t v = b < tiles ? row[b] : 0u;
        const uint32_t ex = block_excl_scan256(v, sh);
        if (b < tiles) row[b] = carry + ex;
        if (threadIdx.x == kRsThreads - 1) sh[kRsThreads / 64] = ex + v;
        __syncthreads();
        carry += sh[kRsThreads / 64];
        __syncthreads();
    }
    if (threadIdx.x == 0) tot[blockIdx.x] = carry;
}

template <int ROUNDS, class K, class V>
__global__ __launch_bounds__(kRsThreads) void k_rs_scatter(const K* kin, const V* vin, K* kout, V* vout, int64_t n,
                                                          int shift, const uint32_t* off, int64_t tiles,
                                                          const uint32_t* tot) {
    constexpr int kW = kRsThreads / 64;
    __shared__ uint32_t next[kRsBins];       // this tile's next output position per digit
    __shared__ uint32_t wcnt[kW][kRsBins];   // keys per digit in each wavefront of the current round
    __shared__ uint32_t sh[kW];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t before = (1ull << lane) - 1ull;
    // digit d starts after every smaller digit's keys and this digit's keys of earlier tiles
    const uint32_t digit_base = block_excl_scan256(tot[threadIdx.x], sh);
    next[threadIdx.x] = digit_base + off[(int64_t)threadIdx.x * tiles + blockIdx.x];
    const int64_t base = (int64_t)blockIdx.x * (ROUNDS * kRsThreads);
    for (int j = 0; j < ROUNDS; ++j) {
        const int64_t i = base + (int64_t)j * kRsThreads + threadIdx.x;
        const bool valid = i < n;
        const K k = valid ? kin[i] : K(0);
        const uint32_t d = (uint32_t)(k >> shift) & (kRsBins - 1);
        uint64_t same = __ballot(valid);   // lanes holding a key with this lane's digit
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            const bool set = (d >> bit) & 1u;
            const uint64_t m = __ballot(set);
            same &= set ? m : ~m;
        }
        for (int q = threadIdx.x; q < kW * kRsBins; q += kRsThreads) (&wcnt[0][0])[q] = 0u;
        __syncthreads();
        const uint32_t rank = (uint32_t)__popcll(same & before);
        if (valid && rank == 0) wcnt[w][d] = (uint32_t)__popcll(same);
        __syncthreads();
        uint32_t pos = 0;
        if (valid) {
            pos = next[d] + rank;
            for (int q = 0; q < w; ++q) pos += wcnt[q][d];
        }
        __syncthreads();
        uint32_t round_total = 0;
        for (int q = 0; q < kW; ++q) round_total += wcnt[q][threadIdx.x];
        next[threadIdx.x] += round_total;
        if (valid) {
            kout[pos] = k;
            if (vout) vout[pos] = vin[i];
        }
        __syncthreads();
    }
}

// sorts keys (and vals, when given) in place; n below 2^32
template <int ROUNDS, class K, class V>
void radix_sort_tiles(DBuf<K>& keys, DBuf<V>* vals, int64_t n, int bits, hipStream_t st) {
    const int64_t tiles = (n + ROUNDS * kRsThreads - 1) / (ROUNDS * kRsThreads);
    DBuf<K> k2(n);
    DBuf<V> v2(vals ? n : 0);
    DBuf<uint32_t> hist(kRsBins * tiles), tot(kRsBins);
    for (int shift = 0; shift < bits; shift += 8) {
        hipLaunchKernelGGL((k_rs_hist<ROUNDS, K>), dim3((unsigned)tiles), dim3(kRsThreads), 0, st, (const K*)keys.p, n,
                           shift, hist.p, tiles);
        ITS_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_rs_offsets, dim3(kRsBins), dim3(kRsThreads), 0, st, hist.p, tiles, tot.p);
        ITS_LAUNCH_CHECK();
        hipLaunchKernelGGL((k_rs_scatter<ROUNDS, K, V>), dim3((unsigned)tiles), dim3(kRsThreads), 0, st,
                           (const K*)keys.p, vals ? (const V*)vals->p : (const V*)nullptr, k2.p,
                           vals ? v2.p : (V*)nullptr, n, shift, (const uint32_t*)hist.p, tiles, (const uint32_t*)tot.p);
        ITS_LAUNCH_CHECK();
        std::swap(keys, k2);
        if (vals) std::swap(*vals, v2);
    }
}
// Tiles of 2048 keys, or of 512 below kRsSmall keys: a tile's rounds follow
// one another, and 2048-key tiles would leave most CUs without one.
constexpr int64_t kRsSmall = int64_t(1) << 20;
template <class K, class V>
void radix_sort(DBuf<K>& keys, DBuf<V>* vals, int64_t n, int bits, hipStream_t st) {
    if (n <= 1 || bits <= 0) return;
    ITS_REQUIRE(n < (int64_t(1) << 32), ITS_E_RANGE, "radix sort of 2^32 keys or more");
    if (n < kRsSmall) radix_sort_tiles<2>(keys, vals, n, bits, st);
    else radix_sort_tiles<8>(keys, vals, n, bits, st);
}

struct TriTree {
    Shape s{};
    int64_t nodes = 0, fans = 0;
    DBuf<Quant> q;
    DBuf<double> tris;
    DBuf<float> fan;
    DBuf<float4> sph, nrm, node;
    DBuf<int32_t> tid;
    DBuf<uint32_t> code, cell_lb;
    int cell_bits = 0;
    // half edges sorted by undirected edge, for the fans
    DBuf<uint64_t> hkeys;
    DBuf<uint32_t> hvals;
    DBuf<int32_t> pos;       // sorted position per triangle
    // open flag, boundary half edges (boundary_edge); points passed on by the
    // two packet kernels, undecided points
    DBuf<int> counts;
    DBuf<RimEdge> rim;
    int64_t M = 0;
    uint64_t none = 0;
    int vb = 0;
    TreeView view() const {
        return TreeView{s, q.p, tris.p, sph.p, nrm.p, tid.p, code.p, node.p, fan.p, cell_lb.p, cell_bits};
    }
};

// lower bound of each code prefix's range in the sorted codes: entry C
// (0 <= C <= 2^bits) is the first position whose code is >= C << (30 - bits)
__global__ void k_cell_lb(const uint32_t* code, int64_t T, int bits, uint32_t* lb) {
    const int64_t C = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (C > ((int64_t)1 << bits)) return;
    const uint64_t target = (uint64_t)C << (30 - bits);
    int64_t a = 0, b = T;
    while (a < b) {
        const int64_t m = (a + b) >> 1;
        if ((uint64_t)code[m] < target) a = m + 1; else b = m;
    }
    lb[C] = (uint32_t)a;
}

void sort_half_edges(TriTree& tr, hipStream_t st, const int32_t* d_F) {
    const int64_t M = tr.M;
    tr.hkeys.alloc(M);
    tr.hvals.alloc(M);
    hipLaunchKernelGGL(k_half_edges, dim3(blocks_for(M, kT)), dim3(kT), 0, st, d_F, M / 3, (const int32_t*)tr.pos.p,
                       tr.vb, tr.none, tr.hkeys.p, tr.hvals.p);
    ITS_LAUNCH_CHECK();
    radix_sort(tr.hkeys, &tr.hvals, M, std::min(64, 2 * tr.vb), st);
}

// Most half edges for the hash table: 2^24 slots, 256 MB, the size of the
// Infinity Cache.
constexpr int64_t kHashEdges = int64_t(1) << 23;

void tree_build(TriTree& tr, hipStream_t st, const double* d_V, int64_t nV, const int32_t* d_F, int64_t nF) {
    ITS_REQUIRE(nF > 0 && nF < (1ll << 30) && nV < (1ll << 31), ITS_E_RANGE, "mesh too large for the triangle tree (2^30 triangles, 2^31 vertices)");
    Shape& s = tr.s;
    s.T = (int32_t)nF;
    s.count[0] = (int32_t)((nF + kBucket - 1) / kBucket);
    s.off[0] = 0;
    s.H = 0;
    while (s.count[s.H] > 1) {
        ITS_REQUIRE(s.H + 1 < kMaxLevels, ITS_E_INVALID, "triangle tree too deep");
        s.count[s.H + 1] = (s.count[s.H] + 1) / 2;
        s.off[s.H + 1] = s.off[s.H] + s.count[s.H];
        ++s.H;
    }
    tr.nodes = (int64_t)s.off[s.H] + 1;

    // Morton quantisation over the centroid box
    const int nb = (int)std::min<int64_t>(256, blocks_for(nF, kT));
    DBuf<double> part(6 * (size_t)nb);
    hipLaunchKernelGGL(k_centroid_box, dim3(nb), dim3(kT), 0, st, d_V, d_F, nF, part.p);
    ITS_LAUNCH_CHECK();
    tr.q.alloc(1);
    hipLaunchKernelGGL(k_quant, dim3(1), dim3(kT), 0, st, (const double*)part.p, nb, tr.q.p);
    ITS_LAUNCH_CHECK();

    // sort triangles by centroid code (stable: ties by index)
    tr.code.alloc(nF);
    DBuf<uint32_t> tidx(nF);
    hipLaunchKernelGGL(k_tri_keys, dim3(blocks_for(nF, kT)), dim3(kT), 0, st, d_V, d_F, nF, (const Quant*)tr.q.p, tr.code.p,
                       tidx.p);
    ITS_LAUNCH_CHECK();
    radix_sort(tr.code, &tidx, nF, 30, st);
    tr.tris.alloc(9 * (size_t)nF);
    tr.sph.alloc(nF);
    tr.nrm.alloc(nF);
    tr.tid.alloc(nF);
    tr.pos.alloc(nF);
    hipLaunchKernelGGL(k_tri_gather, dim3(blocks_for(nF, kT)), dim3(kT), 0, st, (const uint32_t*)tidx.p, nF, d_V, d_F,
                       tr.tris.p, tr.sph.p, tr.nrm.p, tr.tid.p, tr.pos.p);
    ITS_LAUNCH_CHECK();
    // code-prefix table with about one prefix per triangle (3 to 21 bits)
    tr.cell_bits = 3;
    while (tr.cell_bits < 21 && ((int64_t)1 << tr.cell_bits) < nF) ++tr.cell_bits;
    const int64_t ncell = ((int64_t)1 << tr.cell_bits) + 1;
    tr.cell_lb.alloc(ncell);
    hipLaunchKernelGGL(k_cell_lb, dim3(blocks_for(ncell, kT)), dim3(kT), 0, st, (const uint32_t*)tr.code.p, nF,
                       tr.cell_bits, tr.cell_lb.p);
    ITS_LAUNCH_CHECK();

    // node boxes, one level per launch
    tr.node.alloc(2 * tr.nodes);
    hipLaunchKernelGGL(k_bucket_box, dim3(blocks_for(s.count[0], kT)), dim3(kT), 0, st, tr.tris.p, s, tr.node.p);
    ITS_LAUNCH_CHECK();
    for (int h = 1; h <= s.H; ++h) {
        hipLaunchKernelGGL(k_level_box, dim3(blocks_for(s.count[h], kT)), dim3(kT), 0, st, s, h, tr.node.p);
        ITS_LAUNCH_CHECK();
    }

    // half edges grouped by undirected edge: whether the mesh is closed, and
    // its boundary
    const int64_t M = 3 * nF;
    const int vb = bits_for((uint64_t)(nV - 1));
    tr.M = M;
    tr.vb = vb;
    tr.none = (2 * vb >= 64) ? ~0ull : ((1ull << (2 * vb)) - 1);
    tr.counts.alloc(5);
    tr.rim.alloc(kRimMost);
    ITS_HIP(hipMemsetAsync(tr.counts.p, 0, tr.counts.bytes(), st));
    if (M <= kHashEdges) {
        int bits = 1;
        while ((int64_t(1) << bits) < M + M / 2) ++bits;
        const int64_t n = int64_t(1) << bits;
        DBuf<EdgeSlot> slots(n);
        ITS_HIP(hipMemsetAsync(slots.p, 0, slots.bytes(), st));
        hipLaunchKernelGGL(k_edge_insert, dim3(blocks_for(M, kT)), dim3(kT), 0, st, d_F, nF, vb, slots.p, bits,
                           tr.counts.p);
        ITS_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_edge_check, dim3(blocks_for(n, kT)), dim3(kT), 0, st, (const EdgeSlot*)slots.p, n, vb,
                           d_V, tr.counts.p, tr.rim.p);
        ITS_LAUNCH_CHECK();
    } else {
        sort_half_edges(tr, st, d_F);
        hipLaunchKernelGGL(k_closed_check, dim3(blocks_for(M, kT)), dim3(kT), 0, st, (const uint64_t*)tr.hkeys.p,
                           (const uint32_t*)tr.hvals.p, M, tr.none, vb, d_V, tr.counts.p, tr.rim.p);
        ITS_LAUNCH_CHECK();
    }
}

// Boundary fans of the tree's nodes, for the winding-number walk; built only
// when some point needs that walk.
void fans_build(TriTree& tr, hipStream_t st, const double* d_V, const int32_t* d_F) {
    if (!tr.hkeys.p) sort_half_edges(tr, st, d_F);
    const Shape& s = tr.s;
    const int64_t M = tr.M;
    const int vb = tr.vb;
    const uint64_t none = tr.none;
    const uint64_t* hkeys = tr.hkeys.p;
    const uint32_t* hvals = tr.hvals.p;
    DBuf<uint32_t> node_cnt(tr.nodes);
    ITS_HIP(hipMemsetAsync(node_cnt.p, 0, tr.nodes * sizeof(uint32_t), st));
    hipLaunchKernelGGL(k_fan_node_count, dim3(blocks_for(M, kT)), dim3(kT), 0, st, hkeys, hvals, M, s, none,
                       node_cnt.p);
    ITS_LAUNCH_CHECK();
    DBuf<uint8_t> keep(tr.nodes);
    {
        std::vector<uint32_t> h_cnt(tr.nodes);
        ITS_HIP(hipMemcpyAsync(h_cnt.data(), node_cnt.p, tr.nodes * sizeof(uint32_t), hipMemcpyDeviceToHost, st));
        ITS_HIP(hipStreamSynchronize(st));
        const std::vector<uint8_t> h_keep = fan_choice(s, std::min(kLeafLevel, (int)s.H), h_cnt);
        ITS_HIP(hipMemcpyAsync(keep.p, h_keep.data(), tr.nodes, hipMemcpyHostToDevice, st));
        ITS_HIP(hipStreamSynchronize(st));
    }
    DBuf<uint32_t> ecnt(M);
    hipLaunchKernelGGL(k_fan_edge_count, dim3(blocks_for(M, kT)), dim3(kT), 0, st, hkeys, hvals, M, s, none,
                       (const uint8_t*)keep.p, ecnt.p);
    ITS_LAUNCH_CHECK();
    const uint64_t E = scan_exclusive_u32(ecnt.p, ecnt.p, M, st);
    ITS_REQUIRE(E < (1ull << 31), ITS_E_RANGE, "triangle tree: more than 2^31 boundary fan edges");
    tr.fans = (int64_t)E;
    DBuf<uint32_t> fan_node(std::max<uint64_t>(E, 1));
    DBuf<uint64_t> fan_edge(std::max<uint64_t>(E, 1));
    if (E) {
        hipLaunchKernelGGL(k_fan_emit, dim3(blocks_for(M, kT)), dim3(kT), 0, st, hkeys, hvals, M, s, none, vb,
                           (const uint8_t*)keep.p, (const uint32_t*)ecnt.p, fan_node.p, fan_edge.p);
        ITS_LAUNCH_CHECK();
        // stable: within a node, fan edges stay in edge-key order
        radix_sort(fan_node, &fan_edge, (int64_t)E, bits_for((uint64_t)tr.nodes), st);
    }
    DBuf<uint32_t> fan_off(tr.nodes);
    hipLaunchKernelGGL(k_fan_kept_count, dim3(blocks_for(tr.nodes, kT)), dim3(kT), 0, st, tr.nodes,
                       (const uint32_t*)node_cnt.p, (const uint8_t*)keep.p, fan_off.p);
    ITS_LAUNCH_CHECK();
    const uint64_t E2 = scan_exclusive_u32(fan_off.p, fan_off.p, tr.nodes, st);
    ITS_REQUIRE(E2 == E, ITS_E_STATE, "triangle tree: fan edge counts disagree");
    hipLaunchKernelGGL(k_fan_table, dim3(blocks_for(tr.nodes, kT)), dim3(kT), 0, st, tr.nodes,
                       (const uint32_t*)node_cnt.p, (const uint8_t*)keep.p, (const uint32_t*)fan_off.p, tr.node.p);
    ITS_LAUNCH_CHECK();
    tr.fan.alloc(6 * std::max<uint64_t>(E, 1));
    if (E) {
        hipLaunchKernelGGL(k_fan_coords, dim3(blocks_for((int64_t)E, kT)), dim3(kT), 0, st, (const uint64_t*)fan_edge.p,
                           (const uint32_t*)fan_node.p, (int64_t)E, d_V, (const float4*)tr.node.p, tr.fan.p);
        ITS_LAUNCH_CHECK();
    }
    ITS_HIP(hipStreamSynchronize(st));
}

// -------------------------------------------------------------- query -----
// The node-by-node and winding walks run one wavefront per point: the walk is the same for all
// lanes, and nodes of level kLeafLevel and below (at most 64 triangles) are
// leaves whose triangles the 64 lanes take one each.  Per-lane results are
// combined by a fixed butterfly, so nothing depends on timing.
constexpr int kWavesPerBlock = kT / 64;

struct NodeRec {
    float4 lo, hi;
    int first, count;
};
__device__ inline NodeRec load_node(const TreeView& t, int node) {
    const float4 lo = t.node[2 * node], hi = t.node[2 * node + 1];
    return NodeRec{lo, hi, __float_as_int(lo.w), __float_as_int(hi.w)};
}

// minimum of (d2, index) over the wavefront, ties to the lower index
__device__ inline void wave_argmin(double& d2, int32_t& id) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double od = __shfl_xor(d2, o, 64);
        const int32_t oi = __shfl_xor(id, o, 64);
        if (od < d2 || (od == d2 && oi < id)) {
            d2 = od;
            id = oi;
        }
    }
}

// Values that are equal in every lane are moved to scalar registers, which
// the compiler cannot infer from threadIdx.x >> 6 or from shuffles.
__device__ inline int wave_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline double wave_uniform(double v) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

__device__ inline float wave_uniform_f(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// false when the bounding sphere of sorted triangle i, or its plane, is
// farther than the best distance so far.  Far from the surface the sphere's
// radius is most of what separates the candidates; the plane's distance is
// within the triangle's tilt of the true one.
__device__ inline bool sphere_within(const TreeView& t, int64_t i, const double p[3], float pm, double best) {
    const float4 S = t.sph[i];
    const float dx = (float)p[0] - S.x, dy = (float)p[1] - S.y, dz = (float)p[2] - S.z;
    const float m = bound_margin(pm + fmaxf(fabsf(S.x), fmaxf(fabsf(S.y), fabsf(S.z))) + S.w);
    const float lb = sqrtf(dx * dx + dy * dy + dz * dz) - S.w - m;
    if (lb > 0.f && (double)lb * (double)lb > best) return false;
    const float4 n = t.nrm[i];
    const float pb = fabsf(n.x * dx + n.y * dy + n.z * dz) - m;
    return !(pb > 0.f && (double)pb * (double)pb > best);
}
// binary64 distance of sorted triangle i (when take), merged over the
// wavefront into (best, bt)
__device__ inline void tri_nearest(const TreeView& t, int64_t i, bool take, const double p[3], double& best,
                                   int32_t& bt) {
    double d2 = INFINITY;
    int32_t id = 0x7fffffff;
    if (take) {
        const double* T = t.tris + 9 * i;
        d2 = point_tri_dist2(p, T, T + 3, T + 6);
        id = t.tid[i];
        // a degenerate triangle can give 0/0; like a plain "d2 < best"
        // scan, a NaN never wins (and must not reach the butterfly)
        if (!(d2 <= INFINITY)) {
            d2 = INFINITY;
            id = 0x7fffffff;
        }
    }
    wave_argmin(d2, id);
    if (d2 < best || (d2 == best && id < bt)) {
        best = d2;
        bt = id;
    }
    best = wave_uniform(best);
    bt = wave_uniform(bt);
}
// nearest triangle of a leaf, one triangle per lane; a triangle whose
// bounding sphere is farther than the best so far is skipped
__device__ inline void leaf_nearest(const TreeView& t, int h, int64_t k, int lane, const double p[3], float pm,
                                    double& best, int32_t& bt) {
    const int64_t i = node_first(h, k) + lane;
    const bool take = i < node_last(t.s, h, k) && sphere_within(t, i, p, pm, best);
    tri_nearest(t, i, take, p, best, bt);
}

// true when no point of the box can be within the best distance found so
// far: binary32 distance to the box (boxes are rounded outward, so they hold
// every vertex), reduced by a margin that covers its rounding
__device__ inline float box_lb(const float pf[3], float pm, float4 lo, float4 hi) {
    const float l[3] = {lo.x, lo.y, lo.z}, u[3] = {hi.x, hi.y, hi.z};
    float d2 = 0.f, sc = pm;
    for (int a = 0; a < 3; ++a) {
        const float e = fmaxf(fmaxf(l[a] - pf[a], pf[a] - u[a]), 0.f);
        d2 += e * e;
        sc = fmaxf(sc, fmaxf(fabsf(l[a]), fabsf(u[a])));
    }
    return sqrtf(d2) - bound_margin(sc);
}
__device__ inline bool lb_beyond(float lb, double best) { return lb > 0.f && (double)lb * (double)lb > best; }
__device__ inline bool box_beyond(const float pf[3], float pm, float4 lo, float4 hi, double best) {
    return lb_beyond(box_lb(pf, pm, lo, hi), best);
}

// the writes of some lanes are read by other lanes of the same wavefront
__device__ inline void lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// The frontier walks start at the lowest level of at most `most` nodes (not
// below the leaves), testing all its nodes at once, several per lane,
// instead of descending from the root one level per round.  A box holds its
// children's boxes, so a node that the walk from the root would have dropped
// with an ancestor only makes the frontier larger, never changes the result.
__device__ inline int start_level(const Shape& s, int leaf, int most) {
    int h = s.H;
    while (h > leaf && s.count[h - 1] <= most) --h;
    return h;
}

__device__ inline bool box_outside(const double p[3], float4 lo, float4 hi) {
    return p[0] < (double)lo.x || p[0] > (double)hi.x || p[1] < (double)lo.y || p[1] > (double)hi.y ||
           p[2] < (double)lo.z || p[2] > (double)hi.z;
}

// The node-by-node walk: depth first, skipping a node whose box is farther
// than the best distance so far.  For points whose frontier overflows.
__device__ void dist_dfs(const TreeView& t, int leaf, int lane, const double p[3], const float pf[3], float pm,
                         double& best, int32_t& bt) {
    int h = t.s.H, k = 0;
    while (true) {
        const NodeRec r = load_node(t, t.s.off[h] + k);
        if (!box_beyond(pf, pm, r.lo, r.hi, best)) {
            if (h > leaf) {
                --h;
                k <<= 1;
                continue;
            }
            leaf_nearest(t, h, k, lane, p, pm, best, bt);
        }
        if (!tree_next(t.s, h, k)) break;
    }
}

// ------------------------------------------------------------- packets ----
// Many points near one another (the octree's vertices above all) need almost
// the same nodes and triangles, which a wavefront per point would read and test
// once per point.  The packet kernels give a wavefront kPk neighbouring points
// and walk the tree once for all of them:
//   - k_pt_seed gives every point the exact distance to one triangle near its
//     Morton position and a sort key: the size of that distance (powers of
//     two of the mesh box), then the Morton prefix.  Points of like distance
//     and place end up side by side, so one far point does not widen the
//     search of the near ones.
//   - A packet keeps the frontier of one tree level in LDS, nodes that the
//     box of its points can need, one node per lane and round, down to the
//     buckets of 8 triangles.
//   - Every (point, bucket) pair is tested, kPk points by 64 / kPk buckets a
//     round; the pairs that pass go to an LDS queue.
//   - 64 queued pairs at a time test their bucket's 8 bounding spheres, in
//     binary32 with the margins of sphere_within; the (point, triangle) pairs
//     that pass go to a second queue and take the exact binary64 test 64 at a
//     time, whatever their points.
// Every triangle that the exact minimum (or crossing count) needs passes
// these tests, and the exact tests are those of the node-by-node walks, so the
// results are theirs bit for bit.  Bound by vector instructions (about 3,800
// per packet of 16 points, 65 % of the issue slots; a wavefront per point took
// over 1,200 per point): 200,000 triangles and 554,122 octree vertices,
// distances 2,736 -> 370 us and 169 us for the 2 % of points on the second
// pass, crossings 1,692 -> 270 us, seeds 58 us and their sort 75 us.
//
// Packets whose frontier would overflow put their points on a list, which the
// second pass walks one point a wavefront (k_dist_point, k_ray_point), down to
// leaves of 64 triangles.  There a frontier that would overflow stays at its
// level, and all leaves below its nodes are tested.
constexpr int kPk = 16;
constexpr int kFrontPacket = 384, kFrontPoint = 512;   // nodes per frontier of the two passes
constexpr int kPairQueue = 128;  // (point, bucket): below 64 before a round, up to 64 a round
constexpr int kTriQueue = 576;   // (point, triangle): below 64 before a round, up to 512 a round
constexpr int kSeedWindow = 16;  // sorted triangles looked at around the Morton position

// The points of a pass: n, in the given order, or those of a list whose length
// is in device memory; both null: points 0 .. n - 1.
struct Work {
    int64_t n;
    const uint32_t* list;
    const unsigned* list_n;
    __device__ int64_t size() const { return list_n ? (int64_t)*list_n : n; }
    __device__ int64_t point(int64_t at) const { return list ? (int64_t)list[at] : at; }
};

// Margin for binary32 tests of a point (largest coordinate pm) against any
// box or sphere of the tree
__device__ inline float root_scale(const NodeRec& root) {
    float sc = 0.f;
    const float l[3] = {root.lo.x, root.lo.y, root.lo.z}, u[3] = {root.hi.x, root.hi.y, root.hi.z};
    for (int a = 0; a < 3; ++a) sc = fmaxf(sc, fmaxf(fabsf(l[a]), fabsf(u[a])));
    return sc;
}

__device__ inline float wave_min_f(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
    return wave_uniform_f(v);
}
__device__ inline float wave_max_f(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return wave_uniform_f(v);
}

constexpr int kSeedKeyBits = 24;
// d2_out, at_out: exact squared distance and sorted position of the triangle near p
__global__ void k_pt_seed(TreeView t, const double* pts, int64_t N, uint32_t* key, uint32_t* idx, double* d2_out,
                          int32_t* at_out) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (int64_t)gridDim.x * blockDim.x) {
        const double p[3] = {pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]};
        const uint32_t c = quant_code(*t.q, p);
        const uint32_t C = c >> (30 - t.cell_bits);
        int64_t a = t.cell_lb[C], b = t.cell_lb[C + 1];
        while (a < b) {
            const int64_t m = (a + b) >> 1;
            if (t.code[m] < c) a = m + 1; else b = m;
        }
        const int64_t lo = max((int64_t)0, min(a, (int64_t)t.s.T) - kSeedWindow / 2);
        const int64_t hi = min((int64_t)t.s.T, lo + kSeedWindow);
        const float pf[3] = {(float)p[0], (float)p[1], (float)p[2]};
        float near2 = INFINITY;
        int64_t j = min(a, (int64_t)t.s.T - 1);
        for (int64_t k = lo; k < hi; ++k) {
            const float4 S = t.sph[k];
            const float dx = pf[0] - S.x, dy = pf[1] - S.y, dz = pf[2] - S.z;
            const float d2 = dx * dx + dy * dy + dz * dz;
            if (d2 < near2) {
                near2 = d2;
                j = k;
            }
        }
        const NodeRec root = load_node(t, t.s.off[t.s.H]);
        const float ext = fmaxf(root.hi.x - root.lo.x, fmaxf(root.hi.y - root.lo.y, root.hi.z - root.lo.z));
        // Away from the surface the Morton position says little (a tenth of the
        // seeds are over twice as far as the nearest triangle), and the reach of
        // a packet grows with it: such a point also descends the tree, to the
        // child whose box is nearer by its nearest and farthest corner together,
        // and looks at that bucket.
        if (near2 > ext * ext * (1.f / (128.f * 128.f))) {
            int k = 0;
            for (int h = t.s.H; h > 0; --h) {
                float m[2] = {INFINITY, INFINITY};
                for (int c = 0; c < 2; ++c) {
                    if (2 * k + c >= t.s.count[h - 1]) break;
                    const NodeRec r = load_node(t, t.s.off[h - 1] + 2 * k + c);
                    const float l[3] = {r.lo.x, r.lo.y, r.lo.z}, u[3] = {r.hi.x, r.hi.y, r.hi.z};
                    m[c] = 0.f;
                    for (int x = 0; x < 3; ++x) {
                        const float e = fmaxf(fmaxf(l[x] - pf[x], pf[x] - u[x]), 0.f);
                        const float f = fmaxf(fabsf(pf[x] - l[x]), fabsf(pf[x] - u[x]));
                        m[c] += e * e + f * f;
                    }
                }
                k = 2 * k + (m[1] < m[0] ? 1 : 0);
            }
            for (int q = k * kBucket; q < min((k + 1) * kBucket, t.s.T); ++q) {
                const float4 S = t.sph[q];
                const float dx = pf[0] - S.x, dy = pf[1] - S.y, dz = pf[2] - S.z;
                const float d2 = dx * dx + dy * dy + dz * dz;
                if (d2 < near2) {
                    near2 = d2;
                    j = q;
                }
            }
        }
        const double* T = t.tris + 9 * j;
        double best = point_tri_dist2(p, T, T + 3, T + 6);
        if (!(best <= INFINITY)) best = INFINITY;   // a degenerate triangle never wins
        // distance classes: below 1/128 of the box, then one per power of two
        const float rel = sqrtf((float)best) * 128.f;
        uint32_t cls = 0;
        for (float lim = ext; cls < 7 && !(rel < lim); lim *= 2.f) ++cls;
        key[i] = (cls << 21) | (c >> 9);   // kSeedKeyBits bits
        idx[i] = (uint32_t)i;
        d2_out[i] = best;
        at_out[i] = (int32_t)j;
    }
}

// bucket j of the frontier: its nodes are of `level`, each standing for the
// 2^level buckets below it
__device__ inline int front_bucket(const uint32_t* list, int level, uint32_t j) {
    return (int)((list[j >> level] << level) | (j & ((1u << level) - 1u)));
}

// appends v of the lanes with take to a queue of n entries
__device__ inline void queue_push(uint32_t* queue, int& n, bool take, uint32_t v, uint64_t below) {
    const uint64_t m = __ballot(take);
    if (take) queue[n + __popcll(m & below)] = v;
    n += __popcll(m);
}

// The walk starts at the lowest level of at most this many nodes, all loaded
// at once.  Packets go down to the buckets.  A single point (P = 1) stops at the
// leaves, nodes of 64 triangles.
constexpr int start_nodes(int P) { return P > 1 ? 256 : 512; }
constexpr int stop_level(int P) { return P > 1 ? 0 : 3; }
static_assert(start_nodes(1) <= kFrontPoint, "the start level always fits");

// 64 boxes, loaded one per lane and read by the lanes of any point
struct BoxStage {
    float4 lo[64], hi[64];
    __device__ void fill(const TreeView& t, int node, int lane) {
        const float4 l = t.node[2 * node], h = t.node[2 * node + 1];
        lds_fence();
        lo[lane] = l;
        hi[lane] = h;
        lds_fence();
    }
};

// Frontier of a packet: nodes of one level that some point needs, from the
// start level down, one node (pair) per lane and round.  keep(lo, hi) is the
// test with the box of all points; lists longer than kPkRefine are cut down
// to the nodes that need(lo, hi) holds for with one of the points (P points
// by 64 / P nodes a round).  Both must hold for a node whenever they hold
// for one of its children.  Returns the count (list in fk[cur], nodes of
// `level`).  A list that would overflow ends the walk: -1 with several
// points, the list of the level above with one.
constexpr int kPkRefine = 40;
template <int P, int FRONT, class Keep, class Need>
__device__ inline int packet_frontier(const TreeView& t, int start, int lane, uint32_t (*fk)[FRONT], BoxStage* box,
                                      int& cur, int& level, Keep&& keep, Need&& need) {
    constexpr int SUB = 64 / P, kQ = start_nodes(P) / 64, stop = stop_level(P);
    const uint64_t below = (1ull << lane) - 1ull;
    const int slot = lane / P;
    const int count = t.s.count[start];
    int n = 0;
    cur = 0;
    bool kp[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
        kp[q] = false;
        if (lane + 64 * q < count) {
            const NodeRec r = load_node(t, t.s.off[start] + lane + 64 * q);
            kp[q] = keep(r.lo, r.hi);
        }
    }
    lds_fence();   // the lists of the packet before
    level = start;
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
        if (P > 1 && n + __popcll(__ballot(kp[q])) > FRONT) return -1;
        queue_push(fk[0], n, kp[q], (uint32_t)(lane + 64 * q), below);
    }
    lds_fence();
    for (int h = start; h > stop && n > 0; --h) {
        if (P > 1 && n > kPkRefine) {
            int m = 0;
            for (int j0 = 0; j0 < n; j0 += 64) {
                const uint32_t k = j0 + lane < n ? fk[cur][j0 + lane] : 0u;
                box->fill(t, t.s.off[h] + (int)k, lane);
                uint64_t used = 0;   // nodes of this round that some point needs
                const int rounds = (min(64, n - j0) + SUB - 1) / SUB;
                for (int r = 0; r < rounds; ++r) {
                    const int b = r * SUB + slot;
                    const uint64_t votes = __ballot(need(box->lo[b], box->hi[b]));
#pragma unroll
                    for (int q = 0; q < SUB; ++q)
                        if ((votes >> (q * P)) & ((1ull << P) - 1ull)) used |= 1ull << (r * SUB + q);
                }
                queue_push(fk[cur ^ 1], m, j0 + lane < n && ((used >> lane) & 1ull), k, below);
            }
            lds_fence();
            cur ^= 1;
            n = m;
        }
        const int64_t coff = t.s.off[h - 1];
        const int ccount = t.s.count[h - 1];
        int m = 0;
        for (int j0 = 0; j0 < n; j0 += 64) {
            const int j = j0 + lane;
            bool keep0 = false, keep1 = false;
            uint32_t c0 = 0;
            if (j < n) {
                c0 = 2u * fk[cur][j];
                const NodeRec r0 = load_node(t, (int)(coff + c0));
                const bool two = (int)c0 + 1 < ccount;
                const NodeRec r1 = load_node(t, (int)(coff + c0 + (two ? 1u : 0u)));
                keep0 = keep(r0.lo, r0.hi);
                keep1 = two && keep(r1.lo, r1.hi);
            }
            const uint64_t m0 = __ballot(keep0), m1 = __ballot(keep1);
            const int tot = __popcll(m0) + __popcll(m1);
            if (m + tot > FRONT) return P > 1 ? -1 : n;
            const int pos = m + __popcll(m0 & below) + __popcll(m1 & below);
            if (keep0) fk[cur ^ 1][pos] = c0;
            if (keep1) fk[cur ^ 1][pos + (keep0 ? 1 : 0)] = c0 + 1u;
            m += tot;
        }
        lds_fence();
        cur ^= 1;
        n = m;
        level = h - 1;
    }
    return n;
}

// The frontier of a single point
template <class Keep>
__device__ inline int point_frontier(const TreeView& t, int start, int lane, uint32_t (*fk)[kFrontPoint], int& cur,
                                     int& level, Keep&& keep) {
    return packet_frontier<1, kFrontPoint>(t, start, lane, fk, nullptr, cur, level, keep, keep);
}

// The second pass: one point a wavefront.  Its frontier's nodes, of `level`, each
// stand for the 2^(level - leaf) leaves below.  64 leaves are tested a round,
// one per lane: box(lo, hi) gives a number, and keep(number) tells whether the
// leaf is needed, now and after the exact tests before it.  The triangles of
// the leaves that are, one per lane and kLeaves leaves at a time, go through tri
// to a queue, and exact takes them 64 at a time.
//
// Leaves, and not the packets' pairs of point and bucket: with one point those
// read 8 spheres per lane from 64 places of memory at once, and a bucket's box
// saves little where most triangles below a leaf are needed.  Bound by vector
// instructions, mostly the exact tests', and by latency for few points.
// 300,000 points in the middle of a torus of 20,000 triangles, as far from all
// of it: 14.6 ms in pairs, 8.0 so (the whole call); 300,000 around a mesh of two
// parts far apart: 16.9 and 8.4; the second pass of the 554,122 vertices of the
// 200,000-triangle knot: 306 and 169 us.  Two leaves at a time were 1 % slower
// over 245 sets of points, and so was the exact distance of the seed's leaf
// before the frontier.
constexpr int kLeaves = 4;
constexpr int kLeafQueue = 64 + 64 * kLeaves;   // below 64 before a round
template <class Box, class Keep, class Tri, class Exact>
__device__ inline void point_leaves(const TreeView& t, const uint32_t* list, int n, int level, int leaf, int lane,
                                    uint32_t* queue, Box&& box, Keep&& keep, Tri&& tri, Exact&& exact) {
    const uint64_t below = (1ull << lane) - 1ull;
    const int shift = level - leaf, nl = n << shift;
    int qn = 0;
    auto flush = [&](int cnt) {   // the last cnt queued triangles
        lds_fence();
        qn -= cnt;
        const uint32_t k = queue[qn + (lane < cnt ? lane : 0)];
        lds_fence();
        exact((int64_t)k, lane < cnt);
    };
    for (int j0 = 0; j0 < nl; j0 += 64) {
        const int j = j0 + lane;
        int l = 0;
        bool have = false;
        float far = 0.f;
        if (j < nl) {
            l = (int)((list[j >> shift] << shift) | (uint32_t)(j & ((1 << shift) - 1)));
            have = l < t.s.count[leaf];
            if (have) {
                const NodeRec r = load_node(t, t.s.off[leaf] + l);
                far = box(r.lo, r.hi);
            }
        }
        uint64_t left = __ballot(have && keep(far));
        while (left != 0ull) {
            int k[kLeaves];
            bool pass[kLeaves];
            float4 S[kLeaves];
#pragma unroll
            for (int q = 0; q < kLeaves; ++q) {
                const int b = left != 0ull ? __ffsll((unsigned long long)left) - 1 : 0;
                const int64_t lk = __builtin_amdgcn_readlane(l, b);
                k[q] = (int)node_first(leaf, lk) + lane;
                pass[q] = left != 0ull && k[q] < node_last(t.s, leaf, lk);
                S[q] = t.sph[pass[q] ? k[q] : 0];
                left &= left - 1ull;
            }
#pragma unroll
            for (int q = 0; q < kLeaves; ++q)
                queue_push(queue, qn, pass[q] && tri(k[q], S[q]), (uint32_t)k[q], below);
            if (qn < 64) continue;
            while (qn >= 64) flush(64);
            left &= __ballot(keep(far));
        }
    }
    if (qn > 0) flush(qn);
}

// out holds the seeds' squared distances on entry
__global__ __launch_bounds__(64, 5) void k_dist_point(TreeView t, const double* pts, Work work, const int32_t* seed_at,
                                                     double* out, int32_t* tri_out) {
    __shared__ uint32_t fk[2][kFrontPoint];
    __shared__ uint32_t queue[kLeafQueue];
    const int lane = threadIdx.x;
    const int64_t N = work.size();
    const NodeRec root = load_node(t, t.s.off[t.s.H]);
    const float rs = root_scale(root);
    const int leaf = std::min(kLeafLevel, (int)t.s.H);
    const int start = start_level(t.s, leaf, start_nodes(1));
    for (int64_t g = blockIdx.x; g < N; g += gridDim.x) {
        const int64_t i = work.point(N - 1 - g);
        const double p[3] = {wave_uniform(pts[3 * i]), wave_uniform(pts[3 * i + 1]), wave_uniform(pts[3 * i + 2])};
        const float pf[3] = {(float)p[0], (float)p[1], (float)p[2]};
        const float pm = fmaxf(fabsf(pf[0]), fmaxf(fabsf(pf[1]), fabsf(pf[2])));
        const float M = bound_margin(pm + 4.f * rs);   // covers any centre and radius of the tree
        const int seed = wave_uniform(seed_at[i]);
        double best = wave_uniform(out[i]);
        int32_t bt = best < INFINITY ? t.tid[seed] : 0x7fffffff;
        if (isfinite(pf[0]) && isfinite(pf[1]) && isfinite(pf[2])) {
            auto upper = [M](double d2) { return wave_uniform_f(sqrtf((float)d2) * 1.000001f + M); };
            float ubm = upper(best);   // upper bound of the distance, with the margin
            // points much farther than a triangle's size also test the planes
            const float near = 4.f * t.sph[seed].w;
            auto box = [&](float4 lo, float4 hi) {
                const float ex = fmaxf(fmaxf(lo.x - pf[0], pf[0] - hi.x), 0.f);
                const float ey = fmaxf(fmaxf(lo.y - pf[1], pf[1] - hi.y), 0.f);
                const float ez = fmaxf(fmaxf(lo.z - pf[2], pf[2] - hi.z), 0.f);
                return ex * ex + ey * ey + ez * ez;
            };
            auto keep = [&](float d2) { return !(d2 > ubm * ubm); };
            int cur = 0, level = 0;
            const int n = point_frontier(t, start, lane, fk, cur, level,
                                         [&](float4 lo, float4 hi) { return keep(box(lo, hi)); });
            point_leaves(t, fk[cur], n, level, leaf, lane, queue, box, keep, [&](int k, float4 S) {
                const float dx = pf[0] - S.x, dy = pf[1] - S.y, dz = pf[2] - S.z, lim = ubm + S.w;
                if (dx * dx + dy * dy + dz * dz > lim * lim) return false;
                if (!(ubm > near)) return true;
                const float4 nr = t.nrm[k];
                return !(fabsf(nr.x * dx + nr.y * dy + nr.z * dz) > ubm);
            }, [&](int64_t k, bool take) {
                tri_nearest(t, k, take, p, best, bt);
                ubm = fminf(ubm, upper(best));
            });
        } else {   // a coordinate beyond binary32, or NaN
            dist_dfs(t, leaf, lane, p, pf, pm, best, bt);
        }
        if (lane == 0) {
            out[i] = sqrt(best);
            if (tri_out) tri_out[i] = bt;
        }
    }
}

// points of a packet that goes to the second pass
__device__ inline void packet_pass_on(bool valid, int64_t i, int lane, uint32_t* rest, unsigned* rest_n) {
    const uint64_t m = __ballot(valid);
    unsigned base = 0;
    if (lane == 0) base = atomicAdd(rest_n, (unsigned)__popcll(m));
    base = (unsigned)wave_uniform((int)base);
    if (valid) rest[base + __popcll(m & ((1ull << lane) - 1ull))] = (uint32_t)i;
}

// Point sets below this take the second pass alone: 3,000 packets or fewer
// leave most of the chip's 1,024 SIMDs with few wavefronts or none, 16 times as
// many wavefronts hide more, and the points' sort takes 9 launches.  In packets
// and one by one, whole call in ms: 24,000 points in the box of a
// 10,000-triangle torus 0.50 and 0.37, 48,000 0.56 and 0.50, 64,000 0.59 and
// 0.57, 100,000 0.68 and 0.74; near its surface 48,000 0.48 and 0.44, 64,000
// 0.49 and 0.50; 200,000-triangle knot, near the surface, 48,000 1.02 and 1.01,
// 64,000 1.02 and 1.11.
constexpr int64_t kPacketPoints = 49152;

// out holds the seeds' squared distances on entry
__global__ __launch_bounds__(64, 5) void k_dist_packet(TreeView t, const double* pts, Work work, const int32_t* seed_at,
                                                    double* out, int32_t* tri_out, uint32_t* rest, unsigned* rest_n) {
    constexpr int P = kPk, FRONT = kFrontPacket, SUB = 64 / P;   // buckets tested at once
    __shared__ uint32_t fk[2][FRONT];
    __shared__ BoxStage box;
    __shared__ uint32_t pairs[kPairQueue];   // frontier slot * P + point
    __shared__ uint32_t cand[kTriQueue];     // (frontier slot * 8 + triangle) * P + point
    __shared__ double sp[3][P];
    __shared__ float sub[P];               // upper bounds with margin
    __shared__ float4 sseed[P];            // bounding spheres of the points' seed triangles (centre at infinity: no bound)
    __shared__ unsigned long long sbest[P];   // bits of the best squared distance (order of non-negative doubles)
    __shared__ int32_t sid[P];
    const int lane = threadIdx.x, pt = lane & (P - 1), slot = lane / P;
    const uint64_t below = (1ull << lane) - 1ull;
    const int64_t N = work.size(), groups = (N + P - 1) / P;
    const NodeRec root = load_node(t, t.s.off[t.s.H]);
    const float rs = root_scale(root);
    const int start = start_level(t.s, std::min(stop_level(P), (int)t.s.H), start_nodes(P));
    for (int64_t g = blockIdx.x; g < groups; g += gridDim.x) {
    // the far points' packets, the longest, are last in the order and taken first
    const int64_t at = (groups - 1 - g) * P + pt;
    const bool valid = at < N;
    const int64_t i = work.point(valid ? at : N - 1);
    const double p[3] = {pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]};
    const float pf[3] = {(float)p[0], (float)p[1], (float)p[2]};
    // a coordinate beyond binary32 (or NaN) is for the node-by-node walk
    const bool wild = __ballot(!(isfinite(pf[0]) && isfinite(pf[1]) && isfinite(pf[2]))) != 0ull;
    const float pm = fmaxf(fabsf(pf[0]), fmaxf(fabsf(pf[1]), fabsf(pf[2])));
    const float M = bound_margin(pm + 4.f * rs);   // covers any centre and radius of the tree
    auto upper = [M](double d2) { return sqrtf((float)d2) * 1.000001f + M; };
    const double seed_d2 = out[i];
    float ubm = upper(seed_d2);   // upper bound of the distance, with the margin
    lds_fence();   // the packet before has been read
    if (slot == 0) {
        const int32_t j = seed_at[i];
        for (int a = 0; a < 3; ++a) sp[a][pt] = p[a];
        // A triangle with a unit normal has a distance to every point, no larger
        // than its centre's.  A face (a, a, c) has none (0 / 0) for the points
        // on the c side of a: it never wins, so its centre bounds nothing.
        const float4 S = t.sph[j], nr = t.nrm[j];
        const bool sound = nr.x * nr.x + nr.y * nr.y + nr.z * nr.z > 0.5f;
        sseed[pt] = sound ? S : make_float4(INFINITY, 0.f, 0.f, S.w);
        sbest[pt] = (unsigned long long)__double_as_longlong(seed_d2);
        sid[pt] = seed_d2 < INFINITY ? t.tid[j] : 0x7fffffff;
    }
    lds_fence();
    // A point's Morton position can miss a triangle that a neighbour's found:
    // the centres of all the packet's sound seeds bound its distance too.
    for (int q = slot; q < P; q += SUB) {
        const float4 S = sseed[q];
        const float dx = pf[0] - S.x, dy = pf[1] - S.y, dz = pf[2] - S.z;
        ubm = fminf(ubm, sqrtf(dx * dx + dy * dy + dz * dz) + M);
    }
#pragma unroll
    for (int o = P; o < 64; o <<= 1) ubm = fminf(ubm, __shfl_xor(ubm, o, 64));
    if (slot == 0) sub[pt] = ubm;
    // the packet's box, grown by the largest upper bound
    float blo[3], bhi[3];
    for (int a = 0; a < 3; ++a) {
        blo[a] = wave_min_f(pf[a]);
        bhi[a] = wave_max_f(pf[a]);
    }
    const float reach = wave_max_f(ubm), reach2 = reach * reach;
    // can the box hold a triangle nearer than this lane's point has found?
    auto needs = [&](float4 lo, float4 hi) {
        const float ex = fmaxf(fmaxf(lo.x - pf[0], pf[0] - hi.x), 0.f);
        const float ey = fmaxf(fmaxf(lo.y - pf[1], pf[1] - hi.y), 0.f);
        const float ez = fmaxf(fmaxf(lo.z - pf[2], pf[2] - hi.z), 0.f);
        return valid && !(ex * ex + ey * ey + ez * ez > ubm * ubm);
    };
    int cur = 0;
    int level = 0;
    const int n = wild ? -1 : packet_frontier<P, FRONT>(t, start, lane, fk, &box, cur, level, [&](float4 lo, float4 hi) {
        const float ex = fmaxf(fmaxf(lo.x - bhi[0], blo[0] - hi.x), 0.f);
        const float ey = fmaxf(fmaxf(lo.y - bhi[1], blo[1] - hi.y), 0.f);
        const float ez = fmaxf(fmaxf(lo.z - bhi[2], blo[2] - hi.z), 0.f);
        return !(ex * ex + ey * ey + ez * ez > reach2);
    }, needs);
    if (n < 0) {
        packet_pass_on(valid && slot == 0, i, lane, rest, rest_n);
        continue;
    }
    // points much farther than a triangle's size also test the planes
    const bool planes = reach > 4.f * sseed[0].w;
    int qp = 0, qt = 0;
    const int nb = n << level;   // buckets of the frontier
    uint64_t have = 0;           // which of the 64 staged buckets exist
    for (int j0 = 0;; j0 += SUB) {
        const bool more = j0 < nb;
        if (more) {
            const int j = j0 + slot;
            bool pass = false;
            if ((j0 & 63) == 0) {   // the next 64 buckets
                const int b = j0 + lane < nb ? front_bucket(fk[cur], level, (uint32_t)(j0 + lane)) : 0;
                have = __ballot(j0 + lane < nb && b < t.s.count[0]);
                box.fill(t, t.s.off[0] + min(b, t.s.count[0] - 1), lane);
            }
            if ((have >> (j & 63)) & 1ull) pass = needs(box.lo[j & 63], box.hi[j & 63]);
            queue_push(pairs, qp, pass, (uint32_t)(j * P + pt), below);
        }
        if (qp >= 64 || (!more && qp > 0)) {
            lds_fence();
            const int cnt = min(qp, 64);
            qp -= cnt;
            const bool take = lane < cnt;
            const uint32_t e = pairs[qp + (take ? lane : 0)];
            const int o = (int)(e & (P - 1));
            const uint32_t js = e / P;
            const float ox = (float)sp[0][o], oy = (float)sp[1][o], oz = (float)sp[2][o], ou = sub[o];
            const int first = front_bucket(fk[cur], level, js) * kBucket;
#pragma unroll
            for (int q = 0; q < kBucket; ++q) {
                const int k = first + q;
                const float4 S = t.sph[min(k, t.s.T - 1)];
                const float dx = ox - S.x, dy = oy - S.y, dz = oz - S.z, lim = ou + S.w;
                bool pass = take && k < t.s.T && !(dx * dx + dy * dy + dz * dz > lim * lim);
                if (planes && pass) {
                    const float4 nr = t.nrm[k];
                    pass = !(fabsf(nr.x * dx + nr.y * dy + nr.z * dz) > ou);
                }
                queue_push(cand, qt, pass, (js * kBucket + q) * P + o, below);
            }
        }
        while (qt >= 64 || (!more && qp == 0 && qt > 0)) {
            lds_fence();
            const int cnt = min(qt, 64);
            qt -= cnt;
            const bool take = lane < cnt;
            const uint32_t e = cand[qt + (take ? lane : 0)];
            const int o = (int)(e & (P - 1));
            const uint32_t jq = e / P;
            const int64_t k = (int64_t)front_bucket(fk[cur], level, jq / kBucket) * kBucket + jq % kBucket;
            const double q[3] = {sp[0][o], sp[1][o], sp[2][o]};
            const double* T = t.tris + 9 * k;
            double d2 = point_tri_dist2(q, T, T + 3, T + 6);
            int32_t id = t.tid[k];
            if (!take || !(d2 <= INFINITY)) {   // a degenerate triangle never wins
                d2 = INFINITY;
                id = 0x7fffffff;
            }
            const unsigned long long bits = (unsigned long long)__double_as_longlong(d2), pre = sbest[o];
            lds_fence();
            if (take) atomicMin(&sbest[o], bits);
            lds_fence();
            const unsigned long long now = sbest[o];
            const bool win = take && bits == now;
            if (win && now < pre) sid[o] = 0x7fffffff;   // a smaller distance: the old index does not count
            lds_fence();
            if (win) atomicMin(&sid[o], id);
            lds_fence();
            ubm = fminf(ubm, upper(__longlong_as_double((long long)sbest[pt])));
            sub[pt] = ubm;   // the same value from every lane of the point
            lds_fence();
        }
        if (!more && qp == 0 && qt == 0) break;
    }
    if (valid && slot == 0) {
        out[i] = sqrt(__longlong_as_double((long long)sbest[pt]));
        if (tri_out) tri_out[i] = sid[pt];
    }
    }
}

// Winding number: fans of the nodes the point is outside of, triangles of
// the leaves it reaches.  Level by level: the wavefront classifies all nodes
// of a level at once (one per lane) into leaves, fans (the point is outside
// the box) and nodes to descend, keeping the lists in LDS; fans carry their
// edge range and apex - p, so their sums start without another node read.
// Lists that would overflow send the point to the node-by-node walk.
constexpr int kWindFront = 128, kWindFans = 128, kWindLeaves = 64;
struct FanItem {
    int first, count;
    float z[3], lz;
};

__device__ inline float leaf_wind(const TreeView& t, int h, int64_t k, int lane, const double p[3]) {
    const int64_t j = node_first(h, k) + lane;
    if (j >= node_last(t.s, h, k)) return 0.f;
    const double* T = t.tris + 9 * j;
    return solid_angle(p, T, T + 3, T + 6);
}
__device__ inline float fan_wind(const TreeView& t, int first, int count, const float z[3], float lz, int lane) {
    float acc = 0.f;
    for (int e = lane; e < count; e += 64) {
        const float* ab = t.fan + 6 * ((int64_t)first + e);
        const float u[3] = {ab[0] + z[0], ab[1] + z[1], ab[2] + z[2]};
        const float v[3] = {ab[3] + z[0], ab[4] + z[1], ab[5] + z[2]};
        acc += fan_angle(z, lz, u, v);
    }
    return acc;
}
__device__ inline FanItem fan_item(const NodeRec& r, const double p[3]) {
    // apex - p once per node in binary64; the edge ends are stored relative
    // to the apex, so a - p = (a - apex) + (apex - p)
    FanItem f;
    f.first = r.first;
    f.count = r.count;
    f.z[0] = (float)(fan_apex(r.lo.x, r.hi.x) - p[0]);
    f.z[1] = (float)(fan_apex(r.lo.y, r.hi.y) - p[1]);
    f.z[2] = (float)(fan_apex(r.lo.z, r.hi.z) - p[2]);
    f.lz = __builtin_amdgcn_sqrtf(f.z[0] * f.z[0] + f.z[1] * f.z[1] + f.z[2] * f.z[2]);
    return f;
}

// the node-by-node walk (lists overflowed)
__device__ float wind_dfs(const TreeView& t, int leaf, int lane, const double p[3]) {
    float acc = 0.f;
    int h = t.s.H, k = 0;
    while (true) {
        const NodeRec r = load_node(t, t.s.off[h] + k);
        if (h <= leaf) {
            acc += leaf_wind(t, h, k, lane, p);
        } else if (r.count >= 0 && box_outside(p, r.lo, r.hi)) {
            const FanItem f = fan_item(r, p);
            acc += fan_wind(t, f.first, f.count, f.z, f.lz, lane);
        } else {
            --h;
            k <<= 1;
            continue;
        }
        if (!tree_next(t.s, h, k)) break;
    }
    return acc;
}

// Orientation signs with static error filters (Shewchuk 1997, the first
// stage of orient2d and orient3d): +1 or -1 when the binary64 determinant
// exceeds the bound on its rounding error, 0 when the sign is not certain.
// Nothing here may be contracted into fused multiply-adds: the bounds count
// every rounding of the products and sums as written.
constexpr double kO2dBound = 3.3306690738754716e-16;   // (3 + 16 eps) eps, eps = 2^-53
constexpr double kO3dBound = 7.7715611723761027e-16;   // (7 + 56 eps) eps
// (a - p) x (b - p), z component: > 0 when p lies left of a -> b in xy
__device__ inline int o2d_sign(double ax, double ay, double bx, double by, double px, double py) {
#pragma clang fp contract(off)
    const double l = (ax - px) * (by - py);
    const double r = (ay - py) * (bx - px);
    const double det = l - r;
    const double bound = kO2dBound * (fabs(l) + fabs(r));
    return det > bound ? 1 : (-det > bound ? -1 : 0);
}
// (a - p) . ((b - p) x (c - p))
__device__ inline int o3d_sign(const double* a, const double* b, const double* c, const double p[3]) {
#pragma clang fp contract(off)
    const double adx = a[0] - p[0], ady = a[1] - p[1], adz = a[2] - p[2];
    const double bdx = b[0] - p[0], bdy = b[1] - p[1], bdz = b[2] - p[2];
    const double cdx = c[0] - p[0], cdy = c[1] - p[1], cdz = c[2] - p[2];
    const double bdxcdy = bdx * cdy, cdxbdy = cdx * bdy;
    const double cdxady = cdx * ady, adxcdy = adx * cdy;
    const double adxbdy = adx * bdy, bdxady = bdx * ady;
    const double det = adz * (bdxcdy - cdxbdy) + bdz * (cdxady - adxcdy) + cdz * (adxbdy - bdxady);
    const double perm = (fabs(bdxcdy) + fabs(cdxbdy)) * fabs(adz) + (fabs(cdxady) + fabs(adxcdy)) * fabs(bdz) +
                        (fabs(adxbdy) + fabs(bdxady)) * fabs(cdz);
    const double bound = kO3dBound * perm;
    return det > bound ? 1 : (-det > bound ? -1 : 0);
}

// An axis ray from p: along axis w in direction sg (+1 or -1), with u, v the
// next two axes in cyclic order, so (u, v, w) is oriented like (x, y, z) and
// the (u, v) orientation of a triangle has the sign of its normal's w
// component.  Any ray gives the winding number; each point takes the axis
// direction that leaves the mesh's box soonest, which meets the fewest nodes.
struct Ray {
    int u, v, w, sg;
};
__device__ inline double sel3(const double* x, int i) { return i == 0 ? x[0] : (i == 1 ? x[1] : x[2]); }
__device__ inline float sel3(float4 x, int i) { return i == 0 ? x.x : (i == 1 ? x.y : x.z); }
__device__ inline Ray choose_ray(const double p[3], float4 lo, float4 hi) {
    Ray R{0, 1, 2, 1};
    float len = INFINITY;
    for (int a = 0; a < 3; ++a) {
        const float pa = (float)sel3(p, a);
        const float ahead = sel3(hi, a) - pa, behind = pa - sel3(lo, a);
        if (ahead < len) {
            len = ahead;
            R = Ray{(a + 1) % 3, (a + 2) % 3, a, 1};
        }
        if (behind < len) {
            len = behind;
            R = Ray{(a + 1) % 3, (a + 2) % 3, a, -1};
        }
    }
    return R;
}

// Signed crossing of the ray from p with one triangle: +1 / -1 (the sign of
// n . d, its normal against the ray direction) when the ray crosses it ahead
// of p, else 0; unsure is set when an orientation that decides this is not
// certain.
__device__ inline int tri_ray(const double* T, const double p[3], const Ray& R, bool& unsure) {
    const double* a = T;
    const double* b = T + 3;
    const double* c = T + 6;
    const double pu = sel3(p, R.u), pv = sel3(p, R.v), pw = sel3(p, R.w);
    const double au = a[R.u], av = a[R.v], aw = a[R.w];
    const double bu = b[R.u], bv = b[R.v], bw = b[R.w];
    const double cu = c[R.u], cv = c[R.v], cw = c[R.w];
    const double wmin = fmin(aw, fmin(bw, cw)), wmax = fmax(aw, fmax(bw, cw));
    // outside the (u, v) bounding rectangle, or wholly behind p: no crossing
    if (pu < fmin(au, fmin(bu, cu)) || pu > fmax(au, fmax(bu, cu)) || pv < fmin(av, fmin(bv, cv)) ||
        pv > fmax(av, fmax(bv, cv)) || (R.sg > 0 ? wmax < pw : wmin > pw))
        return 0;
    const int s1 = o2d_sign(au, av, bu, bv, pu, pv);
    const int s2 = o2d_sign(bu, bv, cu, cv, pu, pv);
    const int s3 = o2d_sign(cu, cv, au, av, pu, pv);
    const bool pos = s1 > 0 || s2 > 0 || s3 > 0, neg = s1 < 0 || s2 < 0 || s3 < 0;
    if (pos && neg) return 0;   // two certain signs disagree: outside the projection
    if (s1 == 0 || s2 == 0 || s3 == 0) {
        unsure = true;
        return 0;
    }
    // inside the projection; s1 is the (u, v) orientation of (a, b, c), the
    // sign of n_w, so n . d has the sign dir.  The ray meets the plane at
    // t = ((a - p) . n) / (n . d), n = (b - a) x (c - a), and (a - p) . n is
    // the orientation of (a, b, c, p): ahead of p when it has the sign dir
    const int dir = R.sg > 0 ? s1 : -s1;
    if (R.sg > 0 ? wmin > pw : wmax < pw) return dir;   // wholly ahead
    const int s4 = o3d_sign(a, b, c, p);
    if (s4 == 0) {
        unsure = true;
        return 0;
    }
    return s4 == dir ? dir : 0;
}

// Crossings of a packet: all its rays take the axis direction that leaves the
// mesh's box soonest from the middle of the packet (any ray gives the winding
// number), so one walk serves them all.
// decided[i] = 1 and the sign is applied when every orientation was certain
// and the lists fitted; otherwise decided[i] = 0 and the fan walk takes the
// point.  With cross given (an open mesh) the crossings and the ray's axis and
// direction are left there instead, and k_rim applies the sign.
__global__ __launch_bounds__(64, 5) void k_ray_packet(TreeView t, const double* pts, Work work, double* out,
                                                   uint8_t* decided, int* cross, unsigned* undecided, uint32_t* rest,
                                                   unsigned* rest_n) {
    constexpr int P = kPk, FRONT = kFrontPacket, SUB = 64 / P;   // buckets tested at once
    __shared__ uint32_t fk[2][FRONT];
    __shared__ BoxStage box;
    __shared__ uint32_t pairs[kPairQueue];   // frontier slot * P + point
    __shared__ uint32_t cand[kTriQueue];     // (frontier slot * 8 + triangle) * P + point
    __shared__ double sp[3][P];
    __shared__ float sf[4][P];             // u, v, place along the ray, margin
    __shared__ int scross[P], sunsure[P];
    const int lane = threadIdx.x, pt = lane & (P - 1), slot = lane / P;
    const uint64_t below = (1ull << lane) - 1ull;
    const int64_t N = work.size(), groups = (N + P - 1) / P;
    const NodeRec root = load_node(t, t.s.off[t.s.H]);
    const float rs = root_scale(root);
    const int start = start_level(t.s, std::min(stop_level(P), (int)t.s.H), start_nodes(P));
    for (int64_t g = blockIdx.x; g < groups; g += gridDim.x) {
    const int64_t at = (groups - 1 - g) * P + pt;
    const bool valid = at < N;
    const int64_t i = work.point(valid ? at : N - 1);
    const double p[3] = {pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]};
    const float pf[3] = {(float)p[0], (float)p[1], (float)p[2]};
    const bool wild = __ballot(!(isfinite(pf[0]) && isfinite(pf[1]) && isfinite(pf[2]))) != 0ull;
    double mid[3];
    for (int a = 0; a < 3; ++a) mid[a] = 0.5 * ((double)wave_min_f(pf[a]) + (double)wave_max_f(pf[a]));
    Ray R = choose_ray(mid, root.lo, root.hi);
    R.w = wave_uniform(R.w);
    R.sg = wave_uniform(R.sg);
    R.u = R.w == 2 ? 0 : R.w + 1;
    R.v = R.u == 2 ? 0 : R.u + 1;
    const bool fwd = R.sg > 0;
    const float pm = fmaxf(fabsf(pf[0]), fmaxf(fabsf(pf[1]), fabsf(pf[2])));
    const float M = bound_margin(pm + 4.f * rs);
    auto at3 = [](float x, float y, float z, int a) { return a == 0 ? x : (a == 1 ? y : z); };
    const float pu = at3(pf[0], pf[1], pf[2], R.u), pv = at3(pf[0], pf[1], pf[2], R.v);
    const float pw = at3(pf[0], pf[1], pf[2], R.w) * (fwd ? 1.f : -1.f);   // place along the ray
    lds_fence();   // the packet before has been read
    if (slot == 0) {
        for (int a = 0; a < 3; ++a) sp[a][pt] = p[a];
        sf[0][pt] = pu;
        sf[1][pt] = pv;
        sf[2][pt] = pw;
        sf[3][pt] = M;
        scross[pt] = 0;
        sunsure[pt] = 0;
    }
    const float ulo = wave_min_f(pu - M), uhi = wave_max_f(pu + M);
    const float vlo = wave_min_f(pv - M), vhi = wave_max_f(pv + M);
    const float wlo = wave_min_f(pw - M);
    // last place of a box along the ray
    auto box_far = [&](float4 lo, float4 hi) { return fwd ? sel3(hi, R.w) : -sel3(lo, R.w); };
    // does the ray of this lane's point meet the box?
    auto needs = [&](float4 lo, float4 hi) {
        return valid && !(sel3(hi, R.u) < pu - M || sel3(lo, R.u) > pu + M || sel3(hi, R.v) < pv - M ||
                          sel3(lo, R.v) > pv + M || box_far(lo, hi) < pw - M);
    };
    int cur = 0;
    int level = 0;
    const int n = wild ? -1 : packet_frontier<P, FRONT>(t, start, lane, fk, &box, cur, level, [&](float4 lo, float4 hi) {
        return !(sel3(hi, R.u) < ulo || sel3(lo, R.u) > uhi || sel3(hi, R.v) < vlo || sel3(lo, R.v) > vhi ||
                 box_far(lo, hi) < wlo);
    }, needs);
    if (n < 0) {
        packet_pass_on(valid && slot == 0, i, lane, rest, rest_n);
        continue;
    }
    int qp = 0, qt = 0;
    const int nb = n << level;   // buckets of the frontier
    uint64_t have = 0;           // which of the 64 staged buckets exist
    for (int j0 = 0;; j0 += SUB) {
        const bool more = j0 < nb;
        if (more) {
            const int j = j0 + slot;
            bool pass = false;
            if ((j0 & 63) == 0) {   // the next 64 buckets
                const int b = j0 + lane < nb ? front_bucket(fk[cur], level, (uint32_t)(j0 + lane)) : 0;
                have = __ballot(j0 + lane < nb && b < t.s.count[0]);
                box.fill(t, t.s.off[0] + min(b, t.s.count[0] - 1), lane);
            }
            if ((have >> (j & 63)) & 1ull) pass = needs(box.lo[j & 63], box.hi[j & 63]);
            queue_push(pairs, qp, pass, (uint32_t)(j * P + pt), below);
        }
        if (qp >= 64 || (!more && qp > 0)) {
            lds_fence();
            const int cnt = min(qp, 64);
            qp -= cnt;
            const bool take = lane < cnt;
            const uint32_t e = pairs[qp + (take ? lane : 0)];
            const int o = (int)(e & (P - 1));
            const uint32_t js = e / P;
            const float ou = sf[0][o], ov = sf[1][o], ow = sf[2][o], om = sf[3][o];
            const int first = front_bucket(fk[cur], level, js) * kBucket;
#pragma unroll
            for (int q = 0; q < kBucket; ++q) {
                const int k = first + q;
                const float4 S = t.sph[min(k, t.s.T - 1)];
                // wholly beside the ray or behind its start: no crossing
                const float du = ou - sel3(S, R.u), dv = ov - sel3(S, R.v), lim = S.w + om;
                const float behind = ow - sel3(S, R.w) * (fwd ? 1.f : -1.f);
                const bool pass = take && k < t.s.T && !(du * du + dv * dv > lim * lim) && !(behind > lim);
                queue_push(cand, qt, pass, (js * kBucket + q) * P + o, below);
            }
        }
        while (qt >= 64 || (!more && qp == 0 && qt > 0)) {
            lds_fence();
            const int cnt = min(qt, 64);
            qt -= cnt;
            if (lane < cnt) {
                const uint32_t e = cand[qt + lane];
                const int o = (int)(e & (P - 1));
                const uint32_t jq = e / P;
                const int64_t k = (int64_t)front_bucket(fk[cur], level, jq / kBucket) * kBucket + jq % kBucket;
                const double q[3] = {sp[0][o], sp[1][o], sp[2][o]};
                bool unsure = false;
                const int c = tri_ray(t.tris + 9 * k, q, R, unsure);
                if (c) atomicAdd(&scross[o], c);
                if (unsure) sunsure[o] = 1;
            }
            lds_fence();
        }
        if (!more && qp == 0 && qt == 0) break;
    }
    const bool mine = valid && slot == 0, unsure = mine && sunsure[pt] != 0;
    const uint64_t mu = __ballot(unsure);
    if (mu != 0ull && lane == 0) atomicAdd(undecided, (unsigned)__popcll(mu));
    if (mine) {
        decided[i] = unsure ? 0 : 1;
        if (cross) cross[i] = scross[pt] * 8 + R.w * 2 + (fwd ? 1 : 0);
        else if (!unsure && scross[pt] >= 1) out[i] = -out[i];   // winding number > 1/2
    }
    }
}

// The same for one point a wavefront
__global__ __launch_bounds__(64, 5) void k_ray_point(TreeView t, const double* pts, Work work, double* out,
                                                    uint8_t* decided, int* cross, unsigned* undecided) {
    __shared__ uint32_t fk[2][kFrontPoint];
    __shared__ uint32_t queue[kLeafQueue];
    const int lane = threadIdx.x;
    const int64_t N = work.size();
    const NodeRec root = load_node(t, t.s.off[t.s.H]);
    const float rs = root_scale(root);
    const int leaf = std::min(kLeafLevel, (int)t.s.H);
    const int start = start_level(t.s, leaf, start_nodes(1));
    for (int64_t g = blockIdx.x; g < N; g += gridDim.x) {
        const int64_t i = work.point(N - 1 - g);
        const double p[3] = {wave_uniform(pts[3 * i]), wave_uniform(pts[3 * i + 1]), wave_uniform(pts[3 * i + 2])};
        const float pf[3] = {(float)p[0], (float)p[1], (float)p[2]};
        Ray R = choose_ray(p, root.lo, root.hi);
        bool unsure = !(isfinite(pf[0]) && isfinite(pf[1]) && isfinite(pf[2]));
        int c = 0;
        if (!unsure) {
            R.w = wave_uniform(R.w);
            R.sg = wave_uniform(R.sg);
            R.u = R.w == 2 ? 0 : R.w + 1;
            R.v = R.u == 2 ? 0 : R.u + 1;
            const float dir = R.sg > 0 ? 1.f : -1.f;
            const float pm = fmaxf(fabsf(pf[0]), fmaxf(fabsf(pf[1]), fabsf(pf[2])));
            const float M = bound_margin(pm + 4.f * rs);
            const float4 pf4 = make_float4(pf[0], pf[1], pf[2], 0.f);
            const float pu = sel3(pf4, R.u), pv = sel3(pf4, R.v), pw = sel3(pf4, R.w) * dir;   // pw: place along the ray
            // does the ray meet the box?
            auto meets = [&](float4 lo, float4 hi) {
                const float last = R.sg > 0 ? sel3(hi, R.w) : -sel3(lo, R.w);
                return !(sel3(hi, R.u) < pu - M || sel3(lo, R.u) > pu + M || sel3(hi, R.v) < pv - M ||
                         sel3(lo, R.v) > pv + M || last < pw - M);
            };
            int cur = 0, level = 0;
            const int n = point_frontier(t, start, lane, fk, cur, level, meets);
            point_leaves(t, fk[cur], n, level, leaf, lane, queue,
                         [&](float4 lo, float4 hi) { return meets(lo, hi) ? 0.f : 1.f; },
                         [](float miss) { return miss == 0.f; }, [&](int, float4 S) {
                // wholly beside the ray or behind its start: no crossing
                const float du = pu - sel3(S, R.u), dv = pv - sel3(S, R.v), lim = S.w + M;
                return !(du * du + dv * dv > lim * lim) && !(pw - sel3(S, R.w) * dir > lim);
            }, [&](int64_t k, bool take) {
                if (take) c += tri_ray(t.tris + 9 * k, p, R, unsure);
            });
        }
        unsure = __ballot(unsure) != 0ull;
        c = wave_sum(c);
        if (lane == 0) {
            decided[i] = unsure ? 0 : 1;
            if (unsure) atomicAdd(undecided, 1u);
            if (cross) cross[i] = c * 8 + R.w * 2 + (R.sg > 0 ? 1 : 0);
            else if (!unsure && c >= 1) out[i] = -out[i];   // winding number > 1/2
        }
    }
}

// Signs of a mesh with a boundary, from the crossings of the ray from p along r.
// The cone over the boundary whose apex lies infinitely far along -r closes the
// mesh; the ray meets that cone nowhere.  So the winding number of mesh and cone
// together is the count of crossings, and that of the mesh is the count plus
// 1 / 4 pi times the sum over boundary half edges (a, b) of the solid angle of
// the triangle (-r, a, b).  With a, b relative to p, (u, v) across the ray and
// alpha(x) = |x| - x . r, half that angle is
//     atan2(-(a_u b_v - a_v b_u) sg, alpha(a) alpha(b) + a_u b_u + a_v b_v),
// sg the ray's direction on its axis and alpha taken without cancellation.  It
// jumps by 2 pi where the ray crosses the edge, as the count does.  Left to the
// fan walk (decided = 0): points whose ray passes an edge so closely that
// binary32 may jump on the other side, and winding numbers within 1e-5 and 1e-7
// an edge of 1/2, the sum's error away from the boundary.  One angle's error
// grows with the inverse of the point's distance to its edge: a million random
// edges in binary32 against binary64 gave at most 1.3e-5 turns at 1e-3 of the
// edge's length (mostly 6e-7) and 1.3e-4 at 1e-4, and rays that pass the edge
// closely do worse.  So a point that close to the boundary and that close to 1/2
// can get either sign, as it can from the fans, whose formula is no better there.
// Angles are summed in multiples of 2^-27: the sum does not depend on the edges'
// order.
//
// 64 points a block; its wavefronts share the edges, which are uniform and come
// by scalar loads.  Bound by vector instructions: 2 ps per (point, edge) over
// the chip, 100 us per 100 edges at 500,000 points.  Knot tube with a hole, 20,000
// triangles at 128^3: crossings 63 us and this kernel 13, where the fan walk took 1,065
// and its fans 350 with their host step.
constexpr int kRimWaves = 8;
__global__ __launch_bounds__(64 * kRimWaves) void k_rim(const RimEdge* __restrict__ rim, int n,
                                                       const double* __restrict__ pts, int64_t N, double* out,
                                                       uint8_t* decided, const int* __restrict__ cross,
                                                       unsigned* undecided) {
#pragma clang fp contract(fast)
    __shared__ long long sum[kRimWaves][64];
    __shared__ int bad[kRimWaves][64];
    const int lane = threadIdx.x & 63, wave = wave_uniform((int)(threadIdx.x >> 6));
    for (int64_t i0 = (int64_t)blockIdx.x * 64; i0 < N; i0 += (int64_t)gridDim.x * 64) {
    const int64_t i = i0 + lane, at = i < N ? i : N - 1;
    const double p[3] = {pts[3 * at], pts[3 * at + 1], pts[3 * at + 2]};
    const int c = cross[at], w = (c >> 1) & 3;
    const float sg = (c & 1) ? 1.f : -1.f;
    long long acc = 0;
    bool unsure = false;
    auto split = [&](const double* x, float& u, float& v, float& alpha) {
        const float dx = (float)(x[0] - p[0]), dy = (float)(x[1] - p[1]), dz = (float)(x[2] - p[2]);
        u = w == 0 ? dy : (w == 1 ? dz : dx);
        v = w == 0 ? dz : (w == 1 ? dx : dy);
        const float along = sg * (w == 0 ? dx : (w == 1 ? dy : dz));
        const float across = u * u + v * v;
        const float m = __builtin_amdgcn_sqrtf(across + along * along) + fabsf(along);
        alpha = along > 0.f ? across * __builtin_amdgcn_rcpf(m) : m;
    };
    for (int e = wave; e < n; e += kRimWaves) {
        float au, av, aa, bu, bv, ba;
        split(rim[e].a, au, av, aa);
        split(rim[e].b, bu, bv, ba);
        const float n1 = au * bv, n2 = av * bu, d1 = au * bu, d2 = av * bv, d0 = aa * ba;
        const float num = -sg * (n1 - n2), den = d0 + (d1 + d2);
        if (!(fabsf(num) > 1e-6f * (fabsf(n1) + fabsf(n2))) && !(den > 1e-6f * (d0 + (fabsf(d1) + fabsf(d2)))))
            unsure = true;
        acc += (long long)(int)(atan2_fit(num, den) * 134217728.f);
    }
    __syncthreads();   // the points before have been read
    sum[wave][lane] = acc;
    bad[wave][lane] = unsure ? 1 : 0;
    __syncthreads();
    if (wave != 0) continue;
    for (int k = 1; k < kRimWaves; ++k) {
        acc += sum[k][lane];
        unsure = unsure || bad[k][lane] != 0;
    }
    const bool mine = i < N && decided[at] != 0;
    const double wn = (double)(c >> 3) + (double)acc * (1.0 / (134217728.0 * 2.0 * M_PI));
    if (!(fabs(wn - 0.5) > 1e-5 + 1e-7 * n)) unsure = true;
    const uint64_t mu = __ballot(mine && unsure);
    if (mu != 0ull && lane == 0) atomicAdd(undecided, (unsigned)__popcll(mu));
    if (mine && unsure) decided[i] = 0;
    else if (mine && wn > 0.5) out[i] = -out[i];
    }
}

__global__ __launch_bounds__(kT) void k_sdf_wind(TreeView t, const double* pts, int64_t N, double* out,
                                                 const uint8_t* decided) {
    __shared__ uint32_t fk[2][kWavesPerBlock][kWindFront];   // nodes of the level being classified
    __shared__ FanItem fans[kWavesPerBlock][kWindFans];
    __shared__ uint32_t leaves[kWavesPerBlock][kWindLeaves];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t below = (1ull << lane) - 1ull;
    const int64_t nw = (int64_t)gridDim.x * kWavesPerBlock;
    const int leaf = std::min(kLeafLevel, (int)t.s.H);
    for (int64_t i = (int64_t)blockIdx.x * kWavesPerBlock + w; i < N; i += nw) {
        if (decided && decided[i]) continue;   // the ray settled its sign
        const double p[3] = {pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]};
        int n = 1, cur = 0, nf = 0, nl = 0;
        bool overflow = false;
        lds_fence();
        if (lane == 0) fk[0][w][0] = 0u;
        lds_fence();
        for (int h = t.s.H; n > 0; --h) {
            if (h <= leaf) {   // every node of this level is a leaf
                if (nl + n > kWindLeaves) {
                    overflow = true;
                    break;
                }
                for (int j = lane; j < n; j += 64) leaves[w][nl + j] = fk[cur][w][j];
                nl += n;
                lds_fence();
                break;
            }
            const int64_t off = t.s.off[h];
            const int cnext = t.s.count[h - 1];
            int m = 0;
            for (int j0 = 0; j0 < n; j0 += 64) {
                const int j = j0 + lane;
                bool is_fan = false, down = false;
                uint32_t k = 0;
                NodeRec r{};
                if (j < n) {
                    k = fk[cur][w][j];
                    r = load_node(t, (int)(off + k));
                    is_fan = r.count >= 0 && box_outside(p, r.lo, r.hi);
                    down = !is_fan;
                }
                const bool two = down && (int)(2 * k + 1) < cnext;
                const uint64_t mf = __ballot(is_fan), md = __ballot(down), m2 = __ballot(two);
                const int tf = __popcll(mf), td = __popcll(md) + __popcll(m2);
                if (nf + tf > kWindFans || m + td > kWindFront) {
                    overflow = true;
                    break;
                }
                if (is_fan) fans[w][nf + __popcll(mf & below)] = fan_item(r, p);
                if (down) {
                    const int pos = m + __popcll(md & below) + __popcll(m2 & below);
                    fk[cur ^ 1][w][pos] = 2 * k;
                    if (two) fk[cur ^ 1][w][pos + 1] = 2 * k + 1;
                }
                nf += tf;
                m += td;
            }
            lds_fence();
            if (overflow) break;
            cur ^= 1;
            n = m;
        }
        float acc = 0.f;
        if (overflow) {
            acc = wind_dfs(t, leaf, lane, p);
        } else {
            for (int f = 0; f < nf; ++f) {
                const FanItem it = fans[w][f];
                acc += fan_wind(t, it.first, it.count, it.z, it.lz, lane);
            }
            for (int l = 0; l < nl; ++l) acc += leaf_wind(t, leaf, leaves[w][l], lane, p);
        }
        const float wn = wave_sum(acc) * (float)(0.25 / M_PI);
        if (lane == 0) {
            const double d = out[i];
            out[i] = (wn > 0.5f) ? -d : d;
        }
    }
}
}  // namespace

void signed_distance(its_ctx ctx, const double* d_V, int64_t nV, const int32_t* d_F, int64_t nF,
                     const double* d_pts, int64_t N, double* d_out, int32_t* d_tri) {
    if (N <= 0) return;
    const hipStream_t st = ctx->stream;
    TriTree tr;
    tree_build(tr, st, d_V, nV, d_F, nF);
    // the boundary, read while the distance kernels run
    ITS_HIP(hipMemcpyAsync(ctx->pinned, tr.counts.p, 2 * sizeof(int), hipMemcpyDeviceToHost, st));
    ITS_HIP(hipEventRecord(ctx->pinned_ev, st));
    // grid-strided launches: as many blocks as the CUs hold at once
    int dev = 0, cus = 256;
    ITS_HIP(hipGetDevice(&dev));
    ITS_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    auto grid_of = [&](const void* kernel, int threads, int64_t most) {
        int per_cu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0) != hipSuccess || per_cu < 1) {
            (void)hipGetLastError();
            per_cu = 1;
        }
        return (unsigned)std::min<int64_t>(most, (int64_t)per_cu * cus);
    };
    // every point's seed; with packets, also their order
    const bool packets = N >= kPacketPoints && N < (int64_t(1) << 32);
    DBuf<uint32_t> key(N), order(N), rest;
    DBuf<int32_t> seed_at(N);
    hipLaunchKernelGGL(k_pt_seed, dim3(strided_blocks(N, kT, kT)), dim3(kT), 0, st, tr.view(), d_pts, N, key.p, order.p, d_out,
                       seed_at.p);
    ITS_LAUNCH_CHECK();
    unsigned* counts = (unsigned*)tr.counts.p + 2;   // passed on, twice, and undecided
    const unsigned pgrid = strided_blocks(N, kPk, 64);   // a packet a block
    Work all{N, nullptr, nullptr}, left = all;
    if (packets) {
        radix_sort(key, &order, N, kSeedKeyBits, st);
        rest.alloc(N);
        all.list = order.p;
        left = Work{N, rest.p, counts};
        hipLaunchKernelGGL(k_dist_packet, dim3(pgrid), dim3(64), 0, st, tr.view(), d_pts, all, (const int32_t*)seed_at.p, d_out,
                           d_tri, rest.p, counts);
        ITS_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_dist_point, dim3(grid_of((const void*)k_dist_point, 64, N)), dim3(64), 0, st, tr.view(), d_pts, left,
                       (const int32_t*)seed_at.p, d_out, d_tri);
    ITS_LAUNCH_CHECK();
    // Signs by the ray, and the rim where there is a boundary, for the points
    // that they decide; the fans are built and walked only for the others.
    // The rim's time grows with the boundary, the fan walk's hardly, so long
    // boundaries stay with the fans: more than one half edge per two triangles
    // (1,300 separate triangles, 60,000 points: 1.25 ms with the rim, 0.94
    // without; sphere of 879 triangles with 835: 0.76 and 0.74; of 1,150 with
    // 344: 0.50 and 0.76) or more than kRimMost (knot tube of 38,798 with 3,516,
    // 60,000 points: 1.23 and 1.97; torus of 8,638 with 3,566: about equal).
    DBuf<uint8_t> decided;
    DBuf<int> cross;
    const int most = (int)std::min<int64_t>(kRimMost, nF / 2);
    ITS_HIP(hipEventSynchronize(ctx->pinned_ev));
    const bool open = ctx->pinned[0] != 0;
    const int rim = ctx->pinned[1];
    const bool by_ray = rim <= most && tune_get(ITS_TUNE_SDF_RAY);
    bool fans = true;
    if (by_ray) {
        decided.alloc(N);
        if (open) cross.alloc(N);
        if (packets) {
            left.list_n = counts + 1;
            hipLaunchKernelGGL(k_ray_packet, dim3(pgrid), dim3(64), 0, st, tr.view(), d_pts, all, d_out, decided.p,
                               cross.p, counts + 2, rest.p, counts + 1);
            ITS_LAUNCH_CHECK();
        }
        hipLaunchKernelGGL(k_ray_point, dim3(grid_of((const void*)k_ray_point, 64, N)), dim3(64), 0, st, tr.view(), d_pts, left,
                           d_out, decided.p, cross.p, counts + 2);
        ITS_LAUNCH_CHECK();
        if (open) {
            hipLaunchKernelGGL(k_rim, dim3(strided_blocks(N, 64, 64 * kRimWaves)), dim3(64 * kRimWaves), 0, st,
                               (const RimEdge*)tr.rim.p,
                               rim, d_pts, N, d_out, decided.p, (const int*)cross.p, counts + 2);
            ITS_LAUNCH_CHECK();
        }
        fans = read1(counts + 2, st) != 0;
    }
    if (fans) {
        fans_build(tr, st, d_V, d_F);
        hipLaunchKernelGGL(k_sdf_wind, dim3(grid_of((const void*)k_sdf_wind, kT, (N + kWavesPerBlock - 1) / kWavesPerBlock)), dim3(kT), 0, st, tr.view(), d_pts, N, d_out,
                           by_ray ? (const uint8_t*)decided.p : (const uint8_t*)nullptr);
        ITS_LAUNCH_CHECK();
    }
    ITS_HIP(hipStreamSynchronize(st));
}

namespace {
// unit normal of each point's nearest triangle (zero for a degenerate one, and
// for a point to which no triangle has a distance)
__global__ void k_tri_normal(int64_t N, const double* V, const int32_t* F, int64_t nF, const int32_t* tri,
                             float4* nrm) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int32_t t = tri[i];
    if (t < 0 || t >= nF) {
        nrm[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        return;
    }
    const double* a = V + 3 * (int64_t)F[3 * (int64_t)t];
    const double* b = V + 3 * (int64_t)F[3 * (int64_t)t + 1];
    const double* c = V + 3 * (int64_t)F[3 * (int64_t)t + 2];
    const double u[3] = {b[0] - a[0], b[1] - a[1], b[2] - a[2]}, v[3] = {c[0] - a[0], c[1] - a[1], c[2] - a[2]};
    const double x = u[1] * v[2] - u[2] * v[1], y = u[2] * v[0] - u[0] * v[2], z = u[0] * v[1] - u[1] * v[0];
    const double l = sqrt(x * x + y * y + z * z);
    nrm[i] = l > 0 ? make_float4((float)(x / l), (float)(y / l), (float)(z / l), 0.f) : make_float4(0.f, 0.f, 0.f, 0.f);
}
}  // namespace

void nearest_normals(hipStream_t st, const double* d_V, const int32_t* d_F, int64_t nF, const int32_t* d_tri,
                     int64_t N, float4* d_nrm) {
    if (N <= 0) return;
    hipLaunchKernelGGL(k_tri_normal, dim3(blocks_for(N, kT)), dim3(kT), 0, st, N, d_V, d_F, nF, d_tri, d_nrm);
    ITS_LAUNCH_CHECK();
}

void sort_u64(DBuf<uint64_t>& keys, int64_t n, int bits, hipStream_t st) {
    radix_sort(keys, (DBuf<uint32_t>*)nullptr, n, bits, st);
}

}  // namespace its
