// Sparse voxel octree construction for gfx950.
//
// Replaces SparseVoxelOctree::createOctree (reference src/cuAcc/SVO.cu:674-856),
// constructNodeNeighbors (858-911) and the per-level vertex dedup
// (913-963, 1010-1096).  The reference keeps a dense Morton-indexed uint32
// occupancy array and runs thrust scans/sorts over it level by level.  Here
// every set of cells or lattice points is a bitset with a rank directory
// (RankWord), so compaction is a popcount scan, membership and rank are one
// word read, and nothing is sorted: Morton order of the bitset is the order
// of the reference's compacted arrays, and the x-major lattice bitset order
// is the reference's lexicographic vertex order.
//
// Floating point: node origins and voxel tests are binary64 in exactly the
// operation order of the reference expressions, compiled without FMA
// contraction, so they agree bit for bit with the CPU restatement.
#include <algorithm>
#include <cmath>

#include "internal.hpp"

namespace its {
namespace {

constexpr int kT = 256;

// ------------------------------------------------------------ voxelizer ----
struct Grid {
    double go[3];
    double unit[3];
    int R;
};

__device__ inline double dmin(double a, double b) { return a < b ? a : b; }
__device__ inline double dmax(double a, double b) { return a > b ? a : b; }
__device__ inline double dot3(const double a[3], const double b[3]) { return a[0] * b[0] + (a[1] * b[1] + a[2] * b[2]); }
__device__ inline double dot2(double a0, double a1, double b0, double b1) { return a0 * b0 + a1 * b1; }

// triangle's clamped voxel box (surfaceVoxelize, SVO.cu:394-404)
__device__ inline void tri_box(const double* t, const Grid& g, int bo[3], int be[3]) {
    for (int a = 0; a < 3; ++a) {
        double v0 = t[a] - g.go[a], v1 = t[3 + a] - g.go[a], v2 = t[6 + a] - g.go[a];
        double lo = dmin(v0, dmin(v1, v2)), hi = dmax(v0, dmax(v1, v2));
        int l = (int)(lo / g.unit[a]), h = (int)(hi / g.unit[a]);
        bo[a] = max(0, min(l, g.R - 1));
        be[a] = max(bo[a], min(h, g.R - 1));   // never empty: a triangle has a candidate
    }
}

__global__ void k_tri_count(const double* tris, int64_t T, Grid g, uint64_t* cnt) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= T) return;
    int bo[3], be[3];
    tri_box(tris + 9 * t, g, bo, be);
    cnt[t] = (uint64_t)(be[0] - bo[0] + 1) * (uint64_t)(be[1] - bo[1] + 1) * (uint64_t)(be[2] - bo[2] + 1);
}

// First triangle of every 256 candidates: the last whose offset is not beyond
// theirs.  One thread per entry, so that a triangle with many candidates takes no
// longer than the others.  One thread per triangle, writing its run of entries,
// took 2.5 us where this takes 7.3 (200,000 small triangles at 256^3), but 1.4 ms
// for 3 on a slanted tetrahedron at 256^3 and 79 ms for 0.02 at 1024^3.
__global__ void k_cand_starts(const uint64_t* off, int64_t T, uint64_t entries, uint32_t* start) {
    const uint64_t step = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; b < entries; b += step) {
        const uint64_t c = b * kT;
        int64_t lo = 0, hi = T - 1;
        while (lo < hi) {
            const int64_t mid = (lo + hi + 1) >> 1;
            if (off[mid] <= c) lo = mid;
            else hi = mid - 1;
        }
        start[b] = (uint32_t)lo;
    }
}

// One thread per (triangle, candidate voxel); the triangle set-up is
// recomputed per candidate, in the reference's expression order.  A block's
// 256 candidates belong to at most 256 consecutive triangles, since every
// triangle has one: they start at the block's entry of start (k_cand_starts),
// and each thread searches their offsets in LDS.
__global__ __launch_bounds__(kT) void k_voxelize(const double* tris, int64_t T, const uint64_t* off, uint64_t total,
                                                 const uint32_t* start, Grid g, RankWord* occ) {
    __shared__ uint64_t s_off[kT + 1];
    for (uint64_t b = blockIdx.x; b * kT < total; b += gridDim.x) {
        const uint64_t c0 = b * kT;
        const int64_t t0 = start[b], t1 = c0 + kT < total ? (int64_t)start[b + 1] : T - 1;
        const int nt = (int)min(t1 - t0 + 1, (int64_t)kT);
        __syncthreads();
        if ((int)threadIdx.x < nt) s_off[threadIdx.x] = off[t0 + threadIdx.x];
        __syncthreads();
        const uint64_t c = c0 + threadIdx.x;
        if (c >= total) continue;
        int lq = 0, hq = nt - 1;
        while (lq < hq) {
            const int mid = (lq + hq + 1) >> 1;
            if (s_off[mid] <= c) lq = mid;
            else hq = mid - 1;
        }
        const int64_t lo = t0 + lq;
        const double* tri = tris + 9 * lo;
        int bo[3], be[3];
        tri_box(tri, g, bo, be);
        uint64_t local = c - s_off[lq];
        uint64_t nx = be[0] - bo[0] + 1, ny = be[1] - bo[1] + 1;
        int x = bo[0] + (int)(local % nx);
        int y = bo[1] + (int)((local / nx) % ny);
        int z = bo[2] + (int)(local / (nx * ny));

        double v0[3], v1[3], v2[3], e0[3], e1[3], e2[3], n[3];
        for (int a = 0; a < 3; ++a) {
            v0[a] = tri[a] - g.go[a];
            v1[a] = tri[3 + a] - g.go[a];
            v2[a] = tri[6 + a] - g.go[a];
        }
        for (int a = 0; a < 3; ++a) {
            e0[a] = v1[a] - v0[a];
            e1[a] = v2[a] - v1[a];
            e2[a] = v0[a] - v2[a];
        }
        n[0] = e0[1] * e1[2] - e0[2] * e1[1];
        n[1] = e0[2] * e1[0] - e0[0] * e1[2];
        n[2] = e0[0] * e1[1] - e0[1] * e1[0];
        double z2 = dot3(n, n);
        if (z2 > 0.0) {
            double s = sqrt(z2);
            n[0] = n[0] / s;
            n[1] = n[1] / s;
            n[2] = n[2] / s;
        }
        const double* u = g.unit;
        double cc[3] = {n[0] > 0.0 ? u[0] : 0.0, n[1] > 0.0 ? u[1] : 0.0, n[2] > 0.0 ? u[2] : 0.0};
        double cv[3], dv[3];
        for (int a = 0; a < 3; ++a) {
            cv[a] = cc[a] - v0[a];
            dv[a] = (u[a] - cc[a]) - v0[a];
        }
        double d1 = dot3(n, cv), d2 = dot3(n, dv);
        double p[3] = {(double)x * u[0], (double)y * u[1], (double)z * u[2]};
        double nDOTp = dot3(n, p);
        if ((nDOTp + d1) * (nDOTp + d2) > 0.0) continue;

        const double* vs[3] = {v0, v1, v2};
        const double* es[3] = {e0, e1, e2};
        bool ok = true;
        // XY
        for (int i = 0; i < 3 && ok; ++i) {
            double a0 = -1.0 * es[i][1], a1 = es[i][0];
            if (n[2] < 0.0) { a0 = -a0; a1 = -a1; }
            double d = (-1.0 * dot2(a0, a1, vs[i][0], vs[i][1])) + dmax(0.0, u[0] * a0) + dmax(0.0, u[1] * a1);
            if ((dot2(a0, a1, p[0], p[1]) + d) < 0.0) ok = false;
        }
        // YZ
        for (int i = 0; i < 3 && ok; ++i) {
            double a0 = -1.0 * es[i][2], a1 = es[i][1];
            if (n[0] < 0.0) { a0 = -a0; a1 = -a1; }
            double d = (-1.0 * dot2(a0, a1, vs[i][1], vs[i][2])) + dmax(0.0, u[1] * a0) + dmax(0.0, u[2] * a1);
            if ((dot2(a0, a1, p[1], p[2]) + d) < 0.0) ok = false;
        }
        // ZX
        for (int i = 0; i < 3 && ok; ++i) {
            double a0 = -1.0 * es[i][0], a1 = es[i][2];
            if (n[1] < 0.0) { a0 = -a0; a1 = -a1; }
            double d = (-1.0 * dot2(a0, a1, vs[i][2], vs[i][0])) + dmax(0.0, u[2] * a0) + dmax(0.0, u[0] * a1);
            if ((dot2(a0, a1, p[2], p[0]) + d) < 0.0) ok = false;
        }
        if (!ok) continue;
        uint32_t m = morton3((uint32_t)x, (uint32_t)y, (uint32_t)z);
        const uint32_t bit = 1u << (m & 31);
        if (!(__hip_atomic_load(&occ[m >> 5].bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit))
            atomicOr(&occ[m >> 5].bits, bit);
    }
}

// --------------------------------------------------------------- levels ----
// All levels side by side, finest first: every kernel below takes the nodes,
// cells or vertices of all levels in one launch, since most levels are far
// too small to fill the chip or even a launch.
//
// The occupied cells are a pyramid of Morton bitsets.  A node is a child of
// an occupied cell, and the children of the cell of rank r sit at 8r .. 8r+7
// of their level, so a node's index, its parent, its children and its 27
// neighbours are each one bit and rank of the level above or its own.
struct Tree {
    int top;                          // levels of the pyramid
    int depth;                        // levels up to the root
    int R0;
    double go[3];
    double width[kMaxLevels];
    int64_t word[kMaxLevels + 1];     // first word of each level's occupancy
    int64_t first[kMaxLevels + 1];    // first occupied cell of each level (ranks count over the levels)
    int64_t node[kMaxLevels + 1];     // first node of each level
    int64_t lat[kMaxLevels + 1];      // first word of each level's corner lattice
    int64_t vert[kMaxLevels + 1];     // first vertex of each level
};
__device__ inline int level_of(const int64_t* first, int n, int64_t i) {
    int d = 0;
    while (d + 1 < n && i >= first[d + 1]) ++d;
    return d;
}

// parents' bits from the children's: a parent is one byte of its level below
__device__ inline uint32_t parent_bits(const RankWord* child, int64_t nchild, int64_t w) {
    uint32_t bits = 0;
    for (int q = 0; q < 8; ++q) {
        const uint32_t b = 8 * w + q < nchild ? child[8 * w + q].bits : 0u;
        for (int y = 0; y < 4; ++y)
            if ((b >> (8 * y)) & 255u) bits |= 1u << (4 * q + y);
    }
    return bits;
}
__global__ void k_occ_up(const RankWord* child, int64_t nchild, RankWord* up, int64_t nup) {
    const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w < nup) up[w].bits = parent_bits(child, nchild, w);
}
// the upper levels in one workgroup
constexpr int kOccTopThreads = 1024;
__global__ __launch_bounds__(kOccTopThreads) void k_occ_top(Tree T, int from, RankWord* occ) {
    for (int d = from; d + 1 < T.top; ++d) {
        const int64_t nup = T.word[d + 2] - T.word[d + 1];
        for (int64_t w = threadIdx.x; w < nup; w += kOccTopThreads)
            occ[T.word[d + 1] + w].bits = parent_bits(occ + T.word[d], T.word[d + 1] - T.word[d], w);
        __threadfence_block();
        __syncthreads();
    }
}

// ranks at the starts of n consecutive bitsets, and the total
struct Starts {
    int n;
    int64_t word[kMaxLevels + 1];
};
__global__ void k_level_first(const RankWord* g, Starts S, const uint32_t* total, uint32_t* first) {
    const int d = threadIdx.x;
    if (d < S.n) first[d] = g[S.word[d]].rank;
    if (d == S.n) first[d] = *total;
}

// codes of the occupied cells, by rank
__global__ void k_occ_codes(const RankWord* occ, Tree T, uint32_t* codes) {
    const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= T.word[T.top]) return;
    const RankWord rw = occ[w];
    if (rw.bits == 0) return;
    const uint32_t base = (uint32_t)(w - T.word[level_of(T.word, T.top, w)]) * 32u;
    uint32_t b = rw.bits, r = rw.rank;
    while (b) {
        codes[r++] = base + (uint32_t)(__ffs(b) - 1);
        b &= b - 1;
    }
}

// rank of the occupied cell m of level d within its level, or ITS_NONE
__device__ inline uint32_t occ_rank(const Tree& T, const RankWord* occ, int d, uint32_t m) {
    const uint32_t r = bit_find(occ + T.word[d], m);
    return r == ITS_NONE ? ITS_NONE : r - (uint32_t)T.first[d];
}
// global index of the node m of level d, or ITS_NONE
__device__ inline uint32_t node_of(const Tree& T, const RankWord* occ, const uint32_t* codes, int d, uint32_t m) {
    if (d + 1 == T.depth) return m == codes[T.first[d]] ? (uint32_t)T.node[d] : ITS_NONE;
    const uint32_t r = occ_rank(T, occ, d + 1, m >> 3);
    return r == ITS_NONE ? ITS_NONE : (uint32_t)T.node[d] + 8u * r + (m & 7u);
}

struct NodeOut {
    uint32_t* morton;
    uint8_t* is_leaf;
    double* origin;
    double* width;
    uint32_t* parent;
    uint32_t* childbase;
};
// nodes of all levels: octets of the children of each occupied parent, and
// the root (createNode_1/2 + createRemainNode, SVO.cu:560-672)
__global__ void k_nodes(Tree T, const RankWord* occ, const uint32_t* codes, NodeOut o) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= T.node[T.depth]) return;
    const int d = level_of(T.node, T.depth, g);
    const int64_t j = g - T.node[d];
    const bool root = d + 1 == T.depth;
    const uint32_t m = root ? codes[T.first[d]] : ((codes[T.first[d + 1] + (j >> 3)] << 3) | (uint32_t)(j & 7));
    const double w = T.width[d];
    uint32_t x, y, z;
    demorton3(m, x, y, z);
    o.morton[g] = m;
    o.origin[3 * g + 0] = T.go[0] + w * (double)x;
    o.origin[3 * g + 1] = T.go[1] + w * (double)y;
    o.origin[3 * g + 2] = T.go[2] + w * (double)z;
    o.width[g] = w;
    o.parent[g] = root ? ITS_NONE : node_of(T, occ, codes, d + 1, m >> 3);
    const uint32_t r = d > 0 ? occ_rank(T, occ, d, m) : ITS_NONE;
    o.is_leaf[g] = r == ITS_NONE ? 1 : 0;
    o.childbase[g] = r == ITS_NONE ? ITS_NONE : (uint32_t)T.node[d - 1] + 8u * r;
}

// Neighbour index k = (dx+1) + 3(dy+1) + 9(dz+1), as findNeighbors
// (SVO.cu:858-890): the node at the neighbouring cell of the same level.  One
// thread per (node, neighbour slot), so a wavefront stores 64 consecutive
// entries of the 27-per-node table.
__global__ void k_neighbors(Tree T, const RankWord* occ, const uint32_t* codes, const uint32_t* morton, uint32_t* nb) {
    const int64_t n = 27 * T.node[T.depth], step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += step) {
        const int64_t g = t / 27;
        const int k = (int)(t - 27 * g);
        uint32_t v = ITS_NONE;
        if (k == 13) {
            v = (uint32_t)g;
        } else {
            const int d = level_of(T.node, T.depth, g);
            if (d + 1 < T.depth) {
                uint32_t x, y, z;
                demorton3(morton[g], x, y, z);
                const uint32_t R = (uint32_t)(T.R0 >> d);
                x += (uint32_t)(k % 3 - 1);
                y += (uint32_t)((k / 3) % 3 - 1);
                z += (uint32_t)(k / 9 - 1);
                if (x < R && y < R && z < R) v = node_of(T, occ, codes, d, morton3(x, y, z));
            }
        }
        nb[t] = v;
    }
}

// -------------------------------------------------------------- vertices ----
__device__ inline uint32_t lat_index(uint32_t X, uint32_t Y, uint32_t Z, uint32_t D) { return (X * D + Y) * D + Z; }

// Corners of all nodes.  The eight nodes of an octet share a block of 3 x 3 x 3
// lattice points: one thread per octet and (x, y), which sets three
// consecutive bits of the lattice, instead of 64 atomics for the octet's
// nodes one by one.  The last item is the root, 2 x 2 x 2 points.
__global__ void k_mark_corners(Tree T, const uint32_t* codes, RankWord* lat) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    // octets of levels 0 .. depth - 2 are the occupied cells of levels 1 .. depth - 1
    const int64_t octets = T.first[T.depth] - T.first[1];
    const int64_t q = t / 9;
    const int c = (int)(t - 9 * q);
    if (q > octets) return;
    const bool root = q == octets;
    const int64_t i = root ? T.first[T.depth - 1] : T.first[1] + q;   // the cell whose corners these are
    const int up = level_of(T.first, T.depth, i), d = root ? up : up - 1;
    const uint32_t dx = (uint32_t)(c % 3), dy = (uint32_t)(c / 3);
    if (root && (dx == 2 || dy == 2)) return;
    uint32_t x, y, z;
    demorton3(codes[i], x, y, z);
    const uint32_t scale = root ? 1u : 2u, D = (uint32_t)(T.R0 >> d) + 1u;
    const uint32_t key = lat_index(scale * x + dx, scale * y + dy, scale * z, D);
    const uint64_t bits = (uint64_t)(root ? 3u : 7u) << (key & 31);
    RankWord* g = lat + T.lat[d] + (key >> 5);
    for (int h = 0; h < 2; ++h) {
        const uint32_t b = (uint32_t)(bits >> (32 * h));
        if (b && (__hip_atomic_load(&g[h].bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & b) != b)
            atomicOr(&g[h].bits, b);
    }
}

// lattice keys of the vertices, by rank; the ranks, counted over all levels so
// far, become ranks within the level
__global__ void k_vert_keys(Tree T, RankWord* lat, uint32_t* keys) {
    const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= T.lat[T.depth]) return;
    const RankWord rw = lat[w];
    const int d = level_of(T.lat, T.depth, w);
    lat[w].rank = rw.rank - (uint32_t)T.vert[d];
    uint32_t b = rw.bits, r = rw.rank;
    const uint32_t base = (uint32_t)(w - T.lat[d]) * 32u;
    while (b) {
        keys[r++] = base + (uint32_t)(__ffs(b) - 1);
        b &= b - 1;
    }
}

struct VertOut {
    uint16_t *x, *y, *z;
    uint8_t* level;
    uint32_t* owner;
    double* xyz;
};
// Vertices of all levels: lattice coordinates; the owner, the smallest index
// of the nodes sharing the corner (the min over d_vertSharedLUT neighbours in
// determineNodeVertex, SVO.cu:950-960), which within a level is the smallest
// code; and the position from it, origin + width * (offset), the copy the
// reference's stable sort + unique keeps (SVO.cu:1081-1082).
__global__ void k_vertices(Tree T, const RankWord* occ, const uint32_t* codes, const uint32_t* keys, VertOut o) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= T.vert[T.depth]) return;
    const int d = level_of(T.vert, T.depth, v);
    const uint32_t R = (uint32_t)(T.R0 >> d), D = R + 1u, key = keys[v];
    const uint32_t XY = key / D, Z = key - XY * D, X = XY / D, Y = XY - X * D;
    uint32_t own = ITS_NONE, ox = 0, oy = 0, oz = 0;
    for (int k = 0; k < 8; ++k) {
        const uint32_t x = X - (k & 1), y = Y - ((k >> 1) & 1), z = Z - ((k >> 2) & 1);
        if (x >= R || y >= R || z >= R) continue;
        const uint32_t g = node_of(T, occ, codes, d, morton3(x, y, z));
        if (g < own) {
            own = g;
            ox = x;
            oy = y;
            oz = z;
        }
    }
    const double w = T.width[d];
    o.x[v] = (uint16_t)X;
    o.y[v] = (uint16_t)Y;
    o.z[v] = (uint16_t)Z;
    o.level[v] = (uint8_t)d;
    o.owner[v] = own;
    o.xyz[3 * v + 0] = (T.go[0] + w * (double)ox) + w * (double)(X - ox);
    o.xyz[3 * v + 1] = (T.go[1] + w * (double)oy) + w * (double)(Y - oy);
    o.xyz[3 * v + 2] = (T.go[2] + w * (double)oz) + w * (double)(Z - oz);
}

// ranks of n bitsets in a row and the count before each of them and in all,
// in one read-back
std::vector<int64_t> rank_levels(RankWord* g, const Starts& S, int64_t words, hipStream_t st) {
    DBuf<uint32_t> first(S.n + 2);
    uint32_t* total = first.p + S.n + 1;
    rank_build_async(g, words, st, total);
    hipLaunchKernelGGL(k_level_first, dim3(1), dim3(64), 0, st, (const RankWord*)g, S, (const uint32_t*)total, first.p);
    ITS_LAUNCH_CHECK();
    std::vector<uint32_t> h;
    to_host(h, first.p, S.n + 1, st);
    return std::vector<int64_t>(h.begin(), h.end());
}

}  // namespace

void svo_build(its_svo s, const double* d_tris, int64_t n_tris) {
    hipStream_t st = s->ctx->stream;
    const int R = s->R;
    Grid g;
    for (int a = 0; a < 3; ++a) {
        g.go[a] = s->origin[a];
        g.unit[a] = s->width[a] / R;   // unitVoxelSize (SVO.cu:683-685)
    }
    g.R = R;
    s->voxel_width = g.unit[0];        // unitNodeWidth = unitVoxelSize.x()

    Tree T{};
    T.R0 = R;
    for (int a = 0; a < 3; ++a) T.go[a] = g.go[a];
    T.top = 1;
    while ((R >> (T.top - 1)) > 1) ++T.top;
    ITS_REQUIRE(T.top <= kMaxLevels, ITS_E_RANGE, "octree deeper than supported");
    Starts S{};
    S.n = T.top;
    for (int d = 0; d < T.top; ++d) {
        const int64_t side = R >> d;
        T.word[d + 1] = T.word[d] + std::max<int64_t>(1, (side * side * side + 31) / 32);
        S.word[d] = T.word[d];
    }
    const int64_t words = T.word[T.top];

    // ---- occupancy: voxels, then the pyramid above them
    DBuf<RankWord> occ(words);
    ITS_HIP(hipMemsetAsync(occ.p, 0, occ.bytes(), st));
    if (n_tris > 0) {
        DBuf<uint64_t> cnt(n_tris);
        hipLaunchKernelGGL(k_tri_count, dim3(blocks_for(n_tris, kT)), dim3(kT), 0, st, d_tris, n_tris, g, cnt.p);
        ITS_LAUNCH_CHECK();
        const uint64_t total = scan_exclusive_u64(cnt.p, cnt.p, n_tris, st);
        if (total) {
            unsigned nb = (unsigned)std::min<uint64_t>((total + kT - 1) / kT, 1u << 20);
            const int64_t entries = (int64_t)((total + kT - 1) / kT);
            DBuf<uint32_t> start(entries);
            hipLaunchKernelGGL(k_cand_starts, dim3(strided_blocks(entries, kT, kT)), dim3(kT), 0, st,
                               (const uint64_t*)cnt.p, n_tris, (uint64_t)entries, start.p);
            ITS_LAUNCH_CHECK();
            hipLaunchKernelGGL(k_voxelize, dim3(nb), dim3(kT), 0, st, d_tris, n_tris, (const uint64_t*)cnt.p, total,
                               (const uint32_t*)start.p, g, occ.p);
            ITS_LAUNCH_CHECK();
        }
    }
    int d0 = 0;
    for (; d0 + 1 < T.top && T.word[d0 + 2] - T.word[d0 + 1] > kOccTopThreads; ++d0) {
        const int64_t nup = T.word[d0 + 2] - T.word[d0 + 1];
        hipLaunchKernelGGL(k_occ_up, dim3(blocks_for(nup, kT)), dim3(kT), 0, st, (const RankWord*)occ.p + T.word[d0],
                           T.word[d0 + 1] - T.word[d0], occ.p + T.word[d0 + 1], nup);
        ITS_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_occ_top, dim3(1), dim3(kOccTopThreads), 0, st, T, d0, occ.p);
    ITS_LAUNCH_CHECK();

    // ---- levels (SVO.cu:717-815): the first with a single occupied cell is
    // the root; the levels above it are dropped
    const std::vector<int64_t> first = rank_levels(occ.p, S, words, st);
    for (int d = 0; d <= T.top; ++d) T.first[d] = first[d];
    s->num_voxels = first[1];
    s->occ_codes.alloc(std::max<int64_t>(first[T.top], 1));
    s->depth = 0;
    s->num_nodes = 0;
    if (s->num_voxels == 0) return;
    hipLaunchKernelGGL(k_occ_codes, dim3(blocks_for(words, kT)), dim3(kT), 0, st, (const RankWord*)occ.p, T,
                       s->occ_codes.p);
    ITS_LAUNCH_CHECK();
    double w = g.unit[0];
    for (int d = 0; d < T.top && s->depth == 0; ++d, w *= 2.0) {
        Level& L = s->lv[d];
        L.R = R >> d;
        L.width = w;
        T.width[d] = w;
        L.n_occ = first[d + 1] - first[d];
        if (L.n_occ == 1) s->depth = d + 1;
        L.n_nodes = L.n_occ == 1 ? 1 : 8 * (first[d + 2] - first[d + 1]);
        T.node[d + 1] = T.node[d] + L.n_nodes;
    }
    ITS_REQUIRE(s->depth > 0, ITS_E_STATE, "octree level loop did not reach a single cell");
    const int depth = T.depth = s->depth;
    for (int d = 0; d <= depth; ++d) s->esum_nodes[d] = T.node[d];
    const int64_t total = s->num_nodes = T.node[depth];

    // ---- node arrays
    s->morton.alloc(total);
    s->is_leaf.alloc(total);
    s->node_origin.alloc(3 * total);
    s->node_width.alloc(total);
    s->parent.alloc(total);
    s->childbase.alloc(total);
    s->neighbors.alloc(27 * total);
    const NodeOut o{s->morton.p, s->is_leaf.p, s->node_origin.p, s->node_width.p, s->parent.p, s->childbase.p};
    const RankWord* d_occ = occ.p;
    const uint32_t* codes = s->occ_codes.p;
    hipLaunchKernelGGL(k_nodes, dim3(blocks_for(total, kT)), dim3(kT), 0, st, T, d_occ, codes, o);
    ITS_LAUNCH_CHECK();

    // ---- corner lattices
    S.n = depth;
    for (int d = 0; d < depth; ++d) {
        const int64_t D = s->lv[d].R + 1;
        T.lat[d + 1] = T.lat[d] + (D * D * D + 31) / 32;
        S.word[d] = T.lat[d];
    }
    const int64_t lat_words = T.lat[depth];
    s->lattice.alloc(lat_words);
    ITS_HIP(hipMemsetAsync(s->lattice.p, 0, s->lattice.bytes(), st));
    for (int d = 0; d < depth; ++d) s->lv[d].lattice.p = s->lattice.p + T.lat[d];
    const int64_t items = 9 * (T.first[depth] - T.first[1] + 1);
    hipLaunchKernelGGL(k_mark_corners, dim3(blocks_for(items, kT)), dim3(kT), 0, st, T, codes, s->lattice.p);
    ITS_LAUNCH_CHECK();
    // queued behind the marks, in front of the read-back
    hipLaunchKernelGGL(k_neighbors, dim3(strided_blocks(27 * total, kT, kT)), dim3(kT), 0, st, T, d_occ, codes,
                       (const uint32_t*)s->morton.p, s->neighbors.p);
    ITS_LAUNCH_CHECK();
    const std::vector<int64_t> vert = rank_levels(s->lattice.p, S, lat_words, st);
    for (int d = 0; d <= depth; ++d) s->esum_verts[d] = T.vert[d] = vert[d];
    for (int d = 0; d < depth; ++d) s->lv[d].n_verts = vert[d + 1] - vert[d];
    const int64_t nv = s->num_verts = vert[depth];

    // ---- vertices
    s->vx.alloc(nv);
    s->vy.alloc(nv);
    s->vz.alloc(nv);
    s->vlevel.alloc(nv);
    s->vowner.alloc(nv);
    s->vxyz.alloc(3 * nv);
    DBuf<uint32_t> keys(nv);
    hipLaunchKernelGGL(k_vert_keys, dim3(blocks_for(lat_words, kT)), dim3(kT), 0, st, T, s->lattice.p, keys.p);
    ITS_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_vertices, dim3(blocks_for(nv, kT)), dim3(kT), 0, st, T, d_occ, codes, (const uint32_t*)keys.p,
                       VertOut{s->vx.p, s->vy.p, s->vz.p, s->vlevel.p, s->vowner.p, s->vxyz.p});
    ITS_LAUNCH_CHECK();
    ITS_HIP(hipStreamSynchronize(st));
}

// An octree object that holds only a vertex set, its levels and lattices:
// the inputs of MC::marching_cubes (MarchingCubes.h:136-139), nodeVertexArray
// (corner position and owner node per vertex) and nodeWidthArray (per node).
// A vertex's level follows from its owner's width, w_d = w_0 * 2^d with w_0
// the smallest width; the grid origin is the smallest coordinate of every
// axis (the root's first corner); a vertex's lattice key is its position in
// units of w_d from there.  The evaluation field and marching cubes then work
// as on a built octree: f(x) = sum_i lambda_i B_i(x) with B_i the hat of
// width w_level(i) centred on vertex i (CUDACompute.cu:468).
void svo_from_vertices(its_svo s, const double* xyz, const uint32_t* owner, int64_t n, const double* node_width,
                       int64_t n_nodes) {
    ITS_REQUIRE(n > 0, ITS_E_INVALID, "no vertices");
    ITS_REQUIRE(n < (int64_t)UINT32_MAX, ITS_E_RANGE, "too many vertices");
    double w0 = 0;
    for (int64_t i = 0; i < n; ++i) {
        ITS_REQUIRE(owner[i] < (uint64_t)n_nodes, ITS_E_INVALID, "vertex owner outside the node array");
        const double w = node_width[3 * (int64_t)owner[i]];
        ITS_REQUIRE(std::isfinite(w) && w > 0, ITS_E_INVALID, "node widths must be positive");
        if (i == 0 || w < w0) w0 = w;
    }
    double origin[3] = {xyz[0], xyz[1], xyz[2]};
    for (int64_t i = 0; i < n; ++i)
        for (int a = 0; a < 3; ++a) {
            ITS_REQUIRE(std::isfinite(xyz[3 * i + a]), ITS_E_INVALID, "vertex coordinates must be finite");
            origin[a] = std::min(origin[a], xyz[3 * i + a]);
        }
    std::vector<uint8_t> level(n);
    int depth = 0;
    for (int64_t i = 0; i < n; ++i) {
        const double w = node_width[3 * (int64_t)owner[i]];
        int d = 0;
        while (d < kMaxLevels && std::ldexp(w0, d) < w) ++d;
        ITS_REQUIRE(d < kMaxLevels && std::ldexp(w0, d) == w, ITS_E_INVALID,
                    "node widths must be the smallest width times a power of two");
        level[i] = (uint8_t)d;
        depth = std::max(depth, d + 1);
    }
    const int R = 1 << (depth - 1);
    ITS_REQUIRE(R <= 1024, ITS_E_RANGE, "more than 1024 cells per axis");
    std::vector<uint64_t> key(n);   // level in the high byte, lattice key below
    std::vector<uint16_t> kx(n), ky(n), kz(n);
    for (int64_t i = 0; i < n; ++i) {
        const int d = level[i];
        const double w = std::ldexp(w0, d);
        const int Rd = R >> d;
        int64_t k[3];
        for (int a = 0; a < 3; ++a) {
            const double u = (xyz[3 * i + a] - origin[a]) / w;
            k[a] = std::llround(u);
            ITS_REQUIRE(k[a] >= 0 && k[a] <= Rd && std::fabs(u - (double)k[a]) <= 1e-6, ITS_E_INVALID,
                        "a vertex is not a corner of its level's lattice");
        }
        kx[i] = (uint16_t)k[0];
        ky[i] = (uint16_t)k[1];
        kz[i] = (uint16_t)k[2];
        key[i] = ((uint64_t)d << 56) | (uint64_t)((k[0] * (Rd + 1) + k[1]) * (Rd + 1) + k[2]);
    }
    std::vector<int64_t> ord(n);
    for (int64_t i = 0; i < n; ++i) ord[i] = i;
    bool sorted = true;
    for (int64_t i = 1; i < n && sorted; ++i) sorted = key[i - 1] < key[i];
    if (!sorted) std::stable_sort(ord.begin(), ord.end(), [&](int64_t a, int64_t b) { return key[a] < key[b]; });
    for (int64_t i = 1; i < n; ++i)
        ITS_REQUIRE(key[ord[i - 1]] != key[ord[i]], ITS_E_INVALID, "two vertices share a level and a lattice point");
    if (!sorted) {
        s->vperm.assign(n, 0);
        for (int64_t j = 0; j < n; ++j) s->vperm[ord[j]] = j;
    }
    s->vertices_only = true;
    s->depth = depth;
    s->R = R;
    s->voxel_width = w0;
    for (int a = 0; a < 3; ++a) {
        s->origin[a] = origin[a];
        s->width[a] = (double)R * w0;
    }
    s->num_voxels = 0;
    s->num_nodes = 0;
    s->num_verts = n;
    hipStream_t st = s->ctx->stream;
    std::vector<uint16_t> hx(n), hy(n), hz(n);
    std::vector<uint8_t> hl(n);
    std::vector<uint32_t> ho(n);
    std::vector<double> hxyz(3 * n);
    for (int64_t j = 0; j < n; ++j) {
        const int64_t i = ord[j];
        hx[j] = kx[i];
        hy[j] = ky[i];
        hz[j] = kz[i];
        hl[j] = level[i];
        ho[j] = owner[i];
        for (int a = 0; a < 3; ++a) hxyz[3 * j + a] = xyz[3 * i + a];
    }
    int64_t at = 0, words = 0;
    std::vector<int64_t> lat_off(depth);
    for (int d = 0; d < depth; ++d) {
        const int64_t D = (int64_t)(R >> d) + 1;
        lat_off[d] = words;
        words += (D * D * D + 31) / 32;
    }
    std::vector<RankWord> lat(words, RankWord{0, 0});
    s->lattice.alloc(words);
    for (int d = 0; d < depth; ++d) {
        Level& L = s->lv[d];
        L.R = R >> d;
        L.width = std::ldexp(w0, d);
        L.lattice.p = s->lattice.p + lat_off[d];
        const int64_t D = (int64_t)L.R + 1;
        RankWord* g = lat.data() + lat_off[d];
        s->esum_verts[d] = at;
        int64_t cnt = 0;
        while (at < n && hl[at] == d) {
            const uint64_t b = (uint64_t)((hx[at] * D + hy[at]) * D + hz[at]);
            g[b >> 5].bits |= 1u << (b & 31);
            ++at;
            ++cnt;
        }
        L.n_verts = cnt;
        uint32_t run = 0;
        for (int64_t w = 0; w < (D * D * D + 31) / 32; ++w) {
            g[w].rank = run;
            run += (uint32_t)__builtin_popcount(g[w].bits);
        }
    }
    ITS_HIP(hipMemcpyAsync(s->lattice.p, lat.data(), words * sizeof(RankWord), hipMemcpyHostToDevice, st));
    s->esum_verts[depth] = n;
    s->vx.alloc(n);
    s->vy.alloc(n);
    s->vz.alloc(n);
    s->vlevel.alloc(n);
    s->vowner.alloc(n);
    s->vxyz.alloc(3 * n);
    ITS_HIP(hipMemcpyAsync(s->vx.p, hx.data(), n * sizeof(uint16_t), hipMemcpyHostToDevice, st));
    ITS_HIP(hipMemcpyAsync(s->vy.p, hy.data(), n * sizeof(uint16_t), hipMemcpyHostToDevice, st));
    ITS_HIP(hipMemcpyAsync(s->vz.p, hz.data(), n * sizeof(uint16_t), hipMemcpyHostToDevice, st));
    ITS_HIP(hipMemcpyAsync(s->vlevel.p, hl.data(), n * sizeof(uint8_t), hipMemcpyHostToDevice, st));
    ITS_HIP(hipMemcpyAsync(s->vowner.p, ho.data(), n * sizeof(uint32_t), hipMemcpyHostToDevice, st));
    ITS_HIP(hipMemcpyAsync(s->vxyz.p, hxyz.data(), 3 * n * sizeof(double), hipMemcpyHostToDevice, st));
    ITS_HIP(hipStreamSynchronize(st));   // the host staging vectors go out of scope
}

}  // namespace its
