// Solver state of the matrix-free collocation operator (internal).
#pragma once
#include "internal.hpp"

namespace its {

struct Coarse {
    int L, lc;
    uint32_t off[kMaxLevels + 1];   // global vertex offsets
};

// Operator lists, shared by the single-mesh and the batched solver.
//
// The parents of a vertex and the children of a coarse vertex are runs of
// lattice points, and consecutive points along z that exist are consecutive
// vertices.  A list is therefore stored by its (x, y) columns:
//   - parents: up to 4 columns of 1 or 2 points (2 where the vertex's z is
//     odd, bit 28 of the first column), one 16-byte word per vertex;
//   - children, at 2 (X, Y, Z) + {-1, 0, 1}^3: 9 columns, each the first
//     child's index with a 3-bit mask of the points that exist in bits 28 to
//     30, in slices of 64 vertices, column by column, so that a wavefront
//     reads whole lines.  A child's weight, 2^-(its odd coordinates), follows
//     from its place.
// Lists by offset and length cost two dependent reads before the entries, and
// the entries of neighbouring vertices lay 27 apart.  256^3 knot, average of
// the levels' launches: restriction 5.3 -> 4.3 us (one-workgroup levels 11.4
// -> 7.1), prolongation 3.9 -> 3.5; with a branch around every read instead
// of a safe address it was 6.9 and 11.5.  Sums run over the parents z-major
// and over the children x-major, ascending.
struct Lists {
    const uint4* par;
    const uint32_t* kid;
    int64_t kid0;   // first vertex with children (of level 1)
};
constexpr uint32_t kListIdx = 0x0FFFFFFFu;
__host__ __device__ inline int64_t kid_slot(int64_t c, int q) { return ((c >> 6) * 9 + q) * 64 + (c & 63); }

// Points that do not exist are read from `safe` and not added: the loads are
// straight-line code, all in flight at once, with no branch around each.
// sum of g over the parents P; w = 1 / their count (0 without parents)
template <class T, class Read>
__device__ inline T gather_parents(uint4 P, T& w, uint32_t safe, Read&& g) {
    const bool any = P.x != ITS_NONE, two = P.y != ITS_NONE, four = P.z != ITS_NONE, zz = any && ((P.x >> 28) & 1u);
    const uint32_t c[4] = {P.x & kListIdx, P.y, P.z, P.w};
    const bool has[4] = {any, two, four, four};
    T v[8];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        v[q] = g(has[q] ? c[q] : safe);
        v[4 + q] = g(has[q] && zz ? c[q] + 1u : safe);
    }
    T s = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) s = has[q & 3] && (q < 4 || zz) ? s + v[q] : s;
    w = any ? (four ? (T)0.25 : two ? (T)0.5 : (T)1) * (zz ? (T)0.5 : (T)1) : (T)0;
    return s;
}
// sum of 2^-k h over the children in the columns e
template <class T, class Read>
__device__ inline T sum_children(const uint32_t e[9], uint32_t safe, Read&& h) {
    T v[27];
#pragma unroll
    for (int q = 0; q < 9; ++q) {
        const uint32_t b = e[q] & kListIdx, m = e[q] >> 28;
        const uint32_t b1 = b + (m & 1u), b2 = b1 + ((m >> 1) & 1u);
        v[3 * q] = h((m & 1u) ? b : safe);
        v[3 * q + 1] = h((m & 2u) ? b1 : safe);
        v[3 * q + 2] = h((m & 4u) ? b2 : safe);
    }
    T s = 0;
#pragma unroll
    for (int q = 0; q < 9; ++q)
#pragma unroll
        for (int z = 0; z < 3; ++z) {
            const int k = (q / 3 != 1) + (q % 3 != 1) + (z != 1);   // odd coordinates of the child
            const T weight = k == 0 ? (T)1 : k == 1 ? (T)0.5 : k == 2 ? (T)0.25 : (T)0.125;
            s = ((e[q] >> (28 + z)) & 1u) ? s + v[3 * q + z] * weight : s;
        }
    return s;
}
__device__ inline void load_kids(const Lists& A, int64_t c, uint32_t e[9]) {
#pragma unroll
    for (int q = 0; q < 9; ++q) e[q] = A.kid[kid_slot(c - A.kid0, q)];
}
// over the children of vertex c (of level 1 or above)
template <class T>
__device__ inline T gather_children(const Lists& A, int64_t c, const T* h) {
    uint32_t e[9];
    load_kids(A, c, e);
    return sum_children<T>(e, 0u, [&](uint32_t y) { return h[y]; });
}

// ---------------------------------------------------------------- solver
// Per-vertex and per-block bodies of the CGLS passes, shared by the
// single-mesh solver (lscg.hip) and the many-mesh solver (lscg_batch.hip),
// so both compute every value with the same operations in the same order.
constexpr int kFitT = 256;     // threads per block of the passes
constexpr int kFitRed = 512;   // most partials of a reduction (fixed per mesh size)
__host__ __device__ inline unsigned fit_red_blocks(int64_t n) {
    const int64_t b = (n + kFitT - 1) / kFitT;
    return (unsigned)(b < 1 ? 1 : (b < kFitRed ? b : kFitRed));
}
// device scalar slots of a solve
enum FitScal { S_ABSNEW = 0, S_ALPHA, S_BETA, S_TT, S_RN2, S_THRESH, S_RN2_0, S_ZZ, S_ZZ2, S_COUNT };

// g_i = p_i + 2^-k sum_{c in pro(i)} g_c; with UPD the new search direction
// p_i = z_i + beta p_i first
template <class T, bool UPD>
__device__ inline void prolong_at(int64_t i, const Lists& A, T* p, const T* z, T* g, const double* scal) {
    T pi = p[i];
    if (UPD) {
        pi = z[i] + (T)scal[S_BETA] * pi;
        p[i] = pi;
    }
    T w;
    const T s = gather_parents<T>(A.par[i], w, 0u, [&](uint32_t j) { return g[j]; });
    g[i] = pi + w * s;
}
// h_c += sum_{y in res(c)} 2^-k(y) h_y
template <class T>
__device__ inline void restrict_at(int64_t c, const Lists& A, T* h) {
    h[c] += gather_children(A, c, (const T*)h);
}
// x += alpha p; r -= alpha t along the coincidence chain of i; h_i = (D^T r)_i
__device__ inline void update_dt_at(int64_t i, const uint8_t* finest, const uint32_t* up, float* x, const float* p,
                                    float* r, const float* t, float* h, const double* scal, int do_update) {
    float alpha = do_update ? (float)scal[S_ALPHA] : 0.f;
    if (do_update) x[i] = fmaf(alpha, p[i], x[i]);
    if (!finest[i]) {
        h[i] = 0.f;
        return;
    }
    float s = 0.f;
    for (uint32_t j = (uint32_t)i; j != ITS_NONE; j = up[j]) {
        float rj = r[j];
        if (do_update) {
            rj = fmaf(-alpha, t[j], rj);
            r[j] = rj;
        }
        s += rj;
    }
    h[i] = s;
}
// binary64 h_i = (D^T r)_i
__device__ inline void dt64_at(int64_t i, const uint8_t* finest, const uint32_t* up, const double* r, double* h) {
    if (!finest[i]) {
        h[i] = 0.0;
        return;
    }
    double s = 0.0;
    for (uint32_t j = (uint32_t)i; j != ITS_NONE; j = up[j]) s += r[j];
    h[i] = s;
}

// block sum of a blockDim.x-thread block; valid in thread 0
__device__ inline double block_sum(double v, double* sh) {
    v = wave_sum(v);
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) sh[wid] = v;
    __syncthreads();
    double s = 0;
    if (threadIdx.x == 0)
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += sh[w];
    __syncthreads();
    return s;
}
// Reductions write one partial per block; a one-workgroup kernel that
// follows sums them (kernel boundaries order the writes, so no fences or
// atomics are needed) in a fixed order: per-thread strided sums, then a
// fixed tree.  The total is valid in thread 0.
__device__ inline double sum_partials(const double* part, unsigned np, int stride, int o, double* sh) {
    double v = 0;
    for (unsigned b = threadIdx.x; b < np; b += blockDim.x) v += part[b * stride + o];
    return block_sum(v, sh);
}
// Block blk of nb: t = D g over its grid-stride share and the block's
// partial of ||t||^2 into part[blk]
__device__ inline void apply_down_block(int64_t n, unsigned blk, unsigned nb, const uint32_t* down, const float* g,
                                        float* t, double* part, double* sh) {
    double acc = 0;
    for (int64_t i = (int64_t)blk * blockDim.x + threadIdx.x; i < n; i += (int64_t)nb * blockDim.x) {
        float v = g[down[i]];
        t[i] = v;
        acc += (double)v * (double)v;
    }
    double s = block_sum(acc, sh);
    if (threadIdx.x == 0) part[blk] = s;
}
// z = M^-1 nr and the block's partials of nr.nr and nr.z
__device__ inline void precond_block(int64_t n, unsigned blk, unsigned nb, const float* nr, const float* invd, float* z,
                                     double* part, double* sh) {
    double a = 0, c = 0;
    for (int64_t i = (int64_t)blk * blockDim.x + threadIdx.x; i < n; i += (int64_t)nb * blockDim.x) {
        float v = nr[i];
        float zi = invd[i] * v;
        z[i] = zi;
        a += (double)v * (double)v;
        c += (double)v * (double)zi;
    }
    double sa = block_sum(a, sh);
    double sc = block_sum(c, sh);
    if (threadIdx.x == 0) {
        part[2 * blk] = sa;
        part[2 * blk + 1] = sc;
    }
}
__device__ inline void dot64_block(int64_t n, unsigned blk, unsigned nb, const double* a, const double* b,
                                   double* part, double* sh) {
    double acc = 0;
    for (int64_t i = (int64_t)blk * blockDim.x + threadIdx.x; i < n; i += (int64_t)nb * blockDim.x)
        acc += a[i] * b[i];
    double s = block_sum(acc, sh);
    if (threadIdx.x == 0) part[blk] = s;
}
// alpha = absNew / ||t||^2
__device__ inline void scalar_alpha_body(const double* part, unsigned np, double* scal, double* sh) {
    double tt = sum_partials(part, np, 1, 0, sh);
    if (threadIdx.x == 0) {
        scal[S_TT] = tt;
        scal[S_ALPHA] = tt > 0 ? scal[S_ABSNEW] / tt : 0.0;
    }
}
// rn2, absNew', the stopping test of Eigen's loop, beta.  ctl: [0] done,
// [1] iterations, [3] iteration limit
__device__ inline void scalar_beta_body(const double* part, unsigned np, double* scal, int* ctl, int init, double* sh) {
    double rn2 = sum_partials(part, np, 2, 0, sh);
    double zz = sum_partials(part, np, 2, 1, sh);
    if (threadIdx.x == 0) {
        scal[S_RN2] = rn2;
        if (init) {
            scal[S_RN2_0] = rn2;
            scal[S_ABSNEW] = zz;
            scal[S_BETA] = 0.0;
            if (rn2 < scal[S_THRESH] || zz == 0.0) ctl[0] = 1;
        } else {
            ctl[1] += 1;
            if (rn2 < scal[S_THRESH] || ctl[1] >= ctl[3]) {
                ctl[0] = 1;
            } else {
                double absOld = scal[S_ABSNEW];
                scal[S_ABSNEW] = zz;
                scal[S_BETA] = zz / absOld;
            }
        }
    }
}

// The coarse levels [lc, L) hold few vertices (at most kCoarse).  One
// workgroup runs all of them with the level values in LDS and a barrier
// between levels, replacing one launch per level.
constexpr int kCoarse = 12288;
constexpr int kCoarseT = 1024;
// vertices per thread whose lists and values a thread loads before the level
// loop; larger ranges load them level by level
constexpr int kCoarseHold = 2;
// level of coarse vertex i (C.lc <= level < C.L)
__device__ inline int coarse_level(const Coarse& C, uint32_t i) {
    int d = C.lc;
    while (d + 1 < C.L && i >= C.off[d + 1]) ++d;
    return d;
}

// g = G p on the coarse levels (with the search direction update when upd).
// When the range holds at most kCoarseHold vertices per thread, every thread
// loads its vertices' lists and values before the level loop, which then waits
// only for the LDS values of the level above; the sums keep the same order.
__device__ inline void prolong_coarse_body(const Coarse& C, const Lists& A, float* p, const float* z, float* g,
                                           const double* scal, int upd, float* sg) {
    const uint32_t base = C.off[C.lc], end = C.off[C.L];
    const float beta = upd ? (float)scal[S_BETA] : 0.f;
    auto value = [&](uint32_t i) {
        float pi = p[i];
        if (upd) {
            pi = z[i] + beta * pi;
            p[i] = pi;
        }
        return pi;
    };
    auto step = [&](uint32_t i, uint4 P, float pi) {
        float w;
        const float s = gather_parents<float>(P, w, base, [&](uint32_t j) { return sg[j - base]; });
        const float v = pi + w * s;
        sg[i - base] = v;
        g[i] = v;
    };
    if (end - base <= kCoarseHold * blockDim.x) {
        int lev[kCoarseHold];
        uint4 P[kCoarseHold];
        float pi[kCoarseHold];
#pragma unroll
        for (int v = 0; v < kCoarseHold; ++v) {
            const uint32_t i = base + threadIdx.x + v * blockDim.x;
            lev[v] = -1;
            if (i < end) {
                lev[v] = coarse_level(C, i);
                P[v] = A.par[i];
                pi[v] = value(i);
            }
        }
        for (int d = C.L - 1; d >= C.lc; --d) {
#pragma unroll
            for (int v = 0; v < kCoarseHold; ++v)
                if (lev[v] == d) step(base + threadIdx.x + v * blockDim.x, P[v], pi[v]);
            __syncthreads();
        }
        return;
    }
    for (int d = C.L - 1; d >= C.lc; --d) {
        for (uint32_t i = C.off[d] + threadIdx.x; i < C.off[d + 1]; i += blockDim.x) step(i, A.par[i], value(i));
        __syncthreads();
    }
}
// restriction over the coarse levels [C.lc, C.L) (C.lc >= 1), as in
// prolong_coarse_body; the lowest of them reads its children from memory
__device__ inline void restrict_coarse_body(const Coarse& C, const Lists& A, float* h, float* sh) {
    const uint32_t base = C.off[C.lc], end = C.off[C.L];
    auto put = [&](uint32_t c, float hc) {
        sh[c - base] = hc;
        h[c] = hc;
    };
    if (end - base <= kCoarseHold * blockDim.x) {
        int lev[kCoarseHold];
        uint32_t e[kCoarseHold][9];
        float hc[kCoarseHold];
#pragma unroll
        for (int v = 0; v < kCoarseHold; ++v) {
            const uint32_t c = base + threadIdx.x + v * blockDim.x;
            lev[v] = -1;
            if (c < end) {
                lev[v] = coarse_level(C, c);
                load_kids(A, c, e[v]);
                hc[v] = h[c];
            }
        }
#pragma unroll
        for (int v = 0; v < kCoarseHold; ++v)
            if (lev[v] == C.lc)
                put(base + threadIdx.x + v * blockDim.x,
                    hc[v] + sum_children<float>(e[v], base, [&](uint32_t y) { return h[y]; }));
        __syncthreads();
        for (int d = C.lc + 1; d < C.L; ++d) {
#pragma unroll
            for (int v = 0; v < kCoarseHold; ++v)
                if (lev[v] == d)
                    put(base + threadIdx.x + v * blockDim.x,
                        hc[v] + sum_children<float>(e[v], base, [&](uint32_t y) { return sh[y - base]; }));
            __syncthreads();
        }
        return;
    }
    for (int d = C.lc; d < C.L; ++d) {
        for (uint32_t c = C.off[d] + threadIdx.x; c < C.off[d + 1]; c += blockDim.x) {
            uint32_t e[9];
            load_kids(A, c, e);
            put(c, h[c] + sum_children<float>(e, base, [&](uint32_t y) { return d == C.lc ? h[y] : sh[y - base]; }));
        }
        __syncthreads();
    }
}

struct Fit {
    int64_t n = 0;
    int L = 0;
    int64_t off[kMaxLevels + 1] = {0};
    DBuf<uint4> par;                   // prolongation: coarse parents of each vertex (Lists)
    DBuf<uint32_t> kid;                // restriction: fine children of each vertex from level 1 on (Lists)
    int64_t entries = 0;               // parents in all
    DBuf<uint32_t> down, up;           // finest coincident vertex; coincident vertex one level up
    DBuf<uint8_t> finest;
    DBuf<float> invd32;
    DBuf<double> invd64;
    // inner CGLS vectors (binary32)
    DBuf<float> x, r, p, z, t, g, h;
    // binary64 work vectors
    DBuf<double> g64, h64, r64, nr64, b64, tmp64;
    // reductions and device scalars
    DBuf<double> part;
    DBuf<double> scal;     // see Scal
    DBuf<int> ctl;         // [0] done, [1] iterations, [2] structure error
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    int graph_chunk = 0;
    int lc = 0;            // first level handled by the one-workgroup coarse kernels
    Coarse coarse{};
    Lists lists() const { return Lists{par.p, kid.p, L > 1 ? off[1] : n}; }
    ~Fit() {
        if (gexec) (void)hipGraphExecDestroy(gexec);
        if (graph) (void)hipGraphDestroy(graph);
    }
};
Fit* fit_get(its_svo s);

}  // namespace its
