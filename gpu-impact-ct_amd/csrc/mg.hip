// Multigrid V cycle (BiCGstab preconditioner 1) on the device (gfx950).
//
// multigridV(.TRUE., 1, bb, phi) (src/mod_solvers.f90:456-585) with its parts:
// relax_restrict (relaxation, product_div_grad_relax, restrict), relax_bottom
// and interpolate_relax (interpolate, relaxation).  The relaxation is the
// Jacobi branch of relaxation_div_grad / relaxation_div_grad_inv with omega
// 0.98 (src/mod_laplace.f90:466-597, 712-790) on each level's pressure range;
// the reference's exchange_relax (src/mod_exchange.f90:1273-1480) becomes
// wrapped reads across periodic directions.  Every value is formed with the
// reference's operation order, so the cycle is bit-identical to the loop
// restatement.
//
// Large levels run one launch per step (the JOR sweeps of kernels.hip, and one
// thread per coarse point or cell for the transfers).  A launch of a few
// microseconds costs about as much as the work of a small level, so the levels
// from the first of at most MG_FUSED_POINTS points run inside one
// single-workgroup kernel that walks the rest of the cycle in LDS.
#include "ih_device.h"
#include "ih_mg.h"

#include <type_traits>
#include <utility>

namespace ih {

using namespace dev;

namespace {

// index along d after exchange_relax: periodic directions wrap onto S?p..N?p
__device__ inline int wrapd(const Geo &g, int d, int idx) {
    if (!g.per[d]) return idx;
    const int P = g.Np[d] - g.Sp[d] + 1;
    if (idx < g.Sp[d]) return idx + P;
    if (idx > g.Np[d]) return idx - P;
    return idx;
}

__device__ inline int64_t wix(const Geo &g, int i, int j, int k) {
    return gidx(g, wrapd(g, 0, i), wrapd(g, 1, j), wrapd(g, 2, k));
}

// ---- per-point steps (T: the arithmetic type of the cycle)

// first relaxation of a level (r == 1 with init_yes): rel = omega bb / diag
template <typename T>
__device__ inline void pt_init(const Geo &g, const T *const *dg, int i, int j, int k, T omega, const T *bb, T *x) {
    const int64_t p = gidx(g, i, j, k);
    const T d = (dg[0][g.cst[0] + i] + dg[1][g.cst[1] + j]) + dg[2][g.cst[2] + k];
    x[p] = omega * bb[p] / d;
}

// Averaging on the edges of wall pairs, the reference's statements in order:
// direction pairs (1,2), (1,3), (2,3), per pair the sides (L,L), (L,U), (U,L),
// (U,U), each a line over 1..N of the third direction.  THREE = false: two
// neighbours / 2 (restrict, src/mod_solvers.f90:632-661); true: three neighbours
// / 3 (interpolate, :1028-1043).
// The pairs write only points with walls of two or more directions, and the last pair
// to write a point reads points with fewer walls or ones that an earlier pair wrote
// from such points, so the value after all three pairs is a function of the field
// before them, of its points with at most one wall: a reader forms it where it needs
// it, and it can be stored by one thread while others form theirs.  The corner's is
// formed by the pair (2,3) from values that the pairs (1,3) and (1,2) left.
template <typename T, bool THREE, typename F>
__device__ inline T edge_value(const int *N, const bool *wall, int i, int j, int k, F f) {
    const int ii = i == 1 ? 2 : N[0] - 1, jj = j == 1 ? 2 : N[1] - 1, kk = k == 1 ? 2 : N[2] - 1;
    auto avg = [](T a, T b, T c) { return THREE ? (a + b + c) / T(3) : (a + b) / T(2); };
    auto e01 = [&](int c) { return avg(f(ii, j, c), f(i, jj, c), THREE ? f(ii, jj, c) : T(0)); };
    auto e02 = [&](int b) { return avg(f(ii, b, k), f(i, b, kk), THREE ? f(ii, b, kk) : T(0)); };
    if (wall[1] && wall[2]) {
        if (wall[0]) return avg(e02(jj), e01(kk), THREE ? f(i, jj, kk) : T(0));
        return avg(f(i, jj, k), f(i, j, kk), THREE ? f(i, jj, kk) : T(0));
    }
    return wall[2] ? e02(j) : e01(k);
}

// walls at (i, j, k), and whether they are two or more
__device__ inline bool edge_point(const int *N, const int *per, int i, int j, int k, bool *wall) {
    wall[0] = !per[0] && (i == 1 || i == N[0]);
    wall[1] = !per[1] && (j == 1 || j == N[1]);
    wall[2] = !per[2] && (k == 1 || k == N[2]);
    return (int)wall[0] + (int)wall[1] + (int)wall[2] >= 2;
}

template <typename T, bool THREE>
__device__ inline T edge_value(const Geo &g, int i, int j, int k, const T *f) {
    bool w[3];
    edge_point(g.N, g.per, i, j, k, w);
    return edge_value<T, THREE>(g.N, w, i, j, k, [&](int a, int b, int c) { return f[gidx(g, a, b, c)]; });
}

// a point of a level's field as the averages need it: its walls, and the points that a
// two-wall point is averaged from (inward along the one, the other and both walls'
// directions; else the point itself), for loads without a branch
struct EdgeAt {
    int64_t p, a, b, c;
    int walls;
};
__device__ inline EdgeAt edge_at(const Geo &g, int i, int j, int k) {
    EdgeAt q;
    bool w[3];
    const bool in = i >= 1 && j >= 1 && k >= 1 && i <= g.N[0] && j <= g.N[1] && k <= g.N[2];
    edge_point(g.N, g.per, i, j, k, w);
    q.walls = in ? (int)w[0] + (int)w[1] + (int)w[2] : 0;
    q.p = gidx(g, i, j, k);
    const int64_t d0 = i == 1 ? 1 : -1, d1 = j == 1 ? g.px : -(int64_t)g.px, d2 = k == 1 ? g.pxy : -g.pxy;
    const int64_t da = w[0] ? d0 : d1, db = w[2] ? d2 : d1;
    q.a = q.walls == 2 ? q.p + da : q.p;
    q.b = q.walls == 2 ? q.p + db : q.p;
    q.c = q.walls == 2 ? q.p + da + db : q.p;
    return q;
}
__device__ inline void point_of(const Geo &g, int64_t p, int &i, int &j, int &k) {
    p -= g.lead;
    k = (int)(p / g.pxy) - 3;
    p -= (int64_t)(k + 3) * g.pxy;
    j = (int)(p / g.px) - 3;
    i = (int)(p - (int64_t)(j + 3) * g.px) - 3;
}

template <typename T>
__device__ inline const T *const *dg_of(const Coef &c);
template <>
__device__ inline const double *const *dg_of<double>(const Coef &c) {
    return c.dg;
}
template <>
__device__ inline const float *const *dg_of<float>(const Coef &c) {
    return c.dgf;
}

// ---- one launch per step (large levels) ------------------------------------

template <typename T>
__global__ void k_mg_init(Geo g, Coef c, Range3 r, T omega, const T *__restrict__ bb, T *__restrict__ x,
                          const int *active) {
    if (active && !*active) return;
    IH_POINT(r);
    pt_init<T>(g, dg_of<T>(c), i, j, k, omega, bb, x);
}

// the FP32 cycle's first relaxation on level 1, from the FP64 right-hand side:
// b32 = (float) v is stored for the later steps
__global__ void k_mg_init_f32_first(Geo g, Coef c, Range3 r, float omega, const double *__restrict__ v,
                                    float *__restrict__ b32, float *__restrict__ x, const int *active) {
    if (active && !*active) return;
    IH_POINT(r);
    const int64_t p = gidx(g, i, j, k);
    b32[p] = (float)v[p];
    pt_init<float>(g, c.dgf, i, j, k, omega, b32, x);
}


template <typename T>
struct LevelW {
    const T *w[3];
    int d[3];
};

// restrict(.TRUE., g, coarse, bb, lap) (src/mod_solvers.f90:632-714) by coarse points:
// bb - lap on the seven fine points with both averaged on the edges; the averaged bb
// (the later sweeps read it) is stored by the thread whose fine cell holds the point,
// v's as well if given (the FP32 cycle's right-hand side is a copy of it).  With xinit
// the coarse level's first relaxation too (omega A / diag at the same point, the value
// pt_init forms).  Bound by latency but on level 1; with the averages in a launch of
// their own, 7.8 + 5.7 microseconds over the levels of 257x129x129 (4.7 + 4.8 at 97^3),
// here 11.7 (8.2).
template <typename T>
__global__ __launch_bounds__(BX * BY) void k_mg_restrict(Geo gf, Geo gc, LevelW<T> R, Coef cc, Range3 r, T *bb, const T *__restrict__ lap,
                              double *v, T *__restrict__ out, T *__restrict__ xinit, T omega, const int *active) {
    if (active && !*active) return;
    const int ii = r.lo0 + (int)(blockIdx.x * BX + threadIdx.x);
    const int jj = r.lo1 + (int)(blockIdx.y * BY + threadIdx.y);
    const int kk = r.lo2 + (int)blockIdx.z;
    if (ii >= r.lo0 + r.n0 || jj >= r.lo1 + r.n1) return;
    const int i = R.d[0] * (ii - 1) + 1, j = R.d[1] * (jj - 1) + 1, k = R.d[2] * (kk - 1) + 1;
    auto near_wall = [&](int d, int t) { return !gf.per[d] && (t <= 2 || t >= gf.N[d] - 1); };
    T df[7];
    auto raw = [&](int a, int b, int c) {
        const int64_t p = wix(gf, a, b, c);
        return bb[p] - lap[p];
    };
    if ((int)near_wall(0, i) + (int)near_wall(1, j) + (int)near_wall(2, k) < 2) {
        df[0] = raw(i, j, k);
        df[1] = raw(i - 1, j, k);
        df[2] = raw(i + 1, j, k);
        df[3] = raw(i, j - 1, k);
        df[4] = raw(i, j + 1, k);
        df[5] = raw(i, j, k - 1);
        df[6] = raw(i, j, k + 1);
    } else {
        // all loads first: an edge point's two neighbours, else the point twice
        EdgeAt q[7];
        T fa[7], fb[7], la[7], lb[7];
#pragma unroll
        for (int e = 0; e < 7; ++e) {
            q[e] = edge_at(gf, wrapd(gf, 0, i + (e == 2) - (e == 1)), wrapd(gf, 1, j + (e == 4) - (e == 3)),
                           wrapd(gf, 2, k + (e == 6) - (e == 5)));
            fa[e] = bb[q[e].a];
            fb[e] = bb[q[e].b];
            la[e] = lap[q[e].a];
            lb[e] = lap[q[e].b];
        }
        auto store = [&](int64_t p, T value) {
            bb[p] = value;
            if (v) {
                int a, b, c;
                point_of(gf, p, a, b, c);
                v[p] = edge_value<double, false>(gf, a, b, c, v);
            }
        };
#pragma unroll
        for (int e = 0; e < 7; ++e) {
            T f = q[e].walls == 2 ? (fa[e] + fb[e]) / T(2) : fa[e], l = q[e].walls == 2 ? (la[e] + lb[e]) / T(2) : la[e];
            if (q[e].walls == 3) {
                int a, b, c;
                point_of(gf, q[e].a, a, b, c);
                f = edge_value<T, false>(gf, a, b, c, bb);
                l = edge_value<T, false>(gf, a, b, c, lap);
            }
            df[e] = f - l;
            // the thread's fine points: its own and, along a halved direction, the next
            if (q[e].walls >= 2 && (e == 0 || (e % 2 == 0 && R.d[e / 2 - 1] == 2 && (e == 2 ? i : e == 4 ? j : k) < gf.N[e / 2 - 1])))
                store(q[e].p, f);
        }
        // the last point along a periodic direction: no level reads it, its average is
        // part of the field all the same
        if (q[0].walls == 2) {
            const bool last[3] = {ii == r.lo0 + r.n0 - 1, jj == r.lo1 + r.n1 - 1, kk == r.lo2 + r.n2 - 1};
            for (int d = 0; d < 3; ++d) {
                if (!gf.per[d] || !last[d]) continue;
                const int a = d == 0 ? gf.N[0] : i, b = d == 1 ? gf.N[1] : j, c = d == 2 ? gf.N[2] : k;
                store(gidx(gf, a, b, c), edge_value<T, false>(gf, a, b, c, bb));
            }
        }
    }
    const int s1 = gc.cst[0], s2 = gc.cst[1], s3 = gc.cst[2];
    const T *const *w = R.w;
    const T wc = (w[0][s1 + ii] + w[1][s2 + jj]) + w[2][s3 + kk];
    const T wn[6] = {w[0][ii], w[0][2 * s1 + ii], w[1][jj], w[1][2 * s2 + jj], w[2][kk], w[2][2 * s3 + kk]};
    T t = wc * df[0];
#pragma unroll
    for (int e = 0; e < 6; ++e) t = t + wn[e] * df[1 + e];
    const T a = t / T(3);
    out[gidx(gc, ii, jj, kk)] = a;
    if (xinit) {
        const T *const *dg = dg_of<T>(cc);
        const T d = (dg[0][gc.cst[0] + ii] + dg[1][gc.cst[1] + jj]) + dg[2][gc.cst[2] + kk];
        xinit[gidx(gc, ii, jj, kk)] = omega * a / d;
    }
}

// interpolate(.TRUE., g, coarse, fine, work) (src/mod_solvers.f90:1028-1141) added to
// fine, by coarse cells: the thread of cell (I, J, K) writes the fine points
// dn*(T-1)+1+s, s < dn (s = 0 only at T = Nc), from the eight coarse values around it
// (averaged on the edges; nothing else reads those, so they are not stored): the
// injected values, then the z, y and x passes with the operands each pass reads.
// 8.9 + 5.7 microseconds over the levels of 257x129x129 with the averages in a launch
// of their own, here 11.9 (97^3: 6.2 + 4.8, here 9.5)
template <typename T>
__global__ __launch_bounds__(BX * BY) void k_mg_interp_cells(Geo gf, Geo gc, LevelW<T> W, const T *__restrict__ coarse, T *__restrict__ fine,
                                  const int *active) {
    if (active && !*active) return;
    const int I = 1 + (int)(blockIdx.x * BX + threadIdx.x);
    const int J = 1 + (int)(blockIdx.y * BY + threadIdx.y);
    const int K = 1 + (int)blockIdx.z;
    if (I > gc.N[0] || J > gc.N[1]) return;
    const int Tc[3] = {I, J, K};
    int ns[3];
    for (int d = 0; d < 3; ++d) ns[d] = (W.d[d] == 2 && Tc[d] < gc.N[d]) ? 2 : 1;
    // coarse values at (I + a, J + b, K + e); a direction with one fine point
    // per cell reads index 0 only
    const int i0 = W.d[0] * (I - 1) + 1, j0 = W.d[1] * (J - 1) + 1, k0 = W.d[2] * (K - 1) + 1;
    const int s1 = gf.cst[0], s2 = gf.cst[1], s3 = gf.cst[2];
    // the weights of the points off the lattice and the fine values do not wait for the
    // coarse ones
    const int ix = i0 + ns[0] - 1, jx = j0 + ns[1] - 1, kx = k0 + ns[2] - 1;
    const T w1a = W.w[0][ix], w1b = W.w[0][s1 + ix], w2a = W.w[1][jx], w2b = W.w[1][s2 + jx], w3a = W.w[2][kx],
            w3b = W.w[2][s3 + kx];
    typedef T T2 __attribute__((ext_vector_type(2)));
    T2 fv[2][2];  // i0 is odd where a direction is halved: a pair of points is aligned
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const T *const f = fine + gidx(gf, i0, j0 + ((q & 1) < ns[1] ? q & 1 : 0), k0 + (q >> 1 < ns[2] ? q >> 1 : 0));
        if (ns[0] == 2)
            fv[q & 1][q >> 1] = *(const T2 *)f;
        else
            fv[q & 1][q >> 1] = T2{*f, T(0)};
    }
    T cv[2][2][2];
    auto near_wall = [&](int d, int t) { return !gc.per[d] && (t == 1 || t >= gc.N[d] - 1); };
    const bool edges = (int)near_wall(0, I) + (int)near_wall(1, J) + (int)near_wall(2, K) >= 2;
    auto corner = [&](int q, int d) { return Tc[d] + ((q >> d & 1) < ns[d] ? q >> d & 1 : 0); };
    if (!edges) {
#pragma unroll
        for (int q = 0; q < 8; ++q)
            cv[q & 1][q >> 1 & 1][q >> 2] = coarse[wix(gc, corner(q, 0), corner(q, 1), corner(q, 2))];
    } else {
        T f[8][3];
        int walls[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const EdgeAt at =
                edge_at(gc, wrapd(gc, 0, corner(q, 0)), wrapd(gc, 1, corner(q, 1)), wrapd(gc, 2, corner(q, 2)));
            walls[q] = at.walls;
            f[q][0] = coarse[at.a];
            f[q][1] = coarse[at.b];
            f[q][2] = coarse[at.c];
        }
        T three = T(0);  // a cell has one point on three walls at most
        bool any = false;
#pragma unroll
        for (int q = 0; q < 8; ++q) any = any || walls[q] == 3;
        if (any)
            three = edge_value<T, true>(gc, I == 1 ? 1 : gc.N[0], J == 1 ? 1 : gc.N[1], K == 1 ? 1 : gc.N[2], coarse);
#pragma unroll
        for (int q = 0; q < 8; ++q)
            cv[q & 1][q >> 1 & 1][q >> 2] =
                walls[q] == 3 ? three : (walls[q] == 2 ? (f[q][0] + f[q][1] + f[q][2]) / T(3) : f[q][0]);
    }
#pragma unroll
    for (int se = 0; se < 2; ++se) {
        // z pass at the four lattice columns (a, b)
        T wz[2][2];
        for (int b = 0; b < 2; ++b)
            for (int a = 0; a < 2; ++a) wz[a][b] = se == 0 ? cv[a][b][0] : w3a * cv[a][b][0] + w3b * cv[a][b][1];
#pragma unroll
        for (int sb = 0; sb < 2; ++sb) {
            if (se >= ns[2] || sb >= ns[1]) continue;
            // y pass at the two lattice x positions
            T wy[2];
            for (int a = 0; a < 2; ++a) wy[a] = sb == 0 ? wz[a][0] : w2a * wz[a][0] + w2b * wz[a][1];
            T *const f = fine + gidx(gf, i0, j0 + sb, k0 + se);
            const T2 v = {fv[sb][se][0] + wy[0], fv[sb][se][1] + (w1a * wy[0] + w1b * wy[1])};
            if (ns[0] == 2)
                *(T2 *)f = v;
            else
                *f = v[0];
        }
    }
}

// ---- levels g0..G in one workgroup ------------------------------------------

constexpr int MG_FUSED_THREADS = 1024;
constexpr int MG_FUSED_OWN = (int)(MG_FUSED_POINTS / MG_FUSED_THREADS);  // points of a level a thread owns

struct MgFusedLevel {
    int P[3], N[3], dn[3], cst[3];  // points of the range, sizes, ratios to the next level, table strides
    int tab;                        // its tables: per direction dg, cR (3 cst) and cI (2 cst)
    int A, X;                       // right-hand side and iterate in the pool (X[0] is a zero, points from X[1])
};
struct MgFusedArgs {
    MgFusedLevel L[MG_LEVELS_MAX + 1];
    Geo g;  // of level g0
    int g0, G, n_down, n_up, n_bottom;
    int per[3];
    int ntab, tmp;  // table elements (from 0 in the pool), the second iterate of any level (as X)
};

// The rest of the cycle from level g0: its right-hand side A is in place, its last
// iterate goes to out.  Everything lives in LDS: the tables, and per level the points
// of the pressure range without halos (a neighbour past a wall is the zero in front of
// the iterate, one across a periodic pair the wrapped point).  A thread owns the same
// points of a level through all its steps, with their coefficients, neighbours and
// right-hand side in registers, so a sweep is seven LDS reads, the point's chain and a
// barrier.  One workgroup's chain of about 40 steps a cycle: the latency of a step, and
// the one compute unit's issue on its larger levels, bound it.  17x9x9 and coarser:
// 111 -> 31 microseconds with the fields in LDS instead of the levels' arrays.
template <typename T>
__global__ __launch_bounds__(MG_FUSED_THREADS) void k_mg_fused(MgFusedArgs args, const T *__restrict__ tables,
                                                               const T *__restrict__ Ag, T *__restrict__ out, T omega,
                                                               const int *active) {
    if (active && !*active) return;
    __shared__ T pool[MG_FUSED_LDS / sizeof(T)];
    // the levels are indexed where they are passed (a reference to the parameter would
    // be a copy of it in scratch memory)
    (void)args;
    const auto *const a =
        (const __attribute__((address_space(4))) MgFusedArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    const int tid = (int)threadIdx.x;
    const int g0 = a->g0, G = a->G, n_down = a->n_down, n_up = a->n_up, n_bottom = a->n_bottom, tmp = a->tmp;
    const int per[3] = {a->per[0], a->per[1], a->per[2]};
    constexpr int OWN = MG_FUSED_OWN;
    // an owned point: its neighbours (a direction's two, 16 bits each, from the iterate's
    // zero), coefficients, diagonal and right-hand side
    struct Own {
        unsigned nb[3];
        T c[6], d, A;
    };
    Own o[OWN];
    struct Level {
        int P[3], N[3], dn[3], cst[3], tab, A, X, n;
    };
    auto level = [&](int g) {
        const auto &q = a->L[g];
        Level l;
        for (int d = 0; d < 3; ++d) {
            l.P[d] = q.P[d];
            l.N[d] = q.N[d];
            l.dn[d] = q.dn[d];
            l.cst[d] = q.cst[d];
        }
        l.tab = q.tab;
        l.A = q.A;
        l.X = q.X;
        l.n = l.P[0] * l.P[1] * l.P[2];
        return l;
    };
    auto split = [](const Level &l, int q, int &i, int &j, int &k) {
        const int r = q / l.P[0];
        i = 1 + q - r * l.P[0];
        k = 1 + r / l.P[1];
        j = 1 + r - (k - 1) * l.P[1];
    };
    const int lead = a->g.lead, px = a->g.px;
    const int64_t pxy = a->g.pxy;
    auto at = [&](int i, int j, int k) {  // gidx
        return lead + (i + 3) + (int64_t)px * (j + 3) + pxy * (k + 3);
    };
    for (int t = tid; t < a->ntab; t += MG_FUSED_THREADS) pool[t] = tables[t];
    if (tid == 0) {
        for (int g = g0; g <= G; ++g) pool[a->L[g].X] = T(0);
        pool[tmp] = T(0);
    }
    {
        const Level l = level(g0);
        for (int q = tid; q < l.n; q += MG_FUSED_THREADS) {
            int i, j, k;
            split(l, q, i, j, k);
            pool[l.A + q] = Ag[at(i, j, k)];
        }
    }
    __syncthreads();
    auto enter = [&](const Level &l) {
        const T *const t0 = pool + l.tab, *const t1 = t0 + 8 * l.cst[0], *const t2 = t1 + 8 * l.cst[1];
#pragma unroll
        for (int m = 0; m < OWN; ++m) {
            const int q = tid + m * MG_FUSED_THREADS;
            if (q >= l.n) continue;
            Own &p = o[m];
            int i, j, k;
            split(l, q, i, j, k);
            auto nb = [&](int x, int P, int pr, int stride) {
                const int lo = x > 1 ? q + 1 - stride : (pr ? q + 1 + (P - 1) * stride : 0);
                const int hi = x < P ? q + 1 + stride : (pr ? q + 1 - (P - 1) * stride : 0);
                return (unsigned)(lo | hi << 16);
            };
            p.nb[0] = nb(i, l.P[0], per[0], 1);
            p.nb[1] = nb(j, l.P[1], per[1], l.P[0]);
            p.nb[2] = nb(k, l.P[2], per[2], l.P[0] * l.P[1]);
            p.c[0] = t0[i];
            p.c[1] = t0[2 * l.cst[0] + i];
            p.c[2] = t1[j];
            p.c[3] = t1[2 * l.cst[1] + j];
            p.c[4] = t2[k];
            p.c[5] = t2[2 * l.cst[2] + k];
            p.d = (t0[l.cst[0] + i] + t1[l.cst[1] + j]) + t2[l.cst[2] + k];
            p.A = pool[l.A + q];
        }
    };
    auto nbr = [](const Own &p, int e) { return (int)(e & 1 ? p.nb[e >> 1] >> 16 : p.nb[e >> 1] & 0xffffu); };
    int x = 0, y = 0;  // the level's iterate and the other buffer
    auto sweeps = [&](const Level &l, int n) {
        for (; n > 0; --n) {
#pragma unroll
            for (int m = 0; m < OWN; ++m) {
                const int q = tid + m * MG_FUSED_THREADS;
                if (q >= l.n) continue;
                const Own &p = o[m];
                T v[6];
#pragma unroll
                for (int e = 0; e < 6; ++e) v[e] = pool[x + nbr(p, e)];
                const T own = pool[x + q + 1];
                T t = p.A;
#pragma unroll
                for (int e = 0; e < 6; ++e) t = t - p.c[e] * v[e];
                pool[y + q + 1] = omega * t / p.d + (T(1) - omega) * own;
            }
            __syncthreads();
            const int z = x;
            x = y;
            y = z;
        }
    };
    // the first relaxation, from zero; flips: the sweeps that follow before the iterate
    // has to be in X
    auto first = [&](const Level &l, int flips) {
        x = flips & 1 ? tmp : l.X;
        y = flips & 1 ? l.X : tmp;
#pragma unroll
        for (int m = 0; m < OWN; ++m) {
            const int q = tid + m * MG_FUSED_THREADS;
            if (q < l.n) pool[x + q + 1] = omega * o[m].A / o[m].d;
        }
        __syncthreads();
    };
    // the averages on the edges of the arrays at f1 and (if >= 0) f2
    auto edges = [&](const Level &l, auto three, int f1, int f2) {
        for (int q = tid; q < l.n; q += MG_FUSED_THREADS) {
            int i, j, k;
            split(l, q, i, j, k);
            bool w[3];
            if (!edge_point(l.N, per, i, j, k, w)) continue;
            for (int f = f1; f >= 0; f = f == f1 ? f2 : -1)
                pool[f + q] = edge_value<T, decltype(three)::value>(l.N, w, i, j, k, [&](int u, int v, int t) {
                    return pool[f + (u - 1) + l.P[0] * ((v - 1) + l.P[1] * (t - 1))];
                });
        }
        __syncthreads();
    };
    Level l = level(g0);
    for (int g = g0; g < G; ++g) {
        const Level lc = level(g + 1);
        enter(l);
        first(l, n_down - 1);
        sweeps(l, n_down - 1);
        // the residual product, then the averages on the edges of it and of A
        const int A = l.A, C = tmp + 1;
#pragma unroll
        for (int m = 0; m < OWN; ++m) {
            const int q = tid + m * MG_FUSED_THREADS;
            if (q >= l.n) continue;
            const Own &p = o[m];
            T t = p.c[0] * pool[l.X + nbr(p, 0)];
#pragma unroll
            for (int e = 1; e < 6; ++e) t = t + p.c[e] * pool[l.X + nbr(p, e)];
            pool[C + q] = t + p.d * pool[l.X + q + 1];
        }
        __syncthreads();
        edges(l, std::false_type{}, A, C);
        // A - C on the points of the coarse level
        const T *const w0 = pool + lc.tab + 3 * lc.cst[0], *const w1 = w0 + 5 * lc.cst[0] + 3 * lc.cst[1],
                       *const w2 = w1 + 5 * lc.cst[1] + 3 * lc.cst[2];
        for (int q = tid; q < lc.n; q += MG_FUSED_THREADS) {
            int ii, jj, kk;
            split(lc, q, ii, jj, kk);
            const int st1 = l.P[0], st2 = l.P[0] * l.P[1];
            const int c0 = l.dn[0] * (ii - 1), c1 = l.dn[1] * (jj - 1), c2 = l.dn[2] * (kk - 1);  // from 0
            const int p = c0 + st1 * c1 + st2 * c2;
            auto lo = [&](int c, int P, int pr, int st) { return c > 0 ? p - st : (pr ? p + (P - 1) * st : -1); };
            auto hi = [&](int c, int P, int pr, int st) { return c < P - 1 ? p + st : (pr ? p - (P - 1) * st : -1); };
            auto df = [&](int u) { return u < 0 ? T(0) : pool[A + u] - pool[C + u]; };
            T t = ((w0[lc.cst[0] + ii] + w1[lc.cst[1] + jj]) + w2[lc.cst[2] + kk]) * df(p);
            t = t + w0[ii] * df(lo(c0, l.P[0], per[0], 1));
            t = t + w0[2 * lc.cst[0] + ii] * df(hi(c0, l.P[0], per[0], 1));
            t = t + w1[jj] * df(lo(c1, l.P[1], per[1], st1));
            t = t + w1[2 * lc.cst[1] + jj] * df(hi(c1, l.P[1], per[1], st1));
            t = t + w2[kk] * df(lo(c2, l.P[2], per[2], st2));
            t = t + w2[2 * lc.cst[2] + kk] * df(hi(c2, l.P[2], per[2], st2));
            pool[lc.A + q] = t / T(3);
        }
        __syncthreads();
        l = lc;
    }
    enter(l);
    first(l, 0);
    sweeps(l, 2 * n_bottom - 1);
    for (int g = G - 1; g >= g0; --g) {
        const Level lc = l;
        l = level(g);
        const int xc = x + 1;
        edges(lc, std::true_type{}, xc, -1);
        enter(l);
        const T *const i0 = pool + l.tab + 6 * l.cst[0], *const i1 = i0 + 2 * l.cst[0] + 6 * l.cst[1],
                       *const i2 = i1 + 2 * l.cst[1] + 6 * l.cst[2];
        for (int q = tid; q < l.n; q += MG_FUSED_THREADS) {
            int i, j, k;
            split(l, q, i, j, k);
            // a direction's coarse neighbours below and above; the same one on the lattice
            auto below = [](int t, int dn) { return (t - 1) >> (dn - 1); };  // from 0
            auto above = [](int b, bool on, int P) { return on ? b : (b + 1 < P ? b + 1 : 0); };
            const bool li = l.dn[0] == 1 || (i & 1), lj = l.dn[1] == 1 || (j & 1), lk = l.dn[2] == 1 || (k & 1);
            const int I0 = below(i, l.dn[0]), J0 = below(j, l.dn[1]), K0 = below(k, l.dn[2]);
            const int I1 = above(I0, li, lc.P[0]), J1 = above(J0, lj, lc.P[1]), K1 = above(K0, lk, lc.P[2]);
            const T k0 = i2[k], k1 = i2[l.cst[2] + k], j0 = i1[j], j1 = i1[l.cst[1] + j], x0 = i0[i],
                    x1 = i0[l.cst[0] + i];
            auto wz = [&](int I, int J) {
                const int r = xc + I + lc.P[0] * J, s2 = lc.P[0] * lc.P[1];
                const T lo = pool[r + s2 * K0], hi = pool[r + s2 * K1];
                return lk ? lo : k0 * lo + k1 * hi;
            };
            auto wy = [&](int I) {
                const T lo = wz(I, J0), hi = wz(I, J1);
                return lj ? lo : j0 * lo + j1 * hi;
            };
            const T lo = wy(I0), hi = wy(I1);
            pool[l.X + q + 1] = pool[l.X + q + 1] + (li ? lo : x0 * lo + x1 * hi);
        }
        __syncthreads();
        x = l.X;
        y = tmp;
        sweeps(l, n_up);
    }
    for (int q = tid; q < l.n; q += MG_FUSED_THREADS) {
        int i, j, k;
        split(l, q, i, j, k);
        out[at(i, j, k)] = pool[x + q + 1];
    }
}

// the layout of levels g0..G in the pool; false if it does not fit
bool fused_layout(const MgDev &m, int g0, MgFusedArgs &a) {
    a = MgFusedArgs{};
    a.g0 = g0;
    a.G = m.G;
    a.n_down = m.n_down;
    a.n_up = m.n_up;
    a.n_bottom = m.n_bottom;
    a.g = m.L[g0].g;
    int64_t at = 0, most = 0;
    for (int g = g0; g <= m.G; ++g) {
        MgFusedLevel &l = a.L[g];
        l.tab = (int)at;
        for (int d = 0; d < 3; ++d) {
            const Geo &q = m.L[g].g;
            l.P[d] = q.Np[d] - q.Sp[d] + 1;
            l.N[d] = q.N[d];
            l.dn[d] = m.L[g].dn[d];
            l.cst[d] = q.cst[d];
            a.per[d] = q.per[d];
            at += 8 * l.cst[d];
        }
    }
    a.ntab = (int)at;
    for (int g = g0; g <= m.G; ++g) {
        MgFusedLevel &l = a.L[g];
        const int64_t n = (int64_t)l.P[0] * l.P[1] * l.P[2];
        if (n > MG_FUSED_POINTS || l.P[0] > 1023 || l.P[1] > 1023 || l.P[2] > 1023) return false;
        most = std::max(most, n);
        l.A = (int)at;
        at += n;
        l.X = (int)at;
        at += n + 1;
    }
    a.tmp = (int)at;
    at += most + 1;
    return at * (int64_t)sizeof(double) <= MG_FUSED_LDS;
}

inline Range3 full_range(const Geo &g) { return Range3{1, 1, 1, g.N[0], g.N[1], g.N[2]}; }


// The cycle for arithmetic type T.  Level 1: right-hand side b1 (v itself for
// FP64; the float copy the first relaxation stores for FP32), iterate buffers
// x/y; the last sweep of level 1 writes z (for FP32 widened to double).
template <typename T>
struct CycleBufs;
template <>
struct CycleBufs<double> {
    static double *A(const MgLevel &L) { return L.A; }
    static double *B(const MgLevel &L) { return L.B; }
    static double *C(const MgLevel &L) { return L.C; }
    static double *D(const MgLevel &L) { return L.D; }
    static const double *const *cR(const MgLevel &L) { return L.cR; }
    static const double *const *cI(const MgLevel &L) { return L.cI; }
    static JorLaunch shape(const MgLevel &L) { return L.shape; }
    static const double *tables(const MgLevel &L) { return L.c.dg[0]; }
};
template <>
struct CycleBufs<float> {
    static float *A(const MgLevel &L) { return L.Af; }
    static float *B(const MgLevel &L) { return L.Bf; }
    static float *C(const MgLevel &L) { return L.Cf; }
    static float *D(const MgLevel &L) { return L.Df; }
    static const float *const *cR(const MgLevel &L) { return L.cRf; }
    static const float *const *cI(const MgLevel &L) { return L.cIf; }
    static JorLaunch shape(const MgLevel &L) { return L.shape32; }
    static const float *tables(const MgLevel &L) { return L.c.dgf[0]; }
};

// launches of n sweeps of a level: two a launch where its range takes pairs
inline bool level_pairs(const MgLevel &L, bool fp32) { return jor_pair_ok(L.g, L.c, L.pr, fp32); }
inline int sweep_launches(int n, bool pairs) { return pairs ? (n + 1) / 2 : n; }

inline void jor_any(hipStream_t s, const MgLevel &L, double omega, const double *x, const double *b, double *y,
                    const int *act, JorLaunch sh) {
    launch_jor(s, L.g, L.c, L.pr, omega, x, b, y, act, sh);
}
inline void jor_any(hipStream_t s, const MgLevel &L, float omega, const float *x, const float *b, float *y,
                    const int *act, JorLaunch sh) {
    launch_jor_f32(s, L.g, L.c, L.pr, omega, x, b, y, act, sh);
}

template <typename T>
void mg_cycle(hipStream_t s, const MgDev &m, double *v, double *z, const int *act) {
    using B_ = CycleBufs<T>;
    const int G = m.G;
    const int g0 = m.g0;  // levels g0..G run fused (g0 >= 2)
    const T omega = (T)m.omega;
    const bool fp64 = sizeof(T) == 8;
    T *b[MG_LEVELS_MAX + 1], *x[MG_LEVELS_MAX + 1], *y[MG_LEVELS_MAX + 1];
    if (fp64) {
        // level 1 alternates between z and D over the cycle's sweeps; starting on
        // the buffer that makes the last sweep write z leaves the result in place
        const bool p1 = level_pairs(m.L[1], false);
        const int flips1 = G > 1 ? sweep_launches(m.n_down - 1, p1) + sweep_launches(m.n_up, p1)
                                 : sweep_launches(m.n_bottom - 1, p1) + sweep_launches(m.n_bottom, p1);
        b[1] = (T *)v;
        x[1] = (flips1 % 2 == 0) ? (T *)z : B_::D(m.L[1]);
        y[1] = (x[1] == (T *)z) ? B_::D(m.L[1]) : (T *)z;
    } else {
        b[1] = B_::A(m.L[1]);
        x[1] = B_::B(m.L[1]);
        y[1] = B_::D(m.L[1]);
    }
    for (int g = 2; g <= G; ++g) {
        b[g] = B_::A(m.L[g]);
        x[g] = B_::B(m.L[g]);
        y[g] = B_::D(m.L[g]);
    }
    // relaxation of level g; init_done: the restriction into g already wrote the first
    // relaxation; last_to_z: the FP32 cycle's final sweep, written to z as double
    auto relax = [&](int g, bool init, int n, bool init_done = false, bool last_to_z = false) {
        const MgLevel &L = m.L[g];
        const Range3 r = make_range(L.pr);
        int q = 1;
        if (init && n >= 1) {
            if (!init_done) {
                if (!fp64 && g == 1)
                    hipLaunchKernelGGL(k_mg_init_f32_first, grid_for(r), dim3(BX, BY, 1), 0, s, L.g, L.c, r,
                                       (float)omega, (const double *)v, (float *)b[1], (float *)x[1], act);
                else
                    hipLaunchKernelGGL(k_mg_init<T>, grid_for(r), dim3(BX, BY, 1), 0, s, L.g, L.c, r, omega, b[g],
                                       x[g], act);
            }
            q = 2;
        }
        const bool pairs = level_pairs(L, !fp64);
        while (q <= n) {
            const int two = pairs && (n - q) % 2 == 1 ? 2 : 1;  // an odd count's single sweep comes first
            q += two;
            const bool to_z = last_to_z && q > n;
            if (two == 2) {
                if (to_z)
                    launch_jor_pair(s, L.g, L.c, L.pr, (float)omega, (const float *)x[g], (const float *)b[g], z, act);
                else
                    launch_jor_pair(s, L.g, L.c, L.pr, omega, (const T *)x[g], (const T *)b[g], y[g], act);
            } else {
                if (to_z)
                    launch_jor_f32_to64(s, L.g, L.c, L.pr, (float)omega, (const float *)x[g], (const float *)b[g], z,
                                        act, B_::shape(L));
                else
                    jor_any(s, L, omega, x[g], b[g], y[g], act, B_::shape(L));
            }
            std::swap(x[g], y[g]);
        }
    };
    if (G == 1) {
        relax(1, true, m.n_bottom);
        relax(1, false, m.n_bottom, false, !fp64);
        return;
    }
    const int gl = std::min(g0, G) - 1;  // last level with launches of its own on the way down
    for (int g = 1; g <= gl; ++g) {
        const MgLevel &L = m.L[g], &Lc = m.L[g + 1];
        relax(g, true, m.n_down, g >= 2);
        // the residual product with the JOR sweep's 16-byte lanes and launch shape
        // (one point a lane with seven 8-byte loads is bound by address issue)
        launch_lap(s, L.g, L.c, L.pr, (const T *)x[g], B_::C(L), act, B_::shape(L));
        LevelW<T> R;
        int nmax[3];
        for (int d = 0; d < 3; ++d) {
            R.w[d] = B_::cR(Lc)[d];
            R.d[d] = L.dn[d];
            nmax[d] = Lc.g.N[d] - (L.g.per[d] ? 1 : 0);
        }
        const Range3 cr{1, 1, 1, nmax[0], nmax[1], nmax[2]};
        // a launched coarse level takes its first relaxation from here (the fused
        // levels run their own); nmax spans that level's pressure range
        const bool coarse_launched = g + 1 < g0;
        hipLaunchKernelGGL(k_mg_restrict<T>, grid_for(cr), dim3(BX, BY, 1), 0, s, L.g, Lc.g, R, Lc.c, cr, b[g],
                           B_::C(L), !fp64 && g == 1 ? v : (double *)nullptr, B_::A(Lc), coarse_launched ? x[g + 1] : (T *)nullptr, omega, act);
    }
    if (g0 <= G) {
        MgFusedArgs a;
        fused_layout(m, g0, a);
        hipLaunchKernelGGL(k_mg_fused<T>, dim3(1), dim3(MG_FUSED_THREADS), 0, s, a, B_::tables(m.L[g0]), b[g0], x[g0],
                           omega, act);
    } else {
        relax(G, true, m.n_bottom, true);
        relax(G, false, m.n_bottom);
    }
    for (int g = gl; g >= 1; --g) {
        const MgLevel &L = m.L[g], &Lc = m.L[g + 1];
        LevelW<T> W;
        for (int d = 0; d < 3; ++d) {
            W.w[d] = B_::cI(L)[d];
            W.d[d] = L.dn[d];
        }
        const Range3 cr = full_range(Lc.g);
        hipLaunchKernelGGL(k_mg_interp_cells<T>, grid_for(cr), dim3(BX, BY, 1), 0, s, L.g, Lc.g, W, x[g + 1], x[g],
                           act);
        relax(g, false, m.n_up, false, !fp64 && g == 1);
    }
}

}  // namespace

int mg_first_fused(const MgDev &m) {
    MgFusedArgs a;
    for (int g = 2; g <= m.G; ++g)
        if (fused_layout(m, g, a)) return g;
    return MG_LEVELS_MAX + 1;
}

void launch_mg_vcycle(hipStream_t s, const MgDev &m, double *v, double *z, const int *act) {
    mg_cycle<double>(s, m, v, z, act);
}

void launch_mg_vcycle_f32(hipStream_t s, const MgDev &m, double *v, double *z, const int *act) {
    mg_cycle<float>(s, m, v, z, act);
}

}  // namespace ih
