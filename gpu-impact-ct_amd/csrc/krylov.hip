// Fused Poisson operator and device-controlled BiCGstab (gfx950).
//
// k_apply evaluates product_div_grad (src/mod_laplace.f90:38-197): for each
// direction m the gradient G_m p (src/mod_diff.f90:309-414, zero on the wall
// planes of its component, exchanged with the vel_dir = m rules) followed by
// the divergence D_m (src/mod_diff.f90:52-118), accumulated in the reference's
// order.  Instead of writing the three gradient fields to HBM it keeps them on
// chip: a 16 x 16 column tile marches through a z chunk of up to 32 planes;
// per plane the pressure cross (the tile plus x and y halos of 5) is staged in
// LDS, every G_1 and G_2 value of the tile and its halo is formed once, and G_3
// lives in a per-thread register queue along z.  Every gradient value is
// computed with the reference's operation order, so Ap is bit-identical to the
// three-pass evaluation, while HBM traffic drops to one read of p and one
// write of Ap.
//
// The BiCGstab recurrences (src/mod_solvers.f90:1509-1935; preconditioner 0,
// or the right-preconditioned form with FP32 JOR sweeps or the multigrid V
// cycle as M) run without host round trips: one-block control kernels reduce the partial
// dot products with the fixed tree and update the scalars in device memory; an
// active flag turns the remaining launches of a batch into no-ops once the
// iteration has stopped, so the host checks convergence once per batch.
#include "ih_device.h"
#include "ih_krylov.h"
#include "ih_mg.h"

#include <type_traits>
#include <utility>

namespace ih {

using namespace dev;

namespace {


__device__ inline int wrap_p(const Geo &g, int d, int idx) {
    const int P = g.Np[d] - g.Sp[d] + 1;
    if (idx < g.Sp[d]) return idx + P;
    if (idx > g.Np[d]) return idx - P;
    return idx;
}

// Source index of the pressure-like field along d after exchange(d, 0, .):
// periodic ghosts are copies, wall ghosts (<= 0, > N) are zero.
__device__ inline bool p_src(const Geo &g, int d, int &idx) {
    if (g.per[d]) {
        idx = wrap_p(g, d, idx);
        return true;
    }
    return idx >= 1 && idx <= g.N[d];
}

// Coefficient index of G_d at position idx along d; false where the exchanged
// gradient field is zero (wall planes 0 and N, wall ghosts).
__device__ inline bool g_src(const Geo &g, int d, int &idx) {
    if (g.per[d]) {
        idx = wrap_p(g, d, idx);
        return true;
    }
    return idx >= 1 && idx <= g.N[d] - 1;
}

__device__ inline bool wall_plane(const Geo &g, int e, int idx) { return !g.per[e] && (idx == 1 || idx == g.N[e]); }

// p_src and wall_plane along z with the periodicity of z a compile-time
// constant: the plane loop of k_apply then has no branches on it (they cost
// scalar instructions and branch joins every plane)
template <bool PZ>
__device__ inline bool p_src_z(const Geo &g, int &idx) {
    if (PZ) {
        idx = wrap_p(g, 2, idx);
        return true;
    }
    return idx >= 1 && idx <= g.N[2];
}
template <bool PZ>
__device__ inline bool wall_z(const Geo &g, int idx) {
    return !PZ && (idx == 1 || idx == g.N[2]);
}

// dot modes of k_apply
enum { DOT_NONE = 0, DOT_W = 1, DOT_SELF = 2, DOT_PAIR = 3 };

// Two forms of the operator on a 16 x 16 column tile marching through a z chunk.
//
// Teams (apply_teams): two teams of 256 threads, one thread of each team per
// (x, y) column:
//   team 0 stages the halo of the pressure cross and forms the G_1 and G_2 values
//   of the tile and its halo from the staged plane;
//   team 1 stages the tile's own pressures, keeps p and G_3 of its column in
//   register queues along z, and forms the divergence from the gradient tiles.
// Cross and gradient tiles are double buffered: between two barriers team 0 forms
// the gradients of plane k while team 1 forms the divergence of plane k-1, so a
// plane costs one barrier and each team about half of its instructions.
//
// Column (apply_column): one thread per column does all of a plane.
//
// What bounds them: where the tiles do not fill the compute units (65^3 has 75) the
// chain of one plane, barrier to barrier, which the teams halve; beyond two tiles a
// compute unit the waits of its wavefronts, with the vector ALU 34 to 40 % and LDS 33 to
// 36 % busy at 257x129x129 (column form), and there two teams (8 wavefronts, two
// blocks a compute unit) gain nothing over three blocks of 4 wavefronts.  Operator
// with <Ap, w>, teams against column: 14.0 / 20.5 us at 33x17x17, 17.3 / 25.7 at
// 65^3, 28.8 / 36.7 at 193x97x97; a whole BiCGstab iteration 108.7 / 122.2 us at
// 193x97x97 (364 tiles), 177.8 / 177.3 at 257x129x129 (765), 603.5 / 596.7 at
// 385x193x193 (2275): teams up to two tiles a compute unit, column beyond.
// Measured and not taken: segments of four points a thread in each direction in
// turn with all coefficients scalar (9/4 gradients a point, bound by VALU: 48 us
// at 257x129x129 against 45); the teams at 80 VGPRs for three blocks (spills).
static int64_t apply_team_tiles(int cus) { return 2 * (int64_t)cus; }
constexpr int APPLY_THREADS = 2 * RED_TX * RED_TY;

// Keeps the compiler to the order written: nothing moves across.
__device__ inline void pin() { __builtin_amdgcn_sched_barrier(0); }

// Loaded values that a loop only reads: waited for here, before the loop.  (With
// their loads possibly still in flight at its head, the first use in the loop
// would wait, every trip, for everything in flight, the prefetches included.)
template <int N>
__device__ inline void arrive(double (&v)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(v[i]));
}

using cdbl = const __attribute__((address_space(4))) double;

// the tables of direction d from position pos on (six taps a position)
__device__ inline cdbl *row6(const double *t, int pos) { return (cdbl *)(t + 6 * (pos + COEF6_LEAD)); }

// DM = DOT_W accumulates <Ap, w>, DOT_SELF <p, Ap> and <Ap, Ap>, DOT_PAIR
// <w, Ap> and <Ap, Ap>, per column in plane order over the planes kc0..kc1 (a
// reduction chunk), then over the tile with the fixed tree into entry pi.
// The block functions of one tile serve the single-case and the batched kernels, and
// both forms give the same bits, so a batched case is bit-identical to its own launch.
template <int DM, bool PZ>
__device__ inline void apply_teams(const Geo &g, const Coef &c, const Range3 &r, int bx, int by, int kc0, int kc1,
                                   int64_t pi, const double *__restrict__ src, double *__restrict__ dst,
                                   const double *__restrict__ w, double *part1, double *part2) {
    constexpr int TX = RED_TX, TY = RED_TY, NT = TX * TY;
    constexpr int PW = TX + 10, PH = TY + 10, PS = PW * PH;
    constexpr int NHX = 10 * TY, NH = NHX + 10 * TX;  // halo positions of a plane
    constexpr int NG1X = 5 * TY, NG2X = 5 * TX;
    static_assert(NG1X + NG2X <= NT && NH - NT == 64 && NT == 256, "one halo gradient per thread, the last 64 halo loads");
    constexpr int G1S = TX + 5;                  // row stride of the G_1 tile
    constexpr int OG2 = TY * G1S;                // offset of the G_2 tile
    constexpr int GS = OG2 + (TY + 5) * TX;
    __shared__ double sP[2][PS];
    __shared__ double sG[2][GS + 1];
    __shared__ double sm[8];

    const int tx = threadIdx.x, ty = threadIdx.y;
    const int tid = tx + TX * ty;
    const int team = __builtin_amdgcn_readfirstlane((int)threadIdx.z);
    const int x0 = r.lo0 + bx * TX, y0 = r.lo1 + by * TY;
    const int x = x0 + tx, y = y0 + ty;
    const int xe = r.lo0 + r.n0 - 1, ye = r.lo1 + r.n1 - 1;
    const int64_t pxy = g.pxy;
    // A load outside the field reads some element of its plane instead and its
    // value is replaced by zero where it is used, planes later (a select at the load
    // would make the wave wait for it at once).  Bases are uniform, offsets 32-bit.
    const double *hb = src + gidx(g, -3, -3, 0);
    double acc1 = 0.0, acc2 = 0.0;

    if (team == 0) {
        const int c0 = g.cst[0], c1 = g.cst[1];
        const int b1 = (ty + 5) * PW + tx, w1 = ty * G1S + tx;     // G_1 at x0-3+tx, row ty
        const int b2 = ty * PW + tx + 5, w2 = OG2 + ty * TX + tx;  // G_2 at y0-3+ty, column tx
        int p1 = x0 - 3 + tx;
        const bool v1 = p1 <= xe + 2 && g_src(g, 0, p1) && !wall_plane(g, 1, y);
        int p2 = y0 - 3 + ty;
        const bool v2 = p2 <= ye + 2 && g_src(g, 1, p2) && !wall_plane(g, 0, x);
        double cg1[6], cg2[6];
#pragma unroll
        for (int s = 0; s < 6; ++s) {
            cg1[s] = v1 ? c.G[0][s * c0 + p1] : 0.0;
            cg2[s] = v2 ? c.G[1][s * c1 + p2] : 0.0;
        }
        arrive(cg1);
        arrive(cg2);
        // position e of the plane's halo: its place in the cross and in the field
        auto halo_at = [&](int e, int &slot, unsigned &off) -> bool {
            int hx, hy;
            if (e < NHX) {
                const int row = e / 10, cc = e % 10;
                const int col = cc < 5 ? cc : TX + cc;
                hx = x0 - 5 + col;
                hy = y0 + row;
                slot = (row + 5) * PW + col;
            } else {
                const int rr = (e - NHX) / TX, col = (e - NHX) % TX;
                const int row = rr < 5 ? rr : TY + rr;
                hx = x0 + col;
                hy = y0 - 5 + row;
                slot = row * PW + col + 5;
            }
            const bool v = hx <= xe + 5 && hy <= ye + 5 && p_src(g, 0, hx) && p_src(g, 1, hy);
            off = v ? (unsigned)(gidx(g, hx, hy, 0) - gidx(g, -3, -3, 0)) : 0u;
            return v;
        };
        // Three wavefronts form a halo gradient each thread (the last 32 threads of
        // the third none), the fourth loads the 64 halo positions left over instead:
        // a loop of its own for each, so that neither holds the other's registers.
        auto march = [&](auto job_) {
            constexpr bool JOB = decltype(job_)::value;
            constexpr int NL = JOB ? 1 : 2;
            unsigned hoff[NL];
            int hslot[NL];
            bool hval[NL];
            hval[0] = halo_at(tid, hslot[0], hoff[0]);
            if constexpr (!JOB) hval[1] = halo_at(NT + (tid & 63), hslot[1], hoff[1]);
            auto load_halo = [&](int kk, double (&hv)[NL]) {
                const double *b = hb + (int64_t)(kk <= kc1 ? kk : kc1) * pxy;  // planes past the chunk are not staged
#pragma unroll
                for (int h = 0; h < NL; ++h) hv[h] = b[hoff[h]];
            };
            auto stage_halo = [&](double *P, const double (&hv)[NL]) {
#pragma unroll
                for (int h = 0; h < NL; ++h) P[hslot[h]] = hval[h] ? hv[h] : 0.0;
            };
            // halo gradient: LDS base, stride, destination and coefficients
            double cgx[6];
            int bxj = 0, sxj = 1, wxj = GS;  // GS: a slot past the tiles for the threads without one
            bool vx = false;
            if constexpr (JOB) {
                const double *cx = c.G[0];
                int cix = 0, cstx = c0;
                if (tid < NG2X) {
                    const int c2x = tid % TX, v2r = TY + tid / TX;
                    int py_ = y0 - 3 + v2r;
                    vx = py_ <= ye + 2 && g_src(g, 1, py_) && !wall_plane(g, 0, x0 + c2x);
                    cx = c.G[1];
                    cix = py_;
                    cstx = c1;
                    bxj = v2r * PW + c2x + 5;
                    sxj = PW;
                    wxj = OG2 + v2r * TX + c2x;
                } else if (tid < NG2X + NG1X) {
                    const int e1 = tid - NG2X;
                    const int r1x = e1 / 5, u1x = TX + e1 % 5;
                    int px_ = x0 - 3 + u1x;
                    vx = px_ <= xe + 2 && g_src(g, 0, px_) && !wall_plane(g, 1, y0 + r1x);
                    cix = px_;
                    bxj = (r1x + 5) * PW + u1x;
                    wxj = r1x * G1S + u1x;
                }
#pragma unroll
                for (int s = 0; s < 6; ++s) cgx[s] = vx ? cx[s * cstx + cix] : 0.0;
                arrive(cgx);
            }
            double hvA[NL], hvB[NL];
            load_halo(kc0, hvA);
            pin();
            load_halo(kc0 + 1, hvB);
            // the gradients of plane k, then the halo of plane k+1 and the load of plane k+2's
            auto body = [&](int k, int buf, double (&hv)[NL], double (&hnext)[NL]) {
                __syncthreads();
                load_halo(k + 2, hv);
                const bool zk = wall_z<PZ>(g, k);
                const double *P = sP[buf];
                double *G = sG[buf];
                double pa[6], pb[6], pe[6];
#pragma unroll
                for (int s = 0; s < 6; ++s) pa[s] = P[b1 + s];
#pragma unroll
                for (int s = 0; s < 6; ++s) pb[s] = P[b2 + s * PW];
                if constexpr (JOB) {
#pragma unroll
                    for (int s = 0; s < 6; ++s) pe[s] = P[bxj + s * sxj];
                }
                pin();
                double a = cg1[0] * pa[0], b = cg2[0] * pb[0], e = JOB ? cgx[0] * pe[0] : 0.0;
#pragma unroll
                for (int s = 1; s < 6; ++s) {
                    a = a + cg1[s] * pa[s];
                    b = b + cg2[s] * pb[s];
                    if (JOB) e = e + cgx[s] * pe[s];
                }
                G[w1] = (v1 && !zk) ? a : 0.0;
                G[w2] = (v2 && !zk) ? b : 0.0;
                if constexpr (JOB) G[wxj] = (vx && !zk) ? e : 0.0;
                stage_halo(sP[buf ^ 1], hnext);  // past the chunk: written and not read
            };
            stage_halo(sP[0], hvA);
            for (int k = kc0;;) {
                body(k, 0, hvA, hvB);
                if (++k > kc1) break;
                body(k, 1, hvB, hvA);
                if (++k > kc1) break;
            }
        };
        if (__builtin_amdgcn_readfirstlane(tid >> 6) < 3)
            march(std::true_type{});
        else
            march(std::false_type{});
        __syncthreads();
    } else {
        const bool own = (x <= xe) && (y <= ye);
        int xs = x, ys = y;
        const bool vcol = x <= xe + 5 && y <= ye + 5 && p_src(g, 0, xs) && p_src(g, 1, ys);
        const unsigned colo = vcol ? (unsigned)(gidx(g, xs, ys, 0) - gidx(g, -3, -3, 0)) : 0u;
        const unsigned selfo = own ? (unsigned)(gidx(g, x, y, 0) - gidx(g, -3, -3, 0)) : 0u;
        double *const db = dst + gidx(g, -3, -3, 0);
        const double *const wb = DM == DOT_W || DM == DOT_PAIR ? w + gidx(g, -3, -3, 0) : nullptr;
        const bool g3on = own && !(wall_plane(g, 0, x) || wall_plane(g, 1, y));
        const int gz_lo = PZ ? kc0 - 4 : 1, gz_hi = PZ ? kc1 + 4 : g.N[2] - 1;
        // p of the own column at plane kk (at most kc1 + 5), and whether the field has it
        auto col_ok = [&](int &kk) { return p_src_z<PZ>(g, kk); };
        auto load_col = [&](int kk) -> double {
            kk = kk <= kc1 + 5 ? kk : kc1 + 5;
            return hb[(int64_t)(col_ok(kk) ? kk : kc1) * pxy + colo];
        };
        auto load_w = [&](int kk) -> double {
            if (DM != DOT_W && DM != DOT_PAIR) return 0.0;  // w is only a valid pointer in these modes
            return wb[(int64_t)(kk <= kc1 ? kk : kc1) * pxy + selfo];
        };
        // at the divergence of plane k: q = p(k .. k+5), g3 = G_3(k-3 .. k+2)
        const int c0 = g.cst[0], c1 = g.cst[1];
        double q[6], g3[6], cd1[6], cd2[6], pz[11];
#pragma unroll
        for (int s = 0; s < 11; ++s) pz[s] = load_col(kc0 - 5 + s);
#pragma unroll
        for (int s = 0; s < 6; ++s) {
            cd1[s] = own ? c.D[0][s * c0 + x] : 0.0;
            cd2[s] = own ? c.D[1][s * c1 + y] : 0.0;
        }
        {
            cdbl *Gz = row6(c.G6[2], kc0 - 3);
#pragma unroll
            for (int s = 0; s < 11; ++s) {
                int kk = kc0 - 5 + s;
                pz[s] = vcol && col_ok(kk) ? pz[s] : 0.0;
            }
            sP[0][(ty + 5) * PW + tx + 5] = pz[5];
#pragma unroll
            for (int t = 0; t < 6; ++t) {
                double v = Gz[6 * t] * pz[t];
#pragma unroll
                for (int s = 1; s < 6; ++s) v = v + Gz[6 * t + s] * pz[t + s];
                const int kk = kc0 - 3 + t;
                g3[t] = (g3on && kk >= gz_lo && kk <= gz_hi) ? v : 0.0;
            }
#pragma unroll
            for (int s = 0; s < 6; ++s) q[s] = pz[5 + s];
        }
        arrive(cd1);
        arrive(cd2);
        double pA = load_col(kc0 + 6), wA = load_w(kc0);
        pin();
        double pB = load_col(kc0 + 7), wB = load_w(kc0 + 1);
        // the z coefficients of a plane: G_3 at k+3, then D_3 at k
        double cz[12];
        auto load_cz = [&](int k) {
            cdbl *Gz = row6(c.G6[2], k + 3), *Dz = row6(c.D6[2], k);
#pragma unroll
            for (int s = 0; s < 6; ++s) {
                cz[s] = Gz[s];
                cz[6 + s] = Dz[s];
            }
        };
        load_cz(kc0);
        // the divergence of plane k (its gradients are in sG[buf]), staging p of plane k+2
        auto body = [&](int k, int buf, double &pn, double &wv) {
            __syncthreads();
            double G1[6], G2[6];
#pragma unroll
            for (int t = 0; t < 6; ++t) G1[t] = sG[buf][ty * G1S + tx + t];
#pragma unroll
            for (int t = 0; t < 6; ++t) G2[t] = sG[buf][OG2 + (ty + t) * TX + tx];
            sP[buf][(ty + 5) * PW + tx + 5] = q[2];  // past the chunk: written and not read
            pin();
            // what was loaded two planes ago is taken over before this plane's store
            // is issued: a wait for it would then be a wait for the store as well
            const double q0 = q[0], wk = wv;
#pragma unroll
            for (int s = 0; s < 5; ++s) q[s] = q[s + 1];
            int kn = k + 6;
            q[5] = vcol && col_ok(kn) ? pn : 0.0;
            double v = cz[0] * q[0];
#pragma unroll
            for (int s = 1; s < 6; ++s) v = v + cz[s] * q[s];
            pn = load_col(k + 8);
            wv = load_w(k + 2);
            double lap = cd1[0] * G1[0];
#pragma unroll
            for (int t = 1; t < 6; ++t) lap = lap + cd1[t] * G1[t];
#pragma unroll
            for (int t = 0; t < 6; ++t) lap = lap + cd2[t] * G2[t];
#pragma unroll
            for (int t = 0; t < 6; ++t) lap = lap + cz[6 + t] * g3[t];
#pragma unroll
            for (int t = 0; t < 5; ++t) g3[t] = g3[t + 1];
            asm volatile("" : "+v"(v));  // a select, not a branch around the sum
            g3[5] = (g3on && k + 3 >= gz_lo && k + 3 <= gz_hi) ? v : 0.0;
            pin();
            load_cz(k + 1);
            pin();
            if (DM == DOT_W) {
                acc1 = acc1 + (own ? lap * wk : 0.0);
            } else if (DM == DOT_SELF) {
                acc1 = acc1 + (own ? q0 * lap : 0.0);
                acc2 = acc2 + (own ? lap * lap : 0.0);
            } else if (DM == DOT_PAIR) {
                acc1 = acc1 + (own ? wk * lap : 0.0);
                acc2 = acc2 + (own ? lap * lap : 0.0);
            }
            if (own) db[(int64_t)k * pxy + selfo] = lap;
        };
        __syncthreads();  // plane kc0 is staged
        sP[1][(ty + 5) * PW + tx + 5] = q[1];
        // the loop leaves from between its two halves: with a way around the second
        // one the first half's wait for its loads would be a wait for all loads
        for (int k = kc0;;) {
            body(k, 0, pA, wA);
            if (++k > kc1) break;
            body(k, 1, pB, wB);
            if (++k > kc1) break;
        }
    }
    if (DM != DOT_NONE) {
        // the fixed tree over the tile, the partial sums of team 1
        if (team == 1) {
            const double s1 = wave_sum(acc1);
            const double s2 = DM == DOT_W ? 0.0 : wave_sum(acc2);
            if ((tid & 63) == 0) {
                sm[tid >> 6] = s1;
                sm[4 + (tid >> 6)] = s2;
            }
        }
        __syncthreads();
        if (team == 1 && tid == 0) {
            part1[pi] = (sm[0] + sm[1]) + (sm[2] + sm[3]);
            if (DM == DOT_SELF || DM == DOT_PAIR) part2[pi] = (sm[4] + sm[5]) + (sm[6] + sm[7]);
        }
    }
}

// The column form: one thread per (x, y) column.  Pressure cross and gradient
// tiles are double buffered, and the divergence of plane k-1 is formed after the
// gradients of plane k, so each plane costs one barrier.  The halo of plane k+2,
// p(k+7) of the column queue and w(k+1) are loaded while planes k and k+1 are
// computed (the plane loop is unrolled twice so that the two register sets
// alternate).  The gradient coefficients of a thread's positions stay in registers
// for the whole chunk, those in z are scalar loads a plane ahead (from LDS they were
// 13 of a plane's 45 LDS accesses: 600.5 against 596.7 us an iteration at
// 385x193x193, 177.9 against 177.3 at 257x129x129); every thread forms one G_1, one
// G_2 and at most one halo gradient per plane without divergent branches.
// 3 wavefronts per SIMD (at most 168 VGPRs).
template <int DM, bool PZ>
__device__ inline void apply_column(const Geo &g, const Coef &c, const Range3 &r, int bx, int by, int kc0, int kc1,
                                    int64_t pi, const double *__restrict__ src, double *__restrict__ dst,
                                    const double *__restrict__ w, double *part1, double *part2) {
    constexpr int TX = RED_TX, TY = RED_TY;
    constexpr int NT = TX * TY;
    constexpr int PW = TX + 10, PH = TY + 10, PS = PW * PH;
    constexpr int NHX = 10 * TY;
    constexpr int NH = NHX + 10 * TX;
    constexpr int HL = (NH + NT - 1) / NT;
    constexpr int NG1X = 5 * TY, NG2X = 5 * TX;
    static_assert(NG1X + NG2X <= NT, "one extra gradient job per thread at most");
    constexpr int G1S = TX + 5;                 // row stride of the G_1 tile
    constexpr int OG2 = TY * G1S;               // offset of the G_2 tile
    constexpr int GS = OG2 + (TY + 5) * TX + 1; // + one dummy slot
    __shared__ double sP[2][PS];
    __shared__ double sG[2][GS];
    __shared__ double sm[8];

    const int tx = threadIdx.x, ty = threadIdx.y;
    const int tid = tx + TX * ty;
    const int x0 = r.lo0 + bx * TX, y0 = r.lo1 + by * TY;
    const int x = x0 + tx, y = y0 + ty;
    const int xe = r.lo0 + r.n0 - 1, ye = r.lo1 + r.n1 - 1;
    const bool own = (x <= xe) && (y <= ye);
    const int c0 = g.cst[0], c1 = g.cst[1];
    const int64_t pxy = g.pxy;
    // loads outside the field read c.zero, so no value is masked after its load
    // (a select on the loaded value would make the wave wait for it at once)
    const double *zero = c.zero;

    const int64_t hbase = gidx(g, -3, -3, 0);  // a valid element; offsets below are >= 0 from it
    int xs = x, ys = y;
    const bool vcol = x <= xe + 5 && y <= ye + 5 && p_src(g, 0, xs) && p_src(g, 1, ys);
    const int64_t colb = vcol ? gidx(g, xs, ys, 0) : hbase;
    const int64_t selfb = own ? gidx(g, x, y, 0) : hbase;

    int hoff[HL], hslot[HL];
#pragma unroll
    for (int h = 0; h < HL; ++h) {
        const int e = tid + h * NT;
        hoff[h] = -1;
        hslot[h] = PS;  // past the tile: not written
        if (e < NHX) {
            const int row = e / 10, cc = e % 10;
            const int col = cc < 5 ? cc : TX + cc;
            int hx = x0 - 5 + col, hy = y0 + row;
            hslot[h] = (row + 5) * PW + col;
            if (hx <= xe + 5 && hy <= ye + 5 && p_src(g, 0, hx) && p_src(g, 1, hy))
                hoff[h] = (int)(gidx(g, hx, hy, 0) - hbase);
        } else if (e < NH) {
            const int e2 = e - NHX;
            const int rr = e2 / TX, col = e2 % TX;
            const int row = rr < 5 ? rr : TY + rr;
            int hx = x0 + col, hy = y0 - 5 + row;
            hslot[h] = row * PW + col + 5;
            if (hx <= xe + 5 && hy <= ye + 5 && p_src(g, 0, hx) && p_src(g, 1, hy))
                hoff[h] = (int)(gidx(g, hx, hy, 0) - hbase);
        }
    }

    // gradient jobs (LDS base, stride, destination) and coefficients
    double cg1[6], cg2[6], cgx[6], cd1[6], cd2[6];
    bool v1, v2, vx;
    const int b1 = (ty + 5) * PW + tx, w1 = ty * G1S + tx;           // G_1 at x0-3+tx, row ty
    const int b2 = ty * PW + tx + 5, w2 = OG2 + ty * TX + tx;         // G_2 at y0-3+ty, column tx
    int bxj = 0, sxj = 1, wxj = GS - 1;
    {
        int p1 = x0 - 3 + tx;
        v1 = p1 <= xe + 2 && g_src(g, 0, p1) && !wall_plane(g, 1, y);
        int p2 = y0 - 3 + ty;
        v2 = p2 <= ye + 2 && g_src(g, 1, p2) && !wall_plane(g, 0, x);
        const double *cx = c.G[0];
        int cix = 0, cstx = c0;
        vx = false;
        const int e1 = tid - NG2X;
        if (e1 >= 0 && e1 < NG1X) {
            const int r1x = e1 / 5, u1x = TX + e1 % 5;
            int px_ = x0 - 3 + u1x;
            vx = px_ <= xe + 2 && g_src(g, 0, px_) && !wall_plane(g, 1, y0 + r1x);
            cix = px_;
            bxj = (r1x + 5) * PW + u1x;
            sxj = 1;
            wxj = r1x * G1S + u1x;
        } else if (tid < NG2X) {
            const int c2x = tid % TX, v2r = TY + tid / TX;
            int py_ = y0 - 3 + v2r;
            vx = py_ <= ye + 2 && g_src(g, 1, py_) && !wall_plane(g, 0, x0 + c2x);
            cx = c.G[1];
            cix = py_;
            cstx = c1;
            bxj = v2r * PW + c2x + 5;
            sxj = PW;
            wxj = OG2 + v2r * TX + c2x;
        }
#pragma unroll
        for (int s = 0; s < 6; ++s) {
            cg1[s] = v1 ? c.G[0][s * c0 + p1] : 0.0;
            cg2[s] = v2 ? c.G[1][s * c1 + p2] : 0.0;
            cgx[s] = vx ? cx[s * cstx + cix] : 0.0;
            cd1[s] = own ? c.D[0][s * c0 + x] : 0.0;
            cd2[s] = own ? c.D[1][s * c1 + y] : 0.0;
        }
    }
    const bool g3on = own && !(wall_plane(g, 0, x) || wall_plane(g, 1, y));
    const int gz_lo = PZ ? kc0 - 8 : 1, gz_hi = PZ ? kc1 + 8 : g.N[2] - 1;

    // queue at iteration k: q = p(k-1 .. k+4), g3 = G_3(k-4 .. k+1)
    double q[6], g3[6];
    {
        double pz[11];
#pragma unroll
        for (int s = 0; s < 11; ++s) {
            int kk = kc0 - 6 + s;
            const bool v = vcol && p_src_z<PZ>(g, kk);
            pz[s] = *(v ? src + colb + (int64_t)kk * pxy : zero);
        }
        cdbl *Gz = row6(c.G6[2], kc0 - 4);
#pragma unroll
        for (int t = 0; t < 6; ++t) {
            double v = Gz[6 * t] * pz[t];
#pragma unroll
            for (int s = 1; s < 6; ++s) v = v + Gz[6 * t + s] * pz[t + s];
            const int kk = kc0 - 4 + t;
            g3[t] = (g3on && kk >= gz_lo && kk <= gz_hi) ? v : 0.0;
        }
#pragma unroll
        for (int s = 0; s < 6; ++s) q[s] = pz[5 + s];
    }
    auto load_halo = [&](int kk, double (&hv)[HL]) {
        const bool vk = kk <= kc1 && p_src_z<PZ>(g, kk);
#pragma unroll
        for (int h = 0; h < HL; ++h) {
            const bool v = vk && hoff[h] >= 0;
            hv[h] = *(v ? src + hbase + hoff[h] + (int64_t)kk * pxy : zero);
        }
    };
    auto load_col = [&](int kk) -> double {
        const bool v = vcol && kk <= kc1 + 5 && p_src_z<PZ>(g, kk);
        return *(v ? src + colb + (int64_t)kk * pxy : zero);
    };
    auto load_w = [&](int kk) -> double {
        if (DM != DOT_W && DM != DOT_PAIR) return 0.0;  // w is only a valid pointer in these modes
        const bool v = own && kk <= kc1;
        return *(v ? w + selfb + (int64_t)kk * pxy : zero);
    };
    double hvA[HL], hvB[HL];
    load_halo(kc0, hvA);
    load_halo(kc0 + 1, hvB);
    double pA = load_col(kc0 + 5), pB = load_col(kc0 + 6);
    double wA = load_w(kc0), wB = load_w(kc0 + 1);
    double acc1 = 0.0, acc2 = 0.0;
    // z coefficients of plane k's step, scalar operands loaded a plane ahead: G_3 at
    // k+2, D_3 at k-1
    double cz[12];
    auto load_cz = [&](int k) {
        cdbl *Gz = row6(c.G6[2], k + 2), *Dz = row6(c.D6[2], k - 1);
#pragma unroll
        for (int s = 0; s < 6; ++s) {
            cz[s] = Gz[s];
            cz[6 + s] = Dz[s];
        }
    };
    load_cz(kc0);

    auto divergence = [&](int k, const double *G, double wv) {
        // plane k from the gradient tile G, g3 = G_3(k-3 .. k+2), q[0] = p(k)
        double lap = cd1[0] * G[ty * G1S + tx];
#pragma unroll
        for (int t = 1; t < 6; ++t) lap = lap + cd1[t] * G[ty * G1S + tx + t];
#pragma unroll
        for (int t = 0; t < 6; ++t) lap = lap + cd2[t] * G[OG2 + (ty + t) * TX + tx];
#pragma unroll
        for (int t = 0; t < 6; ++t) lap = lap + cz[6 + t] * g3[t];
        if (own) dst[selfb + (int64_t)k * pxy] = lap;
        if (DM == DOT_W) {
            acc1 = acc1 + (own ? lap * wv : 0.0);
        } else if (DM == DOT_SELF) {
            acc1 = acc1 + (own ? q[0] * lap : 0.0);
            acc2 = acc2 + (own ? lap * lap : 0.0);
        } else if (DM == DOT_PAIR) {
            acc1 = acc1 + (own ? wv * lap : 0.0);
            acc2 = acc2 + (own ? lap * lap : 0.0);
        }
    };
    auto body = [&](int k, int buf, double (&hv)[HL], double &pn, double &wprev, double &wcur) {
        // stage plane k
        double *P = sP[buf];
        P[(ty + 5) * PW + tx + 5] = q[1];
#pragma unroll
        for (int h = 0; h < HL; ++h)
            if (hslot[h] < PS) P[hslot[h]] = hv[h];
        __syncthreads();
        load_halo(k + 2, hv);
        // gradients of plane k
        const bool zk = wall_z<PZ>(g, k);
        double *G = sG[buf];
        {
            double a = cg1[0] * P[b1];
#pragma unroll
            for (int s = 1; s < 6; ++s) a = a + cg1[s] * P[b1 + s];
            G[w1] = (v1 && !zk) ? a : 0.0;
            double b = cg2[0] * P[b2];
#pragma unroll
            for (int s = 1; s < 6; ++s) b = b + cg2[s] * P[b2 + s * PW];
            G[w2] = (v2 && !zk) ? b : 0.0;
            if (tid < NG1X + NG2X) {  // halo gradient jobs; the last wavefront has none
                double e = cgx[0] * P[bxj];
#pragma unroll
                for (int s = 1; s < 6; ++s) e = e + cgx[s] * P[bxj + s * sxj];
                G[wxj] = (vx && !zk) ? e : 0.0;
            }
        }
        // divergence of plane k-1 (its gradient tile is the other buffer)
        if (k > kc0) {
            divergence(k - 1, sG[buf ^ 1], wprev);
            wprev = load_w(k + 1);
        }
        // advance: q = p(k .. k+5), g3 = G_3(k-3 .. k+2)
#pragma unroll
        for (int s = 0; s < 5; ++s) q[s] = q[s + 1];
        q[5] = pn;
        pn = load_col(k + 7);
#pragma unroll
        for (int t = 0; t < 5; ++t) g3[t] = g3[t + 1];
        double v = cz[0] * q[0];
#pragma unroll
        for (int s = 1; s < 6; ++s) v = v + cz[s] * q[s];
        g3[5] = (g3on && k + 2 >= gz_lo && k + 2 <= gz_hi) ? v : 0.0;
        pin();
        load_cz(k + 1);
        pin();
        (void)wcur;
    };
    // w(k-1) is consumed in iteration k: the A set serves even offsets k-kc0, the B set odd ones
    for (int k = kc0; k <= kc1; k += 2) {
        body(k, 0, hvA, pA, wB, wA);
        if (k + 1 <= kc1) body(k + 1, 1, hvB, pB, wA, wB);
    }
    __syncthreads();
    {
        const int n = kc1 - kc0 + 1;
        const int buf = (n - 1) & 1;
        divergence(kc1, sG[buf], buf == 0 ? wA : wB);
    }
    if (DM != DOT_NONE) {
        const double s1 = block_sum(acc1, sm);
        __syncthreads();
        if (tid == 0) part1[pi] = s1;
        if (DM == DOT_SELF || DM == DOT_PAIR) {
            const double s2 = block_sum(acc2, sm + 4);
            if (tid == 0) part2[pi] = s2;
        }
    }
}

template <bool TEAMS, int DM, bool PZ>
__device__ inline void apply_block(const Geo &g, const Coef &c, const Range3 &r, int bx, int by, int bz, int nbz,
                                   int64_t pi, const double *src, double *dst, const double *w, double *part1,
                                   double *part2) {
    int kc0, kc1;
    red_chunk(r, bz, nbz, kc0, kc1);
    if constexpr (TEAMS)
        apply_teams<DM, PZ>(g, c, r, bx, by, kc0, kc1, pi, src, dst, w, part1, part2);
    else
        apply_column<DM, PZ>(g, c, r, bx, by, kc0, kc1, pi, src, dst, w, part1, part2);
}

constexpr int apply_threads(bool teams) { return teams ? APPLY_THREADS : RED_THREADS; }
constexpr int apply_waves(bool teams) { return teams ? 4 : 3; }  // wavefronts per SIMD

template <bool TEAMS, int DM, bool PZ>
__global__ __launch_bounds__(apply_threads(TEAMS), apply_waves(TEAMS)) void k_apply(
    Geo g, Coef c, Range3 r, int nbx, int nby, int nbz, const double *__restrict__ src, double *__restrict__ dst,
    const double *__restrict__ w, double *part1, double *part2, const int *active) {
    if (active && !*active) return;
    int bx, by, bz;
    if (!xcd_tile(nbx, nby, nbz, bx, by, bz)) return;
    const int64_t pi = (int64_t)bx + (int64_t)nbx * ((int64_t)by + (int64_t)nby * bz);
    apply_block<TEAMS, DM, PZ>(g, c, r, bx, by, bz, nbz, pi, src, dst, w, part1, part2);
}

// ---------------------------------------------------------------------------
// BiCGstab vector kernels (reduction tiles, so that fused partials follow
// the fixed tree) and the one-block control kernels.
// ---------------------------------------------------------------------------
// The reduction-tile kernels below are block functions of tile (bx, by, bz)
// out of nbz z chunks, partial index pi = bx + nbx*(by + nby*bz), run by the
// single-case kernels (tile = block index) and by the batched ones.
__device__ inline void init_rr_block(const Geo &g, const Range3 &r, int bx, int by, int bz, int nbz, int64_t pi,
                                     const double *bb, double *rr, double *rh, double *pmax, double *pdot) {
    __shared__ double sm[8];
    const int i = r.lo0 + bx * RED_TX + (int)threadIdx.x;
    const int j = r.lo1 + by * RED_TY + (int)threadIdx.y;
    double m = 0.0, d = 0.0;
    if (i < r.lo0 + r.n0 && j < r.lo1 + r.n1) {
        int kc0, kc1;
        red_chunk(r, bz, nbz, kc0, kc1);
        for (int k = kc0; k <= kc1; ++k) {
            const int64_t x = gidx(g, i, j, k);
            const double v = bb[x] - rr[x];
            rr[x] = v;
            rh[x] = v;
            const double a = fabs(v);
            m = max_nan(a, m);
            d = d + v * v;
        }
    }
    const double bm = block_max(m, sm);
    __syncthreads();
    const double bs = block_sum(d, sm + 4);
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        pmax[pi] = bm;
        pdot[pi] = bs;
    }
}

__global__ __launch_bounds__(256) void k_init_rr(Geo g, Range3 r, const double *bb, double *rr, double *rh,
                                                 double *pmax, double *pdot) {
    init_rr_block(g, r, (int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, (int)gridDim.z, part_index(), bb, rr, rh,
                  pmax, pdot);
}

// The first FP32 preconditioner sweep at one point, from the zero start: b32 =
// (float) v and e = the JOR update with every neighbour 0, in the operands and
// order of the sweep kernels (jor_f32_first_block), so the values are the same
// bits.  The update kernels that produce v call it when the preconditioner is
// FP32 sweeps (FIRST), which saves the first sweep's own pass over v.
struct FirstSweep {
    const float *g1, *g2, *g3;
    float omega;
    float *b32, *e;
};

__device__ inline void first_sweep_point(const Geo &g, const FirstSweep &f, int i, int j, int k, int64_t x,
                                         double v) {
    const int c0 = g.cst[0], c1 = g.cst[1], c2 = g.cst[2];
    const float z = 0.0f;
    const float bv = (float)v;
    float s = bv;
    s = s - f.g1[0 * c0 + i] * z;
    s = s - f.g1[2 * c0 + i] * z;
    s = s - f.g2[0 * c1 + j] * z;
    s = s - f.g2[2 * c1 + j] * z;
    s = s - f.g3[0 * c2 + k] * z;
    s = s - f.g3[2 * c2 + k] * z;
    const float diag = (f.g1[1 * c0 + i] + f.g2[1 * c1 + j]) + f.g3[1 * c2 + k];
    f.b32[x] = bv;
    f.e[x] = f.omega * s / diag + (1.0f - f.omega) * z;
}

template <bool FIRST>
__global__ void k_p_update(Geo g, Range3 r, const double *rr, double *pk, const double *Ap, const double *sc,
                           const int *fl, FirstSweep fs) {
    if (!fl[KF_ACTIVE]) return;
    IH_POINT(r);
    const int64_t x = gidx(g, i, j, k);
    double p;
    if (fl[KF_MODE])
        p = rr[x] + sc[KS_BETA] * pk[x] + sc[KS_OM2] * Ap[x];
    else
        p = rr[x];
    pk[x] = p;
    if (FIRST) first_sweep_point(g, fs, i, j, k, x, p);
}

__device__ inline double reduce_sum_parts(const double *part, int64_t nb, double *sm) {
    const int tid = threadIdx.x + threadIdx.y * blockDim.x;
    return block_sum(thread_sum_parts(part, nb, tid), sm);
}

__device__ inline double reduce_max_parts(const double *part, int64_t nb, double *sm) {
    const int tid = threadIdx.x + threadIdx.y * blockDim.x;
    return block_max(thread_max_parts(part, nb, tid), sm);
}

// status_iteration + the scalar part of the iteration head (mod_solvers.f90:1589-1666)
__device__ inline void ctl_head_tail(double *sc, int *fl, int counter) {
    if (counter >= 2) {
        if (sc[KS_OMEGA] == 0.0 || sc[KS_RHR_PREV] == 0.0) {
            fl[KF_EXIT] = 2;
            fl[KF_ACTIVE] = 0;
            fl[KF_DONE] = 1;
            return;
        }
        const double beta = (sc[KS_ALPHA] / sc[KS_OMEGA]) * (sc[KS_RHR] / sc[KS_RHR_PREV]);
        const double om2 = -beta * sc[KS_OMEGA];
        sc[KS_BETA] = beta;
        sc[KS_OM2] = om2;
        sc[KS_OMEGA] = om2;
        fl[KF_MODE] = 1;
    } else {
        fl[KF_MODE] = 0;
    }
}

// The head of an iteration: stop test, counter, rho rotation and beta.  It runs
// in the same thread right after the scalars it reads were written, at the end
// of k_ctl_setup and of k_ctl_end (the head of the next iteration), so no
// launch of its own is needed.
__device__ inline void ctl_begin(double *sc, int *fl) {
    if (!fl[KF_ACTIVE]) return;
    const double norm = sc[KS_NORM];
    int counter = fl[KF_COUNTER];
    bool ex = norm < sc[KS_EPS];
    if (!ex && counter == fl[KF_NMAX]) {
        ex = true;
        fl[KF_EXIT] = 1;
    }
    if (counter < 1 && norm != 0.0) ex = false;
    if (!(norm == norm) || norm > 1.0e300) {  // a non-finite residual: stop as a breakdown
        ex = true;
        fl[KF_EXIT] = 2;
    }
    if (ex) {
        fl[KF_ACTIVE] = 0;
        fl[KF_DONE] = 1;
        return;
    }
    counter = counter + 1;
    fl[KF_COUNTER] = counter;
    sc[KS_RHR_PREV] = sc[KS_RHR];
    sc[KS_RHR] = sc[KS_RHR_NEXT];
    if (fabs(sc[KS_RHR]) == 0.0) {
        // new reference vector needed: the host resets rh and resumes
        fl[KF_RESET] = 1;
        fl[KF_ACTIVE] = 0;
        return;
    }
    ctl_head_tail(sc, fl, counter);
}

// after the initial residual: norm, rhr_next; reset the iteration state
__global__ __launch_bounds__(256) void k_ctl_setup(const double *pmax, const double *pdot, int64_t nb, double *sc,
                                                   int *fl, double eps, int nmax) {
    __shared__ double sm[8];
    const double nm = reduce_max_parts(pmax, nb, sm);
    __syncthreads();
    const double dt = reduce_sum_parts(pdot, nb, sm + 4);
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        sc[KS_NORM] = nm;
        sc[KS_NORM0] = nm;
        sc[KS_RHR_NEXT] = dt;
        sc[KS_RHR] = 0.0;
        sc[KS_ALPHA] = 0.0;
        sc[KS_OMEGA] = 0.0;
        sc[KS_EPS] = eps;
        fl[KF_ACTIVE] = 1;
        fl[KF_COUNTER] = 0;
        fl[KF_NMAX] = nmax;
        fl[KF_EXIT] = 0;
        fl[KF_RESET] = 0;
        fl[KF_MODE] = 0;
        fl[KF_DONE] = 0;
        ctl_begin(sc, fl);  // the head of the first iteration
    }
}

__global__ void k_ctl_resume(double *sc, int *fl) {
    fl[KF_RESET] = 0;
    fl[KF_ACTIVE] = 1;
    ctl_head_tail(sc, fl, fl[KF_COUNTER]);
}

// Every workgroup of the two update kernels below first reduces the partials
// of the operator kernel before it (the same fixed tree as the single-workgroup
// control kernels), so the scalar step of BiCGstab needs no launch of its own.
// Workgroup 0 publishes the scalar, or the breakdown flags, in which case no
// workgroup updates.  The active flag is read once per workgroup: workgroup 0
// may clear it while later workgroups start, and either value they see leads
// to the same decision.
__device__ inline bool wg_active(const int *fl, int *s_go) {
    if (threadIdx.x == 0 && threadIdx.y == 0 && threadIdx.z == 0) *s_go = fl[KF_ACTIVE];
    __syncthreads();
    return *s_go != 0;
}

__device__ inline void breakdown(int *fl) {
    fl[KF_EXIT] = 2;
    fl[KF_ACTIVE] = 0;
    fl[KF_DONE] = 1;
}

// The planes of a reduction chunk (at most 32) on UPD_ZG groups of 256 threads, at
// most UPD_KP planes each: all of a thread's loads are in flight before the scalar
// of the step is reduced from the operator's partials.
constexpr int UPD_ZG = 4, UPD_KP = RED_KC / UPD_ZG;

// the planes k0 .. k0 + cnt - 1 of group zg out of the chunk kc0..kc1
__device__ inline void split_planes(int zg, int kc0, int kc1, int &k0, int &cnt) {
    const int per = (kc1 - kc0 + UPD_ZG) / UPD_ZG;
    k0 = kc0 + zg * per;
    cnt = kc1 - k0 + 1 < per ? kc1 - k0 + 1 : per;
}

// the sum of the partials by the 256 threads of a group, as wave sums sm[0..3]
__device__ inline void split_sum_parts(const double *part, int64_t nb, int tid, double *sm) {
    const double v = wave_sum(thread_sum_parts(part, nb, tid));
    if ((tid & 63) == 0) sm[tid >> 6] = v;
}

// alpha = rhr/<rh, Ap> (a vanishing <rh, Ap> is a breakdown), then rr = rr - alpha*Ap
// (src/mod_solvers.f90:1709-1740).  Bound by HBM from 257x129x129 on, below by latency:
// a thread that walks its chunk's planes one by one waits once a plane.  Four groups
// of planes against one: 5.4 -> 3.7 us at 33x17x17, 6.6 -> 4.4 at 65^3, 12.3 -> 8.1 at
// 193x97x97, 18.9 -> 18.0 at 257x129x129 (5.7 TB/s), 58.2 -> 54.6 at 385x193x193.
// ASK: the flag is asked before anything is loaded, so an iteration enqueued past the stop
// (up to seven a solve, and a batch's stopped cases) moves nothing; else it is read with
// the loads, which is the faster form of an iteration that runs (KrylovPtrs::ask).
template <bool FIRST, bool ASK>
__device__ inline void s_update_block(const Geo &g, const Range3 &r, int bx, int by, int bz, int nbz, int64_t pi,
                                      double *rr, const double *Ap, const double *part, int64_t nb, double *sc,
                                      int *fl, const FirstSweep &fs) {
    __shared__ double sm[4];
    __shared__ int s_go;
    const int tid = (int)(threadIdx.x + RED_TX * threadIdx.y);
    const int zg = __builtin_amdgcn_readfirstlane((int)threadIdx.z);
    if (ASK && !wg_active(fl, &s_go)) return;
    if (!ASK && tid == 0 && zg == 0) s_go = fl[KF_ACTIVE];
    const int i = r.lo0 + bx * RED_TX + (int)threadIdx.x;
    const int j = r.lo1 + by * RED_TY + (int)threadIdx.y;
    const bool own = i < r.lo0 + r.n0 && j < r.lo1 + r.n1;
    int kc0, kc1;
    red_chunk(r, bz, nbz, kc0, kc1);
    int k0, cnt;
    split_planes(zg, kc0, kc1, k0, cnt);
    const int64_t x0 = gidx(g, own ? i : r.lo0, own ? j : r.lo1, 0);
    double v[UPD_KP], a[UPD_KP];
#pragma unroll
    for (int u = 0; u < UPD_KP; ++u) {
        v[u] = a[u] = 0.0;
        if (u < cnt) {
            const int64_t x = x0 + (int64_t)(k0 + u) * g.pxy;
            v[u] = rr[x];
            a[u] = Ap[x];
        }
    }
    if (zg == 0) split_sum_parts(part, nb, tid, sm);
    __syncthreads();
    if (!s_go) return;
    const double rhAp = (sm[0] + sm[1]) + (sm[2] + sm[3]);
    const bool ok = !(fabs(rhAp) == 0.0);
    const double alpha = ok ? sc[KS_RHR] / rhAp : 0.0;
    if (tid == 0 && zg == 0 && pi == 0) {
        if (ok)
            sc[KS_ALPHA] = alpha;
        else
            breakdown(fl);
    }
    if (!ok || !own) return;
#pragma unroll
    for (int u = 0; u < UPD_KP; ++u) {
        if (u >= cnt) break;
        const int k = k0 + u;
        const int64_t x = x0 + (int64_t)k * g.pxy;
        const double w = v[u] - alpha * a[u];
        rr[x] = w;
        if (FIRST) first_sweep_point(g, fs, i, j, k, x, w);
    }
}

template <bool FIRST, bool ASK>
__global__ __launch_bounds__(RED_THREADS *UPD_ZG) void k_s_update_alpha(Geo g, Range3 r, double *rr, const double *Ap,
                                                                        const double *part, int64_t nb, double *sc,
                                                                        int *fl, FirstSweep fs) {
    s_update_block<FIRST, ASK>(g, r, (int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, (int)gridDim.z, part_index(),
                               rr, Ap, part, nb, sc, fl, fs);
}

// omega = <r, Ar>/<Ar, Ar> (a vanishing <Ar, Ar> is a breakdown), then
// phi = phi + omega*ra + alpha*pa; rr = rr - omega*Ar, with the max-norm and
// <rr, rh> partials of the new residual in pmax/pdot (ra = rr, pa = pk without
// a preconditioner; ra = z2, pa = z1 with one, src/mod_solvers.f90:1782-1797, 1855-1899).
// pmax/pdot must not alias p1/p2, which other workgroups may still be reducing.
__device__ inline void x_update_block(const Geo &g, const Range3 &r, int bx, int by, int bz, int nbz, int64_t pi,
                                      double *phi, double *rr, const double *ra, const double *pa, const double *Ar,
                                      const double *rh, const double *p1, const double *p2, int64_t nb, double *sc,
                                      int *fl, double *pmax, double *pdot) {
    __shared__ double sm[8];
    __shared__ double s_om;
    __shared__ int s_go;
    if (!wg_active(fl, &s_go)) return;
    double t1, t2;
    thread_sum_parts2(p1, p2, nb, (int)(threadIdx.x + threadIdx.y * blockDim.x), t1, t2);
    const double rAr = block_sum(t1, sm);
    __syncthreads();
    const double ArAr = block_sum(t2, sm + 4);
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        const bool ok = !(fabs(ArAr) == 0.0);
        const double om = ok ? rAr / ArAr : 0.0;
        s_om = om;
        s_go = ok;
        if (pi == 0) {
            if (ok)
                sc[KS_OMEGA] = om;
            else
                breakdown(fl);
        }
    }
    __syncthreads();
    if (!s_go) return;
    const double om = s_om, alpha = sc[KS_ALPHA];
    const int i = r.lo0 + bx * RED_TX + (int)threadIdx.x;
    const int j = r.lo1 + by * RED_TY + (int)threadIdx.y;
    double m = 0.0, d = 0.0;
    if (i < r.lo0 + r.n0 && j < r.lo1 + r.n1) {
        int kc0, kc1;
        red_chunk(r, bz, nbz, kc0, kc1);
        // two register sets: the loads of plane k+1 are in flight while plane k is
        // updated (a thread's planes are distinct elements, so no store changes a
        // value loaded for a later plane; ra is rr itself without a preconditioner,
        // and both then read the old r).  No memory access sits on a branch, so the
        // waits can count exactly: past the chunk, the loads read its last plane
        // again, and the one update past it (odd chunk lengths) rewrites that plane
        // from the values loaded before its first update, the same bits again,
        // while the norm and the dot skip it.
        const int64_t x0 = gidx(g, i, j, kc0);
        const int64_t pxy = g.pxy;
        struct In {
            double ph, ra, pa, rr, Ar, rh;
        };
        In A, B;
        auto ld = [&](int k, In &v) {
            const int64_t x = x0 + (int64_t)((k < kc1 ? k : kc1) - kc0) * pxy;
            v.ph = phi[x];
            v.ra = ra[x];
            v.pa = pa[x];
            v.rr = rr[x];
            v.Ar = Ar[x];
            v.rh = rh[x];
        };
        auto up = [&](int k, const In &v) {
            const int64_t x = x0 + (int64_t)((k < kc1 ? k : kc1) - kc0) * pxy;
            phi[x] = v.ph + om * v.ra + alpha * v.pa;
            const double w = v.rr - om * v.Ar;
            rr[x] = w;
            const double a = fabs(w);
            const bool in = k <= kc1;
            m = in ? max_nan(a, m) : m;
            d = in ? d + w * v.rh : d;
        };
        if (kc0 <= kc1) ld(kc0, A);
        for (int k = kc0; k <= kc1; k += 2) {
            ld(k + 1, B);
            up(k, A);
            ld(k + 2, A);
            up(k + 1, B);
        }
    }
    const double bm = block_max(m, sm);
    __syncthreads();
    const double bs = block_sum(d, sm + 4);
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        pmax[pi] = bm;
        pdot[pi] = bs;
    }
}

__global__ __launch_bounds__(256) void k_x_update_omega(Geo g, Range3 r, double *phi, double *rr, const double *ra,
                                                        const double *pa, const double *Ar, const double *rh,
                                                        const double *p1, const double *p2, int64_t nb, double *sc,
                                                        int *fl, double *pmax, double *pdot) {
    x_update_block(g, r, (int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, (int)gridDim.z, part_index(), phi, rr,
                   ra, pa, Ar, rh, p1, p2, nb, sc, fl, pmax, pdot);
}

// The same update with the chunk's planes on UPD_ZG groups.  The chunk's sum is still
// formed in plane order: the groups take turns, each adding its products to what the
// group below passes on, so the partials are the same bits.  PRE: ra is another
// field than rr (the preconditioned direction); ASK as in the s update.  8.3 -> 7.1 us
// at 33x17x17, 11.0 -> 9.2 at 65^3, 16.9 -> 11.7 at 118x71x91, 17.0 -> 14.5 at 129x97x97.
template <bool PRE, bool ASK>
__device__ inline void x_update_split_block(const Geo &g, const Range3 &r, int bx, int by, int bz, int nbz, int64_t pi,
                                            double *phi, double *rr, const double *ra, const double *pa,
                                            const double *Ar, const double *rh, const double *p1, const double *p2,
                                            int64_t nb, double *sc, int *fl, double *pmax, double *pdot) {
    __shared__ double sm[8], smax[4 * UPD_ZG], carry[RED_THREADS];
    __shared__ int s_go;
    const int tid = (int)(threadIdx.x + RED_TX * threadIdx.y);
    const int zg = __builtin_amdgcn_readfirstlane((int)threadIdx.z);
    if (ASK && !wg_active(fl, &s_go)) return;
    if (!ASK && tid == 0 && zg == 0) s_go = fl[KF_ACTIVE];
    const int i = r.lo0 + bx * RED_TX + (int)threadIdx.x;
    const int j = r.lo1 + by * RED_TY + (int)threadIdx.y;
    const bool own = i < r.lo0 + r.n0 && j < r.lo1 + r.n1;
    int kc0, kc1;
    red_chunk(r, bz, nbz, kc0, kc1);
    int k0, cnt;
    split_planes(zg, kc0, kc1, k0, cnt);
    const int64_t x0 = gidx(g, own ? i : r.lo0, own ? j : r.lo1, 0);
    double vph[UPD_KP], vra[UPD_KP], vpa[UPD_KP], vrr[UPD_KP], vAr[UPD_KP], vrh[UPD_KP];
#pragma unroll
    for (int u = 0; u < UPD_KP; ++u) {
        vph[u] = vra[u] = vpa[u] = vrr[u] = vAr[u] = vrh[u] = 0.0;
        if (u < cnt) {
            const int64_t x = x0 + (int64_t)(k0 + u) * g.pxy;
            vph[u] = phi[x];
            vpa[u] = pa[x];
            vrr[u] = rr[x];
            vra[u] = PRE ? ra[x] : vrr[u];
            vAr[u] = Ar[x];
            vrh[u] = rh[x];
        }
    }
    const double alpha = sc[KS_ALPHA];
    if (zg == 0) split_sum_parts(p1, nb, tid, sm);
    if (zg == 1) split_sum_parts(p2, nb, tid, sm + 4);
    __syncthreads();
    if (!s_go) return;
    const double rAr = (sm[0] + sm[1]) + (sm[2] + sm[3]);
    const double ArAr = (sm[4] + sm[5]) + (sm[6] + sm[7]);
    const bool ok = !(fabs(ArAr) == 0.0);
    const double om = ok ? rAr / ArAr : 0.0;
    if (tid == 0 && zg == 0 && pi == 0) {
        if (ok)
            sc[KS_OMEGA] = om;
        else
            breakdown(fl);
    }
    if (!ok) return;
    double m = 0.0;
#pragma unroll
    for (int u = 0; u < UPD_KP; ++u) {
        const int64_t x = x0 + (int64_t)(k0 + u) * g.pxy;
        const double w = vrr[u] - om * vAr[u];
        const bool in = own && u < cnt;
        if (in) {
            phi[x] = vph[u] + om * vra[u] + alpha * vpa[u];
            rr[x] = w;
        }
        m = in ? max_nan(fabs(w), m) : m;
        vrh[u] = w * vrh[u];
    }
    m = wave_max(m);
    if ((tid & 63) == 0) smax[zg * 4 + (tid >> 6)] = m;
#pragma unroll
    for (int z = 0; z < UPD_ZG; ++z) {
        if (z > 0) __syncthreads();
        if (zg == z) {
            double d = z == 0 ? 0.0 : carry[tid];
#pragma unroll
            for (int u = 0; u < UPD_KP; ++u) d = own && u < cnt ? d + vrh[u] : d;
            if (z < UPD_ZG - 1) {
                carry[tid] = d;
            } else {
                const double s = wave_sum(d);
                if ((tid & 63) == 0) sm[tid >> 6] = s;
            }
        }
    }
    __syncthreads();
    if (tid == 0 && zg == 0) {
        m = smax[0];
        for (int q = 1; q < 4 * UPD_ZG; ++q) m = max_nan(smax[q], m);
        pmax[pi] = m;
        pdot[pi] = (sm[0] + sm[1]) + (sm[2] + sm[3]);
    }
}

// The operator's dot products from memory, for an operator launched in shorter z chunks
// than the reduction's: <o, Ap>, and <Ap, Ap> with TWO, the planes of a reduction chunk
// on UPD_ZG groups that take turns in plane order, so the partials are the fused ones'
// bits.
template <bool TWO>
__global__ __launch_bounds__(UPD_ZG * RED_THREADS) void k_dots(Geo g, Range3 r, int nbx, int nby, int nbz,
                                                               const double *__restrict__ Ap,
                                                               const double *__restrict__ o, double *part1,
                                                               double *part2, const int *active) {
    if (active && !*active) return;
    int bx, by, bz;
    if (!xcd_tile(nbx, nby, nbz, bx, by, bz)) return;
    const int64_t pi = (int64_t)bx + (int64_t)nbx * ((int64_t)by + (int64_t)nby * bz);
    __shared__ double sm[8], carry[TWO ? 2 : 1][RED_THREADS];
    const int tid = (int)(threadIdx.x + RED_TX * threadIdx.y);
    const int zg = __builtin_amdgcn_readfirstlane((int)threadIdx.z);
    const int i = r.lo0 + bx * RED_TX + (int)threadIdx.x;
    const int j = r.lo1 + by * RED_TY + (int)threadIdx.y;
    const bool own = i < r.lo0 + r.n0 && j < r.lo1 + r.n1;
    int kc0, kc1;
    red_chunk(r, bz, nbz, kc0, kc1);
    int k0, cnt;
    split_planes(zg, kc0, kc1, k0, cnt);
    const int64_t x0 = gidx(g, own ? i : r.lo0, own ? j : r.lo1, 0);
    double a[UPD_KP], b[UPD_KP];
#pragma unroll
    for (int u = 0; u < UPD_KP; ++u) {
        a[u] = b[u] = 0.0;
        if (u < cnt) {
            const int64_t x = x0 + (int64_t)(k0 + u) * g.pxy;
            a[u] = Ap[x];
            b[u] = o[x];
        }
    }
#pragma unroll
    for (int u = 0; u < UPD_KP; ++u) {
        b[u] = b[u] * a[u];
        a[u] = a[u] * a[u];
    }
#pragma unroll
    for (int z = 0; z < UPD_ZG; ++z) {
        if (z > 0) __syncthreads();
        if (zg == z) {
            double s1 = z == 0 ? 0.0 : carry[0][tid], s2 = z == 0 || !TWO ? 0.0 : carry[TWO][tid];
#pragma unroll
            for (int u = 0; u < UPD_KP; ++u) {
                s1 = own && u < cnt ? s1 + b[u] : s1;
                if (TWO) s2 = own && u < cnt ? s2 + a[u] : s2;
            }
            if (z < UPD_ZG - 1) {
                carry[0][tid] = s1;
                if (TWO) carry[TWO][tid] = s2;
            } else {
                s1 = wave_sum(s1);
                if (TWO) s2 = wave_sum(s2);
                if ((tid & 63) == 0) {
                    sm[tid >> 6] = s1;
                    sm[4 + (tid >> 6)] = s2;
                }
            }
        }
    }
    __syncthreads();
    if (tid == 0 && zg == 0) {
        part1[pi] = (sm[0] + sm[1]) + (sm[2] + sm[3]);
        if (TWO) part2[pi] = (sm[4] + sm[5]) + (sm[6] + sm[7]);
    }
}

// One block of it fills a compute unit (1024 threads of 104 or 120 VGPRs), so it is
// taken where its blocks fill their rounds over the device: up to one round, or with
// the last round at most an eighth of all empty.  A BiCGstab iteration with it and
// without: 118x71x91 (120 tiles) 78.1 / 82 us, 193x97x97 (364, the second round 42 %
// full) 105.3 / 104.7, 257x129x129 (765) 175.1 / 175.1, 385x193x193 (2275) 584 / 589.
static bool x_split(int64_t tiles, int64_t cus) {
    const int64_t rounds = (tiles + cus - 1) / cus;
    return rounds <= 1 || 8 * tiles >= 7 * rounds * cus;
}

template <bool PRE, bool ASK>
__global__ __launch_bounds__(RED_THREADS *UPD_ZG) void k_x_update_split(
    Geo g, Range3 r, double *phi, double *rr, const double *ra, const double *pa, const double *Ar, const double *rh,
    const double *p1, const double *p2, int64_t nb, double *sc, int *fl, double *pmax, double *pdot) {
    x_update_split_block<PRE, ASK>(g, r, (int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, (int)gridDim.z,
                                   part_index(), phi, rr, ra, pa, Ar, rh, p1, p2, nb, sc, fl, pmax, pdot);
}

// The end of an iteration by one workgroup: the norm and <rr, rh> from the partials,
// then the head of the next iteration, on copies of the scalars and flags that are
// loaded with the partials (each read behind a store would be a trip to the cache of
// its own, a dozen one after the other).
__device__ inline void ctl_end_block(const double *pmax, const double *pdot, int64_t nb, double *sc, int *fl) {
    __shared__ double sm[8];
    double s[KS_NSLOTS];
    int f[KF_NSLOTS];
#pragma unroll
    for (int q = 0; q < KS_NSLOTS; ++q) s[q] = sc[q];
#pragma unroll
    for (int q = 0; q < KF_NSLOTS; ++q) f[q] = fl[q];
    if (!f[KF_ACTIVE]) return;
    double tm, ts;
    thread_max_sum_parts(pmax, pdot, nb, (int)(threadIdx.x + threadIdx.y * blockDim.x), tm, ts);
    tm = wave_max(tm);
    ts = wave_sum(ts);
    const int tid = (int)(threadIdx.x + threadIdx.y * blockDim.x);
    if ((tid & 63) == 0) {
        sm[tid >> 6] = tm;
        sm[4 + (tid >> 6)] = ts;
    }
    __syncthreads();
    if (tid == 0) {
        double nm = sm[0];
        for (int q = 1; q < 4; ++q) nm = max_nan(sm[q], nm);
        s[KS_NORM] = nm;
        s[KS_RHR_NEXT] = (sm[4] + sm[5]) + (sm[6] + sm[7]);
        ctl_begin(s, f);
#pragma unroll
        for (int q = 0; q < KS_NSLOTS; ++q) sc[q] = s[q];
#pragma unroll
        for (int q = 0; q < KF_NSLOTS; ++q) fl[q] = f[q];
    }
}

__global__ __launch_bounds__(256) void k_ctl_end(const double *pmax, const double *pdot, int64_t nb, double *sc,
                                                 int *fl) {
    ctl_end_block(pmax, pdot, nb, sc, fl);
}

__global__ __launch_bounds__(256) void k_set_rhr(const double *part, int64_t nb, double *sc) {
    __shared__ double sm[4];
    const double v = reduce_sum_parts(part, nb, sm);
    if (threadIdx.x == 0 && threadIdx.y == 0) sc[KS_RHR] = v;
}

// ---------------------------------------------------------------------------
// Batched BiCGstab.  One launch covers the tiles of many cases (any grid
// sizes): tile_case maps a global tile to its case, and a case's tiles are its
// operator/reduction tiles in the single-case numbering from its tile0.  Every
// block runs the block function of the single-case kernel for that tile and
// writes the partial of the same index into the case's own buffers, and every
// scalar step reads the case's own scalars, so each case's iteration is
// bit-identical to its own solve.  A case whose solve has stopped (its active
// flag cleared) makes its blocks return at once.
// ---------------------------------------------------------------------------
__device__ inline int batch_tile(const KBatchCase *cases, const int *tile_case, int ntiles, int &bx, int &by,
                                 int &bz, int64_t &pi) {
    int t, d1, d2;
    if (!xcd_tile(ntiles, 1, 1, t, d1, d2)) return -1;
    const int q = tile_case[t];
    const int local = t - cases[q].tile0;
    const int nbx = cases[q].nbx, nby = cases[q].nby;
    bx = local % nbx;
    const int rem = local / nbx;
    by = rem % nby;
    bz = rem / nby;
    pi = local;
    return q;
}

template <bool TEAMS, int DM, bool PZ>
__global__ __launch_bounds__(apply_threads(TEAMS), apply_waves(TEAMS)) void k_apply_batch(
    const KBatchCase *__restrict__ cases, const int *__restrict__ tile_case, int ntiles, int form, int pre) {
    int bx, by, bz;
    int64_t pi;
    const int q = batch_tile(cases, tile_case, ntiles, bx, by, bz, pi);
    if (q < 0) return;
    const KBatchCase &K = cases[q];
    if ((K.g.per[2] != 0) != PZ) return;  // the other launch of this form covers it
    if (form != KB_APPLY_PHI && !K.fl[KF_ACTIVE]) return;
    const double *src = K.phi, *w = nullptr;
    double *dst = K.rr;
    if (form == KB_APPLY_W) {
        src = pre ? K.z1 : K.pk;
        dst = K.Ap;
        w = K.rh;
    } else if (form == KB_APPLY_SELF) {
        src = K.rr;
        dst = K.Ar;
    } else if (form == KB_APPLY_PAIR) {
        src = K.z2;
        dst = K.Ar;
        w = K.rr;
    }
    apply_block<TEAMS, DM, PZ>(K.g, K.c, K.r, bx, by, bz, K.nbz, pi, src, dst, w, K.part1, K.part2);
}

// the first-sweep operands of a batched case
__device__ inline FirstSweep batch_first(const KBatchCase &K, float omega) {
    return FirstSweep{K.c.dgf[0], K.c.dgf[1], K.c.dgf[2], omega, K.b32, K.e32};
}

// pk = rr + beta*pk + om2*Ap (rr in the first iteration) over a reduction tile;
// FIRST: with M's first FP32 sweep of pk
template <bool FIRST>
__global__ __launch_bounds__(256) void k_p_update_batch(const KBatchCase *__restrict__ cases,
                                                        const int *__restrict__ tile_case, int ntiles, float omega) {
    int bx, by, bz;
    int64_t pi;
    const int q = batch_tile(cases, tile_case, ntiles, bx, by, bz, pi);
    if (q < 0) return;
    const KBatchCase &K = cases[q];
    if (!K.fl[KF_ACTIVE]) return;
    const Range3 &r = K.r;
    const int i = r.lo0 + bx * RED_TX + (int)threadIdx.x;
    const int j = r.lo1 + by * RED_TY + (int)threadIdx.y;
    if (i >= r.lo0 + r.n0 || j >= r.lo1 + r.n1) return;
    int kc0, kc1;
    red_chunk(r, bz, K.nbz, kc0, kc1);
    const bool mode = K.fl[KF_MODE] != 0;
    const double beta = K.sc[KS_BETA], om2 = K.sc[KS_OM2];
    const FirstSweep fs = batch_first(K, omega);
    for (int k = kc0; k <= kc1; ++k) {
        const int64_t x = gidx(K.g, i, j, k);
        const double p = mode ? K.rr[x] + beta * K.pk[x] + om2 * K.Ap[x] : K.rr[x];
        K.pk[x] = p;
        if (FIRST) first_sweep_point(K.g, fs, i, j, k, x, p);
    }
}

template <bool FIRST>
__global__ __launch_bounds__(RED_THREADS *UPD_ZG) void k_s_update_batch(const KBatchCase *__restrict__ cases,
                                                        const int *__restrict__ tile_case, int ntiles, float omega) {
    int bx, by, bz;
    int64_t pi;
    const int q = batch_tile(cases, tile_case, ntiles, bx, by, bz, pi);
    if (q < 0) return;
    const KBatchCase &K = cases[q];
    s_update_block<FIRST, true>(K.g, K.r, bx, by, bz, K.nbz, pi, K.rr, K.Ap, K.part1, K.nb, K.sc, K.fl,
                                batch_first(K, omega));
}

template <bool SPLIT>
__global__ __launch_bounds__(SPLIT ? RED_THREADS * UPD_ZG : RED_THREADS) void k_x_update_batch(
    const KBatchCase *__restrict__ cases, const int *__restrict__ tile_case, int ntiles, int pre) {
    int bx, by, bz;
    int64_t pi;
    const int q = batch_tile(cases, tile_case, ntiles, bx, by, bz, pi);
    if (q < 0) return;
    const KBatchCase &K = cases[q];
    const double *ra = pre ? K.z2 : K.rr, *pa = pre ? K.z1 : K.pk;
    if constexpr (SPLIT)
        x_update_split_block<true, true>(K.g, K.r, bx, by, bz, K.nbz, pi, K.phi, K.rr, ra, pa, K.Ar, K.rh, K.part1,
                                         K.part2, K.nb, K.sc, K.fl, K.part3, K.part4);
    else
        x_update_block(K.g, K.r, bx, by, bz, K.nbz, pi, K.phi, K.rr, ra, pa, K.Ar, K.rh, K.part1, K.part2, K.nb, K.sc,
                       K.fl, K.part3, K.part4);
}

// one workgroup per case
__global__ __launch_bounds__(256) void k_ctl_end_batch(const KBatchCase *__restrict__ cases) {
    const KBatchCase &K = cases[blockIdx.x];
    ctl_end_block(K.part3, K.part4, K.nb, K.sc, K.fl);
}

// rr = bb - rr, rh = rr with their partials, and max|bb| partials (part3)
__global__ __launch_bounds__(256) void k_init_rr_batch(const KBatchCase *__restrict__ cases,
                                                       const int *__restrict__ tile_case, int ntiles) {
    int bx, by, bz;
    int64_t pi;
    const int q = batch_tile(cases, tile_case, ntiles, bx, by, bz, pi);
    if (q < 0) return;
    const KBatchCase &K = cases[q];
    init_rr_block(K.g, K.r, bx, by, bz, K.nbz, pi, K.bb, K.rr, K.rh, K.part1, K.part2);
    __syncthreads();
    __shared__ double sm[4];
    const Range3 &r = K.r;
    const int i = r.lo0 + bx * RED_TX + (int)threadIdx.x;
    const int j = r.lo1 + by * RED_TY + (int)threadIdx.y;
    double m = 0.0;
    if (i < r.lo0 + r.n0 && j < r.lo1 + r.n1) {
        int kc0, kc1;
        red_chunk(r, bz, K.nbz, kc0, kc1);
        for (int k = kc0; k <= kc1; ++k) {
            const double a = fabs(K.bb[gidx(K.g, i, j, k)]);
            m = max_nan(a, m);
        }
    }
    const double bm = block_max(m, sm);
    if (threadIdx.x == 0 && threadIdx.y == 0) K.part3[pi] = bm;
}

// per case: eps = tol * max|bb| (the host's bnorm product, here on the device),
// then k_ctl_setup's work on the initial residual's partials
__global__ __launch_bounds__(256) void k_ctl_setup_batch(const KBatchCase *__restrict__ cases, double tol, int nmax) {
    const KBatchCase &K = cases[blockIdx.x];
    __shared__ double sm[8];
    const double bmax = reduce_max_parts(K.part3, K.nb, sm);
    __syncthreads();
    const double nm = reduce_max_parts(K.part1, K.nb, sm + 4);
    __syncthreads();
    const double dt = reduce_sum_parts(K.part2, K.nb, sm);
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        double *sc = K.sc;
        int *fl = K.fl;
        sc[KS_NORM] = nm;
        sc[KS_NORM0] = nm;
        sc[KS_RHR_NEXT] = dt;
        sc[KS_RHR] = 0.0;
        sc[KS_ALPHA] = 0.0;
        sc[KS_OMEGA] = 0.0;
        sc[KS_EPS] = tol * bmax;
        fl[KF_ACTIVE] = 1;
        fl[KF_COUNTER] = 0;
        fl[KF_NMAX] = nmax;
        fl[KF_EXIT] = 0;
        fl[KF_RESET] = 0;
        fl[KF_MODE] = 0;
        fl[KF_DONE] = 0;
        ctl_begin(sc, fl);
    }
}

// every case's flags and scalars into one array each, for a single copy to the host
__global__ void k_gather_batch(const KBatchCase *__restrict__ cases, int ncases, int *fl_out, double *sc_out) {
    const int q = blockIdx.x;
    const int t = threadIdx.x;
    if (q >= ncases) return;
    if (t < KF_NSLOTS) fl_out[q * KF_NSLOTS + t] = cases[q].fl[t];
    if (t < KS_NSLOTS) sc_out[q * KS_NSLOTS + t] = cases[q].sc[t];
}

}  // namespace

// ===========================================================================
static inline Range3 Rk(const Box &b) { return make_range(b); }

// z chunks of an operator that leaves its dot products to k_dots: as many as fill the
// device with two blocks of teams a compute unit, of about three planes (balanced: where
// the planes limit their number some have two).  A block
// marches its chunk and six planes more at 0.6 us a plane, so a grid of few columns is
// bound by the 32 planes of the reduction's chunk; k_dots costs 3.5 to 5 us.  Operator
// fused / split without k_dots, a BiCGstab iteration fused / split, microseconds:
//   33x17x17     14.1 /  6.5   48.1 / 45.0     118x71x91   22.5 / 12.9   83.1 / 70.9
//   65^3         17.3 /  9.2   61.1 / 54.8     97^3        20.0 / 15.9   (not taken)
//   129x65x65    17.6 / 11.4   65.5 / 61.2     193x97x97   28.9 / 27.1   (not taken)
// hence at least APPLY_SPLIT times the reduction's chunks (97^3 has 10 for 4).
static int apply_split(int columns, int planes, int cus) {
    return (int)std::min<int64_t>((planes + 2) / 3, apply_team_tiles(cus) / columns);
}
constexpr int APPLY_SPLIT = 3;

void launch_apply_A(hipStream_t s, const Geo &g, const Coef &c, const Box &pb, const double *src, double *dst,
                    const double *w, int dot_mode, double *part1, double *part2, const int *active) {
    Range3 r = Rk(pb);
    if (empty(r)) return;
    // the operator tile is the reduction tile, so the fused dot partials follow the fixed tree
    const int nbx = (r.n0 + RED_TX - 1) / RED_TX, nby = (r.n1 + RED_TY - 1) / RED_TY, nbz = (r.n2 + RED_KC - 1) / RED_KC;
    const int64_t tiles = (int64_t)nbx * nby * nbz;
    const int nsplit = apply_split(nbx * nby, r.n2, g.cus);
    if (nsplit >= APPLY_SPLIT * nbz) {
        const dim3 grid(xcd_grid((int64_t)nbx * nby * nsplit)), block(RED_TX, RED_TY, 2);
        if (g.per[2])
            hipLaunchKernelGGL((k_apply<true, DOT_NONE, true>), grid, block, 0, s, g, c, r, nbx, nby, nsplit, src, dst,
                               nullptr, nullptr, nullptr, active);
        else
            hipLaunchKernelGGL((k_apply<true, DOT_NONE, false>), grid, block, 0, s, g, c, r, nbx, nby, nsplit, src, dst,
                               nullptr, nullptr, nullptr, active);
        const dim3 dgrid(xcd_grid(tiles)), dblock(RED_TX, RED_TY, UPD_ZG);
        if (dot_mode == DOT_W)
            hipLaunchKernelGGL(k_dots<false>, dgrid, dblock, 0, s, g, r, nbx, nby, nbz, dst, w, part1, part2, active);
        else if (dot_mode != DOT_NONE)
            hipLaunchKernelGGL(k_dots<true>, dgrid, dblock, 0, s, g, r, nbx, nby, nbz, dst,
                               dot_mode == DOT_SELF ? src : w, part1, part2, active);
        return;
    }
    const bool teams = tiles <= apply_team_tiles(g.cus);
    const dim3 grid(xcd_grid(tiles)), block(RED_TX, RED_TY, teams ? 2 : 1);
#define IH_APPLY_AS(T, DMV, PZV)                                                                               \
    hipLaunchKernelGGL((k_apply<T, DMV, PZV>), grid, block, 0, s, g, c, r, nbx, nby, nbz, src, dst, w, part1, part2, \
                       active)
#define IH_APPLY(DMV)                         \
    do {                                      \
        if (teams && g.per[2])                \
            IH_APPLY_AS(true, DMV, true);     \
        else if (teams)                       \
            IH_APPLY_AS(true, DMV, false);    \
        else if (g.per[2])                    \
            IH_APPLY_AS(false, DMV, true);    \
        else                                  \
            IH_APPLY_AS(false, DMV, false);   \
    } while (0)
    if (dot_mode == DOT_W)
        IH_APPLY(DOT_W);
    else if (dot_mode == DOT_SELF)
        IH_APPLY(DOT_SELF);
    else if (dot_mode == DOT_PAIR)
        IH_APPLY(DOT_PAIR);
    else
        IH_APPLY(DOT_NONE);
#undef IH_APPLY
#undef IH_APPLY_AS
}

void launch_krylov_init(hipStream_t s, const Geo &g, const Box &b, const double *bb, double *rr, double *rh,
                        double *pmax, double *pdot, double *sc, int *fl, double eps, int nmax) {
    Range3 r = Rk(b);
    hipLaunchKernelGGL(k_init_rr, red_grid(r), dim3(RED_TX, RED_TY, 1), 0, s, g, r, bb, rr, rh, pmax, pdot);
    hipLaunchKernelGGL(k_ctl_setup, dim3(1), dim3(RED_TX, RED_TY, 1), 0, s, pmax, pdot, red_blocks(b), sc, fl, eps,
                       nmax);
}

// z = M v: `sweeps` FP32 JOR sweeps on A_cdg e = (float)v from e = 0, z = (double)e.
// The first sweep reads v itself (and stores b = (float)v), the last writes z
// widened to double, so M costs sweeps passes over the box and no more.  With
// first_done the kernel that wrote v has formed the first sweep already.
static void launch_precond(hipStream_t s, const Geo &g, const Coef &c, const Box &b, double *v, double *z,
                           const KrylovPtrs &k, bool first_done = false) {
    const int *act = k.fl + KF_ACTIVE;
    if (k.mg) {
        // multigridV(.TRUE.,1,v,z) (src/mod_solvers.f90:1688, 1751)
        if (k.mg_fp32)
            launch_mg_vcycle_f32(s, *k.mg, v, z, act);
        else
            launch_mg_vcycle(s, *k.mg, v, z, act);
        return;
    }
    if (k.sweeps64 > 0) {
        // FP64 sweeps on A e = v from e = 0 (the like-for-like FP64 form of the FP32 M):
        // the first reads the zero field, the last writes z
        const bool pairs = jor_pair_ok(g, c, b, false);
        const double *x = k.zero64;
        for (int q = 0; q < k.sweeps64;) {
            // an odd count's single sweep comes first
            const int n = pairs && (k.sweeps64 - q) % 2 == 0 ? 2 : 1;
            q += n;
            double *y = q == k.sweeps64 ? z : (x == k.e64a ? k.e64b : k.e64a);
            if (n == 2)
                launch_jor_pair(s, g, c, b, k.omega64, x, v, y, act);
            else
                launch_jor(s, g, c, b, k.omega64, x, v, y, act, k.shape64);
            x = y;
        }
        return;
    }
    if (k.sweeps == 1) {
        launch_jor_f32_first(s, g, c, b, k.omega, v, k.b32, nullptr, z, act);
        return;
    }
    if (!first_done) launch_jor_f32_first(s, g, c, b, k.omega, v, k.b32, k.e0, nullptr, act);
    // the sweeps after the first, two a launch where the box takes pairs
    const bool pairs = jor_pair_ok(g, c, b, true);
    float *x = k.e0, *y = k.e1;
    for (int left = k.sweeps - 1; left > 0;) {
        const int n = pairs && left % 2 == 0 ? 2 : 1;
        left -= n;
        if (left == 0 && n == 2)
            launch_jor_pair(s, g, c, b, k.omega, x, k.b32, z, act);
        else if (left == 0)
            launch_jor_f32_to64(s, g, c, b, k.omega, x, k.b32, z, act, k.shape);
        else if (n == 2)
            launch_jor_pair(s, g, c, b, k.omega, x, k.b32, y, act);
        else
            launch_jor_f32(s, g, c, b, k.omega, x, k.b32, y, act, k.shape);
        std::swap(x, y);
    }
}

static void launch_s_update(hipStream_t s, const Geo &g, const Range3 &r, int64_t nb, const KrylovPtrs &k, bool first,
                            const FirstSweep &fs) {
    auto *const kern = first ? (k.ask ? k_s_update_alpha<true, true> : k_s_update_alpha<true, false>)
                             : (k.ask ? k_s_update_alpha<false, true> : k_s_update_alpha<false, false>);
    hipLaunchKernelGGL(kern, red_grid(r), dim3(RED_TX, RED_TY, UPD_ZG), 0, s, g, r, k.rr, k.Ap, k.part1, nb, k.sc, k.fl,
                       fs);
}

static void launch_x_update(hipStream_t s, const Geo &g, const Range3 &r, int64_t nb, const KrylovPtrs &k, bool pre) {
    const double *ra = pre ? k.z2 : k.rr, *pa = pre ? k.z1 : k.pk;
    if (!x_split(nb, g.cus)) {
        hipLaunchKernelGGL(k_x_update_omega, red_grid(r), dim3(RED_TX, RED_TY, 1), 0, s, g, r, k.phi, k.rr, ra, pa,
                           k.Ar, k.rh, k.part1, k.part2, nb, k.sc, k.fl, k.part3, k.part4);
        return;
    }
    auto *const kern = pre ? (k.ask ? k_x_update_split<true, true> : k_x_update_split<true, false>)
                           : (k.ask ? k_x_update_split<false, true> : k_x_update_split<false, false>);
    hipLaunchKernelGGL(kern, red_grid(r), dim3(RED_TX, RED_TY, UPD_ZG), 0, s, g, r, k.phi, k.rr, ra, pa, k.Ar, k.rh,
                       k.part1, k.part2, nb, k.sc, k.fl, k.part3, k.part4);
}

void launch_krylov_iteration(hipStream_t s, const Geo &g, const Coef &c, const Box &b, const KrylovPtrs &k) {
    Range3 r = Rk(b);
    const int64_t nb = red_blocks(b);
    const bool pre = k.sweeps > 0 || k.sweeps64 > 0 || k.mg;
    // FP32 sweeps as M (two or more): the p and s updates also form M's first sweep
    const bool fuse = !k.mg && k.sweeps64 == 0 && k.sweeps >= 2;
    const FirstSweep fs{c.dgf[0], c.dgf[1], c.dgf[2], k.omega, k.b32, k.e0};
    if (fuse)
        hipLaunchKernelGGL(k_p_update<true>, grid_for(r), dim3(BX, BY, 1), 0, s, g, r, k.rr, k.pk, k.Ap, k.sc, k.fl,
                           fs);
    else
        hipLaunchKernelGGL(k_p_update<false>, grid_for(r), dim3(BX, BY, 1), 0, s, g, r, k.rr, k.pk, k.Ap, k.sc, k.fl,
                           FirstSweep{});
    if (pre) launch_precond(s, g, c, b, k.pk, k.z1, k, fuse);
    launch_apply_A(s, g, c, b, pre ? k.z1 : k.pk, k.Ap, k.rh, DOT_W, k.part1, nullptr, k.fl + KF_ACTIVE);
    launch_s_update(s, g, r, nb, k, fuse, fs);
    if (pre) {
        launch_precond(s, g, c, b, k.rr, k.z2, k, fuse);
        launch_apply_A(s, g, c, b, k.z2, k.Ar, k.rr, DOT_PAIR, k.part1, k.part2, k.fl + KF_ACTIVE);
    } else {
        launch_apply_A(s, g, c, b, k.rr, k.Ar, nullptr, DOT_SELF, k.part1, k.part2, k.fl + KF_ACTIVE);
    }
    launch_x_update(s, g, r, nb, k, pre);
    hipLaunchKernelGGL(k_ctl_end, dim3(1), dim3(RED_TX, RED_TY, 1), 0, s, k.part3, k.part4, nb, k.sc, k.fl);
}

void launch_krylov_part(hipStream_t s, const Geo &g, const Coef &c, const Box &b, const KrylovPtrs &k, int which) {
    Range3 r = Rk(b);
    const int64_t nb = red_blocks(b);
    switch (which) {
    case KPART_P_UPDATE:
        hipLaunchKernelGGL(k_p_update<false>, grid_for(r), dim3(BX, BY, 1), 0, s, g, r, k.rr, k.pk, k.Ap, k.sc, k.fl,
                           FirstSweep{});
        break;
    case KPART_APPLY_W:
        launch_apply_A(s, g, c, b, k.pk, k.Ap, k.rh, DOT_W, k.part1, nullptr, k.fl + KF_ACTIVE);
        break;
    case KPART_S_UPDATE:
        launch_s_update(s, g, r, nb, k, false, FirstSweep{});
        break;
    case KPART_APPLY_SELF:
        launch_apply_A(s, g, c, b, k.rr, k.Ar, nullptr, DOT_SELF, k.part1, k.part2, k.fl + KF_ACTIVE);
        break;
    case KPART_X_UPDATE:
        launch_x_update(s, g, r, nb, k, false);
        break;
    default:
        break;
    }
}

void launch_apply_batch(hipStream_t s, const KBatchCase *cases, const int *tile_case, int ntiles, int form, bool pre,
                        bool any_pz, bool any_nonpz, int cus) {
    if (ntiles <= 0) return;
    const bool teams = ntiles <= apply_team_tiles(cus);
    const dim3 grid(xcd_grid(ntiles)), block(RED_TX, RED_TY, teams ? 2 : 1);
#define IH_APB_AS(T, DMV, PZV)                                                                                    \
    hipLaunchKernelGGL((k_apply_batch<T, DMV, PZV>), grid, block, 0, s, cases, tile_case, ntiles, form, (int)pre)
#define IH_APB(DMV)                               \
    do {                                          \
        if (any_nonpz && teams)                   \
            IH_APB_AS(true, DMV, false);          \
        else if (any_nonpz)                       \
            IH_APB_AS(false, DMV, false);         \
        if (any_pz && teams)                      \
            IH_APB_AS(true, DMV, true);           \
        else if (any_pz)                          \
            IH_APB_AS(false, DMV, true);          \
    } while (0)
    if (form == KB_APPLY_W)
        IH_APB(DOT_W);
    else if (form == KB_APPLY_SELF)
        IH_APB(DOT_SELF);
    else if (form == KB_APPLY_PAIR)
        IH_APB(DOT_PAIR);
    else
        IH_APB(DOT_NONE);
#undef IH_APB
#undef IH_APB_AS
}

void launch_krylov_init_batch(hipStream_t s, const KBatchCase *cases, int ncases, const int *tile_case, int ntiles,
                              double tol, int nmax) {
    if (ntiles <= 0) return;
    hipLaunchKernelGGL(k_init_rr_batch, dim3(xcd_grid(ntiles)), dim3(RED_TX, RED_TY, 1), 0, s, cases, tile_case,
                       ntiles);
    hipLaunchKernelGGL(k_ctl_setup_batch, dim3(ncases), dim3(RED_TX, RED_TY, 1), 0, s, cases, tol, nmax);
}

void launch_p_update_batch(hipStream_t s, const KBatchCase *cases, const int *tile_case, int ntiles, bool first,
                           float omega) {
    if (ntiles <= 0) return;
    if (first)
        hipLaunchKernelGGL(k_p_update_batch<true>, dim3(xcd_grid(ntiles)), dim3(RED_TX, RED_TY, 1), 0, s, cases,
                           tile_case, ntiles, omega);
    else
        hipLaunchKernelGGL(k_p_update_batch<false>, dim3(xcd_grid(ntiles)), dim3(RED_TX, RED_TY, 1), 0, s, cases,
                           tile_case, ntiles, omega);
}

void launch_s_update_batch(hipStream_t s, const KBatchCase *cases, const int *tile_case, int ntiles, bool first,
                           float omega) {
    if (ntiles <= 0) return;
    if (first)
        hipLaunchKernelGGL(k_s_update_batch<true>, dim3(xcd_grid(ntiles)), dim3(RED_TX, RED_TY, UPD_ZG), 0, s, cases,
                           tile_case, ntiles, omega);
    else
        hipLaunchKernelGGL(k_s_update_batch<false>, dim3(xcd_grid(ntiles)), dim3(RED_TX, RED_TY, UPD_ZG), 0, s, cases,
                           tile_case, ntiles, omega);
}

void launch_x_update_batch(hipStream_t s, const KBatchCase *cases, const int *tile_case, int ntiles, bool pre,
                           int cus) {
    if (ntiles <= 0) return;
    if (x_split(ntiles, cus))
        hipLaunchKernelGGL(k_x_update_batch<true>, dim3(xcd_grid(ntiles)), dim3(RED_TX, RED_TY, UPD_ZG), 0, s, cases,
                           tile_case, ntiles, (int)pre);
    else
        hipLaunchKernelGGL(k_x_update_batch<false>, dim3(xcd_grid(ntiles)), dim3(RED_TX, RED_TY, 1), 0, s, cases,
                           tile_case, ntiles, (int)pre);
}

void launch_gather_batch(hipStream_t s, const KBatchCase *cases, int ncases, int *fl_out, double *sc_out) {
    if (ncases > 0) hipLaunchKernelGGL(k_gather_batch, dim3(ncases), dim3(64), 0, s, cases, ncases, fl_out, sc_out);
}

void launch_ctl_end_batch(hipStream_t s, const KBatchCase *cases, int ncases) {
    if (ncases > 0) hipLaunchKernelGGL(k_ctl_end_batch, dim3(ncases), dim3(RED_TX, RED_TY, 1), 0, s, cases);
}

void launch_krylov_resume(hipStream_t s, const Geo &g, const Box &b, const KrylovPtrs &k) {
    // rh = rr, rhr = <rr, rh>, then the tail of the iteration head
    launch_copy_box(s, g, b, k.rr, k.rh);
    launch_dot_partial(s, g, b, k.rr, k.rh, k.part1);
    hipLaunchKernelGGL(k_set_rhr, dim3(1), dim3(RED_TX, RED_TY, 1), 0, s, k.part1, red_blocks(b), k.sc);
    hipLaunchKernelGGL(k_ctl_resume, dim3(1), dim3(1), 0, s, k.sc, k.fl);
}

}  // namespace ih
