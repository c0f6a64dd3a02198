// tpsph_adjoint.hip -- reverse mode of the right-hand side (the pullback of kick!) and of a
// CarpenterKennedy2N54 trajectory with step checkpoints.
//
// The reference has no automatic differentiation through its right-hand side; the pullback
// here is written by hand from the terms of the forward pass (wcsph/rhs.jl:5-127,
// fluid.jl:160-197, density_diffusion.jl:213-240, pressure_acceleration.jl:34-41,
// viscosity.jl:89-132, dummy_particles.jl:489-569 and 586-672, state_equations.jl:100-139).
// Differentiated: the fluid state (v, rho, x) and the scalars alpha (Monaghan), delta
// (Molteni-Colagrossi) and g (gravity = g * unit direction of the acceleration).  Options:
// WendlandC2, StateEquationCole with a fixed sound speed, ArtificialViscosityMonaghan,
// Molteni-Colagrossi or no density diffusion, Adami walls without viscosity, FP64.
//
// Every pass is a gather, so no floating-point atomics and the results are deterministic:
//
//   phi_ab = Gbar_a . dv_ab + rbar_a drho_ab
//
// is the adjoint-weighted pair term of particle a's rates (Gbar_a, rbar_a: the adjoint of a's
// dv and drho).  Fluid particle c collects d phi / d state_c over its own terms (phi_ca) and
// its partners' terms (phi_ac): the neighbour relation is symmetric, so the partners are its
// own neighbours.  The wall pressures and densities of the Adami pass depend on the fluid
// near each wall particle; their adjoints are gathered per wall particle first (k_adj_wall),
// which turns them into two coefficients per wall particle that the fluid pass (k_adj_fluid)
// then reads.  Non-smooth points take the branch the forward pass took: the viscosity switch
// v_ab.r_ab < 0, the clipping of the wall pressure, the volume bound of the Adami pass.
//
// Checkpoints: tpsph_adjoint_forward keeps the state at the start of every segment of
// `checkpoint_every` steps; tpsph_adjoint_reverse runs the segments backwards, recomputes each
// from its checkpoint while keeping the state of every stage, and sweeps the stages in
// reverse.  The stage map of the 2N-storage scheme,
//     tmp_i = A_i tmp_{i-1} + dt k(y_{i-1}),   y_i = y_{i-1} + B_i tmp_i,
// reverses to
//     tbar += B_i ybar,   kbar = dt tbar,   ybar += J(y_{i-1})^T kbar,   tbar *= A_i
// with k = (kick!, drift!) and J^T kbar the pullback of kick! plus the drift's vbar += kbar_u.
#include "tpsph_internal.h"

#include <algorithm>

using namespace tpsph;

namespace {

constexpr int kRedBlocks = 256;  // blocks of the deterministic parameter reduction
constexpr int kAdjLanes = 4;     // lanes per particle of the adjoint passes

// Constants of the parameter derivatives (d dd2 / d delta and d (alpha c) / d alpha, zero without
// the diffusion or the viscosity, and the unit gravity direction) and of the fluid pairs: alpha c
// and beta of the viscosity (zero without) and -1/(2 h), -3/(2 h).
struct AdjConsts {
    double dd2_per_delta, visc_per_alpha;
    double ghat[3];
    double visc, beta, minus_half_h_inv, minus_3half_h_inv;
};

// d phi_ab / d(inputs) of the term of fluid particle a with wall partner b (at rest, without
// viscosity and density diffusion): r_ab (r), its square d2, v_a (va), the density and pressure
// of a, rho_b and V_b = m_b / rho_b of the wall and its pressure, and the adjoint weights G (of
// dv_a) and gr (of drho_a).
// Outputs: d phi / d r_ab, d phi / d vr (d phi / d v_a = vr r_ab), d phi / d rho_a,
// d phi / d rho_b (total: also through V_b) and d phi / d p_a = d phi / d p_b.  sqrt and the
// reciprocals are the refined hardware approximations of the forward pass (within a few ulp).
struct WallAdj {
    double r[3];
    double vr;
    double rho_a, rho_b, p;
};

template <int ND>
__device__ __forceinline__ WallAdj wall_adj(const DevParams &P, const double *r, double d2,
                                            const double *va, double rho_a, double inv_rho_a,
                                            double inv_rho_b, double p_a, double p_b, double V_b,
                                            const double *G, double gr)
{
    WallAdj o;
    const double d = sqrt_pos(d2);
    const double w = 1.0 - 0.5 * P.h_inv * d;
    const double kdr = P.kgrad_c * (w * w * w);  // grad W = kdr r_ab
    const double dkdr = P.kgrad_c * (-1.5 * P.h_inv) * (w * w) * rcp_pos(d);  // d kdr / d r_ab = dkdr r_ab
    double A = G[0] * r[0] + G[1] * r[1], vr = va[0] * r[0] + va[1] * r[1];
    if constexpr (ND == 3) A += G[2] * r[2], vr += va[2] * r[2];
    const double fac = -V_b * (p_a + p_b) * inv_rho_a;
    const double E = rho_a * vr;  // drho_ab = V_b kdr E
    const double kA = kdr * A;    // dv_ab = fac kdr r_ab
    const double radial = (fac * A + gr * V_b * E) * dkdr;
    o.vr = gr * V_b * kdr * rho_a;
#pragma unroll
    for (int k = 0; k < 3; k++) o.r[k] = 0.0;
#pragma unroll
    for (int k = 0; k < ND; k++) o.r[k] = kdr * fac * G[k] + o.vr * va[k] + radial * r[k];
    o.p = -kA * V_b * inv_rho_a;
    o.rho_a = kA * (V_b * (p_a + p_b) * (inv_rho_a * inv_rho_a)) + gr * V_b * kdr * vr;
    o.rho_b = (kA * (p_a + p_b) * inv_rho_a - gr * kdr * E) * V_b * inv_rho_b;
    return o;
}

// A fluid particle of the fluid-fluid pullback: its state and the adjoint weights of its rates.
struct AdjRec {
    double x[3], rho, v[3], p, V, G[3], gr;
};

// What the fluid-fluid pairs of one particle c (the target) add to d L / d state_c, and their
// parts of the alpha and delta derivatives.
//
// Both terms of a pair at once, phi_cj + phi_jc.  With K the kernel factor (grad W = K r),
// r = x_c - x_j, v = v_c - v_j, w = 1 / (rho_c rho_j), D = m_j G_c - m_c G_j, T = D.r,
// B = Pi - (p_c + p_j) w and Pi the viscosity per partner mass,
//   phi_cj + phi_jc = K (T B + dd2 (rho_c - rho_j) X + v.r Z),
//   X = g_c V_j - g_j V_c,   Z = g_c V_j rho_c + g_j V_c rho_j   (g: the weight of drho)
// so the sums share all but a few of their operations (two terms one after the other: about 190
// instructions for a pair, this form 120).  Every unordered pair meets both its particles, so
// alpha and delta take half of its two terms from each.
template <int ND>
struct AdjTarget {
    AdjRec c;
    double m, inv_rho;
    double xb[3] = {0.0, 0.0, 0.0}, vb[3] = {0.0, 0.0, 0.0};
    double rhob = 0.0, pb = 0.0, alpha = 0.0, delta = 0.0;

    __device__ __forceinline__ void set(const AdjRec &target)
    {
        c = target;
        m = c.rho * c.V;
        inv_rho = rcp_pos(c.rho);
    }

    __device__ __forceinline__ void pair(const DevParams &P, const AdjConsts &C, const AdjRec &j)
    {
        const double r0 = c.x[0] - j.x[0], r1 = c.x[1] - j.x[1];
        const double r2 = (ND == 3) ? c.x[2] - j.x[2] : 0.0;
        const double d2 = dist2<ND>(r0, r1, r2);
        if (!(d2 <= P.R2 && d2 >= P.az2)) return;
        // sqrt_pos and the reciprocal of its result
        const double y = __builtin_amdgcn_rsq(d2);
        const double g = d2 * y;
        const double d = fma(g, fma(-0.5 * y, g, 0.5), g);
        const double inv_d = fma(y, fma(-d, y, 1.0), y);
        const double w1 = fma(C.minus_half_h_inv, d, 1.0);
        const double w2 = w1 * w1;
        const double K = w2 * w1;  // without its constant (scale)
        const double dK = C.minus_3half_h_inv * w2 * inv_d;
        // one reciprocal for 1 / (d^2 + eps h^2), 1 / (rho_c + rho_j) and 1 / (rho_c rho_j)
        const double q = d2 + P.eps_h2, sum = c.rho + j.rho, prod = c.rho * j.rho;
        const double ps = prod * sum;
        const double qps = q * ps, R1 = rcp_pos(qps);
        const double R = fma(R1, fma(-qps, R1, 1.0), R1);  // (three results share its error)
        const double inv_q = R * ps, Rq = R * q;
        const double w = Rq * sum, inv_sum = Rq * prod;

        const double v0 = c.v[0] - j.v[0], v1 = c.v[1] - j.v[1];
        const double v2 = (ND == 3) ? c.v[2] - j.v[2] : 0.0;
        double vr = v0 * r0 + v1 * r1;
        const double mj = j.rho * j.V;
        const double D0 = mj * c.G[0] - m * j.G[0], D1 = mj * c.G[1] - m * j.G[1];
        const double D2 = (ND == 3) ? mj * c.G[2] - m * j.G[2] : 0.0;
        double T = D0 * r0 + D1 * r1;
        if constexpr (ND == 3) {
            vr += v2 * r2;
            T += D2 * r2;
        }
        // Pi = 2 (alpha c mu + beta mu^2) / (rho_c + rho_j), mu = h min(vr, 0) / q
        const double mu = P.h * (fmin(vr, 0.0) * inv_q);
        const double two_inv = 2.0 * inv_sum;
        const double t1 = fma(C.beta, mu, C.visc), t2 = fma(C.beta, mu, t1);
        const double Pi = two_inv * (mu * t1);
        const double dmu = two_inv * t2;  // d Pi / d mu
        const double Pi_vr = vr < 0.0 ? dmu * (P.h * inv_q) : 0.0;

        const double Sw = (c.p + j.p) * w, B = Pi - Sw;
        const double gV = c.gr * j.V, gj = j.gr * c.V;
        const double X = gV - gj, Z = fma(gV, c.rho, gj * j.rho);
        const double diff = c.rho - j.rho, dd = P.dd2 * diff;
        const double all = fma(T, B, fma(dd, X, vr * Z));
        const double KT = K * T;
        const double Kv = fma(KT, Pi_vr, K * Z);                       // along v (x) and r (v)
        const double rad = fma(dK, all, -2.0 * KT * (dmu * mu) * inv_q);  // along r (x)
        const double KB = K * B;
        xb[0] += fma(KB, D0, fma(Kv, v0, rad * r0));
        xb[1] += fma(KB, D1, fma(Kv, v1, rad * r1));
        vb[0] = fma(Kv, r0, vb[0]);
        vb[1] = fma(Kv, r1, vb[1]);
        if constexpr (ND == 3) {
            xb[2] += fma(KB, D2, fma(Kv, v2, rad * r2));
            vb[2] = fma(Kv, r2, vb[2]);
        }
        pb = fma(-KT, w, pb);
        const double dens = fma(P.dd2, X, fma(vr, gV, (dd - vr * j.rho) * (gj * inv_rho)));
        rhob = fma(KT, Sw * inv_rho - Pi * inv_sum, fma(K, dens, rhob));
        alpha = fma(KT, two_inv * mu, alpha);
        delta = fma(K, diff * X, delta);
    }

    // the kernel's constant, common to all pairs
    __device__ __forceinline__ void scale(const DevParams &P)
    {
        const double f = P.kgrad_c;
#pragma unroll
        for (int k = 0; k < ND; k++) {
            xb[k] *= f;
            vb[k] *= f;
        }
        rhob *= f;
        pb *= f;
        alpha *= f;
        delta *= f;
    }
};

// d p / d rho of StateEquationCole (state_equations.jl:100-129), zero where it clips
__host__ __device__ __forceinline__ double dpressure_drho(const DevParams &P, double rho)
{
    const double x = rho / P.rho0;
    if (P.clip_fluid && !(P.B * (pow(x, P.gamma) - 1.0) + P.p_bg > 0.0)) return 0.0;
    return P.B * P.gamma / P.rho0 * pow(x, P.gamma - 1.0);
}

// Every candidate of one particle: its Verlet list (list != nullptr, n >= 0), else the cell
// walk around (x, y, z) with cells grown by hs.  fn(j) applies the exact radius test.  LANES
// lanes share the particle: lane q takes list entries q, q + LANES, ...; the cell walk of an
// overflowed list runs on lane 0 alone.
template <int ND, int LANES = 1, typename Fn>
__device__ __forceinline__ void for_each_candidate(const DevParams &P, const int *__restrict__ list,
                                                   int n, int stride, int col,
                                                   const int *__restrict__ start, double hs,
                                                   double x, double y, double z, int q, Fn &&fn)
{
    if (list && n >= 0) {
        // the next entry is loaded before the current one is evaluated
        int j = q < n ? list[(size_t)q * stride + col] : 0;
        for (int k = q; k < n; k += LANES) {
            const int kn = min(k + LANES, n - 1);
            const int jn = list[(size_t)kn * stride + col];
            fn(j);
            j = jn;
        }
    } else if (q == 0) {
        Pencils<ND> it;
        it.init(P, x, y, z, hs);
        int jb, je;
        while (it.next(P, start, jb, je))
            for (int j = jb; j < je; j++) fn(j);
    }
}

// Sum of v over the LANES lanes of a group (a fixed butterfly: every lane gets the total).
template <int LANES>
__device__ __forceinline__ double group_sum(double v)
{
#pragma unroll
    for (int o = 1; o < LANES; o <<= 1) v += __shfl_xor(v, o);
    return v;
}

// The adjoint weights of the rates in cell-sorted order: kb[s] = {Gbar (3), rbar}.
//   STAGE = false: from a caller's dv_bar (the pullback of one kick);
//   STAGE = true: the reversed stage map, tbar += B ybar, kbar = dt tbar, the drift's
//   vbar += kbar_u, tbar *= A (register adjoints tvb / tub, state adjoints vb / ub).
// GATHER: also the cell-sorted records of the stage's state (v, u) in the order of the last
// rebuild, which stands (the segment is 2D and small more often than not, and then as long as
// its launches take).
template <int ND, bool STAGE, bool GATHER>
__global__ void __launch_bounds__(kBlock)
    k_adj_weights(const DevHandle *__restrict__ H, const double *__restrict__ v,
                  const double *__restrict__ u, const double *__restrict__ dv_bar,
                  double *__restrict__ vb, double *__restrict__ ub, double *__restrict__ tvb,
                  double *__restrict__ tub, double a, double b, double dt,
                  double4 *__restrict__ kb)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= H->P.nf) return;
    const int s = H->iperm[i];
    if constexpr (GATHER) {
        const DevParams P = H->params();
        double x[3] = {0.0, 0.0, 0.0}, vv[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int d = 0; d < ND; d++) {
            x[d] = u[(size_t)i * ND + d];
            vv[d] = v[(size_t)i * (ND + 1) + d];
        }
        const double rho = v[(size_t)i * (ND + 1) + ND], m = H->mass[i];
        H->rec[2 * (size_t)s] = make_double4(x[0], x[1], x[2], rho);
        H->rec[2 * (size_t)s + 1] = make_double4(vv[0], vv[1], vv[2], state_equation(P, rho));
        H->vol[s] = make_double2(m / rho, m);
        // for the cell walks (see k_gather)
        const int *noverflow = H->noverflow;
        if (!noverflow || *noverflow != 0) {
            H->xs[s] = x[0];
            H->ys[s] = x[1];
            if constexpr (ND == 3) H->zs[s] = x[2];
        }
    }
    double k[ND + 1];
    if constexpr (STAGE) {
#pragma unroll
        for (int c = 0; c <= ND; c++) {
            const size_t e = (size_t)i * (ND + 1) + c;
            const double t = fma(b, vb[e], tvb[e]);
            k[c] = dt * t;
            tvb[e] = a * t;
        }
#pragma unroll
        for (int d = 0; d < ND; d++) {
            const size_t e = (size_t)i * ND + d;
            const double t = fma(b, ub[e], tub[e]);
            tub[e] = a * t;
            vb[(size_t)i * (ND + 1) + d] += dt * t;  // drift!: du = v
        }
    } else {
#pragma unroll
        for (int c = 0; c <= ND; c++) k[c] = dv_bar[(size_t)i * (ND + 1) + c];
    }
    kb[s] = make_double4(k[0], k[1], ND == 3 ? k[2] : 0.0, k[ND]);
}

// Adjoint of the Adami pass, four lanes per wall particle (wall-sorted order w): the adjoints
// of p_w and rho_w from the fluid-wall terms of the fluid near w, through the inverse state
// equation and the clipping to the adjoint of the unclipped p_w = N_w / V_w with
//   N_w = sum_f (p_offset + p_f + rho_f g.(x_w - x_f)) W_wf,   V_w = sum_f W_wf,
// stored as coef[w] = {cN, cV}: d L / d N_w = cN, d L / d V_w = cV.  gw[w] accumulates (ACC) or
// takes the partial along g: cN sum_f rho_f ghat.(x_w - x_f) W_wf.
template <int ND, bool ACC>
__global__ void __launch_bounds__(kBlock)
    k_adj_wall(const DevHandle *__restrict__ H, AdjConsts K, const double4 *__restrict__ kb,
               double2 *__restrict__ coef, double *__restrict__ gw)
{
    const DevParams P = H->params();
    const FluidView F = H->fluid();
    const double4 *wpos = H->wpos;
    const double *pw = H->pw, *rhow = H->rhow;
    const double2 *wpv = H->wpv;
    const int *alist = H->anbr, *acnt = H->acnt;
    const int lw = H->lw;
    // four lanes per wall particle (the loop bound is uniform per group of lanes, so the
    // partners shuffle together); lane q takes the list entries q, q + 4, ...
    const int q = threadIdx.x % kAdjLanes;
    const int w = (blockIdx.x * kBlock + (int)threadIdx.x) / kAdjLanes;
    if (w >= P.nw) return;  // whole groups
    const int n = alist ? acnt[w] : -1;
    if (n == 0) {  // no fluid within reach: p_w and rho_w are constants
        if (q == 0) coef[w] = make_double2(0.0, 0.0);
        if (!ACC && q == 0) gw[w] = 0.0;
        return;
    }
    const double4 xw = wpos[w];
    const double p_w = pw[w], rho_w = rhow[w], V_w = wpv[w].y;
    const double inv_rho_w = rcp_pos(rho_w);
    double pbar = 0.0, rbar = 0.0, vol = 0.0, gsum = 0.0;
    for_each_candidate<ND, kAdjLanes>(P, alist, n, lw, w, F.start, P.hs_fluid, xw.x, xw.y, xw.z, q, [&](int j) {
        const double4 a = F.rec[2 * (size_t)j];
        // the Adami pass's difference x_w - x_f
        const double p0 = xw.x - a.x, p1 = xw.y - a.y, p2 = (ND == 3) ? xw.z - a.z : 0.0;
        const double d2 = dist2<ND>(p0, p1, p2);
        if (d2 > P.R2) return;
        const double W = wendland_c2(P, sqrt(d2));
        vol += W;
        double gp = K.ghat[0] * p0 + K.ghat[1] * p1;
        if constexpr (ND == 3) gp += K.ghat[2] * p2;
        gsum += a.w * gp * W;
        if (d2 < P.az2) return;
        const double4 b = F.rec[2 * (size_t)j + 1];
        const double4 g = kb[j];
        const double r[3] = {-p0, -p1, -p2};  // r_ab = x_f - x_w
        const double va[3] = {b.x, b.y, b.z};
        const double G[3] = {g.x, g.y, g.z};
        const WallAdj o = wall_adj<ND>(P, r, d2, va, a.w, rcp_pos(a.w), inv_rho_w, b.w, p_w, V_w, G, g.w);
        pbar += o.p;
        rbar += o.rho_b;
    });
    pbar = group_sum<kAdjLanes>(pbar);
    rbar = group_sum<kAdjLanes>(rbar);
    vol = group_sum<kAdjLanes>(vol);
    gsum = group_sum<kAdjLanes>(gsum);
    if (q != 0) return;
    // inverse state equation: d rho_w / d p_w = rho_w / (gamma (p_w - p_bg + B))
    const double ptot = pbar + rbar * rho_w / (P.gamma * (p_w - P.p_bg + P.B));
    double cN = 0.0, cV = 0.0;
    if (!(P.clip_wall && !(p_w > 0.0))) {
        if (vol > DBL_EPSILON) {
            cN = ptot / vol;
            cV = -ptot * p_w / vol;
        } else {
            cN = ptot;
        }
    }
    coef[w] = make_double2(cN, cV);
    gw[w] = ACC ? gw[w] + cN * gsum : cN * gsum;
}

// The record of sorted particle s from global memory.
template <int ND>
__device__ __forceinline__ AdjRec adj_load(const FluidView &F, const double4 *__restrict__ kb, int s)
{
    const double4 a = F.rec[2 * (size_t)s], b = F.rec[2 * (size_t)s + 1], g = kb[s];
    return {{a.x, a.y, a.z}, a.w, {b.x, b.y, b.z}, b.w, F.vol[s].x, {g.x, g.y, g.z}, g.w};
}

// The wall part of d L / d state_c (list column t, lane q of LANES): c's own fluid-wall terms and
// its part in the Adami sums of the wall particles near it.  The parameters are read again:
// held through the fluid pairs' loop they do not fit the scalar registers.
template <int ND, int LANES>
__device__ __forceinline__ void adj_walls(const DevHandle *handle, const double2 *__restrict__ coef,
                                          int t, int q, AdjTarget<ND> &T)
{
    const DevHandle *H = read_again(handle);
    const DevParams P = H->params();
    const WallView Wv = H->walls();
    const int *wnbr = H->wnbr;
    const int nw = wnbr ? (int)H->wcnt[t] : -1;
    const double *xc = T.c.x, *v_c = T.c.v;
    for_each_candidate<ND, LANES>(P, wnbr, nw, H->ls, t, Wv.start, P.hs_wall, xc[0], xc[1], xc[2], q, [&](int w) {
        const double4 xw = Wv.pos[w];
        double r[3] = {xc[0] - xw.x, xc[1] - xw.y, (ND == 3) ? xc[2] - xw.z : 0.0};
        const double d2 = dist2<ND>(r[0], r[1], r[2]);
        if (d2 > P.R2) return;
        const double2 pv = Wv.pv[w];
        const double2 cf = coef[w];
        // the Adami sums of w: N_w and V_w depend on p_c, rho_c and x_c
        const double dist = sqrt(d2);  // d2 may be 0 here
        const double W = wendland_c2(P, dist);
        const double ww = 1.0 - 0.5 * P.h_inv * dist;
        const double kdrW = dist < P.two_h ? P.kgrad_c * (ww * ww * ww) : 0.0;
        double gx = -(P.g[0] * r[0] + P.g[1] * r[1]);  // g.(x_w - x_c)
        if constexpr (ND == 3) gx -= P.g[2] * r[2];
        T.pb += cf.x * W;
        T.rhob += cf.x * gx * W;
        const double radial = cf.x * ((P.p_offset + T.c.p) + T.c.rho * gx) + cf.y;
#pragma unroll
        for (int k = 0; k < ND; k++) T.xb[k] += -cf.x * T.c.rho * P.g[k] * W + radial * kdrW * r[k];
        if (d2 < P.az2) return;
        // own fluid-wall term (v_w = 0)
        const WallAdj o = wall_adj<ND>(P, r, d2, v_c, T.c.rho, T.inv_rho, pv.y / xw.w, T.c.p, pv.x, pv.y, T.c.G, T.c.gr);
#pragma unroll
        for (int k = 0; k < ND; k++) {
            T.xb[k] += o.r[k];
            T.vb[k] += o.vr * r[k];
        }
        T.rhob += o.rho_a;
        T.pb += o.p;
    });
}

// Sums over the LANES lanes of a target, then the state equation and gravity; lane 0 of an active
// target adds (ACC) or writes d L / d state_c into vb (v, rho) and ub (x) at row i of the
// caller's order, and the partials along alpha, delta and g into th[3 i ..].
template <int ND, int LANES, bool ACC>
__device__ __forceinline__ void adj_finish(const DevHandle *handle, const AdjConsts &K, AdjTarget<ND> &T,
                                           bool write, int i, double *__restrict__ vb,
                                           double *__restrict__ ub, double *__restrict__ th)
{
#pragma unroll
    for (int k = 0; k < ND; k++) {
        T.xb[k] = group_sum<LANES>(T.xb[k]);
        T.vb[k] = group_sum<LANES>(T.vb[k]);
    }
    T.rhob = group_sum<LANES>(T.rhob);
    T.pb = group_sum<LANES>(T.pb);
    T.alpha = group_sum<LANES>(T.alpha);
    T.delta = group_sum<LANES>(T.delta);
    if (!write) return;
    const DevParams P = read_again(handle)->params();
    T.rhob += T.pb * dpressure_drho(P, T.c.rho);
    double gpart = T.c.G[0] * K.ghat[0] + T.c.G[1] * K.ghat[1];  // gravity: dv += g ghat
    if constexpr (ND == 3) gpart += T.c.G[2] * K.ghat[2];
    double *vi = vb + (size_t)i * (ND + 1), *ui = ub + (size_t)i * ND, *ti = th + 3 * (size_t)i;
#pragma unroll
    for (int k = 0; k < ND; k++) {
        vi[k] = ACC ? vi[k] + T.vb[k] : T.vb[k];
        ui[k] = ACC ? ui[k] + T.xb[k] : T.xb[k];
    }
    vi[ND] = ACC ? vi[ND] + T.rhob : T.rhob;
    // half of both terms of every pair (see AdjTarget)
    const double alpha = 0.5 * K.visc_per_alpha * T.alpha, delta = 0.5 * K.dd2_per_delta * T.delta;
    ti[0] = ACC ? ti[0] + alpha : alpha;
    ti[1] = ACC ? ti[1] + delta : delta;
    ti[2] = ACC ? ti[2] + gpart : gpart;
}

// Adjoint of the fluid terms of fluid particle c, four lanes per particle (lane q takes the
// list entries q, q + 4, ...; the partial sums are added across the four lanes in a fixed
// order): its fluid-fluid pairs, its fluid-wall terms and its part in the Adami sums of the
// wall particles near it, the state equation and gravity.
// What bounds it: the gathers of the candidates through the L1 (116 bytes of a record, its volume,
// its weights and its index) at three waves per SIMD.  250k particles in 3D, pullback of one
// kick: 203 us with the two terms of a pair one after the other, 187 with AdjTarget's; held to
// 128 registers (four waves) 48 bytes spill and it takes 29 us more.  Candidates from unions staged in
// LDS brick by brick took 239 us (a block of 512 threads, the FP64 chains of two waves per SIMD
// exposed) and 264 (1,024 threads, which spill). 
template <int ND, bool ACC>
__global__ void __launch_bounds__(kBlock)
    k_adj_fluid(const DevHandle *__restrict__ H, AdjConsts K,
                const double4 *__restrict__ kb, const double2 *__restrict__ coef,
                double *__restrict__ vb, double *__restrict__ ub, double *__restrict__ th)
{
    const DevParams P = H->params();
    const FluidView F = H->fluid();
    const int *ord = H->ord, *nbr = H->nbr, *cnt = H->cnt;
    if (blockIdx.x == 0 && threadIdx.x == 0) *H->flag = 0;  // the rebuild (if any) is done
    const int q = threadIdx.x % kAdjLanes;
    const int tt = (xcd_tile(blockIdx.x, gridDim.x) * kBlock + (int)threadIdx.x) / kAdjLanes;
    // the loop bound is uniform per group of lanes, so the partners shuffle together
    const bool active = tt < P.nf;
    const int t = active ? tt : P.nf - 1;
    const int s = ord ? ord[t] : t;
    AdjTarget<ND> T;
    T.set(adj_load<ND>(F, kb, s));
    const int n = nbr ? cnt[t] : -1;
    auto pair = [&](int j) { T.pair(P, K, adj_load<ND>(F, kb, j)); };
    const int *uidx = H->uidx;
    const int first = uidx ? (int)H->tbase[t] : -1;
    if (first >= 0) {
        // the list of union records of the target's brick (list_place), a row of four entries
        // and their sorted indices one row ahead of the pair terms
        const ushort4 *l4 = reinterpret_cast<const ushort4 *>((const unsigned short *)H->nbr16);
        const int ls = H->ls;
        const int rows = active ? list_rows(n) : 0;
        ushort4 e4 = l4[(size_t)min(q, max(rows - 1, 0)) * ls + t];
        for (int r = q; r < rows; r += kAdjLanes) {
            const ushort4 next = l4[(size_t)min(r + kAdjLanes, rows - 1) * ls + t];
            const int k = list_row_entries(n, r);
            const int j4[4] = {uidx[first + (e4.x >> 4)], k > 1 ? uidx[first + (e4.y >> 4)] : 0,
                               k > 2 ? uidx[first + (e4.z >> 4)] : 0,
                               k > 3 ? uidx[first + (e4.w >> 4)] : 0};
#pragma unroll 1
            for (int i = 0; i < k; i++) pair(i == 0 ? j4[0] : i == 1 ? j4[1] : i == 2 ? j4[2] : j4[3]);
            e4 = next;
        }
    } else {
        for_each_candidate<ND, kAdjLanes>(P, nbr, active ? n : 0, H->ls, t, F.start, P.hs_fluid, T.c.x[0],
                                          T.c.x[1], T.c.x[2], active ? q : kAdjLanes, pair);
    }
    T.scale(P);
    if (P.nw > 0 && active) adj_walls<ND, kAdjLanes>(H, coef, t, q, T);
    adj_finish<ND, kAdjLanes, ACC>(H, K, T, active && q == 0, F.perm[s], vb, ub, th);
}

__global__ void __launch_bounds__(kBlock) k_adj_fill(double *p, size_t n, double value)
{
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock)
        p[i] = value;
}

// Deterministic sums of the parameter partials: block k sums a fixed strided share of the
// fluid partials th (3 per particle) and of the wall partials gw (added to g) with a fixed
// tree; k_adj_sum_final adds the block results with another (one thread after the other took
// 28 us).
__global__ void __launch_bounds__(kBlock)
    k_adj_sum(int nf, const double *__restrict__ th, int nw, const double *__restrict__ gw,
              double *__restrict__ part)
{
    __shared__ double s[3][kBlock];
    double acc[3] = {0.0, 0.0, 0.0};
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < nf; i += gridDim.x * kBlock) {
#pragma unroll
        for (int k = 0; k < 3; k++) acc[k] += th[3 * (size_t)i + k];
    }
    for (int w = blockIdx.x * kBlock + threadIdx.x; w < nw; w += gridDim.x * kBlock) acc[2] += gw[w];
#pragma unroll
    for (int k = 0; k < 3; k++) s[k][threadIdx.x] = acc[k];
    __syncthreads();
    for (int o = kBlock / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
#pragma unroll
            for (int k = 0; k < 3; k++) s[k][threadIdx.x] += s[k][threadIdx.x + o];
        }
        __syncthreads();
    }
    if ((int)threadIdx.x < 3) part[(size_t)blockIdx.x * 3 + threadIdx.x] = s[threadIdx.x][0];
}

__global__ void __launch_bounds__(kRedBlocks)
    k_adj_sum_final(int nparts, const double *__restrict__ part, double *__restrict__ out)
{
    __shared__ double s[3][kRedBlocks];
    const int b = threadIdx.x;
#pragma unroll
    for (int k = 0; k < 3; k++) s[k][b] = b < nparts ? part[(size_t)b * 3 + k] : 0.0;
    __syncthreads();
    for (int o = kRedBlocks / 2; o > 0; o >>= 1) {
        if (b < o) {
#pragma unroll
            for (int k = 0; k < 3; k++) s[k][b] += s[k][b + o];
        }
        __syncthreads();
    }
    if (b < 3) out[b] = s[b][0];
}

int check_supported(tpsph_handle *h)
{
    const tpsph_params &p = h->params;
    if (is_host(h))
        return fail(h, TPSPH_ERR_ARGUMENT, "reverse mode needs device pointers (TPSPH_MEM_DEVICE)");
    if (p.adaptive_sound_speed || p.use_density_diffusion == TPSPH_DIFFUSION_ANTUONO ||
        p.wall_viscosity || p.precision != TPSPH_PRECISION_FP64 ||
        p.density_calculator != TPSPH_DENSITY_CONTINUITY)
        return fail(h, TPSPH_ERR_ARGUMENT,
                    "reverse mode supports ContinuityDensity, StateEquationCole with a fixed "
                    "sound speed, Molteni-Colagrossi or no density diffusion, walls without "
                    "viscosity and FP64");
    return TPSPH_OK;
}

AdjConsts adj_consts(const tpsph_handle *h)
{
    AdjConsts K{};
    const DevParams &P = h->P;
    K.dd2_per_delta = P.use_dd ? 2.0 * P.h * P.c : 0.0;  // Molteni-Colagrossi: dd2 = 2 delta h c
    double g2 = 0.0;
    for (int d = 0; d < 3; d++) g2 += P.g[d] * P.g[d];
    const double g = std::sqrt(g2);
    for (int d = 0; d < 3; d++) K.ghat[d] = g > 0.0 ? P.g[d] / g : 0.0;
    K.visc_per_alpha = P.use_visc ? P.c : 0.0;
    K.visc = P.use_visc ? P.alpha * P.c : 0.0;
    K.beta = P.use_visc ? P.beta : 0.0;
    K.minus_half_h_inv = -0.5 * P.h_inv;
    K.minus_3half_h_inv = -1.5 * P.h_inv;
    return K;
}

int fill(tpsph_handle *h, double *p, size_t n, double value)
{
    if (n == 0) return TPSPH_OK;
    const int grid = (int)std::max<size_t>(1, std::min<size_t>((n + kBlock - 1) / kBlock, 2048));
    hipLaunchKernelGGL(k_adj_fill, dim3(grid), dim3(kBlock), 0, h->stream, p, n, value);
    return launch_check(h, "k_adj_fill");
}

int ensure_buffers(tpsph_handle *h)
{
    if (h->adj_kb) return TPSPH_OK;
    TRY(dalloc(h, &h->adj_kb, (size_t)h->nf));
    TRY(dalloc(h, &h->adj_coef, (size_t)h->nw));
    TRY(dalloc(h, &h->adj_th, 3 * (size_t)h->nf));
    TRY(dalloc(h, &h->adj_gw, (size_t)h->nw));
    TRY(dalloc(h, &h->adj_red, 3 * (size_t)kRedBlocks + 3));
    TRY(dalloc(h, &h->adj_vb, v_len(h)));
    TRY(dalloc(h, &h->adj_ub, u_len(h)));
    TRY(dalloc(h, &h->adj_tvb, v_len(h)));
    TRY(dalloc(h, &h->adj_tub, u_len(h)));
    return TPSPH_OK;
}

int grow(tpsph_handle *h, double **p, size_t *cap, size_t n)
{
    if (*cap >= n) return TPSPH_OK;
    if (*p) HIP_TRY(h, hipFree(*p));
    *p = nullptr;
    *cap = 0;
    TRY(dalloc(h, p, n));
    *cap = n;
    return TPSPH_OK;
}

// The adjoint passes at the state the handle has just prepared: kb must hold the weights.
// Adds (ACC) or writes d L / d (v, u) into vb / ub; the parameter partials go to adj_th /
// adj_gw.
template <int ND, bool ACC>
int adjoint_passes(tpsph_handle *h, double *vb, double *ub)
{
    TimedScope ts(h, TPSPH_TIME_ADJOINT);
    const AdjConsts K = adj_consts(h);
    if (h->nw > 0) {
        hipLaunchKernelGGL((k_adj_wall<ND, ACC>), dim3(nblocks(kAdjLanes * (int64_t)h->nw)), dim3(kBlock), 0, h->stream,
                           h->dev, K, h->adj_kb, h->adj_coef, h->adj_gw);
        TRY(launch_check(h, "k_adj_wall"));
    }
    hipLaunchKernelGGL((k_adj_fluid<ND, ACC>), dim3(nblocks(kAdjLanes * (int64_t)h->nf)), dim3(kBlock), 0, h->stream,
                       h->dev, K, h->adj_kb, h->adj_coef, vb, ub, h->adj_th);
    return launch_check(h, "k_adj_fluid");
}

int reduce_params(tpsph_handle *h, double *param_bar)
{
    const int grid = std::max(1, std::min(nblocks(std::max(h->nf, h->nw)), kRedBlocks));
    hipLaunchKernelGGL(k_adj_sum, dim3(grid), dim3(kBlock), 0, h->stream, h->nf, h->adj_th, h->nw,
                       h->adj_gw, h->adj_red);
    double *res = h->adj_red + 3 * (size_t)kRedBlocks;
    hipLaunchKernelGGL(k_adj_sum_final, dim3(1), dim3(kRedBlocks), 0, h->stream, grid, h->adj_red, res);
    TRY(launch_check(h, "k_adj_sum"));
    if (param_bar) {
        HIP_TRY(h, hipMemcpyAsync(param_bar, res, 3 * sizeof(double), hipMemcpyDefault, h->stream));
        HIP_TRY(h, hipStreamSynchronize(h->stream));
    }
    return TPSPH_OK;
}

template <int ND>
int kick_vjp_impl(tpsph_handle *h, const double *dv_bar, const double *v, const double *u,
                  double *v_bar, double *u_bar, double *param_bar)
{
    TRY(prepare_dispatch(h, v, u));
    hipLaunchKernelGGL((k_adj_weights<ND, false, false>), dim3(nblocks(h->nf)), dim3(kBlock), 0,
                       h->stream, h->dev, nullptr, nullptr, dv_bar, nullptr, nullptr, nullptr, nullptr,
                       0.0, 0.0, 0.0, h->adj_kb);
    TRY(launch_check(h, "k_adj_weights"));
    TRY((adjoint_passes<ND, false>(h, v_bar, u_bar)));
    h->have_kick = false;
    return reduce_params(h, param_bar);
}

template <int ND>
int reverse_impl(tpsph_handle *h, const double *vT_bar, const double *uT_bar, double *v0_bar,
                 double *u0_bar, double *param_bar)
{
    const size_t nv = v_len(h), nu = u_len(h);
    const int64_t every = h->adj_every, nsteps = h->adj_nsteps;
    const int64_t nseg = (nsteps + every - 1) / every;
    // the stage states of one segment, then the working state of its recomputation
    TRY(grow(h, &h->adj_st, &h->adj_st_cap, (size_t)(5 * every + 1) * (nv + nu)));
    double *st_v = h->adj_st, *st_u = h->adj_st + (size_t)5 * every * nv;
    double *wv = st_u + (size_t)5 * every * nu, *wu = wv + nv;
    HIP_TRY(h, hipMemcpyAsync(h->adj_vb, vT_bar, nv * sizeof(double), hipMemcpyDeviceToDevice, h->stream));
    HIP_TRY(h, hipMemcpyAsync(h->adj_ub, uT_bar, nu * sizeof(double), hipMemcpyDeviceToDevice, h->stream));
    TRY(fill(h, h->adj_tvb, nv, 0.0));
    TRY(fill(h, h->adj_tub, nu, 0.0));
    TRY(fill(h, h->adj_th, 3 * (size_t)h->nf, 0.0));
    TRY(fill(h, h->adj_gw, (size_t)h->nw, 0.0));
    for (int64_t k = nseg - 1; k >= 0; k--) {
        const int64_t steps = std::min(every, nsteps - k * every);
        const double *ck = h->adj_ck + (size_t)k * (nv + nu);
        HIP_TRY(h, hipMemcpyAsync(wv, ck, nv * sizeof(double), hipMemcpyDeviceToDevice, h->stream));
        HIP_TRY(h, hipMemcpyAsync(wu, ck + nv, nu * sizeof(double), hipMemcpyDeviceToDevice, h->stream));
        int64_t n0 = 0, n1 = 0;
        TRY(tpsph_rebuild_count(h, &n0));
        TRY(run_ck2n54(h, wv, wu, h->adj_dt, steps, st_v, st_u));
        TRY(tpsph_rebuild_count(h, &n1));
        int moved = 1;
        HIP_TRY(h, hipMemcpyAsync(&moved, h->flag, sizeof(int), hipMemcpyDeviceToHost, h->stream));
        HIP_TRY(h, hipStreamSynchronize(h->stream));
        // no rebuild in the recomputation and the last stored state (which no kick saw) within
        // its skin: every stored state is within the skin of the current lists, so the reverse
        // stages keep the order
        const bool keep_order = n1 == n0 && moved == 0;
        for (int64_t s = steps - 1; s >= 0; s--) {
            for (int i = 4; i >= 0; i--) {
                const size_t e = (size_t)(5 * s + i);
                const double *yv = st_v + e * nv, *yu = st_u + e * nu;
                // (with a rebuild the weights follow it: they go to the new order)
                if (!keep_order) TRY(prepare_dispatch(h, yv, yu));
                const auto weights = keep_order ? k_adj_weights<ND, true, true> : k_adj_weights<ND, true, false>;
                hipLaunchKernelGGL(weights, dim3(nblocks(h->nf)), dim3(kBlock), 0,
                                   h->stream, h->dev, yv, yu, nullptr, h->adj_vb, h->adj_ub,
                                   h->adj_tvb, h->adj_tub, kCkA[i], kCkB[i], h->adj_dt, h->adj_kb);
                TRY(launch_check(h, "k_adj_weights"));
                if (keep_order) TRY(prepare_dispatch(h, yv, yu, true));
                TRY((adjoint_passes<ND, true>(h, h->adj_vb, h->adj_ub)));
            }
        }
    }
    h->have_kick = false;
    HIP_TRY(h, hipMemcpyAsync(v0_bar, h->adj_vb, nv * sizeof(double), hipMemcpyDeviceToDevice, h->stream));
    HIP_TRY(h, hipMemcpyAsync(u0_bar, h->adj_ub, nu * sizeof(double), hipMemcpyDeviceToDevice, h->stream));
    return reduce_params(h, param_bar);
}

}  // namespace

extern "C" {

int tpsph_kick_vjp(tpsph_handle *h, const double *dv_bar, const double *v_ode,
                   const double *u_ode, double t, double *v_bar, double *u_bar,
                   double *param_bar)
{
    (void)t;
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    TRY(check_supported(h));
    if (h->nf == 0) {
        if (param_bar) {
            const double zero[3] = {0.0, 0.0, 0.0};
            HIP_TRY(h, hipMemcpy(param_bar, zero, sizeof(zero), hipMemcpyDefault));
        }
        return TPSPH_OK;
    }
    if (!dv_bar || !v_ode || !u_ode || !v_bar || !u_bar)
        return fail(h, TPSPH_ERR_ARGUMENT, "dv_bar, v_ode, u_ode, v_bar and u_bar must not be NULL");
    TRY(ensure_buffers(h));
    return h->nd == 2 ? kick_vjp_impl<2>(h, dv_bar, v_ode, u_ode, v_bar, u_bar, param_bar)
                      : kick_vjp_impl<3>(h, dv_bar, v_ode, u_ode, v_bar, u_bar, param_bar);
}

int tpsph_adjoint_forward(tpsph_handle *h, const double *v0_ode, const double *u0_ode,
                          double t0, double dt, int64_t nsteps, int64_t checkpoint_every,
                          double *v_ode, double *u_ode)
{
    (void)t0;
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    TRY(check_supported(h));
    if (nsteps < 0) return fail(h, TPSPH_ERR_ARGUMENT, "nsteps must be non-negative");
    if (checkpoint_every < 1) return fail(h, TPSPH_ERR_ARGUMENT, "checkpoint_every must be at least 1");
    if (h->nf > 0 && (!v0_ode || !u0_ode || !v_ode || !u_ode))
        return fail(h, TPSPH_ERR_ARGUMENT, "v0_ode, u0_ode, v_ode and u_ode must not be NULL");
    h->adj_ready = false;
    if (h->nf == 0) {
        h->adj_nsteps = nsteps;
        h->adj_every = checkpoint_every;
        h->adj_dt = dt;
        h->adj_ready = true;
        return TPSPH_OK;
    }
    TRY(ensure_buffers(h));
    const size_t nv = v_len(h), nu = u_len(h);
    const int64_t nseg = (nsteps + checkpoint_every - 1) / checkpoint_every;
    TRY(grow(h, &h->adj_ck, &h->adj_ck_cap, (size_t)std::max<int64_t>(nseg, 1) * (nv + nu)));
    if (v_ode != v0_ode)
        HIP_TRY(h, hipMemcpyAsync(v_ode, v0_ode, nv * sizeof(double), hipMemcpyDeviceToDevice, h->stream));
    if (u_ode != u0_ode)
        HIP_TRY(h, hipMemcpyAsync(u_ode, u0_ode, nu * sizeof(double), hipMemcpyDeviceToDevice, h->stream));
    for (int64_t k = 0; k < nseg; k++) {
        double *ck = h->adj_ck + (size_t)k * (nv + nu);
        HIP_TRY(h, hipMemcpyAsync(ck, v_ode, nv * sizeof(double), hipMemcpyDeviceToDevice, h->stream));
        HIP_TRY(h, hipMemcpyAsync(ck + nv, u_ode, nu * sizeof(double), hipMemcpyDeviceToDevice, h->stream));
        TRY(run_ck2n54(h, v_ode, u_ode, dt, std::min(checkpoint_every, nsteps - k * checkpoint_every),
                       nullptr, nullptr));
    }
    h->adj_nsteps = nsteps;
    h->adj_every = checkpoint_every;
    h->adj_dt = dt;
    h->adj_ready = true;
    return TPSPH_OK;
}

int tpsph_adjoint_reverse(tpsph_handle *h, const double *v_bar, const double *u_bar,
                          double *v0_bar, double *u0_bar, double *param_bar)
{
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    TRY(check_supported(h));
    if (!h->adj_ready)
        return fail(h, TPSPH_ERR_STATE, "no trajectory stored: call tpsph_adjoint_forward first");
    if (h->nf == 0) {
        if (param_bar) {
            const double zero[3] = {0.0, 0.0, 0.0};
            HIP_TRY(h, hipMemcpy(param_bar, zero, sizeof(zero), hipMemcpyDefault));
        }
        return TPSPH_OK;
    }
    if (!v_bar || !u_bar || !v0_bar || !u0_bar)
        return fail(h, TPSPH_ERR_ARGUMENT, "v_bar, u_bar, v0_bar and u0_bar must not be NULL");
    return h->nd == 2 ? reverse_impl<2>(h, v_bar, u_bar, v0_bar, u0_bar, param_bar)
                      : reverse_impl<3>(h, v_bar, u_bar, v0_bar, u0_bar, param_bar);
}

}  // extern "C"
