// tpsph_mixed.hip -- the fluid-fluid pass of the mixed-precision right-hand side
// (tpsph_params.precision == TPSPH_PRECISION_MIXED).
//
// The same bricks, unions and 16-bit LDS lists as k_fluid_brick (tpsph.hip), with the pair
// arithmetic in FP32:
//   - positions are staged relative to the centre of the brick (FP64 difference, rounded
//     once to FP32), so the pair differences carry the FP32 error of coordinates of a few R
//     instead of the domain's extent;
//   - densities are staged as rho - rho0 (FP64 difference, rounded once), so the
//     Molteni-Colagrossi term rho_a - rho_b keeps its relative precision;
//   - the density rate is summed with Kahan's compensated summation (one compensated add per
//     group of four list slots); the factors common to a target's pairs multiply the finished
//     sums in FP64, and the two lanes of a target combine their (sum,
//     compensation) pairs in FP64;
//   - FP64 stays where it is: the state, the state equation (pressures come from the FP64
//     density of the stage kernel), the wall sums (k_fluid_walls), the Adami pass, the
//     stage update and the written dv / drho.
// Bricks that do not stage (a union beyond the LDS records, an overflowed list) run the FP64
// terms from global memory in k_fluid_brick_global.
//
// LDS: 36 bytes per record (two float4 and one float) instead of 72, so two blocks of 1024
// threads share a CU and one block's staging overlaps the other's pair terms.
#include "tpsph_internal.h"

using namespace tpsph;

namespace {

constexpr float kFar32 = 1e18f;  // coordinate of the far record: d^2 = 1e36 stays finite

template <int ND>
struct BrickSmem32 {
    // (vol first: the fields of a record lie at constant offsets from 16 times its number)
    float vol[kBrickCap];  // V = m / rho
    float4 pa[kBrickCap];  // {x, y, z, rho - rho0} relative to the brick centre
    float4 pb[kBrickCap];  // {vx, vy, vz, p}
    int item;
    double org[3];         // the brick centre
};

// What the FP32 pass needs, packed small so that it stays in scalar registers: the pair
// constants in FP32 and the brick geometry in FP64.  Under StateEquationAdaptiveCole the
// viscosity and diffusion constants of this kick are read from dyn ({c, B, alpha c h,
// 2 delta h c}, written by the gather).
struct Pair32 {
    float az2, minus_half_h_inv, eps_h2, two_av_c, dd2, rho0;
    int use_visc;
    int nb0, nb1, bc[3];
    double lo[3], cs[3], g[3], rho0_64, kgrad_c;
    const double *dyn;
};

Pair32 pair32(const DevParams &P)
{
    Pair32 q;
    q.az2 = (float)P.az2;
    q.minus_half_h_inv = (float)(-0.5 * P.h_inv);
    // (at least az2: with epsilon = 0 or no viscosity the reciprocal of a coincident pair is finite)
    q.eps_h2 = std::fmax((float)P.eps_h2, q.az2);
    q.two_av_c = P.use_visc ? (float)(2.0 * P.av_c) : 0.0f;
    q.dd2 = (float)P.dd2;
    q.rho0 = (float)P.rho0;
    q.use_visc = P.use_visc;
    q.nb0 = P.nb[0];
    q.nb1 = P.nb[1];
    for (int d = 0; d < 3; d++) {
        q.bc[d] = P.bc[d];
        q.lo[d] = P.lo[d];
        q.cs[d] = P.cs[d];
        q.g[d] = P.g[d];
    }
    q.rho0_64 = P.rho0;
    q.kgrad_c = P.kgrad_c;
    q.dyn = P.dyn;
    return q;
}

// Kahan's compensated sum: s + c carries the running total, c the negated rounding error.
struct Kahan {
    float s = 0.0f, c = 0.0f;
    __device__ __forceinline__ void add(float x)
    {
        const float y = x - c;
        const float t = s + y;
        c = (t - s) - y;
        s = t;
    }
};

// A target of the pair loop and its terms in FP32, in the form of BrickTarget (tpsph.hip): with
// k = (1 - r / 2h)^3 of a pair the sums are
//   acc  += V_b k [-(p_a + p_b) + 2 alpha c h rho_a rho_b min(v_ab.r_ab, 0) /
//                  ((r^2 + eps h^2)(rho_a + rho_b))] r_ab
//   part += V_b k [2 delta h c (rho_a - rho_b) + rho_a v_ab.r_ab]
// and the range test is the clamp of 1 - r / 2h, with a NaN in place of an r^2 below az2
// (max(NaN, 0) = 0); the far record has no volume.  acc and part are the plain sums of one
// list row (at most four terms), which the caller adds to the totals.
template <int ND>
struct Target32 {
    float x[3], v[3], drho, rho, p, visc;

    __device__ __forceinline__ Target32(const Pair32 &q, const float4 &a, const float4 &b)
        : x{a.x, a.y, a.z}, v{b.x, b.y, b.z}, drho(a.w), rho((float)(q.rho0_64 + (double)a.w)),
          p(b.w), visc(q.two_av_c * rho)
    {
    }

    __device__ __forceinline__ void add(const Pair32 &q, const float4 &a, const float4 &b,
                                        float V_b, float *acc, float &part) const
    {
        const float p0 = x[0] - a.x, p1 = x[1] - a.y, p2 = (ND == 3) ? x[2] - a.z : 0.0f;
        float d2 = p0 * p0 + p1 * p1;
        if constexpr (ND == 3) d2 = d2 + p2 * p2;
        const float near = d2 >= q.az2 ? d2 : __builtin_nanf("");
        const float r = near * __builtin_amdgcn_rsqf(near);
        const float w = __builtin_fmaxf(__builtin_fmaf(q.minus_half_h_inv, r, 1.0f), 0.0f);
        const float Vk = V_b * (w * w * w);
        const float v0 = v[0] - b.x, v1 = v[1] - b.y, v2 = (ND == 3) ? v[2] - b.z : 0.0f;
        float vr = v0 * p0 + v1 * p1;
        if constexpr (ND == 3) vr = vr + v2 * p2;
        const float rho_b = q.rho0 + a.w;
        const float num = visc * (rho_b * __builtin_fminf(vr, 0.0f));
        float f = __builtin_fmaf(num, __builtin_amdgcn_rcpf((d2 + q.eps_h2) * (rho + rho_b)), -(p + b.w));
        f *= Vk;
        acc[0] = __builtin_fmaf(f, p0, acc[0]);
        acc[1] = __builtin_fmaf(f, p1, acc[1]);
        if constexpr (ND == 3) acc[2] = __builtin_fmaf(f, p2, acc[2]);
        part = __builtin_fmaf(Vk, __builtin_fmaf(q.dd2, drho - a.w, rho * vr), part);
    }
};

__device__ __forceinline__ float4 lds_at(const float4 *p, int e16)
{
    return *reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(p) + e16);
}
__device__ __forceinline__ float lds_at(const float *p, int e16)
{
    return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(p) + (e16 >> 2));
}

// Fluid-fluid pass over the staged bricks, one block of kBrickThreads per brick taken from
// the work counter work[0] (two blocks per CU).
// What bounds it: the VALU (FP32 terms issue at the FP64 rate, a candidate of 75 instructions was
// 285 of 332 us at 2M particles).  The factored terms of Target32, two candidates a step without
// selects between them and the targets' own records from the staged union took it to 291 us,
// and 299 with the velocity sums row by row, which keeps the error against FP64 at the plain
// form's (rows summed in FP64: 320, the registers run out).
// Bricks that do not stage are listed in bfall
// (work[1] of them) for k_fluid_brick_global (FP64, global memory), launched after this
// kernel.
template <int ND>
__global__ void __launch_bounds__(kBrickThreads, 8)
    k_fluid_brick32(const DevHandle *__restrict__ H, Pair32 q, double *__restrict__ dv)
{
    const FluidView F = H->fluid();
    const int *nel = H->nel, *uidx = H->uidx;
    const int4 *bhead = H->bhead;
    const int2 *thead = H->thead;
    const unsigned short *nbr16 = H->nbr16;
    const int *nne = H->counters;
    int *work = H->bwork, *bfall = H->bfall;
    const int ls = H->ls;
    if (q.dyn) {  // the sound speed of this kick
        q.two_av_c = q.use_visc ? (float)(2.0 * q.dyn[2]) : 0.0f;
        q.dd2 = (float)q.dyn[3];
    }
    __shared__ BrickSmem32<ND> S;
    const int tid = threadIdx.x;
    if (blockIdx.x == 0 && tid == 0) *H->flag = 0;  // the rebuild (if any) is done
    const int ne = *nne;
    while (true) {
        if (tid == 0) S.item = atomicAdd(work, 1);
        __syncthreads();
        const int item = S.item;
        if (item >= ne) break;
        const int b = nel[item];
        const int4 hd = bhead[item];
        const int ntot = hd.z;
        if (ntot > kBrickCap - 1) {  // left to the FP64 pass (uniform per block)
            if (tid == 0) bfall[atomicAdd(&work[1], 1)] = item;
        } else {
            const int t0 = hd.x, t1 = hd.y;
            if (tid == 0) {
                const int bx = b % q.nb0, by = (b / q.nb0) % q.nb1, bz = b / (q.nb0 * q.nb1);
                const int bc[3] = {bx, by, bz};
#pragma unroll
                for (int d = 0; d < 3; d++)
                    S.org[d] = d < ND ? q.lo[d] + (bc[d] * q.bc[d] + 0.5 * q.bc[d]) * q.cs[d] : 0.0;
                constexpr int f = kBrickCap - 1;  // the far record
                S.pa[f] = make_float4(kFar32, kFar32, kFar32, 0.0f);
                S.pb[f] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                S.vol[f] = 0.0f;
            }
            __syncthreads();
            const double o0 = S.org[0], o1 = S.org[1], o2 = S.org[2];
            for (int i = tid; i < ntot; i += kBrickThreads) {
                const int g = uidx[hd.w + i];
                const double4 a = F.rec[2 * (size_t)g];
                const double4 c = F.rec[2 * (size_t)g + 1];
                S.pa[i] = make_float4((float)(a.x - o0), (float)(a.y - o1),
                                      ND == 3 ? (float)(a.z - o2) : 0.0f, (float)(a.w - q.rho0_64));
                S.pb[i] = make_float4((float)c.x, (float)c.y, ND == 3 ? (float)c.z : 0.0f, (float)c.w);
                S.vol[i] = (float)F.vol[g].x;
            }
            __syncthreads();
            // two lanes per target take alternate rows of the list
            const int half = tid & 1;
            const ushort4 *l4 = reinterpret_cast<const ushort4 *>(nbr16);
            for (int base = t0; base < t1; base += kBrickThreads / 2) {
                const int t = base + (tid >> 1);
                const bool active = t < t1;
                const int col = active ? t : t0;
                const int2 th = thead[col];
                ushort4 cur4 = l4[(size_t)half * ls + col];
                const int self = (th.y & (kBrickCap - 1)) * 16;
                const int m = active ? (th.y >> kHeadCount) & kHeadCountMask : 0;
                const Target32<ND> T(q, lds_at(S.pa, self), lds_at(S.pb, self));
                float acc[3] = {0.0f, 0.0f, 0.0f};
                Kahan drho;
                const int rows = list_rows(m);
                for (int r = half; r < rows; r += 2) {
                    // list rows clamped into the list rather than selected (a select made the
                    // compiler issue flat loads, whose waits hold up the LDS reads)
                    const ushort4 nxt4 = l4[(size_t)min(r + 2, rows - 1) * ls + col];
                    float row[3] = {0.0f, 0.0f, 0.0f}, part = 0.0f;
                    // two candidates at a time; entries past the list are the far record's
                    auto two = [&](int ea, int eb) {
                        const float4 a0 = lds_at(S.pa, ea), b0 = lds_at(S.pb, ea);
                        const float4 a1 = lds_at(S.pa, eb), b1 = lds_at(S.pb, eb);
                        const float V0 = lds_at(S.vol, ea), V1 = lds_at(S.vol, eb);
                        T.add(q, a0, b0, V0, row, part);
                        T.add(q, a1, b1, V1, row, part);
                    };
                    two(cur4.x, cur4.y);
                    if (list_row_entries(m, r) > 2) two(cur4.z, cur4.w);
#pragma unroll
                    for (int d = 0; d < ND; d++) acc[d] += row[d];  // (a row at a time: fewer roundings)
                    drho.add(part);
                    cur4 = nxt4;
                }
                // the partner's sums in FP64, the compensation folded in
                const double f = q.kgrad_c / (q.rho0_64 + (double)T.drho);
                double acc64[3] = {f * (double)acc[0], f * (double)acc[1], f * (double)acc[2]};
                double drho64 = q.kgrad_c * ((double)drho.s - (double)drho.c);
#pragma unroll
                for (int d = 0; d < 3; d++) acc64[d] += __shfl_xor(acc64[d], 1);
                drho64 += __shfl_xor(drho64, 1);
                if (active && half == 0) {
                    double *o = dv + (size_t)th.x * (ND + 1);
                    const bool walls = (th.y & kHeadWalls) != 0;  // k_fluid_walls adds the wall sum, then gravity
#pragma unroll
                    for (int d = 0; d < ND; d++) o[d] = walls ? acc64[d] : acc64[d] + q.g[d];
                    o[ND] = drho64;
                }
            }
        }
        __syncthreads();  // the LDS is staged again for the next brick
    }
}

}  // namespace

int tpsph::launch_fluid_brick_mixed(tpsph_handle *h, double *dv)
{
    const int grid = std::max(1, std::min(h->nbricks, 2 * h->n_cu));
    const auto kernel = h->nd == 2 ? k_fluid_brick32<2> : k_fluid_brick32<3>;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBrickThreads), 0, h->stream, h->dev, pair32(h->P), dv);
    return launch_check(h, "k_fluid_brick32");
}
