// tpsph.hip -- MI355X (gfx950) WCSPH right-hand side behind the C ABI of include/tpsph.h.
//
// One kick! (semidiscretization.jl:589-612) runs, on the handle's stream:
//   1. k_gather<0>   gather the fluid state into cell-sorted order with the current
//                    permutation, fluid state equation, and flag a rebuild if any particle
//                    moved by more than half the skin since the last cell-list build;
//   2. rebuild, only when flagged (every kernel reads the flag and returns otherwise; the
//      fluid kernel of step 4 lowers the flag again): k_links + k_scan + k_gather<1> (a stable
//      counting sort on the linear cell index that gathers again, with a snapshot of the build
//      positions; one kernel, k_sort, for small fluids) and, with Verlet lists, k_brick_lists (bricks, unions,
//      fluid and wall candidates within R + skin);
//   3. the Adami pressure extrapolation + inverse state equation per wall particle (adami_pass):
//      with Verlet lists in the launch of k_brick_lists, otherwise k_wall;
//   4. the fused fluid-fluid + fluid-wall interaction + gravity, results scattered back to
//      the caller's particle order: k_fluid_brick + k_fluid_walls (Verlet lists with the
//      candidates staged brick by brick in LDS), k_fluid_list (Verlet lists) or k_fluid
//      (cell walk).
// The wall cell list is static and built once at create.
//
// Neighbour search.  Cells have edge R/k (k = cell_divisions, R = compact support 2h).  For
// a target at x_a the candidate cells are enumerated as x-rows ("pencils") of cells: for
// every (y, z) cell pair the transverse distance d_t from x_a to the pencil (cell interval
// grown by half the skin) prunes the pencil when d_t > R, and otherwise only the x-cells
// within sqrt(R^2 - d_t^2) + skin/2 of x_a are visited -- one contiguous range of the
// cell-sorted arrays.  Border cells extend to infinity outwards, so clamped particles
// (outside the grid box) are always visited.  Every candidate then passes the exact test
// d^2 = (dx*dx + dy*dy) + dz*dz <= R^2 (FP contraction off, the oracle's evaluation order),
// so the neighbour relation is exactly the reference's.
//
// Pair evaluation.  k_fluid is two-phase per wavefront: phase 1 runs the exact radius test
// over the candidates and appends hits to a per-lane list in LDS (kCap entries per lane);
// phase 2 evaluates the pair terms on the dense lists.  Phases alternate until every lane
// has exhausted its pencils, so any neighbour count is handled.  k_fluid_list streams the
// Verlet lists instead (about 1.1x the neighbour count per particle, read as contiguous
// 256-byte rows per wavefront) and applies the same exact test to every entry.
#include "tpsph_internal.h"

#include <mutex>

namespace tpsph {
thread_local std::string g_create_error;
}  // namespace tpsph

using namespace tpsph;

namespace {


// ------------------------------------------------------------------------------------------
// cell list (counting sort), every kernel gated by the rebuild flag (nullptr = always)
// ------------------------------------------------------------------------------------------

template <int ND>
__device__ __forceinline__ int cell_of(const DevParams &P, double x0, double x1, double x2)
{
    const int c0 = cell_1d(x0, P.lo[0], P.inv_cs[0], P.n[0]);
    const int c1 = cell_1d(x1, P.lo[1], P.inv_cs[1], P.n[1]);
    const int c2 = (ND == 3) ? cell_1d(x2, P.lo[2], P.inv_cs[2], P.n[2]) : 0;
    return c0 + P.n[0] * (c1 + P.n[1] * c2);
}

template <int ND>
__global__ void k_cells(const DevHandle *__restrict__ H, const int *flag, int n,
                        const double *__restrict__ x, int *__restrict__ cell,
                        int *__restrict__ rank, int *__restrict__ count)
{
    if (skip(flag)) return;
    const DevParams P = H->params();
    clear_scan_state(H->scan_state, H->scan_words, blockIdx.x, gridDim.x);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const double *xi = x + (size_t)i * ND;
        const int c = cell_of<ND>(P, xi[0], xi[1], ND == 3 ? xi[2] : 0.0);
        cell[i] = c;
        rank[i] = atomicAdd(&count[c], 1);
    }
}

// The fluid's cells as chains: head[c] is the member of cell c that came last, next[i] the one
// before i; count[c] of them belong to the cell, whatever head and the first member's next held
// before (so neither is ever cleared).  k_gather<1> finds a particle's place by the chain and
// the scanned counts, without the two passes that write and order the members of every cell.
// Also clears the scan's state and the list build's counters.  Block bx of nb.
template <int ND>
__device__ __forceinline__ void links_body(const DevHandle *H, int bx, int nb, const double *__restrict__ x)
{
    const DevParams P = H->params();
    int *head = H->f_head, *next = H->f_next, *count = H->f_count, *counters = H->counters;
    clear_scan_state(H->scan_state, H->scan_words, bx, nb);
    if (counters && bx == 0 && (int)threadIdx.x < kCounters) counters[threadIdx.x] = 0;
    for (int i = bx * (int)blockDim.x + (int)threadIdx.x; i < P.nf; i += nb * (int)blockDim.x) {
        const double *xi = x + (size_t)i * ND;
        const int c = cell_of<ND>(P, xi[0], xi[1], ND == 3 ? xi[2] : 0.0);
        atomicAdd(&count[c], 1);
        next[i] = atomicExch(&head[c], i);
    }
}

template <int ND>
__global__ void k_links(const DevHandle *__restrict__ H, const double *__restrict__ x)
{
    if (skip(H->flag)) return;
    links_body<ND>(H, blockIdx.x, gridDim.x, x);
}

// ------------------------------------------------------------------------------------------
// gather into cell-sorted order + fluid state equation (wcsph/system.jl:426-438)
//   MODE 0: runs when no rebuild is pending; flags one if a particle left its skin.  A block
//           that starts after another block raised the flag returns early: the rebuild that
//           follows gathers everything again.
//   MODE 1: runs at a rebuild; stores the build positions.
//   MODE 2: the same with a finished permutation (tpsph_kick_noalloc).
// ------------------------------------------------------------------------------------------
// MODE 1 puts particle i behind the members of its cell with a smaller index (the stable counting
// sort, whatever order the atomics of k_links were served in), which it counts along the cell's
// chain.  With bcount it also counts the particles of every brick of cells and lists the bricks
// that hold any (nel, nne of them; k_links cleared it).
// The counters of the brick kernels (work) and of k_sort, cleared by the first kernel of every kick
__device__ __forceinline__ void reset_counters(int *work, int *sort_ctl)
{
    if (work && threadIdx.x < 3) work[threadIdx.x] = 0;
    if (sort_ctl && threadIdx.x < kSortCtl) sort_ctl[threadIdx.x] = 0;
}

// FP32 position for the list builds: relative to the grid origin, clamped to one box length beyond
// the grid box on every side.  Clamping brings no two points further apart, so the FP32 test
// leaves out no neighbour, and a particle farther out (or without a position: NaN) is no
// candidate of the particles in the box.  (With every candidate of a particle outside the box
// listed, lists overflowed: 45k particles in 2D, the upper half outside: 1182 us per kick, 31 so.)
template <int ND>
__device__ __forceinline__ float4 list_f32(const DevParams &P, double x0, double x1, double x2)
{
    const double x[3] = {x0, x1, x2};
    float c[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < ND; d++) c[d] = (float)fmin(fmax(x[d] - P.lo[d], -P.box[d]), 2.0 * P.box[d]);
    return make_float4(c[0], c[1], c[2], 0.f);
}

template <int ND>
__global__ void k_wall_f32(DevParams P, int nw, const double4 *__restrict__ wpos,
                           float4 *__restrict__ wxf)
{
    const int w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= nw) return;
    const double4 x = wpos[w];
    wxf[w] = list_f32<ND>(P, x.x, x.y, x.z);
}

// StateEquationAdaptiveCole: the sound speed of this kick from the nparts block maxima of v.v that
// k_vmax left, c = min(c_max, max(c_min, sqrt(max v.v) / Ma)), and the constants that depend on
// it, computed as tpsph_create computes them from a fixed c.  Every block of the gather takes the
// maximum itself (at most kGateBlocks numbers) and the first one writes dyn for the kernels that
// follow: a kernel of one block between k_vmax and the gather took 2.2 us and its launch (kick at
// rest with it -> so, 48k particles in 3D 50.1 -> 49.1 us, 250k 108.1 -> 107.7, 913k 265 -> 265).
__device__ __forceinline__ void adaptive_sound(const DevHandle *H, DevParams &P, int nparts, bool write)
{
    __shared__ double s[kBlock / 64];
    const double *part = H->vmax_part;
    double m = 0.0;
    for (int i = threadIdx.x; i < nparts; i += kBlock) m = fmax(m, part[i]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kBlock / 64; w++) m = fmax(m, s[w]);
    const double c = fmin(P.c_max, fmax(P.c_min, sqrt(m) / P.mach));
    P.c = c;
    P.B = P.rho0 * (c * c) / P.gamma;
    if (write && threadIdx.x == 0) {
        double *dyn = H->dyn;
        dyn[0] = c;
        dyn[1] = P.B;
        dyn[2] = H->alpha * c * P.h;
        dyn[3] = P.use_dd ? 2.0 * H->delta * P.h * c : 0.0;
    }
}

// nparts: adaptive_sound (MODE 0 with an adaptive sound speed, blocks of kBlock threads), or 0.
template <int ND, int MODE>
__device__ __forceinline__ void gather_body(const DevHandle *H, int bx, int nb,
                                            const double *__restrict__ u,
                                            const double *__restrict__ v, int nparts = 0)
{
    DevParams P = H->params();
    int *flag = H->flag, *work = H->bwork, *iperm = H->iperm, *perm = H->f_perm;
    const double *m = H->mass;
    double *xs = H->xs, *ys = H->ys, *zs = H->zs, *snap = H->snap;
    double4 *rec = H->rec;
    double2 *vol = H->vol;
    const int *start = H->f_start, *head = H->f_head, *next = H->f_next, *noverflow = H->noverflow;
    int *bcount = H->bcount, *nel = H->nel, *nne = H->counters;
    float4 *xf = H->xf;
    if (MODE == 0 && nparts > 0)
        adaptive_sound(H, P, nparts, bx == 0);
    else
        P = with_sound(P);
    const int f = *flag;
    // MODE 0 runs first in every kick: it resets the counters of the kernels that follow
    if (MODE == 0 && bx == 0) reset_counters(work, H->sort_ctl);
    if ((MODE == 0) == (f != 0)) return;
    const size_t nf = (size_t)P.nf;
    // with Verlet lists the SoA coordinates are read between rebuilds only by the cell walk
    // of overflowed lists (noverflow counts them; nullptr = always needed)
    const bool soa = !noverflow || *noverflow != 0;
    // the loop bound is uniform per wavefront (blockDim is a multiple of 64): the brick
    // counting below works on whole wavefronts
    for (int s0 = bx * (int)blockDim.x; s0 < P.nf; s0 += nb * (int)blockDim.x) {
        int s = s0 + (int)threadIdx.x;
        const bool in = s < P.nf;
        int b = -1;          // brick of the particle (at a rebuild with bcount)
        bool moved = false;  // left its skin (MODE 0)
        if (in) {
            const int i = MODE == 1 ? s : perm[s];
            double x[3] = {0.0, 0.0, 0.0}, vv[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int d = 0; d < ND; d++) {
                x[d] = u[(size_t)i * ND + d];
                vv[d] = v[(size_t)i * P.vrows + d];
            }
            if constexpr (MODE == 1) {
                const int c = cell_of<ND>(P, x[0], x[1], x[2]);
                const int b0 = start[c], members = start[c + 1] - b0;
                s = b0;
                for (int k = 0, j = head[c]; k < members; k++) {
                    s += j < i ? 1 : 0;
                    if (k + 1 < members) j = next[j];
                }
                perm[s] = i;
            }
            // SummationDensity: density and pressure are written by k_sum_finish
            const double rho = P.summation ? 1.0 : v[(size_t)i * (ND + 1) + ND];
            const double mass = m[i];
            if (MODE != 0 || soa) {
                xs[s] = x[0];
                ys[s] = x[1];
                if constexpr (ND == 3) zs[s] = x[2];
            }
            rec[2 * (size_t)s] = make_double4(x[0], x[1], x[2], rho);
            rec[2 * (size_t)s + 1] = make_double4(vv[0], vv[1], vv[2], state_equation(P, rho));
            vol[s] = make_double2(mass / rho, mass);
            if constexpr (MODE == 0) {
                // Euclidean displacement since the build (bounds the per-axis drift the grown
                // cells allow for, and the drift the Verlet lists allow for)
                double e2 = 0.0;
#pragma unroll
                for (int d = 0; d < ND; d++) {
                    const double e = x[d] - snap[d * nf + s];
                    e2 = fma(e, e, e2);
                }
                moved = !(e2 <= P.half_skin2);
            } else {
#pragma unroll
                for (int d = 0; d < ND; d++) snap[d * nf + s] = x[d];
                iperm[i] = s;
                if (xf) xf[s] = list_f32<ND>(P, x[0], x[1], x[2]);
                if (bcount) {
                    const int c0 = cell_1d(x[0], P.lo[0], P.inv_cs[0], P.n[0]);
                    const int c1 = cell_1d(x[1], P.lo[1], P.inv_cs[1], P.n[1]);
                    const int c2 = (ND == 3) ? cell_1d(x[2], P.lo[2], P.inv_cs[2], P.n[2]) : 0;
                    b = c0 / P.bc[0] + P.nb[0] * (c1 / P.bc[1] + P.nb[1] * (c2 / P.bc[2]));
                }
            }
        }
        if constexpr (MODE == 0) raise_rebuild_flag(flag, moved);
        if (MODE != 0 && bcount) {
            // neighbouring particles mostly share a brick, so equal bricks come in runs: the first lane of a run adds the run with one atomic, and whoever finds a
            // brick empty lists it
            const int lane = (int)threadIdx.x & 63;
            const int prev = __shfl_up(b, 1);
            const bool head = lane == 0 || b != prev;
            const unsigned long long heads = __ballot(head);
            const unsigned long long after = heads & ~((2ull << lane) - 1);
            const int end = after ? __ffsll((long long)after) - 1 : 64;
            if (head && b >= 0 && atomicAdd(&bcount[b], end - lane) == 0)
                nel[atomicAdd(nne, 1)] = b;
        }
    }
    if (MODE != 0 && H->nrebuild && bx == 0 && threadIdx.x == 0) *H->nrebuild += 1;
}

template <int ND, int MODE>
__global__ void k_gather(const DevHandle *__restrict__ H, const double *__restrict__ u,
                         const double *__restrict__ v, int nparts)
{
    gather_body<ND, MODE>(H, blockIdx.x, gridDim.x, u, v, nparts);
}

// k_links, k_scan and k_gather<1> in one launch, which like theirs returns at once while the flag
// is down: a launch costs a kick of a small fluid 2.5 us, whether it does anything or not.
//
// Items are handed out by a ticket in the order of the phases (`items` of the particles, `tiles`
// of the scan, `items` of the gather), and an item waits until every item of the phase before
// is done.  Those are in the hands of blocks that run already and that wait for still earlier
// phases only, so the waits end whatever number of blocks the device holds at a time.  What a
// phase wrote is released by its block at device scope and acquired by the waiting one.
//
// A kick without a rebuild saves two launches, one with a rebuild is longer than with three kernels
// (each phase waits for tickets, counts and cold caches, and 64 blocks scan the cells).  us per
// kick, three kernels -> this one, at rest and rebuilding every time, over the cells of the grid:
//                      0.2M                     1M            2M            4M            20M
//   1,800 in 2D    21.2 -> 14.2, 41 -> 48    46 -> 51      50 -> 62      55 -> 84     113 -> 256
//   45k in 2D      22.1 -> 17.7, 58 -> 67    64 -> 70      66 -> 83      73 -> 105    127 -> 270
//   48k in 3D      33.5 -> 29.7, 101 -> 111  107 -> 115    122 -> 137    127 -> 158   183 -> 323
//   125k in 3D     60.9 -> 56.6, 154 -> 167  152 -> 165    155 -> 177    160 -> 198   224 -> 372
// (at rest the cells do not matter).  The line lies at three turns of the blocks over the scan's
// tiles, kSortMaxCells: there a rebuild costs what four kicks without one save.  Larger fluids
// (kSortMax) take the three kernels too: their rebuild needs the whole device (1.02M particles:
// 350 us more with 128 blocks).
template <int ND>
__global__ void __launch_bounds__(kSortThreads)
    k_sort(const DevHandle *__restrict__ H, const double *__restrict__ u,
           const double *__restrict__ v, int items, int tiles)
{
    if (skip(H->flag)) return;
    __shared__ int s[kSortThreads / 64];
    __shared__ int s_ticket, s_before;
    int *ctl = H->sort_ctl;  // lines of kSortLine ints: the ticket, then the items done of every phase
    const int ncells = H->P.ncells;
    if (threadIdx.x == 0) s_ticket = atomicAdd(&ctl[0], 1);
    __syncthreads();
    while (true) {
        int item = s_ticket, phase = 0, before = 0;
        for (int n = items; phase < 3 && item >= n; n = phase == 1 ? tiles : items) {
            item -= n;
            before = n;
            phase++;
        }
        if (phase == 3) return;  // uniform: every item is taken
        if (phase > 0) {
            if (threadIdx.x == 0) {
                while (__hip_atomic_load(&ctl[phase * kSortLine], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < before)
                    __builtin_amdgcn_s_sleep(1);
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            }
            __syncthreads();
        }
        if (phase == 0)
            links_body<ND>(H, item, items, u);
        else if (phase == 1)
            scan_tile<true, kSortThreads>(H->f_count, H->f_start, H->scan_state, ncells + 1, item, s, s_before);
        else
            gather_body<ND, 1>(H, item, items, u, v);
        // every wavefront's stores have left it, then one release for the block
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) {
            if (phase < 2)
                __hip_atomic_fetch_add(&ctl[(1 + phase) * kSortLine], 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            s_ticket = atomicAdd(&ctl[0], 1);
        }
        __syncthreads();
    }
}


// The Adami pass of wall particle w: kWallLanes lanes share it (lane q takes the entries q,
// q + kWallLanes, ... of its list of n fluid candidates, or for n < 0, an overflowed list or the
// cell search, its share of the rows of the cell walk; the partial sums are added at the end).
template <int ND>
__device__ __forceinline__ void adami_wall(const DevHandle *H, const DevParams &P, const FluidView &F,
                                           int w, int q, int n)
{
    constexpr int LANES = kWallLanes;
    const double4 xw = H->wpos[w];
    double pressure = 0.0, volume = 0.0, vs[3] = {0.0, 0.0, 0.0};
    if (n >= 0) {
        const int *alist = H->anbr;
        const int lw = H->lw;
        // the next list entry is loaded before the current one is evaluated
        int j = q < n ? alist[(size_t)q * lw + w] : 0;
        for (int k = q; k < n; k += LANES) {
            const int jn = alist[(size_t)min(k + LANES, n - 1) * lw + w];
            adami_term<ND>(P, F, xw, j, pressure, volume, vs);
            j = jn;
        }
    } else {
        Pencils<ND, LANES> it;
        it.init(P, xw.x, xw.y, xw.z, P.hs_fluid, q);
        int jb, je;
        while (it.next(P, F.start, jb, je))
            for (int j = jb; j < je; j++) adami_term<ND>(P, F, xw, j, pressure, volume, vs);
    }
#pragma unroll
    for (int o = 1; o < LANES; o <<= 1) {
        pressure += __shfl_xor(pressure, o);
        volume += __shfl_xor(volume, o);
        if (P.visc_w) {
#pragma unroll
            for (int d = 0; d < ND; d++) vs[d] += __shfl_xor(vs[d], o);
        }
    }
    if (q == 0) adami_finish(P, w, xw.w, pressure, volume, H->pw, H->rhow, H->wpv, vs, H->wvel);
}

// The Adami pass of all wall particles, as block bx of nb.  With Verlet lists only the active
// ones (a non-empty list, listed at the rebuild) are visited: the others keep the values the
// rebuild gave them.
template <int ND>
__device__ __forceinline__ void adami_pass(const DevHandle *H, int bx, int nb)
{
    const DevParams P = with_sound(H->params());
    const FluidView F = H->fluid();
    const int *active = H->wactive, *acnt = H->acnt;
    const int na = active ? H->counters[kCountActive] : P.nw;
    // the loop bound is uniform per group of lanes, so the partners shuffle together
    for (int g = (bx * (int)blockDim.x + (int)threadIdx.x) / kWallLanes; g < na; g += nb * (int)blockDim.x / kWallLanes) {
        const int w = active ? active[g] : g;
        adami_wall<ND>(H, P, F, w, threadIdx.x % kWallLanes, active ? acnt[w] : -1);
    }
}

template <int ND>
__global__ void __launch_bounds__(kBlock)
    k_wall(const DevHandle *__restrict__ H)
{
    adami_pass<ND>(H, blockIdx.x, gridDim.x);
}


// SUM: SummationDensity (the pressure acceleration of pair_fluid<ND, true>, velocity rows
// of dv only).  ANT: DensityDiffusionAntuono.  Without either the pairs take pair_factored.
template <int ND, bool SUM = false, bool ANT = false>
__global__ void __launch_bounds__(kBlock)
    k_fluid(const DevHandle *__restrict__ H, double *__restrict__ dv)
{
    const DevParams P = with_sound(H->params());
    const FluidView F = H->fluid();
    const WallView Wv = H->walls();
    const unsigned char *wall_near = H->wall_near;
    if (blockIdx.x == 0 && threadIdx.x == 0) *H->flag = 0;  // the rebuild (if any) is done
    __shared__ int lists[kCap * kBlock];
    int *lst = lists + threadIdx.x;
    const int s = xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    const bool active = s < P.nf;
    double xa[3] = {0.0, 0.0, 0.0}, va[3] = {0.0, 0.0, 0.0}, rho_a = 1.0, p_a = 0.0;
    if (active) {
        const double4 a = F.rec[2 * (size_t)s];
        const double4 b = F.rec[2 * (size_t)s + 1];
        xa[0] = a.x;
        xa[1] = a.y;
        xa[2] = a.z;
        rho_a = a.w;
        va[0] = b.x;
        va[1] = b.y;
        va[2] = b.z;
        p_a = b.w;
    }
    const double inv_rho_a = 1.0 / rho_a;
    if constexpr (SUM) p_a = p_a / (rho_a * rho_a);  // the target's p / rho^2
    double ga[3] = {0.0, 0.0, 0.0};  // DensityDiffusionAntuono: this particle's gradient
    if (ANT && active) {
#pragma unroll
        for (int d = 0; d < ND; d++) ga[d] = P.ddgrad[(size_t)s * ND + d];
    }

    double acc[3] = {0.0, 0.0, 0.0}, drho = 0.0;
    constexpr bool kFactored = !SUM && !ANT;
    neighbour_sweep<ND, false, kCap, kBlock, SUM, kFactored>(
        P, F.start, F.x, F.y, F.z, P.hs_fluid, active, F, Wv, lst, xa, va, rho_a, p_a,
        kFactored ? (P.use_visc ? 2.0 * P.av_c * rho_a : 0.0) : inv_rho_a, acc, drho, 0.0,
        ANT ? ga : nullptr);
    if constexpr (kFactored) {
#pragma unroll
        for (int d = 0; d < ND; d++) acc[d] *= P.kgrad_c / rho_a;
        drho *= P.kgrad_c;
    }
    double accw[3] = {0.0, 0.0, 0.0}, drhow = 0.0;
    if (P.nw > 0) {
        // walls are static: only cells flagged at create can have wall neighbours
        bool near = false;
        if (active) {
            const int c0 = cell_1d(xa[0], P.lo[0], P.inv_cs[0], P.n[0]);
            const int c1 = cell_1d(xa[1], P.lo[1], P.inv_cs[1], P.n[1]);
            const int c2 = (ND == 3) ? cell_1d(xa[2], P.lo[2], P.inv_cs[2], P.n[2]) : 0;
            near = wall_near[c0 + P.n[0] * (c1 + P.n[1] * c2)] != 0;
        }
        if (__any(near)) {
            const double m_a = (P.visc_w == 2 && active) ? F.vol[s].y : 1.0;
            neighbour_sweep<ND, true, kCap, kBlock, SUM>(P, Wv.start, Wv.x, Wv.y, Wv.z,
                                                         P.hs_wall, near, F, Wv, lst, xa, va,
                                                         rho_a, p_a, inv_rho_a, accw, drhow, m_a);
        }
    }
    if (!active) return;
    const int i = F.perm[s];
    constexpr int rows = SUM ? ND : ND + 1;
#pragma unroll
    for (int d = 0; d < ND; d++) dv[(size_t)i * rows + d] = (acc[d] + accw[d]) + P.g[d];
    if constexpr (!SUM) dv[(size_t)i * rows + ND] = drho + drhow;
}

// SummationDensity (summation_density!, density_calculators.jl:26-48): the density of every
// cell-sorted fluid particle s, sum_b m_b W(|x_s - x_b|) over the fluid particles within the
// compact support (itself included, W(0)) and then over the wall particles, the neighbour
// systems in the semidiscretization's order.  Written to rho (cell-sorted); k_sum_finish
// then sets the records, so that no lane reads a record another lane writes.
template <int ND>
__global__ void __launch_bounds__(kBlock)
    k_sum_density(const DevHandle *__restrict__ H)
{
    const DevParams P = H->params();
    const FluidView F = H->fluid();
    const WallView Wv = H->walls();
    const unsigned char *wall_near = H->wall_near;
    double *rho = H->sum_rho;
    const int s = xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    if (s >= P.nf) return;
    const double x0 = F.x[s], x1 = F.y[s], x2 = (ND == 3) ? F.z[s] : 0.0;
    double sum = 0.0;
    Pencils<ND> it;
    it.init(P, x0, x1, x2, P.hs_fluid);
    int jb, je;
    while (it.next(P, F.start, jb, je))
        for (int j = jb; j < je; j++) {
            const double d2 = dist2<ND>(x0 - F.x[j], x1 - F.y[j], (ND == 3) ? x2 - F.z[j] : 0.0);
            if (d2 <= P.R2) sum += F.vol[j].y * wendland_c2(P, sqrt(d2));
        }
    if (P.nw > 0) {
        const int c0 = cell_1d(x0, P.lo[0], P.inv_cs[0], P.n[0]);
        const int c1 = cell_1d(x1, P.lo[1], P.inv_cs[1], P.n[1]);
        const int c2 = (ND == 3) ? cell_1d(x2, P.lo[2], P.inv_cs[2], P.n[2]) : 0;
        if (wall_near[c0 + P.n[0] * (c1 + P.n[1] * c2)]) {
            Pencils<ND> iw;
            iw.init(P, x0, x1, x2, P.hs_wall);
            while (iw.next(P, Wv.start, jb, je))
                for (int w = jb; w < je; w++) {
                    const double4 xw = Wv.pos[w];
                    const double d2 = dist2<ND>(x0 - xw.x, x1 - xw.y, (ND == 3) ? x2 - xw.z : 0.0);
                    if (d2 <= P.R2) sum += xw.w * wendland_c2(P, sqrt(d2));
                }
        }
    }
    rho[s] = sum;
}

// The same sums over the Verlet lists (group t of four lanes takes the particle ord[t]): the
// particle itself (m W(0)), its fluid list and its wall list, each within the compact
// support; an overflowed list walks the cells instead (the SoA coordinates are current
// while some list overflows; the walls are static).  The four lanes' partial sums are added
// in a fixed order.
template <int ND>
__global__ void __launch_bounds__(kBlock)
    k_sum_density_lists(const DevHandle *__restrict__ H)
{
    const DevParams P = H->params();
    const FluidView F = H->fluid();
    const WallView Wv = H->walls();
    const int *ord = H->ord, *nbr = H->nbr, *cnt = H->cnt, *wnbr = H->wnbr, *wcnt = H->wcnt;
    const int ls = H->ls;
    double *rho = H->sum_rho;
    const int q = threadIdx.x % 4;
    const int t = (blockIdx.x * blockDim.x + threadIdx.x) / 4;
    const bool active = t < P.nf;
    const int tc = active ? t : P.nf - 1;  // an in-bounds particle for the idle lanes
    const int s = ord[tc];
    const double4 a = F.rec[2 * (size_t)s];
    const double x0 = a.x, x1 = a.y, x2 = (ND == 3) ? a.z : 0.0;
    double sum = (q == 0) ? F.vol[s].y * wendland_c2(P, 0.0) : 0.0;
    const int n = active ? cnt[tc] : 0;
    if (n >= 0) {
        for (int k = q; k < n; k += 4) {
            const int j = nbr[(size_t)k * ls + tc];
            const double4 b = F.rec[2 * (size_t)j];
            const double d2 = dist2<ND>(x0 - b.x, x1 - b.y, (ND == 3) ? x2 - b.z : 0.0);
            if (d2 <= P.R2) sum += F.vol[j].y * wendland_c2(P, sqrt(d2));
        }
    } else {
        Pencils<ND> it;
        it.init(P, x0, x1, x2, P.hs_fluid);
        int jb, je;
        while (it.next(P, F.start, jb, je))
            for (int j = jb + q; j < je; j += 4) {
                const double d2 = dist2<ND>(x0 - F.x[j], x1 - F.y[j], (ND == 3) ? x2 - F.z[j] : 0.0);
                if (d2 <= P.R2 && j != s) sum += F.vol[j].y * wendland_c2(P, sqrt(d2));
            }
    }
    const int nw = (active && P.nw > 0) ? wcnt[tc] : 0;
    if (nw > 0) {
        for (int k = q; k < nw; k += 4) {
            const double4 xw = Wv.pos[wnbr[(size_t)k * ls + tc]];
            const double d2 = dist2<ND>(x0 - xw.x, x1 - xw.y, (ND == 3) ? x2 - xw.z : 0.0);
            if (d2 <= P.R2) sum += xw.w * wendland_c2(P, sqrt(d2));
        }
    } else if (nw < 0) {
        Pencils<ND> iw;
        iw.init(P, x0, x1, x2, P.hs_wall);
        int jb, je;
        while (iw.next(P, Wv.start, jb, je))
            for (int w = jb + q; w < je; w += 4) {
                const double4 xw = Wv.pos[w];
                const double d2 = dist2<ND>(x0 - xw.x, x1 - xw.y, (ND == 3) ? x2 - xw.z : 0.0);
                if (d2 <= P.R2) sum += xw.w * wendland_c2(P, sqrt(d2));
            }
    }
    sum += __shfl_xor(sum, 1);
    sum += __shfl_xor(sum, 2);
    if (active && q == 0) rho[s] = sum;
}

// The brick kernels' part of the handle (see tpsph_handle).
struct BrickArgs {
    const int *ord, *nne;
    int *work;
    const int4 *bhead;
    const int *uidx;
    const unsigned short *nbr16;
    const int2 *thead;
    const int *nbr, *cnt, *wcnt;
    int ls;
    double *dv;
    const int *bfall;

    __device__ __forceinline__ explicit BrickArgs(const DevHandle &H, double *rates = nullptr)
        : ord(H.ord), nne(H.counters), work(H.bwork), bhead(H.bhead), uidx(H.uidx),
          nbr16(H.nbr16), thead(H.thead), nbr(H.nbr), cnt(H.cnt), wcnt(H.wcnt), ls(H.ls),
          dv(rates), bfall(H.bfall)
    {
    }
};

// The 16-byte (8-byte) field of the record at byte offset e16 (16 times its number).
__device__ __forceinline__ double2 lds_at(const double2 *p, int e16)
{
    return *reinterpret_cast<const double2 *>(reinterpret_cast<const char *>(p) + e16);
}
__device__ __forceinline__ double lds_at(const double *p, int e16)
{
    return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(p) + (e16 >> 1));
}

// The fluid part of the sums brick by brick: the union staged in LDS as {x, y} and {z, m}
// fields (the far record: far away, zero mass), each target summing m W over its list's LDS
// indices, four lanes per target; the particle itself (m W(0)) and the wall part as in
// k_sum_density_lists.  Bricks that do not stage take the global lists.  Blocks take bricks
// from work[2].
template <int ND>
struct SumSmem {
    double2 p0[kBrickCap], p1[kBrickCap];  // {x, y}, {z, m} (2D: {0, m})
    int item;
};

template <int ND>
__global__ void __launch_bounds__(kBrickThreads)
    k_sum_density_brick(const DevHandle *__restrict__ H)
{
    const DevParams P = H->params();
    const FluidView F = H->fluid();
    const WallView Wv = H->walls();
    const BrickArgs A(*H);
    const int *wnbr = H->wnbr;
    double *rho = H->sum_rho;
    __shared__ SumSmem<ND> S;
    const int tid = threadIdx.x;
    const int ne = *A.nne, ls = A.ls;
    const int cap = P.brick_cap;
    while (true) {
        if (tid == 0) S.item = atomicAdd(&A.work[2], 1);
        __syncthreads();
        const int item = S.item;
        if (item >= ne) break;
        const int4 hd = A.bhead[item];
        const int t0 = hd.x, t1 = hd.y, ntot = hd.z;
        const bool staged = ntot <= cap - 1;
        if (staged) {
            if (tid == 0) {  // the far record
                S.p0[cap - 1] = make_double2(kFar, kFar);
                S.p1[cap - 1] = make_double2(kFar, 0.0);
            }
            for (int i = tid; i < ntot; i += kBrickThreads) {
                const int g = A.uidx[hd.w + i];
                const double4 a = F.rec[2 * (size_t)g];
                S.p0[i] = make_double2(a.x, a.y);
                S.p1[i] = make_double2(ND == 3 ? a.z : 0.0, F.vol[g].y);
            }
            __syncthreads();
        }
        const int q = tid & 3;
        for (int base = t0; base < t1; base += kBrickThreads / 4) {
            const int t = base + tid / 4;
            const bool active = t < t1;
            const int col = active ? t : t0;
            const int s = A.ord[col];
            const double4 a = F.rec[2 * (size_t)s];
            const double x0 = a.x, x1 = a.y, x2 = (ND == 3) ? a.z : 0.0;
            double sum = (q == 0) ? F.vol[s].y * wendland_c2(P, 0.0) : 0.0;
            const int n = active ? A.cnt[col] : 0;
            if (staged) {
                const ushort4 *l4 = reinterpret_cast<const ushort4 *>(A.nbr16);
                const int ng = list_rows(max(n, 0));
                // rows clamped into the list rather than a select between a load and a
                // register (which made the compiler issue flat loads)
                ushort4 cur4 = l4[(size_t)min(q, max(ng - 1, 0)) * ls + col];
                for (int g = q; g < ng; g += 4) {
                    const ushort4 nxt4 = l4[(size_t)min(g + 4, ng - 1) * ls + col];
                    const unsigned short e4[4] = {cur4.x, cur4.y, cur4.z, cur4.w};
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const double2 b0 = lds_at(S.p0, e4[k]), b1 = lds_at(S.p1, e4[k]);
                        const double d2 = dist2<ND>(x0 - b0.x, x1 - b0.y, (ND == 3) ? x2 - b1.x : 0.0);
                        // the far record (and the slots past the list) add zero mass
                        if (d2 <= P.R2) sum += b1.y * wendland_c2(P, sqrt(d2));
                    }
                    cur4 = nxt4;
                }
            } else if (n >= 0) {
                for (int k = q; k < n; k += 4) {
                    const int j = A.nbr[(size_t)k * ls + col];
                    const double4 c = F.rec[2 * (size_t)j];
                    const double d2 = dist2<ND>(x0 - c.x, x1 - c.y, (ND == 3) ? x2 - c.z : 0.0);
                    if (d2 <= P.R2) sum += F.vol[j].y * wendland_c2(P, sqrt(d2));
                }
            } else {
                Pencils<ND> it;
                it.init(P, x0, x1, x2, P.hs_fluid);
                int jb, je;
                while (it.next(P, F.start, jb, je))
                    for (int j = jb + q; j < je; j += 4) {
                        const double d2 = dist2<ND>(x0 - F.x[j], x1 - F.y[j], (ND == 3) ? x2 - F.z[j] : 0.0);
                        if (d2 <= P.R2 && j != s) sum += F.vol[j].y * wendland_c2(P, sqrt(d2));
                    }
            }
            const int nw = (active && P.nw > 0) ? A.wcnt[col] : 0;
            if (nw > 0) {
                for (int k = q; k < nw; k += 4) {
                    const double4 xw = Wv.pos[wnbr[(size_t)k * ls + col]];
                    const double d2 = dist2<ND>(x0 - xw.x, x1 - xw.y, (ND == 3) ? x2 - xw.z : 0.0);
                    if (d2 <= P.R2) sum += xw.w * wendland_c2(P, sqrt(d2));
                }
            } else if (nw < 0) {
                Pencils<ND> iw;
                iw.init(P, x0, x1, x2, P.hs_wall);
                int jb, je;
                while (iw.next(P, Wv.start, jb, je))
                    for (int w = jb + q; w < je; w += 4) {
                        const double4 xw = Wv.pos[w];
                        const double d2 = dist2<ND>(x0 - xw.x, x1 - xw.y, (ND == 3) ? x2 - xw.z : 0.0);
                        if (d2 <= P.R2) sum += xw.w * wendland_c2(P, sqrt(d2));
                    }
            }
            sum += __shfl_xor(sum, 1);
            sum += __shfl_xor(sum, 2);
            if (active && q == 0) rho[s] = sum;
        }
        __syncthreads();  // the LDS is staged again for the next brick
    }
}

// The records of the summed densities: rho, the state equation's pressure and V = m / rho.
__global__ void __launch_bounds__(kBlock)
    k_sum_finish(const DevHandle *__restrict__ H)
{
    const DevParams P = with_sound(H->params());
    const int nf = P.nf;
    const double *rho = H->sum_rho;
    double4 *rec = H->rec;
    double2 *vol = H->vol;
    const int s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= nf) return;
    const double r = rho[s];
    rec[2 * (size_t)s].w = r;
    rec[2 * (size_t)s + 1].w = state_equation(P, r);
    const double m = vol[s].y;
    vol[s] = make_double2(m / r, m);
}

// Flag every cell that has a wall particle within the wall list radius of some point of the
// cell (static).
template <int ND>
__global__ void k_wall_near(DevParams P, int nw, const double4 *__restrict__ wpos,
                            unsigned char *__restrict__ near)
{
    int w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= nw) return;
    const double4 x = wpos[w];
    // the wall list radius R + skin/2 (and margins) of the Verlet lists, which covers the
    // radius R of the cell walk
    const double reach = P.R + P.hs_wall + P.hs_list_wall;
    const int x0 = cell_1d(x.x - reach, P.lo[0], P.inv_cs[0], P.n[0]);
    const int x1 = cell_1d(x.x + reach, P.lo[0], P.inv_cs[0], P.n[0]);
    const int y0 = cell_1d(x.y - reach, P.lo[1], P.inv_cs[1], P.n[1]);
    const int y1 = cell_1d(x.y + reach, P.lo[1], P.inv_cs[1], P.n[1]);
    const int z0 = (ND == 3) ? cell_1d(x.z - reach, P.lo[2], P.inv_cs[2], P.n[2]) : 0;
    const int z1 = (ND == 3) ? cell_1d(x.z + reach, P.lo[2], P.inv_cs[2], P.n[2]) : 0;
    for (int cz = z0; cz <= z1; cz++)
        for (int cy = y0; cy <= y1; cy++)
            for (int cx = x0; cx <= x1; cx++) near[cx + P.n[0] * (cy + P.n[1] * cz)] = 1;
}

// ------------------------------------------------------------------------------------------
// Verlet lists, rebuilt together with the cell list.  Until the next rebuild no particle
// moves by more than half the skin, so a fluid pair within R now was within R + skin at the
// build and a fluid-wall pair within R + skin/2 (walls do not move).  The lists hold those
// candidates; every kick still applies the exact radius test, so the neighbour sets are the
// same as those of a full search.  Entry k of sorted particle s sits at k * ls + s: the 64
// lanes of a wavefront read one contiguous 256-byte row per slot.  A particle with more
// candidates than the capacity stores count -1 and walks the cells in the kick instead.
// ------------------------------------------------------------------------------------------
// Broadcast of lane I of each quad (four consecutive lanes) to the whole quad (DPP).
template <int I>
__device__ __forceinline__ int quad_bcast(int v)
{
    return __builtin_amdgcn_mov_dpp(v, I * 0x55, 0xF, 0xF, false);
}

// Verlet list of fluid particle s (sorted index) in column col: the candidates within the
// list radius, in the pencils' order (the walls' lists and the bricks that do not stage).
template <int ND, bool WALL>
__device__ __forceinline__ void build_list(const DevParams &P, const FluidView &F,
                                           const WallView &Wv, int s, int col, int ls, int cap,
                                           int *__restrict__ nbr, int *__restrict__ cnt)
{
    const double xa = F.x[s], ya = F.y[s], za = (ND == 3) ? F.z[s] : 0.0;
    const int *start = WALL ? Wv.start : F.start;
    // the FP32 test takes what is not surely beyond the list radius
    const float4 xaf = F.xf[s];
    const float4 *cf = WALL ? Wv.xf : F.xf;
    const float out2 = WALL ? P.wlist_out2 : P.list_out2;
    Pencils<ND> it;
    it.init(P, xa, ya, za, WALL ? P.hs_list_wall : P.hs_list_fluid);
    int n = 0, j, je;
    while (it.next(P, start, j, je)) {
        // four candidates per step, their loads in flight together: the SoA arrays carry
        // kPad entries past their end, so the loads stay in bounds, and j + k < je masks the
        // candidates past the range (the list order is the candidates' order)
        for (; j < je; j += 4) {
            bool hit[4];
            float4 q[4];
#pragma unroll
            for (int k = 0; k < 4; k++) q[k] = cf[j + k];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float ex = xaf.x - q[k].x, ey = xaf.y - q[k].y;
                const float ez = (ND == 3) ? xaf.z - q[k].z : 0.f;
                const float d2f = ex * ex + ey * ey + ez * ez;
                hit[k] = !(d2f > out2);
            }
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if (j + k < je && hit[k] && (WALL || j + k != s)) {
                    if (n < cap) nbr[(size_t)n * ls + col] = j + k;
                    n++;
                }
            }
        }
    }
    cnt[col] = n <= cap ? n : -1;
}

// Verlet lists of the wall particles (wall-sorted order w) over the fluid: candidates within
// R + skin/2 of the static wall particle, for the Adami pass, which follows with `pass`.  Block
// bx of gx.
template <int ND>
__device__ __forceinline__ void wall_lists_body(const DevHandle *H, int bx, int gx, bool pass)
{
    const DevParams P = with_sound(H->params());
    const FluidView F = H->fluid();
    const double4 *wpos = H->wpos;
    const int lw = H->lw, cap = H->cap_a;
    int *nbr = H->anbr, *cnt = H->acnt, *active = H->wactive, *nactive = H->counters + kCountActive;
    for (int base = bx * kListThreads; base < P.nw; base += gx * kListThreads) {  // uniform
        const int w = base + (int)threadIdx.x;
        if (w < P.nw) {
            const double4 xw = wpos[w];
            const float4 xwf = list_f32<ND>(P, xw.x, xw.y, xw.z);
            Pencils<ND> it;
            it.init(P, xw.x, xw.y, xw.z, P.hs_list_wall);
            int n = 0, j, je;
            while (it.next(P, F.start, j, je)) {
                for (; j < je; j++) {
                    // what is not surely beyond the list radius (see build_list)
                    const float4 q = F.xf[j];
                    const float ex = xwf.x - q.x, ey = xwf.y - q.y, ez = (ND == 3) ? xwf.z - q.z : 0.f;
                    const float d2f = ex * ex + ey * ey + ez * ez;
                    if (!(d2f > P.wlist_out2)) {
                        if (n < cap) nbr[(size_t)n * lw + w] = j;
                        n++;
                    }
                }
            }
            cnt[w] = n <= cap ? n : -1;
            if (n == 0) {  // no fluid within reach until the next rebuild: the values of empty sums
                const double vs0[3] = {0.0, 0.0, 0.0};
                adami_finish(P, w, xw.w, 0.0, 0.0, H->pw, H->rhow, H->wpv, vs0, H->wvel);
            } else {
                active[atomicAdd(nactive, 1)] = w;
            }
        }
        if (!pass) continue;  // uniform
        __syncthreads();  // the block's lists
        for (int k = threadIdx.x / kWallLanes; k < kListThreads; k += kListThreads / kWallLanes) {
            const int v = base + k;
            const int n = v < P.nw ? cnt[v] : 0;
            if (n != 0) adami_wall<ND>(H, P, F, v, threadIdx.x % kWallLanes, n);
        }
    }
}

// Fluid kernel over the Verlet lists.
//
// Loads are quad-cooperative.  In slot k every lane needs the 64-byte record rec[2j], rec[2j+1]
// of its own candidate j.  The four lanes of a quad fetch the four records of the quad
// together: one 16-byte chunk per lane and record, so each load instruction reads 16 whole
// records (half cache lines) instead of 64 scattered 16-byte pieces.  The chunks pass
// through a wavefront-private LDS stage (80-byte stride: the writes and the reads are both
// free of bank conflicts), from which each lane reads its own record.  The candidate
// indices are read two slots ahead, the records one slot ahead of the pair terms.  The exact
// radius test (and the zero-distance skip) selects the pairs.
template <int ND>
__global__ void __launch_bounds__(kBlock)
    k_fluid_list(const DevHandle *__restrict__ H, double *__restrict__ dv)
{
    const DevParams P = with_sound(H->params());
    const FluidView F = H->fluid();
    const WallView Wv = H->walls();
    const int *ord = H->ord, *nbr = H->nbr, *cnt = H->cnt, *wnbr = H->wnbr, *wcnt = H->wcnt;
    const int ls = H->ls;
    if (blockIdx.x == 0 && threadIdx.x == 0) *H->flag = 0;  // the rebuild (if any) is done
    // 8 KiB per wavefront: the staging area (64 records x 80 bytes) while the lists are
    // streamed, then the int lists (kCap x 64 lanes) of the cell-walk fallback
    constexpr int kWaveUnits = 64 * kCap / 4;  // 16-byte units
    __shared__ double2 smem[kBlock / 64][kWaveUnits];
    const int lane = threadIdx.x & 63;
    double2 *stg = smem[threadIdx.x >> 6];
    int *lst = reinterpret_cast<int *>(stg) + lane;  // fallback lists, stride 64
    // t: position in the processing order (the list column), s: the cell-sorted particle
    const int t = xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    const bool active = t < P.nf;
    const int col = active ? t : 0;  // in-bounds column for the inactive lanes' loads
    const int s = ord[col];
    const int sl = s;
    double xa[3] = {0.0, 0.0, 0.0}, va[3] = {0.0, 0.0, 0.0}, rho_a = 1.0, p_a = 0.0;
    int n = 0, nw = 0;
    if (active) {
        const double4 a = F.rec[2 * (size_t)s];
        const double4 b = F.rec[2 * (size_t)s + 1];
        xa[0] = a.x;
        xa[1] = a.y;
        xa[2] = a.z;
        rho_a = a.w;
        va[0] = b.x;
        va[1] = b.y;
        va[2] = b.z;
        p_a = b.w;
        n = cnt[col];
        if (P.nw > 0) nw = wcnt[col];
    }
    const double inv_rho_a = 1.0 / rho_a;
    double ga[3] = {0.0, 0.0, 0.0};  // DensityDiffusionAntuono: this particle's gradient
    if (P.ddgrad && active) {
#pragma unroll
        for (int d = 0; d < ND; d++) ga[d] = P.ddgrad[(size_t)s * ND + d];
    }
    const double *gap = P.ddgrad ? ga : nullptr;

    double acc[3] = {0.0, 0.0, 0.0}, drho = 0.0;
    {
        const int m = max(n, 0);
        int mw = m;  // longest list of the wavefront
        for (int o = 32; o > 0; o >>= 1) mw = max(mw, __shfl_xor(mw, o));
        const double2 *rec2 = reinterpret_cast<const double2 *>(F.rec);
        const uint32_t r16 = 16u * (uint32_t)(lane & 3);
        double2 *mine = stg + 5 * (lane & ~3) + (lane & 3);  // chunk (lane & 3) of the quad's records
        const double2 *own = stg + 5 * lane;
        double2 c0, c1, c2, c3, vb;
        auto issue = [&](int j) {
            c0 = ldo(rec2, (uint32_t)quad_bcast<0>(j) * 64u + r16);
            c1 = ldo(rec2, (uint32_t)quad_bcast<1>(j) * 64u + r16);
            c2 = ldo(rec2, (uint32_t)quad_bcast<2>(j) * 64u + r16);
            c3 = ldo(rec2, (uint32_t)quad_bcast<3>(j) * 64u + r16);
            vb = ldo(F.vol, (uint32_t)j * 16u);
        };
        int jc = (m > 0) ? nbr[col] : sl;  // candidate whose record is in flight
        if (mw > 0) issue(jc);
        int jn = (1 < m) ? nbr[(size_t)ls + col] : sl;  // candidate of the next slot
        for (int k = 0; k < mw; k++) {
            mine[0] = c0;
            mine[5] = c1;
            mine[10] = c2;
            mine[15] = c3;
            __builtin_amdgcn_wave_barrier();
            const double2 a0 = own[0], a1 = own[1], b0 = own[2], b1 = own[3];
            const FluidNbr cur = {make_double4(a0.x, a0.y, a1.x, a1.y),
                                  make_double4(b0.x, b0.y, b1.x, b1.y), vb, jc};
            __builtin_amdgcn_wave_barrier();
            if (k + 1 < mw) issue(jn);
            jc = jn;
            jn = (k + 2 < m) ? nbr[(size_t)(k + 2) * ls + col] : sl;
            if (k < m) {
                const double p0 = xa[0] - cur.a.x, p1 = xa[1] - cur.a.y;
                const double p2 = (ND == 3) ? xa[2] - cur.a.z : 0.0;
                const double d2 = dist2<ND>(p0, p1, p2);
                if (d2 <= P.R2 && d2 >= P.az2)
                    pair_fluid<ND>(P, cur, xa, va, rho_a, p_a, inv_rho_a, acc, drho, gap);
            }
        }
    }
    if (__any(n < 0))
        neighbour_sweep<ND, false, kCap, 64>(P, F.start, F.x, F.y, F.z, P.hs_fluid, n < 0, F,
                                             Wv, lst, xa, va, rho_a, p_a, inv_rho_a, acc, drho,
                                             0.0, gap);

    double accw[3] = {0.0, 0.0, 0.0}, drhow = 0.0;
    if (__any(nw != 0)) {
        const double m_a = P.visc_w == 2 ? F.vol[s].y : 1.0;
        const int m = max(nw, 0);
        int j = (m > 0) ? wnbr[col] : 0;
        WallNbr cur = load_wall(Wv, j);
        for (int k = 0; k < m; k++) {
            const int jn = (k + 1 < m) ? wnbr[(size_t)(k + 1) * ls + col] : j;
            const WallNbr nxt = load_wall(Wv, jn);
            const double p0 = xa[0] - cur.a.x, p1 = xa[1] - cur.a.y;
            const double p2 = (ND == 3) ? xa[2] - cur.a.z : 0.0;
            const double d2 = dist2<ND>(p0, p1, p2);
            if (d2 <= P.R2 && d2 >= P.az2)
                pair_wall<ND>(P, cur, xa, va, rho_a, p_a, inv_rho_a, accw, drhow, m_a);
            cur = nxt;
            j = jn;
        }
        if (__any(nw < 0))
            neighbour_sweep<ND, true, kCap, 64>(P, Wv.start, Wv.x, Wv.y, Wv.z, P.hs_wall, nw < 0,
                                                F, Wv, lst, xa, va, rho_a, p_a, inv_rho_a, accw,
                                                drhow, m_a);
    }
    if (!active) return;
    const int i = F.perm[s];
#pragma unroll
    for (int d = 0; d < ND; d++) dv[(size_t)i * (ND + 1) + d] = (acc[d] + accw[d]) + P.g[d];
    dv[(size_t)i * (ND + 1) + ND] = drho + drhow;
}


// ------------------------------------------------------------------------------------------
// Bricks in LDS.  A brick is a block of bc[0] x bc[1] x bc[2] cells; its targets are the
// fluid particles in those cells (ord[t0 .. t1), columns of the lists).  Its union is every fluid
// particle in a cell row (y, z) near the brick, trimmed in x: the cells within the list radius
// R + skin of the brick box, as contiguous ranges of the cell-sorted arrays.  Every Verlet list
// entry of a target lies in the union of its brick, so after one staging pass of the union
// into LDS the pair terms read every candidate from LDS, and the list of a target holds record
// numbers of the union (16 bits, list_place; the places past the end of a list in its last
// rows hold the far record, brick_cap - 1, which no target reaches).  uidx holds the sorted
// index of every union record, the union of a brick from bhead.w on.  A brick whose union
// does not leave room for the far record, or with a target whose list overflowed, is marked
// (union size INT_MAX) and its targets have int lists and read their candidates from global
// memory.
//
// Without staging (h->bricks false: the union rows of a brick exceed kBrickMaxRows) every brick
// takes the int lists.
// ------------------------------------------------------------------------------------------
// The list build's part of the handle (see tpsph_handle).
struct ListsArgs {
    const int *nel;
    int *nne;  // counters (kCountBricks ...)
    int *bcount, *ord, *tbase, *uidx;
    int uidx_cap;
    int4 *bhead;
    int ls, cap_f, cap_w;
    int *nbr, *cnt, *wnbr, *wcnt, *wtargets;
    const unsigned char *wall_near;
    unsigned short *nbr16;  // nullptr: no brick stages
    int2 *thead;

    __device__ __forceinline__ explicit ListsArgs(const DevHandle &H)
        : nel(H.nel), nne(H.counters), bcount(H.bcount), ord(H.ord), tbase(H.tbase), uidx(H.uidx),
          uidx_cap(H.uidx_cap), bhead(H.bhead), ls(H.ls), cap_f(H.cap_f), cap_w(H.cap_w),
          nbr(H.nbr), cnt(H.cnt), wnbr(H.wnbr), wcnt(H.wcnt), wtargets(H.wtargets),
          wall_near(H.wall_near), nbr16(H.nbr16), thead(H.thead)
    {
    }
};

// ND, WIDE: cell rows of a target along y (kRows) and cell offsets of a union (kCellTab).  3D: bricks
// stage with one or two cell divisions (at most 144 union rows x 42 cells), and, WIDE, with
// DensityDiffusionAntuono's smaller bricks also with three (256 x 42, and one block per compute
// unit instead of two); 2D: with one to four (42 x 84).
template <int ND, bool WIDE>
struct ListsSmem {
    static constexpr int kRows = ND == 2 ? 9 : WIDE ? 7 : 5;
    static constexpr int kCellTab = ND == 2 ? 42 * 84 : WIDE ? 256 * 42 : 144 * 42;
    // the last entries of every thread's list, slot-major: 64 lanes write 64 banks whatever
    // slots they are at (aligned to a wave's ring: the slot is or-ed into the address)
    alignas(kListRing * 128) unsigned short ring[kListThreads / 64][kListRing * 64];
    // FP32 positions of the union (relative to the grid origin) and their padding
    float x[kBrickCap + 4], y[kBrickCap + 4], z[kBrickCap + 4];
    unsigned short ctab[kCellTab];
    unsigned short near[kBrickCap];  // the targets with walls near their cell
    int row_gb[kBrickMaxRows], row_lds[kBrickMaxRows + 1];
    int row_x0[kBrickMaxRows], row_x1[kBrickMaxRows];  // first and last cell along x (a grid has up to 2^20)
    int trow_s[kBrickMaxRows], trow_t[kBrickMaxRows + 1];
    int scan[kListThreads / 64];
    int item, col0, ubase, bad, nnear;
};

static_assert(sizeof(ListsSmem<2, false>) <= 80 * 1024 && sizeof(ListsSmem<3, false>) <= 80 * 1024,
              "two blocks per compute unit");

// Exclusive scan over the kListThreads threads of a block.
__device__ __forceinline__ int lists_scan(int value, int *s, int &total)
{
    const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
    int x = value;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) s[wave] = x;
    __syncthreads();
    int below = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < kListThreads / 64; w++) {
        const int y = s[w];
        below += w < wave ? y : 0;
        total += y;
    }
    __syncthreads();  // s is free again
    return below + x - value;
}

// Target `k` of the brick: its sorted index.
template <typename Smem>
__device__ __forceinline__ int lists_target(const Smem &S, int nrows, int k)
{
    const int r = bsearch_le(S.trow_t, nrows, k);
    return S.trow_s[r] + (k - S.trow_t[r]);
}

// The FP32 positions and the cell offsets of the union whose rows are in S (n records of the
// cell-sorted points with cell offsets `start`); uidx: also their sorted indices.
template <int ND, typename Smem>
__device__ __forceinline__ void stage_union(const DevParams &P, const int *__restrict__ start,
                                            const float4 *__restrict__ xf, Smem &S, int n,
                                            int uy0, int uz0, int nuy, int *__restrict__ uidx)
{
    // four records per thread at a time: their row searches and loads overlap
    static_assert(kBrickCap <= 4 * kListThreads && kBrickMaxRows == 256, "one pass of four, eight steps");
    int r[4], s[4];
    float4 c[4];
#pragma unroll
    for (int k = 0; k < 4; k++) r[k] = 0;
#pragma unroll
    for (int step = 128; step > 0; step >>= 1) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int to = r[k] + step;
            if (to < P.maxr && S.row_lds[to] <= (int)threadIdx.x + k * kListThreads) r[k] = to;
        }
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int i = (int)threadIdx.x + k * kListThreads;
        s[k] = i < n ? S.row_gb[r[k]] + (i - S.row_lds[r[k]]) : 0;
        c[k] = xf[s[k]];
    }
    // (the division: exact for these sizes, i + 1/2 is at least 1 / 2 ctab off a multiple)
    const float per_row = 1.0f / (float)P.ctab;
    for (int i = threadIdx.x; i < P.maxr * P.ctab; i += kListThreads) {
        const int u = (int)(((float)i + 0.5f) * per_row), x = S.row_x0[u] + (i - u * P.ctab);
        if (S.row_x1[u] < S.row_x0[u] || x > S.row_x1[u] + 1) continue;
        const int cy = uy0 + u % nuy, cz = (ND == 3) ? uz0 + u / nuy : 0;
        S.ctab[i] = (unsigned short)(S.row_lds[u] + start[P.n[0] * (cy + P.n[1] * cz) + x] - S.row_gb[u]);
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int i = (int)threadIdx.x + k * kListThreads;
        if (i >= n) continue;
        if (uidx) uidx[i] = s[k];
        S.x[i] = c[k].x;
        S.y[i] = c[k].y;
        if constexpr (ND == 3) S.z[i] = c[k].z;
    }
}

// 16 entries of a thread's ring, from list entry `first` (a multiple of 16) on, as the four rows
// of list_place.
__device__ __forceinline__ void ring_rows(const unsigned short *ring, int first,
                                          ushort4 *__restrict__ out, int ls, int col)
{
    const unsigned short *r = ring + (first & (kListRing - 1)) * 64;
#pragma unroll
    for (int q = 0; q < 4; q++)
        out[(size_t)(first / 4 + q) * ls + col] = make_ushort4(r[64 * q], r[64 * (q + 4)], r[64 * (q + 8)], r[64 * (q + 12)]);
}

// The list of the target at sorted index s in column col, one thread per target: the candidates
// of the staged union (of the fluid, WALL: of the walls) in the rows of cells near the target,
// as Pencils enumerates them.  A row's candidates are tested four at a time without branches:
// each is written behind the list (in the ring of the fluid list, whose 16 oldest entries go
// to memory when it fills; a wall list is short and goes to memory as it is found), which
// grows on a hit only.  Returns the number of entries (which may exceed the capacity: the
// surplus is not written).
template <int ND, bool WALL, typename Smem>
__device__ __forceinline__ int union_list(const DevParams &P, const FluidView &F,
                                          const ListsArgs &A, Smem &S, int s, bool active,
                                          int col, int self, double xa, double ya, double za,
                                          int c1, int c2, int uy0, int uz0, int nuy)
{
    constexpr int kRows = Smem::kRows;
    const float4 xaf = F.xf[s];
    const double hs = WALL ? P.hs_list_wall : P.hs_list_fluid;
    const float out2 = WALL ? P.wlist_out2 : P.list_out2;
    const int cap = WALL ? A.cap_w : A.cap_f;
    ushort4 *out = reinterpret_cast<ushort4 *>(A.nbr16);
    char *const ring = reinterpret_cast<char *>(S.ring);
    const uint32_t lane_ring = (threadIdx.x >> 6) * (kListRing * 128u) + (threadIdx.x & 63) * 2u;
    const double xc = (xa - P.lo[0]) * P.inv_cs[0];  // in cells
    double y2[kRows];
#pragma unroll
    for (int j = 0; j < kRows; j++) {
        const double y = transverse(P, 1, c1 + j - P.lr[1], ya, hs);
        y2[j] = y * y;
    }
    uint32_t n = 0;  // 128 times the number of entries: the offset of the ring's next slot
    uint32_t written = 0;
    for (int dz = ND == 3 ? -P.lr[2] : 0; dz <= (ND == 3 ? P.lr[2] : 0); dz++) {
        const int cz = ND == 3 ? c2 + dz : 0;
        const double z = (ND == 3) ? transverse(P, 2, cz, za, hs) : 0.0;
        const double rz2 = fma(-z, z, P.R2);
        const bool okz = active && (ND == 2 || (cz >= 0 && cz < P.n[2]));
        const int uz = (c1 - P.lr[1] - uy0) + nuy * (cz - uz0);
#pragma unroll
        for (int j = 0; j < kRows; j++) {
            if (j > 2 * P.lr[1]) break;  // uniform
            const int cy = c1 + j - P.lr[1], u = uz + j;
            const double r2 = rz2 - y2[j];
            int b = 0, e = 0;
            if (okz && cy >= 0 && cy < P.n[1] && r2 >= 0.0) {
                // conservative half-width: FP32 sqrt, enlarged well past its rounding error
                const double rx = ((double)(__builtin_amdgcn_sqrtf((float)r2) * 1.000001f) + hs) * P.inv_cs[0];
                const double last = (double)(P.n[0] - 1);  // cell_1d's clamping
                const int x0 = max((int)fmin(fmax(xc - rx, 0.0), last), S.row_x0[u]);
                const int x1 = min((int)fmin(fmax(xc + rx, 0.0), last), S.row_x1[u]);
                const unsigned short *ct = S.ctab + u * P.ctab - S.row_x0[u];
                if (x0 <= x1) {
                    b = ct[x0];
                    e = ct[x1 + 1];
                }
            }
            // the target's own row in two parts, without the target
            const bool own = !WALL && j == P.lr[1] && dz == 0;
            const int e_last = e;
            if (own) e = min(e, self);
            for (int part = 0; part <= (own ? 1 : 0); part++) {
                if (part == 1) {
                    b = max(b, self + 1);
                    e = e_last;
                }
                for (int k = b; k < e; k += 4) {
                    bool hit[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float ex = xaf.x - S.x[k + i], ey = xaf.y - S.y[k + i];
                        const float ez = (ND == 3) ? xaf.z - S.z[k + i] : 0.f;
                        // not surely beyond the list radius
                        hit[i] = !(ex * ex + ey * ey + ez * ez > out2) & (k + i < e);
                    }
                    if constexpr (WALL) {
                        const int w = S.row_gb[u] + (k - S.row_lds[u]);
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            if (hit[i] && (int)n < cap) A.wnbr[(size_t)n * A.ls + col] = w + i;
                            n += hit[i] ? 1u : 0u;
                        }
                    } else {
                        const int k16 = k * 16;
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            *reinterpret_cast<unsigned short *>(ring + (lane_ring | (n & (kListRing * 128u - 1)))) =
                                (unsigned short)(k16 + 16 * i);
                            n += hit[i] ? 128u : 0u;
                        }
                        // (one slot stays free for the candidate that does not hit)
                        if (__any(n - written > (kListRing - 5) * 128u) && n - written >= 16 * 128u) {
                            if ((int)(written >> 7) < cap)
                                ring_rows(S.ring[threadIdx.x >> 6] + (threadIdx.x & 63), (int)(written >> 7), out, A.ls, col);
                            written += 16 * 128u;
                        }
                    }
                }
            }
        }
    }
    if constexpr (WALL) return (int)n;
    const int count = (int)(n >> 7);
    if (active) {
        for (int p = count; p < ((count + 15) & ~15); p++)
            *reinterpret_cast<unsigned short *>(ring + (lane_ring | (((uint32_t)p * 128u) & (kListRing * 128u - 1)))) =
                (unsigned short)((P.brick_cap - 1) * 16);
        for (int w = (int)(written >> 7); w < min(count, cap); w += 16)
            ring_rows(S.ring[threadIdx.x >> 6] + (threadIdx.x & 63), w, out, A.ls, col);
    }
    return count;
}

// The lists of one brick's targets over the fluid (its union is staged); lists the targets with
// walls near their cell.  S.bad is set when a list overflowed (the brick then does not stage).
template <int ND, typename Smem>
__device__ __forceinline__ void brick_lists(const DevParams &P, const FluidView &F,
                                            const WallView &Wv, const ListsArgs &A, Smem &S,
                                            int ntargets, int nrows, int uy0, int uz0, int nuy)
{
    for (int base = 0; base < ntargets; base += kListThreads) {
        const int k = base + (int)threadIdx.x;
        const bool active = k < ntargets;
        const int s = lists_target(S, nrows, active ? k : 0), col = S.col0 + k;
        const double xa = F.x[s], ya = F.y[s], za = (ND == 3) ? F.z[s] : 0.0;
        const int c0 = cell_1d(xa, P.lo[0], P.inv_cs[0], P.n[0]);
        const int c1 = cell_1d(ya, P.lo[1], P.inv_cs[1], P.n[1]);
        const int c2 = (ND == 3) ? cell_1d(za, P.lo[2], P.inv_cs[2], P.n[2]) : 0;
        const int own = (c1 - uy0) + nuy * (c2 - uz0);
        const int self = S.row_lds[own] + (s - S.row_gb[own]);
        const int n = union_list<ND, false>(P, F, A, S, s, active, col, self, xa, ya, za,
                                            c1, c2, uy0, uz0, nuy);
        if (active) {
            A.ord[col] = s;
            A.cnt[col] = n <= A.cap_f ? n : -1;
            A.tbase[col] = S.ubase;
            A.thead[col] = make_int2(F.perm[s], self | n << kHeadCount);
            if (n > A.cap_f) S.bad = 1;
            if (P.nw > 0) {
                if (A.wall_near[c0 + P.n[0] * (c1 + P.n[1] * c2)])
                    S.near[atomicAdd(&S.nnear, 1)] = (unsigned short)k;
                else
                    A.wcnt[col] = 0;
            }
        }
    }
}

// The wall lists of the targets in S.near, the walls' union staged.
template <int ND, typename Smem>
__device__ __forceinline__ void brick_wall_lists(const DevParams &P, const FluidView &F,
                                                 const WallView &Wv, const ListsArgs &A,
                                                 Smem &S, int nrows, int uy0, int uz0,
                                                 int nuy, bool staged)
{
    for (int base = 0; base < S.nnear; base += kListThreads) {
        const int i = base + (int)threadIdx.x;
        const bool active = i < S.nnear;
        const int k = S.near[active ? i : 0];
        const int s = lists_target(S, nrows, k), col = S.col0 + k;
        int n;
        if (staged) {
            const double xa = F.x[s], ya = F.y[s], za = (ND == 3) ? F.z[s] : 0.0;
            const int c1 = cell_1d(ya, P.lo[1], P.inv_cs[1], P.n[1]);
            const int c2 = (ND == 3) ? cell_1d(za, P.lo[2], P.inv_cs[2], P.n[2]) : 0;
            n = union_list<ND, true>(P, F, A, S, s, active, col, 0, xa, ya, za, c1, c2,
                                     uy0, uz0, nuy);
            if (!active) continue;
            n = n <= A.cap_w ? n : -1;
            A.wcnt[col] = n;
        } else {
            if (!active) continue;
            build_list<ND, true>(P, F, Wv, s, col, A.ls, A.cap_w, A.wnbr, A.wcnt);
            n = A.wcnt[col];
        }
        if (n != 0) {
            A.thead[col].y |= kHeadWalls;
            if (A.wtargets) A.wtargets[atomicAdd(&A.nne[kCountWallTargets], 1)] = col;
        }
    }
}

// Int lists of the targets of a brick that does not stage, one thread per target.
// walls: also their wall lists and headers (not when brick_lists has written them).
template <int ND, typename Smem>
__device__ __forceinline__ void brick_int_lists(const DevParams &P, const FluidView &F,
                                                const WallView &Wv, const ListsArgs &A,
                                                const Smem &S, int ntargets, int nrows,
                                                bool walls)
{
    for (int k = threadIdx.x; k < ntargets; k += kListThreads) {
        const int s = lists_target(S, nrows, k), col = S.col0 + k;
        build_list<ND, false>(P, F, Wv, s, col, A.ls, A.cap_f, A.nbr, A.cnt);
        // an overflowed list walks the cells, which need the SoA coordinates every kick
        if (A.cnt[col] < 0) atomicAdd(&A.nne[kCountOverflow], 1);
        A.tbase[col] = -1;
        if (!walls) continue;
        A.ord[col] = s;
        if (P.nw > 0) {
            const int c0 = cell_1d(F.x[s], P.lo[0], P.inv_cs[0], P.n[0]);
            const int c1 = cell_1d(F.y[s], P.lo[1], P.inv_cs[1], P.n[1]);
            const int c2 = (ND == 3) ? cell_1d(F.z[s], P.lo[2], P.inv_cs[2], P.n[2]) : 0;
            if (A.wall_near[c0 + P.n[0] * (c1 + P.n[1] * c2)]) {
                build_list<ND, true>(P, F, Wv, s, col, A.ls, A.cap_w, A.wnbr, A.wcnt);
                if (A.wtargets && A.wcnt[col] != 0) A.wtargets[atomicAdd(&A.nne[kCountWallTargets], 1)] = col;
            } else {
                A.wcnt[col] = 0;
            }
        }
    }
}

// The rebuild after the cell-sorted gather, in one launch: the first nwall blocks build the
// Verlet lists of the wall particles, the others take the bricks (columns of the targets, union,
// lists of the targets over the fluid and the walls); both read only the new cell-sorted order.
// adami: the blocks of the wall particles also run the Adami pass, with the flag down nothing
// else (one launch of a kick less).
//
// The list build is bound by the VALU work of the candidates' tests (1.02M particles: 88k of
// 146k cycles per brick).  The candidates' FP32 positions come from the staged union (from
// global memory the address units were busy for 470 of 680 us); one thread per target tests
// four candidates per step (four lanes per target: a row of cells holds about five
// candidates, so the lanes idle, and what a row costs besides its tests is paid by four times
// as many waves); the test is the FP32 one alone; the int list of a staged target (4 bytes per
// entry) is not written any more; the walls of a brick are staged the same way, for the
// targets near one only (four lanes per target on global memory: 157 us, here 40).  Bricks,
// unions and lists took 860 us and five launches, four lanes per target 720, this form 495.
// Two blocks of 512 threads share a compute unit (80 KB each; WIDE: one of 88 KB).  A brick takes
// its columns, its part of uidx and the block's next brick from three counters, each on a line of
// its own: on one line they bounded the build of many bricks of few targets (700k particles in
// 2D: 96 -> 74 us, with one in a hundred dispersed as spray 235 -> 150).
template <int ND, bool WIDE>
__global__ void __launch_bounds__(kListThreads, WIDE ? 2 : 4)
    k_brick_lists(const DevHandle *__restrict__ H, int nwall, bool adami)
{
    const bool rebuild = !skip(H->flag);
    if ((int)blockIdx.x < nwall) {
        if (rebuild)
            wall_lists_body<ND>(H, blockIdx.x, nwall, adami);
        else if (adami)
            adami_pass<ND>(H, blockIdx.x, nwall);
        return;
    }
    if (!rebuild) return;
    const DevParams P = H->params();
    const FluidView F = H->fluid();
    const int block = (int)blockIdx.x - nwall, nblocks = (int)gridDim.x - nwall;
    const WallView Wv = H->walls();
    const ListsArgs A(*H);
    __shared__ ListsSmem<ND, WIDE> S;
    const int tid = threadIdx.x;
    const int ne = A.nne[kCountBricks];
    const int nuy = P.bc[1] + 2 * P.ur[1];
    for (int turn = block;; ) {
        if (turn >= ne) break;  // uniform over the block
        const int b = A.nel[turn];
        const int bx = b % P.nb[0], by = (b / P.nb[0]) % P.nb[1], bz = b / (P.nb[0] * P.nb[1]);
        const int X0 = bx * P.bc[0], X1 = min(X0 + P.bc[0], P.n[0]) - 1;
        const int Y0 = by * P.bc[1], Y1 = min(Y0 + P.bc[1], P.n[1]) - 1;
        const int Z0 = (ND == 3) ? bz * P.bc[2] : 0;
        const int Z1 = (ND == 3) ? min(Z0 + P.bc[2], P.n[2]) - 1 : 0;
        // the targets: the brick's cell rows
        const int nty = Y1 - Y0 + 1, nrows = nty * (Z1 - Z0 + 1);
        int ts = 0, tn = 0;
        if (tid < nrows) {
            const int row = P.n[0] * (Y0 + tid % nty + P.n[1] * (Z0 + tid / nty));
            ts = F.start[row + X0];
            tn = F.start[row + X1 + 1] - ts;
        }
        int ntargets;
        const int tt = lists_scan(tn, S.scan, ntargets);
        if (tid < nrows) {
            S.trow_s[tid] = ts;
            S.trow_t[tid] = tt;
        }
        // the union: its rows, then (where it fits) its records
        const int uy0 = Y0 - P.ur[1], uz0 = (ND == 3) ? Z0 - P.ur[2] : 0;
        int tot = INT_MAX;
        if (A.nbr16) {
            const double m = P.hs_union;
            const double bxlo = cell_lo(P, 0, X0, m), bxhi = cell_hi(P, 0, X1, m);
            const double bylo = cell_lo(P, 1, Y0, m), byhi = cell_hi(P, 1, Y1, m);
            const double bzlo = (ND == 3) ? cell_lo(P, 2, Z0, m) : 0.0;
            const double bzhi = (ND == 3) ? cell_hi(P, 2, Z1, m) : 0.0;
            int cntr = 0, gb = 0, x0 = 0, x1 = -1;
            if (tid < P.maxr) {
                const int cy = uy0 + tid % nuy;
                const int cz = (ND == 3) ? uz0 + tid / nuy : 0;
                if (cy >= 0 && cy < P.n[1] && cz >= 0 && cz < P.n[2]) {
                    const double dy = fmax(0.0, fmax(cell_lo(P, 1, cy, m) - byhi, bylo - cell_hi(P, 1, cy, m)));
                    double dz = 0.0;
                    if constexpr (ND == 3)
                        dz = fmax(0.0, fmax(cell_lo(P, 2, cz, m) - bzhi, bzlo - cell_hi(P, 2, cz, m)));
                    const double r2 = P.rl_union2 - (dy * dy + dz * dz);
                    if (r2 >= 0.0) {
                        const double rx = sqrt(r2) * (1.0 + 1e-9) + m;
                        x0 = cell_1d(bxlo - rx, P.lo[0], P.inv_cs[0], P.n[0]);
                        x1 = min(cell_1d(bxhi + rx, P.lo[0], P.inv_cs[0], P.n[0]), x0 + P.ctab - 2);
                        const int row = P.n[0] * (cy + P.n[1] * cz);
                        gb = F.start[row + x0];
                        cntr = F.start[row + x1 + 1] - gb;
                    }
                }
            }
            const int lds0 = lists_scan(cntr, S.scan, tot);
            if (tid < P.maxr) {
                S.row_gb[tid] = gb;
                S.row_lds[tid] = lds0;
                S.row_x0[tid] = x0;
                S.row_x1[tid] = x1;
            }
            if (tid == 0) S.row_lds[P.maxr] = tot;
            if (tot > P.brick_cap - 1) tot = INT_MAX;
        }
        if (tid == 0) {
            A.bcount[b] = 0;  // clear for the next rebuild
            S.col0 = atomicAdd(&A.nne[kCountTargets], ntargets);
            S.ubase = tot < INT_MAX ? atomicAdd(&A.nne[kCountRecords], tot) : 0;
            S.bad = 0;
            S.nnear = 0;
            S.item = atomicAdd(&A.nne[kCountClaims], 1);
        }
        __syncthreads();
        const int next = nblocks + S.item;
        if (tot < INT_MAX && S.ubase > A.uidx_cap - tot) tot = INT_MAX;  // uniform
        if (tot < INT_MAX) {
            stage_union<ND>(P, F.start, F.xf, S, tot, uy0, uz0, nuy, A.uidx + S.ubase);
            __syncthreads();
            brick_lists<ND>(P, F, Wv, A, S, ntargets, nrows, uy0, uz0, nuy);
            __syncthreads();
            if (S.bad) {  // some list overflowed
                tot = INT_MAX;
                brick_int_lists<ND>(P, F, Wv, A, S, ntargets, nrows, false);
            }
            if (S.nnear > 0) {
                // the union of the walls: the same cell rows (the fluid's list radius reaches
                // further than the walls')
                int gb = 0, cntr = 0;
                if (tid < P.maxr && S.row_x0[tid] <= S.row_x1[tid]) {
                    const int cy = uy0 + tid % nuy, cz = (ND == 3) ? uz0 + tid / nuy : 0;
                    const int row = P.n[0] * (cy + P.n[1] * cz);
                    gb = Wv.start[row + S.row_x0[tid]];
                    cntr = Wv.start[row + S.row_x1[tid] + 1] - gb;
                }
                int wtot;
                const int lds0 = lists_scan(cntr, S.scan, wtot);
                const bool staged = wtot <= kBrickCap - 1;
                if (tid < P.maxr) {
                    S.row_gb[tid] = gb;
                    S.row_lds[tid] = lds0;
                }
                if (tid == 0) S.row_lds[P.maxr] = wtot;
                __syncthreads();
                if (staged) {
                    stage_union<ND>(P, Wv.start, Wv.xf, S, wtot, uy0, uz0, nuy, nullptr);
                    __syncthreads();
                }
                brick_wall_lists<ND>(P, F, Wv, A, S, nrows, uy0, uz0, nuy, staged);
            }
        } else {
            brick_int_lists<ND>(P, F, Wv, A, S, ntargets, nrows, true);
        }
        if (tid == 0) A.bhead[turn] = make_int4(S.col0, S.col0 + ntargets, tot, tot < INT_MAX ? S.ubase : 0);
        turn = next;
        __syncthreads();  // S is written again
    }
}

// Staged union: one record per particle as four 16-byte fields and one 8-byte field, each in
// an array of its own, read with one ds_read_b128 (ds_read_b64) per field.  The 16-byte
// stride spreads random candidates over all banks; 72- or 64-byte records made the lanes of
// a read collide on fewer bank groups (measured 2% and 12% slower).  The last record is the
// far record that pads the list groups (finite values, zero volume).
// ANT (DensityDiffusionAntuono): also the renormalised density gradient, g0 {gx, gy} and in
// 3D g1 {gz}, in CAP = kBrickCapGrad records there (96 bytes each: the LDS holds fewer).
template <int ND, bool ANT = false>
struct BrickSmem {
    static constexpr int CAP = (ANT && ND == 3) ? kBrickCapGrad : kBrickCap;
    // 3D: p0 {x, y}, p1 {z, rho}, p2 {vx, vy}, p3 {vz, p};  2D: p0 {x, y}, p1 {rho, vx},
    // p2 {vy, p} (p3 unused); vol: V = m / rho (SummationDensity: m)
    // (vol first: the other fields of a record lie at constant offsets from 16 times its number)
    double vol[CAP];
    double2 p0[CAP], p1[CAP], p2[CAP], p3[ND == 3 ? CAP : 1];
    double2 g0[ANT ? CAP : 1];
    double g1[(ANT && ND == 3) ? CAP : 1];
    int4 head[2];  // bhead of this brick and of the next one
};

// A staged record in registers.
struct BrickRec {
    double x[3], rho, v[3], p, V;
};

template <int ND, bool ANT>
__device__ __forceinline__ BrickRec lds_rec(const BrickSmem<ND, ANT> &S, int e16)
{
    BrickRec n;
    const double2 a = lds_at(S.p0, e16), b = lds_at(S.p1, e16), c = lds_at(S.p2, e16);
    n.x[0] = a.x;
    n.x[1] = a.y;
    if constexpr (ND == 3) {
        const double2 d = lds_at(S.p3, e16);
        n.x[2] = b.x;
        n.rho = b.y;
        n.v[0] = c.x;
        n.v[1] = c.y;
        n.v[2] = d.x;
        n.p = d.y;
    } else {
        n.x[2] = 0.0;
        n.rho = b.x;
        n.v[0] = b.y;
        n.v[1] = c.x;
        n.v[2] = 0.0;
        n.p = c.y;
    }
    n.V = lds_at(S.vol, e16);
    return n;
}

// The density gradient of staged record e (DensityDiffusionAntuono).
template <int ND, bool ANT>
__device__ __forceinline__ void lds_grad(const BrickSmem<ND, ANT> &S, int e16, double *g)
{
    const double2 a = lds_at(S.g0, e16);
    g[0] = a.x;
    g[1] = a.y;
    g[2] = (ND == 3) ? lds_at(S.g1, e16) : 0.0;
}

// The pair constants of the staged pair loop (scalar registers).
struct BrickConsts {
    double az2, minus_half_h_inv, eps_h2, two_av_c, dd2, h, two_beta, kgrad_c;

    __device__ __forceinline__ explicit BrickConsts(const DevParams &P)
        : az2(P.az2), minus_half_h_inv(-0.5 * P.h_inv), eps_h2(P.eps_h2), two_av_c(2.0 * P.av_c),
          dd2(P.dd2), h(P.h), two_beta(2.0 * P.beta), kgrad_c(P.kgrad_c)
    {
    }
};

// A target of the staged pair loop and its fluid-fluid terms (pair_fluid's) without branches.
// With k = (1 - r / 2h)^3 of a pair the sums are
//   acc  += V_b k [-(p_a + p_b) + 2 alpha c h rho_a rho_b min(v_ab.r_ab, 0) /
//                  ((r^2 + eps h^2)(rho_a + rho_b)) + ...beta] r_ab
//   drho += V_b k [2 delta h c (rho_a - rho_b) + rho_a v_ab.r_ab]
// and what is common to all pairs of the target, kgrad_c / rho_a and kgrad_c, multiplies the
// finished sums: 8 instructions fewer per candidate than with the factors in every term.
// SUM (SummationDensity): acc += m_b k [-(p_a/rho_a^2 + p_b/rho_b^2) + 2 alpha c h ...], with
// p / rho^2 staged in the pressure slot and m in the volume slot, and no density rate.
//
// The range test is the kernel factor itself: max(1 - r / 2h, 0) is zero for every candidate
// beyond R (up to rounding at exactly R, where (1 - r / 2h)^3 is below 1e-46), for the far
// record (whose volume is zero too) and, as max(NaN, 0), for a pair at d^2 < az2, whose
// high word is replaced by a NaN's.
template <int ND, int VISC, bool ANT, bool SUM>
struct BrickTarget {
    double x[3], v[3], rho, p, visc, g[ANT ? 3 : 1];

    __device__ __forceinline__ BrickTarget(const BrickConsts &C, const BrickRec &me)
    {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            x[d] = me.x[d];
            v[d] = me.v[d];
        }
        rho = me.rho;
        p = me.p;
        visc = SUM ? C.two_av_c : C.two_av_c * me.rho;
    }

    // gb: the candidate's renormalised density gradient (ANT)
    __device__ __forceinline__ void add(const BrickConsts &C, const BrickRec &n, double *acc,
                                        double &drho, const double *gb) const
    {
        const double p0 = x[0] - n.x[0], p1 = x[1] - n.x[1];
        const double p2 = (ND == 3) ? x[2] - n.x[2] : 0.0;
        double d2 = dist2<ND>(p0, p1, p2);
        const double near = __hiloint2double(d2 >= C.az2 ? __double2hiint(d2) : 0x7ff80000,
                                             __double2loint(d2));
        const double w = fmax(fma(C.minus_half_h_inv, sqrt_pos(near), 1.0), 0.0);
        const double Vk = n.V * (w * w * w);
        const double v0 = v[0] - n.v[0], v1 = v[1] - n.v[1];
        const double v2 = (ND == 3) ? v[2] - n.v[2] : 0.0;
        double vr = v0 * p0 + v1 * p1;
        if constexpr (ND == 3) vr += v2 * p2;
        double f = -(p + n.p);
        if constexpr (VISC != kViscNone) {
            const double q = d2 + C.eps_h2;
            const double sum_rho = rho + n.rho;
            const double vn = fmin(vr, 0.0);
            const double num = SUM ? visc * vn : visc * (n.rho * vn);
            f = fma(num, rcp_pos(q * sum_rho), f);
            if constexpr (VISC == kViscAlphaBeta) {
                const double mu = C.h * vn * rcp_pos(q);
                const double b = C.two_beta * (mu * mu) * rcp_pos(sum_rho);
                f += SUM ? b : (rho * n.rho) * b;
            }
        }
        f *= Vk;
        acc[0] = fma(f, p0, acc[0]);
        acc[1] = fma(f, p1, acc[1]);
        if constexpr (ND == 3) acc[2] = fma(f, p2, acc[2]);
        if constexpr (!SUM) {
            double drr = rho - n.rho;
            if constexpr (ANT) {
                double gr = (g[0] + gb[0]) * p0 + (g[1] + gb[1]) * p1;
                if constexpr (ND == 3) gr += (g[2] + gb[2]) * p2;
                drr = fma(-0.5, gr, drr);
            }
            drho = fma(Vk, fma(C.dd2, drr, rho * vr), drho);
        }
    }

    // the factors common to all pairs of the target
    __device__ __forceinline__ void scale(const BrickConsts &C, double *acc, double &drho) const
    {
        const double f = SUM ? C.kgrad_c : C.kgrad_c / rho;
#pragma unroll
        for (int d = 0; d < 3; d++) acc[d] *= f;
        drho *= C.kgrad_c;
    }
};

// One thread's share of a union on its way from global memory to LDS: records tid and
// tid + kBrickThreads (a union holds fewer than 2 kBrickThreads).
template <int ND, bool ANT, bool SUM>
struct UnionShare {
    double4 a[2], c[2];
    double V[2], g[2][ANT ? ND : 1];

    // s: the sorted indices of the two records
    __device__ __forceinline__ void load(const DevParams &P, const FluidView &F, int2 s)
    {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t o = (uint32_t)(h ? s.y : s.x);
            a[h] = ldo(F.rec, o * 64u);
            c[h] = ldo(F.rec, o * 64u + 32u);
            const double2 vm = ldo(F.vol, o * 16u);
            V[h] = SUM ? vm.y : vm.x;
            if constexpr (ANT) {
#pragma unroll
                for (int d = 0; d < ND; d++) g[h][d] = P.ddgrad[(size_t)o * ND + d];
            }
        }
    }

    __device__ __forceinline__ void store(BrickSmem<ND, ANT> &S, int ntot) const
    {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int i = (int)threadIdx.x + h * kBrickThreads;
            if (i >= ntot) continue;
            const double pslot = SUM ? c[h].w / (a[h].w * a[h].w) : c[h].w;
            S.p0[i] = make_double2(a[h].x, a[h].y);
            if constexpr (ND == 3) {
                S.p1[i] = make_double2(a[h].z, a[h].w);
                S.p2[i] = make_double2(c[h].x, c[h].y);
                S.p3[i] = make_double2(c[h].z, pslot);
            } else {
                S.p1[i] = make_double2(a[h].w, c[h].x);
                S.p2[i] = make_double2(c[h].y, pslot);
            }
            S.vol[i] = V[h];
            if constexpr (ANT) {
                S.g0[i] = make_double2(g[h][0], g[h][1]);
                if constexpr (ND == 3) S.g1[i] = g[h][2];
            }
        }
    }
};

// The fluid-fluid sums of the targets of a brick that does not stage (four lanes per target):
// the int Verlet lists, or the cell walk (lane 0) of an overflowed list.
template <int ND, bool SUM, typename Args>
__device__ __forceinline__ void brick_from_global(const DevParams &P, const FluidView &F,
                                                  const Args &A, int t0, int t1)
{
    const int q = (int)threadIdx.x & 3;
    for (int base = t0; base < t1; base += kBrickThreads / 4) {
        const int t = base + (int)threadIdx.x / 4;
        const bool active = t < t1;
        const int col = active ? t : t0;
        const int s = A.ord[col];
        const double4 a = F.rec[2 * (size_t)s], c = F.rec[2 * (size_t)s + 1];
        const double xa[3] = {a.x, a.y, a.z}, va[3] = {c.x, c.y, c.z};
        const double rho_a = a.w, inv_rho_a = 1.0 / a.w;
        const double p_a = SUM ? c.w / (rho_a * rho_a) : c.w;
        double ga[3] = {0.0, 0.0, 0.0};  // DensityDiffusionAntuono: the target's gradient
        const bool ant = !SUM && P.ddgrad;
        if (ant) {
#pragma unroll
            for (int d = 0; d < ND; d++) ga[d] = P.ddgrad[(size_t)s * ND + d];
        }
        double acc[3] = {0.0, 0.0, 0.0}, drho = 0.0;
        auto pair = [&](int j) {
            const FluidNbr nb = load_fluid(F, j);
            const double p0 = xa[0] - nb.a.x, p1 = xa[1] - nb.a.y;
            const double p2 = (ND == 3) ? xa[2] - nb.a.z : 0.0;
            const double d2 = dist2<ND>(p0, p1, p2);
            if (d2 <= P.R2 && d2 >= P.az2)
                pair_fluid<ND, SUM>(P, nb, xa, va, rho_a, p_a, inv_rho_a, acc, drho, ant ? ga : nullptr);
        };
        const int n = active ? A.cnt[col] : 0;
        if (n >= 0) {
            for (int k = q; k < n; k += 4) pair(A.nbr[(size_t)k * A.ls + col]);
        } else if (q == 0) {
            Pencils<ND> it;
            it.init(P, xa[0], xa[1], xa[2], P.hs_fluid);
            int jb, je;
            while (it.next(P, F.start, jb, je))
                for (int j = jb; j < je; j++) pair(j);
        }
#pragma unroll
        for (int o = 1; o < 4; o <<= 1) {
#pragma unroll
            for (int d = 0; d < 3; d++) acc[d] += __shfl_xor(acc[d], o);
            drho += __shfl_xor(drho, o);
        }
        if (active && q == 0) {
            constexpr int rows = SUM ? ND : ND + 1;
            const bool walls = P.nw > 0 && A.wcnt[col] != 0;
            const int i = F.perm[s];
#pragma unroll
            for (int d = 0; d < ND; d++)
                A.dv[(size_t)i * rows + d] = walls ? acc[d] : acc[d] + P.g[d];
            if constexpr (!SUM) A.dv[(size_t)i * rows + ND] = drho;
        }
    }
}

// The sorted indices of this thread's two records of a union of n records from entry `first`
// of uidx on (past n those of its last record, 0 of an empty union).
__device__ __forceinline__ int2 union_share(const int *__restrict__ uidx, int first, int n)
{
    const int last = max(n - 1, 0);
    const int a = uidx[first + min((int)threadIdx.x, last)];
    const int b = uidx[first + min((int)threadIdx.x + kBrickThreads, last)];
    return n > 0 ? make_int2(a, b) : make_int2(0, 0);
}

// Fluid-fluid kernel over the bricks, one block of kBrickThreads per compute unit.  Targets
// with wall candidates are completed by k_fluid_walls.
//
// What bounds it: 1024 threads with one 147 KB union leave a compute unit one block, so
// nothing hides a brick's chain of dependent loads (claim, brick header, record numbers,
// records, target headers: 24k of 57k cycles per brick at 1.02M particles) but the block
// itself.  So the chain runs one brick ahead: while a brick's pair loop runs, wave 0 claims
// the brick after the next one and reads its header; every wave that has finished its targets
// loads its share of the next union into registers before it waits for the others, and then
// the headers and first list rows of its next targets; and the targets' own records come from
// the staged union (thead).  Measured at 1.02M particles, with the pair terms of BrickTarget:
// 299 -> 247 us per launch, and with uidx in place of searches of the union rows, the list
// layout of list_place and the target headers read ahead 222 us.
// Bricks: the first gridDim.x in the order of the blocks, then from the work counter (which
// k_gather<0> and the stage kernel reset).  A brick that does not stage takes several times as long
// as one that does, so its block claims none before it is done: held by their blocks meanwhile,
// the other bricks made the tail of the launch (128k particles in 3D at h = 1.5 dx, 144 of 396
// bricks: 282 us per launch with the next ones claimed ahead, 155 so).
// VISC: visc_mode(P), the viscosity form of the pair loop.  ANT: DensityDiffusionAntuono
// (P.ddgrad), whose gradients are staged beside the records.  SUM: SummationDensity
// (pressure slot staged as p / rho^2, no density rate, dv of ND rows).
template <int ND, int VISC = kViscAlpha, bool ANT = false, bool SUM = false>
__global__ void __launch_bounds__(kBrickThreads)
    k_fluid_brick(const DevHandle *__restrict__ H, double *__restrict__ dv)
{
    const DevParams P = with_sound(H->params());
    const FluidView F = H->fluid();
    const BrickArgs A(*H, dv);
    using Smem = BrickSmem<ND, ANT>;
    __shared__ Smem S;
    const int tid = threadIdx.x;
    if (blockIdx.x == 0 && tid == 0) *H->flag = 0;  // the rebuild (if any) is done
    const int ne = *A.nne;
    if ((int)blockIdx.x >= ne) return;  // uniform: a block without a brick
    constexpr int kFarSlot = Smem::CAP - 1;
    if (tid == 0) {  // the far record: coordinates kFar, rho 1, the rest 0
        if constexpr (ANT) {
            S.g0[kFarSlot] = make_double2(0.0, 0.0);
            if constexpr (ND == 3) S.g1[kFarSlot] = 0.0;
        }
        S.p0[kFarSlot] = make_double2(kFar, kFar);
        S.p2[kFarSlot] = make_double2(0.0, 0.0);
        if constexpr (ND == 3) {
            S.p1[kFarSlot] = make_double2(kFar, 1.0);
            S.p3[kFarSlot] = make_double2(0.0, 0.0);
        } else {
            S.p1[kFarSlot] = make_double2(1.0, 0.0);
        }
        S.vol[kFarSlot] = 0.0;
    }
    auto claim = [&] { return (int)gridDim.x + atomicAdd(A.work, 1); };
    auto read_head = [&](int item, int k) {  // lane 0 of wave 0
        S.head[k] = item < ne ? A.bhead[item] : make_int4(-1, -1, 0, 0);
    };
    int4 hd = A.bhead[blockIdx.x];  // {first target, one past the last, union size, first entry}
    int nstage = hd.z <= kFarSlot ? hd.z : 0;
    {
        UnionShare<ND, ANT, SUM> share;
        share.load(P, F, union_share(A.uidx, hd.w, nstage));
        if (tid == 0) read_head((int)gridDim.x < ne && hd.z <= kFarSlot ? claim() : ne, 1);
        share.store(S, nstage);
    }
    // Four lanes per target: lane q of target i takes the entries q, q + 4, ... of its list;
    // the four partial sums are added across the lanes (a fixed butterfly) and lane 0 writes.
    // With four lanes a brick's targets (about 385) take two passes of 256 whose waves spread
    // evenly over the four SIMDs; two lanes left a quarter of the waves idle and one SIMD
    // with the most work (8% slower).
    constexpr int kL = 4;
    const int q = tid & (kL - 1);
    const ushort4 *l4 = reinterpret_cast<const ushort4 *>(A.nbr16);
    const BrickConsts C(P);
    // header and first list row of this thread's first target
    auto column = [&](const int4 &head, int base) {
        const int t = base + tid / kL;
        return t < head.y ? t : head.x;
    };
    int2 th = A.thead[column(hd, hd.x)];
    ushort4 cur4 = l4[(size_t)q * A.ls + column(hd, hd.x)];
    __syncthreads();
    for (int cur = 0;; cur ^= 1) {
        const bool staged = hd.z <= kFarSlot;
        if (!staged) {
            brick_from_global<ND, SUM>(P, F, A, hd.x, hd.y);
            if (tid == 0) read_head(claim(), cur ^ 1);
            __syncthreads();
        }
        const int4 nx = S.head[cur ^ 1];
        const int nx_stage = nx.z <= kFarSlot ? nx.z : 0;
        const int2 us = union_share(A.uidx, nx.w, nx_stage);
        int item = ne;  // the brick after the next one: its number arrives during the pair loop
        if (tid == 0 && nx.x >= 0 && nx.z <= kFarSlot) item = claim();
        if (staged) {
            for (int base = hd.x; base < hd.y; base += kBrickThreads / kL) {
                const bool active = base + tid / kL < hd.y;
                const int col = column(hd, base);
                if (base > hd.x) {
                    th = A.thead[col];
                    cur4 = l4[(size_t)q * A.ls + col];
                }
                const int self = (th.y & (kBrickCap - 1)) * 16;
                const int m = active ? (th.y >> kHeadCount) & kHeadCountMask : 0;
                BrickTarget<ND, VISC, ANT, SUM> T(C, lds_rec<ND>(S, self));
                if constexpr (ANT) lds_grad<ND>(S, self, T.g);
                double acc[3] = {0.0, 0.0, 0.0}, drho = 0.0;
                // four entries per 8-byte load, one row ahead of the pair terms
                const int rows = list_rows(m);
                for (int r = q; r < rows; r += kL) {
                    // rows clamped into the list rather than a select between a load and a
                    // register: the select made the compiler keep cur4 in scratch and issue
                    // a flat load, whose wait also held up every LDS read
                    const ushort4 nxt4 = l4[(size_t)min(r + kL, rows - 1) * A.ls + col];
                    // the candidates are independent chains without branches: two at a time
                    // interleave within the register budget of four waves per SIMD; entries
                    // past the end of the list are the far record's: exact zeros
                    auto two = [&](int ea, int eb) {
                        const BrickRec na = lds_rec<ND>(S, ea);
                        const BrickRec nb = lds_rec<ND>(S, eb);
                        double gna[3], gnb[3];
                        if constexpr (ANT) {
                            lds_grad<ND>(S, ea, gna);
                            lds_grad<ND>(S, eb, gnb);
                        }
                        T.add(C, na, acc, drho, gna);
                        T.add(C, nb, acc, drho, gnb);
                    };
                    two(cur4.x, cur4.y);
                    if (list_row_entries(m, r) > 2) two(cur4.z, cur4.w);
                    cur4 = nxt4;
                }
                T.scale(C, acc, drho);
#pragma unroll
                for (int o = 1; o < kL; o <<= 1) {
#pragma unroll
                    for (int d = 0; d < 3; d++) acc[d] += __shfl_xor(acc[d], o);
                    drho += __shfl_xor(drho, o);
                }
                if (active && q == 0) {
                    // with wall candidates k_fluid_walls adds the wall sum and then gravity
                    constexpr int vrows = SUM ? ND : ND + 1;
                    const bool walls = (th.y & kHeadWalls) != 0;
                    double *o = A.dv + (size_t)th.x * vrows;
#pragma unroll
                    for (int d = 0; d < ND; d++) o[d] = walls ? acc[d] : acc[d] + P.g[d];
                    if constexpr (!SUM) o[ND] = drho;
                }
            }
        }
        if (nx.x < 0) break;  // uniform: no brick after this one
        // (a load without a branch around it keeps the share in registers; a brick that does
        // not stage reads some valid record)
        UnionShare<ND, ANT, SUM> share;
        share.load(P, F, us);
        th = A.thead[column(nx, nx.x)];
        cur4 = l4[(size_t)q * A.ls + column(nx, nx.x)];
        // wave 0 is the first to finish (the oldest wave wins the issue), and this brick's
        // header is no longer read
        if (tid == 0) read_head(item, cur);
        __syncthreads();  // every wave has finished with the staged union
        hd = nx;
        share.store(S, nx_stage);
        __syncthreads();
    }
}

// The bricks that do not stage, which the mixed-precision pass (tpsph_mixed.hip) leaves to
// FP64: the work[1] bricks it listed in bfall, taken by blocks in turn.
template <int ND>
__global__ void __launch_bounds__(kBrickThreads)
    k_fluid_brick_global(const DevHandle *__restrict__ H, double *__restrict__ dv)
{
    const DevParams P = with_sound(H->params());
    const FluidView F = H->fluid();
    const BrickArgs A(*H, dv);
    const int ne = A.work[1];
    for (int k = blockIdx.x; k < ne; k += gridDim.x) {
        const int4 hd = A.bhead[A.bfall[k]];
        brick_from_global<ND, false>(P, F, A, hd.x, hd.y);
    }
}

// Wall sums of the targets with wall candidates (wtargets, built at the rebuild) after
// k_fluid_brick: dv = (dv + wall sum) + gravity, the reference's order of the sums.
// Four lanes share a target: lane q takes list entries q, q + 4, ...; the sums are added
// across the four lanes before the write.
// SUM: SummationDensity (the target's p / rho^2 in the pressure slot, dv of ND rows).
template <int ND, bool SUM = false>
__global__ void __launch_bounds__(kBlock)
    k_fluid_walls(const DevHandle *__restrict__ H, double *__restrict__ dv)
{
    const DevParams P = with_sound(H->params());
    const FluidView F = H->fluid();
    const WallView Wv = H->walls();
    const int *ord = H->ord, *wtargets = H->wtargets, *nwtargets = H->counters + kCountWallTargets;
    const int *wnbr = H->wnbr, *wcnt = H->wcnt;
    const int ls = H->ls;
    constexpr int kLanes = 4;
    __shared__ int lists[kCap * kBlock];  // only for particles whose wall list overflowed
    int *lst = lists + threadIdx.x;
    const int nt = *nwtargets;
    const int q = threadIdx.x % kLanes;
    for (int base = blockIdx.x * (kBlock / kLanes); base < nt; base += gridDim.x * (kBlock / kLanes)) {
        const int idx = base + (int)threadIdx.x / kLanes;
        const bool active = idx < nt;
        const int t = wtargets[active ? idx : base];
        const int s = ord[t];
        const double4 a = F.rec[2 * (size_t)s];
        const double4 c = F.rec[2 * (size_t)s + 1];
        const double xa[3] = {a.x, a.y, a.z}, va[3] = {c.x, c.y, c.z};
        const double rho_a = a.w, inv_rho_a = 1.0 / rho_a;
        const double p_a = SUM ? c.w / (rho_a * rho_a) : c.w;
        const double m_a = P.visc_w == 2 ? F.vol[s].y : 1.0;
        const int nw = active ? wcnt[t] : 0;
        double accw[3] = {0.0, 0.0, 0.0}, drhow = 0.0;
        const int m = max(nw, 0);
        // the next list entry is loaded before the current one is evaluated
        int jw = q < m ? wnbr[(size_t)q * ls + t] : 0;
        for (int k = q; k < m; k += kLanes) {
            const WallNbr cur = load_wall(Wv, jw);
            jw = wnbr[(size_t)min(k + kLanes, m - 1) * ls + t];
            const double p0 = xa[0] - cur.a.x, p1 = xa[1] - cur.a.y;
            const double p2 = (ND == 3) ? xa[2] - cur.a.z : 0.0;
            const double d2 = dist2<ND>(p0, p1, p2);
            if (d2 <= P.R2 && d2 >= P.az2)
                pair_wall<ND, SUM>(P, cur, xa, va, rho_a, p_a, inv_rho_a, accw, drhow, m_a);
        }
        if (__any(nw < 0))
            neighbour_sweep<ND, true, kCap, kBlock, SUM>(P, Wv.start, Wv.x, Wv.y, Wv.z, P.hs_wall,
                                                         nw < 0 && q == 0, F, Wv, lst, xa, va,
                                                         rho_a, p_a, inv_rho_a, accw, drhow, m_a);
#pragma unroll
        for (int o = 1; o < kLanes; o <<= 1) {
#pragma unroll
            for (int d = 0; d < 3; d++) accw[d] += __shfl_xor(accw[d], o);
            drhow += __shfl_xor(drhow, o);
        }
        if (active && q == 0) {
            double *o = dv + (size_t)F.perm[s] * (SUM ? ND : ND + 1);
#pragma unroll
            for (int d = 0; d < ND; d++) o[d] = (o[d] + accw[d]) + P.g[d];
            if constexpr (!SUM) o[ND] = o[ND] + drhow;
        }
    }
}

// DensityDiffusionAntuono's update! (density_diffusion.jl:176-211), over the fluid
// neighbours b of fluid particle a:
//   M_a = -sum_b V_b grad W_ab (x) r_ab        (compute_gradient_correction_matrix!,
//                                               corrections.jl:329-354)
//   L_a = M_a^-1, or the identity where |det M_a| < 1f-9
//                                              (correction_matrix_inversion_step!,
//                                               corrections.jl:425-457)
//   grad rho_a = -sum_b (rho_a - rho_b) V_b L_a grad W_ab = -L_a s_a,
//   s_a = sum_b (rho_a - rho_b) V_b grad W_ab  (L_a is the same for every pair of a, so it
//                                               multiplies the sum once)
// with V_b = m_b / rho_b and grad W zero at distance >= R and at distance^2 < eps(h^2)
// (smoothing_kernel_grad, abstract_system.jl:142-155).  M_a is symmetric: its upper
// triangle is summed.  Four lanes share a particle; their partial sums are added with
// shuffles.
struct GradSums {
    double m[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};  // M_00 M_01 M_02 M_11 M_12 M_22
    double sv[3] = {0.0, 0.0, 0.0};
};

// One pair's terms; vk = V_b |grad W| / r (zero for a pair outside the kernel's support).
template <int ND>
__device__ __forceinline__ void grad_add(GradSums &g, double vk, double drr, double p0,
                                         double p1, double p2)
{
    const double f = drr * vk;
    g.m[0] -= vk * p0 * p0;
    g.m[1] -= vk * p0 * p1;
    g.m[3] -= vk * p1 * p1;
    g.sv[0] += f * p0;
    g.sv[1] += f * p1;
    if constexpr (ND == 3) {
        g.m[2] -= vk * p0 * p2;
        g.m[4] -= vk * p1 * p2;
        g.m[5] -= vk * p2 * p2;
        g.sv[2] += f * p2;
    }
}

// V_b |grad W| / r of a pair at squared distance d2, zero outside [eps(h^2), R^2) without a
// branch (the square root of an excluded d2 may be NaN: it is selected away).
__device__ __forceinline__ double grad_vk(const DevParams &P, double V_b, double d2)
{
    const bool in = (d2 < P.R2) & (d2 >= P.eps_hh);
    const double r = sqrt_pos(d2);
    const double w = fma(-0.5 * P.h_inv, r, 1.0);
    return in ? V_b * (P.kgrad_c * (w * w * w)) : 0.0;
}

// Sums of the four lanes of a quad (a fixed butterfly), then the inversion and the gradient
// of particle s (lane 0 of an active quad writes it).
template <int ND>
__device__ __forceinline__ void grad_finish(const DevParams &P, GradSums &g, bool write, int s)
{
#pragma unroll
    for (int o = 1; o < 4; o <<= 1) {
#pragma unroll
        for (int i = 0; i < 6; i++)
            if (ND == 3 || i == 0 || i == 1 || i == 3) g.m[i] += __shfl_xor(g.m[i], o);
#pragma unroll
        for (int i = 0; i < ND; i++) g.sv[i] += __shfl_xor(g.sv[i], o);
    }
    if (!write) return;
    const double *m = g.m, *sv = g.sv;
    constexpr double kSingular = (double)1.0e-9f;  // the Float32 literal 1.0f-9
    double gr[3];
    if constexpr (ND == 2) {
        const double det = m[0] * m[3] - m[1] * m[1];
        if (fabs(det) < kSingular) {
            gr[0] = -sv[0];
            gr[1] = -sv[1];
        } else {
            const double id = 1.0 / det;
            gr[0] = -(m[3] * sv[0] - m[1] * sv[1]) * id;
            gr[1] = -(m[0] * sv[1] - m[1] * sv[0]) * id;
        }
    } else {
        // cofactors of the symmetric M (its adjugate is symmetric too)
        const double c00 = m[3] * m[5] - m[4] * m[4];
        const double c01 = m[2] * m[4] - m[1] * m[5];
        const double c02 = m[1] * m[4] - m[2] * m[3];
        const double c11 = m[0] * m[5] - m[2] * m[2];
        const double c12 = m[1] * m[2] - m[0] * m[4];
        const double c22 = m[0] * m[3] - m[1] * m[1];
        const double det = m[0] * c00 + m[1] * c01 + m[2] * c02;
        if (fabs(det) < kSingular) {
            gr[0] = -sv[0];
            gr[1] = -sv[1];
            gr[2] = -sv[2];
        } else {
            const double id = 1.0 / det;
            gr[0] = -(c00 * sv[0] + c01 * sv[1] + c02 * sv[2]) * id;
            gr[1] = -(c01 * sv[0] + c11 * sv[1] + c12 * sv[2]) * id;
            gr[2] = -(c02 * sv[0] + c12 * sv[1] + c22 * sv[2]) * id;
        }
    }
#pragma unroll
    for (int d = 0; d < ND; d++) P.ddgrad[(size_t)s * ND + d] = gr[d];
}

// The sums of particle s from global memory: its Verlet list (n >= 0 entries in column t,
// lane q takes entries q, q + 4, ...) or, for an overflowed list or the cell search
// (n < 0), the cell walk over the SoA coordinates, which are current whenever they are
// walked.
template <int ND>
__device__ __forceinline__ void grad_sums_global(const DevParams &P, const FluidView &F,
                                                 GradSums &g, const double *xa, double rho_a,
                                                 int n, const int *__restrict__ nbr, int t,
                                                 int ls, int q)
{
    if (n >= 0) {
        for (int k = q; k < n; k += 4) {
            const int j = nbr[(size_t)k * ls + t];
            const double4 b = F.rec[2 * (size_t)j];
            const double p0 = xa[0] - b.x, p1 = xa[1] - b.y;
            const double p2 = (ND == 3) ? xa[2] - b.z : 0.0;
            const double d2 = dist2<ND>(p0, p1, p2);
            if (d2 < P.R2 && d2 >= P.eps_hh)
                grad_add<ND>(g, grad_vk(P, F.vol[j].x, d2), rho_a - b.w, p0, p1, p2);
        }
    } else {
        Pencils<ND> it;
        it.init(P, xa[0], xa[1], xa[2], P.hs_fluid);
        int jb, je;
        while (it.next(P, F.start, jb, je)) {
            for (int j = jb + q; j < je; j += 4) {
                const double p0 = xa[0] - F.x[j], p1 = xa[1] - F.y[j];
                const double p2 = (ND == 3) ? xa[2] - F.z[j] : 0.0;
                const double d2 = dist2<ND>(p0, p1, p2);
                if (d2 < P.R2 && d2 >= P.eps_hh)
                    grad_add<ND>(g, grad_vk(P, F.vol[j].x, d2), rho_a - F.rec[2 * (size_t)j].w,
                                 p0, p1, p2);
            }
        }
    }
}

// The gradients over the Verlet lists (group t takes the particle ord[t] and its list) or,
// without lists (nbr == nullptr), the cell walk of every particle.
template <int ND>
__global__ void __launch_bounds__(kBlock)
    k_antuono_gradient(const DevHandle *__restrict__ H, bool lists)
{
    const DevParams P = H->params();
    const FluidView F = H->fluid();
    const int *ord = H->ord, *nbr = lists ? (const int *)H->nbr : nullptr, *cnt = H->cnt;
    const int ls = H->ls;
    const int q = threadIdx.x % 4;
    const int t = (blockIdx.x * blockDim.x + threadIdx.x) / 4;
    const bool active = t < P.nf;
    const int tc = active ? t : P.nf - 1;  // an in-bounds particle for the idle lanes
    const int s = nbr ? ord[tc] : tc;
    const double4 a = F.rec[2 * (size_t)s];
    const double xa[3] = {a.x, a.y, a.z};
    GradSums g;
    const int n = !active ? 0 : (nbr ? cnt[t] : -1);
    grad_sums_global<ND>(P, F, g, xa, a.w, n, nbr, t, ls, q);
    grad_finish<ND>(P, g, active && q == 0, s);
}

// The gradients brick by brick (the lists' LDS indices, the union staged in LDS as
// {x, y} and {z, rho} fields and V, the far record padding the list groups), as
// k_fluid_brick takes the fluid pass; bricks that do not stage read global memory.  Blocks
// take bricks from work[2].
template <int ND>
struct GradSmem {
    double2 p0[kBrickCap], p1[kBrickCap];  // {x, y}, {z, rho} (2D: {0, rho})
    double vol[kBrickCap];
    int item;
};

template <int ND>
__global__ void __launch_bounds__(kBrickThreads)
    k_antuono_gradient_brick(const DevHandle *__restrict__ H)
{
    const DevParams P = H->params();
    const FluidView F = H->fluid();
    const BrickArgs A(*H);
    __shared__ GradSmem<ND> S;
    const int tid = threadIdx.x;
    const int ne = *A.nne, ls = A.ls;
    const int cap = P.brick_cap;
    while (true) {
        if (tid == 0) S.item = atomicAdd(&A.work[2], 1);
        __syncthreads();
        const int item = S.item;
        if (item >= ne) break;
        const int4 hd = A.bhead[item];
        const int t0 = hd.x, t1 = hd.y, ntot = hd.z;
        const bool staged = ntot <= cap - 1;
        if (staged) {
            if (tid == 0) {  // the far record: far away, zero volume
                S.p0[cap - 1] = make_double2(kFar, kFar);
                S.p1[cap - 1] = make_double2(kFar, 1.0);
                S.vol[cap - 1] = 0.0;
            }
            for (int i = tid; i < ntot; i += kBrickThreads) {
                const int g = A.uidx[hd.w + i];
                const double4 a = F.rec[2 * (size_t)g];
                S.p0[i] = make_double2(a.x, a.y);
                S.p1[i] = make_double2(ND == 3 ? a.z : 0.0, a.w);
                S.vol[i] = F.vol[g].x;
            }
            __syncthreads();
        }
        const int q = tid & 3;
        for (int base = t0; base < t1; base += kBrickThreads / 4) {
            const int t = base + tid / 4;
            const bool active = t < t1;
            const int col = active ? t : t0;
            const int s = A.ord[col];
            const double4 a = F.rec[2 * (size_t)s];
            const double xa[3] = {a.x, a.y, ND == 3 ? a.z : 0.0};
            const int n = active ? A.cnt[col] : 0;
            GradSums gs;
            if (staged) {
                const ushort4 *l4 = reinterpret_cast<const ushort4 *>(A.nbr16);
                const int ng = list_rows(max(n, 0));
                // rows clamped into the list rather than a select between a load and a
                // register (which made the compiler issue flat loads)
                ushort4 cur4 = l4[(size_t)min(q, max(ng - 1, 0)) * ls + col];
                for (int g = q; g < ng; g += 4) {
                    const ushort4 nxt4 = l4[(size_t)min(g + 4, ng - 1) * ls + col];
                    const unsigned short e4[4] = {cur4.x, cur4.y, cur4.z, cur4.w};
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const int e = e4[k];
                        const double2 b0 = lds_at(S.p0, e), b1 = lds_at(S.p1, e);
                        const double p0 = xa[0] - b0.x, p1 = xa[1] - b0.y;
                        const double p2 = (ND == 3) ? xa[2] - b1.x : 0.0;
                        const double d2 = dist2<ND>(p0, p1, p2);
                        grad_add<ND>(gs, grad_vk(P, lds_at(S.vol, e), d2), a.w - b1.y, p0, p1, p2);
                    }
                    cur4 = nxt4;
                }
            } else {
                grad_sums_global<ND>(P, F, gs, xa, a.w, n, A.nbr, col, ls, q);
            }
            grad_finish<ND>(P, gs, active && q == 0, s);
        }
        __syncthreads();  // the LDS is staged again for the next brick
    }
}

// drift!: du = v (semidiscretization.jl:561-571; delta_v = 0 without shifting)
// (vrows rows of v per particle: ND + 1, or ND under SummationDensity)
template <int ND>
__global__ void k_drift(int nf, int vrows, const double *__restrict__ v, double *__restrict__ du)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nf) return;
#pragma unroll
    for (int d = 0; d < ND; d++) du[(size_t)i * ND + d] = v[(size_t)i * vrows + d];
}

// One 2N-storage stage of the partition (v, u) with slopes (dv, v): the drift slope is read
// before v is updated, as the integrator evaluates kick! and drift! at the same stage state.
// A block owns kBlock particles and walks their u and then their v entries as flat,
// contiguous ranges, so every load and store of a wavefront covers whole cache lines.
// Then, what k_gather<0> does for the next kick: the cell-sorted records of the new state
// (positions, velocity, density, pressure by the state equation, volume), the skin check
// and the reset of the brick work counter.  iperm[i] is the sorted index of particle i of
// the last rebuild.
template <int ND>
__global__ void __launch_bounds__(kBlock)
    k_ck_stage_gather(const DevHandle *__restrict__ H, double *__restrict__ v,
                      double *__restrict__ u, double *__restrict__ tv, double *__restrict__ tu,
                      const double *__restrict__ dv, double a, double b, double dt, int first)
{
    DevParams P = H->params();
    int *flag = H->flag, *work = H->bwork;
    const int *iperm = H->iperm, *noverflow = H->noverflow;
    const double *m = H->mass, *snap = H->snap;
    double *xs = H->xs, *ys = H->ys, *zs = H->zs;
    double4 *rec = H->rec;
    double2 *vol = H->vol;
    const int nf = P.nf;
    P = with_sound(P);
    const int i0 = blockIdx.x * kBlock;
    const int np = min(kBlock, nf - i0);
    const size_t u0 = (size_t)i0 * ND, v0 = (size_t)i0 * (ND + 1);
    for (int e = threadIdx.x; e < np * ND; e += kBlock) {
        const int p = e / ND, d = e - p * ND;
        const double slope = v[v0 + (size_t)p * (ND + 1) + d];
        const size_t k = u0 + e;
        const double t = first ? dt * slope : fma(dt, slope, a * tu[k]);
        tu[k] = t;
        u[k] = fma(b, t, u[k]);
    }
    __syncthreads();  // the v entries read above are written below
    for (int e = threadIdx.x; e < np * (ND + 1); e += kBlock) {
        const size_t k = v0 + e;
        const double t = first ? dt * dv[k] : fma(dt, dv[k], a * tv[k]);
        tv[k] = t;
        v[k] = fma(b, t, v[k]);
    }
    __syncthreads();  // the block's new u and v are complete
    if (blockIdx.x == 0) reset_counters(work, H->sort_ctl);
    const int i = i0 + (int)threadIdx.x;
    bool moved = false;  // left its skin
    if (i < nf) {
        const size_t nfs = (size_t)nf;
        const int s = iperm[i];
        double x[3] = {0.0, 0.0, 0.0}, vv[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int d = 0; d < ND; d++) {
            x[d] = u[(size_t)i * ND + d];
            vv[d] = v[(size_t)i * (ND + 1) + d];
        }
        const double rho = v[(size_t)i * (ND + 1) + ND];
        const double mass = m[i];
        if (!noverflow || *noverflow != 0) {  // see k_gather
            xs[s] = x[0];
            ys[s] = x[1];
            if constexpr (ND == 3) zs[s] = x[2];
        }
        rec[2 * (size_t)s] = make_double4(x[0], x[1], x[2], rho);
        rec[2 * (size_t)s + 1] = make_double4(vv[0], vv[1], vv[2], state_equation(P, rho));
        vol[s] = make_double2(mass / rho, mass);
        double e2 = 0.0;
#pragma unroll
        for (int d = 0; d < ND; d++) {
            const double e = x[d] - snap[d * nfs + s];
            e2 = fma(e, e, e2);
        }
        moved = !(e2 <= P.half_skin2);
    }
    raise_rebuild_flag(flag, moved);
}

// ------------------------------------------------------------------------------------------
// StateEquationAdaptiveCole: update_speed_of_sound! (wcsph/system.jl:307-320) at the start
// of every kick.  k_vmax: per-block maxima of v.v over the fluid's current velocities (the
// caller-order v_ode), from which the gather takes the sound speed (adaptive_sound).
// ------------------------------------------------------------------------------------------
template <int ND>
__global__ void __launch_bounds__(kBlock)
    k_vmax(int nf, int vrows, const double *__restrict__ v, double *__restrict__ part)
{
    __shared__ double s[kBlock];
    double m = 0.0;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < nf; i += gridDim.x * kBlock) {
        double d = v[(size_t)i * vrows] * v[(size_t)i * vrows];
#pragma unroll
        for (int k = 1; k < ND; k++) d += v[(size_t)i * vrows + k] * v[(size_t)i * vrows + k];
        m = fmax(m, d);
    }
    s[threadIdx.x] = m;
    __syncthreads();
    for (int o = kBlock / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) s[threadIdx.x] = fmax(s[threadIdx.x], s[threadIdx.x + o]);
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

// ------------------------------------------------------------------------------------------
// FP64 integrals of the fluid state (tpsph_integrals): per-block partial sums over a fixed
// assignment of particles to blocks and a fixed tree inside each block, then one block sums
// the partials in block order -- the result does not depend on scheduling.
// ------------------------------------------------------------------------------------------
constexpr int kIntegrals = 8;
constexpr int kIntegralBlocks = 1024;

template <int ND>
__global__ void __launch_bounds__(kBlock)
    k_integrals(int nf, const double *__restrict__ v, const double *__restrict__ u,
                const double *__restrict__ m, DevParams P, double *__restrict__ part)
{
    __shared__ double s[kIntegrals][kBlock];
    double acc[kIntegrals] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < nf; i += gridDim.x * kBlock) {
        const double mi = m[i];
        const double rho = v[(size_t)i * (ND + 1) + ND];
        double v2 = 0.0, gx = 0.0;
#pragma unroll
        for (int d = 0; d < ND; d++) {
            const double vd = v[(size_t)i * (ND + 1) + d];
            acc[1 + d] += mi * vd;
            v2 += vd * vd;
            gx += P.g[d] * u[(size_t)i * ND + d];
        }
        acc[0] += mi;
        acc[4] += 0.5 * mi * v2;
        acc[5] -= mi * gx;
        acc[6] += mi / rho;
        acc[7] += rho;
    }
#pragma unroll
    for (int k = 0; k < kIntegrals; k++) s[k][threadIdx.x] = acc[k];
    __syncthreads();
    for (int o = kBlock / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
#pragma unroll
            for (int k = 0; k < kIntegrals; k++) s[k][threadIdx.x] += s[k][threadIdx.x + o];
        }
        __syncthreads();
    }
    if ((int)threadIdx.x < kIntegrals) part[(size_t)blockIdx.x * kIntegrals + threadIdx.x] = s[threadIdx.x][0];
}

__global__ void __launch_bounds__(kBlock) k_integrals_final(int nparts, const double *__restrict__ part,
                                                            double *__restrict__ out)
{
    if ((int)threadIdx.x >= kIntegrals) return;
    double acc = 0.0;
    for (int b = 0; b < nparts; b++) acc += part[(size_t)b * kIntegrals + threadIdx.x];
    out[threadIdx.x] = acc;
}

__global__ void k_rk_stage(int64_t n, double *__restrict__ y, double *__restrict__ tmp,
                           const double *__restrict__ k, double a, double b, double dt,
                           int first)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double t = first ? dt * k[i] : fma(dt, k[i], a * tmp[i]);
    tmp[i] = t;
    y[i] = fma(b, t, y[i]);
}

// y = a y + b x, the broadcasts of a low-storage Runge-Kutta step one at a time: b == 0 reads
// only y (y = a y), a == 0 only x (y = b x), both zero write zeros; otherwise fma(b, x, a y)
// (the rounding of muladd(b, x, a y)).
__global__ void k_axpby(int64_t n, double *__restrict__ y, double a, const double *x, double b)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (b == 0.0)
        y[i] = a == 0.0 ? 0.0 : a * y[i];
    else if (a == 0.0)
        y[i] = b * x[i];
    else
        y[i] = fma(b, x[i], a * y[i]);
}

// ------------------------------------------------------------------------------------------
// neighbour CSR export (parity tests): rows = cell-sorted points (rx, ry, rz; row_perm to the
// caller's order), columns = cell-sorted points with cell offsets col_start
// ------------------------------------------------------------------------------------------
template <int ND, bool FILL>
__global__ void k_nbr(DevParams P, int nrows, const double *__restrict__ rx,
                      const double *__restrict__ ry, const double *__restrict__ rz,
                      const int *__restrict__ row_perm, const int *__restrict__ col_start,
                      const double *__restrict__ cx, const double *__restrict__ cy,
                      const double *__restrict__ cz, const int *__restrict__ col_perm,
                      double hs, int *__restrict__ counts, const int64_t *__restrict__ offsets,
                      int *__restrict__ idx)
{
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nrows) return;
    const double xa = rx[s], ya = ry[s], za = (ND == 3) ? rz[s] : 0.0;
    Pencils<ND> it;
    it.init(P, xa, ya, za, hs);
    const int row = row_perm[s];
    int64_t o = FILL ? offsets[row] : 0;
    const int64_t b = o;
    int cnt = 0, jb, je;
    while (it.next(P, col_start, jb, je)) {
        for (int j = jb; j < je; j++) {
            const double d2 = dist2<ND>(xa - cx[j], ya - cy[j], (ND == 3) ? za - cz[j] : 0.0);
            if (d2 <= P.R2) {
                if (FILL) idx[o++] = col_perm[j];
                cnt++;
            }
        }
    }
    if (!FILL) {
        counts[row] = cnt;
        return;
    }
    for (int64_t k = b + 1; k < o; k++) {  // ascending columns
        int key = idx[k];
        int64_t j = k - 1;
        while (j >= b && idx[j] > key) {
            idx[j + 1] = idx[j];
            j--;
        }
        idx[j + 1] = key;
    }
}

// Pairs that the last kick's kernels evaluated (parity tests of the pair search): for every
// row particle, the candidates its kernel read -- the brick list (LDS indices mapped back to
// sorted indices through the brick's row tables, as the staging pass maps them), the int
// Verlet list, or the cell walk of an overflowed list or of the cell search -- that pass the
// kernel's exact test on the kick's positions: az2 <= d^2 <= R^2 for the fluid-fluid and
// fluid-wall sums (the pair terms), d^2 <= R^2 for the Adami sums of the walls.
struct EvalPairsArgs {
    int pair;           // TPSPH_PAIR_*
    int lists, bricks;  // the kick's pair search
    const int *ord, *tbase, *uidx;
    const unsigned short *nbr16;
    const int *nbr, *cnt, *wnbr, *wcnt;
    int ls;
    const int *anbr, *acnt;
    int lw;
    const int *w_perm;
};

template <int ND, bool FILL>
__global__ void k_eval_pairs(DevParams P, FluidView F, WallView Wv, EvalPairsArgs a,
                             int *__restrict__ counts, const int64_t *__restrict__ offsets,
                             int *__restrict__ idx)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    const bool wall_rows = a.pair == TPSPH_PAIR_WALL_FLUID;
    const int nrows = wall_rows ? P.nw : P.nf;
    if (r >= nrows) return;
    // the row particle: sorted index s (fluid rows in the kernels' target order)
    const int s = (!wall_rows && a.lists) ? a.ord[r] : r;
    double xa[3];
    if (wall_rows) {
        const double4 w = Wv.pos[s];
        xa[0] = w.x, xa[1] = w.y, xa[2] = w.z;
    } else {
        const double4 f = F.rec[2 * (size_t)s];
        xa[0] = f.x, xa[1] = f.y, xa[2] = f.z;
    }
    const int row = wall_rows ? a.w_perm[s] : F.perm[s];
    const bool wall_cols = a.pair == TPSPH_PAIR_FLUID_WALL;
    const double lower = wall_rows ? -1.0 : P.az2;
    int64_t o = FILL ? offsets[row] : 0;
    const int64_t o0 = o;
    int n_hit = 0;
    auto consider = [&](int j) {
        double xb[3];
        if (wall_cols) {
            const double4 w = Wv.pos[j];
            xb[0] = w.x, xb[1] = w.y, xb[2] = w.z;
        } else {
            const double4 f = F.rec[2 * (size_t)j];
            xb[0] = f.x, xb[1] = f.y, xb[2] = f.z;
        }
        const double d2 = dist2<ND>(xa[0] - xb[0], xa[1] - xb[1], (ND == 3) ? xa[2] - xb[2] : 0.0);
        if (d2 <= P.R2 && d2 >= lower) {
            if (FILL) idx[o++] = wall_cols ? a.w_perm[j] : F.perm[j];
            n_hit++;
        }
    };
    auto walk = [&](const int *start, double hs) {
        Pencils<ND> it;
        it.init(P, xa[0], xa[1], xa[2], hs);
        int jb, je;
        while (it.next(P, start, jb, je))
            for (int j = jb; j < je; j++) consider(j);
    };
    if (!a.lists) {
        if (wall_cols)
            walk(Wv.start, P.hs_wall);
        else
            walk(F.start, P.hs_fluid);
    } else if (wall_rows) {
        const int n = a.acnt[s];
        if (n >= 0)
            for (int k = 0; k < n; k++) consider(a.anbr[(size_t)k * a.lw + s]);
        else
            walk(F.start, P.hs_fluid);
    } else if (wall_cols) {
        const int n = a.wcnt[r];
        if (n >= 0)
            for (int k = 0; k < n; k++) consider(a.wnbr[(size_t)k * a.ls + r]);
        else
            walk(Wv.start, P.hs_wall);
    } else {
        const int n = a.cnt[r];
        const int first = a.bricks ? a.tbase[r] : -1;
        if (first >= 0) {  // the list of union records
            for (int k = 0; k < n; k++) {
                const int p = list_place(k);
                consider(a.uidx[first + a.nbr16[((size_t)(p >> 2) * a.ls + r) * 4 + (p & 3)] / 16]);
            }
        } else if (n >= 0) {
            for (int k = 0; k < n; k++) consider(a.nbr[(size_t)k * a.ls + r]);
        } else {
            walk(F.start, P.hs_fluid);
        }
    }
    if (!FILL) {
        counts[row] = n_hit;
        return;
    }
    for (int64_t k = o0 + 1; k < o; k++) {  // ascending columns
        const int key = idx[k];
        int64_t j = k - 1;
        while (j >= o0 && idx[j] > key) {
            idx[j + 1] = idx[j];
            j--;
        }
        idx[j + 1] = key;
    }
}

// cell-sorted SoA coordinates (and optionally {x, y, z, mass} records) of n points
template <int ND>
__global__ void k_positions(int n, const double *__restrict__ x, const int *__restrict__ perm,
                            double *__restrict__ xs, double *__restrict__ ys,
                            double *__restrict__ zs, double4 *__restrict__ pos,
                            const double *__restrict__ mass)
{
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int i = perm[s];
    const double a = x[(size_t)i * ND], b = x[(size_t)i * ND + 1];
    const double c = (ND == 3) ? x[(size_t)i * ND + 2] : 0.0;
    xs[s] = a;
    ys[s] = b;
    if (zs) zs[s] = c;
    if (pos) pos[s] = make_double4(a, b, c, mass ? mass[i] : 0.0);
}

template <typename T>
__global__ void k_unpermute(int n, const int *__restrict__ perm, const T *__restrict__ sorted,
                            T *__restrict__ out)
{
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    out[perm[s]] = sorted[s];
}

// tpsph_sort_particles: row j of the sorted state is row perm[j] of the caller's state (v
// with `vrows` doubles per particle, u with ND, the mass with one); po[j] = perm[j]
template <int ND>
__global__ void k_permute_state(int n, int vrows, const int *__restrict__ perm,
                                const double *__restrict__ v, const double *__restrict__ u,
                                const double *__restrict__ m, double *__restrict__ vo,
                                double *__restrict__ uo, double *__restrict__ mo,
                                int64_t *__restrict__ po)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const int i = perm[j];
    for (int d = 0; d < vrows; d++) vo[(size_t)j * vrows + d] = v[(size_t)i * vrows + d];
#pragma unroll
    for (int d = 0; d < ND; d++) uo[(size_t)j * ND + d] = u[(size_t)i * ND + d];
    mo[j] = m[i];
    if (po) po[j] = i;
}

// fluid pressure (p = .w of the second double4 of each record, half = 1) or density (.w of
// the first, half = 0) of the cell-sorted records
__global__ void k_record_pressure(int n, const double4 *__restrict__ rec, double *__restrict__ p,
                                  int half = 1)
{
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    p[s] = rec[2 * (size_t)s + half].w;
}


}  // namespace

namespace {



// Cell list of n points x (ND doubles per point, caller order) into start / perm, the members
// of a cell by their index.
template <int ND>
int build_cells(tpsph_handle *h, const int *flag, int n, const double *x, int *cell, int *rank,
                int *count, int *start, int *perm)
{
    // count is zero on entry (cleared at create, and again by k_scatter)
    const int nc = h->P.ncells;
    // (n = 0 too: it clears the scan's state)
    hipLaunchKernelGGL((k_cells<ND>), dim3(gate_blocks(n)), dim3(kBlock), 0, h->stream, h->dev, flag, n, x,
                       cell, rank, count);
    TRY(launch_check(h, "k_cells"));
    TRY(scan(h, flag, count, start, nc + 1));
    if (n > 0) {
        hipLaunchKernelGGL((k_scatter), dim3(gate_blocks(n)), dim3(kBlock), 0, h->stream, flag, n, cell, rank, start, perm, count);
        hipLaunchKernelGGL((k_sort_cells), dim3(gate_blocks(nc)), dim3(kBlock), 0, h->stream, flag, nc, start, perm);
    }
    return launch_check(h, "k_scatter/k_sort_cells");
}

// Whether the list kernel also runs the Adami pass: not before the densities are summed, and as a
// kernel of its own while the kernels are timed.
bool adami_in_lists(const tpsph_handle *h)
{
    return h->search == TPSPH_SEARCH_LISTS && !h->P.summation && !h->timing;
}

// Whether the bricks stage: the union rows of a brick of full size fit (small fluids have smaller
// bricks, but whether a call is accepted does not depend on the number of particles).
bool brick_rows_ok(const DevParams &P) { return P.full_rows <= kBrickMaxRows; }

// Whether the list build needs its larger tables.
bool wide_lists(const DevParams &P) { return P.nd == 3 && P.lr[1] > 2 && brick_rows_ok(P); }

// Fluid cell list (rebuilt only when flagged) + cell-sorted gather of (v, u).
template <int ND>
int update_fluid(tpsph_handle *h, const double *v, const double *u, bool gathered,
                 bool keep_order = false)
{
    const int nf = h->nf;
    if (nf == 0) return TPSPH_OK;
    if (keep_order) return TPSPH_OK;  // the order and the lists stand, the caller wrote the records
    if (!gathered) {  // else the stage kernel wrote the records of (v, u)
        TimedScope t(h, TPSPH_TIME_GATHER);
        hipLaunchKernelGGL((k_gather<ND, 0>), dim3(nblocks(nf)), dim3(kBlock), 0, h->stream, h->dev, u, v,
                           h->dyn ? gate_blocks(nf) : 0);
        TRY(launch_check(h, "k_gather<0>"));
    }
    {
        TimedScope t(h, TPSPH_TIME_CELL_LIST);
        const bool lists = h->search == TPSPH_SEARCH_LISTS;
        if (!h->f_head) {
            TRY(build_cells<ND>(h, h->flag, nf, u, h->f_cell, h->f_rank, h->f_count, h->f_start, h->f_perm));
            hipLaunchKernelGGL((k_gather<ND, 2>), dim3(gate_blocks(nf)), dim3(kBlock), 0, h->stream, h->dev, u, v, 0);
        } else if (h->sort_ctl) {
            const int items = std::min((nf + kSortThreads - 1) / kSortThreads, kSortItems);
            const int tiles = h->P.ncells / (kSortThreads * kScanItems) + 1;
            hipLaunchKernelGGL((k_sort<ND>), dim3(std::min(std::max(items, tiles), kSortItems)), dim3(kSortThreads), 0,
                               h->stream, h->dev, u, v, items, tiles);
        } else {
            hipLaunchKernelGGL((k_links<ND>), dim3(gate_blocks(nf)), dim3(kBlock), 0, h->stream, h->dev, u);
            launch_scan<true>(h->stream, h->flag, h->f_count, h->f_start, h->scan_state, h->P.ncells + 1);
            hipLaunchKernelGGL((k_gather<ND, 1>), dim3(gate_blocks(nf)), dim3(kBlock), 0, h->stream, h->dev, u, v, 0);
        }
        TRY(launch_check(h, "k_sort / k_gather<1>"));
        if (lists) {
            const int gb = std::max(1, std::min(h->nbricks, 2 * h->n_cu));
            // as many blocks for the walls as the Adami pass has lanes for, at most one turn
            const int gw = (int)std::min<int64_t>((kWallLanes * (int64_t)h->nw + kListThreads - 1) / kListThreads, 2 * h->n_cu);
            const auto build = wide_lists(h->P) ? k_brick_lists<ND, ND == 3> : k_brick_lists<ND, false>;
            hipLaunchKernelGGL(build, dim3(gw + gb), dim3(kListThreads), 0, h->stream, h->dev, gw, adami_in_lists(h));
            TRY(launch_check(h, "k_brick_lists"));
        }
        // the fluid kernel of this kick lowers the flag
    }
    return TPSPH_OK;
}

// Everything a kick does before the fluid pass: the sound speed (adaptive), the cell-sorted
// records of (v, u) with the fluid pressures, the rebuild of the cell list and the lists (if
// a particle left its skin), and the Adami pass of the walls.
template <int ND>
int prepare_impl(tpsph_handle *h, const double *v, const double *u, bool gathered,
                 bool keep_order = false)
{
    const int nf = h->nf, nw = h->nw;
    if (h->dyn && nf > 0) {
        // the sound speed of this kick comes from its velocities, before any pressure: the
        // records are then gathered again with it
        TimedScope t(h, TPSPH_TIME_GATHER);
        const int nb = gate_blocks(nf);
        hipLaunchKernelGGL((k_vmax<ND>), dim3(nb), dim3(kBlock), 0, h->stream, nf, h->P.vrows, v, h->vmax_part);
        TRY(launch_check(h, "k_vmax"));
        gathered = false;
    }
    TRY(update_fluid<ND>(h, v, u, gathered, keep_order));
    if (h->P.summation && nf > 0) {
        // compute_density! before the state equation (wcsph/system.jl:291-301, 323-326)
        TimedScope t(h, TPSPH_TIME_GATHER);
        if (h->search == TPSPH_SEARCH_LISTS && h->bricks)
            hipLaunchKernelGGL((k_sum_density_brick<ND>), dim3(std::max(1, std::min(h->nbricks, h->n_cu))),
                               dim3(kBrickThreads), 0, h->stream, h->dev);
        else if (h->search == TPSPH_SEARCH_LISTS)
            hipLaunchKernelGGL((k_sum_density_lists<ND>), dim3(nblocks(4 * (int64_t)nf)), dim3(kBlock), 0, h->stream, h->dev);
        else
            hipLaunchKernelGGL((k_sum_density<ND>), dim3(nblocks(nf)), dim3(kBlock), 0, h->stream, h->dev);
        hipLaunchKernelGGL((k_sum_finish), dim3(nblocks(nf)), dim3(kBlock), 0, h->stream, h->dev);
        TRY(launch_check(h, "k_sum_density"));
    }
    if (nw > 0 && (nf == 0 || keep_order || !adami_in_lists(h))) {
        TimedScope t(h, TPSPH_TIME_WALL);
        hipLaunchKernelGGL((k_wall<ND>), dim3(gate_blocks(kWallLanes * (int64_t)nw)), dim3(kBlock), 0, h->stream, h->dev);
        TRY(launch_check(h, "k_wall"));
    }
    return TPSPH_OK;
}

template <int ND>
int kick_impl(tpsph_handle *h, double *dv, const double *v, const double *u, bool gathered)
{
    const int nf = h->nf, nw = h->nw;
    TRY(prepare_impl<ND>(h, v, u, gathered));
    if (nf > 0) {
        TimedScope t(h, TPSPH_TIME_FLUID);
        if (h->P.ddgrad) {
            const bool lists = h->search == TPSPH_SEARCH_LISTS;
            if (lists && h->bricks)
                hipLaunchKernelGGL((k_antuono_gradient_brick<ND>),
                    dim3(std::max(1, std::min(h->nbricks, h->n_cu))), dim3(kBrickThreads), 0, h->stream, h->dev);
            else
                hipLaunchKernelGGL((k_antuono_gradient<ND>), dim3(nblocks(4 * (int64_t)nf)), dim3(kBlock), 0,
                                   h->stream, h->dev, lists);
            TRY(launch_check(h, "k_antuono_gradient"));
        }
        if (h->search == TPSPH_SEARCH_LISTS && h->bricks && h->mixed) {
            TRY(launch_fluid_brick_mixed(h, dv));
            hipLaunchKernelGGL((k_fluid_brick_global<ND>), dim3(std::max(1, std::min(h->nbricks, h->n_cu))),
                dim3(kBrickThreads), 0, h->stream, h->dev, dv);
            if (nw > 0)
                hipLaunchKernelGGL((k_fluid_walls<ND>), dim3(gate_blocks(4 * (int64_t)nf)), dim3(kBlock), 0, h->stream, h->dev, dv);
        } else if (h->search == TPSPH_SEARCH_LISTS && h->bricks) {
            const int vm = visc_mode(h->P);
            const bool ant = h->P.ddgrad != nullptr, sum = h->P.summation != 0;
            const auto brick =
                ant   ? (vm == kViscNone    ? k_fluid_brick<ND, kViscNone, true>
                         : vm == kViscAlpha ? k_fluid_brick<ND, kViscAlpha, true>
                                            : k_fluid_brick<ND, kViscAlphaBeta, true>)
                : sum ? (vm == kViscNone    ? k_fluid_brick<ND, kViscNone, false, true>
                         : vm == kViscAlpha ? k_fluid_brick<ND, kViscAlpha, false, true>
                                            : k_fluid_brick<ND, kViscAlphaBeta, false, true>)
                      : (vm == kViscNone    ? k_fluid_brick<ND, kViscNone>
                         : vm == kViscAlpha ? k_fluid_brick<ND, kViscAlpha>
                                            : k_fluid_brick<ND, kViscAlphaBeta>);
            hipLaunchKernelGGL(brick, dim3(std::max(1, std::min(h->nbricks, h->n_cu))), dim3(kBrickThreads), 0,
                h->stream, h->dev, dv);
            const auto walls = sum ? k_fluid_walls<ND, true> : k_fluid_walls<ND, false>;
            if (nw > 0)
                hipLaunchKernelGGL(walls, dim3(gate_blocks(4 * (int64_t)nf)), dim3(kBlock), 0, h->stream, h->dev, dv);
        } else if (h->search == TPSPH_SEARCH_LISTS) {
            hipLaunchKernelGGL((k_fluid_list<ND>), dim3(nblocks(nf)), dim3(kBlock), 0, h->stream, h->dev, dv);
        } else if (h->P.summation) {
            hipLaunchKernelGGL((k_fluid<ND, true>), dim3(nblocks(nf)), dim3(kBlock), 0, h->stream, h->dev, dv);
        } else {
            const auto cells = h->P.ddgrad ? k_fluid<ND, false, true> : k_fluid<ND>;
            hipLaunchKernelGGL(cells, dim3(nblocks(nf)), dim3(kBlock), 0, h->stream, h->dev, dv);
        }
        TRY(launch_check(h, "k_fluid"));
    }
    h->have_kick = true;
    return TPSPH_OK;
}



}  // namespace

// The device parameters of params for nf fluid and nw wall particles on the grid of the box
// [lo, hi] (one padding cell per side): kernel and state-equation constants, cells, skin
// radii and bricks.  Failures go to the create error (tpsph_last_error(NULL)).
int tpsph::derive_params(const tpsph_params *params, int nf, int nw, const double *lo,
                  const double *hi, DevParams &P, int &nbricks, double volume, int slots)
{
    const int nd = params->ndims;
    // --- derived parameters
    const double hl = params->smoothing_length;
    const double R = 2.0 * hl;  // compact_support(WendlandC2, h)
    P.nd = nd;
    P.nf = nf;
    P.nw = nw;
    P.use_visc = params->use_viscosity ? 1 : 0;
    P.summation = params->density_calculator == TPSPH_DENSITY_SUMMATION ? 1 : 0;
    P.vrows = nd + (P.summation ? 0 : 1);
    // density diffusion acts through the continuity equation, which SummationDensity has not
    P.use_dd = (params->use_density_diffusion && !P.summation) ? 1 : 0;
    P.clip_fluid = params->clip_fluid_eos ? 1 : 0;
    P.clip_wall = params->clip_wall_pressure ? 1 : 0;
    P.h = hl;
    P.h_inv = 1.0 / hl;
    P.R = R;
    P.R2 = R * R;
    P.two_h = 2.0 * hl;
    P.az2 = std::nextafter(R * R, INFINITY) - R * R;  // sqrt(eps(R^2))^2
    const double sigma = nd == 2 ? (7.0 / (4.0 * M_PI)) * (P.h_inv * P.h_inv)
                                 : (21.0 / (16.0 * M_PI)) * (P.h_inv * P.h_inv * P.h_inv);
    P.kval_c = sigma;
    P.kgrad_c = -5.0 * sigma * (P.h_inv * P.h_inv);
    P.rho0 = params->reference_density;
    P.c = params->sound_speed;
    P.gamma = params->exponent;
    P.inv_gamma = 1.0 / params->exponent;
    P.p_bg = params->background_pressure;
    P.B = P.rho0 * (P.c * P.c) / P.gamma;
    P.alpha = params->alpha;
    P.beta = params->beta;
    P.eps_h2 = params->epsilon * (hl * hl);
    P.av_c = params->alpha * P.c * hl;
    P.dd2 = P.use_dd ? 2.0 * params->delta * hl * P.c : 0.0;
    P.ddgrad = nullptr;  // set below for DensityDiffusionAntuono
    P.eps_hh = std::nextafter(hl * hl, INFINITY) - hl * hl;
    for (int d = 0; d < 3; d++) P.g[d] = d < nd ? params->acceleration[d] : 0.0;
    P.p_offset = params->pressure_offset;
    P.dyn = nullptr;  // set below for an adaptive state equation
    P.visc_w = params->wall_viscosity;
    P.w_alpha = params->wall_alpha;
    P.w_ac = params->wall_alpha * P.c;
    P.w_beta = params->wall_beta;
    P.w_eps_h2 = params->wall_epsilon * hl * hl;
    P.w_nu = params->wall_nu;
    P.nu_kin = params->alpha * hl * P.c / (2 * nd + 4);
    P.mach = params->mach_number_target;
    P.c_min = params->min_sound_speed;
    P.c_max = params->max_sound_speed;

    const int div = params->cell_divisions > 0 ? params->cell_divisions : 2;
    const int xdiv = params->x_cell_divisions > 0 ? params->x_cell_divisions : 2 * div;
    const double skin = params->skin >= 0.0 ? params->skin : 0.04;
    double extent = R;
    for (int d = 0; d < nd; d++) extent = std::fmax(extent, std::fmax(std::fabs(lo[d]), std::fabs(hi[d])) + 4.0 * R);
    // cell-interval rounding margin: far above the error of floor((x - lo) / cs)
    const double margin = 1e-9 * R + 64.0 * DBL_EPSILON * extent;
    P.half_skin = 0.5 * skin * R;
    P.half_skin2 = P.half_skin * P.half_skin;
    P.hs_fluid = P.half_skin + margin;
    P.hs_wall = margin;
    {
        const double rlf = R + 2.0 * P.half_skin + margin, rlw = R + P.half_skin + margin;
        P.rl2_fluid = rlf * rlf;
        P.rl2_wall = rlw * rlw;
        P.hs_list_fluid = 2.0 * P.half_skin + 2.0 * margin;
        P.hs_list_wall = P.half_skin + 2.0 * margin;
    }
    // k cells span the reach of a point: R (as bounded by the FP32 square roots of the pencil
    // widths, which run at most 2e-6 R above it), its own drift and a neighbour's drift
    const double span = (R * 1.00001 + 2.0 * P.hs_fluid) * (1.0 + 1e-9);
    int64_t ncells = 1;
    for (int d = 0; d < 3; d++) {
        const double cs = span / (d == 0 ? xdiv : div);
        P.cs[d] = cs;
        P.inv_cs[d] = 1.0 / cs;
        if (d < nd) {
            P.lo[d] = lo[d] - cs;
            int64_t n = (int64_t)std::ceil((hi[d] + cs - P.lo[d]) * P.inv_cs[d]) + 1;
            if (n < 1) n = 1;
            if (n > (1 << 20))
                return fail(nullptr, TPSPH_ERR_ARGUMENT, "domain box too large for the cell grid");
            P.n[d] = (int)n;
        } else {
            P.lo[d] = 0.0;
            P.n[d] = 1;
        }
        ncells *= P.n[d];
    }
    if (ncells > (int64_t)INT32_MAX / 4)
        return fail(nullptr, TPSPH_ERR_ARGUMENT, "cell grid too large (domain / smoothing_length)");
    P.ncells = (int)ncells;
    // FP32 test of the list builds.  A position up to a box length outside the grid box (list_f32)
    // is stored as fl32(x - lo), off by at most 2^-23 L (L the box's longest side), so an FP32
    // distance d' is off by at most 7 * 2^-24 L + 2^-24 d from the FP64 one d, and its square by
    // a further 3.1 * 2^-24 relative: with e = 8 * 2^-24 (L + rl) the bound leaves a margin of
    // at least 2^-24 rl beyond the list radius rl.  The lists take whatever is within it: a
    // few candidates more than the list radius holds (every kick applies the exact radius
    // test), in exchange for no FP64 test in the build
    {
        const double u = 0x1p-24;
        double L = 0.0;
        for (int d = 0; d < 3; d++) {
            P.box[d] = d < nd ? P.n[d] * P.cs[d] : 0.0;
            L = std::fmax(L, P.box[d]);
        }
        auto bound = [&](double rl2) {
            const double rl = std::sqrt(rl2), e = 8.0 * u * (L + rl);
            const double out2 = (rl + e) * (rl + e) * (1.0 + 4.0 * u);
            const float fo = (float)out2;
            return (double)fo < out2 ? std::nextafter(fo, INFINITY) : fo;
        };
        P.list_out2 = bound(P.rl2_fluid);
        P.wlist_out2 = bound(P.rl2_wall);
    }
    {
        // bricks of 3 (3D) or 8 (2D) cell spans per side, about 3.1 R (8.3 R) wide, in 3D
        // shortened along x to 2.75 spans: at h = 1.2 dx a 3D brick holds up to 448 targets
        // and a union of at most about 2020 particles at rest, inside the LDS records of the
        // brick kernel (full 3-span bricks: 512 targets, and the unions of 5-10 % of the
        // bricks exceed the records and take the slower global path)
        // DensityDiffusionAntuono stages the density gradients too: in 3D its records hold
        // kBrickCapGrad particles, so its bricks are one cell shorter along y and z (unions of
        // about 5/6 the size, about 320 targets)
        const int per = nd == 3 ? 3 : 8;
        const bool grad = params->use_density_diffusion == TPSPH_DIFFUSION_ANTUONO && nd == 3;
        P.brick_cap = grad ? kBrickCapGrad : kBrickCap;
        for (int d = 0; d < 3; d++) {
            P.bc[d] = d < nd ? per * (d == 0 ? xdiv : div) : 1;
            if (nd == 3 && d == 0) P.bc[d] = std::max(1, P.bc[d] * 11 / 12);
            if (grad && d >= 1) P.bc[d] = std::max(1, P.bc[d] - 1);
        }
        // union rows: cells within the list radius of the brick box (grown by the margin)
        const double rl = R + 2.0 * P.half_skin + margin, reach = R + P.hs_list_fluid;
        auto union_rows = [&] {
            int rows = 1;
            for (int d = 1; d < nd; d++) rows *= P.bc[d] + 2 * P.ur[d];
            return rows;
        };
        auto union_cells = [&] { return P.bc[0] + 2 * ((int)std::floor((rl + 4.0 * margin) / P.cs[0]) + 1) + 2; };
        for (int d = 0; d < 3; d++) {
            const bool yz = d >= 1 && d < nd;
            P.ur[d] = yz ? (int)std::ceil(rl / P.cs[d]) + 1 : 0;
            P.lr[d] = yz ? (int)std::ceil(reach / P.cs[d]) : 0;  // of a target's pencils
        }
        P.full_rows = union_rows();
        // (they do not fit only where the margin is no longer small against a cell: a box more
        // than 1e12 R from the origin)
        if (P.full_rows * union_cells() > (nd == 2 ? ListsSmem<2, false>::kCellTab
                                           : P.lr[1] > 2 ? ListsSmem<3, true>::kCellTab
                                                         : ListsSmem<3, false>::kCellTab))
            P.full_rows = INT_MAX;
        // A small fluid in full bricks leaves most of the chip without one: its bricks shrink
        // until they are about as many as the device takes at a time (3/4 of it: the bricks on
        // the surface are not full), down to 50 targets.  Beyond that a second turn costs
        // more than the smaller bricks save.  Fluid pass at 1,800 / 7,200 / 45,000 particles
        // in 2D: 15.8 / 17.0 / 17.4 us with full bricks, 12.4 / 13.3 / 15.9 with these; at
        // 9,537 / 31,250 / 48,778 in 3D 31.6 / 33.3 / 35.7 against 19.5 / 27.6 / 29.0; bricks of
        // half the size at 45,000 and 48,778: 21.0 and 38.5.  The order of every sum is
        // the same whatever the bricks.
        // (Not for more particles than that many bricks hold: masses that do not fit the spacing
        // would ask for bricks of single cells, whose unions add up beyond 32 bits.)
        if (volume > 0.0 && slots > 0 && nf <= 0.75 * slots * P.brick_cap) {
            double cells = 1.0, cell_volume = 1.0;
            for (int d = 0; d < nd; d++) {
                cells *= P.bc[d];
                cell_volume *= P.cs[d];
            }
            const double targets = std::fmax(50.0, nf / (0.75 * slots));
            const double f = std::pow(targets * volume / cell_volume / cells, 1.0 / nd);
            for (int d = 0; d < nd && f < 1.0; d++)
                P.bc[d] = std::max(1, (int)std::floor(P.bc[d] * f + 0.5));
        }
        int64_t nb = 1;
        for (int d = 0; d < 3; d++) {
            P.nb[d] = (P.n[d] + P.bc[d] - 1) / P.bc[d];
            nb *= P.nb[d];
        }
        nbricks = (int)nb;
        P.maxr = union_rows();
        P.ctab = union_cells();
        P.rl_union2 = (rl + margin) * (rl + margin);
        P.hs_union = margin;
    }
    return TPSPH_OK;
}

int tpsph::validate(const tpsph_params *p, int64_t nf, int64_t nw, const double *fm, const double *wx,
             const double *wm)
{
    auto bad = [](const std::string &m) { return fail(nullptr, TPSPH_ERR_ARGUMENT, m); };
    if (!p) return bad("params is NULL");
    if (p->ndims != 2 && p->ndims != 3) return bad("ndims must be 2 or 3");
    if (p->kernel != TPSPH_KERNEL_WENDLAND_C2) return bad("only WendlandC2Kernel is implemented");
    if (p->memory != TPSPH_MEM_DEVICE && p->memory != TPSPH_MEM_HOST)
        return bad("memory must be TPSPH_MEM_DEVICE or TPSPH_MEM_HOST");
    if (nf < 0 || nw < 0) return bad("particle counts must be non-negative");
    if (nf > (int64_t)1 << 26 || nw > (int64_t)1 << 26)
        return bad("particle counts above 2^26 per system exceed the 32-bit byte offsets of "
                   "this build");
    if (!(p->smoothing_length > 0.0)) return bad("`smoothing_length` must be positive");
    if (!(p->reference_density > DBL_EPSILON))
        return bad("`reference_density` needs to be positive and larger than eps()");
    if (!(p->sound_speed > 0.0)) return bad("`sound_speed` must be positive");
    if (p->wall_viscosity < 0 || p->wall_viscosity > 2)
        return bad("wall_viscosity must be 0 (nothing), 1 (ArtificialViscosityMonaghan) or 2 "
                   "(ViscosityAdami)");
    if (p->wall_viscosity && p->use_viscosity != 1)
        return bad("a wall viscosity needs the fluid's ArtificialViscosityMonaghan (its "
                   "kinematic viscosity enters the wall terms)");
    if (p->wall_viscosity && !(p->wall_epsilon > 0.0)) return bad("`wall_epsilon` must be positive");
    if (p->adaptive_sound_speed) {
        if (!(p->mach_number_target > 0.0)) return bad("`mach_number_target` must be positive");
        if (!(p->min_sound_speed > 0.0)) return bad("`min_sound_speed` must be positive");
        if (!(p->max_sound_speed >= p->min_sound_speed))
            return bad("`max_sound_speed` must not be below `min_sound_speed`");
    }
    if (!(p->exponent > 0.0)) return bad("`exponent` must be positive");
    if (p->cell_divisions < 0 || p->cell_divisions > 4) return bad("cell_divisions must be in 0..4");
    if (p->x_cell_divisions < 0 || p->x_cell_divisions > 8)
        return bad("x_cell_divisions must be in 0..8");
    if (p->pair_search < TPSPH_SEARCH_AUTO || p->pair_search > TPSPH_SEARCH_CELLS)
        return bad("pair_search must be one of enum tpsph_pair_search");
    if (p->use_density_diffusion < TPSPH_DIFFUSION_NONE ||
        p->use_density_diffusion > TPSPH_DIFFUSION_ANTUONO)
        return bad("use_density_diffusion must be one of enum tpsph_density_diffusion");
    if (!(p->skin < 1.0)) return bad("skin must be below 1 (a fraction of the compact support)");
    if (p->precision != TPSPH_PRECISION_FP64 && p->precision != TPSPH_PRECISION_MIXED)
        return bad("precision must be TPSPH_PRECISION_FP64 or TPSPH_PRECISION_MIXED");
    if (p->density_calculator != TPSPH_DENSITY_CONTINUITY &&
        p->density_calculator != TPSPH_DENSITY_SUMMATION)
        return bad("density_calculator must be one of enum tpsph_density_calculator");
    if (p->density_calculator == TPSPH_DENSITY_SUMMATION && p->precision != TPSPH_PRECISION_FP64)
        return bad("SummationDensity runs in FP64 (TPSPH_PRECISION_FP64)");
    if (p->precision == TPSPH_PRECISION_MIXED && p->use_viscosity && p->beta != 0.0)
        return bad("precision TPSPH_PRECISION_MIXED evaluates ArtificialViscosityMonaghan with "
                   "beta = 0 only");
    if (nf > 0 && !fm) return bad("fluid_mass is NULL");
    if (nw > 0 && (!wx || !wm)) return bad("wall_coordinates / wall_mass is NULL");
    return TPSPH_OK;
}

int tpsph::kick_dispatch(tpsph_handle *h, double *dv, const double *v, const double *u,
                         bool gathered)
{
    return h->nd == 2 ? kick_impl<2>(h, dv, v, u, gathered) : kick_impl<3>(h, dv, v, u, gathered);
}

int tpsph::prepare_dispatch(tpsph_handle *h, const double *v, const double *u, bool keep_order)
{
    return h->nd == 2 ? prepare_impl<2>(h, v, u, false, keep_order)
                      : prepare_impl<3>(h, v, u, false, keep_order);
}

const double tpsph::kCkA[5] = {0.0, -567301805773.0 / 1357537059087.0,
                               -2404267990393.0 / 2016746695238.0,
                               -3550918686646.0 / 2091501179385.0,
                               -1275806237668.0 / 842570457699.0};
const double tpsph::kCkB[5] = {1432997174477.0 / 9575080441755.0,
                               5161836677717.0 / 13612068292357.0,
                               1720146321549.0 / 2090206949498.0,
                               3134564353537.0 / 4481467310338.0,
                               2277821191437.0 / 14882151754819.0};

int tpsph::run_ck2n54(tpsph_handle *h, double *v, double *u, double dt, int64_t nsteps,
                      double *store_v, double *store_u)
{
    if (!h->sol_dv) {
        TRY(dalloc(h, &h->sol_dv, v_len(h)));
        TRY(dalloc(h, &h->sol_tv, v_len(h)));
        TRY(dalloc(h, &h->sol_tu, u_len(h)));
    }
    if (h->P.summation) {
        // SummationDensity: v is the velocity, so the drift slope of u is v itself; the stage
        // updates u (with the v of the stage state) before v, then the next kick gathers and
        // sums the densities of the new state
        const int64_t n = (int64_t)h->nf * h->nd;
        const unsigned grid = (unsigned)((n + kBlock - 1) / kBlock);
        if (store_v) return fail(h, TPSPH_ERR_ARGUMENT, "reverse mode needs ContinuityDensity");
        for (int64_t s = 0; s < nsteps; s++) {
            for (int i = 0; i < 5; i++) {
                TRY(kick_dispatch(h, h->sol_dv, v, u, false));
                TimedScope ts(h, TPSPH_TIME_STAGE);
                hipLaunchKernelGGL((k_rk_stage), dim3(grid), dim3(kBlock), 0, h->stream, n, u,
                                   h->sol_tu, v, kCkA[i], kCkB[i], dt, (int)(i == 0));
                hipLaunchKernelGGL((k_rk_stage), dim3(grid), dim3(kBlock), 0, h->stream, n, v,
                                   h->sol_tv, h->sol_dv, kCkA[i], kCkB[i], dt, (int)(i == 0));
                TRY(launch_check(h, "k_rk_stage"));
            }
        }
        h->have_kick = false;
        return TPSPH_OK;
    }
    // every stage kernel also writes the cell-sorted records of the new state, so the kicks
    // after the first skip the gather
    bool gathered = false;
    for (int64_t s = 0; s < nsteps; s++) {
        for (int i = 0; i < 5; i++) {
            if (store_v) {  // the state this stage's kick sees
                const size_t k = (size_t)(5 * s + i);
                HIP_TRY(h, hipMemcpyAsync(store_v + k * v_len(h), v, v_len(h) * sizeof(double),
                                          hipMemcpyDeviceToDevice, h->stream));
                HIP_TRY(h, hipMemcpyAsync(store_u + k * u_len(h), u, u_len(h) * sizeof(double),
                                          hipMemcpyDeviceToDevice, h->stream));
                // the stored states are what the caller keeps: the last kick and stage would
                // only advance (v, u) past them
                if (s == nsteps - 1 && i == 4) break;
            }
            TRY(kick_dispatch(h, h->sol_dv, v, u, gathered));
            TimedScope ts(h, TPSPH_TIME_STAGE);
            hipLaunchKernelGGL(h->nd == 2 ? k_ck_stage_gather<2> : k_ck_stage_gather<3>, dim3(nblocks(h->nf)),
                               dim3(kBlock), 0, h->stream, h->dev, v, u, h->sol_tv, h->sol_tu, h->sol_dv,
                               kCkA[i], kCkB[i], dt, (int)(i == 0));
            TRY(launch_check(h, "k_ck_stage_gather"));
            gathered = true;
        }
    }
    // the state has advanced past the last kick: its pressures belong to no current state
    h->have_kick = false;
    return TPSPH_OK;
}

namespace {


__global__ void k_put_handle(DevHandle image, DevHandle *dev) { *dev = image; }

// Writes what the kernels read of the handle to h->dev (by a kernel: no host memory is read
// later, so the write can be captured in a graph).
int put_handle(tpsph_handle *h)
{
    DevHandle d;
    d.P = h->P;
    d.f_start = h->f_start; d.f_perm = h->f_perm; d.xs = h->xs; d.ys = h->ys; d.zs = h->zs;
    d.rec = h->rec; d.vol = h->vol; d.xf = h->xf;
    d.w_start = h->w_start; d.wx = h->wx; d.wy = h->wy; d.wz = h->wz; d.wpos = h->wpos;
    d.wpv = h->wpv; d.wvel = h->wvel; d.wxf = h->wxf; d.pw = h->pw; d.rhow = h->rhow;
    d.flag = h->flag; d.f_head = h->f_head; d.f_next = h->f_rank; d.iperm = h->iperm;
    d.nrebuild = h->nrebuild; d.counters = h->counters; d.scan_state = h->scan_state;
    d.scan_words = scan_words(h->P.ncells + 1);
    d.f_count = h->f_count; d.sort_ctl = h->sort_ctl;
    d.snap = h->snap; d.mass = h->f_mass; d.wall_near = h->wall_near;
    d.bcount = h->bcount; d.nel = h->nel; d.ord = h->ord; d.tbase = h->tbase; d.uidx = h->uidx;
    d.nbr = h->nbr; d.cnt = h->cnt; d.wnbr = h->wnbr; d.wcnt = h->wcnt; d.wtargets = h->wtargets;
    d.noverflow = h->search == TPSPH_SEARCH_LISTS ? h->counters + kCountOverflow : nullptr;
    d.bwork = h->bwork; d.bfall = h->bfall; d.bhead = h->bhead; d.nbr16 = h->nbr16; d.thead = h->thead;
    d.uidx_cap = (int)h->uidx_cap; d.ls = h->ls; d.cap_f = h->cap_f; d.cap_w = h->cap_w;
    // (without fluid no list is ever built: the walls walk the cells, which are empty)
    d.wactive = h->nf > 0 ? h->wactive : nullptr;
    d.anbr = h->anbr; d.acnt = h->acnt; d.lw = h->lw; d.cap_a = h->cap_a;
    d.dyn = h->dyn; d.ddgrad = h->ddgrad; d.vmax_part = h->vmax_part; d.sum_rho = h->sum_rho;
    d.alpha = h->params.alpha; d.delta = h->params.delta;
    hipLaunchKernelGGL((k_put_handle), dim3(1), dim3(1), 0, h->stream, d, h->dev);
    return launch_check(h, "k_put_handle");
}

// CSR of nrows rows in the caller's order from a count launch and a fill launch of the same
// kernel: launch(fill, counts, offsets, idx).  offsets / idx may be host or device memory.
template <typename Launch>
int emit_csr(tpsph_handle *h, int nrows, Launch launch, int64_t *offsets, int32_t *idx,
             int64_t capacity)
{
    int *counts = nullptr;
    int64_t *doff = nullptr;
    int *didx = nullptr;
    TRY(dalloc(h, &counts, (size_t)nrows));
    std::vector<int> hc((size_t)nrows);
    std::vector<int64_t> ho((size_t)nrows + 1, 0);
    int rc = TPSPH_OK;
    if (nrows > 0) {
        launch(false, counts, nullptr, nullptr);
        rc = launch_check(h, "pair count");
        if (rc == TPSPH_OK) {
            hipError_t e = hipMemcpyAsync(hc.data(), counts, (size_t)nrows * sizeof(int), hipMemcpyDeviceToHost, h->stream);
            if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
            if (e != hipSuccess) rc = fail(h, TPSPH_ERR_HIP, std::string("neighbour counts: ") + hipGetErrorString(e));
        }
    }
    for (int r = 0; r < nrows; r++) ho[(size_t)r + 1] = ho[(size_t)r] + hc[(size_t)r];
    const int64_t total = ho[(size_t)nrows];
    if (rc == TPSPH_OK) {
        hipError_t e = hipMemcpy(offsets, ho.data(), ho.size() * sizeof(int64_t), hipMemcpyDefault);
        if (e != hipSuccess) rc = fail(h, TPSPH_ERR_HIP, std::string("offsets: ") + hipGetErrorString(e));
    }
    if (rc == TPSPH_OK && idx != nullptr && capacity < total)
        rc = fail(h, TPSPH_ERR_CAPACITY, "idx capacity is smaller than the number of pairs");
    if (rc == TPSPH_OK && idx != nullptr && total > 0) {
        rc = dalloc(h, &doff, ho.size());
        if (rc == TPSPH_OK) rc = dalloc(h, &didx, (size_t)total);
        if (rc == TPSPH_OK) {
            hipError_t e = hipMemcpy(doff, ho.data(), ho.size() * sizeof(int64_t), hipMemcpyHostToDevice);
            if (e != hipSuccess) rc = fail(h, TPSPH_ERR_HIP, "offsets upload failed");
        }
        if (rc == TPSPH_OK) {
            launch(true, nullptr, doff, didx);
            rc = launch_check(h, "pair fill");
        }
        if (rc == TPSPH_OK) {
            hipError_t e = hipMemcpyAsync(idx, didx, (size_t)total * sizeof(int), hipMemcpyDefault, h->stream);
            if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
            if (e != hipSuccess) rc = fail(h, TPSPH_ERR_HIP, std::string("neighbour lists: ") + hipGetErrorString(e));
        }
    }
    (void)hipFree(counts);
    (void)hipFree(doff);
    (void)hipFree(didx);
    return rc;
}

// ------------------------------------------------------------------------------------------
// Kick without allocation (tpsph_kick_noalloc): every intermediate array of one kick lives in
// a file-scope device array, `scratch`, laid out anew on each call.  Host code reaches the
// array through the address hipGetSymbolAddress returns on each device (the symbol itself is
// a host-side stand-in and never a device address).  Counters and histograms are cleared
// by kernels, so the call records no memset (it can be captured in a HIP graph).
// ------------------------------------------------------------------------------------------
constexpr size_t kScratchBytes = size_t(64) << 20;  // 64 MiB per device
// behind them what depends on no particle: the kernels' copy of the handle and the scan's state
// (at most one word per kScanTile of the cells that fit, 17 bytes each)
constexpr size_t kScratchHandle = 2048, kScratchTail = size_t(16) << 10;
static_assert(sizeof(DevHandle) <= kScratchHandle &&
                  kScratchHandle + 8 * (kScratchBytes / 17 / kScanTile + 2) <= kScratchTail,
              "the tail holds the handle and the scan's state");
constexpr int kMaxDevices = 64;

__device__ __align__(256) unsigned char scratch[kScratchBytes + kScratchTail];

__global__ void k_fill_i32(int *p, int value, int n)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        p[i] = value;
}

__global__ void k_fill_u8(unsigned char *p, unsigned char value, int n)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        p[i] = value;
}

__global__ void k_fill_f64(double *p, double value, int n)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        p[i] = value;
}

// device address of `scratch` on the current device, looked up once per device
int scratch_base(unsigned char **base)
{
    static std::mutex mu;
    static unsigned char *addr[kMaxDevices] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
        return fail(nullptr, TPSPH_ERR_HIP, "tpsph_kick_noalloc: no current HIP device");
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(nullptr, TPSPH_ERR_HIP,
                        std::string("tpsph_kick_noalloc: hipGetSymbolAddress(scratch): ") +
                            hipGetErrorString(e));
        addr[dev] = static_cast<unsigned char *>(p);
    }
    *base = addr[dev];
    return TPSPH_OK;
}

// Bump allocator over the scratch array (256-byte aligned regions).
struct ScratchLayout {
    unsigned char *base;
    size_t used = 0;
    template <typename T>
    T *take(size_t count)
    {
        T *p = reinterpret_cast<T *>(base ? base + used : nullptr);
        used += (std::max<size_t>(count, 1) * sizeof(T) + 255) / 256 * 256;
        return p;
    }
};

// The kick of kick_impl with the cell walk (TPSPH_SEARCH_CELLS), fluid and wall cell lists
// built from scratch, on a handle whose arrays all point into the scratch array.  With
// base == nullptr only the layout is measured (h->... stay null, nothing is launched).
template <int ND>
int noalloc_kick(tpsph_handle *h, unsigned char *base, size_t *bytes, const double *fluid_mass,
                 const double *wall_x, const double *wall_mass, double *dv, const double *v,
                 const double *u)
{
    const int nf = h->nf, nw = h->nw;
    const int nc = h->P.ncells;
    ScratchLayout L{base};
    h->flag = L.take<int>(1);
    // a word per 2,048 cells, which the scan once kept here: the sizes that fit are an interface
    L.take<int>(((size_t)nc + 1 + 2047) / 2048 + 1);
    h->f_cell = L.take<int>(nf);
    h->f_rank = L.take<int>(nf);
    h->f_perm = L.take<int>(nf);
    h->iperm = L.take<int>(nf);
    h->f_count = L.take<int>((size_t)nc + 1);
    h->f_start = L.take<int>((size_t)nc + 1);
    h->xs = L.take<double>((size_t)nf + kPad);
    h->ys = L.take<double>((size_t)nf + kPad);
    h->zs = L.take<double>((size_t)nf + kPad);
    h->snap = L.take<double>((size_t)ND * nf);
    h->rec = L.take<double4>(2 * (size_t)nf);
    h->vol = L.take<double2>(nf);
    int *w_cell = L.take<int>(nw), *w_rank = L.take<int>(nw), *w_count = L.take<int>((size_t)nc + 1);
    h->w_start = L.take<int>((size_t)nc + 1);
    h->w_perm = L.take<int>(nw);
    h->wx = L.take<double>((size_t)nw + kPad);
    h->wy = L.take<double>((size_t)nw + kPad);
    h->wz = L.take<double>((size_t)nw + kPad);
    h->wpos = L.take<double4>(nw);
    h->wpv = L.take<double2>(nw);
    h->pw = L.take<double>(nw);
    h->rhow = L.take<double>(nw);
    h->wall_near = L.take<unsigned char>(nc);
    *bytes = L.used;
    if (!base) return TPSPH_OK;
    h->dev = reinterpret_cast<DevHandle *>(base + kScratchBytes);
    h->scan_state = reinterpret_cast<unsigned long long *>(base + kScratchBytes + kScratchHandle);
    hipStream_t st = h->stream;
    const double nan = __builtin_nan("");
    // what must start at zero (or NaN): histograms, the wall-near flags, the SoA padding
    hipLaunchKernelGGL((k_fill_i32), dim3(gate_blocks(nc + 1)), dim3(kBlock), 0, st, h->f_count, 0, nc + 1);
    hipLaunchKernelGGL((k_fill_i32), dim3(gate_blocks(nc + 1)), dim3(kBlock), 0, st, w_count, 0, nc + 1);
    if (nf == 0)  // no cell list is built then
        hipLaunchKernelGGL((k_fill_i32), dim3(gate_blocks(nc + 1)), dim3(kBlock), 0, st, h->f_start, 0, nc + 1);
    hipLaunchKernelGGL((k_fill_u8), dim3(gate_blocks(nc)), dim3(kBlock), 0, st, h->wall_near, (unsigned char)0, nc);
    for (double *a : {h->xs, h->ys, h->zs})
        hipLaunchKernelGGL((k_fill_f64), dim3(gate_blocks(nf + kPad)), dim3(kBlock), 0, st, a, nan, nf + kPad);
    for (double *a : {h->wx, h->wy, h->wz})
        hipLaunchKernelGGL((k_fill_f64), dim3(gate_blocks(nw + kPad)), dim3(kBlock), 0, st, a, nan, nw + kPad);
    hipLaunchKernelGGL((k_set_i32), dim3(1), dim3(1), 0, st, h->flag, 1);
    TRY(launch_check(h, "tpsph_kick_noalloc clearing"));
    h->f_mass = const_cast<double *>(fluid_mass);
    TRY(put_handle(h));
    // static walls: cell list, sorted positions and masses, cells near walls
    if (nw > 0) {
        TRY(build_cells<ND>(h, nullptr, nw, wall_x, w_cell, w_rank, w_count, h->w_start, h->w_perm));
        hipLaunchKernelGGL((k_positions<ND>), dim3(nblocks(nw)), dim3(kBlock), 0, st, nw, wall_x,
                           h->w_perm, h->wx, h->wy, ND == 3 ? h->wz : nullptr, h->wpos, wall_mass);
        hipLaunchKernelGGL((k_wall_near<ND>), dim3(nblocks(nw)), dim3(kBlock), 0, st, h->P, nw, h->wpos, h->wall_near);
        TRY(launch_check(h, "tpsph_kick_noalloc walls"));
    }
    return kick_impl<ND>(h, dv, v, u, false);
}

}  // namespace

// ==========================================================================================
// C ABI
// ==========================================================================================
extern "C" {

int tpsph_abi_version(void) { return TPSPH_ABI_VERSION; }

const char *tpsph_last_error(const tpsph_handle *h)
{
    return h ? h->last_error.c_str() : g_create_error.c_str();
}

int tpsph_create(const tpsph_params *params, int64_t n_fluid, int64_t n_wall,
                 const double *fluid_mass, const double *wall_coordinates,
                 const double *wall_mass, void *stream, tpsph_handle **out)
{
    if (!out) return fail(nullptr, TPSPH_ERR_ARGUMENT, "out is NULL");
    *out = nullptr;
    TRY(validate(params, n_fluid, n_wall, fluid_mass, wall_coordinates, wall_mass));
    tpsph_handle *h = new (std::nothrow) tpsph_handle();
    if (!h) return fail(nullptr, TPSPH_ERR_HIP, "out of host memory");
    h->params = *params;
    h->nd = params->ndims;
    h->nf = (int)n_fluid;
    h->nw = (int)n_wall;
    h->stream = (hipStream_t)stream;
    const int nd = h->nd;
    const bool host = is_host(h);
    const hipMemcpyKind in_kind = host ? hipMemcpyHostToDevice : hipMemcpyDeviceToDevice;

    std::vector<double> wxh((size_t)nd * h->nw);
    if (h->nw > 0) {
        hipError_t e = hipMemcpy(wxh.data(), wall_coordinates, wxh.size() * sizeof(double),
                                 host ? hipMemcpyHostToHost : hipMemcpyDeviceToHost);
        if (e != hipSuccess) {
            std::string m = std::string("copy of wall_coordinates: ") + hipGetErrorString(e);
            delete h;
            return fail(nullptr, TPSPH_ERR_HIP, m);
        }
    }

    // --- grid: the domain box (or the wall box when unset), one padding cell per side
    double lo[3], hi[3];
    bool have_box = true;
    for (int d = 0; d < nd; d++)
        if (!(params->domain_min[d] < params->domain_max[d])) have_box = false;
    for (int d = 0; d < nd; d++) {
        lo[d] = have_box ? params->domain_min[d] : INFINITY;
        hi[d] = have_box ? params->domain_max[d] : -INFINITY;
    }
    for (int i = 0; i < h->nw; i++)
        for (int d = 0; d < nd; d++) {
            lo[d] = std::fmin(lo[d], wxh[(size_t)i * nd + d]);
            hi[d] = std::fmax(hi[d], wxh[(size_t)i * nd + d]);
        }
    for (int d = 0; d < nd; d++)
        if (!(lo[d] <= hi[d])) {
            lo[d] = 0.0;
            hi[d] = 0.0;
        }
    {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0)
            h->n_cu = cus;
    }
    // mean masses, for the capacities of the Verlet lists and the size of the bricks
    double mf = 0.0, mw = 0.0;
    if (params->pair_search != TPSPH_SEARCH_CELLS) {
        std::vector<double> mh((size_t)std::max(h->nf, h->nw));
        auto mean = [&](const double *src, int n) {
            if (n == 0) return 0.0;
            if (hipMemcpy(mh.data(), src, (size_t)n * sizeof(double),
                          host ? hipMemcpyHostToHost : hipMemcpyDeviceToHost) != hipSuccess)
                return -1.0;
            double acc = 0.0;
            for (int i = 0; i < n; i++) acc += mh[i];
            return acc / n;
        };
        mf = mean(fluid_mass, h->nf);
        mw = mean(wall_mass, h->nw);
        if (mf < 0.0 || mw < 0.0) {
            delete h;
            return fail(nullptr, TPSPH_ERR_HIP, "copy of the masses failed");
        }
    }
    {
        const int slots = params->precision == TPSPH_PRECISION_MIXED ? 2 * h->n_cu : h->n_cu;
        const int rc = derive_params(params, h->nf, h->nw, lo, hi, h->P, h->nbricks,
                                     mf / params->reference_density, slots);
        if (rc != TPSPH_OK) {
            delete h;
            return rc;
        }
    }
    DevParams &P = h->P;
    const int64_t ncells = P.ncells;
    h->search = params->pair_search;
    // SummationDensity on the Verlet lists needs the brick kernel (P.maxr within one scan
    // block); the automatic choice takes the cell walk otherwise
    const bool sum_lists_ok = !P.summation || brick_rows_ok(P);
    if (h->search == TPSPH_SEARCH_AUTO)
        h->search = (P.half_skin > 0.0 && sum_lists_ok) ? TPSPH_SEARCH_LISTS : TPSPH_SEARCH_CELLS;
    if (h->search == TPSPH_SEARCH_LISTS && !sum_lists_ok) {
        delete h;
        return fail(nullptr, TPSPH_ERR_ARGUMENT,
                    "SummationDensity with TPSPH_SEARCH_LISTS needs the brick kernel: the "
                    "default cell divisions, or TPSPH_SEARCH_CELLS");
    }
    if (h->search == TPSPH_SEARCH_LISTS) {
        // capacities: 1.5 x the expected count in the list ball (particle volume m / rho0)
        // plus 16; walls fill at most 7/8 (3D) or 3/4 (2D) of the ball around a corner
        auto ball = [&](double r) { return nd == 2 ? M_PI * r * r : 4.0 / 3.0 * M_PI * r * r * r; };
        auto cap = [&](double expected) {
            const double c = std::ceil(1.5 * expected) + 16.0;
            return (int)std::min(4096.0, std::ceil(c / 8.0) * 8.0);
        };
        const double rlf = std::sqrt(P.rl2_fluid), rlw = std::sqrt(P.rl2_wall);
        h->cap_f = cap(mf > 0.0 ? ball(rlf) / (mf / P.rho0) : 0.0);
        h->cap_w = h->nw > 0 ? cap(mw > 0.0 ? (nd == 2 ? 0.75 : 0.875) * ball(rlw) / (mw / P.rho0) : 0.0) : 0;
        h->ls = (h->nf + 63) / 64 * 64;
        // a wall particle of a flat wall sees fluid in at most half its ball
        h->cap_a = h->nw > 0 ? cap(mf > 0.0 ? 0.6 * ball(rlw) / (mf / P.rho0) : 0.0) : 0;
        h->lw = (h->nw + 63) / 64 * 64;
    }
    auto cleanup_fail = [&](int rc) {
        std::string m = h->last_error;
        tpsph_destroy(h);
        return fail(nullptr, rc, m);
    };
    int rc;
#define CTRY(expr) \
    if ((rc = (expr)) != TPSPH_OK) return cleanup_fail(rc)
    const int nf = h->nf, nw = h->nw;
    h->mixed = params->precision == TPSPH_PRECISION_MIXED;
    if (h->mixed && !(h->search == TPSPH_SEARCH_LISTS && brick_rows_ok(P) &&
                      params->use_density_diffusion != TPSPH_DIFFUSION_ANTUONO)) {
        delete h;
        return fail(nullptr, TPSPH_ERR_ARGUMENT,
                    "precision TPSPH_PRECISION_MIXED runs on the brick kernel: it needs the "
                    "Verlet lists (skin > 0), the default brick sizes and no "
                    "DensityDiffusionAntuono");
    }
    CTRY(dalloc(h, &h->flag, 1));
    CTRY(dalloc(h, &h->nrebuild, 1));
    if (hipMemset(h->nrebuild, 0, sizeof(int)) != hipSuccess) {
        h->last_error = "clearing the rebuild count failed";
        return cleanup_fail(TPSPH_ERR_HIP);
    }
    if (params->wall_viscosity && nw > 0) CTRY(dalloc(h, &h->wvel, 3 * (size_t)nw));
    if (params->use_density_diffusion == TPSPH_DIFFUSION_ANTUONO && !P.summation && nf > 0) {
        CTRY(dalloc(h, &h->ddgrad, (size_t)nd * nf));
        P.ddgrad = h->ddgrad;
    }
    if (P.summation) CTRY(dalloc(h, &h->sum_rho, (size_t)std::max(nf, 1)));
    if (params->adaptive_sound_speed) {
        CTRY(dalloc(h, &h->dyn, 4));
        CTRY(dalloc(h, &h->vmax_part, kGateBlocks));
        // until the first kick: the constants of params.sound_speed
        const double init[4] = {P.c, P.B, P.av_c, P.dd2};
        if (hipMemcpy(h->dyn, init, sizeof(init), hipMemcpyHostToDevice) != hipSuccess) {
            h->last_error = "copy of the sound speed failed";
            return cleanup_fail(TPSPH_ERR_HIP);
        }
        P.dyn = h->dyn;
    }
    CTRY(dalloc(h, &h->scan_state, (size_t)scan_words((int)ncells + 1)));
    if (h->search == TPSPH_SEARCH_LISTS && nf <= kSortMax && ncells <= kSortMaxCells)
        CTRY(dalloc(h, &h->sort_ctl, kSortCtl));
    CTRY(dalloc(h, &h->f_cell, nf));
    CTRY(dalloc(h, &h->f_rank, nf));
    CTRY(dalloc(h, &h->f_perm, nf));
    CTRY(dalloc(h, &h->f_head, (size_t)ncells));
    CTRY(dalloc(h, &h->f_count, (size_t)ncells + 1));
    CTRY(dalloc(h, &h->f_start, (size_t)ncells + 1));
    CTRY(dalloc(h, &h->f_mass, nf));
    CTRY(dalloc(h, &h->xs, (size_t)nf + kPad));
    CTRY(dalloc(h, &h->ys, (size_t)nf + kPad));
    CTRY(dalloc(h, &h->zs, (size_t)nf + kPad));
    if (h->search == TPSPH_SEARCH_LISTS) CTRY(dalloc(h, &h->xf, (size_t)nf + kPad));
    if (h->search == TPSPH_SEARCH_LISTS && nw > 0) CTRY(dalloc(h, &h->wxf, (size_t)nw + kPad));
    CTRY(dalloc(h, &h->snap, (size_t)nd * nf));
    CTRY(dalloc(h, &h->iperm, nf));
    CTRY(dalloc(h, &h->rec, 2 * (size_t)nf));
    CTRY(dalloc(h, &h->vol, nf));
    CTRY(dalloc(h, &h->w_start, (size_t)ncells + 1));
    CTRY(dalloc(h, &h->w_perm, nw));
    CTRY(dalloc(h, &h->wx, (size_t)nw + kPad));
    CTRY(dalloc(h, &h->wy, (size_t)nw + kPad));
    CTRY(dalloc(h, &h->wz, (size_t)nw + kPad));
    CTRY(dalloc(h, &h->wall_near, (size_t)ncells));
    if (h->search == TPSPH_SEARCH_LISTS) {
        CTRY(dalloc(h, &h->nbr, (size_t)h->cap_f * h->ls));
        CTRY(dalloc(h, &h->cnt, nf));
        CTRY(dalloc(h, &h->ord, nf));
        CTRY(dalloc(h, &h->counters, kCounters));
        // the brick kernel (with DensityDiffusionAntuono its records also carry the density
        // gradients) whenever every brick's union rows fit one scan block
        h->bricks = brick_rows_ok(P);
        if (h->bricks) {
            // a cell lies in the unions of at most `times` bricks along an axis
            int64_t times = 1;
            for (int d = 0; d < nd; d++) {
                const int beyond = (int)std::floor((std::sqrt(P.rl_union2) + 4.0 * P.hs_union) / P.cs[d]) + 1;
                times *= (2 * beyond + P.bc[d] - 1) / P.bc[d] + 1;
            }
            h->uidx_cap = std::min<int64_t>(std::max<int64_t>(times * nf, 1), INT_MAX);
            CTRY(dalloc(h, &h->uidx, (size_t)h->uidx_cap));
            // [0] the brick kernels' work counter, [1] the bricks the mixed-precision pass
            // leaves to the FP64 pass (listed in bfall), [2] the work counter of the brick
            // gradient pass (DensityDiffusionAntuono); all cleared by the kick's gather or
            // the stage kernel
            CTRY(dalloc(h, &h->bwork, 3));
            if (h->mixed) CTRY(dalloc(h, &h->bfall, (size_t)h->nbricks));
            CTRY(dalloc(h, &h->nbr16, (size_t)((h->cap_f + 15) / 16 * 16) * h->ls));
            CTRY(dalloc(h, &h->thead, (size_t)h->ls));
        }
        CTRY(dalloc(h, &h->bcount, (size_t)h->nbricks));
        CTRY(dalloc(h, &h->nel, (size_t)std::min<int64_t>(h->nbricks, nf)));
        CTRY(dalloc(h, &h->bhead, (size_t)std::min<int64_t>(h->nbricks, nf)));
        CTRY(dalloc(h, &h->tbase, nf));
        if (hipMemset(h->bcount, 0, (size_t)h->nbricks * sizeof(int)) != hipSuccess) {
            h->last_error = "clearing the brick counts failed";
            return cleanup_fail(TPSPH_ERR_HIP);
        }
        if (nw > 0) {
            CTRY(dalloc(h, &h->wnbr, (size_t)h->cap_w * h->ls));
            CTRY(dalloc(h, &h->wcnt, nf));
            CTRY(dalloc(h, &h->anbr, (size_t)h->cap_a * h->lw));
            CTRY(dalloc(h, &h->acnt, nw));
            CTRY(dalloc(h, &h->wactive, nw));
            if (h->bricks) CTRY(dalloc(h, &h->wtargets, nf));
        }
    }
    // NaN (all bits set) in the coordinate arrays, including their padding; never zero so a
    // padded entry can not pass the radius test
    for (double *a : {h->xs, h->ys, h->zs})
        CTRY(hip_fill(h, a, (size_t)nf + kPad));
    if ((h->xf && hipMemset(h->xf, 0xff, ((size_t)nf + kPad) * sizeof(float4)) != hipSuccess) ||
        (h->wxf && hipMemset(h->wxf, 0xff, ((size_t)nw + kPad) * sizeof(float4)) != hipSuccess)) {
        h->last_error = "clearing the FP32 positions failed";
        return cleanup_fail(TPSPH_ERR_HIP);
    }
    for (double *a : {h->wx, h->wy, h->wz})
        CTRY(hip_fill(h, a, (size_t)nw + kPad));
    if (hipMemset(h->f_count, 0, ((size_t)ncells + 1) * sizeof(int)) != hipSuccess) {
        h->last_error = "clearing the cell counts failed";
        return cleanup_fail(TPSPH_ERR_HIP);
    }
    if (nf == 0 && hipMemset(h->f_start, 0, ((size_t)ncells + 1) * sizeof(int)) != hipSuccess) {
        h->last_error = "clearing the cell offsets failed";
        return cleanup_fail(TPSPH_ERR_HIP);
    }
    if (hipMemset(h->wall_near, 0, (size_t)ncells) != hipSuccess) {
        h->last_error = "clearing wall_near failed";
        return cleanup_fail(TPSPH_ERR_HIP);
    }
    CTRY(dalloc(h, &h->wpos, nw));
    CTRY(dalloc(h, &h->wpv, nw));
    CTRY(dalloc(h, &h->pw, nw));
    CTRY(dalloc(h, &h->rhow, nw));
    hipLaunchKernelGGL((k_set_i32), dim3(1), dim3(1), 0, h->stream, h->flag, 1);  // the first kick builds the fluid cells
    CTRY(launch_check(h, "k_set_i32"));
    if (nf > 0) {
        hipError_t e = hipMemcpy(h->f_mass, fluid_mass, (size_t)nf * sizeof(double), in_kind);
        if (e != hipSuccess) {
            h->last_error = std::string("copy of fluid_mass: ") + hipGetErrorString(e);
            return cleanup_fail(TPSPH_ERR_HIP);
        }
    }
    CTRY(dalloc(h, &h->dev, 1));
    CTRY(put_handle(h));
    // static wall cell list
    if (nw > 0) {
        double *wx_d = nullptr, *wm_d = nullptr;
        int *wcell = nullptr, *wrank = nullptr, *wcount = nullptr;
        rc = dalloc(h, &wx_d, (size_t)nd * nw);
        if (rc == TPSPH_OK) rc = dalloc(h, &wm_d, nw);
        if (rc == TPSPH_OK) rc = dalloc(h, &wcell, nw);
        if (rc == TPSPH_OK) rc = dalloc(h, &wrank, nw);
        if (rc == TPSPH_OK) rc = dalloc(h, &wcount, (size_t)ncells + 1);
        if (rc == TPSPH_OK && hipMemset(wcount, 0, ((size_t)ncells + 1) * sizeof(int)) != hipSuccess)
            rc = fail(h, TPSPH_ERR_HIP, "clearing the wall cell counts failed");
        if (rc == TPSPH_OK) {
            hipError_t e1 = hipMemcpy(wx_d, wxh.data(), wxh.size() * sizeof(double), hipMemcpyHostToDevice);
            hipError_t e2 = hipMemcpy(wm_d, wall_mass, (size_t)nw * sizeof(double), in_kind);
            if (e1 != hipSuccess || e2 != hipSuccess) rc = fail(h, TPSPH_ERR_HIP, "copy of wall data failed");
        }
        if (rc == TPSPH_OK)
            rc = nd == 2 ? build_cells<2>(h, nullptr, nw, wx_d, wcell, wrank, wcount, h->w_start, h->w_perm)
                         : build_cells<3>(h, nullptr, nw, wx_d, wcell, wrank, wcount, h->w_start, h->w_perm);
        if (rc == TPSPH_OK) {
            if (nd == 2)
                hipLaunchKernelGGL((k_positions<2>), dim3(nblocks(nw)), dim3(kBlock), 0, h->stream, nw, wx_d, h->w_perm, h->wx, h->wy, nullptr, h->wpos, wm_d);
            else
                hipLaunchKernelGGL((k_positions<3>), dim3(nblocks(nw)), dim3(kBlock), 0, h->stream, nw, wx_d, h->w_perm, h->wx, h->wy, h->wz, h->wpos, wm_d);
            if (nd == 2)
                hipLaunchKernelGGL((k_wall_near<2>), dim3(nblocks(nw)), dim3(kBlock), 0, h->stream, h->P, nw, h->wpos, h->wall_near);
            else
                hipLaunchKernelGGL((k_wall_near<3>), dim3(nblocks(nw)), dim3(kBlock), 0, h->stream, h->P, nw, h->wpos, h->wall_near);
            if (h->wxf && nd == 2)
                hipLaunchKernelGGL((k_wall_f32<2>), dim3(nblocks(nw)), dim3(kBlock), 0, h->stream, h->P, nw, h->wpos, h->wxf);
            else if (h->wxf)
                hipLaunchKernelGGL((k_wall_f32<3>), dim3(nblocks(nw)), dim3(kBlock), 0, h->stream, h->P, nw, h->wpos, h->wxf);
            rc = launch_check(h, "wall setup");
        }
        hipError_t es = hipStreamSynchronize(h->stream);
        (void)hipFree(wx_d);
        (void)hipFree(wm_d);
        (void)hipFree(wcell);
        (void)hipFree(wrank);
        (void)hipFree(wcount);
        if (rc == TPSPH_OK && es != hipSuccess)
            rc = fail(h, TPSPH_ERR_HIP, std::string("wall setup: ") + hipGetErrorString(es));
        if (rc != TPSPH_OK) return cleanup_fail(rc);
    }
#undef CTRY
    *out = h;
    return TPSPH_OK;
}

int tpsph_kick(tpsph_handle *h, double *dv_ode, const double *v_ode, const double *u_ode,
               double t)
{
    (void)t;
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    if (h->nf > 0 && (!dv_ode || !v_ode || !u_ode))
        return fail(h, TPSPH_ERR_ARGUMENT, "dv_ode, v_ode and u_ode must not be NULL");
    if (!is_host(h)) return kick_dispatch(h, dv_ode, v_ode, u_ode);
    TRY(ensure_staging(h));
    HIP_TRY(h, hipMemcpyAsync(h->st_v, v_ode, v_len(h) * sizeof(double), hipMemcpyHostToDevice, h->stream));
    HIP_TRY(h, hipMemcpyAsync(h->st_u, u_ode, u_len(h) * sizeof(double), hipMemcpyHostToDevice, h->stream));
    TRY(kick_dispatch(h, h->st_dv, h->st_v, h->st_u));
    HIP_TRY(h, hipMemcpyAsync(dv_ode, h->st_dv, v_len(h) * sizeof(double), hipMemcpyDeviceToHost, h->stream));
    HIP_TRY(h, hipStreamSynchronize(h->stream));
    return TPSPH_OK;
}

int tpsph_drift(tpsph_handle *h, double *du_ode, const double *v_ode, const double *u_ode,
                double t)
{
    (void)t;
    (void)u_ode;
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    if (h->nf == 0) return TPSPH_OK;
    if (!du_ode || !v_ode) return fail(h, TPSPH_ERR_ARGUMENT, "du_ode and v_ode must not be NULL");
    if (!is_host(h)) {
        if (h->nd == 2)
            hipLaunchKernelGGL((k_drift<2>), dim3(nblocks(h->nf)), dim3(kBlock), 0, h->stream, h->nf, h->P.vrows, v_ode, du_ode);
        else
            hipLaunchKernelGGL((k_drift<3>), dim3(nblocks(h->nf)), dim3(kBlock), 0, h->stream, h->nf, h->P.vrows, v_ode, du_ode);
        return launch_check(h, "k_drift");
    }
    for (int i = 0; i < h->nf; i++)
        for (int d = 0; d < h->nd; d++)
            du_ode[(size_t)i * h->nd + d] = v_ode[(size_t)i * h->P.vrows + d];
    return TPSPH_OK;
}

int tpsph_get_pressures(tpsph_handle *h, double *fluid_pressure, double *wall_pressure,
                        double *wall_density)
{
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    if (!h->have_kick) return fail(h, TPSPH_ERR_STATE, "no kick has been evaluated yet");
    const size_t n = (size_t)std::max(h->nf, h->nw);
    double *tmp = nullptr, *pf_sorted = nullptr;
    TRY(dalloc(h, &tmp, n));
    int rc = dalloc(h, &pf_sorted, (size_t)h->nf);
    auto emit = [&](double *dst, const double *sorted, const int *perm, int cnt) -> int {
        if (!dst || cnt == 0) return TPSPH_OK;
        hipLaunchKernelGGL((k_unpermute<double>), dim3(nblocks(cnt)), dim3(kBlock), 0, h->stream, cnt, perm, sorted, tmp);
        TRY(launch_check(h, "k_unpermute"));
        HIP_TRY(h, hipMemcpyAsync(dst, tmp, (size_t)cnt * sizeof(double), hipMemcpyDefault, h->stream));
        HIP_TRY(h, hipStreamSynchronize(h->stream));
        return TPSPH_OK;
    };
    if (rc == TPSPH_OK && fluid_pressure && h->nf > 0) {
        hipLaunchKernelGGL((k_record_pressure), dim3(nblocks(h->nf)), dim3(kBlock), 0, h->stream, h->nf, h->rec, pf_sorted);
        rc = launch_check(h, "k_record_pressure");
        if (rc == TPSPH_OK) rc = emit(fluid_pressure, pf_sorted, h->f_perm, h->nf);
    }
    if (rc == TPSPH_OK) rc = emit(wall_pressure, h->pw, h->w_perm, h->nw);
    if (rc == TPSPH_OK) rc = emit(wall_density, h->rhow, h->w_perm, h->nw);
    (void)hipFree(tmp);
    (void)hipFree(pf_sorted);
    return rc;
}

int tpsph_get_density(tpsph_handle *h, double *fluid_density)
{
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    if (!fluid_density) return fail(h, TPSPH_ERR_ARGUMENT, "fluid_density is NULL");
    if (!h->have_kick) return fail(h, TPSPH_ERR_STATE, "no kick has been evaluated yet");
    if (h->nf == 0) return TPSPH_OK;
    double *sorted = nullptr, *tmp = nullptr;
    TRY(dalloc(h, &sorted, (size_t)h->nf));
    int rc = dalloc(h, &tmp, (size_t)h->nf);
    if (rc == TPSPH_OK) {
        hipLaunchKernelGGL((k_record_pressure), dim3(nblocks(h->nf)), dim3(kBlock), 0, h->stream,
                           h->nf, h->rec, sorted, 0);
        hipLaunchKernelGGL((k_unpermute<double>), dim3(nblocks(h->nf)), dim3(kBlock), 0, h->stream,
                           h->nf, h->f_perm, sorted, tmp);
        rc = launch_check(h, "k_record_pressure/k_unpermute");
    }
    if (rc == TPSPH_OK &&
        (hipMemcpyAsync(fluid_density, tmp, (size_t)h->nf * sizeof(double), hipMemcpyDefault,
                        h->stream) != hipSuccess ||
         hipStreamSynchronize(h->stream) != hipSuccess))
        rc = fail(h, TPSPH_ERR_HIP, "reading the densities failed");
    (void)hipFree(sorted);
    (void)hipFree(tmp);
    return rc;
}

int tpsph_get_sound_speed(tpsph_handle *h, double *sound_speed)
{
    if (!h || !sound_speed) return fail(h, TPSPH_ERR_ARGUMENT, "handle or sound_speed is NULL");
    if (!h->dyn) {
        *sound_speed = h->P.c;
        return TPSPH_OK;
    }
    if (hipMemcpyAsync(sound_speed, h->dyn, sizeof(double), hipMemcpyDeviceToHost, h->stream) !=
            hipSuccess ||
        hipStreamSynchronize(h->stream) != hipSuccess)
        return fail(h, TPSPH_ERR_HIP, "reading the sound speed failed");
    return TPSPH_OK;
}

int tpsph_neighbors_csr(tpsph_handle *h, const double *u_ode, int32_t pair, int64_t *offsets,
                        int32_t *idx, int64_t capacity)
{
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    if (pair < 0 || pair > 2) return fail(h, TPSPH_ERR_ARGUMENT, "unknown pair kind");
    if (!offsets) return fail(h, TPSPH_ERR_ARGUMENT, "offsets must not be NULL");
    if (h->nf > 0 && !u_ode) return fail(h, TPSPH_ERR_ARGUMENT, "u_ode must not be NULL");
    const int nd = h->nd, nf = h->nf, nw = h->nw;
    const double *u = u_ode;
    if (is_host(h)) {
        TRY(ensure_staging(h));
        HIP_TRY(h, hipMemcpyAsync(h->st_u, u_ode, u_len(h) * sizeof(double), hipMemcpyHostToDevice, h->stream));
        u = h->st_u;
    }
    // fluid cell list of the current positions; the flag stays raised, so the next kick
    // rebuilds and gathers its own state again
    hipLaunchKernelGGL((k_set_i32), dim3(1), dim3(1), 0, h->stream, h->flag, 1);
    TRY(nd == 2 ? build_cells<2>(h, h->flag, nf, u, h->f_cell, h->f_rank, h->f_count, h->f_start, h->f_perm)
                : build_cells<3>(h, h->flag, nf, u, h->f_cell, h->f_rank, h->f_count, h->f_start, h->f_perm));
    if (nf > 0) {
        if (nd == 2)
            hipLaunchKernelGGL((k_positions<2>), dim3(nblocks(nf)), dim3(kBlock), 0, h->stream, nf, u, h->f_perm, h->xs, h->ys, nullptr, nullptr, nullptr);
        else
            hipLaunchKernelGGL((k_positions<3>), dim3(nblocks(nf)), dim3(kBlock), 0, h->stream, nf, u, h->f_perm, h->xs, h->ys, h->zs, nullptr, nullptr);
        TRY(launch_check(h, "k_positions"));
    }
    h->have_kick = false;
    int nrows;
    const double *rx, *ry, *rz, *cx, *cy, *cz;
    const int *row_perm, *col_start, *col_perm;
    double hs;
    if (pair == TPSPH_PAIR_FLUID_FLUID) {
        nrows = nf; rx = h->xs; ry = h->ys; rz = h->zs; row_perm = h->f_perm;
        col_start = h->f_start; cx = h->xs; cy = h->ys; cz = h->zs; col_perm = h->f_perm;
        hs = h->P.hs_fluid;
    } else if (pair == TPSPH_PAIR_FLUID_WALL) {
        nrows = nf; rx = h->xs; ry = h->ys; rz = h->zs; row_perm = h->f_perm;
        col_start = h->w_start; cx = h->wx; cy = h->wy; cz = h->wz; col_perm = h->w_perm;
        hs = h->P.hs_wall;
    } else {
        nrows = nw; rx = h->wx; ry = h->wy; rz = h->wz; row_perm = h->w_perm;
        col_start = h->f_start; cx = h->xs; cy = h->ys; cz = h->zs; col_perm = h->f_perm;
        hs = h->P.hs_fluid;
    }
    auto launch = [&](bool fill, int *counts, const int64_t *doff, int *didx) {
        const dim3 g(nblocks(nrows)), b(kBlock);
        if (nd == 2 && !fill)
            hipLaunchKernelGGL((k_nbr<2, false>), g, b, 0, h->stream, h->P, nrows, rx, ry, rz, row_perm, col_start, cx, cy, cz, col_perm, hs, counts, nullptr, nullptr);
        else if (nd == 2)
            hipLaunchKernelGGL((k_nbr<2, true>), g, b, 0, h->stream, h->P, nrows, rx, ry, rz, row_perm, col_start, cx, cy, cz, col_perm, hs, nullptr, doff, didx);
        else if (!fill)
            hipLaunchKernelGGL((k_nbr<3, false>), g, b, 0, h->stream, h->P, nrows, rx, ry, rz, row_perm, col_start, cx, cy, cz, col_perm, hs, counts, nullptr, nullptr);
        else
            hipLaunchKernelGGL((k_nbr<3, true>), g, b, 0, h->stream, h->P, nrows, rx, ry, rz, row_perm, col_start, cx, cy, cz, col_perm, hs, nullptr, doff, didx);
    };
    return emit_csr(h, nrows, launch, offsets, idx, capacity);
}

int tpsph_kick_pairs_csr(tpsph_handle *h, int32_t pair, int64_t *offsets, int32_t *idx,
                         int64_t capacity)
{
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    if (pair < 0 || pair > 2) return fail(h, TPSPH_ERR_ARGUMENT, "unknown pair kind");
    if (!offsets) return fail(h, TPSPH_ERR_ARGUMENT, "offsets must not be NULL");
    if (!h->have_kick) return fail(h, TPSPH_ERR_STATE, "no kick has been evaluated yet");
    const bool lists = h->search == TPSPH_SEARCH_LISTS;
    const EvalPairsArgs a{pair, lists ? 1 : 0, h->bricks ? 1 : 0, h->ord, h->tbase, h->uidx, h->nbr16, h->nbr, h->cnt,
                          h->wnbr, h->wcnt, h->ls, h->anbr, h->acnt, h->lw, h->w_perm};
    const int nrows = pair == TPSPH_PAIR_WALL_FLUID ? h->nw : h->nf;
    if ((pair != TPSPH_PAIR_FLUID_FLUID && h->nw == 0) || h->nf == 0) {
        // no pairs: all offsets zero
        std::vector<int64_t> zero((size_t)nrows + 1, 0);
        HIP_TRY(h, hipMemcpy(offsets, zero.data(), zero.size() * sizeof(int64_t), hipMemcpyDefault));
        return TPSPH_OK;
    }
    auto launch = [&](bool fill, int *counts, const int64_t *doff, int *didx) {
        const dim3 g(nblocks(nrows)), b(kBlock);
        const FluidView F = h->fluid_view();
        const WallView W = h->wall_view();
        if (h->nd == 2 && !fill)
            hipLaunchKernelGGL((k_eval_pairs<2, false>), g, b, 0, h->stream, h->P, F, W, a, counts, nullptr, nullptr);
        else if (h->nd == 2)
            hipLaunchKernelGGL((k_eval_pairs<2, true>), g, b, 0, h->stream, h->P, F, W, a, nullptr, doff, didx);
        else if (!fill)
            hipLaunchKernelGGL((k_eval_pairs<3, false>), g, b, 0, h->stream, h->P, F, W, a, counts, nullptr, nullptr);
        else
            hipLaunchKernelGGL((k_eval_pairs<3, true>), g, b, 0, h->stream, h->P, F, W, a, nullptr, doff, didx);
    };
    return emit_csr(h, nrows, launch, offsets, idx, capacity);
}

int tpsph_axpby(tpsph_handle *h, int64_t n, double *y, double a, const double *x, double b)
{
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    if (n < 0) return fail(h, TPSPH_ERR_ARGUMENT, "n must be non-negative");
    if (n == 0) return TPSPH_OK;
    if (!y || (b != 0.0 && !x)) return fail(h, TPSPH_ERR_ARGUMENT, "y (and x when b != 0) must not be NULL");
    if (is_host(h)) {
        for (int64_t i = 0; i < n; i++) {
            if (b == 0.0)
                y[i] = a == 0.0 ? 0.0 : a * y[i];
            else if (a == 0.0)
                y[i] = b * x[i];
            else
                y[i] = std::fma(b, x[i], a * y[i]);
        }
        return TPSPH_OK;
    }
    TimedScope ts(h, TPSPH_TIME_STAGE);
    hipLaunchKernelGGL((k_axpby), dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, h->stream, n, y, a, x, b);
    return launch_check(h, "k_axpby");
}

int tpsph_rk_stage(tpsph_handle *h, double *y, double *tmp, const double *k, double a,
                   double b, double dt, int64_t n, int32_t first_stage)
{
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    if (n < 0) return fail(h, TPSPH_ERR_ARGUMENT, "n must be non-negative");
    if (n == 0) return TPSPH_OK;
    if (!y || !tmp || !k) return fail(h, TPSPH_ERR_ARGUMENT, "y, tmp and k must not be NULL");
    if (is_host(h)) {
        for (int64_t i = 0; i < n; i++) {
            double t = first_stage ? dt * k[i] : std::fma(dt, k[i], a * tmp[i]);
            tmp[i] = t;
            y[i] = std::fma(b, t, y[i]);
        }
        return TPSPH_OK;
    }
    TimedScope ts(h, TPSPH_TIME_STAGE);
    hipLaunchKernelGGL((k_rk_stage), dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, h->stream, n, y, tmp, k, a, b, dt, first_stage);
    return launch_check(h, "k_rk_stage");
}

int tpsph_solve_ck2n54(tpsph_handle *h, double *v_ode, double *u_ode, double t0, double dt,
                       int64_t nsteps)
{
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    if (nsteps < 0) return fail(h, TPSPH_ERR_ARGUMENT, "nsteps must be non-negative");
    if (h->nf == 0 || nsteps == 0) return TPSPH_OK;
    if (!v_ode || !u_ode) return fail(h, TPSPH_ERR_ARGUMENT, "v_ode and u_ode must not be NULL");
    (void)t0;
    double *v = v_ode, *u = u_ode;
    if (is_host(h)) {
        TRY(ensure_staging(h));
        HIP_TRY(h, hipMemcpyAsync(h->st_v, v_ode, v_len(h) * sizeof(double), hipMemcpyHostToDevice, h->stream));
        HIP_TRY(h, hipMemcpyAsync(h->st_u, u_ode, u_len(h) * sizeof(double), hipMemcpyHostToDevice, h->stream));
        v = h->st_v;
        u = h->st_u;
    }
    TRY(run_ck2n54(h, v, u, dt, nsteps, nullptr, nullptr));
    if (is_host(h)) {
        HIP_TRY(h, hipMemcpyAsync(v_ode, v, v_len(h) * sizeof(double), hipMemcpyDeviceToHost, h->stream));
        HIP_TRY(h, hipMemcpyAsync(u_ode, u, u_len(h) * sizeof(double), hipMemcpyDeviceToHost, h->stream));
        HIP_TRY(h, hipStreamSynchronize(h->stream));
    }
    return TPSPH_OK;
}

int tpsph_kick_noalloc(const tpsph_params *params, int64_t n_fluid, int64_t n_wall,
                       const double *fluid_mass, const double *wall_coordinates,
                       const double *wall_mass, double *dv_ode, const double *v_ode,
                       const double *u_ode, double t, void *stream)
{
    (void)t;
    TRY(validate(params, n_fluid, n_wall, fluid_mass, wall_coordinates, wall_mass));
    auto bad = [](const std::string &m) { return fail(nullptr, TPSPH_ERR_ARGUMENT, "tpsph_kick_noalloc: " + m); };
    if (params->memory != TPSPH_MEM_DEVICE) return bad("needs device pointers (TPSPH_MEM_DEVICE)");
    if (params->adaptive_sound_speed || params->use_density_diffusion == TPSPH_DIFFUSION_ANTUONO ||
        params->wall_viscosity || params->precision != TPSPH_PRECISION_FP64 ||
        params->density_calculator != TPSPH_DENSITY_CONTINUITY)
        return bad("supports ContinuityDensity, StateEquationCole, Molteni-Colagrossi diffusion, "
                   "walls without viscosity and FP64");
    if (n_fluid > 0 && (!dv_ode || !v_ode || !u_ode))
        return bad("dv_ode, v_ode and u_ode must not be NULL");
    double lo[3] = {0.0, 0.0, 0.0}, hi[3] = {0.0, 0.0, 0.0};
    for (int d = 0; d < params->ndims; d++) {
        if (!(params->domain_min[d] < params->domain_max[d]))
            return bad("needs the grid box (domain_min < domain_max on every axis)");
        lo[d] = params->domain_min[d];
        hi[d] = params->domain_max[d];
    }
    // a handle on the stack whose arrays point into the scratch array; it owns nothing
    tpsph_handle h;
    h.params = *params;
    h.nd = params->ndims;
    h.nf = (int)n_fluid;
    h.nw = (int)n_wall;
    h.stream = (hipStream_t)stream;
    h.search = TPSPH_SEARCH_CELLS;
    TRY(derive_params(params, h.nf, h.nw, lo, hi, h.P, h.nbricks));
    size_t bytes = 0;
    TRY(h.nd == 2 ? noalloc_kick<2>(&h, nullptr, &bytes, fluid_mass, wall_coordinates, wall_mass, dv_ode, v_ode, u_ode)
                  : noalloc_kick<3>(&h, nullptr, &bytes, fluid_mass, wall_coordinates, wall_mass, dv_ode, v_ode, u_ode));
    if (bytes > kScratchBytes)
        return bad("needs " + std::to_string(bytes) + " bytes of scratch for " +
                   std::to_string(n_fluid) + " fluid, " + std::to_string(n_wall) +
                   " wall particles and " + std::to_string(h.P.ncells) +
                   " cells; the limit is " + std::to_string(kScratchBytes) + " bytes");
    unsigned char *base = nullptr;
    TRY(scratch_base(&base));
    const int rc = h.nd == 2 ? noalloc_kick<2>(&h, base, &bytes, fluid_mass, wall_coordinates, wall_mass, dv_ode, v_ode, u_ode)
                             : noalloc_kick<3>(&h, base, &bytes, fluid_mass, wall_coordinates, wall_mass, dv_ode, v_ode, u_ode);
    if (rc != TPSPH_OK) return fail(nullptr, rc, h.last_error);
    return TPSPH_OK;
}

int tpsph_integrals(tpsph_handle *h, const double *v_ode, const double *u_ode, double *out)
{
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    if (!out) return fail(h, TPSPH_ERR_ARGUMENT, "out must not be NULL");
    if (h->nf > 0 && (!v_ode || !u_ode)) return fail(h, TPSPH_ERR_ARGUMENT, "v_ode and u_ode must not be NULL");
    if (h->P.summation)
        return fail(h, TPSPH_ERR_ARGUMENT, "tpsph_integrals reads the density rows of v_ode "
                                           "(ContinuityDensity)");
    const double *v = v_ode, *u = u_ode;
    if (is_host(h) && h->nf > 0) {
        TRY(ensure_staging(h));
        HIP_TRY(h, hipMemcpyAsync(h->st_v, v_ode, v_len(h) * sizeof(double), hipMemcpyHostToDevice, h->stream));
        HIP_TRY(h, hipMemcpyAsync(h->st_u, u_ode, u_len(h) * sizeof(double), hipMemcpyHostToDevice, h->stream));
        v = h->st_v;
        u = h->st_u;
    }
    if (!h->integ) TRY(dalloc(h, &h->integ, (size_t)(kIntegralBlocks + 1) * kIntegrals));
    const int nb = std::max(1, std::min(nblocks(h->nf), kIntegralBlocks));
    if (h->nd == 2)
        hipLaunchKernelGGL((k_integrals<2>), dim3(nb), dim3(kBlock), 0, h->stream, h->nf, v, u, h->f_mass, h->P, h->integ);
    else
        hipLaunchKernelGGL((k_integrals<3>), dim3(nb), dim3(kBlock), 0, h->stream, h->nf, v, u, h->f_mass, h->P, h->integ);
    double *res = h->integ + (size_t)kIntegralBlocks * kIntegrals;
    hipLaunchKernelGGL((k_integrals_final), dim3(1), dim3(kBlock), 0, h->stream, nb, h->integ, res);
    TRY(launch_check(h, "k_integrals"));
    HIP_TRY(h, hipMemcpyAsync(out, res, kIntegrals * sizeof(double), hipMemcpyDefault, h->stream));
    HIP_TRY(h, hipStreamSynchronize(h->stream));
    return TPSPH_OK;
}

int tpsph_rebuild_count(tpsph_handle *h, int64_t *count)
{
    if (!h || !count) return fail(h, TPSPH_ERR_ARGUMENT, "handle or count is NULL");
    int n = 0;
    if (h->nrebuild) {
        HIP_TRY(h, hipMemcpyAsync(&n, h->nrebuild, sizeof(int), hipMemcpyDeviceToHost, h->stream));
        HIP_TRY(h, hipStreamSynchronize(h->stream));
    }
    *count = n;
    return TPSPH_OK;
}

int tpsph_sort_particles(tpsph_handle *h, double *v_ode, double *u_ode, int64_t *perm)
{
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    const int nf = h->nf, nd = h->nd;
    if (nf == 0) return TPSPH_OK;
    if (!v_ode || !u_ode) return fail(h, TPSPH_ERR_ARGUMENT, "v_ode and u_ode must not be NULL");
    TRY(ensure_staging(h));
    const size_t vl = v_len(h), ul = u_len(h);
    const bool host = is_host(h);
    // device copies of the state before the sort (st_v, st_u) and of the masses (st_dv);
    // host mode writes the sorted state to temporaries and copies it back
    double *vo = v_ode, *uo = u_ode, *tmp = nullptr;
    int64_t *po = perm;
    const hipMemcpyKind in_kind = host ? hipMemcpyHostToDevice : hipMemcpyDeviceToDevice;
    HIP_TRY(h, hipMemcpyAsync(h->st_v, v_ode, vl * sizeof(double), in_kind, h->stream));
    HIP_TRY(h, hipMemcpyAsync(h->st_u, u_ode, ul * sizeof(double), in_kind, h->stream));
    HIP_TRY(h, hipMemcpyAsync(h->st_dv, h->f_mass, (size_t)nf * sizeof(double),
                              hipMemcpyDeviceToDevice, h->stream));
    if (host) {
        TRY(dalloc(h, &tmp, vl + ul + (size_t)nf));
        vo = tmp;
        uo = tmp + vl;
        po = perm ? reinterpret_cast<int64_t *>(tmp + vl + ul) : nullptr;
    }
    // the cell-sorted order of the current positions (the flag stays raised until the
    // preparation below has rebuilt everything from the sorted state)
    hipLaunchKernelGGL((k_set_i32), dim3(1), dim3(1), 0, h->stream, h->flag, 1);
    int rc = nd == 2 ? build_cells<2>(h, h->flag, nf, h->st_u, h->f_cell, h->f_rank, h->f_count,
                                      h->f_start, h->f_perm)
                     : build_cells<3>(h, h->flag, nf, h->st_u, h->f_cell, h->f_rank, h->f_count,
                                      h->f_start, h->f_perm);
    if (rc == TPSPH_OK) {
        if (nd == 2)
            hipLaunchKernelGGL((k_permute_state<2>), dim3(nblocks(nf)), dim3(kBlock), 0, h->stream, nf,
                               h->P.vrows, h->f_perm, h->st_v, h->st_u, h->st_dv, vo, uo, h->f_mass, po);
        else
            hipLaunchKernelGGL((k_permute_state<3>), dim3(nblocks(nf)), dim3(kBlock), 0, h->stream, nf,
                               h->P.vrows, h->f_perm, h->st_v, h->st_u, h->st_dv, vo, uo, h->f_mass, po);
        rc = launch_check(h, "k_permute_state");
    }
    // rebuild from the sorted state: the cell-sorted order is the one just computed (within
    // a cell the order is by caller index, which now increases along it), so the internal
    // permutation is the identity; pressures and wall values of the sorted state are ready
    // for tpsph_get_pressures, and the next kick need not rebuild
    if (rc == TPSPH_OK) rc = prepare_dispatch(h, vo, uo);
    if (rc == TPSPH_OK) {
        hipLaunchKernelGGL((k_set_i32), dim3(1), dim3(1), 0, h->stream, h->flag, 0);
        rc = launch_check(h, "k_set_i32");
    }
    if (rc == TPSPH_OK && host) {
        if (hipMemcpyAsync(v_ode, vo, vl * sizeof(double), hipMemcpyDeviceToHost, h->stream) != hipSuccess ||
            hipMemcpyAsync(u_ode, uo, ul * sizeof(double), hipMemcpyDeviceToHost, h->stream) != hipSuccess ||
            (perm && hipMemcpyAsync(perm, po, (size_t)nf * sizeof(int64_t), hipMemcpyDeviceToHost,
                                    h->stream) != hipSuccess) ||
            hipStreamSynchronize(h->stream) != hipSuccess)
            rc = fail(h, TPSPH_ERR_HIP, "copy of the sorted state to the host failed");
    }
    if (tmp) (void)hipFree(tmp);
    // a recorded trajectory (reverse mode) belongs to the old order
    h->adj_ready = false;
    h->have_kick = rc == TPSPH_OK;
    return rc;
}

int tpsph_synchronize(tpsph_handle *h)
{
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    HIP_TRY(h, hipStreamSynchronize(h->stream));
    return TPSPH_OK;
}

int tpsph_enable_timing(tpsph_handle *h, int32_t enable)
{
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    HIP_TRY(h, hipStreamSynchronize(h->stream));
    h->timing = enable != 0;
    h->records.clear();
    h->events_used = 0;
    return TPSPH_OK;
}

int tpsph_kernel_time(tpsph_handle *h, int32_t which, int64_t *launches, double *total_ms)
{
    if (!h) return fail(nullptr, TPSPH_ERR_ARGUMENT, "handle is NULL");
    if (which < 0 || which >= TPSPH_TIME_COUNT) return fail(h, TPSPH_ERR_ARGUMENT, "unknown kernel id");
    HIP_TRY(h, hipStreamSynchronize(h->stream));
    int64_t n = 0;
    double sum = 0.0;
    for (const auto &r : h->records) {
        if (r.kind != which) continue;
        float ms = 0.0f;
        HIP_TRY(h, hipEventElapsedTime(&ms, r.a, r.b));
        sum += ms;
        n++;
    }
    if (launches) *launches = n;
    if (total_ms) *total_ms = sum;
    return TPSPH_OK;
}

void tpsph_destroy(tpsph_handle *h)
{
    if (!h) return;
    (void)hipStreamSynchronize(h->stream);
    void *ptrs[] = {h->flag, h->f_cell, h->f_rank, h->f_count, h->f_start, h->f_perm,
                    h->scan_state, h->sort_ctl, h->f_head, h->f_mass, h->xs, h->ys, h->zs, h->xf, h->wxf, h->snap, h->rec, h->vol,
                    h->w_start, h->w_perm, h->wx, h->wy, h->wz, h->wpos, h->wpv, h->wall_near,
                    h->pw, h->nbr, h->cnt, h->wnbr, h->wcnt, h->anbr, h->acnt, h->ord, h->bcount, h->tbase,
                    h->uidx, h->bhead, h->nel, h->counters, h->wactive, h->bwork, h->nbr16,
                    h->wtargets, h->iperm, h->dyn, h->vmax_part, h->wvel, h->ddgrad,
                    h->rhow, h->st_v, h->st_u, h->st_dv, h->st_du, h->sol_dv, h->sol_tv,
                    h->sol_tu, h->integ, h->nrebuild, h->adj_kb, h->adj_coef, h->adj_th,
                    h->adj_gw, h->adj_red, h->adj_vb, h->adj_ub, h->adj_tvb, h->adj_tub,
                    h->adj_ck, h->adj_st, h->sum_rho, h->bfall, h->thead, h->dev};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    for (hipEvent_t e : h->event_pool) (void)hipEventDestroy(e);
    delete h;
}

}  // extern "C"
