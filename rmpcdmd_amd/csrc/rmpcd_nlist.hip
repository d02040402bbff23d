// rmpcd_nlist.hip -- stencil neighbour list of the colloids, colloid-solvent and
// colloid-colloid Lennard-Jones forces and the catalytic helpers of the drivers
// (src/neighbor_list.f90:76-264, programs/single_dimer_pbc.f90:493-565).
//
// update_list keeps the reference's list order (stencil order, then the cell's sorted
// order) with two passes over (point, stencil cell): a count pass, a per-point scan of
// the counts, and a fill pass that writes every accepted particle at its final offset.
#include "rmpcd_internal.hpp"
#include "rmpcd_pairforce.hpp"
#include "rmpcd_steps.hpp"

namespace rmpcd {

constexpr int NL_THREADS = 256;

// cell of a colloid and the Hilbert key of stencil cell j (neighbor_list.f90:111-121)
__device__ inline int stencil_key(const Box &b, const double *x, const int32_t *st, int j)
{
    int p0, p1, p2;
    cell_of<double>(b, x[0], x[1], x[2], p0, p1, p2);
    int a0 = (p0 + st[3 * j]) % b.L[0], a1 = (p1 + st[3 * j + 1]) % b.L[1],
        a2 = (p2 + st[3 * j + 2]) % b.L[2];
    a0 += a0 < 0 ? b.L[0] : 0;
    a1 += a1 < 0 ? b.L[1] : 0;
    a2 += a2 < 0 ? b.L[2] : 0;
    return compact_key(a0, a1, a2, b.M[0], b.M[1], b.M[2]);
}

// pass 1 (fill == 0) counts accepted particles per (point, stencil cell) and marks
// is_md / is_reac; pass 2 (fill == 1) writes them at offset[point*ns + j].  LANES lanes
// take a stencil cell, a particle each (a thread per cell walked its ten particles one
// after the other: 15 us a pass for one point with 1500 stencil cells, FP64), fewer for
// less dense cells (by_density).
template <class F, int LANES>
__global__ void __launch_bounds__(NL_THREADS)
    k_nl_pass(Box b, PView<F64> pts, PView<F> sol, const int32_t *__restrict__ start,
              const int32_t *__restrict__ count, const int32_t *__restrict__ st, int ns,
              double radiussq, double L0, double L1, double L2, int do_lj, LJ lj,
              int32_t *__restrict__ cnt, uint8_t *__restrict__ is_md, uint8_t *__restrict__ is_reac,
              int fill, int32_t nmax, int32_t *__restrict__ list)
{
    const int j = (blockIdx.x * blockDim.x + threadIdx.x) / LANES;
    const int i = blockIdx.y;
    if (j >= ns) return;  // all lanes of a cell alike
    const int lane = threadIdx.x & 63, sub = lane & (LANES - 1), first = lane - sub;
    double x[3] = {pts.pos[i], pts.pos[pts.n + i], pts.pos[2 * pts.n + i]};
    int si = pts.species[i];
    int key = stencil_key(b, x, st, j);
    int s = start[key], n = count[key];
    int64_t slot = (int64_t)i * ns + j;
    int off = fill ? cnt[slot] : 0;
    int k = 0;
    bool noreac = false;
    for (int q0 = s; q0 < s + n; q0 += LANES) {
        const int q = q0 + sub;
        const int sp = q < s + n ? (int)sol.species[q] : 0;
        bool in = false;
        if (sp > 0) {
            double y0 = (double)sol.pos[q], y1 = (double)sol.pos[sol.n + q], y2 = (double)sol.pos[2 * sol.n + q];
            double d0 = min_image(x[0] - y0, L0), d1 = min_image(x[1] - y1, L1), d2 = min_image(x[2] - y2, L2);
            double rsq = (d0 * d0 + d1 * d1) + d2 * d2;
            in = rsq < radiussq;
            if (in && do_lj && rsq <= lj.cut_sq[(sp - 1) + lj.n1 * (si - 1)]) noreac = true;
        }
        // the accepted lanes of this cell, in the cell's order
        const unsigned m = (unsigned)(__ballot(in) >> first) & ((1u << LANES) - 1);
        if (fill && in) {
            const int pos = off + k + __popc(m & ((1u << sub) - 1));
            if (pos < nmax) list[(int64_t)i * nmax + pos] = q;
        }
        k += __popc(m);
    }
    if (!fill) {
        const unsigned nr = (unsigned)(__ballot(noreac) >> first) & ((1u << LANES) - 1);
        if (sub == 0) {
            cnt[slot] = k;
            if (k > 0) {
                is_md[key] = 1;
                if (nr) is_reac[key] = 0;
            }
        }
    }
}

// per point: exclusive scan of the stencil counts in place; n[i] = total; flags overflow
__global__ void __launch_bounds__(1024)
    k_nl_scan(int32_t *cnt, int ns, int32_t nmax, int32_t *__restrict__ nout, int32_t *__restrict__ overflow)
{
    __shared__ int lds[16];
    int i = blockIdx.x;
    int32_t *c = cnt + (int64_t)i * ns;
    int carry = 0;
    for (int base = 0; base < ns; base += blockDim.x) {
        int q = base + threadIdx.x;
        int v = q < ns ? c[q] : 0;
        int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
        int inc = wave_inclusive_scan(v);
        if (lane == 63) lds[wid] = inc;
        __syncthreads();
        int off = 0, tot = 0;
        for (int w = 0; w < nw; ++w) {
            int t = lds[w];
            if (w < wid) off += t;
            tot += t;
        }
        __syncthreads();
        if (q < ns) c[q] = carry + off + inc - v;
        carry += tot;
    }
    if (threadIdx.x == 0) {
        // the reference stops here on overflow (neighbor_list.f90:135-137); the count is
        // clamped so that no consumer reads past the list capacity
        nout[i] = carry > nmax ? nmax : carry;
        if (carry > nmax) *overflow = 1;
    }
}

__global__ void k_init_cells(int ncells, uint8_t *is_md, uint8_t *is_reac)
{
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncells) return;
    is_md[c] = 0;
    is_reac[c] = 1;
}

// compute_force part 1 (neighbor_list.f90:180-188): PAST_MD <- MD, MD cleared
template <class F>
__global__ void k_roll_md(int64_t n, typename F::small *flags)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int f = (int)flags[i];
    f = (f & MD_MASK) ? (f | PAST_MD_MASK) : (f & ~PAST_MD_MASK);
    flags[i] = (typename F::small)(f & ~MD_MASK);
}

// The colloids c0 .. c0 + gridDim.y - 1, one thread per list entry.  The reference adds
// the forces on a solvent particle in colloid order.  One colloid meets a particle once,
// and its thread adds the force at once (next null).  With several, the entries inside the
// cutoff chain up per particle, head[particle] = the last to arrive, next[entry] = the one
// before (entries counted from 1, 0 ends a chain, OUTSIDE marks the entries beyond the
// cutoff), and k_force_nl_apply adds each chain in order.  The colloid force and energy go
// to per-block partials, summed in block order by k_force_nl_sum.  Bound by launches and the
// latency of the entries' reads: a launch per colloid, which kept the order before, took
// 390 us an MD step with 52 colloids (30.0 ms a cycle of 50 steps, 10.8 with the chains).
constexpr uint32_t OUTSIDE = 0xffffffffu;
// List entries of one launch's chains, 4 B each, which the workspace holds until the process
// ends: 64 MiB.  More colloids are taken in several pairs of launches, in their order.
constexpr int32_t CHAIN_ENTRIES = 1 << 24;

template <class F>
__global__ void __launch_bounds__(256)
    k_force_nl(PView<F64> c, PView<F> sol, const int32_t *__restrict__ list,
               const int32_t *__restrict__ nl, int32_t nmax, double L0, double L1, double L2, LJ lj,
               double *__restrict__ part, int c0, uint32_t *__restrict__ head, uint32_t *__restrict__ next)
{
    using R = typename F::real;
    __shared__ double red[16];
    const int i = c0 + (int)blockIdx.y;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int n_i = min(nl[i], nmax);
    double *pp = part + ((int64_t)i * gridDim.x + blockIdx.x) * 4;
    if ((int)(blockIdx.x * blockDim.x) >= n_i) {  // past the list: nothing to add
        if (threadIdx.x < 4) pp[threadIdx.x] = 0;
        return;
    }
    double f[3] = {0, 0, 0}, e = 0;
    if (k < n_i) {
        const int idx = list[(int64_t)i * nmax + k];
        const bool in = pair_force<F>(c, sol, i, idx, L0, L1, L2, lj, f, &e);
        if (next) {
            const uint32_t ent = (uint32_t)blockIdx.y * (uint32_t)nmax + (uint32_t)k + 1;
            next[ent - 1] = in ? atomicExch(&head[idx], ent) : OUTSIDE;
        } else if (in) {
            for (int q = 0; q < 3; ++q) sol.force[q * sol.n + idx] = sol.force[q * sol.n + idx] - (R)f[q];
            sol.flags[idx] = (typename F::small)((int)sol.flags[idx] | MD_MASK |
                                                 (c.species[i] == 1 ? CATALYZED_MASK : 0));
        }
    }
    const double b0 = block_sum(f[0], red), b1 = block_sum(f[1], red), b2 = block_sum(f[2], red),
                 be = block_sum(e, red);
    if (threadIdx.x == 0) {
        pp[0] = b0;
        pp[1] = b1;
        pp[2] = b2;
        pp[3] = be;
    }
}

// the chains of k_force_nl: the thread of a chain's last arrival adds its entries in
// colloid order (the next larger entry each time: two or three colloids meet at most) and
// clears the head.  The other entries of the chain read a head that is not their own before
// as after that.  The first CHAIN_REG entries are read once and kept; a longer chain's rest is
// walked for each addition, and holds no more than the launch's entries, so the walk ends.
// (200 overlapping colloids in an L = 16 box, FP64, a call: 56 us walking the chain for each
// addition, 52.5 like this.)
constexpr int CHAIN_REG = 8;

template <class F>
__global__ void __launch_bounds__(256)
    k_force_nl_apply(PView<F64> c, PView<F> sol, const int32_t *__restrict__ list, const int32_t *__restrict__ nl,
                     int32_t nmax, double L0, double L1, double L2, LJ lj, int c0, uint32_t *__restrict__ head,
                     const uint32_t *__restrict__ next)
{
    using R = typename F::real;
    const int i = c0 + (int)blockIdx.y;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= min(nl[i], nmax)) return;
    const uint32_t ent = (uint32_t)blockIdx.y * (uint32_t)nmax + (uint32_t)k + 1;
    const uint32_t most = gridDim.y * (uint32_t)nmax, before = next[ent - 1];
    if (before == OUTSIDE) return;
    const int idx = list[(int64_t)i * nmax + k];
    if (head[idx] != ent) return;
    R a[3] = {sol.force[idx], sol.force[sol.n + idx], sol.force[2 * sol.n + idx]};
    int fl = (int)sol.flags[idx];
    uint32_t id[CHAIN_REG], rest = before, done = 0;
    id[0] = ent;
#pragma unroll
    for (int j = 1; j < CHAIN_REG; ++j) {
        id[j] = rest ? rest : OUTSIDE;
        if (rest) rest = next[rest - 1];
    }
    for (;;) {
        uint32_t least = OUTSIDE, len = 0;
#pragma unroll
        for (int j = 0; j < CHAIN_REG; ++j)
            if (id[j] > done && id[j] < least) least = id[j];
        for (uint32_t q = rest; q && len < most; q = next[q - 1], ++len)
            if (q > done && q < least) least = q;
        if (least == OUTSIDE) break;
        done = least;
        const int ci = c0 + (int)((least - 1) / (uint32_t)nmax);
        double f[3] = {0, 0, 0}, e;
        pair_force<F>(c, sol, ci, idx, L0, L1, L2, lj, f, &e);
        for (int q = 0; q < 3; ++q) a[q] = a[q] - (R)f[q];
        fl |= MD_MASK | (c.species[ci] == 1 ? CATALYZED_MASK : 0);
    }
    for (int q = 0; q < 3; ++q) sol.force[q * sol.n + idx] = a[q];
    sol.flags[idx] = (typename F::small)fl;
    head[idx] = 0;
}

// the colloid force and energy of compute_force: a colloid's block partials added to the
// force it holds
__global__ void __launch_bounds__(64)
    k_force_nl_sum(PView<F64> c, const double *__restrict__ part, int nb, double *__restrict__ e_out)
{
    const int i = blockIdx.x, q = threadIdx.x;
    const double a = list_force_sum(part, nb, i);
    if (q < 3)
        c.force[q * c.n + i] = c.force[q * c.n + i] + a;
    else if (q == 3)
        e_out[i] = a;
}

// sum of n doubles in index order by one thread (the small colloid count)
__global__ void k_sum_serial(const double *a, int64_t n, double *out)
{
    if (threadIdx.x || blockIdx.x) return;
    double s = 0;
    for (int64_t i = 0; i < n; ++i) s = s + a[i];
    out[0] = s;
}

// ---- driver helpers -------------------------------------------------------------
// flag_particles_nl (single_dimer_pbc.f90:493-509)
template <class F>
__global__ void k_flag_nl(PView<F> sol, PView<F64> c, const int32_t *__restrict__ list,
                          const int32_t *__restrict__ nl, int32_t nmax, double L0, double L1, double L2,
                          double cut_sq_c)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= min(nl[0], nmax)) return;
    int r = list[k];
    if ((int)sol.species[r] != 1) return;
    double d0 = min_image(c.pos[0] - (double)sol.pos[r], L0);
    double d1 = min_image(c.pos[c.n] - (double)sol.pos[sol.n + r], L1);
    double d2 = min_image(c.pos[2 * c.n] - (double)sol.pos[2 * sol.n + r], L2);
    if ((d0 * d0 + d1 * d1) + d2 * d2 < cut_sq_c)
        sol.flags[r] = (typename F::small)((int)sol.flags[r] | REAC_MASK);
}

// change_species (single_dimer_pbc.f90:511-542)
template <class F>
__global__ void k_change_species(PView<F> sol, PView<F64> c, double L0, double L1, double L2,
                                 double cut_sq_c, double cut_sq_n, double prob,
                                 const double *__restrict__ draws, uint64_t seed, uint64_t step)
{
    int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= sol.n) return;
    int f = (int)sol.flags[m];
    if (!(f & REAC_MASK)) return;
    double y0 = (double)sol.pos[m], y1 = (double)sol.pos[sol.n + m], y2 = (double)sol.pos[2 * sol.n + m];
    double a0 = min_image(c.pos[0] - y0, L0), a1 = min_image(c.pos[c.n] - y1, L1),
           a2 = min_image(c.pos[2 * c.n] - y2, L2);
    double dc = (a0 * a0 + a1 * a1) + a2 * a2;
    double b0 = min_image(c.pos[1] - y0, L0), b1 = min_image(c.pos[c.n + 1] - y1, L1),
           b2 = min_image(c.pos[2 * c.n + 1] - y2, L2);
    double dn = (b0 * b0 + b1 * b1) + b2 * b2;
    if (dc > cut_sq_c && dn > cut_sq_n) {
        double u;
        if (draws) {
            u = draws[m];
        } else {
            uint64_t a, b;
            threefry2x64(step, (uint64_t)sol.id[m], seed, STREAM_CHANGE, a, b);
            u = u01(a);
        }
        if (u <= prob) sol.species[m] = (typename F::small)2;
        sol.flags[m] = (typename F::small)(f & ~REAC_MASK);
    }
}

// flag_particles_nl of the fixed-sphere driver
// (setup_single_catalytic_fixed_sphere.f90:311-329): a species-1 list particle inside
// the cutoff draws u (list slot k: draws[k], or threefry((step, id), (seed, CHANGE)))
// and is flagged when u <= prob
template <class F>
__global__ void k_flag_nl_prob(PView<F> sol, PView<F64> c, const int32_t *__restrict__ list,
                               const int32_t *__restrict__ nl, int32_t nmax, double L0, double L1, double L2,
                               double cut_sq_c, double prob, const double *__restrict__ draws, uint64_t seed,
                               uint64_t step)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= min(nl[0], nmax)) return;
    int r = list[k];
    if ((int)sol.species[r] != 1) return;
    double d0 = min_image(c.pos[0] - (double)sol.pos[r], L0);
    double d1 = min_image(c.pos[c.n] - (double)sol.pos[sol.n + r], L1);
    double d2 = min_image(c.pos[2 * c.n] - (double)sol.pos[2 * sol.n + r], L2);
    if ((d0 * d0 + d1 * d1) + d2 * d2 < cut_sq_c) {
        double u;
        if (draws) {
            u = draws[k];
        } else {
            uint64_t a, b;
            threefry2x64(step, (uint64_t)sol.id[r], seed, STREAM_CHANGE, a, b);
            u = u01(a);
        }
        if (u <= prob) sol.flags[r] = (typename F::small)((int)sol.flags[r] | REAC_MASK);
    }
}

// change_species of the fixed-sphere driver (setup_single_catalytic_fixed_sphere.f90:331-349)
template <class F>
__global__ void k_change_species_sphere(PView<F> sol, PView<F64> c, double L0, double L1, double L2,
                                        double cut_sq_c)
{
    int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= sol.n) return;
    int f = (int)sol.flags[m];
    if (!(f & REAC_MASK)) return;
    double a0 = min_image(c.pos[0] - (double)sol.pos[m], L0);
    double a1 = min_image(c.pos[c.n] - (double)sol.pos[sol.n + m], L1);
    double a2 = min_image(c.pos[2 * c.n] - (double)sol.pos[2 * sol.n + m], L2);
    if ((a0 * a0 + a1 * a1) + a2 * a2 > cut_sq_c) {
        sol.species[m] = (typename F::small)2;
        sol.flags[m] = (typename F::small)(f & ~REAC_MASK);
    }
}

// refuel (single_dimer_pbc.f90:544-565)
template <class F>
__global__ void k_refuel(PView<F> sol, PView<F64> c, double L0, double L1, double L2, double far)
{
    int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= sol.n) return;
    if ((int)sol.species[m] != 2) return;
    double y0 = (double)sol.pos[m], y1 = (double)sol.pos[sol.n + m], y2 = (double)sol.pos[2 * sol.n + m];
    double a0 = min_image(c.pos[0] - y0, L0), a1 = min_image(c.pos[c.n] - y1, L1),
           a2 = min_image(c.pos[2 * c.n] - y2, L2);
    double b0 = min_image(c.pos[1] - y0, L0), b1 = min_image(c.pos[c.n + 1] - y1, L1),
           b2 = min_image(c.pos[2 * c.n + 1] - y2, L2);
    if ((a0 * a0 + a1 * a1) + a2 * a2 > far && (b0 * b0 + b1 * b1) + b2 * b2 > far)
        sol.species[m] = (typename F::small)1;
}

// ---------------------------------------------------------------------------------
template <class F>
int update_list_impl(const rmpcd_box_t *box, rmpcd_cells_t *cells, const rmpcd_particles_t *points,
                     const rmpcd_particles_t *solvent, double radius, const int32_t *stencil, int ns,
                     const rmpcd_lj_t *lj, int32_t nmax, int32_t *list, int32_t *n)
{
    Box b = make_box(box);
    int np = (int)points->n;
    int32_t *cnt = (int32_t *)workspace(WS_NLCNT, sizeof(int32_t) * (size_t)np * ns);
    // the overflow flag, written where the host reads it: no other call uses this word, and
    // each call of this one waits for its kernels
    char *pin = (char *)pinned(64);
    if (!cnt || !pin) return set_error(RMPCD_ERR_HIP, "update_list: workspace allocation failed");
    hipStream_t s = stream();
    double L0 = b.L[0] * b.a, L1 = b.L[1] * b.a, L2 = b.L[2] * b.a;  // neighbor_list.f90:92
    LJ l{};
    if (lj) l = make_lj(lj);
    k_init_cells<<<blocks_for(b.ncells, 256), 256, 0, s>>>(b.ncells, cells->is_md, cells->is_reac);
    volatile int32_t *host = (int32_t *)(pin + 32);
    *host = 0;
    auto pass = [&](int fill) {
        by_density(box, solvent->n, [&](auto lanes) {
            constexpr int LANES = decltype(lanes)::value;
            const dim3 grid(blocks_for((int64_t)ns * LANES, NL_THREADS), np);
            k_nl_pass<F, LANES><<<grid, NL_THREADS, 0, s>>>(b, view<F64>(points), view<F>(solvent), cells->cell_start,
                                                            cells->cell_count, stencil, ns, radius * radius, L0, L1, L2,
                                                            lj ? 1 : 0, l, cnt, cells->is_md, cells->is_reac, fill, nmax,
                                                            list);
        });
    };
    pass(0);
    RMPCD_LAUNCHED();
    k_nl_scan<<<np, 1024, 0, s>>>(cnt, ns, nmax, n, (int32_t *)(pin + 32));
    RMPCD_LAUNCHED();
    pass(1);
    RMPCD_LAUNCHED();
    RMPCD_HIP(hipStreamSynchronize(s));
    if (*host) return set_error(RMPCD_ERR_OVERFLOW, "maximum of neighbor list reached");
    return RMPCD_OK;
}

// the solvent's share of compute_force after the roll of the MD bits, and the colloids'
// block partials (4 per block of 256 entries, nb blocks each)
template <class F>
int force_list(const rmpcd_particles_t *ps1, const rmpcd_particles_t *ps2, const int32_t *list, const int32_t *nl,
               int32_t nmax, const double *L, const rmpcd_lj_t *lj, double *part)
{
    const int np = (int)ps1->n;
    const unsigned nb = blocks_for(nmax, 256);
    const PView<F> sol = view<F>(ps2);
    // colloids of one launch
    const int group = nmax >= CHAIN_ENTRIES ? 1 : np < CHAIN_ENTRIES / nmax ? np : CHAIN_ENTRIES / nmax;
    const bool chains = group > 1;
    uint32_t *head = nullptr, *next = nullptr;
    int rc;
    if (chains) {
        head = (uint32_t *)workspace(WS_HEAD, sizeof(uint32_t) * (size_t)sol.n);
        next = (uint32_t *)workspace(WS_AUX, sizeof(uint32_t) * (size_t)group * nmax);
        if (!head || !next) return set_error(RMPCD_ERR_HIP, "compute_force: workspace allocation failed");
        if ((rc = zeroed_open(WS_HEAD))) return rc;
    }
    hipStream_t s = stream();
    const LJ l = make_lj(lj);
    for (int c0 = 0; c0 < np; c0 += group) {
        const dim3 grid(nb, group < np - c0 ? group : np - c0);
        k_force_nl<F><<<grid, 256, 0, s>>>(view<F64>(ps1), sol, list, nl, nmax, L[0], L[1], L[2], l, part, c0, head,
                                           next);
        if (chains)
            k_force_nl_apply<F><<<grid, 256, 0, s>>>(view<F64>(ps1), sol, list, nl, nmax, L[0], L[1], L[2], l, c0, head,
                                                     next);
        RMPCD_LAUNCHED();
    }
    if (chains) zeroed_close(WS_HEAD);
    return RMPCD_OK;
}

int energy_sum_unchecked(const double *e, int64_t n, double *out)
{
    k_sum_serial<<<1, 64, 0, stream()>>>(e, n, out);
    RMPCD_LAUNCHED();
    return RMPCD_OK;
}

int force_list_unchecked(const rmpcd_particles_t *ps1, const rmpcd_particles_t *ps2, const int32_t *list,
                         const int32_t *nl, int32_t nmax, const double *L, const rmpcd_lj_t *lj, double *part)
{
    return RMPCD_DISPATCH_FORM(ps2, force_list, ps1, ps2, list, nl, nmax, L, lj, part);
}

int force_sum_unchecked(const rmpcd_particles_t *ps1, const double *part, int nb, double *e_out)
{
    k_force_nl_sum<<<(unsigned)ps1->n, 64, 0, stream()>>>(view<F64>(ps1), part, nb, e_out);
    RMPCD_LAUNCHED();
    return RMPCD_OK;
}

template <class F>
int force_impl(rmpcd_particles_t *ps1, rmpcd_particles_t *ps2, const int32_t *list, const int32_t *nl,
               int32_t nmax, const double *L, const rmpcd_lj_t *lj, double *e)
{
    const int np = (int)ps1->n;
    const unsigned nb = blocks_for(nmax, 256);
    double *part = (double *)workspace(WS_PART, sizeof(double) * 4 * (size_t)nb * np);
    double *eb = (double *)workspace(WS_RED, sizeof(double) * np);
    double *host = (double *)pinned(64);
    if (!part || !eb || !host) return set_error(RMPCD_ERR_HIP, "compute_force: workspace allocation failed");
    hipStream_t s = stream();
    const PView<F> sol = view<F>(ps2);
    k_roll_md<F><<<blocks_for(sol.n, 256), 256, 0, s>>>(sol.n, sol.flags);
    RMPCD_LAUNCHED();
    int rc = force_list<F>(ps1, ps2, list, nl, nmax, L, lj, part);
    if (rc) return rc;
    if ((rc = force_sum_unchecked(ps1, part, (int)nb, eb))) return rc;
    k_sum_serial<<<1, 64, 0, s>>>(eb, np, host);
    RMPCD_LAUNCHED();
    RMPCD_HIP(hipStreamSynchronize(s));
    *e = host[0];
    return RMPCD_OK;
}

}  // namespace rmpcd

using namespace rmpcd;

extern "C" {

int rmpcd_update_list(const rmpcd_box_t *box, rmpcd_cells_t *cells, const rmpcd_particles_t *points,
                      const rmpcd_particles_t *solvent, double radius, const int32_t *stencil,
                      int32_t n_stencil, const rmpcd_lj_t *lj, int32_t nmax, int32_t *list, int32_t *n)
{
    int rc = check_box(box, "update_list");
    if (!rc) rc = check_particles(points, "update_list", false);
    if (!rc) rc = check_particles(solvent, "update_list", false);
    if (rc) return rc;
    RMPCD_CHECK(points->form == RMPCD_FP64, "update_list: points (colloids) must use the FP64 form");
    RMPCD_CHECK(points->n <= 65535, "update_list: at most 65535 points");
    RMPCD_CHECK(cells && cells->cell_count && cells->cell_start && cells->is_md && cells->is_reac,
                "update_list: null cell arrays");
    RMPCD_CHECK(stencil && n_stencil > 0 && list && n && nmax > 0, "update_list: bad list arguments");
    return RMPCD_DISPATCH_FORM(solvent, update_list_impl, box, cells, points, solvent, radius, stencil,
                               n_stencil, lj, nmax, list, n);
}

int rmpcd_compute_force(rmpcd_particles_t *ps1, rmpcd_particles_t *ps2, const int32_t *list,
                        const int32_t *n, int32_t nmax, const double L[3], const rmpcd_lj_t *lj, double *e)
{
    int rc = check_particles(ps1, "compute_force", true);
    if (!rc) rc = check_particles(ps2, "compute_force", true);
    if (rc) return rc;
    RMPCD_CHECK(ps1->form == RMPCD_FP64, "compute_force: colloids must use the FP64 form");
    RMPCD_CHECK(ps1->n <= 65535, "compute_force: at most 65535 colloids");
    RMPCD_CHECK(list && n && nmax > 0 && L && lj && e, "compute_force: null argument");
    return RMPCD_DISPATCH_FORM(ps2, force_impl, ps1, ps2, list, n, nmax, L, lj, e);
}

int rmpcd_compute_force_n2(rmpcd_particles_t *ps, const double L[3], const rmpcd_lj_t *lj, double *e)
{
    int rc = check_particles(ps, "compute_force_n2", true);
    if (rc) return rc;
    RMPCD_CHECK(ps->form == RMPCD_FP64, "compute_force_n2: colloids must use the FP64 form");
    RMPCD_CHECK(L && lj && e, "compute_force_n2: null argument");
    int64_t n = ps->n;
    double *ep = (double *)workspace(WS_PART, sizeof(double) * (n + 1));
    double *host = (double *)pinned(64);
    if (!ep || !host) return set_error(RMPCD_ERR_HIP, "compute_force_n2: workspace allocation failed");
    hipStream_t s = stream();
    const PView<F64> c = view<F64>(ps);
    k_force_n2_blocks<256><<<(unsigned)n, 256, 0, s>>>(c.pos, c.species, n, c.force, L[0], L[1], L[2], make_lj(lj), ep);
    RMPCD_LAUNCHED();
    k_sum_block<256><<<1, 256, 0, s>>>(ep, n, host);
    RMPCD_LAUNCHED();
    RMPCD_HIP(hipStreamSynchronize(s));
    *e = host[0];
    return RMPCD_OK;
}

int rmpcd_flag_particles_nl(rmpcd_particles_t *solvent, const rmpcd_particles_t *colloids,
                            const int32_t *list, const int32_t *n, int32_t nmax, const double edges[3],
                            double cut_sq_c)
{
    int rc = check_particles(solvent, "flag_particles_nl", false);
    if (!rc) rc = check_particles(colloids, "flag_particles_nl", false);
    if (rc) return rc;
    RMPCD_CHECK(colloids->form == RMPCD_FP64, "flag_particles_nl: colloids must use the FP64 form");
    RMPCD_CHECK(list && n && edges && nmax > 0, "flag_particles_nl: null argument");
    // the list length is read on the device; launch for the list capacity of colloid 0
    int64_t cap = nmax;
    hipStream_t s = stream();
    if (solvent->form == RMPCD_FP64)
        k_flag_nl<F64><<<blocks_for(cap, 256), 256, 0, s>>>(view<F64>(solvent), view<F64>(colloids), list, n,
                                                            nmax, edges[0], edges[1], edges[2], cut_sq_c);
    else
        k_flag_nl<F32><<<blocks_for(cap, 256), 256, 0, s>>>(view<F32>(solvent), view<F64>(colloids), list, n,
                                                            nmax, edges[0], edges[1], edges[2], cut_sq_c);
    RMPCD_LAUNCHED();
    return RMPCD_OK;
}

int rmpcd_change_species(rmpcd_particles_t *solvent, const rmpcd_particles_t *colloids, const double edges[3],
                         double cut_sq_c, double cut_sq_n, double prob, const double *draws, uint64_t seed,
                         uint64_t step)
{
    int rc = check_particles(solvent, "change_species", false);
    if (!rc) rc = check_particles(colloids, "change_species", false);
    if (rc) return rc;
    RMPCD_CHECK(colloids->form == RMPCD_FP64 && colloids->n >= 2, "change_species: needs two FP64 colloids");
    RMPCD_CHECK(edges && (draws || solvent->id), "change_species: null argument");
    hipStream_t s = stream();
    if (solvent->form == RMPCD_FP64)
        k_change_species<F64><<<blocks_for(solvent->n, 256), 256, 0, s>>>(
            view<F64>(solvent), view<F64>(colloids), edges[0], edges[1], edges[2], cut_sq_c, cut_sq_n, prob,
            draws, seed, step);
    else
        k_change_species<F32><<<blocks_for(solvent->n, 256), 256, 0, s>>>(
            view<F32>(solvent), view<F64>(colloids), edges[0], edges[1], edges[2], cut_sq_c, cut_sq_n, prob,
            draws, seed, step);
    RMPCD_LAUNCHED();
    return RMPCD_OK;
}

int rmpcd_flag_particles_nl_prob(rmpcd_particles_t *solvent, const rmpcd_particles_t *colloids,
                                 const int32_t *list, const int32_t *n, int32_t nmax, const double edges[3],
                                 double cut_sq_c, double prob, const double *draws, uint64_t seed, uint64_t step)
{
    int rc = check_particles(solvent, "flag_particles_nl", false);
    if (!rc) rc = check_particles(colloids, "flag_particles_nl", false);
    if (rc) return rc;
    RMPCD_CHECK(colloids->form == RMPCD_FP64, "flag_particles_nl: colloids must use the FP64 form");
    RMPCD_CHECK(list && n && edges && nmax > 0, "flag_particles_nl: null argument");
    RMPCD_CHECK(draws || solvent->id, "flag_particles_nl: null argument");
    hipStream_t s = stream();
    if (solvent->form == RMPCD_FP64)
        k_flag_nl_prob<F64><<<blocks_for(nmax, 256), 256, 0, s>>>(view<F64>(solvent), view<F64>(colloids), list,
                                                                  n, nmax, edges[0], edges[1], edges[2],
                                                                  cut_sq_c, prob, draws, seed, step);
    else
        k_flag_nl_prob<F32><<<blocks_for(nmax, 256), 256, 0, s>>>(view<F32>(solvent), view<F64>(colloids), list,
                                                                  n, nmax, edges[0], edges[1], edges[2],
                                                                  cut_sq_c, prob, draws, seed, step);
    RMPCD_LAUNCHED();
    return RMPCD_OK;
}

int rmpcd_change_species_sphere(rmpcd_particles_t *solvent, const rmpcd_particles_t *colloids,
                                const double edges[3], double cut_sq_c)
{
    int rc = check_particles(solvent, "change_species", false);
    if (!rc) rc = check_particles(colloids, "change_species", false);
    if (rc) return rc;
    RMPCD_CHECK(colloids->form == RMPCD_FP64 && colloids->n >= 1, "change_species: needs an FP64 colloid");
    RMPCD_CHECK(edges != nullptr, "change_species: null edges");
    hipStream_t s = stream();
    if (solvent->form == RMPCD_FP64)
        k_change_species_sphere<F64><<<blocks_for(solvent->n, 256), 256, 0, s>>>(
            view<F64>(solvent), view<F64>(colloids), edges[0], edges[1], edges[2], cut_sq_c);
    else
        k_change_species_sphere<F32><<<blocks_for(solvent->n, 256), 256, 0, s>>>(
            view<F32>(solvent), view<F64>(colloids), edges[0], edges[1], edges[2], cut_sq_c);
    RMPCD_LAUNCHED();
    return RMPCD_OK;
}

int rmpcd_refuel(rmpcd_particles_t *solvent, const rmpcd_particles_t *colloids, const double edges[3], int32_t L1)
{
    int rc = check_particles(solvent, "refuel", false);
    if (!rc) rc = check_particles(colloids, "refuel", false);
    if (rc) return rc;
    RMPCD_CHECK(colloids->form == RMPCD_FP64 && colloids->n >= 2, "refuel: needs two FP64 colloids");
    RMPCD_CHECK(edges != nullptr, "refuel: null edges");
    // far = (L(1)*0.45)**2 evaluated in default (single precision) REAL (single_dimer_pbc.f90:551)
    float farf = (float)L1 * 0.45f;
    farf = farf * farf;
    double far = (double)farf;
    hipStream_t s = stream();
    if (solvent->form == RMPCD_FP64)
        k_refuel<F64><<<blocks_for(solvent->n, 256), 256, 0, s>>>(view<F64>(solvent), view<F64>(colloids),
                                                                  edges[0], edges[1], edges[2], far);
    else
        k_refuel<F32><<<blocks_for(solvent->n, 256), 256, 0, s>>>(view<F32>(solvent), view<F64>(colloids),
                                                                  edges[0], edges[1], edges[2], far);
    RMPCD_LAUNCHED();
    return RMPCD_OK;
}

}  // extern "C"
