// rmpcd_programs.hip -- the driver loops other than the dimer's, on device-resident state,
// in the reference's call order through this library's own entry points:
//   FLUID     test/setup_simple_fluid.f90:45-127
//   SPHERE    test/setup_single_catalytic_fixed_sphere.f90:89-253 and its helpers :311-349
//   COLLOIDS  programs/n_colloids_pbc.f90:123-346: the thermostat phase (:227-280) for
//             the first n_thermo cycles, then the production loop (:286-346) with its
//             temperature ramp
// Random numbers come from Threefry-2x64-20 keyed by (seed, stream), with the counters
// given next to each use, so that a test can reproduce every draw:
//   grid shift s        threefry((s, 0)) a, b and threefry((s, 1)) a, stream SHIFT
//   SRD axes, cycle s   Marsaglia pairs from threefry((s, cell + 2^40 k)), stream SRD
//   bulk reaction       threefry((cycle, cell)) a, stream REACTION
//   sphere flag draw    threefry((md_step, id)) a, stream CHANGE
//   colloid placement   draw k: threefry((k, 2^62)) a, stream PLACE
//   MPC-AT, cycle s     the normals of particle id: Box-Muller on threefry((2s, id)) and
//                       threefry((2s + 1, id)), stream THERMO
#include <math.h>
#include <string.h>

#include <new>
#include <vector>

#include "rmpcd_pairforce.hpp"
#include "rmpcd_programs.hpp"
#include "rmpcd_steps.hpp"

namespace rmpcd {

// ---- the MD steps, their passes fused ------------------------------------------------------
// Each kernel makes the reference's passes of one region of the step in the reference's
// order per particle.  What bounds these loops at their size (10^5 to 10^6 particles) is
// launches and waits: one wait per step, for the displacements that decide on a sort; the
// energies and the temperature stay on the device until a run ends.  As separate passes with
// four waits per step a cycle of ten SPHERE steps took 0.94 ms (L = 32, FP64) and one of
// fifty COLLOIDS steps 7.9 ms (L = 48, FP64, 52 colloids), 0.63 and 4.8 ms like this.
constexpr unsigned STEP_BLOCKS = 1024;  // workgroups of a pass over all particles that leaves a partial each

// The solvent's force reset of a SPHERE step (the new force array zeroed, the MD bits rolled;
// neighbor_list.f90:180-188) falls on two kernels: the list's particles have it in
// k_sphere_list, which marks them, the others in k_sphere_finish, which removes the mark.  A
// step that stops at a failed list build has then touched neither, as in the reference.
constexpr int LISTED_MASK = 1 << 7;  // a bit of the flags that no state shows between steps

__device__ inline int roll_md(int f)
{
    f = (f & MD_MASK) ? (f | PAST_MD_MASK) : (f & ~PAST_MD_MASK);
    return f & ~MD_MASK;
}

// SPHERE, before the decision: md_pos and maximum_displacement
template <class F>
__global__ void __launch_bounds__(256)
    k_sphere_move(PView<F> p, const typename F::real *__restrict__ pos_old, double dt, double *__restrict__ part)
{
    using R = typename F::real;
    __shared__ double red[16];
    const R rdt = (R)dt, dt_sq = (R)((dt * dt) / 2);
    double r_sq = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < p.n; i += (int64_t)gridDim.x * blockDim.x) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int64_t q = k * p.n + i;
            p.pos[q] = (p.pos[q] + rdt * p.vel[q]) + dt_sq * p.force[q];
        }
        r_sq = fmax(r_sq, disp_sq<F>(p, pos_old, i));
    }
    const double m = block_max(r_sq, red);
    if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// SPHERE: compute_force on the list of colloid 0, and flag_particles_nl of its driver
// (setup_single_catalytic_fixed_sphere.f90:311-329), which reads neither the velocities nor
// the bits that md_vel writes in between
template <class F>
__global__ void __launch_bounds__(256)
    k_sphere_list(PView<F64> c, PView<F> sol, const int32_t *__restrict__ list, const int32_t *__restrict__ nl,
                  int32_t nmax, double L0, double L1, double L2, LJ lj, double prob, uint64_t seed, uint64_t step,
                  double *__restrict__ part)
{
    using R = typename F::real;
    __shared__ double red[16];
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int n = min(nl[0], nmax);
    double f[3] = {0, 0, 0}, e = 0;
    if (k < n) {
        const int idx = list[k];
        int fl = (int)sol.flags[idx];
        // (a stencil wider than the box lists a particle twice)
        R g[3] = {0, 0, 0};
        if (fl & LISTED_MASK)
            for (int q = 0; q < 3; ++q) g[q] = sol.force[q * sol.n + idx];
        else
            fl = roll_md(fl) | LISTED_MASK;
        if (pair_force<F>(c, sol, 0, idx, L0, L1, L2, lj, f, &e)) {
            for (int q = 0; q < 3; ++q) g[q] = g[q] - (R)f[q];
            fl |= MD_MASK | (c.species[0] == 1 ? CATALYZED_MASK : 0);
        }
        for (int q = 0; q < 3; ++q) sol.force[q * sol.n + idx] = g[q];
        if ((int)sol.species[idx] == 1) {
            const double d0 = min_image(c.pos[0] - (double)sol.pos[idx], L0);
            const double d1 = min_image(c.pos[c.n] - (double)sol.pos[sol.n + idx], L1);
            const double d2 = min_image(c.pos[2 * c.n] - (double)sol.pos[2 * sol.n + idx], L2);
            if ((d0 * d0 + d1 * d1) + d2 * d2 < lj.cut_sq[0]) {
                uint64_t a, b;
                threefry2x64(step, (uint64_t)sol.id[idx], seed, STREAM_CHANGE, a, b);
                if (u01(a) <= prob) fl |= REAC_MASK;
            }
        }
        sol.flags[idx] = (typename F::small)fl;
    }
    double *pp = part + 4 * (int64_t)blockIdx.x;
    if ((int)(blockIdx.x * blockDim.x) >= n) {
        if (threadIdx.x < 4) pp[threadIdx.x] = 0;
        return;
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

// SPHERE, the end of the step: md_vel (md.f90:219-237) and change_species
// (setup_single_catalytic_fixed_sphere.f90:331-349)
template <class F>
__global__ void __launch_bounds__(256)
    k_sphere_finish(PView<F> p, PView<F64> c, double dt, double L0, double L1, double L2, double cut_sq_c)
{
    using R = typename F::real;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= p.n) return;
    const int old = (int)p.flags[i];
    const bool listed = (old & LISTED_MASK) != 0;
    int f = listed ? old & ~LISTED_MASK : roll_md(old);
    R fn[3];  // read beside the flags, not after them
    for (int k = 0; k < 3; ++k) fn[k] = p.force[k * p.n + i];
    if (!listed)
        for (int k = 0; k < 3; ++k) p.force[k * p.n + i] = fn[k] = 0;
    if (!(f & WALL_MASK)) {
        const R rdt = (R)dt;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int64_t q = k * p.n + i;
            p.vel[q] = p.vel[q] + (rdt * (fn[k] + p.force_old[q])) / (R)2;
        }
    } else {
        f &= ~WALL_MASK;
    }
    if (f & REAC_MASK) {
        const double a0 = min_image(c.pos[0] - (double)p.pos[i], L0);
        const double a1 = min_image(c.pos[c.n] - (double)p.pos[p.n + i], L1);
        const double a2 = min_image(c.pos[2 * c.n] - (double)p.pos[2 * p.n + i], L2);
        if ((a0 * a0 + a1 * a1) + a2 * a2 > cut_sq_c) {
            p.species[i] = (typename F::small)2;
            f &= ~REAC_MASK;
        }
    }
    if (f != old) p.flags[i] = (typename F::small)f;
}

// COLLOIDS: cell_md_pos with md_flag true and cell_maximum_displacement over the same cells
template <class F, int LANES>
__global__ void __launch_bounds__(256)
    k_cells_move(int ncells, const int32_t *__restrict__ start, const int32_t *__restrict__ count,
                 const uint8_t *__restrict__ is_md, PView<F> p, const typename F::real *__restrict__ pos_old, double dt,
                 double *__restrict__ part)
{
    using R = typename F::real;
    __shared__ double red[16];
    const R rdt = (R)dt, dt_sq = (R)((dt * dt) / 2);
    double r_sq = 0;
    for_md_cells<LANES>(ncells, start, count, is_md, 1, [&](int64_t j) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int64_t q = k * p.n + j;
            p.pos[q] = (p.pos[q] + rdt * p.vel[q]) + dt_sq * p.force[q];
        }
        r_sq = fmax(r_sq, disp_sq<F>(p, pos_old, j));
    });
    const double m = block_max(r_sq, red);
    if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// COLLOIDS: the colloids' Verlet position and their displacement
__global__ void __launch_bounds__(256)
    k_colloids_move(PView<F64> c, const double *__restrict__ mass, const double *__restrict__ pos_old, double dt,
                    double *__restrict__ part)
{
    __shared__ double red[16];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    double r_sq = 0;
    if (i < c.n) {
        for (int k = 0; k < 3; ++k) {
            const int64_t q = k * c.n + i;
            c.pos[q] = (c.pos[q] + dt * c.vel[q]) + ((dt * dt) * c.force[q]) / (2 * mass[i]);
        }
        r_sq = disp_sq<F64>(c, pos_old, i);
    }
    const double m = block_max(r_sq, red);
    if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// the solvent's force reset of a step: zeroed, the MD bits rolled (neighbor_list.f90:180-188)
template <class F>
__global__ void __launch_bounds__(256) k_force_reset(PView<F> p)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= p.n) return;
    for (int k = 0; k < 3; ++k) p.force[k * p.n + i] = 0;
    p.flags[i] = (typename F::small)roll_md((int)p.flags[i]);
}

// COLLOIDS, one workgroup per colloid: its list partials, compute_force_n2 and its Verlet
// velocity
template <int T>
__global__ void __launch_bounds__(T)
    k_colloids_finish(PView<F64> c, const double *__restrict__ mass, const double *__restrict__ part, int nb, double L0,
                      double L1, double L2, LJ lj, double dt, double *__restrict__ e1, double *__restrict__ e2)
{
    __shared__ double red[16], sum[4];
    const int64_t i = blockIdx.x;
    const double a = list_force_sum(part, nb, i);
    if (threadIdx.x < 4) sum[threadIdx.x] = a;
    double f[3], e;
    n2_pair_sums<T>(c.pos, c.species, c.n, i, L0, L1, L2, lj, red, f[0], f[1], f[2], e);
    if (threadIdx.x < 3) {
        const int64_t q = threadIdx.x * c.n + i;
        const double s = threadIdx.x == 0 ? f[0] : threadIdx.x == 1 ? f[1] : f[2];
        const double fn = (0.0 + a) + s;
        c.force[q] = fn;
        c.vel[q] = c.vel[q] + (dt * (fn + c.force_old[q])) / (2 * mass[i]);
    }
    if (threadIdx.x == 0) {
        e1[i] = sum[3];
        e2[i] = e;
    }
}

// sqrt of the maxima of a step's displacement partials: the one wait of an MD step
static int fetch_max2(const double *part, int64_t n, const double *part2, int64_t n2, double *r, double *r2)
{
    double *host = (double *)pinned(64);
    if (!host) return set_error(RMPCD_ERR_HIP, "program: pinned staging allocation failed");
    k_max_final<1024><<<part2 ? 2 : 1, 1024, 0, stream()>>>(part, n, host, part2, n2);
    RMPCD_LAUNCHED();
    RMPCD_HIP(hipStreamSynchronize(stream()));
    *r = sqrt(host[0]);
    if (r2) *r2 = sqrt(host[1]);
    return RMPCD_OK;
}

int ProgramSim::fetch_scalars()
{
    double *host = (double *)pinned(64);
    if (!host) return set_error(RMPCD_ERR_HIP, "program: pinned staging allocation failed");
    hipStream_t st = stream();
    int rc;
    if (have_e) {
        if ((rc = energy_sum_unchecked(dev_e1, nc, host))) return rc;
        if (cfg.kind == RMPCD_PROG_COLLOIDS) {
            k_sum_block<256><<<1, 256, 0, st>>>(dev_e2, nc, host + 1);
            RMPCD_LAUNCHED();
        }
    }
    if (have_te) RMPCD_HIP(hipMemcpyAsync(host + 2, dev_te, sizeof(double), hipMemcpyDeviceToHost, st));
    RMPCD_HIP(hipStreamSynchronize(st));
    if (have_e) {
        e1 = host[0];
        if (cfg.kind == RMPCD_PROG_COLLOIDS) e2 = host[1];
    }
    if (have_te) temperature = host[2];
    have_e = have_te = false;
    return RMPCD_OK;
}

int ProgramSim::setup(const rmpcd_program_config_t &c)
{
    cfg = c;
    RMPCD_CHECK(cfg.kind == RMPCD_PROG_FLUID || cfg.kind == RMPCD_PROG_SPHERE || cfg.kind == RMPCD_PROG_COLLOIDS,
                "program: unknown kind");
    RMPCD_CHECK(cfg.n_md > 0 && cfg.tau > 0 && cfg.rho > 0, "program: N_MD, tau and rho must be positive");
    RMPCD_CHECK(cfg.form == RMPCD_FP64 || cfg.form == RMPCD_FP32, "program: unknown form");
    RMPCD_CHECK(!cfg.graph || (cfg.kind == RMPCD_PROG_COLLOIDS && cfg.n_thermo == 0 && !cfg.thermostat),
                "program: the graph mode runs the COLLOIDS production loop with SRD (no thermostat)");
    int rc = rmpcd_box_init(&box, cfg.L, 1.0, 0);
    if (rc) return rc;
    seed = cfg.seed;
    dt = cfg.tau / cfg.n_md;
    int64_t vol = (int64_t)cfg.L[0] * cfg.L[1] * cfg.L[2];
    n = (int64_t)cfg.rho * vol;
    double sigma = cfg.sigma, f6 = pow(2.0, 1.0 / 6.0);
    double sigma_cut = sigma * f6;
    if (cfg.kind == RMPCD_PROG_SPHERE) {
        nc = 1;
        // mass = rho * sigma**3 * 4 * 3.14159265/3, the literal in default REAL (:103)
        mass = (((cfg.rho * (sigma * sigma * sigma)) * 4) * (double)3.14159265f) / 3;
        double eps[2] = {cfg.epsilon, cfg.epsilon}, sig[2] = {sigma, sigma}, cut[2] = {sigma_cut, sigma_cut};
        if ((rc = rmpcd_lj_params_init(&lj_sc, 2, 1, eps, sig, cut))) return rc;
        skin = cfg.skin > 0 ? cfg.skin : 1.5;  // :175
        nmax = (int)(300 * (sigma * sigma * sigma));  // neigh%init(colloids%Nmax, int(300*sigma**3)), :173
    } else if (cfg.kind == RMPCD_PROG_COLLOIDS) {
        nc = cfg.n_colloids;
        RMPCD_CHECK(nc > 0 && nc <= 100000, "program: n_colloids must be in [1, 100000]");
        // mass = rho * sigma**3 * 4 * 3.141/3 (n_colloids_pbc.f90:123)
        mass = (((cfg.rho * (sigma * sigma * sigma)) * 4) * (double)3.141f) / 3;
        // N = rho*L(1)*L(2)*L(3) - int(rho*4*3.142/3 * sigma**3*colloids%Nmax) (:147): the
        // left factor is evaluated in default REAL
        float lf = (float)(cfg.rho * 4) * 3.142f;
        lf = lf / 3.0f;
        double excl = ((double)lf * (sigma * sigma * sigma)) * (double)nc;
        n = (int64_t)cfg.rho * vol - (int64_t)excl;
        if (n <= 0) return set_error(RMPCD_ERR_ARG, "Not enough volume available for solvent");
        double eps = cfg.epsilon, e2c = cfg.epsilon_colloids;
        if ((rc = rmpcd_lj_params_init(&lj_sc, 1, 1, &eps, &sigma, &sigma_cut))) return rc;
        double csig = 2 * sigma, ccut = 2 * (3 * sigma);  // colloid_lj (:160-163)
        if ((rc = rmpcd_lj_params_init(&lj_cc, 1, 1, &e2c, &csig, &ccut))) return rc;
        skin = cfg.skin > 0 ? cfg.skin : 0.8;  // :212
        double rs = sigma_cut + skin;
        nmax = (int)(250 * (rs * rs));  // neigh%init(colloids%Nmax, int(250*(sigma_cut+skin)**2)), :213
    } else {
        nc = 0;
    }
    if (cfg.nmax_list > 0) nmax = cfg.nmax_list;
    RMPCD_CHECK(n > 0 && n < ((int64_t)1 << 31), "program: solvent count out of range");
    radius = sigma_cut + skin;

    size_t RS = rsize(cfg.form), SS = ssize(cfg.form);
    for (int b = 0; b < 2; ++b) {
        if ((rc = alloc(&sol_pos[b], 3 * n * RS))) return rc;
        if ((rc = alloc(&sol_vel[b], 3 * n * RS))) return rc;
        if ((rc = alloc((void **)&sol_image[b], 3 * n * 4))) return rc;
        if ((rc = alloc((void **)&sol_id[b], n * 4))) return rc;
        if ((rc = alloc(&sol_species[b], n * SS))) return rc;
        if ((rc = alloc(&sol_flags[b], n * SS))) return rc;
    }
    for (int b = 0; b < 4; ++b)
        if ((rc = alloc(&sol_force[b], 3 * n * RS))) return rc;
    if ((rc = alloc((void **)&cell_count, box.ncells * 4))) return rc;
    if ((rc = alloc((void **)&cell_start, box.ncells * 4))) return rc;
    if ((rc = alloc((void **)&is_md, box.ncells))) return rc;
    if ((rc = alloc((void **)&is_reac, box.ncells))) return rc;
    if ((rc = alloc((void **)&scratch, 1 << 16))) return rc;
    dev_te = scratch + 64;
    if (nc) {
        size_t c3 = 3 * (size_t)nc * sizeof(double);
        if ((rc = alloc((void **)&col_pos, c3))) return rc;
        if ((rc = alloc((void **)&col_pos_old, c3))) return rc;
        if ((rc = alloc((void **)&col_vel, c3))) return rc;
        if ((rc = alloc((void **)&col_force[0], c3))) return rc;
        if ((rc = alloc((void **)&col_force[1], c3))) return rc;
        if ((rc = alloc((void **)&col_image, 3 * (size_t)nc * 4))) return rc;
        if ((rc = alloc((void **)&col_id, (size_t)nc * 4))) return rc;
        if ((rc = alloc((void **)&col_species, (size_t)nc * 4))) return rc;
        if ((rc = alloc((void **)&col_flags, (size_t)nc * 4))) return rc;
        if ((rc = alloc((void **)&col_mass, (size_t)nc * 8))) return rc;
        if ((rc = alloc((void **)&list, (size_t)nc * nmax * 4))) return rc;
        if ((rc = alloc((void **)&nlist, (size_t)nc * 4))) return rc;
        if ((rc = alloc((void **)&dev_e1, (size_t)nc * 8))) return rc;
        if ((rc = alloc((void **)&dev_e2, (size_t)nc * 8))) return rc;
        n_stencil = rmpcd_make_stencil(1.0, radius, nullptr, 0);
        std::vector<int32_t> st(3 * (size_t)n_stencil);
        rmpcd_make_stencil(1.0, radius, st.data(), n_stencil);
        if ((rc = alloc((void **)&stencil, st.size() * 4))) return rc;
        RMPCD_HIP(hipMemcpy(stencil, st.data(), st.size() * 4, hipMemcpyHostToDevice));
        std::vector<int32_t> ids(nc), sp(nc, 1);
        std::vector<double> ms(nc, mass);
        for (int i = 0; i < nc; ++i) ids[i] = i;
        RMPCD_HIP(hipMemcpy(col_id, ids.data(), 4 * (size_t)nc, hipMemcpyHostToDevice));
        RMPCD_HIP(hipMemcpy(col_species, sp.data(), 4 * (size_t)nc, hipMemcpyHostToDevice));
        RMPCD_HIP(hipMemcpy(col_mass, ms.data(), 8 * (size_t)nc, hipMemcpyHostToDevice));
        if ((rc = place_colloids())) return rc;
    }
    if ((rc = init_solvent())) return rc;

    rmpcd_particles_t s, p;
    switch (cfg.kind) {
    case RMPCD_PROG_FLUID:
        // sort, count, first grid shift (setup_simple_fluid.f90:82-86)
        if ((rc = sort(false))) return rc;
        if ((rc = shift(0))) return rc;
        break;
    case RMPCD_PROG_SPHERE:
        // sort, list, first forces (:171-184); pos_old keeps the unsorted positions
        if ((rc = sort(false))) return rc;
        if ((rc = build_list())) return rc;
        s = sv();
        p = cv();
        if ((rc = rmpcd_compute_force(&p, &s, list, nlist, nmax, box.edges, &lj_sc, &e1))) return rc;
        RMPCD_HIP(hipMemcpyAsync(s.force_old, s.force, 3 * n * RS, hipMemcpyDeviceToDevice, stream()));
        RMPCD_HIP(hipMemcpyAsync(p.force_old, p.force, 3 * nc * 8, hipMemcpyDeviceToDevice, stream()));
        break;
    case RMPCD_PROG_COLLOIDS:
        // sort, list, first forces, pos_old = pos (n_colloids_pbc.f90:209-226)
        if ((rc = sort(false))) return rc;
        if ((rc = build_list())) return rc;
        s = sv();
        p = cv();
        if ((rc = rmpcd_compute_force(&p, &s, list, nlist, nmax, box.edges, &lj_sc, &e1))) return rc;
        if ((rc = rmpcd_compute_force_n2(&p, box.edges, &lj_cc, &e2))) return rc;
        RMPCD_HIP(hipMemcpyAsync(s.force_old, s.force, 3 * n * RS, hipMemcpyDeviceToDevice, stream()));
        RMPCD_HIP(hipMemcpyAsync(p.force_old, p.force, 3 * nc * 8, hipMemcpyDeviceToDevice, stream()));
        if ((rc = copy_pos_old())) return rc;
        break;
    }
    RMPCD_HIP(hipStreamSynchronize(stream()));
    return RMPCD_OK;
}

// colloid positions: the box centre (setup_single_catalytic_fixed_sphere.f90:150), or
// uniform draws rejected within colloid_lj sigma of an earlier colloid
// (n_colloids_pbc.f90:189-205)
int ProgramSim::place_colloids()
{
    std::vector<double> pos(3 * (size_t)nc);
    if (cfg.kind == RMPCD_PROG_SPHERE) {
        for (int k = 0; k < 3; ++k) pos[k] = box.edges[k] / 2.0;
    } else {
        double s2 = lj_cc.sigma[0] * lj_cc.sigma[0];
        uint64_t draw = 0;
        auto uni = [&]() {
            uint64_t a, b;
            threefry2x64(draw++, 1ull << 62, seed, STREAM_PLACE, a, b);
            return u01(a);
        };
        int i = 0;
        while (i < nc) {
            RMPCD_CHECK(draw < 3000000000ull, "program: no room for the colloids");
            double x[3];
            for (int k = 0; k < 3; ++k) x[k] = uni() * cfg.L[k];
            bool tooclose = false;
            for (int j = 0; j < i && !tooclose; ++j) {
                double r[3];
                for (int k = 0; k < 3; ++k) r[k] = min_image(x[k] - pos[(size_t)k * nc + j], box.edges[k]);
                if ((r[0] * r[0] + r[1] * r[1]) + r[2] * r[2] < s2) tooclose = true;
            }
            if (!tooclose) {
                for (int k = 0; k < 3; ++k) pos[(size_t)k * nc + i] = x[k];
                ++i;
            }
        }
    }
    RMPCD_HIP(hipMemcpy(col_pos, pos.data(), 8 * pos.size(), hipMemcpyHostToDevice));
    return RMPCD_OK;
}

template <class F>
static int init_solvent_t(ProgramSim &s)
{
    hipStream_t st = stream();
    rmpcd_particles_t sv = s.sv();
    PView<F> p = view<F>(&sv);
    k_fill_state<F><<<blocks_for(s.n, 256), 256, 0, st>>>(p);
    RMPCD_LAUNCHED();
    unsigned nb = blocks_for(s.n, 256);
    double *part = (double *)workspace(WS_PART, sizeof(double) * 3 * (nb + 1));
    if (!part) return set_error(RMPCD_ERR_HIP, "program: workspace allocation failed");
    double *sum = s.scratch;
    // SPHERE: uniform velocities (random_number - 0.5) * sqrt(12 T) (:143-144);
    // FLUID, COLLOIDS: sqrt(T) times normals
    bool uniform = s.cfg.kind == RMPCD_PROG_SPHERE;
    double scale = uniform ? sqrt(12 * s.cfg.T) : sqrt(s.cfg.T);
    k_init_velocities<F><<<nb, 256, 0, st>>>(p, s.seed, scale, part, uniform ? 1 : 0);
    RMPCD_LAUNCHED();
    k_sum_blocks3<3><<<1, 256, 0, st>>>(part, (int)nb, sum);
    RMPCD_LAUNCHED();
    k_remove_mean<F><<<nb, 256, 0, st>>>(p, sum);
    RMPCD_LAUNCHED();
    rmpcd_particles_t cv = s.cv();
    int32_t *fail = (int32_t *)(sum + 4);
    RMPCD_HIP(hipMemsetAsync(fail, 0, 4, st));
    const rmpcd_lj_t &l = s.lj_sc;
    k_place_random<F><<<nb, 256, 0, st>>>(p, view<F64>(&cv), s.nc, s.box.edges[0], s.box.edges[1], s.box.edges[2],
                                          l.n1 > 0 ? l.n1 : 1, l.cut_sq[0], l.cut_sq[1], l.cut_sq[2], l.cut_sq[3],
                                          s.seed, fail);
    RMPCD_LAUNCHED();
    int32_t hf = 0;
    RMPCD_HIP(hipMemcpyAsync(&hf, fail, 4, hipMemcpyDeviceToHost, st));
    RMPCD_HIP(hipStreamSynchronize(st));
    if (hf) return set_error(RMPCD_ERR_ARG, "program: random placement found no free position");
    return RMPCD_OK;
}

int ProgramSim::init_solvent()
{
    return cfg.form == RMPCD_FP64 ? init_solvent_t<F64>(*this) : init_solvent_t<F32>(*this);
}

// FLUID collision cycle c (setup_simple_fluid.f90:108-118): SRD on the cells of the last
// sort, streaming, the next grid shift, sort
int ProgramSim::fluid_cycle()
{
    rmpcd_particles_t s = sv(), d = alt();
    rmpcd_cells_t c = cells();
    int rc = shift((uint64_t)cycles + 1);
    if (rc) return rc;
    if ((rc = fluid_cycle_unchecked(&box, &s, &d, &c, seed, (uint64_t)cycles, cfg.n_md, dt))) return rc;
    cur = 1 - cur;
    md_steps += cfg.n_md;
    ++cycles;
    return RMPCD_OK;
}

// SPHERE MD step (setup_single_catalytic_fixed_sphere.f90:190-228)
template <class F>
static int sphere_step_t(ProgramSim &m)
{
    hipStream_t st = stream();
    rmpcd_particles_t s = m.sv();
    const unsigned nb = blocks_for(m.n, 256) < STEP_BLOCKS ? blocks_for(m.n, 256) : STEP_BLOCKS;
    const unsigned lb = blocks_for(m.nmax, 256);
    double *part = (double *)workspace(WS_PART, sizeof(double) * (4 * (size_t)lb > nb ? 4 * (size_t)lb : nb));
    if (!part) return set_error(RMPCD_ERR_HIP, "program: workspace allocation failed");
    k_sphere_move<F><<<nb, 256, 0, st>>>(view<F>(&s), (const typename F::real *)m.alt().pos, m.dt, part);
    RMPCD_LAUNCHED();
    int rc;
    double so_max;
    if ((rc = fetch_max2(part, nb, nullptr, 0, &so_max, nullptr))) return rc;
    if (so_max >= m.skin) {
        if ((rc = m.sort(true))) return rc;  // apply_pbc, sort
        if ((rc = m.build_list())) return rc;
        if ((rc = m.copy_pos_old())) return rc;
        ++m.n_extra;
    }
    // switch(force, force_old) for both; the driver zeroes the solvent forces only
    m.fpar = 1 - m.fpar;
    m.cfpar = 1 - m.cfpar;
    s = m.sv();
    rmpcd_particles_t p = m.cv();
    const double *L = m.box.edges;
    k_sphere_list<F><<<lb, 256, 0, st>>>(view<F64>(&p), view<F>(&s), m.list, m.nlist, m.nmax, L[0], L[1], L[2],
                                         make_lj(&m.lj_sc), m.cfg.prob, m.seed, (uint64_t)m.md_steps, part);
    k_sphere_finish<F><<<blocks_for(m.n, 256), 256, 0, st>>>(view<F>(&s), view<F64>(&p), m.dt, L[0], L[1], L[2],
                                                             m.lj_sc.cut_sq[0]);
    RMPCD_LAUNCHED();
    if ((rc = force_sum_unchecked(&p, part, (int)lb, m.dev_e1))) return rc;
    m.have_e = true;
    ++m.md_steps;
    return RMPCD_OK;
}

int ProgramSim::sphere_step()
{
    return cfg.form == RMPCD_FP64 ? sphere_step_t<F64>(*this) : sphere_step_t<F32>(*this);
}

// SPHERE collision (:230-253): temperature, grid shift, sort without apply_pbc, list,
// SRD, bulk B->A reaction
int ProgramSim::sphere_collide()
{
    rmpcd_particles_t s = sv();
    rmpcd_cells_t c = cells();
    int rc = temperature_unchecked(&box, &c, &s, dev_te);
    if (rc) return rc;
    have_te = true;
    if ((rc = shift((uint64_t)cycles))) return rc;
    if ((rc = sort(false))) return rc;
    if ((rc = build_list())) return rc;
    s = sv();
    if ((rc = rmpcd_simple_mpcd_step(&box, &c, &s, nullptr, seed, (uint64_t)cycles, 0, 0.0, 0, cfg.T, 1))) return rc;
    if ((rc = rmpcd_bulk_reaction(&box, &c, &s, 2, 1, cfg.bulk_rate, cfg.tau, nullptr, seed, (uint64_t)cycles)))
        return rc;
    ++cycles;
    return RMPCD_OK;
}

// COLLOIDS MD step (n_colloids_pbc.f90:288-320): lazy streaming of the cells holding
// list particles; the others catch up (cell_md_pos/vel with md_flag false) at a sort
template <class F>
static int colloids_step_t(ProgramSim &m)
{
    hipStream_t st = stream();
    rmpcd_particles_t s = m.sv(), p = m.cv();
    rmpcd_cells_t c = m.cells();
    const unsigned nb = cell_blocks(m.box.ncells), cb = blocks_for(m.nc, 256), lb = blocks_for(m.nmax, 256);
    const size_t moves = (size_t)nb + cb, lists = 4 * (size_t)lb * m.nc;
    double *part = (double *)workspace(WS_PART, sizeof(double) * (moves > lists ? moves : lists));
    if (!part) return set_error(RMPCD_ERR_HIP, "program: workspace allocation failed");
    by_density(&m.box, m.n, [&](auto lanes) {
        k_cells_move<F, decltype(lanes)::value><<<nb, 256, 0, st>>>(m.box.ncells, c.cell_start, c.cell_count, c.is_md,
                                                                    view<F>(&s), (const typename F::real *)m.alt().pos,
                                                                    m.dt, part);
    });
    RMPCD_LAUNCHED();
    k_colloids_move<<<cb, 256, 0, st>>>(view<F64>(&p), m.col_mass, m.col_pos_old, m.dt, part + nb);
    RMPCD_LAUNCHED();
    const double k1 = (double)(m.md_steps + 1 - m.last_sort);
    int rc;
    double so_max, co_max;
    if ((rc = fetch_max2(part, nb, part + nb, cb, &so_max, &co_max))) return rc;
    // cell_maximum_displacement is at least max_v dt (particle_system.f90:408)
    const double bound = m.box.max_v * (m.dt * k1);
    if (bound > so_max) so_max = bound;
    if (co_max >= m.skin * 0.1 || so_max >= m.skin * 0.9) {
        if ((rc = rmpcd_cell_md_pos(&m.box, &c, &s, k1 * m.dt, 0))) return rc;
        if ((rc = rmpcd_cell_md_vel(&m.box, &c, &s, k1 * m.dt, 0))) return rc;
        if ((rc = rmpcd_apply_pbc(&p, m.box.edges))) return rc;
        if ((rc = m.sort(true))) return rc;
        m.last_sort = m.md_steps + 1;
        if ((rc = m.build_list())) return rc;
        if ((rc = m.copy_pos_old())) return rc;
        ++m.n_extra;
    }
    // switch(force, force_old) for both systems, then the new forces from zero
    m.fpar = 1 - m.fpar;
    m.cfpar = 1 - m.cfpar;
    s = m.sv();
    p = m.cv();
    const double *L = m.box.edges;
    k_force_reset<F><<<blocks_for(m.n, 256), 256, 0, st>>>(view<F>(&s));
    RMPCD_LAUNCHED();
    if ((rc = force_list_unchecked(&p, &s, m.list, m.nlist, m.nmax, L, &m.lj_sc, part))) return rc;
    k_colloids_finish<256><<<(unsigned)m.nc, 256, 0, st>>>(view<F64>(&p), m.col_mass, part, (int)lb, L[0], L[1], L[2],
                                                           make_lj(&m.lj_cc), m.dt, m.dev_e1, m.dev_e2);
    RMPCD_LAUNCHED();
    m.have_e = true;
    if ((rc = rmpcd_cell_md_vel(&m.box, &c, &s, m.dt, 1))) return rc;
    ++m.md_steps;
    return RMPCD_OK;
}

int ProgramSim::colloids_step()
{
    return cfg.form == RMPCD_FP64 ? colloids_step_t<F64>(*this) : colloids_step_t<F32>(*this);
}

// COLLOIDS collision (:322-344)
int ProgramSim::colloids_collide()
{
    int rc = shift((uint64_t)cycles);
    if (rc) return rc;
    rmpcd_particles_t s = sv(), p = cv();
    rmpcd_cells_t c = cells();
    double k2 = (double)(md_steps - last_sort);
    if ((rc = rmpcd_cell_md_pos(&box, &c, &s, k2 * dt, 0))) return rc;
    if ((rc = rmpcd_cell_md_vel(&box, &c, &s, k2 * dt, 0))) return rc;
    if ((rc = rmpcd_apply_pbc(&p, box.edges))) return rc;
    if ((rc = sort(true))) return rc;
    last_sort = md_steps;
    if ((rc = build_list())) return rc;
    if ((rc = copy_pos_old())) return rc;
    s = sv();
    if (cycles < cfg.n_thermo) {
        // thermostat phase: MPC-AT at T, rescale_cells every 10th loop (:277-279)
        if ((rc = rmpcd_simple_mpcd_step(&box, &c, &s, nullptr, seed, (uint64_t)cycles, 0, 0.0, 1, cfg.T,
                                          cfg.hydro)))
            return rc;
        if ((cycles + 1) % 10 == 0 && (rc = rmpcd_rescale_cells(&box, &c, &s, cfg.T))) return rc;
    } else {
        // production loop i (1-based): T ramped from T to T_final over n_loop loops (:334-336)
        const int64_t i = cycles - cfg.n_thermo + 1;
        const double T = cfg.n_loop > 1 ? cfg.T + (double)(i - 1) * (cfg.T_final - cfg.T) / (double)(cfg.n_loop - 1)
                                        : cfg.T;
        if ((rc = rmpcd_simple_mpcd_step(&box, &c, &s, nullptr, seed, (uint64_t)cycles, 0, 0.0, cfg.thermostat ? 1 : 0,
                                          T, cfg.hydro)))
            return rc;
    }
    if ((rc = temperature_unchecked(&box, &c, &s, dev_te))) return rc;
    have_te = true;
    ++cycles;
    return RMPCD_OK;
}

int ProgramSim::run(int n_cycles)
{
    if (cfg.kind == RMPCD_PROG_COLLOIDS && cfg.graph) return colloids_graph_run(*this, n_cycles);
    const int rc = run_cycles(n_cycles);
    // a run that stopped at a failed list build leaves the scalars of the steps before it
    const int rf = (have_e || have_te) && rc != RMPCD_ERR_HIP ? fetch_scalars() : RMPCD_OK;
    if (rc || rf) return rc ? rc : rf;
    RMPCD_HIP(hipStreamSynchronize(stream()));
    return RMPCD_OK;
}

int ProgramSim::run_cycles(int n_cycles)
{
    int rc;
    for (int cy = 0; cy < n_cycles; ++cy) {
        switch (cfg.kind) {
        case RMPCD_PROG_FLUID:
            if ((rc = fluid_cycle())) return rc;
            break;
        case RMPCD_PROG_SPHERE:
            for (int j = 0; j < cfg.n_md; ++j)
                if ((rc = sphere_step())) return rc;
            if ((rc = sphere_collide())) return rc;
            break;
        default:
            for (int j = 0; j < cfg.n_md; ++j)
                if ((rc = colloids_step())) return rc;
            if ((rc = colloids_collide())) return rc;
        }
    }
    return RMPCD_OK;
}

}  // namespace rmpcd

using namespace rmpcd;

extern "C" {

int rmpcd_program_create(const rmpcd_program_config_t *cfg, rmpcd_program_t **out)
{
    RMPCD_CHECK(cfg && out, "rmpcd_program_create: null argument");
    *out = nullptr;
    ProgramSim *s = new (std::nothrow) ProgramSim();
    if (!s) return set_error(RMPCD_ERR_ARG, "rmpcd_program_create: out of host memory");
    int rc = s->setup(*cfg);
    if (rc) {
        delete s;
        return rc;
    }
    *out = (rmpcd_program_t *)s;
    return RMPCD_OK;
}

int rmpcd_program_run(rmpcd_program_t *prog, int32_t n_cycles)
{
    RMPCD_CHECK(prog && n_cycles >= 0, "rmpcd_program_run: bad argument");
    return ((ProgramSim *)prog)->run(n_cycles);
}

int rmpcd_program_state(rmpcd_program_t *prog, rmpcd_particles_t *solvent, rmpcd_particles_t *colloids,
                        rmpcd_box_t *box, rmpcd_cells_t *cells, rmpcd_program_stats_t *stats)
{
    RMPCD_CHECK(prog, "rmpcd_program_state: null program");
    ProgramSim *s = (ProgramSim *)prog;
    RMPCD_HIP(hipStreamSynchronize(stream()));
    if (solvent) *solvent = s->sv();
    if (colloids) *colloids = s->cv();
    if (box) *box = s->box;
    if (cells) *cells = s->cells();
    if (stats) {
        memset(stats, 0, sizeof(*stats));
        stats->n_solvent = s->n;
        stats->n_colloids = s->nc;
        stats->md_steps = s->md_steps;
        stats->cycles = s->cycles;
        stats->n_extra_sorting = s->n_extra;
        stats->e1 = s->e1;
        stats->e2 = s->e2;
        stats->temperature = s->temperature;
        stats->dt = s->dt;
        stats->mass = s->mass;
        stats->nmax = s->nmax;
        stats->last_sort = (int32_t)s->last_sort;
        stats->list = s->list;
        stats->nlist = s->nlist;
        stats->pos_old = s->alt().pos;
        stats->colloid_pos_old = s->col_pos_old;
    }
    return RMPCD_OK;
}

int rmpcd_program_destroy(rmpcd_program_t *prog)
{
    delete (ProgramSim *)prog;
    return RMPCD_OK;
}

}  // extern "C"
