// rmpcd_steps.hpp -- pieces of the MD step shared by the entry points (rmpcd_md.hip,
// rmpcd_nlist.hip) and the programs that fuse them (rmpcd_programs.hip): the walk over the
// cells with is_md set or clear, displacements and their maximum, the pair force.
#pragma once
#include <type_traits>

#include "rmpcd_internal.hpp"

namespace rmpcd {

// cell_md_pos / cell_md_vel / cell_md_pos_{y,z}wall (md.f90:79-263) and
// cell_maximum_displacement (particle_system.f90:380-410) touch the particles of the cells
// with is_md equal to md_flag.  A wave takes CELL_WAVE consecutive cells: it reads their
// marks, starts and counts together, then goes through those that qualify with LANES lanes
// each, so that neighbouring lanes move neighbouring particles (a thread per cell walked its
// ten particles one after the other, each wave's lanes ten particles apart: for the
// velocities, positions and displacements of the md cells of an L = 48 box with 52 colloids,
// FP64, 33, 24 and 22 us then, 16, 10 and 12 us now).  LANES by the density: see by_density.
constexpr int CELL_WAVE = 32;

template <int LANES, class Fn>
__device__ inline void for_md_cells(int ncells, const int32_t *__restrict__ start, const int32_t *__restrict__ count,
                                    const uint8_t *__restrict__ is_md, int md_flag, Fn each)
{
    constexpr int GROUPS = 64 / LANES;
    const int lane = threadIdx.x & 63, sub = lane & (LANES - 1), grp = lane / LANES;
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t c = wave * CELL_WAVE + (lane & (CELL_WAVE - 1));
    int s = 0, m = 0;
    bool on = false;
    if (c < ncells) {
        s = start[c];
        m = count[c];
        on = m > 0 && (is_md[c] != 0) == (md_flag != 0);
    }
    // one bit per cell (the two halves of the wave hold the same cells)
    uint32_t todo = (uint32_t)__ballot(on);
    if constexpr (LANES < 16) {  // every cell in its turn: one or two rounds
        if (todo == 0) return;
        for (int r = 0; r < CELL_WAVE / GROUPS; ++r) {
            const int from = r * GROUPS + grp;
            const int cs = __shfl(s, from), cm = __shfl(m, from);
            const int n = todo >> from & 1 ? cm : 0;
            for (int j = sub; j < n; j += LANES) each((int64_t)cs + j);
        }
        return;
    }
    while (todo) {
        uint32_t t = todo;
        for (int k = 0; k < grp; ++k) t &= t - 1;
        const int from = t ? __ffs(t) - 1 : 0;
        const int cs = __shfl(s, from), cm = __shfl(m, from);
        const int n = t ? cm : 0;
        for (int j = sub; j < n; j += LANES) each((int64_t)cs + j);
        for (int k = 0; k < GROUPS; ++k) todo &= todo - 1;
    }
}

inline unsigned cell_blocks(int ncells) { return blocks_for(ncells, 256 / 64 * CELL_WAVE); }

// The lanes that take a cell, by the mean number of particles in one.  Lists of 1000 points,
// L = 64, FP64, at 1, 3 and 10 particles a cell: 54, 73 and 162 us; 16 lanes throughout 158, 159
// and 162; a thread per cell 62, 91 and 380.  Velocities of all cells, L = 100, FP64: 46 us at 1
// (16 lanes 86, a thread per cell 49) and 248 at 10 (a thread per cell 1536).
template <class Fn>
inline void by_density(const rmpcd_box_t *box, int64_t n, Fn fn)
{
    const double per_cell = (double)n / ((double)box->L[0] * box->L[1] * box->L[2]);
    if (per_cell >= 6)
        fn(std::integral_constant<int, 16>{});
    else if (per_cell >= 1.5)
        fn(std::integral_constant<int, 4>{});
    else
        fn(std::integral_constant<int, 2>{});
}

// the squared displacement of particle j from pos_old (particle_system.f90:357-378)
template <class F>
__device__ inline double disp_sq(const PView<F> &p, const typename F::real *__restrict__ pos_old, int64_t j)
{
    if ((int)p.species[j] < 0) return 0;
    const double d0 = (double)(p.pos[j] - pos_old[j]);
    const double d1 = (double)(p.pos[p.n + j] - pos_old[p.n + j]);
    const double d2 = (double)(p.pos[2 * p.n + j] - pos_old[2 * p.n + j]);
    return (d0 * d0 + d1 * d1) + d2 * d2;
}

// compute_force part 2 (neighbor_list.f90:191-222): the force of colloid i on entry k of
// its list, f = 0 beyond the cutoff; true when the pair is inside it
template <class F>
__device__ inline bool pair_force(const PView<F64> &c, const PView<F> &sol, int i, int idx, double L0, double L1,
                                  double L2, const LJ &lj, double f[3], double *e)
{
    const int s2 = (int)sol.species[idx];
    if (s2 <= 0) return false;
    const double d0 = min_image(c.pos[i] - (double)sol.pos[idx], L0);
    const double d1 = min_image(c.pos[c.n + i] - (double)sol.pos[sol.n + idx], L1);
    const double d2 = min_image(c.pos[2 * c.n + i] - (double)sol.pos[2 * sol.n + idx], L2);
    const double r_sq = (d0 * d0 + d1 * d1) + d2 * d2;
    const int pidx = (s2 - 1) + lj.n1 * (c.species[i] - 1);
    if (!(r_sq <= lj.cut_sq[pidx])) return false;
    const double fr = lj_force_over_r(r_sq, lj.eps[pidx], lj.sigma[pidx]);
    f[0] = fr * d0;
    f[1] = fr * d1;
    f[2] = fr * d2;
    *e = lj_energy(r_sq, lj.eps[pidx], lj.sigma[pidx], lj.cut_energy[pidx]);
    return true;
}

// component q = threadIdx.x (force 0..2, energy 3) of colloid i's block partials, staged in
// LDS and added in block order by one lane per component; any workgroup, all threads call
__device__ inline double list_force_sum(const double *__restrict__ part, int nb, int64_t i)
{
    __shared__ double lp[256][4];
    const int q = threadIdx.x;
    double a = 0;
    for (int b0 = 0; b0 < nb; b0 += 256) {
        const int m = min(256, nb - b0);
        __syncthreads();
        for (int x = q; x < 4 * m; x += blockDim.x) lp[x >> 2][x & 3] = part[4 * (i * nb + b0) + x];
        __syncthreads();
        if (q < 4)
            for (int b = 0; b < m; ++b) a += lp[b][q];
    }
    return a;
}

// the maximum of n values, written where the host reads it; the second workgroup, if any,
// takes those of a second array
template <int T>
__global__ void __launch_bounds__(T)
    k_max_final(const double *__restrict__ part, int64_t n, double *__restrict__ out, const double *__restrict__ part2,
                int64_t n2)
{
    __shared__ double red[16];
    const double *p = blockIdx.x ? part2 : part;
    const int64_t m = blockIdx.x ? n2 : n;
    double a = 0;
    for (int64_t q = threadIdx.x; q < m; q += T) a = fmax(a, p[q]);
    a = block_max(a, red);
    if (threadIdx.x == 0) out[blockIdx.x] = a;
}

}  // namespace rmpcd
