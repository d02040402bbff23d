// rmpcd_srdtile.hpp -- the SRD collision of a run of cells whose particles a workgroup holds
// in LDS (mpcd.f90:120-180), all its threads at work: the cell sums keep the reference's
// order on one thread per cell, while the other waves draw the axes; the rotation, which
// is per particle, runs over all threads.
#pragma once
#include "rmpcd_internal.hpp"

namespace rmpcd {

constexpr int SRD_CELLS = 64;  // cells of a run at most (the lanes of one wave)

template <class R, class S, int M>
struct SrdTile {
    S sp[M];                    // the particles' species
    uint8_t cell[M];            // and their cells in the run
    R u[3][SRD_CELLS];          // cell means
    R o[9][SRD_CELLS];          // rotation matrices, row-major
    uint8_t on[SRD_CELLS];      // cells that collide
    double cand[2][192];        // candidate points of Marsaglia's method
};

// The workgroup has 256 threads; cells [c0, c0 + ncell), ncell a power of two up to
// SRD_CELLS, the first particle in slot s; the velocities v and t.sp are staged (a barrier
// before the call, the new velocities behind the barrier that ends it).  Threefry axes keyed
// by (seed, step, cell).
template <class R, class S, int M>
__device__ inline void srd_tile(SrdTile<R, S, M> &t, R v[3][M], int64_t s, int m, int c0, int ncell,
                                const int32_t *__restrict__ start, const int32_t *__restrict__ count, uint64_t seed,
                                uint64_t step, double sin_a, double cos_a)
{
    const int tid = threadIdx.x;
    Acc3<R> old;
    int n = 0, a = 0, n_eff = 0;
    const int tries = 192 / ncell < 8 ? 192 / ncell : 8;
    if (tid < 64) {
        // the ordered sums, one lane per cell
        if (tid < ncell) {
            n = count[c0 + tid];
            a = (int)(start[c0 + tid] - s);
            for (int i = a; i < a + n; ++i) {
                t.cell[i] = (uint8_t)tid;
                if ((int)t.sp[i] > 0) {
                    for (int k = 0; k < 3; ++k) old.add(k, v[k][i]);
                    ++n_eff;
                }
            }
            const bool on = n > 1 && n_eff > 1;
            t.on[tid] = on;
            if (on)
                for (int k = 0; k < 3; ++k) t.u[k][tid] = old.sum(k) / (R)n_eff;
        }
    } else if (tid - 64 < tries * ncell) {
        // the first candidates of every cell's axis at once (the tries of rand_sphere_threefry)
        const int x = tid - 64, c = c0 + (x & (ncell - 1)), k = x / ncell;
        uint64_t p, q;
        threefry2x64(step, (uint64_t)c + ((uint64_t)k << 40), seed, STREAM_SRD, p, q);
        t.cand[0][x] = 2 * u01(p) - 1;
        t.cand[1][x] = 2 * u01(q) - 1;
    }
    __syncthreads();
    if (tid < ncell && t.on[tid]) {
        double n1 = 0, n2 = 0, r = 2;
        for (int k = 0; k < tries && !(r < 1.0); ++k) {
            n1 = t.cand[0][k * ncell + tid];
            n2 = t.cand[1][k * ncell + tid];
            r = n1 * n1 + n2 * n2;
        }
        for (uint64_t k = tries; k < 64 && !(r < 1.0); ++k) {
            uint64_t p, q;
            threefry2x64(step, (uint64_t)(c0 + tid) + (k << 40), seed, STREAM_SRD, p, q);
            n1 = 2 * u01(p) - 1;
            n2 = 2 * u01(q) - 1;
            r = n1 * n1 + n2 * n2;
        }
        const Sphere sph = marsaglia_from(n1, n2, r);
        R o[9];
        srd_matrix(sph.n[0], sph.n[1], sph.n[2], sin_a, cos_a, o);
        for (int k = 0; k < 9; ++k) t.o[k][tid] = o[k];
    }
    __syncthreads();
    for (int q = tid; q < m; q += 256) {
        const int c = t.cell[q];
        if (!t.on[c]) continue;
        R o[9];
        for (int k = 0; k < 9; ++k) o[k] = t.o[k][c];
        R w[3] = {v[0][q], v[1][q], v[2][q]};
        srd_rotate_one(w, o, t.u[0][c], t.u[1][c], t.u[2][c]);
        for (int k = 0; k < 3; ++k) v[k][q] = w[k];
    }
    __syncthreads();
    if constexpr (sizeof(R) == 4) {
        // FP32: the cell's momentum put back (srd_rotate), where every particle entered the mean
        if (tid < ncell && t.on[tid] && n_eff == n)
            srd_conserve(v[0] + a, v[1] + a, v[2] + a, n, old);
        __syncthreads();
    }
}

}  // namespace rmpcd
