// rmpcd_internal.hpp -- host-side runtime shared by the translation units of the
// library: error reporting, the launch stream, the grow-only device workspace and
// argument checks.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstdarg>
#include <cstdio>

#include "rmpcd_capi.h"
#include "rmpcd_device.hpp"

namespace rmpcd {

int set_error(int code, const char *fmt, ...);
hipStream_t stream();

// device workspace: named slots that grow on demand and live until process exit
enum Slot {
    WS_KEY = 0,     // per-particle cell key
    WS_SLOT,        // per-particle place in its tile's list
    WS_TMP,         // the tiles' particle lists
    WS_TILE,        // sort tile starts
    WS_TCOUNT,      // sort tile counts, zero between sorts
    WS_SCAN,        // scan tile sums
    WS_RED,         // reductions (doubles)
    WS_FLAG,        // status flags (ints)
    WS_LUT,         // Hilbert table of the current box
    WS_NLCNT,       // neighbour-list per-stencil-cell counts
    WS_PART,        // per-block partial sums
    WS_AUX,         // misc
    WS_HEAD,        // chains of list entries by particle, zero between calls of compute_force
    WS_COUNT
};
void *workspace(Slot s, size_t bytes);
// A slot whose words are zero between calls.  A call opens it before its first kernel that
// writes there and closes it when the one that leaves the words zero is queued; the words of
// a slot that is new, or that a call left open when it stopped at an error, are cleared when
// it is opened next (by a kernel: a call may be captured).
int zeroed_open(Slot s);
void zeroed_close(Slot s);
// host-pinned staging for synchronous scalar results
void *pinned(size_t bytes);

// the current device's address of the fixed scratch array of
// rmpcd_compute_temperature_noalloc (looked up on the device's first use)
int noalloc_scratch(double **out);

// Hilbert table of a box (cached by box shape)
const int32_t *hilbert_lut(const Box &b);

#define RMPCD_HIP(call)                                                                  \
    do {                                                                                 \
        hipError_t e_ = (call);                                                          \
        if (e_ != hipSuccess)                                                            \
            return ::rmpcd::set_error(RMPCD_ERR_HIP, "%s failed: %s", #call,             \
                                      hipGetErrorString(e_));                            \
    } while (0)

#define RMPCD_LAUNCHED()                                                                 \
    do {                                                                                 \
        hipError_t e_ = hipGetLastError();                                               \
        if (e_ != hipSuccess)                                                            \
            return ::rmpcd::set_error(RMPCD_ERR_HIP, "kernel launch failed: %s",         \
                                      hipGetErrorString(e_));                            \
    } while (0)

#define RMPCD_CHECK(cond, ...)                                                           \
    do {                                                                                 \
        if (!(cond)) return ::rmpcd::set_error(RMPCD_ERR_ARG, __VA_ARGS__);              \
    } while (0)

int check_particles(const rmpcd_particles_t *p, const char *who, bool need_force);
int check_box(const rmpcd_box_t *b, const char *who);

// rmpcd_sort on sets that the caller has checked; id_to_idx may be null (not written); even:
// the particles are known to lie about evenly in the box
int sort_unchecked(const rmpcd_box_t *box, const rmpcd_particles_t *src, rmpcd_particles_t *dst, int32_t *id_to_idx,
                   rmpcd_cells_t *cells, int wrap, bool even);

// a plain fluid's cycle on checked sets whose forces are zero: SRD on the cells of the last
// sort, n_md streaming steps, then the sort under the next grid shift
int fluid_cycle_unchecked(const rmpcd_box_t *next, const rmpcd_particles_t *src, rmpcd_particles_t *dst,
                          rmpcd_cells_t *cells, uint64_t seed, uint64_t step, int n_md, double dt);

// the parts of compute_force after the roll of the MD bits, on checked sets: the solvent's
// forces and the colloids' block partials (4 doubles per block of 256 entries), the
// partials' sums added to the colloid forces, the energies' sum in colloid order
int force_list_unchecked(const rmpcd_particles_t *ps1, const rmpcd_particles_t *ps2, const int32_t *list,
                         const int32_t *nl, int32_t nmax, const double *L, const rmpcd_lj_t *lj, double *part);
int force_sum_unchecked(const rmpcd_particles_t *ps1, const double *part, int nb, double *e_out);
int energy_sum_unchecked(const double *e, int64_t n, double *out);
// compute_temperature on checked sets, left in device (or pinned) memory
int temperature_unchecked(const rmpcd_box_t *box, const rmpcd_cells_t *cells, const rmpcd_particles_t *p, double *te);

inline unsigned blocks_for(int64_t n, int threads)
{
    int64_t b = (n + threads - 1) / threads;
    return (unsigned)(b < 1 ? 1 : b);
}

// dispatch on the numeric form of a particle set
#define RMPCD_DISPATCH_FORM(p, FN, ...)                                                  \
    ((p)->form == RMPCD_FP64 ? FN<::rmpcd::F64>(__VA_ARGS__)                             \
                             : FN<::rmpcd::F32>(__VA_ARGS__))

}  // namespace rmpcd
