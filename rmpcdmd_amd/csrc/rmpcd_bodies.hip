// rmpcd_bodies.hip -- colloids held together by links: iterative RATTLE over a link list
// (src/md.f90:321-480), the elastic network (516-544) and the rigid body with
// quaternion velocity Verlet (547-700).
//
// The reference updates the links one after the other, each correction seeing the ones
// before it, sweep after sweep until the constraints hold.  That order is kept exactly.
// On the host the link list becomes a schedule: an update waits for the earlier updates
// that share a particle with it, and updates that share none may run side by side, so that
// every particle is read and written in the order of the sequential loops and the results
// are the reference's bit for bit.
//
// The schedule covers a block of K consecutive sweeps as one unrolled sequence, so the first
// links of sweep s + 1 start while the last ones of sweep s are still running (on a
// 300-bead shell one sweep alone takes 155 steps, each further sweep of the block about 15),
// and a step holds at most 64 updates, those with the longest way to go first: one wave runs
// it, a lane per update, and needs no barrier between steps.  The stopping test of a sweep
// needs the state at its end: the update that is a particle's last in a sweep copies the
// particle to that sweep's snapshot in LDS, the block's tests then run on the snapshots with
// all waves, and the state of the first sweep that passes is put back.  Bodies too large for
// that run sweep by sweep, level by level, from global memory.
#include <math.h>
#include <string.h>

#include <type_traits>
#include <vector>

#include "rmpcd_internal.hpp"

namespace rmpcd {

constexpr int BT = 256;           // threads of the one workgroup
constexpr int RATTLE_MAX = 1000;  // md.f90:341, :432
constexpr int KMAX = 16;          // sweeps per block at most (4 bits of the entry)
constexpr int AHEAD = 4;          // steps that a link's constants are read ahead of their use
constexpr int LC = 10;            // doubles per link of its constants
// particles of the one-wave rattle at most, for its 16-bit offsets (with 160 KiB of LDS the
// snapshot of one sweep ends it at 1687 for positions and 2250 for velocities)
constexpr int WAVE_N = 2700;
// Entries of its schedule at most, 64 MiB: every step takes 64, however few updates may run
// side by side, so a list that is one long chain would take 64 times its updates.
constexpr int64_t WAVE_ENTRIES = 1 << 22;

struct BodyMass {
    double m[16];    // particle_system%mass by species (species s at s - 1)
    double inv[16];  // 1 / mass, as the reference's i_mass
};

__device__ inline double dot3b(const double a[3], const double b[3]) { return (a[0] * b[0] + a[1] * b[1]) + a[2] * b[2]; }

// ---- the link schedules -----------------------------------------------------------------
// Built on the host from the caller's link list and kept on the device while the list is
// unchanged (compared by content on every call).
struct BlockSched {
    int K = 0, n_steps = 0;   // n_steps a multiple of 2 AHEAD
    bool too_long = false;    // more than WAVE_ENTRIES: not built
    // 64 per step, all as byte offsets that a lane can use as they are: {a | b << 16 in the
    // particles, the link's constants | sweep, where a's and b's state go in the snapshots}
    uint4 *d_ent = nullptr;
    void *block = nullptr;
};

struct Schedule {
    std::vector<int32_t> links;  // the caller's list, for the comparison
    std::vector<double> dist;
    int device = -1;             // the device whose memory holds it
    int64_t n = 0;
    int n_links = 0, n_levels = 0;
    // one sweep by level (the global-memory rattle)
    int32_t *d_i1 = nullptr, *d_i2 = nullptr, *d_start = nullptr;
    double *d_d = nullptr;
    // by link: a, b, distance; per particle: the links
    // touching it in link order (bit 31 set where it is the second particle)
    int32_t *d_la = nullptr, *d_lb = nullptr;
    double *d_dist = nullptr;
    int32_t *d_cstart = nullptr, *d_csr = nullptr;
    void *block = nullptr;
    BlockSched blocks[KMAX + 1];  // by K, built on first use
};

static Schedule g_sched[4];
static int g_sched_next = 0;

static void free_schedule(Schedule &s)
{
    for (auto &b : s.blocks) {
        if (b.block) (void)hipFree(b.block);
        b = BlockSched();
    }
    if (s.block) (void)hipFree(s.block);
    s.block = nullptr;
}

template <class T>
static int upload(T *dst, const std::vector<T> &src)
{
    if (!src.empty()) RMPCD_HIP(hipMemcpy(dst, src.data(), sizeof(T) * src.size(), hipMemcpyHostToDevice));
    return RMPCD_OK;
}

static int get_schedule(const int32_t *links, const double *dist, int n_links, int64_t n, const char *who,
                        Schedule **out)
{
    int device = 0;
    RMPCD_HIP(hipGetDevice(&device));
    for (auto &s : g_sched)
        if (s.block && s.device == device && s.n == n && s.n_links == n_links && n_links > 0 &&
            !memcmp(s.links.data(), links, sizeof(int32_t) * 2 * (size_t)n_links) &&
            !memcmp(s.dist.data(), dist, sizeof(double) * (size_t)n_links)) {
            *out = &s;
            return RMPCD_OK;
        }
    for (int l = 0; l < 2 * n_links; ++l)
        RMPCD_CHECK(links[l] >= 0 && links[l] < n, "%s: link %d names particle %d, outside [0, %lld)", who, l / 2,
                    links[l], (long long)n);
    std::vector<int32_t> last((size_t)n, 0), lvl((size_t)n_links);
    int n_levels = 0;
    for (int l = 0; l < n_links; ++l) {
        const int a = links[2 * l], b = links[2 * l + 1];
        const int v = last[a] > last[b] ? last[a] : last[b];
        lvl[l] = v;
        last[a] = last[b] = v + 1;
        if (v + 1 > n_levels) n_levels = v + 1;
    }
    const size_t nl = (size_t)n_links;
    std::vector<int32_t> start((size_t)n_levels + 1, 0), i1(nl), i2(nl), la(nl), lb(nl);
    std::vector<double> dd(nl);
    for (int l = 0; l < n_links; ++l) ++start[lvl[l] + 1];
    for (int v = 0; v < n_levels; ++v) start[v + 1] += start[v];
    std::vector<int32_t> fill(start.begin(), start.end() - 1);
    for (int l = 0; l < n_links; ++l) {
        const int k = fill[lvl[l]]++;
        i1[k] = links[2 * l];
        i2[k] = links[2 * l + 1];
        dd[k] = dist[l];
        la[l] = links[2 * l];
        lb[l] = links[2 * l + 1];
    }
    std::vector<int32_t> cstart((size_t)n + 1, 0), csr(2 * nl);
    for (int l = 0; l < n_links; ++l) {
        ++cstart[links[2 * l] + 1];
        ++cstart[links[2 * l + 1] + 1];
    }
    for (int64_t p = 0; p < n; ++p) cstart[p + 1] += cstart[p];
    std::vector<int32_t> cf(cstart.begin(), cstart.end() - 1);
    for (int l = 0; l < n_links; ++l) {
        csr[cf[links[2 * l]]++] = l;
        csr[cf[links[2 * l + 1]]++] = (int32_t)((uint32_t)l | 0x80000000u);
    }
    Schedule &s = g_sched[g_sched_next];
    g_sched_next = (g_sched_next + 1) % 4;
    if (s.block) {
        // a kernel may still read it; its memory belongs to the device it was made on
        int cur = device;
        RMPCD_HIP(hipSetDevice(s.device));
        RMPCD_HIP(hipDeviceSynchronize());
        free_schedule(s);
        RMPCD_HIP(hipSetDevice(cur));
    }
    const size_t nl1 = nl > 0 ? nl : 1;
    const size_t bytes = nl1 * 16 + nl1 * 4 * 4 + ((size_t)n_levels + 1) * 4 + ((size_t)n + 1) * 4 + 2 * nl1 * 4 + 256;
    RMPCD_HIP(hipMalloc(&s.block, bytes));
    s.d_d = (double *)s.block;
    s.d_dist = s.d_d + nl1;
    s.d_i1 = (int32_t *)(s.d_dist + nl1);
    s.d_i2 = s.d_i1 + nl1;
    s.d_la = s.d_i2 + nl1;
    s.d_lb = s.d_la + nl1;
    s.d_csr = s.d_lb + nl1;
    s.d_cstart = s.d_csr + 2 * nl1;
    s.d_start = s.d_cstart + n + 1;
    std::vector<double> dist_v(dist, dist + n_links);
    int rc;
    if ((rc = upload(s.d_d, dd)) || (rc = upload(s.d_dist, dist_v)) || (rc = upload(s.d_i1, i1)) ||
        (rc = upload(s.d_i2, i2)) || (rc = upload(s.d_la, la)) || (rc = upload(s.d_lb, lb)) ||
        (rc = upload(s.d_csr, csr)) || (rc = upload(s.d_cstart, cstart)) ||
        (rc = upload(s.d_start, start)))
        return rc;
    s.links.assign(links, links + 2 * nl);
    s.dist = dist_v;
    s.device = device;
    s.n = n;
    s.n_links = n_links;
    s.n_levels = n_levels;
    *out = &s;
    return RMPCD_OK;
}

// the unrolled schedule of K sweeps, built once per list and K (null if it is too long): each
// step takes, of the updates whose predecessors have run, the up to 64 with the longest chain
// behind them
static int get_block(Schedule &s, int K, const BlockSched **out)
{
    BlockSched &b = s.blocks[K];
    if (b.block) {
        *out = &b;
        return RMPCD_OK;
    }
    *out = nullptr;
    if (b.too_long || (int64_t)K * s.n_links > WAVE_ENTRIES) return RMPCD_OK;
    const int nl = s.n_links, nt = K * nl;
    const int32_t *links = s.links.data();
    // the next update of a's and of b's particle, the number of updates waited for, the
    // length of the longest chain from here on
    std::vector<int32_t> next(2 * (size_t)nt, -1), wait((size_t)nt, 0), height((size_t)nt, 0), last((size_t)s.n, -1),
        lastlink((size_t)s.n, -1);
    for (int l = 0; l < nl; ++l) lastlink[links[2 * l]] = lastlink[links[2 * l + 1]] = l;
    for (int t = nt - 1; t >= 0; --t) {
        const int x[2] = {links[2 * (t % nl)], links[2 * (t % nl) + 1]};
        int h = 0;
        for (int e = 0; e < 2; ++e)
            if (last[x[e]] >= 0 && !(e == 1 && x[1] == x[0])) {
                next[2 * (size_t)t + e] = last[x[e]];
                ++wait[last[x[e]]];
                if (height[last[x[e]]] > h) h = height[last[x[e]]];
            }
        height[t] = h + 1;
        last[x[0]] = last[x[1]] = t;
        if ((int64_t)height[t] * 64 > WAVE_ENTRIES) {
            b.too_long = true;
            return RMPCD_OK;
        }
    }
    // the longest chain first, the one that became ready first among equals: a list per height
    int top = 0;
    for (int t = 0; t < nt; ++t)
        if (height[t] > top) top = height[t];
    std::vector<int32_t> front((size_t)top + 1, -1), back((size_t)top + 1), behind((size_t)nt);
    auto push = [&](int32_t t) {
        const int h = height[t];
        behind[t] = -1;
        if (front[h] < 0)
            front[h] = t;
        else
            behind[back[h]] = t;
        back[h] = t;
        if (h > top) top = h;
    };
    auto any_ready = [&] {
        while (top > 0 && front[top] < 0) --top;
        return top > 0;
    };
    for (int t = 0; t < nt; ++t)
        if (wait[t] == 0) push(t);
    std::vector<uint4> ent;
    const uint32_t spare = (uint32_t)(K * s.n * 24);  // in the snapshots: a place per lane
    const uint4 idle{(uint32_t)(s.n * 24) | ((uint32_t)((s.n + 1) * 24) << 16), (uint32_t)nl * LC * 8, 0, 0};
    std::vector<int32_t> step;
    ent.reserve(2 * (size_t)nt);
    while (any_ready()) {
        step.clear();
        while (step.size() < 64 && any_ready()) {
            step.push_back(front[top]);
            front[top] = behind[front[top]];
        }
        for (const int32_t t : step) {
            const int l = t % nl, q = t / nl, a = links[2 * l], c = links[2 * l + 1];
            const uint32_t lane = (uint32_t)(ent.size() % 64);
            uint4 e;
            e.x = (uint32_t)a * 24 | ((uint32_t)c * 24 << 16);
            e.y = (uint32_t)l * LC * 8 | (uint32_t)q;
            e.z = lastlink[a] == l ? (uint32_t)((q * s.n + a) * 24) : spare + lane * 24;
            e.w = lastlink[c] == l ? (uint32_t)((q * s.n + c) * 24) : spare + lane * 24;
            ent.push_back(e);
            for (int k = 0; k < 2; ++k) {
                const int32_t w = next[2 * (size_t)t + k];
                if (w >= 0 && --wait[w] == 0) push(w);
            }
        }
        auto pad = [&] {
            uint4 e = idle;
            e.z = e.w = spare + (uint32_t)(ent.size() % 64) * 24;
            ent.push_back(e);
        };
        while (ent.size() % 64) pad();
        if (!any_ready())  // idle steps up to a whole turn, and one more turn to read ahead
            while (ent.size() % (64 * 2 * AHEAD)) pad();
        if ((int64_t)ent.size() > WAVE_ENTRIES) {
            b.too_long = true;
            return RMPCD_OK;
        }
    }
    const size_t n_ent = ent.size();
    for (int k = 0; k < 64 * 2 * AHEAD; ++k) {
        ent.push_back(idle);
        ent.back().z = ent.back().w = spare + (uint32_t)(k % 64) * 24;
    }
    RMPCD_HIP(hipMalloc(&b.block, ent.size() * sizeof(uint4)));
    b.d_ent = (uint4 *)b.block;
    int rc = upload(b.d_ent, ent);
    if (rc) return rc;
    b.K = K;
    b.n_steps = (int)(n_ent / 64);
    *out = &b;
    return RMPCD_OK;
}

// bytes of LDS the one-wave rattle takes: the particles' positions and velocities (for the
// velocities alone: velocities) with two spare particles for idle lanes, a copy of what a
// block starts from, K snapshots with a spare place per lane, flags
static size_t wave_lds_bytes(int64_t n, int K, bool with_pr)
{
    return 24 * ((size_t)(n + 2) * (with_pr ? 3 : 2) + (size_t)K * n + 64) + 2 * KMAX * 4 + 64;
}

static int lds_limit()
{
    static int limit = 0;
    if (!limit) {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v <= 0)
            v = 64 * 1024;
        limit = v;
    }
    return limit;
}

constexpr int WT = 512;  // threads of the one-wave rattle: one wave updates, all set up and test

struct WaveView {
    const uint4 *ent;
    const int32_t *la, *lb;
    const double *dist;
    const int32_t *cstart;  // links per particle, to see which have any
    int n_links, n_steps, K;
};

// a / b, correctly rounded, from y = the rounded 1 / b: Markstein's correction of a quotient
// by its exact remainder (P. W. Markstein, IBM J. Res. Dev. 34, 1990), twice; the second
// starts from a quotient within one unit in the last place, for which it is proven.  The
// caller keeps |a| and b away from the ends of the exponent range.
__device__ inline double div_by(double a, double b, double y)
{
    double q = a * y;
    q = fma(fma(-b, q, a), y, q);
    return fma(fma(-b, q, a), y, q);
}

// sqrt(x), correctly rounded, for 1e-200 < x < 1e200: a Goldschmidt step from the hardware's
// reciprocal square root, then two corrections by the exact remainder (same source); without
// the scaling and the special cases of sqrt()
__device__ inline double sqrt_mid(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    g = fma(fma(-g, g, x), h, g);
    return fma(fma(-g, g, x), h, g);
}
// how far |x| lies above 1e-200 in units of its upper word, doubled; more than MID_SPAN from
// 1e200 on, and for 0, infinities and NaN
constexpr uint32_t MID_LOW = (1023u - 665u) << 21, MID_SPAN = (665u + 664u) << 21;
__device__ inline uint32_t mid_off(double x) { return ((uint32_t)__double2hiint(x) << 1) - MID_LOW; }
// the same in single units for an x that has to be positive: more than MID_SPAN / 2 for the rest
__device__ inline uint32_t mid_off_pos(double x) { return (uint32_t)__double2hiint(x) - MID_LOW / 2; }

// The steps of a block for one wave.  A lane's update needs its entry, then the constants of
// the entry's link (and with kG the update's multiplier from g): they are read from memory
// 2 AHEAD and AHEAD steps before their use and looked at no earlier, so that a step waits
// for LDS alone.  each(entry, constants, step) runs with every lane; the idle ones, and with
// kLimit those of sweeps from ns on, have the two spare particles for their ends.
template <int NC_, bool kG, bool kLimit, class Fn>
__device__ inline void for_steps(const WaveView &w, const double *lc, const double *g, int n, int ns, Fn each)
{
    const int lane = threadIdx.x & 63;
    uint4 e[2 * AHEAD];
    double c[AHEAD][NC_ + 1];
    auto entry = [&](int s) {
        const uint4 *at = w.ent + (size_t)s * 64;
        uint4 f = at[lane];
        return f;
    };
    auto constants = [&](int d, uint32_t y, int s) {
        const double *q = (const double *)((const char *)lc + (y & ~15u));
#pragma unroll
        for (int k = 0; k < NC_; ++k) c[d][k] = q[k];
        if (kG) {
            const double *at = g + (size_t)s * 64;
            c[d][NC_] = at[lane];
        }
    };
#pragma unroll
    for (int d = 0; d < 2 * AHEAD; ++d) e[d] = entry(d);
#pragma unroll
    for (int d = 0; d < AHEAD; ++d) constants(d, e[d].y, d);
    for (int s0 = 0; s0 < w.n_steps; s0 += 2 * AHEAD) {
#pragma unroll
        for (int d = 0; d < 2 * AHEAD; ++d) {
            const int s = s0 + d;
            uint4 f = e[d];
            if (kLimit && (int)(f.y & 15) >= ns) {
                f.x = (uint32_t)(n * 24) | ((uint32_t)((n + 1) * 24) << 16);
                f.z = f.w = (uint32_t)(w.K * n * 24 + lane * 24);
            }
            each(f, c[d % AHEAD], s);
            constants(d % AHEAD, e[(d + AHEAD) % (2 * AHEAD)].y, s + AHEAD);
            e[d] = entry(s + 2 * AHEAD);
            // LDS serves a wave in order: what this step wrote, the next one reads
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// ---- rattle_body_pos (kPos) / rattle_body_vel, one wave --------------------------------
// Every particle but the first is unfolded next to particle 0 (md.f90:343-353, :427-431) and
// folded back at the end (md.f90:400-402, :474-476); pos_rattle is left unfolded, as the
// reference leaves it.  What does not change during the call is made once per link: the
// separation of pos_rattle (positions) or of the positions (velocities), its square, the
// denominator of the multiplier and its reciprocal.  The position updates do not read the
// velocities, so a second wave makes the velocity updates of a block, from the multipliers,
// while the first runs the next block.
//
// The square root and the division of an update are made without the general forms' scaling
// and special cases; what they leave out is watched for (the largest mid_off of their
// operands), and a block that met it is run again from its start with the general forms.  A
// position's multiplier needs no watch of its own: with the root between 1e-100 and 1e100 its
// numerator is +0, for which div_by is exact, or at least an ulp of the root, 1e-117, and it
// is at most 1e155, beyond which the discriminant is not finite.  (Watched too, the zeros of
// a body at rest or of links at their exact length sent blocks to the general forms: a
// 60-bead shell with half its beads at rest 459 us a call, 372 like this.)
//
// Bound by one wave's issue and the latency of a step's chain of LDS reads and FP64
// operations (one update after the other along the longest chain of links): 0.21 us a step.
// An MD step of a 300-bead shell with 1202 links, 229 and 364 sweeps: 1.9 ms for the
// positions and 2.0 for the velocities; 256 threads with a barrier per level and 12 sweeps
// per block took 4.8 and 5.0.
template <bool kPos>
__global__ void __launch_bounds__(WT)
    k_rattle_wave(PView<F64> p, double *__restrict__ gpr, WaveView w, BodyMass bm, double dt, double e0, double e1,
                  double e2, double precision, int32_t *__restrict__ out, int32_t *__restrict__ gim, double *lc,
                  double *gg)
{
    extern __shared__ double smem[];
    const int n = (int)p.n, n3 = 3 * (n + 2);
    const int tid = threadIdx.x, wave = tid >> 6;
    const int nl = w.n_links, K = w.K;
    const double edges[3] = {e0, e1, e2};
    double *X = smem;                  // positions (kPos) or velocities, x y z per particle
    double *V = kPos ? X + n3 : X;     // velocities
    double *XS = V + n3;               // X at the start of a block
    double *SN = XS + n3;              // snapshots of X, n particles per sweep, and a place per lane
    // failed sweeps of a block; those of the next block are cleared while a slow wave may
    // still look at these, so they lie apart
    int32_t *const NC2 = (int32_t *)(SN + 3 * ((size_t)K * n + 64));
    // unfold; the velocities' positions go to the snapshots' place until the links are made
    double *Q = kPos ? X : SN;
    for (int i = tid; i < n; i += WT)
        for (int k = 0; k < 3; ++k) {
            const double x0 = p.pos[k * p.n], x = p.pos[k * p.n + i];
            const int j = i == 0 ? 0 : (int)floor(((x - x0) / edges[k]) + 0.5);
            gim[k * n + i] = j;
            Q[3 * i + k] = i == 0 ? x : x - j * edges[k];
            V[3 * i + k] = p.vel[k * p.n + i];
            if (kPos) {
                const double r0 = gpr[k * p.n], r = gpr[k * p.n + i];
                const int jr = i == 0 ? 0 : (int)floor(((r - r0) / edges[k]) + 0.5);
                gpr[k * p.n + i] = i == 0 ? r : r - jr * edges[k];
            }
        }
    // the spare particles lie one apart along x; the link behind the last one, theirs, has
    // constants that keep their update harmless and in range
    if (tid < 6) X[3 * n + tid] = V[3 * n + tid] = tid == 0 ? 1 : 0;
    if (tid < LC) lc[(size_t)nl * LC + tid] = tid == 0 || (tid >= 5 && tid <= 7) ? 1 : tid == 8 ? 0.75 : 0;
    __threadfence_block();
    __syncthreads();
    for (int l = tid; l < nl; l += WT) {
        const int a = w.la[l], b = w.lb[l];
        const double ma = bm.inv[((int)p.species[a] - 1) & 15], mb = bm.inv[((int)p.species[b] - 1) & 15];
        const double d = w.dist[l];
        double *c = lc + (size_t)l * LC;
        double r[3], den;
        for (int k = 0; k < 3; ++k) {
            r[k] = kPos ? gpr[k * p.n + a] - gpr[k * p.n + b] : Q[3 * a + k] - Q[3 * b + k];
            c[k] = r[k];
        }
        const double rsq = dot3b(r, r);
        den = kPos ? (dt * (ma + mb)) * rsq : (d * d) * (ma + mb);
        c[3] = ma;
        c[4] = mb;
        c[5] = den;
        // a NaN sends the block to the general division
        c[6] = den > 1e-90 && den < 1e90 ? 1 / den : NAN;
        c[7] = rsq;
        c[8] = d * d;
    }
    __threadfence_block();
    __syncthreads();
    char *const xb = (char *)X, *const vb = (char *)V, *const sb = (char *)SN;
    // (a link from a particle to itself has r = 0: its update is NaN, or changes nothing)
    // velocity updates of a block up to sweep ns, from the block's multipliers
    auto velocity = [&](const uint4 e, const double *c, int) {
        double *va = (double *)(vb + (e.x & 0xFFFF)), *vc = (double *)(vb + (e.x >> 16));
        const double a[3] = {va[0], va[1], va[2]}, b[3] = {vc[0], vc[1], vc[2]}, g = c[5];
        for (int k = 0; k < 3; ++k) va[k] = a[k] - (g * c[k]) * c[3];
        for (int k = 0; k < 3; ++k) vc[k] = b[k] + (g * c[k]) * c[4];
    };
    // the updates of a block; kFast: false when an operand left the range of the short forms
    auto block = [&](double *g_now, int ns, auto fast, auto limit) {
        constexpr bool kFast = decltype(fast)::value, kLimit = decltype(limit)::value;
        uint32_t off = 0;
        for_steps<kPos ? 9 : 7, false, kLimit>(w, lc, nullptr, n, ns, [&](const uint4 e, const double *c, int s) {
            double *xa = (double *)(xb + (e.x & 0xFFFF)), *xc = (double *)(xb + (e.x >> 16));
            double *sa = (double *)(sb + e.z), *sc = (double *)(sb + e.w);
            const double a[3] = {xa[0], xa[1], xa[2]}, b[3] = {xc[0], xc[1], xc[2]};
            const double d[3] = {a[0] - b[0], a[1] - b[1], a[2] - b[2]};
            double g;  // the multiplier
            if (kPos) {
                const double ssq = dot3b(d, d), rs = dot3b(c, d);
                const double disc = rs * rs - c[7] * (ssq - c[8]);
                if (kFast) {
                    g = rs - sqrt_mid(disc);
                    off = max(off, mid_off_pos(disc));
                } else {
                    g = rs - sqrt(disc);
                }
            } else {
                g = dot3b(d, c);
                if (kFast) off = max(off, mid_off(g));
            }
            g = kFast ? div_by(g, c[5], c[6]) : g / c[5];
            if (kFast) off = max(off, c[6] != c[6] ? 0xffffffffu : 0u);
            const double h = kPos ? g * dt : g;
            double na[3], nb[3];
            for (int k = 0; k < 3; ++k) {
                na[k] = a[k] - (h * c[k]) * c[3];
                nb[k] = b[k] + (h * c[k]) * c[4];
            }
            for (int k = 0; k < 3; ++k) xa[k] = na[k];
            for (int k = 0; k < 3; ++k) xc[k] = nb[k];
            for (int k = 0; k < 3; ++k) sa[k] = na[k];
            for (int k = 0; k < 3; ++k) sc[k] = nb[k];
            if (kPos) {
                double *at = g_now + (size_t)s * 64;
                at[tid & 63] = g;
            }
        });
        return !__any(off > (kPos ? MID_SPAN / 2 : MID_SPAN));
    };
    const std::true_type yes{};
    const std::false_type no{};
    int it = RATTLE_MAX + 1, conv = -1, blk = 0, ns = 0;
    for (int base = 0; base < RATTLE_MAX && conv < 0; base += K, ++blk) {
        ns = K < RATTLE_MAX - base ? K : RATTLE_MAX - base;
        int32_t *const NC = NC2 + (blk & 1) * KMAX;
        double *g_now = gg + (size_t)(blk & 1) * w.n_steps * 64;
        if (wave == 0) {
            for (int i = tid; i < n3; i += 64) XS[i] = X[i];
            if (ns < K || !block(g_now, ns, yes, no)) {
                for (int i = tid; i < n3; i += 64) X[i] = XS[i];
                block(g_now, ns, no, yes);
            }
        } else if (kPos && wave == 1 && blk > 0) {
            for_steps<5, true, false>(w, lc, gg + (size_t)((blk - 1) & 1) * w.n_steps * 64, n, K, velocity);
        }
        if (tid >= WT - 64 && tid - (WT - 64) < K) NC[tid - (WT - 64)] = 0 < precision ? 0 : 1;
        __threadfence_block();
        __syncthreads();
        // the stopping test of each sweep of the block (md.f90:385-392, :454-465): a sweep
        // passes when no link reaches the precision (a NaN never does).  Items run sweep
        // fastest and skip sweeps already failed.
        const int n_items = ns * nl;
        for (int y = tid; y < n_items; y += WT) {
            const int q = y % ns, l = y / ns;
            if (((volatile int32_t *)NC)[q]) continue;
            const int a = w.la[l], b = w.lb[l];
            double r[3], err;
            for (int k = 0; k < 3; ++k) r[k] = SN[3 * (q * n + a) + k] - SN[3 * (q * n + b) + k];
            if (kPos)
                err = fabs(sqrt(dot3b(r, r)) - w.dist[l]);
            else
                err = fabs(dot3b(r, lc + (size_t)l * LC) / lc[(size_t)l * LC + 5]);
            if (err >= precision) NC[q] = 1;
        }
        __syncthreads();
        for (int q = 0; q < ns; ++q)
            if (!NC[q]) {
                conv = q;
                break;
            }
        if (conv >= 0) it = base + conv + 1;
    }
    // the velocity updates of the last block, and the state after the sweep that passed
    if (kPos && wave == 0 && blk > 0)
        for_steps<5, true, true>(w, lc, gg + (size_t)((blk - 1) & 1) * w.n_steps * 64, n, conv >= 0 ? conv + 1 : ns,
                                 velocity);
    __syncthreads();
    for (int i = tid; i < n; i += WT) {
        const bool put_back = conv >= 0 && w.cstart[i + 1] > w.cstart[i];
        for (int k = 0; k < 3; ++k) {
            const double x = put_back ? SN[3 * (conv * n + i) + k] : X[3 * i + k];
            if (kPos) p.pos[k * p.n + i] = i == 0 ? x : x + gim[k * n + i] * edges[k];
            p.vel[k * p.n + i] = kPos ? V[3 * i + k] : x;
        }
        if (!kPos && i > 0)  // unfolded and folded back as the reference does
            for (int k = 0; k < 3; ++k) {
                const int j = gim[k * n + i];
                p.pos[k * p.n + i] = (p.pos[k * p.n + i] - j * edges[k]) + j * edges[k];
            }
    }
    if (tid == 0) out[0] = it;
}

__device__ inline double body_max(double v, double *red)
{
    // every value is >= 0; max is exact in any order
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[w] = v;
    __syncthreads();
    double r = red[0];
    for (int k = 1; k < BT / 64; ++k) r = fmax(r, red[k]);
    return r;
}

struct SchedView {
    const int32_t *i1, *i2, *start;
    const double *d;
    int n_links, n_levels;
};

// ---- rattle_body_pos (kPos) / rattle_body_vel from global memory ----------------------
// For bodies whose links and schedule do not fit in LDS: one sweep at a time, its levels
// in turn, the particles updated in place.
template <bool kPos>
__global__ void __launch_bounds__(BT) k_rattle_global(PView<F64> p, double *__restrict__ pr, SchedView sv,
                                                      BodyMass bm, double dt, double e0, double e1, double e2,
                                                      double precision, int32_t *__restrict__ out,
                                                      double *__restrict__ minv, int32_t *__restrict__ im)
{
    __shared__ double red[64];
    const int64_t n = p.n;
    const int tid = threadIdx.x;
    const double edges[3] = {e0, e1, e2};
    double *pos = p.pos, *vel = p.vel;
    for (int64_t i = tid; i < n; i += BT) {
        minv[i] = bm.inv[((int)p.species[i] - 1) & 15];
        for (int k = 0; k < 3; ++k) {
            const double x0 = pos[k * n], x = pos[k * n + i];
            const int j = i == 0 ? 0 : (int)floor(((x - x0) / edges[k]) + 0.5);
            im[k * n + i] = j;
            pos[k * n + i] = i == 0 ? x : x - j * edges[k];
            if (kPos) {
                const double r0 = pr[k * n], r = pr[k * n + i];
                const int jr = i == 0 ? 0 : (int)floor(((r - r0) / edges[k]) + 0.5);
                pr[k * n + i] = i == 0 ? r : r - jr * edges[k];
            }
        }
    }
    __syncthreads();
    int it;
    for (it = 1; it <= RATTLE_MAX; ++it) {
        for (int v = 0; v < sv.n_levels; ++v) {
            for (int l = sv.start[v] + tid; l < sv.start[v + 1]; l += BT) {
                const int a = sv.i1[l], b = sv.i2[l];
                const double ma = minv[a], mb = minv[b], dl = sv.d[l];
                double s[3];
                for (int k = 0; k < 3; ++k) s[k] = pos[k * n + a] - pos[k * n + b];
                if (kPos) {
                    double r[3];
                    for (int k = 0; k < 3; ++k) r[k] = pr[k * n + a] - pr[k * n + b];
                    const double rsq = dot3b(r, r), ssq = dot3b(s, s), rs = dot3b(r, s);
                    double g = rs - sqrt(rs * rs - rsq * (ssq - dl * dl));
                    g = g / ((dt * (ma + mb)) * rsq);
                    for (int k = 0; k < 3; ++k) {
                        pos[k * n + a] = pos[k * n + a] - ((g * dt) * r[k]) * ma;
                        pos[k * n + b] = pos[k * n + b] + ((g * dt) * r[k]) * mb;
                        vel[k * n + a] = vel[k * n + a] - (g * r[k]) * ma;
                        vel[k * n + b] = vel[k * n + b] + (g * r[k]) * mb;
                    }
                } else {
                    double dv[3];
                    for (int k = 0; k < 3; ++k) dv[k] = vel[k * n + a] - vel[k * n + b];
                    const double kk = dot3b(dv, s) / ((dl * dl) * (ma + mb));
                    for (int k = 0; k < 3; ++k) {
                        vel[k * n + a] = vel[k * n + a] - (kk * s[k]) * ma;
                        vel[k * n + b] = vel[k * n + b] + (kk * s[k]) * mb;
                    }
                }
            }
            __syncthreads();
        }
        double err = 0;
        for (int l = tid; l < sv.n_links; l += BT) {
            const int a = sv.i1[l], b = sv.i2[l];
            double s[3];
            for (int k = 0; k < 3; ++k) s[k] = pos[k * n + a] - pos[k * n + b];
            double e;
            if (kPos) {
                e = fabs(sqrt(dot3b(s, s)) - sv.d[l]);
            } else {
                double dv[3];
                for (int k = 0; k < 3; ++k) dv[k] = vel[k * n + a] - vel[k * n + b];
                e = fabs(dot3b(dv, s) / ((sv.d[l] * sv.d[l]) * (minv[a] + minv[b])));
            }
            if (e > err) err = e;
        }
        err = body_max(err, red);
        if (err < precision) break;
    }
    __syncthreads();
    for (int64_t i = tid + 1; i < n; i += BT)
        for (int k = 0; k < 3; ++k) pos[k * n + i] = pos[k * n + i] + im[k * n + i] * edges[k];
    if (tid == 0) out[0] = it;
}

// elastic_network (md.f90:516-544).  The link forces are independent: made in parallel
// first.  Each particle then adds the forces of its links in link order (the per-particle
// lists of the schedule), which is the order of the reference's loop, and the energy
// terms are summed in link order.  kLds: the terms and forces of the links in LDS.
template <bool kLds>
__global__ void __launch_bounds__(BT) k_elastic_network(PView<F64> p, const int32_t *__restrict__ la,
                                                        const int32_t *__restrict__ lb, const double *__restrict__ dist,
                                                        const int32_t *__restrict__ cstart,
                                                        const int32_t *__restrict__ csr, int n_links, double kk,
                                                        double e0, double e1, double e2, double *__restrict__ gterms,
                                                        double *__restrict__ out)
{
    extern __shared__ double smem[];
    const int64_t n = p.n;
    const int tid = threadIdx.x;
    const double L[3] = {e0, e1, e2};
    double *T = kLds ? smem : gterms;
    double *F = T + n_links;
    for (int l = tid; l < n_links; l += BT) {
        const int a = la[l], b = lb[l];
        const double r0 = dist[l];
        double x[3];
        for (int k = 0; k < 3; ++k) x[k] = min_image(p.pos[k * n + a] - p.pos[k * n + b], L[k]);
        const double r = sqrt(dot3b(x, x));
        T[l] = (kk * ((r - r0) * (r - r0))) / 2;
        for (int k = 0; k < 3; ++k) F[3 * l + k] = ((-kk) * (r - r0)) * x[k] / r;
    }
    __syncthreads();
    for (int64_t i = tid; i < n; i += BT) {
        const int j0 = cstart[i], j1 = cstart[i + 1];
        if (j0 == j1) continue;
        double f[3] = {p.force[i], p.force[n + i], p.force[2 * n + i]};
        for (int j = j0; j < j1; ++j) {
            const uint32_t c = (uint32_t)csr[j];
            const int l = (int)(c & 0x7FFFFFFFu);
            if (c >> 31)
                for (int k = 0; k < 3; ++k) f[k] = f[k] - F[3 * l + k];
            else
                for (int k = 0; k < 3; ++k) f[k] = f[k] + F[3 * l + k];
        }
        for (int k = 0; k < 3; ++k) p.force[k * n + i] = f[k];
    }
    if (tid == 0) {
        double e = 0;
#pragma unroll 8
        for (int l = 0; l < n_links; ++l) e = e + T[l];
        out[0] = e;
    }
}

// ---- the rigid body (md.f90:547-700) -------------------------------------------------
// Quaternions scalar first, q = (s, v).  The reference takes them from its quaternion
// module (an absent submodule); these are the textbook definitions: Hamilton product,
// conjugate, rotation v -> q (0, v) q*.
__device__ inline void qmul(const double a[4], const double b[4], double r[4])
{
    const double s = a[0] * b[0] - ((a[1] * b[1] + a[2] * b[2]) + a[3] * b[3]);
    const double x = (a[0] * b[1] + b[0] * a[1]) + (a[2] * b[3] - a[3] * b[2]);
    const double y = (a[0] * b[2] + b[0] * a[2]) + (a[3] * b[1] - a[1] * b[3]);
    const double z = (a[0] * b[3] + b[0] * a[3]) + (a[1] * b[2] - a[2] * b[1]);
    r[0] = s;
    r[1] = x;
    r[2] = y;
    r[3] = z;
}
__device__ inline void qconj(const double q[4], double r[4])
{
    r[0] = q[0];
    r[1] = -q[1];
    r[2] = -q[2];
    r[3] = -q[3];
}
__device__ inline void qrot(const double q[4], const double v[3], double r[3])
{
    const double p[4] = {0, v[0], v[1], v[2]};
    double t[4], c[4], u[4];
    qmul(q, p, t);
    qconj(q, c);
    qmul(t, c, u);
    r[0] = u[1];
    r[1] = u[2];
    r[2] = u[3];
}
__device__ inline double qnorm(const double q[4]) { return sqrt(((q[0] * q[0] + q[1] * q[1]) + q[2] * q[2]) + q[3] * q[3]); }
__device__ inline void qnormalize(double q[4])
{
    const double s = qnorm(q);
    for (int k = 0; k < 4; ++k) q[k] = q[k] / s;
}
__device__ inline void cross3(const double a[3], const double b[3], double r[3])
{
    r[0] = a[1] * b[2] - a[2] * b[1];
    r[1] = a[2] * b[0] - a[0] * b[2];
    r[2] = a[0] * b[1] - a[1] * b[0];
}

__device__ inline bool body_range_ok(const rmpcd_rigid_body_t *b, int64_t n)
{
    return b->i_start >= 0 && b->i_stop >= b->i_start && b->i_stop < n;
}

// Sums over the body's particles keep the reference's order: the terms of a chunk of BT
// particles are made in parallel into LDS and added by thread 0 one after the other.
__global__ void __launch_bounds__(BT) k_rigid_init(rmpcd_rigid_body_t *b, PView<F64> p, BodyMass bm, double e0,
                                                   double e1, double e2)
{
    __shared__ double t[7][BT];
    __shared__ double acc[7];
    const int64_t n = p.n;
    const int tid = threadIdx.x;
    const double edges[3] = {e0, e1, e2};
    if (!body_range_ok(b, n)) return;
    const int i0 = b->i_start, i1 = b->i_stop;
    if (tid == 0)
        for (int k = 0; k < 7; ++k) acc[k] = 0;
    // mass, mass * unfolded position, mass * velocity (md.f90:561-568)
    for (int c0 = i0; c0 <= i1; c0 += BT) {
        const int i = c0 + tid;
        if (i <= i1) {
            const double m = bm.m[((int)p.species[i] - 1) & 15];
            t[0][tid] = m;
            for (int k = 0; k < 3; ++k) {
                t[1 + k][tid] = m * (p.pos[k * n + i] + p.image[k * n + i] * edges[k]);
                t[4 + k][tid] = m * p.vel[k * n + i];
            }
        }
        __syncthreads();
        if (tid == 0) {
            const int m = i1 - c0 + 1 < BT ? i1 - c0 + 1 : BT;
            for (int j = 0; j < m; ++j)
                for (int k = 0; k < 7; ++k) acc[k] = acc[k] + t[k][j];
        }
        __syncthreads();
    }
    const double mass = acc[0];
    const double com[3] = {acc[1] / mass, acc[2] / mass, acc[3] / mass};
    const double cv[3] = {acc[4] / mass, acc[5] / mass, acc[6] / mass};
    __syncthreads();
    if (tid == 0)
        for (int k = 0; k < 3; ++k) acc[k] = 0;
    // body-frame positions and the diagonal of the inertia tensor (md.f90:574-580)
    for (int c0 = i0; c0 <= i1; c0 += BT) {
        const int i = c0 + tid;
        if (i <= i1) {
            const double m = bm.m[((int)p.species[i] - 1) & 15];
            double r[3];
            for (int k = 0; k < 3; ++k) r[k] = (p.pos[k * n + i] + p.image[k * n + i] * edges[k]) - com[k];
            for (int k = 0; k < 3; ++k) b->pos_body[3 * (i - i0) + k] = r[k];
            const double r2 = (r[0] * r[0] + r[1] * r[1]) + r[2] * r[2];
            for (int k = 0; k < 3; ++k) t[k][tid] = m * (r2 - r[k] * r[k]);
        }
        __syncthreads();
        if (tid == 0) {
            const int m = i1 - c0 + 1 < BT ? i1 - c0 + 1 : BT;
            for (int j = 0; j < m; ++j)
                for (int k = 0; k < 3; ++k) acc[k] = acc[k] + t[k][j];
        }
        __syncthreads();
    }
    if (tid == 0) {
        b->mass = mass;
        for (int k = 0; k < 3; ++k) {
            b->pos[k] = com[k];
            b->vel[k] = cv[k];
            b->I_body[k] = acc[k];
            b->force[k] = 0;
            b->torque[k] = 0;
            b->L[k] = 0;
            b->omega_body[k] = 0;
        }
        b->q[0] = 1;
        b->q[1] = b->q[2] = b->q[3] = 0;
    }
}

// rigid_body_compute_force_torque (md.f90:591-607)
__global__ void __launch_bounds__(BT) k_rigid_force_torque(rmpcd_rigid_body_t *b, PView<F64> p)
{
    __shared__ double t[6][BT];
    __shared__ double acc[6];
    const int64_t n = p.n;
    const int tid = threadIdx.x;
    if (!body_range_ok(b, n)) return;
    const int i0 = b->i_start, i1 = b->i_stop;
    const double q[4] = {b->q[0], b->q[1], b->q[2], b->q[3]};
    if (tid == 0)
        for (int k = 0; k < 6; ++k) acc[k] = 0;
    for (int c0 = i0; c0 <= i1; c0 += BT) {
        const int i = c0 + tid;
        if (i <= i1) {
            const double f[3] = {p.force[i], p.force[n + i], p.force[2 * n + i]};
            double r[3], c[3];
            qrot(q, b->pos_body + 3 * (i - i0), r);
            cross3(r, f, c);
            for (int k = 0; k < 3; ++k) {
                t[k][tid] = f[k];
                t[3 + k][tid] = c[k];
            }
        }
        __syncthreads();
        if (tid == 0) {
            const int m = i1 - c0 + 1 < BT ? i1 - c0 + 1 : BT;
            for (int j = 0; j < m; ++j)
                for (int k = 0; k < 6; ++k) acc[k] = acc[k] + t[k][j];
        }
        __syncthreads();
    }
    if (tid == 0)
        for (int k = 0; k < 3; ++k) {
            b->force[k] = acc[k];
            b->torque[k] = acc[3 + k];
        }
}

// rigid_body_vv1 (md.f90:613-673): thread 0 advances the orientation (the half-step
// quaternion iterated to the threshold, at most 1000 rounds) and the centre of mass; the
// particles are then placed in parallel
__global__ void __launch_bounds__(BT) k_rigid_vv1(rmpcd_rigid_body_t *b, PView<F64> p, double dt, double threshold,
                                                  double e0, double e1, double e2, int32_t *__restrict__ out)
{
    __shared__ double sq[8];
    const int64_t n = p.n;
    const int tid = threadIdx.x;
    const double edges[3] = {e0, e1, e2};
    if (!body_range_ok(b, n)) {
        if (tid == 0) out[0] = -1;
        return;
    }
    if (tid == 0) {
        double I_inv[3], q[4], qc[4], L[3], Lb[3], tb[3], ob[3], Lbd[3], c[3], qd[4], w[4];
        for (int k = 0; k < 3; ++k) I_inv[k] = 1 / b->I_body[k];
        for (int k = 0; k < 4; ++k) q[k] = b->q[k];
        for (int k = 0; k < 3; ++k) L[k] = b->L[k];
        qconj(q, qc);
        qrot(qc, L, Lb);
        qrot(qc, b->torque, tb);
        for (int k = 0; k < 3; ++k) ob[k] = Lb[k] * I_inv[k];
        cross3(ob, Lb, c);
        for (int k = 0; k < 3; ++k) Lbd[k] = tb[k] - c[k];
        for (int k = 0; k < 3; ++k) Lb[k] = Lb[k] + (dt * Lbd[k]) / 2;
        for (int k = 0; k < 3; ++k) ob[k] = Lb[k] * I_inv[k];
        w[0] = 0;
        for (int k = 0; k < 3; ++k) w[k + 1] = ob[k];
        qmul(q, w, qd);
        for (int k = 0; k < 4; ++k) qd[k] = qd[k] / 2;
        for (int k = 0; k < 4; ++k) q[k] = q[k] + (qd[k] * dt) / 2;
        qnormalize(q);
        for (int k = 0; k < 3; ++k) L[k] = b->L[k] + (b->torque[k] * dt) / 2;
        double q_old[4] = {q[0], q[1], q[2], q[3]};
        int it;
        for (it = 1; it <= RATTLE_MAX; ++it) {
            qconj(q, qc);
            qrot(qc, L, Lb);
            for (int k = 0; k < 3; ++k) w[k + 1] = I_inv[k] * Lb[k];
            qmul(q, w, qd);
            for (int k = 0; k < 4; ++k) qd[k] = qd[k] / 2;
            for (int k = 0; k < 4; ++k) q[k] = b->q[k] + (qd[k] * dt) / 2;
            qnormalize(q);
            double dq[4];
            for (int k = 0; k < 4; ++k) dq[k] = q[k] - q_old[k];
            if (qnorm(dq) < threshold) break;
            for (int k = 0; k < 4; ++k) q_old[k] = q[k];
        }
        double qn[4];
        for (int k = 0; k < 4; ++k) qn[k] = b->q[k] + dt * qd[k];
        qnormalize(qn);
        for (int k = 0; k < 4; ++k) b->q[k] = sq[k] = qn[k];
        for (int k = 0; k < 3; ++k) {
            const double x = (b->pos[k] + b->vel[k] * dt) + (b->force[k] * (dt * dt)) / (2 * b->mass);
            b->pos[k] = sq[4 + k] = x;
        }
        out[0] = it;
    }
    __syncthreads();
    const double q[4] = {sq[0], sq[1], sq[2], sq[3]};
    const double com[3] = {sq[4], sq[5], sq[6]};
    const int i0 = b->i_start, i1 = b->i_stop;
    for (int i = i0 + tid; i <= i1; i += BT) {
        double r[3];
        qrot(q, b->pos_body + 3 * (i - i0), r);
        for (int k = 0; k < 3; ++k) {
            const double old = p.pos[k * n + i];
            const double x = com[k] + r[k];
            const double delta = (x - old) + edges[k] / 2;
            p.pos[k * n + i] = x - floor(delta / edges[k]) * edges[k];
        }
    }
    __syncthreads();
    if (tid == 0)
        for (int k = 0; k < 3; ++k) {
            b->L[k] = b->L[k] + (b->torque[k] * dt) / 2;
            b->vel[k] = b->vel[k] + (b->force[k] * dt) / (2 * b->mass);
        }
}

// rigid_body_vv2 (md.f90:679-700)
__global__ void __launch_bounds__(BT) k_rigid_vv2(rmpcd_rigid_body_t *b, PView<F64> p, double dt)
{
    __shared__ double s[10];
    const int64_t n = p.n;
    const int tid = threadIdx.x;
    if (!body_range_ok(b, n)) return;
    if (tid == 0) {
        double qc[4], Lb[3], om[3];
        for (int k = 0; k < 3; ++k) b->L[k] = b->L[k] + (b->torque[k] * dt) / 2;
        qconj(b->q, qc);
        qrot(qc, b->L, Lb);
        for (int k = 0; k < 3; ++k) b->omega_body[k] = Lb[k] / b->I_body[k];
        qrot(b->q, b->omega_body, om);
        for (int k = 0; k < 3; ++k) b->vel[k] = b->vel[k] + (b->force[k] * dt) / (2 * b->mass);
        for (int k = 0; k < 4; ++k) s[k] = b->q[k];
        for (int k = 0; k < 3; ++k) {
            s[4 + k] = om[k];
            s[7 + k] = b->vel[k];
        }
    }
    __syncthreads();
    const double q[4] = {s[0], s[1], s[2], s[3]};
    const double om[3] = {s[4], s[5], s[6]};
    const int i0 = b->i_start, i1 = b->i_stop;
    for (int i = i0 + tid; i <= i1; i += BT) {
        double r[3], c[3];
        qrot(q, b->pos_body + 3 * (i - i0), r);
        cross3(om, r, c);
        for (int k = 0; k < 3; ++k) p.vel[k * n + i] = s[7 + k] + c[k];
    }
}

static int body_mass(const double *mass, int32_t n_mass, BodyMass &m)
{
    if (!mass || n_mass < 1 || n_mass > 16) return set_error(RMPCD_ERR_ARG, "mass table must hold 1..16 species");
    for (int k = 0; k < 16; ++k) {
        m.m[k] = k < n_mass ? mass[k] : 0.0;
        m.inv[k] = k < n_mass ? 1 / mass[k] : 0.0;
    }
    return RMPCD_OK;
}

static int check_body(const rmpcd_particles_t *p, const int32_t *links, const double *dist, int32_t n_links,
                      const char *who, bool need_force)
{
    int rc = check_particles(p, who, need_force);
    if (rc) return rc;
    RMPCD_CHECK(p->form == RMPCD_FP64, "%s: colloids must use the FP64 form", who);
    RMPCD_CHECK(n_links >= 0 && (n_links == 0 || (links && dist)), "%s: bad link arguments", who);
    return RMPCD_OK;
}

// a synchronous int32 result from the device
static int fetch_i32(const int32_t *dev, int32_t *host_out)
{
    int32_t *h = (int32_t *)pinned(64);
    if (!h) return set_error(RMPCD_ERR_HIP, "host staging allocation failed");
    RMPCD_HIP(hipMemcpyAsync(h, dev, sizeof(int32_t), hipMemcpyDeviceToHost, stream()));
    RMPCD_HIP(hipStreamSynchronize(stream()));
    *host_out = h[0];
    return RMPCD_OK;
}

// which rattle runs: the one-wave one with the most sweeps per block whose snapshots fit in
// LDS and whose schedule is not too long, else the global one
static int pick_k(Schedule &s, bool with_pr, const BlockSched **blk, size_t *lds)
{
    *blk = nullptr;
    *lds = 0;
    if (s.n > WAVE_N || s.n_links >= (1 << 24) || s.n_links == 0) return RMPCD_OK;
    for (int K = KMAX; K >= 1; --K) {
        const size_t need = wave_lds_bytes(s.n, K, with_pr);
        if (need > (size_t)lds_limit()) continue;
        int rc = get_block(s, K, blk);
        if (rc) return rc;
        *lds = need;
        if (*blk) return RMPCD_OK;
    }
    return RMPCD_OK;
}

template <bool kPos>
static int rattle_body(rmpcd_particles_t *p, double *pos_rattle, const int32_t *links, const double *distances,
                       int32_t n_links, const double *mass, int32_t n_mass, double dt, const double edges[3],
                       double precision, int32_t *iterations, const char *who)
{
    int rc = check_body(p, links, distances, n_links, who, false);
    if (rc) return rc;
    RMPCD_CHECK(edges && (!kPos || pos_rattle), "%s: null argument", who);
    BodyMass bm;
    if ((rc = body_mass(mass, n_mass, bm))) return rc;
    const int64_t n = p->n;
    int32_t *out = (int32_t *)workspace(WS_FLAG, 64);
    RMPCD_CHECK(out != nullptr, "%s: workspace allocation failed", who);
    // no links: nothing to correct, the first sweep meets any positive precision, and
    // the positions still go through the reference's unfold and fold
    Schedule *s = nullptr;
    if (n_links > 0 && (rc = get_schedule(links, distances, n_links, n, who, &s))) return rc;
    const BlockSched *blk = nullptr;
    size_t lds = 0;
    if (s && (rc = pick_k(*s, kPos, &blk, &lds))) return rc;
    if (blk) {
        // images, the links' constants, the updates' multipliers of two blocks
        const size_t im_b = (3 * (size_t)n * 4 + 255) & ~(size_t)255, lc_b = ((size_t)n_links + 1) * LC * 8;
        const size_t n_ent = (size_t)blk->n_steps * 64, ahead = 64 * AHEAD;
        char *w = (char *)workspace(WS_AUX, im_b + lc_b + (kPos ? (2 * n_ent + ahead) * 8 : 0) + 256);
        RMPCD_CHECK(w != nullptr, "%s: workspace allocation failed", who);
        if (lds > 64 * 1024)
            RMPCD_HIP(hipFuncSetAttribute((const void *)k_rattle_wave<kPos>,
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        const WaveView wv{blk->d_ent, s->d_la, s->d_lb, s->d_dist, s->d_cstart, s->n_links, blk->n_steps, blk->K};
        k_rattle_wave<kPos><<<1, WT, lds, stream()>>>(view<F64>(p), pos_rattle, wv, bm, dt, edges[0], edges[1], edges[2],
                                                      precision, out, (int32_t *)w, (double *)(w + im_b),
                                                      (double *)(w + im_b + lc_b));
    } else {
        char *w = (char *)workspace(WS_AUX, (size_t)n * 8 + 3 * (size_t)n * 4 + 256);
        RMPCD_CHECK(w != nullptr, "%s: workspace allocation failed", who);
        SchedView sv{nullptr, nullptr, nullptr, nullptr, 0, 0};
        if (s) sv = SchedView{s->d_i1, s->d_i2, s->d_start, s->d_d, s->n_links, s->n_levels};
        k_rattle_global<kPos><<<1, BT, 0, stream()>>>(view<F64>(p), pos_rattle, sv, bm, dt, edges[0], edges[1],
                                                       edges[2], precision, out, (double *)w,
                                                       (int32_t *)(w + (size_t)n * 8));
    }
    RMPCD_LAUNCHED();
    if (iterations) return fetch_i32(out, iterations);
    return RMPCD_OK;
}

}  // namespace rmpcd

using namespace rmpcd;

extern "C" {

int rmpcd_rattle_body_pos(rmpcd_particles_t *p, double *pos_rattle, const int32_t *links, const double *distances,
                          int32_t n_links, const double *mass, int32_t n_mass, double dt, const double edges[3],
                          double precision, int32_t *iterations)
{
    return rattle_body<true>(p, pos_rattle, links, distances, n_links, mass, n_mass, dt, edges, precision, iterations,
                             "rattle_body_pos");
}

int rmpcd_rattle_body_vel(rmpcd_particles_t *p, const int32_t *links, const double *distances, int32_t n_links,
                          const double *mass, int32_t n_mass, double dt, const double edges[3], double precision,
                          int32_t *iterations)
{
    return rattle_body<false>(p, nullptr, links, distances, n_links, mass, n_mass, dt, edges, precision, iterations,
                              "rattle_body_vel");
}

int rmpcd_elastic_network(rmpcd_particles_t *p, const int32_t *links, const double *distances, int32_t n_links,
                          double k, const double edges[3], double *energy)
{
    const char *who = "elastic_network";
    int rc = check_body(p, links, distances, n_links, who, true);
    if (rc) return rc;
    RMPCD_CHECK(edges && energy, "%s: null argument", who);
    if (n_links == 0) {
        *energy = 0;
        return RMPCD_OK;
    }
    Schedule *s;
    if ((rc = get_schedule(links, distances, n_links, p->n, who, &s))) return rc;
    const size_t tbytes = (size_t)n_links * 32;  // a term and a force per link
    double *w = (double *)workspace(WS_AUX, tbytes + 256);
    double *h = (double *)pinned(64);
    RMPCD_CHECK(w && h, "%s: workspace allocation failed", who);
    double *out = w + 4 * (size_t)n_links;
    if (tbytes <= (size_t)lds_limit()) {
        if (tbytes > 64 * 1024)
            RMPCD_HIP(hipFuncSetAttribute((const void *)k_elastic_network<true>,
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)tbytes));
        k_elastic_network<true><<<1, BT, tbytes, stream()>>>(view<F64>(p), s->d_la, s->d_lb, s->d_dist, s->d_cstart,
                                                             s->d_csr, n_links, k, edges[0], edges[1], edges[2], w,
                                                             out);
    } else {
        k_elastic_network<false><<<1, BT, 0, stream()>>>(view<F64>(p), s->d_la, s->d_lb, s->d_dist, s->d_cstart,
                                                          s->d_csr, n_links, k, edges[0], edges[1], edges[2], w, out);
    }
    RMPCD_LAUNCHED();
    RMPCD_HIP(hipMemcpyAsync(h, out, sizeof(double), hipMemcpyDeviceToHost, stream()));
    RMPCD_HIP(hipStreamSynchronize(stream()));
    *energy = h[0];
    return RMPCD_OK;
}

int rmpcd_rigid_body_init(rmpcd_rigid_body_t *body, const rmpcd_particles_t *p, const double *mass, int32_t n_mass,
                          const double edges[3], int32_t i_start, int32_t i_stop, double *pos_body)
{
    int rc = check_particles(p, "rigid_body_init", false);
    if (rc) return rc;
    RMPCD_CHECK(p->form == RMPCD_FP64 && p->image, "rigid_body_init: colloids must use the FP64 form, with images");
    RMPCD_CHECK(body && edges && pos_body, "rigid_body_init: null argument");
    RMPCD_CHECK(i_start >= 0 && i_stop >= i_start && i_stop < p->n, "rigid_body_init: particle range out of bounds");
    BodyMass bm;
    if ((rc = body_mass(mass, n_mass, bm))) return rc;
    rmpcd_rigid_body_t h{};
    h.i_start = i_start;
    h.i_stop = i_stop;
    h.pos_body = pos_body;
    RMPCD_HIP(hipMemcpyAsync(body, &h, sizeof(h), hipMemcpyHostToDevice, stream()));
    k_rigid_init<<<1, BT, 0, stream()>>>(body, view<F64>(p), bm, edges[0], edges[1], edges[2]);
    RMPCD_LAUNCHED();
    RMPCD_HIP(hipStreamSynchronize(stream()));
    return RMPCD_OK;
}

int rmpcd_rigid_body_compute_force_torque(rmpcd_rigid_body_t *body, const rmpcd_particles_t *p)
{
    const char *who = "rigid_body_compute_force_torque";
    int rc = check_particles(p, who, true);
    if (rc) return rc;
    RMPCD_CHECK(p->form == RMPCD_FP64, "%s: colloids must use the FP64 form", who);
    RMPCD_CHECK(body != nullptr, "%s: null body", who);
    k_rigid_force_torque<<<1, BT, 0, stream()>>>(body, view<F64>(p));
    RMPCD_LAUNCHED();
    return RMPCD_OK;
}

int rmpcd_rigid_body_vv1(rmpcd_rigid_body_t *body, rmpcd_particles_t *p, double dt, double threshold,
                         const double edges[3], int32_t *iterations)
{
    const char *who = "rigid_body_vv1";
    int rc = check_particles(p, who, false);
    if (rc) return rc;
    RMPCD_CHECK(p->form == RMPCD_FP64, "%s: colloids must use the FP64 form", who);
    RMPCD_CHECK(body && edges, "%s: null argument", who);
    int32_t *out = (int32_t *)workspace(WS_FLAG, 64);
    RMPCD_CHECK(out != nullptr, "%s: workspace allocation failed", who);
    k_rigid_vv1<<<1, BT, 0, stream()>>>(body, view<F64>(p), dt, threshold, edges[0], edges[1], edges[2], out);
    RMPCD_LAUNCHED();
    if (!iterations) return RMPCD_OK;
    if ((rc = fetch_i32(out, iterations))) return rc;
    RMPCD_CHECK(*iterations >= 0, "%s: the body's particles are outside [0, n)", who);
    return RMPCD_OK;
}

int rmpcd_rigid_body_vv2(rmpcd_rigid_body_t *body, rmpcd_particles_t *p, double dt)
{
    const char *who = "rigid_body_vv2";
    int rc = check_particles(p, who, false);
    if (rc) return rc;
    RMPCD_CHECK(p->form == RMPCD_FP64, "%s: colloids must use the FP64 form", who);
    RMPCD_CHECK(body != nullptr, "%s: null body", who);
    k_rigid_vv2<<<1, BT, 0, stream()>>>(body, view<F64>(p), dt);
    RMPCD_LAUNCHED();
    return RMPCD_OK;
}

}  // extern "C"
