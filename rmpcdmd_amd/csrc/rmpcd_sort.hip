// rmpcd_sort.hip -- cell keys, cell counts, the cell_start scan and the stable
// counting sort of the solvent (src/cell_system.f90:86-129,
// src/particle_system.f90:304-355, src/md.f90:202-217 fused).
//
// Sort pipeline (all launches on the library stream).  The unit is a tile: 2^k cells with
// consecutive Hilbert keys, at most 1382 particles on average in FP32 and 460 in FP64.
//   k_tile_key    per particle: optional periodic wrap, cell key from the box's Hilbert
//                 table, and its place in its tile's list (an LDS hash counts the tiles of
//                 1024 consecutive particles, one global atomic per tile met there)
//   k_tile_scan   exclusive scan of the tile counts
//   k_tile_place  list[start of the tile + place] = particle
//   k_tile_gather one workgroup per tile: counts its cells (cell_count, cell_start), ranks
//                 each particle among its cell's by original index, and moves the planes
//                 through LDS, read in list order and written in slot order
//   k_tile_spill  ranks and moves the particles of the tiles that the LDS does not hold (in
//                 smaller sorts the first workgroups of k_tile_gather do)
// The order within a tile's list is not deterministic, the rank does not depend on it: the
// result equals the reference's single-thread order, where each cell keeps increasing
// original index.
#include <type_traits>

#include "rmpcd_internal.hpp"
#include "rmpcd_srdtile.hpp"

namespace rmpcd {

// cell key of a position given in the particle's precision
template <class R>
__device__ inline int key_of(const Box &b, const int32_t *lut, R x, R y, R z)
{
    int p0, p1, p2;
    cell_of<R>(b, x, y, z, p0, p1, p2);
    if ((unsigned)p0 < (unsigned)b.L[0] && (unsigned)p1 < (unsigned)b.L[1] &&
        (unsigned)p2 < (unsigned)b.L[2])
        return lut[p0 + b.L[0] * (p1 + b.L[1] * p2)];
    // outside the box (the reference keys it anyway, through the low bits of p)
    return compact_key(p0, p1, p2, b.M[0], b.M[1], b.M[2]);
}

template <class F>
__global__ void k_key_count(Box b, const int32_t *__restrict__ lut, PView<F> p,
                            int32_t *__restrict__ count)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= p.n) return;
    atomicAdd(&count[key_of<typename F::real>(b, lut, p.pos[i], p.pos[p.n + i], p.pos[2 * p.n + i])], 1);
}

__global__ void k_fill_i32(int32_t *a, int64_t n, int32_t v)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}

// ---- exclusive scan of int32 over n (n up to 2^30) ------------------------------
constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

// block-wide exclusive scan of one value per thread; returns the block total in *total
__device__ inline int block_exclusive_scan(int v, int *lds_waves, int *total)
{
    int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    int inc = wave_inclusive_scan(v);
    if (lane == 63) lds_waves[wid] = inc;
    __syncthreads();
    int off = 0, tot = 0;
    for (int w = 0; w < nw; ++w) {
        int t = lds_waves[w];
        if (w < wid) off += t;
        tot += t;
    }
    __syncthreads();
    *total = tot;
    return off + inc - v;
}

// phase 1: per tile exclusive scan (in place into out) and the tile's total
__global__ void __launch_bounds__(SCAN_THREADS)
    k_scan_tiles(const int32_t *__restrict__ in, int32_t *__restrict__ out, int64_t n,
                 int32_t *__restrict__ tile_sums)
{
    __shared__ int lds[SCAN_THREADS / 64];
    int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    int v[SCAN_ITEMS];
    int s = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        v[k] = (base + k < n) ? in[base + k] : 0;
        s += v[k];
    }
    int tot;
    int off = block_exclusive_scan(s, lds, &tot);
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        if (base + k < n) out[base + k] = off;
        off += v[k];
    }
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = tot;
}

// phase 2: one block scans the tile totals (any count, in chunks of blockDim)
__global__ void __launch_bounds__(1024) k_scan_top(int32_t *tile_sums, int64_t ntiles)
{
    __shared__ int lds[16];
    int carry = 0;
    for (int64_t c = 0; c < ntiles; c += blockDim.x) {
        int64_t i = c + threadIdx.x;
        int v = i < ntiles ? tile_sums[i] : 0;
        int tot;
        int ex = block_exclusive_scan(v, lds, &tot);
        if (i < ntiles) tile_sums[i] = ex + carry;
        carry += tot;
        __syncthreads();
    }
}

// phase 3: add each tile's offset
__global__ void __launch_bounds__(SCAN_THREADS)
    k_scan_add(int32_t *__restrict__ out, int64_t n, const int32_t *__restrict__ tile_sums)
{
    int64_t base = (int64_t)blockIdx.x * SCAN_TILE;
    int add = tile_sums[blockIdx.x];
    for (int k = threadIdx.x; k < SCAN_TILE; k += SCAN_THREADS)
        if (base + k < n) out[base + k] += add;
}

int exclusive_scan(const int32_t *in, int32_t *out, int64_t n)
{
    int64_t ntiles = (n + SCAN_TILE - 1) / SCAN_TILE;
    int32_t *sums = (int32_t *)workspace(WS_SCAN, sizeof(int32_t) * (ntiles + 1));
    if (!sums) return set_error(RMPCD_ERR_HIP, "scan: workspace allocation failed");
    hipStream_t s = stream();
    k_scan_tiles<<<(unsigned)ntiles, SCAN_THREADS, 0, s>>>(in, out, n, sums);
    RMPCD_LAUNCHED();
    k_scan_top<<<1, 1024, 0, s>>>(sums, ntiles);
    RMPCD_LAUNCHED();
    k_scan_add<<<(unsigned)ntiles, SCAN_THREADS, 0, s>>>(out, n, sums);
    RMPCD_LAUNCHED();
    return RMPCD_OK;
}

// ---- counting sort ---------------------------------------------------------------
constexpr int SORT_T = 256;
constexpr int KEY_ITEMS = 4, KEY_CHUNK = SORT_T * KEY_ITEMS;  // particles per workgroup of the key pass
constexpr int HASH_BITS = 11, HASH = 1 << HASH_BITS;          // LDS hash entries, 2 x KEY_CHUNK
// a thread's particles of a tile that is moved through LDS (three planes at a time): 1536
// particles in FP32; 512 in FP64, where 1536 leave three waves per SIMD (a step of 837,000
// particles 174 against 219 us; FP32 at 21 million 1.79 ms, 1.84 with 768 or 1024)
template <class F>
constexpr int TILE_ITEMS = sizeof(typename F::real) == 4 ? 6 : 2;
template <class F>
constexpr int TILE_MAX = SORT_T * TILE_ITEMS<F>;
// tiles in a run that one XCD takes.  An eighth of the tiles per XCD left half of them with
// the empty cells of a 60 x 31 x 45 box (its particles in no order: 528 us a step, 459 with
// runs of 16, 485 with 4, 64 or 256; 21 million particles in order: 1.38 ms, 1.35 ms with
// runs of 4 to 64).
constexpr int TILE_RUN = 16;
// Cells of a tile at most: TILE_CELLS, or TILE_THIN where the particles of twice as many still
// fit.  (1 particle a cell: a tile of 128 cells, half of them outside an L=100 box, gives a
// workgroup 60 particles, a sort of a million FP32 152 us; 84 like this; 102 without tiles.  The
// larger counts cost the move two of six workgroups per CU where a tile is full.)
constexpr int TILE_CELLS = 128, TILE_THIN = 1024;
// Particles on average in a tile inside the box up to which a thread takes two at most (a
// small box's tiles: 5120 FP32 particles 39.1 us a sort with room for six a thread, 35.8 like
// this).
constexpr int TILE_FEW = 200;
constexpr int SCAN1_TILES = 1 << 14;                          // tile counts that one workgroup scans
// The counts of up to SCAN1_TILES tiles are spread over 128 KiB, a cache line each up to 2048:
// particles in no order (the first sort of a run) meet a few thousand counts from
// everywhere, and atomics on one line wait for each other (a step's key pass on 4096
// tiles: 201 us side by side, 50 spread).
constexpr int COUNT_SPAN = 1 << 15;
static int count_stride(int nt)
{
    int s = 1;
    while (s < 16 && nt <= SCAN1_TILES && nt * 2 * s <= COUNT_SPAN) s *= 2;
    return s;
}

// Places in the tiles' lists for up to three quarters as many particles as the hash has
// entries: each particle takes a place among its tile's of this workgroup from the LDS hash, and one
// global atomic per tile met turns these into places in the tile's list, so a run of
// consecutive particles of one tile stays together there.  All threads call clear, a
// barrier, put per particle, a barrier, commit, a barrier; then place(at, in).
template <int BITS>
struct TileHash {
    int key[1 << BITS], cnt[1 << BITS];
    __device__ inline void clear()
    {
        for (int h = threadIdx.x; h < (1 << BITS); h += SORT_T) {
            key[h] = -1;
            cnt[h] = 0;
        }
    }
    __device__ inline void put(int t, int &at, int &in)
    {
        unsigned h = ((unsigned)t * 2654435769u) >> (32 - BITS);
        for (;;) {  // a quarter of the entries at least stays free
            int q = key[h];
            if (q == -1) q = atomicCAS(&key[h], -1, t);
            if (q == t || q == -1) break;
            h = (h + 1) & ((1 << BITS) - 1);
        }
        at = (int)h;
        in = atomicAdd(&cnt[h], 1);
    }
    __device__ inline void commit(int32_t *__restrict__ tile_count, int stride)
    {
        for (int h = threadIdx.x; h < (1 << BITS); h += SORT_T)
            if (cnt[h] > 0) cnt[h] = atomicAdd(&tile_count[(int64_t)key[h] * stride], cnt[h]);
    }
    __device__ inline int place(int at, int in) const { return cnt[at] + in; }
};

// cell key and place in the tile's list of every particle, a thread's positions loaded
// before anything is done with them.  21 million particles FP32: 0.15 ms, 0.77 ms with an
// atomic per particle on its cell.
template <class F>
__global__ void __launch_bounds__(SORT_T)
    k_tile_key(Box b, const int32_t *__restrict__ lut, PView<F> p, int wrap, int shift,
               int stride, int32_t *__restrict__ tile_count, int32_t *__restrict__ key, int32_t *__restrict__ slot)
{
    using R = typename F::real;
    __shared__ TileHash<HASH_BITS> hash;
    const int64_t base = (int64_t)blockIdx.x * KEY_CHUNK + threadIdx.x;
    R x[KEY_ITEMS][3];
#pragma unroll
    for (int u = 0; u < KEY_ITEMS; ++u) {
        const int64_t i = base + u * SORT_T;
        if (i < p.n)
            for (int k = 0; k < 3; ++k) x[u][k] = p.pos[k * p.n + i];
    }
    hash.clear();
    __syncthreads();
    int at[KEY_ITEMS], in[KEY_ITEMS];
#pragma unroll
    for (int u = 0; u < KEY_ITEMS; ++u) {
        const int64_t i = base + u * SORT_T;
        if (i >= p.n) continue;
        if (wrap) {
            for (int k = 0; k < 3; ++k) fold_pbc<R>(x[u][k], (R)b.edges[k]);
        }
        const int c = key_of<R>(b, lut, x[u][0], x[u][1], x[u][2]);
        key[i] = c;
        hash.put(c >> shift, at[u], in[u]);
    }
    __syncthreads();
    hash.commit(tile_count, stride);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < KEY_ITEMS; ++u) {
        const int64_t i = base + u * SORT_T;
        if (i < p.n) slot[i] = hash.place(at[u], in[u]);
    }
}

// A plain fluid's cycle up to its sort (setup_simple_fluid.f90:108-118): SRD on the cells
// of the last sort, n_md steps of mpcd_stream_periodic, then key and place in the tile's
// list under the next grid shift (b).  One workgroup takes 2^cshift cells, collides their
// velocities in LDS while the positions are on their way to registers, and goes on with the
// particles it holds; one with more particles than its LDS collides from memory, a thread
// per cell, and goes through them in pieces.  Bound by instructions (0.18 ms of them for 21
// million FP32 particles) and by their phases: 0.37 ms with eight workgroups per CU, 0.42
// with six, 0.56 with four.  The hash takes the place of the collision's LDS for that, the
// axes are drawn by the waves that do not add up the cells (one wave per workgroup
// colliding its cells alone: 0.61 ms), and a position inside the box is not divided by it.
// As separate collision, streaming and key passes: 0.55 ms.
template <class F>
constexpr int FLUID_ITEMS = sizeof(typename F::real) == 4 ? 3 : 2;
template <class F>
constexpr int FLUID_MAX = SORT_T * FLUID_ITEMS<F>;

template <class F>
__global__ void __launch_bounds__(SORT_T, 8)
    k_fluid_key(Box b, const int32_t *__restrict__ lut, PView<F> p, const int32_t *__restrict__ start,
                const int32_t *__restrict__ count, int cshift, uint64_t seed, uint64_t step, int n_md, double dt,
                int shift, int stride, int32_t *__restrict__ tile_count, int32_t *__restrict__ key,
                int32_t *__restrict__ slot)
{
    using R = typename F::real;
    constexpr int N = FLUID_ITEMS<F>, M = FLUID_MAX<F>;
    constexpr int BITS = 10;
    static_assert(M <= 3 << (BITS - 2), "the hash holds a workgroup's particles");
    // the hash is used after the collision, in its place
    __shared__ union U {
        TileHash<BITS> hash;
        SrdTile<R, typename F::small, M> srd;
        __device__ U() {}
    } sh;
    __shared__ R v[3][M];
    const int tid = threadIdx.x;
    const int c0 = (int)blockIdx.x << cshift, ncell = 1 << cshift;
    const int64_t s = start[c0];
    const int m = (int)(start[c0 + ncell - 1] + count[c0 + ncell - 1] - s);
    if (m == 0) return;
    R x[N][3];
    auto load = [&](int base) {
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const int q = base + tid + u * SORT_T;
            if (q < m)
                for (int k = 0; k < 3; ++k) x[u][k] = p.pos[k * p.n + s + q];
        }
    };
    const R rdt = (R)dt;
    // the particles from base on that the registers hold, their velocities from vel(k, q)
    auto piece = [&](int base, bool write_vel, auto vel) {
        sh.hash.clear();
        __syncthreads();
        int at[N], in[N];
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const int q = base + tid + u * SORT_T;
            if (q >= m) continue;
            const int64_t i = s + q;
            for (int k = 0; k < 3; ++k) {
                const R w = vel(k, q);
                int jump = 0;
                for (int j = 0; j < n_md; ++j) {
                    x[u][k] = x[u][k] + w * rdt;
                    jump += fold_pbc<R>(x[u][k], (R)b.edges[k]);
                }
                if (write_vel) p.vel[k * p.n + i] = w;
                p.pos[k * p.n + i] = x[u][k];
                if (jump != 0) p.image[k * p.n + i] += jump;
            }
            const int c = key_of<R>(b, lut, x[u][0], x[u][1], x[u][2]);
            key[i] = c;
            sh.hash.put(c >> shift, at[u], in[u]);
        }
        __syncthreads();
        sh.hash.commit(tile_count, stride);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const int q = base + tid + u * SORT_T;
            if (q < m) slot[s + q] = sh.hash.place(at[u], in[u]);
        }
    };
    // the LDS and memory in separate calls, so each is addressed directly
    if (m <= M) {
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const int q = tid + u * SORT_T;
            if (q < m) {
                for (int k = 0; k < 3; ++k) v[k][q] = p.vel[k * p.n + s + q];
                sh.srd.sp[q] = p.species[s + q];
            }
        }
        load(0);
        __syncthreads();
        srd_tile(sh.srd, v, s, m, c0, ncell, start, count, seed, step, 1.0, 0.0);
        piece(0, true, [&](int k, int q) { return v[k][q]; });
        return;
    }
    for (int c = tid; c < ncell; c += SORT_T) {
        const int n = count[c0 + c];
        if (n <= 1) continue;
        const int64_t a = start[c0 + c];
        srd_cell(p.vel + a, p.vel + p.n + a, p.vel + 2 * p.n + a, p.species + a, n, c0 + c, b.ncells,
                 (const double *)nullptr, seed, step, 1.0, 0.0);
    }
    __threadfence_block();
    __syncthreads();
    for (int base = 0; base < m; base += M) {
        load(base);
        piece(base, false, [&](int k, int q) { return p.vel[k * p.n + s + q]; });
        __syncthreads();
    }
}

// start[t] for t in [0, nt], start[nt] = the particle count, from the counts that lie
// stride apart; the counts are left zero, as the next sort needs them.  The counts are read
// and the starts written in order, with the runs that the threads add up in LDS between
// (bit-mixed against bank conflicts): 7 us for 8192 tiles, 10 for 16,384; each thread
// reading its own run from memory took 20 and 24.
__global__ void __launch_bounds__(1024)
    k_tile_scan(int32_t *__restrict__ count, int stride, int nt, int32_t *__restrict__ start)
{
    __shared__ int v[SCAN1_TILES];
    __shared__ int lds[16];
    const int tid = threadIdx.x;
    auto at = [](int i) { return i ^ ((i >> 5) & 31); };
    for (int i = tid; i < nt; i += 1024) {
        v[at(i)] = count[i * stride];
        count[i * stride] = 0;
    }
    __syncthreads();
    const int per = (nt + 1023) >> 10, lo = min(per * tid, nt), hi = min(lo + per, nt);
    int s = 0;
    for (int i = lo; i < hi; ++i) s += v[at(i)];
    int tot;
    int off = block_exclusive_scan(s, lds, &tot);
    for (int i = lo; i < hi; ++i) {
        const int c = v[at(i)];
        v[at(i)] = off;
        off += c;
    }
    __syncthreads();
    for (int i = tid; i < nt; i += 1024) start[i] = v[at(i)];
    if (tid == 0) start[nt] = tot;
}

// Pieces of the tiles that hold more particles than the LDS: how many, and each one's tile
// and number in it.
struct SpillWork {
    int32_t *count;
    int2 *item;
};
// Who moves such a tile's particles.  Its own workgroup any number of them (ALONE), or up to
// HELP_OWN and above that the first HELPERS workgroups of the launch (HELPED), or up to SPILL_OWN
// and above that the launch of k_tile_spill that follows (SPREAD): clustered particles fill
// few tiles, and would leave the rest of the device idle.  The helpers wait for nobody, so each
// counts and groups the cells that it moves from the tile's whole list; k_tile_spill finds
// them grouped, but its launch takes 2 us, mostly for nothing.  It follows sorts of SPREAD_FROM
// particles or more (200 us a step and above).  The device-resident programs, whose particles
// spread evenly from the start, go alone.
enum Spill { ALONE, HELPED, SPREAD };
constexpr int64_t SPREAD_FROM = 1 << 20;
constexpr int SPILL_PIECE = 512, SPILL_AHEAD = 8, SPILL_OWN = 1024;
constexpr unsigned SPILL_BLOCKS = 1024;  // 2048 idle 1 us longer
// The helpers' units are of about SPILL_PIECE particles.  327,680 particles in an eighth, a 64th
// and a 512th of the box (in order): FP64 0.08, 0.17 and 3.3 ms a sort, FP32 0.07, 0.24 and 3.7;
// by the tiles' own workgroups 0.10, 1.7, 85 and 0.17, 2.9, 138; without tiles FP64 0.14, 0.56 and
// 3.2.  (256 and 512 helpers: 0.34 and 0.25 for the FP64 64th.)  Where no tile overflows they cost
// nothing that shows with 5120 to 327,680 particles (21 to 88 us a sort), and 1 us of the 154 of
// a step of 837,000 FP64 particles.  A flag from the scan or the place pass instead of
// their own look at the starts, and helpers that have moved a tile first, were not faster.
constexpr int HELPERS = 1024, HELP_OWN = 2048, HELP_CELL = 2048;
// A cell of a tile of m particles that all units share: each unit of 512 then looks through all of
// the tile instead of the cell, but one workgroup is not left with the whole cell (64 cells
// of 5000 FP64 particles 2.7 ms a sort, shared 0.24).
__device__ inline bool help_shared(int count, int m)
{
    return count > HELP_CELL && (int64_t)count * count > (int64_t)1024 * m;
}

// a thread's next particles of such a tile and their cells, -1 beyond its m particles
__device__ inline void spill_load(int32_t w[SPILL_AHEAD], int k[SPILL_AHEAD], const int32_t *__restrict__ list,
                                  const int32_t *__restrict__ key, int cmask, int64_t q0, int m)
{
#pragma unroll
    for (int u = 0; u < SPILL_AHEAD; ++u) w[u] = q0 + u * SORT_T < m ? list[q0 + u * SORT_T] : -1;
#pragma unroll
    for (int u = 0; u < SPILL_AHEAD; ++u) k[u] = w[u] >= 0 ? key[w[u]] & cmask : 0;
}

__global__ void k_tile_place(int64_t n, const int32_t *__restrict__ key, int shift,
                             const int32_t *__restrict__ slot, const int32_t *__restrict__ start,
                             int32_t *__restrict__ list, SpillWork work)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (i == 0) *work.count = 0;
    list[start[key[i] >> shift] + slot[i]] = (int32_t)i;
}

// one plane of a tile's particles: the loads of a thread's N particles, their way to the
// slots in LDS, and the slots' way out
template <int N, class T>
__device__ inline void tile_load(T r[N], const T *__restrict__ plane, const int32_t v[N])
{
#pragma unroll
    for (int u = 0; u < N; ++u)
        if (v[u] >= 0) r[u] = plane[v[u]];
}
template <int N, class T>
__device__ inline void tile_put(T *lds, const T r[N], const int32_t v[N], const int d[N])
{
#pragma unroll
    for (int u = 0; u < N; ++u)
        if (v[u] >= 0) lds[d[u]] = r[u];
}
template <int N, class T>
__device__ inline void tile_store(T *__restrict__ plane, const T *lds, int m)
{
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const int q = (int)threadIdx.x + u * SORT_T;
        if (q < m) plane[q] = lds[q];
    }
}

// particle w of src to slot o of dst
template <class F, bool FORCES>
__device__ inline void spill_move(const Box &b, const PView<F> &src, const PView<F> &dst, int wrap, int32_t w, int64_t o,
                                  int32_t *__restrict__ id_to_idx)
{
    using R = typename F::real;
    const int64_t n = src.n;
    for (int j = 0; j < 3; ++j) {
        R x = src.pos[j * n + w];
        int32_t im = src.image[j * n + w];
        if (wrap) im += fold_pbc<R>(x, (R)b.edges[j]);
        dst.pos[j * n + o] = x;
        dst.image[j * n + o] = im;
        dst.vel[j * n + o] = src.vel[j * n + w];
        if (FORCES) {
            dst.force[j * n + o] = src.force[j * n + w];
            dst.force_old[j * n + o] = src.force_old[j * n + w];
        }
    }
    const int32_t id = src.id[w];
    dst.id[o] = id;
    dst.species[o] = src.species[w];
    dst.flags[o] = src.flags[w];
    if (id_to_idx && (uint32_t)id < (uint32_t)n) id_to_idx[id] = (int32_t)o;
}

// Of a tile of m particles: the counts of its cells, added to lcnt, and their starts in the tile.
// All threads call, with a barrier before and after.
__device__ inline void spill_count(int *lcnt, const int32_t *list, const int32_t *key, int cmask, int m)
{
    for (int64_t q0 = threadIdx.x; q0 < m; q0 += SPILL_AHEAD * SORT_T) {
        int32_t w[SPILL_AHEAD];
        int k[SPILL_AHEAD];
        spill_load(w, k, list, key, cmask, q0, m);
#pragma unroll
        for (int u = 0; u < SPILL_AHEAD; ++u)
            if (w[u] >= 0) atomicAdd(&lcnt[k[u]], 1);
    }
}
__device__ inline void cell_starts(int *lstart, const int *lcnt, int ncell)
{
    if (threadIdx.x >= 64) return;  // one wave scans the tile's cells
    int carry = 0;
    for (int c0 = 0; c0 < ncell; c0 += 64) {
        const int k = c0 + (int)threadIdx.x, w = k < ncell ? lcnt[k] : 0;
        const int inc = wave_inclusive_scan(w);
        if (k < ncell) lstart[k] = carry + inc - w;
        carry += __shfl(inc, 63);
    }
}

// the list's particles of the cells [c0, c1] grouped by cell, to a stretch that starts with the
// tile; those cells' lcnt is zero before and their counts after
__device__ inline void spill_group(int32_t *grouped, int *lcnt, const int *lstart, const int32_t *list, const int32_t *key,
                                   int cmask, int m, int c0, int c1)
{
    for (int64_t q0 = threadIdx.x; q0 < m; q0 += SPILL_AHEAD * SORT_T) {
        int32_t w[SPILL_AHEAD];
        int k[SPILL_AHEAD];
        spill_load(w, k, list, key, cmask, q0, m);
#pragma unroll
        for (int u = 0; u < SPILL_AHEAD; ++u)
            if (w[u] >= 0 && k[u] >= c0 && k[u] <= c1) grouped[lstart[k[u]] + atomicAdd(&lcnt[k[u]], 1)] = w[u];
    }
}

// Particles [q0, q1) of a tile's list that is grouped by cell, at most P a thread: a thread ranks
// its own in their cells by original index, the cells' lists staged in LDS, and moves them
// straight between the planes, to slots from s on.  lcnt and lstart are the tile's cells in that
// list.  All threads call.
constexpr int SPILL_STAGE = 1536;
template <class F, bool FORCES, int P>
__device__ inline void spill_piece(const Box &b, const PView<F> &src, const PView<F> &dst, int wrap, int64_t s,
                                   const int32_t *key, int cmask, const int32_t *grouped, const int *lcnt,
                                   const int *lstart, int q0, int q1, int32_t *stage, int *range,
                                   int32_t *__restrict__ id_to_idx)
{
    const int tid = threadIdx.x;
    int32_t w[P];
    int a[P], z[P], rank[P];  // the particles' cells in the list
#pragma unroll
    for (int u = 0; u < P; ++u) {
        const int q = q0 + tid + u * SORT_T;
        w[u] = q < q1 ? grouped[q] : -1;
        const int c = w[u] >= 0 ? key[w[u]] & cmask : 0;
        a[u] = w[u] >= 0 ? lstart[c] : 0;
        z[u] = w[u] >= 0 ? a[u] + lcnt[c] : 0;
        rank[u] = 0;
        // the piece's first and last particle bound the cells that are needed
        if (q == q0) range[0] = a[u];
        if (q == q1 - 1) range[1] = z[u];
    }
    __syncthreads();
    const int r0 = range[0], r1 = range[1];
    for (int base = r0; base < r1; base += SPILL_STAGE) {
        const int m = r1 - base < SPILL_STAGE ? r1 - base : SPILL_STAGE;
        __syncthreads();
        for (int k = tid; k < m; k += SORT_T) stage[k] = grouped[base + k];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < P; ++u) {
            const int lo = a[u] > base ? a[u] - base : 0, hi = z[u] - base < m ? z[u] - base : m;
            int r = 0;
#pragma unroll 4
            for (int k = lo; k < hi; ++k) r += stage[k] < w[u] ? 1 : 0;
            rank[u] += r;
        }
    }
#pragma unroll
    for (int u = 0; u < P; ++u)
        if (w[u] >= 0) spill_move<F, FORCES>(b, src, dst, wrap, w[u], s + a[u] + rank[u], id_to_idx);
    __syncthreads();
}

// Particles [q0, q0 + SPILL_PIECE) of a tile's list, those in cells that all units share: ranked by
// cell and original index among all of the tile's.  All threads call.
template <class F>
__device__ inline void help_cells(const Box &b, const PView<F> &src, const PView<F> &dst, int wrap, int64_t s,
                                  const int32_t *key, int cmask, const int32_t *list, int m, const int *lcnt, int q0,
                                  uint64_t *stage, int32_t *__restrict__ id_to_idx)
{
    constexpr int P = SPILL_PIECE / SORT_T, STAGE = SPILL_STAGE / 2;
    const int tid = threadIdx.x;
    int32_t w[P];
    uint64_t o[P];
    int rank[P];
#pragma unroll
    for (int u = 0; u < P; ++u) {
        const int q = q0 + tid + u * SORT_T;
        w[u] = q < m ? list[q] : -1;
        const int c = w[u] >= 0 ? key[w[u]] & cmask : 0;
        if (!help_shared(lcnt[c], m)) w[u] = -1;
        o[u] = (uint64_t)c << 32 | (uint32_t)w[u];
        rank[u] = 0;
    }
    for (int base = 0; base < m; base += STAGE) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < STAGE / SORT_T; ++u) {
            const int q = base + tid + u * SORT_T;
            const int32_t x = q < m ? list[q] : -1;
            stage[tid + u * SORT_T] = x >= 0 ? (uint64_t)(key[x] & cmask) << 32 | (uint32_t)x : ~(uint64_t)0;
        }
        __syncthreads();
#pragma unroll 4
        for (int k = 0; k < STAGE; ++k) {
            const uint64_t y = stage[k];
#pragma unroll
            for (int u = 0; u < P; ++u) rank[u] += y < o[u] ? 1 : 0;
        }
    }
#pragma unroll
    for (int u = 0; u < P; ++u)
        if (w[u] >= 0) spill_move<F, true>(b, src, dst, wrap, w[u], s + rank[u], id_to_idx);
    __syncthreads();
}

// The tiles of more than HELP_OWN particles, their units to the HELPERS workgroups in turn.  A
// unit is the cells that begin in SPILL_PIECE consecutive places of the tile (that are not shared by
// all units), their list made in the unit's own stretch of `spill`.  `some` holds
// HELP_WORDS words: the particles of SORT_T tiles, which of them are large, flags and ranges.
constexpr int HELP_MASK = SORT_T, HELP_FLAG = HELP_MASK + SORT_T / 32, HELP_RANGE = HELP_FLAG + 2,
              HELP_WORDS = HELP_RANGE + 4;
template <class F>
__device__ inline void help(const Box &b, const PView<F> &src, const PView<F> &dst, int wrap, int shift, int nt,
                            const int32_t *key, const int32_t *start, const int32_t *list, int32_t *spill, int *lcnt,
                            int *lstart, void *stage, int *some, int32_t *__restrict__ id_to_idx)
{
    const int tid = threadIdx.x, ncell = 1 << shift, cmask = ncell - 1;
    int any = 0;
#pragma unroll 4
    for (int t = tid; t < nt; t += SORT_T) any |= start[t + 1] - start[t] > HELP_OWN;
    if (tid == 0) some[HELP_FLAG] = 0;
    __syncthreads();
    if (any) some[HELP_FLAG] = 1;
    __syncthreads();
    if (!some[HELP_FLAG]) return;
    int unit = blockIdx.x;  // the next one of this workgroup, counted from the tile at hand
    for (int t0 = 0; t0 < nt; t0 += SORT_T) {
        const int mine = t0 + tid < nt ? start[t0 + tid + 1] - start[t0 + tid] : 0;
        const uint64_t large = __ballot(mine > HELP_OWN);
        some[tid] = mine;
        if ((tid & 31) == 0) some[HELP_MASK + tid / 32] = (int)(large >> (tid & 32));
        __syncthreads();
        for (int word = 0; word < SORT_T / 32; ++word) {
            for (uint32_t left = (uint32_t)some[HELP_MASK + word]; left; left &= left - 1) {
                const int t = 32 * word + __ffs(left) - 1, m = some[t], units = (m - 1) / SPILL_PIECE + 1;
                if (unit >= units) {
                    unit -= units;
                    continue;
                }
                const int64_t s = start[t0 + t];
                for (int c = tid; c < ncell; c += SORT_T) lcnt[c] = 0;
                if (tid == 0) some[HELP_FLAG + 1] = 0;
                __syncthreads();
                spill_count(lcnt, list + s, key, cmask, m);
                __syncthreads();
                cell_starts(lstart, lcnt, ncell);
                for (int c = tid; c < ncell; c += SORT_T)
                    if (help_shared(lcnt[c], m)) some[HELP_FLAG + 1] = 1;
                __syncthreads();
                for (; unit < units; unit += HELPERS) {
                    int *range = some + HELP_RANGE;  // the unit's cells, first and last
                    __syncthreads();
                    if (tid == 0) range[0] = ncell, range[1] = -1;
                    __syncthreads();
                    for (int c = tid; c < ncell; c += SORT_T)
                        if (lstart[c] / SPILL_PIECE == unit && lcnt[c] > 0 && !help_shared(lcnt[c], m)) {
                            atomicMin(&range[0], c);
                            atomicMax(&range[1], c);
                        }
                    __syncthreads();
                    const int c0 = range[0], c1 = range[1];
                    if (c0 <= c1) {
                        const int q0 = lstart[c0], q1 = lstart[c1] + lcnt[c1];
                        __syncthreads();
                        for (int c = c0 + tid; c <= c1; c += SORT_T) lcnt[c] = 0;
                        __syncthreads();
                        spill_group(spill + s, lcnt, lstart, list + s, key, cmask, m, c0, c1);
                        __threadfence_block();
                        __syncthreads();
                        for (int q = q0; q < q1; q += SPILL_PIECE)
                            spill_piece<F, true, SPILL_PIECE / SORT_T>(
                                b, src, dst, wrap, s, key, cmask, spill + s, lcnt, lstart, q,
                                q + SPILL_PIECE < q1 ? q + SPILL_PIECE : q1, (int32_t *)stage, range + 2, id_to_idx);
                    }
                    if (some[HELP_FLAG + 1])
                        help_cells<F>(b, src, dst, wrap, s, key, cmask, list + s, m, lcnt, unit * SPILL_PIECE,
                                      (uint64_t *)stage, id_to_idx);
                }
                unit -= units;
                __syncthreads();
            }
        }
        __syncthreads();
    }
}

// The cell sort's move.  Bound by memory: FP32 it reads 74 B and writes 66 B per particle.
// For 21 million particles on a newly shifted grid it fetches 110 B (tiles read the edges of
// their neighbours' stretches) and writes 67 in 0.70 ms, 5.3 TB/s; on the grid of the last sort
// 78 and 67 B in 0.645 ms.  Moved one particle per thread
// straight from the planes, each load touched a cache line per lane and the pass took 2.08
// ms; in list order a tile's loads run along the source, and LDS puts them in slot order so
// that the stores are contiguous too.  id_to_idx costs 0.43 ms of the 1.13 ms with it: its
// 4-byte stores go anywhere once the particles have mixed, each fetching and writing a piece of
// a line (170 and 100 B a particle in all).  FORCES false leaves the force planes out, for a
// program whose forces are zero in both buffers (72 and 43 B, 0.43 ms).  With two particles a thread
// it is held to eight waves per SIMD, which its scalar registers would make seven (a step of
// 390,000 FP64 particles 95 us, 90 with eight).
template <class F, bool FORCES, int CELLS, int N, Spill MODE>
__global__ void __launch_bounds__(SORT_T, CELLS > TILE_CELLS ? 1 : N == 2 ? 8 : FORCES ? 6 : 1)
    k_tile_gather(Box b, PView<F> src, PView<F> dst, int wrap, int shift, int nt, const int32_t *__restrict__ key,
                  const int32_t *__restrict__ start, const int32_t *__restrict__ list, int32_t *__restrict__ spill,
                  int32_t *__restrict__ cell_count, int32_t *__restrict__ cell_start, SpillWork work,
                  int32_t *__restrict__ id_to_idx)
{
    using R = typename F::real;
    using S = typename F::small;
    constexpr int M = SORT_T * N, PLANES = FORCES ? 4 : 2;
    __shared__ alignas(8) R buf[3][M];
    __shared__ int lv[M];
    __shared__ int lcnt[CELLS], lstart[CELLS];
    constexpr int OWN = MODE == ALONE ? INT32_MAX : MODE == HELPED ? HELP_OWN : SPILL_OWN > M ? SPILL_OWN : M;
    static_assert(sizeof(buf) >= SPILL_STAGE * sizeof(int32_t) && M >= HELP_WORDS && M <= OWN, "the stages");
    if constexpr (MODE == HELPED)
        if (blockIdx.x < HELPERS) {
            help<F>(b, src, dst, wrap, shift, nt, key, start, list, spill, lcnt, lstart, buf, lv, id_to_idx);
            return;
        }
    // consecutive workgroups go to the XCDs in turn: each XCD takes runs of TILE_RUN tiles,
    // so that the tiles in flight there read neighbouring stretches.  The runs are short
    // enough that the empty cells of a padded box fall to all XCDs alike.
    const int block = (int)blockIdx.x - (MODE == HELPED ? HELPERS : 0), j = block >> 3;
    const int t = ((j / TILE_RUN) * 8 + (block & 7)) * TILE_RUN + j % TILE_RUN;
    if (t >= nt) return;
    const int tid = threadIdx.x;
    const int64_t n = src.n;
    const int64_t s = start[t];
    const int m = (int)(start[t + 1] - s);
    const int ncell = 1 << shift, cmask = ncell - 1;
    for (int c = tid; c < ncell; c += SORT_T) lcnt[c] = 0;
    __syncthreads();
    int v[N], c[N], d[N];
    R x[3][N];
    R *const from[4] = {src.pos, src.vel, src.force, src.force_old};
    R *const to[4] = {dst.pos, dst.vel, dst.force, dst.force_old};
    const bool fits = m <= M;
    if (fits) {
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const int q = tid + u * SORT_T;
            v[u] = q < m ? list[s + q] : -1;
        }
#pragma unroll
        for (int u = 0; u < N; ++u) c[u] = v[u] >= 0 ? key[v[u]] & cmask : 0;
        // the positions are on their way while the particles are ranked
        for (int k = 0; k < 3; ++k) tile_load<N>(x[k], src.pos + k * n, v);
#pragma unroll
        for (int u = 0; u < N; ++u) d[u] = v[u] >= 0 ? atomicAdd(&lcnt[c[u]], 1) : 0;
    } else {
        spill_count(lcnt, list + s, key, cmask, m);
    }
    __syncthreads();
    cell_starts(lstart, lcnt, ncell);
    __syncthreads();
    for (int k = tid; k < ncell; k += SORT_T) {
        cell_count[((int64_t)t << shift) + k] = lcnt[k];
        cell_start[((int64_t)t << shift) + k] = (int32_t)s + lstart[k];
    }
    if (fits) {
#pragma unroll
        for (int u = 0; u < N; ++u)
            if (v[u] >= 0) lv[lstart[c[u]] + d[u]] = v[u];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < N; ++u) {
            if (v[u] < 0) continue;
            const int a = lstart[c[u]], e = a + lcnt[c[u]];
            int rank = 0;
            for (int q = a; q < e; ++q) rank += lv[q] < v[u] ? 1 : 0;
            d[u] = a + rank;
        }
        // the planes, three at a time; the next three are loaded before these are written
        int32_t im[3][N];
        for (int k = 0; k < 3; ++k) tile_load<N>(im[k], src.image + k * n, v);
        if (wrap)
            for (int k = 0; k < 3; ++k)
                for (int u = 0; u < N; ++u)
                    if (v[u] >= 0) im[k][u] += fold_pbc<R>(x[k][u], (R)b.edges[k]);
#pragma unroll
        for (int g = 0; g < PLANES; ++g) {
            for (int k = 0; k < 3; ++k) tile_put<N>(buf[k], x[k], v, d);
            if (g + 1 < PLANES)
                for (int k = 0; k < 3; ++k) tile_load<N>(x[k], from[(g + 1) & 3] + k * n, v);
            __syncthreads();
            for (int k = 0; k < 3; ++k) tile_store<N>(to[g] + k * n + s, buf[k], m);
            __syncthreads();
        }
        int32_t id[N];
        S sp[N], fl[N];
        tile_load<N>(id, src.id, v);
        tile_load<N>(sp, src.species, v);
        tile_load<N>(fl, src.flags, v);
        int32_t *ib[3] = {(int32_t *)buf[0], (int32_t *)buf[1], (int32_t *)buf[2]};
        for (int k = 0; k < 3; ++k) tile_put<N>(ib[k], im[k], v, d);
        __syncthreads();
        for (int k = 0; k < 3; ++k) tile_store<N>(dst.image + k * n + s, ib[k], m);
        __syncthreads();
        S *sb = (S *)buf[1], *fb = (S *)buf[2];
        tile_put<N>(ib[0], id, v, d);
        tile_put<N>(sb, sp, v, d);
        tile_put<N>(fb, fl, v, d);
        if (id_to_idx)
            for (int u = 0; u < N; ++u)
                if (v[u] >= 0 && (uint32_t)id[u] < (uint32_t)n) id_to_idx[id[u]] = (int32_t)(s + d[u]);
        __syncthreads();
        tile_store<N>(dst.id + s, ib[0], m);
        tile_store<N>(dst.species + s, sb, m);
        tile_store<N>(dst.flags + s, fb, m);
        return;
    }
    // more particles than the LDS holds: the list grouped by cell goes to memory (each
    // workgroup writes and reads its own stretch), and each particle is ranked and moved from
    // there, by the helpers, or by k_tile_spill
    if (MODE == HELPED && m > OWN) return;
    for (int k = tid; k < ncell; k += SORT_T) lcnt[k] = 0;
    __syncthreads();
    spill_group(spill + s, lcnt, lstart, list + s, key, cmask, m, 0, ncell - 1);
    if (MODE == SPREAD && m > OWN) {
        const int pieces = (m - 1) / SPILL_PIECE + 1;
        if (tid == 0) lv[0] = atomicAdd(work.count, pieces);
        __syncthreads();
        for (int k = tid; k < pieces; k += SORT_T) work.item[lv[0] + k] = make_int2(t, k);
        return;
    }
    __threadfence_block();
    __syncthreads();
    if constexpr (FORCES) {
        for (int q = 0; q < m; q += SORT_T)
            spill_piece<F, true, 1>(b, src, dst, wrap, s, key, cmask, spill + s, lcnt, lstart, q,
                                    q + SORT_T < m ? q + SORT_T : m, (int32_t *)buf, lv, id_to_idx);
    } else {
        // an even fluid's tile overflows where one cell does; what is above costs its usual
        // way registers (21 million FP32 particles 953 us a cycle, 941 like this)
        for (int q = tid; q < m; q += SORT_T) {
            const int32_t w = spill[s + q];
            const int k = key[w] & cmask;
            const int a = lstart[k], e = a + lcnt[k];
            int rank = 0;
            for (int y = a; y < e; ++y) rank += spill[s + y] < w ? 1 : 0;
            spill_move<F, false>(b, src, dst, wrap, w, s + a + rank, id_to_idx);
        }
    }
}

// The tiles too large for their own workgroup, a piece of one per workgroup at a time: a sort
// with all particles in a half, an eighth, a 64th and a 512th of an L=64 box (2.6 million FP32, in
// order) takes 0.29, 0.30, 0.66 and 3.6 ms; without tiles 0.42, 0.68, 1.7 and 9.7; by helpers 0.27, 0.72,
// 3.2 and 15.  In no order 1.13, 1.12, 1.43 and 3.6 ms; without tiles 1.11, 1.10, 1.29 and 4.2.
template <class F>
__global__ void __launch_bounds__(SORT_T)
    k_tile_spill(Box b, PView<F> src, PView<F> dst, int wrap, int shift, const int32_t *__restrict__ key,
                 const int32_t *__restrict__ start, const int32_t *__restrict__ spill,
                 const int32_t *__restrict__ cell_count, const int32_t *__restrict__ cell_start, SpillWork work,
                 int32_t *__restrict__ id_to_idx)
{
    __shared__ int32_t stage[SPILL_STAGE];
    __shared__ int range[2];
    const int items = *work.count;
    for (int it = blockIdx.x; it < items; it += gridDim.x) {
        const int2 e = work.item[it];
        const int q0 = start[e.x] + e.y * SPILL_PIECE, end = start[e.x + 1];
        const int64_t c = (int64_t)e.x << shift;  // (the lists' starts are the box's)
        spill_piece<F, true, SPILL_PIECE / SORT_T>(b, src, dst, wrap, 0, key, (1 << shift) - 1, spill, cell_count + c,
                                                   cell_start + c, q0, end - q0 > SPILL_PIECE ? q0 + SPILL_PIECE : end,
                                                   stage, range, id_to_idx);
    }
}

template <class F>
int count_impl(const rmpcd_box_t *box, const rmpcd_particles_t *pp, rmpcd_cells_t *cells)
{
    Box b = make_box(box);
    PView<F> p = view<F>(pp);
    const int32_t *lut = hilbert_lut(b);
    if (!lut) return set_error(RMPCD_ERR_HIP, "count: Hilbert table allocation failed");
    hipStream_t s = stream();
    k_fill_i32<<<blocks_for(b.ncells, 256), 256, 0, s>>>(cells->cell_count, b.ncells, 0);
    RMPCD_LAUNCHED();
    k_key_count<F><<<blocks_for(p.n, 256), 256, 0, s>>>(b, lut, p, cells->cell_count);
    RMPCD_LAUNCHED();
    return exclusive_scan(cells->cell_count, cells->cell_start, b.ncells);
}

// cells per tile (a power of two): the most whose particles, at the mean density of the
// cells inside the box, fill at most 0.9 of the LDS (in FP32 a tile above that by chance still
// fits: three standard deviations of 1382 particles are 112, and 154 are spare; in FP64 52 are
// spare, 2.4 standard deviations of 460, and a tile above that is moved from memory), and small
// enough that a box has two workgroups for every compute unit (a floor of 1024 or 2048 tiles made
// no difference)
static int tile_shift(const Box &b, int64_t n, int tile_max, int tile_cells)
{
    const double per_cell = (double)n / ((double)b.L[0] * b.L[1] * b.L[2]);
    int shift = 0;
    while ((2 << shift) <= tile_cells && (2 << shift) <= b.ncells && per_cell * (2 << shift) <= tile_max * 0.9 &&
           (b.ncells >> (shift + 1)) >= 512)
        ++shift;
    return shift;
}

// a sort's workspace and tiles
struct TileSort {
    Box b;
    const int32_t *lut;
    int shift, nt, stride;
    double per_tile;  // particles, in tiles inside the box
    int32_t *key, *slot, *list, *start, *count;
    SpillWork work;
};

template <class F>
static int tile_sort_begin(const rmpcd_box_t *box, int64_t n, TileSort &t)
{
    t.b = make_box(box);
    t.shift = tile_shift(t.b, n, TILE_MAX<F>, TILE_THIN);
    t.nt = t.b.ncells >> t.shift;
    t.per_tile = (double)n / ((double)t.b.L[0] * t.b.L[1] * t.b.L[2]) * (1 << t.shift);
    t.stride = count_stride(t.nt);
    t.key = (int32_t *)workspace(WS_KEY, sizeof(int32_t) * n);
    t.slot = (int32_t *)workspace(WS_SLOT, sizeof(int32_t) * n);
    t.list = (int32_t *)workspace(WS_TMP, sizeof(int32_t) * n);
    // the tiles' starts, the spill pieces' number, the pieces: one per SPILL_PIECE particles, and
    // a last, shorter one per tile that overflows
    const size_t words = ((size_t)t.nt + 2 + 1) & ~(size_t)1;
    const size_t most = (size_t)(n / SPILL_PIECE + n / SPILL_OWN + 1);
    t.start = (int32_t *)workspace(WS_TILE, sizeof(int32_t) * words + sizeof(int2) * most);
    if (t.start) t.work = {t.start + t.nt + 1, (int2 *)(t.start + words)};
    t.count = (int32_t *)workspace(WS_TCOUNT, sizeof(int32_t) * ((size_t)t.nt + 1) * t.stride);  // zero between sorts
    if (!t.key || !t.slot || !t.list || !t.start || !t.count)
        return set_error(RMPCD_ERR_HIP, "rmpcd_sort: workspace allocation failed");
    t.lut = hilbert_lut(t.b);
    if (!t.lut) return set_error(RMPCD_ERR_HIP, "rmpcd_sort: Hilbert table allocation failed");
    return zeroed_open(WS_TCOUNT);  // the keys' kernel comes next
}

// the sort after its keys
template <class F, bool FORCES>
static int tile_sort_finish(const TileSort &t, const rmpcd_particles_t *src, rmpcd_particles_t *dst,
                            int32_t *id_to_idx, rmpcd_cells_t *cells, int wrap, bool even)
{
    const int64_t n = src->n;
    hipStream_t s = stream();
    const Spill mode = even ? ALONE : n >= SPREAD_FROM || t.nt > SCAN1_TILES ? SPREAD : HELPED;
    if (t.nt <= SCAN1_TILES) {
        k_tile_scan<<<1, 1024, 0, s>>>(t.count, t.stride, t.nt, t.start);
        RMPCD_LAUNCHED();
    } else {
        int rc = exclusive_scan(t.count, t.start, (int64_t)t.nt + 1);
        if (rc) return rc;
        k_fill_i32<<<blocks_for(t.nt, 256), 256, 0, s>>>(t.count, t.nt, 0);
        RMPCD_LAUNCHED();
    }
    zeroed_close(WS_TCOUNT);
    k_tile_place<<<blocks_for(n, 256), 256, 0, s>>>(n, t.key, t.shift, t.slot, t.start, t.list, t.work);
    RMPCD_LAUNCHED();
    const unsigned runs = (unsigned)((t.nt + 8 * TILE_RUN - 1) / (8 * TILE_RUN));
    auto move = [&](auto cells_max, auto items, auto spill) {
        constexpr Spill MODE = decltype(spill)::value;
        k_tile_gather<F, FORCES, decltype(cells_max)::value, decltype(items)::value, MODE>
            <<<(MODE == HELPED ? HELPERS : 0) + 8 * TILE_RUN * runs, SORT_T, 0, s>>>(
                t.b, view<F>(src), view<F>(dst), wrap, t.shift, t.nt, t.key, t.start, t.list, t.slot, cells->cell_count,
                cells->cell_start, t.work, id_to_idx);
    };
    auto tiles = [&](auto spill) {
        const std::integral_constant<int, TILE_ITEMS<F>> items{};
        const std::integral_constant<int, TILE_CELLS> some{};
        if ((1 << t.shift) > TILE_CELLS)
            move(std::integral_constant<int, TILE_THIN>{}, items, spill);
        else if (t.per_tile <= TILE_FEW)
            move(some, std::integral_constant<int, 2>{}, spill);
        else
            move(some, items, spill);
    };
    if (mode == ALONE) tiles(std::integral_constant<Spill, ALONE>{});
    if constexpr (FORCES) {  // the others are the programs'
        if (mode == HELPED) tiles(std::integral_constant<Spill, HELPED>{});
        if (mode == SPREAD) tiles(std::integral_constant<Spill, SPREAD>{});
    }
    RMPCD_LAUNCHED();
    if constexpr (FORCES) {
        if (mode != SPREAD) return RMPCD_OK;
        const unsigned pieces = blocks_for(n, SPILL_PIECE);
        k_tile_spill<F><<<pieces < SPILL_BLOCKS ? pieces : SPILL_BLOCKS, SORT_T, 0, s>>>(
            t.b, view<F>(src), view<F>(dst), wrap, t.shift, t.key, t.start, t.slot, cells->cell_count, cells->cell_start,
            t.work, id_to_idx);
        RMPCD_LAUNCHED();
    }
    return RMPCD_OK;
}

template <class F>
int sort_impl(const rmpcd_box_t *box, const rmpcd_particles_t *src, rmpcd_particles_t *dst,
              int32_t *id_to_idx, rmpcd_cells_t *cells, int wrap, bool even)
{
    TileSort t;
    int rc = tile_sort_begin<F>(box, src->n, t);
    if (rc) return rc;
    k_tile_key<F><<<blocks_for(src->n, KEY_CHUNK), SORT_T, 0, stream()>>>(t.b, t.lut, view<F>(src), wrap, t.shift,
                                                                          t.stride, t.count, t.key, t.slot);
    RMPCD_LAUNCHED();
    return tile_sort_finish<F, true>(t, src, dst, id_to_idx, cells, wrap, even);
}

template <class F>
int fluid_cycle_impl(const rmpcd_box_t *next, const rmpcd_particles_t *src, rmpcd_particles_t *dst,
                     rmpcd_cells_t *cells, uint64_t seed, uint64_t step, int n_md, double dt)
{
    TileSort t;
    int rc = tile_sort_begin<F>(next, src->n, t);
    if (rc) return rc;
    // the collision's cells per workgroup, by the same rule as a tile's
    int cshift = tile_shift(t.b, src->n, FLUID_MAX<F>, SRD_CELLS);
    k_fluid_key<F><<<(unsigned)(t.b.ncells >> cshift), SORT_T, 0, stream()>>>(
        t.b, t.lut, view<F>(src), cells->cell_start, cells->cell_count, cshift, seed, step, n_md, dt, t.shift, t.stride,
        t.count, t.key, t.slot);
    RMPCD_LAUNCHED();
    return tile_sort_finish<F, false>(t, src, dst, nullptr, cells, 0, true);
}

int fluid_cycle_unchecked(const rmpcd_box_t *next, const rmpcd_particles_t *src, rmpcd_particles_t *dst,
                          rmpcd_cells_t *cells, uint64_t seed, uint64_t step, int n_md, double dt)
{
    return RMPCD_DISPATCH_FORM(src, fluid_cycle_impl, next, src, dst, cells, seed, step, n_md, dt);
}

int sort_unchecked(const rmpcd_box_t *box, const rmpcd_particles_t *src, rmpcd_particles_t *dst, int32_t *id_to_idx,
                   rmpcd_cells_t *cells, int wrap, bool even)
{
    return RMPCD_DISPATCH_FORM(src, sort_impl, box, src, dst, id_to_idx, cells, wrap, even);
}

template <class F>
__global__ void k_cartesian(Box b, PView<F> p, int32_t *out)
{
    using R = typename F::real;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= p.n) return;
    int p0, p1, p2;
    cell_of<R>(b, p.pos[i], p.pos[p.n + i], p.pos[2 * p.n + i], p0, p1, p2);
    out[i] = p0;
    out[p.n + i] = p1;
    out[2 * p.n + i] = p2;
}

template <class F>
int cartesian_impl(const rmpcd_box_t *box, const rmpcd_particles_t *pp, int32_t *out)
{
    PView<F> p = view<F>(pp);
    k_cartesian<F><<<blocks_for(p.n, 256), 256, 0, stream()>>>(make_box(box), p, out);
    RMPCD_LAUNCHED();
    return RMPCD_OK;
}

}  // namespace rmpcd

using namespace rmpcd;

extern "C" {

int rmpcd_count_particles(const rmpcd_box_t *box, const rmpcd_particles_t *p,
                          rmpcd_cells_t *cells)
{
    int rc = check_box(box, "rmpcd_count_particles");
    if (!rc) rc = check_particles(p, "rmpcd_count_particles", false);
    if (rc) return rc;
    RMPCD_CHECK(cells && cells->cell_count && cells->cell_start,
                "rmpcd_count_particles: null cell arrays");
    return RMPCD_DISPATCH_FORM(p, count_impl, box, p, cells);
}

int rmpcd_cartesian_indices(const rmpcd_box_t *box, const rmpcd_particles_t *p, int32_t *xyz)
{
    int rc = check_box(box, "rmpcd_cartesian_indices");
    if (!rc) rc = check_particles(p, "rmpcd_cartesian_indices", false);
    if (rc) return rc;
    RMPCD_CHECK(xyz != nullptr, "rmpcd_cartesian_indices: null output");
    return RMPCD_DISPATCH_FORM(p, cartesian_impl, box, p, xyz);
}

int rmpcd_sort(const rmpcd_box_t *box, const rmpcd_particles_t *src, rmpcd_particles_t *dst,
               int32_t *id_to_idx, rmpcd_cells_t *cells, int32_t apply_pbc)
{
    int rc = check_box(box, "rmpcd_sort");
    if (!rc) rc = check_particles(src, "rmpcd_sort", true);
    if (!rc) rc = check_particles(dst, "rmpcd_sort", true);
    if (rc) return rc;
    RMPCD_CHECK(src->n == dst->n && src->form == dst->form,
                "rmpcd_sort: source and destination differ in size or form");
    RMPCD_CHECK(src->image && dst->image && src->id && dst->id && id_to_idx,
                "rmpcd_sort: null image/id/id_to_idx");
    RMPCD_CHECK(cells && cells->cell_count && cells->cell_start, "rmpcd_sort: null cell arrays");
    // the gather reads every source slot while it writes the destination: the two sets
    // must be different buffers (the reference sorts into its second buffer and swaps)
    RMPCD_CHECK(src->pos != dst->pos && src->vel != dst->vel && src->force != dst->force &&
                    src->force_old != dst->force_old && src->image != dst->image &&
                    src->id != dst->id && src->species != dst->species && src->flags != dst->flags,
                "rmpcd_sort: source and destination share an array (the sort is out of place)");
    return sort_unchecked(box, src, dst, id_to_idx, cells, apply_pbc ? 1 : 0, false);
}

}  // extern "C"
