// DEM hot path on gfx950: spheres and half-spaces, linear spring-dashpot
// contacts with per-contact tangential history (examples/dem.py).
//
// Storage: structure of arrays in the reference's particle order (slot i is
// the reference's particle i: exchange and borders move particles exactly as
// the generated program does, so every order-dependent rule -- exchange tail
// fill, ghost order, cell order, contact slot order -- is the reference's).
// Contact history is [slot k][particle i] (k-major) so that the lanes of a
// wave, which hold consecutive particles, touch consecutive words.
//
// One step is a fixed sequence of kernels whose grids depend on capacities
// only; every count lives in device memory (DemCounters), so the step is
// captured once as a hipGraph and replayed.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.hpp"
#include "dem_kernels.hpp"

namespace dk {

// copy table entry blockIdx.y, grid-strided over its rows x words
__global__ __launch_bounds__(256) void k_copy_rows(const CopyDesc *__restrict__ table) {
    const CopyDesc c = table[blockIdx.y];
    const uint32_t *__restrict__ src = (const uint32_t *) c.src;
    uint32_t *__restrict__ dst = (uint32_t *) c.dst;
    const size_t total = (size_t) c.words * (size_t) c.rows;
    for (size_t e = (size_t) blockIdx.x * 256 + threadIdx.x; e < total; e += (size_t) gridDim.x * 256) {
        const size_t r = e / (size_t) c.words, w = e - r * (size_t) c.words;
        dst[r * c.dst_pitch + w] = src[r * c.src_pitch + w];
    }
}

void launch_copy_rows(hipStream_t s, const CopyDesc *table, int ncopies, int n) {
    if (ncopies <= 0 || n <= 0) return;
    // the widest entry: a double array of 9 rows of n particles
    const size_t most = (size_t) 2 * n * 9;
    const int gx = (int) std::min<size_t>((most + 255) / 256, 1024);
    hipLaunchKernelGGL(k_copy_rows, dim3(gx, ncopies), dim3(256), 0, s, table);
}

__global__ void k_fill_i32(int *__restrict__ p, int v, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = v;
}

// ---------------------------------------------------------------- scans

template <int BS>
__device__ __forceinline__ int block_scan_excl(int v, int *lds, int *total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) lds[wave] = x;
    __syncthreads();
    // every wave sums the wave totals itself
    constexpr int NW = BS / 64;
    const int w = lane < NW ? lds[lane] : 0;
    int t = w;
#pragma unroll
    for (int off = 1; off < NW; off <<= 1) {
        const int y = __shfl_up(t, off, 64);
        if (lane >= off) t += y;
    }
    *total = __shfl(t, NW - 1, 64);
    const int r = __shfl(t - w, wave, 64) + x - v;
    __syncthreads();
    return r;
}

// ---------------------------------------------------------------- selection (exchange / borders)

// DimensionRanges predicates (src/pairs/sim/domain_partitioning.py:31-65):
// side 0 "x_d < min + offset", side 1 "x_d > max - offset", Infinite and
// Global particles excluded (flags & 9).
__device__ __forceinline__ void dsel(double xd, int fl, double lo, double hi, double off, bool &s0, bool &s1) {
    const bool ok = (fl & (DFLAG_INFINITE | DFLAG_GLOBAL)) == 0;
    s0 = ok && xd < lo + off;
    s1 = ok && xd > hi - off;
}

// a particle outside the box along a periodic dimension joins the list that the
// next exchange reads.  An exchange shifts a particle only along its own
// dimension, so whoever leaves along any of them is outside before the first.
__device__ __forceinline__ void note_leaver(const DemPtrs &p, int *__restrict__ c, const DemGeom &g, int i, int fl,
                                            double x, double y, double z) {
    const double xs[3] = {x, y, z};
    bool out = false;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        bool a, b;
        dsel(xs[d], fl, g.lo[d], g.hi[d], 0.0, a, b);
        out = out || (g.periodic[d] && (a || b));
    }
    if (!out) return;
    const int k = atomicAdd(&c[D_LEAVE], 1);
    if (k < LEAVE_CAP) p.leavers[k] = i;
}

__global__ __launch_bounds__(256) void k_find_leavers(DemPtrs p, int *__restrict__ c, DemGeom g) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < c[D_NLOCAL]) note_leaver(p, c, g, i, p.flags[i], p.x[i], p.y[i], p.z[i]);
}

// ---------------------------------------------------------------- exchange with contact history

// remove_exchanged_particles_pt1 (src/pairs/sim/comm.py:445-470): holes of
// leavers below nlocal - n are filled from the tail, skipping leavers
__device__ __forceinline__ void exch_pt1(int n, int nl, const int *__restrict__ send_map,
                                         const int *__restrict__ exchg_flag, int *__restrict__ copy_to) {
    int pos = nl - 1;
    for (int i = 0; i < n; i++) {
        if (send_map[i] < nl - n) {
            while (exchg_flag[pos] == 1) pos--;
            copy_to[i] = pos;
            pos--;
        } else {
            copy_to[i] = -1;
        }
    }
}

// what travels with a particle (comm.py:61-72, the property list of the
// exchange): arrays of doubles, then of words
constexpr int EXD = 36, EXI = 4, EXB = EXD + EXI;

__device__ __forceinline__ double *exch_array(const DemPtrs &p, int f) {
    double *const a[14] = {p.x, p.y, p.z, p.m, p.vx, p.vy, p.vz, p.wx, p.wy, p.wz, p.r, p.nx, p.ny, p.nz};
    double *r = a[0];
#pragma unroll
    for (int k = 1; k < 14; k++) r = f == k ? a[k] : r;
    if (f >= 14) r = p.inv_i + (size_t) (f - 14) * p.cap;
    if (f >= 23) r = p.rot_m + (size_t) (f - 23) * p.cap;
    if (f >= 32) r = p.rot_q + (size_t) (f - 32) * p.cap;
    return r;
}

__device__ __forceinline__ int *exch_words(const DemPtrs &p, int f) {
    return f == 0 ? p.uid : f == 1 ? p.shape : f == 2 ? p.flags : p.type;
}

// slot k of the contact history of src written to dst
__device__ __forceinline__ void copy_contact(const DemPtrs &p, int k, int dst, int src) {
    const size_t a = (size_t) k * p.cap + dst, b = (size_t) k * p.cap + src;
    const size_t ta = 3 * (size_t) k * p.cap + dst, tb = 3 * (size_t) k * p.cap + src, C = p.cap;
    const int u = p.c_uid[b], w = p.c_used[b], s = p.c_stick[b];
    const double t0 = p.c_tsd[tb], t1 = p.c_tsd[tb + C], t2 = p.c_tsd[tb + 2 * C], v = p.c_ivm[b];
    p.c_uid[a] = u; p.c_used[a] = w; p.c_stick[a] = s;
    p.c_tsd[ta] = t0; p.c_tsd[ta + C] = t1; p.c_tsd[ta + 2 * C] = t2;
    p.c_ivm[a] = v;
}

// The leavers of one dimension moved: properties packed with the position
// shifted (comm.py:312-318), the holes filled from the tail with their contact
// history (remove_exchanged_particles_pt2, comm.py:473-506; copy guard "src >
// 0"), the leavers unpacked at nlocal - n + i, and the history of the leaver's
// slot as it is after the hole filling packed and unpacked (the reference packs
// it then); every contact's uid lands in one buffer word, so the last contact's
// uid is the one that travels.  Each phase is finished before the next begins.
// A thread moves one word or one contact of one leaver.
__device__ __forceinline__ void exch_move(const DemPtrs &p, double *const *s_arr, int n, int nl, int dim,
                                          const DemGeom &g) {
    const int nt = blockDim.x, base = nl - n, hb = 2 + 5 * p.ccap;
    const size_t C = p.cap;
    for (int e = threadIdx.x; e < n * EXB; e += nt) {
        const int i = e / EXB, f = e - i * EXB, m = p.send_map[i];
        double v;
        if (f < EXD) {
            v = s_arr[f][m];
            if (f < 3) v = v + (f == dim ? (p.send_side[i] == 0 ? 1 : -1) : 0) * g.len[f];
        } else {
            v = exch_words(p, f - EXD)[m];
        }
        p.buf[e] = v;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < n * EXB; e += nt) {
        const int i = e / EXB, f = e - i * EXB, src = p.copy_to[i];
        if (src <= 0) continue;
        const int dst = p.send_map[i];
        if (f < EXD) s_arr[f][dst] = s_arr[f][src];
        else exch_words(p, f - EXD)[dst] = exch_words(p, f - EXD)[src];
    }
    for (int e = threadIdx.x; e < n * p.ccap; e += nt) {
        const int i = e / p.ccap, k = e - i * p.ccap, src = p.copy_to[i];
        if (src <= 0) continue;
        const int dst = p.send_map[i], nc = p.num_contacts[src];
        if (k < nc) copy_contact(p, k, dst, src);
        if (k == 0) p.num_contacts[dst] = nc;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < n * EXB; e += nt) {
        const int i = e / EXB, f = e - i * EXB;
        if (f < EXD) s_arr[f][base + i] = p.buf[e];
        else exch_words(p, f - EXD)[base + i] = (int) p.buf[e];
    }
    for (int e = threadIdx.x; e < n * p.ccap; e += nt) {
        const int i = e / p.ccap, k = e - i * p.ccap, m = p.send_map[i], nc = p.num_contacts[m];
        double *b = p.hbuf + (size_t) hb * i;
        if (k == 0) {
            b[0] = nc;
            if (nc == 0) b[1] = 0.0;
        }
        if (k >= nc) continue;
        const size_t a = (size_t) k * C + m, t = 3 * (size_t) k * C + m;
        if (k == nc - 1) b[1] = p.c_uid[a];
        const int stick = p.c_stick[a];
        const double t0 = p.c_tsd[t], t1 = p.c_tsd[t + C], t2 = p.c_tsd[t + 2 * C], v = p.c_ivm[a];
        b += 2 + 5 * k;
        b[0] = stick; b[1] = t0; b[2] = t1; b[3] = t2; b[4] = v;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < n * p.ccap; e += nt) {
        const int i = e / p.ccap, k = e - i * p.ccap, to = base + i;
        const double *b = p.hbuf + (size_t) hb * i;
        const int nc = (int) b[0], uid = (int) b[1];
        if (k == 0) p.num_contacts[to] = nc;
        if (k >= nc) continue;
        b += 2 + 5 * k;
        const size_t a = (size_t) k * C + to, t = 3 * (size_t) k * C + to;
        const double v0 = b[0], t0 = b[1], t1 = b[2], t2 = b[3], v = b[4];
        p.c_uid[a] = uid; p.c_used[a] = 1; p.c_stick[a] = (int) v0;
        p.c_tsd[t] = t0; p.c_tsd[t + C] = t1; p.c_tsd[t + 2 * C] = t2;
        p.c_ivm[a] = v;
    }
    __syncthreads();
}

// The exchange, dimension by dimension (comm.py:100-151), in one workgroup: a
// step moves few particles across a face, and they are on the list that the
// integration before has left.  A thread holds one of them, follows it where an
// exchange moves it, and ranks it among the leavers of a dimension (side 0
// before side 1, each in index order: the reference's send order); the tail
// that fills the holes is planned with two scans.  More leavers than the list
// holds are found by a scan of the locals instead.  Bound by the latency of its
// phases.  It replaces, per dimension, a count and a scatter pass over the
// locals and a kernel whose thread 0 walked the tail through memory (bed of
// 187200 spheres, two dimensions: 46 us -> 7.9).
__global__ __launch_bounds__(1024) void k_exchange(DemPtrs p, int *__restrict__ c, DemGeom g) {
    __shared__ int lds[20];
    __shared__ double *s_arr[EXD];
    __shared__ __align__(16) unsigned s_key[LEAVE_CAP];
    __shared__ int s_map[LEAVE_CAP], s_fill[LEAVE_CAP], s_hole[LEAVE_CAP], s_tail[LEAVE_CAP];
    const int tid = threadIdx.x, cnt = c[D_LEAVE], nl = c[D_NLOCAL], ovf = c[D_OVF];
    __syncthreads();
    if (tid == 0) c[D_LEAVE] = 0;
    if (ovf || cnt == 0) return;
    if (tid < EXD) s_arr[tid] = exch_array(p, tid);
    const bool listed = cnt <= LEAVE_CAP;
    int me = listed && tid < cnt ? p.leavers[tid] : -1;
    for (int dim = 0; dim < 3; dim++) {
        if (!g.periodic[dim]) continue;
        const double *Xd = dim == 0 ? p.x : (dim == 1 ? p.y : p.z);
        int n;
        if (listed) {
            bool a = false, b = false;
            if (me >= 0) dsel(Xd[me], p.flags[me], g.lo[dim], g.hi[dim], 0.0, a, b);
            const bool out = a || b;
            const unsigned key = a ? (unsigned) me : b ? (unsigned) me | 0x80000000u : 0xffffffffu;
            s_key[tid] = key;
            s_tail[tid] = 0;
            n = __syncthreads_count(out);
            if (n == 0) continue;
            if (n <= p.send_cap) {
                int rank = 0;
                if (__ballot(out)) {  // (the entries past cnt are the largest key)
                    const uint4 *k4 = (const uint4 *) s_key;
#pragma unroll 4
                    for (int u = 0; u < (cnt + 3) / 4; u++) {
                        const uint4 k = k4[u];
                        rank += (k.x < key ? 1 : 0) + (k.y < key ? 1 : 0) + (k.z < key ? 1 : 0) + (k.w < key ? 1 : 0);
                    }
                }
                if (out) {
                    s_map[rank] = me;
                    p.send_map[rank] = me;
                    p.send_side[rank] = a ? 0 : 1;
                    if (me >= nl - n) s_tail[nl - 1 - me] = 1;
                }
                __syncthreads();
                int total;
                const bool fills = tid < n && !s_tail[tid], hole = tid < n && s_map[tid] < nl - n;
                const int ef = block_scan_excl<1024>(fills ? 1 : 0, lds, &total);
                const int eh = block_scan_excl<1024>(hole ? 1 : 0, lds, &total);
                if (fills) { s_fill[ef] = nl - 1 - tid; s_tail[tid] = 2 + ef; }
                if (hole) s_hole[eh] = s_map[tid];
                __syncthreads();
                if (tid < n) p.copy_to[tid] = hole ? s_fill[eh] : -1;
                if (out) me = nl - n + rank;
                else if (me >= nl - n) me = s_hole[s_tail[nl - 1 - me] - 2];
            }
        } else {
            // totals, then places in index order within each side
            int t0 = 0, t1 = 0;
            for (int i0 = 0; i0 < nl; i0 += 1024) {
                const int i = i0 + tid;
                bool a = false, b = false;
                if (i < nl) dsel(Xd[i], p.flags[i], g.lo[dim], g.hi[dim], 0.0, a, b);
                if (i < nl) p.exchg_flag[i] = a || b ? 1 : 0;
                t0 += __syncthreads_count(a);
                t1 += __syncthreads_count(b);
            }
            n = t0 + t1;
            if (n == 0) continue;
            if (n <= p.send_cap) {
                int o0 = 0, o1 = t0;
                for (int i0 = 0; i0 < nl; i0 += 1024) {
                    const int i = i0 + tid;
                    bool a = false, b = false;
                    if (i < nl) dsel(Xd[i], p.flags[i], g.lo[dim], g.hi[dim], 0.0, a, b);
                    int s0, s1;
                    const int q0 = block_scan_excl<1024>(a ? 1 : 0, lds, &s0);
                    const int q1 = block_scan_excl<1024>(b ? 1 : 0, lds, &s1);
                    if (a) { p.send_map[o0 + q0] = i; p.send_side[o0 + q0] = 0; }
                    if (b) { p.send_map[o1 + q1] = i; p.send_side[o1 + q1] = 1; }
                    o0 += s0;
                    o1 += s1;
                }
                __syncthreads();
                if (tid == 0) exch_pt1(n, nl, p.send_map, p.exchg_flag, p.copy_to);
            }
        }
        if (n > p.send_cap) {
            if (tid == 0) {
                atomicMax(&c[D_REQ_SEND], n);
                atomicMax(&c[D_OVF], DOVF_SEND);
            }
            return;
        }
        __syncthreads();
        exch_move(p, s_arr, n, nl, dim, g);
    }
}

// ---------------------------------------------------------------- borders and cell counts

__device__ __forceinline__ int dcell_dim(double x, int d, const DemGeom &g) {
    const double q = (x - (g.lo[d] - g.width)) / g.width;
    const int cc = (int) q >= 0 ? (int) q : 0;
    return cc < g.dim_cells[d] ? cc : g.dim_cells[d] - 1;
}

__device__ __forceinline__ int dcell_index(int cx, int cy, int cz, const DemGeom &g) {
    return (cx * g.dim_cells[1] + cy) * g.dim_cells[2] + cz + 1;
}

__device__ __forceinline__ int dcell_of(double x, double y, double z, const DemGeom &g) {
    return dcell_index(dcell_dim(x, 0, g), dcell_dim(y, 1, g), dcell_dim(z, 2, g), g);
}

constexpr int pow3(int n) { return n == 0 ? 1 : 3 * pow3(n - 1); }

// the k-th periodic dimension
__device__ __forceinline__ int periodic_dim(const DemGeom &g, int k) {
    int d = 0;
    for (; d < 3; d++)
        if (g.periodic[d] && k-- == 0) break;
    return d;
}

// Borders (comm.py:56-98): dimension by dimension, side 0 then side 1, every
// local and every ghost of the dimensions before that lies within a cell width
// of the face gets a ghost behind all others.  A ghost keeps its particle's
// other coordinates, so whether it is selected along a later dimension depends
// on the particle alone, and the ghosts of all dimensions fall into kinds: one
// digit per periodic dimension (0 not shifted, 1 side 0, 2 side 1), the later
// dimension the higher digit.  The order of the ghosts is that of their kind as
// a number in base 3, and within a kind the index order of the particles.  So
// one count per kind and block of particles (k_border_count) places them all.
template <int ND>
struct Kinds {
    bool side[ND > 0 ? ND : 1][2];
    __device__ __forceinline__ void set(const DemGeom &g, const double (&xs)[3], int fl, bool in) {
#pragma unroll
        for (int k = 0; k < ND; k++) {
            const int d = ND == 3 ? k : periodic_dim(g, k);
            const double xd = d == 0 ? xs[0] : d == 1 ? xs[1] : xs[2];
            bool a, b;
            dsel(xd, fl, g.lo[d], g.hi[d], g.width, a, b);
            side[k][0] = in && a;
            side[k][1] = in && b;
        }
    }
    __device__ __forceinline__ bool any() const {
        bool r = false;
#pragma unroll
        for (int k = 0; k < ND; k++) r = r || side[k][0] || side[k][1];
        return r;
    }
    __device__ __forceinline__ bool has(int kind) const {
        bool r = true;
#pragma unroll
        for (int k = 0; k < ND; k++) {
            const int digit = kind % 3;
            kind /= 3;
            r = r && (digit == 0 || side[k][digit == 2 ? 1 : 0]);
        }
        return r;
    }
};

// Locals into their cells (BuildCellLists, src/pairs/sim/cell_lists.py:90-134;
// Infinite -> cell 0) and the ghosts of each kind counted by block.  Bound by
// the returning atomics of the cell counts.
template <int ND>
__global__ __launch_bounds__(256) void k_cell_count(DemPtrs p, int *__restrict__ c, DemGeom g, int pitch) {
    constexpr int NK = pow3(ND);
    __shared__ int s_n[NK][4];
    const int nl = c[D_NLOCAL];
    if (ND == 0 && blockIdx.x == 0 && threadIdx.x == 0) c[D_NGHOST] = 0;
    if ((int) blockIdx.x * 256 >= nl) return;
    const int i = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Kinds<ND> K;
    double xs[3] = {0.0, 0.0, 0.0};
    int fl = 0, cell = 0, slot = 0;
    if (i < nl) {
        xs[0] = p.x[i]; xs[1] = p.y[i]; xs[2] = p.z[i]; fl = p.flags[i];
        cell = (fl & DFLAG_INFINITE) ? 0 : dcell_of(xs[0], xs[1], xs[2], g);
        slot = atomicAdd(&p.cell_count[cell], 1);  // its place among the cell's entries
    }
    if (ND > 0) {
        K.set(g, xs, fl, i < nl);
        const bool some = __ballot(K.any()) != 0;
#pragma unroll
        for (int k = 1; k < NK; k++) {
            const int m = some ? __popcll(__ballot(K.has(k))) : 0;
            if (lane == 0) s_n[k][wave] = m;
        }
        __syncthreads();
        const int k = threadIdx.x;
        if (k >= 1 && k < NK) p.blk[(size_t) k * pitch + blockIdx.x] = s_n[k][0] + s_n[k][1] + s_n[k][2] + s_n[k][3];
    }
    if (i < nl) {
        p.particle_cell[i] = cell;
        p.cell_slot[i] = slot;
    }
}

// The ghosts at nlocal + place (uid, type, mass, radius, position + shift,
// linear and angular velocity, shape; flags are not sent, comm.py:61-72), and
// their cells counted.  Every workgroup sums the counts of the blocks itself,
// so the places need no pass of their own, and takes the same capacity
// decision, dimension by dimension; without room no ghost is made and the cells
// hold the locals.  Bound by latency: the particle's fields are loaded before
// the sums and the atomics of all kinds are in flight before the first place
// is stored.  2080 | 187200 spheres, us: with the locals' atomics here, a kind
// and its cell at a time 12 | 22 on top of 2.6 | 4.7 for the counts; so 7.7 |
// 9.4 on top of 3.1 | 9.6 for k_cell_count.
template <int ND>
__global__ __launch_bounds__(256) void k_border_ghosts(DemPtrs p, int *__restrict__ c, DemGeom g, int pitch) {
    constexpr int NK = pow3(ND);
    __shared__ int s_total[NK], s_before[NK], s_wave[NK][4];
    const int nl = c[D_NLOCAL], ovf = c[D_OVF];
    const int nblk = (nl + 255) / 256;
    if (blockIdx.x > 0 && (int) blockIdx.x >= nblk) return;  // workgroup 0 always writes the count
    const int i = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Kinds<ND> K;
    double xs[3] = {0.0, 0.0, 0.0};
    int fl = 0;
    if (i < nl) { xs[0] = p.x[i]; xs[1] = p.y[i]; xs[2] = p.z[i]; fl = p.flags[i]; }
    K.set(g, xs, fl, i < nl);
    int uid = 0, type = 0, shape = 0;
    double m = 0.0, r = 0.0, v[3] = {0.0, 0.0, 0.0}, w[3] = {0.0, 0.0, 0.0};
    const bool mine = K.any();
    if (mine) {
        uid = p.uid[i]; type = p.type[i]; shape = p.shape[i]; m = p.m[i]; r = p.r[i];
        v[0] = p.vx[i]; v[1] = p.vy[i]; v[2] = p.vz[i]; w[0] = p.wx[i]; w[1] = p.wy[i]; w[2] = p.wz[i];
    }
    const bool some = __ballot(mine) != 0;
#pragma unroll
    for (int k = 1; k < NK; k++) {
        const int n = some ? __popcll(__ballot(K.has(k))) : 0;
        if (lane == 0) s_wave[k][wave] = n;
    }
    constexpr int PER = (NK + 2) / 4;  // kinds of a wave: 1 + wave, 5 + wave, ..
    constexpr int AHEAD = ND == 3 ? 1 : 8;
    int t[PER] = {}, q[PER] = {};
#pragma unroll AHEAD
    for (int u = lane; u < nblk; u += 64) {
#pragma unroll
        for (int e = 0; e < PER; e++) {
            const int k = 1 + wave + 4 * e;
            const int x = k < NK ? p.blk[(size_t) k * pitch + u] : 0;
            t[e] += x;
            q[e] += u < (int) blockIdx.x ? x : 0;
        }
    }
#pragma unroll
    for (int e = 0; e < PER; e++) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            t[e] += __shfl_xor(t[e], o, 64);
            q[e] += __shfl_xor(q[e], o, 64);
        }
        const int k = 1 + wave + 4 * e;
        if (lane == 0 && k < NK) { s_total[k] = t[e]; s_before[k] = q[e]; }
    }
    __syncthreads();
    int need = 0, short_of = DOVF_NONE;
#pragma unroll
    for (int d = 0; d < ND; d++) {
        if (short_of) break;
        for (int k = pow3(d); k < pow3(d + 1); k++) need += s_total[k];
        short_of = need > p.send_cap ? DOVF_SEND : nl + need > p.cap ? DOVF_PART : DOVF_NONE;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c[D_NGHOST] = ovf || short_of ? 0 : need;
        if (!ovf && short_of) {
            atomicMax(&c[short_of == DOVF_SEND ? D_REQ_SEND : D_REQ_PART], short_of == DOVF_SEND ? need : nl + need);
            atomicMax(&c[D_OVF], short_of);
        }
    }
    if (ovf || short_of || !some) return;
    // places by kind, cells by dimension and shift
    int to[NK], slot[NK], at = nl;
#pragma unroll
    for (int k = 1; k < NK; k++) {
        int n = 0;
#pragma unroll
        for (int u = 0; u < 3; u++) n += u < wave ? s_wave[k][u] : 0;
        to[k] = at + s_before[k] + n + lane_rank(__ballot(K.has(k)));
        at += s_total[k];
    }
    if (!mine) return;
    double y[3][3];
    int cc[3][3];
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int e = 0; e < 3; e++) {
            // src += send_mult * length (comm.py:312-318)
            y[d][e] = xs[d] + (double) (e == 1 ? 1 : e == 2 ? -1 : 0) * g.len[d];
            cc[d][e] = e == 0 || g.periodic[d] ? dcell_dim(y[d][e], d, g) : 0;
        }
#pragma unroll
    for (int k = 1; k < NK; k++) {
        if (!K.has(k)) continue;
        int digits = k, cell[3];
        double z[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            int e = 0;
            if (g.periodic[d]) { e = digits % 3; digits /= 3; }
            z[d] = e == 0 ? y[d][0] : e == 1 ? y[d][1] : y[d][2];
            cell[d] = e == 0 ? cc[d][0] : e == 1 ? cc[d][1] : cc[d][2];
        }
        const int to_k = to[k], ck = dcell_index(cell[0], cell[1], cell[2], g);
        slot[k] = atomicAdd(&p.cell_count[ck], 1);
        p.particle_cell[to_k] = ck;
        p.uid[to_k] = uid; p.type[to_k] = type; p.shape[to_k] = shape; p.m[to_k] = m; p.r[to_k] = r;
        p.x[to_k] = z[0]; p.y[to_k] = z[1]; p.z[to_k] = z[2];
        p.vx[to_k] = v[0]; p.vy[to_k] = v[1]; p.vz[to_k] = v[2];
        p.wx[to_k] = w[0]; p.wy[to_k] = w[1]; p.wz[to_k] = w[2];
    }
#pragma unroll
    for (int k = 1; k < NK; k++)
        if (K.has(k)) p.cell_slot[to[k]] = slot[k];
}

// exclusive scan of the cell counts: each block's own, and the block totals;
// the counts are cleared behind the reads (nothing else uses them, so the next
// binning starts from zeros)
__global__ __launch_bounds__(1024) void k_scan_partial(int *__restrict__ in, int *__restrict__ out,
                                                       int *__restrict__ bsum, int n) {
    __shared__ int lds[20];
    const int i = blockIdx.x * 1024 + threadIdx.x;
    int t;
    const int v = i < n ? in[i] : 0;
    if (v) in[i] = 0;
    const int e = block_scan_excl<1024>(v, lds, &t);
    if (i < n) out[i] = e;
    if (threadIdx.x == 0) bsum[blockIdx.x] = t;
}

// each block adds the totals of the blocks before it to the scan of its own
__global__ __launch_bounds__(1024) void k_scan_add(const int *__restrict__ in, int *__restrict__ out,
                                                   const int *__restrict__ bsum, int n) {
    __shared__ int red[16];
    int q = 0;
    for (int b = threadIdx.x; b < (int) blockIdx.x; b += 1024) q += bsum[b];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) q += __shfl_xor(q, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = q;
    __syncthreads();
    int off = 0;
#pragma unroll
    for (int w = 0; w < 16; w++) off += red[w];
    const int i = blockIdx.x * 1024 + threadIdx.x;
    if (i < n) out[i] = in[i] + off;
}

// The particles into their cells (a half-space's entry carries a mark).  ADD: the blocks' offsets are not in
// cell_start yet: every workgroup scans the block totals (at most SCAN_LDS of
// them) in LDS and adds them where it needs them, and the workgroups share the
// writing of cell_start for the passes behind.
constexpr int SCAN_LDS = 2048;
constexpr int CELL_PLANE = (int) 0x80000000;
// what a half-space's ordered record holds in place of its radius (a value that
// no sphere has, also one of negative radius)
constexpr double PLANE_MARK = -__builtin_inf();
template <bool ADD>
__global__ __launch_bounds__(256) void k_cell_fill(DemPtrs p, const int *__restrict__ c, int nstart, int nblk) {
    __shared__ int s_off[ADD ? SCAN_LDS : 1];
    __shared__ int lds[8];
    const int n = c[D_NLOCAL] + c[D_NGHOST];
    const int i = blockIdx.x * 256 + threadIdx.x;
    int cell = 0, start = 0, slot = 0, sh = 0;
    if (i < n) {
        sh = p.shape[i];
        cell = p.particle_cell[i];
        slot = p.cell_slot[i];
        start = (ADD ? p.cell_scan : p.cell_start)[cell];
    }
    if (ADD) {
        int at = 0;
        for (int b0 = 0; b0 < nblk; b0 += 256) {
            const int b = b0 + threadIdx.x;
            int total;
            const int e = block_scan_excl<256>(b < nblk ? p.scan_tmp[b] : 0, lds, &total);
            if (b < nblk) s_off[b] = at + e;
            at += total;
        }
        __syncthreads();
        for (int k = i; k < nstart; k += gridDim.x * 256) p.cell_start[k] = p.cell_scan[k] + s_off[k >> 10];
        start += s_off[cell >> 10];
    }
    if (i < n) p.cell_particles[start + slot] = i | (sh != DSHAPE_SPHERE ? CELL_PLANE : 0);
}

// PartitionCellLists (src/pairs/sim/cell_lists.py:137-171) of one cell, whose
// entries cp[0, cnt) come in any order: index order (the CPU's insertion
// order), then the in-place two-pointer partition by shape, spheres then
// half-spaces
__device__ __forceinline__ void partition_cell(const int *__restrict__ shape, int *cp, int cnt) {
    for (int a = 1; a < cnt; a++) {
        const int v = cp[a];
        int b = a - 1;
        while (b >= 0 && cp[b] > v) { cp[b + 1] = cp[b]; b--; }
        cp[b + 1] = v;
    }
    int lo = 0;
    for (int sh = 0; sh < 2; sh++) {
        int hi = cnt - 1;
        while (lo <= hi) {
            const int q = cp[lo];
            if (shape[q] != sh) {
                if (lo != hi) { cp[lo] = cp[hi]; cp[hi] = q; }
                hi--;
            } else {
                lo++;
            }
        }
    }
}

// One thread per particle: its place in its cell's order, and the records the
// contact kernels read -- by place: index, cell (bit 31: FIXED) and (x, y, z,
// r); by index: everything a contact needs of its partner in one 128-byte line
// (a gather of twelve arrays touches twelve lines).  In a cell of spheres the
// order is the index order, so a particle's place is the number of smaller
// indices in the cell; a cell that holds a half-space is ordered by the thread
// of its first particle and written by it.  Bound by memory: 100 bytes in and
// 136 out per particle, the records through LDS so that a wave writes whole
// lines (13 us at 190000 particles; 42 with each thread storing its record).
// A cell's entries are read four at a time and say themselves which of them is
// a half-space (15 us with an entry and its shape at a time).
__global__ __launch_bounds__(256) void k_cell_order(DemPtrs p, const int *__restrict__ c) {
    constexpr int W = 13;  // LDS row of a record (doubles, one of padding)
    __shared__ double s_rec[256 * W];
    const int n = c[D_NLOCAL] + c[D_NGHOST];
    const int b0 = blockIdx.x * 256;
    const int i = b0 + threadIdx.x;
    if (b0 >= n) return;
    int sh = DSHAPE_SPHERE, fl = 0, cell = 0, s0 = 0, cnt = 0;
    double x = 0.0, y = 0.0, z = 0.0, r = 0.0;
    if (i < n) {
        cell = p.particle_cell[i];
        sh = p.shape[i];
        fl = p.flags[i];
        x = p.x[i]; y = p.y[i]; z = p.z[i]; r = p.r[i];
        double *R = s_rec + threadIdx.x * W;
        R[0] = x; R[1] = y; R[2] = z; R[3] = r;
        R[4] = p.vx[i]; R[5] = p.vy[i]; R[6] = p.vz[i]; R[7] = p.m[i];
        R[8] = p.wx[i]; R[9] = p.wy[i]; R[10] = p.wz[i];
        R[11] = __longlong_as_double((long long) p.uid[i] << 32 | (unsigned) p.type[i]);
        s0 = p.cell_start[cell];
        cnt = p.cell_start[cell + 1] - s0;
    }
    __syncthreads();
    // the block's records, 16 bytes per thread at consecutive addresses
    const int nb = min(256, n - b0);
    for (int u = threadIdx.x; u < 6 * nb; u += 256) {
        const int k = u / 6, w = u - 6 * k;
        const double *R = s_rec + k * W + 2 * w;
        ((double2 *) (p.rec + b0 + k))[w] = make_double2(R[0], R[1]);
    }
    if (i >= n) return;
    int rank = 0;
    bool mixed = sh != DSHAPE_SPHERE;
    if (cnt > 1)
        for (int k0 = 0; k0 < cnt; k0 += 4) {
            int e[4];
#pragma unroll
            for (int u = 0; u < 4; u++) e[u] = p.cell_particles[s0 + min(k0 + u, cnt - 1)];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                rank += k0 + u < cnt && (e[u] & ~CELL_PLANE) < i ? 1 : 0;
                mixed = mixed || e[u] < 0;
            }
        }
    auto put = [&](int q, int j, int jf, double jx, double jy, double jz, double jr, int jsh) {
        p.corder[q] = make_int2(j, cell | ((jf & DFLAG_FIXED) ? (int) 0x80000000 : 0));
        p.crec[q] = make_double4(jx, jy, jz, jsh == DSHAPE_SPHERE ? jr : PLANE_MARK);
    };
    if (!mixed) {
        put(s0 + rank, i, fl, x, y, z, r, sh);
    } else if (rank == 0) {
        int *cp = p.cmixed + s0;
        for (int k = 0; k < cnt; k++) cp[k] = p.cell_particles[s0 + k] & ~CELL_PLANE;
        partition_cell(p.shape, cp, cnt);
        for (int k = 0; k < cnt; k++) {
            const int j = cp[k];
            put(s0 + k, j, p.flags[j], p.x[j], p.y[j], p.z[j], p.r[j], p.shape[j]);
        }
    }
}

// ---------------------------------------------------------------- integration

// euler (examples/dem.py:77-85) of particle i under force f and torque tq, with
// quaternion(phi, |phi|) and quaternion_to_rotation_matrix
// (src/pairs/mapping/keywords.py:190-252); a particle it moves out of the box is
// noted for the next exchange
__device__ __forceinline__ void euler_particle(const DemPtrs &p, int *__restrict__ c, const DemGeom &g, double dt,
                                               int i, int fl, const double (&f)[3], const double (&tq)[3]) {
    if (fl & DFLAG_FIXED) {
        note_leaver(p, c, g, i, fl, p.x[i], p.y[i], p.z[i]);
        return;
    }
    const size_t C = p.cap;
    const double im = 1.0 / p.m[i];
    const double hm = 0.5 * im;
    double x[3] = {p.x[i], p.y[i], p.z[i]}, v[3] = {p.vx[i], p.vy[i], p.vz[i]}, w[3] = {p.wx[i], p.wy[i], p.wz[i]};
    for (int d = 0; d < 3; d++) x[d] = x[d] + (((hm * f[d]) * dt) * dt + v[d] * dt);
    for (int d = 0; d < 3; d++) v[d] = v[d] + (im * f[d]) * dt;
    double I[9], R[9], q[4];
    for (int k = 0; k < 9; k++) { I[k] = p.inv_i[k * C + i]; R[k] = p.rot_m[k * C + i]; }
    for (int k = 0; k < 4; k++) q[k] = p.rot_q[k * C + i];
    double a[3], b[3], wd[3];
    for (int r = 0; r < 3; r++) a[r] = (I[3 * r] * tq[0] + I[3 * r + 1] * tq[1]) + I[3 * r + 2] * tq[2];
    for (int r = 0; r < 3; r++) b[r] = (R[3 * r] * a[0] + R[3 * r + 1] * a[1]) + R[3 * r + 2] * a[2];
    for (int cc = 0; cc < 3; cc++) wd[cc] = (b[0] * R[cc] + b[1] * R[3 + cc]) + b[2] * R[6 + cc];
    double phi[3];
    for (int d = 0; d < 3; d++) phi[d] = w[d] * dt + ((0.5 * wd[d]) * dt) * dt;
    const double plen = sqrt((phi[0] * phi[0] + phi[1] * phi[1]) + phi[2] * phi[2]);
    double dq[4];
    if (fabs(plen) < 1e-06) {
        dq[0] = 1.0; dq[1] = 0.0; dq[2] = 0.0; dq[3] = 0.0;
    } else {
        const double cs = cos(plen * 0.5), sn = sin(plen * 0.5), inv = 1.0 / plen;
        dq[0] = cs;
        for (int d = 0; d < 3; d++) dq[1 + d] = sn * (phi[d] * inv);
    }
    const double p0 = ((dq[0] * q[0] - dq[1] * q[1]) - dq[2] * q[2]) - dq[3] * q[3];
    const double p1 = ((dq[0] * q[1] + dq[1] * q[0]) + dq[2] * q[3]) - dq[3] * q[2];
    const double p2 = ((dq[0] * q[2] + dq[2] * q[0]) + dq[3] * q[1]) - dq[1] * q[3];
    const double p3 = ((dq[0] * q[3] + dq[3] * q[0]) + dq[1] * q[2]) - dq[2] * q[1];
    const double n2 = ((p0 * p0 + p1 * p1) + p2 * p2) + p3 * p3;
    const double sc = (fabs(n2 - 1.0) < 1e-08) ? 1.0 : 1.0 / sqrt(n2);
    q[0] = p0 * sc; q[1] = p1 * sc; q[2] = p2 * sc; q[3] = p3 * sc;
    R[0] = (1.0 - (2.0 * q[2]) * q[2]) - (2.0 * q[3]) * q[3];
    R[1] = 2.0 * (q[1] * q[2] - q[0] * q[3]);
    R[2] = 2.0 * (q[1] * q[3] + q[0] * q[2]);
    R[3] = 2.0 * (q[1] * q[2] + q[0] * q[3]);
    R[4] = (1.0 - (2.0 * q[1]) * q[1]) - (2.0 * q[3]) * q[3];
    R[5] = 2.0 * (q[2] * q[3] - q[0] * q[1]);
    R[6] = 2.0 * (q[1] * q[3] - q[0] * q[2]);
    R[7] = 2.0 * (q[2] * q[3] + q[0] * q[1]);
    R[8] = (1.0 - (2.0 * q[1]) * q[1]) - (2.0 * q[2]) * q[2];
    for (int d = 0; d < 3; d++) w[d] = w[d] + wd[d] * dt;
    note_leaver(p, c, g, i, fl, x[0], x[1], x[2]);
    p.x[i] = x[0]; p.y[i] = x[1]; p.z[i] = x[2];
    p.vx[i] = v[0]; p.vy[i] = v[1]; p.vz[i] = v[2];
    p.wx[i] = w[0]; p.wy[i] = w[1]; p.wz[i] = w[2];
    for (int k = 0; k < 9; k++) p.rot_m[k * C + i] = R[k];
    for (int k = 0; k < 4; k++) p.rot_q[k * C + i] = q[k];
}

__global__ __launch_bounds__(256) void k_euler(DemPtrs p, int *__restrict__ c, DemGeom g, double dt) {
    const int nl = c[D_NLOCAL];
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nl || c[D_OVF]) return;
    const double f[3] = {p.fx[i], p.fy[i], p.fz[i]}, tq[3] = {p.tx[i], p.ty[i], p.tz[i]};
    euler_particle(p, c, g, dt, i, p.flags[i], f, tq);
}

// ---------------------------------------------------------------- contacts

struct Acc3 { double x, y, z; };

// linear_spring_dashpot (examples/dem.py:18-74) for one contact: normal n,
// penetration delta, contact point cp, history slot k (fresh: a new slot, whose
// history is zero and is not read); updates the slot and
// returns the contact's force F and torque term T = (cp - x_i) x F
__device__ __forceinline__ void spring_dashpot(const DemPtrs &p, const DemParams &prm, const DemRec &ri,
                                               const DemRec &rj, int i, int k, bool fresh, const double n[3],
                                               double delta, const double cp[3], double F[3], double T[3]) {
    const size_t a = (size_t) k * p.cap + i;
    const bool sticking = !fresh && p.c_stick[a] == 1;
    const double xi[3] = {ri.x, ri.y, ri.z}, xj[3] = {rj.x, rj.y, rj.z};
    const double vi[3] = {ri.vx, ri.vy, ri.vz}, vj[3] = {rj.vx, rj.vy, rj.vz};
    const double wi[3] = {ri.wx, ri.wy, ri.wz}, wj[3] = {rj.wx, rj.wy, rj.wz};
    double ai[3], aj[3], rel[3], reln[3], relt[3];
    for (int d = 0; d < 3; d++) { ai[d] = cp[d] - xi[d]; aj[d] = cp[d] - xj[d]; }
    double vwi[3], vwj[3];
    vwi[0] = vi[0] + (wi[1] * ai[2] - wi[2] * ai[1]);
    vwi[1] = vi[1] + (wi[2] * ai[0] - wi[0] * ai[2]);
    vwi[2] = vi[2] + (wi[0] * ai[1] - wi[1] * ai[0]);
    vwj[0] = vj[0] + (wj[1] * aj[2] - wj[2] * aj[1]);
    vwj[1] = vj[1] + (wj[2] * aj[0] - wj[0] * aj[2]);
    vwj[2] = vj[2] + (wj[0] * aj[1] - wj[1] * aj[0]);
    for (int d = 0; d < 3; d++) rel[d] = -(vwi[d] - vwj[d]);
    const double rn = (rel[0] * n[0] + rel[1] * n[1]) + rel[2] * n[2];
    for (int d = 0; d < 3; d++) { reln[d] = rn * n[d]; relt[d] = rel[d] - reln[d]; }
    const double relt_len = sqrt((relt[0] * relt[0] + relt[1] * relt[1]) + relt[2] * relt[2]);
    const bool cond_a = sticking && relt_len < 1e-08;
    const double meff = 1.0 / (1.0 / ri.m + 1.0 / rj.m);
    // stiffness from the collision time (examples/dem.py:34-35), or fixed
    const double kn = prm.kn_fixed > 0.0 ? prm.kn_fixed
                                         : (meff * (prm.pi * prm.pi + prm.ln_e * prm.ln_e)) / (prm.t_c * prm.t_c);
    const double kt = prm.kappa * kn;
    double h[3] = {0.0, 0.0, 0.0}, iv = 0.0;
    if (!fresh) {
        for (int d = 0; d < 3; d++) h[d] = p.c_tsd[(3 * (size_t) k + d) * p.cap + i];
        iv = p.c_ivm[a];
    }
    const double hn = (h[0] * n[0] + h[1] * n[1]) + h[2] * n[2];
    double rot[3], ntsd[3];
    for (int d = 0; d < 3; d++) rot[d] = h[d] - n[d] * hn;
    const double rot2 = (rot[0] * rot[0] + rot[1] * rot[1]) + rot[2] * rot[2];
    const double h2 = (h[0] * h[0] + h[1] * h[1]) + h[2] * h[2];
    const double scale = sqrt(h2 / rot2);
    for (int d = 0; d < 3; d++) ntsd[d] = prm.dt * relt[d] + ((rot2 <= 0.0) ? 0.0 : rot[d] * scale);
    // damping for the restitution coefficient: from the collision time
    // (examples/dem.py:36), or for the fixed stiffness
    const double dn = prm.kn_fixed > 0.0 ? ((-(2.0) * prm.ln_e) * sqrt(meff * kn)) / prm.sqrt_pl
                                         : ((-(2.0) * meff) * prm.ln_e) / prm.t_c;
    const double dtan = prm.sqrt_kappa * dn;
    double ftls[3];
    for (int d = 0; d < 3; d++) ftls[d] = kt * ntsd[d] + dtan * relt[d];
    const double ftls_len = sqrt((ftls[0] * ftls[0] + ftls[1] * ftls[1]) + ftls[2] * ftls[2]);
    const int tk = ri.type * prm.ntypes + rj.type;
    double fn[3];
    for (int d = 0; d < 3; d++) fn[d] = (kn * delta) * n[d] + dn * reln[d];
    const double fn_len = sqrt((fn[0] * fn[0] + fn[1] * fn[1]) + fn[2] * fn[2]);
    const double f_static = prm.mu_s[tk] * fn_len;
    const double f_dynamic = prm.mu_d[tk] * fn_len;
    const bool cond1 = cond_a && ftls_len < f_static;
    const bool cond2 = sticking && ftls_len < f_dynamic;
    const bool slide = (!cond1 && !cond2) && kt > 0.0;
    const double f_fric = cond1 ? f_static : f_dynamic;
    const double inv_len = 1.0 / ftls_len;
    double tdir[3];
    for (int d = 0; d < 3; d++) tdir[d] = (ftls_len > 0.0) ? ftls[d] * inv_len : 0.0;
    for (int d = 0; d < 3; d++)
        p.c_tsd[(3 * (size_t) k + d) * p.cap + i] = slide ? (f_fric * tdir[d] - dtan * relt[d]) / kt : ntsd[d];
    const double rel_len = sqrt((rel[0] * rel[0] + rel[1] * rel[1]) + rel[2] * rel[2]);
    p.c_ivm[a] = (iv > 0.0) ? iv : rel_len;
    p.c_stick[a] = ((cond1 || cond2) || ftls_len < f_dynamic) ? 1 : 0;
    const double ft_abs = (f_fric < ftls_len) ? f_fric : ftls_len;
    for (int d = 0; d < 3; d++) F[d] = fn[d] + ft_abs * tdir[d];
    const double c0 = cp[0] - xi[0], c1 = cp[1] - xi[1], c2 = cp[2] - xi[2];
    T[0] = c1 * F[2] - c2 * F[1];
    T[1] = c2 * F[0] - c0 * F[2];
    T[2] = c0 * F[1] - c1 * F[0];
}

// force += F, torque += T of one contact, in the caller's contact order
__device__ __forceinline__ void accumulate(Acc3 &fa, Acc3 &ta, const double F[3], const double T[3]) {
    fa.x = fa.x + F[0]; fa.y = fa.y + F[1]; fa.z = fa.z + F[2];
    ta.x = ta.x + T[0]; ta.y = ta.y + T[1]; ta.z = ta.z + T[2];
}

// contact slot of uid_j in i's history: the last match, or a new slot with
// zeroed history (src/pairs/mapping/funcs.py:230-270); marks it used
__device__ __forceinline__ int contact_slot(const DemPtrs &p, int *c, int i, int uid_j) {
    const int nc = p.num_contacts[i];
    int slot = -1;
    for (int k = 0; k < nc; k++)
        if (p.c_uid[(size_t) k * p.cap + i] == uid_j) slot = k;
    if (slot == -1) {
        if (nc >= p.ccap) {
            atomicMax(&c[D_REQ_CONTACT], nc + 1);
            atomicMax(&c[D_OVF], DOVF_CONTACT);
            return -1;
        }
        slot = nc;
        p.num_contacts[i] = nc + 1;
        const size_t a = (size_t) slot * p.cap + i;
        p.c_uid[a] = uid_j;
        p.c_stick[a] = 0;
        p.c_tsd[3 * (size_t) slot * p.cap + i] = 0.0;
        p.c_tsd[(3 * (size_t) slot + 1) * p.cap + i] = 0.0;
        p.c_tsd[(3 * (size_t) slot + 2) * p.cap + i] = 0.0;
        p.c_ivm[a] = 0.0;
    }
    p.c_used[(size_t) slot * p.cap + i] = 1;
    return slot;
}

// contact test of i (position xi, radius ri) against a sphere (xj, rj), as
// linear_spring_dashpot's guard (examples/dem.py:18-30 with the sphere
// geometry of src/pairs/sim/interaction.py); on contact fills the normal, the
// contact point and the penetration depth
__device__ __forceinline__ bool sphere_contact(const double xi[3], double ri, const double xj[3], double rj,
                                               double nv[3], double cpt[3], double &delta) {
    const double d[3] = {xi[0] - xj[0], xi[1] - xj[1], xi[2] - xj[2]};
    const double rsq = (d[0] * d[0] + d[1] * d[1]) + d[2] * d[2];
    const double rs = ri + rj;
    if (!(rsq < rs * (rs + 0.0))) return false;
    const double dist = sqrt(rsq);
    const double pen = (dist - ri) - rj;
    delta = -(pen);
    if (delta < 0.0) return false;
    const double inv = 1.0 / dist;
    for (int e = 0; e < 3; e++) nv[e] = d[e] * inv;
    const double reach = rj + 0.5 * pen;
    for (int e = 0; e < 3; e++) cpt[e] = xj[e] + nv[e] * reach;
    return true;
}

// the same against half-space j at xj
__device__ __forceinline__ bool plane_contact(const DemPtrs &p, const double xi[3], double ri, int j,
                                              const double xj[3], double nv[3], double cpt[3], double &delta) {
    const double nj[3] = {p.nx[j], p.ny[j], p.nz[j]};
    const double pen = (((nj[0] * xi[0] + nj[1] * xi[1]) + nj[2] * xi[2]) - ri) -
                       ((nj[0] * xj[0] + nj[1] * xj[1]) + nj[2] * xj[2]);
    if (!(pen < 0.0)) return false;
    delta = -(pen);
    if (delta < 0.0) return false;
    const double reach = ri + pen;
    for (int e = 0; e < 3; e++) { nv[e] = nj[e]; cpt[e] = xi[e] - reach * nj[e]; }
    return true;
}

__device__ __forceinline__ bool contact_geom(const DemPtrs &p, const double xi[3], double ri, int j, const DemRec &rj,
                                             int pass, double nv[3], double cpt[3], double &delta) {
    const double xj[3] = {rj.x, rj.y, rj.z};
    return pass == 0 ? sphere_contact(xi, ri, xj, rj.r, nv, cpt, delta) : plane_contact(p, xi, ri, j, xj, nv, cpt, delta);
}

// Candidates of i in the reference's visiting order: the spheres of cell 0
// and of the 27 stencil cells, then the half-spaces of the same cells
// (cell_lists.py partitions each cell spheres-first).  fn(j, pass) is called
// for each candidate j != i and returns false to stop the walk.
template <typename F>
__device__ __forceinline__ void walk_candidates(const DemPtrs &p, const DemGeom &g, int i, int ci, F &&fn) {
    for (int pass = 0; pass < 2; pass++) {
        for (int s = -1; s < 27; s++) {
            const int cell = s < 0 ? 0 : ci + g.stencil[s];
            if (!(s < 0 || (cell > 0 && cell < g.ncells))) continue;
            for (int q = p.cell_start[cell]; q < p.cell_start[cell + 1]; q++) {
                const int j = p.corder[q].x;
                if (j == i || p.shape[j] != pass) continue;
                if (!fn(j, pass)) return;
            }
        }
    }
}

// inclusive sum over each group of W lanes
template <int W>
__device__ __forceinline__ int group_scan(int x) {
    const int l = threadIdx.x & (W - 1);
#pragma unroll
    for (int off = 1; off < W; off <<= 1) {
        const int y = __shfl_up(x, off, W);
        if (l >= off) x += y;
    }
    return x;
}

// Contact search, LPS lanes per local sphere, spheres in cell order (the
// groups of a wave are neighbours and read the same records).  The visiting
// order's 28 cells (cell 0, then the 27 stencil cells) are ten runs of the
// cell order: cell 0, and the three cells of each of the nine z-columns, which
// are consecutive.  Lane l finds the bounds of column l, lane 0 those of cell 0
// and lane 7 those of the last column too; the runs are laid end to end in LDS
// (a window of FIND_WIN candidates at a time) and the lanes take the candidates
// in turn, so that all have the same number whatever the runs' lengths.  A
// group's part of the wave's ballot gives every hit its place in the visiting
// order (all spheres, then all half-spaces); they are stored to cand[i][t]
// (half-spaces as ~j).
// cand_n[i] = DCAND + 1 when more than DCAND touch (the contact kernel then
// walks the cells itself).  Only geometry is read: no history is touched.
// Bound by vector work, then by the latency of its dependent loads (place, run
// bounds, candidates).  Bed of 187200 spheres | 200000 falling, us: by particle
// index, cell by cell, from four arrays 105 | 59; a lane per column of the
// the ordered records, as slow as its longest column, 41 | 28; so 31 | 25.
constexpr int LPS = 8, FIND_WIN = 64;
__global__ __launch_bounds__(256) void k_contact_find(DemPtrs p, const int *__restrict__ c, DemGeom g) {
    constexpr int GROUPS = 256 / LPS;
    __shared__ int s_place[GROUPS][FIND_WIN + 1];
    __shared__ int s_hit[GROUPS][DCAND + 1], s_wall[GROUPS][DCAND + 1];
    if (c[D_OVF]) return;
    const int nl = c[D_NLOCAL], n = nl + c[D_NGHOST];
    const int q0 = (blockIdx.x * 256 + threadIdx.x) / LPS;
    const int l = threadIdx.x & (LPS - 1), grp = threadIdx.x / LPS;
    const bool in = q0 < n;
    if (!__ballot(in)) return;
    const int qi = in ? q0 : 0;
    const int2 own = p.corder[qi];
    const int i = own.x, cc = own.y;
    const double4 me = p.crec[qi];
    const bool act = in && i < nl, look = act && cc >= 0;
    const int ci = cc & 0x7fffffff;
    // the lane's two runs [st, st + len)
    int st[2] = {0, 0}, len[2] = {0, 0};
    auto column = [&](int col, int &s0, int &ln) {
        const int base = ci + g.stencil[3 * col + 1];
        const int lo = max(base - 1, 1), hi = min(base + 1, g.ncells - 1);
        if (lo <= hi) {
            s0 = p.cell_start[lo];
            ln = p.cell_start[hi + 1] - s0;
        }
    };
    if (look) {
        if (l == 0) { st[0] = p.cell_start[0]; len[0] = p.cell_start[1] - st[0]; }
        column(l, st[1], len[1]);
        if (l == LPS - 1) {
            st[0] = st[1]; len[0] = len[1];
            column(LPS, st[1], len[1]);
        }
    }
    const double xi[3] = {me.x, me.y, me.z};
    // a half-space that is not FIXED looks for partners itself, as a point of its own radius
    const double ri = me.w == PLANE_MARK ? p.r[i] : me.w;
    const int upto = group_scan<LPS>(len[0] + len[1]);
    const int total = __shfl(upto, LPS - 1, LPS);
    const int at[2] = {upto - len[0] - len[1], upto - len[1]};  // the runs' first candidates
    // 0: no contact, 1: sphere, 2: half-space
    auto touch = [&](int q, const double4 &r) {
        double nv[3], cpt[3], delta;
        const double xj[3] = {r.x, r.y, r.z};
        if (q == qi) return 0;
        if (r.w != PLANE_MARK) {
            // sqrt(d2) - ri - rj <= 0 without the root where d2 is below (ri +
            // rj)^2 by more than 1e-12 of it (the rounding errors are 1e-15)
            const double d0 = xi[0] - xj[0], d1 = xi[1] - xj[1], d2 = xi[2] - xj[2], rs = ri + r.w;
            const double dd = (d0 * d0 + d1 * d1) + d2 * d2, rr = rs * rs;
            if (ri >= 0.0 && r.w >= 0.0 && rr > 1e-280 && dd < rr * (1.0 - 1e-12)) return 1;
            return sphere_contact(xi, ri, xj, r.w, nv, cpt, delta) ? 1 : 0;
        }
        return plane_contact(p, xi, ri, p.corder[q].x, xj, nv, cpt, delta) ? 2 : 0;
    };
    const int shift = (threadIdx.x & 63) & ~(LPS - 1);
    const unsigned below = (1u << l) - 1u;
    int ns = 0, nh = 0;  // hits of the group
    for (int w0 = 0; __ballot(w0 < total); w0 += FIND_WIN) {
#pragma unroll
        for (int e = 0; e < 2; e++)
            for (int k = max(0, w0 - at[e]); k < min(len[e], w0 + FIND_WIN - at[e]); k++)
                s_place[grp][at[e] + k - w0] = st[e] + k;
        wave_lds_sync();
        const int m = min(total - w0, FIND_WIN);
        for (int b = 0; __ballot(b < m); b += 2 * LPS) {
            const int ba = b + l, bb = b + LPS + l;
            const bool ina = ba < m, inb = bb < m;
            const int qa = ina ? s_place[grp][ba] : qi, qb = inb ? s_place[grp][bb] : qi;
            const double4 ra = p.crec[qa], rb = p.crec[qb];
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int q = e == 0 ? qa : qb;
                const int t = touch(q, e == 0 ? ra : rb);  // none for its own record
                const unsigned sph = (unsigned) (__ballot(t == 1) >> shift) & 0xffu;
                if (t == 1) {
                    const int r = ns + __popc(sph & below);
                    if (r < DCAND) s_hit[grp][r] = q;
                }
                ns += __popc(sph);
                const unsigned long long walls = __ballot(t == 2);
                if (walls) {
                    const unsigned pl = (unsigned) (walls >> shift) & 0xffu;
                    if (t == 2) {
                        const int r = nh + __popc(pl & below);
                        if (r < DCAND) s_wall[grp][r] = q;
                    }
                    nh += __popc(pl);
                }
            }
        }
        wave_lds_sync();
    }
    const int nt = ns + nh;
    if (!act) return;
    if (nt <= DCAND)
        for (int t = l; t < nt; t += LPS) {
            const int j = p.corder[t < ns ? s_hit[grp][t] : s_wall[grp][t - ns]].x;
            p.cand[(size_t) i * DCAND + t] = t < ns ? j : ~j;
        }
    if (l == 0) p.cand_n[i] = nt <= DCAND ? nt : DCAND + 1;
}

// The contacts of SPW consecutive local particles, one wave.  The wave's
// contacts are numbered particle by particle in visiting order and dealt to
// the lanes densely, 64 at a time, whichever particle they belong to:
//  1. each contact looks its partner's uid up in its particle's history
//     (reset_contact_history_usage_status and the slot rule of
//     src/pairs/mapping/funcs.py:230-270: the last match, or a new slot); the
//     particle's lane numbers the new slots in order;
//  2. linear_spring_dashpot per contact, history updated, force and torque
//     terms through LDS; the particle's lane adds them in contact order, with
//     the reference's sphere / half-space grouping (force += sphere + plane
//     sums, torque += plane + sphere sums) on top of gravity;
//  3. clear_unused_contact_history from the particle's mask of used slots;
//  4. EULER: the particle integrated (nothing here reads another particle's
//     position but from the records made before).
// A particle with more than DCAND touching partners, more history than the
// mask holds, or two contacts in one slot (a partner and its image) walks its
// cells in its lane instead, one contact after the other, as the reference.
// Bound by the gathers of the partners' records (0.9 M of 128 bytes in a bed of
// 187200 spheres) and the FP64 divisions and roots of the contact law.  One
// dense pass in place of a kernel per phase: the phases ran one thread per
// possible contact (16 per particle) or per particle, and gathered a partner
// from twelve arrays: 134 -> 53 us in that bed, 29 -> 11 us at 2080 spheres;
// eight history slots compared at a time 53 -> 48.  With the integration 60,
// for 48 and 18 us apart; 12.0 for 10.8 and 4.3 at 2080 spheres.
template <int SPW, bool EULER>
__global__ __launch_bounds__(64) void k_contact_solve(DemPtrs p, int *__restrict__ c, DemGeom g, DemParams prm) {
    __shared__ double s_term[64][7];
    __shared__ int s_kind[64];
    __shared__ int s_off[SPW], s_nc[SPW];
    __shared__ int s_cand[SPW * DCAND], s_uid[SPW * DCAND], s_slot[SPW * DCAND];
    __shared__ unsigned char s_own[SPW * DCAND];
    if (c[D_OVF]) return;
    const int nl = c[D_NLOCAL];
    const int i0 = blockIdx.x * SPW, lane = threadIdx.x;
    if (i0 >= nl) return;
    const int i = i0 + lane;
    const bool sph = lane < SPW && i < nl;
    const size_t C = p.cap;
    int nc = 0, nt = 0;
    if (sph) { nc = p.num_contacts[i]; nt = p.cand_n[i]; }
    const int nc0 = nc;
    bool slow = nt > DCAND || nc + nt > 64;
    const int n = slow ? 0 : nt;
    int off = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(off, o, 64);
        if (lane >= o) off += y;
    }
    const int total = __shfl(off, 63, 64);
    off -= n;
    if (lane < SPW) { s_off[lane] = off; s_nc[lane] = nc0; }
    for (int t = 0; t < n; t++) s_own[off + t] = (unsigned char) lane;
    __syncthreads();
    for (int k = lane; k < total; k += 64) {
        const int s = s_own[k], ii = i0 + s;
        const int e = p.cand[(size_t) ii * DCAND + (k - s_off[s])];
        const int uid = p.rec[e < 0 ? ~e : e].uid;
        const int m = s_nc[s];
        int slot = -1;
        for (int h0 = 0; h0 < m; h0 += 8) {
            int u[8];
#pragma unroll
            for (int v = 0; v < 8; v++) u[v] = p.c_uid[min(h0 + v, m - 1) * C + ii];
#pragma unroll
            for (int v = 0; v < 8; v++)
                if (h0 + v < m && u[v] == uid) slot = h0 + v;
        }
        s_cand[k] = e;
        s_uid[k] = uid;
        s_slot[k] = slot;
    }
    __syncthreads();
    unsigned long long used = 0ull;
    if (n > 0) {
        // two contacts in one slot: not independent
        bool fresh = false;
        for (int t = 0; t < n; t++) {
            const int slot = s_slot[off + t];
            if (slot < 0) { fresh = true; continue; }
            if (used >> slot & 1ull) slow = true;
            used |= 1ull << slot;
        }
        if (fresh)
            for (int t = 1; t < n; t++)
                for (int u = 0; u < t; u++)
                    if (s_slot[off + t] < 0 && s_slot[off + u] < 0 && s_uid[off + t] == s_uid[off + u]) slow = true;
        if (slow) {
            for (int t = 0; t < n; t++) s_slot[off + t] = -1;
        } else if (fresh) {
            for (int t = 0; t < n; t++) {
                if (s_slot[off + t] >= 0) continue;
                if (nc >= p.ccap) {
                    atomicMax(&c[D_REQ_CONTACT], nc + 1);
                    atomicMax(&c[D_OVF], DOVF_CONTACT);
                    continue;
                }
                s_slot[off + t] = nc;
                used |= 1ull << nc;
                nc++;
            }
        }
    }
    __syncthreads();
    Acc3 fs = {0.0, 0.0, 0.0}, fp = {0.0, 0.0, 0.0}, ts = {0.0, 0.0, 0.0}, tp = {0.0, 0.0, 0.0};
    for (int k0 = 0; k0 < total; k0 += 64) {
        const int k = k0 + lane;
        int kind = 2;
        if (k < total && s_slot[k] >= 0) {
            const int s = s_own[k], ii = i0 + s, slot = s_slot[k];
            const int e = s_cand[k], j = e < 0 ? ~e : e;
            const DemRec ri = p.rec[ii], rj = p.rec[j];
            const double xi[3] = {ri.x, ri.y, ri.z};
            const bool fresh = slot >= s_nc[s];
            double nv[3], cpt[3], delta, F[3], T[3];
            if (contact_geom(p, xi, ri.r, j, rj, e < 0 ? 1 : 0, nv, cpt, delta)) {
                spring_dashpot(p, prm, ri, rj, ii, slot, fresh, nv, delta, cpt, F, T);
                if (fresh) p.c_uid[slot * C + ii] = s_uid[k];
                for (int d = 0; d < 3; d++) { s_term[lane][d] = F[d]; s_term[lane][3 + d] = T[d]; }
                kind = e < 0 ? 1 : 0;
            }
        }
        s_kind[lane] = kind;
        __syncthreads();
        for (int q = max(off, k0); q < min(off + n, k0 + 64); q++) {
            const double *t = s_term[q - k0];
            const int kd = s_kind[q - k0];
            const double F[3] = {t[0], t[1], t[2]}, T[3] = {t[3], t[4], t[5]};
            if (kd == 0) accumulate(fs, ts, F, T);
            else if (kd == 1) accumulate(fp, tp, F, T);
        }
        __syncthreads();
    }
    if (!sph) return;
    double f0 = 0.0, f1 = 0.0, f2 = 0.0, t0 = 0.0, t1 = 0.0, t2 = 0.0;
    if (slow) {
        for (int k = 0; k < nc0; k++) p.c_used[k * C + i] = 0;
        p.num_contacts[i] = nc0;
    }
    const int fl = p.flags[i];
    if (!(fl & DFLAG_FIXED)) {
        // gravity (examples/dem.py:88-90)
        const double ri = p.r[i];
        const double vol = (((4.0 / 3.0) * prm.pi) * ri * ri) * ri;
        f2 = f2 - (prm.drho * vol) * prm.grav;
        if (slow) {
            const DemRec me = p.rec[i];
            const double xi[3] = {me.x, me.y, me.z};
            walk_candidates(p, g, i, p.particle_cell[i], [&](int j, int pass) {
                double nv[3], cpt[3], delta, F[3], T[3];
                const DemRec rj = p.rec[j];
                if (!contact_geom(p, xi, ri, j, rj, pass, nv, cpt, delta)) return true;
                const int slot = contact_slot(p, c, i, rj.uid);
                if (slot < 0) return true;
                spring_dashpot(p, prm, me, rj, i, slot, false, nv, delta, cpt, F, T);
                if (pass == 0) accumulate(fs, ts, F, T);
                else accumulate(fp, tp, F, T);
                return true;
            });
        }
        f0 = f0 + (fs.x + fp.x); f1 = f1 + (fs.y + fp.y); f2 = f2 + (fs.z + fp.z);
        t0 = t0 + (tp.x + ts.x); t1 = t1 + (tp.y + ts.y); t2 = t2 + (tp.z + ts.z);
    }
    p.fx[i] = f0; p.fy[i] = f1; p.fz[i] = f2;
    p.tx[i] = t0; p.ty[i] = t1; p.tz[i] = t2;
    // clear_unused_contact_history (src/pairs/sim/contact_history.py:91-127)
    if (slow) nc = p.num_contacts[i];
    int k = 0;
    while (k < nc) {
        const size_t a = k * C + i;
        if (slow ? p.c_used[a] == 0 : !(used >> k & 1ull)) {
            const int last = nc - 1;
            if (last > 0) {
                const size_t b = last * C + i;
                p.c_stick[a] = p.c_stick[b];
                for (int d = 0; d < 3; d++) p.c_tsd[(3 * (size_t) k + d) * C + i] = p.c_tsd[(3 * (size_t) last + d) * C + i];
                p.c_ivm[a] = p.c_ivm[b];
                p.c_uid[a] = p.c_uid[b];
                if (slow) p.c_used[a] = p.c_used[b];
                else used = (used & ~(1ull << k)) | (used >> last & 1ull) << k;
            }
            nc = nc - 1;
        } else {
            k++;
        }
    }
    p.num_contacts[i] = nc;
    if (EULER) {
        const double f[3] = {f0, f1, f2}, tq[3] = {t0, t1, t2};
        euler_particle(p, c, g, prm.dt, i, fl, f, tq);
    }
}

// update_mass_and_inertia (examples/dem.py:6-15)
__global__ __launch_bounds__(256) void k_mass_inertia(DemPtrs p, int nl) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nl) return;
    const size_t C = p.cap;
    for (int k = 0; k < 9; k++) p.rot_m[k * C + i] = (k % 4 == 0) ? 1.0 : 0.0;
    p.rot_q[i] = 1.0; p.rot_q[C + i] = 0.0; p.rot_q[2 * C + i] = 0.0; p.rot_q[3 * C + i] = 0.0;
    if (p.shape[i] == DSHAPE_SPHERE) {
        double a = 0.4 * p.m[i];
        a = a * p.r[i];
        a = a * p.r[i];
        const double M[9] = {a, 0.0, 0.0, 0.0, a, 0.0, 0.0, 0.0, a};
        double det = M[0] * (M[4] * M[8] - M[7] * M[5]);
        det = det + M[1] * (M[5] * M[6] - M[8] * M[3]);
        det = det + M[2] * (M[3] * M[7] - M[4] * M[6]);
        const double id = 1.0 / det;
        const double inv[9] = {id * (M[4] * M[8] - M[5] * M[7]), id * (M[7] * M[2] - M[8] * M[1]),
                               id * (M[1] * M[5] - M[2] * M[4]), id * (M[5] * M[6] - M[3] * M[8]),
                               id * (M[8] * M[0] - M[6] * M[2]), id * (M[2] * M[3] - M[0] * M[5]),
                               id * (M[3] * M[7] - M[4] * M[6]), id * (M[6] * M[1] - M[7] * M[0]),
                               id * (M[0] * M[4] - M[1] * M[3])};
        for (int k = 0; k < 9; k++) p.inv_i[k * C + i] = inv[k];
    } else {
        p.m[i] = __longlong_as_double(0x7ff0000000000000LL);  // +infinity
        for (int k = 0; k < 9; k++) p.inv_i[k * C + i] = 0.0;
    }
}

// ---------------------------------------------------------------- launchers

static int grid_of(int n, int bs) { return n <= 0 ? 1 : (n + bs - 1) / bs; }

void launch_fill(hipStream_t s, int *p, int v, int n) {
    hipLaunchKernelGGL(k_fill_i32, dim3(std::max(1, std::min(grid_of(n, 256), 4096))), dim3(256), 0, s, p, v, n);
}

void launch_mass_inertia(hipStream_t s, const DemPtrs &p, int nl) {
    hipLaunchKernelGGL(k_mass_inertia, dim3(grid_of(nl, 256)), dim3(256), 0, s, p, nl);
}

template <int ND>
static void launch_borders(hipStream_t s, const DemPtrs &p, int *c, const DemGeom &g) {
    const int nb = grid_of(p.cap, 256);
    hipLaunchKernelGGL(k_cell_count<ND>, dim3(nb), dim3(256), 0, s, p, c, g, nb);
    if constexpr (ND > 0) hipLaunchKernelGGL(k_border_ghosts<ND>, dim3(nb), dim3(256), 0, s, p, c, g, nb);
}

void launch_find_leavers(hipStream_t s, const DemPtrs &p, int *c, const DemGeom &g) {
    if (!g.periodic[0] && !g.periodic[1] && !g.periodic[2]) return;
    launch_fill(s, c + D_LEAVE, 0, 1);
    hipLaunchKernelGGL(k_find_leavers, dim3(grid_of(p.cap, 256)), dim3(256), 0, s, p, c, g);
}

// exchange, borders, cells of one step (the cell counts are zero on entry:
// allocated zeroed, cleared by every scan); one rank: only the periodic
// dimensions send
void launch_prepare(hipStream_t s, const DemPtrs &p, int *c, const DemGeom &g) {
    const int nd = g.periodic[0] + g.periodic[1] + g.periodic[2];
    if (nd > 0) hipLaunchKernelGGL(k_exchange, dim3(1), dim3(1024), 0, s, p, c, g);
    if (nd == 0) launch_borders<0>(s, p, c, g);
    else if (nd == 1) launch_borders<1>(s, p, c, g);
    else if (nd == 2) launch_borders<2>(s, p, c, g);
    else launch_borders<3>(s, p, c, g);
    // (one entry past the cells, whose count stays zero: cell_start[ncells] is the total)
    const int n = g.ncells + 1, nb = grid_of(n, 1024), pg = grid_of(p.cap, 256);
    hipLaunchKernelGGL(k_scan_partial, dim3(nb), dim3(1024), 0, s, p.cell_count, p.cell_scan, p.scan_tmp, n);
    if (nb <= SCAN_LDS) {
        hipLaunchKernelGGL(k_cell_fill<true>, dim3(pg), dim3(256), 0, s, p, c, n, nb);
    } else {
        hipLaunchKernelGGL(k_scan_add, dim3(nb), dim3(1024), 0, s, p.cell_scan, p.cell_start, p.scan_tmp, n);
        hipLaunchKernelGGL(k_cell_fill<false>, dim3(pg), dim3(256), 0, s, p, c, n, nb);
    }
    hipLaunchKernelGGL(k_cell_order, dim3(pg), dim3(256), 0, s, p, c);
}

template <bool EULER>
static void launch_solve(hipStream_t s, const DemPtrs &p, int *c, int nlocal, const DemGeom &g, const DemParams &prm) {
    // particles per wave: a wave's chain of look-ups is shorter with fewer (a
    // small system is one wave of the chip long), its lanes fuller with more:
    // beds of 2080 / 9600 / 39200 / 187200 spheres, ms a pass on 8, 16, 32:
    // 16.1 16.8 17.8 / 4.58 4.76 4.99 / 6.41 6.24 6.45 / 28.8 27.3 26.4
    const int spw = nlocal < 16384 ? 8 : nlocal < 65536 ? 16 : 32;
    const dim3 grid(grid_of(nlocal, spw));
    if (spw == 8) hipLaunchKernelGGL((k_contact_solve<8, EULER>), grid, dim3(64), 0, s, p, c, g, prm);
    else if (spw == 16) hipLaunchKernelGGL((k_contact_solve<16, EULER>), grid, dim3(64), 0, s, p, c, g, prm);
    else hipLaunchKernelGGL((k_contact_solve<32, EULER>), grid, dim3(64), 0, s, p, c, g, prm);
}

// forces, history bookkeeping and integration
void launch_contacts(hipStream_t s, const DemPtrs &p, int *c, int nlocal, const DemGeom &g, const DemParams &prm,
                     const hipEvent_t *between) {
    hipLaunchKernelGGL(k_contact_find, dim3(grid_of(p.cap, 256 / LPS)), dim3(256), 0, s, p, c, g);
    if (between) hipEventRecord(between[0], s);
    if (between) launch_solve<false>(s, p, c, nlocal, g, prm);
    else launch_solve<true>(s, p, c, nlocal, g, prm);
    if (between) hipEventRecord(between[1], s);
}

void launch_euler(hipStream_t s, const DemPtrs &p, int *c, const DemGeom &g, const DemParams &prm) {
    hipLaunchKernelGGL(k_euler, dim3(grid_of(p.cap, 256)), dim3(256), 0, s, p, c, g, prm.dt);
}

}  // namespace dk
