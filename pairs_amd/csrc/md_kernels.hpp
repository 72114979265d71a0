// Device state and launchers of the LJ molecular-dynamics path.
//
// Storage layout in HBM.  Particles live in "physical" slots: locals first,
// sorted by cell, then ghosts, sorted by cell; every per-particle array is SoA
// (x, y, z, vx, ..., one array per component).  The reference's own particle
// index ("reference index": the slot the generated CPU program would use) is
// kept as a relabeling, ref[physical] and phys[reference], updated exactly as
// the reference's exchange and borders would move particles; every
// order-dependent rule (exchange tail fill, ghost order, cell order, half-list
// i < j, neighbour order) is applied to reference indices.  Positions are
// double-buffered (X[2], Y[2], Z[2]) so that the fused force/integrate kernel
// never overwrites a position another thread gathers.
//
// Work decomposition.  The neighbour build works on "segments": ZC
// consecutive cells of one z-column of the cell grid, whose home particles
// are one contiguous range of physical local slots, and whose candidate cells
// (cell 0 plus the 3x3 columns around it, z range widened by one) are 20
// contiguous physical runs: the segment's tile, staged in LDS once and shared
// by all its home particles.  Neighbour lists hold physical slots (32 bits),
// in the reference's candidate order.  The force kernels work on "waves" of 2
// to 64 consecutive physical locals, 32 lanes to one lane per local by the size
// of the system, gathering neighbour positions from a packed (x, y, z, type) copy
// of the position buffer; large systems of one type stage them in LDS, a tile
// per group of locals.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

#include "common.hpp"

namespace pk {

enum { FLAG_INFINITE = 1, FLAG_GHOST = 2, FLAG_FIXED = 4, FLAG_GLOBAL = 8 };
enum { SHAPE_SPHERE = 0, SHAPE_HALFSPACE = 1, SHAPE_POINT_MASS = 2 };

// device-resident counters (read by kernels so launches need no host round trip)
enum {
    C_NLOCAL = 0,
    C_NGHOST = 1,
    C_NSEND_ALL = 2,
    C_NSEND = 3,  // 6 entries: per dimension, side 0 then side 1
    C_RANGE = 9,  // particle range of the current compaction
    C_BASE0 = 10,
    C_BASE1 = 11,
    C_OVF = 12,   // first overflow kind (0 = none)
    C_REQ_NEIGH = 13,
    C_REQ_SEND = 14,
    C_REQ_PART = 15,
    C_TILE_MAX = 16,  // largest segment tile of the current lists
    C_UNSUPPORTED = 17,
    C_IMG_OVF = 18,   // a local has more periodic images than IMG_MAX
    C_LEAVE = 19,     // locals outside a periodic dimension, listed for the exchange
    C_LEAVE_MAX = 20, // their number at the last exchange
    C_NGROUPS = 21,   // groups of the force tiles
    C_BIG = 22,       // those whose tile does not fit
    C_COUNT = 23
};
enum { OVF_NONE = 0, OVF_PART = 1, OVF_NEIGH = 2, OVF_SEND = 3, OVF_TILE = 4 };

// cell grid and domain, passed by value
struct Geom {
    double lo[3], hi[3], len[3];
    double spacing;
    int dim_cells[3];
    int ncells;
    int nstencil;
    int stencil[27];
    int zc;        // cells per segment along z
    int nchunks;   // segments per z-column
    int nsegs;     // dim_cells[0] * dim_cells[1] * nchunks
};

// Neighbour lists: entry k of physical local i.  Rows come in groups of four
// so that one 16-byte load gives a lane four consecutive entries; a group
// holds, for every particle, its four entries side by side in the order 0, 2,
// 1, 3 (list_pos): the halves of a group are then the entries that one lane
// pair of the force kernel takes, so that its two pairs gather consecutive
// entries -- often records of one cache line -- with one instruction.
__host__ __device__ __forceinline__ int list_pos(int k) { return ((k & 1) << 1) | ((k >> 1) & 1); }
__host__ __device__ __forceinline__ size_t nl_at(int k, int i, int nl_stride) {
    return ((size_t) (k >> 2) * nl_stride + i) * 4 + list_pos(k);
}

// list rows are allocated in multiples of this: the force kernel reads a
// local's list up to 32 rows at a time, by whole rounds
constexpr int LIST_ROWS = 32;
__host__ __device__ __forceinline__ int list_rows(int ncap) { return (ncap + LIST_ROWS - 1) / LIST_ROWS * LIST_ROWS; }

// force tiles: locals of a group, cells it spans, particles of a tile (six
// tiles in a CU's LDS)
constexpr int TILE_G = 128;
constexpr int TILE_SPAN = 8;
constexpr int TILE_CAP = 1088;
// the local of a group of n whose list thread t of the force kernel walks: its
// own, or, without one, its wave's first (a local's 16-bit rows are padded to
// the depth of its own wave, and not further)
__host__ __device__ __forceinline__ int tile_lane_row(int t, int n) {
    if (t < n) return t;
    const int first = t & ~63;
    return first < n ? first : n - 1;
}

constexpr int IMG_MAX = 8;
// leavers that the one-workgroup exchange takes from its list
constexpr int LEAVE_CAP = 4096;
// ghost kinds: per periodic dimension none, side 0 or side 1
constexpr int MAX_KIND = 27;

// The runs of a group's candidate cells as the tile build searches them: sorted
// by first slot, so that a slot's place among the candidates is that of the last
// run that begins at or before it.  Runs of neighbouring columns may overlap (a
// column's range of flat cells reaches into the next column's first cell), and
// then begin at one slot where the cells between are empty: the longer of them
// comes last, as it holds all of the shorter.
constexpr int NRUNS = 20;
// run t's rank among the runs that are not empty (off: their exclusive sums)
__host__ __device__ __forceinline__ int tile_run_rank(const int *start, const int *off, int t) {
    const int len = off[t + 1] - off[t];
    int rank = 0;
    for (int k = 0; k < NRUNS; k++) {
        const int n = off[k + 1] - off[k];
        if (n == 0 || start[k] > start[t]) continue;
        rank += start[k] < start[t] || n < len || (n == len && k < t) ? 1 : 0;
    }
    return rank;
}
// slot j's place (from, delta by rank: first slot, place minus slot; from is
// the largest number behind the last)
__host__ __device__ __forceinline__ int tile_place(const int *from, const int *delta, int j) {
    int p = 0;
#pragma unroll
    for (int s = 16; s > 0; s >>= 1) p += from[p + s] <= j ? s : 0;
    return j + delta[p];
}

// what a position-advancing kernel needs to refresh the ghost images
struct Images {
    const int *cnt;
    const int4 *tab;
    int cap, on;
};

struct LJTab {
    int nt;
    int unit;  // one type with epsilon = sigma6 = 1
    double eps[16], sig6[16];  // ntypes <= 4
};

struct LJParams {
    double rc2, dt, hdt;
    int ntypes;
    double eps[16], sig6[16];
};

struct DevState {
    int cap, ncap, send_cap, ncells_cap, nl_stride;
    int nlocal;   // host mirror (constant between uploads on one domain)
    int cur;      // which position buffer holds the current state
    int tile_cap; // LDS tile entries the neighbour build may stage
    int pstride;  // row stride of the partials array
    int max_lds;  // shared memory a workgroup may allocate
    double *X[2], *Y[2], *Z[2];
    double4 *P[2];       // (x, y, z, type) of each position buffer, packed for the force kernels' gathers; one
                         // more record, at the origin, for padded list entries
    double *vx, *vy, *vz, *fx, *fy, *fz, *mass;
    int *type, *flags, *uid, *shape, *ref;
    int *phys;    // physical slot of each reference index
    // spare arrays the rebuild permutes into (swapped with the live ones)
    double *alt_vx, *alt_vy, *alt_vz, *alt_mass;
    int *alt_type, *alt_flags, *alt_uid, *alt_shape, *alt_ref, *alt_cell;
    int *numneighs;
    uint32_t *nl;  // entry k of physical local i at nl_at(k, i, nl_stride): physical slot
    // half lists: rows [rev0, 2 rev0) hold each local's mirror part (the
    // earlier-index locals whose half list holds it, by reference index);
    // rev0 = 0 for full lists
    int rev0;
    int *nrev;
    int *particle_cell, *slot, *perm;
    int *lcount, *gcount, *lstart, *gstart;  // per-cell counts and CSR starts (locals / ghosts)
    int *send_map, *send_mult, *exchg_flag;
    int *sync_src;       // per ghost (physical order): physical source slot
    int *sync_mult;      // per ghost (physical order): 3 image multipliers
    // periodic images of each local (its ghosts, and ghosts of those): the
    // kernel that advances a local's position also writes its images' next
    // positions, so no separate ghost refresh runs between steps
    int *img_cnt;        // per physical local
    int4 *img_tab;       // [k][cap]: image k's ghost index (physical - nlocal), its source slot (-1: the
                         // local itself), its shift (2 bits per dimension, + 1)
    int img_on;          // host: every local's images fit IMG_MAX
    // force tiles of a large system (k_ljt): a group's locals and its tile's
    // size (0: does not fit), the tile's slots, the lists as offsets into it
    int tiles;           // host: the neighbour build makes them
    int tile_gmax;
    int4 *tile_grp, *tile_tab;
    int *tile_slots;
    uint4 *nl16;
    int *tile_cnt;
    int *leavers;        // [LEAVE_CAP] physical slots
    int exch_listed;     // host: the exchange works from the list of leavers
    int *counters;
    int *scratch_i;      // 4 * send_cap
    double *stage;       // 10 * send_cap doubles
    double *partials;    // 3 rows of pstride: per force wave (kinetic, energy, virial)
    double *thermo;      // 5 per thermo record
};

void launch_fill_i32(hipStream_t s, int *p, int v, int n);
// P[cur] = (X[cur], Y[cur], Z[cur], 0) for locals and ghosts
void launch_pack_p(hipStream_t s, const DevState &d, int cur);
// waves of the force kernels: 64 locals each
int force_waves(const DevState &d);
// waves of the timestep's LJ force kernel (two to 32 lanes per local)
int lj_waves(const DevState &d);
// the older API's modules (examples/lj_onetype.py): forces with its pair
// expression (full lists), and its Euler update in the current buffer
void launch_lj_older(hipStream_t s, const DevState &d, const Geom &g, const LJParams &prm);
void launch_euler_md(hipStream_t s, const DevState &d, double dt);
void launch_fill_f64(hipStream_t s, double *p, double v, int n);
void launch_set_counters(hipStream_t s, int *c, int first, int count, int v);
// dst[r * C_COUNT + k] = src[r][k] for r < n (device array of counter pointers)
void launch_gather_counters(hipStream_t s, const int *const *src, int n, int *dst);
// the locals' state a rebuild changes in place, and the counters
struct CkptArrays {
    double *X, *Y, *Z, *vx, *vy, *vz, *mass;
    int *type, *flags, *uid, *shape, *ref, *phys, *counters;
};
// copy the first n locals' entries (and all counters) from a to b
void launch_checkpoint(hipStream_t s, const CkptArrays &a, const CkptArrays &b, int n);
void launch_identity(hipStream_t s, int *p, int n);
void launch_exchange(hipStream_t s, const DevState &d, const Geom &g, const int *periodic);
void launch_borders(hipStream_t s, const DevState &d, const Geom &g, const int *periodic);
// bins locals and ghosts into cells and permutes every particle array into
// cell order (swapping d's spare arrays in), then builds the ghost sync maps
// (pack: and the packed copy of the new positions)
void launch_bin_sort(hipStream_t s, DevState &d, const Geom &g, bool pack = false);
void launch_build_neighbors(hipStream_t s, const DevState &d, const Geom &g, int half, double rc2);
// largest tile (entries) the build and force kernels can stage in LDS
int build_tile_limit(const DevState &d, const Geom &g, int half);

// one system of a batched cell phase
struct RepDesc {
    DevState d;       // d.cur: the position buffer before the phase
    Geom g;
    int periodic[3];
};
// exchange, borders and cell binning of n systems, each kernel one launch
// (blockIdx.y = system); max_cap / max_ncells: the largest system's
void launch_cells_batch(hipStream_t s, const RepDesc *D, int n, int max_cap, int max_ncells);
// thermo rows (T, P, PE, W, P total) of n systems after a fused step with
// reduction, out[5 r + k]
void launch_thermo_batch(hipStream_t s, const RepDesc *D, int n, double *out);

// the neighbour build's arguments for one system (position buffer d.cur)
struct BuildArgs {
    const int *counters;
    int *counters_rw;
    Geom g;
    const int *lstart, *gstart;
    const double *X, *Y, *Z;
    const int *ref, *flags;
    double rc2;
    uint32_t *nl;
    int nl_stride, ncap, tcap, zt, rev0;
    int *numneighs, *nrev;
};
BuildArgs build_args(const DevState &d, const Geom &g, int half, double rc2);
// the force tiles of one system
struct TileArgs {
    int *counters;
    Geom g;
    const int *lstart, *gstart, *numneighs, *nrev;
    const uint32_t *nl;
    uint4 *nl16;         // row r of local i: entries 8 r .. 8 r + 7; half lists: mirror rows from rows / 8 on
    int nlocal, nl_stride, ncap, rows, rev0;
    int4 *grp;           // first local, locals, first cell, last cell
    int4 *tile;          // by workgroup: first local, locals (0: none), the tile's size (0: does not fit)
    int *slots;
    int gmax;
};
// the most groups of a system's tiles: the length of its table
int tile_groups_max(int nlocal, const Geom &g);
// the table before a build has made tiles: every local, none with a tile (their
// forces come from the 32-bit lists); the rest is empty, as the force kernel
// reads all of it
inline std::vector<int4> tiles_before_build(int nlocal, int gmax) {
    std::vector<int4> tab(gmax, make_int4(0, 0, 0, 0));
    for (int k = 0; k * TILE_G < nlocal; k++) tab[k] = make_int4(k * TILE_G, std::min(TILE_G, nlocal - k * TILE_G), 0, 0);
    return tab;
}
// threads of a build workgroup: of one system (BB, or BB_SMALL in small ones),
// of a batch (BB); and its dynamic LDS
constexpr int BB = 128;
constexpr int BB_SMALL = 512;
int build_threads(const DevState &d, const Geom &g, int half);
size_t build_lds_bytes(const DevState &d, const Geom &g, int half, int threads);
// the builds of many systems in one launch (block b: system rep[b], its
// segment b - seg_base[rep[b]]); lds = the largest system's need
void launch_build_batch(hipStream_t s, const BuildArgs *desc, const int *rep, const int *seg_base, int nblocks,
                        size_t lds, int half);
void launch_expand_neighbors(hipStream_t s, const DevState &d, const Geom &g, int *out_ref, int ncap_out);
void launch_sync_pp(hipStream_t s, const DevState &d, const Geom &g, int cur, int prev, int grid);
void launch_sync_inplace(hipStream_t s, const DevState &d, const Geom &g, int grid, int with_vel);
// mode: 0 force only, 1 force + integrators (fused), 2 energy only (no writes)
// The force kernel gathers positions from P[cur]: with pack, a pass first
// packs it from X, Y, Z; after_pack, if given, is recorded between that pass
// and the force kernel.  With fuse and do_vv1 the kernel also writes P[next]
// for every local and (images on) every ghost.
void launch_lj_full(hipStream_t s, const DevState &d, const Geom &g, const LJParams &prm, int cur, int next, int fuse,
                    int do_vv2, int do_vv1, int reduce, int pack = 1, hipEvent_t after_pack = nullptr);
void launch_energy(hipStream_t s, const DevState &d, const Geom &g, const LJParams &prm, int half, double *eatom);
void launch_vv_initial(hipStream_t s, const DevState &d, const LJParams &prm);
void launch_vv_post(hipStream_t s, const DevState &d, const Geom &g, const LJParams &prm, int cur, int next,
                    int do_vv2, int do_vv1, int reduce, double4 *Pn = nullptr);
void launch_ke_partial(hipStream_t s, const DevState &d);
// thermo row from the partials: kinetic row over nb_ke entries, energy and
// virial rows over nb_f entries
void launch_thermo_reduce(hipStream_t s, const DevState &d, int nb_ke, int nb_f, int which_mask, const Geom &g,
                          double *out);

// every argument of the full-list force kernel (one system)
struct LJArgs {
    const int *counters;
    int nlocal, rows;    // locals; allocated list rows of each part
    Geom g;
    const double *X, *Y, *Z;
    const double4 *P;    // packed (x, y, z, type) of X, Y, Z, and the spare record
    double4 *Pn;         // packed copy of the next positions, or null
    double *Xn, *Yn, *Zn;
    const int *type;
    const uint32_t *nl;
    int nl_stride;
    const int *numneighs, *flags;
    const int *nrev;     // half lists: length of each particle's mirror part
    int rev0;            // half lists: first list row of the mirror part
    int ncap;            // list rows of each part: counts are clamped to it
    double *fx, *fy, *fz, *vx, *vy, *vz;
    const double *mass;
    double rc2, dt, hdt;
    LJTab tab;
    int do_vv2, do_vv1, pstride;
    double *partials, *eatom;
    Images im;
};
// the fused force + integrate arguments of one system (cur -> next buffer)
LJArgs lj_args(const DevState &d, const Geom &g, const LJParams &prm, int cur, int next, int do_vv2, int do_vv1,
               int fused, double *eatom, bool packed = true);
// the packed copy (P) of the buffer each of n descriptors reads (max_cap:
// the largest system's particle capacity)
void launch_pack_p_batch(hipStream_t s, const LJArgs *desc, int n, int max_cap);
// fused force + integrate for many systems: block b is wave b - wave_base[rep[b]] of system rep[b]
// the ghost-image table of a kernel that advances positions (on only when
// it writes the next positions into the other buffer and every local's
// images fit the table)
Images images_of(const DevState &d, bool writes_next);
// one persistent launch over the wave table of many systems: the resident
// workgroups, or at most max_wg of them when max_wg > 0
void launch_lj_full_batch(hipStream_t s, const LJArgs *desc, const int *rep, const int *wave_base, int nblocks,
                          int ntypes1, int unit, int reduce, int max_wg);

}  // namespace pk
