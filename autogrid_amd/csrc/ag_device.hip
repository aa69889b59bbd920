// Device side of the MI355X AutoGrid4 engine (gfx950, wave64).
//
// One call of ag_maps_plain runs, on the context's stream:
//   1. cell list   : atoms within 8 A of the box binned into cubic cells by a
//                    counting sort; each cell's atoms are then ordered by atom
//                    index so every later traversal is deterministic.
//   2. near kernel : one workgroup per brick of grid points, 8x8x4 on large grids,
//                    8x4x4 or 4x4x4 on smaller ones, where two or four waves
//                    share the atoms of a 4x4x4 cube.  It stages
//                    the atoms within 8.03 A of the brick (cells in fixed
//                    order, ballot compaction) and evaluates, per point, the
//                    8 A part of the reference's per-point loop
//                    (main.cpp:2866-3431): covalent maps, closest donor H,
//                    directional H-bond factors, vdW/H-bond table terms,
//                    desolvation, the d map, the H-bond min/max fix-up, and
//                    the electrostatic terms of every atom the far kernel
//                    leaves out.  Bin indices floor(128 r) are taken from an
//                    FP32 distance unless 128 r lies within 4e-4 of an
//                    integer, where the reference's FP64 distance is
//                    recomputed, so the table bins match the reference's.
//   3. far kernel  : the electrostatic sum over all atoms (main.cpp:2940-2982)
//                    for every pair whose FP32 bin is >= 1025 (r > 8 A).  A wave
//                    takes a patch of 64 rows of 16 points.  Atoms near the
//                    patch go pair by pair through the dielectric table in
//                    LDS, with zeros below bin 1025; the others are summed at
//                    80 Chebyshev nodes of the patch's box and interpolated
//                    to its points; in large receptors most of those at the
//                    512 nodes of a coarse box of patches first.  How far off
//                    an atom has to be follows its charge, the table's steps
//                    and the patch's own distance from the receptor.  The sums
//                    join the near kernel's value.
// Where kernels do not depend on each other they overlap: a small plan's far field
// goes first and makes the cell list, and in a constant dielectric the far field
// runs beside the near one.
// No atomics touch map values; every sum has a fixed order.

#include <hip/hip_runtime.h>
#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <functional>
#include <memory>
#include <string>
#include <thread>
#include <vector>

#include "ag_internal.h"
#include "ag_devcommon.h"

// Device scratch of the allocation-free entry point (ag_maps_plain_noalloc):
// one array per GPU, present from the library's load until the process
// ends.  Host code never uses this name as an address: each device's
// address comes from hipGetSymbolAddress at context creation (ag_ctx::scratch).
static __device__ __align__(256) unsigned char scratch[AG_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kBX = 8, kBY = 8, kBZ = 4;          // brick of the near kernel
constexpr int kNearThreads = kBX * kBY * kBZ;     // 256
constexpr int kStage = 3;                         // atoms per thread of a staging round
constexpr int kMapSlots = 16;                     // maps per near-kernel pass
constexpr int kPlainSlots = 12;                   // of which without H-bond terms
constexpr int kHbSlots = kMapSlots - kPlainSlots; // of which H-bonding probes
constexpr int kCandCap = 2048;                    // candidates per brick
constexpr int kHCap = 256;                        // donor-H candidates per brick
// The near kernel's bins, as rows of its tables: 0 to 1023, whose rows hold
// values; 1024 to 1039, past the 8 A cutoff, whose rows are zeros (a distance is
// clamped to 1039.5 bins), so a lane out of range needs no test; the pair at 8 A
// exactly (bin 1024, not past the cutoff: the last value row); and bin 1025 as
// the near field's, where the far kernel's bin is 1024.
constexpr int kNearZeroRow = 1039, kNearExactRow = 1040, kNearEdgeRow = 1041, kNearRows = 1042;
constexpr float kNearRadius = 8.03f;              // staging radius (A)
constexpr int kFarK = 16;                         // points per lane, far kernel
constexpr int kFarWaves = 4;                      // waves of a far-kernel workgroup: parts of the atom list
constexpr int kFarThreads = 64 * kFarWaves;
constexpr int kFarAtomChunk = 64;                 // Kahan block (at least)
constexpr int kFarNx = 5, kFarNy = 4;             // interpolation nodes of a patch along x, and along y and z
constexpr double kFarQRef = 0.85;                 // charge of level 0 over the conformation's rms charge
constexpr int kFarLevels = 12;                    // charge levels, each with its own distance
constexpr int kFarStrict = 20;                    // stricter levels before them, for patches far from the atoms
constexpr int kReachTab = 256;                    // distances (half A) of k_far_reach's table
constexpr int kFarSplitMax = 8;                   // workgroups that may share a patch's atoms
constexpr int kBoxN = 8;                          // interpolation nodes of a coarse box along each axis
constexpr int kBoxNodes = kBoxN * kBoxN * kBoxN;
constexpr int kFarNodes = kFarNx * kFarNy * kFarNy;  // of a patch
constexpr int kBoxRuns = 2, kBoxRows = 32;        // a coarse box: x-runs, and rows along y and z (whole patches, about)
constexpr int kFarBinMin = 1025;                  // far kernel takes bins >= this
constexpr float kGuardBins = 4.0e-4f;             // FP64 recompute band around bin edges

// Map roles.
enum : int { ROLE_NONE = 0, ROLE_AFF = 1, ROLE_DES = 2, ROLE_COV = 4 };
// Coefficient bits of an H-bonding slot for one atom class.
enum : int { HC_PLAIN = 1, HC_HRAMP = 2, HC_MINMAX = 4, HC_RACC = 8 };
// H-bond cases (main.cpp:3286-3390).
enum : int { HBC_PLAIN = 0, HBC_ACC_PROBE = 1, HBC_MINMAX_RACC = 2, HBC_DON_PROBE = 3 };

struct __align__(16) NearAtom {   // 80 bytes
    double x, y, z;               // grid frame, as the reference holds them
    float qe;                     // charge * coeff_estat
    float vol;
    float solq;                   // solpar + solpar_q * |charge|
    int meta;                     // type | hbond << 8 | rexp << 16 | disorder << 24
    int index;                    // atom index in the receptor
    float rv2rest;                // 1 - |rv2|^2
    float rv[3];
    float pad0;
    float rv2[3];
    float pad1;
};
static_assert(sizeof(NearAtom) == 80, "NearAtom layout");

// One receptor conformation on its own grid, as the kernels see it.  A plan
// holds one; a batch holds many, their atoms, cells, bricks and far-kernel
// tiles concatenated in conformation order.
struct ConfDev {
    int n1[3], ne[3];
    double spacing;
    float s128;                   // (float)(spacing * 128)
    float near_band;              // far_band: half-width (bins) of the shell where the far kernel's bin decides
    int near_share;               // near kernel: waves (1, 2 or 4) that share a cube's atoms
    int nb[3];                    // bricks per axis
    double cell_origin[3];
    int nc[3];
    int cell_base;                // first cell of this conformation in the cell arrays
    int atom_base, n_atoms;       // atom range in the concatenated atom arrays
    long long P;
    long long map_off;            // offset of its [n_maps][P] block in the map output
    long long pt_off;             // offset of its [P] block in the fmap / cmap outputs
    int runs_per_row;             // far-kernel runs of kFarK points along x
    int far_py, far_pz;           // far-kernel patch: rows along y and z, one per lane (far_py * far_pz <= 64)
    int far_npy, far_npz;         // patches along y and z
    int far_split;                // workgroups sharing each patch's atoms
    int far_clamp;                // far kernel: a direct pair may pass the table's end
    float far_r2[kFarStrict + kFarLevels];   // squared distances (bins^2) from a patch's box past which atoms are interpolated
    float far_qscale;             // an atom's level is that of |its far charge| times this (far_level)
    long long part_off;           // far_split > 1: offset of its [far_split][P] partial e maps
    int box_parts;                // coarse boxes: workgroups sharing one's atoms; 0: no coarse boxes
    int box_py, box_pz;           // patches of a box along y and z
    int box_n[3];                 // boxes per axis
    float box_r2[kFarStrict + kFarLevels];   // as far_r2, from a box
    long long reach_off;          // offset of its patches' shifts (k_far_reach)
    long long box_off;            // offsets of its boxes' node sums ([box][part][kBoxNodes] doubles), of their
    long long box_mask_off;       // atom sets ([box][groups of 64 atoms]) and of its patches' node values
    long long box_patch_off;      // ([patch][kFarNodes] doubles)
};

// Read-only device tables (conformation records, work prefixes) are read
// through the constant address space: no kernel writes them, so uniform
// reads become scalar loads the compiler may repeat instead of holding the
// values in registers across the hot loops.
#define AG_CONST __attribute__((address_space(4)))
// float4 layout without HIP_vector_type's constructors.
struct __align__(16) PlainF4 {
    float x, y, z, w;
};
template <typename T>
__device__ __forceinline__ const AG_CONST T *as_const(const T *p) {
    return (const AG_CONST T *)(p);
}

// Work lists: item k of a launch belongs to conformation c with
// prefix[c] <= k < prefix[c + 1].
__device__ __forceinline__ int find_conf(const AG_CONST int *prefix, int nconf, int item) {
    int lo = 0, hi = nconf;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (prefix[mid] <= item) lo = mid;
        else hi = mid;
    }
    return lo;
}

// When a kernel began, by its first thread (wall_clock64; null: not wanted).
__device__ __forceinline__ void stamp_start(unsigned long long *stamp) {
    if (stamp && blockIdx.x == 0 && threadIdx.x == 0) *stamp = wall_clock64();
}

struct NearParams {
    // conformations and work distribution
    const ConfDev *confs;
    const int *brick_prefix;      // [nconf + 1]
    int nconf, total_bricks;
    int item_base;                // first brick of this launch
    double cell_size;
    const int *cell_start;        // [total cells + 1]
    const NearAtom *atoms;        // sorted by (cell, index)
    const double *coord64;        // [n][3] by atom index
    const double *rvec64;         // [n][3]
    // tables
    const float *tab;             // [T][kNearRows][row slots] for this pass's maps (near_row)
    const float *sol;             // [1025]
    const float *reps;            // [8192] electrostatic factor (r_eps or 332/diel)
    // map slots of this pass: [0, kPlainSlots) maps without H-bond terms,
    // [kPlainSlots, kMapSlots) H-bonding probes
    float sp[kMapSlots];          // solpar_probe, 0 when the slot carries no desolvation
    float volp[kMapSlots];        // vol_probe, 0 when the slot carries no desolvation
    int hcode[kHbSlots][7];       // per atom H-bond class: bits 0-3 ordered atom, 4-7 disordered
                                  // atom; each nibble kP | kH << 1 | kM << 2 | use_racc << 3
    int out_slot[kMapSlots];      // output map of each slot, -1 if unused
    int e_slot, d_slot;           // -1 when not produced in this pass
    int has_affinity;             // any slot in use, or the d map
    float solpar_q;
    int disorder_h, hydrogen_type;
    int *cmap;                    // constriction count per point, or null (pass 0 only)
    double ccut;                  // constriction distance cutoff (<= 8 A)
    int bhtree;                   // ag_mapset.bhtree: Loop 2 and cmap by the tree's FP32 test
    unsigned char *collide;       // tree build, collisions tested: 1 per point within 1.5 A of an atom (pass 0)
    float *maps;
    const float *far_part;        // the far kernel's parts of the e map when it has run before, or null
    int *status;
    unsigned long long *stamp;
};

// An atom of the far kernel: coordinates in bins (exact) and charge times the
// electrostatic coefficient.
struct __align__(16) FarAtom {
    double x, y, z;
    float w, pad;
};

struct FarParams {
    const ConfDev *confs;
    const int *tile_prefix;       // [nconf + 1], items: patches x x-runs x parts
    int nconf, total_tiles;
    int item_base, item_end;      // tiles [item_base, item_end) of this launch
    int *queue;                   // null: one tile per workgroup; else a persistent work counter
    const FarAtom *atoms;
    const float *tab;             // [AG_NDIEL] electrostatic factor
    float *maps;                  // e map slot: in = near part, out = total
    float *part;                  // partial e maps of the conformations with far_split > 1
    double *wide;                 // where not null, the whole far field goes here (one conformation, far_split 1)
    double *box_sums;             // coarse boxes (ConfDev::box_*)
    unsigned long long *box_mask;
    double *box_patch;
    const unsigned char *shift;   // per patch, how many levels stricter its distances are (k_far_reach)
    int e_slot;
    unsigned long long *stamp;
};

// Consecutive workgroup ids go round-robin over the 8 XCDs; here XCD x takes
// chunks x, x + 8, x + 16, ... of C consecutive items, so that every XCD
// gets items from all over the grid (the work per item varies with the
// local atom density, and in the far kernel with the distance to the
// atoms) while the items of a chunk share its L2.  Ids past
// the last whole round of 8 chunks map to themselves.
template <int C>
__device__ __forceinline__ int xcd_chunked(int bid, int nblocks) {
    const int full = nblocks / (8 * C) * (8 * C);
    if (bid >= full) return bid;
    const int x = bid % 8, k = bid / 8;
    return ((k / C) * 8 + x) * C + k % C;
}

// Table offset of the far kernel's bin: with r = rb2 * rsq(rb2) (128 r in
// bins), y = fma(rb2, rsq(rb2), 2^21 - 1/8) lies in [2^21, 2^22), where the
// float spacing is 1/4, so the low 23 bits of y hold m = round(4 r - 1/2)
// (ties to even).  For n <= r < n + 1, 4n - 1/2 <= 4r - 1/2 < 4n + 7/2 puts m
// in {4n, ..., 4n + 3} (the tie at r = n goes to the even 4n), so
// m & ~3 = 4 floor(r): the byte offset of bin floor(r) in a float table, in
// one fma and one and.  Valid for r < 2^21 - 1.
constexpr float kBinMagic = 2097151.875f;         // 2^21 - 1/8
__device__ __forceinline__ unsigned bin4_of(float rb2, float rs) {
    return __float_as_uint(__builtin_fmaf(rb2, rs, kBinMagic)) & 0x7FFFFCu;
}

// Far-kernel geometry.  An atom and a patch's points are taken from the centre
// of the patch's box: the difference is formed in FP64 and rounded once, so a
// pair's bin does not depend on how far from the origin it lies (coordinates
// rounded to FP32 before the difference put 20 to 90 % more variance into the
// bins: 7.2e-7 of the e map for 6.1e-7 with 5,000 atoms, 9.0e-7 for 6.5e-7 with
// 20,000).  Along x the box is a run of kFarK points at dk = (k - kFarMid) s128
// (k = 0..kFarK-1), and with u the atom's x
//   rb2 = (u - dk)^2 + dyz2,  dyz2 = max(dy^2 + dz^2, floor)
//       = fma(u s128, 15 - 2k, fma(s128^2, (j + 1/2)^2, fma(u, u, dyz2))),
// j = |k - kFarMid| - 1/2: the points k and kFarK-1-k share the middle
// term, and both factors 15 - 2k and (j + 1/2)^2 are exact small constants
// the instructions carry as literals, so no register holds them.  Per point
// that is 1.5 operations instead of a subtract and an fma.  The roundings
// of the three products and sums are below 2^-21 (7.5 s128)^2 in total when
// u = dk, where the exact value is only dyz2; its floor, four times that,
// keeps rb2 > 0 and rsq finite, and changes nothing further off the run's
// line than 0.5 bins at 0.375 A spacing.  (The floor was a term added to every
// pair, 1.1e-4 of a bin at r = 1,100: without it 40 % fewer far-field bins
// differ from the FP64 ones.)
constexpr float kFarMid = 0.5f * (kFarK - 1);

__device__ __forceinline__ float far_floor(float s128) {
    const float d = kFarMid * s128;
    return fmaxf(1.0e-3f, d * d * 0x1p-19f);
}
// Centre (bins) of the n points from point i0 on.
__device__ __forceinline__ double far_centre(int i0, int n, int ne, double spacing) {
    return ((double)(i0 - ne) + 0.5 * (double)(n - 1)) * (spacing * 128.0);
}
// Offset of a box's j-th of n points from its centre.
__device__ __forceinline__ float far_offset(int j, int n, float s128) {
    return ((float)j - 0.5f * (float)(n - 1)) * s128;
}
// (j + 1/2)^2 for point k, and the factor 15 - 2k of u s128
__device__ __forceinline__ constexpr float far_c2(int k) {
    return (k >= kFarK / 2 ? (float)(k - kFarK / 2) + 0.5f : (float)(kFarK / 2 - 1 - k) + 0.5f) *
           (k >= kFarK / 2 ? (float)(k - kFarK / 2) + 0.5f : (float)(kFarK / 2 - 1 - k) + 0.5f);
}
__device__ __forceinline__ constexpr float far_m(int k) { return (float)(kFarK - 1 - 2 * k); }

// The far kernel's table offset for an atom (in bins) and point (ix, iy, iz),
// reproduced bit for bit by the near kernel when it decides which atoms
// the far kernel left out, and by the audit (same operations in the same
// order; the build turns off FP contraction).
struct FarPatch {
    int ne[3], py, pz;
    double spacing;
    float s128;
};
// An atom's y or z distance from row i, in patches of p rows.
__device__ __forceinline__ float far_row(double a, int i, int p, int ne, double spacing, float s128) {
    const int l = i % p;
    return (float)(a - far_centre(i - l, p, ne, spacing)) - far_offset(l, p, s128);
}
// The offset from the distances along y and z and the atom's x from the run's centre.
__device__ __forceinline__ unsigned far_bin4(float u, float dy, float dz, int k, float s128) {
    const float dyz2 = fmaxf(__builtin_fmaf(dy, dy, dz * dz), far_floor(s128));
    const float U = __builtin_fmaf(u, u, dyz2);
    const float W = __builtin_fmaf(s128 * s128, far_c2(k), U);
    const float rb2 = __builtin_fmaf(u * s128, far_m(k), W);
    return bin4_of(rb2, __builtin_amdgcn_rsqf(rb2));
}
__device__ __forceinline__ unsigned far_bin4(double ax, double ay, double az, const FarPatch &f, int ix, int iy,
                                             int iz) {
    const int k = ix % kFarK;
    return far_bin4((float)(ax - far_centre(ix - k, kFarK, f.ne[0], f.spacing)),
                    far_row(ay, iy, f.py, f.ne[1], f.spacing, f.s128),
                    far_row(az, iz, f.pz, f.ne[2], f.spacing, f.s128), k, f.s128);
}

// ---------------------------------------------------------------------------
// cell list
// ---------------------------------------------------------------------------

__device__ __forceinline__ int cell_of(const ConfDev &c, double cs, const double *p) {
    int ix = (int)floor((p[0] - c.cell_origin[0]) / cs);
    int iy = (int)floor((p[1] - c.cell_origin[1]) / cs);
    int iz = (int)floor((p[2] - c.cell_origin[2]) / cs);
    if (ix < 0 || iy < 0 || iz < 0 || ix >= c.nc[0] || iy >= c.nc[1] || iz >= c.nc[2]) return -1;
    return c.cell_base + ix + c.nc[0] * (iy + c.nc[1] * iz);
}

// atom_conf: conformation of each atom, or null when there is one.
__global__ void k_cell_count(const ConfDev *confs, const int *atom_conf, int n, double cs, const double *coord,
                             int *atom_cell, int *count) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int cell = cell_of(confs[atom_conf ? atom_conf[i] : 0], cs, coord + 3 * (size_t)i);
    atom_cell[i] = cell;
    if (cell >= 0) atomicAdd(&count[cell], 1);
}

// Clears the cell counts [0, n), the overflow word and the nq
// work counters of one map set, in one launch: a kernel rather than memset
// nodes, since a plan's map set is captured in a graph.
__global__ void k_zero_cells(int *count, int n, int *status, int *queue, int nq,
                             unsigned long long *stamp) {
    stamp_start(stamp);
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) count[i] = 0;
    if (i < nq) queue[i] = 0;
    if (i == 0) *status = 0;
}

// Exclusive scan of count[0..n) into start[0..n], one workgroup of 1024
// walking tiles of 1024 * kScanPer cells.  Each thread takes kScanPer
// consecutive cells of a tile (16-byte loads and stores, so a wave covers
// one contiguous 4 KiB span); the thread sums are scanned within each wave
// by shuffles and across the 16 waves through LDS, and the total of the
// tiles before is carried in a register.
constexpr int kScanPer = 16;

__global__ void __launch_bounds__(1024) k_scan(const int *count, int *start, int n) {
    __shared__ int wave_sum[16];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    int carry = 0;
    for (int base = 0; base < n; base += 1024 * kScanPer) {   // uniform: every thread reaches both barriers
        const int i0 = base + t * kScanPer;
        const bool whole = i0 + kScanPer <= n;
        int v[kScanPer];
        if (whole) {
            const int4 *q = reinterpret_cast<const int4 *>(count + i0);
#pragma unroll
            for (int j = 0; j < kScanPer / 4; j++) {
                const int4 a = q[j];
                v[4 * j] = a.x;
                v[4 * j + 1] = a.y;
                v[4 * j + 2] = a.z;
                v[4 * j + 3] = a.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < kScanPer; j++) v[j] = i0 + j < n ? count[i0 + j] : 0;
        }
        int s = 0;
#pragma unroll
        for (int j = 0; j < kScanPer; j++) s += v[j];
        int x = s;   // inclusive scan over the wave
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(x, off);
            if (lane >= off) x += y;
        }
        if (lane == 63) wave_sum[w] = x;
        __syncthreads();
        int before = 0, total = 0;
        for (int k = 0; k < 16; k++) {
            const int ws = wave_sum[k];
            before += k < w ? ws : 0;
            total += ws;
        }
        __syncthreads();   // the next tile rewrites wave_sum
        int run = carry + before + x - s;
        if (whole) {
            int4 *o = reinterpret_cast<int4 *>(start + i0);
#pragma unroll
            for (int j = 0; j < kScanPer / 4; j++) {
                int4 r;
                r.x = run;
                r.y = r.x + v[4 * j];
                r.z = r.y + v[4 * j + 1];
                r.w = r.z + v[4 * j + 2];
                run = r.w + v[4 * j + 3];
                o[j] = r;
            }
        } else {
#pragma unroll
            for (int j = 0; j < kScanPer; j++) {
                if (i0 + j < n) start[i0 + j] = run;
                run += v[j];
            }
        }
        carry += total;
    }
    if (t == 0) start[n] = carry;
}

// Counts the cells down again (k_gather finds the order within a cell).
__global__ void k_cell_scatter(int n, const int *atom_cell, const int *start, int *count, int *slot_atom) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int cell = atom_cell[i];
    if (cell < 0) return;
    int pos = start[cell] + atomicSub(&count[cell], 1) - 1;
    slot_atom[pos] = i;
}

// What one workgroup needs to make the cell list of a small plan by itself.
struct CellParams {
    const ConfDev *confs;
    const int *atom_conf;         // null when there is one conformation
    int n, ncells;
    double cs;
    const double *coord;
    int *start, *atom_cell, *slot_atom;
    int *status, *queue;
    int nq;
    unsigned long long *stamp, *stamp_end;
};

// k_zero_cells, k_cell_count, k_scan and k_cell_scatter by one workgroup, the
// counts (ncells + 1 of them) in its LDS.
template <int THREADS>
__device__ void cell_list(const CellParams &p, int *cnt, int *wave_sum) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    stamp_start(p.stamp);
    for (int k = t; k < p.ncells; k += THREADS) cnt[k] = 0;
    for (int k = t; k < p.nq; k += THREADS) p.queue[k] = 0;
    if (t == 0) *p.status = 0;
    __syncthreads();
    for (int i = t; i < p.n; i += THREADS) {
        const int cell = cell_of(p.confs[p.atom_conf ? p.atom_conf[i] : 0], p.cs, p.coord + 3 * (size_t)i);
        p.atom_cell[i] = cell;
        if (cell >= 0) atomicAdd(&cnt[cell], 1);
    }
    __syncthreads();
    // exclusive scan: 64 consecutive cells per wave and round, the waves'
    // parts one after the other
    const int per = ((p.ncells + THREADS - 1) / THREADS) * 64;   // cells of a wave
    const int c0 = w * per, c1 = min(c0 + per, p.ncells);
    int sum = 0;
    for (int c = c0 + lane; c < c1; c += 64) sum += cnt[c];
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    if (lane == 0) wave_sum[w] = sum;
    __syncthreads();
    int run = 0;
    for (int k = 0; k < w; k++) run += wave_sum[k];
    for (int base = c0; base < c1; base += 64) {
        const int c = base + lane, v = c < c1 ? cnt[c] : 0;
        int x = v;
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(x, off);
            if (lane >= off) x += y;
        }
        if (c < c1) cnt[c] = p.start[c] = run + x - v;
        run += __shfl(x, 63);
    }
    if (w == THREADS / 64 - 1 && lane == 0) p.start[p.ncells] = run;
    __syncthreads();
    for (int i = t; i < p.n; i += THREADS) {
        const int cell = p.atom_cell[i];
        if (cell >= 0) p.slot_atom[atomicAdd(&cnt[cell], 1)] = i;
    }
    if (p.stamp_end) {
        __syncthreads();
        if (t == 0) *p.stamp_end = wall_clock64();
    }
}

// The cell list in one launch.  Its four parts take 2 to 4 us each, most of that
// the launch, and as much again between them: 1,000 atoms 11.4 us in all and 4.9
// here, 5,000 atoms 13.9 and 14.9, 20,000 atoms 21 and 69 (the gaps not counted).
constexpr int kCellsOne = 32768, kCellsOneAtoms = 6144;
__global__ void __launch_bounds__(1024) k_cells(CellParams p) {
    __shared__ int cnt[kCellsOne];
    __shared__ int wave_sum[16];
    cell_list<1024>(p, cnt, wave_sum);
}

struct AtomSrc {
    const double *coord, *charge, *vol, *solpar, *rvec, *rvec2;
    const int *type, *hbond, *rexp;
    const unsigned char *disorder;
    double coeff_estat, solpar_q;
};

// The atoms' records in cell order, by atom index within a cell (a cell holds
// few atoms: each counts those before it).
__global__ void k_gather(int ncells, const int *atom_cell, const int *start, const int *slot_atom, AtomSrc s,
                         NearAtom *out, unsigned long long *stamp) {
    stamp_start(stamp);
    const int slot = blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= start[ncells]) return;
    const int i = slot_atom[slot], cell = atom_cell[i];
    const int b = start[cell], e = start[cell + 1];
    int k = b;
    for (int j = b; j < e; j++) k += slot_atom[j] < i;
    NearAtom a;
    a.x = s.coord[3 * i];
    a.y = s.coord[3 * i + 1];
    a.z = s.coord[3 * i + 2];
    double q = s.charge[i];
    a.qe = (float)(q * s.coeff_estat);
    a.vol = (float)s.vol[i];
    a.solq = (float)(s.solpar[i] + s.solpar_q * fabs(q));
    const double *u = s.rvec + 3 * (size_t)i, *v = s.rvec2 + 3 * (size_t)i;
    a.rv2rest = (float)(1.0 - (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]));
    for (int d = 0; d < 3; d++) {
        a.rv[d] = (float)u[d];
        a.rv2[d] = (float)v[d];
    }
    a.meta = (s.type[i] & 0xff) | ((s.hbond[i] & 0xff) << 8) | ((s.rexp[i] & 0xff) << 16) |
             ((s.disorder[i] ? 1 : 0) << 24);
    a.index = i;
    a.pad0 = a.pad1 = 0.f;
    out[k] = a;
}

__global__ void k_far_atoms(int n, const double *coord, const double *charge, double coeff_estat,
                            FarAtom *out) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[i] = FarAtom{coord[3 * i] * 128.0, coord[3 * i + 1] * 128.0, coord[3 * i + 2] * 128.0,
                     (float)(charge[i] * coeff_estat * 128.0), 0.f};
}

// ---------------------------------------------------------------------------
// near kernel
// ---------------------------------------------------------------------------

__device__ __forceinline__ double ref_dist(double ax, double ay, double az, double cx, double cy, double cz,
                                           double &dx, double &dy, double &dz) {
#pragma clang fp contract(off)
    // hypotenuse(): sqrt(dx*dx + dy*dy + dz*dz), no fused operations
    dx = ax - cx;
    dy = ay - cy;
    dz = az - cz;
    return sqrt(dx * dx + dy * dy + dz * dz);
}

// Orders a wave's own LDS accesses: its lanes see what the others wrote before.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Smaller and larger of two values neither of which is NaN, in one
// instruction: fminf and fmaxf first quieten an operand that might be a
// signalling NaN.
__device__ __forceinline__ float min_of(float a, float b) {
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float max_of(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// min(g, 1039.5) and min(inv_r, 2), the limit in the instruction.
__device__ __forceinline__ float clamp_bins(float g) {
    float r;
    asm("v_min_f32 %0, 0x4481f000, %1" : "=v"(r) : "v"(g));
    return r;
}
__device__ __forceinline__ float half_at_least(float inv_r) {
    float r;
    asm("v_min_f32 %0, 2.0, %1" : "=v"(r) : "v"(inv_r));
    return r;
}

// Uniform per-atom values: every lane reads the same LDS record, so its
// fields are moved to scalar registers and branches on them stay scalar.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float unif(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// A thread's point inside the brick: each wave takes a 4x4x4 cube, shared by
// `share` consecutive waves, or (CUBE false, nothing shared) an 8x8x1 slab.
template <bool CUBE>
__device__ __forceinline__ void brick_lane(int tid, int share, int &lx, int &ly, int &lz) {
    if (CUBE || share > 1) {
        const int cube = (tid >> 6) / share, lane = tid & 63;
        lx = (cube & 1) * 4 + (lane & 3);
        ly = (cube >> 1) * 4 + ((lane >> 2) & 3);
        lz = lane >> 4;
    } else {
        lx = tid % kBX;
        ly = (tid / kBX) % kBY;
        lz = tid / (kBX * kBY);
    }
}

// Slots of a table row: NPLAIN == 4 keeps four plain and four H-bond slots (32
// bytes), the others all sixteen (64 bytes).
__host__ __device__ constexpr int near_row(int nplain) { return nplain == 4 ? 8 : 16; }

// One value of a lane in each lane of its group of Q (2 or 4) neighbours, J the
// lane's place in the group.
template <int Q, int J>
__device__ __forceinline__ int group_lane(int v) {
    constexpr int ctrl = Q == 4 ? J * 0x55 : (J | J << 2 | (2 + J) << 4 | (2 + J) << 6);
    return __builtin_amdgcn_mov_dpp(v, ctrl, 0xf, 0xf, true);
}

// With 32-byte rows bound by its vector operations (49 per pair of a wave and a
// plain atom, 90 to 140 where the atom is directional), with 64-byte rows by the
// vector caches: 13 Vina maps make 4.3e8 accesses, 0.70 ms at one per clock and
// CU.  5,000 atoms, 127^3 points: 13 Vina maps 1,096 -> 731 us, 15 AutoDock maps
// 1,099 -> 836; 41^3 points and 1,000 atoms 157 -> 61.  CUBE selects the lane
// layout inside the brick (brick_lane).  FORM:
//   kNearPlain   neither the tree build's queries, a constriction count
//                nor disordered hydroxyls (their branches compiled out);
//   kNearGeneral every map-set option;
//   kNearPaged   every option, and candidate / donor-H lists longer than
//                one LDS page.
// The unpaged forms leave a brick whose candidates (or donor H) do not fit
// one LDS list: they set the overflow word, and the host runs the whole map
// set again with the paged form (whose page loops keep state beside the
// accumulators, with spills the common case should not pay for).
enum : int { kNearPlain = 0, kNearGeneral = 1, kNearPaged = 2 };
struct NearLists {
    double hpos[kHCap][3];
    int cand[kCandCap];
    int hidx[kHCap];
    float hrvs[kHCap][3];
};
template <int NPLAIN, bool CUBE, int FORM>
__global__ void __launch_bounds__(kNearThreads) __attribute__((amdgpu_waves_per_eu(FORM == kNearPlain ? 5 : 4))) k_near(NearParams p) {
    constexpr bool PAGED = FORM == kNearPaged;
    constexpr bool GENERAL = FORM != kNearPlain;
    __shared__ NearLists lists;   // reused at the end for the table sums
    int *const cand = lists.cand, *const hidx = lists.hidx;
    double(*const hpos)[3] = lists.hpos;
    float(*const hrvs)[3] = lists.hrvs;
    float *const scratch_f = reinterpret_cast<float *>(&lists);
    static_assert(sizeof(NearLists) >= sizeof(float) * kNearThreads * (kMapSlots + 1), "room for the table sums");
    __shared__ float2 rs_s[kNearRows];   // (electrostatic factor, sol_fn) per row; zeros past the near field's
    __shared__ int2 wave_tot[2][kStage][kNearThreads / 64];

    const int tid = threadIdx.x;
    stamp_start(p.stamp);
    // read here, stored once the staging's own reads are on their way
    constexpr int kRsPer = (kNearRows + kNearThreads - 1) / kNearThreads;
    float2 rs[kRsPer];
#pragma unroll
    for (int u = 0; u < kRsPer; u++) {
        const int k = min(tid + u * kNearThreads, kNearRows - 1);
        const int bin = k == kNearExactRow ? AG_NEINT : k == kNearEdgeRow ? kFarBinMin : min(k, kFarBinMin);
        rs[u] = make_float2(k < kFarBinMin || k > kNearZeroRow ? p.reps[bin] : 0.f,
                            k < AG_NEINT || k == kNearExactRow ? p.sol[min(bin, AG_NEINT)] : 0.f);
    }

    // one workgroup per brick of all conformations, in chunks of 16 bricks
    // spread over the XCDs: a brick's time follows the local atom density,
    // and contiguous eighths of the grid per XCD left the XCDs that hold a
    // protein's dense core finishing last.  (A persistent loop
    // over a work counter keeps more uniform state live than the scalar
    // register file holds and spills; the far kernel, whose state is
    // small, is the persistent one.)
    const int item = p.item_base + xcd_chunked<16>(blockIdx.x, gridDim.x);
    if (item >= p.total_bricks) return;
    const int ci = find_conf(as_const(p.brick_prefix), p.nconf, item);
    const AG_CONST ConfDev &cf = as_const(p.confs)[ci];
    const int brick = item - as_const(p.brick_prefix)[ci];
    const int n1x = cf.n1[0], n1y = cf.n1[1], n1z = cf.n1[2];
    const int nex = cf.ne[0], ney = cf.ne[1], nez = cf.ne[2];
    const double spacing = cf.spacing;
    const float s128 = cf.s128;
    const int bx = brick % cf.nb[0];
    const int by = (brick / cf.nb[0]) % cf.nb[1];
    const int bz = brick / (cf.nb[0] * cf.nb[1]);
    // With share > 1 the workgroup has a brick of 4 / share cubes of 4x4x4
    // points, and the share waves of a cube hold the same points and take each
    // share-th candidate (and donor H), the sums added up at the end.
    const int share = cf.near_share;
    const bool shared = share > 1;
    const int first = uni((tid >> 6) & (share - 1));
    const int ex = share > 2 ? kBX / 2 : kBX, ey = shared ? kBY / 2 : kBY;
    const int ix0 = bx * ex, iy0 = by * ey, iz0 = bz * kBZ;
    int lx, ly, lz;
    brick_lane<CUBE>(tid, share, lx, ly, lz);
    const int ix = ix0 + lx;
    const int iy = iy0 + ly;
    const int iz = iz0 + lz;

    // brick box in the grid frame
    const int ix1 = min(ix0 + ex, n1x) - 1, iy1 = min(iy0 + ey, n1y) - 1, iz1 = min(iz0 + kBZ, n1z) - 1;
    const double bmin[3] = {(ix0 - nex) * spacing, (iy0 - ney) * spacing, (iz0 - nez) * spacing};
    const double bmax[3] = {(ix1 - nex) * spacing, (iy1 - ney) * spacing, (iz1 - nez) * spacing};

    // point, reference arithmetic: c = (double)(i - ne) * spacing
    const double cx = (double)(ix - nex) * spacing;
    const double cy = (double)(iy - ney) * spacing;
    const double cz = (double)(iz - nez) * spacing;
    // (the far kernel's coordinates of the point and the tree build's FP32
    // query point are formed where they are used, in rare branches of the
    // candidate loop, so they hold no registers across it)
    const int bh = GENERAL ? p.bhtree : 0;
    const float ccf = (float)p.ccut, ccf2 = ccf * ccf;
    bool collide = false;

    // ---- stage candidate atoms: cells overlapping the brick box + radius ----
    int c0[3], c1[3];
    for (int d = 0; d < 3; d++) {
        c0[d] = (int)floor((bmin[d] - kNearRadius - cf.cell_origin[d]) / p.cell_size);
        c1[d] = (int)floor((bmax[d] + kNearRadius - cf.cell_origin[d]) / p.cell_size);
        c0[d] = max(c0[d], 0);
        c1[d] = min(c1[d], cf.nc[d] - 1);
    }
    const int ncx = c1[0] - c0[0] + 1, ncy = c1[1] - c0[1] + 1, ncz = c1[2] - c0[2] + 1;
    // Cells along x follow each other in the sorted atoms, so the cells of one
    // (y, z) are one run of slots: nrun runs, looked at 64 at a time, one per lane.
    const int nrun = (ncx > 0 && ncy > 0 && ncz > 0) ? ncy * ncz : 0;
    const int wave = tid >> 6, wlane = tid & 63;
    // Staging pass: the brick's candidates (atoms within 8.03 A of the box),
    // in cell order and slot order within a cell, are numbered from 0 as
    // found, and the donor H among them likewise.  Candidates numbered
    // cpage .. cpage + kCandCap - 1 go to cand[] and donor H numbered hpage ..
    // hpage + kHCap - 1 to the H lists (a negative page stores none); ncand
    // and nh end as the totals.  A brick with more than fits is processed
    // page by page, each page staged by another pass, in the same order, so
    // its sums are those one unbounded list would give.  Every wave scans
    // the run lengths for itself, so the only exchange is each wave's count of
    // what it found, one barrier per 256 atoms (two buffers: a wave may be one
    // round ahead).
    const float r2cut = kNearRadius * kNearRadius;
    const float lo_f[3] = {(float)bmin[0], (float)bmin[1], (float)bmin[2]};
    const float hi_f[3] = {(float)bmax[0], (float)bmax[1], (float)bmax[2]};
    int ncand = 0, nh = 0;
    auto stage = [&](int cpage, int hpage) {
        int found = 0, found_h = 0, buf = 0;
        for (int rbase = 0; rbase < nrun; rbase += 64) {
            int rstart = 0, rcount = 0;
            if (rbase + wlane < nrun) {
                const int gy = c0[1] + (rbase + wlane) % ncy, gz = c0[2] + (rbase + wlane) / ncy;
                const int g = cf.cell_base + c0[0] + cf.nc[0] * (gy + cf.nc[1] * gz);
                rstart = p.cell_start[g];
                rcount = p.cell_start[g + ncx] - rstart;
            }
            int rend = rcount;   // inclusive prefix
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int v = __shfl_up(rend, o);
                rend += wlane >= o ? v : 0;
            }
            const int total = __shfl(rend, 63);
            const int rslot = rstart - (rend - rcount);   // slot of the run's atom j is rslot + j
            for (int j0 = 0; j0 < total; j0 += kStage * kNearThreads, buf ^= 1) {
                bool ok[kStage], is_h[kStage];
                int slot[kStage];
#pragma unroll
                for (int u = 0; u < kStage; u++) {
                    const int j = j0 + u * kNearThreads + tid;
                    int lo = 0;   // runs that end at or before j
#pragma unroll
                    for (int o = 32; o > 0; o >>= 1) lo += __shfl(rend, lo + o - 1) <= j ? o : 0;
                    slot[u] = __shfl(rslot, lo) + j;
                    ok[u] = j < total;
                }
#pragma unroll
                for (int u = 0; u < kStage; u++) {
                    // an index past the last atom reads the first atom
                    const NearAtom &a = p.atoms[ok[u] ? slot[u] : 0];
                    // FP32: off by 1e-5 A at most, and an atom more than 8.02 A
                    // away adds nothing
                    const float av[3] = {(float)a.x, (float)a.y, (float)a.z};
                    float dd = 0.f;
                    for (int d = 0; d < 3; d++) {
                        const float t = fmaxf(fmaxf(lo_f[d] - av[d], av[d] - hi_f[d]), 0.f);
                        dd = __builtin_fmaf(t, t, dd);
                    }
                    ok[u] = ok[u] & (dd <= r2cut);
                    const int hb = (a.meta >> 8) & 0xff;
                    is_h[u] = ok[u] & ((hb == AG_HB_DS) | (hb == AG_HB_D1));
                }
                unsigned long long mo[kStage], mh[kStage];
                const unsigned long long below = (1ull << wlane) - 1ull;
#pragma unroll
                for (int u = 0; u < kStage; u++) {
                    mo[u] = __ballot(ok[u]);
                    mh[u] = __ballot(is_h[u]);
                    if (wlane == 0) wave_tot[buf][u][wave] = make_int2(__popcll(mo[u]), __popcll(mh[u]));
                }
                __syncthreads();
#pragma unroll
                for (int u = 0; u < kStage; u++) {
                    int cj = found + __popcll(mo[u] & below) - cpage, hj = found_h + __popcll(mh[u] & below) - hpage;
#pragma unroll
                    for (int w = 0; w < kNearThreads / 64; w++) {
                        const int2 n = wave_tot[buf][u][w];
                        found += n.x;
                        found_h += n.y;
                        cj += w < wave ? n.x : 0;
                        hj += w < wave ? n.y : 0;
                    }
                    if (cpage >= 0 && ok[u] && cj >= 0 && cj < kCandCap) cand[cj] = slot[u] * (int)sizeof(NearAtom);
                    if (hpage >= 0 && is_h[u] && hj >= 0 && hj < kHCap) {
                        const NearAtom &a = p.atoms[slot[u]];
                        hpos[hj][0] = a.x; hpos[hj][1] = a.y; hpos[hj][2] = a.z;
                        hidx[hj] = a.index;
                        hrvs[hj][0] = a.rv[0]; hrvs[hj][1] = a.rv[1]; hrvs[hj][2] = a.rv[2];
                    }
                }
            }
        }
        ncand = uni(found);
        nh = uni(found_h);
    };
    stage(0, 0);
#pragma unroll
    for (int u = 0; u < kRsPer; u++)
        if (tid + u * kNearThreads < kNearRows) rs_s[tid + u * kNearThreads] = rs[u];
    __syncthreads();
    if constexpr (!PAGED) {
        if (ncand > kCandCap || nh > kHCap) {   // uniform per workgroup
            if (tid == 0) __hip_atomic_store(p.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);   // host memory
            return;
        }
    }

    // Table sums.  A table row is read by the Q lanes of a group together, 16
    // bytes each: for each of the group's Q points in turn, lane c takes chunk c
    // (four slots) of that point's row, and adds it to its own sums.  So accT[j]
    // holds chunk c of point j; after the loop the group's lanes trade them.  The
    // vector cache serves one 128-byte line per cycle, so a load whose 64 lanes
    // read 64 rows took about 45 cycles and four of them 180 per candidate; now
    // each touches 64 / Q rows (2.7e8 line reads instead of 7.4e8 in 13 maps of
    // 127^3 points, 1,085 -> 712 us).  The H-bond slots of an atom whose class
    // mixes there are read by the point's own lane (acc_hb).
    constexpr int ROW = near_row(NPLAIN), Q = ROW / 4;
    float accT[Q][4], acc_hb[kHbSlots];
#pragma unroll
    for (int j = 0; j < Q; j++)
#pragma unroll
        for (int s = 0; s < 4; s++) accT[j][s] = 0.f;
#pragma unroll
    for (int k = 0; k < kHbSlots; k++) acc_hb[k] = 0.f;
    // min/max of the H-bond pairs of each H-bonding slot (main.cpp:3300-3374)
    float hmin[kHbSlots], hmax[kHbSlots];
#pragma unroll
    for (int k = 0; k < kHbSlots; k++) {
        hmin[k] = 999999.f;
        hmax[k] = -999999.f;
    }

    // ---- closest donor H (main.cpp:2985-3015), FP64, lowest index on ties ----
    // The reference compares r = sqrt(d2), which is correctly rounded and so
    // monotone in d2: squared distances more than 2^-49 apart (relative)
    // order the same way, strictly.  Within that band the two rounded
    // distances may tie, so there they are formed and compared as the
    // reference does.  The start, 999999^2, is exact and its root is 999999.
    double best_d2 = 999999.0 * 999999.0;
    int best_idx = 0x7fffffff;
    float hrv[3] = {0.f, 0.f, 0.f};   // bond vector of the closest H so far
    const auto closer = [&](double d2, int index) {
        if (d2 < best_d2 * (1.0 - 0x1p-49)) return true;
        if (d2 > best_d2 * (1.0 + 0x1p-49)) return false;
        const double r = sqrt(d2), rb = sqrt(best_d2);
        return r < rb || (r == rb && index < best_idx);
    };
    for (int h0 = 0; h0 < nh; h0 += kHCap) {   // pages of donor H
        if constexpr (PAGED) {
            if (h0 > 0) {
                __syncthreads();
                stage(-1, h0);
                __syncthreads();
            }
        }
        const int hn = min(nh - h0, kHCap);
        for (int h = first; h < hn; h += share) {
#pragma clang fp contract(off)
            const double dx = hpos[h][0] - cx, dy = hpos[h][1] - cy, dz = hpos[h][2] - cz;
            const double d2 = dx * dx + dy * dy + dz * dz;   // as ref_dist forms it
            if (closer(d2, hidx[h])) {
                best_d2 = d2;
                best_idx = hidx[h];
                hrv[0] = hrvs[h][0]; hrv[1] = hrvs[h][1]; hrv[2] = hrvs[h][2];
            }
        }
        if constexpr (!PAGED) break;
    }
    if (shared && nh > 0) {   // the closest of the sharing waves' (the order is total, so any split gives the same)
        static_assert(kHCap == kNearThreads, "the donor-H lists hold one entry per thread");
        double *const hd2 = &hpos[0][0];
        __syncthreads();
        hd2[tid] = best_d2;
        hidx[tid] = best_idx;
        hrvs[tid][0] = hrv[0]; hrvs[tid][1] = hrv[1]; hrvs[tid][2] = hrv[2];
        __syncthreads();
        for (int w = 0; w < share; w++) {
            const int o = (wave - first + w) * 64 + wlane;
            if (closer(hd2[o], hidx[o])) {
                best_d2 = hd2[o];
                best_idx = hidx[o];
                hrv[0] = hrvs[o][0]; hrv[1] = hrvs[o][1]; hrv[2] = hrvs[o][2];
            }
        }
    }

    // With 64-byte rows a lane keeps its H's bond vector in the H list, which is
    // done with, for the donor hydrogens among the candidates: in registers two of
    // its components went to scratch (whole map set of 127^3 points 1,618 -> 1,600
    // us).  With 32-byte rows there are registers for it (47 x 83 x 119 points 428 us,
    // 435 from LDS).
    constexpr bool H_IN_LDS = NPLAIN > 4;
    if constexpr (H_IN_LDS) {
        static_assert(kHCap >= kNearThreads, "a bond vector per thread");
        __syncthreads();
        hrvs[tid][0] = hrv[0]; hrvs[tid][1] = hrv[1]; hrvs[tid][2] = hrv[2];
    }

    // The point indices are formed again from the thread index where they
    // are needed after this point (a rare branch of the candidate loop and
    // the stores), so three indices do not stay live across the loop: one
    // register instead of three, and no spill.
    const auto point_index = [&](int &qx, int &qy, int &qz) {
        int t = tid;
        asm volatile("" : "+v"(t));   // opaque at each use: not hoisted out of the loop
        brick_lane<CUBE>(t, share, qx, qy, qz);
        qx += ix0;
        qy += iy0;
        qz += iz0;
    };
    float e_near = 0.f, dv_acc = 0.f, dq_acc = 0.f;
    int ccount = 0;
    const bool want_cmap = GENERAL && p.cmap != nullptr;
    const float *tab = p.tab;
    const bool want_e = p.e_slot >= 0;
    const float band = cf.near_band;
    // cos and sin of 1.24791 rad, the disordered-hydroxyl offset angle
    const float cdis = 0.31936680f, sdis = 0.94763168f;

    // H-bond codes of the pass, one word per atom class (lane hb holds
    // hcode[k][hb] in byte k), read with readlane instead of a load per atom.
    // Cross-lane reads (this one and the candidate index) happen only at the
    // top of a candidate iteration, where every lane of the wave is active:
    // a register reloaded from a spill under a partial exec mask would hold
    // stale values in the inactive lanes.
    const unsigned lane_chunk = 16u * (tid & (Q - 1));
    const bool last_chunk = (tid & (Q - 1)) == Q - 1;
    const int hcw = wlane < 7 ? (p.hcode[0][wlane] | p.hcode[1][wlane] << 8 | p.hcode[2][wlane] << 16 |
                                 p.hcode[3][wlane] << 24)
                              : 0;
    for (int cpage = 0; cpage < ncand; cpage += kCandCap) {   // pages of candidates
        if constexpr (PAGED) {
            if (cpage > 0) {
                __syncthreads();
                stage(cpage, -1);
                __syncthreads();
            }
        }
        const int cpn = min(ncand - cpage, kCandCap);
        const int cn = (cpn - first + share - 1) / share;   // this wave's: first, first + share, ...
        // candidate records go straight into scalar registers through the
        // constant address space (the atom array is read-only here).  The
        // wave holds 64 candidate indices in one register and loads the
        // next record's coordinates, class and index one candidate ahead,
        // which also brings both of its cache lines into the scalar cache.
        // The list holds byte offsets of the records (below 4 GiB, checked
        // when the plan is built), so a record's address is the array base
        // plus an unsigned 32-bit scalar, which the scalar loads take as
        // their offset operand: no 64-bit multiply-add per record.
        const AG_CONST char *cbase = reinterpret_cast<const AG_CONST char *>(as_const(p.atoms));
        const auto rec = [&](unsigned off) {
            return reinterpret_cast<const AG_CONST NearAtom *>(cbase + off);
        };
        for (int j0 = 0; j0 < cn; j0 += 64) {
            const int vcand = cand[min(j0 + wlane, cn - 1) * share + first];
            const int jn = min(64, cn - j0);
            unsigned off = (unsigned)__builtin_amdgcn_readlane(vcand, 0);
            double nx = rec(off)->x, ny = rec(off)->y, nz = rec(off)->z;
            int nmeta = rec(off)->meta, nindex = rec(off)->index;
            float nqe = rec(off)->qe, nvol = rec(off)->vol, nsolq = rec(off)->solq;
            for (int jj = 0; jj < jn; jj++) {
                // this record's address, formed once: its fields load from it
                // with immediate offsets in whichever branch needs them
                const AG_CONST NearAtom *ap = rec(off);
                asm volatile("" : "+s"(ap));
                const AG_CONST NearAtom &a = *ap;
                const double ax = nx, ay = ny, az = nz;
                const int ameta = nmeta, aindex = nindex;
                const float aqe = nqe, avol = nvol, asolq = nsolq;
                const unsigned hw = (unsigned)__builtin_amdgcn_readlane(hcw, (ameta >> 8) & 63);
                unsigned noff = (unsigned)__builtin_amdgcn_readlane(vcand, min(jj + 1, jn - 1));
                // the next loads may issue only once this record has arrived:
                // scalar loads complete out of order, so the wait for this
                // record would otherwise also wait for the next one
                asm volatile("" : "+s"(noff) : "s"(ameta), "s"(aindex), "s"(ax), "s"(ay), "s"(az), "s"(aqe), "s"(avol), "s"(asolq));
                nx = rec(noff)->x;
                ny = rec(noff)->y;
                nz = rec(noff)->z;
                nmeta = rec(noff)->meta;
                nindex = rec(noff)->index;
                nqe = rec(noff)->qe;
                nvol = rec(noff)->vol;
                nsolq = rec(noff)->solq;
                off = noff;   // a still names this record
                // geometry: FP64 difference as the reference forms it, FP32 after
                const double dx64 = ax - cx, dy64 = ay - cy, dz64 = az - cz;
                const float dxf = (float)dx64, dyf = (float)dy64, dzf = (float)dz64;
                // (1e-14 A^2 keeps the root's argument positive)
                const float r2 = __builtin_fmaf(dxf, dxf, __builtin_fmaf(dyf, dyf, __builtin_fmaf(dzf, dzf, 1.0e-14f)));
                // beyond 8.02 A: neither cutoff pass nor near e term.  A lane out of
                // range goes along where another is in range (the table reads are
                // shared) and adds zeros.
                const bool in = r2 <= 64.33f;
                if (!__ballot(in)) continue;
                // hardware rsq (1 ulp): 128 r is good to 5.5 x 2^-24 of itself, 3.4e-4
                // bins here, inside the guard band (a 1e-3 band sent 13 % of the
                // wave's atoms through FP64 for some lane, 4e-4 sends 5 %);
                // the same rsq is 1/r for the near e term and the unit vector
                float inv_r = __builtin_amdgcn_rsqf(r2);
                float r = r2 * inv_r;
                const float g = clamp_bins(r * 128.f);
                int bin = (int)g;
                bool cut = r > 8.0f;
                if (fabsf(g - rintf(g)) < kGuardBins) {
                    double rdx, rdy, rdz;
                    const double r64 = ref_dist(ax, ay, az, cx, cy, cz, rdx, rdy, rdz);
                    cut = r64 > 8.0;
                    bin = (int)(r64 * 128.0);
                    if (bin == AG_NEINT && !cut) bin = kNearExactRow;
                    r = (float)r64;
                    inv_r = __builtin_amdgcn_rcpf(fmaxf(r, 1.0e-6f));
                }
                // which of the pairs at 1,025 bins are the near kernel's: the far
                // kernel's own bin says
                bool no_e = false;   // (general forms, at spacings where the band reaches below 8 A)
                if (want_e && fabsf(g - (float)kFarBinMin) <= band) {
                    // the far kernel's coordinates of the atom and the point: run centre, offset in the run, y, z
                    // (one axis after the other: few registers beside the sums)
                    int q, qy, qz, unused;
                    point_index(unused, qy, unused);
                    float dyE = far_row(ay * 128.0, qy, cf.far_py, ney, spacing, s128);
                    asm volatile("" : "+v"(dyE));
                    point_index(unused, unused, qz);
                    float dzE = far_row(az * 128.0, qz, cf.far_pz, nez, spacing, s128);
                    asm volatile("" : "+v"(dzE));
                    point_index(q, unused, unused);
                    const int k = q % kFarK;
                    const float uE = (float)(ax * 128.0 - far_centre(q - k, kFarK, nex, spacing));
                    const bool near_e = far_bin4(uE, dyE, dzE, k, s128) < 4u * kFarBinMin;
                    if (!GENERAL || (bin >= AG_NEINT && bin != kNearExactRow))
                        bin = !near_e ? kNearZeroRow : bin >= kFarBinMin ? kNearEdgeRow : bin;
                    else no_e = !near_e;
                }
                // the tree build's radius queries (bhtree.cpp:341-362): FP32 point
                // and atom, each component within the radius, then the rounded
                // squared distance against the rounded squared radius
                bool in8 = false;
                float rB = 0.f;
                int bin_bh = 0;
                if (bh) {
                    // the tree build's query point: the grid point as float (main.cpp:2860)
                    const float e0 = (float)cx - (float)ax, e1 = (float)cy - (float)ay, e2 = (float)cz - (float)az;
                    const float a0 = fabsf(e0), a1 = fabsf(e1), a2 = fabsf(e2);
                    const float D = (e0 * e0 + e1 * e1) + e2 * e2;
                    in8 = a0 <= 8.f && a1 <= 8.f && a2 <= 8.f && D <= 64.f;
                    if (a0 <= 1.5f && a1 <= 1.5f && a2 <= 1.5f && D <= 2.25f) collide = true;
                    if (want_cmap) ccount += a0 <= ccf && a1 <= ccf && a2 <= ccf && D <= ccf2;
                    rB = sqrtf(D);   // correctly rounded, as the tree's sqrt of a float
                    bin_bh = (int)((double)rB * 128.0);
                }
                // The pairs' vdW/H-bond table rows, loaded here so that the loads
                // are in flight during the constriction, electrostatic and
                // directional work below.  The type's rows start at a scalar base,
                // a bin's row is a 32-bit byte offset from it; the bin is the one
                // Loop 2 uses (the tree build's FP32 distance in that mode).  A
                // pair past the cutoff reads the row of zeros.
                const int meta = ameta;
                const int type = meta & 0xff, hb = (meta >> 8) & 0xff, rexp = (meta >> 16) & 0xff;
                const bool dis = GENERAL && ((meta >> 24) & 1);
                const bool skip_atom = !p.has_affinity || (p.disorder_h && dis && type == p.hydrogen_type);   // uniform
                // whether the pair has terms (the plain form asks only where a class has
                // directional terms or mixes: its other rows are zeros)
                const auto selected = [&] {
                    return GENERAL ? in & !(bh ? !in8 : cut) & !skip_atom : (bin < AG_NEINT) | (bin == kNearExactRow);
                };
                const int row = !GENERAL ? bin : !selected() ? kNearZeroRow
                                : !bh ? bin : bin_bh >= AG_NEINT ? kNearExactRow : bin_bh;
                // H-bonding slots (main.cpp:3286-3374): the (probe, atom) case is a
                // set of 0/1 coefficients chosen per atom class, uniform across
                // the wave.  For a class that mixes in some slot, each lane reads
                // its own point's H-bond slots, and the lanes that would take that
                // chunk for the group read zeros.
                constexpr unsigned kMixBits = (HC_HRAMP | HC_MINMAX) * 0x01010101u;
                const unsigned codes = hw >> (dis ? 4 : 0);
                const bool mixes = (codes & kMixBits) != 0;   // uniform
                float4 E[Q], Eo;
                {
                    constexpr unsigned kTypeBytes = kNearRows * ROW * sizeof(float);
                    const char *trow = reinterpret_cast<const char *>(tab) + (size_t)type * kTypeBytes;
                    constexpr unsigned zero = kNearZeroRow * ROW * sizeof(float);
                    const unsigned roff = (unsigned)row * (unsigned)(ROW * sizeof(float));
                    unsigned at[4];
                    at[0] = (unsigned)group_lane<Q, 0>((int)roff) + lane_chunk;
                    at[1] = (unsigned)group_lane<Q, 1>((int)roff) + lane_chunk;
                    if constexpr (Q == 4) {
                        at[2] = (unsigned)group_lane<Q, 2>((int)roff) + lane_chunk;
                        at[3] = (unsigned)group_lane<Q, 3>((int)roff) + lane_chunk;
                    }
                    if (mixes) {
                        Eo = *reinterpret_cast<const float4 *>(trow + (roff + 16u * (Q - 1)));
    #pragma unroll
                        for (int j = 0; j < Q; j++) at[j] = last_chunk ? zero : at[j];
                    }
    #pragma unroll
                    for (int j = 0; j < Q; j++) E[j] = *reinterpret_cast<const float4 *>(trow + at[j]);
                }
                // electrostatic factor and sol_fn of the bin, one LDS read
                const float2 rsv = rs_s[bin];
                // constriction grid: atoms within the cutoff (main.cpp:2969-2973)
                if (want_cmap && !bh && in) {
                    if (fabsf(r - (float)p.ccut) < 1.0e-5f) {
                        double rdx, rdy, rdz;
                        ccount += ref_dist(ax, ay, az, cx, cy, cz, rdx, rdy, rdz) <= p.ccut;
                    } else {
                        ccount += r <= (float)p.ccut;
                    }
                }
                // electrostatics of pairs the far kernel leaves out
                if (want_e) {
                    // 1/max(r, 0.5) with r clamped at APPROX_ZERO
                    const float te = aqe * half_at_least(inv_r);
                    e_near = __builtin_fmaf(GENERAL && no_e ? 0.f : te, rsv.x, e_near);
                }
                // Loop 2 of the tree build takes the atoms its 8 A query returns,
                // at their FP32 distance (main.cpp:3019-3028)
                if (bh) {
                    r = rB;
                    inv_r = __builtin_amdgcn_rcpf(fmaxf(rB, 1.0e-6f));
                }
                float racc = 1.f, rdon = 1.f, Hramp = 1.f;
                // directional classes only (D1, A1, A2): the unit vector to the point
                constexpr unsigned kDirClasses = (1u << AG_HB_D1) | (1u << AG_HB_A1) | (1u << AG_HB_A2);
                if (((kDirClasses >> hb) & 1u) && selected()) {
                    const float dn0 = dxf * inv_r, dn1 = dyf * inv_r, dn2 = dzf * inv_r;
                    const float rv0 = unif(a.rv[0]), rv1 = unif(a.rv[1]), rv2 = unif(a.rv[2]);
                    const int aidx = aindex;
                    if (hb == AG_HB_D1 || (hb == AG_HB_A2 && !dis)) {
                        // cos(theta) of the D1 / ordered-A2 branches; FP64 near 0
                        float cos_t = -(dn0 * rv0) - dn1 * rv1 - dn2 * rv2;
                        bool pos;
                        if (fabsf(cos_t) < 1.0e-5f) {
                            double rdx, rdy, rdz;
                            double r64 = ref_dist(ax, ay, az, cx, cy, cz, rdx, rdy, rdz);
                            if (bh) r64 = (double)rB;   // the tree build's r (main.cpp:3026)
                            if (r64 < 1.0e-6) r64 = 1.0e-6;
                            const double ir = 1. / r64;
                            const double *rv64 = p.rvec64 + 3 * (size_t)aidx;
                            double c = 0.;
                            c -= rdx * ir * rv64[0];
                            c -= rdy * ir * rv64[1];
                            c -= rdz * ir * rv64[2];
                            pos = hb == AG_HB_D1 ? c > 0. : c >= 0.;
                            cos_t = (float)c;
                        } else {
                            pos = hb == AG_HB_D1 ? cos_t > 0.f : cos_t >= 0.f;
                        }
                        if (hb == AG_HB_D1) {
                            if (!pos) {
                                racc = 0.f;
                            } else {
                                const float c2 = cos_t * cos_t;
                                racc = rexp == 2 ? c2 : (rexp == 4 ? c2 * c2 : cos_t);
                                if (aidx != best_idx) {
                                    const float *const h = H_IN_LDS ? hrvs[tid] : hrv;
                                    float ct = h[0] * rv0 + h[1] * rv1 + h[2] * rv2;
                                    Hramp = hramp_value(__builtin_amdgcn_fmed3f(ct, -1.f, 1.f));
                                }
                            }
                        } else {
                            // Goodford lone-pair terms.  With x = dn.rv2 and
                            // y = (dn x rv2).rv / |dn x rv2|:
                            //   t0 = pi/2 - acos(x)         -> cos(t0) = sqrt(1 - x^2)
                            //   ti = |acos(y) - pi/2|       -> sin(2 ti) = 2|y| sqrt(1 - y^2)
                            // with dn a unit vector, 1 - x^2 = (1 - |rv2|^2) + |dn x rv2|^2: formed
                            // from x it loses all digits along the axis.
                            const float rw0 = unif(a.rv2[0]), rw1 = unif(a.rv2[1]), rw2 = unif(a.rv2[2]);
                            const float cr0 = __builtin_fmaf(dn1, rw2, -(dn2 * rw1)),
                                        cr1 = __builtin_fmaf(dn2, rw0, -(dn0 * rw2)),
                                        cr2 = __builtin_fmaf(dn0, rw1, -(dn1 * rw0));
                            const float cross2 = __builtin_fmaf(cr0, cr0, __builtin_fmaf(cr1, cr1, cr2 * cr2));
                            const float cos_t0 = __builtin_amdgcn_sqrtf(max_of(unif(a.rv2rest) + cross2, 0.f));
                            rdon = 0.f;
                            if (pos) {
                                const float yn = __builtin_fmaf(cr0, rv0, __builtin_fmaf(cr1, rv1, cr2 * rv2));
                                const float y = min_of(fabsf(yn) * __builtin_amdgcn_rsqf(max_of(cross2, 1.0e-6f)), 1.f);
                                const float s2 = y * __builtin_amdgcn_sqrtf(max_of(__builtin_fmaf(-y, y, 1.f), 0.f));
                                rdon = __builtin_fmaf(0.2f, s2, 0.9f) * cos_t0;
                            } else if (cos_t >= -0.34202f) {
                                const float u = 0.116978f - cos_t * cos_t;
                                rdon = 562.25f * (u * u * u) * cos_t0;
                            }
                        }
                    } else if (hb == AG_HB_A1) {
                        const float cos_t = -(dn0 * rv0) - dn1 * rv1 - dn2 * rv2;
                        rdon = cos_t <= 0.f ? 0.f : cos_t * cos_t;
                    } else if (hb == AG_HB_A2 && dis) {
                        // cos(theta - 1.24791) = c cos(1.24791) + sqrt(1 - c^2) sin(1.24791);
                        // theta <= 1.24791 + pi/2  <=>  c >= -sin(1.24791)
                        float c = -(dn0 * rv0) - dn1 * rv1 - dn2 * rv2;
                        c = fminf(fmaxf(c, -1.f), 1.f);
                        racc = 0.f;
                        rdon = 0.f;
                        if (c >= -sdis) {
                            const float cc = c * cdis + __builtin_amdgcn_sqrtf(fmaxf(1.f - c * c, 0.f)) * sdis;
                            rdon = (cc * cc) * (cc * cc);
                            racc = rdon;
                        }
                    }
                }  // directional classes
                const float S = !GENERAL ? rsv.y : !selected() ? 0.f : rs_s[row].y;   // sol_fn[min(bin, 1024)]
                // desolvation (main.cpp:3375-3390): slot m gains
                // (sp[m] vol + volp[m] solq) S per pair, i.e. sp[m] sum(vol S) +
                // volp[m] sum(solq S) over the point's pairs: two sums per point
                // instead of a term per slot, combined after the loop
                dv_acc = __builtin_fmaf(avol, S, dv_acc);
                dq_acc = __builtin_fmaf(asolq, S, dq_acc);
    #pragma unroll
                for (int j = 0; j < Q; j++) {
                    accT[j][0] += E[j].x;
                    accT[j][1] += E[j].y;
                    accT[j][2] += E[j].z;
                    accT[j][3] += E[j].w;
                }
                // The mix runs in scalar branches, one per slot.  A disordered
                // partner uses the hydrogen-type row at r - 1.10 A
                // (main.cpp:3313-3349), FP64 like the reference.
                if (mixes && selected()) {
                    const float e4[kHbSlots] = {Eo.x, Eo.y, Eo.z, Eo.w};
                    float Eh[kHbSlots] = {0.f, 0.f, 0.f, 0.f};
                    if (dis && p.hydrogen_type >= 0) {
                        double rdx, rdy, rdz;
                        const double r64 = bh ? (double)rB : ref_dist(ax, ay, az, cx, cy, cz, rdx, rdy, rdz);
                        const int hb_bin = min(max(0, (int)((r64 - 1.10) * 128.0)), AG_NEINT - 1);
                        const float4 v = reinterpret_cast<const float4 *>(
                            tab + ((size_t)p.hydrogen_type * kNearRows + hb_bin) * ROW)[Q - 1];
                        Eh[0] = v.x; Eh[1] = v.y; Eh[2] = v.z; Eh[3] = v.w;
                    }
    #pragma unroll
                    for (int k = 0; k < kHbSlots; k++) {
                        const int code = (codes >> (8 * k)) & 15;   // scalar
                        const float e = e4[k];
                        if (code & HC_PLAIN) acc_hb[k] += e;
                        if (!(code & (HC_HRAMP | HC_MINMAX))) continue;
                        const float f = (code & HC_RACC) ? racc : rdon;
                        const float rsph = __builtin_amdgcn_fmed3f(e * 0.01f, 0.f, 1.f);
                        const float mix = __builtin_fmaf(1.f - f, rsph, f);
                        if (code & HC_HRAMP)
                            acc_hb[k] = __builtin_fmaf((dis ? Eh[k] : e) * Hramp, mix, acc_hb[k]);
                        if (code & HC_MINMAX) {
                            const float v = e * mix;
                            hmin[k] = min_of(hmin[k], v);
                            hmax[k] = max_of(hmax[k], v);
                        }
                    }
                }
            }
        }
        if constexpr (!PAGED) break;
    }

    // each point's sums back to its lane, through LDS (the lists are done with)
    float acc[kMapSlots];
    {
        __syncthreads();
        constexpr int PITCH = ROW + 1, WAVE = 64 * PITCH;
        float *const tr = scratch_f + wave * WAVE;
        const int c = tid & (Q - 1), g0 = wlane - c;
#pragma unroll
        for (int j = 0; j < Q; j++)
#pragma unroll
            for (int s = 0; s < 4; s++) tr[(g0 + j) * PITCH + 4 * c + s] = accT[j][s];
        wave_sync();
#pragma unroll
        for (int k = 0; k < kHbSlots; k++) tr[wlane * PITCH + ROW - 4 + k] += acc_hb[k];
        if (shared) __syncthreads();
        else wave_sync();
#pragma unroll
        for (int m = 0; m < kMapSlots; m++) {
            if (m >= NPLAIN && m < kPlainSlots) continue;
            const int at = wlane * PITCH + (m < kPlainSlots ? m : ROW - 4 + (m - kPlainSlots));
            acc[m] = 0.f;
            if (!shared) {
                acc[m] = tr[at];
            } else if ((m & (share - 1)) == first) {   // the maps this wave stores
                for (int w = 0; w < share; w++) acc[m] += scratch_f[(wave - first + w) * WAVE + at];
            }
        }
    }
    if (shared) {   // the other sums of the sharing waves
        constexpr int VALUES = 5 + 2 * kHbSlots;
        static_assert(sizeof(NearLists) >= sizeof(float) * kNearThreads * VALUES, "room for the shared sums");
        __syncthreads();
        float *const mine = scratch_f + wave * (64 * VALUES) + wlane;
        mine[0] = e_near;
        mine[64] = dv_acc;
        mine[128] = dq_acc;
        mine[192] = __int_as_float(ccount);
        mine[256] = __int_as_float(collide);
#pragma unroll
        for (int k = 0; k < kHbSlots; k++) {
            mine[320 + 64 * k] = hmin[k];
            mine[320 + 64 * (kHbSlots + k)] = hmax[k];
        }
        __syncthreads();
        e_near = dv_acc = dq_acc = 0.f;
        ccount = 0;
        for (int w = 0; w < share; w++) {
            const float *const v = scratch_f + (wave - first + w) * (64 * VALUES) + wlane;
            e_near += v[0];
            dv_acc += v[64];
            dq_acc += v[128];
            ccount += __float_as_int(v[192]);
            collide |= __float_as_int(v[256]) != 0;
#pragma unroll
            for (int k = 0; k < kHbSlots; k++) {
                hmin[k] = min_of(hmin[k], v[320 + 64 * k]);
                hmax[k] = max_of(hmax[k], v[320 + 64 * (kHbSlots + k)]);
            }
        }
    }

    int qx, qy, qz;
    point_index(qx, qy, qz);
    if (qx < n1x && qy < n1y && qz < n1z) {
        // output pointers are formed here, after the candidate loop, so they
        // hold no registers during it; each wave of a shared cube stores
        // its part of the maps
        int *const cmap = p.cmap ? p.cmap + cf.pt_off : nullptr;
        float *const maps = p.maps + cf.map_off;
        const long long P = cf.P;
        const long long pt = (long long)qx + (long long)n1x * ((long long)qy + (long long)n1y * qz);
        const auto stores = [&](int k) { return (k & (share - 1)) == first; };
#pragma unroll
        for (int m = 0; m < kMapSlots; m++) {
            if ((m >= NPLAIN && m < kPlainSlots) || p.out_slot[m] < 0 || !stores(m)) continue;
            float v = acc[m] + __builtin_fmaf(p.sp[m], dv_acc, p.volp[m] * dq_acc);
            if (m >= kPlainSlots && hmin[m - kPlainSlots] < 999999.f)
                v += hmin[m - kPlainSlots] + fmaxf(hmax[m - kPlainSlots], 0.f);
            maps[(long long)p.out_slot[m] * P + pt] = v;
        }
        if (want_e && stores(0)) {
            if (p.far_part) {   // as k_far_sum adds them
                double v = e_near;
                for (int q = 0; q < cf.far_split; q++) v += (double)p.far_part[cf.part_off + q * P + pt];
                e_near = (float)v;
            }
            maps[(long long)p.e_slot * P + pt] = e_near;
        }
        if (cmap && stores(1)) cmap[pt] = ccount;
        if (p.collide && stores(2)) p.collide[cf.pt_off + pt] = collide ? 1 : 0;
        if (p.d_slot >= 0 && stores(3)) maps[(long long)p.d_slot * P + pt] = p.solpar_q * dv_acc;   // solpar_q sum(vol S)
    }
}

// The tree build's collision rule (main.cpp:2906-2927): a point within
// 1.5 A of a receptor atom has e = 0 and floating value 1.5 (Loop 1 is
// skipped there).  Runs after the near, far and floating-grid kernels.
__global__ void k_collide(long long P, const unsigned char *mask, float *emap, float *fmap) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P || !mask[i]) return;
    if (emap) emap[i] = 0.f;
    if (fmap) fmap[i] = 1.5f;
}

__global__ void k_fill(float *out, long long n, float v) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = v;
}

// Covalent maps (main.cpp:2866-2879): a Gaussian well around the
// attachment point, no receptor atoms involved.
struct CovParams {
    int n1[3], ne[3];
    double spacing;
    double pos[3], half_width, barrier;
    int n_cov;
    int slot[16];
    float *maps;
    long long P;
};

__global__ void k_covalent(CovParams c) {
    const long long pt = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (pt >= c.P) return;
    const int ix = (int)(pt % c.n1[0]);
    const int iy = (int)((pt / c.n1[0]) % c.n1[1]);
    const int iz = (int)(pt / ((long long)c.n1[0] * c.n1[1]));
    const double dx = c.pos[0] - (double)(ix - c.ne[0]) * c.spacing;
    const double dy = c.pos[1] - (double)(iy - c.ne[1]) * c.spacing;
    const double dz = c.pos[2] - (double)(iz - c.ne[2]) * c.spacing;
    double rcov = sqrt(dx * dx + dy * dy + dz * dz) / c.half_width;
    if (rcov < 1.0e-6) rcov = 1.0e-6;
    const float v = (float)(c.barrier * (1. - exp(-0.69314718055994530942 * rcov * rcov)));
    for (int k = 0; k < c.n_cov; k++) c.maps[(long long)c.slot[k] * c.P + pt] = v;
}

// Floating grid (main.cpp:2962-2966): the distance to the nearest receptor
// atom, each distance clamped at APPROX_ZERO.  A workgroup owns 8x8x8 points,
// two per lane.  No atom farther from the box than the smallest distance at which
// some atom is sure to be (to the box's farthest point) can be nearest to any of
// them: a first pass over the atoms finds that distance, a second packs the
// atoms within it (a hundred of 3,000 at protein density) into LDS, 256 tested
// at a time.  The distances and their minimum are those of every pair, bit for
// bit.  3,000 atoms, 81^3 points: 430 us (all pairs) -> 17.
constexpr int kFminEdge = 8;
struct FminParams {
    int n1[3], ne[3];
    float spacing;
    int nb[3];
    const float4 *atoms;          // (x, y, z, 0) grid frame, A
    int n_atoms;
    float *fmap;
};

__global__ void __launch_bounds__(256) k_fmin(FminParams p) {
    __shared__ float4 list[256];
    __shared__ int wave_n[2][4];
    __shared__ float wave_min[4];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int b = blockIdx.x;
    const int x0 = b % p.nb[0] * kFminEdge, y0 = b / p.nb[0] % p.nb[1] * kFminEdge,
              z0 = b / (p.nb[0] * p.nb[1]) * kFminEdge;
    const int ix = x0 + (tid & 7), iy = y0 + ((tid >> 3) & 7), iz = z0 + (tid >> 6);   // and iz + 4
    const auto at = [&](int i, int d) { return (float)(i - p.ne[d]) * p.spacing; };
    const float px = at(ix, 0), py = at(iy, 1), pz[2] = {at(iz, 2), at(iz + 4, 2)};
    const float lo[3] = {at(x0, 0), at(y0, 1), at(z0, 2)};
    const float hi[3] = {at(min(x0 + kFminEdge, p.n1[0]) - 1, 0), at(min(y0 + kFminEdge, p.n1[1]) - 1, 1),
                         at(min(z0 + kFminEdge, p.n1[2]) - 1, 2)};
    const float4 *__restrict__ atoms = p.atoms;
    float reach = 3.0e38f;
    for (int a = tid; a < p.n_atoms; a += 256) {
        const float4 q = atoms[a];
        const float dx = fmaxf(q.x - lo[0], hi[0] - q.x), dy = fmaxf(q.y - lo[1], hi[1] - q.y),
                    dz = fmaxf(q.z - lo[2], hi[2] - q.z);
        reach = fminf(reach, __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz)));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) reach = fminf(reach, __shfl_xor(reach, o));
    if (lane == 0) wave_min[wave] = reach;
    __syncthreads();
    // a few rounding errors of 2^-24 on either side; at most 3e38, finite
    reach = fminf(fminf(wave_min[0], wave_min[1]), fminf(wave_min[2], wave_min[3]));
    reach = fminf(reach, 3.0e38f) * (1.f + 0x1p-20f) + 1.0e-30f;
    float m2[2] = {3.0e38f, 3.0e38f};
    for (int a0 = 0, buf = 0; a0 < p.n_atoms; a0 += 256, buf ^= 1) {
        float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
        bool near = a0 + tid < p.n_atoms;
        if (near) {
            q = atoms[a0 + tid];
            const float dx = fmaxf(fmaxf(lo[0] - q.x, q.x - hi[0]), 0.f),
                        dy = fmaxf(fmaxf(lo[1] - q.y, q.y - hi[1]), 0.f),
                        dz = fmaxf(fmaxf(lo[2] - q.z, q.z - hi[2]), 0.f);
            near = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz)) <= reach;
        }
        const unsigned long long m = __ballot(near);
        if (lane == 0) wave_n[buf][wave] = __popcll(m);
        __syncthreads();   // and every wave is done with the last list
        int n = 0, at_i = __popcll(m & ((1ull << lane) - 1ull));
#pragma unroll
        for (int w = 0; w < 4; w++) {
            at_i += w < wave ? wave_n[buf][w] : 0;
            n += wave_n[buf][w];
        }
        if (n == 0) continue;
        if (near) list[at_i] = q;
        __syncthreads();
        for (int i = 0; i < n; i++) {
            const float4 c = list[i];
            const float dx = c.x - px, dy = c.y - py;
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const float dz = c.z - pz[k];
                m2[k] = fminf(m2[k], __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz)));
            }
        }
    }
    if (ix < p.n1[0] && iy < p.n1[1]) {
#pragma unroll
        for (int k = 0; k < 2; k++)
            if (iz + 4 * k < p.n1[2])
                p.fmap[(long long)ix + (long long)p.n1[0] * ((long long)iy + (long long)p.n1[1] * (iz + 4 * k))] =
                    p.n_atoms > 0 ? fmaxf(__builtin_amdgcn_sqrtf(m2[k]), 1.0e-6f) : 1.0e12f;
    }
}

__global__ void k_fmin_atoms(int n, const double *coord, float4 *out) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[i] = make_float4((float)coord[3 * i], (float)coord[3 * i + 1], (float)coord[3 * i + 2], 0.f);
}

// Bin audit (diagnostic, not part of a map set): for every (point, atom)
// pair compare the bin floor(128 r) the device path uses with the one the
// reference's FP64 distance gives.
//   far pairs  (the far kernel's FP32 bin >= 1025): the FP32 bin is used
//              as is, so every mismatch is a table-bin flip;
//   near pairs: the near kernel recomputes in FP64 whenever 128 r is within
//              kGuardBins of an integer, so a mismatch outside that band
//              would be an unguarded flip (expected: none).
struct AuditParams {
    int n1[3];
    FarPatch far;
    const double *coord;         // [n][3]
    int n_atoms;
    long long P;
    unsigned long long *out;     // [0] far pairs, [1] far flips, [2] near unguarded flips, [3] max flips/point
};

__global__ void __launch_bounds__(256) k_audit(AuditParams p) {
    const long long pt = (long long)blockIdx.x * 256 + threadIdx.x;
    unsigned long long far_pairs = 0, far_flips = 0, near_bad = 0;
    if (pt < p.P) {
        const int ix = (int)(pt % p.n1[0]);
        const int iy = (int)((pt / p.n1[0]) % p.n1[1]);
        const int iz = (int)(pt / ((long long)p.n1[0] * p.n1[1]));
        const double cx = (double)(ix - p.far.ne[0]) * p.far.spacing, cy = (double)(iy - p.far.ne[1]) * p.far.spacing,
                     cz = (double)(iz - p.far.ne[2]) * p.far.spacing;
        for (int a = 0; a < p.n_atoms; a++) {
            const int fb = (int)(far_bin4(p.coord[3 * a] * 128.0, p.coord[3 * a + 1] * 128.0, p.coord[3 * a + 2] * 128.0,
                                          p.far, ix, iy, iz) >> 2);
            double dx, dy, dz;
            const double r64 = ref_dist(p.coord[3 * a], p.coord[3 * a + 1], p.coord[3 * a + 2], cx, cy, cz, dx, dy, dz);
            const int b64 = min((int)(r64 * 128.0), AG_NDIEL - 1);
            if (fb >= kFarBinMin) {
                far_pairs++;
                far_flips += min(fb, AG_NDIEL - 1) != b64;
            } else {
                const float dxf = (float)dx, dyf = (float)dy, dzf = (float)dz;
                const float r2 = __builtin_fmaf(dxf, dxf, __builtin_fmaf(dyf, dyf, __builtin_fmaf(dzf, dzf, 1.0e-14f)));
                const float g = r2 * __builtin_amdgcn_rsqf(r2) * 128.f;
                if (fabsf(g - rintf(g)) >= kGuardBins && min((int)g, AG_NDIEL - 1) != b64) near_bad++;
            }
        }
    }
    // wave sums, then one atomic per wave
    for (int off = 32; off > 0; off >>= 1) {
        far_pairs += __shfl_xor(far_pairs, off);
        near_bad += __shfl_xor(near_bad, off);
    }
    unsigned long long mx = far_flips;
    unsigned long long sum_f = far_flips;
    for (int off = 32; off > 0; off >>= 1) {
        sum_f += __shfl_xor(sum_f, off);
        const unsigned long long o = __shfl_xor(mx, off);
        mx = o > mx ? o : mx;
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&p.out[0], far_pairs);
        atomicAdd(&p.out[1], sum_f);
        atomicAdd(&p.out[2], near_bad);
        atomicMax(&p.out[3], mx);
    }
}

// ---------------------------------------------------------------------------
// far kernel
// ---------------------------------------------------------------------------

// Bins at and beyond kFarLastBin all read r_eps[8191]: the reference clamps
// the index there (main.cpp:2956).
constexpr int kFarLastBin = AG_NDIEL - 1;

// How a far-kernel launch reads its table.
//   kFarTable   a bin's entry from LDS;
//   kFarClamped the same, offsets capped at the last entry: for launches where a
//               conformation's direct pairs may pass it (spacings of about 1 A
//               and more; the cap changes no other pair's value);
//   kFarFlat    one value from bin 1025 on (constant dielectric): no table, only
//               the test for the pairs the near kernel takes, and that only for
//               atoms near the patch (kFarFlatBeyond: pairs of the others).
enum : int { kFarTable = 0, kFarClamped = 1, kFarFlat = 2, kFarFlatBeyond = 3 };

// One pair of an atom with the 16 points of a lane's run, accumulated into
// part[]: the squared distance in bins^2 by the run-centre expansion, rsq,
// the bin's table offset in one fma and one and, the LDS read.
template <int KIND>
__device__ __forceinline__ void far_pair(const PlainF4 &at, float py, float pz, float floor2, float s128, float s2,
                                         const float *T, float *part) {
    const float dy = at.y - py, dz = at.z - pz;
    const float dyz2 = fmaxf(__builtin_fmaf(dy, dy, dz * dz), floor2);
    const float U = __builtin_fmaf(at.x, at.x, dyz2);
    const float us = at.x * s128;
    float W[kFarK / 2];
#pragma unroll
    for (int j = 0; j < kFarK / 2; j++) W[j] = __builtin_fmaf(s2, far_c2(kFarK / 2 + j), U);
    float rs[kFarK];
    unsigned off[kFarK];
#pragma unroll
    for (int k = 0; k < kFarK; k++) {
        const int j = k >= kFarK / 2 ? k - kFarK / 2 : kFarK / 2 - 1 - k;
        const float rb2 = __builtin_fmaf(us, far_m(k), W[j]);
        rs[k] = __builtin_amdgcn_rsqf(rb2);
        if (KIND == kFarFlat) rs[k] = bin4_of(rb2, rs[k]) >= 4u * kFarBinMin ? rs[k] : 0.f;
        if (KIND < kFarFlat) off[k] = bin4_of(rb2, rs[k]);
        if (KIND == kFarClamped) off[k] = min(off[k], 4u * kFarLastBin);
    }
    if (KIND >= kFarFlat) {   // the weight holds the table's value
#pragma unroll
        for (int k = 0; k < kFarK; k++) part[k] = __builtin_fmaf(at.w, rs[k], part[k]);
        return;
    }
    float tv[kFarK];
#pragma unroll
    for (int k = 0; k < kFarK; k++)
        tv[k] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(T) + off[k]);
#pragma unroll
    for (int k = 0; k < kFarK; k++) part[k] = __builtin_fmaf(at.w, rs[k] * tv[k], part[k]);
}

// Place among the levels of an atom's charge over the conformation's: level 0
// for ratios from sqrt(1/2) to 2 sqrt(2), one more for each factor of sqrt(1/2) below,
// the last for all that are smaller, and one stricter for each factor of sqrt(2) above.
__device__ __forceinline__ int far_level(float ratio) {
    const int l = 126 - (int)(__float_as_uint(ratio * ratio) >> 23);
    return min(max(l > 0 ? l : min(l + 3, 0), -kFarStrict) + kFarStrict, kFarStrict + kFarLevels - 1);
}

// A wave-uniform value moved to a scalar register.
__device__ __forceinline__ float sreg(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

__device__ __forceinline__ double sreg(double v) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

// Lane i's value, in a scalar register.
__device__ __forceinline__ float lane_of(float v, int i) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), i));
}

__device__ __forceinline__ unsigned long long lane_of(unsigned long long v, int i) {
    const unsigned lo = __builtin_amdgcn_readlane((int)v, i), hi = __builtin_amdgcn_readlane((int)(v >> 32), i);
    return (unsigned long long)hi << 32 | lo;
}

// Chebyshev nodes of [-1, 1]: cos((2i + 1) pi / 2n), in increasing order.
__host__ __device__ __forceinline__ constexpr float far_node5(int i) {
    return i == 0 ? -0.95105652f : i == 1 ? -0.58778525f : i == 2 ? 0.f : i == 3 ? 0.58778525f : 0.95105652f;
}
constexpr float kNode4a = 0.92387953f, kNode4b = 0.38268343f;   // the four: -a, -b, b, a

// Lagrange weight of x-node i at point k of a run: t = (k - 7.5) / 7.5.
__device__ __forceinline__ constexpr double far_wx(int i, int k) {
    const double t = (k - 0.5 * (kFarK - 1)) / (0.5 * (kFarK - 1));
    double w = 1.0;
    for (int j = 0; j < kFarNx; j++)
        if (j != i) w *= (t - (double)far_node5(j)) / ((double)far_node5(i) - (double)far_node5(j));
    return w;
}
// The four Lagrange weights of the y (or z) nodes at t in [-1, 1].
__device__ __forceinline__ void far_wy(double t, double w[4]) {
    constexpr double a = kNode4a, b = kNode4b;
    constexpr double ka = 1. / (2. * a * (a * a - b * b)), kb = 1. / (2. * b * (a * a - b * b));
    const double t2 = t * t, pb = (t2 - b * b) * ka, pa = (a * a - t2) * kb;
    w[0] = -pb * (t - a);
    w[1] = -pa * (t - b);
    w[2] = pa * (t + b);
    w[3] = pb * (t + a);
}

// Coarse boxes.  In a large receptor most atoms are far from many patches
// together, so they are summed at the nodes of a box of patches (2 x-runs and
// about 32 rows each way: 16 patches of 8 x 8), 8 x 8 x 8 nodes for 32,768 points
// instead of 16 times 80.  The sums go to the patches' own nodes by
// interpolation, and the far kernel leaves out the atoms in them.  20,000 atoms
// on 257^3 points: the far field 8.5 -> 4.4 ms, and with the patches outside the
// receptor as strict as k_far_reach has them 5.7 (boxes 1.33, transfer 0.02,
// patches 4.35).
__host__ __device__ __forceinline__ constexpr double box_node(int i) {   // Chebyshev nodes, increasing
    constexpr double c[4] = {0.98078528040323044913, 0.83146961230254523708, 0.55557023301960222474,
                             0.19509032201612826785};
    return i < 4 ? -c[i] : c[7 - i];
}
// Lagrange weight of node j at t.
__device__ __forceinline__ double box_weight(int j, double t) {
    double num = 1.0, den = 1.0;
#pragma unroll
    for (int m = 0; m < kBoxN; m++) {
        const double x = box_node(m);
        double xj = 0.0;
#pragma unroll
        for (int q = 0; q < kBoxN; q++) xj = q == j ? box_node(q) : xj;
        num *= m == j ? 1.0 : t - x;
        den *= m == j ? 1.0 : xj - x;
    }
    return num / den;
}

// The sums at a box's nodes of one part of the atoms beyond its distances, and
// which atoms those are.  A lane has the eight x-nodes of one (y, z) node; the
// atoms go one after the other, as the far kernel's direct pairs do.
template <bool FLAT>
__global__ void __launch_bounds__(kFarThreads) __attribute__((amdgpu_waves_per_eu(4))) k_far_boxes(FarParams p, int conf) {
    __shared__ float T[FLAT ? kFarStrict + kFarLevels : AG_NDIEL];
    __shared__ double XD[2 * kBoxNodes];   // 40 KiB in all: four workgroups per CU
    stamp_start(p.stamp);
    const AG_CONST ConfDev &cf = as_const(p.confs)[conf];
    const float flat = FLAT ? as_const(p.tab)[kFarLastBin] : 1.f;
    // the bins below the far kernel's are not read: the distances are there instead
    float *const level_r2 = T;
    static_assert(kFarStrict + kFarLevels <= kFarBinMin / 4 * 4, "room for the distances");
    for (int i = kFarBinMin / 4 + threadIdx.x; !FLAT && i < AG_NDIEL / 4; i += kFarThreads)
        reinterpret_cast<float4 *>(T)[i] = reinterpret_cast<const float4 *>(p.tab)[i];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const int part = blockIdx.x % cf.box_parts, box = blockIdx.x / cf.box_parts;
    const int ibx = box % cf.box_n[0], iby = box / cf.box_n[0] % cf.box_n[1], ibz = box / cf.box_n[0] / cf.box_n[1];
    // as strict as its strictest patch (every wave for itself; at most 2 x 5 x 5 patches)
    int shift = 0;
    {
        const int r = ibx * kBoxRuns + lane % kBoxRuns, y = iby * cf.box_py + lane / kBoxRuns % cf.box_py,
                  z = ibz * cf.box_pz + lane / (kBoxRuns * cf.box_py);
        if (lane < kBoxRuns * cf.box_py * cf.box_pz && r < cf.runs_per_row && y < cf.far_npy && z < cf.far_npz)
            shift = p.shift[cf.reach_off + r + (long long)cf.runs_per_row * (y + (long long)cf.far_npy * z)];
        for (int o = 32; o > 0; o >>= 1) shift = max(shift, __shfl_xor(shift, o));
    }
    if (threadIdx.x < kFarStrict + kFarLevels)
        level_r2[threadIdx.x] = reinterpret_cast<const float *>(&p.confs[conf].box_r2)[max((int)threadIdx.x - shift, 0)];
    __syncthreads();
    const int nx = kBoxRuns * kFarK, ny = cf.box_py * cf.far_py, nz = cf.box_pz * cf.far_pz;   // points of the box
    const double bx = sreg(far_centre(ibx * nx, nx, cf.ne[0], cf.spacing)),
                 by = sreg(far_centre(iby * ny, ny, cf.ne[1], cf.spacing)),
                 bz = sreg(far_centre(ibz * nz, nz, cf.ne[2], cf.spacing));
    const float hx = sreg(far_offset(nx - 1, nx, cf.s128)), hy = sreg(far_offset(ny - 1, ny, cf.s128)),
                hz = sreg(far_offset(nz - 1, nz, cf.s128));
    float cy = 0.f, cz = 0.f;   // this lane's y and z node
#pragma unroll
    for (int i = 0; i < kBoxN; i++) {
        cy = (lane & 7) == i ? hy * (float)box_node(i) : cy;
        cz = lane >> 3 == i ? hz * (float)box_node(i) : cz;
    }
    float d[kBoxN / 2], dq[kBoxN / 2];
#pragma unroll
    for (int j = 0; j < kBoxN / 2; j++) {
        d[j] = sreg(hx * (float)-box_node(j));
        dq[j] = sreg(d[j] * d[j]);
    }
    double sum[kBoxN];
    float acc[kBoxN];
#pragma unroll
    for (int j = 0; j < kBoxN; j++) {
        sum[j] = 0.;
        acc[j] = 0.f;
    }
    const float qscale = sreg(cf.far_qscale);
    const FarAtom *const atoms = p.atoms + cf.atom_base;
    const int n_atoms = cf.n_atoms, groups = (n_atoms + 63) / 64;
    unsigned long long *const mask = p.box_mask + cf.box_mask_off + (long long)box * groups;
    const int step = 64 * kFarWaves * cf.box_parts, a_first = 64 * (part * kFarWaves + wave);
    int n_acc = 0;
    FarAtom A{};
    if (a_first + lane < n_atoms) A = atoms[a_first + lane];
    for (int a0 = a_first; a0 < n_atoms; a0 += step) {
        const float4 at = make_float4((float)(A.x - bx), (float)(A.y - by), (float)(A.z - bz), A.w);
        const bool valid = a0 + lane < n_atoms;
        if (a0 + step + lane < n_atoms) A = atoms[a0 + step + lane];
        const float ex = fmaxf(fabsf(at.x) - hx, 0.f), ey = fmaxf(fabsf(at.y) - hy, 0.f),
                    ez = fmaxf(fabsf(at.z) - hz, 0.f);
        const bool beyond = __builtin_fmaf(ex, ex, __builtin_fmaf(ey, ey, ez * ez)) >= level_r2[far_level(at.w * qscale)];
        unsigned long long set = __ballot(beyond && valid);
        if (lane == 0) mask[a0 / 64] = set;
        n_acc += __popcll(set);
        while (set) {
            const int i = __builtin_ctzll(set);
            set &= set - 1;
            const float qx = lane_of(at.x, i), dy = lane_of(at.y, i) - cy, dz = lane_of(at.z, i) - cz;
            const float qw = FLAT ? lane_of(at.w, i) * flat : lane_of(at.w, i);
            const float U = __builtin_fmaf(qx, qx, __builtin_fmaf(dy, dy, dz * dz)), u2 = qx + qx;
            float rs[kBoxN], tv[kBoxN];
#pragma unroll
            for (int j = 0; j < kBoxN; j++) {
                const int h = j < kBoxN / 2 ? j : kBoxN - 1 - j;
                const float rb2 = __builtin_fmaf(j < kBoxN / 2 ? u2 : -u2, d[h], U + dq[h]);
                rs[j] = __builtin_amdgcn_rsqf(rb2);
                if (FLAT) continue;
                const unsigned off = min(bin4_of(rb2, rs[j]), 4u * kFarLastBin);
                tv[j] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(T) + off);
            }
#pragma unroll
            for (int j = 0; j < kBoxN; j++) acc[j] = __builtin_fmaf(qw, FLAT ? rs[j] : rs[j] * tv[j], acc[j]);
        }
        if (n_acc >= kFarAtomChunk) {
            n_acc = 0;
#pragma unroll
            for (int j = 0; j < kBoxN; j++) {
                sum[j] += (double)acc[j];
                acc[j] = 0.f;
            }
        }
    }
#pragma unroll
    for (int j = 0; j < kBoxN; j++) sum[j] += (double)acc[j];
    // waves 2 and 3 hand their sums to 0 and 1, then 1 to 0
    if (wave >= 2) {
#pragma unroll
        for (int j = 0; j < kBoxN; j++) XD[((wave - 2) * kBoxN + j) * 64 + lane] = sum[j];
    }
    __syncthreads();
    if (wave < 2) {
#pragma unroll
        for (int j = 0; j < kBoxN; j++) sum[j] += XD[(wave * kBoxN + j) * 64 + lane];
    }
    __syncthreads();
    if (wave == 1) {
#pragma unroll
        for (int j = 0; j < kBoxN; j++) XD[j * 64 + lane] = sum[j];
    }
    __syncthreads();
    if (wave == 0) {
        double *const out = p.box_sums + cf.box_off + (long long)blockIdx.x * kBoxNodes;
#pragma unroll
        for (int j = 0; j < kBoxN; j++) out[j * 64 + lane] = sum[j] + XD[j * 64 + lane];
    }
}

// The boxes' sums at their patches' nodes, one wave per patch: the parts
// added, then axis by axis 8 -> 5, 8 -> 4 and 8 -> 4 nodes.
__global__ void __launch_bounds__(64) k_far_down(FarParams p, int conf) {
    __shared__ double w[kFarNx + 2 * kFarNy][kBoxN], t[64][kFarNx], u[kBoxN][kFarNy][kFarNx];
    const AG_CONST ConfDev &cf = as_const(p.confs)[conf];
    const int patch = blockIdx.x, lane = threadIdx.x;
    const int prow = patch / cf.runs_per_row;
    const int pr = patch - prow * cf.runs_per_row, pzi = prow / cf.far_npy, pyi = prow - pzi * cf.far_npy;
    const int ib[3] = {pr / kBoxRuns, pyi / cf.box_py, pzi / cf.box_pz};
    const int box = ib[0] + cf.box_n[0] * (ib[1] + cf.box_n[1] * ib[2]);
    double c[kBoxN];
#pragma unroll
    for (int j = 0; j < kBoxN; j++) c[j] = 0.;
    for (int q = 0; q < cf.box_parts; q++) {
        const double *const in = p.box_sums + cf.box_off + ((long long)box * cf.box_parts + q) * kBoxNodes;
#pragma unroll
        for (int j = 0; j < kBoxN; j++) c[j] += in[j * 64 + lane];
    }
    // weights: the place of a patch's node in its box, in box half widths
    for (int k = lane; k < (kFarNx + 2 * kFarNy) * kBoxN; k += 64) {
        const int row = k / kBoxN, j = k % kBoxN;
        const int axis = row < kFarNx ? 0 : row < kFarNx + kFarNy ? 1 : 2;
        const int i = axis == 0 ? row : axis == 1 ? row - kFarNx : row - kFarNx - kFarNy;
        const int n = axis == 0 ? kFarK : axis == 1 ? cf.far_py : cf.far_pz;          // points of the patch
        const int m = axis == 0 ? kBoxRuns : axis == 1 ? cf.box_py : cf.box_pz;       // patches of the box
        const int at = axis == 0 ? pr - ib[0] * m : axis == 1 ? pyi - ib[1] * m : pzi - ib[2] * m;
        const double node = axis == 0 ? (i == 0 ? far_node5(0) : i == 1 ? far_node5(1) : i == 2 ? far_node5(2) : i == 3 ? far_node5(3) : far_node5(4))
                                      : (i & 2 ? 1. : -1.) * (i == 0 || i == 3 ? kNode4a : kNode4b);
        const double half = 0.5 * (n - 1), centre = at * n + half;
        const double big = 0.5 * (m * n - 1);
        w[row][j] = box_weight(j, (centre + half * node - big) / big);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kFarNx; i++) {
        double v = 0.;
#pragma unroll
        for (int j = 0; j < kBoxN; j++) v = __builtin_fma(w[i][j], c[j], v);
        t[lane][i] = v;
    }
    __syncthreads();
    for (int k = lane; k < kBoxN * kFarNy * kFarNx; k += 64) {
        const int i = k % kFarNx, y = k / kFarNx % kFarNy, jz = k / (kFarNx * kFarNy);
        double v = 0.;
#pragma unroll
        for (int j = 0; j < kBoxN; j++) v = __builtin_fma(w[kFarNx + y][j], t[jz * 8 + j][i], v);
        u[jz][y][i] = v;
    }
    __syncthreads();
    double *const out = p.box_patch + cf.box_patch_off + (long long)patch * kFarNodes;
    for (int k = lane; k < kFarNodes; k += 64) {
        const int i = k % kFarNx, y = k / kFarNx % kFarNy, z = k / (kFarNx * kFarNy);
        double v = 0.;
#pragma unroll
        for (int j = 0; j < kBoxN; j++) v = __builtin_fma(w[kFarNx + kFarNy + z][j], u[j][y][i], v);
        out[k] = v;
    }
}

// How much stricter a patch's distances have to be.  Interpolation replaces the
// table's steps by their mean, an error of a third of a step a pair, where the
// sum pair by pair only puts one pair in 6,000 on the wrong side of a step.
// Beside the pairs around a patch in or near the receptor that is nothing: their
// steps are larger by more than that.  Away from it, it shows: in the shell 12
// to 30 A outside, distances meant for the inside left up to 20 times the error
// of the all-pairs sum.  So each patch finds the largest error a pair summed there
// may have, max over the atoms of |charge| G(distance), and goes as many levels
// of 2^(-1/2) stricter as that is below what level 0 leaves (far_shape makes the
// table, 2 log2(level 0 / G) at each half A from the patch's centre).  A
// workgroup takes 16 patches, each 16 lanes' group of its 1,024 threads another of
// the atoms; once, when the plan is made, as it depends on the conformation
// alone (20,000 atoms, 18,513 patches: 193 us, 5,000 and 2,048: 17).
constexpr int kReachThreads = 1024, kReachPatches = 16;
__global__ void __launch_bounds__(kReachThreads) k_far_reach(FarParams p, int conf, const float *tables, unsigned char *shift) {
    constexpr int kParts = kReachThreads / kReachPatches;
    __shared__ float table[kReachTab];
    __shared__ float4 list[kReachThreads];   // x, y, z, level of the charge
    __shared__ float least_s[kParts][kReachPatches];
    const AG_CONST ConfDev &cf = as_const(p.confs)[conf];
    const int own = threadIdx.x % kReachPatches, part = threadIdx.x / kReachPatches;
    const int patches = cf.runs_per_row * cf.far_npy * cf.far_npz, mine = blockIdx.x * kReachPatches + own;
    const int patch = min(mine, patches - 1);
    const int prow = patch / cf.runs_per_row, pzi = prow / cf.far_npy;
    const float cx = (float)far_centre((patch - prow * cf.runs_per_row) * kFarK, kFarK, cf.ne[0], cf.spacing),
                cy = (float)far_centre((prow - pzi * cf.far_npy) * cf.far_py, cf.far_py, cf.ne[1], cf.spacing),
                cz = (float)far_centre(pzi * cf.far_pz, cf.far_pz, cf.ne[2], cf.spacing);
    if (threadIdx.x < kReachTab) table[threadIdx.x] = tables[(size_t)conf * kReachTab + threadIdx.x];
    const FarAtom *const atoms = p.atoms + cf.atom_base;
    float least = (float)kFarStrict;
    for (int a0 = 0; a0 < cf.n_atoms; a0 += kReachThreads) {
        const int n = min(kReachThreads, cf.n_atoms - a0);
        __syncthreads();   // the last atoms' readers are done
        if ((int)threadIdx.x < n) {
            const FarAtom q = atoms[a0 + threadIdx.x];
            list[threadIdx.x] = make_float4((float)q.x, (float)q.y, (float)q.z,
                                            -2.f * __builtin_amdgcn_logf(fabsf(q.w) * cf.far_qscale));
        }
        __syncthreads();
        for (int i = part; i < n; i += kParts) {
            const float4 q = list[i];
            const float dx = q.x - cx, dy = q.y - cy, dz = q.z - cz;
            const float d = __builtin_amdgcn_sqrtf(__builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz))) * (2.f / 128.f);
            least = fminf(least, table[(int)fminf(d, (float)(kReachTab - 1))] + q.w);   // (no charge: infinite, or NaN, which fminf drops)
        }
    }
    least_s[part][own] = least;
    __syncthreads();
    if (part == 0 && mine < patches) {
        for (int k = 1; k < kParts; k++) least = fminf(least, least_s[k][own]);
        shift[cf.reach_off + patch] = (unsigned char)(int)ceilf(fmaxf(least, 0.f));
    }
}

// Far-field electrostatics.  An item is one patch of rows (far_py x far_pz,
// one per lane of a wave) times one x-run of 16 points, and one of far_split
// parts of the atom list; the workgroup's four waves take the same points
// and a quarter of the part each (every fourth group of 64 atoms), and add
// up in a fixed order through LDS.
//
// Atoms near the patch's box (closer than their level's sqrt(far_r2)) go pair by pair
// through the dielectric table, as the reference sums them (main.cpp:2940-2982):
// the table sits in LDS at address 0, so a bin's byte offset is its LDS
// address, with zeros below bin 1025 for the pairs the near kernel takes.
//
// The others vary smoothly over the box (the host picks the distance so
// that a table step there is below 6.5e-5 of its value and the box subtends a
// small angle, smaller distances for smaller charges, far_radii, and larger ones
// away from the atoms, k_far_reach): their sum is formed at 5 x 4 x 4 Chebyshev nodes of
// the box with the same table, and interpolated to its points.  An atom then
// costs 80 terms instead of 1,024.  Four atoms go at once, one for each 16
// lanes; a lane takes the five x-nodes of one (y, z) node.
//
// The split follows the wave: one lane tests one atom, a ballot gives the
// direct atoms (a scalar loop, their records read from the lanes) and
// packs the others into the wave's LDS strip, all in index order, so results
// repeat and depend on the conformation alone.
//
// Measured against every pair through the table (and, in large boxes, the
// constant beyond 64 A), at protein density: 20,000 atoms on 257^3 points
// 62.2 -> 8.6 ms (5.7 with the coarse boxes), 5,000 on 127^3 2.00 -> 0.81 ms,
// 1,849 on 61^3 0.42 -> 0.11 ms.
// Of the 127^3 launch's wave instructions three quarters are direct pairs (28 %
// of all pairs), a quarter the nodes; it is bound by the vector unit (65 %
// busy) and the table reads in LDS (60 %, 3.9 conflict cycles each) together.
// Eight waves per workgroup instead of four: 0.94 ms, 9.7 ms on 257^3 (for 8.6).
//
// KIND: kFarTable, kFarClamped or kFarFlat.  Without the table 3,000 atoms on 81^3
// points take 336 us for 444.
// CELLS: the launch's first workgroup makes the plan's cell list, which the
// near kernel will want (small plans, whose parts the near kernel adds up).
constexpr int kFarLds = AG_NDIEL + 2 * 64 * kFarK;
template <int KIND, bool CELLS>
__global__ void __launch_bounds__(kFarThreads) __attribute__((amdgpu_waves_per_eu(4))) k_far(FarParams p, CellParams cp) {
    // 40 KiB: four workgroups per CU
    __shared__ float lds[kFarLds];
    if (CELLS && blockIdx.x == 0) {
        int *const cnt = reinterpret_cast<int *>(lds);
        cell_list<kFarThreads>(cp, cnt + kFarWaves, cnt);
        return;
    }
    if (!CELLS) stamp_start(p.stamp);
    float *const T = lds, *const X = lds + AG_NDIEL;
    static_assert(kFarBinMin == AG_NEINT + 1, "the table's zeros below end one bin into a float4");
    constexpr bool FLAT = KIND == kFarFlat;
    const float flat = FLAT ? as_const(p.tab)[kFarLastBin] : 1.f;
    for (int i = threadIdx.x; !FLAT && i < AG_NDIEL / 4; i += kFarThreads) {
        float4 v = reinterpret_cast<const float4 *>(p.tab)[i];
        if (i <= AG_NEINT / 4) v.x = 0.f;
        if (i < AG_NEINT / 4) v.y = v.z = v.w = 0.f;
        reinterpret_cast<float4 *>(T)[i] = v;
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int lane = threadIdx.x % 64;
    int item;
    if (p.queue) {
        if (threadIdx.x == 0) reinterpret_cast<int *>(X)[0] = p.item_base + atomicAdd(p.queue, 1);
        __syncthreads();
        item = reinterpret_cast<int *>(X)[0];
    } else {
        item = p.item_base + (CELLS ? xcd_chunked<16>(blockIdx.x - 1, gridDim.x - 1) : xcd_chunked<16>(blockIdx.x, gridDim.x));
    }
    __syncthreads();
    item = __builtin_amdgcn_readfirstlane(item);
    while (item < p.item_end) {
        const int ci = find_conf(as_const(p.tile_prefix), p.nconf, item);
        const AG_CONST ConfDev &cf = as_const(p.confs)[ci];
        const int n1x = cf.n1[0];
        const int local = item - as_const(p.tile_prefix)[ci];
        const int patch = local / cf.far_split, part_i = local - patch * cf.far_split;
        const int prow = patch / cf.runs_per_row;
        const int pzi = prow / cf.far_npy;
        const int ix0 = (patch - prow * cf.runs_per_row) * kFarK;
        const int iy0 = (prow - pzi * cf.far_npy) * cf.far_py, iz0 = pzi * cf.far_pz;
        const int ly = lane % cf.far_py, lz = lane / cf.far_py;
        const bool active = lz < cf.far_pz && iy0 + ly < cf.n1[1] && iz0 + lz < cf.n1[2];
        const int iy = iy0 + (active ? ly : 0), iz = iz0 + (active ? lz : 0);   // idle lanes: the patch's corner
        const float s128 = cf.s128;
        const float py = far_offset(iy - iy0, cf.far_py, s128), pz = far_offset(iz - iz0, cf.far_pz, s128);
        const float floor2 = far_floor(s128), s2 = s128 * s128;
        // the patch's box (whole, also where the grid ends inside it): centre and half widths
        const double bx = sreg(far_centre(ix0, kFarK, cf.ne[0], cf.spacing)),
                     by = sreg(far_centre(iy0, cf.far_py, cf.ne[1], cf.spacing)),
                     bz = sreg(far_centre(iz0, cf.far_pz, cf.ne[2], cf.spacing));
        const float my = 0.5f * (float)(cf.far_py - 1), mz = 0.5f * (float)(cf.far_pz - 1);
        const float hx = sreg(kFarMid * s128), hy = sreg(my * s128), hz = sreg(mz * s128);
        const float d1 = sreg(hx * far_node5(3)), d2 = sreg(hx * far_node5(4));
        const float d1q = sreg(d1 * d1), d2q = sreg(d2 * d2);
        float s[kFarK], c[kFarK], part[kFarK];
        double ns[kFarNx];
#pragma unroll
        for (int k = 0; k < kFarK; k++) s[k] = c[k] = part[k] = 0.f;
#pragma unroll
        for (int i = 0; i < kFarNx; i++) ns[i] = 0.;
        float4 *const strip = reinterpret_cast<float4 *>(X) + 64 * wave;
        static_assert(kFarStrict + kFarLevels <= 64, "a lane for each level");
        float *const level_r2 = X + 4 * 64 * kFarWaves + 64 * wave;   // the wave's copy, as strict as the patch is
        if (lane < kFarStrict + kFarLevels)
            level_r2[lane] = reinterpret_cast<const float *>(
                &p.confs[ci].far_r2)[max(lane - (int)p.shift[cf.reach_off + patch], 0)];
        wave_sync();
        const float qscale = sreg(FLAT ? cf.far_qscale / flat : cf.far_qscale);   // (zero charges: any level)
        const FarAtom *const atoms = p.atoms + cf.atom_base;
        const int n_atoms = cf.n_atoms;
        const int step = 64 * kFarWaves * cf.far_split;
        int n_part = 0;   // atoms in part[] since it was last flushed
        const int a_first = 64 * (part_i * kFarWaves + wave);
        // the coarse box's atoms are in its own sums
        const unsigned long long *box_mask = nullptr;
        if (cf.box_parts)
            box_mask = p.box_mask + cf.box_mask_off +
                       (long long)((n_atoms + 63) / 64) *
                           (ix0 / (kFarK * kBoxRuns) +
                            cf.box_n[0] * ((prow - pzi * cf.far_npy) / cf.box_py + cf.box_n[1] * (pzi / cf.box_pz)));
        // 64 groups of 64 atoms at a time: lane l has the set of the l-th's that are left
        for (int c0 = a_first; c0 < n_atoms; c0 += 64 * step) {
            unsigned long long todo = 0;
            {
                const int a = c0 + step * lane;
                if (a < n_atoms) {
                    const int nb = min(64, n_atoms - a);
                    todo = nb == 64 ? ~0ull : ((1ull << nb) - 1);
                    if (box_mask) todo &= ~box_mask[a / 64];
                }
            }
            unsigned long long live = __ballot(todo != 0);
            FarAtom A{};
            if (live) A = atoms[min(c0 + step * __builtin_ctzll(live) + lane, n_atoms - 1)];
            while (live) {
                const int group = __builtin_ctzll(live);
                live &= live - 1;
                const unsigned long long all = lane_of(todo, group);
                const float4 at = make_float4((float)(A.x - bx), (float)(A.y - by), (float)(A.z - bz), FLAT ? A.w * flat : A.w);
                if (live) A = atoms[min(c0 + step * __builtin_ctzll(live) + lane, n_atoms - 1)];
                const float ex = fmaxf(fabsf(at.x) - hx, 0.f), ey = fmaxf(fabsf(at.y) - hy, 0.f),
                            ez = fmaxf(fabsf(at.z) - hz, 0.f);
                const float box2 = __builtin_fmaf(ex, ex, __builtin_fmaf(ey, ey, ez * ez));
                const bool beyond = box2 >= level_r2[far_level(at.w * qscale)];
                const unsigned long long far_set = __ballot(beyond) & all;
                const unsigned long long past =
                    FLAT ? __ballot(box2 >= (float)(kFarBinMin + 1) * (float)(kFarBinMin + 1)) : 0;
                unsigned long long dir_set = ~far_set & all;
                if (far_set) {
                    const int nf = __popcll(far_set);
                    if ((far_set >> lane) & 1) strip[__popcll(far_set & ((1ull << lane) - 1))] = at;
                    // the last four filled up with zero weights
                    if (lane >= nf && lane < ((nf + 3) & ~3)) strip[lane] = make_float4(4096.f, 0.f, 0.f, 0.f);
                    wave_sync();
                    // this lane's y and z node (formed here: no register holds it through the direct loop)
                    int jl = lane;
                    asm volatile("" : "+v"(jl));
                    const int jy = jl & 3, jz = (jl >> 2) & 3;
                    const float ny = hy * ((jy & 2 ? 1.f : -1.f) * ((jy == 0 || jy == 3) ? kNode4a : kNode4b));
                    const float nz = hz * ((jz & 2 ? 1.f : -1.f) * ((jz == 0 || jz == 3) ? kNode4a : kNode4b));
                    float np[kFarNx];
#pragma unroll
                    for (int j = 0; j < kFarNx; j++) np[j] = 0.f;
                    for (int i = 0; i < nf; i += 4) {
                        const float4 q = strip[i + (jl >> 4)];
                        const float dy = q.y - ny, dz = q.z - nz;
                        const float U = __builtin_fmaf(q.x, q.x, __builtin_fmaf(dy, dy, dz * dz));
                        const float W1 = U + d1q, W2 = U + d2q, u2 = q.x + q.x;
                        const float rb2[kFarNx] = {__builtin_fmaf(u2, d2, W2), __builtin_fmaf(u2, d1, W1), U,
                                                   __builtin_fmaf(-u2, d1, W1), __builtin_fmaf(-u2, d2, W2)};
                        float rs[kFarNx], tv[kFarNx];
#pragma unroll
                        for (int j = 0; j < kFarNx; j++) {
                            rs[j] = __builtin_amdgcn_rsqf(rb2[j]);
                            if (FLAT) continue;
                            const unsigned off = min(bin4_of(rb2[j], rs[j]), 4u * kFarLastBin);
                            tv[j] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(T) + off);
                        }
#pragma unroll
                        for (int j = 0; j < kFarNx; j++) np[j] = __builtin_fmaf(q.w, FLAT ? rs[j] : rs[j] * tv[j], np[j]);
                    }
                    wave_sync();   // the strip is rewritten for the next 64 atoms
                    // (16 atoms of a lane at most: what a node's value loses here, the
                    // points near the patch's ends get up to three times over)
#pragma unroll
                    for (int j = 0; j < kFarNx; j++) ns[j] += (double)np[j];
                }
                if (dir_set) {
                    n_part += __popcll(dir_set);
                    do {
                        const int i = __builtin_ctzll(dir_set);
                        dir_set &= dir_set - 1;
                        const PlainF4 q{lane_of(at.x, i), lane_of(at.y, i), lane_of(at.z, i), lane_of(at.w, i)};
                        // (no point of the box within a bin of the near kernel's pairs)
                        if (FLAT && ((past >> i) & 1)) far_pair<kFarFlatBeyond>(q, py, pz, floor2, s128, s2, T, part);
                        else far_pair<KIND>(q, py, pz, floor2, s128, s2, T, part);
                    } while (dir_set);
                    if (n_part >= kFarAtomChunk) {
                        n_part = 0;
#pragma unroll
                        for (int k = 0; k < kFarK; k++) {
                            const float y = part[k] - c[k];
                            const float t = s[k] + y;
                            c[k] = (t - s[k]) - y;
                            s[k] = t;
                            part[k] = 0.f;
                        }
                    }
                }
            }
        }
        // the nodes' sums over the four atom groups, then the points' values
        // from all 80 nodes through the wave's strip, in FP64: 250 of the
        // wave's 40,000 operations, and one rounding instead of several
        double *const V = reinterpret_cast<double *>(strip);
        {
            double v[kFarNx];
#pragma unroll
            for (int j = 0; j < kFarNx; j++) {
                v[j] = ns[j];
                v[j] += __shfl_xor(v[j], 16);
                v[j] += __shfl_xor(v[j], 32);
            }
            if (lane < 16) {
                if (box_mask && wave == 0 && part_i == 0) {
                    const double *const more = p.box_patch + cf.box_patch_off + (long long)patch * kFarNodes + lane * kFarNx;
#pragma unroll
                    for (int j = 0; j < kFarNx; j++) v[j] += more[j];
                }
#pragma unroll
                for (int j = 0; j < kFarNx; j++) V[lane * kFarNx + j] = v[j];
            }
        }
        wave_sync();
        double g[kFarNx];
        {
            double wy[4], wz[4];
            far_wy(((double)(iy - iy0) - my) / my, wy);
            far_wy(((double)(iz - iz0) - mz) / mz, wz);
#pragma unroll
            for (int j = 0; j < kFarNx; j++) g[j] = 0.;
#pragma unroll
            for (int m = 0; m < 16; m++) {
                const double w = wy[m & 3] * wz[m >> 2];
#pragma unroll
                for (int j = 0; j < kFarNx; j++) g[j] = __builtin_fma(w, V[m * kFarNx + j], g[j]);
            }
        }
        // eight points at a time: the direct sums plus the interpolated ones;
        // waves 2 and 3 hand theirs to 0 and 1, then 1 to 0
        double *const XD = reinterpret_cast<double *>(X);
        const long long base = (long long)ix0 + (long long)n1x * ((long long)iy + (long long)cf.n1[1] * iz);
        float *const out = cf.far_split == 1 ? p.maps + cf.map_off + (long long)p.e_slot * cf.P
                                             : p.part + cf.part_off + (long long)part_i * cf.P;
#pragma unroll
        for (int k0 = 0; k0 < kFarK; k0 += 8) {
            double f[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                f[k] = (double)s[k0 + k] + ((double)part[k0 + k] - (double)c[k0 + k]);
#pragma unroll
                for (int j = 0; j < kFarNx; j++) f[k] = __builtin_fma(far_wx(j, k0 + k), g[j], f[k]);
            }
            __syncthreads();
            if (wave >= 2) {
#pragma unroll
                for (int k = 0; k < 8; k++) XD[((wave - 2) * 8 + k) * 64 + lane] = f[k];
            }
            __syncthreads();
            if (wave < 2) {
#pragma unroll
                for (int k = 0; k < 8; k++) f[k] += XD[(wave * 8 + k) * 64 + lane];
            }
            __syncthreads();
            if (wave == 1) {
#pragma unroll
                for (int k = 0; k < 8; k++) XD[k * 64 + lane] = f[k];
            }
            __syncthreads();
            if (wave == 0 && active) {
#pragma unroll
                for (int k = 0; k < 8; k++)
                    if (ix0 + k0 + k < n1x) {
                        const double v = f[k] + XD[k * 64 + lane];
                        float *const o = out + base + k0 + k;
                        if (p.wide) p.wide[base + k0 + k] = v;
                        else *o = cf.far_split == 1 ? (float)((double)*o + v) : (float)v;
                    }
            }
        }
        if (!p.queue) break;
        __syncthreads();
        if (threadIdx.x == 0) reinterpret_cast<int *>(X)[0] = p.item_base + atomicAdd(p.queue, 1);
        __syncthreads();
        item = __builtin_amdgcn_readfirstlane(reinterpret_cast<int *>(X)[0]);
        __syncthreads();
    }
}

// When a stream gets here.
__global__ void k_stamp(unsigned long long *stamp) { stamp_start(stamp); }

// The e map where the far field was summed beside the near one.
__global__ void __launch_bounds__(256) k_far_add(const double *wide, float *emap, long long P) {
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < P; i += (long long)gridDim.x * 256)
        emap[i] = (float)((double)emap[i] + wide[i]);
}

// The e map of conformations whose patches were shared by several
// workgroups: the near kernel's value plus the parts, in part order.  One
// workgroup column per conformation of the launch.
__global__ void __launch_bounds__(256) k_far_sum(FarParams p, int conf0) {
    const AG_CONST ConfDev &cf = as_const(p.confs)[conf0 + blockIdx.y];
    if (cf.far_split == 1) return;
    float *const emap = p.maps + cf.map_off + (long long)p.e_slot * cf.P;
    const float *const part = p.part + cf.part_off;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < cf.P; i += (long long)gridDim.x * 256) {
        double s = emap[i];
        for (int q = 0; q < cf.far_split; q++) s += (double)part[q * cf.P + i];
        emap[i] = (float)s;
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// context, plans and host orchestration
// ---------------------------------------------------------------------------


// Near-kernel layout chosen by the autotuner.
struct Tune {
    double cell_size = 4.0;     // cell edge of the cell list (A)
    bool cube = true;           // lanes of a wave on a 4x4x4 cube instead of an 8x8x1 slab
                                // (the cube measures faster on the 5,000-atom, 127^3 map set)
};


// Receptor conformations (one for a plan, many for a batch) on their grids,
// with a shared map set and tables, resident on one device.
struct ag_plan {
    explicit ag_plan(std::shared_ptr<DevPool> pl) : pool(std::move(pl)) {}
    std::shared_ptr<DevPool> pool;     // first: the buffers below draw on it
    ag_ctx *ctx = nullptr;
    int nconf = 0, N = 0, M = 0, T = 0, n_maps = 0, groups = 0;
    bool vina = false, persistent = false;
    long long P_total = 0;
    std::vector<ConfDev> confs;
    std::vector<int> brick_prefix, tile_prefix;
    int total_cells = 0, total_bricks = 0, total_tiles = 0;
    Tune tune;
    double tune_ms = 0.0;              // time the autotuner spent
    DevBuf confs_d{pool}, brick_prefix_d{pool}, tile_prefix_d{pool}, atom_conf_d{pool}, queue_d{pool};
    DevBuf coord{pool}, charge{pool}, vol{pool}, solpar{pool}, rvec{pool}, rvec2{pool}, type{pool}, hbond{pool},
        rexp{pool}, disorder{pool};
    DevBuf atom_cell{pool}, cell_count{pool}, cell_start{pool}, slot_atom{pool},
        near_atoms{pool}, far_atoms{pool}, fmin_atoms{pool};
    DevBuf tab{pool}, sol{pool}, reps{pool}, far_part{pool}, far_box{pool}, far_reach{pool}, status{pool};
    DevBuf collide{pool};              // tree build: collision mask per point
    bool want_collide = false;
    int e_index = -1;                  // e map slot, -1 if none
    AtomSrc src{};
    std::vector<NearParams> near;      // one per pass of 16 map slots
    int nplain = 12;                   // plain slots in use (4, 8 or 12)
    std::vector<int> cov_slots;
    double cov_pos[3] = {0, 0, 0}, cov_half_width = 1.0, cov_barrier = 0.0;
    bool want_fmap = false, want_cmap = false;
    std::vector<int> zero_slots;       // output maps that are all zero (Vina e/d)
    FarParams far{};
    bool run_far = false;
    bool has_boxes = false;            // some conformation's far field has coarse boxes
    bool far_flat = false;             // the electrostatic factor is one value from the far kernel's bins on
    bool beside = false;               // the far field may run beside the near one, into the context's far_wide
    double coeff_estat = 0.0;
    int far_grid = 0;                  // persistent far-kernel grid
    bool paged = false;                // near kernel in its paged form (a brick overflowed one LDS list)
    bool any_disorder = false;         // some atom flagged as a disordered hydroxyl
    // captured map set (persistent mode): the cell list and near field, then
    // the far field of conformations [0, far_split) and of [far_split,
    // nconf), as graphs launched back to back (the second far graph is
    // empty when far_split == nconf)
    hipGraphExec_t graph = nullptr, graph_far = nullptr, graph_far2 = nullptr;
    int far_split = 0;
    std::vector<float> reach_tables;   // k_far_reach's, on their way up
    std::shared_ptr<StatusPage> status_page;   // owner of report, if any
    MapReport *report = nullptr;       // pinned: what the kernels of a map set report
    float *g_maps = nullptr, *g_fmap = nullptr;
    int32_t *g_cmap = nullptr;
    void drop_graphs() {
        if (graph) (void)hipGraphExecDestroy(graph);
        if (graph_far) (void)hipGraphExecDestroy(graph_far);
        if (graph_far2) (void)hipGraphExecDestroy(graph_far2);
        graph = graph_far = graph_far2 = nullptr;
    }
    int *overflow_flag() const { return report ? &report->overflow : (int *)status.ptr; }
    unsigned long long *stamp(int phase) const { return report && !persistent ? &report->start[phase] : nullptr; }
    ~ag_plan() {
        drop_graphs();
        if (report) status_page->give_back(report);
    }
};

namespace agdev {

// The device address of `scratch` on `device` (current), looked up once
// per device and kept: every GPU holds its own copy of the array.
static void *scratch_address(int device) {
    static std::mutex mu;
    static std::vector<void *> addr;
    std::lock_guard<std::mutex> lk(mu);
    if ((int)addr.size() <= device) addr.resize(device + 1, nullptr);
    if (!addr[device]) {
        void *p = nullptr;
        HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        addr[device] = p;
    }
    return addr[device];
}

ag_status context_create(ag_ctx **out, int device) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0)
        ag::fail(AG_ERR_DEVICE, "no HIP device is available (this engine has no CPU fallback)");
    if (device < 0 || device >= n) ag::fail(AG_ERR_DEVICE, "HIP device index out of range");
    HIP_CHECK(hipSetDevice(device));
    ag_ctx *c = new ag_ctx();
    c->device = device;
    HIP_CHECK(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
    HIP_CHECK(hipStreamCreateWithFlags(&c->copy_stream, hipStreamNonBlocking));
    HIP_CHECK(hipStreamCreateWithFlags(&c->stream2, hipStreamNonBlocking));
    HIP_CHECK(hipEventCreateWithFlags(&c->cells_ev, hipEventDisableTiming));
    HIP_CHECK(hipEventCreateWithFlags(&c->near_ev, hipEventDisableTiming));
    HIP_CHECK(hipEventCreateWithFlags(&c->far_ev, hipEventDisableTiming));
    HIP_CHECK(hipEventCreateWithFlags(&c->far2_ev, hipEventDisableTiming));
    for (auto &e : c->ev) HIP_CHECK(hipEventCreate(&e));
    for (auto &e : c->chunk_ev) HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    HIP_CHECK(hipDeviceGetAttribute(&c->n_cu, hipDeviceAttributeMultiprocessorCount, device));
    int khz = 0;
    HIP_CHECK(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device));
    c->clock_khz = khz > 0 ? khz : 100000.0;
    c->scratch = scratch_address(device);
    *out = c;
    return AG_OK;
}

void *host_alloc_pinned(ag_ctx *c, size_t bytes) {
    HIP_CHECK(hipSetDevice(c->device));
    void *p = nullptr;
    if (hipHostMalloc(&p, bytes, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return p;
}

void host_free_pinned(void *p) {
    if (p) (void)hipHostFree(p);
}

void context_destroy(ag_ctx *c) {
    if (!c) return;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    if (c->copy_stream) (void)hipStreamSynchronize(c->copy_stream);
    if (c->stream2) (void)hipStreamSynchronize(c->stream2);
    if (c->cells_ev) (void)hipEventDestroy(c->cells_ev);
    if (c->near_ev) (void)hipEventDestroy(c->near_ev);
    if (c->far_ev) (void)hipEventDestroy(c->far_ev);
    if (c->far2_ev) (void)hipEventDestroy(c->far2_ev);
    if (c->stream2) (void)hipStreamDestroy(c->stream2);
    for (auto &e : c->ev)
        if (e) (void)hipEventDestroy(e);
    for (auto &e : c->chunk_ev)
        if (e) (void)hipEventDestroy(e);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    if (c->copy_stream) (void)hipStreamDestroy(c->copy_stream);
    delete c;
}

void context_timing(ag_ctx *c, float *ms) {
    for (int i = 0; i < 4; i++) ms[i] = c->last_ms[i];
}

template <typename T>
static T *upload(hipStream_t st, DevBuf &b, const T *src, size_t n) {
    T *d = (T *)b.get(sizeof(T) * n);
    if (n) HIP_CHECK(hipMemcpyAsync(d, src, sizeof(T) * n, hipMemcpyHostToDevice, st));
    return d;
}

static void validate(const ag_receptor *rec, const ag_grid *grid, const ag_mapset *ms, const ag_tables *tab,
                     bool vina) {
    const int N = rec->n_atoms, M = ms->n_atom_maps, T = tab->n_rec_types;
    if (N < 0 || N > AG_MAX_ATOMS) ag::fail(AG_ERR_BAD_INPUT, "atom count out of range");
    if (M < 0 || M + 2 > AG_MAX_MAPS) ag::fail(AG_ERR_BAD_INPUT, "map count out of range");
    if (T < 0 || T > AG_MAX_REC_TYPES) ag::fail(AG_ERR_BAD_INPUT, "receptor type count out of range");
    for (int d = 0; d < 3; d++)
        if (grid->n1[d] < 1 || grid->n1[d] > AG_MAX_GRID_PTS || grid->ne[d] < 0)
            ag::fail(AG_ERR_BAD_INPUT, "grid dimensions out of range");
    if (!(grid->spacing > 0)) ag::fail(AG_ERR_BAD_INPUT, "grid spacing must be positive");
    if (ms->constriction_grid && !(ms->constriction_cutoff <= 8.0))
        ag::fail(AG_ERR_UNSUPPORTED, "constriction_distance_cutoff above 8 A is not supported on the device");
    const int n_maps = M + (ms->elec_index >= 0) + (ms->dsolv_index >= 0);
    if (ms->n_maps != n_maps) ag::fail(AG_ERR_BAD_INPUT, "n_maps does not match the map set");
    if ((ms->elec_index >= 0 && ms->elec_index >= n_maps) || (ms->dsolv_index >= 0 && ms->dsolv_index >= n_maps))
        ag::fail(AG_ERR_BAD_INPUT, "e/d map slot out of range");
    if (N > 0 && (!rec->coord || !rec->charge || !rec->vol || !rec->solpar || !rec->type || !rec->hbond ||
                  !rec->rexp || !rec->rvector || !rec->rvector2 || !rec->disorder))
        ag::fail(AG_ERR_BAD_INPUT, "receptor arrays missing");
    for (int i = 0; i < N; i++) {
        if (rec->type[i] < 0 || rec->type[i] >= T) ag::fail(AG_ERR_BAD_INPUT, "atom type index out of range");
        if (rec->hbond[i] < 0 || rec->hbond[i] > 6) ag::fail(AG_ERR_BAD_INPUT, "atom hbond class out of range");
    }
    if (vina && ms->separate_desolvation)
        ag::fail(AG_ERR_UNSUPPORTED, "Vina-potential maps do not combine with separate_desolvation_maps");
    if (ms->bhtree < 0 || ms->bhtree > 2) ag::fail(AG_ERR_BAD_INPUT, "bhtree mode must be 0, 1 or 2");
    if (vina && ms->bhtree) ag::fail(AG_ERR_UNSUPPORTED, "Vina-potential maps have no tree-build mode");
    if (M > 0 && !vina) {
        bool any_h = false;
        for (int i = 0; i < N && !any_h; i++) any_h = rec->hbond[i] == AG_HB_DS || rec->hbond[i] == AG_HB_D1;
        if (!any_h) ag::fail(AG_ERR_NO_DONOR_H, "no closestH atom was found");
    }
    if (ms->hydrogen_type < -1 || ms->hydrogen_type >= T) ag::fail(AG_ERR_BAD_INPUT, "hydrogen type index out of range");
    if (M > 0 && !ms->maps) ag::fail(AG_ERR_BAD_INPUT, "map descriptors missing");
    if (M > 0 && T > 0 && !tab->e_vdw_hb) ag::fail(AG_ERR_BAD_INPUT, "vdW/H-bond tables missing");
    if (!tab->sol_fn || (ms->dddiel && !tab->r_eps)) ag::fail(AG_ERR_BAD_INPUT, "desolvation/dielectric tables missing");
}

// Role of map m: the second map of each separate-desolvation pair carries
// that type's desolvation (main.cpp:3385).
static int map_role(const ag_mapset *ms, int m) {
    if (ms->maps[m].is_covalent) return ROLE_COV;
    if (!ms->separate_desolvation) return ROLE_AFF | ROLE_DES;
    int k = 0;
    while (k < m) k += ms->maps[k].is_covalent ? 1 : 2;
    return k == m ? ROLE_AFF : ROLE_DES;
}

// H-bond case of (probe class mh, atom class ah) (main.cpp:3286-3374).
static int hb_case(int mh, int ah) {
    const bool atom_don = (ah == 1 || ah == 2 || ah == 6);
    if ((mh == 3 || mh == 5 || mh == 6) && atom_don) return HBC_ACC_PROBE;
    if ((mh == 4 || mh == 6) && atom_don) return HBC_MINMAX_RACC;
    if ((mh == 1 || mh == 2 || mh == 6) && (ah > 2 || ah == 6)) return HBC_DON_PROBE;
    return HBC_PLAIN;
}

static void launch_near(const ag_plan &p, int grid, const NearParams &np, hipStream_t st) {
    // the plain form takes a band that stays past 8 A (spacings up to about 50 A)
    const bool wide = std::any_of(p.confs.begin(), p.confs.end(), [](const ConfDev &c) { return c.near_band > 0.9f; });
#define AG_NEAR(NP, CB)                                                                 \
    do {                                                                                \
        if (p.paged) k_near<NP, CB, kNearPaged><<<grid, kNearThreads, 0, st>>>(np);     \
        else if (np.bhtree || np.cmap || p.any_disorder || wide)                        \
            k_near<NP, CB, kNearGeneral><<<grid, kNearThreads, 0, st>>>(np);            \
        else k_near<NP, CB, kNearPlain><<<grid, kNearThreads, 0, st>>>(np);             \
    } while (0)
    if (p.tune.cube) {
        if (p.nplain == 4) AG_NEAR(4, true);
        else if (p.nplain == 8) AG_NEAR(8, true);
        else AG_NEAR(12, true);
    } else {
        if (p.nplain == 4) AG_NEAR(4, false);
        else if (p.nplain == 8) AG_NEAR(8, false);
        else AG_NEAR(12, false);
    }
#undef AG_NEAR
    HIP_CHECK(hipGetLastError());
}

// How the far kernel treats a conformation: the distance (bins) past which
// atoms are interpolated, the shape of its patches, and how many workgroups
// share a patch's atoms.  All of it depends on the conformation and the
// tables alone, so its maps are the same in a batch as in a plan of its own.
struct FarShape {
    float radius2[kFarStrict + kFarLevels] = {};
    float reach[kReachTab] = {};   // k_far_reach's table
    float qscale = 0.f;
    bool clamp = false;
    int clamp_from = kFarStrict + 1;   // least shift of a patch at which it is needed (plan_build)
    int py = 8, pz = 8, split = 1;
    // coarse boxes (ConfDev::box_*): parts (0: none), patches along y and z
    int box_parts = 0, box_py = 4, box_pz = 4;
    float box_radius2[kFarStrict + kFarLevels] = {};
};

// Least distance (A) of a level whatever the table (far_radii): 48.75 spacings,
// 6.5 half-lengths of an x-run, for the 1/r, 75 where the table has no steps
// at all (constant dielectric), whose sum has no table error beside the
// interpolation's.  A level allows sqrt(2) times the error of the one
// before: with five x-nodes 2^-0.1 of the distance from the run's centre, with
// the Mehler-Solmajer dielectric's steps (they fall by e in 3.2 A) 1.1 A.  The
// near kernel has the pairs up to 8.01 A.
static double far_floor_radius(bool flat, double spacing, int level, int nodes, double half_points) {
    // (coarse boxes: far_boxes adds what their nodes need)
    const double half = half_points * spacing, g = std::pow(2.0, -level / (2.0 * nodes));
    const double z = nodes == kBoxN ? 1.0 : flat ? 11.0 : 7.5;
    if (flat) return std::max({8.25, 20.0 * g, (z * g - 1.0) * half});
    const double base = std::min(21.0, std::max(18.5, 26.0 - 20.0 * spacing)) - 1.1 * level;
    return std::max({8.25, base, (z * g - 1.0) * half});
}

static bool flat_table(const std::vector<float> &reps) {
    return std::all_of(reps.begin() + kFarBinMin, reps.end(), [&](float v) { return v == reps.back(); });
}

// Distances (A) past which an atom's term varies over a patch of a grid of
// the given spacing the way 5 x 4 x 4 nodes follow, for each level of its charge.
// Level 0: (a) no table step beyond it exceeds 6.5e-5 of the value there, (b)
// 5 Chebyshev nodes over any x-run's length beyond it reproduce the table to
// 1e-5, and (c) it is at least far_floor_radius.  An atom of level l has at
// most 2^(-l/2) of the reference charge, so its term may be off by 2^(l/2)
// times as much, and (a) and (b) ask for that.  Bins from 8191 on hold one
// value, so past 64 A only (c) is asked for.
// With the Mehler-Solmajer dielectric the steps decide: they leave 2e-7 of
// the e map (2-norm, 5,000-atom protein) at 20 A, 5e-7 at 18 A and 8e-7 at 16 A,
// beside the 6e-7 that FP32 bins of the direct pairs leave.  The floor and the
// reference charge keep the map's error below the all-pairs sum's (whose
// coordinates were rounded in the grid's frame): 6.2e-7 for 6.9e-7 at 0.25 A (2,743
// atoms), at 0.375 A 9.5e-7 for 1.07e-6 (5,000 atoms) and 1.28e-6 for 1.31e-6 (20,000,
// 257^3 points).  That is a whole map's, which points in and at the receptor make
// up; outside it k_far_reach takes the distances of stricter levels.  One distance for every charge: 3 % less error, 830 us instead of 772
// for 5,000 atoms on 127^3 points, 460 instead of 430 for 3,000 on 81^3 in a constant
// dielectric.
static void far_radii(const std::vector<float> &reps, double spacing, int nodes, double half_points,
                      double radius[kFarLevels]) {
    const bool flat = flat_table(reps);
    const double run = 2.0 * half_points * spacing * 128.0;   // bins along it
    const auto node = [&](int i) { return nodes == kBoxN ? box_node(i) : (double)far_node5(i); };
    const auto g = [&](double bin) {                     // the table as a function, between bin centres
        const double y = std::min(std::max(bin - 0.5, 0.0), (double)(AG_NDIEL - 1));
        const int k = std::min((int)y, AG_NDIEL - 2);
        return reps[k] + (y - k) * ((double)reps[k + 1] - reps[k]);
    };
    double W[17][kBoxN];
    for (int q = 0; q <= 16; q++)
        for (int i = 0; i < nodes; i++) {
            W[q][i] = 1.0;
            for (int j = 0; j < nodes; j++)
                if (j != i) W[q][i] *= (-1.0 + q / 8.0 - node(j)) / (node(i) - node(j));
        }
    double floor_r[kFarLevels], ok[kFarLevels];
    for (int l = 0; l < kFarLevels; l++) {
        floor_r[l] = far_floor_radius(flat, spacing, l, nodes, half_points);
        ok[l] = (AG_NDIEL - 1) / 128.0 + 1.0 / 64.0;
    }
    // outwards in: a level's distance is the last before its first fault
    int first = 0, bin = AG_NDIEL - 1;   // levels below first have ended
    for (double r = AG_NDIEL - 1; first < kFarLevels; r -= 32.0) {
        double step = 0.0, off = 0.0;
        for (; bin > kFarBinMin && bin > r; bin--)
            step = std::max(step, std::fabs((double)reps[bin - 1] - reps[bin]) / std::fabs((double)reps[bin]));
        double f[kBoxN];
        for (int i = 0; i < nodes; i++) f[i] = g(r + 0.5 * run * (1.0 + node(i)));
        for (int q = 0; q <= 16; q++) {
            double v = 0.0;
            for (int i = 0; i < nodes; i++) v += W[q][i] * f[i];
            const double want = g(r + run * (q / 16.0));
            off = std::max(off, std::fabs(v - want) / std::fabs(want));
        }
        for (int l = first; l < kFarLevels; l++) {
            const bool good = step <= 6.5e-5 * std::pow(2.0, 0.5 * l) && off <= 1.0e-5 * std::pow(2.0, 0.5 * l);
            if (good && r >= floor_r[l] * 128.0 - 64.0) ok[l] = r / 128.0;
            else if (l == first) first++;   // the levels end in order
        }
    }
    for (int l = 0; l < kFarLevels; l++) radius[l] = std::max(floor_r[l], ok[l]);
}

// The table as a function of the distance (A), over the distance.
static double far_term(const std::vector<float> &reps, double r) {
    const double y = std::min(std::max(r * 128.0 - 0.5, 0.0), (double)(AG_NDIEL - 1));
    const int k = std::min((int)y, AG_NDIEL - 2);
    return (reps[k] + (y - k) * ((double)reps[k + 1] - reps[k])) / r;
}

// The interpolation along an axis: its nodes, and their weights at the ends and
// between them, where it is furthest off.
struct FarNodes {
    int n;
    double node[kBoxN], at[kBoxN + 1], weight[kBoxN + 1][kBoxN];
    explicit FarNodes(int count) : n(count) {
        const double four[4] = {-kNode4a, -kNode4b, kNode4b, kNode4a};
        for (int i = 0; i < n; i++) node[i] = n == kBoxN ? box_node(i) : n == kFarNx ? (double)far_node5(i) : four[i];
        for (int q = 0; q <= n; q++) {
            at[q] = q == 0 ? -1.0 : q == n ? 1.0 : 0.5 * (node[q - 1] + node[q]);
            for (int i = 0; i < n; i++) {
                weight[q][i] = 1.0;
                for (int j = 0; j < n; j++)
                    if (j != i) weight[q][i] *= (at[q] - node[j]) / (node[i] - node[j]);
            }
        }
    }
};
static const FarNodes kFarAxisX(kFarNx), kFarAxisY(kFarNy), kBoxAxis(kBoxN);

// Its error over an axis of half-length `half` (A), for an atom r off the box: ahead
// of it, beside its middle and beside its end.
static double far_axis_error(const std::vector<float> &reps, double r, double half, const FarNodes &x) {
    double worst = 0.0;
    for (int place = 0; place < 3; place++) {
        const auto f = [&](double t) {
            const double a = half * (place == 1 ? t : 1.0 + t);
            return far_term(reps, place == 0 ? r + a : std::sqrt(r * r + a * a));
        };
        double v[kBoxN];
        for (int i = 0; i < x.n; i++) v[i] = f(x.node[i]);
        for (int q = 0; q <= x.n; q++) {
            double s = 0.0;
            for (int i = 0; i < x.n; i++) s += x.weight[q][i] * v[i];
            worst = std::max(worst, std::fabs(s - f(x.at[q])));
        }
    }
    return worst;
}

// The largest table step beyond a distance, over that distance.
struct FarError {
    const std::vector<float> &reps;
    std::vector<float> step;      // largest step beyond k / 2 A, over the distance
    explicit FarError(const std::vector<float> &tab) : reps(tab), step(129, 0.f) {
        for (int k = 127; k >= 0; k--) {
            float s = 0.f;
            for (int b = std::max(64 * k, 1); b < 64 * (k + 1); b++) s = std::max(s, std::fabs(tab[b] - tab[b - 1]));
            step[k] = std::max(step[k + 1], s / std::max(0.5f, 0.5f * (float)k));
        }
    }
    double steps(double r) const { return step[std::min((int)(2.0 * r), 128)]; }
};

// What a patch leaves of the term of an atom r off it: half of the steps each way and
// the nodes' error, the half-lengths of its axes given.
static double far_error(const FarError &e, double r, const double half[2]) {
    const double nodes = std::max(far_axis_error(e.reps, r, half[0], kFarAxisX), far_axis_error(e.reps, r, half[1], kFarAxisY));
    return std::hypot(e.steps(r) / std::sqrt(12.0), nodes);
}

// Distances at which error(r) keeps to h0 2^(-n/2), h0 2^(-(n-1)/2), ...: from
// `most` inwards to r0, so that nothing beyond a distance is worse, between two hops
// as the error's logarithm has it.
template <typename F>
static void far_distances(F &&error, double r0, double most, double hop, double h0, int n, int levels, double *radius) {
    for (int l = 0; l < levels; l++) radius[l] = std::max(most, r0);
    int first = 0;   // levels before it have ended
    double outer = 0.0;
    for (double r = most; r > r0 && first < levels; r -= hop) {
        const double h = error(r);
        for (int l = first; l < levels; l++) {
            const double allowed = h0 * std::pow(2.0, 0.5 * (l - n));
            if (h <= allowed) {
                radius[l] = r;
            } else if (l == first) {
                const double x = std::log(h / allowed) / std::log(h / outer);
                if (r < most && x >= 0.0 && x < 1.0) radius[l] = r + hop * x;
                first++;
            }
        }
        outer = h;
    }
}

// Share of the pairs that an all-pairs sum in FP32 puts on the wrong side of a
// table step (5,000 atoms on 127^3 points, 0.375 A; fewer on finer grids), what its
// roundings leave of a term (in wider patches the nodes' error is the same for many
// atoms, and counts for more), and levels between one such pair and a patch's sum
// over many.  Chosen so that the error is the all-pairs sum's or less in the shells
// around receptors of 600 to 20,000 atoms: 0.8 to 0.9 times it at 0.375 A, 1.0 in the
// shell 16 to 20 A off (1.15 with a margin of 3; without the stricter levels 13 to
// 16 times).  20,000 atoms on 257^3 points, two thirds of them outside the
// receptor: 9.1 ms, without 7.9 (10.9 with a rounding of 6e-8, which does not show);
// boxes of which little is outside take the same time.
constexpr double kFarFlips = 1.6e-4, kFarRounding = 4.0e-7, kFarMargin = 4.0;

static FarShape far_shape(const ag_grid &g, int n_atoms, const double radius[kFarLevels], const FarError &err,
                          const double *coord, const double *charge, double coeff) {
    FarShape f;
    double q2 = 0.0;
    for (int a = 0; a < n_atoms; a++) q2 += charge[a] * charge[a];
    const double ref = kFarQRef * std::sqrt(q2 / std::max(1, n_atoms)) * std::fabs(coeff) * 128.0;
    f.qscale = ref > 0.0 ? (float)(1.0 / ref) : 0.f;
    // patches of 6 to 10 rows along y and what 64 lanes leave along z: the
    // shape that needs the fewest, the squarest of equals
    int best = INT32_MAX, best_d = 0;
    for (int py = 6; py <= 10; py++) {
        const int pz = 64 / py;
        const int n = ((g.n1[1] + py - 1) / py) * ((g.n1[2] + pz - 1) / pz), d = std::abs(py - pz);
        if (n < best || (n == best && d < best_d)) {
            best = n;
            best_d = d;
            f.py = py;
            f.pz = pz;
        }
    }
    // the stricter levels, and the pair sum's error over the distance
    const double half[2] = {kFarMid * g.spacing, 0.5 * (std::max(f.py, f.pz) - 1) * g.spacing};
    const double h0 = far_error(err, radius[0], half);
    double strict[kFarStrict];
    const double s = g.spacing * 128.0;
    const double diag = s * std::sqrt((double)((kFarK - 1) * (kFarK - 1) + (f.py - 1) * (f.py - 1) +
                                               (f.pz - 1) * (f.pz - 1)));
    // up to where direct pairs reach the table's end, if not 17 half-lengths
    const double inside = (kFarLastBin - 5.0 - diag) / 128.0;
    far_distances([&](double r) { return far_error(err, r, half); }, radius[0], std::max(inside, 17.0 * half[0]),
                  std::max(4.0, half[0] / 2.0), h0, kFarStrict, kFarStrict, strict);
    const double flips = kFarFlips * std::min(1.0, std::pow(g.spacing / 0.375, 4));
    const double rounding = kFarRounding * std::min(1.0, 0.375 * 0.375 / (g.spacing * g.spacing));
    for (int k = 0; k < kReachTab; k++) {
        const double d = std::max(1.0, 0.5 * k), step = std::sqrt(flips) * err.steps(std::max(d, 8.0)),
                     round = rounding * std::fabs(far_term(err.reps, d));
        f.reach[k] = (float)(2.0 * std::log2(std::max(h0, 1e-300) / std::max(std::hypot(step, round), 1e-300)) + kFarMargin);
    }
    for (int l = 0; l < kFarStrict + kFarLevels; l++) {
        const double d = 128.0 * (l < kFarStrict ? strict[l] : radius[l - kFarStrict]);
        f.radius2[l] = (float)(d * d);
    }
    // how many levels stricter than 0 the largest charge is (far_level)
    double q_max = 0.0;
    for (int a = 0; a < n_atoms; a++) q_max = std::max(q_max, std::fabs(charge[a]));
    int large = 0;
    if (ref > 0.0 && q_max > 0.0)
        large = (int)std::min(std::max(std::floor(2.0 * std::log2(q_max * std::fabs(coeff) * 128.0 / ref) + 1e-5) - 2.0, 0.0),
                              (double)kFarStrict);
    if (!std::isfinite(q2) || !std::isfinite(f.qscale)) large = kFarStrict;
    // the largest bin of a direct pair: its atom lies within the radius of the patch's box
    int passes = kFarStrict + 1;   // least level past 0 with which one may pass the table's end
    for (int q = kFarStrict; q >= 0; q--)
        if (std::sqrt(f.radius2[kFarStrict - q]) + diag + 4.0 >= kFarLastBin) passes = q;
    double rmax = 0.0;
    if (passes <= kFarStrict)
        for (int a = 0; a < n_atoms; a++) {
            double q = 0.0;
            for (int d = 0; d < 3; d++) {
                const double x = coord[3 * (size_t)a + d];
                const double e = std::max(std::fabs(x + g.ne[d] * g.spacing),
                                          std::fabs(x - (g.n1[d] - 1 - g.ne[d]) * g.spacing));
                q += e * e;
            }
            rmax = std::max(rmax, q);
        }
    if (std::sqrt(rmax) * 128.0 + 20.0 * s + 4.0 >= kFarLastBin) f.clamp_from = std::max(0, passes - large);
    f.clamp = f.clamp_from == 0;
    // a grid of few patches shares each among workgroups until there are
    // about four workgroups per CU, at least 256 atoms each (one group of 64
    // per wave)
    const long long items = (long long)best * ((g.n1[0] + kFarK - 1) / kFarK);
    f.split = (int)std::max<long long>(1, std::min<long long>({1024 / items, n_atoms / 256, kFarSplitMax}));
    return f;
}

// Coarse boxes where they pay.  A patch spends 80 node terms on an atom beyond
// it, a box 512 for its 16 patches, at 4e12 terms/s; two more launches and the
// transfer to the patches' nodes cost about 20 us.  Atoms at protein density
// (0.068 / A^3) within the distance of a box are no box's: a receptor has to
// hold half as many again before a part of it worth the launches is beyond.
// (5,000 atoms on 127^3 points, where that is 5,470: 794 us with boxes for 807; a
// batch of twelve conformations of 1,500 to 6,000 atoms 5.19 ms for 4.96.)
static void far_boxes(FarShape &f, const ag_grid &g, int n_atoms, const std::vector<float> &reps, const FarError &err) {
    f.box_py = std::max(1, (kBoxRows + f.py / 2) / f.py);
    f.box_pz = std::max(1, (kBoxRows + f.pz / 2) / f.pz);
    const int edge = std::max({kBoxRuns * kFarK, f.box_py * f.py, f.box_pz * f.pz});
    const double a = edge * g.spacing;
    const auto dilated = [&](double r) { return a * a * a + r * (6 * a * a + M_PI * r * (3 * a + 4. / 3. * r)); };
    if (n_atoms < 1.5 * 0.068 * dilated(18.5)) return;   // (no distance is less)
    // as far_radii has it for the table, and where its nodes leave half of what a
    // level allows; the stricter levels no nearer than a patch's.  (What counts is the
    // atom ahead of a face: the two axes along it see the pole of 1/r beside them,
    // at 1.8 half-edges 2.6e-5 of the term where a patch's run leaves 5e-6.)
    constexpr int kLevels = kFarStrict + kFarLevels;
    const double patch_half[2] = {kFarMid * g.spacing, 0.5 * (std::max(f.py, f.pz) - 1) * g.spacing};
    const double half = 0.5 * (edge - 1) * g.spacing;
    const double r0 = std::sqrt((double)f.radius2[kFarStrict]) / 128.0;   // a patch's level 0
    double table[kFarLevels], radius[kLevels];
    far_radii(reps, g.spacing, kBoxN, 0.5 * (edge - 1), table);
    far_distances([&](double r) { return 2.0 * far_axis_error(err.reps, r, half, kBoxAxis); }, 8.25,
                  std::max(30.0, 8.0 * half), std::max(3.0, half / 2.0), far_error(err, r0, patch_half), kFarStrict,
                  kLevels, radius);
    for (int l = 0; l < kLevels; l++)
        radius[l] = std::max(radius[l], l < kFarStrict ? std::sqrt((double)f.radius2[l]) / 128.0 : table[l - kFarStrict]);
    const double beyond = n_atoms - 0.068 * dilated(radius[kFarStrict]);
    const double patches = (double)((g.n1[0] + kFarK - 1) / kFarK) * ((g.n1[1] + f.py - 1) / f.py) *
                           ((g.n1[2] + f.pz - 1) / f.pz);
    const double boxes = std::ceil(g.n1[0] / (double)(kBoxRuns * kFarK)) * std::ceil(g.n1[1] / (double)(f.box_py * f.py)) *
                         std::ceil(g.n1[2] / (double)(f.box_pz * f.pz));
    if (beyond < n_atoms / 3.0 || beyond * (kFarNodes * patches - kBoxNodes * boxes) < 8e7) return;
    // about eight workgroups per CU, at least 256 atoms each
    f.box_parts = (int)std::max(1.0, std::min({2048 / boxes, n_atoms / 256.0, 16.0}));
    for (int l = 0; l < kLevels; l++) f.box_radius2[l] = (float)(radius[l] * 128.0 * (radius[l] * 128.0));
}

// The far kernel with, if cp is given, the cell list in one more workgroup.
static void launch_far(int blocks, const FarParams &fp, int kind, const CellParams *cp, hipStream_t st) {
#define AG_FAR(K)                                                                              \
    case K:                                                                                    \
        if (cp) k_far<K, true><<<blocks + 1, kFarThreads, 0, st>>>(fp, *cp);                   \
        else k_far<K, false><<<blocks, kFarThreads, 0, st>>>(fp, CellParams{});                \
        break
    switch (kind) {
        AG_FAR(kFarTable);
        AG_FAR(kFarClamped);
        AG_FAR(kFarFlat);
    }
#undef AG_FAR
    HIP_CHECK(hipGetLastError());
}
// The kind of a launch of conformations [c0, c1).
static int far_kind(const ag_plan &p, int c0, int c1) {
    if (p.far_flat) return kFarFlat;
    for (int ci = c0; ci < c1; ci++)
        if (p.confs[ci].far_clamp) return kFarClamped;
    return kFarTable;
}

// Waves of the near kernel that share a cube's atoms, from the number of 8x8x4
// bricks of the grid.  The kernel is bound by its vector operations, so what
// counts is that every SIMD has waves until the end: 256 CUs hold 1,280
// workgroups at once.  Sharing by s cuts the list into s parts and makes s
// times as many workgroups, whose staging and final sums are the cost.
// Measured (us) at s = 1, 2, 4: 396 bricks (41^3 points) 147, 80, 62;
// 1,024 (61^3) 201, 180, 170; 1,980 (47 x 83 x 119) 239, 215, 226; 2,541 (81^3)
// 263, 231, 233 and twelve of these in a batch 5,137, 5,212, 5,397 in all; 8,448
// (127^3) 810, 807, 935; 70,785 (257^3) 3,398, 3,817, 4,768.
static int near_share(long long bricks) {
    return bricks <= 1024 ? 4 : bricks <= 4096 ? 2 : 1;
}

// How far (bins) a pair's distance in the near kernel may lie from the far
// kernel's bin limit and the two still disagree on which of them has it.  The
// far kernel's distances from the patch's centre are good to 2^-25 of them on
// each side, three times at most per axis, its squared distance sums four products of up to
// (limit + kFarMid s128)^2 with an error of 2^-24 each, the near kernel's
// distance is good to 3e-4 bins; doubled.  At 0.375 A spacing 0.003: the shell
// in which the near kernel repeats the far kernel's arithmetic held some lane
// of 3 waves in 10 when it was 5 bins wide for every grid.
static float far_band(const ag_grid &g) {
    const double s128 = g.spacing * 128.0, reach = kFarBinMin + kFarMid * s128;
    const double coord = 9 * 0x1p-25 * reach;
    const double square = 4 * 0x1p-24 * 2 * reach * reach / (2.0 * kFarBinMin);
    return (float)(2 * (coord + square + 3e-4));
}

static long long far_box_count(const ConfDev &cf) { return (long long)cf.box_n[0] * cf.box_n[1] * cf.box_n[2]; }
static long long far_patch_count(const ConfDev &cf) { return (long long)cf.runs_per_row * cf.far_npy * cf.far_npz; }

// Memory that a plan can do without: null where there is none left.
static void *room_for(DevBuf &b, size_t bytes) {
    if (b.pool && b.pool->arena && !b.pool->fits(bytes)) return nullptr;
    try {
        return b.get(bytes);
    } catch (const ag::Error &e) {
        if (e.status != AG_ERR_OOM) throw;
        return nullptr;
    }
}

// Where a far field beside the near one goes: 8 bytes a point (268 MB at most),
// one block for all plans of a context, which run one after the other.  A plan that
// finds no room runs one field after the other.
static double *wide_field(ag_plan *p) {
    if (!p->beside) return nullptr;
    void *const block = room_for(p->ctx->far_wide, sizeof(double) * (size_t)p->confs[0].P);
    p->beside = block != nullptr;
    return (double *)block;
}

// Per-conformation geometry, work prefixes and cell arrays for the plan's
// cell size.
static void plan_geometry(ag_plan &p, const ag_grid *grids, const int *natoms, const FarShape *far) {
    const int n = p.nconf;
    const double cs = p.tune.cell_size;
    p.confs.assign(n, ConfDev{});
    p.brick_prefix.assign(n + 1, 0);
    p.tile_prefix.assign(n + 1, 0);
    long long brick = 0, tile = 0, moff = 0, poff = 0, part = 0, box_sums = 0, box_mask = 0, box_patch = 0, reach = 0;
    int cell_base = 0, atom_base = 0;
    for (int c = 0; c < n; c++) {
        ConfDev &cf = p.confs[c];
        memset(&cf, 0, sizeof cf);
        const ag_grid &g = grids[c];
        for (int d = 0; d < 3; d++) {
            cf.n1[d] = g.n1[d];
            cf.ne[d] = g.ne[d];
            const double lo = -g.ne[d] * g.spacing - 8.1;
            const double hi = (g.n1[d] - 1 - g.ne[d]) * g.spacing + 8.1;
            cf.cell_origin[d] = lo;
            cf.nc[d] = (int)ceil((hi - lo) / cs) + 1;
        }
        cf.spacing = g.spacing;
        cf.s128 = (float)(g.spacing * 128.0);
        cf.near_band = far_band(g);
        const int brick_edge[3] = {kBX, kBY, kBZ};
        long long bricks = 1;
        for (int d = 0; d < 3; d++) bricks *= (g.n1[d] + brick_edge[d] - 1) / brick_edge[d];
        cf.near_share = near_share(bricks);
        for (int d = 0; d < 3; d++) {
            const int e = brick_edge[d] / (cf.near_share > (d == 0 ? 2 : 1) && d < 2 ? 2 : 1);
            cf.nb[d] = (g.n1[d] + e - 1) / e;
        }
        cf.cell_base = cell_base;
        cf.atom_base = atom_base;
        cf.n_atoms = natoms[c];
        cf.P = (long long)g.n1[0] * g.n1[1] * g.n1[2];
        cf.map_off = moff;
        cf.pt_off = poff;
        cf.runs_per_row = (g.n1[0] + kFarK - 1) / kFarK;
        const FarShape fs = far ? far[c] : FarShape();
        cf.far_py = fs.py;
        cf.far_pz = fs.pz;
        cf.far_npy = (g.n1[1] + fs.py - 1) / fs.py;
        cf.far_npz = (g.n1[2] + fs.pz - 1) / fs.pz;
        cf.far_split = fs.split;
        cf.far_clamp = fs.clamp;
        for (int l = 0; l < kFarStrict + kFarLevels; l++) cf.far_r2[l] = fs.radius2[l];
        cf.far_qscale = fs.qscale;
        cf.part_off = part;
        cf.box_parts = fs.box_parts;
        cf.box_py = fs.box_py;
        cf.box_pz = fs.box_pz;
        cf.box_n[0] = (cf.runs_per_row + kBoxRuns - 1) / kBoxRuns;
        cf.box_n[1] = (cf.far_npy + fs.box_py - 1) / fs.box_py;
        cf.box_n[2] = (cf.far_npz + fs.box_pz - 1) / fs.box_pz;
        for (int l = 0; l < kFarStrict + kFarLevels; l++) cf.box_r2[l] = fs.box_radius2[l];
        cf.reach_off = reach;
        reach += far_patch_count(cf);
        if (cf.box_parts) {
            const long long boxes = far_box_count(cf);
            cf.box_off = box_sums;
            cf.box_mask_off = box_mask;
            cf.box_patch_off = box_patch;
            box_sums += boxes * cf.box_parts * kBoxNodes;
            box_mask += boxes * ((natoms[c] + 63) / 64);
            box_patch += far_patch_count(cf) * kFarNodes;
        }
        if (fs.split > 1) part += fs.split * cf.P;
        p.brick_prefix[c] = (int)brick;
        p.tile_prefix[c] = (int)tile;
        brick += (long long)cf.nb[0] * cf.nb[1] * cf.nb[2];
        tile += (long long)cf.far_npy * cf.far_npz * cf.runs_per_row * cf.far_split;
        const long long cells = (long long)cf.nc[0] * cf.nc[1] * cf.nc[2];
        if (cell_base + cells > INT32_MAX / 2 || brick > INT32_MAX / 2 || tile > INT32_MAX / 2)
            ag::fail(AG_ERR_UNSUPPORTED, "batch too large for one plan");
        cell_base += (int)cells;
        atom_base += natoms[c];
        moff += (long long)p.n_maps * cf.P;
        poff += cf.P;
    }
    p.brick_prefix[n] = (int)brick;
    p.tile_prefix[n] = (int)tile;
    p.total_bricks = (int)brick;
    p.total_tiles = (int)tile;
    p.total_cells = cell_base;
    p.P_total = poff;
    if (p.want_collide) {
        p.near[0].collide = (unsigned char *)p.collide.get((size_t)p.P_total);
    }
    p.cell_count.get(sizeof(int) * (size_t)p.total_cells);
    p.cell_start.get(sizeof(int) * ((size_t)p.total_cells + 1));
    p.confs_d.get(sizeof(ConfDev) * p.confs.size());
    p.brick_prefix_d.get(sizeof(int) * p.brick_prefix.size());
    p.tile_prefix_d.get(sizeof(int) * p.tile_prefix.size());
    const size_t reach_tables = sizeof(float) * kReachTab * (size_t)n;
    unsigned char *const d_reach = far ? (unsigned char *)p.far_reach.get(reach_tables + (size_t)reach) : nullptr;
    // the partial e maps come last: where a fixed arena has no room left for
    // them, no patch is shared
    if (part && p.pool->arena && !p.pool->fits(sizeof(float) * (size_t)part)) {
        part = tile = 0;
        for (int c = 0; c < n; c++) {
            ConfDev &cf = p.confs[c];
            cf.far_split = 1;
            p.tile_prefix[c] = (int)tile;
            tile += (long long)cf.far_npy * cf.far_npz * cf.runs_per_row;
        }
        p.tile_prefix[n] = p.total_tiles = (int)tile;
    }
    p.far.part = part ? (float *)p.far_part.get(sizeof(float) * (size_t)part) : nullptr;
    p.beside = far && p.far_flat && !p.persistent && n == 1 && !p.pool->arena && !p.want_collide &&
               p.confs[0].far_split == 1 && p.confs[0].P <= (1ll << 25);
    // the coarse boxes' sums, patch values and atom sets, in one block; no boxes
    // where there is no room for it
    p.has_boxes = box_sums > 0;
    if (p.has_boxes) {
        p.far.box_sums = (double *)room_for(p.far_box, 8 * (size_t)(box_sums + box_patch + box_mask));
        if (p.far.box_sums) {
            p.far.box_patch = p.far.box_sums + box_sums;
            p.far.box_mask = (unsigned long long *)(p.far.box_patch + box_patch);
        } else {
            p.has_boxes = false;
            for (ConfDev &cf : p.confs) cf.box_parts = 0;
        }
    }
    hipStream_t st = p.ctx->stream;
    upload(st, p.confs_d, p.confs.data(), p.confs.size());
    upload(st, p.brick_prefix_d, p.brick_prefix.data(), p.brick_prefix.size());
    upload(st, p.tile_prefix_d, p.tile_prefix.data(), p.tile_prefix.size());
    const ConfDev *d_confs = (const ConfDev *)p.confs_d.ptr;
    for (auto &q : p.near) {
        q.confs = d_confs;
        q.brick_prefix = (const int *)p.brick_prefix_d.ptr;
        q.nconf = n;
        q.total_bricks = p.total_bricks;
        q.cell_size = cs;
        q.cell_start = (const int *)p.cell_start.ptr;
    }
    p.far.confs = d_confs;
    p.far.tile_prefix = (const int *)p.tile_prefix_d.ptr;
    p.far.nconf = n;
    p.far.total_tiles = p.total_tiles;
    int occ = 0;
    HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, reinterpret_cast<const void *>(&k_far<kFarClamped, false>),
                                                           kFarThreads, 0));
    p.far_grid = std::max(1, std::min(p.total_tiles, std::max(occ, 1) * p.ctx->n_cu));
    if (far) {
        p.reach_tables.clear();
        for (int c = 0; c < n; c++) p.reach_tables.insert(p.reach_tables.end(), far[c].reach, far[c].reach + kReachTab);
        HIP_CHECK(hipMemcpyAsync(d_reach, p.reach_tables.data(), reach_tables, hipMemcpyHostToDevice, st));
        p.far.shift = d_reach + reach_tables;
        for (int c = 0; c < n; c++)
            k_far_reach<<<(unsigned)((far_patch_count(p.confs[c]) + kReachPatches - 1) / kReachPatches), kReachThreads, 0, st>>>(
                p.far, c, (const float *)d_reach, d_reach + reach_tables);
        HIP_CHECK(hipGetLastError());
    }
}

// Build a plan over n conformations (a single plan is n = 1).
// An arena pool (the allocation-free entry point) also keeps the host
// staging in pageable memory instead of the context's pinned buffer.
static ag_plan *plan_build(ag_ctx *c, int n, const ag_receptor *recs, const ag_grid *grids, const ag_mapset *ms,
                           const ag_tables *tab, int potential, bool persistent, const Tune &tune,
                           std::shared_ptr<DevPool> pool = nullptr) {
    const bool vina = potential == AG_POTENTIAL_VINA;
    if (potential != AG_POTENTIAL_AD4 && !vina) ag::fail(AG_ERR_BAD_INPUT, "unknown potential");
    if (n < 1) ag::fail(AG_ERR_BAD_INPUT, "a plan needs at least one conformation");
    for (int i = 0; i < n; i++) validate(&recs[i], &grids[i], ms, tab, vina);
    HIP_CHECK(hipSetDevice(c->device));
    if (!pool) pool = c->pool;
    const bool no_alloc = pool->arena != nullptr;
    std::unique_ptr<ag_plan> pl(new ag_plan(pool));
    ag_plan &p = *pl;
    p.ctx = c;
    p.nconf = n;
    p.vina = vina;
    p.persistent = persistent;
    p.tune = tune;
    const int M = p.M = ms->n_atom_maps;
    const int T = p.T = tab->n_rec_types;
    p.n_maps = ms->n_maps;
    p.coeff_estat = ms->coeff_estat;
    hipStream_t st = c->stream;

    // concatenated atoms
    std::vector<int> natoms(n);
    long long Nl = 0;
    for (int i = 0; i < n; i++) Nl += (natoms[i] = recs[i].n_atoms);
    if (Nl > INT32_MAX / 4) ag::fail(AG_ERR_UNSUPPORTED, "too many atoms in one batch");
    const int N = p.N = (int)Nl;
    // concatenated receptor arrays, staged in the context's pinned buffer
    size_t off = 0;
    auto carve = [&](size_t bytes) {
        const size_t o = off;
        off += (bytes + 255) & ~size_t(255);
        return o;
    };
    const size_t n3 = 3 * (size_t)N, nn = (size_t)N;
    const size_t o_coord = carve(8 * n3), o_charge = carve(8 * nn), o_vol = carve(8 * nn), o_solpar = carve(8 * nn);
    const size_t o_rvec = carve(8 * n3), o_rvec2 = carve(8 * n3), o_type = carve(4 * nn), o_hbond = carve(4 * nn);
    const size_t o_rexp = carve(4 * nn), o_conf = carve(4 * nn), o_dis = carve(nn);
    std::vector<char> pageable(no_alloc ? off + 256 : 0);
    char *const h = no_alloc ? pageable.data() : (char *)c->stage.get(off + 256);
    double *const coord = (double *)(h + o_coord), *const charge = (double *)(h + o_charge);
    double *const vol = (double *)(h + o_vol), *const solpar = (double *)(h + o_solpar);
    double *const rvec = (double *)(h + o_rvec), *const rvec2 = (double *)(h + o_rvec2);
    int *const type = (int *)(h + o_type), *const hbond = (int *)(h + o_hbond), *const rexp = (int *)(h + o_rexp);
    int *const atom_conf = (int *)(h + o_conf);
    unsigned char *const dis = (unsigned char *)(h + o_dis);
    std::vector<int> first_atom(n + 1, 0);
    for (int i = 0; i < n; i++) first_atom[i + 1] = first_atom[i] + natoms[i];
    auto stage_conf = [&](int i) {
        const int o = first_atom[i];
        const ag_receptor &r = recs[i];
        const size_t k = natoms[i];
        if (!k) return;
        std::copy(r.coord, r.coord + 3 * k, coord + 3 * (size_t)o);
        std::copy(r.charge, r.charge + k, charge + o);
        std::copy(r.vol, r.vol + k, vol + o);
        std::copy(r.solpar, r.solpar + k, solpar + o);
        std::copy(r.rvector, r.rvector + 3 * k, rvec + 3 * (size_t)o);
        std::copy(r.rvector2, r.rvector2 + 3 * k, rvec2 + 3 * (size_t)o);
        std::copy(r.type, r.type + k, type + o);
        std::copy(r.hbond, r.hbond + k, hbond + o);
        std::copy(r.rexp, r.rexp + k, rexp + o);
        std::copy(r.disorder, r.disorder + k, dis + o);
        std::fill(atom_conf + o, atom_conf + o + k, i);
    };
    // large batches copy on several host threads (at most 16), one
    // conformation at a time
    const int n_thr = N > 200000 ? std::max(1, std::min({16, n, (int)std::thread::hardware_concurrency()})) : 1;
    if (n_thr > 1) {
        std::atomic<int> next{0};
        std::vector<std::thread> th;
        for (int t = 0; t < n_thr; t++)
            th.emplace_back([&] {
                for (int i; (i = next.fetch_add(1)) < n;) stage_conf(i);
            });
        for (auto &x : th) x.join();
    } else {
        for (int i = 0; i < n; i++) stage_conf(i);
    }
    double *d_coord = upload(st, p.coord, coord, n3);
    double *d_charge = upload(st, p.charge, charge, nn);
    double *d_vol = upload(st, p.vol, vol, nn);
    double *d_solpar = upload(st, p.solpar, solpar, nn);
    double *d_rvec = upload(st, p.rvec, rvec, n3);
    double *d_rvec2 = upload(st, p.rvec2, rvec2, n3);
    int *d_type = upload(st, p.type, type, nn);
    int *d_hbond = upload(st, p.hbond, hbond, nn);
    int *d_rexp = upload(st, p.rexp, rexp, nn);
    unsigned char *d_dis = upload(st, p.disorder, dis, nn);
    p.any_disorder = std::any_of(dis, dis + N, [](unsigned char v) { return v != 0; });
    if (n > 1) upload(st, p.atom_conf_d, atom_conf, nn);
    p.src = AtomSrc{d_coord, d_charge, d_vol, d_solpar, d_rvec, d_rvec2, d_type, d_hbond, d_rexp, d_dis,
                    ms->coeff_estat, ms->solpar_q};
    p.atom_cell.get(sizeof(int) * (size_t)N);
    p.slot_atom.get(sizeof(int) * (size_t)N);
    // the near kernel's candidate lists hold 32-bit byte offsets of records
    if ((unsigned long long)N * sizeof(NearAtom) > UINT32_MAX)
        ag::fail(AG_ERR_UNSUPPORTED, "too many atoms in one plan for the near kernel (at most 53,687,091)");
    p.near_atoms.get(sizeof(NearAtom) * (size_t)N);
    // an arena pool allocates no pinned memory: its plans keep the flag on the device
    if (!p.pool->arena) {
        p.status_page = c->status_page;
        p.report = p.status_page->take();
    }
    if (!p.report) p.status.get(sizeof(int));

    // electrostatic factor per bin: 332/eps for the distance-dependent
    // dielectric, 332/diel for a constant one (main.cpp:2960-2978)
    std::vector<float> reps(AG_NDIEL);
    for (int k = 0; k < AG_NDIEL; k++) reps[k] = ms->dddiel ? (float)tab->r_eps[k] : (float)ms->inv_diel_cal;
    float *d_reps = upload(st, p.reps, reps.data(), AG_NDIEL);
    std::vector<float> sol(AG_NEINT + 1);
    for (int k = 0; k <= AG_NEINT; k++) sol[k] = (float)tab->sol_fn[k];
    float *d_sol = upload(st, p.sol, sol.data(), AG_NEINT + 1);

    // Map slots of the near-kernel passes.  Maps without H-bond terms (and
    // the desolvation halves of separate_desolvation_maps) take plain slots,
    // H-bonding probes take the H-bond slots; covalent maps take none.  With
    // the Vina potential every map is a plain table sum: no directional
    // H-bond terms, no desolvation, no e or d map.
    std::vector<int> plain_maps, hb_maps;
    for (int m = 0; m < M; m++) {
        const int role = map_role(ms, m);
        if (role == ROLE_COV) p.cov_slots.push_back(m);
        else if (!vina && (role & ROLE_AFF) && ms->maps[m].is_hbonder) hb_maps.push_back(m);
        else plain_maps.push_back(m);
    }
    // A pass has kPlainSlots plain slots and kHbSlots H-bond slots; plain
    // maps beyond the plain slots take free H-bond slots, whose code is then
    // the plain table add for every atom class (13 Vina maps: one pass).
    const int n_plain = (int)plain_maps.size(), n_hb = (int)hb_maps.size();
    p.groups = std::max({1, (n_hb + kHbSlots - 1) / kHbSlots, (n_plain + n_hb + kMapSlots - 1) / kMapSlots});
    std::vector<std::array<int, kMapSlots>> slot_map(p.groups);
    std::vector<std::array<bool, kHbSlots>> hb_plain(p.groups);
    int nplain_max = 0;
    for (int g = 0; g < p.groups; g++) {
        slot_map[g].fill(-1);
        hb_plain[g].fill(false);
        int np_g = 0;
        for (int j = 0; j < kPlainSlots; j++) {
            const size_t i = (size_t)g * kPlainSlots + j;
            if (i < plain_maps.size()) { slot_map[g][j] = plain_maps[i]; np_g = j + 1; }
        }
        nplain_max = std::max(nplain_max, np_g);
        for (int k = 0; k < kHbSlots; k++) {
            const size_t i = (size_t)g * kHbSlots + k;
            if (i < hb_maps.size()) slot_map[g][kPlainSlots + k] = hb_maps[i];
        }
    }
    for (size_t i = (size_t)p.groups * kPlainSlots; i < plain_maps.size(); i++) {
        bool placed = false;
        for (int g = 0; g < p.groups && !placed; g++)
            for (int k = 0; k < kHbSlots && !placed; k++)
                if (slot_map[g][kPlainSlots + k] < 0) {
                    slot_map[g][kPlainSlots + k] = plain_maps[i];
                    hb_plain[g][k] = true;
                    placed = true;
                }
        if (!placed) ag::fail(AG_ERR_UNSUPPORTED, "near-kernel slot assignment left a map without a slot");
    }
    p.nplain = nplain_max <= 4 ? 4 : (nplain_max <= 8 ? 8 : 12);
    // rows of near_row slots: the bins, zeros past the cutoff, and the last bin's
    // again for 8 A exactly
    const int row = near_row(p.nplain);
    const size_t gstride = (size_t)(T > 0 ? T : 1) * kNearRows * row;
    std::vector<float> gtab(gstride * p.groups, 0.f);
    for (int g = 0; g < p.groups; g++) {
        for (int t = 0; t < T; t++)
            for (int j = 0; j < kMapSlots; j++) {
                const int m = slot_map[g][j];
                // a slot without an affinity term (desolvation only) keeps
                // zeros, so the kernel adds every slot's table value
                if (m < 0 || !(map_role(ms, m) & ROLE_AFF)) continue;
                const float *srcrow = tab->e_vdw_hb + ((size_t)t * M + m) * AG_NEINT;
                const int at = j < kPlainSlots ? j : row - 4 + (j - kPlainSlots);
                float *dst = gtab.data() + g * gstride + (size_t)t * kNearRows * row + at;
                for (int k = 0; k < AG_NEINT; k++) dst[(size_t)k * row] = srcrow[k];
                dst[(size_t)kNearExactRow * row] = srcrow[AG_NEINT - 1];
            }
    }
    float *d_tab = upload(st, p.tab, gtab.data(), gtab.size());
    p.queue_d.get(sizeof(int) * kMaxChunks);

    NearParams np;
    memset(&np, 0, sizeof np);
    np.atoms = (const NearAtom *)p.near_atoms.ptr;
    np.coord64 = d_coord;
    np.rvec64 = d_rvec;
    np.sol = d_sol;
    np.reps = d_reps;
    np.disorder_h = ms->disorder_h;
    np.hydrogen_type = ms->hydrogen_type;
    np.solpar_q = (float)ms->solpar_q;
    np.status = p.overflow_flag();
    for (int g = 0; g < p.groups; g++) {
        NearParams q = np;
        bool used = false;
        for (int j = 0; j < kMapSlots; j++) {
            const int m = slot_map[g][j];
            q.out_slot[j] = m;
            q.sp[j] = 0.f;
            q.volp[j] = 0.f;
            if (m < 0) continue;
            used = true;
            const int role = map_role(ms, m);
            const ag_map_desc &md = ms->maps[m];
            if ((role & ROLE_DES) && !vina) {
                q.sp[j] = (float)md.solpar_probe;
                q.volp[j] = (float)md.vol_probe;
            }
            if (j >= kPlainSlots) {
                const int k = j - kPlainSlots;
                for (int ah = 0; ah <= 6; ah++) {
                    if (hb_plain[g][k]) {   // a plain map in an H-bond slot
                        q.hcode[k][ah] = HC_PLAIN | (HC_PLAIN << 4);
                        continue;
                    }
                    const int cse = hb_case(md.hbond, ah);
                    int ordered = 0, disordered = 0;
                    if (cse == HBC_PLAIN) ordered = disordered = HC_PLAIN;
                    else if (cse == HBC_ACC_PROBE) ordered = disordered = HC_HRAMP | HC_RACC;
                    else if (cse == HBC_MINMAX_RACC) ordered = disordered = HC_MINMAX | HC_RACC;
                    else {  // HBC_DON_PROBE
                        ordered = HC_MINMAX;
                        disordered = HC_HRAMP;
                    }
                    q.hcode[k][ah] = ordered | (disordered << 4);
                }
            }
        }
        q.tab = d_tab + g * gstride;
        q.e_slot = (g == 0 && !vina) ? ms->elec_index : -1;
        q.d_slot = (g == 0 && !vina) ? ms->dsolv_index : -1;
        q.has_affinity = used || q.d_slot >= 0;
        p.near.push_back(q);
    }

    // floating and constriction grids
    p.want_fmap = ms->floating_grid != 0;
    p.want_cmap = ms->constriction_grid != 0;
    if (p.want_cmap) p.near[0].ccut = ms->constriction_cutoff;
    // the tree build's semantics (every pass: Loop 2; pass 0: cmap, collisions)
    for (auto &q : p.near) q.bhtree = ms->bhtree;
    p.want_collide = ms->bhtree == 1 && (ms->elec_index >= 0 || ms->floating_grid);
    p.e_index = vina ? -1 : ms->elec_index;
    if (p.want_fmap && N > 0) {
        float4 *d_fa = (float4 *)p.fmin_atoms.get(sizeof(float4) * (size_t)N);
        k_fmin_atoms<<<(N + 255) / 256, 256, 0, st>>>(N, d_coord, d_fa);
        HIP_CHECK(hipGetLastError());
    }
    if (p.cov_slots.size() > 16) ag::fail(AG_ERR_UNSUPPORTED, "more than 16 covalent maps");
    for (int d = 0; d < 3; d++) p.cov_pos[d] = ms->cov_pos[d];
    p.cov_half_width = ms->cov_half_width;
    p.cov_barrier = ms->cov_barrier;
    // Vina: the e and d maps stay zero (main.cpp:2968, 3391)
    if (vina) {
        if (ms->elec_index >= 0) p.zero_slots.push_back(ms->elec_index);
        if (ms->dsolv_index >= 0) p.zero_slots.push_back(ms->dsolv_index);
    }

    // far kernel (e map)
    p.run_far = !vina && ms->elec_index >= 0 && N > 0;
    p.far_flat = flat_table(reps) && std::isfinite(reps.back());   // (its pairs are weighted before they are left out)
    std::vector<FarShape> far_shapes;
    if (p.run_far) {
        FarAtom *d_far = (FarAtom *)p.far_atoms.get(sizeof(FarAtom) * (size_t)N);
        k_far_atoms<<<(N + 255) / 256, 256, 0, st>>>(N, d_coord, d_charge, ms->coeff_estat, d_far);
        HIP_CHECK(hipGetLastError());
        const FarError err(reps);
        double radius[kFarLevels] = {}, spacing = -1.0;
        for (int i = 0, o = 0; i < n; o += natoms[i], i++) {
            if (grids[i].spacing != spacing) far_radii(reps, spacing = grids[i].spacing, kFarNx, kFarMid, radius);
            far_shapes.push_back(
                far_shape(grids[i], natoms[i], radius, err, coord + 3 * (size_t)o, charge + o, ms->coeff_estat));
            far_boxes(far_shapes.back(), grids[i], natoms[i], reps, err);
        }
        FarParams &fp = p.far;
        memset(&fp, 0, sizeof fp);
        fp.atoms = d_far;
        fp.tab = d_reps;
        fp.e_slot = ms->elec_index;
    }
    plan_geometry(p, grids, natoms.data(), p.run_far ? far_shapes.data() : nullptr);
    // A batch's far field is captured as two graphs: conformations [0,
    // far_split), then the rest, so that the first part's e maps can go to
    // the host while the second part computes.  The second part is sized so
    // that its far field (at about 5.5e12 pairs/s) lasts about as long as
    // that copy (at about 45 GB/s): what is left after the map set is the
    // second part's e maps.
    p.far_split = n;
    if (persistent && n > 1 && p.run_far) {
        double work = 0.0, ebytes = 0.0;
        for (const ConfDev &cf : p.confs) {
            work += (double)cf.P * cf.n_atoms;
            ebytes += 4.0 * (double)cf.P;
        }
        const double t_far = work / 5.5e12, t_copy = ebytes / 45e9;
        const double want_b = work * t_copy / (t_far + t_copy);
        double acc = 0.0;
        int split = n;
        while (split > 1 && acc < want_b) {
            --split;
            acc += (double)p.confs[split].P * p.confs[split].n_atoms;
        }
        p.far_split = split;
    }
    // whether some patch's direct pairs may pass the table's end (spacings past
    // 0.48 A, patches far from the atoms)
    bool ask = false;
    for (int i = 0; i < n && p.run_far && !p.far_flat; i++)
        ask = ask || (far_shapes[i].clamp_from > 0 && far_shapes[i].clamp_from <= kFarStrict);
    std::vector<unsigned char> shift;
    if (ask) {
        shift.resize((size_t)(p.confs[n - 1].reach_off + far_patch_count(p.confs[n - 1])));
        HIP_CHECK(hipMemcpyAsync(shift.data(), p.far.shift, shift.size(), hipMemcpyDeviceToHost, st));
    }
    HIP_CHECK(hipStreamSynchronize(st));   // host staging vectors go out of scope
    for (int i = 0; i < n && ask; i++) {
        const auto first = shift.begin() + p.confs[i].reach_off;
        const int most = *std::max_element(first, first + far_patch_count(p.confs[i]));
        p.confs[i].far_clamp = most >= far_shapes[i].clamp_from;
    }
    return pl.release();
}


// Host destinations of a batch: conformation i's maps / fmap / cmap.
struct HostOut {
    float *const *maps;
    float *const *fmap;
    int32_t *const *cmap;
};

// Contiguous conformation ranges of about equal work (points x atoms).
// Chunks of consecutive conformations for a batch with host outputs: `want`
// chunks whose work (points x atoms) follows the weights 1, ..., 1, 1/2,
// 1/4, ..., 1/2^taper.  The last chunks shrink so that the copy left after
// the final kernel is short; fewer, larger chunks before them keep the
// number of chunk boundaries low.
static std::vector<std::pair<int, int>> plan_chunks(const ag_plan &p, int want, int taper) {
    std::vector<std::pair<int, int>> out;
    const int n = p.nconf;
    want = std::max(1, std::min({want, n, kMaxChunks}));
    taper = std::max(0, std::min(taper, want - 1));
    std::vector<double> bound(want);   // cumulative work fraction at the end of each chunk
    {
        double sum = 0.0;
        for (int k = 0; k < want; k++) sum += k < want - taper ? 1.0 : std::ldexp(1.0, -(k - (want - taper) + 1));
        double acc = 0.0;
        for (int k = 0; k < want; k++) {
            acc += k < want - taper ? 1.0 : std::ldexp(1.0, -(k - (want - taper) + 1));
            bound[k] = acc / sum;
        }
    }
    double total = 0.0;
    for (const ConfDev &cf : p.confs) total += (double)cf.P * (cf.n_atoms + 64);
    int c0 = 0;
    double acc = 0.0;
    for (int c = 0; c < n; c++) {
        acc += (double)p.confs[c].P * (p.confs[c].n_atoms + 64);
        const int k = (int)out.size();
        if (c == n - 1 || (k < want - 1 && acc >= total * bound[k])) {
            out.emplace_back(c0, c + 1);
            c0 = c + 1;
        }
    }
    return out;
}

enum : int { kPartAll = 0, kPartNear = 1, kPartFar = 2 };
// Stamps of MapReport: the starts of the first kernel (the cell list, or with it
// the far field), the gather behind a far field that went first, the near field, the
// far field; the end of a cell list beside the far field, and of a near and a far
// field beside each other.
enum : int { kStampFirst = 0, kStampGather = 1, kStampNear = 2, kStampFar = 3, kStampCellsEnd = 4, kStampNearEnd = 5,
             kStampFarEnd = 6 };

// One conformation whose far field is in parts, with a cell list that one
// workgroup makes in the far kernel's LDS before the others are done.
static bool far_goes_first(const ag_plan &p) {
    return !p.persistent && p.nconf == 1 && p.run_far && p.confs[0].far_split > 1 && !p.has_boxes && p.N <= kCellsOneAtoms &&
           p.total_cells <= kFarLds - kFarWaves;
}

// Enqueue one map set on the context's stream, conformation chunk by chunk.
// With events, HIP events bracket the cell list, the near-field and the
// far-field phases (single chunk).  With host outputs, each chunk's maps
// are copied to the host on the context's copy stream as soon as the chunk
// is done, while the next chunk computes.  `part` (single chunk) enqueues
// only the cell list and near field (kPartNear) or only the far field
// (kPartFar); with kPartAll, mark_near records the context's near_ev once the
// near field of every conformation is enqueued.
static void enqueue(ag_plan *p, float *d_maps, float *d_fmap, int32_t *d_cmap, bool events, bool skip_far,
                    const std::vector<std::pair<int, int>> &chunks, const HostOut *host, bool mark_near = false,
                    int part = kPartAll, int queue_base = 0) {
    ag_ctx *c = p->ctx;
    hipStream_t st = c->stream;
    const int N = p->N;
    const int tpb = 256;
    int *d_atom_cell = (int *)p->atom_cell.ptr, *d_count = (int *)p->cell_count.ptr;
    int *d_start = (int *)p->cell_start.ptr;
    int *d_slot_atom = (int *)p->slot_atom.ptr;
    int *d_status = p->overflow_flag();
    int *d_queue = (int *)p->queue_d.ptr;
    const int nchunks = (int)chunks.size();
    if (nchunks < 1 || nchunks > kMaxChunks) ag::fail(AG_ERR_BAD_INPUT, "bad chunking of the batch");
    if (part != kPartAll && (nchunks != 1 || host)) ag::fail(AG_ERR_BAD_INPUT, "bad chunking of the batch");
    const unsigned cgrid = (unsigned)((p->total_cells + tpb - 1) / tpb);
    if (events) HIP_CHECK(hipEventRecord(c->ev[0], st));
    // A small plan's far field, in parts, goes first with the cell list in one
    // of its workgroups, and the near kernel adds the parts: 3 launches instead
    // of 5.  (With one part the far kernel adds to the near field's e map, and
    // a copy to the host overlaps the far field behind it.)
    const bool far_first = far_goes_first(*p) && part == kPartAll && !skip_far && !host && !mark_near && nchunks == 1;
    // In a constant dielectric the far field is vector operations alone, and the
    // near field waits for its table rows: they run beside each other (3,000
    // atoms on 81^3 points with floating and constriction grids 808 -> 700 us; with a
    // table, 5,000 atoms on 127^3 points 1,600 -> 1,563).  Not where copies to the host
    // start behind the near field: it would end later (800 -> 937 us).
    double *const wide = part == kPartAll && !skip_far && !host && !mark_near && nchunks == 1 ? wide_field(p) : nullptr;
    const bool beside = wide != nullptr;
    const bool stamps = events && p->report && !p->persistent && !skip_far;
    const auto stamp = [&](int phase) { return stamps ? p->stamp(phase) : nullptr; };
    if (part != kPartFar) {
        const int *atom_conf = p->nconf > 1 ? (const int *)p->atom_conf_d.ptr : nullptr;
        const ConfDev *d_confs = (const ConfDev *)p->confs_d.ptr;
        const CellParams cp{d_confs, atom_conf, N, p->total_cells, p->tune.cell_size, (const double *)p->coord.ptr,
                            d_start, d_atom_cell, d_slot_atom, d_status, d_queue, kMaxChunks, stamp(kStampFirst),
                            far_first ? stamp(kStampCellsEnd) : nullptr};
        if (far_first) {
            FarParams fp = p->far;
            fp.maps = d_maps;
            fp.item_end = p->total_tiles;
            launch_far(p->total_tiles, fp, far_kind(*p, 0, 1), &cp, st);
        } else if (N <= kCellsOneAtoms && p->total_cells <= kCellsOne) {
            k_cells<<<1, 1024, 0, st>>>(cp);
        } else {
            k_zero_cells<<<std::max(cgrid, (unsigned)((kMaxChunks + tpb - 1) / tpb)), tpb, 0, st>>>(
                d_count, p->total_cells, d_status, d_queue, kMaxChunks, stamp(kStampFirst));
            if (N > 0)
                k_cell_count<<<(N + tpb - 1) / tpb, tpb, 0, st>>>(d_confs, atom_conf, N, p->tune.cell_size,
                                                                  (const double *)p->coord.ptr, d_atom_cell, d_count);
            k_scan<<<1, 1024, 0, st>>>(d_count, d_start, p->total_cells);
            if (N > 0)
                k_cell_scatter<<<(N + tpb - 1) / tpb, tpb, 0, st>>>(N, d_atom_cell, d_start, d_count, d_slot_atom);
        }
        if (N > 0)
            k_gather<<<(N + tpb - 1) / tpb, tpb, 0, st>>>(p->total_cells, d_atom_cell, d_start, d_slot_atom, p->src,
                                                          (NearAtom *)p->near_atoms.ptr,
                                                          far_first ? stamp(kStampGather) : nullptr);
        HIP_CHECK(hipGetLastError());
    }
    if (events && !stamps) HIP_CHECK(hipEventRecord(c->ev[1], st));
    // The near field (near kernel, floating grid, covalent and zero maps) of
    // conformations [c0, c1) on stream s.
    auto near_pass = [&](int c0, int c1, hipStream_t s) {
        const int b0 = p->brick_prefix[c0], b1 = p->brick_prefix[c1];
        for (int g = 0; g < p->groups; g++) {
            NearParams np = p->near[g];
            np.maps = d_maps;
            np.cmap = (g == 0 && p->want_cmap) ? d_cmap : nullptr;
            np.item_base = b0;
            np.far_part = far_first ? p->far.part : nullptr;
            np.stamp = g == 0 ? stamp(kStampNear) : nullptr;
            if (!(np.has_affinity || np.e_slot >= 0 || np.cmap) || b1 <= b0) continue;
            launch_near(*p, b1 - b0, np, s);
        }
        for (int ci = c0; ci < c1; ci++) {
            const ConfDev &cf = p->confs[ci];
            const unsigned pgrid = (unsigned)((cf.P + 255) / 256);
            if (p->want_fmap) {
                FminParams fm;
                memset(&fm, 0, sizeof fm);
                for (int d = 0; d < 3; d++) {
                    fm.n1[d] = cf.n1[d];
                    fm.ne[d] = cf.ne[d];
                }
                fm.spacing = (float)cf.spacing;
                for (int d = 0; d < 3; d++) fm.nb[d] = (cf.n1[d] + kFminEdge - 1) / kFminEdge;
                fm.atoms = (const float4 *)p->fmin_atoms.ptr + cf.atom_base;
                fm.n_atoms = cf.n_atoms;
                fm.fmap = d_fmap + cf.pt_off;
                k_fmin<<<(unsigned)(fm.nb[0] * fm.nb[1] * fm.nb[2]), 256, 0, s>>>(fm);
            }
            if (!p->cov_slots.empty()) {
                CovParams cv;
                memset(&cv, 0, sizeof cv);
                for (int d = 0; d < 3; d++) {
                    cv.n1[d] = cf.n1[d];
                    cv.ne[d] = cf.ne[d];
                    cv.pos[d] = p->cov_pos[d];
                }
                cv.spacing = cf.spacing;
                cv.half_width = p->cov_half_width;
                cv.barrier = p->cov_barrier;
                cv.n_cov = (int)p->cov_slots.size();
                for (int q = 0; q < cv.n_cov; q++) cv.slot[q] = p->cov_slots[q];
                cv.P = cf.P;
                cv.maps = d_maps + cf.map_off;
                k_covalent<<<pgrid, 256, 0, s>>>(cv);
            }
            for (int m : p->zero_slots)
                k_fill<<<pgrid, 256, 0, s>>>(d_maps + cf.map_off + (size_t)m * cf.P, cf.P, 0.f);
        }
        HIP_CHECK(hipGetLastError());
    };
    // The far field of chunk k ([c0, c1), work counter k) and the tree
    // build's collision rule after it, on stream s.
    auto far_pass = [&](int k, int c0, int c1, hipStream_t s) {
        const int t0 = p->tile_prefix[c0], t1 = p->tile_prefix[c1];
        if (p->run_far && !skip_far && !far_first && t1 > t0) {
            FarParams fp = p->far;
            fp.maps = d_maps;
            fp.stamp = stamp(kStampFar);
            fp.wide = wide;
            fp.item_base = t0;
            fp.item_end = t1;
            fp.queue = p->persistent ? d_queue + queue_base + k : nullptr;
            const int blocks = p->persistent ? std::min(p->far_grid, t1 - t0) : t1 - t0;
            if (p->has_boxes)
                for (int ci = c0; ci < c1; ci++) {
                    const ConfDev &cf = p->confs[ci];
                    if (!cf.box_parts) continue;
                    const unsigned items = (unsigned)(far_box_count(cf) * cf.box_parts);
                    if (p->far_flat) k_far_boxes<true><<<items, kFarThreads, 0, s>>>(fp, ci);
                    else k_far_boxes<false><<<items, kFarThreads, 0, s>>>(fp, ci);
                    fp.stamp = nullptr;   // (the far field has begun)
                    k_far_down<<<(unsigned)far_patch_count(cf), 64, 0, s>>>(fp, ci);
                }
            launch_far(blocks, fp, far_kind(*p, c0, c1), nullptr, s);
            long long most = 0;   // points of the largest conformation with parts to add
            for (int ci = c0; ci < c1; ci++)
                if (p->confs[ci].far_split > 1) most = std::max(most, p->confs[ci].P);
            if (most)
                k_far_sum<<<dim3((unsigned)((most + 255) / 256), (unsigned)(c1 - c0)), 256, 0, s>>>(fp, c0);
        }
        if (p->want_collide)
            for (int ci = c0; ci < c1; ci++) {
                const ConfDev &cf = p->confs[ci];
                k_collide<<<(unsigned)((cf.P + 255) / 256), 256, 0, s>>>(
                    cf.P, (const unsigned char *)p->collide.ptr + cf.pt_off,
                    p->e_index >= 0 ? d_maps + cf.map_off + (size_t)p->e_index * cf.P : nullptr,
                    d_fmap ? d_fmap + cf.pt_off : nullptr);
            }
        HIP_CHECK(hipGetLastError());
    };
    // Chunk k's outputs to the host on the copy stream, once s has them.
    auto copy_out = [&](int k, int c0, int c1, hipStream_t s) {
        HIP_CHECK(hipEventRecord(c->chunk_ev[k], s));
        HIP_CHECK(hipStreamWaitEvent(c->copy_stream, c->chunk_ev[k], 0));
        for (int ci = c0; ci < c1; ci++) {
            const ConfDev &cf = p->confs[ci];
            HIP_CHECK(hipMemcpyAsync(host->maps[ci], d_maps + cf.map_off, sizeof(float) * (size_t)p->n_maps * cf.P,
                                     hipMemcpyDeviceToHost, c->copy_stream));
            if (d_fmap)
                HIP_CHECK(hipMemcpyAsync(host->fmap[ci], d_fmap + cf.pt_off, sizeof(float) * (size_t)cf.P,
                                         hipMemcpyDeviceToHost, c->copy_stream));
            if (d_cmap)
                HIP_CHECK(hipMemcpyAsync(host->cmap[ci], d_cmap + cf.pt_off, sizeof(int32_t) * (size_t)cf.P,
                                         hipMemcpyDeviceToHost, c->copy_stream));
        }
    };
    const hipStream_t st_main = st;
    if (host && nchunks > 1) {
        // Pipelined batch: the whole batch's near field first, on the main
        // stream, then the chunks' far fields alternating between the two
        // compute streams (chunks touch disjoint conformations), each chunk's
        // copies behind its far kernel.  Copies start after the first chunk's
        // far field and overlap the rest; two far launches in flight fill
        // each other's tails.  (Near and far passes interleaved chunk by
        // chunk measured 8 ms slower on the 64-conformation ensemble: a near
        // pass beside the other stream's persistent far kernel waits for CU
        // slots.)
        near_pass(0, p->nconf, st_main);
        HIP_CHECK(hipEventRecord(c->cells_ev, st_main));
        HIP_CHECK(hipStreamWaitEvent(c->stream2, c->cells_ev, 0));
        for (int k = 0; k < nchunks; k++) {
            const hipStream_t s = (k & 1) ? c->stream2 : st_main;
            far_pass(k, chunks[k].first, chunks[k].second, s);
            copy_out(k, chunks[k].first, chunks[k].second, s);
        }
    } else {
        for (int k = 0; k < nchunks; k++) {
            if (beside) {
                HIP_CHECK(hipEventRecord(c->cells_ev, st_main));
                HIP_CHECK(hipStreamWaitEvent(c->stream2, c->cells_ev, 0));
                far_pass(k, chunks[k].first, chunks[k].second, c->stream2);
                if (stamps) k_stamp<<<1, 1, 0, c->stream2>>>(stamp(kStampFarEnd));
                HIP_CHECK(hipEventRecord(c->far2_ev, c->stream2));
            }
            if (part != kPartFar) near_pass(chunks[k].first, chunks[k].second, st_main);
            if (events && !stamps && k == nchunks - 1) HIP_CHECK(hipEventRecord(c->ev[2], st_main));
            if (mark_near && k == nchunks - 1) HIP_CHECK(hipEventRecord(c->near_ev, st_main));
            if (beside) {
                if (stamps) k_stamp<<<1, 1, 0, st_main>>>(stamp(kStampNearEnd));
                HIP_CHECK(hipStreamWaitEvent(st_main, c->far2_ev, 0));
                const ConfDev &cf = p->confs[0];
                k_far_add<<<(unsigned)std::min<long long>((cf.P + 255) / 256, 4096), 256, 0, st_main>>>(
                    wide, d_maps + cf.map_off + (long long)p->far.e_slot * cf.P, cf.P);
                continue;
            }
            if (part != kPartNear) far_pass(k, chunks[k].first, chunks[k].second, st_main);
            if (host) copy_out(k, chunks[k].first, chunks[k].second, st_main);
        }
    }
    st = st_main;
    if (host) {
        // the copy stream has waited for every chunk, so this joins both
        // compute streams as well
        HIP_CHECK(hipEventRecord(c->chunk_ev[kMaxChunks], c->copy_stream));
        HIP_CHECK(hipStreamWaitEvent(st, c->chunk_ev[kMaxChunks], 0));
    }
    if (events) HIP_CHECK(hipEventRecord(c->ev[3], st));
}

static void enqueue(ag_plan *p, float *d_maps, float *d_fmap, int32_t *d_cmap, bool events, bool skip_far,
                    bool mark_near = false, int part = kPartAll) {
    enqueue(p, d_maps, d_fmap, d_cmap, events, skip_far, {{0, p->nconf}}, nullptr, mark_near, part);
}

// Whether a brick of the last map set overflowed the near kernel's LDS lists
// (syncs the context's stream).
static bool overflowed(ag_plan *p) {
    if (p->report) {   // written by the kernels themselves
        HIP_CHECK(hipStreamSynchronize(p->ctx->stream));
        return __atomic_load_n(&p->report->overflow, __ATOMIC_ACQUIRE) != 0;
    }
    int status = 0;
    HIP_CHECK(hipMemcpyAsync(&status, p->status.ptr, sizeof(int), hipMemcpyDeviceToHost, p->ctx->stream));
    HIP_CHECK(hipStreamSynchronize(p->ctx->stream));
    return status != 0;
}

// Runs one map set of p through `run` and checks the overflow word: when a
// brick had more than 2048 candidate atoms or 256 donor H within 8.03 A, the
// plan switches to the paged near kernel for good (its graph, if any, is
// captured again) and runs the map set once more.
template <class F>
static void run_checked(ag_plan *p, F &&run) {
    run();
    if (!overflowed(p)) return;
    if (p->paged) ag::fail(AG_ERR_DEVICE, "the paged near kernel reported an overflow");
    p->paged = true;
    p->drop_graphs();
    run();
    if (overflowed(p)) ag::fail(AG_ERR_DEVICE, "the paged near kernel reported an overflow");
}

// Autotuner: times the near-field pass of every candidate layout on a
// sample of the batch (up to 8 conformations spread over its sizes) and
// keeps the fastest.  Results differ between cell sizes only in the order
// of the FP32 sums; for a fixed choice every run is bitwise repeatable.
static Tune autotune(ag_ctx *c, int n, const ag_receptor *recs, const ag_grid *grids, const ag_mapset *ms,
                     const ag_tables *tab, int potential, double *spent_ms) {
    const auto t0 = std::chrono::steady_clock::now();
    std::vector<int> order(n);
    for (int i = 0; i < n; i++) order[i] = i;
    std::sort(order.begin(), order.end(), [&](int a, int b) {
        const long long pa = (long long)grids[a].n1[0] * grids[a].n1[1] * grids[a].n1[2] * std::max(recs[a].n_atoms, 1);
        const long long pb = (long long)grids[b].n1[0] * grids[b].n1[1] * grids[b].n1[2] * std::max(recs[b].n_atoms, 1);
        return pa != pb ? pa < pb : a < b;
    });
    const int ns = std::min(n, 8);
    std::vector<ag_receptor> srec(ns);
    std::vector<ag_grid> sgrid(ns);
    for (int k = 0; k < ns; k++) {
        const int i = order[ns == 1 ? n - 1 : (int)((long long)k * (n - 1) / (ns - 1))];
        srec[k] = recs[i];
        sgrid[k] = grids[i];
    }
    long long sp = 0;
    for (int k = 0; k < ns; k++) sp += (long long)sgrid[k].n1[0] * sgrid[k].n1[1] * sgrid[k].n1[2];
    DevBuf out;
    float *d_maps = (float *)out.get(sizeof(float) * (size_t)sp * ms->n_maps + 256);
    DevBuf extra;
    char *x = (char *)extra.get(2 * sizeof(float) * (size_t)sp + 256);
    float *d_fmap = ms->floating_grid ? (float *)x : nullptr;
    int32_t *d_cmap = ms->constriction_grid ? (int32_t *)(x + sizeof(float) * (size_t)sp) : nullptr;
    const double cells[3] = {3.0, 4.0, 5.0};
    Tune best;
    float best_ms = 1e30f;
    for (int cube = 0; cube < 2; cube++)
        for (double cs : cells) {
            Tune t;
            t.cell_size = cs;
            t.cube = cube != 0;
            std::unique_ptr<ag_plan> p(plan_build(c, ns, srec.data(), sgrid.data(), ms, tab, potential, true, t));
            float ms_near = 0.f;
            for (int rep = 0; rep < 2; rep++) {
                run_checked(p.get(), [&] { enqueue(p.get(), d_maps, d_fmap, d_cmap, true, true); });
                HIP_CHECK(hipEventElapsedTime(&ms_near, c->ev[1], c->ev[2]));
            }
            if (ms_near < best_ms) {
                best_ms = ms_near;
                best = t;
            }
        }
    *spent_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return best;
}

ag_plan *plan_create(ag_ctx *c, const ag_receptor *rec, const ag_grid *grid, const ag_mapset *ms,
                     const ag_tables *tab, int potential) {
    std::unique_ptr<ag_plan, void (*)(ag_plan *)> p(plan_build(c, 1, rec, grid, ms, tab, potential, false, Tune()), plan_destroy);
    (void)wide_field(p.get());   // here rather than in the first map set
    return p.release();
}

ag_plan *batch_create(ag_ctx *c, int n, const ag_receptor *recs, const ag_grid *grids, const ag_mapset *ms,
                      const ag_tables *tab, int potential, const ag_tune *tune) {
    Tune t;
    double spent = 0.0;
    if (tune) {
        if (!(tune->cell_size >= 2.0 && tune->cell_size <= 8.0))
            ag::fail(AG_ERR_BAD_INPUT, "cell size must lie in [2, 8] A");
        t.cell_size = tune->cell_size;
        t.cube = tune->cube != 0;
    } else {
        for (int i = 0; i < n; i++) validate(&recs[i], &grids[i], ms, tab, potential == AG_POTENTIAL_VINA);
        t = autotune(c, n, recs, grids, ms, tab, potential, &spent);
    }
    ag_plan *p = plan_build(c, n, recs, grids, ms, tab, potential, true, t);
    p->tune_ms = spent;
    return p;
}

void plan_tune(const ag_plan *p, ag_tune *out) {
    out->cell_size = p->tune.cell_size;
    out->cube = p->tune.cube ? 1 : 0;
    out->reserved = 0;
    out->tune_ms = p->tune_ms;
}

void plan_layout(const ag_plan *p, long long *map_off, long long *pt_off, long long *map_floats, long long *points) {
    for (int i = 0; i < p->nconf; i++) {
        if (map_off) map_off[i] = p->confs[i].map_off;
        if (pt_off) pt_off[i] = p->confs[i].pt_off;
    }
    if (map_floats) *map_floats = p->P_total * p->n_maps;
    if (points) *points = p->P_total;
}

int plan_count(const ag_plan *p) { return p->nconf; }

void plan_destroy(ag_plan *p) {
    if (!p) return;
    (void)hipSetDevice(p->ctx->device);
    (void)hipStreamSynchronize(p->ctx->stream);
    (void)hipStreamSynchronize(p->ctx->stream2);
    (void)hipStreamSynchronize(p->ctx->copy_stream);
    delete p;
}

// One map set (all conformations of the plan) into d_maps
// ([sum n_maps * P] float, device) and, when asked for, d_fmap / d_cmap
// ([sum P]), enqueued on the context's stream.  A single plan runs its
// kernels directly with phase timing; a batch replays captured hipGraphs
// (re-captured when the outputs move): the cell list and near field, then
// the persistent far field in two parts (conformations split at
// far_split).  Either way the context's near_ev is recorded once the near
// field is done; a batch records far_ev after its first far-field part.
// The second part goes on stream2 behind near_ev, submitted after the
// first: the first part's persistent grid fills the GPU, and the second
// part's workgroups take the CUs as the first part's drain, instead of
// starting after its last one.  The parts write different conformations
// and take separate work counters; the main stream joins the second part
// before ev[3].
static hipGraphExec_t capture(ag_plan *p, float *d_maps, float *d_fmap, int32_t *d_cmap, int part, int c0, int c1,
                              int queue_base) {
    hipStream_t st = p->ctx->stream;
    hipGraph_t g = nullptr;
    HIP_CHECK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    try {
        enqueue(p, d_maps, d_fmap, d_cmap, false, false, {{c0, c1}}, nullptr, false, part, queue_base);
    } catch (...) {
        hipGraph_t dead = nullptr;
        (void)hipStreamEndCapture(st, &dead);
        if (dead) (void)hipGraphDestroy(dead);
        throw;
    }
    HIP_CHECK(hipStreamEndCapture(st, &g));
    hipGraphExec_t exec = nullptr;
    hipError_t e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess)
        ag::fail(AG_ERR_DEVICE, std::string("HIP error: ") + hipGetErrorString(e) + " at hipGraphInstantiate");
    return exec;
}

static void launch_mapset(ag_plan *p, float *d_maps, float *d_fmap, int32_t *d_cmap, bool mark_near) {
    ag_ctx *c = p->ctx;
    hipStream_t st = c->stream;
    if (!p->persistent) {
        if (p->report) *p->report = MapReport{};   // (the plan's last map set was waited for)
        enqueue(p, d_maps, d_fmap, d_cmap, true, false, mark_near);
        return;
    }
    if (!p->graph || p->g_maps != d_maps || p->g_fmap != d_fmap || p->g_cmap != d_cmap) {
        p->drop_graphs();
        p->graph = capture(p, d_maps, d_fmap, d_cmap, kPartNear, 0, p->nconf, 0);
        p->graph_far = capture(p, d_maps, d_fmap, d_cmap, kPartFar, 0, p->far_split, 0);
        if (p->far_split < p->nconf)
            p->graph_far2 = capture(p, d_maps, d_fmap, d_cmap, kPartFar, p->far_split, p->nconf, 1);
        p->g_maps = d_maps;
        p->g_fmap = d_fmap;
        p->g_cmap = d_cmap;
    }
    HIP_CHECK(hipEventRecord(c->ev[0], st));
    HIP_CHECK(hipGraphLaunch(p->graph, st));
    HIP_CHECK(hipEventRecord(c->near_ev, st));
    HIP_CHECK(hipGraphLaunch(p->graph_far, st));
    HIP_CHECK(hipEventRecord(c->far_ev, st));
    if (p->graph_far2) {
        HIP_CHECK(hipStreamWaitEvent(c->stream2, c->near_ev, 0));
        HIP_CHECK(hipGraphLaunch(p->graph_far2, c->stream2));
        HIP_CHECK(hipEventRecord(c->far2_ev, c->stream2));
        HIP_CHECK(hipStreamWaitEvent(st, c->far2_ev, 0));
    }
    HIP_CHECK(hipEventRecord(c->ev[3], st));
}

static void read_timing(ag_plan *p) {
    ag_ctx *c = p->ctx;
    float total = 0.f;
    HIP_CHECK(hipEventElapsedTime(&total, c->ev[0], c->ev[3]));
    if (p->persistent) {
        c->last_ms[0] = c->last_ms[1] = c->last_ms[2] = -1.f;
    } else if (p->report) {
        // the phases' starts by the device's clock; the last one ends with the total
        const unsigned long long *const t = p->report->start;
        const auto span = [&](int from, int to) {
            return t[from] && t[to] > t[from] ? (float)((double)(t[to] - t[from]) / c->clock_khz) : 0.f;
        };
        if (t[kStampGather]) {   // the far field went first, the cell list beside it
            const float gather = span(kStampGather, kStampNear);
            c->last_ms[2] = span(kStampFirst, kStampGather);
            c->last_ms[0] = span(kStampFirst, kStampCellsEnd) + gather;
            c->last_ms[1] = std::max(0.f, total - gather - c->last_ms[2]);
        } else if (t[kStampFarEnd]) {   // the fields ran beside each other
            c->last_ms[0] = t[kStampFar] < t[kStampNear] ? span(kStampFirst, kStampFar) : span(kStampFirst, kStampNear);
            c->last_ms[1] = span(kStampNear, kStampNearEnd);
            c->last_ms[2] = span(kStampFar, kStampFarEnd);
        } else {
            c->last_ms[0] = span(kStampFirst, kStampNear);
            c->last_ms[1] = t[kStampFar] ? span(kStampNear, kStampFar) : std::max(0.f, total - c->last_ms[0]);
            c->last_ms[2] = std::max(0.f, total - c->last_ms[0] - c->last_ms[1]);
        }
    } else {
        HIP_CHECK(hipEventElapsedTime(&c->last_ms[0], c->ev[0], c->ev[1]));
        HIP_CHECK(hipEventElapsedTime(&c->last_ms[1], c->ev[1], c->ev[2]));
        HIP_CHECK(hipEventElapsedTime(&c->last_ms[2], c->ev[2], c->ev[3]));
    }
    c->last_ms[3] = total;
}

void plan_execute(ag_plan *p, float *d_maps, float *d_fmap, int32_t *d_cmap) {
    if ((p->want_fmap && !d_fmap) || (p->want_cmap && !d_cmap))
        ag::fail(AG_ERR_BAD_INPUT, "the map set asks for a floating/constriction grid but no output was given");
    HIP_CHECK(hipSetDevice(p->ctx->device));
    run_checked(p, [&] { launch_mapset(p, d_maps, d_fmap, d_cmap, false); });
    read_timing(p);
}

// plan_execute, then every conformation's outputs into host memory
// (maps_out[i]: [n_maps][P_i] floats; fmap_out[i] / cmap_out[i]: [P_i]).
// Only the e map is written after the near field (by the far kernel and the
// tree build's collision rule, which also sets fmap), so the copy stream
// takes the other maps, cmap and -- without the collision rule -- fmap as
// soon as near_ev is reached, while the far kernel runs; the e maps (and
// fmap) of a batch's first far-field graph follow far_ev, during its second
// far-field graph, and the rest the end of the map set.  Host memory pinned
// with hipHostMalloc lets the copies overlap the kernels.
void plan_execute_host(ag_plan *p, float *d_maps, float *d_fmap, int32_t *d_cmap, float *const *maps_out,
                       float *const *fmap_out, int32_t *const *cmap_out) {
    if ((p->want_fmap && !d_fmap) || (p->want_cmap && !d_cmap))
        ag::fail(AG_ERR_BAD_INPUT, "the map set asks for a floating/constriction grid but no output was given");
    if (!maps_out) ag::fail(AG_ERR_BAD_INPUT, "no map outputs");
    for (int i = 0; i < p->nconf; i++)
        if (!maps_out[i] || (p->want_fmap && (!fmap_out || !fmap_out[i])) ||
            (p->want_cmap && (!cmap_out || !cmap_out[i])))
            ag::fail(AG_ERR_BAD_INPUT, "missing output for a conformation");
    ag_ctx *c = p->ctx;
    HIP_CHECK(hipSetDevice(c->device));
    hipStream_t st = c->stream, cs = c->copy_stream;
    const int e = p->e_index;
    const bool fmap_late = p->want_collide;
    auto copy = [&](void *dst, const void *src, size_t bytes) {
        if (bytes) HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, cs));
    };
    run_checked(p, [&] {
        launch_mapset(p, d_maps, d_fmap, d_cmap, true);
        HIP_CHECK(hipStreamWaitEvent(cs, c->near_ev, 0));
        for (int i = 0; i < p->nconf; i++) {
            const ConfDev &cf = p->confs[i];
            const size_t pb = sizeof(float) * (size_t)cf.P;
            const float *src = d_maps + cf.map_off;
            if (e < 0) {
                copy(maps_out[i], src, pb * p->n_maps);
            } else {
                copy(maps_out[i], src, pb * e);
                copy(maps_out[i] + (size_t)(e + 1) * cf.P, src + (size_t)(e + 1) * cf.P, pb * (p->n_maps - e - 1));
            }
            if (d_cmap) copy(cmap_out[i], d_cmap + cf.pt_off, sizeof(int32_t) * (size_t)cf.P);
            if (d_fmap && !fmap_late) copy(fmap_out[i], d_fmap + cf.pt_off, pb);
        }
        // the e maps (and late fmaps) of a batch's first far-field graph,
        // then of the rest
        const auto late = [&](int c0, int c1) {
            for (int i = c0; i < c1; i++) {
                const ConfDev &cf = p->confs[i];
                const size_t pb = sizeof(float) * (size_t)cf.P;
                if (e >= 0) copy(maps_out[i] + (size_t)e * cf.P, d_maps + cf.map_off + (size_t)e * cf.P, pb);
                if (d_fmap && fmap_late) copy(fmap_out[i], d_fmap + cf.pt_off, pb);
            }
        };
        const int split = p->persistent ? p->far_split : p->nconf;
        if (split < p->nconf) {
            HIP_CHECK(hipStreamWaitEvent(cs, c->far_ev, 0));
            late(0, split);
        }
        HIP_CHECK(hipEventRecord(c->chunk_ev[0], st));
        HIP_CHECK(hipStreamWaitEvent(cs, c->chunk_ev[0], 0));
        late(split < p->nconf ? split : 0, p->nconf);
        HIP_CHECK(hipEventRecord(c->chunk_ev[kMaxChunks], cs));
        HIP_CHECK(hipStreamWaitEvent(st, c->chunk_ev[kMaxChunks], 0));
    });
    read_timing(p);
}

// ag_maps_plain with device outputs, every device buffer drawn from this
// device's scratch array: a plan on an arena pool over it, built, run and
// dropped.  Nothing is allocated on the device or pinned on the host.
void maps_plain_noalloc(ag_ctx *c, const ag_receptor *rec, const ag_grid *grid, const ag_mapset *ms,
                        const ag_tables *tab, float *maps, float *fmap, int32_t *cmap) {
    HIP_CHECK(hipSetDevice(c->device));
    if (!c->scratch) ag::fail(AG_ERR_DEVICE, "no scratch address for this device");
    auto arena = std::make_shared<DevPool>(c->scratch, (size_t)AG_NOALLOC_SCRATCH_BYTES);
    std::unique_ptr<ag_plan, void (*)(ag_plan *)> p(
        plan_build(c, 1, rec, grid, ms, tab, AG_POTENTIAL_AD4, false, Tune(), arena), plan_destroy);
    plan_execute(p.get(), maps, ms->floating_grid ? fmap : nullptr, ms->constriction_grid ? cmap : nullptr);
}

// One map set, handed to the host map by map: each map is copied into host
// memory as soon as the kernels are done and on_ready(j) is called for it
// (j = n_maps for fmap, n_maps + 1 for cmap), so the caller can format and
// write map j while later maps are still in flight.
void maps_plain_streamed(ag_ctx *c, const ag_receptor *rec, const ag_grid *grid, const ag_mapset *ms,
                         const ag_tables *tab, float *maps_out, float *fmap, int32_t *cmap,
                         const std::function<void(int)> &on_ready, int potential) {
    std::unique_ptr<ag_plan, void (*)(ag_plan *)> p(plan_create(c, rec, grid, ms, tab, potential), plan_destroy);
    const long long P = p->P_total;
    const size_t pbytes = sizeof(float) * (size_t)P;
    const size_t bytes = pbytes * (size_t)p->n_maps;
    float *d_maps = (float *)c->maps.get(bytes + 2 * pbytes + 256);
    char *extra = (char *)d_maps + bytes;
    float *d_fmap = ms->floating_grid ? (float *)extra : nullptr;
    int32_t *d_cmap = ms->constriction_grid ? (int32_t *)(extra + pbytes) : nullptr;
    plan_execute(p.get(), d_maps, d_fmap, d_cmap);
    for (int j = 0; j < p->n_maps; j++) {
        HIP_CHECK(hipMemcpyAsync(maps_out + (size_t)j * P, d_maps + (size_t)j * P, pbytes,
                                 hipMemcpyDeviceToHost, c->stream));
        HIP_CHECK(hipStreamSynchronize(c->stream));
        on_ready(j);
    }
    if (d_fmap) {
        HIP_CHECK(hipMemcpyAsync(fmap, d_fmap, pbytes, hipMemcpyDeviceToHost, c->stream));
        HIP_CHECK(hipStreamSynchronize(c->stream));
        on_ready(p->n_maps);
    }
    if (d_cmap) {
        HIP_CHECK(hipMemcpyAsync(cmap, d_cmap, pbytes, hipMemcpyDeviceToHost, c->stream));
        HIP_CHECK(hipStreamSynchronize(c->stream));
        on_ready(p->n_maps + 1);
    }
}

void plan_audit(ag_plan *p, long long out[4]) {
    ag_ctx *c = p->ctx;
    HIP_CHECK(hipSetDevice(c->device));
    hipStream_t st = c->stream;
    if (p->nconf != 1) ag::fail(AG_ERR_UNSUPPORTED, "the bin audit runs on single-conformation plans");
    DevBuf acc;
    unsigned long long *d_out = (unsigned long long *)acc.get(4 * sizeof(unsigned long long));
    HIP_CHECK(hipMemsetAsync(d_out, 0, 4 * sizeof(unsigned long long), st));
    const ConfDev &cf = p->confs[0];
    AuditParams ap;
    memset(&ap, 0, sizeof ap);
    for (int d = 0; d < 3; d++) {
        ap.n1[d] = cf.n1[d];
        ap.far.ne[d] = cf.ne[d];
    }
    ap.far.py = cf.far_py;
    ap.far.pz = cf.far_pz;
    ap.far.spacing = cf.spacing;
    ap.far.s128 = cf.s128;
    ap.coord = (const double *)p->coord.ptr;
    ap.n_atoms = p->N;
    ap.P = cf.P;
    ap.out = d_out;
    k_audit<<<(unsigned)((cf.P + 255) / 256), 256, 0, st>>>(ap);
    HIP_CHECK(hipGetLastError());
    unsigned long long h[4];
    HIP_CHECK(hipMemcpyAsync(h, d_out, sizeof h, hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipStreamSynchronize(st));
    for (int i = 0; i < 4; i++) out[i] = (long long)h[i];
}

void maps_plain(ag_ctx *c, const ag_receptor *rec, const ag_grid *grid, const ag_mapset *ms, const ag_tables *tab,
                float *maps_out, float *fmap, int32_t *cmap, int outputs_on_device, int potential) {
    if ((ms->floating_grid && !fmap) || (ms->constriction_grid && !cmap))
        ag::fail(AG_ERR_BAD_INPUT, "the map set asks for a floating/constriction grid but no output was given");
    std::unique_ptr<ag_plan, void (*)(ag_plan *)> p(
        outputs_on_device ? plan_create(c, rec, grid, ms, tab, potential)
                          : plan_build(c, 1, rec, grid, ms, tab, potential, false, Tune()),
        plan_destroy);
    const long long P = p->P_total;
    const size_t bytes = sizeof(float) * (size_t)p->n_maps * P;
    const size_t pbytes = sizeof(float) * (size_t)P;
    float *d_maps = outputs_on_device ? maps_out : (float *)c->maps.get(bytes + 2 * pbytes + 256);
    float *d_fmap = nullptr;
    int32_t *d_cmap = nullptr;
    if (outputs_on_device) {
        d_fmap = ms->floating_grid ? fmap : nullptr;
        d_cmap = ms->constriction_grid ? cmap : nullptr;
    } else {
        char *base = (char *)d_maps + bytes;
        if (ms->floating_grid) d_fmap = (float *)base;
        if (ms->constriction_grid) d_cmap = (int32_t *)(base + pbytes);
    }
    if (outputs_on_device) {
        plan_execute(p.get(), d_maps, d_fmap, d_cmap);
        return;
    }
    // host outputs: the maps other than e go to the host while the far
    // kernel runs, the e map after it
    float *const mo[1] = {maps_out};
    float *const fo[1] = {fmap};
    int32_t *const co[1] = {cmap};
    plan_execute_host(p.get(), d_maps, d_fmap, d_cmap, mo, d_fmap ? fo : nullptr, d_cmap ? co : nullptr);
}

static bool is_pinned(const void *ptr) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, ptr) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type == hipMemoryTypeHost;
}

// Batch with host outputs: maps_out[i] receives conformation i's
// [n_maps][P_i] floats (fmap_out / cmap_out its [P_i] values when asked).
// When every destination is pinned host memory the conformations run in
// chunks of about equal work, launched directly and alternating between
// the two compute streams, and each chunk's maps are copied to the host on
// the copy stream behind an event while later chunks compute.  (A captured graph would run its
// copy nodes in line with its kernels, serialising the two; a one-shot
// batch has few launches to save, so it is not captured.)  Otherwise the
// plan's graph computes everything and the copies follow it.
void maps_batch(ag_ctx *c, int n, const ag_receptor *recs, const ag_grid *grids, const ag_mapset *ms,
                const ag_tables *tab, float *const *maps_out, float *const *fmap_out, int32_t *const *cmap_out,
                int potential, const ag_tune *tune) {
    if (!maps_out) ag::fail(AG_ERR_BAD_INPUT, "no map outputs");
    for (int i = 0; i < n; i++)
        if (!maps_out[i] || (ms->floating_grid && (!fmap_out || !fmap_out[i])) ||
            (ms->constriction_grid && (!cmap_out || !cmap_out[i])))
            ag::fail(AG_ERR_BAD_INPUT, "missing output for a conformation");
    std::unique_ptr<ag_plan, void (*)(ag_plan *)> p(batch_create(c, n, recs, grids, ms, tab, potential, tune),
                                                   plan_destroy);
    const long long P = p->P_total;
    const size_t bytes = sizeof(float) * (size_t)p->n_maps * P;
    const size_t pbytes = sizeof(float) * (size_t)P;
    float *d_maps = (float *)c->maps.get(bytes + 2 * pbytes + 256);
    char *base = (char *)d_maps + bytes;
    float *d_fmap = ms->floating_grid ? (float *)base : nullptr;
    int32_t *d_cmap = ms->constriction_grid ? (int32_t *)(base + pbytes) : nullptr;
    bool pinned = true;
    for (int i = 0; i < n && pinned; i++)
        pinned = is_pinned(maps_out[i]) && (!d_fmap || is_pinned(fmap_out[i])) && (!d_cmap || is_pinned(cmap_out[i]));
    hipStream_t st = c->stream;
    if (pinned) {
        const HostOut host{maps_out, fmap_out, cmap_out};
        // 10 chunks, the last 3 halving: on the 64-conformation ensemble this
        // measured 112-114 ms of GPU time against 116-117 ms for 16 equal chunks
        const auto chunks = plan_chunks(*p, kBatchChunks, kBatchTaper);
        run_checked(p.get(), [&] {
            HIP_CHECK(hipEventRecord(c->ev[0], st));
            enqueue(p.get(), d_maps, d_fmap, d_cmap, false, false, chunks, &host);
            HIP_CHECK(hipEventRecord(c->ev[3], st));
        });
        HIP_CHECK(hipEventElapsedTime(&c->last_ms[3], c->ev[0], c->ev[3]));
        c->last_ms[0] = c->last_ms[1] = c->last_ms[2] = -1.f;
        return;
    }
    plan_execute(p.get(), d_maps, d_fmap, d_cmap);
    for (int i = 0; i < n; i++) {
        const ConfDev &cf = p->confs[i];
        HIP_CHECK(hipMemcpyAsync(maps_out[i], d_maps + cf.map_off, sizeof(float) * (size_t)p->n_maps * cf.P,
                                 hipMemcpyDeviceToHost, st));
        if (d_fmap)
            HIP_CHECK(hipMemcpyAsync(fmap_out[i], d_fmap + cf.pt_off, sizeof(float) * (size_t)cf.P,
                                     hipMemcpyDeviceToHost, st));
        if (d_cmap)
            HIP_CHECK(hipMemcpyAsync(cmap_out[i], d_cmap + cf.pt_off, sizeof(int32_t) * (size_t)cf.P,
                                     hipMemcpyDeviceToHost, st));
    }
    HIP_CHECK(hipStreamSynchronize(st));
}

}  // namespace agdev
