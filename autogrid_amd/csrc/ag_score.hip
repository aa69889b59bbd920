// Ligand scoring against a map set on gfx950: the consumer side of the maps.
//
// AutoDock reads AutoGrid maps by trilinear interpolation.  The maps are
// [n_maps][n1z][n1y][n1x] floats, x fastest (main.cpp:322), on the grid
// described by the .fld file (main.cpp:1903-1956): point (i, j, k) sits at
// ((i - ne_x) s, (j - ne_y) s, (k - ne_z) s) in the grid frame.  A ligand
// atom of map index t and charge q at x scores
//     E(x) = sum over the 8 corners c of w_c(x) (M_t[c] + q M_e[c] + |q| M_d[c]),
// w_c the trilinear weights of x in its cell, and a pose scores the sum of
// its atoms.  An atom outside the grid scores a fixed penalty with zero
// gradient.
//
// Kernels:
//   k_score      one workgroup per pose, lanes over its atoms: per-atom
//                energy and gradient dE/dx, the pose's sum reduced in FP64
//                in a fixed order;
//   k_score_place, k_sort_zero / _scan / _scatter
//                new positions: each atom's place on the grid, and its eight
//                corners sorted by grid point and by (map, grid point), a
//                stable radix sort, so equal keys stay in atom order;
//   k_score_adj  dL/dmaps = S^T dL/dscores for the scores' sparse matrix S:
//                the first entry of each run of equal keys sums its run: a
//                fixed-order sum, no atomics.

#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "ag_devcommon.h"
#include "ag_internal.h"

namespace {

constexpr int kST = 256;

struct __align__(16) ScoreAtom {   // 32 bytes
    float gx, gy, gz;   // position in grid units: (x + ne s) / s
    float q;
    int map;            // map index of the atom's type, -1 for none
    int pose;
    int inside;         // 1 when the 8 corners lie on the grid
    int pad;
};

struct ScoreParams {
    const ScoreAtom *atoms;
    const int *pose_start;      // [n_poses + 1]
    const float *maps;
    long long P;
    int n1x, n1y, n1z;
    int e_slot, d_slot;
    float inv_spacing;
    float outside;
    float *scores;              // [n_poses]
    float *grad;                // [n_atoms][3] or null
};

__global__ void __launch_bounds__(kST) k_score(ScoreParams p) {
    __shared__ double red[kST];
    const int pose = blockIdx.x;
    const int a0 = p.pose_start[pose], a1 = p.pose_start[pose + 1];
    double part = 0.0;
    for (int a = a0 + (int)threadIdx.x; a < a1; a += kST) {
        const ScoreAtom at = p.atoms[a];
        float e = p.outside, g0 = 0.f, g1 = 0.f, g2 = 0.f;
        if (at.inside) {
            const int i0 = (int)floorf(at.gx), j0 = (int)floorf(at.gy), k0 = (int)floorf(at.gz);
            const float fx = at.gx - (float)i0, fy = at.gy - (float)j0, fz = at.gz - (float)k0;
            const float aq = fabsf(at.q);
            e = 0.f;
#pragma unroll
            for (int c = 0; c < 8; c++) {
                const int dx = c & 1, dy = (c >> 1) & 1, dz = c >> 2;
                const long long idx =
                    (long long)(i0 + dx) + (long long)p.n1x * ((long long)(j0 + dy) + (long long)p.n1y * (k0 + dz));
                float v = 0.f;
                if (at.map >= 0) v = p.maps[(long long)at.map * p.P + idx];
                if (p.e_slot >= 0) v = __builtin_fmaf(at.q, p.maps[(long long)p.e_slot * p.P + idx], v);
                if (p.d_slot >= 0) v = __builtin_fmaf(aq, p.maps[(long long)p.d_slot * p.P + idx], v);
                const float wx = dx ? fx : 1.f - fx, wy = dy ? fy : 1.f - fy, wz = dz ? fz : 1.f - fz;
                const float sx = dx ? 1.f : -1.f, sy = dy ? 1.f : -1.f, sz = dz ? 1.f : -1.f;
                e = __builtin_fmaf(wx * wy * wz, v, e);
                g0 = __builtin_fmaf(sx * wy * wz, v, g0);
                g1 = __builtin_fmaf(wx * sy * wz, v, g1);
                g2 = __builtin_fmaf(wx * wy * sz, v, g2);
            }
        }
        if (p.grad) {
            p.grad[3 * (size_t)a] = g0 * p.inv_spacing;
            p.grad[3 * (size_t)a + 1] = g1 * p.inv_spacing;
            p.grad[3 * (size_t)a + 2] = g2 * p.inv_spacing;
        }
        part += (double)e;
    }
    red[threadIdx.x] = part;
    __syncthreads();
    for (int s = kST / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) p.scores[pose] = (float)red[0];
}

__global__ void k_score_zero(float *out, long long n) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        out[i] = 0.f;
}

// One pass of a stable radix sort of (key, entry) pairs by eight bits: with the
// tiles' digit counts known, each pair's place is that of its digit (a digit's
// tiles follow each other).  A digit comes from the key, or from the entry's
// atom's map (map + 1, so that atoms without one go first).  Whoever places a
// pair counts it for the next pass, so a pass is one launch, which up to
// kSortScanned tiles also adds up the counts itself (each workgroup all of
// them, from the L2 cache).  10,000 atoms, 80,000 pairs: 39 us for all four
// passes; as three launches each (count, scan, scatter) 66 us and the gaps
// between.  (Pairs a workgroup has spread go out one cache line a clock: 40
// workgroups of 2,048 take 9.5 us a pass, ten of 8,192 15.)  The host's sort of
// the 250,000 contributions and their upload took 5.4 ms.
constexpr int kSortThreads = 512, kSortPer = 4;
constexpr int kSortTile = kSortThreads * kSortPer;   // pairs of a workgroup
constexpr int kSortScanned = 64;

// The digits of a pass and its counts.
struct SortDigit {
    const ScoreAtom *by_map;    // null: the digit is (key >> shift) & 255
    int shift;
    int *count;                 // [tiles][256]; null: no pass
};
struct SortPass {
    const uint2 *pair;          // (key, entry)
    uint2 *pair_out;
    int n, tiles;
    int scanned;                // the counts have been through k_sort_scan
    SortDigit digit, next;
    int *clear;                 // the counts of the pass before, left clear for the next sort
};
__device__ __forceinline__ int sort_digit(const SortDigit &p, uint2 pair) {
    return p.by_map ? p.by_map[pair.y >> 3].map + 1 : (int)((pair.x >> p.shift) & 255u);
}
__device__ __forceinline__ void sort_count(const SortDigit &p, uint2 pair, int place) {
    atomicAdd(&p.count[place / kSortTile * 256 + sort_digit(p, pair)], 1);
}

// Clears the counts of all passes, before a scorer's first sort.
__global__ void __launch_bounds__(kST) k_sort_zero(int *count, int n) {
    const int i = blockIdx.x * kST + threadIdx.x;
    if (i < n) count[i] = 0;
}

struct PlaceParams {
    const double *xyz;          // [n][3]
    const float *charge;
    const int *map, *pose;
    int n;
    int n1[3];
    double shift[3], spacing;   // ne * spacing
    unsigned P;                 // grid points; the key of an atom off the grid
    ScoreAtom *atoms;
    uint2 *pair;                // [8 n] (corner's grid point, atom * 8 + corner)
    SortDigit first;            // of the sort
    int *clear;                 // counts of the last sort's last pass, 256 per 256 atoms
};

// An atom's place on the grid and its eight corners' pairs.
__device__ __forceinline__ void place_atom(const PlaceParams &p, int a, int *bin) {
    double g[3];
    bool inside = true;
    for (int d = 0; d < 3; d++) {
        g[d] = (p.xyz[3 * (size_t)a + d] + p.shift[d]) / p.spacing;
        // the 8 corners must lie on the grid: 0 <= g < n1 - 1
        inside = inside && g[d] >= 0.0 && g[d] < (double)(p.n1[d] - 1);
    }
    ScoreAtom at;
    at.gx = (float)g[0];
    at.gy = (float)g[1];
    at.gz = (float)g[2];
    // FP32 rounding may carry g onto n1 - 1: keep such atoms outside
    inside = inside && at.gx < (float)(p.n1[0] - 1) && at.gy < (float)(p.n1[1] - 1) && at.gz < (float)(p.n1[2] - 1);
    at.q = p.charge[a];
    at.map = p.map[a];
    at.pose = p.pose[a];
    at.inside = inside ? 1 : 0;
    at.pad = 0;
    p.atoms[a] = at;
    const int i0 = (int)floorf(at.gx), j0 = (int)floorf(at.gy), k0 = (int)floorf(at.gz);
    for (int c = 0; c < 8; c++) {
        const unsigned pt = inside ? (unsigned)(i0 + (c & 1)) +
                                         (unsigned)p.n1[0] * ((unsigned)(j0 + ((c >> 1) & 1)) +
                                                              (unsigned)p.n1[1] * (unsigned)(k0 + (c >> 2)))
                                   : p.P;
        const uint2 pair = make_uint2(pt, 8u * a + c);
        p.pair[8 * (size_t)a + c] = pair;
        atomicAdd(&bin[sort_digit(p.first, pair)], 1);
    }
}

__global__ void __launch_bounds__(kST) k_score_place(PlaceParams p) {
    const int a = blockIdx.x * kST + threadIdx.x;
    static_assert(kSortTile == 8 * kST && kST == 256, "a workgroup's corners are a tile");
    // the tile's digits for the first pass, counted in LDS
    __shared__ int bin[256];
    bin[threadIdx.x] = 0;
    p.clear[a] = 0;
    __syncthreads();
    if (a < p.n) place_atom(p, a, bin);
    __syncthreads();
    p.first.count[a] = bin[threadIdx.x];
}

// count[b][d] -> pairs of smaller digits plus digit d's of earlier blocks.  One
// workgroup: a thread walks a quarter of the blocks for one digit.
__global__ void __launch_bounds__(1024) k_sort_scan(int *count, int blocks) {
    __shared__ int part[4][256], wave_sum[4];
    const int d = threadIdx.x & 255, g = threadIdx.x >> 8, lane = threadIdx.x & 63;
    const int per = (blocks + 3) / 4, b0 = min(blocks, g * per), b1 = min(blocks, b0 + per);
    int s = 0;
#pragma unroll 8
    for (int b = b0; b < b1; b++) s += count[b * 256 + d];
    part[g][d] = s;
    __syncthreads();
    const int total = part[0][d] + part[1][d] + part[2][d] + part[3][d];
    int x = total;   // inclusive scan over the digits: a wave's 64, then the waves before
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63 && g == 0) wave_sum[d >> 6] = x;
    __syncthreads();
    int run = x - total;
    for (int w = 0; w < (d >> 6); w++) run += wave_sum[w];
    for (int k = 0; k < g; k++) run += part[k][d];
#pragma unroll 8
    for (int b = b0; b < b1; b++) {
        const int c = count[b * 256 + d];
        count[b * 256 + d] = run;
        run += c;
    }
}

// A wave takes its part of the workgroup's tile in order: its digits' counts first,
// then, with the waves' places known, 64 pairs at a time without a barrier.
__global__ void __launch_bounds__(kSortThreads) k_sort_scatter(SortPass p) {
    constexpr int kWaves = kSortThreads / 64;
    __shared__ int place[kWaves][256];   // next free place per wave and digit
    __shared__ int wave_sum[kWaves];
    __shared__ int2 other[256];
    // counts for the next pass: many pairs may share one (few digits, or one
    // map's atoms), so they are added up here before they go to memory
    __shared__ int ahead[kSortScanned * 256];
    const bool gather_ahead = p.next.count && p.tiles <= kSortScanned;
    if (p.clear && threadIdx.x < 256) p.clear[blockIdx.x * 256 + threadIdx.x] = 0;
    if (gather_ahead)
        for (int k = threadIdx.x; k < p.tiles * 256; k += kSortThreads) ahead[k] = 0;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int d = threadIdx.x & 255;
    for (int w = threadIdx.x >> 8; w < kWaves; w += kSortThreads / 256) place[w][d] = 0;
    int run = 0;   // the tile's first place of digit d
    if (p.scanned) {
        run = p.digit.count[blockIdx.x * 256 + d];
    } else {
        // two threads per digit, every other tile each
        static_assert(kSortThreads == 512, "two threads per digit");
        const int half = threadIdx.x >> 8;
        int total = 0;
#pragma unroll 16
        for (int b = half; b < p.tiles; b += 2) {
            const int c = p.digit.count[b * 256 + d];
            total += c;
            run += b < (int)blockIdx.x ? c : 0;
        }
        if (half) other[d] = make_int2(total, run);
        __syncthreads();
        total += other[d].x;
        run += other[d].y;
        int x = total;   // (the lower half's; the upper half's are not used)
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o);
            if (lane >= o) x += y;
        }
        if (lane == 63 && !half) wave_sum[wave] = x;
        __syncthreads();
        run += x - total;
        for (int w = 0; w < (d >> 6); w++) run += wave_sum[w];
    }
    __syncthreads();
    uint2 pair[kSortPer];
    int digit[kSortPer];
    const int first = blockIdx.x * kSortTile + wave * (kSortPer * 64) + lane;
#pragma unroll
    for (int r = 0; r < kSortPer; r++) {
        const int i = first + 64 * r;
        digit[r] = -1;
        if (i < p.n) {
            pair[r] = p.pair[i];
            digit[r] = sort_digit(p.digit, pair[r]);
            atomicAdd(&place[wave][digit[r]], 1);
        }
    }
    __syncthreads();
    if (threadIdx.x < 256)
        for (int w = 0; w < kWaves; w++) {
            const int c = place[w][d];
            place[w][d] = run;
            run += c;
        }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortPer; r++) {
        const bool act = digit[r] >= 0;
        const int dg = act ? digit[r] : 0;
        unsigned long long same = __ballot(act);   // the wave's lanes with this digit
        for (int b = 0; b < 8; b++) {
            const unsigned long long m = __ballot((dg >> b) & 1);
            same &= (dg >> b) & 1 ? m : ~m;
        }
        const int rank = __popcll(same & ((1ull << lane) - 1));
        const int at = place[wave][dg];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // every lane has read its place
        __builtin_amdgcn_wave_barrier();
        if (act) {
            p.pair_out[at + rank] = pair[r];
            if (gather_ahead)
                atomicAdd(&ahead[(at + rank) / kSortTile * 256 + sort_digit(p.next, pair[r])], 1);
            else if (p.next.count)
                sort_count(p.next, pair[r], at + rank);
            if (rank == 0) place[wave][dg] = at + __popcll(same);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    if (gather_ahead) {
        __syncthreads();
        for (int k = threadIdx.x; k < p.tiles * 256; k += kSortThreads)
            if (ahead[k]) atomicAdd(&p.next.count[k], ahead[k]);
    }
}

// Runs of equal keys, summed by their first entry's lane in FP64 in order: e
// and d over all of a grid point's entries, an affinity map over the entries
// of its own atoms.  Slots may coincide (an atom's map with e or d, e with d):
// an entry then adds its map's, e's and d's term in that order.
struct AdjParams {
    const ScoreAtom *atoms;
    int n;                      // entries, 8 per atom
    unsigned P;
    const uint2 *pair;          // (grid point, entry) sorted by grid point
    const uint2 *mpair;         // sorted by map, then grid point
    int e_slot, d_slot;
    const float *dscore;
    float *dmaps;
};
__device__ __forceinline__ float corner_weight(const ScoreAtom &at, int c) {
    const float fx = at.gx - floorf(at.gx), fy = at.gy - floorf(at.gy), fz = at.gz - floorf(at.gz);
    return ((c & 1) ? fx : 1.f - fx) * (((c >> 1) & 1) ? fy : 1.f - fy) * ((c >> 2) ? fz : 1.f - fz);
}

__global__ void __launch_bounds__(kST) k_score_adj(AdjParams p) {
    const int i = blockIdx.x * kST + threadIdx.x;
    if (i >= p.n) return;
    if (blockIdx.y == 0) {
        const unsigned pt = p.pair[i].x;
        if (pt >= p.P || (i > 0 && p.pair[i - 1].x == pt)) return;
        double se = 0.0, sd = 0.0;
        for (int k = i; k < p.n && p.pair[k].x == pt; k++) {
            const int en = (int)p.pair[k].y;
            const ScoreAtom at = p.atoms[en >> 3];
            const float w = corner_weight(at, en & 7);
            const double g = (double)p.dscore[at.pose];
            if (at.map == p.e_slot) se += (double)w * g;
            se += (double)(w * at.q) * g;
            if (p.d_slot == p.e_slot) {
                se += (double)(w * fabsf(at.q)) * g;
            } else {
                if (at.map == p.d_slot) sd += (double)w * g;
                sd += (double)(w * fabsf(at.q)) * g;
            }
        }
        if (p.e_slot >= 0) p.dmaps[(size_t)p.e_slot * p.P + pt] = (float)se;
        if (p.d_slot >= 0 && p.d_slot != p.e_slot) p.dmaps[(size_t)p.d_slot * p.P + pt] = (float)sd;
    } else {
        const unsigned pt = p.mpair[i].x;
        const int m = p.atoms[p.mpair[i].y >> 3].map;
        if (pt >= p.P || m < 0 || m == p.e_slot || m == p.d_slot) return;
        if (i > 0 && p.mpair[i - 1].x == pt && p.atoms[p.mpair[i - 1].y >> 3].map == m) return;
        double s = 0.0;
        for (int k = i; k < p.n && p.mpair[k].x == pt; k++) {
            const int en = (int)p.mpair[k].y;
            const ScoreAtom at = p.atoms[en >> 3];
            if (at.map != m) break;
            s += (double)corner_weight(at, en & 7) * (double)p.dscore[at.pose];
        }
        p.dmaps[(size_t)m * p.P + pt] = (float)s;
    }
}

}  // namespace

struct ag_scorer {
    ag_ctx *ctx = nullptr;
    int n1[3] = {0, 0, 0}, ne[3] = {0, 0, 0};
    double spacing = 0.0;
    long long P = 0;
    int n_maps = 0, e_slot = -1, d_slot = -1;
    int n_poses = 0, n_atoms = 0;
    float outside = 0.f;
    std::vector<int> pose_start;
    std::vector<int> map_index;
    DevBuf atoms, pose_start_d, xyz, charge_d, map_d, pose_d;
    DevBuf pair[3], count;
    bool counts_clear = false;      // every pass's counts but the last's are clear
    int by_point = 0, by_map = 0;   // buffers holding the two sorted lists
};

namespace agdev {

static void scorer_positions(ag_scorer *s, const double *xyz) {
    const int n = s->n_atoms;
    for (size_t i = 0; i < 3 * (size_t)n; i++)
        if (!std::isfinite(xyz[i])) ag::fail(AG_ERR_BAD_INPUT, "ligand position is not finite");
    hipStream_t st = s->ctx->stream;
    const size_t n8 = 8 * (size_t)n;
    if (n8 > (size_t)INT32_MAX) ag::fail(AG_ERR_UNSUPPORTED, "too many ligand atoms for one scorer");
    PlaceParams pp;
    memset(&pp, 0, sizeof pp);
    pp.xyz = (const double *)s->xyz.get(sizeof(double) * 3 * (size_t)n);
    pp.charge = (const float *)s->charge_d.ptr;
    pp.map = (const int *)s->map_d.ptr;
    pp.pose = (const int *)s->pose_d.ptr;
    pp.n = n;
    for (int d = 0; d < 3; d++) {
        pp.n1[d] = s->n1[d];
        pp.shift[d] = s->ne[d] * s->spacing;
    }
    pp.spacing = s->spacing;
    pp.P = (unsigned)s->P;
    pp.atoms = (ScoreAtom *)s->atoms.get(sizeof(ScoreAtom) * (size_t)n);
    const int blocks = (int)((n8 + kSortTile - 1) / kSortTile);
    for (int k = 0; k < 3; k++) {
        s->pair[k].get(sizeof(uint2) * n8);
    }
    // the passes: by grid point, eight bits at a time, then by map
    SortDigit digit[6] = {};
    int passes = 0;
    const size_t counts = 256 * (size_t)std::max(blocks, 1);
    int *count = (int *)s->count.get(sizeof(int) * counts * 5);
    for (int shift = 0; shift < 32 && ((unsigned long long)s->P >> shift) > 0; shift += 8)
        digit[passes++] = SortDigit{nullptr, shift, nullptr};
    digit[passes++] = SortDigit{pp.atoms, 0, nullptr};
    for (int k = 0; k < passes; k++) digit[k].count = count + counts * k;
    if (n == 0) return;
    // pinned staging: one DMA instead of the runtime's own staged copy
    void *stage = s->ctx->stage.get(sizeof(double) * 3 * (size_t)n);
    memcpy(stage, xyz, sizeof(double) * 3 * (size_t)n);
    HIP_CHECK(hipMemcpyAsync(s->xyz.ptr, stage, sizeof(double) * 3 * (size_t)n, hipMemcpyHostToDevice, st));
    pp.pair = (uint2 *)s->pair[0].ptr;
    pp.first = digit[0];
    pp.clear = digit[passes - 1].count;
    if (!s->counts_clear)
        k_sort_zero<<<(unsigned)((counts * passes + kST - 1) / kST), kST, 0, st>>>(count, (int)(counts * passes));
    s->counts_clear = false;
    k_score_place<<<(n + kST - 1) / kST, kST, 0, st>>>(pp);
    // each pass but the last (by map, from the list by grid point) goes to
    // and fro between two buffers
    const bool scan = blocks > kSortScanned;
    for (int k = 0, from = 0; k < passes; k++, from = 1 - from) {
        const bool last = k + 1 == passes;
        const int to = last ? 2 : 1 - from;
        if (scan) k_sort_scan<<<1, 1024, 0, st>>>(digit[k].count, blocks);
        k_sort_scatter<<<blocks, kSortThreads, 0, st>>>(SortPass{
            (const uint2 *)s->pair[from].ptr, (uint2 *)s->pair[to].ptr, (int)n8, blocks, scan, digit[k], digit[k + 1],
            k > 0 ? digit[k - 1].count : nullptr});
        if (last) s->by_point = from;
    }
    s->by_map = 2;
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipStreamSynchronize(st));   // the staging buffer is the context's
    s->counts_clear = true;
}

ag_scorer *scorer_create(ag_ctx *c, const ag_grid *grid, int n_maps, int elec_index, int dsolv_index, int n_poses,
                         const int32_t *pose_start, const double *xyz, const int32_t *map_index,
                         const double *charge, double outside) {
    for (int d = 0; d < 3; d++)
        if (grid->n1[d] < 2 || grid->n1[d] > AG_MAX_GRID_PTS || grid->ne[d] < 0)
            ag::fail(AG_ERR_BAD_INPUT, "grid dimensions out of range (at least 2 points per axis)");
    if (!(grid->spacing > 0)) ag::fail(AG_ERR_BAD_INPUT, "grid spacing must be positive");
    if (n_maps < 1 || n_maps > AG_MAX_MAPS) ag::fail(AG_ERR_BAD_INPUT, "map count out of range");
    if (elec_index >= n_maps || dsolv_index >= n_maps) ag::fail(AG_ERR_BAD_INPUT, "e/d map index out of range");
    if (n_poses < 1) ag::fail(AG_ERR_BAD_INPUT, "no poses");
    if (pose_start[0] != 0) ag::fail(AG_ERR_BAD_INPUT, "pose_start[0] must be 0");
    for (int p = 0; p < n_poses; p++)
        if (pose_start[p + 1] < pose_start[p]) ag::fail(AG_ERR_BAD_INPUT, "pose_start must not decrease");
    const int n = pose_start[n_poses];
    if (n > 0 && (!xyz || !map_index || !charge)) ag::fail(AG_ERR_BAD_INPUT, "ligand arrays missing");
    for (int a = 0; a < n; a++) {
        if (map_index[a] < -1 || map_index[a] >= n_maps) ag::fail(AG_ERR_BAD_INPUT, "ligand map index out of range");
        if (!std::isfinite(charge[a])) ag::fail(AG_ERR_BAD_INPUT, "ligand charge is not finite");
    }
    HIP_CHECK(hipSetDevice(c->device));
    std::unique_ptr<ag_scorer> s(new ag_scorer());
    s->ctx = c;
    for (int d = 0; d < 3; d++) {
        s->n1[d] = grid->n1[d];
        s->ne[d] = grid->ne[d];
    }
    s->spacing = grid->spacing;
    s->P = (long long)grid->n1[0] * grid->n1[1] * grid->n1[2];
    s->n_maps = n_maps;
    s->e_slot = elec_index;
    s->d_slot = dsolv_index;
    s->n_poses = n_poses;
    s->n_atoms = n;
    s->outside = (float)outside;
    s->pose_start.assign(pose_start, pose_start + n_poses + 1);
    s->map_index.assign(map_index, map_index + n);
    std::vector<float> q(std::max(n, 1));
    std::vector<int> pose(std::max(n, 1));
    for (int p = 0; p < n_poses; p++)
        for (int a = pose_start[p]; a < pose_start[p + 1]; a++) {
            q[a] = (float)charge[a];
            pose[a] = p;
        }
    const auto up = [&](DevBuf &b, const void *src, size_t bytes) {
        void *d = b.get(std::max<size_t>(bytes, 16));
        if (bytes) HIP_CHECK(hipMemcpyAsync(d, src, bytes, hipMemcpyHostToDevice, c->stream));
    };
    up(s->pose_start_d, s->pose_start.data(), sizeof(int) * (size_t)(n_poses + 1));
    up(s->charge_d, q.data(), sizeof(float) * (size_t)n);
    up(s->map_d, s->map_index.data(), sizeof(int) * (size_t)n);
    up(s->pose_d, pose.data(), sizeof(int) * (size_t)n);
    HIP_CHECK(hipStreamSynchronize(c->stream));   // host vectors go out of scope
    scorer_positions(s.get(), xyz);
    return s.release();
}

void scorer_set_positions(ag_scorer *s, const double *xyz) {
    HIP_CHECK(hipSetDevice(s->ctx->device));
    if (s->n_atoms > 0 && !xyz) ag::fail(AG_ERR_BAD_INPUT, "ligand positions missing");
    scorer_positions(s, xyz);
}

void scorer_score(ag_scorer *s, const float *d_maps, float *d_scores, float *d_grad) {
    HIP_CHECK(hipSetDevice(s->ctx->device));
    hipStream_t st = s->ctx->stream;
    ScoreParams p;
    memset(&p, 0, sizeof p);
    p.atoms = (const ScoreAtom *)s->atoms.ptr;
    p.pose_start = (const int *)s->pose_start_d.ptr;
    p.maps = d_maps;
    p.P = s->P;
    p.n1x = s->n1[0];
    p.n1y = s->n1[1];
    p.n1z = s->n1[2];
    p.e_slot = s->e_slot;
    p.d_slot = s->d_slot;
    p.inv_spacing = (float)(1.0 / s->spacing);
    p.outside = s->outside;
    p.scores = d_scores;
    p.grad = d_grad;
    k_score<<<s->n_poses, kST, 0, st>>>(p);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipStreamSynchronize(st));
}

void scorer_adjoint(ag_scorer *s, const float *d_dscore, float *d_dmaps) {
    HIP_CHECK(hipSetDevice(s->ctx->device));
    hipStream_t st = s->ctx->stream;
    const long long total = s->P * s->n_maps;
    const unsigned zb = (unsigned)std::min<long long>((total + 255) / 256, 65536);
    k_score_zero<<<zb, 256, 0, st>>>(d_dmaps, total);
    if (s->n_atoms > 0) {
        const int n8 = 8 * s->n_atoms;
        AdjParams p{(const ScoreAtom *)s->atoms.ptr, n8, (unsigned)s->P, (const uint2 *)s->pair[s->by_point].ptr,
                    (const uint2 *)s->pair[s->by_map].ptr, s->e_slot, s->d_slot, d_dscore, d_dmaps};
        k_score_adj<<<dim3((unsigned)((n8 + kST - 1) / kST), 2), kST, 0, st>>>(p);
    }
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipStreamSynchronize(st));
}

void scorer_destroy(ag_scorer *s) {
    if (!s) return;
    (void)hipSetDevice(s->ctx->device);
    (void)hipStreamSynchronize(s->ctx->stream);
    delete s;
}

}  // namespace agdev
