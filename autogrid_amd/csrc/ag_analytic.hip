// Analytic (differentiable) map mode on gfx950.
//
// The map set is evaluated from the functional forms behind the reference's
// tables instead of the tables themselves (main.cpp:2040-2276 tables,
// main.cpp:2805-3431 per-point loop):
//   E_mt(r)  = min(EINTCLAMP, Phi_mt(s(r))), Phi the 12-6 / 12-10 pair
//              potential, s(r) the continuous form of the min-window
//              smoothing (r + w left of the well, r* inside, r - w right);
//   sol(r)   = coeff_desolv exp(-r^2 / (2 * 3.6^2));
//   e        = sum over all atoms of q coeff_estat (332 / eps(r)) / max(r, 0.5),
//              eps the Mehler-Solmajer dielectric at r;
// every 8 A term multiplied by the switch S(r) = 1 - u^3 (10 - 15 u + 6 u^2),
// u = clamp((r - 7.5) / 0.5, 0, 1), in place of the hard cutoff, so the maps
// are continuous in the receptor coordinates.  The per-point assembly (closest
// donor H, racc / rdon / Hramp, the H-bond case split with its min / max,
// desolvation, d map) is the reference's.
//
// Kernels (FP32):
//   k_an_near   one workgroup per cube of 4x4x4 points, its four waves sharing
//               the atoms within 8 A (host-built cell list): affinity, covalent
//               and d maps, plus the tape the adjoint needs (closest H, the
//               atoms that gave each point's H-bond min and max);
//   k_an_e      runs of 13 or 16 points along x per lane over one chunk of
//               atoms, and k_an_esum the chunks' sums per point: the e map; of
//               larger receptors k_an_ebox sums the atoms beyond boxes of about
//               16x16x16 points at 512 Chebyshev nodes of each, and k_an_epatch
//               the rest point by point, with the nodes' values interpolated;
//   k_an_vh     in the cubes of k_an_near: the cotangent of the closest H's
//               bond vector through every Hramp at each point;
//   k_an_hsum   one workgroup per donor H: sums k_an_vh's vectors over the
//               points whose closest H it is (of the points where they are
//               nonzero, packed);
//   k_an_atom   one workgroup per atom: gathers over the grid points within
//               8 A of it the gradients of the 8 A terms with respect to its
//               position, bond vectors, charge, pair parameters and the
//               desolvation weight, beside the kernels on the second stream;
//   k_an_count / k_an_gscan / k_an_pack
//               points where a cotangent is nonzero, packed in point order
//               (the e map's for k_an_eadj, the bond-vector one for
//               k_an_hsum); k_an_gmask flags the points k_an_atom reads;
//   k_an_eadj   atoms x chunks of packed points: the e map's gradients,
//               written as per-chunk partial sums that k_an_ered adds in a
//               fixed order.
// Nothing accumulates through atomics: every gradient is a fixed-order sum,
// so results are bitwise repeatable.

#include <hip/hip_runtime.h>
#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "ag_devcommon.h"
#include "ag_internal.h"

namespace {

#define AN_CONST __attribute__((address_space(4)))   // read-only tables, through scalar loads

constexpr int kAT = 256;                 // threads per workgroup
constexpr int kAMaxAff = 8;              // affinity maps per analytic set (registers, unrolled)
constexpr float kSwOn = 7.5f, kSwInvLen = 2.0f;  // switch from 7.5 A, over 0.5 A
constexpr float kCut2 = 64.0f;
constexpr float kInv2Sig2 = 1.0f / (2.0f * 3.6f * 3.6f);
constexpr float kClamp = 100000.f;       // EINTCLAMP
constexpr float kCellA = 4.0f;           // cell edge (A)
constexpr int kEAtoms = 128;             // atoms per chunk of the forward e kernel (at least)
constexpr int kEMaxChunks = 64;          // chunks of the forward e kernel (at most)
// Mehler-Solmajer constants (distdepdiel.cpp:30-57)
constexpr float kMsA = -8.5525f, kMsB = 78.4f + 8.5525f, kMsK = 7.7839f, kMsLB = 0.003627f * (78.4f + 8.5525f);

enum : int { CASE_PLAIN = 0, CASE_ACC = 1, CASE_MM_RACC = 2, CASE_MM_RDON = 3 };

struct AAtom {            // 64 bytes, in cell order
    float x, y, z, q;     // grid frame; charge
    float vol, solpar;
    int meta;             // type | hbond << 8 | rexp << 16
    int index;
    float rv[3];
    float pad0;
    float rv2[3];
    float pad1;
};
static_assert(sizeof(AAtom) == 64, "AAtom layout");

struct APair {            // one (map, receptor type) pair potential
    float R, eps;         // derived form (eps effective)
    float cA, cB;         // explicit form (nbp_coeffs)
    float rstar;          // minimum of Phi
    int a, b, expl;
};

struct __align__(16) ANear {   // E = c1 (R/s)^a - c2 (R/s)^b, capped (R = 1 for nbp_coeffs pairs)
    float R, c1, c2, rstar;
};
struct __align__(16) ANearType {   // of one receptor type: the forward's form of its pairs
    ANear pair[kAMaxAff];
    int form;                      // 2 bits per map: exponents 12-6 (0), 12-10 (1), others (2)
    int pad[3];
    int a[kAMaxAff], b[kAMaxAff];
};

struct AParams {
    int n1[3], ne[3];
    float h;                          // spacing
    long long P;
    // cells over the box padded by 8 A
    float corg[3];
    int nc[3];
    const int *cell_start;            // [ncells + 1]
    const AAtom *atoms;               // cell order
    const float *rv_by_index;         // [N][3] bond vectors by atom index
    int n_atoms;
    // maps
    int naff;
    int aff_slot[kAMaxAff], des_slot[kAMaxAff];
    float sp[kAMaxAff], volp[kAMaxAff];  // desolvation parameters of des_slot
    int cov_slot[16], n_cov;
    double cov_pos[3], cov_hw, cov_barrier;
    int d_slot;
    const APair *pairs;               // [naff][T]
    const ANearType *near_pairs;      // [T]
    int case_word[7];                 // per atom class, 2 bits per map: its CASE_*
    int T;
    float w_smooth;                   // half window (A)
    float w_desolv, qasp;
    float *maps;                      // [n_maps][P]
    // tape
    int *closest_h;                   // [P]
    int *amin, *amax;                 // [naff][P]
    // adjoint
    const float *dmaps;               // cotangent [n_maps][P]
    float *vh;                        // [P][3]
};

__device__ __forceinline__ float switch_s(float r, float &dS) {
    const float u = fminf(fmaxf((r - kSwOn) * kSwInvLen, 0.f), 1.f);
    const float u2 = u * u;
    dS = -30.f * u2 * (1.f - u) * (1.f - u) * kSwInvLen;
    return 1.f - u2 * u * (10.f - 15.f * u + 6.f * u2);
}

__device__ __forceinline__ float powi(float x, int n) {
    float x2 = x * x, x4 = x2 * x2, x8 = x4 * x4;
    switch (n) {
        case 12: return x8 * x4;
        case 10: return x8 * x2;
        case 6: return x4 * x2;
        case 4: return x4;
        default: {
            float r = 1.f;
            for (int i = 0; i < n; i++) r *= x;
            return r;
        }
    }
}

__device__ __forceinline__ APair load_pair(const AN_CONST APair *p) {
    APair o;
    o.R = p->R;
    o.eps = p->eps;
    o.cA = p->cA;
    o.cB = p->cB;
    o.rstar = p->rstar;
    o.a = p->a;
    o.b = p->b;
    o.expl = p->expl;
    return o;
}

// Smoothed, capped pair energy and its derivatives (FP32).
struct LJ {
    float E, dEdr, dEdR, dEdeps;
};
__device__ __forceinline__ LJ lj_eval(const APair &pp, float r, float w) {
    float s, dsdr;
    if (r < pp.rstar - w) { s = r + w; dsdr = 1.f; }
    else if (r > pp.rstar + w) { s = r - w; dsdr = 1.f; }
    else { s = pp.rstar; dsdr = 0.f; }
    const float a = (float)pp.a, b = (float)pp.b;
    LJ o;
    float dPds, dPdR = 0.f, dPdeps = 0.f;
    // hardware reciprocals (about 1 ulp; rho^12 carries 12 of them, ~1e-6
    // relative, far inside the tolerances); a - b is a small integer
    const float is = __builtin_amdgcn_rcpf(s);
    if (!pp.expl) {
        const float rho = pp.R * is;
        const float pa = powi(rho, pp.a), pb = powi(rho, pp.b);
        const float k = __builtin_amdgcn_rcpf(a - b);
        o.E = pp.eps * k * (b * pa - a * pb);
        dPds = pp.eps * k * a * b * (pb - pa) * is;
        if (dsdr != 0.f) dPdR = pp.eps * k * a * b * (pa - pb) * __builtin_amdgcn_rcpf(pp.R);
        dPdeps = k * (b * pa - a * pb);
    } else {
        const float pa = powi(is, pp.a), pb = powi(is, pp.b);
        o.E = pp.cA * pa - pp.cB * pb;
        dPds = (-a * pp.cA * pa + b * pp.cB * pb) * is;
    }
    if (o.E >= kClamp) {
        o.E = kClamp;
        o.dEdr = o.dEdR = o.dEdeps = 0.f;
        return o;
    }
    o.dEdr = dPds * dsdr;
    o.dEdR = dPdR;
    o.dEdeps = dPdeps;
    return o;
}

__device__ __forceinline__ float racc_of(float c, int rexp, float &dc) {
    if (!(c > 0.f)) { dc = 0.f; return 0.f; }
    if (rexp == 2) { dc = 2.f * c; return c * c; }
    if (rexp == 4) { const float c2 = c * c; dc = 4.f * c2 * c; return c2 * c2; }
    dc = 1.f;
    return c;
}

// Hramp of a D1 atom against the closest H, 0.5 - 0.5 cos(4/3 acos(ct)), and
// its derivative -(2/3) sin(4/3 t) / sin t, t = acos(ct).  With h = cos(t / 2),
// the derivative times h is analytic on [0, 1]: a degree-8 Chebyshev fit,
// 1.7e-8 off at most.  Past |ct| = 1 (clamped) it is 0; where sin t < 1e-4
// beside t = pi (h < 5e-5) it is taken as its value at t = 0.
__device__ __forceinline__ float hramp_of(float ct_raw, float &dct) {
    const float ct = fminf(fmaxf(ct_raw, -1.f), 1.f);
    const float h = __builtin_amdgcn_sqrtf(fmaxf(__builtin_fmaf(0.5f, ct, 0.5f), 0.f));
    float g = -0.00302975586f;
    g = __builtin_fmaf(g, h, 0.0172578153f);
    g = __builtin_fmaf(g, h, -0.0467509426f);
    g = __builtin_fmaf(g, h, 0.0856716455f);
    g = __builtin_fmaf(g, h, -0.13386068f);
    g = __builtin_fmaf(g, h, 0.229579017f);
    g = __builtin_fmaf(g, h, -0.881983904f);
    g = __builtin_fmaf(g, h, -0.444447247f);
    g = __builtin_fmaf(g, h, 0.288675151f);
    dct = ct_raw >= 1.f || ct_raw <= -1.f ? 0.f : h > 5.0e-5f ? g * __builtin_amdgcn_rcpf(h) : -8.f / 9.f;
    return hramp_value(ct);
}

// Ordered A2 lone-pair rdon (main.cpp:3185-3246) with the identities
// cos(pi/2 - acos x) = sqrt(1 - x^2) and sin(2 |acos y - pi/2|) = 2 |y| sqrt(1 - y^2).
// With GRAD, adds gbar * d rdon / d(dn, rv, rv2) into gdn, grv, grv2.
template <bool GRAD>
__device__ __forceinline__ float a2_rdon(const float dn[3], const float rv[3], const float rv2[3], float gbar,
                                         float gdn[3], float grv[3], float grv2[3]) {
    const float cos_t = -(dn[0] * rv[0] + dn[1] * rv[1] + dn[2] * rv[2]);
    const float xr = dn[0] * rv2[0] + dn[1] * rv2[1] + dn[2] * rv2[2];
    const float x = fminf(fmaxf(xr, -1.f), 1.f);
    const float ct0 = sqrtf(fmaxf(1.f - x * x, 0.f));
    float rdon = 0.f, g_ct0 = 0.f;
    if (cos_t >= 0.f) {
        const float cr[3] = {dn[1] * rv2[2] - dn[2] * rv2[1], dn[2] * rv2[0] - dn[0] * rv2[2],
                             dn[0] * rv2[1] - dn[1] * rv2[0]};
        const float rd2r = cr[0] * cr[0] + cr[1] * cr[1] + cr[2] * cr[2];
        const float rd2 = fmaxf(rd2r, 1.0e-6f);
        const float inv = 1.f / sqrtf(rd2);
        const float ch[3] = {cr[0] * inv, cr[1] * inv, cr[2] * inv};
        const float yr = ch[0] * rv[0] + ch[1] * rv[1] + ch[2] * rv[2];
        const float y = fminf(fmaxf(yr, -1.f), 1.f);
        const float sq = sqrtf(fmaxf(1.f - y * y, 0.f));
        const float sin2ti = 2.f * fabsf(y) * sq;
        rdon = (0.9f + 0.1f * sin2ti) * ct0;
        if (GRAD) {
            g_ct0 = gbar * (0.9f + 0.1f * sin2ti);
            const float g_s = gbar * 0.1f * ct0;
            float g_y = 0.f;
            if (yr > -1.f && yr < 1.f && sq > 1.0e-6f) g_y = g_s * 2.f * copysignf(1.f, y) * (1.f - 2.f * y * y) / sq;
            // y = ch . rv
            float gch[3];
            for (int k = 0; k < 3; k++) {
                grv[k] += g_y * ch[k];
                gch[k] = g_y * rv[k];
            }
            // ch = cr / |cr|
            float gcr[3];
            if (rd2r > 1.0e-6f) {
                const float dot = gch[0] * ch[0] + gch[1] * ch[1] + gch[2] * ch[2];
                for (int k = 0; k < 3; k++) gcr[k] = (gch[k] - dot * ch[k]) * inv;
            } else {
                for (int k = 0; k < 3; k++) gcr[k] = gch[k] * inv;
            }
            // cr = dn x rv2: d dn = rv2 x gcr, d rv2 = gcr x dn
            gdn[0] += rv2[1] * gcr[2] - rv2[2] * gcr[1];
            gdn[1] += rv2[2] * gcr[0] - rv2[0] * gcr[2];
            gdn[2] += rv2[0] * gcr[1] - rv2[1] * gcr[0];
            grv2[0] += gcr[1] * dn[2] - gcr[2] * dn[1];
            grv2[1] += gcr[2] * dn[0] - gcr[0] * dn[2];
            grv2[2] += gcr[0] * dn[1] - gcr[1] * dn[0];
        }
    } else if (cos_t >= -0.34202f) {
        const float u = 0.116978f - cos_t * cos_t;
        rdon = 562.25f * (u * u * u) * ct0;
        if (GRAD) {
            g_ct0 = gbar * 562.25f * (u * u * u);
            const float g_c = gbar * 562.25f * 3.f * u * u * (-2.f * cos_t) * ct0;
            for (int k = 0; k < 3; k++) {
                gdn[k] -= g_c * rv[k];
                grv[k] -= g_c * dn[k];
            }
        }
    }
    if (GRAD && g_ct0 != 0.f && xr > -1.f && xr < 1.f && ct0 > 1.0e-6f) {
        const float g_x = -g_ct0 * x / ct0;
        for (int k = 0; k < 3; k++) {
            gdn[k] += g_x * rv2[k];
            grv2[k] += g_x * dn[k];
        }
    }
    return rdon;
}

// Per-pair directional factors (forward).
struct Dir {
    float racc, rdon, Hramp;
};
__device__ __forceinline__ Dir dir_of(const float rv[3], const float rv2[3], int rexp, int index, int hb,
                                      const float dn[3], int closest, const float *rvH) {
    Dir o{1.f, 1.f, 1.f};
    const float c = -(dn[0] * rv[0] + dn[1] * rv[1] + dn[2] * rv[2]);
    if (hb == AG_HB_D1) {
        float dc;
        o.racc = racc_of(c, rexp, dc);
        if (c > 0.f && index != closest && closest >= 0) {
            const float ct = rvH[0] * rv[0] + rvH[1] * rv[1] + rvH[2] * rv[2];
            o.Hramp = hramp_value(fminf(fmaxf(ct, -1.f), 1.f));
        }
    } else if (hb == AG_HB_A1) {
        o.rdon = c > 0.f ? c * c : 0.f;
    } else if (hb == AG_HB_A2) {
        float g3[3] = {0, 0, 0};
        o.rdon = a2_rdon<false>(dn, rv, rv2, 0.f, g3, g3, g3);
    }
    return o;
}

// ---------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------

constexpr int kCube = 4;                 // edge of a workgroup's cube of points
constexpr int kCubeCap = 1024;           // atoms in the workgroup's list
constexpr int kCubeHCap = 256;           // donor H in its list

// A workgroup's cube of points: its corner, this lane's point and the cells
// around its box (points past the grid's end are clamped onto the last one).
struct Cube {
    int ix, iy, iz;          // this lane's point
    bool inside;
    float c[3];              // its position
    float lo[3], hi[3];      // the cube's box
    int clo[3], chi[3];      // cells overlapping the box grown by 8 A
};
__device__ __forceinline__ Cube cube_of(const AParams &p, int block) {
    Cube q;
    const int nx = (p.n1[0] + kCube - 1) / kCube, ny = (p.n1[1] + kCube - 1) / kCube;
    const int b[3] = {block % nx, (block / nx) % ny, block / (nx * ny)};
    const int lane = threadIdx.x & 63;
    const int i[3] = {kCube * b[0] + (lane & 3), kCube * b[1] + ((lane >> 2) & 3), kCube * b[2] + (lane >> 4)};
    q.inside = true;
    int j[3];
    for (int d = 0; d < 3; d++) {
        q.inside = q.inside && i[d] < p.n1[d];
        j[d] = min(i[d], p.n1[d] - 1);
        q.c[d] = (float)(j[d] - p.ne[d]) * p.h;
        q.lo[d] = (float)(kCube * b[d] - p.ne[d]) * p.h;
        q.hi[d] = (float)(min(kCube * b[d] + kCube, p.n1[d]) - 1 - p.ne[d]) * p.h;
        // the margin keeps FP32 rounding of an atom's cell from losing it
        q.clo[d] = max(0, __builtin_amdgcn_readfirstlane((int)floorf((q.lo[d] - 8.01f - p.corg[d]) / kCellA)));
        q.chi[d] = min(p.nc[d] - 1, __builtin_amdgcn_readfirstlane((int)floorf((q.hi[d] + 8.01f - p.corg[d]) / kCellA)));
    }
    q.ix = j[0];
    q.iy = j[1];
    q.iz = j[2];
    return q;
}

// LDS of the staging below.
struct CubeStage {
    int off[kAT + 1];        // first flat index of each cell row
    int first[kAT];          // its first slot
    int wave_tot[kAT / 64];
};

// Walks the atoms of the cube's cells (rows of cells along x are contiguous
// in the atom array) a tile of kAT at a time, in cell order: fn(slot, near)
// is called by every lane, near false where the lane has no atom or its atom
// is past 8 A of the cube's box.  fn may synchronise the workgroup.
template <typename F>
__device__ __forceinline__ void cube_atoms(const AParams &p, const Cube &q, CubeStage &st, F &&fn) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ny = q.chi[1] - q.clo[1] + 1, nz = q.chi[2] - q.clo[2] + 1;
    const int nrows = (q.chi[0] >= q.clo[0] && ny > 0 && nz > 0) ? ny * nz : 0;
    for (int r0 = 0; r0 < nrows; r0 += kAT) {
        int s0 = 0, n = 0;
        if (r0 + tid < nrows) {
            const int row = p.nc[0] * (q.clo[1] + (r0 + tid) % ny + p.nc[1] * (q.clo[2] + (r0 + tid) / ny));
            s0 = p.cell_start[row + q.clo[0]];
            n = p.cell_start[row + q.chi[0] + 1] - s0;
        }
        int x = n;   // inclusive scan: within the wave, then across waves
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o);
            if (lane >= o) x += y;
        }
        __syncthreads();   // the last tile's readers are done
        if (lane == 63) st.wave_tot[wave] = x;
        __syncthreads();
        int before = 0, total = 0;
        for (int w = 0; w < kAT / 64; w++) {
            before += w < wave ? st.wave_tot[w] : 0;
            total += st.wave_tot[w];
        }
        total = __builtin_amdgcn_readfirstlane(total);
        st.off[tid] = before + x - n;
        st.first[tid] = s0;
        if (tid == 0) st.off[kAT] = total;
        __syncthreads();
        for (int j0 = 0; j0 < total; j0 += kAT) {
            const int j = j0 + tid;
            int slot = 0;
            bool near = false;
            if (j < total) {
                int lo = 0, hi = kAT;   // the last row with off <= j
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (st.off[mid] <= j) lo = mid;
                    else hi = mid;
                }
                slot = st.first[lo] + j - st.off[lo];
                const AAtom &a = p.atoms[slot];
                const float ex = fmaxf(fmaxf(q.lo[0] - a.x, a.x - q.hi[0]), 0.f),
                            ey = fmaxf(fmaxf(q.lo[1] - a.y, a.y - q.hi[1]), 0.f),
                            ez = fmaxf(fmaxf(q.lo[2] - a.z, a.z - q.hi[2]), 0.f);
                near = ex * ex + ey * ey + ez * ez < kCut2 * 1.0001f;
            }
            fn(slot, near);
        }
    }
}

// Appends the slots of the flagged lanes to list, in lane order; the count in
// n, the same in every lane, goes up by theirs.  wave_tot holds one int per
// wave.  The caller keeps kAT free places.
__device__ __forceinline__ void append(bool flag, int slot, int *list, int &n, int *wave_tot) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long m = __ballot(flag);
    __syncthreads();
    if (lane == 0) wave_tot[wave] = __popcll(m);
    __syncthreads();
    int at = n + __popcll(m & ((1ull << lane) - 1));
    for (int w = 0; w < kAT / 64; w++) {
        at += w < wave ? wave_tot[w] : 0;
        n += wave_tot[w];
    }
    n = __builtin_amdgcn_readfirstlane(n);
    if (flag) list[at] = slot;
}

// Each point's closest donor H within 8 A (the lowest index of equals), or
// -1: the four waves take every fourth H of the cube's list, and the winners
// meet in LDS.  is_h picks the atoms; every wave returns the point's answer.
__device__ __forceinline__ int cube_closest_h(const AParams &p, const Cube &q, CubeStage &st, int *hlist,
                                              float (*hr2)[64], int (*hix)[64]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float best = 1e30f;
    int bidx = 0x7fffffff, n = 0;
    const auto scan = [&] {
        __syncthreads();
        for (int j = wave; j < n; j += kAT / 64) {
            const int slot = __builtin_amdgcn_readfirstlane(hlist[j]);
            const AN_CONST AAtom &a = ((const AN_CONST AAtom *)p.atoms)[slot];
            const float dx = a.x - q.c[0], dy = a.y - q.c[1], dz = a.z - q.c[2];
            const float r2 = dx * dx + dy * dy + dz * dz;
            const int i = a.index;
            if (r2 < best || (r2 == best && i < bidx)) {
                best = r2;
                bidx = i;
            }
        }
        n = 0;
    };
    cube_atoms(p, q, st, [&](int slot, bool near) {
        if (n > kCubeHCap - kAT) scan();   // uniform
        const int hb = near ? (p.atoms[slot].meta >> 8) & 0xff : 0;
        append(hb == AG_HB_DS || hb == AG_HB_D1, slot, hlist, n, st.wave_tot);
    });
    scan();
    hr2[wave][lane] = best;
    hix[wave][lane] = bidx;
    __syncthreads();
    for (int w = 0; w < kAT / 64; w++) {
        const float r2 = hr2[w][lane];
        const int i = hix[w][lane];
        if (r2 < best || (r2 == best && i < bidx)) {
            best = r2;
            bidx = i;
        }
    }
    return best < kCut2 ? bidx : -1;
}

// The capped energy of map k's pair with an atom of a type, the type (nt, its
// form word) uniform.
__device__ __forceinline__ float pair_energy(const AN_CONST ANearType &nt, int k, unsigned form, float r, float w) {
    // s = r + w left of the well, r* within w of it, r - w right of it
    const float off = __builtin_amdgcn_fmed3f(r - nt.pair[k].rstar, -w, w);
    const float rho = nt.pair[k].R * __builtin_amdgcn_rcpf(r - off);
    const float rho2 = rho * rho, rho4 = rho2 * rho2;
    float pa = rho4 * rho4 * rho4, pb;
    const unsigned f2 = (form >> (2 * k)) & 3;
    if (f2 == 0) {
        pb = rho4 * rho2;
    } else if (f2 == 1) {
        pb = rho4 * rho4 * rho2;
    } else {
        pa = pb = 1.f;
        const int ea = nt.a[k], eb = nt.b[k];
#pragma clang loop unroll(disable)
        for (int i = 0; i < max(ea, eb); i++) {
            pa *= i < ea ? rho : 1.f;
            pb *= i < eb ? rho : 1.f;
        }
    }
    return fminf(__builtin_fmaf(nt.pair[k].c1, pa, -(nt.pair[k].c2 * pb)), kClamp);
}

__device__ __forceinline__ AAtom load_atom(const AN_CONST AAtom *atoms, int slot) {
    const AN_CONST AAtom &s = atoms[slot];
    AAtom a;
    a.x = s.x;
    a.y = s.y;
    a.z = s.z;
    a.q = s.q;
    a.vol = s.vol;
    a.solpar = s.solpar;
    a.meta = s.meta;
    a.index = s.index;
    for (int k = 0; k < 3; k++) {
        a.rv[k] = s.rv[k];
        a.rv2[k] = s.rv2[k];
    }
    return a;
}

// One workgroup per cube of 4 x 4 x 4 points; a lane holds one point, the same
// one in each of the four waves, and the waves take every fourth atom of the
// cube's list (up to kCubeCap at a time), then add up through LDS in wave
// order.  An atom is the same for a whole wave, so its record, its pair
// parameters and its H-bond case come through scalar loads and its branches
// are scalar.  Bound by the vector unit: about 130 operations per (atom, point)
// with five maps, of which the pair potentials take 16 each.  One lane per
// point walking its own cells, with each lane's records and parameters in vector
// registers, measured 3.42 ms (5,000 atoms at protein density, 65^3 points, 5
// affinity maps), now 0.35 ms.
template <int NA>
__global__ void __launch_bounds__(kAT) k_an_near(AParams p) {
    __shared__ CubeStage st;
    __shared__ int list[kCubeCap], hlist[kCubeHCap];
    __shared__ float hr2[kAT / 64][64];
    __shared__ int hix[kAT / 64][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Cube q = cube_of(p, blockIdx.x);
    const int ch = cube_closest_h(p, q, st, hlist, hr2, hix);
    float rvH[3] = {0.f, 0.f, 0.f};
    if (ch >= 0)
        for (int k = 0; k < 3; k++) rvH[k] = p.rv_by_index[3 * ch + k];
    float acc[NA], hmin[NA], hmax[NA];
    int amin[NA], amax[NA];
#pragma unroll
    for (int k = 0; k < NA; k++) {
        acc[k] = 0.f;
        hmin[k] = 999999.f;
        hmax[k] = -999999.f;
        amin[k] = amax[k] = -1;
    }
    // the classes' case words, lane = class; read by readlane at the top of an
    // atom, where every lane is active
    const int case_word = p.case_word[min(lane, 6)];
    // desolvation: map k gains sp[k] sum(vol G) + volp[k] sum(solq G)
    float dv = 0.f, dq = 0.f;
    int n = 0;
    const auto process = [&] {
        __syncthreads();
        const AN_CONST AAtom *atoms = (const AN_CONST AAtom *)p.atoms;
        for (int j0 = wave; j0 < n; j0 += kAT) {
            // 64 of the wave's atoms at a time: their slots in one register,
            // picked by readlane; each record is loaded one atom ahead
            const int mine = list[min(j0 + lane * (kAT / 64), n - 1)];
            const int count = min(64, (n - j0 + kAT / 64 - 1) / (kAT / 64));
            AAtom a = load_atom(atoms, __builtin_amdgcn_readlane(mine, 0));
            for (int jj = 0; jj < count; jj++) {
                const AAtom at = a;
                int next = __builtin_amdgcn_readlane(mine, min(jj + 1, count - 1));
                // the next record's loads issue once this one's have arrived
                asm volatile("" : "+s"(next) : "s"(at.meta), "s"(at.x), "s"(at.index));
                a = load_atom(atoms, next);
                const int type = at.meta & 0xff, hb = (at.meta >> 8) & 0xff;
                const unsigned cases = (unsigned)__builtin_amdgcn_readlane(case_word, hb);
                const float d[3] = {at.x - q.c[0], at.y - q.c[1], at.z - q.c[2]};
                const float r2 = __builtin_fmaf(d[0], d[0], __builtin_fmaf(d[1], d[1], d[2] * d[2]));
                if (!(r2 < kCut2)) continue;
                const AN_CONST ANearType &nt = ((const AN_CONST ANearType *)p.near_pairs)[type];
                const float r2c = fmaxf(r2, 1.0e-12f);
                const float ir = __builtin_amdgcn_rsqf(r2c);   // hardware rsq, exp2 and rcp, about 1 ulp
                const float r = r2c * ir;
                float dS;
                const float S = switch_s(r, dS);
                const float G = p.w_desolv * __builtin_amdgcn_exp2f(r2 * (-kInv2Sig2 * 1.44269504088896341f)) * S;
                dv = __builtin_fmaf(at.vol, G, dv);
                dq = __builtin_fmaf(at.solpar + p.qasp * fabsf(at.q), G, dq);
                Dir dr{1.f, 1.f, 1.f};
                if (hb == AG_HB_D1 || hb == AG_HB_A1 || hb == AG_HB_A2) {
                    const float dn[3] = {d[0] * ir, d[1] * ir, d[2] * ir};
                    dr = dir_of(at.rv, at.rv2, (at.meta >> 16) & 0xff, at.index, hb, dn, ch, rvH);
                }
                const unsigned form = (unsigned)nt.form;
#pragma clang loop unroll(full)
                for (int k = 0; k < NA; k++) {
                    if (k >= p.naff) continue;
                    const float E = pair_energy(nt, k, form, r, p.w_smooth) * S;
                    const unsigned cs = (cases >> (2 * k)) & 3;
                    if (cs == CASE_PLAIN) {
                        acc[k] += E;
                    } else {
                        const float rsph = __builtin_amdgcn_fmed3f(E * 0.01f, 0.f, 1.f);
                        const float f = cs == CASE_MM_RDON ? dr.rdon : dr.racc;
                        const float v = E * __builtin_fmaf(1.f - f, rsph, f);
                        if (cs == CASE_ACC) {
                            acc[k] = __builtin_fmaf(v, dr.Hramp, acc[k]);
                        } else {
                            if (v < hmin[k]) { hmin[k] = v; amin[k] = at.index; }
                            if (v > hmax[k]) { hmax[k] = v; amax[k] = at.index; }
                        }
                    }
                }
            }
        }
        n = 0;
        __syncthreads();
    };
    cube_atoms(p, q, st, [&](int slot, bool near) {
        if (n > kCubeCap - kAT) process();   // uniform
        append(near, slot, list, n, st.wave_tot);
    });
    process();
    // waves 1 to 3 hand over one after the other, so that ties between equal
    // terms go to the earlier wave
    __shared__ float fx[3 * NA + 2][64];
    __shared__ int ix[2 * NA][64];
    for (int w = 1; w < kAT / 64; w++) {
        if (wave == w) {
#pragma unroll
            for (int k = 0; k < NA; k++) {
                fx[3 * k][lane] = acc[k];
                fx[3 * k + 1][lane] = hmin[k];
                fx[3 * k + 2][lane] = hmax[k];
                ix[2 * k][lane] = amin[k];
                ix[2 * k + 1][lane] = amax[k];
            }
            fx[3 * NA][lane] = dv;
            fx[3 * NA + 1][lane] = dq;
        }
        __syncthreads();
        if (wave == 0) {
#pragma unroll
            for (int k = 0; k < NA; k++) {
                acc[k] += fx[3 * k][lane];
                if (fx[3 * k + 1][lane] < hmin[k]) { hmin[k] = fx[3 * k + 1][lane]; amin[k] = ix[2 * k][lane]; }
                if (fx[3 * k + 2][lane] > hmax[k]) { hmax[k] = fx[3 * k + 2][lane]; amax[k] = ix[2 * k + 1][lane]; }
            }
            dv += fx[3 * NA][lane];
            dq += fx[3 * NA + 1][lane];
        }
        __syncthreads();
    }
    if (wave != 0 || !q.inside) return;
    const long long pt = (long long)q.ix + (long long)p.n1[0] * ((long long)q.iy + (long long)p.n1[1] * q.iz);
    // assemble: a desolvation-only map belongs to exactly one affinity map
    // (separate_desolvation_maps), so slot writes do not collide
#pragma unroll
    for (int k = 0; k < NA; k++) {
        if (k >= p.naff) continue;
        float v = acc[k];
        if (amin[k] >= 0) v += hmin[k] + fmaxf(hmax[k], 0.f);
        const float des = __builtin_fmaf(p.sp[k], dv, p.volp[k] * dq);
        if (p.des_slot[k] == p.aff_slot[k]) {
            p.maps[(long long)p.aff_slot[k] * p.P + pt] = v + des;
        } else {
            p.maps[(long long)p.aff_slot[k] * p.P + pt] = v;
            p.maps[(long long)p.des_slot[k] * p.P + pt] = des;
        }
        p.amin[(long long)k * p.P + pt] = amin[k];
        p.amax[(long long)k * p.P + pt] = (amin[k] >= 0 && hmax[k] > 0.f) ? amax[k] : -1;
    }
    if (p.d_slot >= 0) p.maps[(long long)p.d_slot * p.P + pt] = p.qasp * dv;
    p.closest_h[pt] = ch;
    for (int k = 0; k < p.n_cov; k++) {
        const double dx = p.cov_pos[0] - (double)(q.ix - p.ne[0]) * (double)p.h;
        const double dy = p.cov_pos[1] - (double)(q.iy - p.ne[1]) * (double)p.h;
        const double dz = p.cov_pos[2] - (double)(q.iz - p.ne[2]) * (double)p.h;
        double rc = sqrt(dx * dx + dy * dy + dz * dz) / p.cov_hw;
        if (rc < 1.0e-6) rc = 1.0e-6;
        p.maps[(long long)p.cov_slot[k] * p.P + pt] = (float)(p.cov_barrier * (1. - exp(-0.69314718055994530942 * rc * rc)));
    }
}

// Orders a wave's own LDS accesses: its lanes see what the others wrote before.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

struct EParams {
    int n1[3], ne[3];
    float h;
    long long P;
    const float4 *atoms;      // (x, y, z, q * coeff_estat)
    int n_atoms;
    int dddiel;
    float inv_diel;           // 332 / diel for a constant dielectric
    float *emap;
    // forward in runs (k_an_e, k_an_esum)
    const float4 *fatoms;     // (cs x, cs y, cs z, w): coordinates scaled by cs, see k_an_e
    float sc;                 // cs * spacing
    float rcap;               // 2 / cs
    int echunk, nechunks;     // atoms per chunk, chunks
    float *epart;             // [nechunks][P] partial sums
    // forward with boxes (k_an_ebox, k_an_epatch): patches of K x 8 x 8 points, boxes
    // of 2 x 2 of them
    int npatch[3], nbox[3];
    int box_parts;            // workgroups sharing a box's atoms; 0: no boxes
    int split;                // workgroups sharing a patch's atoms
    float box_r2;             // squared distance (scaled) past which a box takes an atom
    double *box_sums;         // [box][part][512]
    unsigned long long *box_mask;   // [box][groups of 64 atoms]: the atoms it takes
    // adjoint
    const float *ge;          // cotangent of the e map
    float4 *partial;          // [chunks][n_atoms]: dx, dy, dz, dq
    int nchunks;
};

struct __align__(16) EAtom {
    float x, y, z, w;
};

template <int K>
struct ERun {
    static constexpr float mid = 0.5f * (K - 1);
    // (k - mid)^2 and the factor K - 1 - 2k of u * spacing
    static __device__ __forceinline__ constexpr float c2(int k) { return ((float)k - mid) * ((float)k - mid); }
    static __device__ __forceinline__ constexpr float m(int k) { return (float)(K - 1 - 2 * k); }
};

// An atom's share of the e map at K points along x.
template <int K, bool DD>
__device__ __forceinline__ void e_pair(const EAtom &at, float py, float pz, float cx, float sc, float s2, float bias,
                                       float rcap, float *part) {
    const float dy = at.y - py, dz = at.z - pz;
    const float dyz2 = __builtin_fmaf(dy, dy, __builtin_fmaf(dz, dz, bias));
    const float u = at.x - cx;
    const float U = __builtin_fmaf(u, u, dyz2);
    const float us = u * sc;
#pragma unroll
    for (int k = 0; k < K; k++) {
        const float rb2 = __builtin_fmaf(us, ERun<K>::m(k), __builtin_fmaf(s2, ERun<K>::c2(k), U));
        const float rs = __builtin_amdgcn_rsqf(rb2);
        const float h = fminf(rs, rcap);
        if (DD) {
            const float e2 = __builtin_amdgcn_exp2f(-(rb2 * rs));
            const float den = __builtin_fmaf(kMsK, e2, 1.f);
            const float g = den * __builtin_amdgcn_rcpf(__builtin_fmaf(kMsA, den, kMsB));
            part[k] = __builtin_fmaf(at.w, h * g, part[k]);
        } else {
            part[k] = __builtin_fmaf(at.w, h, part[k]);
        }
    }
}

template <int K, bool DD>
__global__ void __launch_bounds__(64) k_an_e(EParams p) {
    const int run = blockIdx.x * 64 + threadIdx.x;
    const int rpr = (p.n1[0] + K - 1) / K;
    const int nruns = rpr * p.n1[1] * p.n1[2];
    const bool active = run < nruns;
    const int rr = active ? run : nruns - 1;   // an idle lane computes a real run and stores nothing
    const int row = rr / rpr;
    const int ix0 = (rr - row * rpr) * K;
    const int iy = row % p.n1[1], iz = row / p.n1[1];
    const float sc = p.sc;
    const float py = (float)(iy - p.ne[1]) * sc, pz = (float)(iz - p.ne[2]) * sc;
    const float cx = ((float)(ix0 - p.ne[0]) + ERun<K>::mid) * sc;
    const float s2 = sc * sc;
    const float bias = fmaxf(1.0e-12f, ERun<K>::mid * ERun<K>::mid * s2 * 0x1p-19f);
    const int a0 = blockIdx.y * p.echunk;
    const int a1 = min(a0 + p.echunk, p.n_atoms);
    const float rcap = p.rcap;   // 2 / cs
    float part[K];
#pragma unroll
    for (int k = 0; k < K; k++) part[k] = 0.f;
    // atoms are read-only here: scalar loads through the constant address space
    const __attribute__((address_space(4))) EAtom *atoms = (const __attribute__((address_space(4))) EAtom *)p.fatoms;
    auto ld = [&](int i) {
        const __attribute__((address_space(4))) EAtom &q = atoms[i];
        return EAtom{q.x, q.y, q.z, q.w};
    };
    if (a0 < a1) {
        EAtom nxt = ld(a0);
        for (int a = a0; a < a1; a++) {
            const EAtom at = nxt;
            nxt = ld(min(a + 1, a1 - 1));
            e_pair<K, DD>(at, py, pz, cx, sc, s2, bias, rcap, part);
        }
    }
    if (active) {
        float *out = p.epart + (long long)blockIdx.y * p.P + ix0 + (long long)p.n1[0] * (iy + (long long)p.n1[1] * iz);
#pragma unroll
        for (int k = 0; k < K; k++)
            if (ix0 + k < p.n1[0]) out[k] = part[k];
    }
}

// The e map of larger receptors.  1 / (eps(r) r) is smooth away from the atom, so
// a box of 2 x 2 patches (about 16 x 16 x 16 points) takes the atoms beyond
// box_r2 at 8 x 8 x 8 Chebyshev nodes, and its points interpolate; only the
// atoms around it go pair by pair.  The worst place for an atom is ahead of a
// face, the pole of 1/r beside the two axes along it; evaluated there, eight nodes
// leave 1e-7 of the term on each axis at 4.5 half-edges (2e-7 at 4, 4e-6 at 2.6),
// 8e-8 at 3.5 in a constant dielectric (8e-7 at 2.6): an FP32 term's own roundings.
// Bound by the pairs' and nodes' transcendentals (rsq, exp2, rcp), as the all-pairs
// kernel: 5,000 atoms, 65^3 points 595 -> 395 us (boxes 149, patches 242, sum 4).
constexpr int kEBoxN = 8, kEBoxNodes = kEBoxN * kEBoxN * kEBoxN, kEPatch = 8, kEWaves = 4;
constexpr int kEPart = 32;               // terms of an FP32 partial sum (at least; 95 at most)
__host__ __device__ __forceinline__ constexpr double e_node(int i) {   // Chebyshev nodes, increasing
    constexpr double c[4] = {0.98078528040323044913, 0.83146961230254523708, 0.55557023301960222474,
                             0.19509032201612826785};
    return i < 4 ? -c[i] : c[7 - i];
}
__host__ __device__ __forceinline__ constexpr double e_node_den(int i) {
    double d = 1.0;
    for (int m = 0; m < kEBoxN; m++)
        if (m != i) d *= e_node(i) - e_node(m);
    return d;
}
// The eight Lagrange weights at t.
__device__ __forceinline__ constexpr void e_weights(double t, double w[kEBoxN]) {
    double before[kEBoxN] = {1.0}, after = 1.0;
    for (int m = 1; m < kEBoxN; m++) before[m] = before[m - 1] * (t - e_node(m - 1));
    for (int m = kEBoxN - 1; m >= 0; m--) {
        w[m] = before[m] * after * (1.0 / e_node_den(m));
        after *= t - e_node(m);
    }
}

// The sums at a box's nodes of one part of the atoms beyond it, and which atoms
// those are: a lane has the eight x-nodes of one (y, z) node.
template <int K, bool DD>
__global__ void __launch_bounds__(64 * kEWaves) k_an_ebox(EParams p) {
    __shared__ double XD[(kEWaves - 1) * kEBoxNodes];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const int part = blockIdx.x % p.box_parts, box = blockIdx.x / p.box_parts;
    const int bx = box % p.nbox[0], by = box / p.nbox[0] % p.nbox[1], bz = box / p.nbox[0] / p.nbox[1];
    const float sc = p.sc;
    const float hx = ERun<K>::mid * sc, hr = ((float)kEPatch - 0.5f) * sc;
    const float mx = ((float)(bx * K - p.ne[0]) + ERun<K>::mid) * sc;
    const float my = ((float)(by * 2 * kEPatch - p.ne[1]) + (float)kEPatch - 0.5f) * sc;
    const float mz = ((float)(bz * 2 * kEPatch - p.ne[2]) + (float)kEPatch - 0.5f) * sc;
    float cy = 0.f, cz = 0.f;
#pragma unroll
    for (int i = 0; i < kEBoxN; i++) {
        cy = (lane & 7) == i ? my + hr * (float)e_node(i) : cy;
        cz = lane >> 3 == i ? mz + hr * (float)e_node(i) : cz;
    }
    double sum[kEBoxN];
    float acc[kEBoxN];
#pragma unroll
    for (int j = 0; j < kEBoxN; j++) {
        sum[j] = 0.;
        acc[j] = 0.f;
    }
    const int groups = (p.n_atoms + 63) / 64;
    unsigned long long *const mask = p.box_mask + (size_t)box * groups;
    const AN_CONST EAtom *atoms = (const AN_CONST EAtom *)p.fatoms;   // scalar loads
    int n_acc = 0;
    for (int a0 = 64 * (part * kEWaves + wave); a0 < p.n_atoms; a0 += 64 * kEWaves * p.box_parts) {
        const float4 v = p.fatoms[min(a0 + lane, p.n_atoms - 1)];
        const float ex = fmaxf(fabsf(v.x - mx) - hx, 0.f), ey = fmaxf(fabsf(v.y - my) - hr, 0.f),
                    ez = fmaxf(fabsf(v.z - mz) - hr, 0.f);
        unsigned long long set = __ballot(a0 + lane < p.n_atoms &&
                                          __builtin_fmaf(ex, ex, __builtin_fmaf(ey, ey, ez * ez)) >= p.box_r2);
        if (lane == 0) mask[a0 / 64] = set;
        n_acc += __popcll(set);
        while (set) {
            const AN_CONST EAtom &at = atoms[a0 + __builtin_ctzll(set)];
            set &= set - 1;
            const float dy = at.y - cy, dz = at.z - cz, u = at.x - mx, w = at.w;
            const float U = __builtin_fmaf(u, u, __builtin_fmaf(dy, dy, dz * dz)), u2 = u + u;
#pragma unroll
            for (int j = 0; j < kEBoxN; j++) {
                const float d = hx * (float)e_node(j);
                const float rb2 = __builtin_fmaf(-u2, d, __builtin_fmaf(d, d, U));
                const float rs = __builtin_amdgcn_rsqf(rb2);
                if (DD) {
                    const float e2 = __builtin_amdgcn_exp2f(-(rb2 * rs));
                    const float den = __builtin_fmaf(kMsK, e2, 1.f);
                    const float g = den * __builtin_amdgcn_rcpf(__builtin_fmaf(kMsA, den, kMsB));
                    acc[j] = __builtin_fmaf(w, rs * g, acc[j]);
                } else {
                    acc[j] = __builtin_fmaf(w, rs, acc[j]);
                }
            }
        }
        if (n_acc >= kEPart) {
            n_acc = 0;
#pragma unroll
            for (int j = 0; j < kEBoxN; j++) {
                sum[j] += (double)acc[j];
                acc[j] = 0.f;
            }
        }
    }
#pragma unroll
    for (int j = 0; j < kEBoxN; j++) sum[j] += (double)acc[j];
    if (wave > 0) {
#pragma unroll
        for (int j = 0; j < kEBoxN; j++) XD[((wave - 1) * kEBoxN + j) * 64 + lane] = sum[j];
    }
    __syncthreads();
    if (wave == 0) {
        double *const out = p.box_sums + (size_t)blockIdx.x * kEBoxNodes;
#pragma unroll
        for (int j = 0; j < kEBoxN; j++) {
            for (int q = 0; q < kEWaves - 1; q++) sum[j] += XD[(q * kEBoxN + j) * 64 + lane];
            out[j * 64 + lane] = sum[j];
        }
    }
}

// One patch, and one of its parts of the atoms its box leaves, a run of K
// points per lane; each wave also interpolates a quarter of the box's nodes (in
// the first part).  The waves' sums meet in LDS, in order.
template <int K, bool DD>
__global__ void __launch_bounds__(64 * kEWaves) k_an_epatch(EParams p) {
    __shared__ double XD[(kEWaves - 1) * K * 64];
    __shared__ double V[kEWaves][kEBoxNodes / kEWaves];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const int part = blockIdx.x % p.split, patch = blockIdx.x / p.split;
    const int px = patch % p.npatch[0], pyi = patch / p.npatch[0] % p.npatch[1], pzi = patch / p.npatch[0] / p.npatch[1];
    const int box = px + p.nbox[0] * (pyi / 2 + p.nbox[1] * (pzi / 2));
    const int ix0 = px * K, iy = pyi * kEPatch + lane % kEPatch, iz = pzi * kEPatch + lane / kEPatch;
    const bool active = iy < p.n1[1] && iz < p.n1[2];
    const float sc = p.sc;
    const float py = (float)(iy - p.ne[1]) * sc, pz = (float)(iz - p.ne[2]) * sc;
    const float cx = ((float)(ix0 - p.ne[0]) + ERun<K>::mid) * sc;
    const float s2 = sc * sc, bias = fmaxf(1.0e-12f, ERun<K>::mid * ERun<K>::mid * s2 * 0x1p-19f), rcap = p.rcap;
    const int groups = (p.n_atoms + 63) / 64;
    const AN_CONST unsigned long long *mask = (const AN_CONST unsigned long long *)p.box_mask + (size_t)box * groups;
    const AN_CONST EAtom *atoms = (const AN_CONST EAtom *)p.fatoms;   // scalar loads
    double f[K];
    float sum[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        f[k] = 0.;
        sum[k] = 0.f;
    }
    int n_sum = 0;   // atoms in sum[] since it went to f[]
    for (int a0 = 64 * (part * kEWaves + wave); a0 < p.n_atoms; a0 += 64 * kEWaves * p.split) {
        const int nb = min(64, p.n_atoms - a0);
        unsigned long long set = (nb == 64 ? ~0ull : (1ull << nb) - 1) & ~mask[a0 / 64];
        if (!set) continue;
        const auto ld = [&](int i) {
            const AN_CONST EAtom &q = atoms[a0 + i];
            return EAtom{q.x, q.y, q.z, q.w};
        };
        EAtom nxt = ld(__builtin_ctzll(set));
        n_sum += __popcll(set);
        while (set) {
            const EAtom at = nxt;
            set &= set - 1;
            if (set) nxt = ld(__builtin_ctzll(set));
            e_pair<K, DD>(at, py, pz, cx, sc, s2, bias, rcap, sum);
        }
        if (n_sum >= kEPart) {
            n_sum = 0;
#pragma unroll
            for (int k = 0; k < K; k++) {
                f[k] += (double)sum[k];
                sum[k] = 0.f;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < K; k++) f[k] += (double)sum[k];
    if (part == 0) {
        constexpr int kOwn = 64 / kEWaves;   // (y, z) nodes of a wave: two rows of eight
        for (int t = lane; t < kOwn * kEBoxN; t += 64) {
            double v = 0.;
            for (int q = 0; q < p.box_parts; q++)
                v += p.box_sums[((size_t)box * p.box_parts + q) * kEBoxNodes + t / kOwn * 64 + wave * kOwn + t % kOwn];
            V[wave][t % kOwn * kEBoxN + t / kOwn] = v;
        }
        wave_sync();
        constexpr double half = kEPatch - 0.5;
        double wy[kEBoxN], wz[kEBoxN];
        e_weights(((double)((pyi & 1) * kEPatch + lane % kEPatch) - half) / half, wy);
        e_weights(((double)((pzi & 1) * kEPatch + lane / kEPatch) - half) / half, wz);
        double wz0 = wz[0], wz1 = wz[1];
#pragma unroll
        for (int q = 1; q < kEWaves; q++) {
            wz0 = wave == q ? wz[2 * q] : wz0;
            wz1 = wave == q ? wz[2 * q + 1] : wz1;
        }
        double g[kEBoxN];
#pragma unroll
        for (int j = 0; j < kEBoxN; j++) g[j] = 0.;
#pragma unroll
        for (int l = 0; l < kOwn; l++) {
            const double w = wy[l & 7] * (l < 8 ? wz0 : wz1);
#pragma unroll
            for (int j = 0; j < kEBoxN; j++) g[j] = __builtin_fma(w, V[wave][l * kEBoxN + j], g[j]);
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            double wx[kEBoxN];
            e_weights(((double)k - 0.5 * (K - 1)) / (0.5 * (K - 1)), wx);
#pragma unroll
            for (int j = 0; j < kEBoxN; j++) f[k] = __builtin_fma(wx[j], g[j], f[k]);
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int k = 0; k < K; k++) XD[((wave - 1) * K + k) * 64 + lane] = f[k];
    }
    __syncthreads();
    if (wave == 0 && active) {
        float *const out = p.epart + (long long)part * p.P + ix0 + (long long)p.n1[0] * (iy + (long long)p.n1[1] * iz);
#pragma unroll
        for (int k = 0; k < K; k++) {
            for (int q = 0; q < kEWaves - 1; q++) f[k] += XD[(q * K + k) * 64 + lane];
            if (ix0 + k < p.n1[0]) out[k] = (float)f[k];
        }
    }
}

// The e map: per point the chunks' partial sums in chunk order, Kahan-compensated.
__global__ void k_an_esum(const float *epart, int nchunk, long long P, float *emap) {
    const long long pt = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (pt >= P) return;
    float s = 0.f, c = 0.f;
    for (int j = 0; j < nchunk; j++) {
        const float y = epart[(long long)j * P + pt] - c;
        const float t = s + y;
        c = (t - s) - y;
        s = t;
    }
    emap[pt] = s;
}

// ---------------------------------------------------------------------------
// adjoint
// ---------------------------------------------------------------------------

// Per point: the cotangent of the closest H's bond vector through the Hramp
// factor of every other D1 atom within 8 A.  Cubes and waves as in k_an_near; a
// cube without a point to do leaves zeros.  (One lane per point with its own
// cells: 288 us, now 31 us at the shape above, 184 beside k_an_atom on the other
// stream; 235 and 14 us on 41^3 points.)
__global__ void __launch_bounds__(kAT) k_an_vh(AParams p) {
    __shared__ CubeStage st;
    __shared__ int list[2 * kAT];
    __shared__ float fx[kAT / 64][3][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Cube q = cube_of(p, blockIdx.x);
    const long long pt = (long long)q.ix + (long long)p.n1[0] * ((long long)q.iy + (long long)p.n1[1] * q.iz);
    const int ch = p.closest_h[pt];
    const unsigned cases = (unsigned)p.case_word[AG_HB_D1];
    float g[kAMaxAff];
    bool any = false;
#pragma unroll
    for (int k = 0; k < kAMaxAff; k++) {
        g[k] = k < p.naff && ((cases >> (2 * k)) & 3) == CASE_ACC ? p.dmaps[(long long)p.aff_slot[k] * p.P + pt] : 0.f;
        any = any || g[k] != 0.f;
    }
    any = any && ch >= 0 && q.inside;
    float v[3] = {0.f, 0.f, 0.f};
    if (__ballot(any)) {   // the same in every wave
        float rvH[3] = {0.f, 0.f, 0.f};
        if (ch >= 0)
            for (int k = 0; k < 3; k++) rvH[k] = p.rv_by_index[3 * ch + k];
        int n = 0;
        const auto process = [&] {
            __syncthreads();
            for (int j = wave; j < n; j += kAT / 64) {
                const AAtom a = load_atom((const AN_CONST AAtom *)p.atoms, __builtin_amdgcn_readfirstlane(list[j]));
                if (!any || a.index == ch) continue;
                const float d[3] = {a.x - q.c[0], a.y - q.c[1], a.z - q.c[2]};
                const float r2 = __builtin_fmaf(d[0], d[0], __builtin_fmaf(d[1], d[1], d[2] * d[2]));
                if (!(r2 < kCut2)) continue;
                const float r2c = fmaxf(r2, 1.0e-12f);
                const float ir = __builtin_amdgcn_rsqf(r2c), r = r2c * ir;
                const float cth = -(d[0] * a.rv[0] + d[1] * a.rv[1] + d[2] * a.rv[2]) * ir;
                if (!(cth > 0.f)) continue;
                float dc, dct, dS;
                const float racc = racc_of(cth, (a.meta >> 16) & 0xff, dc);
                hramp_of(rvH[0] * a.rv[0] + rvH[1] * a.rv[1] + rvH[2] * a.rv[2], dct);
                if (dct == 0.f) continue;
                const float S = switch_s(r, dS);
                const AN_CONST ANearType &nt = ((const AN_CONST ANearType *)p.near_pairs)[a.meta & 0xff];
                const unsigned form = (unsigned)nt.form;
                float gH = 0.f;
#pragma clang loop unroll(full)
                for (int k = 0; k < kAMaxAff; k++) {
                    if (k >= p.naff || ((cases >> (2 * k)) & 3) != CASE_ACC) continue;
                    const float E = pair_energy(nt, k, form, r, p.w_smooth) * S;
                    const float rsph = fminf(fmaxf(E * 0.01f, 0.f), 1.f);
                    gH += g[k] != 0.f ? g[k] * E * (racc + (1.f - racc) * rsph) : 0.f;
                }
                for (int k = 0; k < 3; k++) v[k] += gH * dct * a.rv[k];
            }
            n = 0;
            __syncthreads();
        };
        cube_atoms(p, q, st, [&](int slot, bool near) {
            if (n > kAT) process();   // uniform
            append(near && ((p.atoms[slot].meta >> 8) & 0xff) == AG_HB_D1, slot, list, n, st.wave_tot);
        });
        process();
        for (int k = 0; k < 3; k++) fx[wave][k][lane] = v[k];
        __syncthreads();
        for (int k = 0; k < 3; k++) v[k] = ((fx[0][k][lane] + fx[1][k][lane]) + fx[2][k][lane]) + fx[3][k][lane];
    }
    if (wave == 0 && q.inside)
        for (int k = 0; k < 3; k++) p.vh[3 * pt + k] = v[k];
}

// Block reduction of n floats per lane (fixed order): lane 0 of the block
// gets the sums.
template <int NV>
__device__ __forceinline__ void block_sum(float (&v)[NV], float *red) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < NV; k++) {
        float x = v[k];
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
        v[k] = x;
    }
    __syncthreads();
    if (lane == 0)
        for (int k = 0; k < NV; k++) red[wave * NV + k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int k = 0; k < NV; k++) v[k] = red[k] + red[NV + k] + red[2 * NV + k] + red[3 * NV + k];
}

struct HsumParams {
    const int *closest_h;
    const float *vh;
    const int *list;         // points with a nonzero vh, in point order
    const int *count;        // their number (device)
    const int *h_atoms;      // donor H atom indices, one per workgroup
    float *out;              // [n][3]
};

__global__ void __launch_bounds__(kAT) k_an_hsum(HsumParams p) {
    __shared__ float red[4 * 3];
    const int h = p.h_atoms[blockIdx.x];
    const int n = *p.count;
    float v[3] = {0.f, 0.f, 0.f};
    for (int i = threadIdx.x; i < n; i += kAT) {
        const long long pt = p.list[i];
        if (p.closest_h[pt] == h)
            for (int k = 0; k < 3; k++) v[k] += p.vh[3 * pt + k];
    }
    block_sum<3>(v, red);
    if (threadIdx.x == 0)
        for (int k = 0; k < 3; k++) p.out[3 * blockIdx.x + k] = v[k];
}

// Per-atom outputs of k_an_atom: x(3) rv(3) rv2(3) q wdes, then R and eps
// per affinity map.
constexpr int kAtomOut = 11 + 2 * kAMaxAff;

// Bit rows: for each grid row along x, words of 64 points, a bit set where any
// cotangent the atom gather reads (affinity, desolvation and d slots) is
// nonzero.  Where all are zero a point adds exactly nothing to any atom's
// gradient, so k_an_atom skips it.  One wave per word.
__global__ void __launch_bounds__(kAT) k_an_gmask(AParams p, int words, unsigned long long *bits) {
    const long long w = (long long)blockIdx.x * (kAT / 64) + (threadIdx.x >> 6);
    const long long row = w / words;
    const int ix = (int)(w - row * words) * 64 + (threadIdx.x & 63);
    bool any = false;
    if (row < (long long)p.n1[1] * p.n1[2] && ix < p.n1[0]) {
        const long long pt = row * p.n1[0] + ix;
        any = p.d_slot >= 0 && p.dmaps[(long long)p.d_slot * p.P + pt] != 0.f;
        for (int k = 0; k < p.naff; k++)
            any = any || p.dmaps[(long long)p.aff_slot[k] * p.P + pt] != 0.f ||
                  p.dmaps[(long long)p.des_slot[k] * p.P + pt] != 0.f;
    }
    const unsigned long long m = __ballot(any);
    if ((threadIdx.x & 63) == 0 && row < (long long)p.n1[1] * p.n1[2]) bits[w] = m;
}

struct AtomAdjParams {
    AParams a;
    const AAtom *by_index;   // atoms by index
    const int *atom_list;    // atoms whose 8 A sphere meets the box, one per workgroup
    float *out;              // [n_list][kAtomOut]
    const unsigned long long *bits;   // k_an_gmask
    int words;               // 64-point words per grid row
};

// One workgroup per atom.  The rows of the box through its 8 A sphere are
// dealt to the lanes a word of 64 points at a time; a lane keeps the bits
// (k_an_gmask) of its word that lie within the sphere's chord.  Each wave packs
// its lanes' points into its own LDS list in lane order and works through it
// 64 at a time, every lane busy; no barrier until the waves' sums meet.
// The chord is a little wide: points past 8 A are dropped when they are looked at.
// Testing the sphere's cube point by point, with the workgroup's barriers,
// took most of the launch: 865 us (5,000 atoms, 65^3 points, 256 poses), now
// 450 us (490 with the other chain beside it).
template <int NA>
__global__ void __launch_bounds__(kAT) k_an_atom(AtomAdjParams q) {
    constexpr int kList = 512;   // a wave's list; one lane appends at most 64
    __shared__ float red[4 * kAtomOut];
    __shared__ int2 lists[kAT / 64][kList];
    const AParams &p = q.a;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int2 *const list = lists[wave];
    const int idx = __builtin_amdgcn_readfirstlane(q.atom_list[blockIdx.x]);
    const AAtom a = load_atom((const AN_CONST AAtom *)q.by_index, idx);
    const int type = a.meta & 0xff, hb = (a.meta >> 8) & 0xff, rexp = (a.meta >> 16) & 0xff;
    const AN_CONST APair *pairs = (const AN_CONST APair *)p.pairs + type;
    const unsigned cases = (unsigned)p.case_word[hb];
    // rows and words of the box around the atom
    int lo[3], hi[3];
    const float ac[3] = {a.x, a.y, a.z};
    for (int d = 0; d < 3; d++) {
        lo[d] = max(0, __builtin_amdgcn_readfirstlane((int)ceilf((ac[d] - 8.f) / p.h)) + p.ne[d]);
        hi[d] = min(p.n1[d] - 1, __builtin_amdgcn_readfirstlane((int)floorf((ac[d] + 8.f) / p.h)) + p.ne[d]);
    }
    const int w0 = lo[0] / 64, nw = hi[0] / 64 - w0 + 1, ny = hi[1] - lo[1] + 1, nz = hi[2] - lo[2] + 1;
    const int nitem = (hi[0] >= lo[0] && ny > 0 && nz > 0) ? nw * ny * nz : 0;
    float acc[kAtomOut];
#pragma unroll
    for (int k = 0; k < kAtomOut; k++) acc[k] = 0.f;
    const float solq = a.solpar + p.qasp * fabsf(a.q);
    const float sgnq = a.q > 0.f ? 1.f : (a.q < 0.f ? -1.f : 0.f);
    const auto point = [&](int2 e) {   // point index, iy | iz << 16
        const long long pt = e.x;
        const int iy = e.y & 0xffff, iz = e.y >> 16;
        const int ix = e.x - p.n1[0] * (iy + p.n1[1] * iz);
        const float c[3] = {(float)(ix - p.ne[0]) * p.h, (float)(iy - p.ne[1]) * p.h, (float)(iz - p.ne[2]) * p.h};
        const float d[3] = {a.x - c[0], a.y - c[1], a.z - c[2]};
        const float r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
        if (!(r2 < kCut2)) return;   // (a NaN cotangent there is not this atom's)
        const float r2c = fmaxf(r2, 1.0e-12f);
        const float ir = __builtin_amdgcn_rsqf(r2c);   // hardware rsq and exp2, about 1 ulp
        const float r = r2c * ir;
        const float dn[3] = {d[0] * ir, d[1] * ir, d[2] * ir};
        float dS;
        const float S = switch_s(r, dS);
        const float ex = __builtin_amdgcn_exp2f(r2 * (-kInv2Sig2 * 1.44269504088896341f));
        const float G0 = p.w_desolv * ex;               // sol(r)
        const float dG0 = -2.f * r * kInv2Sig2 * G0;    // d sol / dr
        const int ch = p.closest_h[pt];
        float rvH[3] = {0.f, 0.f, 0.f};
        if (ch >= 0)
            for (int k = 0; k < 3; k++) rvH[k] = p.rv_by_index[3 * ch + k];
        // directional factors and the pieces their derivatives need
        float racc = 1.f, rdon = 1.f, Hramp = 1.f, dracc_dc = 0.f, dH_dct = 0.f, cth = 0.f;
        if (hb == AG_HB_D1) {
            cth = -(dn[0] * a.rv[0] + dn[1] * a.rv[1] + dn[2] * a.rv[2]);
            racc = racc_of(cth, rexp, dracc_dc);
            if (cth > 0.f && idx != ch && ch >= 0) {
                const float ct = rvH[0] * a.rv[0] + rvH[1] * a.rv[1] + rvH[2] * a.rv[2];
                Hramp = hramp_of(ct, dH_dct);
            }
        } else if (hb == AG_HB_A1) {
            cth = -(dn[0] * a.rv[0] + dn[1] * a.rv[1] + dn[2] * a.rv[2]);
            rdon = cth > 0.f ? cth * cth : 0.f;
        } else if (hb == AG_HB_A2) {
            float g3[3] = {0, 0, 0};
            rdon = a2_rdon<false>(dn, a.rv, a.rv2, 0.f, g3, g3, g3);
        }
        float g_r = 0.f, g_racc = 0.f, g_rdon = 0.f, g_H = 0.f;
#pragma clang loop unroll(full)
        for (int k = 0; k < NA; k++) {
            if (k >= p.naff) continue;
            const float gE_up = p.dmaps[(long long)p.aff_slot[k] * p.P + pt];
            const float gD_up = p.des_slot[k] == p.aff_slot[k] ? gE_up : p.dmaps[(long long)p.des_slot[k] * p.P + pt];
            const LJ lj = lj_eval(load_pair(pairs + k * p.T), r, p.w_smooth);
            const float E = lj.E * S;
            const float rsph = fminf(fmaxf(E * 0.01f, 0.f), 1.f);
            const float drsph = (E > 0.f && E < 100.f) ? 0.01f : 0.f;
            const unsigned cs = (cases >> (2 * k)) & 3;
            float gE = 0.f;   // dL/dE of this map's pair term
            if (cs == CASE_PLAIN) {
                gE = gE_up;
            } else if (cs == CASE_ACC) {
                const float mix = racc + (1.f - racc) * rsph;
                gE = gE_up * Hramp * (mix + E * (1.f - racc) * drsph);
                g_racc += gE_up * E * Hramp * (1.f - rsph);
                g_H += gE_up * E * mix;
            } else {
                const float wmm = (p.amin[(long long)k * p.P + pt] == idx ? 1.f : 0.f) +
                                  (p.amax[(long long)k * p.P + pt] == idx ? 1.f : 0.f);
                if (wmm != 0.f) {
                    const float f = cs == CASE_MM_RACC ? racc : rdon;
                    const float mix = f + (1.f - f) * rsph;
                    const float gu = gE_up * wmm;
                    gE = gu * (mix + E * (1.f - f) * drsph);
                    if (cs == CASE_MM_RACC) g_racc += gu * E * (1.f - rsph);
                    else g_rdon += gu * E * (1.f - rsph);
                }
            }
            // E = lj.E * S
            g_r += gE * (lj.dEdr * S + lj.E * dS);
            acc[11 + k] += gE * lj.dEdR * S;
            acc[11 + kAMaxAff + k] += gE * lj.dEdeps * S;
            // desolvation (sp vol + solq volp) sol S
            const float coef = p.sp[k] * a.vol + solq * p.volp[k];
            g_r += gD_up * coef * (dG0 * S + G0 * dS);
            acc[9] += gD_up * p.qasp * sgnq * p.volp[k] * G0 * S;
            acc[10] += gD_up * coef * ex * S;   // d / d coeff_desolv
        }
        if (p.d_slot >= 0) {
            const float gd = p.dmaps[(long long)p.d_slot * p.P + pt];
            g_r += gd * p.qasp * a.vol * (dG0 * S + G0 * dS);
            acc[10] += gd * p.qasp * a.vol * ex * S;
        }
        // back through the directional factors to dn and the bond vectors
        float gdn[3] = {0.f, 0.f, 0.f};
        if (hb == AG_HB_D1) {
            const float g_c = g_racc * dracc_dc;
            for (int k = 0; k < 3; k++) {
                gdn[k] -= g_c * a.rv[k];
                acc[3 + k] -= g_c * dn[k];
                acc[3 + k] += g_H * dH_dct * rvH[k];
            }
        } else if (hb == AG_HB_A1) {
            const float g_c = cth > 0.f ? g_rdon * 2.f * cth : 0.f;
            for (int k = 0; k < 3; k++) {
                gdn[k] -= g_c * a.rv[k];
                acc[3 + k] -= g_c * dn[k];
            }
        } else if (hb == AG_HB_A2 && g_rdon != 0.f) {
            float grv[3] = {0.f, 0.f, 0.f}, grv2[3] = {0.f, 0.f, 0.f};
            a2_rdon<true>(dn, a.rv, a.rv2, g_rdon, gdn, grv, grv2);
            for (int k = 0; k < 3; k++) {
                acc[3 + k] += grv[k];
                acc[6 + k] += grv2[k];
            }
        }
        // dn = d / r, r = |d|, d = x - c
        const float dot = gdn[0] * dn[0] + gdn[1] * dn[1] + gdn[2] * dn[2];
        for (int k = 0; k < 3; k++) acc[k] += (gdn[k] - dot * dn[k]) * ir + g_r * dn[k];
    };
    int n = 0;   // entries in the wave's list (uniform)
    for (int i0 = 64 * wave; i0 < nitem; i0 += kAT) {
        unsigned long long m = 0;
        int first = 0, yz = 0;   // the word's first point
        if (i0 + lane < nitem) {
            const int i = i0 + lane, r = i / nw, w = w0 + i - r * nw;
            const int iy = lo[1] + r % ny, iz = lo[2] + r / ny;
            const float dy = a.y - (float)(iy - p.ne[1]) * p.h, dz = a.z - (float)(iz - p.ne[2]) * p.h;
            const float rest = kCut2 - dy * dy - dz * dz;
            if (rest > 0.f) {
                const float half = __builtin_amdgcn_sqrtf(rest) * 1.0001f + 1.0e-4f;
                const int x0 = max(lo[0], (int)ceilf((a.x - half) / p.h) + p.ne[0]) - 64 * w;
                const int x1 = min(hi[0], (int)floorf((a.x + half) / p.h) + p.ne[0]) - 64 * w;
                if (x1 >= 0 && x0 < 64 && x0 <= x1) {
                    const long long row = (long long)iy + (long long)p.n1[1] * iz;
                    m = q.bits[row * q.words + w];
                    m &= ~0ull << max(x0, 0);
                    m &= ~0ull >> (63 - min(x1, 63));
                    first = (int)(row * p.n1[0]) + 64 * w;
                    yz = iy | iz << 16;
                }
            }
        }
        // append the lanes' points in lane order, as many lanes at a time as
        // fit, and work the list off sixty-four at a time
        bool more = true;
        while (more) {
            const int c = __popcll(m);
            int x = c;   // inclusive scan over the wave
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(x, o);
                if (lane >= o) x += y;
            }
            const bool fits = n + x <= kList;   // a prefix of the lanes
            int at = n + x - c;
            const int last = __popcll(__ballot(fits));
            n += last > 0 ? __builtin_amdgcn_readlane(x, last - 1) : 0;
            if (fits) {
                while (m) {
                    list[at++] = make_int2(first + __builtin_ctzll(m), yz);
                    m &= m - 1;
                }
            }
            wave_sync();
            more = last < 64;
            const bool end = !more && i0 + kAT >= nitem;   // the wave's last points
            if (more || end || n > kList - 64) {
                const int todo = end ? n : n & ~63;
                for (int t = 0; t < todo; t += 64)
                    if (t + lane < n) point(list[t + lane]);
                const int2 moved = todo + lane < n ? list[todo + lane] : make_int2(0, 0);
                wave_sync();
                if (todo + lane < n) list[lane] = moved;
                n = end ? 0 : n - todo;
                wave_sync();
            }
        }
    }
    block_sum<kAtomOut>(acc, red);
    if (threadIdx.x == 0)
        for (int k = 0; k < kAtomOut; k++) q.out[(long long)blockIdx.x * kAtomOut + k] = acc[k];
}

// The e map's adjoint (k_an_eadj) gathers, per atom, over the points where the
// cotangent is nonzero (the poses' trilinear footprint, a fraction of the box),
// packed first.
constexpr int kGPack = 1024;             // points per packing block (4 per lane)
constexpr int kEAdjChunk = 1024;         // packed points per e-adjoint chunk

// Points where a predicate holds, packed in point order: k_an_count counts
// them per block of kGPack points, k_an_gscan turns the counts into offsets
// (one workgroup) and k_an_pack writes their indices.
struct NonzeroE {             // the e map's cotangent
    const float *ge;
    __device__ bool operator()(long long pt) const { return ge[pt] != 0.f; }
};
struct NonzeroVh {            // the closest H's bond-vector cotangent (k_an_vh)
    const float *vh;
    __device__ bool operator()(long long pt) const {
        return vh[3 * pt] != 0.f || vh[3 * pt + 1] != 0.f || vh[3 * pt + 2] != 0.f;
    }
};

template <typename Pred>
__global__ void __launch_bounds__(256) k_an_count(Pred pred, long long P, int *counts) {
    __shared__ int wc[4];
    const long long b = (long long)blockIdx.x * kGPack;
    int n = 0;
    for (int k = 0; k < 4; k++) {
        const long long pt = b + k * 256 + threadIdx.x;
        n += pt < P && pred(pt);
    }
    for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
    if ((threadIdx.x & 63) == 0) wc[threadIdx.x >> 6] = n;
    __syncthreads();
    if (threadIdx.x == 0) counts[blockIdx.x] = wc[0] + wc[1] + wc[2] + wc[3];
}

// Exclusive offsets of the block counts, and their total in offs[n].
__global__ void __launch_bounds__(1024) k_an_gscan(const int *counts, int n, int *offs) {
    __shared__ int ws[16];
    const int per = (n + 1023) / 1024;
    const int lo = min(n, threadIdx.x * per), hi = min(n, lo + per);
    int t = 0;
    for (int i = lo; i < hi; i++) t += counts[i];
    // inclusive scan of the lane sums: within each wave, then across waves
    int v = t;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(v, o, 64);
        if (lane >= o) v += u;
    }
    if (lane == 63) ws[w] = v;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int k = 1; k < 16; k++) ws[k] += ws[k - 1];
    __syncthreads();
    int run = v - t + (w ? ws[w - 1] : 0);
    for (int i = lo; i < hi; i++) {
        offs[i] = run;
        run += counts[i];
    }
    if (threadIdx.x == 1023) offs[n] = ws[15];
}

template <typename Pred>
__global__ void __launch_bounds__(256) k_an_pack(Pred pred, long long P, const int *offs, int *packed) {
    __shared__ int wc[4][4];
    const long long b = (long long)blockIdx.x * kGPack;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    unsigned long long m[4];
    for (int k = 0; k < 4; k++) {
        const long long pt = b + k * 256 + threadIdx.x;
        m[k] = __ballot(pt < P && pred(pt));
        if (lane == 0) wc[k][w] = __popcll(m[k]);
    }
    __syncthreads();
    int base = offs[blockIdx.x];
    for (int k = 0; k < 4; k++) {
        int before = base;
        for (int j = 0; j < w; j++) before += wc[k][j];
        if ((m[k] >> lane) & 1) packed[before + __popcll(m[k] & ((1ull << lane) - 1))] = (int)(b + k * 256 + threadIdx.x);
        for (int j = 0; j < 4; j++) base += wc[k][j];
    }
}

// Count, offsets and indices of the points where pred holds; the count
// lands in offs[nblk] (device).
template <typename Pred>
static void pack_points(Pred pred, long long P, int *counts, int *offs, int *packed, hipStream_t st) {
    const int nblk = (int)((P + kGPack - 1) / kGPack);
    k_an_count<<<nblk, 256, 0, st>>>(pred, P, counts);
    k_an_gscan<<<1, 1024, 0, st>>>(counts, nblk, offs);
    k_an_pack<<<nblk, 256, 0, st>>>(pred, P, offs, packed);
}

// One wave per (64 atoms, chunk of kEAdjChunk packed points): per atom
// sum_p g f(r) and sum_p g d(q w f(r))/d(atom position), f = 332 / (eps(r)
// max(r, 0.5)) (inv_diel / max(r, 0.5) for a constant dielectric), with
// hardware rsq / exp2 / rcp.  Chunks past the packed count write nothing.
template <bool DD>
__global__ void __launch_bounds__(64) k_an_eadj(EParams p, const int *packed, const int *count) {
    __shared__ float4 sp[256];
    const int ai = blockIdx.x * 64 + threadIdx.x;
    const bool act = ai < p.n_atoms;
    const float4 at = act ? p.atoms[ai] : make_float4(0.f, 0.f, 0.f, 0.f);
    const int npk = *count;
    const int p0 = blockIdx.y * kEAdjChunk, p1 = min(npk, p0 + kEAdjChunk);
    if (p0 >= p1) return;   // uniform; k_an_ered reads the chunks with points
    float gx = 0.f, gy = 0.f, gz = 0.f, gq = 0.f;
    constexpr float cs = kMsLB * 1.44269504088896341f;      // exp(-lambda B r) = 2^(-cs r)
    constexpr float dk = -kMsB * kMsK * kMsLB;             // d(1/eps)/dr = dk e y^2 (see below)
    for (int b = p0; b < p1; b += 256) {
        __syncthreads();
        if (b + (int)threadIdx.x * 4 < p1)
            for (int k = 0; k < 4; k++) {
                const int q = b + threadIdx.x * 4 + k;
                float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
                if (q < p1) {
                    const long long pt = packed[q];
                    const int ix = (int)(pt % p.n1[0]), iy = (int)((pt / p.n1[0]) % p.n1[1]),
                              iz = (int)(pt / ((long long)p.n1[0] * p.n1[1]));
                    v = make_float4((float)(ix - p.ne[0]) * p.h, (float)(iy - p.ne[1]) * p.h,
                                    (float)(iz - p.ne[2]) * p.h, p.ge[pt]);
                }
                sp[threadIdx.x * 4 + k] = v;
            }
        __syncthreads();
        const int nb = min(256, p1 - b);
        for (int j = 0; j < nb; j++) {
            const float4 P = sp[j];
            const float dx = at.x - P.x, dy = at.y - P.y, dz = at.z - P.z;
            const float r2 = fmaxf(__builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz)), 1.0e-12f);
            const float rs = __builtin_amdgcn_rsqf(r2);
            const bool beyond = rs < 2.f;                   // r > 0.5
            const float rm = beyond ? rs : 2.f;             // 1 / max(r, 0.5)
            const float drm = beyond ? -rs * rs : 0.f;      // d(1 / max(r, 0.5))/dr
            float f, dfdr;
            if (DD) {
                // 1/eps = den y, den = 1 + k e, y = 1 / (A den + B), e = exp(-lambda B r):
                // d(1/eps)/dr = B y^2 dden/dr = -B k lambda B e y^2
                const float e = __builtin_amdgcn_exp2f(-cs * (r2 * rs));
                const float den = __builtin_fmaf(kMsK, e, 1.f);
                const float y = __builtin_amdgcn_rcpf(__builtin_fmaf(kMsA, den, kMsB));
                const float G = den * y;
                const float dG = dk * e * (y * y);
                f = 332.f * G * rm;
                dfdr = 332.f * __builtin_fmaf(dG, rm, G * drm);
            } else {
                f = p.inv_diel * rm;
                dfdr = p.inv_diel * drm;
            }
            gq = __builtin_fmaf(P.w, f, gq);
            const float sc = P.w * at.w * dfdr * rs;       // g q w f'(r) / r
            gx = __builtin_fmaf(sc, dx, gx);
            gy = __builtin_fmaf(sc, dy, gy);
            gz = __builtin_fmaf(sc, dz, gz);
        }
    }
    if (act) p.partial[(long long)blockIdx.y * p.n_atoms + ai] = make_float4(gx, gy, gz, gq);
}

// Each atom's chunks added up in FP64: 16 atoms per workgroup and 16 threads
// per atom, each every 16th chunk with points, the threads' sums in order.  (One
// thread per atom, all chunks: 20 workgroups for 5,000 atoms, 77 us; now 4.2.)
constexpr int kRedAtoms = 16;
__global__ void __launch_bounds__(256) k_an_ered(const float4 *partial, int n_atoms, const int *count, double *out) {
    constexpr int kParts = 256 / kRedAtoms;
    __shared__ double sum[kParts][kRedAtoms][4];
    const int a = threadIdx.x % kRedAtoms, part = threadIdx.x / kRedAtoms;
    const int ai = blockIdx.x * kRedAtoms + a;
    const int nchunks = (*count + kEAdjChunk - 1) / kEAdjChunk;
    double s[4] = {0, 0, 0, 0};
    if (ai < n_atoms)
        for (int c = part; c < nchunks; c += kParts) {
            const float4 v = partial[(long long)c * n_atoms + ai];
            s[0] += v.x;
            s[1] += v.y;
            s[2] += v.z;
            s[3] += v.w;
        }
    for (int k = 0; k < 4; k++) sum[part][a][k] = s[k];
    __syncthreads();
    if (threadIdx.x < kRedAtoms * 4) {
        const int b = threadIdx.x / 4, k = threadIdx.x % 4;
        double v = 0.0;
        for (int q = 0; q < kParts; q++) v += sum[q][b][k];
        const int bi = blockIdx.x * kRedAtoms + b;
        if (bi < n_atoms) out[4 * bi + k] = v;
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

struct ag_analytic {
    ag_ctx *ctx = nullptr;
    int N = 0, M = 0, T = 0, n_maps = 0, naff = 0;
    ag_grid grid{};
    long long P = 0;
    // map set
    std::vector<ag_map_desc> maps;
    int elec = -1, dsolv = -1, dddiel = 0, separate = 0, hydrogen_type = -1;
    double inv_diel = 0, qasp = 0;
    double cov_pos[3] = {0, 0, 0}, cov_hw = 1, cov_barrier = 0;
    std::vector<int> aff_slot, des_slot, cov_slots;
    std::vector<std::array<int, 7>> cases;
    // setup (bond vectors, pair forms)
    ag_setup setup{};
    std::vector<ag_pair> pair_form;    // xA, xB, hbonder, explicit cA/cB ([M][T])
    double r_smooth = 0.5;
    // parameters
    std::vector<double> coord, charge, vol, solpar;
    std::vector<int32_t> type, hbond;
    std::vector<double> rij, eps0;     // [M][T]; eps0 unweighted
    double w[4] = {1, 1, 1, 1};        // vdW, H-bond, electrostatic, desolvation weights
    // derived
    std::vector<int32_t> rexp;
    std::vector<double> rv, rv2;
    std::vector<uint8_t> dis;
    std::vector<ag::BondRecipe> recipes;
    std::vector<int> h_atoms, atom_list;
    // device
    DevBuf d_up, d_eup, d_ebox, d_closest, d_amin, d_amax, d_vh, d_hout, d_aout, d_partial, d_eout, d_epart, d_gcount, d_gpack,
        d_vcount, d_vpack, d_gmask;
    HostStage stage;                   // pinned: parameters up, gradients' sums down
    const AAtom *by_index = nullptr;   // in d_up
    const int *hatoms_d = nullptr, *alist_d = nullptr;
    int eK = 16;                       // run length of the forward e kernel
    AParams ap{};
    EParams ep{};
    int nchunks = 0;
    bool uploaded = false;
    float *last_maps = nullptr;
};

namespace agdev {

// The adjoint's work is on all three of the context's streams.
static void wait_streams(ag_ctx *c) {
    (void)hipStreamSynchronize(c->stream);
    (void)hipStreamSynchronize(c->stream2);
    (void)hipStreamSynchronize(c->copy_stream);
}

// (probe class, atom class) -> case of main.cpp:3286-3374 without disorder.
static int an_case(int mh, int ah) {
    const bool atom_don = (ah == 1 || ah == 2 || ah == 6);
    if ((mh == 3 || mh == 5 || mh == 6) && atom_don) return CASE_ACC;
    if ((mh == 4 || mh == 6) && atom_don) return CASE_MM_RACC;
    if ((mh == 1 || mh == 2 || mh == 6) && (ah > 2 || ah == 6)) return CASE_MM_RDON;
    return CASE_PLAIN;
}

ag_analytic *analytic_create(ag_ctx *c, const ag_receptor *rec, const ag_grid *grid, const ag_mapset *ms,
                             const ag_setup *setup, const double w0[4]) {
    if (ms->disorder_h) ag::fail(AG_ERR_UNSUPPORTED, "disorder_h is not part of the analytic model");
    if (ms->bhtree) ag::fail(AG_ERR_UNSUPPORTED, "the tree build's semantics are not part of the analytic model");
    if (setup->n_atom_maps != ms->n_atom_maps) ag::fail(AG_ERR_BAD_INPUT, "setup and map set disagree");
    if (rec->n_atoms < 0 || rec->n_atoms > AG_MAX_ATOMS) ag::fail(AG_ERR_BAD_INPUT, "atom count out of range");
    for (int d = 0; d < 3; d++)
        if (grid->n1[d] < 1 || grid->n1[d] > AG_MAX_GRID_PTS) ag::fail(AG_ERR_BAD_INPUT, "grid out of range");
    for (int k = 0; k < 4; k++)
        if (!(w0[k] > 0)) ag::fail(AG_ERR_BAD_INPUT, "weights must be positive");
    std::unique_ptr<ag_analytic> a(new ag_analytic());
    a->ctx = c;
    const int N = a->N = rec->n_atoms;
    const int M = a->M = ms->n_atom_maps;
    const int T = a->T = setup->n_rec_types;
    a->n_maps = ms->n_maps;
    a->grid = *grid;
    a->P = (long long)grid->n1[0] * grid->n1[1] * grid->n1[2];
    a->maps.assign(ms->maps, ms->maps + M);
    a->elec = ms->elec_index;
    a->dsolv = ms->dsolv_index;
    a->dddiel = ms->dddiel;
    a->separate = ms->separate_desolvation;
    a->hydrogen_type = ms->hydrogen_type;
    a->inv_diel = ms->inv_diel_cal;
    a->qasp = ms->solpar_q;
    for (int d = 0; d < 3; d++) a->cov_pos[d] = ms->cov_pos[d];
    a->cov_hw = ms->cov_half_width;
    a->cov_barrier = ms->cov_barrier;
    a->setup = *setup;
    a->r_smooth = setup->r_smooth;
    a->pair_form.assign(setup->pairs, setup->pairs + (size_t)M * T);
    a->setup.pairs = a->pair_form.data();
    a->coord.assign(rec->coord, rec->coord + 3 * (size_t)N);
    a->charge.assign(rec->charge, rec->charge + N);
    a->vol.assign(rec->vol, rec->vol + N);
    a->solpar.assign(rec->solpar, rec->solpar + N);
    a->type.assign(rec->type, rec->type + N);
    a->hbond.assign(rec->hbond, rec->hbond + N);
    for (int i = 0; i < N; i++)
        if (a->type[i] < 0 || a->type[i] >= T || a->hbond[i] < 0 || a->hbond[i] > 6)
            ag::fail(AG_ERR_BAD_INPUT, "atom type or H-bond class out of range");
    for (int k = 0; k < 4; k++) a->w[k] = w0[k];
    a->rij.assign((size_t)M * T, 0.0);
    a->eps0.assign((size_t)M * T, 0.0);
    for (size_t k = 0; k < (size_t)M * T; k++) {
        const ag_pair &pp = a->pair_form[k];
        a->rij[k] = pp.Rij;
        a->eps0[k] = pp.eps / (pp.hbonder ? w0[1] : w0[0]);
    }
    // map roles: affinity maps carry E terms, their desolvation goes to the
    // map itself or, with separate_desolvation_maps, to the next one
    for (int m = 0; m < M; m++) {
        if (a->maps[m].is_covalent) {
            a->cov_slots.push_back(m);
            continue;
        }
        a->aff_slot.push_back(m);
        a->des_slot.push_back(a->separate ? m + 1 : m);
        std::array<int, 7> cs{};
        for (int ah = 0; ah <= 6; ah++) cs[ah] = a->maps[m].is_hbonder ? an_case(a->maps[m].hbond, ah) : CASE_PLAIN;
        a->cases.push_back(cs);
        if (a->separate) m++;
    }
    a->naff = (int)a->aff_slot.size();
    if (a->naff > kAMaxAff) ag::fail(AG_ERR_UNSUPPORTED, "more than 8 affinity maps in analytic mode");
    if (a->cov_slots.size() > 16) ag::fail(AG_ERR_UNSUPPORTED, "more than 16 covalent maps");
    return a.release();
}

void analytic_destroy(ag_analytic *a) {
    if (!a) return;
    (void)hipSetDevice(a->ctx->device);
    wait_streams(a->ctx);
    delete a;
}

void analytic_set(ag_analytic *a, const double *coord, const double *charge, const double *rij, const double *eps0,
                  const double *w) {
    if (coord) a->coord.assign(coord, coord + 3 * (size_t)a->N);
    if (charge) a->charge.assign(charge, charge + a->N);
    if (rij) a->rij.assign(rij, rij + (size_t)a->M * a->T);
    if (eps0) a->eps0.assign(eps0, eps0 + (size_t)a->M * a->T);
    if (w)
        for (int k = 0; k < 4; k++) {
            if (!(w[k] > 0)) ag::fail(AG_ERR_BAD_INPUT, "weights must be positive");
            a->w[k] = w[k];
        }
    a->uploaded = false;
}

// Arrays on their way up, packed one after the other in pinned memory and
// copied to one device block.
struct UploadPack {
    char *host, *dev;
    size_t used = 0;
    static size_t padded(size_t bytes) { return (bytes + 255) & ~(size_t)255; }
    template <typename T>
    T *add(size_t n, const T **on_device) {
        T *h = reinterpret_cast<T *>(host + used);
        *on_device = reinterpret_cast<const T *>(dev + used);
        used += padded(sizeof(T) * n);
        return h;
    }
    void copy(hipStream_t st) const {
        if (used) HIP_CHECK(hipMemcpyAsync(dev, host, used, hipMemcpyHostToDevice, st));
    }
};

static void cell_grid(const ag_grid &g, float corg[3], int nc[3]) {   // over the box padded by 8 A
    for (int d = 0; d < 3; d++) {
        const double lo = -g.ne[d] * g.spacing - 8.1, hi = (g.n1[d] - 1 - g.ne[d]) * g.spacing + 8.1;
        corg[d] = (float)lo;
        nc[d] = (int)std::ceil((hi - lo) / kCellA) + 1;
    }
}

// Bytes that upload_e and upload_near pack at most.
static size_t upload_e_bytes(const ag_analytic *a) {
    return 2 * UploadPack::padded(sizeof(float4) * (size_t)std::max(a->N, 1));
}
static size_t upload_near_bytes(const ag_analytic *a) {
    const size_t n = (size_t)std::max(a->N, 1), t = (size_t)std::max(a->T, 1), k = (size_t)std::max(a->naff, 1);
    float corg[3];
    int nc[3];
    cell_grid(a->grid, corg, nc);
    const auto pad = UploadPack::padded;
    return 2 * pad(sizeof(AAtom) * n) + pad(sizeof(float) * 3 * n) +
           pad(sizeof(int) * ((size_t)nc[0] * nc[1] * nc[2] + 1)) + pad(sizeof(APair) * k * t) +
           pad(sizeof(ANearType) * t) + 2 * pad(sizeof(int) * n);
}

static void check_pairs(const ag_analytic *a) {
    for (int k = 0; k < a->naff; k++)
        for (int t = 0; t < a->T; t++) {
            const ag_pair &pf = a->pair_form[(size_t)a->aff_slot[k] * a->T + t];
            if (pf.xA == pf.xB || pf.xA <= 0 || pf.xB <= 0)
                ag::fail(AG_ERR_BAD_INPUT, "pair exponents must differ and be positive");
        }
}

// Boxes for the e map's forward where they pay: a box's 512 nodes stand for its
// about 4,096 points, at two more launches (15 us).  At protein density (0.068
// atoms / A^3) the atoms within the distance of a box are pairs as before, so
// a receptor has to hold twice as many, and what is saved at 2.4e12 terms/s has
// to be worth the launches.  (1,000 atoms on 41^3 points stay with 69 us.)
static void e_boxes(ag_analytic *a) {
    EParams &e = a->ep;
    const ag_grid &g = a->grid;
    const int edge[3] = {a->eK, 2 * kEPatch, 2 * kEPatch}, rows[3] = {a->eK, kEPatch, kEPatch};
    double boxes = 1.0, patches = 1.0;
    for (int d = 0; d < 3; d++) {
        e.npatch[d] = (g.n1[d] + rows[d] - 1) / rows[d];
        e.nbox[d] = (g.n1[d] + edge[d] - 1) / edge[d];
        boxes *= e.nbox[d];
        patches *= e.npatch[d];
    }
    // (1 A: past the point where max(r, 0.5) has its kink)
    const double half = 0.5 * (2 * kEPatch - 1) * g.spacing, w = 2.0 * half;
    const double r = std::max((a->dddiel ? 4.5 : 3.5) * half, 1.0);
    const double inside = 0.068 * (w * w * w + r * (6 * w * w + M_PI * r * (3 * w + 4. / 3. * r)));
    const double pairs = patches * 64 * a->eK;
    if (a->N < 2.0 * inside || (a->N - inside) * (pairs - boxes * kEBoxNodes) < 2.4e8) return;
    e.box_parts = (int)std::max(1.0, std::min({1024 / boxes, a->N / 256.0, 16.0}));
    e.split = (int)std::max(1.0, std::min({1536 / patches, a->N / 256.0, 8.0}));
    const double cs = e.sc / g.spacing;   // coordinates of fatoms are scaled by it
    e.box_r2 = (float)(cs * r * (cs * r));
}

// What the electrostatic kernels read: needs the coordinates and charges only.
static void upload_e(ag_analytic *a, UploadPack up) {
    const int N = a->N;
    const ag_grid &g = a->grid;
    EParams &e = a->ep;
    memset(&e, 0, sizeof e);
    float4 *const eat = up.add<float4>(std::max(N, 1), &e.atoms);
    for (int i = 0; i < N; i++)
        eat[i] = make_float4((float)a->coord[3 * i], (float)a->coord[3 * i + 1], (float)a->coord[3 * i + 2],
                             (float)(a->charge[i] * a->w[2]));
    // the forward's atoms: coordinates scaled by cs, weights with the
    // electrostatic constants (k_an_e)
    const double cs = a->dddiel ? (double)kMsLB * 1.4426950408889634 : 1.0;
    const double wk = a->dddiel ? 332.0 * cs : a->inv_diel;
    float4 *const fat = up.add<float4>(std::max(N, 1), &e.fatoms);
    for (int i = 0; i < N; i++)
        fat[i] = make_float4((float)(cs * a->coord[3 * i]), (float)(cs * a->coord[3 * i + 1]),
                             (float)(cs * a->coord[3 * i + 2]), (float)(a->charge[i] * a->w[2] * wk));
    for (int d = 0; d < 3; d++) {
        e.n1[d] = g.n1[d];
        e.ne[d] = g.ne[d];
    }
    e.h = (float)g.spacing;
    e.P = a->P;
    e.n_atoms = N;
    e.dddiel = a->dddiel;
    e.inv_diel = (float)a->inv_diel;
    e.sc = (float)(cs * g.spacing);
    e.rcap = (float)(2.0 / cs);
    e.echunk = std::max(kEAtoms, (N + kEMaxChunks - 1) / kEMaxChunks);
    e.nechunks = std::max(1, (N + e.echunk - 1) / e.echunk);
    // run length: 13 or 16 points, whichever leaves fewer idle run slots
    a->eK = 13 * ((g.n1[0] + 12) / 13) < 16 * ((g.n1[0] + 15) / 16) ? 13 : 16;
    e_boxes(a);
    if (e.box_parts) {
        const size_t boxes = (size_t)e.nbox[0] * e.nbox[1] * e.nbox[2];
        const size_t sums = sizeof(double) * boxes * e.box_parts * kEBoxNodes;
        char *const block = (char *)a->d_ebox.get(sums + sizeof(unsigned long long) * boxes * ((N + 63) / 64));
        e.box_sums = (double *)block;
        e.box_mask = (unsigned long long *)(block + sums);
        e.nechunks = e.split;
    }
    e.epart = (float *)a->d_epart.get(sizeof(float) * (size_t)e.nechunks * (size_t)a->P);
    a->nchunks = (int)((a->P + kEAdjChunk - 1) / kEAdjChunk);
    e.nchunks = a->nchunks;
    e.partial = (float4 *)a->d_partial.get(sizeof(float4) * (size_t)a->nchunks * std::max(N, 1));
    up.copy(a->ctx->stream);
}

// Host precompute and upload of everything the near kernel and the adjoint read.
static void upload_near(ag_analytic *a, UploadPack up) {
    const int N = a->N, T = a->T;
    const ag_grid &g = a->grid;
    AParams &p = a->ap;
    memset(&p, 0, sizeof p);
    // bond vectors with their construction recipes
    a->rexp.assign(N, 0);
    a->rv.assign(3 * (size_t)N, 0.0);
    a->rv2.assign(3 * (size_t)N, 0.0);
    a->dis.assign(N, 0);
    a->recipes.assign(N, ag::BondRecipe{});
    ag::build_bond_vectors(a->setup, N, a->coord.data(), a->type.data(), a->hbond.data(), a->rexp.data(),
                           a->rv.data(), a->rv2.data(), a->dis.data(), nullptr, a->recipes.data());
    float corg[3];
    int nc[3];
    cell_grid(g, corg, nc);
    const int ncells = nc[0] * nc[1] * nc[2];
    std::vector<int> cell_of(N, -1);
    int *const count = up.add<int>(ncells + 1, &p.cell_start);
    std::fill(count, count + ncells + 1, 0);
    AAtom *const by_index = up.add<AAtom>(N, &a->by_index);
    for (int i = 0; i < N; i++) {
        AAtom &t = by_index[i];
        memset(&t, 0, sizeof t);
        t.x = (float)a->coord[3 * i];
        t.y = (float)a->coord[3 * i + 1];
        t.z = (float)a->coord[3 * i + 2];
        t.q = (float)a->charge[i];
        t.vol = (float)a->vol[i];
        t.solpar = (float)a->solpar[i];
        t.meta = (a->type[i] & 0xff) | ((a->hbond[i] & 0xff) << 8) | ((a->rexp[i] & 0xff) << 16);
        t.index = i;
        for (int k = 0; k < 3; k++) {
            t.rv[k] = (float)a->rv[3 * i + k];
            t.rv2[k] = (float)a->rv2[3 * i + k];
        }
        int cc[3];
        bool in = true;
        const float pos[3] = {t.x, t.y, t.z};
        for (int d = 0; d < 3; d++) {
            cc[d] = (int)std::floor((pos[d] - corg[d]) / kCellA);
            in = in && cc[d] >= 0 && cc[d] < nc[d];
        }
        if (in) {
            cell_of[i] = cc[0] + nc[0] * (cc[1] + nc[1] * cc[2]);
            count[cell_of[i] + 1]++;
        }
    }
    for (int k = 0; k < ncells; k++) count[k + 1] += count[k];
    AAtom *const sorted = up.add<AAtom>(count[ncells], &p.atoms);
    {
        std::vector<int> cur(count, count + ncells);
        for (int i = 0; i < N; i++)   // atom index order within each cell
            if (cell_of[i] >= 0) sorted[cur[cell_of[i]]++] = by_index[i];
    }
    float *const rvf = up.add<float>(3 * (size_t)std::max(N, 1), &p.rv_by_index);
    for (size_t k = 0; k < 3 * (size_t)N; k++) rvf[k] = (float)a->rv[k];
    // pair potentials of the affinity maps, effective eps
    const size_t npairs = (size_t)std::max(a->naff, 1) * std::max(T, 1);
    APair *const pairs = up.add<APair>(npairs, &p.pairs);
    memset(pairs, 0, sizeof(APair) * npairs);
    for (int k = 0; k < a->naff; k++)
        for (int t = 0; t < T; t++) {
            const int m = a->aff_slot[k];
            const ag_pair &pf = a->pair_form[(size_t)m * T + t];
            APair &pp = pairs[(size_t)k * T + t];
            pp.a = pf.xA;
            pp.b = pf.xB;
            if (pf.cA == 0 && pf.cB == 0) {
                pp.R = (float)a->rij[(size_t)m * T + t];
                pp.eps = (float)(a->eps0[(size_t)m * T + t] * (pf.hbonder ? a->w[1] : a->w[0]));
                pp.rstar = pp.R;
                pp.expl = 0;
            } else {
                pp.cA = (float)pf.cA;
                pp.cB = (float)pf.cB;
                pp.rstar = (float)std::pow(pf.xA * pf.cA / (pf.xB * pf.cB), 1.0 / (pf.xA - pf.xB));
                pp.expl = 1;
            }
        }
    ANearType *const near_pairs = up.add<ANearType>(std::max(T, 1), &p.near_pairs);
    memset(near_pairs, 0, sizeof(ANearType) * std::max(T, 1));
    for (int k = 0; k < a->naff; k++)
        for (int t = 0; t < T; t++) {
            const APair &pp = pairs[(size_t)k * T + t];
            ANearType &nt = near_pairs[t];
            ANear &q = nt.pair[k];
            const double ke = (double)pp.eps / (pp.a - pp.b);
            q.R = pp.expl ? 1.f : pp.R;
            q.c1 = pp.expl ? pp.cA : (float)(ke * pp.b);
            q.c2 = pp.expl ? pp.cB : (float)(ke * pp.a);
            q.rstar = pp.rstar;
            nt.a[k] = pp.a;
            nt.b[k] = pp.b;
            nt.form |= (pp.a == 12 && pp.b == 6 ? 0 : pp.a == 12 && pp.b == 10 ? 1 : 2) << (2 * k);
        }
    // donor H atoms and atoms whose 8 A sphere meets the box (adjoint work lists)
    a->h_atoms.clear();
    a->atom_list.clear();
    for (int i = 0; i < N; i++) {
        bool near = true;
        for (int d = 0; d < 3; d++) {
            const double lo = -g.ne[d] * g.spacing - 8.0, hi = (g.n1[d] - 1 - g.ne[d]) * g.spacing + 8.0;
            near = near && a->coord[3 * i + d] >= lo && a->coord[3 * i + d] <= hi;
        }
        if (!near) continue;
        a->atom_list.push_back(i);
        if (a->hbond[i] == AG_HB_D1 || a->hbond[i] == AG_HB_DS) a->h_atoms.push_back(i);
    }
    std::copy(a->h_atoms.begin(), a->h_atoms.end(), up.add<int>(a->h_atoms.size(), &a->hatoms_d));
    std::copy(a->atom_list.begin(), a->atom_list.end(), up.add<int>(a->atom_list.size(), &a->alist_d));
    for (int d = 0; d < 3; d++) {
        p.n1[d] = g.n1[d];
        p.ne[d] = g.ne[d];
        p.corg[d] = corg[d];
        p.nc[d] = nc[d];
    }
    p.h = (float)g.spacing;
    p.P = a->P;
    p.n_atoms = N;
    p.naff = a->naff;
    for (int k = 0; k < a->naff; k++) {
        p.aff_slot[k] = a->aff_slot[k];
        p.des_slot[k] = a->des_slot[k];
        const ag_map_desc &md = a->maps[a->des_slot[k]];
        p.sp[k] = (float)md.solpar_probe;
        p.volp[k] = (float)md.vol_probe;
    }
    p.n_cov = (int)a->cov_slots.size();
    for (int k = 0; k < p.n_cov; k++) p.cov_slot[k] = a->cov_slots[k];
    for (int d = 0; d < 3; d++) p.cov_pos[d] = a->cov_pos[d];
    p.cov_hw = a->cov_hw;
    p.cov_barrier = a->cov_barrier;
    p.d_slot = a->dsolv;
    for (int h = 0; h < 7; h++)
        for (int k = 0; k < a->naff; k++) p.case_word[h] |= a->cases[k][h] << (2 * k);
    p.T = T;
    p.w_smooth = (float)(std::floor(a->r_smooth * AG_A_DIV / 2.) / AG_A_DIV);
    p.w_desolv = (float)a->w[3];
    p.qasp = (float)a->qasp;
    p.closest_h = (int *)a->d_closest.get(sizeof(int) * (size_t)a->P);
    p.amin = (int *)a->d_amin.get(sizeof(int) * (size_t)a->P * std::max(a->naff, 1));
    p.amax = (int *)a->d_amax.get(sizeof(int) * (size_t)a->P * std::max(a->naff, 1));
    p.vh = (float *)a->d_vh.get(sizeof(float) * 3 * (size_t)a->P);
    up.copy(a->ctx->stream);
}

static unsigned cube_count(const ag_grid &g) {
    unsigned n = 1;
    for (int d = 0; d < 3; d++) n *= (unsigned)((g.n1[d] + kCube - 1) / kCube);
    return n;
}

template <int K>
static void launch_e(const ag_analytic &a, const EParams &e, hipStream_t st) {
    if (e.box_parts) {
        const unsigned boxes = (unsigned)(e.nbox[0] * e.nbox[1] * e.nbox[2] * e.box_parts);
        const unsigned patches = (unsigned)(e.npatch[0] * e.npatch[1] * e.npatch[2] * e.split);
        if (a.dddiel) {
            k_an_ebox<K, true><<<boxes, 64 * kEWaves, 0, st>>>(e);
            k_an_epatch<K, true><<<patches, 64 * kEWaves, 0, st>>>(e);
        } else {
            k_an_ebox<K, false><<<boxes, 64 * kEWaves, 0, st>>>(e);
            k_an_epatch<K, false><<<patches, 64 * kEWaves, 0, st>>>(e);
        }
        return;
    }
    const long long nruns = (long long)a.grid.n1[1] * a.grid.n1[2] * ((a.grid.n1[0] + K - 1) / K);
    const dim3 eg((unsigned)((nruns + 63) / 64), (unsigned)e.nechunks);
    if (a.dddiel) k_an_e<K, true><<<eg, 64, 0, st>>>(e);
    else k_an_e<K, false><<<eg, 64, 0, st>>>(e);
}

// The e map needs the coordinates and charges only, so its kernels run while
// the host makes the bond vectors, cells and pair tables of new parameters
// (0.5 ms of host work for 5,000 atoms that the device waited for).
void analytic_forward(ag_analytic *a, float *d_maps) {
    ag_ctx *c = a->ctx;
    HIP_CHECK(hipSetDevice(c->device));
    hipStream_t st = c->stream;
    const bool fresh = !a->uploaded;
    UploadPack eup{}, up{};
    if (fresh) {
        check_pairs(a);
        const size_t eb = upload_e_bytes(a), nb = upload_near_bytes(a);
        char *stage = (char *)a->stage.get(eb + nb);   // free: every call waits for its copies
        eup = UploadPack{stage, (char *)a->d_eup.get(eb)};
        up = UploadPack{stage + eb, (char *)a->d_up.get(nb)};
        upload_e(a, eup);
    }
    HIP_CHECK(hipEventRecord(c->ev[0], st));
    if (a->elec >= 0) {
        EParams e = a->ep;
        e.emap = d_maps + (size_t)a->elec * a->P;
        if (a->eK == 13) launch_e<13>(*a, e, st);
        else launch_e<16>(*a, e, st);
        k_an_esum<<<(unsigned)((a->P + 255) / 256), 256, 0, st>>>(e.epart, e.nechunks, a->P, e.emap);
        HIP_CHECK(hipGetLastError());
    }
    HIP_CHECK(hipEventRecord(c->ev[1], st));
    try {
        if (fresh) upload_near(a, up);
    } catch (...) {
        (void)hipStreamSynchronize(st);   // the e kernels write the caller's maps
        throw;
    }
    AParams p = a->ap;
    p.maps = d_maps;
    const unsigned cubes = cube_count(a->grid);
    HIP_CHECK(hipEventRecord(c->ev[2], st));
    if (a->naff <= 4) k_an_near<4><<<cubes, kAT, 0, st>>>(p);
    else if (a->naff <= 6) k_an_near<6><<<cubes, kAT, 0, st>>>(p);
    else k_an_near<8><<<cubes, kAT, 0, st>>>(p);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipEventRecord(c->ev[3], st));
    HIP_CHECK(hipStreamSynchronize(st));
    a->uploaded = true;
    HIP_CHECK(hipEventElapsedTime(&c->last_ms[1], c->ev[2], c->ev[3]));
    HIP_CHECK(hipEventElapsedTime(&c->last_ms[2], c->ev[0], c->ev[1]));
    HIP_CHECK(hipEventElapsedTime(&c->last_ms[3], c->ev[0], c->ev[3]));
    c->last_ms[0] = 0.f;
    a->last_maps = d_maps;
}

// Gradients of L with respect to the parameters, given dL/dmaps on the
// device (the maps of the last forward are the linearisation point).
void analytic_adjoint(ag_analytic *a, const float *d_dmaps, double *g_coord, double *g_charge, double *g_rij,
                      double *g_eps0, double g_w[4]) {
    ag_ctx *c = a->ctx;
    HIP_CHECK(hipSetDevice(c->device));
    if (!a->uploaded || !a->last_maps) ag::fail(AG_ERR_BAD_INPUT, "ag_analytic_adjoint needs a forward first");
    hipStream_t st = c->stream;
    const int N = a->N, T = a->T, M = a->M;
    AParams p = a->ap;
    p.dmaps = d_dmaps;
    const int nh = (int)a->h_atoms.size(), nl = (int)a->atom_list.size();
    const bool want_e = a->elec >= 0 && N > 0;
    // all buffers before the first launch: a failed allocation leaves no kernel
    // behind that reads the caller's cotangent
    float *d_hout = (float *)a->d_hout.get(sizeof(float) * 3 * (size_t)std::max(nh, 1));
    float *d_aout = (float *)a->d_aout.get(sizeof(float) * kAtomOut * (size_t)std::max(nl, 1));
    double *d_eout = (double *)a->d_eout.get(sizeof(double) * 4 * (size_t)std::max(N, 1));
    const size_t hb = UploadPack::padded(sizeof(float) * 3 * (size_t)nh), ab = UploadPack::padded(sizeof(float) * kAtomOut * (size_t)nl);
    char *const stage = (char *)a->stage.get(hb + ab + sizeof(double) * 4 * (size_t)std::max(N, 1));
    const float *const hout = (const float *)stage, *const aout = (const float *)(stage + hb);
    const double *const eout = (const double *)(stage + hb + ab);
    const int row_words = (a->grid.n1[0] + 63) / 64;
    const long long words = (long long)row_words * a->grid.n1[1] * a->grid.n1[2];
    const int nblk = (int)((a->P + kGPack - 1) / kGPack);   // packing blocks
    const size_t pack_counts = sizeof(int) * (2 * (size_t)nblk + 1), packed_points = sizeof(int) * (size_t)a->P;
    unsigned long long *const bits = nl > 0 ? (unsigned long long *)a->d_gmask.get(sizeof(unsigned long long) * (size_t)words) : nullptr;
    int *const vcounts = nh > 0 ? (int *)a->d_vcount.get(pack_counts) : nullptr;
    int *const vlist = nh > 0 ? (int *)a->d_vpack.get(packed_points) : nullptr;
    int *const gcounts = want_e ? (int *)a->d_gcount.get(pack_counts) : nullptr;
    int *const packed = want_e ? (int *)a->d_gpack.get(packed_points) : nullptr;
    // whatever else throws, no stream is left working on the caller's cotangent
    // or the staging buffer
    struct Join {
        ag_ctx *c;
        ~Join() {
            if (c) wait_streams(c);
        }
    } join{c};
    HIP_CHECK(hipEventRecord(c->ev[0], st));
    // Two independent chains: the atom gather, which waits for scattered reads
    // most of its time, and beside it on the second stream the bond-vector
    // cotangent and the e map's adjoint (one after the other they took 860 us of a
    // 5,000-atom, 65^3-point step, now 715).  The near sums go to the host as soon as
    // they are there, and are worked off there beside the rest.
    const hipStream_t s2 = c->stream2;
    HIP_CHECK(hipEventRecord(c->cells_ev, st));
    HIP_CHECK(hipStreamWaitEvent(s2, c->cells_ev, 0));
    if (nl > 0) {
        AtomAdjParams q;
        q.a = p;
        q.by_index = a->by_index;
        q.atom_list = a->alist_d;
        q.out = d_aout;
        q.words = row_words;
        k_an_gmask<<<(unsigned)((words + kAT / 64 - 1) / (kAT / 64)), kAT, 0, st>>>(p, q.words, bits);
        q.bits = bits;
        if (a->naff <= 4) k_an_atom<4><<<nl, kAT, 0, st>>>(q);
        else if (a->naff <= 6) k_an_atom<6><<<nl, kAT, 0, st>>>(q);
        else k_an_atom<8><<<nl, kAT, 0, st>>>(q);
    }
    HIP_CHECK(hipEventRecord(c->near_ev, st));
    if (nh > 0) {
        k_an_vh<<<cube_count(a->grid), kAT, 0, s2>>>(p);
        pack_points(NonzeroVh{p.vh}, a->P, vcounts, vcounts + nblk, vlist, s2);
        HsumParams hp{p.closest_h, p.vh, vlist, vcounts + 2 * nblk, a->hatoms_d, d_hout};
        k_an_hsum<<<nh, kAT, 0, s2>>>(hp);
    }
    HIP_CHECK(hipEventRecord(c->far_ev, s2));
    if (want_e) {
        EParams e = a->ep;
        e.ge = d_dmaps + (size_t)a->elec * a->P;
        int *const offs = gcounts + nblk;
        pack_points(NonzeroE{e.ge}, a->P, gcounts, offs, packed, s2);
        const dim3 eg((unsigned)((N + 63) / 64), (unsigned)a->nchunks);
        if (a->dddiel) k_an_eadj<true><<<eg, 64, 0, s2>>>(e, packed, offs + nblk);
        else k_an_eadj<false><<<eg, 64, 0, s2>>>(e, packed, offs + nblk);
        k_an_ered<<<(N + kRedAtoms - 1) / kRedAtoms, 256, 0, s2>>>(e.partial, N, offs + nblk, d_eout);
        HIP_CHECK(hipGetLastError());
    }
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipEventRecord(c->far2_ev, s2));
    HIP_CHECK(hipStreamWaitEvent(st, c->far2_ev, 0));
    HIP_CHECK(hipEventRecord(c->ev[3], st));
    if (want_e) HIP_CHECK(hipMemcpyAsync(stage + hb + ab, d_eout, sizeof(double) * 4 * (size_t)N, hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipStreamWaitEvent(c->copy_stream, c->far_ev, 0));
    if (nh) HIP_CHECK(hipMemcpyAsync(stage, d_hout, sizeof(float) * 3 * (size_t)nh, hipMemcpyDeviceToHost, c->copy_stream));
    HIP_CHECK(hipStreamWaitEvent(c->copy_stream, c->near_ev, 0));
    if (nl) HIP_CHECK(hipMemcpyAsync(stage + hb, d_aout, sizeof(float) * kAtomOut * (size_t)nl, hipMemcpyDeviceToHost, c->copy_stream));
    HIP_CHECK(hipStreamSynchronize(c->copy_stream));
    // assemble in FP64
    std::vector<double> gx(3 * (size_t)N, 0.0), grv(3 * (size_t)N, 0.0), grv2(3 * (size_t)N, 0.0), gq(N, 0.0);
    std::vector<double> gR((size_t)M * T, 0.0), gE((size_t)M * T, 0.0);
    double gwd = 0.0;
    for (int l = 0; l < nl; l++) {
        const int i = a->atom_list[l];
        const float *o = aout + (size_t)l * kAtomOut;
        for (int k = 0; k < 3; k++) {
            gx[3 * i + k] += o[k];
            grv[3 * i + k] += o[3 + k];
            grv2[3 * i + k] += o[6 + k];
        }
        gq[i] += o[9];
        gwd += o[10];
        for (int k = 0; k < a->naff; k++) {
            const size_t pm = (size_t)a->aff_slot[k] * T + a->type[i];
            gR[pm] += o[11 + k];
            gE[pm] += o[11 + kAMaxAff + k];
        }
    }
    for (int l = 0; l < nh; l++) {
        const int h = a->h_atoms[l];
        for (int k = 0; k < 3; k++) grv[3 * h + k] += hout[3 * l + k];
    }
    // bond vectors -> coordinates
    ag::bond_vectors_vjp(N, a->coord.data(), a->recipes.data(), grv.data(), grv2.data(), gx.data());
    HIP_CHECK(hipStreamSynchronize(st));   // and with it stream2
    join.c = nullptr;
    HIP_CHECK(hipEventElapsedTime(&c->last_ms[3], c->ev[0], c->ev[3]));
    double gwe = 0.0;
    for (int i = 0; want_e && i < N; i++) {
        // eout: d/dx of sum_p g q w f (the float4 weight holds q w), and
        // sum_p g f
        for (int k = 0; k < 3; k++) gx[3 * i + k] += eout[4 * i + k];
        gq[i] += a->w[2] * eout[4 * i + 3];
        gwe += a->charge[i] * eout[4 * i + 3];
    }
    // effective eps -> unweighted eps and the vdW / H-bond weights
    double gwv = 0.0, gwh = 0.0;
    for (int m = 0; m < M; m++)
        for (int t = 0; t < T; t++) {
            const size_t k = (size_t)m * T + t;
            const ag_pair &pf = a->pair_form[k];
            if (!(pf.cA == 0 && pf.cB == 0)) {
                gR[k] = gE[k] = 0.0;
                continue;
            }
            const double wk = pf.hbonder ? a->w[1] : a->w[0];
            if (pf.hbonder) gwh += gE[k] * a->eps0[k];
            else gwv += gE[k] * a->eps0[k];
            gE[k] *= wk;
        }
    if (g_coord) std::copy(gx.begin(), gx.end(), g_coord);
    if (g_charge) std::copy(gq.begin(), gq.end(), g_charge);
    if (g_rij) std::copy(gR.begin(), gR.end(), g_rij);
    if (g_eps0) std::copy(gE.begin(), gE.end(), g_eps0);
    if (g_w) {
        g_w[0] = gwv;
        g_w[1] = gwh;
        g_w[2] = gwe;
        g_w[3] = gwd;
    }
}

void analytic_info(const ag_analytic *a, int *n_atoms, int *n_maps, int64_t *points, int *n_pairs) {
    if (n_atoms) *n_atoms = a->N;
    if (n_maps) *n_maps = a->n_maps;
    if (points) *points = a->P;
    if (n_pairs) *n_pairs = a->M * a->T;
}

}  // namespace agdev
