// kernels_fp64.hpp -- gfx950 kernels of the plain FP64 time step.
//
// One RK stage is three launches,
//   grad_vis     one thread per cell, gathering its faces in the reference's
//                processing order (calc_gradients[_M2AUSM] + calc_VIS)
//   face_flux    one thread per face, each face once (one_rk_step_* body)
//   cell_update  one thread per cell, gathering face fluxes in the
//                reference's accumulation order, then sponge, RK update and
//                the cell's boundary ghosts (set_boundary_conditions)
// or, for inviscid M1 / M2,
//   stage_fused64  one thread per cell, forming its faces' fluxes as it
//                  gathers them, into a second state buffer
// bc_fill fills the boundary ghosts after the state was set from outside.
// The gathers replace the reference's owner/neighbour scatter: every cell
// sums the same terms in the same order as the reference's in-place loop,
// so no atomics are needed and the result does not depend on scheduling.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "mesh_builder.hpp"

namespace lfm {

struct KArgs {
    int nc, nsm0, ng, nf, ntot;
    int ng_bnd;  // boundary ghosts [nc, nc+ng_bnd); halo ghosts after them
    const int32_t *fP, *fN;
    const double *S;                // [nf][D]: a face's area vector as one record
    const double *d, *w;            // d: [D][nf]
    const int32_t *g_off, *g_ent;   // gather lists
    // each cell's first GatherUnroll gather entries and the cells they lead
    // to (key_at places them; kNoFace and the cell itself past its last)
    const int32_t *g_key, *g_oth;
    const int32_t *s_off, *s_ent;   // slot lists
    const int32_t *ghost_cell, *ghost_role;
    const double *vinv;
    const double *sigma;            // nullptr where every cell's sponge sigma is zero
    const double *smag;             // [nc] Smagorinsky constants, nullptr when laminar
    // per-cell face slots of the one-launch stage (nullptr until built), the
    // first GatherUnroll gather entries of each cell, slot_at places them:
    // either packed words (the other cell in the low pk_shift bits, above
    // them the face's record in the geometry table pk_tab) or, where the mesh
    // has too many distinct records, keys (~other on N entries) with the
    // face's own area vector and weight.  A slot past the cell's last entry
    // holds the cell itself.  s_perm: 3 bits per gather entry, its position
    // in the cell's slot list.  more_faces: some cell has entries beyond the
    // slots.
    const uint32_t *pk;
    const double *pk_tab;
    int pk_shift;
    const int32_t *sl_nb;
    const double *sl_S, *sl_w;
    const int32_t *s_perm;
    int more_faces;
    double *q;                      // cell records (q64_index), ghosts included
    double *dq;                     // [(D+2)][nc]
    double *res_cell;               // [(D+2)][nc]
    // per-cell gradient records (GradRec64; ghosts' stay zero): dudx points
    // at the records, dTdx / rho_grad / p_grad / U_grad into them (component
    // stride 1, cell stride gstride); tauMC / sigmaU (partitions only) are
    // [component][ntot]
    double *dudx, *dTdx, *tauMC, *sigmaU;
    double *rho_grad, *p_grad, *U_grad;
    int gstride;
    double *frhs;                   // face records: [nf][4], then (3D) [nf]
    const double *dt;               // device scalar (deltaT)
    double *partial;                // reduction partials
    // gas
    double gamma, gm1, R_inv, mu, cp, pr_inv;
    double p_inf, T_inf, rho_inf, E_inf, U_inf[3];
};

#define INTERP_LINEAR(w, a, b) ((w) * (a) + (1.0 - (w)) * (b))

// MI355X dispatches workgroup b to XCD b % 8, and each XCD has its own L2.
// Remap so that every XCD runs one contiguous slice of the index space: the
// neighbours a face or cell gathers are then mostly in that XCD's L2.
// Bijection of [0, nb).
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_block(int b, int nb) {
    const int x = b % kXcds, j = b / kXcds;
    const int per = nb / kXcds, rem = nb % kXcds;
    return x * per + (x < rem ? x : rem) + j;
}
#define LFM_TID(blk) (xcd_block((int)(blk), (int)gridDim.x) * (int)blockDim.x + (int)threadIdx.x)
#define LFM_BLK() xcd_block((int)blockIdx.x, (int)gridDim.x)

template <int D>
__device__ __forceinline__ double rpsi(const KArgs &a, const double *q) {
    const double ri = 1.0 / q[0];
    double s = q[1] * q[1];
#pragma unroll
    for (int k = 1; k < D; k++) s += q[k + 1] * q[k + 1];
    return a.gm1 * (q[D + 1] - 0.5 * s * ri) * ri;
}

template <int D>
__device__ __forceinline__ double dotD(const double *x, const double *y) {
    double s = x[0] * y[0];
#pragma unroll
    for (int k = 1; k < D; k++) s += x[k] * y[k];
    return s;
}

// Faces per cell whose gathers are issued together before any arithmetic
// (the cell's faces beyond it are gathered one at a time): every cell of a
// 2D quad/triangle mesh and of a 3D hex mesh fits.
template <int D>
struct GatherUnroll {
    static constexpr int value = D == 2 ? 4 : 6;
};

// Face slot storage: for each group of 64 consecutive cells (one wave's
// cells), slot j's field f (NF fields per slot) at
// [c / 64][j][f][c % 64], so that a wave reads one contiguous block of each
// slot array instead of a separate strided stream per slot and field
// (kSlotBlocked; otherwise [j][f][c]).  Arrays hold whole groups.
constexpr bool kSlotBlocked = true;
template <int D, int NF>
__device__ __forceinline__ size_t slot_at(int nc, int j, int f, int c) {
    if constexpr (kSlotBlocked)
        return ((size_t)(c >> 6) * (GatherUnroll<D>::value * NF) + (size_t)(j * NF + f)) * 64 + (size_t)(c & 63);
    return ((size_t)j * NF + f) * (size_t)nc + c;
}
inline size_t slot_array_len(int nc, int U, int NF) { return (size_t)(nc + 63) / 64 * 64 * U * NF; }

// Loads and stores of data a kernel touches once (face slots, RK register, new
// states, the face kernel's face lists and geometry, face fluxes, gradient
// records, 1/V and sponge), non-temporal where NT: that keeps the gathered
// neighbour records in L2, but what one launch wrote the next then does not
// find in the 256 MB Infinity Cache.  So NT is chosen by what a stage touches
// (Solver::stream_nt).
template <bool NT, class T>
__device__ __forceinline__ T ld_once(const T *p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    return *p;
}
template <bool NT, class T>
__device__ __forceinline__ void st_once(T *p, T v) {
    if constexpr (NT)
        __builtin_nontemporal_store(v, p);
    else
        *p = v;
}
using d2v = double __attribute__((ext_vector_type(2)));

// orders a wave's LDS writes before the reads of its other lanes that follow
// (LDS serves one wave's accesses in order; this keeps the compiler to it)
__device__ __forceinline__ void wave_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
template <bool NT>
__device__ __forceinline__ void st64x2_once(double *p, double x, double y) {
    const d2v v = {x, y};
    st_once<NT>(reinterpret_cast<d2v *>(p), v);
}

// face f's area vector (one 16-byte load in 2D)
template <int D>
__device__ __forceinline__ void load_S64(const double *S, int f, double (&s)[D]) {
    if constexpr (D == 2) {
        const double2 v = reinterpret_cast<const double2 *>(S)[f];
        s[0] = v.x;
        s[1] = v.y;
    } else {
#pragma unroll
        for (int k = 0; k < D; k++) s[k] = S[(size_t)f * D + k];
    }
}

// State layout: components 0-3 of a cell (or ghost) i as one 32-byte
// record, q[4 i + k], then component 4 (the 3D energy) as q[4 ntot + i]: a
// gathered neighbour state is two 16-byte loads (three in 3D).
__host__ __device__ __forceinline__ size_t q64_index(int k, size_t i, size_t ntot) {
    return k < 4 ? 4 * i + (size_t)k : 4 * ntot + i;
}

template <int D>
__device__ __forceinline__ void load_q(const KArgs &a, int i, double *q) {
    const double2 *p = reinterpret_cast<const double2 *>(a.q + 4 * (size_t)i);
    const double2 v0 = p[0], v1 = p[1];
    q[0] = v0.x;
    q[1] = v0.y;
    q[2] = v1.x;
    q[3] = v1.y;
    if (D == 3) q[4] = a.q[(size_t)4 * a.ntot + i];
}

template <int D, bool NT>
__device__ __forceinline__ void store_q(double *qv, size_t ntot, int i, const double *q) {
    st64x2_once<NT>(qv + 4 * (size_t)i, q[0], q[1]);
    st64x2_once<NT>(qv + 4 * (size_t)i + 2, q[2], q[3]);
    if (D == 3) st_once<NT>(qv + 4 * ntot + i, q[4]);
}

// One cell's gradients as one record, padded to whole 16-byte words: dudx
// (D*D), dTdx (D), then with RG (the M2AUSM scheme) the rho and p gradients
// (D each) and U_grad (D*D).
template <int D, bool RG>
struct GradRec64 {
    static constexpr int kDT = D * D;
    static constexpr int kRG = kDT + D;
    static constexpr int kPG = kRG + D;
    static constexpr int kUG = kPG + D;
    static constexpr int kN = RG ? kUG + D * D : kRG;
    static constexpr int kStride = (kN + 1) / 2 * 2;
};
inline int grad_record_stride64(int D, bool rg) {
    const int n = D * D + D + (rg ? 2 * D + D * D : 0);
    return (n + 1) / 2 * 2;
}

// Gather entries of fixed width.  A kernel that walks the gather list waits for
// the list's offsets, then the entry, then (gradients) the face's cells before
// it can ask for the other cell's state; from these arrays the face's data and
// the other cell's state are asked for as soon as the entry is there, at the
// same bytes (32 per 2D cell and gradient launch against 30).  Per step, list
// against these: 2D M2AUSM FP32 50.0 -> 47.6 us (4 k cells), 118 -> 112 (262 k),
// 1429 -> 1328 (4.2 M); FP64 73.6 -> 68.4 (16 k), 470 -> 447 (640 k); FP32 O-grid
// 2377 -> 2303 (4 M).
constexpr int32_t kNoFace = INT32_MIN;
__device__ __forceinline__ int face_of(const int key) {
    return key >= 0 ? (key & kFaceMask) : key == kNoFace ? 0 : ~key;
}
// 2D: a cell's four together (one 16-byte load); 3D: as slots
template <int D>
__device__ __forceinline__ size_t key_at(int nc, int j, int c) {
    if constexpr (D == 2) return (size_t)GatherUnroll<2>::value * c + j;
    return slot_at<D, 1>(nc, j, 0, c);
}
inline size_t keys_len(int D, int nc) {
    return D == 2 ? (size_t)GatherUnroll<2>::value * nc : slot_array_len(nc, GatherUnroll<3>::value, 1);
}
using i2v = int32_t __attribute__((ext_vector_type(2)));
using i4v = int32_t __attribute__((ext_vector_type(4)));
// entries [j0, j0 + N) of cell c (2D: j0 a multiple of N)
template <int D, bool NT, int N>
__device__ __forceinline__ void load_keys(const int32_t *p, const int nc, const int j0, const int c, int (&k)[N]) {
    if constexpr (D == 2 && N == 4) {
        const i4v v = ld_once<NT>(reinterpret_cast<const i4v *>(p) + c);
        k[0] = v.x;
        k[1] = v.y;
        k[2] = v.z;
        k[3] = v.w;
    } else if constexpr (D == 2 && N == 2) {
        const i2v v = ld_once<NT>(reinterpret_cast<const i2v *>(p) + 2 * (size_t)c + j0 / 2);
        k[0] = v.x;
        k[1] = v.y;
    } else {
#pragma unroll
        for (int u = 0; u < N; u++) k[u] = ld_once<NT>(p + key_at<D>(nc, j0 + u, c));
    }
}
template <int D>
__global__ void __launch_bounds__(256) build_keys(int nc, const int32_t *g_off, const int32_t *g_ent, const int32_t *fP,
                                                  const int32_t *fN, int32_t *key, int32_t *oth) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    const int e0 = g_off[c], ne = g_off[c + 1] - e0;
    for (int j = 0; j < GatherUnroll<D>::value; j++) {
        const int ent = j < ne ? g_ent[e0 + j] : kNoFace, f = face_of(ent);
        key[key_at<D>(nc, j, c)] = ent;
        if (oth) oth[key_at<D>(nc, j, c)] = j >= ne ? c : ent >= 0 ? fN[f] : fP[f];
    }
}

// face flux record: components 0-3 as 32 bytes per face, component 4 after
template <int D>
__device__ __forceinline__ void load_frhs(const KArgs &a, int f, double (&r)[D + 2]) {
    const double2 *p = reinterpret_cast<const double2 *>(a.frhs + 4 * (size_t)f);
    const double2 v0 = p[0], v1 = p[1];
    r[0] = v0.x;
    r[1] = v0.y;
    r[2] = v1.x;
    r[3] = v1.y;
    if constexpr (D == 3) r[4] = a.frhs[(size_t)4 * a.nf + f];
}

template <int D, bool RG>
__device__ __forceinline__ void load_grec(const KArgs &a, int c, double (&r)[GradRec64<D, RG>::kStride]) {
    using R = GradRec64<D, RG>;
    const double2 *p = reinterpret_cast<const double2 *>(a.dudx + (size_t)c * R::kStride);
#pragma unroll
    for (int k = 0; k < R::kStride / 2; k++) {
        const double2 v = p[k];
        r[2 * k] = v.x;
        r[2 * k + 1] = v.y;
    }
}

__device__ __forceinline__ double sgn(double x) { return x < 0.0 ? -1.0 : 1.0; }

template <int D>
__device__ __forceinline__ double interp_minmod(double cphi, double aphi, const double *grad, const double *d,
                                                double wl, double flux) {
    const double gradf = aphi - cphi + 1.0e-30;
    double gradcf = 0.0;
#pragma unroll
    for (int k = 0; k < D; k++) gradcf += d[k] * grad[k];
    double r;
    if (fabs(gradcf) >= 1000.0 * fabs(gradf))
        r = 2.0 * 1000.0 * sgn(gradcf) * sgn(gradf) - 1.0;
    else
        r = 2.0 * (gradcf / gradf) - 1.0;
    // std::max(std::min(r, 1), 0) of api/cfdv0_solver.h:364
    const double m1 = (1.0 < r) ? 1.0 : r;
    const double lim = (m1 < 0.0) ? 0.0 : m1;
    const double wt = lim * wl + (1.0 - lim) * (1.0 + flux) * 0.5;
    return wt * cphi + (1.0 - wt) * aphi;
}

__device__ __forceinline__ double p5pos(double M, double alpha) {
    const double M2Pos = 0.25 * (M + 1.0) * (M + 1.0);
    const double M2Neg = -0.25 * (M - 1.0) * (M - 1.0);
    const double M1Pos = 0.5 * (M + fabs(M));
    if (fabs(M) < 1) return M2Pos * ((2.0 - M) - 16.0 * alpha * M * M2Neg);
    return M1Pos / M;
}

__device__ __forceinline__ double p5neg(double M, double alpha) {
    const double M2Pos = 0.25 * (M + 1.0) * (M + 1.0);
    const double M2Neg = -0.25 * (M - 1.0) * (M - 1.0);
    const double M1Neg = 0.5 * (M - fabs(M));
    if (fabs(M) < 1) return M2Neg * ((-2.0 - M) + 16.0 * alpha * M * M2Pos);
    return M1Neg / M;
}

// ---------------------------------------------------------------------------
// Ghost state of one boundary face from its interior cell's state qi
// (cfd_v0.cpp:1010-1133); returns false for an unset patch (the ghost keeps
// q = 0).
// ---------------------------------------------------------------------------
template <int D>
__device__ __forceinline__ bool ghost_state(const KArgs &a, int role, const double *qi, double *qg) {
    if (role == 1) {  // wall
        qg[0] = qi[0];
#pragma unroll
        for (int k = 0; k < D; k++) qg[k + 1] = -qi[k + 1];
        qg[D + 1] = qi[D + 1];
        return true;
    }
    if (role != 2 && role != 3) return false;
    const double rhoInt = qi[0];
    double Uint[D], u2i = 0.0;
#pragma unroll
    for (int k = 0; k < D; k++) {
        Uint[k] = qi[k + 1] / rhoInt;
        u2i += Uint[k] * Uint[k];
    }
    const double pInt = (qi[D + 1] - 0.5 * u2i * rhoInt) * a.gm1;
    double rhoExt, pExt, Uext[D], u2e = 0.0;
    if (role == 2) {  // inlet
        const double TInt = pInt * a.R_inv / rhoInt;
        const double TExt = a.T_inf;
        rhoExt = rhoInt * TInt / TExt;
#pragma unroll
        for (int k = 0; k < D; k++) {
            Uext[k] = a.U_inf[k];
            u2e += Uext[k] * Uext[k];
        }
        pExt = pInt;
    } else {  // outlet
        pExt = a.p_inf;
        rhoExt = rhoInt * pExt / pInt;
#pragma unroll
        for (int k = 0; k < D; k++) {
            Uext[k] = Uint[k];
            u2e += Uext[k] * Uext[k];
        }
    }
    const double EExt = pExt / (rhoExt * a.gm1) + 0.5 * u2e;
    qg[0] = rhoExt;
#pragma unroll
    for (int k = 0; k < D; k++) qg[k + 1] = rhoExt * Uext[k];
    qg[D + 1] = rhoExt * EExt;
    return true;
}

// ---------------------------------------------------------------------------
// set_boundary_conditions (cfd_v0.cpp:1010-1133): ghost state per boundary
// face from its interior cell.  Ghost gradient copies are not stored: the
// interior gradients they copy are zero at this point of every stage, and
// the flux kernels read zero ghost gradients (see grad arrays' ghost part).
// In the fused step the update kernel refreshes the ghosts of the cells it
// updates, so this kernel only runs after the state is set from outside.
// ---------------------------------------------------------------------------
template <int D>
__global__ void __launch_bounds__(256) bc_fill(KArgs a) {
    const int g = LFM_TID(blockIdx.x);
    if (g >= a.ng) return;
    double qi[D + 2], qg[D + 2];
    load_q<D>(a, a.ghost_cell[g], qi);
    if (!ghost_state<D>(a, a.ghost_role[g], qi, qg)) return;
    const int gi = a.nc + g;
    store_q<D, false>(a.q, a.ntot, gi, qg);
}

// ---------------------------------------------------------------------------
// Green-Gauss gradients + viscous tensors, per cell (cfd_v0.cpp:1384-1567,
// 1744-1860).  The reference refreshes tau/sigmaU/tauMC after every touch of
// a cell; the last touch of a cell follows its last contribution, so the
// stored values equal the refresh of the completed sums done here.
// GRAD: 0 none, 1 calc_gradients (results unused by solvers 0/1: skipped),
// 2 calc_gradients_M2AUSM (rho, p, U gradients consumed by the M2AUSM flux).
// VISC false (mu = 0): dTdx, tau, sigmaU and tauMC only ever enter the flux
// multiplied by mu, so they are not formed; dudx is kept for the M2AUSM
// sensor.  (For solvers 0/1 with mu = 0 the kernel is not launched.)
// ---------------------------------------------------------------------------
// tauMC and sigmaU of one cell from its completed dudx (cfd_v0.cpp:1813-1834,
// Smagorinsky 1668-1684 when smag is given): the values calc_VIS leaves in
// the cell.  Used where they are stored and where a face recomputes them.
template <int D>
__device__ __forceinline__ void vis_tensors(const KArgs &a, const double (&dudx)[D][D], const double *qc,
                                            const double *smag_p, double (&tmc)[D][D], double (&sU)[D]) {
    double U[D];
#pragma unroll
    for (int k = 0; k < D; k++) U[k] = qc[k + 1] / qc[0];
    const double mu = a.mu;
    double tau[D][D];
#pragma unroll
    for (int p = 0; p < D; p++) {
        tau[p][p] = 2.0 * dudx[p][p];
#pragma unroll
        for (int b1 = p + 1; b1 < D + p; b1++) {
            const int b = b1 % D;
            tau[p][b] = mu * (dudx[p][b] + dudx[b][p]);
            tau[p][p] -= dudx[b][b];
        }
        tau[p][p] *= 2.0 / 3.0 * mu;
    }
    double diag = 0;
#pragma unroll
    for (int p = 0; p < D; p++) diag -= dudx[p][p];
    diag *= mu * 2.0 / 3.0;
#pragma unroll
    for (int i = 0; i < D; i++) {
#pragma unroll
        for (int j = 0; j < D; j++) tmc[i][j] = mu * dudx[j][i];
        tmc[i][i] += diag;
    }
    if (smag_p) {
        // calc_VIS_Smagorinsky: minus the eddy stress smag |S| S_ij, plus the
        // compressible correction smag |S| div u / 3
        const double smag = *smag_p;
        double strain = 0.0, divu = 0.0;
#pragma unroll
        for (int i = 0; i < D; i++) {
#pragma unroll
            for (int j = 0; j < D; j++) {
                const double sij = 0.5 * (dudx[i][j] + dudx[j][i]);
                strain += sij * sij;
            }
            divu += dudx[i][i];
        }
        strain = sqrt(2.0 * strain);
#pragma unroll
        for (int i = 0; i < D; i++) {
#pragma unroll
            for (int j = 0; j < D; j++) {
                const double sij = 0.5 * (dudx[i][j] + dudx[j][i]);
                tmc[i][j] -= smag * strain * sij;
            }
            tmc[i][i] += smag * strain * divu / 3.0;
        }
    }
#pragma unroll
    for (int i = 0; i < D; i++) sU[i] = dotD<D>(U, tau[i]);
}

// Bound: latency (at a few 100 k cells a launch has 2-3 waves per SIMD to hide
// its dependent loads), so registers decide; in 3D past the cache, memory.
// Faces in groups whose loads are issued together: all four in 2D (176 k-cell
// annulus, four 171, two 176 us per step), two in 3D at 3 waves per SIMD (193
// k-cell O-grid: three spill and take 415, two 397, one 397) and, where the
// stage outgrows the cache, all six at 2 (1 M cells 1400 -> 1351, 4.2 M 5983 ->
// 5873).  There the M1 / M2 gradients are one straight line of six faces: as the
// body of the rolled loop, which is run once, the same faces take 8 % longer
// (4.2 M cells, us of gradients per step: loop 1749, straight 1618; the loop with
// the gather list 1850, straight with it 1684; 3 waves 2140).  With the M2AUSM
// records the two are equal (1 M cells 574 / 574).
template <int D, bool NT>
constexpr int kGradGroup64 = D == 2 ? 4 : NT ? 6 : 2;
template <int D, int GRAD, bool VISC, bool RG, bool NT, bool RNT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kGradGroup64<D, NT> == 6 ? 2 : 3))) grad_vis(KArgs a) {
    const int c = LFM_TID(blockIdx.x);
    using R = GradRec64<D, RG>;
    // every thread reaches the record write-out below (LDS staging)
    const bool valid = c < a.nc;
    double rec[R::kStride];
#pragma unroll
    for (int k = 0; k < R::kStride; k++) rec[k] = 0.0;
    if (valid) {
    const double vinv = a.vinv[c];
    double dudx[D][D], dTdx[D];
    double rg[D], pg[D], ug[D][D];
#pragma unroll
    for (int i = 0; i < D; i++) {
        dTdx[i] = 0.0;
        rg[i] = 0.0;
        pg[i] = 0.0;
#pragma unroll
        for (int j = 0; j < D; j++) {
            dudx[i][j] = 0.0;
            ug[i][j] = 0.0;
        }
    }
    double qself[D + 2];
    load_q<D>(a, c, qself);
    // what a face needs of a cell: velocities as products with 1/rho (dudx,
    // dTdx) and, for M2AUSM, as quotients (ug, p), as the reference forms them
    struct Cell {
        double R, u[D], v[D], p;
    };
    auto cell = [&](const double (&q)[D + 2]) {
        Cell x;
        const double ri = 1.0 / q[0];
        x.R = VISC ? rpsi<D>(a, q) : 0.0;
#pragma unroll
        for (int k = 0; k < D; k++) x.u[k] = q[k + 1] * ri;
        if (GRAD == 2) {
            const double r = q[0], E = q[D + 1] / r;
            double vm = 0.0;
#pragma unroll
            for (int k = 0; k < D; k++) {
                x.v[k] = q[k + 1] / r;
                vm += x.v[k] * x.v[k];
            }
            x.p = r * a.gm1 * (E - 0.5 * vm);
        }
        return x;
    };
    const Cell own = cell(qself);
    // one face's contribution; INTERP_LINEAR's two products are the same ones
    // from either side, so the cell's own come first and no side is selected
    auto add = [&](const bool isP, const double w, const double (&S)[D], const double (&qo)[D + 2]) {
        const Cell o = cell(qo);
        const double omw = 1.0 - w, wc = isP ? w : omw, wo = isP ? omw : w;
        double sv[D];
#pragma unroll
        for (int k = 0; k < D; k++) sv[k] = isP ? S[k] * vinv : -S[k] * vinv;
        if (GRAD == 2) {
            const double rho = wc * qself[0] + wo * qo[0];
            const double pf = wc * own.p + wo * o.p;
#pragma unroll
            for (int i = 0; i < D; i++) {
                pg[i] += pf * sv[i];
                rg[i] += rho * sv[i];
            }
#pragma unroll
            for (int j = 0; j < D; j++) {
                const double UU = wc * own.v[j] + wo * o.v[j];
#pragma unroll
                for (int i = 0; i < D; i++) ug[j][i] += UU * sv[i];
            }
        }
        const double fT = VISC ? (wc * own.R + wo * o.R) * a.R_inv : 0.0;
#pragma unroll
        for (int i = 0; i < D; i++) {
            const double fU = wc * own.u[i] + wo * o.u[i];
#pragma unroll
            for (int j = 0; j < D; j++) dudx[i][j] += fU * sv[j];
            if (VISC) dTdx[i] += fT * sv[i];
        }
    };
    // groups of G faces in gather order, their loads issued together
    constexpr int U = GatherUnroll<D>::value, G = kGradGroup64<D, NT>;
    constexpr bool kStraight = D == 3 && NT && !RG;
    static_assert(U % G == 0 && (!kStraight || G == U));
    int key[G], oth[G], e0 = 0, ne = U;
    load_keys<D, NT>(a.g_key, a.nc, 0, c, key);
    load_keys<D, NT>(a.g_oth, a.nc, 0, c, oth);
    if constexpr (kStraight) {
        double wj[G], Sj[G][D], qj[G][D + 2];
#pragma unroll
        for (int u = 0; u < G; u++) {
            const int f = face_of(key[u]);
            wj[u] = a.w[f];
            load_S64<D>(a.S, f, Sj[u]);
            load_q<D>(a, oth[u], qj[u]);
        }
#pragma unroll
        for (int u = 0; u < G; u++)
            if (key[u] != kNoFace) add(key[u] >= 0, wj[u], Sj[u], qj[u]);
        if (a.more_faces) {  // entries beyond the first U
            const int e2 = a.g_off[c + 1];
            for (int e = a.g_off[c] + U; e < e2; e++) {
                const int ent = a.g_ent[e], f = face_of(ent);
                double S1[D], q1[D + 2];
                load_S64<D>(a.S, f, S1);
                load_q<D>(a, ent >= 0 ? a.fN[f] : a.fP[f], q1);
                add(ent >= 0, a.w[f], S1, q1);
            }
        }
        ne = 0;
    } else if (a.more_faces) {
        e0 = a.g_off[c];
        ne = max(U, a.g_off[c + 1] - e0);
    }
#pragma unroll 1
    for (int j0 = 0; j0 < ne; j0 += G) {
        double wj[G], Sj[G][D], qj[G][D + 2];
        int nkey[G], noth[G];
#pragma unroll
        for (int u = 0; u < G; u++) {
            const int f = face_of(key[u]);
            wj[u] = a.w[f];
            load_S64<D>(a.S, f, Sj[u]);
            load_q<D>(a, oth[u], qj[u]);
        }
        const int jn = j0 + G;
#pragma unroll
        for (int u = 0; u < G; u++) nkey[u] = noth[u] = kNoFace;
        if constexpr (G < U) {
            load_keys<D, NT>(a.g_key, a.nc, jn < U ? jn : 0, c, nkey);
            load_keys<D, NT>(a.g_oth, a.nc, jn < U ? jn : 0, c, noth);
        }
        if (a.more_faces && jn >= U) {  // entries beyond the first U
#pragma unroll
            for (int u = 0; u < G; u++) {
                nkey[u] = jn + u < ne ? a.g_ent[e0 + jn + u] : kNoFace;
                const int f = face_of(nkey[u]);
                noth[u] = nkey[u] >= 0 ? a.fN[f] : a.fP[f];
            }
        }
#pragma unroll
        for (int u = 0; u < G; u++) {
            if (key[u] != kNoFace) add(key[u] >= 0, wj[u], Sj[u], qj[u]);
            key[u] = nkey[u];
            oth[u] = noth[u];
        }
    }
    // refresh of tau / sigmaU / tauMC from the completed dudx (cfd_v0.cpp:1813-1834);
    // stored only where a halo payload needs them (otherwise each face
    // recomputes them from dudx)
    const size_t nt = a.ntot;
    if (VISC && a.tauMC) {
        double tmc[D][D], sU[D];
        vis_tensors<D>(a, dudx, qself, a.smag ? a.smag + c : nullptr, tmc, sU);
#pragma unroll
        for (int i = 0; i < D; i++) {
            a.sigmaU[i * nt + c] = sU[i];
#pragma unroll
            for (int j = 0; j < D; j++) a.tauMC[(i * D + j) * nt + c] = tmc[i][j];
        }
    }
#pragma unroll
    for (int i = 0; i < D; i++) {
#pragma unroll
        for (int j = 0; j < D; j++) rec[i * D + j] = dudx[i][j];
        rec[R::kDT + i] = VISC ? dTdx[i] : 0.0;
        if (RG && GRAD == 2) {
            rec[R::kRG + i] = rg[i];
            rec[R::kPG + i] = pg[i];
#pragma unroll
            for (int j = 0; j < D; j++) rec[R::kUG + i * D + j] = ug[i][j];
        }
    }
    if (!VISC) {
        // dTdx not formed: the formed components only (the record keeps
        // whatever a full calc_VIS left in the dTdx slots)
        double *out = a.dudx + (size_t)c * R::kStride;
#pragma unroll
        for (int k = 0; k < R::kN; k++)
            if (k < R::kDT || k >= R::kRG) out[k] = rec[k];
    }
    }
    if (VISC) {
        // the wave's records are contiguous from its first cell.  In 2D where the
        // stage fits the cache, four 16-byte words of each at a time are staged
        // in LDS and written as 64-byte runs, which L2 joins (176 k-cell
        // annulus 171 against 174 us per step); otherwise the records of 16
        // cells at a time, written as consecutive words (64-byte runs wrote
        // 540 MB where the records of a 4.2 M-cell O-grid are 403).  The face
        // launch reads the records next: non-temporal stores only where they
        // outgrow what the Infinity Cache keeps for it (RNT, from 190 MB; MB of
        // records, us per step plain / non-temporal: M1 / M2 O-grid 101 MB 1312 /
        // 1366, 201 2810 / 2790, 403 5691 / 5611; M2AUSM 117 970 / 1010, 176 1459 /
        // 1485, 235 1993 / 1947; annulus 117 801 / 834, 235 1613 / 1602).
        // Staging whole blocks (57 KB for 3D M2AUSM) held the kernel at 2 waves
        // per SIMD; without minmod the rho / p / U slots are written zero.
        constexpr bool kRuns = D == 2 && !NT;
        constexpr int W = R::kStride / 2, C = 4, M = 16;
        __shared__ double2 stage[256 / 64][kRuns ? 64 * C : M * W];
        double2 *st = stage[threadIdx.x >> 6];
        const int lane = threadIdx.x & 63, c0 = c - lane;
        d2v *dst = reinterpret_cast<d2v *>(a.dudx + (size_t)c0 * R::kStride);
        if constexpr (kRuns) {
#pragma unroll
            for (int w0 = 0; w0 < W; w0 += C) {
                const int n = W - w0 < C ? W - w0 : C;
#pragma unroll
                for (int k = 0; k < n; k++) st[lane * n + k] = make_double2(rec[2 * (w0 + k)], rec[2 * (w0 + k) + 1]);
                wave_sync_lds();
#pragma unroll
                for (int i = 0; i < n; i++) {
                    const int j = i * 64 + lane, r = j / n;
                    const double2 v = st[j];
                    if (c0 + r < a.nc) st_once<false>(dst + r * W + w0 + j % n, d2v{v.x, v.y});
                }
                wave_sync_lds();
            }
        } else {
#pragma unroll
            for (int g = 0; g < 64 / M; g++) {
                if (lane / M == g)
#pragma unroll
                    for (int k = 0; k < W; k++) st[(lane % M) * W + k] = make_double2(rec[2 * k], rec[2 * k + 1]);
                wave_sync_lds();
                const int n = min(a.nc - c0 - g * M, M) * W;
#pragma unroll
                for (int j = lane; j < M * W; j += 64) {
                    const double2 v = st[j];
                    if (j < n) st_once<RNT>(dst + g * M * W + j, d2v{v.x, v.y});
                }
                wave_sync_lds();
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Convective flux of one face (M1 cfd_v0.cpp:2589-2675, M2 1968-2023) seen
// from one of its cells: c that cell, o the other, S pointing out of c, wc / wo
// the weights of INTERP_LINEAR(wc, c, o) and INTERP_LINEAR(wo, o, c) (w and
// 1 - w for the face's P, 1 - w and w for its N).  With c = P these are the
// reference's operations; from N every product and sum is the same one with
// both signs reversed or the two addends exchanged, so the result is P's
// negated, bit for bit, and a cell can form its faces' fluxes without
// selecting which side it is on.
// ---------------------------------------------------------------------------
template <int D>
struct Prim64 {
    double R, c, e;  // p / rho, speed of sound, internal energy (M2: R and e = H)
};
template <int D, int SOLVER>
__device__ __forceinline__ Prim64<D> prim64(const KArgs &a, const double (&q)[D + 2]) {
    Prim64<D> s;
    s.R = rpsi<D>(a, q);
    if constexpr (SOLVER == 0) {
        const double ri = 1.0 / q[0];
        double e = 2 * q[D + 1] * ri;
#pragma unroll
        for (int k = 0; k < D; k++) {
            const double u = q[k + 1] * ri;
            e -= u * u;
        }
        s.e = e * 0.5;
        s.c = sqrt(a.gamma * s.R);
    } else {
        s.e = q[D + 1] / q[0] + s.R;
        s.c = 0.0;
    }
    return s;
}

template <int D>
__device__ __forceinline__ void flux_m1(const double (&qc)[D + 2], const Prim64<D> &sc, const double (&qo)[D + 2],
                                        const Prim64<D> &so, const double (&S)[D], const double Sm, const double wc,
                                        const double wo, double (&rhs)[D + 2]) {
    const double rhoPos = INTERP_LINEAR(wc, qc[0], qo[0]);
    const double rhoNeg = INTERP_LINEAR(wo, qo[0], qc[0]);
    const double rPi = 1.0 / rhoPos, rNi = 1.0 / rhoNeg;
    double rUP[D], rUN[D], uP[D], uN[D];
#pragma unroll
    for (int k = 0; k < D; k++) {
        rUP[k] = INTERP_LINEAR(wc, qc[k + 1], qo[k + 1]);
        rUN[k] = INTERP_LINEAR(wo, qo[k + 1], qc[k + 1]);
    }
    const double eP = INTERP_LINEAR(wc, sc.e, so.e), eN = INTERP_LINEAR(wo, so.e, sc.e);
    const double RP = INTERP_LINEAR(wc, sc.R, so.R), RN = INTERP_LINEAR(wo, so.R, sc.R);
    const double pP = rhoPos * RP, pN = rhoNeg * RN;
    const double cPos = INTERP_LINEAR(wc, sc.c, so.c), cNeg = INTERP_LINEAR(wo, so.c, sc.c);
    double phP = 0.0, phN = 0.0;
#pragma unroll
    for (int k = 0; k < D; k++) {
        uP[k] = rUP[k] * rPi;
        uN[k] = rUN[k] * rNi;
        phP += uP[k] * S[k];
        phN += -uN[k] * S[k];
    }
    // std::max({x1, x2, 0}) / std::min({y1, y2, 0}): first extreme wins
    const double x1 = phP + cPos * Sm, x2 = -phN + cNeg * Sm;
    double psiP = (x1 < x2) ? x2 : x1;
    if (psiP < 0.0) psiP = 0.0;
    const double y1 = phP - cPos * Sm, y2 = -phN - cNeg * Sm;
    double psiN = (y2 < y1) ? y2 : y1;
    if (0.0 < psiN) psiN = 0.0;
    const double a0 = 1.0 / (psiP - psiN);
    const double a1 = psiP * psiN;
    const double aP = psiP * phP, aN = psiN * phN;
    double rEP = eP, rEN = eN;
#pragma unroll
    for (int k = 0; k < D; k++) {
        rEP += 0.5 * uP[k] * uP[k];
        rEN += 0.5 * uN[k] * uN[k];
    }
    rEP *= rhoPos;
    rEN *= rhoNeg;
    rhs[0] = -(aP * rhoPos + aN * rhoNeg + (rhoNeg - rhoPos) * a1) * a0;
#pragma unroll
    for (int k = 0; k < D; k++)
        rhs[k + 1] = -((aP * rUP[k] + aN * rUN[k] + (rUN[k] - rUP[k]) * a1) * a0 +
                       (pP * psiP - pN * psiN) * a0 * S[k]);
    rhs[D + 1] = -(aP * rEP + aN * rEN + (rEN - rEP) * a1 + (aP * pP + aN * pN)) * a0;
}

// flux_m1 where 1 - wc == wo and 1 - wo == wc hold exactly (any w >= 1/2, and
// half of those below): both reconstructed states are then the same sums of
// the same products, so the second one's operations are left out and the
// result is the same to the bit.
template <int D>
__device__ __forceinline__ void flux_m1_sym(const double (&qc)[D + 2], const Prim64<D> &sc, const double (&qo)[D + 2],
                                            const Prim64<D> &so, const double (&S)[D], const double Sm,
                                            const double wc, const double wo, double (&rhs)[D + 2]) {
    const double rho = wc * qc[0] + wo * qo[0];
    const double ri = 1.0 / rho;
    double rU[D], ph = 0.0;
    double rE = wc * sc.e + wo * so.e;
#pragma unroll
    for (int k = 0; k < D; k++) {
        rU[k] = wc * qc[k + 1] + wo * qo[k + 1];
        const double u = rU[k] * ri;
        ph += u * S[k];
        rE += 0.5 * u * u;
    }
    rE *= rho;
    const double p = rho * (wc * sc.R + wo * so.R);
    const double cS = (wc * sc.c + wo * so.c) * Sm;
    double psiP = ph + cS, psiN = ph - cS;
    if (psiP < 0.0) psiP = 0.0;
    if (0.0 < psiN) psiN = 0.0;
    const double a0 = 1.0 / (psiP - psiN);
    const double aP = psiP * ph, aN = psiN * -ph;
    rhs[0] = -(aP * rho + aN * rho) * a0;
    const double pS = (p * psiP - p * psiN) * a0;
#pragma unroll
    for (int k = 0; k < D; k++) rhs[k + 1] = -((aP * rU[k] + aN * rU[k]) * a0 + pS * S[k]);
    rhs[D + 1] = -(aP * rE + aN * rE + (aP * p + aN * p)) * a0;
}

// M2's face pressure and mass flux are formed by the face kernel too, which
// adds the AUSM correction to the pressure in between
template <int D>
__device__ __forceinline__ void flux_m2(const double rhoavg, const double (&rUa)[D], const double Havg,
                                        const double pavg, const double (&S)[D], double (&rhs)[D + 2]) {
    const double rai = 1.0 / rhoavg;
    double phi = 0.0;
#pragma unroll
    for (int k = 0; k < D; k++) phi += (rUa[k] * rai) * S[k];
    rhs[0] = -rhoavg * phi;
#pragma unroll
    for (int k = 0; k < D; k++) rhs[k + 1] = -(rUa[k] * phi + pavg * S[k]);
    rhs[D + 1] = -(rhoavg * Havg * phi);
}

// ---------------------------------------------------------------------------
// Face fluxes: convective (M1 2589-2675, M2 1968-2023, M2AUSM 2256-2366) plus
// the viscous terms shared by all three (2682-2790).  One thread per face.
// VISC false (mu = 0): every viscous term is mu or k = cp mu / Pr times a
// finite value, i.e. a zero the reference adds; it is not formed.
// STORED: tauMC / sigmaU read from the arrays grad_vis filled (partitions,
// whose halo payload carries them); otherwise formed here from dudx.
// In 2D, 3 waves per SIMD: the viscous M2AUSM face then fits 168 VGPRs
// without spills instead of 170 (2 waves), 82 -> 73 us per launch on 1 M
// cells; in 3D the same bound spills and is slower.
// ---------------------------------------------------------------------------
template <int D, int SOLVER, bool VISC, bool STORED, bool NT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 2 ? 3 : 2))) face_flux(KArgs a) {
    const int f = LFM_TID(blockIdx.x);
    if (f >= a.nf) return;
    const int P = ld_once<NT>(a.fP + f), N = ld_once<NT>(a.fN + f);
    // is_ghost: boundary ghosts only; halo ghosts carry the neighbour's tensors
    const bool ghost = (unsigned)(N - a.nc) < (unsigned)a.ng_bnd;
    const double w = ld_once<NT>(a.w + f);
    const size_t nt = a.ntot;
    double S[D], d[D], qP[D + 2], qN[D + 2];
#pragma unroll
    for (int k = 0; k < D; k++) S[k] = ld_once<NT>(a.S + (size_t)f * D + k);
#pragma unroll
    for (int k = 0; k < D; k++) d[k] = ld_once<NT>(a.d + (size_t)k * a.nf + f);
    load_q<D>(a, P, qP);
    load_q<D>(a, N, qN);
    using R = GradRec64<D, SOLVER == 2>;
    double gr[2][R::kStride];  // gradient records of P and N
    if (VISC || SOLVER == 2) {
        load_grec<D, SOLVER == 2>(a, P, gr[0]);
        load_grec<D, SOLVER == 2>(a, N, gr[1]);
    }
    const double cri = 1.0 / qP[0], ari = 1.0 / qN[0];
    double cU[D], aU[D];
#pragma unroll
    for (int k = 0; k < D; k++) {
        cU[k] = qP[k + 1] * cri;
        aU[k] = qN[k + 1] * ari;
    }
    const double cR = rpsi<D>(a, qP), aR = rpsi<D>(a, qN);
    const double cT = cR * a.R_inv, aT = aR * a.R_inv;
    double rhs[D + 2];
    double Sm = 0.0;
#pragma unroll
    for (int k = 0; k < D; k++) Sm += S[k] * S[k];
    Sm = sqrt(Sm);

    if (SOLVER == 0) {
        const Prim64<D> sp = prim64<D, 0>(a, qP), sn = prim64<D, 0>(a, qN);
        flux_m1<D>(qP, sp, qN, sn, S, Sm, w, 1.0 - w, rhs);
    } else {
        const double rhoavg = 0.5 * (qP[0] + qN[0]);
        double rUa[D];
#pragma unroll
        for (int k = 0; k < D; k++) rUa[k] = 0.5 * (qP[k + 1] + qN[k + 1]);
        const double Ravg = 0.5 * (cR + aR);
        double pavg = rhoavg * Ravg;
        const double cH = qP[D + 1] / qP[0] + cR;
        const double aH = qN[D + 1] / qN[0] + aR;
        const double Havg = 0.5 * (cH + aH);
        if (SOLVER == 2) {
            const double cP = sqrt(a.gamma * cR), cN = sqrt(a.gamma * aR);
            const double cavg = 0.5 * (cP + cN);
            double cdiv = 0, ndiv = 0, ccurl = 0, ncurl = 0, cvm = 0, nvm = 0, unP = 0, unN = 0, nrm = 0;
            double cdu[D][D], ndu[D][D];
#pragma unroll
            for (int i = 0; i < D; i++)
#pragma unroll
                for (int j = 0; j < D; j++) {
                    cdu[i][j] = gr[0][i * D + j];
                    ndu[i][j] = gr[1][i * D + j];
                }
#pragma unroll
            for (int p = 0; p < D; p++) {
                cdiv += cdu[p][p];
                ndiv += ndu[p][p];
#pragma unroll
                for (int b = p + 1; b < D; b++) {
                    ccurl += (cdu[p][b] - cdu[b][p]) * (cdu[p][b] - cdu[b][p]);
                    ncurl += (ndu[p][b] - ndu[b][p]) * (ndu[p][b] - ndu[b][p]);
                }
                const double cu = qP[p + 1] / qP[0];
                cvm += cu * cu;
                const double nu = qN[p + 1] / qN[0];
                nvm += nu * nu;
                double gc[D], gn[D];
#pragma unroll
                for (int k = 0; k < D; k++) {
                    gc[k] = gr[0][R::kUG + p * D + k];
                    gn[k] = gr[1][R::kUG + p * D + k];
                }
                const double uPos = interp_minmod<D>(cu, nu, gc, d, w, 1.0);
                const double uNeg = interp_minmod<D>(cu, nu, gn, d, w, -1.0);
                unP += uPos * S[p];
                unN += uNeg * S[p];
                nrm += S[p] * S[p];
            }
            const double cth0 = -(cdiv / sqrt(cdiv * cdiv + ccurl + 4e-2));
            const double nth0 = -(ndiv / sqrt(ndiv * ndiv + ncurl + 4e-2));
            const double cth = (cth0 < 0.) ? 0. : cth0;
            const double nth = (nth0 < 0.) ? 0. : nth0;
            const double tha = 0.5 * (cth + nth);
            double r = qP[0], E = qP[D + 1] / r;
            const double cp_ = r * a.gm1 * (E - 0.5 * cvm);
            r = qN[0];
            E = qN[D + 1] / r;
            const double np_ = r * a.gm1 * (E - 0.5 * nvm);
            double gc[D], gn[D], hc[D], hn[D];
#pragma unroll
            for (int k = 0; k < D; k++) {
                gc[k] = gr[0][R::kRG + k];
                gn[k] = gr[1][R::kRG + k];
                hc[k] = gr[0][R::kPG + k];
                hn[k] = gr[1][R::kPG + k];
            }
            const double rhoP = interp_minmod<D>(qP[0], qN[0], gc, d, w, 1.0);
            const double rhoN = interp_minmod<D>(qP[0], qN[0], gn, d, w, -1.0);
            const double pP = interp_minmod<D>(cp_, np_, hc, d, w, 1.0);
            const double pN = interp_minmod<D>(cp_, np_, hn, d, w, -1.0);
            const double Msq = (unP * unP + unN * unN) / (2. * cavg * cavg * nrm);
            const double MP = unP / (sqrt(nrm) * cavg);
            const double MN = unN / (sqrt(nrm) * cavg);
            const double Minf = 0.2;
            const double mx = (Msq < Minf * Minf) ? Minf * Minf : Msq;
            const double M0 = sqrt((mx < 1.0) ? mx : 1.0);
            const double fa = M0 * (2.0 - M0);
            const double alpha = 3.0 * (5.0 * fa * fa - 4.0) / 16.0;
            const double phalf = pN * (p5pos(MN, alpha) - p5neg(MN, alpha)) - pP * (p5pos(MP, alpha) - p5neg(MP, alpha));
            const double pu = -0.75 * p5pos(MP, alpha) * p5neg(MN, alpha) * (rhoP + rhoN) * cavg * fa * (unN - unP);
            pavg += tha * (pu - 0.5 * phalf);
        }
        flux_m2<D>(rhoavg, rUa, Havg, pavg, S, rhs);
    }

    // viscous terms (cfd_v0.cpp:2682-2790)
    if (VISC) {
    const double mu = a.mu;
    double dmag = 0.0;
#pragma unroll
    for (int k = 0; k < D; k++) dmag += d[k] * d[k];
    dmag = sqrt(dmag);
    const double dmi = 1.0 / dmag;
    double dn[D], du[D][D], dT[D], tau[D][D], tmc[D][D];
    double duP[D][D], duN[D][D], sUP[D], sUN[D];
#pragma unroll
    for (int k = 0; k < D; k++) dn[k] = d[k] * dmi;
    if (ghost) {
#pragma unroll
        for (int i = 0; i < D; i++) {
#pragma unroll
            for (int j = 0; j < D; j++) du[i][j] = (aU[i] - cU[i]) * dn[j] * dmi;
            dT[i] = (aT - cT) * dn[i] * dmi;
        }
    } else {
#pragma unroll
        for (int i = 0; i < D; i++) {
#pragma unroll
            for (int j = 0; j < D; j++) {
                duP[i][j] = gr[0][i * D + j];
                duN[i][j] = gr[1][i * D + j];
                du[i][j] = INTERP_LINEAR(w, duP[i][j], duN[i][j]);
            }
            dT[i] = INTERP_LINEAR(w, gr[0][R::kDT + i], gr[1][R::kDT + i]);
        }
    }
#pragma unroll
    for (int p = 0; p < D; p++) {
        tau[p][p] = 2.0 * du[p][p];
#pragma unroll
        for (int b1 = p + 1; b1 < D + p; b1++) {
            const int b = b1 % D;
            tau[p][b] = mu * (du[p][b] + du[b][p]);
            tau[p][p] -= du[b][b];
        }
        tau[p][p] *= 2.0 / 3.0 * mu;
    }
    const double kcond = a.cp * mu * a.pr_inv;
    if (ghost) {
        double diag = 0;
#pragma unroll
        for (int p = 0; p < D; p++) diag -= du[p][p];
        diag *= mu * 2.0 / 3.0;
#pragma unroll
        for (int i = 0; i < D; i++) {
#pragma unroll
            for (int j = 0; j < D; j++) tmc[i][j] = mu * du[j][i];
            tmc[i][i] += diag;
        }
    } else if constexpr (STORED) {
#pragma unroll
        for (int i = 0; i < D; i++)
#pragma unroll
            for (int j = 0; j < D; j++)
                tmc[i][j] = INTERP_LINEAR(w, a.tauMC[(i * D + j) * nt + P], a.tauMC[(i * D + j) * nt + N]);
    } else {
        // both cells' tensors as calc_VIS leaves them, from their dudx
        double tP[D][D], tN[D][D];
        vis_tensors<D>(a, duP, qP, a.smag ? a.smag + P : nullptr, tP, sUP);
        vis_tensors<D>(a, duN, qN, a.smag ? a.smag + N : nullptr, tN, sUN);
#pragma unroll
        for (int i = 0; i < D; i++)
#pragma unroll
            for (int j = 0; j < D; j++) tmc[i][j] = INTERP_LINEAR(w, tP[i][j], tN[i][j]);
    }
    const double Sd = dotD<D>(S, d);
    double delta[D], K[D], dm = 0.0;
#pragma unroll
    for (int i = 0; i < D; i++) {
        delta[i] = d[i] * Sm * Sm / Sd;
        dm += delta[i] * delta[i];
        K[i] = S[i] - delta[i];
    }
    dm = sqrt(dm);
    double sU[D];
    if (ghost) {
        double Uf[D];
#pragma unroll
        for (int i = 0; i < D; i++) Uf[i] = INTERP_LINEAR(w, cU[i], aU[i]);
#pragma unroll
        for (int i = 0; i < D; i++) sU[i] = dotD<D>(Uf, tau[i]);
    } else if constexpr (STORED) {
#pragma unroll
        for (int i = 0; i < D; i++) sU[i] = INTERP_LINEAR(w, a.sigmaU[i * nt + P], a.sigmaU[i * nt + N]);
    } else {
#pragma unroll
        for (int i = 0; i < D; i++) sU[i] = INTERP_LINEAR(w, sUP[i], sUN[i]);
    }
#pragma unroll
    for (int i = 0; i < D; i++) {
        const double divT = dotD<D>(tmc[i], S);
        const double lapU = mu * (dm * (aU[i] - cU[i]) * dmi + dotD<D>(K, du[i]));
        rhs[i + 1] += divT + lapU;
    }
    const double lapT = kcond * (dm * (aT - cT) * dmi + dotD<D>(K, dT));
    rhs[D + 1] += dotD<D>(sU, S) + lapT;
    }
    st64x2_once<NT>(a.frhs + 4 * (size_t)f, rhs[0], rhs[1]);
    st64x2_once<NT>(a.frhs + 4 * (size_t)f + 2, rhs[2], rhs[3]);
    if (D == 3) st_once<NT>(a.frhs + (size_t)4 * a.nf + f, rhs[D + 1]);
}

// tauMC and sigmaU of every cell from the stored dudx (field read-back of a
// solver that does not store them): [D*D][nc] and [D][nc]
template <int D>
__global__ void __launch_bounds__(256) vis_tensor_field(KArgs a, double *tmc_out, double *sU_out) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= a.nc) return;
    double du[D][D], q[D + 2], tmc[D][D], sU[D];
#pragma unroll
    for (int i = 0; i < D; i++)
#pragma unroll
        for (int j = 0; j < D; j++) du[i][j] = a.dudx[(size_t)c * a.gstride + i * D + j];
    load_q<D>(a, c, q);
    vis_tensors<D>(a, du, q, a.smag ? a.smag + c : nullptr, tmc, sU);
#pragma unroll
    for (int i = 0; i < D; i++) {
        sU_out[(size_t)i * a.nc + c] = sU[i];
#pragma unroll
        for (int j = 0; j < D; j++) tmc_out[(size_t)(i * D + j) * a.nc + c] = tmc[i][j];
    }
}

// dt_c (MODE 0) or cfl_c (MODE 1) from a cell's sum over its faces, combined
// with the block's starting value
template <int D, int MODE>
__device__ __forceinline__ double cfl_value64(const double rho, const double vinv, const double sum,
                                              const double param) {
    double v = MODE == 0 ? 100.0 : 0.0;
    if (MODE == 0) {
        const double vol = 1.0 / vinv;
        const double dtc = param * rho * 2.0 * vol / sum;
        if (v > dtc) v = dtc;
    } else {
        const double cfl = sum * ((1.0 / rho) * vinv * param);
        if (v < cfl) v = cfl;
    }
    return v;
}

// ---------------------------------------------------------------------------
// compute_dt / compute_cfl (cfd_v0.cpp:2887-2942) of one cell from its state
// q: the sum over its faces in slot order, then dt_c (MODE 0) or cfl_c
// (MODE 1).  Returns the block's starting value combined with it, so a NaN
// never wins (as `dt_min > dt`).
// ---------------------------------------------------------------------------
template <int D, int MODE>
__device__ __forceinline__ double cfl_cell(const KArgs &a, const int c, const double (&q)[D + 2], double param) {
    double sum = 0.0;
    auto add = [&](const double (&S)[D]) {
        if (MODE == 0) {
            double sM = 0.0;
#pragma unroll
            for (int k = 0; k < D; k++) sM += S[k] * S[k];
            sM = sqrt(sM);
            double fl = 0.0;
#pragma unroll
            for (int k = 0; k < D; k++) fl += q[k + 1] * S[k] / sM;
            sum += fabs(fl);
        } else {
            double fl = 0.0;
#pragma unroll
            for (int k = 0; k < D; k++) fl += q[k + 1] * S[k];
            sum += fabs(fl);
        }
    };
    // slot-ordered sum; the first slots' area vectors fetched together
    // (slot lists carry no ghost flag)
    const int e0 = a.s_off[c], ne = a.s_off[c + 1] - e0;
    constexpr int U = GatherUnroll<D>::value;
    double Sj[U][D];
#pragma unroll
    for (int j = 0; j < U; j++) {
        const int ent = a.s_ent[e0 + (j < ne ? j : ne - 1)];
        const int f = ent >= 0 ? ent : ~ent;
        double sf[D];
        load_S64<D>(a.S, f, sf);
#pragma unroll
        for (int k = 0; k < D; k++) Sj[j][k] = ent >= 0 ? sf[k] : -sf[k];
    }
#pragma unroll
    for (int j = 0; j < U; j++)
        if (j < ne) add(Sj[j]);
    for (int e = e0 + U; e < e0 + ne; e++) {
        const int ent = a.s_ent[e];
        const int f = ent >= 0 ? ent : ~ent;
        double S[D];
        double sf[D];
        load_S64<D>(a.S, f, sf);
#pragma unroll
        for (int k = 0; k < D; k++) S[k] = ent >= 0 ? sf[k] : -sf[k];
        add(S);
    }
    return cfl_value64<D, MODE>(q[0], a.vinv[c], sum, param);
}

// Block-wide min (MODE 0) / max (MODE 1) of v into *dst; every thread of the
// block calls it.  The values are never NaN, so min / max are exact in any
// order.
template <int MODE>
__device__ __forceinline__ void block_extremum(double v, double *dst) {
    __shared__ double ext[256 / 64];
    auto pick = [](double x, double o) {
        if (MODE == 0) return x > o ? o : x;
        return x < o ? o : x;
    };
    for (int off = 32; off > 0; off >>= 1) v = pick(v, __shfl_down(v, off, 64));
    if ((threadIdx.x & 63) == 0) ext[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = ext[0];
        for (int i = 1; i < (int)(blockDim.x >> 6); i++) r = pick(r, ext[i]);
        *dst = r;
    }
}

// How a stage treats the RK register: zero before it (a step's first stage),
// and not stored after it (the last stage of a step that another follows in the
// same call: nothing reads it before that step starts from zero; 20 of 108 B per
// 3D FP32 cell and stage).  Looked at only by the launches that form the CFL as
// well, which a step's last stage is: the choice costs 0.1 us.
constexpr int kDqZero = 1, kDqDrop = 2;
// the cell's RK register as the last stage left it, zero at a step's first
// stage: every component's load issued before any is used (a choice per
// component compiles to a branch and a wait each)
template <int D, bool NT>
__device__ __forceinline__ void load_dq64(const KArgs &a, const int dq_mode, const int c, double (&dq)[D + 2]) {
#pragma unroll
    for (int k = 0; k < D + 2; k++) dq[k] = 0.0;
    if (!(dq_mode & kDqZero)) {
#pragma unroll
        for (int k = 0; k < D + 2; k++) dq[k] = ld_once<NT>(a.dq + (size_t)k * a.nc + c);
    }
}

// the sponge term of one cell (cfd_v0.cpp:2808-2811)
template <int D, bool NT>
__device__ __forceinline__ void sponge64(const KArgs &a, const int c, const double dt, const double (&q)[D + 2],
                                         double (&dq)[D + 2]) {
    const double sg = ld_once<NT>(a.sigma + c);
    dq[0] += dt * sg * (a.rho_inf - q[0]);
#pragma unroll
    for (int k = 0; k < D; k++) dq[k + 1] += dt * sg * (a.rho_inf * a.U_inf[k] - q[k + 1]);
    dq[D + 1] += dt * sg * (a.rho_inf * a.E_inf - q[D + 1]);
}

// ---------------------------------------------------------------------------
// Residual gather, sponge, RK update (cfd_v0.cpp:2792-2822).  dq starts from
// A_rk * dq (prepare_for_RKstep); dq_mode replaces it by 0 for the first
// stage of a step (prepare_for_timestep zeroed it).  CFL >= 0 (the last
// stage of a step): the step's compute_dt (0) / compute_cfl (1) of the
// updated cells, per-block extrema into a.partial.
// ---------------------------------------------------------------------------
template <int D, bool RES, int CFL, bool NT>
__global__ void __launch_bounds__(256) cell_update(KArgs a, double A, double B, int dq_mode, double cfl_param) {
    static_assert(!(RES && CFL >= 0), "the residual and the CFL share a.partial");
    const int c = LFM_TID(blockIdx.x);
    __shared__ double red[256 / 64][D + 2];
    double cv = CFL == 0 ? 100.0 : 0.0;
    double rsq[D + 2];
#pragma unroll
    for (int k = 0; k < D + 2; k++) rsq[k] = 0.0;
    if (c < a.nc) {
        const double dt = *a.dt;
        const double vinv = ld_once<NT>(a.vinv + c);
        double dq[D + 2], res[D + 2], q[D + 2];
        load_dq64<D, NT>(a, dq_mode, c, dq);
#pragma unroll
        for (int k = 0; k < D + 2; k++) res[k] = 0.0;
        // in 3D the state is asked for after the fluxes, which it would only queue
        // before (O-grid, us of updates per step with it first / last: 4.2 M cells
        // 1530 / 1477, 1 M 381 / 368, 193 k 84 / 81)
        if constexpr (D == 2) load_q<D>(a, c, q);
        constexpr int U = GatherUnroll<D>::value;
        int key[U];
        load_keys<D, NT>(a.g_key, a.nc, 0, c, key);
        unsigned gmask = 0;  // bit j: entry j leads to a boundary ghost
        // owner side adds, neighbour side subtracts (cfd_v0.cpp:2800-2806)
        auto add = [&](const int j, const int ent, const double (&fr)[D + 2]) {
            if (ent >= 0) {
                if (ent & kGhostFaceFlag) gmask |= 1u << j;
#pragma unroll
                for (int k = 0; k < D + 2; k++) {
                    if (RES) res[k] += fr[k];
                    dq[k] += dt * fr[k] * vinv;
                }
            } else {
#pragma unroll
                for (int k = 0; k < D + 2; k++) {
                    if (RES) res[k] -= fr[k];
                    dq[k] -= dt * fr[k] * vinv;
                }
            }
        };
        // the first faces' fluxes fetched together, then added in gather order
        double fr[U][D + 2];
#pragma unroll
        for (int j = 0; j < U; j++) load_frhs<D>(a, face_of(key[j]), fr[j]);
#pragma unroll
        for (int k = 0; k < D + 2; k++) dq[k] *= A;
#pragma unroll
        for (int j = 0; j < U; j++)
            if (key[j] != kNoFace) add(j, key[j], fr[j]);
        int e1 = 0, ne = 0;  // entries beyond the first U
        if (a.more_faces) {
            e1 = a.g_off[c] + U;
            ne = a.g_off[c + 1] - e1;
            for (int j = 0; j < ne; j++) {
                const int ent = a.g_ent[e1 + j];
                double f1[D + 2];
                load_frhs<D>(a, face_of(ent), f1);
                add(U + j, ent, f1);
            }
        }
        if constexpr (D == 3) load_q<D>(a, c, q);
        if (a.sigma) sponge64<D, NT>(a, c, dt, q, dq);
#pragma unroll
        for (int k = 0; k < D + 2; k++) q[k] += B * dq[k];
        store_q<D, NT>(a.q, a.ntot, c, q);
        if (CFL < 0 || !(dq_mode & kDqDrop))
#pragma unroll
            for (int k = 0; k < D + 2; k++) st_once<NT>(a.dq + (size_t)k * a.nc + c, dq[k]);
        // refresh this cell's boundary ghosts for the next stage
        for (unsigned m = gmask; m; m &= m - 1) {
            const int j = __builtin_ctz(m);
            const int ent = j < U ? a.g_key[key_at<D>(a.nc, j, c)] : a.g_ent[e1 + j - U];
            const int g = a.fN[ent & kFaceMask] - a.nc;
            double qg[D + 2];
            if (!ghost_state<D>(a, a.ghost_role[g], q, qg)) continue;
            store_q<D, NT>(a.q, a.ntot, a.nc + g, qg);
        }
        if constexpr (CFL >= 0) cv = cfl_cell<D, CFL>(a, c, q, cfl_param);
        if (RES) {
#pragma unroll
            for (int k = 0; k < D + 2; k++) {
                a.res_cell[(size_t)k * a.nc + c] = res[k];
                rsq[k] = res[k] * res[k];
            }
        }
    }
    if (RES) {
        // per-block partial sums of squared residuals (fixed order)
        const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
        for (int k = 0; k < D + 2; k++) {
            double v = rsq[k];
            for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
            if (lane == 0) red[wid][k] = v;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
#pragma unroll
            for (int k = 0; k < D + 2; k++) {
                double s = 0.0;
                for (int i = 0; i < (int)(blockDim.x >> 6); i++) s += red[i][k];
                a.partial[(size_t)LFM_BLK() * (D + 2) + k] = s;
            }
        }
    }
    if constexpr (CFL >= 0) block_extremum<CFL>(cv, a.partial + LFM_BLK());
}

// Sum of per-block partials in fixed order, one block; all components go down
// the tree together (one after the other took 5.1 us for 256 partials of four).
static __global__ void __launch_bounds__(256) reduce_sum(const double *partial, int nblk, int ncomp, double *out, int accumulate) {
    constexpr int kMax = 5;
    __shared__ double sh[kMax][256];
    const int t = threadIdx.x;
    double v[kMax];
#pragma unroll
    for (int k = 0; k < kMax; k++) v[k] = 0.0;
    for (int i = t; i < nblk; i += 256) {
#pragma unroll
        for (int k = 0; k < kMax; k++)
            if (k < ncomp) v[k] += partial[(size_t)i * ncomp + k];
    }
#pragma unroll
    for (int k = 0; k < kMax; k++) sh[k][t] = v[k];
    for (int st = 128; st >= 64; st >>= 1) {
        __syncthreads();
        if (t < st) {
#pragma unroll
            for (int k = 0; k < kMax; k++) sh[k][t] = v[k] = sh[k][t] + sh[k][t + st];
        }
    }
    if (t >= 64) return;
    for (int st = 32; st > 0; st >>= 1) {
#pragma unroll
        for (int k = 0; k < kMax; k++) v[k] += __shfl_down(v[k], st, 64);
    }
    if (t == 0) {
#pragma unroll
        for (int k = 0; k < kMax; k++)
            if (k < ncomp) out[k] = accumulate ? out[k] + v[k] : v[k];
    }
}

// ---------------------------------------------------------------------------
// compute_dt / compute_cfl (cfd_v0.cpp:2887-2942) as their own launch: per
// cell over its faces in slot order, then min / max.  MODE 0: dt (min, start
// 100), 1: cfl (max, start 0).
// ---------------------------------------------------------------------------
template <int D, int MODE>
__global__ void __launch_bounds__(256) cfl_dt_cells(KArgs a, double param) {
    const int c = LFM_TID(blockIdx.x);
    double v = MODE == 0 ? 100.0 : 0.0;
    if (c < a.nc) {
        double q[D + 2];
        load_q<D>(a, c, q);
        v = cfl_cell<D, MODE>(a, c, q, param);
    }
    block_extremum<MODE>(v, a.partial + LFM_BLK());
}

// Final min / max over the per-block values by one block of NT threads,
// each with 16 loads in flight per round, so the latency of a few rounds
// (65 536 partials on 16.8 M cells: 4 with 1024 threads) bounds it rather
// than a long dependent chain.  Min / max are exact in any order.
template <int MODE, int NT>
__device__ __forceinline__ void cfl_dt_final_block(const double *partial, int nblk, double *out, double *dt_dst) {
    auto pick = [](double x, double o) {
        if (MODE == 0) return x > o ? o : x;
        return x < o ? o : x;
    };
    constexpr int kLoads = 16;
    double v = MODE == 0 ? 100.0 : 0.0;
    for (int i0 = 0; i0 < nblk; i0 += kLoads * NT) {
        double o[kLoads];
#pragma unroll
        for (int j = 0; j < kLoads; j++) {
            const int i = i0 + j * NT + (int)threadIdx.x;
            o[j] = i < nblk ? partial[i] : v;
        }
#pragma unroll
        for (int j = 0; j < kLoads; j++) v = pick(v, o[j]);
    }
    for (int off = 32; off > 0; off >>= 1) v = pick(v, __shfl_down(v, off, 64));
    __shared__ double w[NT / 64];
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = w[0];
        for (int i = 1; i < NT / 64; i++) r = pick(r, w[i]);
        *out = r;
        if (dt_dst) *dt_dst = r;
    }
}

// ---------------------------------------------------------------------------
// One RK stage of the inviscid M1 / M2 schemes in one launch: each cell forms
// its faces' fluxes from its own and the other cells' states as it gathers
// them (every interior face by both of its cells, to the same bits), adds
// sponge and RK update and writes the new state and its boundary ghosts to
// qout, another buffer.  The face fluxes' round trip through memory (write,
// two gathered reads: 120 B of the 773 B per 3D cell and stage that the face
// and update launches move) and the second read of the states are gone.
// PK: the face's area vector and weights come from the geometry table, 4 B
// per slot instead of 36: a uniform mesh has a few dozen distinct records,
// which stay in the L1 caches.
// ---------------------------------------------------------------------------
// Faces whose loads are issued together: two leave 126 VGPRs and 4 waves per
// SIMD (3D box of 1.4 M cells: one 495, two 485, three 526 us per step).
constexpr int kFusedGroup64 = 2;
// geometry table record: S out of the cell [D], |S|, wc, wo, padded to whole
// 16-byte words (6 doubles in 2D and 3D)
constexpr int kTabRec64 = 6;

// the face data of gather entry j of cell c as that cell sees them; key: the
// packed word, or the slot's key
template <int D, bool PK, bool NT>
struct FaceOf64 {
    int other;
    double S[D], Sm, wc, wo;
    __device__ __forceinline__ static int load_key(const KArgs &a, const int j, const int c) {
        const size_t i = slot_at<D, 1>(a.nc, j, 0, c);
        if constexpr (PK) return (int)ld_once<NT>(a.pk + i);
        return ld_once<NT>(a.sl_nb + i);
    }
    __device__ __forceinline__ static int other_of(const KArgs &a, const int key) {
        if constexpr (PK) return (int)((uint32_t)key & ((1u << a.pk_shift) - 1u));
        return key >= 0 ? key : ~key;
    }
    // geometry of a face stored with P's orientation
    __device__ __forceinline__ void from_face(const bool isP, const double (&s)[D], const double w) {
        double m = 0.0;
#pragma unroll
        for (int k = 0; k < D; k++) {
            m += s[k] * s[k];
            S[k] = isP ? s[k] : -s[k];
        }
        Sm = sqrt(m);
        const double omw = 1.0 - w;
        wc = isP ? w : omw;
        wo = isP ? omw : w;
    }
    __device__ __forceinline__ void load(const KArgs &a, const int j, const int c, const int key) {
        other = other_of(a, key);
        if constexpr (PK) {
            const double2 *p =
                reinterpret_cast<const double2 *>(a.pk_tab + (size_t)((uint32_t)key >> a.pk_shift) * kTabRec64);
            const double2 v0 = p[0], v1 = p[1], v2 = p[2];
            const double r[6] = {v0.x, v0.y, v1.x, v1.y, v2.x, v2.y};
#pragma unroll
            for (int k = 0; k < D; k++) S[k] = r[k];
            Sm = r[D];
            wc = r[D + 1];
            wo = r[D + 2];
        } else {
            double s[D];
#pragma unroll
            for (int k = 0; k < D; k++) s[k] = ld_once<NT>(a.sl_S + slot_at<D, D>(a.nc, j, k, c));
            from_face(key >= 0, s, ld_once<NT>(a.sl_w + slot_at<D, 1>(a.nc, j, 0, c)));
        }
    }
    // an entry of the gather list (beyond the slots)
    __device__ __forceinline__ void load_list(const KArgs &a, const int ent) {
        const bool isP = ent >= 0;
        const int f = isP ? (ent & kFaceMask) : ~ent;
        other = isP ? a.fN[f] : a.fP[f];
        double s[D];
        load_S64<D>(a.S, f, s);
        from_face(isP, s, a.w[f]);
    }
};

template <int D, int SOLVER, bool SYM>
__device__ __forceinline__ void own_flux64(const KArgs &a, const double (&qc)[D + 2], const Prim64<D> &sc,
                                           const double (&qo)[D + 2], const double (&S)[D], const double Sm,
                                           const double wc, const double wo, double (&r)[D + 2]) {
    const Prim64<D> so = prim64<D, SOLVER>(a, qo);
    if constexpr (SOLVER == 0) {
        SYM ? flux_m1_sym<D>(qc, sc, qo, so, S, Sm, wc, wo, r) : flux_m1<D>(qc, sc, qo, so, S, Sm, wc, wo, r);
    } else {
        const double rhoavg = 0.5 * (qc[0] + qo[0]);
        double rUa[D];
#pragma unroll
        for (int k = 0; k < D; k++) rUa[k] = 0.5 * (qc[k + 1] + qo[k + 1]);
        const double Ravg = 0.5 * (sc.R + so.R);
        const double Havg = 0.5 * (sc.e + so.e);
        flux_m2<D>(rhoavg, rUa, Havg, rhoavg * Ravg, S, r);
    }
}

// |m.S| (MODE 1) or |m.S| / |S| (MODE 0) of one face, as cfl_cell forms it
template <int D, int MODE>
__device__ __forceinline__ double cfl_term64(const double (&q)[D + 2], const double (&S)[D], const double Sm) {
    double fl = 0.0;
#pragma unroll
    for (int k = 0; k < D; k++) fl += MODE == 0 ? q[k + 1] * S[k] / Sm : q[k + 1] * S[k];
    return fabs(fl);
}

// fin_nblk > 0 (a stage without CFL/dt sums): one block more, the last,
// reduces the fin_nblk per-block CFL maxima that the previous step's last
// stage left in a.partial into *fin_out.
// SYM: every face's weights allow flux_m1_sym.
template <int D, int SOLVER, int CFL, bool PK, bool SYM, bool NT>
__global__ void __launch_bounds__(256) stage_fused64(KArgs a, double *qout, double A, double B, int dq_mode,
                                                     double cfl_param, int fin_nblk, double *fin_out) {
    int nb = (int)gridDim.x;
    if constexpr (CFL < 0) {
        if (fin_nblk > 0) {
            nb -= 1;
            if ((int)blockIdx.x == nb) {
                cfl_dt_final_block<1, 256>(a.partial, fin_nblk, fin_out, nullptr);
                return;
            }
        }
    }
    constexpr int U = GatherUnroll<D>::value;
    using F = FaceOf64<D, PK, NT>;
    const int blk = xcd_block((int)blockIdx.x, nb);
    const int c = blk * (int)blockDim.x + (int)threadIdx.x;
    double cv = CFL == 0 ? 100.0 : 0.0;
    // the CFL/dt terms of a cell's faces in slot order (own thread only)
    __shared__ double terms[CFL >= 0 ? kMaxFaces * 256 : 1];
    // and in 3D its keys, kept for them: read again they come from memory (1.4
    // M-cell box: 89 -> 85 us per launch; in 2D it gains nothing)
    constexpr bool kKeepKey = CFL >= 0 && D == 3;
    __shared__ int keys[kKeepKey ? GatherUnroll<D>::value * 256 : 1];
    if (c < a.nc) {
        constexpr int G = kFusedGroup64;
        int key[G];
#pragma unroll
        for (int u = 0; u < G; u++) key[u] = F::load_key(a, u, c);
        double qc[D + 2], dq[D + 2];
        load_q<D>(a, c, qc);
        const double vinv = ld_once<NT>(a.vinv + c);
        load_dq64<D, NT>(a, dq_mode, c, dq);
        const double dt = *a.dt;
        const Prim64<D> sc = prim64<D, SOLVER>(a, qc);
        unsigned gmask = 0;  // bit j: slot j leads to a boundary ghost
        // a rolled loop over groups of G faces, the next group's keys loaded a
        // group ahead: unrolled, the compiler gathers all faces' loads at the
        // top and spills
#pragma unroll 1
        for (int j0 = 0; j0 < U; j0 += G) {
            F f[G];
            double qo[G][D + 2];
            int next[G];
#pragma unroll
            for (int u = 0; u < G; u++) {
                if constexpr (kKeepKey) keys[(j0 + u) * 256 + threadIdx.x] = key[u];
                f[u].load(a, j0 + u, c, key[u]);
                load_q<D>(a, f[u].other, qo[u]);
                next[u] = F::load_key(a, j0 + G < U ? j0 + G + u : u, c);
            }
            if (j0 == 0)
#pragma unroll
                for (int k = 0; k < D + 2; k++) dq[k] *= A;
#pragma unroll
            for (int u = 0; u < G; u++) {
                if (f[u].other != c) {
                    double r[D + 2];
                    own_flux64<D, SOLVER, SYM>(a, qc, sc, qo[u], f[u].S, f[u].Sm, f[u].wc, f[u].wo, r);
                    gmask |= f[u].other >= a.nc ? 1u << (j0 + u) : 0u;
#pragma unroll
                    for (int k = 0; k < D + 2; k++) dq[k] += dt * r[k] * vinv;
                }
                key[u] = next[u];
            }
        }
        int e1 = 0, e2 = 0;  // gather entries beyond the slots
        if (U < kMaxFaces && a.more_faces) {
            e1 = a.g_off[c] + U;
            e2 = a.g_off[c + 1];
            for (int e = e1; e < e2; e++) {
                F f;
                f.load_list(a, a.g_ent[e]);
                double qo[D + 2], r[D + 2];
                load_q<D>(a, f.other, qo);
                own_flux64<D, SOLVER, false>(a, qc, sc, qo, f.S, f.Sm, f.wc, f.wo, r);
                gmask |= f.other >= a.nc ? 1u << (U + e - e1) : 0u;
#pragma unroll
                for (int k = 0; k < D + 2; k++) dq[k] += dt * r[k] * vinv;
            }
        }
        double q[D + 2];
#pragma unroll
        for (int k = 0; k < D + 2; k++) q[k] = qc[k];
        if (a.sigma) sponge64<D, NT>(a, c, dt, q, dq);
#pragma unroll
        for (int k = 0; k < D + 2; k++) q[k] += B * dq[k];
        store_q<D, NT>(qout, a.ntot, c, q);
        if (CFL < 0 || !(dq_mode & kDqDrop))
#pragma unroll
            for (int k = 0; k < D + 2; k++) st_once<NT>(a.dq + (size_t)k * a.nc + c, dq[k]);
        // this cell's boundary ghosts for the next stage
        for (unsigned m = gmask; m; m &= m - 1) {
            const int j = __builtin_ctz(m);
            int g;
            if (U >= kMaxFaces || j < U) {
                g = F::other_of(a, F::load_key(a, j, c));
            } else {
                g = a.fN[a.g_ent[e1 + j - U] & kFaceMask];
            }
            double qg[D + 2];
            if (!ghost_state<D>(a, a.ghost_role[g - a.nc], q, qg)) load_q<D>(a, g, qg);
            store_q<D, NT>(qout, a.ntot, g, qg);
        }
        if constexpr (CFL >= 0) {
            const int perm = a.s_perm[c];
#pragma unroll
            for (int j = 0; j < U; j++) {
                F f;
                f.load(a, j, c, kKeepKey ? keys[j * 256 + threadIdx.x] : F::load_key(a, j, c));
                if (f.other != c)
                    terms[((perm >> (3 * j)) & 7) * 256 + threadIdx.x] = cfl_term64<D, CFL>(q, f.S, f.Sm);
            }
            for (int e = e1; U < kMaxFaces && e < e2; e++) {
                F f;
                f.load_list(a, a.g_ent[e]);
                terms[((perm >> (3 * (U + e - e1))) & 7) * 256 + threadIdx.x] = cfl_term64<D, CFL>(q, f.S, f.Sm);
            }
            const int n = (perm >> 18) & 7;
            double sum = 0.0;
            for (int j = 0; j < n; j++) sum += terms[j * 256 + threadIdx.x];
            cv = cfl_value64<D, CFL>(q[0], vinv, sum, cfl_param);
        }
    }
    if constexpr (CFL >= 0) block_extremum<CFL>(cv, a.partial + blk);
}

// the one-launch stage's slots from the gather list and, with face_rec, each
// face's record number in the geometry table (2 face_rec + 1 from the N side;
// none: a placeholder's record)
template <int D>
__global__ void __launch_bounds__(256) build_slots64(KArgs a, const uint16_t *face_rec, int none, uint32_t *pk,
                                                     int32_t *nb, double *S, double *w, int32_t *perm) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= a.nc) return;
    const int e0 = a.g_off[c], ne = a.g_off[c + 1] - e0;
    const int s0 = a.s_off[c], ns = a.s_off[c + 1] - s0;
    int p = ns << 18;
    for (int j = 0; j < ne && j < kMaxFaces; j++) {
        const int ent = a.g_ent[e0 + j];
        const int bare = ent >= 0 ? (ent & kFaceMask) : ent;
        for (int i = 0; i < ns; i++)
            if (a.s_ent[s0 + i] == bare) p |= i << (3 * j);
    }
    perm[c] = p;
    constexpr int U = GatherUnroll<D>::value;
    for (int j = 0; j < U; j++) {
        const size_t i1 = slot_at<D, 1>(a.nc, j, 0, c);
        if (j >= ne) {
            // placeholder past the cell's last entry: the cell itself, unit
            // area (read by unbranched gathers, never added)
            if (pk) {
                pk[i1] = (uint32_t)c | (uint32_t)none << a.pk_shift;
            } else {
                nb[i1] = c;
                for (int k = 0; k < D; k++) S[slot_at<D, D>(a.nc, j, k, c)] = 1.0;
                w[i1] = 0.5;
            }
            continue;
        }
        const int ent = a.g_ent[e0 + j];
        const int f = ent >= 0 ? (ent & kFaceMask) : ~ent;
        const int o = ent >= 0 ? a.fN[f] : a.fP[f];
        if (pk) {
            pk[i1] = (uint32_t)o | (uint32_t)(2 * face_rec[f] + (ent >= 0 ? 0 : 1)) << a.pk_shift;
        } else {
            nb[i1] = ent >= 0 ? o : ~o;
            for (int k = 0; k < D; k++) S[slot_at<D, D>(a.nc, j, k, c)] = a.S[(size_t)f * D + k];
            w[i1] = a.w[f];
        }
    }
}

// the final reduction as a launch of its own: one block of kFinalBlock
constexpr int kFinalBlock = 1024;
template <int MODE>
static __global__ void __launch_bounds__(kFinalBlock) cfl_dt_final(const double *partial, int nblk, double *out,
                                                                  double *dt_dst) {
    cfl_dt_final_block<MODE, kFinalBlock>(partial, nblk, out, dt_dst);
}

// conservation integrals sum_c V_c q_c, per-block partials (FP64)
template <int D>
__global__ void __launch_bounds__(256) integrals64(KArgs a) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    __shared__ double red[256 / 64][D + 2];
    double v[D + 2];
#pragma unroll
    for (int k = 0; k < D + 2; k++) v[k] = c < a.nc ? a.q[q64_index(k, c, a.ntot)] / a.vinv[c] : 0.0;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < D + 2; k++) {
        double x = v[k];
        for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
        if (lane == 0) red[wid][k] = x;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < D + 2; k++) {
            double s = 0.0;
            for (int i = 0; i < (int)(blockDim.x >> 6); i++) s += red[i][k];
            a.partial[(size_t)blockIdx.x * (D + 2) + k] = s;
        }
    }
}

template <typename T>
static __global__ void __launch_bounds__(256) fill_zero(T *p, T *r, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = r[i] = 0;
}
static __global__ void __launch_bounds__(64) set_scalar(double *x, double v) {
    if (threadIdx.x == 0) *x = v;
}
// n <= 64 device values to pinned host memory: 2 us less than a copy of theirs
static __global__ void __launch_bounds__(64) export_scalars(const double *x, int n, double *host) {
    if ((int)threadIdx.x < n) host[threadIdx.x] = x[threadIdx.x];
}

template <int D>
__global__ void __launch_bounds__(256) count_nonfinite(const double *q, int nc, int ntot, unsigned long long *cnt) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    int bad = 0;
#pragma unroll
    for (int k = 0; k < D + 2; k++) bad += !isfinite(q[q64_index(k, c, ntot)]);
    if (bad) atomicAdd(cnt, (unsigned long long)bad);
}

}  // namespace lfm
