// kernels_fp32p.hpp -- FP32 time step on deviations from the freestream.
//
// State: q' = q - q_inf in FP32 (q_inf = rho_inf, rho_inf U_inf, rho_inf E_inf
// held as constants).  Every face flux is evaluated as F(q_f).S - F(q_inf).S
// with the deviation formed algebraically, never by subtracting two
// freestream-sized numbers:
//   u' = (m' - u_inf rho') / rho
//   p' = (g-1) [ (rhoE)' - 1/2 (rho' |u_inf|^2 + rho u'.(2 u_inf + u')) ]
//   Rpsi' = (p' - Rpsi_inf rho') / rho
// Subtracting F(q_inf).S face by face leaves every closed cell's sum unchanged
// in exact arithmetic (sum of S over a closed cell is zero) and removes the
// FP32 closure error of the S vectors times the freestream flux.  Green-Gauss
// gradients are taken of the deviations for the same reason.  dt, its
// min-reduction, the CFL and the conservation integrals stay FP64.
//
// M1 (cfd_v0.cpp:2589-2675): both reconstructed states are the same linear
// interpolation (the reference forms rho- with weight 1-w on the swapped pair),
// so the central-upwind combination [psi+ F+ - psi- F- + psi+ psi- (q- - q+)]
// / (psi+ - psi-) equals F+ exactly; this path evaluates F+ directly and so
// carries none of the rounding-level dissipation the FP64 form contains.
#pragma once

#include "solver_state.hpp"

namespace lfm {

struct KArgs32 {
    int nc, nsm0, ng, nf, ntot;
    int ng_bnd;  // boundary ghosts [nc, nc+ng_bnd); halo ghosts after them
    const int32_t *fP, *fN;
    const float *S;  // [nf][D]: a face's area vector as one record
    const float *d, *w;
    const int32_t *g_off, *g_ent;
    // each cell's first GatherUnroll gather entries and the cells they lead to
    // (key_at places them; kNoFace and the cell itself past its last)
    const int32_t *g_key, *g_oth;
    const int32_t *ghost_cell, *ghost_role;
    const float *vinv;
    const float *sigma;  // nullptr where every cell's sponge sigma is zero
    const float *smag;  // [nc] Smagorinsky constants, nullptr when laminar
    float *q, *dq, *res_cell;
    // per-cell gradient records (GradRec32): dudx points at the records,
    // dTdx / rho_grad / p_grad into them (component stride 1, cell stride
    // gstride); tauMC / sigmaU (partitions only) and a U_grad that is not
    // dudx are [component][ntot]
    float *dudx, *dTdx, *tauMC, *sigmaU;
    float *rho_grad, *p_grad, *U_grad;
    int gstride;
    // face fluxes: components 0-3 as one 16-byte record per face ([nf][4]),
    // then (3D) component 4 as [nf]: one vector load per gathered face
    float *frhs;
    const double *dt;
    double *partial;
    const double *vol_d;  // FP64 cell volumes (conservation integrals)
    double *d_cfl, *d_dtmin;  // this solver's FP64 CFL / dt-min scalars
    int nblk_cells;           // blocks of 256 over the cells (reduction partials)
    // per-cell face slots of the one-launch stage and the 3D gradient kernel
    // (the first GatherUnroll gather entries of each cell): either packed
    // words (pk_at; the other cell in the low pk_shift bits, above them the
    // face's record in the geometry table pk_tab) or, where the mesh has too
    // many distinct records, the other cell (~other where the cell is the face's
    // N), the area vector out of the cell and P's weight (sl_*, as slot_at
    // places them).  A slot past
    // the cell's last entry holds the cell itself with zero area, so its flux
    // is zero.  more_faces: some cell has entries beyond the slots.
    const uint32_t *pk;
    const float *pk_tab;
    int pk_shift, pk_half;  // pk_half: every weight in the table is 1/2
    const int32_t *sl_nb;
    const float *sl_S, *sl_w;
    int more_faces;
    int own_nb;  // some cell is its own neighbour: no slots, two entries for such a face
    // the second state buffer, in a batch's copy of a member's arguments
    // (the solver's own copy leaves it null)
    float *q_alt;
    float gamma, gm1, gog, R_inv, mu, cp, pr_inv;
    float rho_inf, p_inf, T_inf, Rpsi_inf, E_inf, H_inf, G_inf, c_inf;
    float uinf[3], minf[3], uinf2;  // uinf2: |u_inf|^2
    double rho_inf_d, m_inf_d[3], rhoE_inf_d;
};

#define LERP32(w, a, b) ((w) * (a) + (1.0f - (w)) * (b))

// The same from the cell's side: wc of its own value, wo of the other's
__device__ __forceinline__ float cell_lerp32(float wc, float c, float wo, float o) {
    return __builtin_fmaf(wc, c, wo * o);
}
// LERP32 at w = 1/2, both products rounded before the sum (they are exact, short
// of the subnormal range): exchanging the cells gives the same bits
__device__ __forceinline__ float half_lerp32(float c, float o) {
#pragma clang fp contract(off)
    const float x = 0.5f * c, y = 0.5f * o;
    return x + y;
}
// LERP32 of a face's P and N where the one-launch stage must find the bits of
// the face kernel: from half_lerp32 where w is 1/2
__device__ __forceinline__ float face_lerp32(float w, float P, float N) {
    const float v = __builtin_fmaf(w, P, (1.0f - w) * N), h = half_lerp32(P, N);
    return w == 0.5f ? h : v;
}
// M2's midpoint
__device__ __forceinline__ float midpoint32(float c, float o) { return 0.5f * (c + o); }

// FP32 reciprocal, quotient, square root and reciprocal square root on the
// hardware instructions (v_rcp_f32, v_sqrt_f32, v_rsq_f32: 1 ulp).  Spelled
// as target builtins so that every kernel instantiating a body, single or
// batched, selects the same instructions: the lowering of a plain `/` or
// sqrtf depends on whether its operands are wave-uniform, which differs
// between the two launch forms.
__device__ __forceinline__ float rcp32(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float div32(float n, float d) { return n * __builtin_amdgcn_rcpf(d); }
__device__ __forceinline__ float sqrt32(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ float rsq32(float x) { return __builtin_amdgcn_rsqf(x); }

// face f's area vector (one 8-byte load in 2D)
template <int D>
__device__ __forceinline__ void load_S32(const float *S, int f, float (&s)[D]) {
    if constexpr (D == 2) {
        const float2 v = reinterpret_cast<const float2 *>(S)[f];
        s[0] = v.x;
        s[1] = v.y;
    } else {
#pragma unroll
        for (int k = 0; k < D; k++) s[k] = S[(size_t)f * D + k];
    }
}

template <int D>
struct Prim32 {
    float rp, rho, ri, up[D], u[D], du2, pp, Rp, R;  // du2 = |u|^2 - |u_inf|^2
};

template <int D>
__device__ __forceinline__ Prim32<D> prim32(const KArgs32 &a, const float *q) {
    Prim32<D> s;
    s.rp = q[0];
    s.rho = a.rho_inf + s.rp;
    s.ri = rcp32(s.rho);
    s.du2 = 0.f;
#pragma unroll
    for (int k = 0; k < D; k++) {
        s.up[k] = (q[k + 1] - a.uinf[k] * s.rp) * s.ri;
        s.u[k] = a.uinf[k] + s.up[k];
        s.du2 += s.up[k] * (2.f * a.uinf[k] + s.up[k]);
    }
    // rho' |u|^2 + rho_inf (|u|^2 - |u_inf|^2) = rho' |u_inf|^2 + rho du2
    s.pp = a.gm1 * (q[D + 1] - 0.5f * (s.rp * a.uinf2 + s.rho * s.du2));
    s.Rp = (s.pp - a.Rpsi_inf * s.rp) * s.ri;
    s.R = a.Rpsi_inf + s.Rp;
    return s;
}

// FP32 state layout: components 0-3 of a cell (or ghost) i as one 16-byte
// record, q[4 i + k], then component 4 (the 3D energy) as q[4 ntot + i]: a
// gathered neighbour state is one vector load (two in 3D).
__host__ __device__ __forceinline__ size_t q32_index(int k, size_t i, size_t ntot) {
    return k < 4 ? 4 * i + (size_t)k : 4 * ntot + i;
}

using f4v = float __attribute__((ext_vector_type(4)));
// a 16-byte record
template <bool NT>
__device__ __forceinline__ void st4_once(float *p, float x, float y, float z, float w) {
    const f4v v = {x, y, z, w};
    st_once<NT>(reinterpret_cast<f4v *>(p), v);
}

template <int D>
__device__ __forceinline__ void load_q32(const KArgs32 &a, int i, float *q) {
    const float4 v = reinterpret_cast<const float4 *>(a.q)[i];
    q[0] = v.x;
    q[1] = v.y;
    q[2] = v.z;
    q[3] = v.w;
    if (D == 3) q[4] = a.q[(size_t)4 * a.ntot + i];
}

template <int D, bool NT>
__device__ __forceinline__ void store_q32(float *qv, size_t ntot, int i, const float *q) {
    st4_once<NT>(qv + 4 * (size_t)i, q[0], q[1], q[2], q[3]);
    if (D == 3) st_once<NT>(qv + 4 * ntot + i, q[4]);
}

template <int D>
__device__ __forceinline__ float dot32(const float *x, const float *y) {
    float s = x[0] * y[0];
#pragma unroll
    for (int k = 1; k < D; k++) s += x[k] * y[k];
    return s;
}

__device__ __forceinline__ float sgn32(float x) { return x < 0.0f ? -1.0f : 1.0f; }

// interp_minmod (api/cfdv0_solver.h:311-370) on deviations: phi' differences
// equal phi differences, and the weights sum to one, so phi_inf is added back
// by the caller.
template <int D>
__device__ __forceinline__ float minmod32(float cphi, float aphi, const float *grad, const float *d, float wl,
                                          float flux) {
    const float gradf = aphi - cphi + 1.0e-30f;
    float gradcf = 0.0f;
#pragma unroll
    for (int k = 0; k < D; k++) gradcf += d[k] * grad[k];
    float r;
    if (fabsf(gradcf) >= 1000.0f * fabsf(gradf))
        r = 2.0f * 1000.0f * sgn32(gradcf) * sgn32(gradf) - 1.0f;
    else
        r = 2.0f * div32(gradcf, gradf) - 1.0f;
    const float m1 = (1.0f < r) ? 1.0f : r;
    const float lim = (m1 < 0.0f) ? 0.0f : m1;
    const float wt = lim * wl + (1.0f - lim) * (1.0f + flux) * 0.5f;
    return wt * cphi + (1.0f - wt) * aphi;
}

__device__ __forceinline__ float p5pos32(float M, float alpha) {
    const float M2Pos = 0.25f * (M + 1.0f) * (M + 1.0f);
    const float M2Neg = -0.25f * (M - 1.0f) * (M - 1.0f);
    if (fabsf(M) < 1.f) return M2Pos * ((2.0f - M) - 16.0f * alpha * M * M2Neg);
    return div32(0.5f * (M + fabsf(M)), M);
}

__device__ __forceinline__ float p5neg32(float M, float alpha) {
    const float M2Pos = 0.25f * (M + 1.0f) * (M + 1.0f);
    const float M2Neg = -0.25f * (M - 1.0f) * (M - 1.0f);
    if (fabsf(M) < 1.f) return M2Neg * ((-2.0f - M) + 16.0f * alpha * M * M2Pos);
    return div32(0.5f * (M - fabsf(M)), M);
}

// ---------------------------------------------------------------------------
// ghost states (cfd_v0.cpp:1010-1133) in deviation form
// ---------------------------------------------------------------------------
template <int D>
__device__ __forceinline__ bool ghost_state32(const KArgs32 &a, int role, const float *qi, float *qg) {
    if (role == 1) {  // wall: rho, -rhoU, rhoE
        qg[0] = qi[0];
#pragma unroll
        for (int k = 0; k < D; k++) qg[k + 1] = -qi[k + 1] - 2.f * a.minf[k];
        qg[D + 1] = qi[D + 1];
        return true;
    }
    if (role != 2 && role != 3) return false;  // unset patch: q = 0, i.e. q' = -q_inf
    const Prim32<D> s = prim32<D>(a, qi);
    if (role == 2) {  // inlet: T = T_inf, U = U_inf, p = p_int
        const float rpg = s.rp + div32(s.rho * (s.Rp * a.R_inv), a.T_inf);
        qg[0] = rpg;
        float u2 = 0.f;
#pragma unroll
        for (int k = 0; k < D; k++) {
            qg[k + 1] = rpg * a.uinf[k];
            u2 += a.uinf[k] * a.uinf[k];
        }
        qg[D + 1] = div32(s.pp, a.gm1) + 0.5f * rpg * u2;
    } else {  // outlet: p = p_inf, U = U_int, rho = rho_int p_inf / p_int
        const float pint = a.p_inf + s.pp;
        const float rpg = div32(s.rp * a.p_inf - a.rho_inf * s.pp, pint);
        const float rhog = a.rho_inf + rpg;
        float u2 = 0.f, du2 = 0.f;
#pragma unroll
        for (int k = 0; k < D; k++) {
            qg[k + 1] = rpg * a.uinf[k] + rhog * s.up[k];
            u2 += s.u[k] * s.u[k];
            du2 += s.up[k] * (2.f * a.uinf[k] + s.up[k]);
        }
        qg[0] = rpg;
        qg[D + 1] = 0.5f * (rpg * u2 + a.rho_inf * du2);
    }
    return true;
}

// ghost states (cfd_v0.cpp:1010-1133) in deviation form; the fused update
// refreshes ghosts, so this runs only after the state is set from outside
template <int D>
__device__ __forceinline__ void bc_fill32_body(const KArgs32 &a, const int g) {
    if (g >= a.ng) return;
    float qi[D + 2], qg[D + 2];
    load_q32<D>(a, a.ghost_cell[g], qi);
    if (!ghost_state32<D>(a, a.ghost_role[g], qi, qg)) return;
    const int gi = a.nc + g;
    store_q32<D, false>(a.q, a.ntot, gi, qg);
}

// ---------------------------------------------------------------------------
// Green-Gauss of deviations + viscous tensors, per cell
// ---------------------------------------------------------------------------
// tauMC and sigmaU of one cell from its completed dudx and velocity (the
// calc_VIS refresh, Smagorinsky stress when smag is given).  Used where they
// are stored and where a face recomputes them.
template <int D>
__device__ __forceinline__ void vis_tensors32(const KArgs32 &a, const float (&dudx)[D][D], const float (&u)[D],
                                              const float *smag_p, float (&tmc)[D][D], float (&sU)[D]) {
    const float mu = a.mu;
    float tau[D][D];
#pragma unroll
    for (int p = 0; p < D; p++) {
        tau[p][p] = 2.0f * dudx[p][p];
#pragma unroll
        for (int b1 = p + 1; b1 < D + p; b1++) {
            const int b = b1 % D;
            tau[p][b] = mu * (dudx[p][b] + dudx[b][p]);
            tau[p][p] -= dudx[b][b];
        }
        tau[p][p] *= 2.0f / 3.0f * mu;
    }
    float diag = 0.f;
#pragma unroll
    for (int p = 0; p < D; p++) diag -= dudx[p][p];
    diag *= mu * (2.0f / 3.0f);
#pragma unroll
    for (int i = 0; i < D; i++) {
#pragma unroll
        for (int j = 0; j < D; j++) tmc[i][j] = mu * dudx[j][i];
        tmc[i][i] += diag;
    }
    if (smag_p) {  // Smagorinsky stress (cfd_v0.cpp:1668-1684)
        const float smag = *smag_p;
        float strain = 0.f, divu = 0.f;
#pragma unroll
        for (int i = 0; i < D; i++) {
#pragma unroll
            for (int j = 0; j < D; j++) {
                const float sij = 0.5f * (dudx[i][j] + dudx[j][i]);
                strain += sij * sij;
            }
            divu += dudx[i][i];
        }
        strain = sqrt32(2.f * strain);
#pragma unroll
        for (int i = 0; i < D; i++) {
#pragma unroll
            for (int j = 0; j < D; j++) tmc[i][j] -= smag * strain * (0.5f * (dudx[i][j] + dudx[j][i]));
            tmc[i][i] += smag * strain * divu * (1.f / 3.f);
        }
    }
#pragma unroll
    for (int i = 0; i < D; i++) sU[i] = dot32<D>(u, tau[i]);
}

// One cell's gradients as one record, padded to whole 8-byte words: dudx
// (D*D), dTdx (D), then with RG (the M2AUSM scheme) the rho and p gradients
// (D each); ghosts' records stay zero.  A gathered neighbour's gradients are
// a few 8-byte vector loads.
template <int D, bool RG>
struct GradRec32 {
    static constexpr int kDT = D * D;
    static constexpr int kRG = kDT + D;
    static constexpr int kPG = kRG + D;
    static constexpr int kN = RG ? kPG + D : kRG;
    static constexpr int kStride = (kN + 1) / 2 * 2;
};
inline int grad_record_stride(int D, bool rg) {
    const int n = D * D + D + (rg ? 2 * D : 0);
    return (n + 1) / 2 * 2;
}

// 2D packed words lie together per cell (one 16-byte load), 3D ones as slots do
template <int D>
__device__ __forceinline__ size_t pk_at(int nc, int j, int c) {
    if constexpr (D == 2) return (size_t)GatherUnroll<2>::value * c + j;
    return slot_at<D, 1>(nc, j, 0, c);
}
inline size_t pk_len(int D, int nc, int U) { return D == 2 ? (size_t)U * nc : slot_array_len(nc, U, 1); }

// one face as one of its cells sees it: the other cell, the area vector out
// of the cell, P's weight and whether the cell is the face's P
template <int D, bool PK, bool NT>
struct FaceOf32 {
    int other;
    float S[D], w;
    bool isP;
    // the weights of the cell's value and of the other's
    __device__ __forceinline__ float wc() const { return isP ? w : 1.0f - w; }
    __device__ __forceinline__ float wo() const { return isP ? 1.0f - w : w; }
    // key: the packed word (an odd record is N's), or the slot's other cell (~other
    // where the cell is the face's N)
    __device__ __forceinline__ static int load_key(const KArgs32 &a, const int j, const int c) {
        if constexpr (PK) return (int)ld_once<NT>(a.pk + pk_at<D>(a.nc, j, c));
        return ld_once<NT>(a.sl_nb + slot_at<D, 1>(a.nc, j, 0, c));
    }
    __device__ __forceinline__ static int other_of(const KArgs32 &a, const int key) {
        if constexpr (PK) return (int)((uint32_t)key & ((1u << a.pk_shift) - 1u));
        return key >= 0 ? key : ~key;
    }
    __device__ __forceinline__ void load(const KArgs32 &a, const int j, const int c, const int key) {
        other = other_of(a, key);
        if constexpr (PK) {
            isP = !((uint32_t)key >> a.pk_shift & 1u);
            const float4 v = reinterpret_cast<const float4 *>(a.pk_tab)[(uint32_t)key >> a.pk_shift];
            const float r[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int k = 0; k < D; k++) S[k] = r[k];
            w = r[D];
        } else {
#pragma unroll
            for (int k = 0; k < D; k++) S[k] = ld_once<NT>(a.sl_S + slot_at<D, D>(a.nc, j, k, c));
            w = ld_once<NT>(a.sl_w + slot_at<D, 1>(a.nc, j, 0, c));
            isP = key >= 0;
        }
    }
    // an entry of the gather list
    __device__ __forceinline__ void load_list(const KArgs32 &a, const int ent) {
        load_face(a, ent);
        other = ent >= 0 ? a.fN[face_of(ent)] : a.fP[face_of(ent)];
    }
    // its face's data alone
    __device__ __forceinline__ void load_face(const KArgs32 &a, const int ent) {
        isP = ent >= 0;
        const int f = face_of(ent);
        w = a.w[f];
        load_S32<D>(a.S, f, S);
#pragma unroll
        for (int k = 0; k < D; k++) S[k] = isP ? S[k] : -S[k];
    }
};

// Green-Gauss sums of one cell over its faces in gather order; returns the
// cell's own primitive state.  SL: every entry from the slots (3D); otherwise
// through the gather entries.  Each face's sums sit in a branch of their own: in one
// block the compiler interleaves all six faces' arithmetic (124 VGPRs instead
// of 96, 4 waves per SIMD instead of 5).
template <int D, int GRAD, bool VISC, bool SL, bool PK, bool NT>
__device__ __forceinline__ Prim32<D> grad32_sums(const KArgs32 &a, const int c, float (&dudx)[D][D],
                                                  float (&dTdx)[D], float (&rg)[D], float (&pg)[D],
                                                  float (&ug)[D][D]) {
    const float vinv = a.vinv[c];
#pragma unroll
    for (int i = 0; i < D; i++) {
        dTdx[i] = rg[i] = pg[i] = 0.f;
#pragma unroll
        for (int j = 0; j < D; j++) dudx[i][j] = ug[i][j] = 0.f;
    }
    float qc0[D + 2];
    load_q32<D>(a, c, qc0);
    const Prim32<D> own = prim32<D>(a, qc0);
    using F = FaceOf32<D, PK, NT>;
    // one face's contribution
    auto add = [&](const F &f, const float (&qo)[D + 2]) {
        const Prim32<D> so = prim32<D>(a, qo);
        const float wc = f.wc(), wo = f.wo();
        float sv[D];
#pragma unroll
        for (int k = 0; k < D; k++) sv[k] = f.S[k] * vinv;
        float fU[D];
#pragma unroll
        for (int k = 0; k < D; k++) fU[k] = cell_lerp32(wc, own.up[k], wo, so.up[k]);
        const float fT = VISC ? cell_lerp32(wc, own.Rp, wo, so.Rp) * a.R_inv : 0.f;
#pragma unroll
        for (int i = 0; i < D; i++) {
#pragma unroll
            for (int j = 0; j < D; j++) dudx[i][j] += fU[i] * sv[j];
            if (VISC) dTdx[i] += fT * sv[i];
        }
        if (GRAD == 2) {
            const float rf = cell_lerp32(wc, own.rp, wo, so.rp);
            const float pf = cell_lerp32(wc, own.pp, wo, so.pp);
#pragma unroll
            for (int i = 0; i < D; i++) {
                pg[i] += pf * sv[i];
                rg[i] += rf * sv[i];
#pragma unroll
                for (int j = 0; j < D; j++) ug[j][i] += fU[j] * sv[i];
            }
        }
    };
    constexpr int U = GatherUnroll<D>::value;
    F f[U];
    float qo[U][D + 2];
    if constexpr (SL) {
#pragma unroll
        for (int j = 0; j < U; j++) {
            f[j].load(a, j, c, F::load_key(a, j, c));
            load_q32<D>(a, f[j].other, qo[j]);
        }
#pragma unroll
        for (int j = 0; j < U; j++)
            if (f[j].other != c) add(f[j], qo[j]);  // not a placeholder's
        return own;
    }
    // the first faces: every load issued before the sums.  Fewer in flight is
    // slower: O-grid gradients 0.97 -> 1.54 ms per step with three, 1.89 with
    // two.
    int e0 = 0, ne = U, key[U], oth[U];
    load_keys<D, NT>(a.g_key, a.nc, 0, c, key);
    load_keys<D, NT>(a.g_oth, a.nc, 0, c, oth);
    if (a.more_faces) {
        e0 = a.g_off[c];
        ne = a.g_off[c + 1] - e0;
    }
#pragma unroll
    for (int j = 0; j < U; j++) {
        f[j].load_face(a, key[j]);
        f[j].other = oth[j];
        load_q32<D>(a, f[j].other, qo[j]);
    }
#pragma unroll
    for (int j = 0; j < U; j++)
        if (key[j] != kNoFace) add(f[j], qo[j]);
    for (int e = e0 + U; e < e0 + ne; e++) {
        F g;
        float q[D + 2];
        g.load_list(a, a.g_ent[e]);
        load_q32<D>(a, g.other, q);
        add(g, q);
    }
    return own;
}

// every thread of the block must call this (the block's records are written
// through LDS); c = the block's first cell + threadIdx.x
template <int D, int GRAD, bool VISC, bool RG, bool SL, bool PK, bool NT>
__device__ __forceinline__ void grad_vis32_body(const KArgs32 &a, const int c) {
    using R = GradRec32<D, RG>;
    const bool valid = c < a.nc;
    float r[R::kStride];
#pragma unroll
    for (int k = 0; k < R::kStride; k++) r[k] = 0.f;
    if (valid) {
        float dudx[D][D], dTdx[D], rg[D], pg[D], ug[D][D];
        const Prim32<D> own = grad32_sums<D, GRAD, VISC, SL, PK, NT>(a, c, dudx, dTdx, rg, pg, ug);
        // tauMC / sigmaU stored only where a halo payload needs them (otherwise
        // each face recomputes them from dudx); U_grad equals dudx bit for bit
        // (same face velocity, same sums) and shares its storage unless a halo
        // payload must leave it zero on the ghosts
        const size_t nt = a.ntot;
        if (VISC && a.tauMC) {
            float tmc[D][D], sU[D];
            vis_tensors32<D>(a, dudx, own.u, a.smag ? a.smag + c : nullptr, tmc, sU);
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
            for (int j = 0; j < D; j++) r[i * D + j] = dudx[i][j];
            r[R::kDT + i] = VISC ? dTdx[i] : 0.f;
            if (RG && GRAD == 2) {
                r[R::kRG + i] = rg[i];
                r[R::kPG + i] = pg[i];
            }
        }
        if (GRAD == 2 && a.U_grad != a.dudx)
#pragma unroll
            for (int i = 0; i < D; i++)
#pragma unroll
                for (int j = 0; j < D; j++) a.U_grad[(i * D + j) * nt + c] = ug[i][j];
        if (!VISC) {
            // dTdx not formed: the formed components only (the record keeps
            // whatever a full calc_VIS left in the dTdx slots)
            float *rec = a.dudx + (size_t)c * R::kStride;
#pragma unroll
            for (int i = 0; i < D; i++) {
#pragma unroll
                for (int j = 0; j < D; j++) rec[i * D + j] = r[i * D + j];
                if (RG && GRAD == 2) {
                    rec[R::kRG + i] = r[R::kRG + i];
                    rec[R::kPG + i] = r[R::kPG + i];
                }
            }
        }
    }
    if (VISC) {
        // the block's records are contiguous from its first cell (a multiple
        // of 256, so 16-byte aligned): staged in LDS, then written as
        // consecutive 16-byte words and a tail of single words (without
        // minmod the rho / p slots are written zero, as they stay)
        constexpr int S = R::kStride;
        __shared__ __align__(16) float st[256 * S];
        const int t = threadIdx.x;
#pragma unroll
        for (int k = 0; k < S / 2; k++)
            reinterpret_cast<float2 *>(st)[t * (S / 2) + k] = make_float2(r[2 * k], r[2 * k + 1]);
        __syncthreads();
        const int c0 = c - t;
        const int nrec = a.nc - c0 < (int)blockDim.x ? a.nc - c0 : (int)blockDim.x;
        float *dst = a.dudx + (size_t)c0 * S;
        const int n = nrec * S, n4 = n / 4;
        for (int j = t; j < n4; j += blockDim.x)
            st_once<NT>(reinterpret_cast<f4v *>(dst) + j, reinterpret_cast<const f4v *>(st)[j]);
        for (int j = 4 * n4 + t; j < n; j += blockDim.x) dst[j] = st[j];
    }
}

// ---------------------------------------------------------------------------
// Where the face kernel reads the cells' gradients (the solver's arrays,
// indexed by cell)
// ---------------------------------------------------------------------------
template <int D, bool RG>
struct GradGlobal32 {
    const KArgs32 &a;
    using R = GradRec32<D, RG>;
    // the gradient record of cell c
    __device__ __forceinline__ void rec(int c, float (&r)[R::kStride]) const {
        if constexpr (R::kStride % 4 == 0) {
            // records of whole 16-byte words (3D without minmod: 48 B)
            const float4 *p = reinterpret_cast<const float4 *>(a.dudx + (size_t)c * R::kStride);
#pragma unroll
            for (int k = 0; k < R::kStride / 4; k++) {
                const float4 v = p[k];
                r[4 * k] = v.x;
                r[4 * k + 1] = v.y;
                r[4 * k + 2] = v.z;
                r[4 * k + 3] = v.w;
            }
        } else {
            const float2 *p = reinterpret_cast<const float2 *>(a.dudx + (size_t)c * R::kStride);
#pragma unroll
            for (int k = 0; k < R::kStride / 2; k++) {
                const float2 v = p[k];
                r[2 * k] = v.x;
                r[2 * k + 1] = v.y;
            }
        }
    }
    // U_grad: dudx itself, or its own [component][ntot] array
    __device__ __forceinline__ float ug(const float (&r)[R::kStride], int c, int i, int j) const {
        return a.U_grad == a.dudx ? r[i * D + j] : a.U_grad[(size_t)(i * D + j) * a.ntot + c];
    }
};

// ---------------------------------------------------------------------------
// face fluxes minus the freestream flux, one thread per face
// ---------------------------------------------------------------------------
// The convective flux of one face (M1 cfd_v0.cpp:2590-2637, M2 1968-2023)
// seen from one of its cells: c the cell, o the other, S out of the cell.
// Every face value is formed from P's and N's, whichever of them c is (isP; M2's
// midpoint and M1 at w = 1/2 are the same with the two exchanged and need no
// selecting), and every other term changes sign with S, so the flux from N is
// P's negated, bit for bit.  HALF: every weight is 1/2.
template <int D>
struct Conv32 {
    float rp, rho, mp[D], phi_inf, phip, phi, pp, Gdev;
};
template <int D, int SOLVER, bool HALF>
__device__ __forceinline__ Conv32<D> conv32(const KArgs32 &a, const float (&qc)[D + 2], const Prim32<D> &sc,
                                            const float (&qo)[D + 2], const Prim32<D> &so, const float (&S)[D],
                                            const float w, const bool isP) {
    Conv32<D> f;
    auto face = [&](const float c, const float o) {
        if constexpr (SOLVER != 0) return midpoint32(c, o);
        if constexpr (HALF) return half_lerp32(c, o);  // the cell's own products are formed once per cell
        return face_lerp32(w, isP ? c : o, isP ? o : c);
    };
    f.rp = face(qc[0], qo[0]);
    f.rho = a.rho_inf + f.rp;
    const float ri = rcp32(f.rho);
    float du2 = 0.f;
    f.phip = f.phi_inf = 0.f;
#pragma unroll
    for (int k = 0; k < D; k++) {
        f.phi_inf += a.uinf[k] * S[k];
        f.mp[k] = face(qc[k + 1], qo[k + 1]);
        const float up = (f.mp[k] - a.uinf[k] * f.rp) * ri;
        f.phip += up * S[k];
        if (SOLVER == 0) du2 += up * (2.f * a.uinf[k] + up);
    }
    f.phi = f.phi_inf + f.phip;
    const float Rp = face(sc.Rp, so.Rp);
    f.pp = f.rp * a.Rpsi_inf + f.rho * Rp;
    // M1: G = rhoE + p = rho (g/(g-1) Rpsi + |u|^2/2) of the face state; M2:
    // rho times the average of the cells' H = rhoE/rho + Rpsi
    float Hp;
    if constexpr (SOLVER == 0) {
        Hp = a.gog * Rp + 0.5f * du2;
    } else {
        const float hc = a.gog * sc.Rp + 0.5f * sc.du2, ho = a.gog * so.Rp + 0.5f * so.du2;
        Hp = midpoint32(hc, ho);
    }
    f.Gdev = f.rp * a.H_inf + f.rho * Hp;
    return f;
}
// the face's rhs from its convective parts and pressure
template <int D>
__device__ __forceinline__ void conv_rhs32(const KArgs32 &a, const Conv32<D> &f, const float pp, const float (&S)[D],
                                           float (&rhs)[D + 2]) {
    float mS = 0.f;
#pragma unroll
    for (int k = 0; k < D; k++) mS += f.mp[k] * S[k];
    rhs[0] = -mS;
#pragma unroll
    for (int k = 0; k < D; k++) rhs[k + 1] = -(f.phip * a.minf[k] + f.phi * f.mp[k] + pp * S[k]);
    rhs[D + 1] = -(f.phip * a.G_inf + f.phi * f.Gdev);
}

// the flux of face f from its cells' states and primitives (qP, sp of P;
// qN, sn of N)
template <int D, int SOLVER, bool VISC, bool STORED, bool NT, class GA>
__device__ __forceinline__ void face_flux32_states(const KArgs32 &a, const int f, const int P, const int N,
                                                   const float (&qP)[D + 2], const float (&qN)[D + 2],
                                                   const Prim32<D> &sp, const Prim32<D> &sn,
                                                   const float (&S)[D], const float w, const GA &ga,
                                                   const int gP, const int gN, float (&rhs)[D + 2]) {
    using R = GradRec32<D, SOLVER == 2>;
    float gr[2][R::kStride];  // gradient records of P and N
    if (VISC || SOLVER == 2) {
        ga.rec(gP, gr[0]);
        ga.rec(gN, gr[1]);
    }
    // is_ghost: boundary ghosts only; halo ghosts carry the neighbour's tensors
    const bool ghost = (unsigned)(N - a.nc) < (unsigned)a.ng_bnd;
    const size_t nt = a.ntot;
    float d[D];
#pragma unroll
    for (int k = 0; k < D; k++) d[k] = ld_once<NT>(a.d + (size_t)k * a.nf + f);
    float Sm2 = 0.f;
#pragma unroll
    for (int k = 0; k < D; k++) Sm2 += S[k] * S[k];
    const float Sm = sqrt32(Sm2);
    const Conv32<D> cv = conv32<D, SOLVER, false>(a, qP, sp, qN, sn, S, w, true);
    float pp = cv.pp;
    if (SOLVER == 2) {
        const float phi_inf = cv.phi_inf;
        const float cP = sqrt32(a.gamma * sp.R), cN = sqrt32(a.gamma * sn.R);
        const float cavg = 0.5f * (cP + cN);
        float cdiv = 0.f, ndiv = 0.f, ccurl = 0.f, ncurl = 0.f, unP = 0.f, unN = 0.f;
        float cdu[D][D], ndu[D][D];
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
            float gc[D], gn[D];
#pragma unroll
            for (int k = 0; k < D; k++) {
                gc[k] = ga.ug(gr[0], gP, p, k);
                gn[k] = ga.ug(gr[1], gN, p, k);
            }
            unP += minmod32<D>(sp.up[p], sn.up[p], gc, d, w, 1.0f) * S[p];
            unN += minmod32<D>(sp.up[p], sn.up[p], gn, d, w, -1.0f) * S[p];
        }
        const float cth0 = -cdiv * rsq32(cdiv * cdiv + ccurl + 4e-2f);
        const float nth0 = -ndiv * rsq32(ndiv * ndiv + ncurl + 4e-2f);
        const float tha = 0.5f * (((cth0 < 0.f) ? 0.f : cth0) + ((nth0 < 0.f) ? 0.f : nth0));
        float gc[D], gn[D], hc[D], hn[D];
#pragma unroll
        for (int k = 0; k < D; k++) {
            gc[k] = gr[0][R::kRG + k];
            gn[k] = gr[1][R::kRG + k];
            hc[k] = gr[0][R::kPG + k];
            hn[k] = gr[1][R::kPG + k];
        }
        const float rhoPos = a.rho_inf + minmod32<D>(sp.rp, sn.rp, gc, d, w, 1.0f);
        const float rhoNeg = a.rho_inf + minmod32<D>(sp.rp, sn.rp, gn, d, w, -1.0f);
        const float pPd = minmod32<D>(sp.pp, sn.pp, hc, d, w, 1.0f);
        const float pNd = minmod32<D>(sp.pp, sn.pp, hn, d, w, -1.0f);
        const float unPf = phi_inf + unP, unNf = phi_inf + unN;
        const float rSc = rcp32(Sm * cavg);
        const float MP = unPf * rSc;
        const float MN = unNf * rSc;
        const float Msq = 0.5f * (MP * MP + MN * MN);
        const float Minf = 0.2f;
        const float mx = (Msq < Minf * Minf) ? Minf * Minf : Msq;
        const float M0 = sqrt32((mx < 1.0f) ? mx : 1.0f);
        const float fa = M0 * (2.0f - M0);
        const float alpha = 3.0f * (5.0f * fa * fa - 4.0f) / 16.0f;
        const float dN = p5pos32(MN, alpha) - p5neg32(MN, alpha);
        const float dP = p5pos32(MP, alpha) - p5neg32(MP, alpha);
        // p_half = pN dN - pP dP = p_inf (dN - dP) + pN' dN - pP' dP.  For
        // |M| < 1, P5+(M) - P5-(M) = M (3 - M^2)/2 + 2 alpha M (1 - M^2)^2, so
        // dN - dP is formed as (MN - MP) times its divided difference, with
        // MN - MP from the normal-velocity deviations (no cancellation).
        float dNP;
        if (fabsf(MN) < 1.f && fabsf(MP) < 1.f) {
            const float s2 = MN * MN + MN * MP + MP * MP;
            const float s4 = MN * MN * MN * MN + MN * MN * MN * MP + MN * MN * MP * MP + MN * MP * MP * MP +
                             MP * MP * MP * MP;
            const float dd = 0.5f * (3.f - s2) + 2.f * alpha * (1.f - 2.f * s2 + s4);
            dNP = (unN - unP) * rSc * dd;
        } else {
            dNP = dN - dP;
        }
        const float phalf = a.p_inf * dNP + pNd * dN - pPd * dP;
        const float pu = -0.75f * p5pos32(MP, alpha) * p5neg32(MN, alpha) * (rhoPos + rhoNeg) * cavg * fa *
                         (unN - unP);
        pp += tha * (pu - 0.5f * phalf);
    }
    conv_rhs32<D>(a, cv, pp, S, rhs);

    // viscous terms (cfd_v0.cpp:2682-2790) on velocity / temperature deviations
    if (VISC) {
    const float mu = a.mu;
    float dmag2 = 0.f;
#pragma unroll
    for (int k = 0; k < D; k++) dmag2 += d[k] * d[k];
    const float dmi = rsq32(dmag2);
    float dn[D], du[D][D], dT[D], tau[D][D], tmc[D][D];
    float duP[D][D], duN[D][D], sUP[D], sUN[D];
#pragma unroll
    for (int k = 0; k < D; k++) dn[k] = d[k] * dmi;
    const float cT = sp.Rp * a.R_inv, aT = sn.Rp * a.R_inv;
    if (ghost) {
#pragma unroll
        for (int i = 0; i < D; i++) {
#pragma unroll
            for (int j = 0; j < D; j++) du[i][j] = (sn.up[i] - sp.up[i]) * dn[j] * dmi;
            dT[i] = (aT - cT) * dn[i] * dmi;
        }
    } else {
#pragma unroll
        for (int i = 0; i < D; i++) {
#pragma unroll
            for (int j = 0; j < D; j++) {
                duP[i][j] = gr[0][i * D + j];
                duN[i][j] = gr[1][i * D + j];
                du[i][j] = LERP32(w, duP[i][j], duN[i][j]);
            }
            dT[i] = LERP32(w, gr[0][R::kDT + i], gr[1][R::kDT + i]);
        }
    }
#pragma unroll
    for (int p = 0; p < D; p++) {
        tau[p][p] = 2.0f * du[p][p];
#pragma unroll
        for (int b1 = p + 1; b1 < D + p; b1++) {
            const int b = b1 % D;
            tau[p][b] = mu * (du[p][b] + du[b][p]);
            tau[p][p] -= du[b][b];
        }
        tau[p][p] *= 2.0f / 3.0f * mu;
    }
    if (ghost) {
        float diag = 0.f;
#pragma unroll
        for (int p = 0; p < D; p++) diag -= du[p][p];
        diag *= mu * (2.0f / 3.0f);
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
                tmc[i][j] = LERP32(w, a.tauMC[(i * D + j) * nt + P], a.tauMC[(i * D + j) * nt + N]);
    } else {
        // both cells' tensors as calc_VIS leaves them, from their dudx
        float tP[D][D], tN[D][D];
        vis_tensors32<D>(a, duP, sp.u, a.smag ? a.smag + P : nullptr, tP, sUP);
        vis_tensors32<D>(a, duN, sn.u, a.smag ? a.smag + N : nullptr, tN, sUN);
#pragma unroll
        for (int i = 0; i < D; i++)
#pragma unroll
            for (int j = 0; j < D; j++) tmc[i][j] = LERP32(w, tP[i][j], tN[i][j]);
    }
    const float Sd = dot32<D>(S, d);
    float K[D], dm2 = 0.f;
#pragma unroll
    for (int i = 0; i < D; i++) {
        const float delta = div32(d[i] * Sm2, Sd);
        dm2 += delta * delta;
        K[i] = S[i] - delta;
    }
    const float dm = sqrt32(dm2);
    float sU[D];
    if (ghost) {
        float Uf[D];
#pragma unroll
        for (int i = 0; i < D; i++) Uf[i] = LERP32(w, sp.u[i], sn.u[i]);
#pragma unroll
        for (int i = 0; i < D; i++) sU[i] = dot32<D>(Uf, tau[i]);
    } else if constexpr (STORED) {
#pragma unroll
        for (int i = 0; i < D; i++) sU[i] = LERP32(w, a.sigmaU[i * nt + P], a.sigmaU[i * nt + N]);
    } else {
#pragma unroll
        for (int i = 0; i < D; i++) sU[i] = LERP32(w, sUP[i], sUN[i]);
    }
    const float kcond = a.cp * mu * a.pr_inv;
#pragma unroll
    for (int i = 0; i < D; i++)
        rhs[i + 1] += dot32<D>(tmc[i], S) + mu * (dm * (sn.up[i] - sp.up[i]) * dmi + dot32<D>(K, du[i]));
    rhs[D + 1] += dot32<D>(sU, S) + kcond * (dm * (aT - cT) * dmi + dot32<D>(K, dT));
    }
}

template <int D, int SOLVER, bool VISC, bool STORED, bool NT, class GA>
__device__ __forceinline__ void face_flux32_rhs(const KArgs32 &a, const int f, const GA &ga, const int gP,
                                                const int gN, float (&rhs)[D + 2]) {
    const int P = ld_once<NT>(a.fP + f), N = ld_once<NT>(a.fN + f);
    float qP[D + 2], qN[D + 2];
    load_q32<D>(a, P, qP);
    load_q32<D>(a, N, qN);
    const Prim32<D> sp = prim32<D>(a, qP), sn = prim32<D>(a, qN);
    float S[D];
#pragma unroll
    for (int k = 0; k < D; k++) S[k] = ld_once<NT>(a.S + (size_t)f * D + k);
    face_flux32_states<D, SOLVER, VISC, STORED, NT>(a, f, P, N, qP, qN, sp, sn, S, ld_once<NT>(a.w + f), ga, gP, gN,
                                                 rhs);
}

template <int D, int SOLVER, bool VISC, bool STORED, bool NT>
__device__ __forceinline__ void face_flux32_body(const KArgs32 &a, const int f) {
    if (f >= a.nf) return;
    float rhs[D + 2];
    face_flux32_rhs<D, SOLVER, VISC, STORED, NT>(a, f, GradGlobal32<D, SOLVER == 2>{a}, a.fP[f], a.fN[f], rhs);
    st4_once<NT>(a.frhs + 4 * (size_t)f, rhs[0], rhs[1], rhs[2], rhs[3]);
    if (D == 3) st_once<NT>(a.frhs + (size_t)4 * a.nf + f, rhs[D + 1]);
}

// ---------------------------------------------------------------------------
// ordered gather of face fluxes, sponge, RK update (deviations)
// ---------------------------------------------------------------------------
// the cell's RK register as the last stage left it, zero at a step's first
// stage: every component's load issued before any is used (a choice per
// component compiles to a branch and a wait each)
template <int D, bool NT>
__device__ __forceinline__ void load_dq32(const KArgs32 &a, const int dq_mode, const int c, float (&dq)[D + 2]) {
#pragma unroll
    for (int k = 0; k < D + 2; k++) dq[k] = 0.f;
    if (!(dq_mode & kDqZero)) {
#pragma unroll
        for (int k = 0; k < D + 2; k++) dq[k] = ld_once<NT>(a.dq + (size_t)k * a.nc + c);
    }
}

// sponge, RK update and stores of one cell: q its state (the updated one on
// return), dq its accumulated register (drop: not stored)
template <int D, bool NT>
__device__ __forceinline__ void finish_cell32(const KArgs32 &a, const int c, const float dt, const float B,
                                              const bool drop, float *qout, float (&q)[D + 2], float (&dq)[D + 2]) {
    // sponge: sigma (q_inf - q) = -sigma q' (no sigma array, and no term,
    // where the case has no sponge layer and every sigma is zero)
    const float sgm = a.sigma ? ld_once<NT>(a.sigma + c) : 0.f;
#pragma unroll
    for (int k = 0; k < D + 2; k++) {
        if (a.sigma) dq[k] -= dt * sgm * q[k];
        q[k] += B * dq[k];
    }
    if (!drop)
#pragma unroll
        for (int k = 0; k < D + 2; k++) st_once<NT>(a.dq + (size_t)k * a.nc + c, dq[k]);
    store_q32<D, NT>(qout, a.ntot, c, q);
}
// boundary ghost g of a cell whose updated state is q, written for the next
// stage
template <int D, bool NT>
__device__ __forceinline__ void refresh_ghost32(const KArgs32 &a, const int g, float *qout, const float (&q)[D + 2]) {
    float qg[D + 2];
    if (!ghost_state32<D>(a, a.ghost_role[g], q, qg)) {
        if (qout == a.q) return;
        load_q32<D>(a, a.nc + g, qg);  // an unset patch's ghost keeps its state
    }
    store_q32<D, NT>(qout, a.ntot, a.nc + g, qg);
}

// ordered gather of one cell's stored face fluxes, sponge and RK update in
// place, with the cell's boundary ghosts refreshed; res receives the
// residual, q the updated state
// MORE: some cell may have gather entries beyond the first U
template <int D, bool RES, bool NT, bool MORE>
__device__ __forceinline__ void cell_update32_cell(const KArgs32 &a, float A, float B, int dq_mode, const bool drop,
                                                   const int c, float (&res)[D + 2], float (&q)[D + 2], float &vinv) {
    const float dt = (float)(*a.dt);
    vinv = ld_once<NT>(a.vinv + c);
    const float sP = dt * vinv;
    float dq[D + 2];
    load_dq32<D, NT>(a, dq_mode, c, dq);
#pragma unroll
    for (int k = 0; k < D + 2; k++) res[k] = 0.f;
    load_q32<D>(a, c, q);
    constexpr int U = GatherUnroll<D>::value;
    int key[U];
    load_keys<D, NT>(a.g_key, a.nc, 0, c, key);
    unsigned gmask = 0;  // bit j: entry j leads to a boundary ghost
    auto load = [&](const int ent, float (&fr)[D + 2]) {
        const int f = face_of(ent);
        const float4 v = reinterpret_cast<const float4 *>(a.frhs)[f];
        fr[0] = v.x;
        fr[1] = v.y;
        fr[2] = v.z;
        fr[3] = v.w;
        if (D == 3) fr[D + 1] = a.frhs[(size_t)4 * a.nf + f];
    };
    auto add = [&](const int j, const int ent, const bool valid, const float (&fr)[D + 2]) {
        gmask |= ent >= 0 && (ent & kGhostFaceFlag) ? 1u << j : 0u;
        const float sg = ent >= 0 ? sP : -sP;
#pragma unroll
        for (int k = 0; k < D + 2; k++) {
            if (RES) res[k] = valid ? res[k] + (ent >= 0 ? fr[k] : -fr[k]) : res[k];
            dq[k] = valid ? dq[k] + sg * fr[k] : dq[k];
        }
    };
    // the faces in gather order, the first U with their loads issued together
    // and without a branch: a placeholder reads face 0 and is selected away
    float fr[U][D + 2];
#pragma unroll
    for (int u = 0; u < U; u++) load(key[u], fr[u]);
#pragma unroll
    for (int k = 0; k < D + 2; k++) dq[k] *= A;
#pragma unroll
    for (int u = 0; u < U; u++) add(u, key[u], key[u] != kNoFace, fr[u]);
    int e1 = 0, ne = 0;  // entries beyond the first U
    if (MORE && a.more_faces) {
        e1 = a.g_off[c] + U;
        ne = a.g_off[c + 1] - e1;
        for (int j = 0; j < ne; j++) {
            const int ent = a.g_ent[e1 + j];
            float f1[D + 2];
            load(ent, f1);
            add(U + j, ent, true, f1);
        }
    }
    finish_cell32<D, NT>(a, c, dt, B, drop, a.q, q, dq);
    // refresh this cell's boundary ghosts for the next stage
    for (unsigned m = gmask; m; m &= m - 1) {
        const int j = __builtin_ctz(m);
        const int ent = !MORE || j < U ? a.g_key[key_at<D>(a.nc, j, c)] : a.g_ent[e1 + j - U];
        refresh_ghost32<D, NT>(a, a.fN[ent & kFaceMask] - a.nc, a.q, q);
    }
}

template <int D, int MODE, bool MORE>
__device__ __forceinline__ double cfl_cell32(const KArgs32 &a, const int c, const float (&qc)[D + 2], float vinv,
                                             double param);

// every thread of the block must call this (block-wide reductions when RES
// or CFL).  CFL >= 0 (the last stage of a step): the step's compute_dt (0) /
// compute_cfl (1) of the updated cells, per-block extrema into a.partial.
template <int D, bool RES, int CFL, bool NT, bool MORE>
__device__ __forceinline__ void cell_update32_body(const KArgs32 &a, float A, float B, int dq_mode, const int c,
                                                   const int lblk, double cfl_param) {
    static_assert(!(RES && CFL >= 0), "the residual and the CFL share a.partial");
    __shared__ double red[256 / 64][D + 2];
    double rsq[D + 2];
    double cv = CFL == 0 ? 100.0 : 0.0;
#pragma unroll
    for (int k = 0; k < D + 2; k++) rsq[k] = 0.0;
    if (c < a.nc) {
        float res[D + 2], q[D + 2], vinv;
        cell_update32_cell<D, RES, NT, MORE>(a, A, B, dq_mode, CFL >= 0 && (dq_mode & kDqDrop), c, res, q, vinv);
        if constexpr (CFL >= 0) cv = cfl_cell32<D, CFL, MORE>(a, c, q, vinv, cfl_param);
        if (RES) {
#pragma unroll
            for (int k = 0; k < D + 2; k++) {
                a.res_cell[(size_t)k * a.nc + c] = res[k];
                rsq[k] = (double)res[k] * (double)res[k];
            }
        }
    }
    if (RES) {
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
                a.partial[(size_t)lblk * (D + 2) + k] = s;
            }
        }
    }
    if constexpr (CFL >= 0) block_extremum<CFL>(cv, a.partial + lblk);
}

// compute_dt / compute_cfl (cfd_v0.cpp:2887-2942) of one cell from its FP32
// deviations: the face terms |m.S| (compute_cfl) or |m.S|/|S| (compute_dt)
// summed in FP32 over the cell's faces in gather order (the update's own
// order; the FP64 path keeps the reference's slot order), then dt_c (MODE 0)
// or cfl_c (MODE 1) in FP64, combined with the block's starting value so a
// NaN never wins; vinv: the cell's 1/V, as the update read it
template <int D, int MODE>
struct CflSum32 {
    float m[D], sum = 0.f;
    __device__ __forceinline__ CflSum32(const KArgs32 &a, const float (&qc)[D + 2]) {
#pragma unroll
        for (int k = 0; k < D; k++) m[k] = a.minf[k] + qc[k + 1];
    }
    // a face of either orientation; valid: false leaves the sum
    __device__ __forceinline__ void add(const float (&S)[D], const bool valid) {
        float fl = 0.f, s2 = 0.f;
#pragma unroll
        for (int k = 0; k < D; k++) fl += m[k] * S[k];
        if (MODE == 0) {
#pragma unroll
            for (int k = 0; k < D; k++) s2 += S[k] * S[k];
            fl *= rsq32(s2);
        }
        sum = valid ? sum + fabsf(fl) : sum;
    }
    __device__ __forceinline__ double value(const KArgs32 &a, const float rp, const float vinv_c,
                                            const double param) const {
        const double rho = a.rho_inf_d + (double)rp;
        const double vinv = (double)vinv_c;
        double v = MODE == 0 ? 100.0 : 0.0;
        if (MODE == 0) {
            const double dtc = param * rho * 2.0 / (vinv * (double)sum);
            if (v > dtc) v = dtc;
        } else {
            const double cfl = (double)sum * ((1.0 / rho) * vinv * param);
            if (v < cfl) v = cfl;
        }
        return v;
    }
};
template <int D, int MODE, bool MORE>
__device__ __forceinline__ double cfl_cell32(const KArgs32 &a, const int c, const float (&qc)[D + 2], float vinv,
                                             double param) {
    CflSum32<D, MODE> t(a, qc);
    constexpr int U = GatherUnroll<D>::value;
    int key[U];
    float S[U][D];
    // a face counts once: a cell's own face not again as its N
    auto counted = [&](const int ent) {
        return ent != kNoFace && !(MORE && a.own_nb && ent < 0 && a.fP[face_of(ent)] == c);
    };
    load_keys<D, false>(a.g_key, a.nc, 0, c, key);
#pragma unroll
    for (int j = 0; j < U; j++) load_S32<D>(a.S, face_of(key[j]), S[j]);
#pragma unroll
    for (int j = 0; j < U; j++) t.add(S[j], counted(key[j]));
    if (MORE && a.more_faces) {
        const int e0 = a.g_off[c], ne = a.g_off[c + 1] - e0;
        for (int j = U; j < ne; j++) {
            const int ent = a.g_ent[e0 + j];
            load_S32<D>(a.S, face_of(ent), S[0]);
            t.add(S[0], counted(ent));
        }
    }
    return t.value(a, qc[0], vinv, param);
}

// compute_dt / compute_cfl as their own launch (every thread of the block
// must call this)
template <int D, int MODE>
__device__ __forceinline__ void cfl_dt_cells32_body(const KArgs32 &a, double param, const int c, const int lblk) {
    double v = MODE == 0 ? 100.0 : 0.0;
    if (c < a.nc) {
        float q[D + 2];
        load_q32<D>(a, c, q);
        v = cfl_cell32<D, MODE, true>(a, c, q, a.vinv[c], param);
    }
    block_extremum<MODE>(v, a.partial + lblk);
}

// FP64 conservation integrals sum_c V_c q_c (per block partials)
template <int D>
__global__ void __launch_bounds__(256) integrals32(KArgs32 a) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    __shared__ double red[256 / 64][D + 2];
    double v[D + 2];
#pragma unroll
    for (int k = 0; k < D + 2; k++) v[k] = 0.0;
    if (c < a.nc) {
        const double vol = a.vol_d[c];
        v[0] = vol * (a.rho_inf_d + (double)a.q[q32_index(0, c, a.ntot)]);
#pragma unroll
        for (int k = 0; k < D; k++) v[k + 1] = vol * (a.m_inf_d[k] + (double)a.q[q32_index(k + 1, c, a.ntot)]);
        v[D + 1] = vol * (a.rhoE_inf_d + (double)a.q[q32_index(D + 1, c, a.ntot)]);
    }
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

template <int D>
__global__ void __launch_bounds__(256) count_nonfinite32(const float *q, int nc, int ntot, unsigned long long *cnt) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    int bad = 0;
#pragma unroll
    for (int k = 0; k < D + 2; k++) bad += !isfinite(q[q32_index(k, c, ntot)]);
    if (bad) atomicAdd(cnt, (unsigned long long)bad);
}

// ---------------------------------------------------------------------------
// single-solver kernels
// ---------------------------------------------------------------------------
template <int D>
__global__ void __launch_bounds__(256) bc_fill32(KArgs32 a) {
    bc_fill32_body<D>(a, LFM_TID(blockIdx.x));
}
// fin_nblk > 0: one block more, the last, reduces the previous step's
// fin_nblk per-block CFL maxima in a.partial into *a.d_cfl (as the one-launch
// stage does)
template <int D, int GRAD, bool VISC, bool RG, bool SL, bool PK, bool NT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 3 && SL && !RG ? 5 : 1)))
grad_vis32(KArgs32 a, int fin_nblk) {
    int nb = (int)gridDim.x;
    if (fin_nblk > 0) {
        nb -= 1;
        if ((int)blockIdx.x == nb) {
            cfl_dt_final_block<1, 256>(a.partial, fin_nblk, a.d_cfl, nullptr);
            return;
        }
    }
    grad_vis32_body<D, GRAD, VISC, RG, SL, PK, NT>(a, xcd_block((int)blockIdx.x, nb) * (int)blockDim.x + (int)threadIdx.x);
}
// 3D M1 / M2 faces: 5 waves per SIMD fit in 96 VGPRs without spills (97
// would allow 4): O-grid face kernel 1.107 -> 1.033 ms per step.  Forcing
// more waves on the update and gradient kernels was measured slower.
template <int D, int SOLVER, bool VISC, bool STORED, bool NT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 3 && SOLVER < 2 ? 5 : 1)))
face_flux32(KArgs32 a) {
    face_flux32_body<D, SOLVER, VISC, STORED, NT>(a, LFM_TID(blockIdx.x));
}
// MORE in 3D only where some cell is its own neighbour: elsewhere no 3D cell
// has more than the U entries (O-grid of 1 M cells: 149 us of updates per step
// without the rest of the list in the kernel, 154 with it)
template <int D, bool RES, int CFL, bool NT, bool MORE>
__global__ void __launch_bounds__(256) cell_update32(KArgs32 a, float A, float B, int dq_mode, double cfl_param) {
    cell_update32_body<D, RES, CFL, NT, MORE>(a, A, B, dq_mode, LFM_TID(blockIdx.x), LFM_BLK(), cfl_param);
}
// ---------------------------------------------------------------------------
// One RK stage in one launch for inviscid M1 / M2: each cell forms its faces'
// fluxes from its own and the other cells' states as it gathers them (every
// interior face by both of its cells, to the face kernel's bits: conv32),
// adds sponge and RK update and writes the new state and its boundary ghosts
// to qout, another buffer.  c: the thread's cell.
// ---------------------------------------------------------------------------
// Bound: HBM in 3D (box of 4.1 M cells: 108 B per cell and stage where a
// face's own data take 204; 821 -> 572 us per step), latency in 2D.  Faces
// whose loads are issued together in 3D: two (box one 637, two 577, three 649
// us per step); in 2D all four, since a 2D stage is bound by the latency of
// its dependent loads.
constexpr int kFusedGroup32 = 2;
template <int D, int SOLVER, int CFL, bool PK, bool HALF, bool NT>
__device__ __forceinline__ void stage32_body(const KArgs32 &a, float *qout, float A, float B, int dq_mode, const int c,
                                             const int lblk, double cfl_param) {
    constexpr int U = GatherUnroll<D>::value;
    constexpr int G = D == 3 ? kFusedGroup32 : U;
    using F = FaceOf32<D, PK, NT>;
    // a face's own data, or its key where they come from the table, are kept
    // for the CFL/dt sums after the update: read again they come from memory
    // (4.1 M-cell box: 128 -> 105 us per launch)
    constexpr bool kKeep = CFL >= 0 && !PK, kKeepKey = CFL >= 0 && PK && G < U;
    __shared__ float keep[kKeep ? U * D * 256 : 1];
    __shared__ int keys[kKeepKey ? U * 256 : 1];
    double cv = CFL == 0 ? 100.0 : 0.0;
    if (c < a.nc) {
        int key[G];
        if constexpr (PK && D == 2) {
            const uint4 v = reinterpret_cast<const uint4 *>(a.pk)[c];
            key[0] = (int)v.x;
            key[1] = (int)v.y;
            key[2] = (int)v.z;
            key[3] = (int)v.w;
        } else {
#pragma unroll
            for (int u = 0; u < G; u++) key[u] = F::load_key(a, u, c);
        }
        float qc[D + 2], dq[D + 2];
        load_q32<D>(a, c, qc);
        const float vinv = ld_once<NT>(a.vinv + c);
        load_dq32<D, NT>(a, dq_mode, c, dq);
        const float dt = (float)(*a.dt);
        const Prim32<D> sc = prim32<D>(a, qc);
        const float s = dt * vinv;
        auto add = [&](const F &f, const float (&qo)[D + 2]) {
            const Prim32<D> so = prim32<D>(a, qo);
            const Conv32<D> cf = conv32<D, SOLVER, HALF>(a, qc, sc, qo, so, f.S, f.w, f.isP);
            float r[D + 2];
            conv_rhs32<D>(a, cf, cf.pp, f.S, r);
#pragma unroll
            for (int k = 0; k < D + 2; k++) dq[k] += s * r[k];
        };
        // groups of G faces in a rolled loop, the next group's keys loaded a
        // group ahead
#pragma unroll 1
        for (int j0 = 0; j0 < U; j0 += G) {
            F f[G];
            float qo[G][D + 2];
            int next[G];
#pragma unroll
            for (int u = 0; u < G; u++) {
                f[u].load(a, j0 + u, c, key[u]);
                load_q32<D>(a, f[u].other, qo[u]);
                if (G < U) next[u] = F::load_key(a, j0 + G < U ? j0 + G + u : u, c);
                if constexpr (kKeepKey) keys[(j0 + u) * 256 + threadIdx.x] = key[u];
                if constexpr (kKeep)
#pragma unroll
                    for (int k = 0; k < D; k++) keep[((j0 + u) * D + k) * 256 + threadIdx.x] = f[u].S[k];
            }
            if (j0 == 0)
#pragma unroll
                for (int k = 0; k < D + 2; k++) dq[k] *= A;
#pragma unroll
            for (int u = 0; u < G; u++) {
                add(f[u], qo[u]);
                if (G < U) key[u] = next[u];
            }
        }
        int e1 = 0, e2 = 0;  // gather entries beyond the slots
        if (U < kMaxFaces && a.more_faces) {
            e1 = a.g_off[c] + U;
            e2 = a.g_off[c + 1];
            for (int e = e1; e < e2; e++) {
                F f;
                float qo[D + 2];
                f.load_list(a, a.g_ent[e]);
                load_q32<D>(a, f.other, qo);
                add(f, qo);
            }
        }
        float q[D + 2];
#pragma unroll
        for (int k = 0; k < D + 2; k++) q[k] = qc[k];
        finish_cell32<D, NT>(a, c, dt, B, CFL >= 0 && (dq_mode & kDqDrop), qout, q, dq);
        // the boundary ghosts of this cell (only cells of the boundary
        // submesh have any) for the next stage
        if (c < a.nsm0) {
#pragma unroll 1
            for (int j = 0; j < U; j++) {
                const int o = F::other_of(a, F::load_key(a, j, c));
                if (o >= a.nc) refresh_ghost32<D, NT>(a, o - a.nc, qout, q);
            }
            for (int e = e1; U < kMaxFaces && e < e2; e++) {
                const int ent = a.g_ent[e];
                if (ent >= 0 && (ent & kGhostFaceFlag)) refresh_ghost32<D, NT>(a, a.fN[ent & kFaceMask] - a.nc, qout, q);
            }
        }
        if constexpr (CFL >= 0) {
            CflSum32<D, CFL> t(a, q);
#pragma unroll
            for (int j = 0; j < U; j++) {
                float S[D];
                if constexpr (kKeep) {
#pragma unroll
                    for (int k = 0; k < D; k++) S[k] = keep[(j * D + k) * 256 + threadIdx.x];
                } else {
                    F f;
                    f.load(a, j, c, kKeepKey ? keys[j * 256 + threadIdx.x] : key[j % G]);
#pragma unroll
                    for (int k = 0; k < D; k++) S[k] = f.S[k];
                }
                // a placeholder's zero area adds zero to the CFL sum
                bool valid = true;
                if constexpr (CFL == 0) {
                    float s2 = 0.f;
#pragma unroll
                    for (int k = 0; k < D; k++) s2 += S[k] * S[k];
                    valid = s2 > 0.f;
                }
                t.add(S, valid);
            }
            for (int e = e1; U < kMaxFaces && e < e2; e++) {
                F f;
                f.load_list(a, a.g_ent[e]);
                t.add(f.S, true);
            }
            cv = t.value(a, q[0], vinv, cfl_param);
        }
    }
    if constexpr (CFL >= 0) block_extremum<CFL>(cv, a.partial + lblk);
}

// the face slots from the gather list: slot j of cell c holds its j-th gather
// entry's other cell, area vector out of the cell and weight, or with
// face_rec the other cell and the face's record number in the geometry table
// (2 face_rec + 1 from the N side; none: a placeholder's record)
template <int D>
__global__ void __launch_bounds__(256) build_slots32(KArgs32 a, const uint16_t *face_rec, int none, uint32_t *pk,
                                                     int32_t *nb, float *S, float *w) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= a.nc) return;
    const int e0 = a.g_off[c], ne = a.g_off[c + 1] - e0;
    constexpr int U = GatherUnroll<D>::value;
    for (int j = 0; j < U; j++) {
        FaceOf32<D, false, false> f;
        f.other = c;
        f.w = 0.5f;
        f.isP = true;
        for (int k = 0; k < D; k++) f.S[k] = 0.f;
        int rec = none;
        if (j < ne) {
            const int ent = a.g_ent[e0 + j];
            f.load_list(a, ent);
            if (pk) rec = 2 * face_rec[ent >= 0 ? (ent & kFaceMask) : ~ent] + (ent >= 0 ? 0 : 1);
        }
        if (pk) {
            pk[pk_at<D>(a.nc, j, c)] = (uint32_t)f.other | (uint32_t)rec << a.pk_shift;
            continue;
        }
        nb[slot_at<D, 1>(a.nc, j, 0, c)] = f.isP ? f.other : ~f.other;
#pragma unroll
        for (int k = 0; k < D; k++) S[slot_at<D, D>(a.nc, j, k, c)] = f.S[k];
        w[slot_at<D, 1>(a.nc, j, 0, c)] = f.w;
    }
}

// fin_nblk > 0 (a stage without CFL/dt sums): the grid has one block more,
// the last, which reduces the fin_nblk per-block CFL maxima that an earlier
// launch left in a.partial into *a.d_cfl (the final reduction of the
// previous step, whose result no stage of this step reads).
template <int D, int SOLVER, int CFL, bool PK, bool HALF, bool NT>
__global__ void __launch_bounds__(256) stage_fused32(KArgs32 a, float *qout, float A, float B, int dq_mode,
                                                     double cfl_param, int fin_nblk) {
    int nb = (int)gridDim.x;
    if constexpr (CFL < 0) {
        if (fin_nblk > 0) {
            nb -= 1;
            if ((int)blockIdx.x == nb) {
                cfl_dt_final_block<1, 256>(a.partial, fin_nblk, a.d_cfl, nullptr);
                return;
            }
        }
    } else {
        (void)fin_nblk;
    }
    const int blk = xcd_block((int)blockIdx.x, nb);
    stage32_body<D, SOLVER, CFL, PK, HALF, NT>(a, qout, A, B, dq_mode, blk * (int)blockDim.x + (int)threadIdx.x, blk,
                                           cfl_param);
}
template <int D, int MODE>
__global__ void __launch_bounds__(256) cfl_dt_cells32(KArgs32 a, double param) {
    cfl_dt_cells32_body<D, MODE>(a, param, LFM_TID(blockIdx.x), LFM_BLK());
}

// tauMC and sigmaU of every cell from the stored dudx (field read-back of a
// solver that does not store them): [D*D][nc] and [D][nc] deviations-free
// tensors (they do not depend on the free stream)
template <int D>
__global__ void __launch_bounds__(256) vis_tensor_field32(KArgs32 a, float *tmc_out, float *sU_out) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= a.nc) return;
    float du[D][D], q[D + 2], tmc[D][D], sU[D];
#pragma unroll
    for (int i = 0; i < D; i++)
#pragma unroll
        for (int j = 0; j < D; j++) du[i][j] = a.dudx[(size_t)c * a.gstride + i * D + j];
    load_q32<D>(a, c, q);
    const Prim32<D> s = prim32<D>(a, q);
    vis_tensors32<D>(a, du, s.u, a.smag ? a.smag + c : nullptr, tmc, sU);
#pragma unroll
    for (int i = 0; i < D; i++) {
        sU_out[(size_t)i * a.nc + c] = sU[i];
#pragma unroll
        for (int j = 0; j < D; j++) tmc_out[(size_t)(i * D + j) * a.nc + c] = tmc[i][j];
    }
}

// ---------------------------------------------------------------------------
// batched kernels: one launch covers several resident solvers of one scheme
// class; each solver computes exactly what its single launch computes.  A
// block's solver and its number within that solver lie together: one load
// before the solver's arguments can be asked for.
// ---------------------------------------------------------------------------
struct BatchMap {
    const int2 *slot;  // [nblocks] solver (sorted) and local block
};

__device__ __forceinline__ void batch_slot(const BatchMap &m, int &r, int &lblk) {
    const int2 v = m.slot[LFM_BLK()];
    r = v.x;
    lblk = v.y;
}

template <int D, int GRAD, bool VISC, bool RG, bool NT>
__global__ void __launch_bounds__(256) grad_vis32_b(const KArgs32 *args, BatchMap m) {
    int r, lb;
    batch_slot(m, r, lb);
    grad_vis32_body<D, GRAD, VISC, RG, false, false, NT>(args[r], lb * 256 + threadIdx.x);
}
// (batch members are undecomposed: their tensors are never stored)
template <int D, int SOLVER, bool VISC, bool NT>
__global__ void __launch_bounds__(256) face_flux32_b(const KArgs32 *args, BatchMap m) {
    int r, lb;
    batch_slot(m, r, lb);
    face_flux32_body<D, SOLVER, VISC, false, NT>(args[r], lb * 256 + threadIdx.x);
}
// CFL 1: the last stage, with compute_cfl at each solver's own deltaT
template <int D, int CFL, bool NT>
__global__ void __launch_bounds__(256) cell_update32_b(const KArgs32 *args, BatchMap m, float A, float B,
                                                       int dq_mode) {
    int r, lb;
    batch_slot(m, r, lb);
    const KArgs32 &a = args[r];
    cell_update32_body<D, false, CFL, NT, true>(a, A, B, dq_mode, lb * 256 + threadIdx.x, lb, CFL >= 0 ? *a.dt : 0.0);
}
// one-launch stage over a batch (inviscid M1 / M2), each member from one
// of its state buffers into the other: flip 0 from a.q into a.q_alt, flip 1
// back
template <int D, int SOLVER, int CFL, bool NT>
__global__ void __launch_bounds__(256) stage_fused32_b(const KArgs32 *args, BatchMap m, float A, float B, int dq_mode,
                                                       int flip) {
    int r, lb;
    batch_slot(m, r, lb);
    KArgs32 a = args[r];
    float *qout = flip ? a.q : a.q_alt;
    if (flip) a.q = a.q_alt;
    const int c = lb * 256 + threadIdx.x;
    const double dt = CFL >= 0 ? *a.dt : 0.0;
    // members may hold either slot form
    if (a.pk && (SOLVER == 1 || a.pk_half))
        stage32_body<D, SOLVER, CFL, true, true, NT>(a, qout, A, B, dq_mode, c, lb, dt);
    else if (a.pk)
        stage32_body<D, SOLVER, CFL, true, SOLVER == 1, NT>(a, qout, A, B, dq_mode, c, lb, dt);
    else
        stage32_body<D, SOLVER, CFL, false, SOLVER == 1, NT>(a, qout, A, B, dq_mode, c, lb, dt);
}
// one block per solver: max of its partials into its CFL scalar
static __global__ void __launch_bounds__(256) cfl_final32_b(const KArgs32 *args) {
    __shared__ double sh[256];
    const KArgs32 &a = args[blockIdx.x];
    double v = 0.0;
    // min / max are exact in any order: keep several loads in flight
#pragma unroll 8
    for (int i = threadIdx.x; i < a.nblk_cells; i += blockDim.x) {
        const double o = a.partial[i];
        if (v < o) v = o;
    }
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int st = blockDim.x / 2; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st && sh[threadIdx.x] < sh[threadIdx.x + st]) sh[threadIdx.x] = sh[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) *a.d_cfl = sh[0];
}

// launchers (defined in solver_fp32p.hip)
template <int D>
void launch_bc32(Solver *s);
template <int D>
void launch_gradvis32(Solver *s, bool full, bool fin = false);
template <int D>
void launch_flux32(Solver *s);
template <int D>
void launch_update32(Solver *s, double A, double B, int dq_mode, bool res, bool accumulate_res,
                     const Solver::CflJob *cfl);
template <int D>
void launch_cfl_dt32(Solver *s, int mode, double param, double *out, double *dt_dst);
template <int D>
void launch_build_slots32(Solver *s, const uint16_t *face_rec, int none, uint32_t *pk, int32_t *nb, float *S,
                          float *w);
template <int D>
void launch_stage_fused32(Solver *s, double A, double B, int dq_mode, const float *qin, float *qout,
                          const Solver::CflJob *cfl, bool fin);

}  // namespace lfm
