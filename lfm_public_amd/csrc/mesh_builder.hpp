// mesh_builder.hpp -- host set-up of one partition: polyMesh -> SoA solver
// layout in the reference's cell and face processing order.
#pragma once

#include <algorithm>
#include <cstdint>
#include <string>
#include <vector>

#include "lfm_hip.h"

namespace lfm {

constexpr int kMaxFaces = 6;        // FACE_CNT in {3,4,5,6} (src/mesh_solver.cpp:56-74)
constexpr int kGhostSubmesh = 10000; // MAX_MPI_RANKS, api/mpi_env.h:4
// gather-list encoding: entry f >= 0 (cell is P), ~f (cell is N); P entries
// of faces whose N is a boundary (not a processor) ghost carry kGhostFaceFlag.
constexpr int32_t kGhostFaceFlag = 1 << 30;
constexpr int32_t kFaceMask = kGhostFaceFlag - 1;

// The reference's two submeshes of one partition, flattened into one index
// space: cells [0, nsm0) are submesh 0 (boundary), [nsm0, nc) submesh 1,
// boundary ghosts [nc, nc+ng).  Faces are listed in the order the
// reference's one_rk_step loops visit them (cell by cell, valid slots in
// reorder_faces order), each once, oriented from P (the visiting cell) to N.
// One processor-patch neighbour of a partition: the reference's MPI ghost
// bookkeeping (cfd_v0.cpp:432-540, 587-748) and neighbour-centre exchange
// (mesh_reader.cpp:390-612).  Halo ghosts are one per processor face.
struct HaloNbr {
    int rank = -1;
    std::vector<int32_t> ghost;       // ghost index (0-based, >= ng_bnd) per processor face
    std::vector<int32_t> face;        // layout face index per processor face
    std::vector<int32_t> key;         // global face key per processor face
    std::vector<int32_t> cell;        // local owner cell (combined index) per processor face
    std::vector<double> xf, xc;       // [3*n] face and owner-cell centres
    std::vector<int32_t> send_cells;  // local cells adjacent to this rank, ascending
    std::vector<int32_t> recv_src;    // after import: record in the neighbour's send list, per face
    bool imported = false;
};

struct SolverLayout {
    int D = 2;
    int nc = 0, nsm0 = 0, ng = 0, nf = 0, max_faces = 0;
    int ng_bnd = 0;                     // boundary ghosts [0, ng_bnd); halo ghosts [ng_bnd, ng)
    int rank = -1;                      // partition rank (-1: undecomposed)
    std::vector<HaloNbr> halo;
    std::vector<int32_t> orig, comb;    // combined -> original cell id, and back
    std::vector<int32_t> fP, fN;        // [nf]
    std::vector<double> S, d, w;        // S,d: [D][nf] SoA; w: [nf]
    std::vector<double> vinv, sigma;    // [nc]
    // Smagorinsky constant -2 (0.16 V^(1/3))^2 each cell's stored tauMC ends
    // with (empty when laminar): its own, or for a cell with no face of its
    // own to process, that of the cell whose face touched it last
    std::vector<double> smag;
    std::vector<double> centre, volume; // [nc*3], [nc] (combined order)
    // gather lists: per cell, faces touching it in processing order;
    // entry f >= 0: the cell is P of face f; entry ~f: the cell is N.
    std::vector<int32_t> g_off, g_ent;
    // slot lists: per cell, all valid faces in reorder_faces slot order
    // (CFL / dt loops, cfd_v0.cpp:2895, 2921), same signed encoding.
    std::vector<int32_t> s_off, s_ent;
    // boundary ghosts: interior cell (combined index) and BC role
    std::vector<int32_t> ghost_cell, ghost_role;
    // per boundary ghost: its patch, and the face postProcForces reads for
    // it (cfd_v0.cpp:3169-3233): boundaries[patch][i] keeps the slot the
    // face had before reorder_faces, the cell's arrays are indexed after it,
    // so the face read is whichever moved into that slot (ref), or the
    // ghost's own face (own).  nb: combined index of the neighbour read;
    // S, d: [D][ng_bnd] as the cell sees that face.
    std::vector<int32_t> ghost_patch;
    std::vector<int32_t> patch_role;  // [n_patches] LFM_BC_* of the polyMesh patches
    std::vector<int32_t> gf_ref_nb;
    std::vector<double> gf_ref_S, gf_ref_d, gf_own_S, gf_own_d;
    // initial conservatives [(D+2)][nc] combined order
    std::vector<double> q0;
};

// Builds the layout and the initial state; returns an empty string on
// success or an error message.
std::string build_layout(const lfm_polymesh &m, const lfm_partition *part, const lfm_params &prm,
                         const double *p, const double *T, const double *U3, const double *alpha,
                         SolverLayout &L);

// Applies a neighbour's set-up message to halo entry `ni`: d and the linear
// weight of its processor faces (mesh_reader.cpp:577-605, cfd_v0.cpp:
// 800-855) and the receive order (the neighbour's ascending send list).
std::string halo_import(SolverLayout &L, int ni, int n, const int32_t *key, const int32_t *cell,
                        const double *disp);

// The distinct face records (area vector and weight as T holds them) of a
// layout, for kernels that read a small table instead of per-face data: a
// uniform mesh has a few dozen.  n = 0 where there are more than max_n; rec:
// each face's record.
template <typename T>
struct FaceTable {
    int n = 0;
    std::vector<T> S, w;        // [n][D], [n]
    std::vector<uint16_t> rec;  // [nf]
};
template <typename T>
FaceTable<T> face_table(const SolverLayout &L, int max_n);

// the most gather entries of a cell (a cell that is its own neighbour has two
// for each such face)
inline int max_entries(const SolverLayout &L) {
    int m = 0;
    for (int c = 0; c < L.nc; c++) m = std::max(m, L.g_off[c + 1] - L.g_off[c]);
    return m;
}

// whether some cell is its own neighbour (a cyclic pair one cell apart): it has
// two gather entries for such a face, as its P and as its N
inline bool own_neighbour(const SolverLayout &L) {
    for (int f = 0; f < L.nf; f++)
        if (L.fP[f] == L.fN[f]) return true;
    return false;
}

// bits that hold an index below n
inline int index_bits(long n) {
    int b = 1;
    while ((1L << b) < n) b++;
    return b;
}

// What one RK stage touches, in bytes, each array once.
struct StageShape {
    int D = 3;
    size_t word = 4, nc = 0, nf = 0;  // bytes per value; cells, faces
    bool one_launch = false;          // stage_fused32 / 64, otherwise gradients, fluxes and update
    bool packed = false;              // slots of one word over a face table
    size_t grad_values = 0;           // values of a cell's gradient record (0: no gradients)
};
inline size_t stage_footprint(const StageShape &s) {
    const size_t D = s.D, w = s.word, U = D == 2 ? 4 : 6, key = sizeof(int32_t);
    size_t cell = (2 * (D + 2) + 2) * w, face = 0;  // state, RK register, 1/V, sponge
    if (s.one_launch) {
        // second state; slots: one word each, or a face's own data
        cell += (D + 2) * w + U * (s.packed ? key : key + (D + 1) * w);
    } else {
        // face fluxes, S, d, w, both cells; the update's gather entries
        face += (3 * D + 3) * w + 2 * key;
        cell += U * key;
        // gradients: the record, and one word more per entry (the cell it leads
        // to, or a packed slot).  Unpacked slots are not counted: gradients read
        // them only past the line that this footprint is held against.
        if (s.grad_values) cell += s.grad_values * w + U * key;
    }
    return s.nc * cell + s.nf * face;
}
// Streams are marked non-temporal from 330 MB touched per stage: below, part of
// what one launch writes is still in the 256 MB Infinity Cache when the next
// reads it, and marking loses that; above, marking keeps the gathered
// neighbours in L2.  us per step plain / marked (MB per stage): FP32 3D box
// 117 / 150 (81), 229 / 307 (193), 383 / 424 (275), 573 / 566 (377), 978 / 946
// (651); viscous 251 / 306 (161), 526 / 542 (313), 659 / 670 (394), 923 / 890
// (541); FP32 O-grid 182 / 218 (92), 327 / 377 (186), 365 / 399 (204), 535 / 548
// (286), 609 / 615 (327), 709 / 695 (368), 1015 / 957 (516), M2AUSM 447 / 484
// (220), 645 / 655 (308); FP32 annulus 317 / 389 (177); FP64 annulus 181 / 188
// (60), 343 / 384 (139), 881 / 837 (356); FP64 O-grid 382 / 441 (157), 756 / 789
// (314), 1440 / 1363 (558); FP64 box 386 / 460 (225), 645 / 654 (336), 915 / 903
// (478).
inline bool outgrows_cache(size_t bytes) { return bytes > (size_t)330 * 1000 * 1000; }

// Gas constants derived as set_init_conditions does (cfd_v0.cpp:880-902).
struct Gas {
    double R, R_inv, gamma, gm1, cp, mu, pr_inv;
    double p_inf, T_inf, rho_inf, E_inf, U_inf[3];
};
Gas derive_gas(const lfm_params &prm);

// Runge-Kutta 2N tables (cfd_v0.cpp:86-128); returns the stage count.
int rk_tables(int rk_order, double A[5], double B[5]);

}  // namespace lfm
