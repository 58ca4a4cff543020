#pragma once
// Flux of an edge vector and the cell field of the flux in one launch (flux_cell.hip), on meshes of one cell shape.
#include "kernels.h"

namespace mhdg
{
// Per cell: its edges (6 of a tetrahedron, 12 of a hexahedron), and per (cell, face) entry the face's edges among them in
// the order of the face's row: 4 bits each from bit 0, their signs from bit 16, kOwnFace if the cell writes the face's flux.
struct CellEdges
{
    const int32_t *edge = nullptr; // null: not built
    const uint32_t *face = nullptr;
};
constexpr uint32_t kOwnFace = 1u << 20;

// the tables; counts[0] the cells with too many edges, counts[1] the faces written
template <int DEG> __global__ void k_cell_edges(DevMesh d, int32_t *edge, uint32_t *face, int32_t *counts);
// phi_f = sum over the face's edges of sgn x_e, x = v, or dir ? 0 : v invdiag; b_c = sum_k recon_k phi_{f_k}: k_d1 then
// k_bcell_g, bit for bit
template <int DEG>
__global__ void k_flux_cell(DevMesh d, CellEdges t, const double *v, const double *invdiag, const int8_t *dir, double *phi, double *b);
// k_d1_f32 then k_bcell_f32_g, bit for bit
template <int DEG> __global__ void k_flux_cell_f32(DevMesh d, CellEdges t, const float *recon, const float *pv, float *phi, float *b);
} // namespace mhdg
