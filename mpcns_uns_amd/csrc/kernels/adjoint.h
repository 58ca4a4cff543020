#pragma once
// Device pointers of the reverse sweep of the explicit step (adjoint.hip).
//
// An entity's adjoint parts for its neighbours go to slots that the neighbours gather in a fixed order (no atomics):
//   FS   (StepFields) per (cell, face) entry and ion, 5: a face replaces the cell's states at it by their adjoints, then
//        the cell replaces these by the adjoints of its stencil neighbours' primitives; each entry is read and written
//        by one thread at a time, so the three share one array.
//   sE   per entry, 9: the face EMF's parts of the cell's u+, B_tot and B_ind.
//   sPhi per entry: the reconstructed field's part of the face's flux.
//   eF   per edge-face entry, 4: the edge's parts of E_f and of the induced flux.    eC per edge-cell entry, 3: of u+.
#include <cstdint>

namespace mhdg
{
struct AdjFields
{
    const int32_t *opp;                   // per c2f entry: the entry across whose cell has this cell in its stencil (-1: none)
    const int32_t *f2e_pos;               // per f2e entry: its position in the edge's e2f row
    const int32_t *cec_ptr, *cec;         // cell -> its edge-cell entries
    int32_t all_active;                   // every face has a cell (Faraday leaves the others alone)
    double *Wb, *rv;                      // per cell, 10: adjoint of the primitives; of the right-hand side, over the volume
    double *Jv, *Btb;                     // per cell, 3: adjoint of the current over the volume; of B_tot
    double *sE, *sPhi, *eF, *eC;
    double *Phib, *PhiAddb, *Baddb;
    // adjoint of the time step: per 256-face block, per cell, per 256-cell block; then (dtb, 14) the total and the
    // derivatives of the step of the cell that sets it by its W (10) and B_tot (3)
    double *dt_f, *dt_c, *dt_cp, *dtb;
    int32_t *dt_cell;                     // that cell (-1: none), and how many sweeps did not find it
    // The free stream's and the inflow EMF's adjoints come from the few 256-entity blocks that touch the inflow: a block's
    // slot or -1, the block of a slot, the rows (10 per entity) of a slot's entities, the blocks' sums
    const int32_t *fs_face, *fs_cell, *inflow_edge, *block_face, *block_cell;
    int32_t n_f, n_c, n_e;
    double *fsf, *fsc, *f_part, *g_part, *e_part;
    const int32_t *wall_slot, *wall_cell; // per cell: its number among the cells with a wall in the stencil, or -1; their list
    int32_t n_wall;
    double *mirror;                       // per wall cell: the parts of the first ion's velocities (3) in its gradients
    double *sums;                         // 14: free stream (10), inflow EMF (3), the second of dt_cell
};
} // namespace mhdg
