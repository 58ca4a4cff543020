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
    double *e_part, *c_part;              // per block: {dt, E_inf (3, summed over the steps)} of the edges, dt of the cells
    double *f_part, *g_part;              // per block, summed over the steps: free stream (10) from the fluxes, the gradients
    double *dtb;                          // 16: adjoint of the time step, then (W 10, B_tot 3) of the cell that sets it
    int32_t *dt_cell;                     // that cell (-1: none), and how many sweeps did not find it
    double *sums;                         // 23: the sums of e_part's E_inf, f_part and g_part
};
} // namespace mhdg
