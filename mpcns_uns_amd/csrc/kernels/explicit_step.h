#pragma once
// Explicit stage of the fused step on the resident state (explicit_step.hip): its layouts and launch entry points.
//
//   rec  per cell, rs doubles a row (a multiple of 8): the primitives of every ion (5 each), the reconstructed induced
//        field (3) and the cell centre (3).  Two ions fill one 128-byte line exactly, so the neighbour gather of the
//        gradients, which reads all of it, takes one line per face.
//   geo  per face, 32 bytes (DevMesh): unit normal and |A|, so that a gathered face needs neither the parts of two arrays
//        nor a division.
//   FS   per (cell, face) entry and ion: the five primitives of the cell's linear state at that face.  The limited
//        gradients are used for nothing else in the step, and a face reads two rows of 40 bytes per ion where it
//        gathered two cells' primitives and gradients (2 x 160 bytes, each cell's read again by all of its faces).
//   FA   per face and ion: the flux through the face (5).
//   Ef   per face, 32 bytes: the EMF candidate (3) and Phi / |A|, what the edge sum reads of a face besides geo.
#include "kernels.h"
#include "krylov.h"

namespace mhdg
{
struct StepFields
{
    double *rec, *Btot, *uplus, *J, *alpha, *FS, *FA, *Ef;
    const int2 *fent;   // per face: the c2f entry that sees it outward, inward (-1: none)
    const int8_t *fcls; // per face: kFluxNone, kFluxInner, kFluxLeft (the inside cell sees it outward), kFluxRight
    int32_t rs, ns;
};
// What a stage reads and writes: a state (U, Phi), the fields formed from it, the edge EMF and the time step
struct StepRun
{
    double *U[kMaxSpecies], *Phi;
    StepFields F;
    double *E, *dt_part, *dt_dev;
};
// How far a stage goes: no update of the state, of its cells, of its cells and faces
enum StageEnd { kStageNone, kStageCells, kStageState };
enum : int8_t { kFluxNone = 0, kFluxInner = 1, kFluxLeft = 2, kFluxRight = 3 };
inline int32_t step_row(int32_t ns) { return (5 * ns + 6 + 7) / 8 * 8; }
// The bytes of a step's fields and tables, about: 1170 a tetrahedron with two ions, 3750 with ten
inline size_t step_bytes(int32_t ns, size_t cells, size_t faces, size_t entries)
{
    return 8 * (size_t(step_row(ns)) * cells + 5 * size_t(ns) * (entries + faces + cells) + 20 * faces + 20 * cells);
}
// Up to this many of them (457k tetrahedra with two ions, 143k with ten) the XCDs take one range each of the step's and the
// products' blocks (near_block, dev.h) and the products' first launch is flux_cell's.  Microseconds without and with the
// order, forced either way.  Two ions, an explicit step: 9.5k tetrahedra 40.5, 36.8; 60k 67.8, 59.3; 150k 127, 114;
// 290k 246, 239; 435k 362, 355; above the line 484k 401, 396; 683k 556, 562; 1.06M 850, 890; 7.8M 6230, 6454.  Ten ions, an
// explicit step and a mixed Hall step (with flux_cell): 60k 164, 519 and 164, 492; 131k 371, 770 and 371, 743; above 150k 421, 918 and
// 426, 905; 387k 1078, 1979 and 1090, 1969.  The line lies where the gain ends for every ion count: above it data passes
// through the L2s and the MALL from HBM, which is read best in one sweep by all XCDs.
constexpr size_t kXcdBytes = size_t(512) << 20;

__global__ void k_face_geo(DevMesh d, double *geo);
__global__ void k_face_entries(DevMesh d, int2 *fent, int8_t *fcls);
__global__ void k_rec_get(const double *rec, int32_t rs, int32_t first, int32_t n, int32_t nc, double *out);
} // namespace mhdg
