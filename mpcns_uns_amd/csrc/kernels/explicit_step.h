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
// Up to this many bytes of a step's fields and tables (620k tetrahedra, two ions) the XCDs take one range each of the
// step's and the products' blocks (near_block, dev.h).  Microseconds per explicit step without and with: 9.5k tetrahedra 40.0, 35.9; 60k 67.7,
// 59.3; 150k (125 MB) 126.7, 114.2; 484k (400 MB) 399.6, 395.7; 1.09M (910 MB) 888, 919; 7.8M 6230, 6454: data that passes through
// the L2s and the MALL from HBM is read best in one sweep by all XCDs.
constexpr size_t kXcdBytes = size_t(512) << 20;
inline int32_t step_row(int32_t ns) { return (5 * ns + 6 + 7) / 8 * 8; }

__global__ void k_face_geo(DevMesh d, double *geo);
__global__ void k_face_entries(DevMesh d, int2 *fent, int8_t *fcls);
__global__ void k_rec_get(const double *rec, int32_t rs, int32_t first, int32_t n, int32_t nc, double *out);
} // namespace mhdg
