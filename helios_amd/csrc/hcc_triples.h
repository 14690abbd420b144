// (T) correction kernel (hcc_triples.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>

namespace hcc {

// Per-molecule operands of the (T) kernel (row-major device arrays).
struct TripMol {
  int n, o, v, pad;
  const double* A;    // (xp|yd) at [p][x][y][d]  (o v^3)
  const double* B;    // (ql|rz) at [q][l][r][z]  (o^3 v)
  const double* L;    // (ia|jb) at [i][j][a][b]  (o^2 v^2)
  const double* t1;   // [i][a]
  const double* t2;   // [i][j][a][b]
  const double* F;    // MO Fock matrix (n x n), orbital energies on its diagonal
};

constexpr int kTripMaxOV = 32;   // o, v <= 32

// Size classes of the work items, a kernel each: v <= 16, v <= 24 and v <= 32.
int trip_class(int v);
// items: per work item (molecule, occupied triple i >= j >= k packed as
// i | j << 8 | k << 16), the items of class 0 first, then 1, then 2 (count[3]
// of each), a molecule's items consecutive: [range.x, range.y); cus: compute
// units of the device; part: 2 per item; out: 2 per molecule (E[T], E[ST])
hipError_t launch_triples(const TripMol* mols, int nm, const int2* range, const int2* items, const int* count, int cus,
                          double* part, double* out, hipStream_t s);

}  // namespace hcc
