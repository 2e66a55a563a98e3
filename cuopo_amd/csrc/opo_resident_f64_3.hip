// opo_resident_f64_3.hip -- the resident crystal pass, complex128 fields, three equations.
#include "opo_resident.h"

namespace opo {
int launch_resident_f64_3(int N1, int N2, int ce, int re, const OpoInst *insts, const ResArgs &a, int grid,
                            hipStream_t s) {
  return launch_resident_t<double, 3>(N1, N2, ce, re, insts, a, grid, s);
}
}  // namespace opo
