// opo_chip_f64.hip -- the whole-chip crystal pass, complex128 fields.
#include "opo_chip.h"

namespace opo {
int launch_chip_f64(int N1, int N2, int NF, const OpoInst *insts, const ResArgs &a, hipStream_t s) {
  if (N1 == 64 && N2 == 512)
    return NF == 3 ? launch_chip_k<double, 64, 512, 3, 8, 8>(insts, a, s) : launch_chip_k<double, 64, 512, 2, 8, 8>(insts, a, s);
  if (N1 == 64 && N2 == 1024)
    return NF == 3 ? launch_chip_k<double, 64, 1024, 3, 8, 8>(insts, a, s) : launch_chip_k<double, 64, 1024, 2, 8, 8>(insts, a, s);
  if (N1 == 64 && N2 == 2048)
    return NF == 3 ? launch_chip_k<double, 64, 2048, 3, 8, 8>(insts, a, s) : launch_chip_k<double, 64, 2048, 2, 8, 8>(insts, a, s);
  if (N1 == 128 && N2 == 2048)
    return NF == 3 ? launch_chip_k<double, 128, 2048, 3, 8, 8>(insts, a, s) : launch_chip_k<double, 128, 2048, 2, 8, 8>(insts, a, s);
  return (int)hipErrorInvalidValue;
}
}  // namespace opo
