// opo_chip_f64.hip -- the whole-chip crystal pass, complex128 fields.
#include "opo_chip.h"

namespace opo {
int launch_chip_f64(int N1, int N2, int NF, int ce, const OpoInst *insts, const ResArgs &a, hipStream_t s) {
  if (N1 == 64 && N2 == 512) return launch_chip_n<double, 64, 512>(NF, ce, insts, a, s);
  if (N1 == 64 && N2 == 1024) return launch_chip_n<double, 64, 1024>(NF, ce, insts, a, s);
  if (N1 == 64 && N2 == 2048) return launch_chip_n<double, 64, 2048>(NF, ce, insts, a, s);
  if (N1 == 128 && N2 == 2048) return launch_chip_n<double, 128, 2048>(NF, ce, insts, a, s);
  return (int)hipErrorInvalidValue;
}
}  // namespace opo
