// SPDX-License-Identifier: BSD-3-Clause
// gemm_planes instances for implicit-GEMM conv2d.
#include "planes_table.hpp"

namespace xtc_hip {

const PlanesEntry* planes_conv(int* count) {
  static const PlanesEntry table[] = {
      planes_instance<float, 64, 64, 32, 2, 2, true, false, true, 1>(),
      planes_instance<float, 64, 64, 32, 2, 2, true, false, false, 1>(),
      planes_instance<float, 128, 64, 32, 4, 2, true, false, false, 1>(),
      planes_instance<__bf16, 64, 64, 64, 2, 2, true, false, true, 2>(),
      planes_instance<__bf16, 64, 64, 64, 2, 2, true, false, false, 1>(),
      planes_instance<__bf16, 64, 64, 64, 2, 4, true, false, true, 2>(2, 2),
      planes_instance<__bf16, 128, 64, 64, 4, 2, true, false, true, 2>(2, 2),
      planes_instance<__bf16, 128, 64, 64, 4, 2, true, false, true, 1, 2>(2, 2),
      planes_instance<__bf16, 128, 128, 64, 2, 4, true, false, true, 2>(2, 2),
      planes_instance<__bf16, 128, 128, 64, 2, 4, true, false, true, 1, 2>(2, 2),
  };
  *count = (int)(sizeof(table) / sizeof(table[0]));
  return table;
}

}  // namespace xtc_hip
