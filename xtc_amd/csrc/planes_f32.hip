// SPDX-License-Identifier: BSD-3-Clause
// gemm_planes instances for fp32 matmuls.
#include "planes_table.hpp"

namespace xtc_hip {

const PlanesEntry* planes_f32(int* count) {
  static const PlanesEntry table[] = {
      planes_instance<float, 256, 128, 32, 4, 2, false, false, true, 1>(),
      planes_instance<float, 128, 256, 32, 2, 4, false, false, true, 1>(),
      planes_instance<float, 128, 128, 32, 2, 4, false, false, true, 1>(),
      planes_instance<float, 64, 64, 32, 2, 2, false, false, true, 1>(),
      planes_instance<float, 64, 64, 32, 2, 2, false, false, false, 1>(),
      planes_instance<float, 256, 128, 32, 4, 2, false, true, true, 1>(),
      planes_instance<float, 128, 256, 32, 2, 4, false, true, true, 1>(),
      planes_instance<float, 128, 128, 32, 2, 4, false, true, true, 1>(),
      planes_instance<float, 64, 64, 32, 2, 2, false, true, true, 1>(),
  };
  *count = (int)(sizeof(table) / sizeof(table[0]));
  return table;
}

}  // namespace xtc_hip
