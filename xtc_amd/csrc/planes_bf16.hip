// SPDX-License-Identifier: BSD-3-Clause
// gemm_planes instances for bf16 matmuls (one plane).
#include "planes_table.hpp"

namespace xtc_hip {

const PlanesEntry* planes_bf16(int* count) {
  static const PlanesEntry table[] = {
      planes_instance<__bf16, 64, 64, 64, 2, 2, false, false, false, 1>(),
      planes_instance<__bf16, 64, 64, 64, 2, 2, false, false, true, 2>(),
      planes_instance<__bf16, 64, 64, 64, 2, 2, false, true, true, 2>(),
      planes_instance<__bf16, 64, 64, 64, 2, 4, false, false, true, 2>(2, 2),
      planes_instance<__bf16, 64, 64, 64, 2, 4, false, true, true, 2>(2, 2),
      planes_instance<__bf16, 128, 128, 64, 2, 4, false, false, true, 2>(2, 2),
      planes_instance<__bf16, 128, 128, 64, 2, 4, false, true, true, 1>(2, 2),
      planes_instance<__bf16, 128, 128, 64, 2, 4, false, false, true, 1, 2>(2, 2),
      planes_instance<__bf16, 128, 128, 64, 2, 4, false, true, true, 1, 2>(2, 2),
  };
  *count = (int)(sizeof(table) / sizeof(table[0]));
  return table;
}

}  // namespace xtc_hip
