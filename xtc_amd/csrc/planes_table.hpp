// SPDX-License-Identifier: BSD-3-Clause
// Compiled instances of gemm_planes (gemm_planes.hpp), one table per
// translation unit so that they compile in parallel.
#pragma once
#include "gemm_planes.hpp"
#include "registry.hpp"

namespace xtc_hip {

struct PlanesEntry {
  int dtype;            // 0 fp32, 1 bf16
  int bm, bn, wgm, wgn; // the tile's block and waves (any slab depth)
  int waves;            // of a k-group of the kernel
  int kg;               // k-groups of a workgroup
  int conv, bt, vec;
  int ring;             // register sets of global loads in flight
  GemmLaunch launch;
};

template <typename T, int BM, int BN, int BK, int WGM, int WGN, bool CONV, bool BT, bool VEC, int RING, int KG>
void launch_planes(const GemmArgs& a, dim3 grid, hipStream_t s) {
  hipLaunchKernelGGL((gemm_planes<T, BM, BN, BK, WGM, WGN, CONV, BT, VEC, RING, KG>), grid, dim3(KG * WGM * WGN * 64), 0, s, a);
}

template <typename T, int BM, int BN, int BK, int WGM, int WGN, bool CONV, bool BT, bool VEC, int RING, int KG = 1>
PlanesEntry planes_instance(int tile_wgm = WGM, int tile_wgn = WGN) {
  return PlanesEntry{sizeof(T) == 4 ? 0 : 1, BM, BN, tile_wgm, tile_wgn, WGM * WGN, KG, CONV, BT, VEC, RING,
                     &launch_planes<T, BM, BN, BK, WGM, WGN, CONV, BT, VEC, RING, KG>};
}

// Filled by planes_*.hip.
const PlanesEntry* planes_f32(int* count);
const PlanesEntry* planes_bf16(int* count);
const PlanesEntry* planes_conv(int* count);

}  // namespace xtc_hip
