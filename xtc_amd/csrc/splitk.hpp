// SPDX-License-Identifier: BSD-3-Clause
// Split-K completion inside the GEMM launch: the workgroup that stores the
// last partial tile of an output tile sums all of them, so a split-K GEMM
// is one kernel (no second reduce launch, no launch gap).
//
// Protocol, per output tile with `splits` workgroups along K:
//   1. every workgroup stores its fp32 partial tile to the workspace with the
//      agent-scope cache policy (gfx950: global_store ... sc1, written
//      through to the device coherence point, so the other XCDs' L2s never
//      hold it dirty): 16-byte stores where the tile allows, else the 4-byte
//      agent-scope atomic store, which compiles to the same policy;
//   2. every thread waits for its stores to complete (vmcnt(0)), the
//      workgroup synchronises and one lane increments the tile's arrival
//      counter (agent-scope atomic add);
//   3. the workgroup that sees splits-1 is the last one: it reads the
//      partials back with sc1 loads (16 bytes, 16 in flight per lane, or
//      4-byte agent-scope atomic loads), sums partial[0..splits-1] in split order (the result does not
//      depend on which workgroup arrived last), applies bias / relu, stores C
//      and sets the counter back to 0 for the next launch.
// Every access to the published data carries the agent-scope policy, so no
// L2 write-back (buffer_wbl2) or invalidate (buffer_inv) is needed: a
// release/acquire fence at agent scope would write back and invalidate the
// whole L2 of the XCD in every workgroup, which costs more than the reduce.
// The 16-byte accesses halve the instructions of the 8-byte atomic pairs
// they replaced and make the C5 MLP 4 % faster.
// Counters start at zero (the host clears them with a kernel when it
// allocates them, and before every call of the no-allocation entry point)
// and every launch leaves them at zero.  Two launches that share the
// counters and the workspace must not overlap: the host keeps both per
// launch stream.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace xtc_hip {

namespace splitk {
typedef float f32x4 __attribute__((ext_vector_type(4)));
// s_waitcnt vmcnt(0), expcnt and lgkmcnt left at their maximum (no wait)
constexpr int kWaitVm0 = (7 << 4) | (15 << 8);
}  // namespace splitk

__device__ __forceinline__ void splitk_store(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ float splitk_load(const float* p) {
  return __hip_atomic_load(const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// 16-byte aligned p: one 16-byte store with the agent-scope cache policy
// (sc1, what an agent-scope atomic store of 8 bytes compiles to), issued from
// asm because no atomic is 16 bytes wide; its completion is waited for in
// splitk_arrive (s_waitcnt vmcnt(0)).  The compiler does not count wait
// states into inline asm, so the asm opens with 24 of them: the most an
// MFMA result needs before a memory instruction reads it (16-pass XDL ops
// need 19).  The trailing s_nop covers the one wait state a VALU write of
// the data registers needs after a store of more than 8 bytes.
__device__ __forceinline__ void splitk_store4(float* p, splitk::f32x4 v) {
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\tglobal_store_dwordx4 %0, %1, off sc1\n\ts_nop 0" ::"v"(p), "v"(v)
               : "memory");
}

// The 16 bytes at byte `off` past the uniform address p, with the agent-scope
// cache policy (sc1).  A buffer load, so that the compiler counts it and many
// stay in flight.
__device__ __forceinline__ splitk::f32x4 splitk_load4(const float* p, unsigned off) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  constexpr int kWords = 0x00027000, kSc1 = 16;  // raw 32-bit data format; gfx940 cache policy bit sc1
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, 0x7fffffff, kWords);
  return __builtin_bit_cast(splitk::f32x4, (u32x4)__builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)off, 0, kSc1));
}

__device__ __forceinline__ float splitk_sum1(const float* p, size_t stride, int splits) {
  constexpr int kBatch = 8;
  float v = 0.f;
  for (int s0 = 0; s0 < splits; s0 += kBatch) {
    float t[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j)
      if (s0 + j < splits) t[j] = splitk_load(p + (size_t)(s0 + j) * stride);
#pragma unroll
    for (int j = 0; j < kBatch; ++j)
      if (s0 + j < splits) v += t[j];
  }
  return v;
}

// Step 2: true in the last-arriving workgroup only.  Called by every thread
// of the workgroup (1-D blocks) after its splitk_store calls.  `flag` is one
// LDS word that no thread touches between the first barrier here and the
// return (a kernel whose LDS is full passes a word of its own, free by then).
__device__ __forceinline__ bool splitk_arrive_in(unsigned* counter, int splits, unsigned* flag) {
  __builtin_amdgcn_s_waitcnt(splitk::kWaitVm0);
  __syncthreads();
  if (threadIdx.x == 0)
    *flag = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(splits - 1)
                ? 1u
                : 0u;
  __syncthreads();
  return *flag != 0;
}

__device__ __forceinline__ bool splitk_arrive(unsigned* counter, int splits) {
  __shared__ unsigned s_last;
  return splitk_arrive_in(counter, splits, &s_last);
}

// Ends the protocol in the last workgroup (after its reads of the partials).
__device__ __forceinline__ void splitk_release(unsigned* counter) {
  if (threadIdx.x == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The last workgroup's sum over one BM x BN output tile at (m0, n0):
// C[m][n] = epilogue( sum_s partial[s * plane + m * ldp + n] ).
// Four columns per thread when ldp and the workspace allow it; the sums are
// the same element by element either way.
template <int BM, int BN, int NT>
__device__ __forceinline__ void splitk_finish_tile(const float* partial, size_t plane, int ldp, float* C,
                                                   const float* bias, int M, int N, int ldc, int splits, int relu,
                                                   float thr, int m0, int n0) {
  using splitk::f32x4;
  const int tid = threadIdx.x;
  if (BN % 4 == 0 && (ldp & 3) == 0 && ((uintptr_t)partial & 15) == 0 && (int64_t)BM * ldp < (1 << 29)) {
    const bool vec_out = ((N | ldc) & 3) == 0 && (((uintptr_t)C | (uintptr_t)bias) & 15) == 0;
    // U quads of columns per thread at once, several splits of each: the loads go
    // past the L2, so it is their round trips that count.  One quad of 4
    // splits at a time took 14 us of a 46 us 256x8192x4608 bf16 product.
    constexpr int QUADS = BM * BN / 4, PER = (QUADS + NT - 1) / NT;
    constexpr int U = PER < 4 ? PER : 4;
    const float* const tile = partial + (size_t)m0 * ldp + n0;
    for (int i0 = 0; i0 < PER; i0 += U) {
      f32x4 v[U];
      unsigned off[U];
      bool any = false;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        // quads outside the tile or the matrix read the tile's first
        const int idx = tid + (i0 + u) * NT;
        const int dm = idx / (BN / 4), dn = 4 * (idx % (BN / 4));
        const bool in = idx < QUADS && m0 + dm < M && n0 + dn < N;
        off[u] = in ? ((unsigned)dm * (unsigned)ldp + dn) * 4u : 0u;
        v[u] = f32x4{0.f, 0.f, 0.f, 0.f};
        any = any || in;
      }
      if (!__any(any)) continue;
      // only the splits that exist, in order, at most 16 loads in flight
      auto add = [&](int s0, auto count) {
        constexpr int C = decltype(count)::value;
        f32x4 t[C][U];
#pragma unroll
        for (int j = 0; j < C; ++j)
#pragma unroll
          for (int u = 0; u < U; ++u) t[j][u] = splitk_load4(tile + (size_t)(s0 + j) * plane, off[u]);
#pragma unroll
        for (int j = 0; j < C; ++j)
#pragma unroll
          for (int u = 0; u < U; ++u) v[u] += t[j][u];
      };
      int s0 = 0;
      if constexpr (U <= 2) {
        for (; s0 + 8 <= splits; s0 += 8) add(s0, std::integral_constant<int, 8>{});
      }
      for (; s0 + 4 <= splits; s0 += 4) add(s0, std::integral_constant<int, 4>{});
      if (s0 + 2 <= splits) {
        add(s0, std::integral_constant<int, 2>{});
        s0 += 2;
      }
      if (s0 < splits) add(s0, std::integral_constant<int, 1>{});
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int idx = tid + (i0 + u) * NT;
        const int m = m0 + idx / (BN / 4);
        const int n = n0 + 4 * (idx % (BN / 4));
        if (idx >= QUADS || m >= M || n >= N) continue;
        if (vec_out) {
          f32x4 x = v[u];
          if (bias) x += *(const f32x4*)(bias + n);
          if (relu) {
#pragma unroll
            for (int r = 0; r < 4; ++r) x[r] = x[r] < thr ? thr : x[r];
          }
          *(f32x4*)(C + (size_t)m * ldc + n) = x;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if (n + r >= N) break;
            float x = v[u][r];
            if (bias) x += bias[n + r];
            if (relu && x < thr) x = thr;
            C[(size_t)m * ldc + n + r] = x;
          }
        }
      }
    }
  } else {
    for (int idx = tid; idx < BM * BN; idx += NT) {
      const int m = m0 + idx / BN;
      const int n = n0 + idx % BN;
      if (m >= M || n >= N) continue;
      float v = splitk_sum1(partial + (size_t)m * ldp + n, plane, splits);
      if (bias) v += bias[n];
      if (relu && v < thr) v = thr;
      C[(size_t)m * ldc + n] = v;
    }
  }
}

}  // namespace xtc_hip
