// SPDX-License-Identifier: BSD-3-Clause
// MFMA GEMM / implicit-GEMM conv2d on bf16 matrix instructions for fp32 and
// bf16 operands, any size and alignment:
//   C[M,N] (fp32) = epilogue( sum_k A[M,K] * B[K,N] )
//
// fp32 operands on bf16 MFMAs.  An fp32 value is the exact sum of three bf16
// values, x = h + m + l (round to nearest, subtract, twice: 8 + 8 + 8
// significant bits), so
//   a b = ah bh + (ah bm + am bh) + (ah bl + al bh + am bm) + O(2^-25 |a b|)
// and six v_mfma_f32_16x16x32_bf16 (16 cycles each) do the work of eight
// v_mfma_f32_16x16x4_f32 (32 cycles each): 96 against 256 matrix cycles per
// 16x16x32 product.  The six products of 32 k are summed from zero, smallest
// first, in a register tile of their own, and that sum is added to the
// accumulator in fp32: one accumulator rounding per 32 products where the
// fp32 MFMA rounds at every product.
//
// What the split cannot hold is computed on fp32 MFMAs instead.  A lane keeps
// the largest and the smallest nonzero |operand| it staged; after the K walk a
// wave looks at its sums.  An infinity or NaN among the operands (or an
// operand above the bf16 range) leaves a non-finite sum; operands below 2^-110,
// denormal or not, lose bits of their m and l parts (bf16 ends at 2^-133), an
// error of at most K 2^-126 max|operand|, which matters only to sums below
// 2^-90 max|operand|, and to zeros only where such operands took part.  A wave
// that finds such a sum repeats its tile with v_mfma_f32_16x16x4_f32 straight
// from global memory (exact in the same cases as the fp32 MFMA).  A zero row
// alone costs nothing; with one operand of 2^-112 in it a workgroup whose
// waves hold zero sums repeats them: 2048x4096x1024 98 us, 286 with one such
// row tile in the matrix, 388 with one in every wave; 4096^3 668, 1789, 2699;
// 1024x1024x256 18, 58, 75.
//
// Structure (per workgroup = one BM x BN output tile, one split of K):
//   * WGM x WGN waves of (BM/WGM) x (BN/WGN), K in slabs of BK through two
//     LDS buffers.  Global loads go to RING register sets, RING slabs ahead;
//     a slab is split into its planes on the way from registers to LDS, so
//     every operand is split once per workgroup, not once per wave.
//   * LDS: A planes [BM][BK] bf16 in 16-byte chunks, chunk c of row r at
//     c ^ swz(r); B planes [BK][BN] in 32-byte chunks, chunk c of row k at
//     c ^ swz(k), read with the transposing ds_read_b64_tr_b16.  B stored
//     transposed (BT) is laid out and read like A.
//   * Loads come in units of 8 consecutive elements (k of A and B^T, n of
//     B).  VEC: strides, K and N are whole 16-byte vectors, a unit is one
//     (bf16) or two (fp32) aligned vectors.  Otherwise whole units are
//     unaligned vector loads (which global memory takes at element alignment)
//     and a unit cut by the edge of K or N is read element by element.  Rows
//     past M and columns past N repeat the last ones; they are not stored.
//   * Conv: A is the im2col view of an NHWC image.  The S*C elements under
//     one window row are contiguous in the image, so k = r * SC + kk reads
//     image row oh * sh + r - ph at element (ow * sw - pw) * C + kk: in
//     bounds when both lie inside the image, no division by C.
//   * B is the first MFMA operand, so a lane holds C[m][n .. n+3].
//   * Split-K: partial planes and arrival counters of splitk.hpp.  KG > 1: the
//     workgroup holds KG groups of WGM x WGN waves, each with its own LDS
//     buffers and its own run of the split's slabs; their sums meet in LDS.
//
// What bounds it.  At 4096^3 the board's power: 6 x 1.37e11 FLOP in 631 us is
// 1.31 PFLOP/s of bf16 MFMAs, where a library bf16 product reaches 1.41
// (fp32 MFMAs: 980 us).  At 2048x4096x1024, one tile per CU, 88-99 us against
// 130-144: 12 us are launch, first loads and stores, a 32-deep step of
// 128x256 takes 2.4 us where its MFMAs alone (operands from registers, same
// power) take 1.6.  Measured there on the way: splitting after the MFMAs
// instead of between them 100-107 us; two groups of waves half a step apart
// 107-119 us; two register sets (spills) 96 us; fragments of the next slab
// read after the barrier instead of behind the last column 91-96 us.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gemm.hpp"
#include "splitk.hpp"

namespace xtc_hip {

namespace planes {

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;

// 16-byte chunk swizzle of an A (or B^T) row of BK bf16
template <int BK>
__device__ __forceinline__ int swz_row(int r) {
  return BK == 64 ? (r & 7) : ((r >> 1) & 3);
}
// 32-byte chunk swizzle of B row k (BN / 16 chunks)
template <int BN>
__device__ __forceinline__ int swz_k(int k) {
  return BN >= 128 ? ((k & 3) | ((k >> 1) & 4)) : BN == 64 ? (k & 3) : (k & 1);
}

// 8 elements as loaded
template <typename T> struct Unit;
template <> struct Unit<float> { float v[8]; };
template <> struct Unit<__bf16> { u32x4 v; };

// VEC: whole 16-byte vectors, `q` per unit (2 for fp32, 1 for bf16)
__device__ __forceinline__ void load_vec(Unit<float>& u, int q, const float* p) {
  const f32x4 t = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
  for (int e = 0; e < 4; ++e) u.v[4 * q + e] = t[e];
}
__device__ __forceinline__ void load_vec(Unit<__bf16>& u, int, const __bf16* p) {
  u.v = *reinterpret_cast<const u32x4*>(p);
}

// the element `off` bytes past the uniform address p (one scalar base and a
// 32-bit lane offset)
template <typename T>
__device__ __forceinline__ const T* at(const T* p, unsigned off) {
  return reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + off);
}

// any alignment: the unit of 8 elements at p, of which the first `n` exist
__device__ __forceinline__ void load_any(Unit<float>& u, const float* p, int n) {
  if (n >= 8) {
    __builtin_memcpy(&u, p, 32);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) u.v[e] = e < n ? p[e] : 0.f;
  }
}
__device__ __forceinline__ void load_any(Unit<__bf16>& u, const __bf16* p, int n) {
  if (n >= 8) {
    __builtin_memcpy(&u, p, 16);
  } else {
    const unsigned short* q = reinterpret_cast<const unsigned short*>(p);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const unsigned lo = 2 * e < n ? q[2 * e] : 0u, hi = 2 * e + 1 < n ? q[2 * e + 1] : 0u;
      u.v[e] = lo | (hi << 16);
    }
  }
}

// element e of a unit (constant e)
__device__ __forceinline__ void put(Unit<float>& u, int e, float v) { u.v[e] = v; }
__device__ __forceinline__ void put(Unit<__bf16>& u, int e, unsigned short v) {
  u.v[e / 2] = (e & 1) ? (u.v[e / 2] & 0xffffu) | ((unsigned)v << 16) : (u.v[e / 2] & 0xffff0000u) | v;
}
// elements from `n` on become zero
__device__ __forceinline__ void cut(Unit<float>& u, int n) {
#pragma unroll
  for (int e = 0; e < 8; ++e) u.v[e] = e < n ? u.v[e] : 0.f;
}
__device__ __forceinline__ void cut(Unit<__bf16>& u, int n) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const unsigned keep = (2 * e < n ? 0xffffu : 0u) | (2 * e + 1 < n ? 0xffff0000u : 0u);
    u.v[e] &= keep;
  }
}
// elements whose bit of `in` is clear become the pad value (STEP elements per bit)
template <int STEP>
__device__ __forceinline__ void pad_out(Unit<float>& u, unsigned in, float pad) {
#pragma unroll
  for (int e = 0; e < 8; ++e) u.v[e] = (in >> (e / STEP)) & 1u ? u.v[e] : pad;
}
template <int STEP>
__device__ __forceinline__ void pad_out(Unit<__bf16>& u, unsigned in, float pad) {
  const unsigned w = splat16(pad, __bf16())[0];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const unsigned keep =
        ((in >> (2 * e / STEP)) & 1u ? 0xffffu : 0u) | ((in >> ((2 * e + 1) / STEP)) & 1u ? 0xffff0000u : 0u);
    u.v[e] = (u.v[e] & keep) | (w & ~keep);
  }
}

typedef __attribute__((address_space(3))) unsigned char lds_byte;
__device__ __forceinline__ void lds_write16(unsigned char* dst, u32x4 v) {
  *reinterpret_cast<lds_u32x4*>((lds_byte*)dst) = v;
}

// twice the bits of |x|, less one: orders nonzero magnitudes, zeros above all
__device__ __forceinline__ unsigned nonzero_key(float x) { return (__float_as_uint(x) << 1) - 1u; }

// dword e of the three planes of a unit: elements 2 e and 2 e + 1 split;
// top: largest magnitude seen, low: key of the smallest nonzero one
__device__ __forceinline__ void split2(const Unit<float>& u, int e, u32x4 (&w)[3], float& top, unsigned& low) {
  f32x2 x = {u.v[2 * e], u.v[2 * e + 1]};
  top = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), top);
  low = min(min(nonzero_key(x[0]), nonzero_key(x[1])), low);
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const unsigned h = __builtin_bit_cast(unsigned, __builtin_convertvector(x, bf16x2));
    w[q][e] = h;
    if (q < 2) x = f32x2{x[0] - __uint_as_float(h << 16), x[1] - __uint_as_float(h & 0xffff0000u)};
  }
}

}  // namespace planes

template <typename T, int BM, int BN, int BK, int WGM, int WGN, bool CONV, bool BT, bool VEC, int RING, int KG = 1>
struct PlanesTile {
  static constexpr int NT = WGM * WGN * 64;  // threads of a k-group
  static constexpr bool F32 = sizeof(T) == 4;
  static constexpr int P = F32 ? 3 : 1;              // planes
  static constexpr int VE = F32 ? 4 : 8, VPU = 8 / VE;  // elements per vector, vectors per unit
  static constexpr int STEP = VEC ? VE : 1;             // conv: elements that share one bounds check
  static constexpr int TM = BM / WGM / 16, TN = BN / WGN / 16;
  static constexpr int A_PLANE = BM * BK * 2, B_PLANE = BK * BN * 2;
  static constexpr int STAGE = P * (A_PLANE + B_PLANE);
  static constexpr int A_UNITS = BM * BK / 8, B_UNITS = BK * BN / 8;
  static constexpr int A_PER = (A_UNITS + NT - 1) / NT, B_PER = (B_UNITS + NT - 1) / NT;
  static constexpr bool A_EVEN = A_UNITS % NT == 0, B_EVEN = B_UNITS % NT == 0, EVEN = A_EVEN && B_EVEN;
  static constexpr bool PIPE = F32 && EVEN && VEC && !CONV && TN > 1 && RING == 1;
  static_assert(BM % (16 * WGM) == 0 && BN % (16 * WGN) == 0, "wave tile");
  static_assert(BK == 32 || BK == 64, "slab");
  static_assert(A_EVEN || A_UNITS < NT, "A units");
  static_assert(B_EVEN || B_UNITS < NT, "B units");
  static_assert(NT % (BK / 8) == 0 && (BT || NT % (BN / 8) == 0), "a thread keeps its column");
  static_assert(KG * 2 * STAGE <= 160 * 1024, "LDS");
  static_assert(KG == 1 || !F32, "the fp32 kernel redoes a whole split's sums");
  static_assert((KG - 1) * BM * BN * 4 <= KG * 2 * STAGE, "the groups' sums fit in the slabs' LDS");
};

template <typename T, int BM, int BN, int BK, int WGM, int WGN, bool CONV, bool BT, bool VEC, int RING, int KG = 1>
__global__ void __attribute__((amdgpu_flat_work_group_size(KG * WGM * WGN * 64, KG * WGM * WGN * 64)))
__attribute__((amdgpu_waves_per_eu(2)))
gemm_planes(GemmArgs args) {
  using namespace planes;
  using X = PlanesTile<T, BM, BN, BK, WGM, WGN, CONV, BT, VEC, RING, KG>;
  constexpr int NT = X::NT, TM = X::TM, TN = X::TN;
  constexpr bool F32 = X::F32;

  __shared__ __attribute__((aligned(1024))) unsigned char shared[KG * 2 * X::STAGE];

  const int wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = KG > 1 ? wave_id / (WGM * WGN) : 0;  // k-group
  unsigned char* const smem = shared + kg * 2 * X::STAGE;
  const unsigned tid = threadIdx.x - kg * NT;  // in the k-group
  const int lane = tid & 63;
  const int wave = wave_id - kg * (WGM * WGN);
  const int wm = wave / WGN, wn = wave % WGN;
  const int l16 = lane & 15, g = lane >> 4;

  int tile_m, tile_n;
  tile_coords(args, tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int split = blockIdx.z;
  // the split's slabs, a run of `steps` of them for each k-group
  const int split_begin = split * args.k_per_split, split_end = min(args.K, split_begin + args.k_per_split);
  const int steps = ((split_end - split_begin + BK - 1) / BK + KG - 1) / KG;
  const int k_begin = min(split_begin + kg * steps * BK, split_end);
  const int k_end = KG > 1 ? min(split_end, k_begin + steps * BK) : split_end;
  const int nk = (k_end - k_begin + BK - 1) / BK;

  const T* const A = reinterpret_cast<const T*>(args.A);
  const T* const B = reinterpret_cast<const T*>(args.B);

  // ---- global sources of this thread's units: byte offsets from the tile's
  // (uniform) corner
  constexpr int AR = NT / (BK / 8), BR = BT ? AR : NT / (BN / 8);  // rows from a unit to the thread's next
  const T* const a_tile = A + (size_t)m0 * args.lda + k_begin;
  const T* const b_tile = BT ? B + (size_t)n0 * args.ldb + k_begin : B + (size_t)k_begin * args.ldb + n0;
  const int a_row = tid / (BK / 8), a_kc = (tid % (BK / 8)) * 8;
  const int b_row = BT ? a_row : tid / (BN / 8);  // of B^T, or k row in the slab
  const int b_col = BT ? a_kc : (tid % (BN / 8)) * 8;
  unsigned a_off[X::A_PER], b_off[X::B_PER];
  const T* a_src[X::A_PER];             // conv: the window's first element
  int a_ih0[X::A_PER], a_e0[X::A_PER];  // conv: its image row and its element in the row
  const int WC = CONV ? args.cW * args.cC : 0;
  const int SC = CONV ? args.cS * args.cC : 0;
#pragma unroll
  for (int i = 0; i < X::A_PER; ++i) {
    const int m = min(m0 + a_row + i * AR, args.M - 1);
    if constexpr (CONV) {
      const int ow = m % args.cOW, t = m / args.cOW;
      const int oh = t % args.cOH, b = t / args.cOH;
      a_ih0[i] = oh * args.cSH - args.cPH;
      a_e0[i] = (ow * args.cSW - args.cPW) * args.cC;
      a_src[i] = A + ((int64_t)b * args.cH + a_ih0[i]) * WC + a_e0[i];
    } else {
      a_off[i] = ((unsigned)(m - m0) * (unsigned)args.lda + a_kc) * (unsigned)sizeof(T);
    }
  }
#pragma unroll
  for (int i = 0; i < X::B_PER; ++i) {
    const int r = BT ? min(n0 + b_row + i * BR, args.N - 1) - n0 : b_row + i * BR;
    b_off[i] = ((unsigned)r * (unsigned)args.ldb + b_col) * (unsigned)sizeof(T);
  }

  // K stagger: tile (tm, tn) starts its K walk at slab (tm + 2 tn) mod 16, so
  // that tiles sharing a panel do not ask for the same lines at once (a K of
  // whole slabs only, so that a partial slab stays the last)
  const int kofs = (KG == 1 || nk > 0) && (k_end - k_begin) % BK == 0 ? ((tile_m + 2 * tile_n) & 15) % nk : 0;
  auto slab_k = [&](int t) {  // k of step t's slab, relative to k_begin
    const int r = t + kofs;
    return (r >= nk ? r - nk : r) * BK;
  };

  Unit<T> areg[RING][X::A_PER], breg[RING][X::B_PER];
  unsigned a_in[RING][X::A_PER];  // conv: which vectors (or elements) of the unit lie inside the image
  float top = 0.f;                // fp32: largest |operand| staged by this lane
  unsigned low = ~0u;             // fp32: key of the smallest nonzero one

  // Unit u of register set `slot` from a whole slab of VEC operands at k = kt.
  const bool inside = BT || n0 + BN <= args.N;
  auto load_whole = [&](int kt, int u, int slot) {
    if (u < X::A_PER) {
#pragma unroll
      for (int q = 0; q < X::VPU; ++q) load_vec(areg[slot][u], q, at(a_tile + kt, a_off[u]) + q * X::VE);
    } else {
      const T* p = at(BT ? b_tile + kt : b_tile + (size_t)kt * args.ldb, b_off[u - X::A_PER]);
#pragma unroll
      for (int q = 0; q < X::VPU; ++q) load_vec(breg[slot][u - X::A_PER], q, p + q * X::VE);
    }
  };
  // Loads of step t's slab.  VEC loads are unconditional, at addresses kept inside
  // the operands (the compiler's wait counts stay exact); what lies past the
  // end of K or outside the image is replaced in store_slab.
  auto load_slab = [&](int t, int slot) {
    const int kt = slab_k(t);
    const int left = k_end - k_begin - kt; // k left in the split
    if constexpr (CONV) {
      const int k = k_begin + kt + a_kc;
      const int r0 = k / SC, kk0 = k - r0 * SC;
#pragma unroll
      for (int i = 0; i < X::A_PER; ++i) {
        if (!X::A_EVEN && tid + i * NT >= X::A_UNITS) continue;
        int r = r0, kk = kk0;
        unsigned in = 0;
#pragma unroll
        for (int q = 0; q < 8; q += X::STEP) {
          const int ih = a_ih0[i] + r, e = a_e0[i] + kk;
          const bool ok = q < left - a_kc && (unsigned)ih < (unsigned)args.cH && (unsigned)e < (unsigned)WC;
          const T* p = ok ? a_src[i] + (int64_t)r * WC + kk : A;
          in |= ok ? 1u << (q / X::STEP) : 0u;
          if constexpr (VEC) load_vec(areg[slot][i], q / X::STEP, p);
          else if constexpr (F32) put(areg[slot][i], q, *p);
          else put(areg[slot][i], q, *reinterpret_cast<const unsigned short*>(p));
          kk += X::STEP;
          if (kk >= SC) {
            kk -= SC;
            ++r;
          }
        }
        a_in[slot][i] = in;
      }
    } else {
#pragma unroll
      for (int i = 0; i < X::A_PER; ++i) {
        if (!X::A_EVEN && tid + i * NT >= X::A_UNITS) continue;
        if (VEC && left >= BK) {
          load_whole(kt, i, slot);
        } else if constexpr (VEC) {
#pragma unroll
          for (int q = 0; q < X::VPU; ++q)
            load_vec(areg[slot][i], q, at(a_tile, a_off[i]) + min(kt + q * X::VE, args.K - X::VE - k_begin - a_kc));
        } else {
          load_any(areg[slot][i], at(a_tile + kt, a_off[i]), left - a_kc);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < X::B_PER; ++i) {
      if (!X::B_EVEN && tid + i * NT >= X::B_UNITS) continue;
      if (VEC && left >= BK && inside) {
        load_whole(kt, X::A_PER + i, slot);
      } else if constexpr (!VEC) {
        const T* p = at(BT ? b_tile + kt : b_tile + (size_t)kt * args.ldb, b_off[i]);
        load_any(breg[slot][i], p, BT ? left - b_col : b_row + i * BR < left ? args.N - (n0 + b_col) : 0);
      } else if constexpr (BT) {
#pragma unroll
        for (int q = 0; q < X::VPU; ++q)
          load_vec(breg[slot][i], q, at(b_tile, b_off[i]) + min(kt + q * X::VE, args.K - X::VE - k_begin - b_col));
      } else {
        const T* row = b_tile + (size_t)min(kt + b_row + i * BR, args.K - 1 - k_begin) * args.ldb;
#pragma unroll
        for (int q = 0; q < X::VPU; ++q)
          load_vec(breg[slot][i], q, row + min(b_col + q * X::VE, args.N - X::VE - n0));
      }
    }
  };

  // Replaces what step t's slab, in register set `slot`, has past the end of K
  // or outside the image.
  auto mask_slab = [&](int t, int slot) {
    const int left = k_end - k_begin - slab_k(t);
    if constexpr (CONV) {
      constexpr unsigned ALL = (1u << (8 / X::STEP)) - 1u;
      unsigned all = ALL;
#pragma unroll
      for (int i = 0; i < X::A_PER; ++i)
        if (X::A_EVEN || tid + i * NT < X::A_UNITS) all &= a_in[slot][i];
      if (__any(all != ALL)) {
#pragma unroll
        for (int i = 0; i < X::A_PER; ++i) pad_out<X::STEP>(areg[slot][i], a_in[slot][i], args.pad_value);
      }
    }
    if (left < BK && (VEC || CONV)) {
#pragma unroll
      for (int i = 0; i < X::A_PER; ++i) cut(areg[slot][i], left - a_kc);
    }
    if (left < BK && VEC) {
#pragma unroll
      for (int i = 0; i < X::B_PER; ++i) cut(breg[slot][i], BT ? left - b_col : b_row + i * BR < left ? 8 : 0);
    }
  };
  // Unit u counts the A units, then the B units.  Its place in an LDS buffer:
  // the swizzles do not change over a thread's units
  static_assert(X::A_PER == 1 || AR % 8 == 0, "A swizzle");
  static_assert(X::B_PER == 1 || BR % (BT ? 8 : 16) == 0, "B swizzle");
  const int a_dst = a_row * (2 * BK) + 16 * ((a_kc >> 3) ^ swz_row<BK>(a_row));
  const int b_dst = X::P * X::A_PLANE +
                    (BT ? b_row * (2 * BK) + 16 * ((b_col >> 3) ^ swz_row<BK>(b_row))
                        : b_row * (2 * BN) + 32 * ((b_col >> 4) ^ swz_k<BN>(b_row)) + 2 * (b_col & 8));
  auto unit_dst = [&](unsigned char* st, int u) {
    return u < X::A_PER ? st + a_dst + u * AR * (2 * BK)
                        : st + b_dst + (u - X::A_PER) * BR * (BT ? 2 * BK : 2 * BN);
  };
  auto split_pair = [&](int u, int slot, int e, u32x4 (&w)[3]) {
    if constexpr (F32) split2(u < X::A_PER ? areg[slot][u] : breg[slot][u - X::A_PER], e, w, top, low);
  };
  auto write_unit = [&](unsigned char* st, int u, const u32x4 (&w)[3]) {
    unsigned char* dst = unit_dst(st, u);
#pragma unroll
    for (int p = 0; p < X::P; ++p) lds_write16(dst + p * (u < X::A_PER ? X::A_PLANE : X::B_PLANE), w[p]);
  };
  auto store_slab = [&](unsigned char* st, int slot) {
#pragma unroll
    for (int u = 0; u < X::A_PER + X::B_PER; ++u) {
      if (!X::A_EVEN && u < X::A_PER && tid + u * NT >= X::A_UNITS) continue;
      if (!X::B_EVEN && u >= X::A_PER && tid + (u - X::A_PER) * NT >= X::B_UNITS) continue;
      u32x4 w[3];
      if constexpr (F32) {
#pragma unroll
        for (int e = 0; e < 4; ++e) split_pair(u, slot, e, w);
      } else {
        w[0] = u < X::A_PER ? areg[slot][u].v : breg[slot][u - X::A_PER].v;
      }
      write_unit(st, u, w);
    }
  };

  // Barrier of a step: this wave's LDS accesses are complete, global loads
  // stay in flight.
  auto step_barrier = [] {
    constexpr int kWaitLgkm0 = 15 | (7 << 4) | (0 << 8) | (3 << 14);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  };

  // ---- fragments
  const int a_row0 = wm * (16 * TM) + l16;
  const int a_h = swz_row<BK>(a_row0);  // unchanged by + 16
  const int b_row0 = BT ? wn * (16 * TN) + l16 : 8 * g + (l16 >> 2);
  const int b_h = BT ? swz_row<BK>(b_row0) : swz_k<BN>(b_row0);  // unchanged by + 16 / by + 4 and + 32
  auto read_a = [&](const unsigned char* sa, int ks, int it) {
    const int off = (a_row0 + it * 16) * (2 * BK) + 16 * ((ks * 4 + g) ^ a_h);
    return __builtin_bit_cast(bf16x8, *(const lds_u32x4*)(sa + off));
  };
  auto read_b = [&](const unsigned char* sb, int ks, int jt) {
    if constexpr (BT) {
      const int off = (b_row0 + jt * 16) * (2 * BK) + 16 * ((ks * 4 + g) ^ b_h);
      return __builtin_bit_cast(bf16x8, *(const lds_u32x4*)(sb + off));
    } else {
      const int off = (ks * 32 + b_row0) * (2 * BN) + 32 * ((wn * TN + jt) ^ b_h) + 8 * (l16 & 3);
      const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(sb + off));
      const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(sb + off + 4 * (2 * BN)));
      return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  };

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Slab t: global -> register set t % RING -> LDS buffer t & 1 -> MFMA.
  // Step t computes slab t, splits slab t + 1 into the other buffer and
  // refills its set with slab t + 1 + RING; one barrier per step.  Unrolled
  // by RING so that the set index is a constant.
  auto refill = [&](int t, unsigned char* nxt, int s1) {
    if (t + 1 < nk) {
      mask_slab(t + 1, s1);
      store_slab(nxt, s1);
      if (t + 1 + RING < nk) load_slab(t + 1 + RING, s1);
    }
  };
#pragma unroll
  for (int r = 0; r < RING; ++r)
    if (r < nk) load_slab(r, r);
  if (KG == 1 || nk > 0) {
    mask_slab(0, 0);
    store_slab(smem, 0);
    if (RING < nk) load_slab(RING, 0);
  }
  __syncthreads();

  if constexpr (F32) {
    // A column is one 16-wide B fragment against the wave's TM A fragments:
    // six groups of TM MFMAs, one per pair of planes.  Planes of A are last
    // used in the order l, m, h, so the barrier of the step sits before its
    // last column: behind the MFMAs of that column the next slab's fragments
    // come in, plane by plane as the registers fall free.  The column's sums
    // are added to the accumulators between the first MFMAs of the next one.
    static_assert(BK == 32, "one k-step per slab");
    constexpr int pb[6] = {0, 1, 0, 2, 1, 0}, pa[6] = {2, 1, 1, 0, 0, 0};
    bf16x8 a[TM][3], b[2][3];
    f32x4 sum[TM];
    auto get_a = [&](const unsigned char* st, int p) {
#pragma unroll
      for (int it = 0; it < TM; ++it) a[it][p] = read_a(st + p * X::A_PLANE, 0, it);
    };
    auto get_b = [&](const unsigned char* st, int jt, int p) {
      b[jt & 1][p] = read_b(st + 3 * X::A_PLANE + p * X::B_PLANE, 0, jt);
    };
    auto group = [&](int jt, int q) {
#pragma unroll
      for (int it = 0; it < TM; ++it) {
        if (q == 0) {
          if (jt > 0) acc[it][jt - 1] += sum[it];
          sum[it] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        sum[it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[jt & 1][pb[q]], a[it][pa[q]], sum[it], 0, 0, 0);
      }
    };
    // The columns before the barrier.  PIPE: register set `slot` (a whole
    // slab) goes to `nxt` and is refilled from k = kt between the MFMAs, a
    // pair of elements after each group: a SIMD issues a wave's vector ALU
    // and LDS instructions while its matrix core works on the wave's MFMAs.
    auto front = [&](const unsigned char* st, auto pipe, unsigned char* nxt, int slot, int kt) {
      constexpr int UNITS = X::A_PER + X::B_PER;
      constexpr int PAIRS = 4 * UNITS, SLOTS = 6 * (TN > 1 ? TN - 1 : 1);
      u32x4 w[3];
#pragma unroll
      for (int jt = 0; jt < TN - 1; ++jt) {
#pragma unroll
        for (int q = 0; q < 6; ++q) {
          if (q < 3) get_b(st, jt + 1, q);
          group(jt, q);
          if constexpr (decltype(pipe)::value) {
#pragma unroll
            for (int x = 0; x < PAIRS; ++x)
              if (x * SLOTS / PAIRS == jt * 6 + q) {
                split_pair(x / 4, slot, x % 4, w);
                if (x % 4 == 3) {
                  write_unit(nxt, x / 4, w);
                  load_whole(kt, x / 4, slot);
                }
              }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    auto back = [&](const unsigned char* nxt) {
      constexpr int jt = TN - 1;
      constexpr bool OWN = TN > 1;  // the last column has its own B fragment registers
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        group(jt, q);
        if (q == 0) get_a(nxt, 2);
        if (q == 1 && OWN && TN % 2 == 0) {
          get_b(nxt, 0, 0);
          get_b(nxt, 0, 1);
        }
        if (q == 2) get_a(nxt, 1);
        if (q == 3 && OWN && TN % 2 == 0) get_b(nxt, 0, 2);
        __builtin_amdgcn_sched_barrier(0);
      }
      get_a(nxt, 0);
      if constexpr (!(OWN && TN % 2 == 0)) {
#pragma unroll
        for (int p = 0; p < 3; ++p) get_b(nxt, 0, p);
      }
#pragma unroll
      for (int it = 0; it < TM; ++it) acc[it][jt] += sum[it];
    };
    get_a(smem, 2);
    get_b(smem, 0, 0);
    get_b(smem, 0, 1);
    get_a(smem, 1);
    get_b(smem, 0, 2);
    get_a(smem, 0);
    int t = 0;
    if constexpr (X::PIPE) {
      // steps whose next two slabs are whole
      for (const int end = inside ? (k_end - k_begin) / BK - 2 : 0; t < end; ++t) {
        unsigned char* nxt = smem + ((t & 1) ^ 1) * X::STAGE;
        front(smem + (t & 1) * X::STAGE, std::bool_constant<X::PIPE>{}, nxt, 0, slab_k(t + 2));
        step_barrier();
        back(nxt);
      }
    }
    for (; t < nk; t += RING) {
#pragma unroll
      for (int u = 0; u < RING; ++u) {
        if (t + u < nk) {
          unsigned char* nxt = smem + (((t + u) & 1) ^ 1) * X::STAGE;
          front(smem + ((t + u) & 1) * X::STAGE, std::false_type{}, nxt, 0, 0);
          refill(t + u, nxt, (u + 1) % RING);
          step_barrier();
          back(nxt);
        }
      }
    }
  } else {
    for (int t0 = 0; t0 < nk; t0 += RING) {
#pragma unroll
      for (int u = 0; u < RING; ++u) {
        const int t = t0 + u;
        if (t < nk) {
          const unsigned char* st = smem + (t & 1) * X::STAGE;
#pragma unroll
          for (int ks = 0; ks < BK / 32; ++ks) {
            bf16x8 a[TM], b[TN];
#pragma unroll
            for (int it = 0; it < TM; ++it) a[it] = read_a(st, ks, it);
#pragma unroll
            for (int jt = 0; jt < TN; ++jt) b[jt] = read_b(st + X::A_PLANE, ks, jt);
#pragma unroll
            for (int jt = 0; jt < TN; ++jt)
#pragma unroll
              for (int it = 0; it < TM; ++it)
                acc[it][jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[jt], a[it], acc[it][jt], 0, 0, 0);
          }
          refill(t, smem + ((t & 1) ^ 1) * X::STAGE, (u + 1) % RING);
          __syncthreads();
        }
      }
    }
  }

  // a k-group with fewer slabs passes every step's barrier with the others
  for (int t = nk; KG > 1 && t < steps; ++t) __syncthreads();

  const int mrow = m0 + wm * (16 * TM) + l16;
  const int ncol = n0 + wn * (16 * TN) + 4 * g;

  // ---- sums the split cannot vouch for: the wave's tile again on fp32 MFMAs
  if constexpr (F32) {
#pragma unroll
    for (int s = 1; s < 64; s *= 2) top = fmaxf(top, __shfl_xor(top, s));
    __shared__ float tops[WGM * WGN];
    __shared__ unsigned smalls[WGM * WGN];
    const bool any = __any(low < nonzero_key(0x1p-110f));
    if (lane == 0) {
      tops[wave] = top;
      smalls[wave] = any;
    }
    __syncthreads();
    unsigned small = 0;
#pragma unroll
    for (int w = 0; w < WGM * WGN; ++w) {
      top = fmaxf(top, tops[w]);
      small |= smalls[w];
    }
    const float floor = top * 0x1p-90f;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = fabsf(acc[i][j][r]);
          bad = bad || !(v < INFINITY) || (v == 0.f ? small != 0 : v < floor);
        }
    if (__ballot(bad)) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int k0 = k_begin; k0 < k_end; k0 += 4) {
        const int k = k0 + g;
        const bool ok = k < k_end;
        float a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int m = min(mrow + 16 * i, args.M - 1);
          a[i] = 0.f;
          if constexpr (CONV) {
            const int ow = m % args.cOW, t = m / args.cOW;
            const int ih = t % args.cOH * args.cSH - args.cPH + k / SC;
            const int e = (ow * args.cSW - args.cPW) * args.cC + k % SC;
            if (ok) {
              const bool in = (unsigned)ih < (unsigned)args.cH && (unsigned)e < (unsigned)WC;
              a[i] = args.pad_value;
              if (in) a[i] = A[((int64_t)(t / args.cOH) * args.cH + ih) * WC + e];
            }
          } else {
            if (ok) a[i] = A[(size_t)m * args.lda + k];
          }
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int n = min(ncol - 4 * g + 16 * j + l16, args.N - 1);
          b[j] = 0.f;
          if (ok) b[j] = BT ? B[(size_t)n * args.ldb + k] : B[(size_t)k * args.ldb + n];
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j], a[i], acc[i][j], 0, 0, 0);
      }
    }
  }

  // ---- the k-groups' sums meet in LDS, added in k order by the first group
  if constexpr (KG > 1) {
    f32x4* const sums = reinterpret_cast<f32x4*>(shared);
    if (kg > 0) {  // the last step's barrier is behind every slab's last read
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) sums[(((kg - 1) * TM + i) * TN + j) * NT + tid] = acc[i][j];
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int q = 0; q < KG - 1; ++q)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] += sums[((q * TM + i) * TN + j) * NT + tid];
    }
  }

  // ---- epilogue: lane holds C[m][n .. n+3]
  const bool to_partial = args.partial != nullptr;
  float* const out = to_partial ? args.partial + (size_t)split * args.M * args.ldp : args.C;
  const int ldo = to_partial ? args.ldp : args.ldc;
  // the workspace has room for whole vectors
  const bool vec_out = to_partial || (((args.N | ldo) & 3) == 0 && ((uintptr_t)out & 15) == 0);
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = ncol + 16 * j;
    if (n >= args.N || kg > 0) continue;
    f32x4 bv = {0.f, 0.f, 0.f, 0.f};
    if (!to_partial && args.bias) {
#pragma unroll
      for (int r = 0; r < 4; ++r) bv[r] = n + r < args.N ? args.bias[n + r] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = mrow + 16 * i;
      if (m >= args.M) continue;
      float* p = out + (size_t)m * ldo + n;
      f32x4 v = acc[i][j];
      if (!to_partial) {
        v += bv;
        if (args.relu) {
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = v[r] < args.relu_threshold ? args.relu_threshold : v[r];
        }
      }
      if (vec_out) {
        if (to_partial) splitk_store4(p, v);
        else *reinterpret_cast<f32x4*>(p) = v;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < args.N) p[r] = v[r];
      }
    }
  }
  if (to_partial && splitk_arrive(args.counters + tile_m * args.tiles_n + tile_n, (int)gridDim.z)) {
    splitk_finish_tile<BM, BN, KG * NT>(args.partial, (size_t)args.M * args.ldp, args.ldp, args.C, args.bias, args.M, args.N, args.ldc, (int)gridDim.z, args.relu,
                                   args.relu_threshold, m0, n0);
    splitk_release(args.counters + tile_m * args.tiles_n + tile_n);
  }
}

}  // namespace xtc_hip
