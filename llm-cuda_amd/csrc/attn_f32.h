// Building blocks of the fp32 attention kernels (forward and backward) on
// v_mfma_f32_32x32x2_f32.
//
// One MFMA contracts two indices: an A (B) operand is one float per lane, row
// (column) l % 32 at k index l / 32; accumulator register r of lane l holds
// column l % 32, row 8 (r / 4) + 4 (l / 32) + r % 4. Two operand forms:
//   * row operands (a contraction over head_dim): lane (l32, hh) holds row
//     l32's dims 8c + 4hh .. + 3 of every 8-dim chunk c, one 16-byte load per
//     chunk; MFMA 4c + e contracts dims 8c + e and 8c + 4 + e, in both
//     operands alike;
//   * column operands (a contraction over 32 tile rows whose B side is the
//     accumulator of the product before: P or dS): MFMA r contracts tile rows
//     n = 8 (r / 4) + r % 4 and n + 4, which are register r of the two lane
//     halves, so the accumulator is the B operand as it stands. Accumulator row
//     i of d tile dt stands for dim DTL i + dt, so a lane reads its DTL dims of
//     row n as one contiguous load (a wave: two whole rows).
// Streamed operands come straight from global memory (L2) into registers: an
// MFMA of this type takes 64 cycles of its SIMD, so a tile's loads (16 row and 16
// column instructions per 32 x 64 operand) are a small share of its time. What a
// workgroup keeps is held in registers in the forward and dQ kernels and, where
// those would cost the second wave (dK/dV: 182 against 95 us at [2, 16/8, 1024,
// 64]), in LDS (f32_stage).
#pragma once

#include "attn_tiles.h"
#include "lc_common.h"

namespace lc_attn {

constexpr int kF32Waves = 4;  // waves per workgroup, sharing one 32-row block
constexpr int kF32Rows = 32;  // rows per block and per tile

// Byte offset past every descriptor's range (loads there return 0): the host
// keeps num_records below it.
constexpr int kF32Oob = 0x7fff0000;

__device__ __forceinline__ f32x16_t f32_mma(float a, float b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t f32_rsrc(const float* base, int nbytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, nbytes, 0x00020000);
}

// Bytes of `rows` rows of D floats, `stride` elements apart.
__device__ __forceinline__ int f32_bytes(int rows, int64_t stride, int D) {
  return rows > 0 ? static_cast<int>(((int64_t)(rows - 1) * stride + D) * 4) : 0;
}

__device__ __forceinline__ void f32_zero(f32x16_t& x) {
#pragma unroll
  for (int r = 0; r < 16; ++r) x[r] = 0.f;
}

// Row operand of the lane's row (rows past the descriptor's range: zeros).
template <int DPAD>
struct F32Row {
  f32x4_t c[DPAD / 8];
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, int row, int stride_b, int hh,
                                       int D) {
    const int base = row * stride_b + hh * 16;
#pragma unroll
    for (int i = 0; i < DPAD / 8; ++i) {
      const int off = i * 8 + hh * 4 < D ? base + i * 32 : kF32Oob;
      c[i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
    }
  }
};

// acc += A B over head_dim (both row operands).
template <int DPAD>
__device__ __forceinline__ void f32_dot(f32x16_t& acc, const F32Row<DPAD>& A,
                                        const F32Row<DPAD>& B) {
#pragma unroll
  for (int i = 0; i < DPAD / 8; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = f32_mma(A.c[i][e], B.c[i][e], acc);
}

// 32 rows from row0 on into LDS, DPAD + 4 floats apart (the whole workgroup;
// rows past the range and dims past D: zeros).
template <int DPAD>
__device__ __forceinline__ void f32_stage(float* dst, const float* base, int nbytes, int row0,
                                          int stride_b, int tid, int D) {
  const __amdgpu_buffer_rsrc_t rs = f32_rsrc(base, nbytes);
#pragma unroll
  for (int e = tid; e < 32 * (DPAD / 4); e += 64 * kF32Waves) {
    const int row = e / (DPAD / 4), d = (e - row * (DPAD / 4)) * 4;
    const int off = d < D ? (row0 + row) * stride_b + d * 4 : kF32Oob;
    *reinterpret_cast<u32x4_t*>(dst + row * (DPAD + 4) + d) =
        __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0);
  }
}

// f32_dot with B rows staged by f32_stage (b: the lane's row + 4 hh).
template <int DPAD>
__device__ __forceinline__ void f32_dot_lds(f32x16_t& acc, const F32Row<DPAD>& A,
                                            const float* b) {
#pragma unroll
  for (int i = 0; i < DPAD / 8; ++i) {
    const f32x4_t B = *reinterpret_cast<const f32x4_t*>(b + i * 8);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = f32_mma(A.c[i][e], B[e], acc);
  }
}

template <int DTL>
struct F32Dims {
  float v[DTL];
};
template <int DTL>
__device__ __forceinline__ F32Dims<DTL> f32_load_dims(__amdgpu_buffer_rsrc_t rs, int off) {
  if constexpr (DTL == 1)
    return __builtin_bit_cast(F32Dims<DTL>, __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
  else if constexpr (DTL == 2)
    return __builtin_bit_cast(F32Dims<DTL>, __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0));
  else
    return __builtin_bit_cast(F32Dims<DTL>, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
}

// Column operand of tile rows row0 .. row0 + 31.
template <int DTL>
struct F32Cols {
  F32Dims<DTL> n[16];
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, int row0, int stride_b, int l32,
                                       int hh, int D) {
    // (dims past D: out of range from any row of the tile, without a wrap)
    const int base = l32 * DTL < D ? (row0 + 4 * hh) * stride_b + l32 * DTL * 4 : kF32Oob;
#pragma unroll
    for (int r = 0; r < 16; ++r)
      n[r] = f32_load_dims<DTL>(
          rs, static_cast<int>(static_cast<unsigned>(base) +
                               static_cast<unsigned>((8 * (r >> 2) + (r & 3)) * stride_b)));
  }
  // Whether any value of the tile is infinite or NaN (in any lane).
  __device__ __forceinline__ bool any_nonfinite() const {
    float z = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int dt = 0; dt < DTL; ++dt) z = fmaf(n[r].v[dt], 0.f, z);
    return __ballot(z != 0.f) != 0;
  }
};

// acc += A B over the tile's 32 rows, B an accumulator (P or dS).
template <int DTL>
__device__ __forceinline__ void f32_outer(f32x16_t (&acc)[DTL], const F32Cols<DTL>& A,
                                          const f32x16_t& B) {
#pragma unroll
  for (int r = 0; r < 16; ++r)
#pragma unroll
    for (int dt = 0; dt < DTL; ++dt) acc[dt] = f32_mma(A.n[r].v[dt], B[r], acc[dt]);
}

// A masked pair's P (or dS) is this value: it adds nothing, and f32_outer_guarded
// can tell it from a probability that underflowed.
constexpr float kF32Masked = -0.0f;

// f32_outer for a tile with infinite or NaN entries in A and masked pairs in B:
// a masked pair must not touch them (0 * inf), so the pairs are taken one by
// one and the masked ones left out. Rare (only tiles that hold both), so a
// rolled loop: B goes through 32 x 33 floats of this wave's LDS.
template <int DTL>
__device__ __forceinline__ void f32_outer_guarded(f32x16_t (&acc)[DTL], __amdgpu_buffer_rsrc_t rs,
                                                  int row0, int stride_b, const f32x16_t& B,
                                                  float* scratch, int l32, int hh, int D) {
#pragma unroll
  for (int r = 0; r < 16; ++r) scratch[(8 * (r >> 2) + 4 * hh + (r & 3)) * 33 + l32] = B[r];
  lc_compiler_fence();
#pragma unroll 1
  for (int n = 0; n < 32; ++n) {
    const float b = scratch[n * 33 + l32];
    const bool seen = __float_as_uint(b) != 0x80000000u;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int d = (8 * (r >> 2) + 4 * hh + (r & 3)) * DTL;
      const F32Dims<DTL> x =
          f32_load_dims<DTL>(rs, d < D ? (row0 + n) * stride_b + d * 4 : kF32Oob);
#pragma unroll
      for (int dt = 0; dt < DTL; ++dt)
        if (seen) acc[dt][r] = fmaf(x.v[dt], b, acc[dt][r]);
    }
  }
  lc_compiler_fence();
}

// This wave's accumulator (dims x 32 columns) into its LDS slab, column-major:
// column c at c * (DPAD + 4), dim d at + d.
template <int DPAD>
__device__ __forceinline__ void f32_put(float* slab, const f32x16_t (&acc)[DPAD / 32], int l32,
                                        int hh) {
  constexpr int DTL = DPAD / 32;
#pragma unroll
  for (int r = 0; r < 16; ++r)
#pragma unroll
    for (int dt = 0; dt < DTL; ++dt)
      slab[l32 * (DPAD + 4) + (8 * (r >> 2) + 4 * hh + (r & 3)) * DTL + dt] = acc[dt][r];
}

// Work item of a causal grid of `units` heads x n blocks, heaviest block rank
// first: rounds of `cus` workgroups in turn up and down, so that the two a CU
// takes together weigh about the same everywhere. (A partial last round keeps
// its order.)
__device__ __forceinline__ int f32_snake(int lin, int total, int cus) {
  const int round = lin / cus;
  if ((round & 1) && (round + 1) * cus <= total) return (2 * round + 1) * cus - 1 - lin;
  return lin;
}

}  // namespace lc_attn
