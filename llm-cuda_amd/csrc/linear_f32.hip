// y = x W^T in fp32 (x [M, K], W [N, K]) for the inference projections of fp32
// models: v_mfma_f32_32x32x2_f32, operands straight from L2 (attn_f32.h).
//
// Workgroup = one 32 x 32 tile of y; its 8 waves each contract an eighth of K
// and the sums are added through LDS in wave order. The projections this takes
// are small (a prompt's rows against a few hundred columns), so what bounds
// them is the length of a wave's chain and the launch, not the matrix rate:
// splitting K inside the workgroup shortens the chain by 8 with no second
// launch, and a tile per workgroup spreads the work over the CUs. Graph-replayed
// us a call against the library's GEMM: [128, 256] x [256, 256] 4.5 / 33.4,
// [128, 688] x [688, 256] 6.6 / 83.1 (it runs one workgroup there),
// [128, 256] x [256, 512] 4.5 / 5.7; four waves 5.1, 7.9 and 5.1.
#include "attn_f32.h"
#include "lc_common.h"

namespace {

using namespace lc_attn;

struct LinF32Args {
  const float* x;
  const float* w;
  float* y;
  int64_t xs, ws, ys;
  int64_t M, N;
  int K;
};

constexpr int kLinWaves = 8;
constexpr int kLinChunks = 4;  // 8-element K chunks per step (32 k: 16 MFMAs)

__global__ __launch_bounds__(64 * kLinWaves) void linear_f32_kernel(LinF32Args a) {
  constexpr int LD = 36;
  __shared__ __align__(16) float slab[kLinWaves][32 * LD];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;
  const int64_t n0 = (int64_t)blockIdx.x * 32, m0 = (int64_t)blockIdx.y * 32;
  const int rows_n = static_cast<int>(min((int64_t)32, a.N - n0));
  const int rows_m = static_cast<int>(min((int64_t)32, a.M - m0));
  // Descriptors over this tile's rows alone (rows past them read zeros).
  const __amdgpu_buffer_rsrc_t wrs = f32_rsrc(a.w + n0 * a.ws, f32_bytes(rows_n, a.ws, a.K));
  const __amdgpu_buffer_rsrc_t xrs = f32_rsrc(a.x + m0 * a.xs, f32_bytes(rows_m, a.xs, a.K));
  const int wbase = static_cast<int>(l32 * a.ws * 4) + hh * 16;
  const int xbase = static_cast<int>(l32 * a.xs * 4) + hh * 16;
  const int chunks = (a.K + 7) / 8;
  const int c0 = static_cast<int>((int64_t)chunks * wave / kLinWaves);
  const int c1 = static_cast<int>((int64_t)chunks * (wave + 1) / kLinWaves);

  f32x4_t aw[2][kLinChunks], ax[2][kLinChunks];
  auto load = [&](int c, int p) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kLinChunks; ++i) {
      const bool ok = c + i < c1 && (c + i) * 8 + hh * 4 < a.K;
      const int off = (c + i) * 32;
      aw[p][i] = __builtin_bit_cast(
          f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(wrs, ok ? wbase + off : kF32Oob, 0, 0));
      ax[p][i] = __builtin_bit_cast(
          f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(xrs, ok ? xbase + off : kF32Oob, 0, 0));
    }
  };
  f32x16_t acc;
  f32_zero(acc);
  auto step = [&](int p) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kLinChunks; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = f32_mma(aw[p][i][e], ax[p][i][e], acc);
  };
  load(c0, 0);
  for (int c = c0; c < c1; c += 2 * kLinChunks) {
    load(c + kLinChunks, 1);
    step(0);
    load(c + 2 * kLinChunks, 0);
    if (c + kLinChunks < c1) step(1);
  }
  // acc: rows n (registers), columns m (lanes); summed as y rows.
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const f32x4_t v = {acc[4 * j], acc[4 * j + 1], acc[4 * j + 2], acc[4 * j + 3]};
    *reinterpret_cast<f32x4_t*>(&slab[wave][l32 * LD + 8 * j + 4 * hh]) = v;
  }
  __syncthreads();
  const int m = tid >> 3, n = (tid & 7) * 4;
  if (m >= rows_m || n >= rows_n) return;  // (and the upper half of the threads: m >= 32)
  f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < kLinWaves; ++w)
    sum += *reinterpret_cast<const f32x4_t*>(&slab[w][m * LD + n]);
  *reinterpret_cast<f32x4_t*>(a.y + (m0 + m) * a.ys + n0 + n) = sum;
}

}  // namespace

extern "C" {

int lc_linear_f32(const float* x, int64_t x_stride, const float* w, int64_t w_stride, float* y,
                  int64_t y_stride, int64_t M, int64_t N, int64_t K, void* stream) {
  LC_REQUIRE(M >= 0 && N >= 0 && K >= 0, "lc_linear_f32: bad shape");
  if (M == 0 || N == 0) return LC_OK;
  LC_REQUIRE(y && ((x && w) || K == 0), "lc_linear_f32: null pointer");
  LC_REQUIRE(N % 4 == 0 && K % 4 == 0, "lc_linear_f32: N and K must be multiples of 4");
  LC_REQUIRE(lc_aligned(y, 16) && y_stride % 4 == 0 && lc_aligned(x, 4) && lc_aligned(w, 4),
             "lc_linear_f32: y rows must be 16-byte aligned");
  LC_REQUIRE(x_stride >= K && w_stride >= K && y_stride >= N, "lc_linear_f32: overlapping rows");
  LC_REQUIRE((32 * x_stride + K) * 4 < kF32Oob && (32 * w_stride + K) * 4 < kF32Oob,
             "lc_linear_f32: rows too far apart");
  const int64_t gm = lc_cdiv(M, 32), gn = lc_cdiv(N, 32);
  LC_REQUIRE(gn < (1LL << 31) && gm < 65536, "lc_linear_f32: grid too large");
  const LinF32Args a{x, w, y, x_stride, w_stride, y_stride, M, N, static_cast<int>(K)};
  linear_f32_kernel<<<dim3((unsigned)gn, (unsigned)gm), 64 * kLinWaves, 0, lc_stream(stream)>>>(a);
  return lc_check_launch("lc_linear_f32");
}

}  // extern "C"
