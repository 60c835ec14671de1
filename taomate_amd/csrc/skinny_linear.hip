// Linear layers over a handful of rows (gfx950): y = act(x) W^T + bias for
// x [M, K], M <= 8, as the timestep MLPs run them (AdaLayerNormSingle,
// ltx_causal/transformer/compat.py:212-275: one row per sample, K up to 4096,
// N up to 24576).
//
// Bound by the read of W, once: 201 MB for 4096 -> 24576.  Every wave streams
// whole rows of W, 16 bytes per lane, two rows at a time; x (after SiLU, rounded
// to bf16 as the tensor op rounds) sits in LDS.  At M = 2 against hipBLASLt:
// 35.9 against 43.2 us (5.6 TB/s) for 4096 -> 24576, 25.4 against 30.8 us for
// 4096 -> 16384, 8.9 against 11.7 us for 4096 -> 4096, 3.0 against 3.6 us for
// 256 -> 4096.  A call queues in 6 us of host time where nn.Linear takes 20 and
// the SiLU is not a launch of its own: a step has 18 of these layers, and the
// two-block step, whose host time shows, went from 4.3 to 4.0 ms.
// Products and sums are float32 (v_dot2_f32_bf16 over bf16 pairs), the result
// is rounded once, after the bias.

#include "ltx_common.h"

namespace ltx {

constexpr int kSkinnyMaxK = LTX_SKINNY_MAX_K;   // x chunk loop bound: K / 512 chunks per lane
constexpr int kSkinnyMaxM = LTX_SKINNY_MAX_ROWS;
constexpr int kSkinnyThreads = 256;

struct SkinnyArgs {
  const uint16_t* x;
  int64_t x_ls;
  const uint16_t* w;
  int64_t w_ls;
  const uint16_t* bias;  // null: none
  uint16_t* y;
  int64_t y_ls;
  int64_t N;
  int M, K, silu;
};

// One wave per row pair of W, grid-strided.  CH: 512-element chunks of K
// (lanes past K read nothing and add nothing).
template <int M, int CH>
__global__ void __launch_bounds__(kSkinnyThreads) skinny_linear_kernel(const SkinnyArgs a) {
  constexpr int kRows = 2;
  extern __shared__ uint4 xs[];  // [M][K / 8]
  const int lane = threadIdx.x & 63;
  const int nch = a.K / 8;
  const int64_t waves = (int64_t)gridDim.x * (kSkinnyThreads / 64);
  int64_t n = ((int64_t)blockIdx.x * (kSkinnyThreads / 64) + (threadIdx.x >> 6)) * kRows;
  uint4 w[kRows][CH];
  auto load = [&](int64_t n0) {
#pragma unroll
    for (int r = 0; r < kRows; ++r)
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int i = c * 64 + lane;
        w[r][c] = make_uint4(0, 0, 0, 0);
        if (n0 + r < a.N && i < nch) w[r][c] = *reinterpret_cast<const uint4*>(a.w + (n0 + r) * a.w_ls + i * 8);
      }
  };
  load(n);  // the first rows of W travel while x is staged
  for (int i = threadIdx.x; i < M * nch; i += kSkinnyThreads) {
    const int m = i / nch, c = i - m * nch;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (m < a.M) v = *reinterpret_cast<const uint4*>(a.x + m * a.x_ls + c * 8);
    if (a.silu) {
      uint32_t* p = &v.x;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float lo = bf16_bits_to_f32(p[e] & 0xFFFFu), hi = bf16_bits_to_f32(p[e] >> 16);
        p[e] = pack_bf16x2(lo / (1.0f + expf(-lo)), hi / (1.0f + expf(-hi)));
      }
    }
    xs[i] = v;
  }
  __syncthreads();
  for (; n < a.N; n += waves * kRows) {
    float acc[kRows][M] = {};
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int i = c * 64 + lane;
      if (i < nch) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
          const uint4 xv = xs[m * nch + i];
          const uint32_t* xp = &xv.x;
#pragma unroll
          for (int r = 0; r < kRows; ++r) {
            const uint32_t* wp = &w[r][c].x;
#pragma unroll
            for (int e = 0; e < 4; ++e)
              acc[r][m] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(ltx_bf16x2_t, wp[e]),
                                                          __builtin_bit_cast(ltx_bf16x2_t, xp[e]), acc[r][m], false);
          }
        }
      }
    }
    const int64_t n0 = n;
    if (n + waves * kRows < a.N) load(n + waves * kRows);  // the next rows travel during the reduction
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
      for (int r = 0; r < kRows; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[r][m] += __shfl_xor(acc[r][m], off, 64);
    // lane r * M + m writes row n0 + r of sample m
    float v = 0.0f;
#pragma unroll
    for (int r = 0; r < kRows; ++r)
#pragma unroll
      for (int m = 0; m < M; ++m) v = lane == r * M + m ? acc[r][m] : v;
    const int r = lane / M, m = lane - r * M;
    if (lane < kRows * M && m < a.M && n0 + r < a.N) {
      if (a.bias != nullptr) v += bf16_bits_to_f32(a.bias[n0 + r]);
      a.y[m * a.y_ls + n0 + r] = (uint16_t)f32_to_bf16_bits(v);
    }
  }
}

template <int M>
void launch_skinny(const SkinnyArgs& a, unsigned blocks, hipStream_t st) {
  const size_t lds = (size_t)M * a.K * 2;
  const int ch = (a.K + 511) / 512;
  if (ch <= 1)
    hipLaunchKernelGGL((skinny_linear_kernel<M, 1>), dim3(blocks), dim3(kSkinnyThreads), lds, st, a);
  else if (ch <= 4)
    hipLaunchKernelGGL((skinny_linear_kernel<M, 4>), dim3(blocks), dim3(kSkinnyThreads), lds, st, a);
  else
    hipLaunchKernelGGL((skinny_linear_kernel<M, 8>), dim3(blocks), dim3(kSkinnyThreads), lds, st, a);
}

}  // namespace ltx

using namespace ltx;

extern "C" int ltx_skinny_linear(int64_t M, int64_t N, int64_t K, const void* x, int64_t x_ls, int silu,
                                 const void* w, int64_t w_ls, const void* bias, void* y, int64_t y_ls,
                                 void* stream) {
  clear_error();
  LTX_REQUIRE(M >= 1 && M <= kSkinnyMaxM, "ltx_skinny_linear: M must be in [1, %d]", kSkinnyMaxM);
  LTX_REQUIRE(K >= 8 && K <= kSkinnyMaxK && K % 8 == 0, "ltx_skinny_linear: K must be a multiple of 8 in [8, %d]",
              kSkinnyMaxK);
  LTX_REQUIRE(N >= 0 && N <= 0x7FFFFFFF, "ltx_skinny_linear: bad N");
  LTX_REQUIRE(x != nullptr && w != nullptr && y != nullptr, "ltx_skinny_linear: null pointer");
  LTX_REQUIRE((uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0 && x_ls % 8 == 0 && w_ls % 8 == 0,
              "ltx_skinny_linear: rows must be 16-byte aligned");
  if (N == 0) return LTX_OK;
  SkinnyArgs a{(const uint16_t*)x, x_ls, (const uint16_t*)w, w_ls, (const uint16_t*)bias, (uint16_t*)y, y_ls,
               N, (int)M, (int)K, silu};
  // two workgroups of four waves per CU at K = 4096 (each wave has two rows of
  // W, 16 KB, in flight), more for shorter rows; fewer rows of W than that
  // take one wave per row pair
  const int64_t want = ceil_div(N, 2 * (kSkinnyThreads / 64)), most = K > 2048 ? 512 : K > 1024 ? 1024 : 2048;
  const unsigned blocks = (unsigned)(want < most ? want : most);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (M == 1)
    launch_skinny<1>(a, blocks, st);
  else if (M == 2)
    launch_skinny<2>(a, blocks, st);
  else if (M <= 4)
    launch_skinny<4>(a, blocks, st);
  else
    launch_skinny<8>(a, blocks, st);
  LTX_LAUNCH_CHECK("ltx_skinny_linear");
  return LTX_OK;
}
