// skinny_linear.hip — out[T, N] = norm(x)[T, K] . w[K, N] for the few rows of
// a decode step (T <= 16), bf16 in and out, fp32 accumulation, the RMS norm of
// the rows optional and in the same launch.
//
// Bound by the latency of one pass over w (12.6 MB for a 2048 x 3072
// projection, ~2 us of HBM time): there is no reuse, so nothing is tiled for
// reuse.  A workgroup of 16 waves owns 32 columns (64 bytes of each w row);
// each wave takes a contiguous share of k, so a workgroup has its whole slab
// in flight at once (K = 2048: 4 steps of 32 rows per wave).  The partial sums
// meet in LDS.
//
// Products on v_mfma_f32_16x16x32_bf16 with the tokens as A (16 rows, rows
// past T are zero) and w as B.  A lane (c = lane % 16, g = lane / 16) reads
// rows 8 g .. 8 g + 7 of a step at columns 2 c and 2 c + 1 (16 lanes cover the
// 64 bytes), so product i takes columns {2 c + i} and its operand is 4 byte
// permutes of the lane's own registers; no LDS transpose.
//
// Norm: the weight loads of the first steps are issued first, then every wave
// sums its share of each row's squares, the shares meet in LDS, and the
// operand is bf16(x * rsqrt * gamma), rounded as row_norm rounds it.
//
// Measured per call (us, graph replays, weights rotated, T = 8; row norm +
// library GEMM against this kernel): 2048 x 3072 15.4 -> 10.1, 4096 x 6144 28.2
// -> 24.9, 2880 x 5120 28.8 -> 21.3, 8192 x 4096 48.6 -> 42.6; without the norm
// 2048 x 2048 8.8 -> 7.2, 4096 x 4096 21.9 -> 19.0.  64 columns per workgroup
// (whole lines, half the workgroups): 2048 x 3072 with norm 11.7; nontemporal
// weight loads 13.8.  Past N = 8192 (more than one workgroup per CU) the
// library is faster: 8192 x 10240 53.8 against 89.9.  A deep K with few columns
// leaves CUs idle: 8192 x 1024 with norm 39.5 against 34.2 at T = 8, 16384 x 32
// 41.9 against 29.0 at T = 16; the wrapper's rule keeps those on the library.
#include "mia_device.h"
#include "mia_internal.h"

namespace mia {
namespace {

constexpr int kSkinnyWaves = 16;
constexpr int kSkinnyCols = 32;
constexpr int kSkinnyRows = 16;  // tokens at most
constexpr int kSkinnyStep = 32;  // k rows per MFMA step
constexpr int kSkinnyBatch = 4;  // steps loaded together

template <bool NORM>
__global__ __launch_bounds__(kSkinnyWaves * 64) void skinny_linear_kernel(
    mia_skinny_linear_args a) {
  __shared__ __attribute__((aligned(16))) float red[kSkinnyWaves][kSkinnyRows][kSkinnyCols];
  __shared__ float sq[kSkinnyWaves][kSkinnyRows];
  const int tid = threadIdx.x;
  const int wave = readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int c = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * kSkinnyCols;
  const int steps = a.k / kSkinnyStep;
  // this wave's steps [s0, s1)
  const int s0 = steps * wave / kSkinnyWaves, s1 = steps * (wave + 1) / kSkinnyWaves;
  const uint16_t *w = (const uint16_t *)a.w + n0 + 2 * c + (int64_t)(8 * g) * a.w_stride;
  const int tok = min(c, a.rows - 1);  // A row of this lane; rows past the last are zeroed
  const bool live = c < a.rows;
  const uint16_t *x = (const uint16_t *)a.x + (int64_t)tok * a.x_stride + 8 * g;

  uint32_t wr[kSkinnyBatch][8];
  auto load_w = [&](int s) {
#pragma unroll
    for (int b = 0; b < kSkinnyBatch; ++b) {
      // past the share: its last step again (not used)
      const uint16_t *p = w + (int64_t)(min(s + b, s1 - 1) * kSkinnyStep) * a.w_stride;
#pragma unroll
      for (int r = 0; r < 8; ++r)
        wr[b][r] = *reinterpret_cast<const uint32_t *>(p + (int64_t)r * a.w_stride);
    }
  };
  if (s0 < s1) load_w(s0);

  float scale = 1.0f;
  if constexpr (NORM) {
    float ss = 0.f;
    for (int s = s0; s < s1; ++s) {
      const u32x4_t v = *reinterpret_cast<const u32x4_t *>(x + s * kSkinnyStep);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float lo = bf16lo(v[e]), hi = bf16hi(v[e]);
        ss += lo * lo + hi * hi;
      }
    }
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    if (g == 0) sq[wave][c] = ss;
    __syncthreads();
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < kSkinnyWaves; ++i) sum += sq[i][c];
    scale = 1.0f / sqrtf(sum / (float)(a.dim_actual > 0 ? a.dim_actual : a.k) + a.eps);
  }

  f32x4_t acc[2] = {};
  for (int s = s0; s < s1; s += kSkinnyBatch) {
#pragma unroll
    for (int b = 0; b < kSkinnyBatch; ++b) {
      if (s + b < s1) {
        const int k = (s + b) * kSkinnyStep;
        u32x4_t xv = *reinterpret_cast<const u32x4_t *>(x + k);
        if constexpr (NORM) {
          float y[8];
#pragma unroll
          for (int e = 0; e < 8; ++e)
            y[e] = ((e & 1) ? bf16hi(xv[e >> 1]) : bf16lo(xv[e >> 1])) * scale;
          if (a.gamma_bf16) {
            const u32x4_t gv = *reinterpret_cast<const u32x4_t *>((const uint16_t *)a.gamma + k + 8 * g);
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] *= (e & 1) ? bf16hi(gv[e >> 1]) : bf16lo(gv[e >> 1]);
          } else if (a.gamma) {
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] *= ((const float *)a.gamma)[k + 8 * g + e];
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) xv[e] = pack2_bf16(y[2 * e], y[2 * e + 1]);
        }
        if (!live) xv = u32x4_t{0u, 0u, 0u, 0u};
        const bf16x8_t av = __builtin_bit_cast(bf16x8_t, xv);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const uint32_t sel = i ? 0x07060302u : 0x05040100u;
          u32x4_t bw;
#pragma unroll
          for (int j = 0; j < 4; ++j)
            bw[j] = __builtin_amdgcn_perm(wr[b][2 * j + 1], wr[b][2 * j], sel);
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, __builtin_bit_cast(bf16x8_t, bw),
                                                           acc[i], 0, 0, 0);
        }
      }
    }
    if (s + kSkinnyBatch < s1) load_w(s + kSkinnyBatch);
  }
  // lane (c, g) holds tokens 4 g .. 4 g + 3 of columns 2 c and 2 c + 1
#pragma unroll
  for (int e = 0; e < 4; ++e)
    *reinterpret_cast<float2 *>(&red[wave][4 * g + e][2 * c]) = make_float2(acc[0][e], acc[1][e]);
  __syncthreads();
  const int t = tid / kSkinnyCols, n = tid % kSkinnyCols;  // at most one output per thread
  if (t < a.rows) {
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < kSkinnyWaves; ++i) v += red[i][t][n];
    ((uint16_t *)a.out)[(int64_t)t * a.out_stride + n0 + n] = (uint16_t)(pack2_bf16(v, 0.f) & 0xffffu);
  }
}

}  // namespace

int launch_skinny_linear(const mia_skinny_linear_args &a, hipStream_t s) {
  const dim3 grid((unsigned)(a.n / kSkinnyCols));
  if (a.norm)
    hipLaunchKernelGGL(skinny_linear_kernel<true>, grid, dim3(kSkinnyWaves * 64), 0, s, a);
  else
    hipLaunchKernelGGL(skinny_linear_kernel<false>, grid, dim3(kSkinnyWaves * 64), 0, s, a);
  return check_hip(hipGetLastError(), "skinny linear launch");
}

}  // namespace mia
