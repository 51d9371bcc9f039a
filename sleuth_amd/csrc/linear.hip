// Linear layers of a decode or verify step: y = x . W^T for at most 16 rows of x (the batch times
// the step's tokens), with the work around it in the same launch: RMSNorm of x before it, the
// bias, the residual sum or the SwiGLU product after it.
//
// What bounds it. W is read once (2 N K bytes) and 16 rows do not fill a GEMM tile, so the call
// is a stream of W: latency at the sizes of one layer (2 to 12 MB), HBM or MALL bandwidth above.
// A step of a layer is a chain of such calls, so launches and their gaps cost as much as the
// streams, hence the fused neighbours.
//
// Split. A block of 8 waves takes 16 output columns; the waves take slices of K, all their W
// loads (16 bytes per lane, up to kAhead k-steps) in flight before anything else, and add their
// tiles through LDS in wave order. On v_mfma_f32_16x16x32 the 16 W rows are the A operand and the
// (up to 16) x rows the B operand, both straight from memory in operand layout, so the same kernel
// serves 1 to 16 rows at the cost of one. A row's result does not depend on the other rows.
// Measured against hipBLASLt (bf16, graph replays of the call alone, one box), N x K at 1 / 5 / 16
// rows: 4096 x 1024: 5.1 / 5.1 / 5.5 us against 6.3; 1024 x 2048: 5.0 / 5.1 / 5.9 against 8.2; 1024 x
// 3072: 7.5 / 7.6 / 8.8 against 9.4; 8192 x 1024: 7.0 / 7.2 / 8.1 against 6.7; 32768 x 4096: 51 / 53 /
// 74 against 62. A four-layer model's decode step (d 1024, hidden 3072; GraphDecoder) with the norms,
// residual sums and SwiGLU product in these launches (and the RoPE rows converted once per pass): 416 -> 207 us.
#include "common.h"
#include "forge_internal.h"

namespace forge {

typedef __bf16 l_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 l_f16x8 __attribute__((ext_vector_type(8)));
typedef float l_floatx4 __attribute__((ext_vector_type(4)));

template <typename T> struct LMfma;
template <> struct LMfma<bf16> {
  typedef l_bf16x8 vec;
  static __device__ __forceinline__ l_floatx4 run(vec a, vec b, l_floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct LMfma<f16> {
  typedef l_f16x8 vec;
  static __device__ __forceinline__ l_floatx4 run(vec a, vec b, l_floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

struct LinearParams {
  const void* x;
  int64_t sx;
  const void* w;
  const void* w2;  // SwiGLU: w is the gate, w2 the up projection
  int64_t sw;
  const void* bias;
  const void* gain;  // RMSNorm of x (norm != 0), or null; fp32 or of x's type, as the module holds it
  int gain_f32;
  int norm;
  float eps;
  const void* res;
  int64_t sr;
  void* out;
  int64_t so;
  int M, N, K;
};

constexpr int kLinWaves = 8;
constexpr int kLinRows = 16;   // rows of x
constexpr int kLinCols = 16;   // output columns per block
constexpr int kAhead = 8;      // k-steps whose W loads are in flight

template <typename T, bool GATED>
__global__ __launch_bounds__(64 * kLinWaves)
void linear_small_kernel(LinearParams p) {
  using V8 = typename LMfma<T>::vec;
  constexpr int NT = GATED ? 2 : 1;  // tiles per wave
  __shared__ float sh_rs[kLinRows];
  __shared__ float sh_acc[kLinWaves][NT][kLinCols * kLinRows];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lane = tid % kWave;
  const int r = lane & 15;  // W row of the tile (A operand), x row (B operand)
  const int g = lane >> 4;  // channels 32 s + 8 g .. + 7 of k-step s
  const int n0 = blockIdx.x * kLinCols;
  const int n = n0 + r < p.N ? n0 + r : p.N - 1;  // columns past N repeat the last one, not written

  // this wave's k-steps
  const int steps = p.K / 32;
  const int s_lo = (int)((int64_t)steps * wave / kLinWaves), s_hi = (int)((int64_t)steps * (wave + 1) / kLinWaves);
  const T* wp[NT];
  wp[0] = static_cast<const T*>(p.w) + n * p.sw + 8 * g;
  if constexpr (GATED) wp[1] = static_cast<const T*>(p.w2) + n * p.sw + 8 * g;
  uint4 wr[NT][kAhead];
  auto load_w = [&](int s0) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int s = s0 + i < s_hi ? s0 + i : s_hi - 1;  // (a wave with no step skips the loop)
#pragma unroll
      for (int t = 0; t < NT; ++t) wr[t][i] = load16(wp[t] + 32 * s);
    }
  };
  if (s_lo < s_hi) load_w(s_lo);

  const bool row = r < p.M;
  const T* xp = static_cast<const T*>(p.x) + (row ? r : 0) * p.sx + 8 * g;
  float rs = 1.0f;
  if (p.norm) {  // RMSNorm factors of the rows: wave w takes rows w and w + 8
#pragma unroll
    for (int j = 0; j < kLinRows / kLinWaves; ++j) {
      const int m = wave + kLinWaves * j;
      if (m < p.M) {
        const T* xr = static_cast<const T*>(p.x) + m * p.sx;
        float ss = 0.0f;
        for (int k = 8 * lane; k < p.K; k += 8 * kWave) {
          float v[8];
          unpack16<T>(load16(xr + k), v);
#pragma unroll
          for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
        }
        ss = group_sum<kWave>(ss);
        if (lane == 0) sh_rs[m] = rsqrtf(ss / (float)p.K + p.eps);
      }
    }
    __syncthreads();
    rs = row ? sh_rs[r] : 0.0f;
  }

  l_floatx4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = l_floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int s0 = s_lo; s0 < s_hi; s0 += kAhead) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int s = s0 + i;
      if (s < s_hi) {  // wave-uniform
        uint4 xr = make_uint4(0, 0, 0, 0);
        if (row) xr = load16(xp + 32 * s);
        if (p.norm) {
          float v[8];
          unpack16<T>(xr, v);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] *= rs;
          if (p.gain) {
            float w[8];
            if (p.gain_f32) load_f32x8(static_cast<const float*>(p.gain) + 32 * s + 8 * g, w);
            else unpack16<T>(load16(static_cast<const T*>(p.gain) + 32 * s + 8 * g), w);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] *= w[e];
          }
          xr = pack16<T>(v);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t)
          acc[t] = LMfma<T>::run(__builtin_bit_cast(V8, wr[t][i]), __builtin_bit_cast(V8, xr), acc[t]);
      }
    }
    if (s0 + kAhead < s_hi) load_w(s0 + kAhead);
  }

  // tile element (column 4 g + j of the block, x row r) of every wave, added in wave order
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) sh_acc[wave][t][r * kLinCols + 4 * g + j] = acc[t][j];
  __syncthreads();
  if (tid >= kLinCols * kLinRows) return;
  const int m = tid / kLinCols, c = n0 + tid % kLinCols;
  if (m >= p.M || c >= p.N) return;
  float v[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    v[t] = sh_acc[0][t][tid];
#pragma unroll
    for (int w = 1; w < kLinWaves; ++w) v[t] += sh_acc[w][t][tid];
  }
  float y = v[0];
  if (p.bias) y += to_f32<T>(static_cast<const T*>(p.bias)[c]);
  // each torch op of the eager layer rounds to the dtype; so do the fused ones
  if constexpr (GATED) {
    const float gt = fp32_result(to_f32<T>(from_f32<T>(v[0])));
    const float up = to_f32<T>(from_f32<T>(v[1]));
    const float act = to_f32<T>(from_f32<T>(gt / (1.0f + expf(-gt))));
    y = act * up;
  }
  if (p.res)
    y = to_f32<T>(from_f32<T>(y)) + to_f32<T>(static_cast<const T*>(p.res)[m * p.sr + c]);
  static_cast<T*>(p.out)[m * p.so + c] = from_f32<T>(y);
}

template <typename T>
static int launch_linear(const LinearParams& p, hipStream_t s) {
  const dim3 grid((unsigned)((p.N + kLinCols - 1) / kLinCols));
  if (p.w2) hipLaunchKernelGGL((linear_small_kernel<T, true>), grid, dim3(64 * kLinWaves), 0, s, p);
  else hipLaunchKernelGGL((linear_small_kernel<T, false>), grid, dim3(64 * kLinWaves), 0, s, p);
  return check_launch();
}

}  // namespace forge

using namespace forge;

extern "C" int forge_linear_small(int dtype, int M, int N, int K, const void* x, int64_t sx, const void* w,
                                  const void* w2, int64_t sw, const void* bias, const void* gain,
                                  int gain_dtype, int norm, float eps, const void* residual, int64_t sr, void* out, int64_t so,
                                  void* stream) {
  clear_error();
  if (dtype != FORGE_BF16 && dtype != FORGE_F16) return set_error("forge_linear_small: dtype must be bf16 or fp16");
  if (M <= 0 || M > kLinRows) return set_error("forge_linear_small: 1 to 16 rows");
  if (N <= 0 || K <= 0 || K % 32) return set_error("forge_linear_small: K must be a positive multiple of 32");
  if (!x || !w || !out) return set_error("null tensor pointer");
  if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)w2 | (uintptr_t)gain) % 16)
    return set_error("forge_linear_small: x, the weights and the gain must be 16-byte aligned");
  if (gain && gain_dtype != FORGE_F32 && gain_dtype != dtype)
    return set_error("forge_linear_small: the gain must be fp32 or of x's type");
  if (sx % 8 || sw % 8 || sw < K || (M > 1 && sx < K))
    return set_error("forge_linear_small: row strides must be multiples of 8 elements and hold a row");
  if (w2 && (bias || residual)) return set_error("forge_linear_small: SwiGLU takes no bias or residual");
  LinearParams p{x, sx, w, w2, sw, bias, gain, gain_dtype == FORGE_F32, norm, eps, residual, sr, out, so, M, N, K};
  hipStream_t s = (hipStream_t)stream;
  return dtype == FORGE_BF16 ? launch_linear<bf16>(p, s) : launch_linear<f16>(p, s);
}
