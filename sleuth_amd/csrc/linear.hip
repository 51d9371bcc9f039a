// Linear layers of a decode or verify step: y = x . W^T for at most 16 rows of x (the batch times
// the step's tokens), with the work around it in the same launch: RMSNorm of x before it, the
// bias, the residual sum or the SwiGLU product after it.
//
// What bounds it. W is read once (2 N K bytes) and 16 rows do not fill a GEMM tile, so the call
// is a stream of W: latency at the sizes of one layer (2 to 12 MB), HBM or MALL bandwidth above.
// A step of a layer is a chain of such calls, so launches and their gaps cost as much as the
// streams, hence the fused neighbours.
//
// Split. A block of 8 waves takes 16 output columns; the waves take slices of K and add their tiles
// through LDS in wave order. On v_mfma_f32_16x16x32 the 16 W rows are the A operand and the (up to
// 16) x rows the B operand, both straight from memory in operand layout, so the same kernel serves 1
// to 16 rows. A row's result does not depend on the other rows. Every load of a slice (x, the gain,
// W; A k-steps of them) goes out before anything is computed, and a slot's next load as soon as the
// slot is used. The RMSNorm sums the squares of the slices that the products read, so x is read
// once and the norm adds one barrier: a pass over x of its own, with W's loads only in flight, took
// 1.3 us more at K 1,024 (5.2 us against 3.9 without the norm; now 3.7 against 2.7).
//
// Measured: bf16, graph replays of the call alone on one W, which the 256 MB MALL then holds; 1 / 5 / 16
// rows, us; in brackets the form before, one box each. (A W of its own per call, as in a model: LinRule
// below. Launched one by one on idle CUs: 1 to 2 us more.) 4096 x 1024 with norm 3.7 / 3.9 / 4.4 (5.2 /
// 5.4 / 6.2), hipBLASLt's product alone 6.3; 1024 x 2048 with residual 3.8 / 4.1 / 5.2 (4.3 / 4.4 / 5.2),
// hipBLASLt 8.2; 3072 x 1024 SwiGLU with norm 4.7 / 4.9 / 5.4 (6.9 / 7.3 / 8.2); 1024 x 3072 with residual
// 4.9 / 5.4 / 6.9 (6.4 / 6.7 / 7.8), hipBLASLt 9.4; 8192 x 1024 with norm 5.0 / 5.3 / 6.2 (7.1 / 7.4 / 8.8),
// hipBLASLt 6.7; 6144 x 4096 with norm 16.1 / 18.3 / 25.1 (17.0 / 17.8 / 23.5; 16 rows go to torch).
// A four-layer model's decode step (d 1024, hidden 3072; GraphDecoder), with the norms, residual sums
// and SwiGLU product in these launches: 175 us (206 the form before, 411 with torch's calls).
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
  const void* gain;  // RMSNorm of x (norm != 0): fp32 or of x's type, as the module holds it
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
constexpr int kLinCols = 16;   // output columns of a tile
// Outputs from which a block takes two tiles: x's rows are then read half as often, and two blocks per
// CU are left. On one W: 32768 x 4096 with norm at 5 rows 54 us against 63 with one tile, at 16 rows 66 against 83.
constexpr int kLinWideN = 16384;

// What the kernel does to x's rows first.
enum LinNorm { kLinPlain, kLinGain, kLinGainF32 };  // nothing; RMSNorm with a gain of x's type; with an fp32 gain

// Unpack the register here, not earlier: the floats of all the k-steps in flight would cost a CU its
// second block.
__device__ __forceinline__ void keep_packed(uint4& u) { asm volatile("" : "+v"(u.x), "+v"(u.y), "+v"(u.z), "+v"(u.w)); }

// TILES: tiles of 16 output columns per block; GATED: each of them twice (gate and up); A: k-steps
// whose loads are in flight.
template <typename T, bool GATED, int TILES, int NORM, int A>
__global__ __launch_bounds__(64 * kLinWaves) __attribute__((amdgpu_waves_per_eu(4)))
void linear_small_kernel(LinearParams p) {
  using V8 = typename LMfma<T>::vec;
  constexpr int NT = GATED ? 2 * TILES : TILES;  // MFMA tiles per wave
  __shared__ float sh_ss[kLinWaves][kLinRows];
  __shared__ float sh_acc[kLinWaves][NT][kLinCols * kLinRows];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lane = tid % kWave;
  const int r = lane & 15;  // W row of the tile (A operand), x row (B operand)
  const int g = lane >> 4;  // channels 32 s + 8 g .. + 7 of k-step s
  const int n0 = blockIdx.x * (kLinCols * TILES);

  // this wave's k-steps
  const int steps = p.K / 32;
  const int s_lo = (int)((int64_t)steps * wave / kLinWaves), s_hi = (int)((int64_t)steps * (wave + 1) / kLinWaves);
  const T* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int c = n0 + kLinCols * (t % TILES) + r;
    const int n = c < p.N ? c : p.N - 1;  // columns past N repeat the last one, not written
    wp[t] = static_cast<const T*>(t < TILES ? p.w : p.w2) + n * p.sw + 8 * g;
  }
  // x through a buffer resource: the lanes of rows past M read zeros without an access
  const __amdgpu_buffer_rsrc_t xs = slab_rsrc(p.x, (unsigned)(((p.M - 1) * p.sx + p.K) * sizeof(T)));
  const unsigned x_off = r < p.M ? (unsigned)((r * p.sx + 8 * g) * sizeof(T)) : 0x80000000u;
  auto load_x = [&](int s) {
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(xs, (int)(x_off + 64 * s), 0, 0));
  };
  const T* gp = static_cast<const T*>(p.gain) + 8 * g;
  uint4 wr[NT][A], xr[A], gr[NORM == kLinGain ? A : 1];
  auto load = [&](int i, int s) {  // k-step s (the last one's again where the wave has fewer) into slot i
    const int last = s < s_hi ? s : s_hi - 1, at = 32 * last;
    xr[i] = load_x(last);
    if constexpr (NORM == kLinGain) gr[i] = load16(gp + at);
#pragma unroll
    for (int t = 0; t < NT; ++t) wr[t][i] = load16(wp[t] + at);
  };
  if (s_lo < s_hi) {  // wave-uniform; a wave with no step contributes zeros
#pragma unroll
    for (int i = 0; i < A; ++i) load(i, s_lo + i);
  }

  float rs = 1.0f;
  if constexpr (NORM != kLinPlain) {
    // RMSNorm factors of the rows: each wave sums the squares of its slice, from the registers that
    // the products read as far as those reach
    float ss = 0.0f;
    auto square = [&](uint4 raw) {
      float v[8];
      unpack16<T>(raw, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
    };
#pragma unroll
    for (int i = 0; i < A; ++i)
      if (s_lo + i < s_hi) {  // wave-uniform
        square(xr[i]);
        keep_packed(xr[i]);
      }
    for (int s = s_lo + A; s < s_hi; s += 4) {
      uint4 more[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) more[i] = load_x(s + i < s_hi ? s + i : s_hi - 1);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (s + i < s_hi) square(more[i]);
    }
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    if (g == 0) sh_ss[wave][r] = ss;
    __syncthreads();
    float all = sh_ss[0][r];
#pragma unroll
    for (int w = 1; w < kLinWaves; ++w) all += sh_ss[w][r];
    rs = rsqrtf(all / (float)p.K + p.eps);
  }

  l_floatx4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = l_floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  auto multiply = [&](int i, int s) {
    uint4 xv = xr[i];
    if constexpr (NORM != kLinPlain) {
      float v[8], w[8];
      unpack16<T>(xv, v);
      if constexpr (NORM == kLinGain) {
        keep_packed(gr[i]);
        unpack16<T>(gr[i], w);
      } else load_f32x8(static_cast<const float*>(p.gain) + 32 * s + 8 * g, w);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = v[e] * rs * w[e];
      xv = pack16<T>(v);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
      acc[t] = LMfma<T>::run(__builtin_bit_cast(V8, wr[t][i]), __builtin_bit_cast(V8, xv), acc[t]);
  };
  int s0 = s_lo;
  for (; s0 + A < s_hi; s0 += A) {  // each slot's next loads go out as soon as it is used
#pragma unroll
    for (int i = 0; i < A; ++i) {
      multiply(i, s0 + i);
      load(i, s0 + A + i);
    }
  }
#pragma unroll
  for (int i = 0; i < A; ++i)
    if (s0 + i < s_hi) multiply(i, s0 + i);  // wave-uniform

  // tile element (column 4 g + j of the block, x row r) of every wave, added in wave order
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) sh_acc[wave][t][r * kLinCols + 4 * g + j] = acc[t][j];
  __syncthreads();
  if (tid >= TILES * kLinCols * kLinRows) return;
  const int tile = tid / (kLinCols * kLinRows), in = tid % (kLinCols * kLinRows);
  const int m = in / kLinCols, c = n0 + tile * kLinCols + in % kLinCols;
  if (m >= p.M || c >= p.N) return;
  float v[GATED ? 2 : 1];
#pragma unroll
  for (int t = 0; t < (GATED ? 2 : 1); ++t) {
    v[t] = sh_acc[0][t * TILES + tile][in];
#pragma unroll
    for (int w = 1; w < kLinWaves; ++w) v[t] += sh_acc[w][t * TILES + tile][in];
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

template <typename T, bool GATED, int TILES, int A>
static void launch_plain(const LinearParams& p, dim3 grid, hipStream_t s) {
  hipLaunchKernelGGL((linear_small_kernel<T, GATED, TILES, kLinPlain, A>), grid, dim3(64 * kLinWaves), 0, s, p);
}

template <typename T, bool GATED, int TILES>
static void launch_tiles(const LinearParams& p, hipStream_t s) {
  const dim3 grid((unsigned)((p.N + kLinCols * TILES - 1) / (kLinCols * TILES))), block(64 * kLinWaves);
  if (p.norm) {
    if (p.gain_f32) hipLaunchKernelGGL((linear_small_kernel<T, GATED, TILES, kLinGainF32, 4>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((linear_small_kernel<T, GATED, TILES, kLinGain, 4>), grid, block, 0, s, p);
    return;
  }
  // k-steps in flight: all of a wave's where 12 or fewer. A slot without a step repeats the last one's
  // loads, so slots fit the steps: 12 slots for 4 steps, and x's rows past M read as row 0, took 4.6 us
  // at 4096 x 1024; 4 slots and no such reads 2.7 us. Kernels with a norm or two tiles have 4 slots:
  // 8 need up to 229 registers, which leaves one block per CU.
  const int steps = (p.K / 32 + kLinWaves - 1) / kLinWaves;  // of a wave
  if (GATED || TILES > 1 || steps <= 4) launch_plain<T, GATED, TILES, 4>(p, grid, s);
  else if (steps > 8 && steps <= 12) launch_plain<T, false, 1, 12>(p, grid, s);
  else launch_plain<T, false, 1, 8>(p, grid, s);
}

// Up to how many rows a caller that can make torch's calls instead should take this launch
// (forge_linear_small_rows). Every block reads all of x, and does the norm's work on it, so the launch
// loses to the library's GEMM as rows, K and blocks grow; what it saves are the launches around the
// product. The lines lie where the whole of it is no slower than torch's calls. us here / torch, bf16,
// graph replays with a W of its own per call (0.7 GB in all, so from HBM), at 1, 4, 8 and 16 rows:
//   plain      4096 x 4096    9.3/15.7   9.4/15.7   9.7/15.6  11.1/15.7
//              8192 x 2048   10.1/14.1   9.3/13.1  10.0/13.2  10.9/13.3
//             12288 x 1024    6.8/9.9    6.7/9.3    7.1/9.3    8.2/9.3
//             10240 x 768     6.3/7.8    6.6/7.9    7.0/8.0    8.1/7.9
//       not    5120 x 3072   11.2/11.5  11.6/11.5  12.2/11.6  14.5/11.5
//       not    5120 x 5120   18.6/14.5  19.8/14.3  22.3/14.9  27.9/15.7
//       not   32768 x 256    10.4/8.1   11.0/8.2   11.8/8.3   13.2/8.4
//   residual   4096 x 14336  25.2/28.7  27.3/28.6  28.4/27.4  34.7/28.0
//              2048 x 8192   13.1/14.7  13.8/14.9  14.8/15.0  18.1/15.3
//       not    4096 x 16384  40.6/32.5  40.9/34.1  42.4/34.6  44.4/33.1
//       not    8192 x 28672  87.6/92.7  96.8/91.6   113/90     132/91
//   norm       6144 x 2048   11.2/20.5  11.8/21.1  12.8/21.8  15.4/21.6
//              6144 x 4096   19.2/25.5  20.2/25.4  22.5/25.6  27.7/25.8
//             12288 x 4096   31.6/38.7  31.7/38.3  35.1/38.7  43.6/38.6
//             13312 x 4096   34.8/38.2  38.3/39.6  43.0/40.5  52.8/39.0
//             32768 x 2048   34.5/44.2  34.9/42.6  37.3/42.8  42.5/43.1
//            151936 x 1024   62.8/72.4  66.6/72.6  69.8/73.5  74.4/75.1
//            163840 x 2048    142/163    155/162    166/168    184/165
//       not    7168 x 5120   24.7/29.6  27.0/28.9  29.2/29.4  37.2/29.8
//       not  128256 x 4096    225/201    237/197    258/197    298/201
//       not  131072 x 512      47/40      49/40      49/41      52/42
//   norm and   9728 x 2560   35.6/53.4  37.5/50.6  40.5/51.9  45.4/49.7
//   SwiGLU    11008 x 4096   46.7/70.9  49.7/73.1  54.6/71.9  62.4/69.0
//             14336 x 4096   59.0/73.2  63.9/75.9  67.3/73.8  78.0/74.1
//             28672 x 4096    106/143    114/142    125/136    138/136
//             13824 x 5120   79.8/90.8  85.3/88.0  92.6/85.7   105/76
//             28672 x 8192    191/262    199/238    222/241    263/242
struct LinRule {
  int n, k, rows;  // up to n outputs of up to k channels: up to `rows` rows
};
// the first line that holds a shape decides; none: 0 rows
constexpr LinRule kLinPlainRule[] = {{4096, 4096, 16}, {8192, 2048, 16}, {16640, 512, 16}, {12288, 895, 12}, {12288, 1024, 16}};
constexpr LinRule kLinResidualRule[] = {{4096, 4096, 16}, {8192, 2048, 16}, {16640, 512, 16}, {12288, 895, 12}, {12288, 1024, 16}, {4096, 16383, 4}};
constexpr LinRule kLinNormRule[] = {{16640, 255, 16}, {1 << 30, 255, 0}, {4096, 4096, 16}, {32768, 2048, 16}, {1 << 30, 767, 0},
                                    {155648, 1024, 16}, {155648, 2048, 8}, {163840, 2048, 4}, {12288, 4096, 8}, {16384, 4096, 4}};
constexpr LinRule kLinGatedRule[] = {{12288, 4096, 16}, {28672, 2048, 16}, {28672, 4096, 8}, {28672, 8192, 4}};

template <int COUNT> static int rule_rows(const LinRule (&rule)[COUNT], int N, int K) {
  for (const LinRule& r : rule)
    if (N <= r.n && K <= r.k) return r.rows;
  return 0;
}

template <typename T>
static int launch_linear(const LinearParams& p, hipStream_t s) {
  if (p.w2) launch_tiles<T, true, 1>(p, s);
  else if (p.N >= kLinWideN) launch_tiles<T, false, 2>(p, s);
  else launch_tiles<T, false, 1>(p, s);
  return check_launch();
}

}  // namespace forge

using namespace forge;

extern "C" int forge_linear_small_rows(int N, int K, int norm, int gated, int residual) {
  if (N <= 0 || K <= 0 || K % 32) return 0;
  return gated ? rule_rows(kLinGatedRule, N, K)
               : norm ? rule_rows(kLinNormRule, N, K)
                      : residual ? rule_rows(kLinResidualRule, N, K) : rule_rows(kLinPlainRule, N, K);
}

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
  if (norm && !gain) return set_error("forge_linear_small: norm needs a gain");
  if (gain && gain_dtype != FORGE_F32 && gain_dtype != dtype)
    return set_error("forge_linear_small: the gain must be fp32 or of x's type");
  if (sx % 8 || sw % 8 || sw < K || (M > 1 && sx < K))
    return set_error("forge_linear_small: row strides must be multiples of 8 elements and hold a row");
  if (M > 1 && sx > (1 << 25)) return set_error("forge_linear_small: rows of x more than 2^25 elements apart");
  if (K > (1 << 25)) return set_error("forge_linear_small: K of more than 2^25");
  if (w2 && (bias || residual)) return set_error("forge_linear_small: SwiGLU takes no bias or residual");
  LinearParams p{x, sx, w, w2, sw, bias, gain, gain_dtype == FORGE_F32, norm, eps, residual, sr, out, so, M, N, K};
  hipStream_t s = (hipStream_t)stream;
  return dtype == FORGE_BF16 ? launch_linear<bf16>(p, s) : launch_linear<f16>(p, s);
}
