// Causal prefill on bf16/fp16 MFMA (gfx950 v_mfma_f32_32x32x16_{bf16,f16}).
//
// A block of 4 waves owns BM = 128 queries of one (b, head); each wave owns 32 of them
// and keeps them for the whole block, together with its output accumulator. Key tiles
// of BN keys (64 for head dim <= 128, 32 for 256) stream through LDS:
//
//   * K and V tiles go from HBM straight into LDS with global_load_lds_dwordx4 (no
//     staging registers, no VALU). Each lane's 16 bytes land at LDS slot `lane`, so the
//     16-byte chunk a lane fetches decides the LDS layout: chunk c of key row r is stored
//     at chunk position c ^ swz(r), an XOR swizzle that keeps the MFMA operand reads
//     below free of bank conflicts. LDS stages (two for every head dim today): the loads
//     of tile j+1 are issued before tile j is computed, one barrier per tile separates
//     the stages, and two blocks share a CU so that its SIMDs interleave two independent
//     waves. At head dim 256 (128 accumulator and 64 Q^T registers of the 256 a wave may use)
//     that needs the load and LDS addresses to come from one register each: two waves per SIMD
//     take 311 us where one took 428 us (4 x 4096 causal, 8 q / 4 KV heads; 642 -> 884 TFLOP/s).
//   * Scores are computed transposed, S^T = K . Q^T: K is the MFMA A operand (128-bit
//     LDS reads), Q^T the B operand held in registers for the whole block. In the 32x32
//     accumulator layout each lane then owns ONE query (column l % 32) and 16 keys of a
//     32-key block (rows 8i + 4(l/32) + j), so the online softmax of a query needs a
//     single cross-lane exchange per tile (lane l <-> l ^ 32) for the running max, and
//     none for the running sum (the two halves are added once at the end).
//   * P^T is fed to the second MFMA (O^T = V^T . P^T) straight from the score registers:
//     MFMA k index 8hi + 4i' + j stands for key 16*half + 8i' + 4hi + j, exactly the keys
//     the lane already holds. The matching V^T operand is read from the row-major V tile
//     with ds_read_b64_tr_b16 (gfx950's transposing LDS read: within each 16-lane group,
//     lane i receives element i % 4 of the 4-element rows addressed by lanes 4k + i / 4,
//     k = 0..3), two reads of 4 keys per MFMA.
//   * The running max only moves when a score exceeds it by 2^8 (log2 units), so the
//     rescale of the accumulator is rare; weights stay <= 2^8, safe in bf16/fp16.
//
// Q gets the per-head RMSNorm and RoPE in its load (fp32 math, one rounding), like
// fused_ops._head_kernel (fused_ops.py:53-85); K and V come from the cache, where
// forge_kv_append wrote them already normalised.
#include <limits.h>

#include "common.h"
#include "forge_internal.h"

namespace forge {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

template <typename T> struct Mfma;
template <> struct Mfma<bf16> {
  typedef bf16x8 vec;
  static __device__ __forceinline__ floatx16 run(vec a, vec b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mfma<f16> {
  typedef f16x8 vec;
  static __device__ __forceinline__ floatx16 run(vec a, vec b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

struct PrefillParams {
  const void* q;
  int64_t sqb, sqh, sqt;
  const float* qw;
  float eps;
  int flags;
  const float* cos;
  const float* sin;
  int64_t cst;
  const void* k;
  const void* v;
  int64_t skb, skh, sks;
  int64_t offset;
  int B, T, H, K, G;
  int nqt;       // query tiles per (b, head)
  int xcd_map;   // 1: blocks of one (b, kv head) pair run on one XCD (B*K % 8 == 0)
  int window;
  float scale_log2;
  void* out;
  int64_t sob, sot, soh;
  // Document masking (forge_attn_prefill_docs): query t of row b also sees no key before
  // position doc_lo[b * sdb + t], the first of its document (non-decreasing in t); or null.
  const int32_t* doc_lo;
  int64_t sdb;
  // Key split (launches whose query tiles leave CUs idle): a query tile's key tiles go to
  // ceil(tiles / split_tiles) blocks, at most nsplit of them, each writing an fp32 partial
  // (m, l, o) that prefill_combine_kernel merges. nsplit 1: no split.
  int nsplit, split_tiles;
  int heads_per_block;  // prefill_wide_kernel only
  float2* ws_ml;  // [nsplit][B*H*T]
  float* ws_o;    // [nsplit][B*H*T][D]
};

// First document position of a row's query tile (its first query's: starts do not decrease).
__device__ __forceinline__ int first_doc(const PrefillParams& p, int b, int qt, int BM) {
  return p.doc_lo ? p.doc_lo[b * p.sdb + (int64_t)qt * BM] : 0;
}

// Key tiles [begin, end] of query tile qt (BM queries, BN keys per tile): from its first
// query's window or document start to its last query.
__host__ __device__ __forceinline__ void tile_span(int64_t offset, int T, int window, int doc0, int qt, int BM,
                                                   int BN, int& begin, int& end) {
  const int64_t i0 = (int64_t)qt * BM;
  const int64_t i1 = i0 + BM < T ? i0 + BM - 1 : T - 1;
  int64_t kmin = window > 0 ? offset + i0 - window + 1 : 0;
  if (kmin < doc0) kmin = doc0;
  begin = (int)(kmin / BN);
  end = (int)((offset + i1) / BN);
}

// Blocks that share a query tile of n key tiles.
__device__ __forceinline__ int split_count(const PrefillParams& p, int n) {
  const int c = (n + p.split_tiles - 1) / p.split_tiles;
  return c < p.nsplit ? c : p.nsplit;
}

// This block's share of its query tile's key tiles: part `part` of split_count. False (the
// same for the whole block) where the query tile has fewer parts.
__device__ __forceinline__ bool take_part(const PrefillParams& p, int part, int& begin, int& end, int& parts) {
  const int n = end - begin + 1;
  parts = split_count(p, n);
  if (part >= parts) return false;
  end = begin + (int)((int64_t)(part + 1) * n / parts) - 1;
  begin += (int)((int64_t)part * n / parts);
  return true;
}

constexpr float kLazyLog2 = 8.0f;

// Block shape per head dim: WAVES waves of 32 queries each, STAGES LDS stages of one K
// and one V tile of BN keys (loads run STAGES - 1 tiles ahead of the compute).
template <int D> struct Tile {
  static constexpr int WAVES = 4;
  static constexpr int STAGES = 2;
  static constexpr int BM = 32 * WAVES;                // queries per block
  static constexpr int BN = D >= 256 ? 32 : 64;        // keys per tile
  static constexpr int NCH = D / 8;                    // 16-byte chunks per key row
  static constexpr int ROWB = 2 * D;                   // bytes per key row
  static constexpr int TILEB = BN * ROWB;              // bytes of one K (or V) tile
  static constexpr int LOADS = TILEB / (WAVES * 1024);   // 16-byte loads per lane per tile
  static constexpr int LDS_BYTES = STAGES * 2 * TILEB;
  static_assert(LOADS * WAVES * 1024 == TILEB, "tile must split into whole wave loads");
};

// XOR swizzles of the 16-byte chunk index by key row (see the reads below).
template <int D> __device__ __forceinline__ int swz_k(int row) {
  return row & ((D / 8 >= 16 ? 16 : D / 8) - 1);
}
template <int D> __device__ __forceinline__ int swz_v(int row) {
  return D / 8 >= 16 ? (row & 3) << 2 : ((row >> 1) & 1) << 2;
}

// Wait until at most N vector-memory loads of this wave are outstanding (loads retire in
// issue order, so everything issued before the last N has landed).
template <int N> __device__ __forceinline__ void wait_vm() {
  static_assert(N == 0 || N == 2 || N == 4 || N == 8, "add the count");
  if constexpr (N == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  else if constexpr (N == 2) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
  else if constexpr (N == 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
  else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
}

// Q rows of one wave as MFMA B operands: load, fused RMSNorm + RoPE (fp32, one rounding).
// Lane (n, hi) holds channels 16s + 8hi + e of query i_q; gains and RoPE rows come in
// 16-byte loads.
template <typename T, int D>
__device__ __forceinline__ void load_q(const PrefillParams& p, int b, int h, int i_q, bool valid_q,
                                       int hi, typename Mfma<T>::vec (&qreg)[D / 16]) {
  constexpr int KSTEPS = D / 16;
  float qf[KSTEPS][8];
  const T* src = static_cast<const T*>(p.q) + b * p.sqb + h * p.sqh + (int64_t)i_q * p.sqt;
#pragma unroll
  for (int s = 0; s < KSTEPS; ++s) {
    if (valid_q) {
      unpack16<T>(load16(src + 16 * s + 8 * hi), qf[s]);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) qf[s][e] = 0.0f;
    }
  }
  if (p.flags & FORGE_NORM_QK) {
    float ss = 0.0f;
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += qf[s][e] * qf[s][e];
    ss += __shfl_xor(ss, 32, kWave);
    const float rs = rsqrtf(ss / (float)D + p.eps);
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) qf[s][e] *= rs;
    if (p.qw) {
      float w[KSTEPS][8];
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s) load_f32x8(p.qw + 16 * s + 8 * hi, w[s]);
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) qf[s][e] *= w[s][e];
    }
  }
  if ((p.flags & FORGE_ROPE) && valid_q) {
    const float* cr = p.cos + (int64_t)i_q * p.cst;
    const float* sr = p.sin + (int64_t)i_q * p.cst;
#pragma unroll
    for (int s = 0; s < KSTEPS / 2; ++s) {
      const int x = 16 * s + 8 * hi;  // first-half channels x..x+7; partners x + D/2
      float c1[8], s1[8], c2[8], s2[8];
      load_f32x8(cr + x, c1);
      load_f32x8(sr + x, s1);
      load_f32x8(cr + x + D / 2, c2);
      load_f32x8(sr + x + D / 2, s2);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float a = qf[s][e], z = qf[s + KSTEPS / 2][e];
        qf[s][e] = a * c1[e] - z * s1[e];
        qf[s + KSTEPS / 2][e] = z * c2[e] + a * s2[e];
      }
    }
  }
#pragma unroll
  for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e) qreg[s][e] = from_f32<T>(qf[s][e]);
}

// SPLIT: the key-split launch (PrefillParams::nsplit > 1); otherwise one block per query tile.
template <typename T, int D, bool SPLIT>
__global__ __launch_bounds__(Tile<D>::WAVES * 64) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_kernel(PrefillParams p) {
  using V8 = typename Mfma<T>::vec;
  using TL = Tile<D>;
  constexpr int BN = TL::BN;
  constexpr int kBM = TL::BM;
  constexpr int KB = BN / 32;       // 32-key blocks per tile
  constexpr int KSTEPS = D / 16;    // MFMA k-steps over the head dim (scores)
  constexpr int DB = D / 32;        // 32-channel blocks of the output
  constexpr int HALVES = BN / 16;   // 16-key MFMA steps of P.V

  extern __shared__ __attribute__((aligned(1024))) char smem[];  // [stage][K|V][TILEB]

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lane = tid % kWave;
  const int n = lane & 31;
  const int hi = lane >> 5;

  // ---- block -> (query tile, head, batch). Heavy (late) causal tiles first. With
  // xcd_map, block i runs on XCD i % 8 and all blocks of one (b, kv head) pair share an
  // XCD, so the K/V they all read stays in that XCD's L2. A split launch does the same with
  // (pair, part) in place of the pair: the blocks of one part read the same keys.
  int qt, b, kvh, gq, part = 0;
  {
    const int bid = blockIdx.x;
    const int NS = SPLIT ? p.nsplit : 1;
    const int P = p.B * p.K * NS;
    if (p.xcd_map) {
      const int x = bid & 7, local = bid >> 3;
      const int per = (P >> 3) * p.G;  // (pair, head) combinations per XCD
      const int rank = local / per, rest = local % per;
      qt = p.nqt - 1 - rank;
      int pair = (rest / p.G) * 8 + x;
      gq = rest % p.G;
      if (SPLIT) {
        part = pair % NS;
        pair /= NS;
      }
      b = pair / p.K;
      kvh = pair % p.K;
    } else {
      const int HB = p.H * p.B * NS;
      qt = p.nqt - 1 - bid / HB;
      const int hb = bid % HB;
      int pair = hb % P;
      gq = hb / P;
      if (SPLIT) {
        part = pair % NS;
        pair /= NS;
      }
      b = pair / p.K;
      kvh = pair % p.K;
    }
  }
  const int h = kvh * p.G + gq;

  const int i_q = qt * kBM + wave * 32 + n;  // this lane's query (index into T)
  const bool valid_q = i_q < p.T;
  const int64_t qpos = p.offset + i_q;
  const int64_t S = p.offset + p.T;

  // ---- key tiles of the block, and the first stage's loads (issued before the Q math)
  const int32_t* dl = p.doc_lo ? p.doc_lo + b * p.sdb : nullptr;
  int kt_begin, kt_end, parts = 1;
  tile_span(p.offset, p.T, p.window, __builtin_amdgcn_readfirstlane(first_doc(p, b, qt, kBM)), qt, kBM, BN,
            kt_begin, kt_end);
  if (SPLIT && !take_part(p, part, kt_begin, kt_end, parts)) return;

  const T* kg = static_cast<const T*>(p.k) + b * p.skb + kvh * p.skh;
  const T* vg = static_cast<const T*>(p.v) + b * p.skb + kvh * p.skh;

  const char* kgb = reinterpret_cast<const char*>(kg);
  const char* vgb = reinterpret_cast<const char*>(vg);
  // Load i of this wave fills LDS slots (wave*LOADS + i)*64 + lane with RL = 64 / NCH key rows, r0 +
  // lane / NCH, in swizzled chunk order. Up to head dim 128 a lane keeps its source byte offset within
  // a tile for every load. At 256, where registers are short, r0 is wave-uniform (its address stays in
  // scalar registers) and the swizzles split over r0 and the lane's part, so a lane's offsets take one
  // xor each from registers shared by all the loads; at 128 those xors in every tile took 184.7 us where
  // the kept offsets take 180.3 (1,017 queries at 6,085, 32 q / 8 KV heads).
  constexpr bool KEEP = D < 256;
  constexpr int RL = kWave / TL::NCH;
  const int ld_row = lane / TL::NCH;
  const int ld_k = ((lane % TL::NCH) ^ swz_k<D>(ld_row)) << 4, ld_v = ((lane % TL::NCH) ^ swz_v<D>(ld_row)) << 4;
  const int ld_off = (int)(ld_row * p.sks * 2);
  int kept_k[KEEP ? TL::LOADS : 1], kept_v[KEEP ? TL::LOADS : 1];
  if constexpr (KEEP) {
#pragma unroll
    for (int i = 0; i < TL::LOADS; ++i) {
      const int row = RL * (wave * TL::LOADS + i) + ld_row, pch = lane % TL::NCH;
      kept_k[i] = (int)(row * p.sks * 2) + ((pch ^ swz_k<D>(row)) << 4);
      kept_v[i] = (int)(row * p.sks * 2) + ((pch ^ swz_v<D>(row)) << 4);
    }
  }
  // The loads are issued from inline asm (lds_dma16), so the compiler does not hold the
  // LDS reads of the current stage back until the next stage's loads have landed; the
  // loop waits for them itself (wait_vm before the barrier).
  auto issue = [&](int kt, int stage) {
    const int64_t key0 = (int64_t)kt * BN;
    const unsigned kdst = lds_offset(smem + (2 * stage) * TL::TILEB + wave * TL::LOADS * 1024);
    const unsigned vdst = kdst + TL::TILEB;
    int lk = ld_k, lv = ld_v, lo = ld_off;
    if constexpr (D >= 256) asm volatile("" : "+v"(lk), "+v"(lv));  // (registers short: not kept over the loop)
    if (key0 + BN <= S) {
      const char* kt_base = kgb + key0 * p.sks * 2;
      const char* vt_base = vgb + key0 * p.sks * 2;
#pragma unroll
      for (int i = 0; i < TL::LOADS; ++i) {
        if constexpr (KEEP) {
          lds_dma16(kt_base, (unsigned)kept_k[i], kdst + i * 1024);
          lds_dma16(vt_base, (unsigned)kept_v[i], vdst + i * 1024);
          continue;
        }
        const int r0 = RL * (wave * TL::LOADS + i);
        const int64_t off = r0 * p.sks * 2;
        lds_dma16(kt_base + off, (unsigned)(lo + (lk ^ (swz_k<D>(r0) << 4))), kdst + i * 1024);
        lds_dma16(vt_base + off, (unsigned)(lo + (lv ^ (swz_v<D>(r0) << 4))), vdst + i * 1024);
      }
    } else {
      // last, partial tile: rows past the end are masked; they read row S - 1 instead (at head dim 256
      // the wave's row is clamped first, so a lane's offset, which is unsigned, stays at least 0)
#pragma unroll
      for (int i = 0; i < TL::LOADS; ++i) {
        if constexpr (KEEP) {
          const int row = RL * (wave * TL::LOADS + i) + ld_row, pch = lane % TL::NCH;
          const int64_t key = key0 + row < S ? key0 + row : S - 1;
          const unsigned rb = (unsigned)((key - key0) * p.sks * 2);
          lds_dma16(kgb + key0 * p.sks * 2, rb + ((pch ^ swz_k<D>(row)) << 4), kdst + i * 1024);
          lds_dma16(vgb + key0 * p.sks * 2, rb + ((pch ^ swz_v<D>(row)) << 4), vdst + i * 1024);
          continue;
        }
        const int r0 = RL * (wave * TL::LOADS + i);
        const int64_t key = key0 + r0 < S ? key0 + r0 : S - 1;
        const int64_t off = key * p.sks * 2;
        const int o = ld_row <= S - 1 - key ? lo : (int)((S - 1 - key) * p.sks * 2);
        lds_dma16(kgb + off, (unsigned)(o + (lk ^ (swz_k<D>(r0) << 4))), kdst + i * 1024);
        lds_dma16(vgb + off, (unsigned)(o + (lv ^ (swz_v<D>(r0) << 4))), vdst + i * 1024);
      }
    }
  };
  issue(kt_begin, 0);
#pragma unroll
  for (int j = 1; j < TL::STAGES - 1; ++j)
    if (kt_begin + j <= kt_end) issue(kt_begin + j, j);

  // ---- Q: load, fused RMSNorm + RoPE, one rounding, kept as MFMA B operands.
  V8 qreg[KSTEPS];
  load_q<T, D>(p, b, h, i_q, valid_q, hi, qreg);

  // this wave's query span (tile skipping and the mask-free fast path); positions fit
  // in 32 bits (host check)
  const int w_first = qt * kBM + wave * 32;
  const int w_last = w_first + 31 < p.T - 1 ? w_first + 31 : p.T - 1;
  const bool wave_any = w_first < p.T;
  const int off = (int)p.offset;
  const int wq_lo = off + w_first, wq_hi = off + w_last;
  const int S32 = (int)S;
  const int qpos32 = (int)qpos;
  // document starts: this lane's query's, and the first (smallest) and last (largest) of the
  // wave's queries (loads of rows past T read row T - 1; those lanes are masked anyway)
  int d_lane = 0, d_wfirst = 0, d_wlast = 0;
  if (dl) {
    d_lane = dl[i_q < p.T ? i_q : p.T - 1];
    d_wfirst = __builtin_amdgcn_readfirstlane(d_lane);
    d_wlast = __builtin_amdgcn_readlane(d_lane, w_last - w_first > 0 ? w_last - w_first : 0);
  }

  // LDS read offsets of a lane within a stage's K and V tiles. K operand: row 32kb + n, chunk
  // 2st + hi, swizzled by the row; V^T operand (tr reads): source lane role g = lane/16,
  // kq = (lane/4)%4, qq = lane%4 addresses key row 16*half + 8i' + 4(g/2) + kq, channel
  // 32db + 16(g%2) + 4qq (rows that differ by multiples of 8 share a swizzle). The swizzles only
  // touch the low four chunk bits, so k-step st lies at k_rd ^ 32 (st % 8) plus 256 bytes per 8
  // steps and channel block d at v_rd ^ 64 (d % 4) plus 256 bytes per 4: one xor from one register.
  const int g = lane >> 4, kq = (lane >> 2) & 3, qq = lane & 3;
  const int v_row = 4 * (g >> 1) + kq;
  const unsigned k_rd = n * TL::ROWB + ((hi ^ swz_k<D>(n)) << 4);
  const unsigned v_rd = v_row * TL::ROWB + (((2 * (g & 1) + (qq >> 1)) ^ swz_v<D>(v_row)) << 4) + 8 * (qq & 1);
  const unsigned lds0 = lds_offset(smem);

  floatx16 oacc[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int x = 0; x < 16; ++x) oacc[d][x] = 0.0f;
  float m_run = kNegInf, l_run = 0.0f;
  const float c = p.scale_log2;

  for (int kt = kt_begin; kt <= kt_end; ++kt) {
    const int idx = kt - kt_begin;
    const int stage = idx % TL::STAGES;
    // Tile kt has landed once at most the loads of the tiles issued after it remain.
    if (TL::STAGES == 3 && kt + 1 <= kt_end) wait_vm<2 * TL::LOADS>();
    else wait_vm<0>();
    __syncthreads();  // tile kt is in LDS for every wave; the stage of tile kt-1 is free
    if (kt + TL::STAGES - 1 <= kt_end) issue(kt + TL::STAGES - 1, (idx + TL::STAGES - 1) % TL::STAGES);

    const int key0 = kt * BN;
    const bool wave_needs = wave_any && key0 <= wq_hi &&
                            (p.window <= 0 || key0 + BN - 1 > wq_lo - p.window) &&
                            key0 + BN - 1 >= d_wfirst;
    if (!wave_needs) continue;
    const bool full = key0 + BN - 1 <= wq_lo && key0 + BN - 1 < S32 &&
                      (p.window <= 0 || wq_hi - key0 < p.window) && w_last - w_first == 31 &&
                      key0 >= d_wlast;

    const unsigned kl = lds0 + (2 * stage) * TL::TILEB + k_rd;
    const unsigned vl = lds0 + (2 * stage + 1) * TL::TILEB + v_rd;

    // ---- S^T = K . Q^T: KB independent accumulation chains. The K operands of step
    // st + 2 are read before the MFMAs of step st are issued (three register sets), so
    // the LDS latency hides under two steps of MFMAs; the scheduling groups pin that
    // order (left alone, the compiler reuses one register set and waits for every read).
    floatx16 sacc[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int x = 0; x < 16; ++x) sacc[kb][x] = 0.0f;
    {
      auto kread = [&](int kb, int st) {
        return *(__attribute__((address_space(3))) const V8*)((kl ^ (32 * (st & 7))) + 256 * (st >> 3) +
                                                              kb * 32 * TL::ROWB);
      };
      V8 a0[KB], a1[KB], a2[KB];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) a0[kb] = kread(kb, 0);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) a1[kb] = kread(kb, 1);
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * KB, 0);
#pragma unroll
      for (int st = 0; st < KSTEPS; ++st) {
        if (st + 2 < KSTEPS) {
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) a2[kb] = kread(kb, st + 2);
          __builtin_amdgcn_sched_group_barrier(0x100, KB, 0);
        }
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) sacc[kb] = Mfma<T>::run(a0[kb], qreg[st], sacc[kb]);
        __builtin_amdgcn_sched_group_barrier(0x008, KB, 0);
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          a0[kb] = a1[kb];
          a1[kb] = a2[kb];
        }
      }
    }

    // ---- mask (boundary tiles only): element (kb, x) of this lane is key
    // key0 + 4hi + ce with ce = 32kb + 8(x/4) + x%4; it is visible iff lo <= ce <= hi.
    if (!full) {
      const int base = key0 + 4 * hi;
      const int top = (qpos32 < S32 - 1 ? qpos32 : S32 - 1) - base;
      const int lim_hi = valid_q ? top : -1;
      int lim_lo = p.window > 0 ? qpos32 - p.window + 1 - base : -(1 << 30);
      if (dl && d_lane - base > lim_lo) lim_lo = d_lane - base;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int x = 0; x < 16; ++x) {
          const int ce = 32 * kb + 8 * (x >> 2) + (x & 3);
          sacc[kb][x] = (ce <= lim_hi && ce >= lim_lo) ? sacc[kb][x] : kNegInf;
        }
    }

    // ---- online softmax (base 2, scale folded into the exponent)
    float mxp[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      mxp[i] = sacc[0][4 * i];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int j = (kb == 0 ? 1 : 0); j < 4; ++j) mxp[i] = fmaxf(mxp[i], sacc[kb][4 * i + j]);
    }
    float mx = fmaxf(fmaxf(mxp[0], mxp[1]), fmaxf(mxp[2], mxp[3]));
    mx = max_xor32(mx);
    const float mxc = mx * c;
    if (mxc > m_run + kLazyLog2) {
      const float alpha = m_run == kNegInf ? 0.0f : __builtin_amdgcn_exp2f(m_run - mxc);
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int x = 0; x < 16; ++x) oacc[d][x] *= alpha;
      m_run = mxc;
    }
    const float neg_m = m_run == kNegInf ? 0.0f : -m_run;  // all -inf so far: weights 0
    float rs[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        const float pv = __builtin_amdgcn_exp2f(fmaf(sacc[kb][x], c, neg_m));
        sacc[kb][x] = pv;
        rs[x & 3] += pv;
      }
    l_run += (rs[0] + rs[1]) + (rs[2] + rs[3]);

    // ---- O^T += V^T . P^T
#pragma unroll
    for (int hf = 0; hf < HALVES; ++hf) {
      const int kb = hf >> 1, half = hf & 1;
      V8 pb;
#pragma unroll
      for (int e = 0; e < 8; ++e) pb[e] = from_f32<T>(sacc[kb][8 * half + e]);
#pragma unroll
      for (int d = 0; d < DB; ++d) {
        const unsigned va = (vl ^ (64 * (d & 3))) + 256 * (d >> 2) + 16 * hf * TL::ROWB;
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)va);
        const i16x4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) i16x4*)(va + 8 * TL::ROWB));
        typedef short i16x8 __attribute__((ext_vector_type(8)));
        const i16x8 av = __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7);
        oacc[d] = Mfma<T>::run(__builtin_bit_cast(V8, av), pb, oacc[d]);
      }
    }
  }

  l_run += __shfl_xor(l_run, 32, kWave);
  if (!valid_q) return;
  if (SPLIT && parts > 1) {  // the row's partial of this part
    const int64_t rows = (int64_t)p.B * p.H * p.T;
    const int64_t slot = part * rows + ((int64_t)b * p.H + h) * p.T + i_q;
    float* po = p.ws_o + slot * D + 4 * hi;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<float4*>(po + d * 32 + 8 * i) =
            make_float4(oacc[d][4 * i], oacc[d][4 * i + 1], oacc[d][4 * i + 2], oacc[d][4 * i + 3]);
    if (hi == 0) p.ws_ml[slot] = make_float2(m_run, l_run);
    return;
  }
  const float inv_l = 1.0f / l_run;
  T* dst = static_cast<T*>(p.out) + b * p.sob + (int64_t)i_q * p.sot + h * p.soh;
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      T vals[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) vals[j] = from_f32<T>(oacc[d][4 * i + j] * inv_l);
      *reinterpret_cast<uint2*>(dst + d * 32 + 8 * i + 4 * hi) = *reinterpret_cast<uint2*>(vals);
    }
}

// Merges the parts of a split launch: D / 4 lanes per (b, h, t) row, four channels each, the
// parts in order. Rows of query tiles that were not split were written by their block.
template <typename T, int D>
__global__ __launch_bounds__(256) void prefill_combine_kernel(PrefillParams p, int BM, int BN) {
  constexpr int LPR = D / 4;
  const int64_t rows = (int64_t)p.B * p.H * p.T;
  const int64_t row = (int64_t)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
  const int x = 4 * (threadIdx.x % LPR);
  if (row >= rows) return;
  const int i_q = (int)(row % p.T);
  const int64_t bh = row / p.T;
  const int h = (int)(bh % p.H), b = (int)(bh / p.H);
  int begin, end;
  tile_span(p.offset, p.T, p.window, 0, i_q / BM, BM, BN, begin, end);
  const int parts = split_count(p, end - begin + 1);
  if (parts < 2) return;
  float M = kNegInf;
  for (int i = 0; i < parts; ++i) M = fmaxf(M, p.ws_ml[i * rows + row].x);
  float L = 0.0f;
  float4 O = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  constexpr int U = 4;  // parts whose loads go out together
  for (int i0 = 0; i0 < parts; i0 += U) {
    float2 ml[U];
    float4 o[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u < parts ? i0 + u : parts - 1;
      ml[u] = p.ws_ml[i * rows + row];
      o[u] = *reinterpret_cast<const float4*>(p.ws_o + (i * rows + row) * D + x);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float a = i0 + u < parts ? rescale(ml[u].x, M) : 0.0f;
      L += a * ml[u].y;
      O.x += a * o[u].x;
      O.y += a * o[u].y;
      O.z += a * o[u].z;
      O.w += a * o[u].w;
    }
  }
  const float inv_l = 1.0f / L;
  T* dst = static_cast<T*>(p.out) + b * p.sob + (int64_t)i_q * p.sot + h * p.soh + x;
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<float4*>(dst) = make_float4(O.x / L, O.y / L, O.z / L, O.w / L);
  } else {
    T v[4] = {from_f32<T>(O.x * inv_l), from_f32<T>(O.y * inv_l), from_f32<T>(O.z * inv_l), from_f32<T>(O.w * inv_l)};
    *reinterpret_cast<uint2*>(dst) = *reinterpret_cast<uint2*>(v);
  }
}

template <typename T, int D>
static int launch_prefill_combine(const PrefillParams& p, int BM, int BN, hipStream_t s) {
  constexpr int RPB = 256 / (D / 4);
  const int64_t rows = (int64_t)p.B * p.H * p.T;
  const int64_t blocks = (rows + RPB - 1) / RPB;
  if (blocks > 0x7fffffff) return set_error("grid too large");
  hipLaunchKernelGGL((prefill_combine_kernel<T, D>), dim3((unsigned)blocks), dim3(256), 0, s, p, BM, BN);
  return check_launch();
}

template <typename T, int D, bool SPLIT>
static int launch_prefill_s(PrefillParams p, hipStream_t s) {
  using TL = Tile<D>;
  constexpr int kThreeLds = 48 * 1024;  // three blocks of it fit a CU's 160 KB, four do not
  static bool attr_set = false;  // raise the dynamic LDS limit once per kernel
  if (!attr_set) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_kernel<T, D, SPLIT>),
                            hipFuncAttributeMaxDynamicSharedMemorySize,
                            TL::LDS_BYTES > kThreeLds ? TL::LDS_BYTES : kThreeLds) != hipSuccess)
      return set_error("forge_attn_prefill: cannot reserve the LDS the kernel needs");
    attr_set = true;
  }
  p.nqt = (p.T + TL::BM - 1) / TL::BM;
  p.xcd_map = ((int64_t)p.B * p.K * p.nsplit) % 8 == 0 ? 1 : 0;
  const int64_t blocks = (int64_t)p.nqt * p.H * p.B * p.nsplit;
  if (blocks > 0x7fffffff) return set_error("grid too large");
  int lds = TL::LDS_BYTES;
  if constexpr (D == 64 && !SPLIT) {
    // A CU holds four blocks. A launch of three to four per CU would then start them all at once, on
    // CUs that cannot even out their blocks' lengths afterwards; with three per CU the last ones go to
    // the CUs that finish first. That pays with documents, whose blocks differ most, and otherwise
    // while few CUs get a fourth block (three against four, us; 16 q / 16 KV heads, 12 / 4 the 792s):
    // documents of 1,250 tokens, 896 blocks 47.5 / 48.8, 1,024 blocks 48.0 / 50.1, of 300 tokens 27.7 /
    // 28.7 and 32.7 / 32.7; whole prompts, 792 blocks 39.6 / 40.5, 896 49.6 / 50.9, 880 39.9 / 37.4, 1,024
    // 57.4 / 54.0; window 512, 792 blocks 29.1 / 29.4, 900 34.7 / 32.7.
    const int64_t cus = device_cus();
    if (blocks > 3 * cus && blocks * 4 <= (p.doc_lo ? 16 : 13) * cus) lds = kThreeLds;
  }
  hipLaunchKernelGGL((prefill_kernel<T, D, SPLIT>), dim3((unsigned)blocks), dim3(TL::WAVES * 64), lds, s, p);
  return check_launch();
}

template <typename T, int D>
static int launch_prefill_d(const PrefillParams& p, hipStream_t s) {
  if (p.nsplit < 2) return launch_prefill_s<T, D, false>(p, s);
  const int st = launch_prefill_s<T, D, true>(p, s);
  return st ? st : launch_prefill_combine<T, D>(p, Tile<D>::BM, Tile<D>::BN, s);
}

// ---------------------------------------------------------------- head dim 512
// Head dim 512 (Gemma 4's full-attention layers: 1 KV head of 512, reference
// kv_cache.py:12-13). A wave's 32 queries would need 128 registers of Q^T and 256 of output
// accumulators, so here the head dim is split over SPLIT waves, each with its D / SPLIT channels
// of a head's 32 queries; a block of NW waves holds NW / SPLIT heads of one KV head, so each K/V
// tile is loaded once for all of them. Per key tile (32 keys, two LDS stages of 32 KB K + 32 KB
// V):
//   * each wave computes the partial scores of its channels, S_w^T = K[:, slice] . Q^T[slice],
//     and stores them in LDS; after a barrier every wave adds its head's partials in slice
//     order, so the waves of a head hold identical scores;
//   * every wave runs the same online softmax (the running max and sum are identical in the
//     waves of a head) and accumulates its own output channels, O^T += V^T[slice] . P^T.
// The q RMSNorm sums the squares of the slices through LDS in the same order; RoPE pairs
// channel c with c ^ 256, so each lane also loads its channels' partners.
// Eight waves (four heads, two waves per SIMD) against four (two heads, one per SIMD): half the
// tile loads per FLOP, and one wave's softmax runs beside the other's MFMAs: 16 q / 1 KV head,
// 4,096 causal: 432 us against 606 us (636 against 454 TFLOP/s). It needs the whole 256-register
// budget of two waves per SIMD, hence the load and LDS addresses made from one register each and
// the K operands held two steps ahead only: every spill reload in the tile loop would wait for
// the tile loads in flight.
template <int NW> struct WideTile {
  static constexpr int D = 512;
  static constexpr int WAVES = NW;
  static constexpr int BM = 32;                          // queries per block
  static constexpr int BN = 32;                          // keys per tile
  static constexpr int NCH = D / 8;
  static constexpr int ROWB = 2 * D;
  static constexpr int TILEB = BN * ROWB;                // 32 KB
  static constexpr int LOADS = TILEB / (WAVES * 1024);   // 8 with four waves, 4 with eight
  static constexpr int STAGES = 2;
  static constexpr int PART_BYTES = WAVES * 64 * 16 * 4; // the waves' partial scores
  static constexpr int LDS_BYTES = STAGES * 2 * TILEB + PART_BYTES;
};

template <typename T, int NW, int SPLIT, bool KSPLIT>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW / 4)))
void prefill_wide_kernel(PrefillParams p) {
  using V8 = typename Mfma<T>::vec;
  using TL = WideTile<NW>;
  constexpr int D = TL::D;
  constexpr int BN = TL::BN;
  // SPLIT waves share a head, each with D / SPLIT channels; the block takes WAVES / SPLIT heads
  // of one KV head, so each K/V tile is loaded once for all of them
  static_assert(SPLIT == 4 || SPLIT == 2, "quarters of one head, or halves of two (four waves) or four (eight)");
  constexpr int HPB = TL::WAVES / SPLIT;     // heads per block
  constexpr int CW = D / SPLIT;              // channels per wave
  constexpr int CCH = CW / 8;                // 16-byte chunks per wave slice
  constexpr int KSTEPS = CW / 16;            // 16-channel MFMA k-steps over a wave's channels
  constexpr int DB = CW / 32;                // 32-channel output blocks per wave
  constexpr int HALVES = BN / 16;

  extern __shared__ __attribute__((aligned(1024))) char smem[];
  float* part = reinterpret_cast<float*>(smem + TL::STAGES * 2 * TL::TILEB);   // [wave][lane][16]
  float* sh_ss = part;  // the q slices' sums of squares [wave][32], before any partial score

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lane = tid % kWave;
  const int n = lane & 31;
  const int hi = lane >> 5;

  // block -> (query tile, head group, batch), heavy (late) causal tiles first; wave w takes
  // slice w % SPLIT of head HPB * hg + w / SPLIT
  // (KSPLIT: the parts of a key-split launch between the query tile and the head group)
  const int NS = KSPLIT ? p.nsplit : 1;
  const int HB = (p.H / HPB) * p.B;
  const int qt = p.nqt - 1 - (int)blockIdx.x / (HB * NS);
  const int kpart = (int)blockIdx.x % (HB * NS) / HB;
  const int hb = (int)blockIdx.x % HB;
  const int b = hb % p.B;
  const int slice = wave % SPLIT;
  const int h = (hb / p.B) * HPB + wave / SPLIT;
  const int kvh = h / p.G;
  const int wbase = wave - slice;  // the head's first wave

  const int i_q = qt * TL::BM + n;
  const bool valid_q = i_q < p.T;
  const int64_t S = p.offset + p.T;
  const int q_last_idx = qt * TL::BM + TL::BM - 1 < p.T - 1 ? qt * TL::BM + TL::BM - 1 : p.T - 1;
  const int32_t* dl = p.doc_lo ? p.doc_lo + b * p.sdb : nullptr;
  int d_lane = 0, d_last = 0;
  if (dl) {
    d_lane = dl[i_q < p.T ? i_q : p.T - 1];
    d_last = __builtin_amdgcn_readlane(d_lane, q_last_idx - qt * TL::BM);
  }
  int kt_begin, kt_end, parts = 1;
  tile_span(p.offset, p.T, p.window, __builtin_amdgcn_readfirstlane(first_doc(p, b, qt, TL::BM)), qt, TL::BM, BN,
            kt_begin, kt_end);
  if (KSPLIT && !take_part(p, kpart, kt_begin, kt_end, parts)) return;

  const char* kgb = reinterpret_cast<const char*>(static_cast<const T*>(p.k) + b * p.skb + kvh * p.skh);
  const char* vgb = reinterpret_cast<const char*>(static_cast<const T*>(p.v) + b * p.skb + kvh * p.skh);
  // A wave's 1 KB load is one key row (64 lanes x 16 bytes), so the row is wave-uniform: with eight
  // waves its address stays in scalar registers and a lane's offset is its swizzled chunk. Four waves
  // have the registers for offsets from the tile's base, which are cheaper than a 64-bit product per
  // row (435 queries, 16 q heads, two rows: 52.8 -> 52.0 us).
  static_assert(TL::NCH == kWave, "one key row per wave load");
  auto issue = [&](int kt, int stage) {
    const unsigned kdst = lds_offset(smem + (2 * stage) * TL::TILEB + wave * TL::LOADS * 1024);
    const int64_t key0 = (int64_t)kt * BN;
    int ln = lane;
    if constexpr (NW == 8) asm volatile("" : "+v"(ln));  // the offsets are made here, one xor each, and not kept in registers
#pragma unroll
    for (int i = 0; i < TL::LOADS; ++i) {
      const int row = wave * TL::LOADS + i;
      const int64_t key = key0 + row < S ? key0 + row : S - 1;   // rows past the end are masked
      if constexpr (NW == 4) {
        const unsigned rb = (unsigned)((key - key0) * p.sks * 2);
        lds_dma16(kgb + key0 * p.sks * 2, rb + ((ln ^ swz_k<D>(row)) << 4), kdst + i * 1024);
        lds_dma16(vgb + key0 * p.sks * 2, rb + ((ln ^ swz_v<D>(row)) << 4), kdst + TL::TILEB + i * 1024);
        continue;
      }
      const int64_t off = key * p.sks * 2;
      lds_dma16(kgb + off, (unsigned)((ln ^ swz_k<D>(row)) << 4), kdst + i * 1024);
      lds_dma16(vgb + off, (unsigned)((ln ^ swz_v<D>(row)) << 4), kdst + TL::TILEB + i * 1024);
    }
  };
  issue(kt_begin, 0);

  // ---- Q^T slice: channels CW slice + 16 s + 8 hi + e, RMSNorm over all 512 channels
  // (slice sums added through LDS in slice order), RoPE with the partner c ^ 256.
  V8 qreg[KSTEPS];
  {
    const int c0 = CW * slice + 8 * hi;
    const int pc0 = (CW * slice + 8 * hi) ^ 256;   // partner channels
    const T* src = static_cast<const T*>(p.q) + b * p.sqb + h * p.sqh + (int64_t)(valid_q ? i_q : 0) * p.sqt;
    // Raw slices stay packed, and each k-step is unpacked, normalised, rotated and rounded in turn.
    // Eight waves read theirs once for the sum of squares and again per k-step: held in between, it
    // and the partners' slice spill. Four waves (twice the registers) hold both: a short call is
    // mostly its prologue, 1.3 to 2 us shorter that way (5 rows of 51 queries 33.1 -> 31.4 us).
    constexpr bool HOLD = NW == 4;
    uint4 held_x[HOLD ? KSTEPS : 1], held_z[HOLD ? KSTEPS : 1];
    if constexpr (HOLD) {
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s) {
        held_x[s] = load16(src + c0 + 16 * s);
        held_z[s] = load16(src + pc0 + 16 * s);
      }
    }
    auto raw_x = [&](int s) { return HOLD ? held_x[HOLD ? s : 0] : load16(src + c0 + 16 * s); };
    auto raw_z = [&](int s) { return HOLD ? held_z[HOLD ? s : 0] : load16(src + pc0 + 16 * s); };
    const bool norm = (p.flags & FORGE_NORM_QK) != 0;
    float rs = 1.0f;
    if (norm) {
      float ss = 0.0f;
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s) {
        float x[8];
        unpack16<T>(raw_x(s), x);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
      }
      ss += __shfl_xor(ss, 32, kWave);
      if (hi == 0) sh_ss[wave * 32 + n] = ss;
      __syncthreads();
      float tot = sh_ss[wbase * 32 + n];
#pragma unroll
      for (int w = 1; w < SPLIT; ++w) tot += sh_ss[(wbase + w) * 32 + n];
      rs = rsqrtf(tot / (float)D + p.eps);
    }
    const bool rope = (p.flags & FORGE_ROPE) && valid_q;
    const float* cr = rope ? p.cos + (int64_t)i_q * p.cst : nullptr;
    const float* sr = rope ? p.sin + (int64_t)i_q * p.cst : nullptr;
    const bool first_half = CW * slice < 256;
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      float x[8], z[8];
      unpack16<T>(raw_x(s), x);
      unpack16<T>(raw_z(s), z);
      if (norm) {
        float wx[8], wz[8];
        if (p.qw) {
          load_f32x8(p.qw + c0 + 16 * s, wx);
          load_f32x8(p.qw + pc0 + 16 * s, wz);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          x[e] *= rs;
          z[e] *= rs;
          if (p.qw) {
            x[e] *= wx[e];
            z[e] *= wz[e];
          }
        }
      }
      if (rope) {
        float cv[8], sv[8];
        load_f32x8(cr + c0 + 16 * s, cv);
        load_f32x8(sr + c0 + 16 * s, sv);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = first_half ? x[e] * cv[e] - z[e] * sv[e] : x[e] * cv[e] + z[e] * sv[e];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) qreg[s][e] = from_f32<T>(valid_q ? x[e] : 0.0f);
    }
  }

  const int off = (int)p.offset;
  const int S32 = (int)S;
  const int qpos32 = (int)(p.offset + i_q);
  const int wq_lo = off + qt * TL::BM, wq_hi = off + q_last_idx;
  // LDS read offsets of a lane within a stage's K and V tiles (the layouts of prefill_kernel).
  // The swizzles only touch the low four chunk bits, so k-step st's operand lies at
  // k_rd ^ 32 (st % 8) plus 256 bytes per 8 steps, and channel block d's at v_rd ^ 64 (d % 4)
  // plus 256 bytes per 4 blocks: one xor from one register each.
  const int g = lane >> 4, kq = (lane >> 2) & 3, qq = lane & 3;
  const int v_row = 4 * (g >> 1) + kq;
  const unsigned k_rd = n * TL::ROWB + CCH * 16 * slice + ((hi ^ swz_k<D>(n)) << 4);
  const unsigned v_rd = v_row * TL::ROWB + CCH * 16 * slice +
                        (((2 * (g & 1) + (qq >> 1)) ^ swz_v<D>(v_row)) << 4) + 8 * (qq & 1);
  const unsigned lds0 = lds_offset(smem);

  floatx16 oacc[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int x = 0; x < 16; ++x) oacc[d][x] = 0.0f;
  float m_run = kNegInf, l_run = 0.0f;
  const float c = p.scale_log2;

  for (int kt = kt_begin; kt <= kt_end; ++kt) {
    const int stage = (kt - kt_begin) & 1;
    wait_vm<0>();
    __syncthreads();   // tile kt in LDS; every wave is done with tile kt - 1 and its partials
    if (kt + 1 <= kt_end) issue(kt + 1, stage ^ 1);
    const unsigned kl = lds0 + (2 * stage) * TL::TILEB + k_rd;
    const unsigned vl = lds0 + (2 * stage + 1) * TL::TILEB + v_rd;

    // partial scores of this wave's channels
    floatx16 sp;
#pragma unroll
    for (int x = 0; x < 16; ++x) sp[x] = 0.0f;
    {
      // K operands two k-steps ahead of their MFMA, pinned as in prefill_kernel (left alone the
      // compiler reads them all first, and with eight waves spills)
      auto kread = [&](int st) {
        return *(__attribute__((address_space(3))) const V8*)((kl ^ (32 * (st & 7))) + 256 * (st >> 3));
      };
      V8 a0 = kread(0), a1 = kread(1), a2 = a1;
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
      for (int st = 0; st < KSTEPS; ++st) {
        if (st + 2 < KSTEPS) {
          a2 = kread(st + 2);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        sp = Mfma<T>::run(a0, qreg[st], sp);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        a0 = a1;
        a1 = a2;
      }
    }
    {
      float4* dst = reinterpret_cast<float4*>(part + (wave * 64 + lane) * 16);
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[i] = make_float4(sp[4 * i], sp[4 * i + 1], sp[4 * i + 2], sp[4 * i + 3]);
    }
    __syncthreads();
    floatx16 sacc;
    {
      // the head's slices added in slice order (the same sums in every wave of the head)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float4 t = reinterpret_cast<const float4*>(part + (wbase * 64 + lane) * 16)[i];
#pragma unroll
        for (int w = 1; w < SPLIT; ++w) {
          const float4 u = reinterpret_cast<const float4*>(part + ((wbase + w) * 64 + lane) * 16)[i];
          t.x += u.x;
          t.y += u.y;
          t.z += u.z;
          t.w += u.w;
        }
        sacc[4 * i + 0] = t.x;
        sacc[4 * i + 1] = t.y;
        sacc[4 * i + 2] = t.z;
        sacc[4 * i + 3] = t.w;
      }
    }

    const int key0 = kt * BN;
    const bool full = key0 + BN - 1 <= wq_lo && key0 + BN - 1 < S32 &&
                      (p.window <= 0 || wq_hi - key0 < p.window) && q_last_idx - qt * TL::BM == TL::BM - 1 &&
                      key0 >= d_last;
    if (!full) {
      const int base = key0 + 4 * hi;
      const int top = (qpos32 < S32 - 1 ? qpos32 : S32 - 1) - base;
      const int lim_hi = valid_q ? top : -1;
      int lim_lo = p.window > 0 ? qpos32 - p.window + 1 - base : -(1 << 30);
      if (dl && d_lane - base > lim_lo) lim_lo = d_lane - base;
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        const int ce = 8 * (x >> 2) + (x & 3);
        sacc[x] = (ce <= lim_hi && ce >= lim_lo) ? sacc[x] : kNegInf;
      }
    }
    float mx = sacc[0];
#pragma unroll
    for (int x = 1; x < 16; ++x) mx = fmaxf(mx, sacc[x]);
    mx = max_xor32(mx);
    const float mxc = mx * c;
    if (mxc > m_run + kLazyLog2) {
      const float alpha = m_run == kNegInf ? 0.0f : __builtin_amdgcn_exp2f(m_run - mxc);
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int x = 0; x < 16; ++x) oacc[d][x] *= alpha;
      m_run = mxc;
    }
    const float neg_m = m_run == kNegInf ? 0.0f : -m_run;
    float rs[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const float pv = __builtin_amdgcn_exp2f(fmaf(sacc[x], c, neg_m));
      sacc[x] = pv;
      rs[x & 3] += pv;
    }
    l_run += (rs[0] + rs[1]) + (rs[2] + rs[3]);

    // O^T += V^T . P^T over this wave's CW channels
#pragma unroll
    for (int hf = 0; hf < HALVES; ++hf) {
      V8 pb;
#pragma unroll
      for (int e = 0; e < 8; ++e) pb[e] = from_f32<T>(sacc[8 * hf + e]);
#pragma unroll
      for (int d = 0; d < DB; ++d) {
        const unsigned va = (vl ^ (64 * (d & 3))) + 256 * (d >> 2) + 16 * hf * TL::ROWB;
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)va);
        const i16x4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) i16x4*)(va + 8 * TL::ROWB));
        typedef short i16x8 __attribute__((ext_vector_type(8)));
        const i16x8 av = __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7);
        oacc[d] = Mfma<T>::run(__builtin_bit_cast(V8, av), pb, oacc[d]);
      }
    }
  }

  l_run += __shfl_xor(l_run, 32, kWave);
  if (!valid_q) return;
  if (KSPLIT && parts > 1) {
    const int64_t rows = (int64_t)p.B * p.H * p.T;
    const int64_t slot = kpart * rows + ((int64_t)b * p.H + h) * p.T + i_q;
    float* po = p.ws_o + slot * D + CW * slice + 4 * hi;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<float4*>(po + d * 32 + 8 * i) =
            make_float4(oacc[d][4 * i], oacc[d][4 * i + 1], oacc[d][4 * i + 2], oacc[d][4 * i + 3]);
    if (hi == 0 && slice == 0) p.ws_ml[slot] = make_float2(m_run, l_run);
    return;
  }
  const float inv_l = 1.0f / l_run;
  T* dst = static_cast<T*>(p.out) + b * p.sob + (int64_t)i_q * p.sot + h * p.soh + CW * slice;
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      T vals[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) vals[j] = from_f32<T>(oacc[d][4 * i + j] * inv_l);
      *reinterpret_cast<uint2*>(dst + d * 32 + 8 * i + 4 * hi) = *reinterpret_cast<uint2*>(vals);
    }
}

template <typename T, int NW, int SPLIT, bool KSPLIT>
static int launch_prefill_wide_s(PrefillParams p, hipStream_t s) {
  using TL = WideTile<NW>;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_wide_kernel<T, NW, SPLIT, KSPLIT>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, TL::LDS_BYTES) != hipSuccess)
      return set_error("forge_attn_prefill: cannot reserve the LDS the kernel needs");
    attr_set = true;
  }
  constexpr int HPB = TL::WAVES / SPLIT;
  p.nqt = (p.T + TL::BM - 1) / TL::BM;
  const int64_t blocks = (int64_t)p.nqt * (p.H / HPB) * p.B * p.nsplit;
  if (blocks > 0x7fffffff) return set_error("grid too large");
  hipLaunchKernelGGL((prefill_wide_kernel<T, NW, SPLIT, KSPLIT>), dim3((unsigned)blocks), dim3(TL::WAVES * 64),
                     TL::LDS_BYTES, s, p);
  return check_launch();
}

template <typename T, int NW, int SPLIT>
static int launch_prefill_wide_w(const PrefillParams& p, hipStream_t s) {
  if (p.nsplit < 2) return launch_prefill_wide_s<T, NW, SPLIT, false>(p, s);
  const int st = launch_prefill_wide_s<T, NW, SPLIT, true>(p, s);
  return st ? st : launch_prefill_combine<T, 512>(p, WideTile<NW>::BM, WideTile<NW>::BN, s);
}

template <typename T>
static int launch_prefill_wide(const PrefillParams& p, hipStream_t s) {
  switch (p.heads_per_block) {
    case 4: return launch_prefill_wide_w<T, 8, 2>(p, s);
    case 2: return launch_prefill_wide_w<T, 4, 2>(p, s);
    default: return launch_prefill_wide_w<T, 4, 4>(p, s);
  }
}

// ---------------------------------------------------------------- fp32
// fp32 prefill on v_mfma_f32_32x32x2_f32 (fp32 products and sums, as the split-K kernel's FMAs).
// That instruction takes 64 clocks for 4,096 FLOP, so a wave needs little bandwidth and the
// operands go from L2 straight into registers, with no LDS and no barrier in the loop: a block is
// 32 queries of one (b, head), and its four waves take the 32-key tiles in turn (wave w tiles w,
// w + 4, ...), each with its own running (m, l, o), merged through LDS at the end in a fixed
// order. Splitting a query tile's keys over the waves keeps the chain of dependent tiles short
// (1,025 causal queries: 9 tiles instead of 33), and small blocks fill the CUs on short calls.
//   * S^T = K . Q^T: lane (n, hi) holds channels 8j + 4hi + e of key n (16-byte loads) and of query
//     n; MFMA step (j, e) contracts channels 8j + e and 8j + 4 + e.
//   * O^T = V^T . P^T straight from the score registers: step x pairs keys 8(x/4) + x%4 and + 4. Row
//     m of output block d stands for channel DB m + d (DB = D / 32 blocks), so one load of DB
//     consecutive channels feeds all the blocks.
// V is requested before the tile's score MFMAs, the next tile's K after them.
// Sums run in short chains added as trees (16 channels of a score, 16 keys of an output, per
// chain). 2-norm error against 64 bits over the split-K path's, means over 4 to 12 inputs of 54 shapes of
// 17 to 1,500 queries: 0.93 to 0.99 from 49 keys on, 0.99 to 1.04 below, where the module takes that path.
// Against the split-K path, whose blocks of 8 rows each take every key through the VALU: 2 x
// 1,025 causal, 8 q / 4 KV heads, head dim 32: 168 -> 23 us (46 TFLOP/s); 4 x 2,048 at head dim
// 64: 3.0 -> 0.21 ms; 2,000 at 16 q / 8 KV heads, head dim 128: 3.1 -> 0.25 ms; 17 queries 11 -> 6 us.
template <int D> struct F32Tile {
  static constexpr int WAVES = 4;
  static constexpr int BM = 32;            // queries per block
  static constexpr int BN = 32 * WAVES;    // keys per step of the block
  static constexpr int DB = D / 32;
  static constexpr int LDS_BYTES = 2 * (32 * D + 64) * 4;  // two waves' partials
};

template <int DB> struct F32Vec;
template <> struct F32Vec<1> { typedef float type __attribute__((ext_vector_type(1))); };
template <> struct F32Vec<2> { typedef float type __attribute__((ext_vector_type(2))); };
template <> struct F32Vec<4> { typedef float type __attribute__((ext_vector_type(4))); };

template <int D, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu((D >= 128 ? 1 : 2))))
void prefill_f32_kernel(PrefillParams p) {
  using TL = F32Tile<D>;
  constexpr int DB = TL::DB;
  constexpr int NJ = D / 8;  // 16-byte pieces of a lane's half row
  typedef typename F32Vec<DB>::type VecV;
  extern __shared__ __attribute__((aligned(16))) float sh[];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lane = tid % kWave;
  const int n = lane & 31;
  const int hi = lane >> 5;

  // block -> (query tile, part, head, batch), heavy (late) causal tiles first
  const int NS = SPLIT ? p.nsplit : 1;
  const int HB = p.H * p.B;
  const int qt = p.nqt - 1 - (int)blockIdx.x / (HB * NS);
  const int part = (int)blockIdx.x % (HB * NS) / HB;
  const int hb = (int)blockIdx.x % HB;
  const int b = hb / p.H, h = hb % p.H;
  const int kvh = h / p.G;
  int kt_begin, kt_end, parts = 1;  // in steps of BN keys
  tile_span(p.offset, p.T, p.window, 0, qt, TL::BM, TL::BN, kt_begin, kt_end);
  if (SPLIT && !take_part(p, part, kt_begin, kt_end, parts)) return;

  const int i0 = qt * TL::BM;
  const int i_q = i0 + n;
  const bool valid_q = i_q < p.T;
  const int S = (int)p.offset + p.T;
  const int qpos = (int)p.offset + i_q;
  const int i_last = i0 + 31 < p.T - 1 ? i0 + 31 : p.T - 1;
  const int q_lo = (int)p.offset + i0, q_hi = (int)p.offset + i_last;

  // K and V through buffer resources that end with key S - 1 (host check: under 2^31 bytes): keys
  // past it, which are masked, read zeros, and an address is one 32-bit offset
  const unsigned row_bytes = (unsigned)p.sks * 4u;
  const unsigned slab_bytes = (unsigned)(S - 1) * row_bytes + D * 4u;
  const __amdgpu_buffer_rsrc_t krs = slab_rsrc(static_cast<const float*>(p.k) + b * p.skb + kvh * p.skh, slab_bytes);
  const __amdgpu_buffer_rsrc_t vrs = slab_rsrc(static_cast<const float*>(p.v) + b * p.skb + kvh * p.skh, slab_bytes);
  const unsigned k_lane = (unsigned)n * row_bytes + 16u * hi, v_lane = 4u * hi * row_bytes + 4u * DB * n;

  // ---- Q^T: RMSNorm + RoPE in fp32 (pairs c, c + D/2 are pieces j, j + NJ/2 of one lane)
  float q[NJ][4];
  {
    const float* src = static_cast<const float*>(p.q) + b * p.sqb + h * p.sqh +
                       (int64_t)(valid_q ? i_q : p.T - 1) * p.sqt + 4 * hi;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const float4 x = *reinterpret_cast<const float4*>(src + 8 * j);
      q[j][0] = x.x; q[j][1] = x.y; q[j][2] = x.z; q[j][3] = x.w;
    }
    if (p.flags & FORGE_NORM_QK) {
      float ss = 0.0f;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += q[j][e] * q[j][e];
      ss += __shfl_xor(ss, 32, kWave);
      const float rs = rsqrtf(ss / (float)D + p.eps);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        float4 w = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
        if (p.qw) w = *reinterpret_cast<const float4*>(p.qw + 8 * j + 4 * hi);
        q[j][0] = q[j][0] * rs * w.x;
        q[j][1] = q[j][1] * rs * w.y;
        q[j][2] = q[j][2] * rs * w.z;
        q[j][3] = q[j][3] * rs * w.w;
      }
    }
    if (p.flags & FORGE_ROPE) {
      const int64_t row = (int64_t)(valid_q ? i_q : p.T - 1) * p.cst + 4 * hi;
#pragma unroll
      for (int j = 0; j < NJ / 2; ++j) {
        const float4 c1 = *reinterpret_cast<const float4*>(p.cos + row + 8 * j);
        const float4 s1 = *reinterpret_cast<const float4*>(p.sin + row + 8 * j);
        const float4 c2 = *reinterpret_cast<const float4*>(p.cos + row + 8 * j + D / 2);
        const float4 s2 = *reinterpret_cast<const float4*>(p.sin + row + 8 * j + D / 2);
        const float c1v[4] = {c1.x, c1.y, c1.z, c1.w}, s1v[4] = {s1.x, s1.y, s1.z, s1.w};
        const float c2v[4] = {c2.x, c2.y, c2.z, c2.w}, s2v[4] = {s2.x, s2.y, s2.z, s2.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float a = q[j][e], z = q[j + NJ / 2][e];
          q[j][e] = a * c1v[e] - z * s1v[e];
          q[j + NJ / 2][e] = z * c2v[e] + a * s2v[e];
        }
      }
    }
  }

  floatx16 oacc[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int x = 0; x < 16; ++x) oacc[d][x] = 0.0f;
  float m_run = kNegInf, l_run = 0.0f;
  const float c = p.scale_log2;

  // first key of this wave's tile of step kt
  auto tile_key = [&](int kt) { return kt * TL::BN + 32 * wave; };
  floatx4 kr[NJ];
  auto load_k = [&](int key0) {
    const unsigned off = (unsigned)key0 * row_bytes + k_lane;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      kr[j] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(krs, (int)(off + 32 * j), 0, 0));
  };
  // a wave's tile lies outside every query's keys in the first and last steps only
  auto needed = [&](int key0) {
    return key0 <= q_hi && (p.window <= 0 || key0 + 31 > q_lo - p.window);
  };
  load_k(tile_key(kt_begin));
  for (int kt = kt_begin; kt <= kt_end; ++kt) {
    const int key0 = tile_key(kt);
    if (!needed(key0)) {  // wave-uniform
      if (kt < kt_end) load_k(tile_key(kt + 1));
      continue;
    }
    VecV vr[16];
    unsigned v_off = v_lane;
    asm volatile("" : "+v"(v_off));  // (the 16 rows' offsets are made here, not kept over the loop)
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const int off = (int)((unsigned)(key0 + 8 * (x >> 2) + (x & 3)) * row_bytes + v_off);
      if constexpr (DB == 1) vr[x] = __builtin_bit_cast(VecV, __builtin_amdgcn_raw_buffer_load_b32(vrs, off, 0, 0));
      else if constexpr (DB == 2) vr[x] = __builtin_bit_cast(VecV, __builtin_amdgcn_raw_buffer_load_b64(vrs, off, 0, 0));
      else vr[x] = __builtin_bit_cast(VecV, __builtin_amdgcn_raw_buffer_load_b128(vrs, off, 0, 0));
    }
    // 16 channels at a time in two chains of four steps: one chain over all the channels would
    // round more often than the split-K path's lanes do
    floatx16 sacc, sodd;  // (at head dim 128 the groups in two running sums)
#pragma unroll
    for (int j0 = 0; j0 < NJ; j0 += 2) {
      floatx16 sc[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int x = 0; x < 16; ++x) sc[i][x] = 0.0f;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 2; ++i) sc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[j0 + i][e], q[j0 + i][e], sc[i], 0, 0, 0);
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        const float u = sc[0][x] + sc[1][x];
        if (D >= 128 && (j0 & 2)) sodd[x] = j0 == 2 ? u : sodd[x] + u;
        else sacc[x] = j0 == 0 ? u : sacc[x] + u;
      }
      // (summed here: two partial tiles live at a time, not all of them)
      if (D >= 128 && (j0 & 2)) asm volatile("" : "+v"(sodd));
      else asm volatile("" : "+v"(sacc));
    }
    if constexpr (D >= 128) {
#pragma unroll
      for (int x = 0; x < 16; ++x) sacc[x] += sodd[x];
    }
    if (kt < kt_end) load_k(tile_key(kt + 1));

    // The exponent is one fma of the raw score; scaled first it would be rounded once more. 2-norm
    // error of the outputs against 64 bits, 2 x 1,025 causal at head dim 32: 2.23e-7 (2.39e-7 scaled
    // first; the split-K path 2.36e-7); 512 queries at 2,000, head dim 64: 3.14e-7 (3.37e-7; 3.24e-7).
    const bool full = key0 + 31 <= q_lo && (p.window <= 0 || q_hi - key0 < p.window);
    float mx = kNegInf;
    if (!full) {
      const int base = key0 + 4 * hi;
      const int top = qpos < S - 1 ? qpos : S - 1;  // (rows past T mask as their own position)
      const int lo = p.window > 0 ? qpos - p.window + 1 : 0;
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        const int key = base + 8 * (x >> 2) + (x & 3);
        sacc[x] = key <= top && key >= lo ? sacc[x] : kNegInf;
        mx = fmaxf(mx, sacc[x] == kNegInf ? kNegInf : sacc[x] * c);
      }
    } else {
#pragma unroll
      for (int x = 0; x < 16; ++x) mx = fmaxf(mx, sacc[x] * c);
    }
    mx = max_xor32(mx);
    if (mx > m_run + kLazyLog2) {
      const float alpha = m_run == kNegInf ? 0.0f : __builtin_amdgcn_exp2f(m_run - mx);
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int x = 0; x < 16; ++x) oacc[d][x] *= alpha;
      m_run = mx;
    }
    const float ref = m_run == kNegInf ? 0.0f : m_run;
#pragma unroll
    for (int x = 0; x < 16; ++x) sacc[x] = sacc[x] == kNegInf ? 0.0f : __builtin_amdgcn_exp2f(fmaf(sacc[x], c, -ref));
    {
      float rs[8];  // summed as a tree
#pragma unroll
      for (int x = 0; x < 8; ++x) rs[x] = sacc[x] + sacc[x + 8];
      l_run += ((rs[0] + rs[4]) + (rs[1] + rs[5])) + ((rs[2] + rs[6]) + (rs[3] + rs[7]));
    }
    // the tile's sum on its own in four chains, then into the running one: the error grows with the
    // tiles and the keys of a chain, not with their product
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      floatx16 sum;
#pragma unroll
      for (int x0 = 0; x0 < 16; x0 += 8) {
        floatx16 ot[2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int x = 0; x < 16; ++x) ot[i][x] = 0.0f;
#pragma unroll
        for (int x = x0; x < x0 + 8; ++x)
          ot[x & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[x][d], sacc[x], ot[x & 1], 0, 0, 0);
#pragma unroll
        for (int x = 0; x < 16; ++x) sum[x] = x0 ? sum[x] + (ot[0][x] + ot[1][x]) : ot[0][x] + ot[1][x];
        asm volatile("" : "+v"(sum));
      }
#pragma unroll
      for (int x = 0; x < 16; ++x) oacc[d][x] += sum[x];
      asm volatile("" : "+v"(oacc[d]));
    }
  }
  l_run += __shfl_xor(l_run, 32, kWave);

  // ---- merge the waves: (0, 2) and (1, 3), then (0, 1)
  auto put = [&](int slot) {
    float* dst = sh + slot * (32 * D + 64);
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int x = 0; x < 16; ++x) dst[(d * 16 + x) * kWave + lane] = oacc[d][x];
    if (hi == 0) {
      dst[32 * D + n] = m_run;
      dst[32 * D + 32 + n] = l_run;
    }
  };
  auto merge = [&](int slot) {
    const float* src = sh + slot * (32 * D + 64);
    const float m_o = src[32 * D + n], l_o = src[32 * D + 32 + n];
    const float m_n = fmaxf(m_run, m_o);
    const float a = rescale(m_run, m_n), z = rescale(m_o, m_n);
    l_run = l_run * a + l_o * z;
    m_run = m_n;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int x = 0; x < 16; ++x) oacc[d][x] = oacc[d][x] * a + src[(d * 16 + x) * kWave + lane] * z;
  };
  if (wave >= 2) put(wave - 2);
  __syncthreads();
  if (wave < 2) merge(wave);
  __syncthreads();
  if (wave == 1) put(0);
  __syncthreads();
  if (wave != 0) return;
  merge(0);
  if (!valid_q) return;
  // channel DB m + d, m = 8(x/4) + 4hi + x%4
  if (SPLIT && parts > 1) {
    const int64_t slot = part * ((int64_t)p.B * p.H * p.T) + ((int64_t)b * p.H + h) * p.T + i_q;
    float* dst = p.ws_o + slot * D;
#pragma unroll
    for (int x = 0; x < 16; ++x)
#pragma unroll
      for (int d = 0; d < DB; ++d) dst[DB * (8 * (x >> 2) + 4 * hi + (x & 3)) + d] = oacc[d][x];
    if (hi == 0) p.ws_ml[slot] = make_float2(m_run, l_run);
    return;
  }
  float* dst = static_cast<float*>(p.out) + b * p.sob + (int64_t)i_q * p.sot + h * p.soh;
#pragma unroll
  for (int x = 0; x < 16; ++x)
#pragma unroll
    for (int d = 0; d < DB; ++d) dst[DB * (8 * (x >> 2) + 4 * hi + (x & 3)) + d] = oacc[d][x] / l_run;
}

template <int D, bool SPLIT>
static int launch_prefill_f32_s(PrefillParams p, hipStream_t s) {
  using TL = F32Tile<D>;
  p.nqt = (p.T + TL::BM - 1) / TL::BM;
  const int64_t blocks = (int64_t)p.nqt * p.H * p.B * p.nsplit;
  if (blocks > 0x7fffffff) return set_error("grid too large");
  hipLaunchKernelGGL((prefill_f32_kernel<D, SPLIT>), dim3((unsigned)blocks), dim3(256), TL::LDS_BYTES, s, p);
  return check_launch();
}

template <int D>
static int launch_prefill_f32(const PrefillParams& p, hipStream_t s) {
  if (p.nsplit < 2) return launch_prefill_f32_s<D, false>(p, s);
  const int st = launch_prefill_f32_s<D, true>(p, s);
  return st ? st : launch_prefill_combine<float, D>(p, F32Tile<D>::BM, F32Tile<D>::BN, s);
}

// How a launch splits its query tiles' keys: parts of at most `tiles` key tiles, nsplit of them
// for the longest query tile. A launch with fewer query tiles than the CUs take (a chunk of a
// long prompt, a short batch) otherwise leaves CUs idle behind its longest blocks: one 512-token
// chunk at position 15,360 (16 q / 8 KV heads, head dim 128) is 64 blocks of 248 tiles.
struct PrefillPlan {
  int nsplit, tiles;
  int heads_per_block;
};
constexpr int kMaxParts = 32;

// Heads per block of an unsplit launch at head dim 512, from the time of its blocks: a tile of four heads
// takes 2.55 us and one of two heads 2.1, what a block does besides (mostly its q prologue) as long as 13
// and 7.6 tiles, and the last, partial round of blocks (the lightest: heavy ones go first) between its
// lightest block and a mean one. Against both forms timed at 33 shapes of 17 to 4,096 queries, one to
// eight rows, the pick is the faster one or within 1% of it (four / two heads, us): 8 x 130 52 / 49, 3 x 435
// 76 / 65, 8 x 300 (8 q / 2 KV heads) 64 / 57, 6 x 435 108 / 112, 3 x 700 99 / 117, 2,000 199 / 179, 2,500 241 / 282.
static int wide_heads(int B, int H, int nqt, int longest, int lightest, int64_t work, int64_t cus) {
  double us[2];
  for (int i = 0; i < 2; ++i) {
    const int heads = i ? 2 : 4;
    const double tile = i ? 2.1 : 2.55, prologue = i ? 7.6 : 13.0;
    const int64_t blocks = (int64_t)nqt * (H / heads) * B, rest = blocks % cus;
    const double mean = (double)work / nqt, last = rest ? lightest + prologue + (mean - lightest) * rest / cus : 0.0;
    const double load = (blocks / cus) * (mean + prologue) + last;
    us[i] = 5.0 + tile * (load > longest + prologue ? load : longest + prologue);
  }
  return us[1] < 0.95 * us[0] ? 2 : 4;  // (by more than the model's error)
}

// Picks the split with the least modelled time. Measured on calls of 1 to 32 parts (graph
// replays, one box; the model is within 15% of each): a tile takes `alone` us in a block that has
// its CU to itself and `shared` us of a CU that holds several (head dims 64 to 256), a block's q
// prologue and epilogue cost about 2.5 tiles, its partial crosses memory twice at about 4 TB/s,
// and the combine launch takes 3 us. So parts pay while CUs are idle and stop paying once the
// partials' traffic grows: 16 q / 8 KV heads, head dim 128, 1 / 2 / 4 / 8 / 16 parts: T 512 at
// 15,360: 279 / 149 / 87 / 83 / 96 us; T 128 there: 267 / 143 / 79 / 49 / 39; T 64 at 1,000:
// 25 / 20 / 16 / 15 / 17; T 1024 at 15,360: 288 / 170 / 143 / 162 / 191; a whole prompt of
// 2,048: 44 / 49 / 53 / 71 / 115 (not split). Head dim 256 (8 q / 4 KV), T 512 at 8,000: 352 /
// 186 / 105 / 69 / 86.
// At head dim 512 the same model picks the heads that share a split launch's blocks and their K/V
// tiles (T 512 at 8,000: 211 us with four, 301 with two), and wide_heads an unsplit one's.
static PrefillPlan prefill_plan(bool f32, int B, int T, int H, int K, int D, int64_t offset, int window,
                                int max_parts) {
  const bool wide = D == 512;
  const int BM = f32 ? F32Tile<32>::BM : wide ? WideTile<4>::BM : Tile<64>::BM;
  const int BN = f32 ? F32Tile<32>::BN : wide ? WideTile<4>::BN : D == 256 ? Tile<256>::BN : Tile<128>::BN;
  const int G = H / K;
  const int most_heads = f32 || !wide ? 1 : G % 4 == 0 ? 4 : G % 2 == 0 ? 2 : 1;
  const int64_t cus = device_cus();
  const int nqt = (T + BM - 1) / BM;
  if ((int64_t)nqt * (H / most_heads) * B >= 4 * cus)  // several rounds of blocks already
    return PrefillPlan{1, 0, most_heads};
  int longest = 0, lightest = INT_MAX;
  int64_t work = 0;
  for (int qt = 0; qt < nqt; ++qt) {
    int begin, end;
    tile_span(offset, T, window, 0, qt, BM, BN, begin, end);
    const int n = end - begin + 1;
    longest = n > longest ? n : longest;
    lightest = n < lightest ? n : lightest;
    work += n;
  }
  PrefillPlan best{1, longest, most_heads};
  double best_us = 0.0;
  for (int c = 1, last = 0; c <= max_parts; ++c) {
    const int tiles = (longest + c - 1) / c;
    if (tiles == last) continue;
    last = tiles;
    int64_t blocks1 = 0, split1 = 0, work1 = 0;  // per head group: blocks, partials, key tiles
    for (int qt = 0; qt < nqt; ++qt) {
      int begin, end;
      tile_span(offset, T, window, 0, qt, BM, BN, begin, end);
      const int n = end - begin + 1, parts = (n + tiles - 1) / tiles;
      blocks1 += parts;
      if (parts > 1) split1 += parts;
      work1 += n;
    }
    bool open = false;  // some split into more parts may still win
    for (int hpb = most_heads; hpb >= (most_heads == 4 ? 2 : most_heads); hpb /= 2) {
      double alone = hpb == 4 ? 2.55 : wide ? 2.1 : D == 256 ? 1.25 : 1.2;
      double shared = wide ? alone : D == 256 ? 1.05 : D == 128 ? 0.95 : 0.65;
      if (f32) {  // four waves' tiles: 128 D / 32 MFMAs of 64 clocks on each SIMD
        alone = 0.6 + 1.0 * D / 32;
        shared = 1.0 * D / 32;
      }
      const int64_t blocks = blocks1 * (H / hpb) * B;
      const double per_block = (double)work1 / blocks1 + 2.5;
      const int64_t rounds = (blocks + cus - 1) / cus;
      double us = (tiles + 2.5) * alone;  // the longest block
      if (rounds > 1 && rounds * per_block * shared > us) us = rounds * per_block * shared;
      const double partials = split1 ? 3.0 + 2.0 * split1 * H * B * BM * D * sizeof(float) / 4e6 : 0.0;
      us += partials;
      // (splitting has to be worth more than the model's error)
      const bool first = c == 1 && hpb == most_heads;
      if (first || us < (c > 1 && best.nsplit == 1 ? 0.8 : 0.95) * best_us) {
        best = PrefillPlan{c, tiles, hpb};
        best_us = us;
      }
      // with the CUs full, blocks and partials only grow with the parts, and the time with them
      open = open || rounds == 1 || blocks * per_block * shared / cus + partials < 0.95 * best_us;
    }
    if (!open) break;
  }
  if (best.nsplit > 1) best.nsplit = (longest + best.tiles - 1) / best.tiles;
  else if (most_heads == 4) best.heads_per_block = wide_heads(B, H, nqt, longest, lightest, work, cus);
  return best;
}

template <typename T>
static int launch_prefill(const PrefillParams& p, int D, hipStream_t s) {
  switch (D) {
    case 64: return launch_prefill_d<T, 64>(p, s);
    case 128: return launch_prefill_d<T, 128>(p, s);
    case 256: return launch_prefill_d<T, 256>(p, s);
    case 512: return launch_prefill_wide<T>(p, s);
    default: return set_error("forge_attn_prefill: head dim must be 64, 128, 256 or 512");
  }
}

}  // namespace forge

using namespace forge;

// Positions up to a tile past the last one fit in 31 bits (without a sum that could wrap).
static bool positions_fit(int64_t offset, int T) { return offset < (1LL << 31) - 256 - (int64_t)T; }

// fp32 (m, l) pairs and partial outputs of every part of every row
static size_t prefill_workspace(const PrefillPlan& plan, int B, int T, int H, int D) {
  const size_t slots = (size_t)plan.nsplit * B * H * T;
  return (slots * sizeof(float2) + 255) / 256 * 256 + slots * D * sizeof(float);
}

// Checks what every prefill entry point takes (`esize` bytes per element) and fills everything
// of p but the documents and the plan. Returns 0, or the status of set_error.
static int prefill_setup(PrefillParams& p, int esize, int B, int T, int H, int K, const void* q, int64_t sqb,
                         int64_t sqh, int64_t sqt, const float* q_weight, float eps, int flags,
                         const float* cos, const float* sin, int64_t s_cos_t, const void* k, const void* v,
                         int64_t skb, int64_t skh, int64_t sks, int64_t offset, int window, float scale,
                         void* out, int64_t sob, int64_t sot, int64_t soh) {
  if (B <= 0 || T <= 0 || H <= 0 || K <= 0) return set_error("sizes must be positive");
  if (H % K) return set_error("n_heads must be a multiple of the KV heads");
  if (offset < 0) return set_error("offset must be >= 0");
  if (window < 0) return set_error("window must be >= 0");
  if (!q || !k || !v || !out) return set_error("null tensor pointer");
  if ((flags & FORGE_ROPE) && (!cos || !sin)) return set_error("FORGE_ROPE needs cos and sin");
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) % 16)
    return set_error("forge_attn_prefill: tensors must be 16-byte aligned");
  if ((sqb | sqh | sqt | skb | skh | sks) % (16 / esize))
    return set_error("forge_attn_prefill: q/k/v strides must be multiples of 16 bytes");
  if ((sob | sot | soh) % 4) return set_error("forge_attn_prefill: out strides must be multiples of 4");
  if (!positions_fit(offset, T)) return set_error("forge_attn_prefill: positions must fit in 31 bits");
  if (sks * esize * 256 >= (1LL << 31)) return set_error("forge_attn_prefill: k/v row stride too large");
  if (((uintptr_t)q_weight | (uintptr_t)cos | (uintptr_t)sin) % 16 || (cos && s_cos_t % 4))
    return set_error("forge_attn_prefill: gain and RoPE rows must be 16-byte aligned");
  p = PrefillParams{};
  p.q = q;
  p.sqb = sqb;
  p.sqh = sqh;
  p.sqt = sqt;
  p.qw = q_weight;
  p.eps = eps;
  p.flags = flags;
  p.cos = cos;
  p.sin = sin;
  p.cst = s_cos_t;
  p.k = k;
  p.v = v;
  p.skb = skb;
  p.skh = skh;
  p.sks = sks;
  p.offset = offset;
  p.B = B;
  p.T = T;
  p.H = H;
  p.K = K;
  p.G = H / K;
  p.window = window;
  p.scale_log2 = scale * kLog2e;
  p.out = out;
  p.sob = sob;
  p.sot = sot;
  p.soh = soh;
  return 0;
}

// Puts a plan and its partials' workspace into p.
static int prefill_bind(PrefillParams& p, const PrefillPlan& plan, int D, void* workspace, size_t workspace_bytes) {
  p.nsplit = plan.nsplit;
  p.split_tiles = plan.tiles;
  p.heads_per_block = plan.heads_per_block;
  if (plan.nsplit < 2) return 0;
  if (workspace_bytes < prefill_workspace(plan, p.B, p.T, p.H, D)) return set_error("workspace too small");
  const size_t slots = (size_t)plan.nsplit * p.B * p.H * p.T;
  p.ws_ml = static_cast<float2*>(workspace);
  p.ws_o = reinterpret_cast<float*>(static_cast<char*>(workspace) + (slots * sizeof(float2) + 255) / 256 * 256);
  return 0;
}

static int prefill_call(int dtype, int B, int T, int H, int K, int D, const void* q, int64_t sqb,
                        int64_t sqh, int64_t sqt, const float* q_weight, float eps, int flags,
                        const float* cos, const float* sin, int64_t s_cos_t, const void* k,
                        const void* v, int64_t skb, int64_t skh, int64_t sks, int64_t offset,
                        int window, float scale, void* out, int64_t sob, int64_t sot, int64_t soh,
                        const int32_t* doc_lo, int64_t sdb, void* workspace, size_t workspace_bytes,
                        void* stream) {
  if (dtype != FORGE_BF16 && dtype != FORGE_F16)
    return set_error("forge_attn_prefill: dtype must be bf16 or fp16 (use forge_attn_decode)");
  if (D != 64 && D != 128 && D != 256 && D != 512)
    return set_error("forge_attn_prefill: head dim must be 64, 128, 256 or 512");
  PrefillParams p;
  int st = prefill_setup(p, 2, B, T, H, K, q, sqb, sqh, sqt, q_weight, eps, flags, cos, sin, s_cos_t, k, v, skb,
                         skh, sks, offset, window, scale, out, sob, sot, soh);
  if (st) return st;
  p.doc_lo = doc_lo;
  p.sdb = sdb;
  st = prefill_bind(p, prefill_plan(false, B, T, H, K, D, offset, window, workspace && !doc_lo ? kMaxParts : 1), D,
                    workspace, workspace_bytes);
  if (st) return st;
  hipStream_t s = (hipStream_t)stream;
  return dtype == FORGE_BF16 ? launch_prefill<bf16>(p, D, s) : launch_prefill<f16>(p, D, s);
}

extern "C" int forge_attn_prefill(int dtype, int B, int T, int H, int K, int D, const void* q,
                                  int64_t sqb, int64_t sqh, int64_t sqt, const float* q_weight,
                                  float eps, int flags, const float* cos, const float* sin,
                                  int64_t s_cos_t, const void* k, const void* v, int64_t skb,
                                  int64_t skh, int64_t sks, int64_t offset, int window,
                                  float scale, void* out, int64_t sob, int64_t sot, int64_t soh,
                                  void* stream) {
  clear_error();
  return prefill_call(dtype, B, T, H, K, D, q, sqb, sqh, sqt, q_weight, eps, flags, cos, sin,
                      s_cos_t, k, v, skb, skh, sks, offset, window, scale, out, sob, sot, soh,
                      nullptr, 0, nullptr, 0, stream);
}

extern "C" int forge_attn_prefill_docs(int dtype, int B, int T, int H, int K, int D,
                                       const void* q, int64_t sqb, int64_t sqh, int64_t sqt,
                                       const float* q_weight, float eps, int flags,
                                       const float* cos, const float* sin, int64_t s_cos_t,
                                       const void* k, const void* v, int64_t skb, int64_t skh,
                                       int64_t sks, int64_t offset, int window, float scale,
                                       const int32_t* doc_start, int64_t s_doc_b, void* out,
                                       int64_t sob, int64_t sot, int64_t soh, void* stream) {
  clear_error();
  if (!doc_start) return set_error("forge_attn_prefill_docs: doc_start is null");
  if ((uintptr_t)doc_start % 4) return set_error("forge_attn_prefill_docs: doc_start must be 4-byte aligned");
  return prefill_call(dtype, B, T, H, K, D, q, sqb, sqh, sqt, q_weight, eps, flags, cos, sin,
                      s_cos_t, k, v, skb, skh, sks, offset, window, scale, out, sob, sot, soh,
                      doc_start, s_doc_b, nullptr, 0, stream);
}

extern "C" size_t forge_attn_prefill_workspace_bytes(int dtype, int B, int T, int H, int K, int D,
                                                     int64_t offset, int window) {
  if ((dtype != FORGE_BF16 && dtype != FORGE_F16) || (D != 64 && D != 128 && D != 256 && D != 512) || B <= 0 ||
      T <= 0 || H <= 0 || K <= 0 || H % K || offset < 0 || window < 0 || !positions_fit(offset, T))
    return 0;
  const PrefillPlan plan = prefill_plan(false, B, T, H, K, D, offset, window, kMaxParts);
  return plan.nsplit > 1 ? prefill_workspace(plan, B, T, H, D) : 0;
}

extern "C" int forge_attn_prefill_ws(int dtype, int B, int T, int H, int K, int D, const void* q, int64_t sqb,
                                     int64_t sqh, int64_t sqt, const float* q_weight, float eps, int flags,
                                     const float* cos, const float* sin, int64_t s_cos_t, const void* k,
                                     const void* v, int64_t skb, int64_t skh, int64_t sks, int64_t offset,
                                     int window, float scale, const int32_t* doc_start, int64_t s_doc_b,
                                     void* out, int64_t sob, int64_t sot, int64_t soh, void* workspace,
                                     size_t workspace_bytes, void* stream) {
  clear_error();
  if ((uintptr_t)doc_start % 4) return set_error("forge_attn_prefill_ws: doc_start must be 4-byte aligned");
  if ((uintptr_t)workspace % 16) return set_error("forge_attn_prefill_ws: the workspace must be 16-byte aligned");
  return prefill_call(dtype, B, T, H, K, D, q, sqb, sqh, sqt, q_weight, eps, flags, cos, sin,
                      s_cos_t, k, v, skb, skh, sks, offset, window, scale, out, sob, sot, soh,
                      doc_start, s_doc_b, workspace, workspace_bytes, stream);
}

extern "C" size_t forge_attn_prefill_f32_workspace_bytes(int B, int T, int H, int K, int D, int64_t offset,
                                                         int window) {
  if ((D != 32 && D != 64 && D != 128) || B <= 0 || T <= 0 || H <= 0 || K <= 0 || H % K || offset < 0 ||
      window < 0 || !positions_fit(offset, T))
    return 0;
  const PrefillPlan plan = prefill_plan(true, B, T, H, K, D, offset, window, kMaxParts);
  return plan.nsplit > 1 ? prefill_workspace(plan, B, T, H, D) : 0;
}

extern "C" int forge_attn_prefill_f32(int B, int T, int H, int K, int D, const void* q, int64_t sqb, int64_t sqh,
                                      int64_t sqt, const float* q_weight, float eps, int flags,
                                      const float* cos, const float* sin, int64_t s_cos_t, const void* k,
                                      const void* v, int64_t skb, int64_t skh, int64_t sks, int64_t offset,
                                      int window, float scale, void* out, int64_t sob, int64_t sot,
                                      int64_t soh, void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  if (D != 32 && D != 64 && D != 128) return set_error("forge_attn_prefill_f32: head dim must be 32, 64 or 128");
  if ((uintptr_t)workspace % 16) return set_error("forge_attn_prefill_f32: the workspace must be 16-byte aligned");
  PrefillParams p;
  int st = prefill_setup(p, 4, B, T, H, K, q, sqb, sqh, sqt, q_weight, eps, flags, cos, sin, s_cos_t, k, v, skb,
                         skh, sks, offset, window, scale, out, sob, sot, soh);
  if (st) return st;
  if (sks < D || sks * 4 * (offset + T + 256) >= (1LL << 31))
    return set_error("forge_attn_prefill_f32: one (batch, kv head) slab of keys must span < 2^31 bytes");
  st = prefill_bind(p, prefill_plan(true, B, T, H, K, D, offset, window, workspace ? kMaxParts : 1), D, workspace,
                    workspace_bytes);
  if (st) return st;
  hipStream_t s = (hipStream_t)stream;
  return D == 32 ? launch_prefill_f32<32>(p, s) : D == 64 ? launch_prefill_f32<64>(p, s) : launch_prefill_f32<128>(p, s);
}
