// FP32 kernels of the encoder-side seam and the original-precision decoder
// projections: linear projections y = x W^T + b (optionally ReLU), and
// non-causal multi-head attention.
//
// These paths have no bit-exact counterpart: the reference's CPU kernels
// already differ in float order between paths (TensorMath.cs:79-200: packed
// AVX/FMA for 16+ frames, FloatRows4Avx below 4, a generic row loop), and
// its device backend checks against a tolerance (2e-4 relative for linear
// projections, 5e-5 for attention, tools/FunAsrNet.Benchmarks
// FloatGpuChecks.cs, AttentionGpuChecks.cs). What is exact here is what the
// reference's checks require to be exact: a projection gives the same bits
// alone, in a group, or as either half of a ReLU chain (one kernel, one
// order per shape).
#include "fah_device.h"
#include "fah_internal.h"

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

namespace fah {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
// Four floats in one load from any float: frames may start anywhere.
typedef float floatx4_any __attribute__((ext_vector_type(4), aligned(4)));

// ---- GEMM: FP32 products on the bf16 matrix cores --------------------------------
// out[f][n] = sum_k x[f][k] * w[n][k] (+ bias[n]) (ReLU), any M (frames), N, K.
//
// What bounds it: fp32 MFMA does 256 flop a cycle and CU, bf16 MFMA 4,096.
// Every fp32 value is the exact sum of three bf16 values (each the rest
// rounded to nearest: 8 + 8 + 8 significand bits), so a product of two is the
// sum of nine bf16 products that fp32 holds exactly; the six largest are
// formed (a0 b0, a0 b1, a1 b0, a1 b1, a0 b2, a2 b0), the other three are below
// 2^-25 of the product, half an ulp of its fp32 rounding. Six bf16 MFMAs of 16
// k take 6 x 32 cycles for a 32 x 32 tile where fp32 ones take 4 x 4 x 32, and
// round the sum six times for 16 k instead of sixteen times.
//
// Layout: a workgroup of WN x KS waves takes 32 TI frames and 32 TJ WN rows in
// v_mfma_f32_32x32x16_bf16 tiles, each wave all the frames and 32 TJ rows, K in
// tiles of 32 KB k of which wave group ks takes the 16-k steps ks HS .. ks HS +
// HS - 1; the groups' sums are added in LDS in order. The weight's planes were
// laid out at upload in the lanes' own order, so a wave reads its operands
// straight from memory, 1 KB at a time (through LDS they took 22.8 us where
// this takes 20.4 for 1000 x 512 -> 2048: LDS reads, then L1 fills of half
// lines). A thread loads 8 k of a frame (32 bytes), splits them and writes 16
// bytes to each of three LDS planes, in the shadow of the previous tile's MFMAs;
// 16-byte chunks are placed so that the rows of an operand read and of a write
// fall on distinct banks (SQ_LDS_BANK_CONFLICT 0). Two LDS buffers, one barrier
// a tile. Results leave by non-temporal stores (18.3 -> 17.6 us: the write-back
// at the kernel's end shortens). Operand lane layout: row l % 32, k 8 (l / 32)
// .. + 7; result register r of lane l: row 8 (r / 4) + 4 (l / 32) + r % 4,
// column l % 32.
//
// Measured against the fp32 MFMA kernel for all weights (fp32 sums of 64 x 64 tiles),
// us: 1000 x 512 -> 2048 25.4 -> 18.6, 333 x 560 -> 1536 17.2 -> 11.5, 4000 x
// 2048 -> 512 85 -> 52, 300 x 1023 -> 700 77 -> 18; error against 64 bits
// (2-norm) 4.0e-7 -> 0.97e-7, 4.2e-7 -> 1.0e-7, 8.1e-7 -> 1.9e-7, 5.7e-7 ->
// 1.0e-7. Of the 18.6, the MFMAs take 6.2 (at the 2.0 GHz seen), the 8 MB of
// stores 3, the launch, first loads and epilogue the rest.
//
// Range: a weight is split only if its values, but zeros, lie in [kSplitTiny,
// kSplitMost] in magnitude, so that its planes hold each exactly, and no row but
// a zero one lies below kSplitRowLeast (checked once, at upload). What bf16 planes
// cannot hold of a frame is then below 2^-126 2^20 K in a sum. Frames with
// infinities, NaN or values that round past the largest bf16 make sums infinite
// or NaN; a workgroup that finds such a sum, one below kSplitLow, or zeros and
// frames with values below kSplitTiny, forms its tile again on fp32 MFMA (tile_f32).
// Other weights run on the fp32 MFMA kernels below.
constexpr uint32_t kSplitLow = 0x1c800000u;      // 2^-70
constexpr uint32_t kSplitTiny = 0x0d800000u;     // 2^-100
constexpr uint32_t kSplitMost = 0x49800000u;     // 2^20
constexpr uint32_t kSplitRowLeast = 0x17800000u; // 2^-80

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  const floatx2 v = {a, b};
  uint32_t r = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  asm("" : "+v"(r));  // (one conversion: the halves are taken from the packed word)
  return r;
}

// Eight floats as three planes of eight bf16. `low`: what lies below each, added
// to what the first two planes leave.
__device__ __forceinline__ void split8(const float* v, uint4* p, const float* low = nullptr) {
  uint32_t w[3][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = v[2 * i], b = v[2 * i + 1];
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      const uint32_t h = pack_bf16(a, b);
      w[s][i] = h;
      if (s < 2) {
        a -= u2f(h << 16);
        b -= u2f(h & 0xffff0000u);
      }
      if (s == 1 && low) {
        a += low[2 * i];
        b += low[2 * i + 1];
      }
    }
  }
#pragma unroll
  for (int s = 0; s < 3; ++s) p[s] = make_uint4(w[s][0], w[s][1], w[s][2], w[s][3]);
}

// Planes of a weight, in the order the GEMM's lanes hold them: for each 32
// rows and 16 k a fragment of [plane 3][lane 64] 16-byte pieces, lane l holding
// row l % 32, k 8 (l / 32) .. + 7. Rows are padded to 32 with the last one (no zero
// sums that the matrix does not have), k with zeros to 128.
__host__ __device__ inline int split_k16(int K) { return ((K + 127) & ~127) / 16; }
__host__ __device__ inline int64_t split_pieces(int64_t rows, int K) { return (rows + 31) / 32 * split_k16(K) * 192; }

__global__ __launch_bounds__(256) void f32_split_planes_kernel(const float* __restrict__ w, int64_t rows, int K,
                                                               uint4* __restrict__ planes) {
  const int64_t fragments = (rows + 31) / 32 * split_k16(K), total = fragments * 64;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int lane = (int)(i & 63);
    const int64_t fragment = i >> 6, r = min(fragment / split_k16(K) * 32 + (lane & 31), rows - 1);
    const int k = (int)(fragment % split_k16(K)) * 16 + 8 * (lane >> 5);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = k + e < K ? w[r * K + k + e] : 0.0f;
    uint4 p[3];
    split8(v, p);
#pragma unroll
    for (int s = 0; s < 3; ++s) planes[fragment * 192 + 64 * s + lane] = p[s];
  }
}

// Sets *outside for a weight that is not to be split (one wave a row).
__global__ __launch_bounds__(256) void f32_split_range_kernel(const float* __restrict__ w, int64_t rows, int K,
                                                              int* outside) {
  const int lane = threadIdx.x & 63;
  for (int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); r < rows; r += (int64_t)gridDim.x * 4) {
    uint32_t most = 0u, least = 0xffffffffu;  // magnitudes; magnitudes less one (zero wraps)
    for (int k = lane; k < K; k += 64) {
      const uint32_t m = f2u(w[r * K + k]) & 0x7fffffffu;
      most = max(most, m);
      least = min(least, m - 1u);
    }
    if (least < kSplitTiny - 1u) *outside = 1;
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) most = max(most, (uint32_t)__shfl_xor((int)most, m, 64));
    if (lane == 0 && (most > kSplitMost || (most != 0u && most < kSplitRowLeast))) *outside = 1;
  }
}

// Eight k of a row from k on, clamped into the row: what lies past K meets the
// weight planes' zeros. VEC: K % 4 == 0.
template <bool VEC>
__device__ __forceinline__ void load8(const float* row, int k, int K, float* v) {
  if (VEC) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const floatx4 q = *reinterpret_cast<const floatx4_any*>(row + min(k + 4 * h, K - 4));
      v[4 * h] = q.x;
      v[4 * h + 1] = q.y;
      v[4 * h + 2] = q.z;
      v[4 * h + 3] = q.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = row[min(k + i, K - 1)];
  }
}

__device__ __forceinline__ void store_linear(float v, const float* bias, float* out, int f, int n, int M, int N,
                                             bool relu) {
  if (f < M && n < N) {
    v = v + (bias ? bias[n] : 0.0f);
    if (relu) v = v < 0.0f ? 0.0f : v;
    out[(size_t)f * N + n] = v;
  }
}

// A TM x TN tile on fp32 MFMA: K in steps of 32 staged in LDS, the next step's
// loads in registers meanwhile (one NaN in 1000 x 512 -> 2048 39 us, 89 with 4-byte
// loads where they are used; in 4000 x 2048 -> 512 140 and 455; the fp32 GEMM for
// all tiles 25 and 85); wave w takes the 16 x 16 blocks w, w + WAVES, ...
// Lane layout of 16x16x4: A[i][k] from lane i + 16k, B[k][j] from lane j + 16k,
// D[4q + r][j] in lane j + 16q. VEC: K % 4 == 0.
template <int TM, int TN, int WAVES, bool VEC>
__device__ __forceinline__ void tile_f32(char* smem, const float* x, const float* w, const float* bias, float* out, int M,
                                      int N, int K, int f0, int n0, bool relu) {
  constexpr int PAD = 33, BLOCKS = (TM / 16) * (TN / 16), PER = BLOCKS / WAVES, NT = 64 * WAVES, PIECES = (TM + TN) * 8 / NT;
  static_assert(BLOCKS % WAVES == 0 && PIECES * NT == (TM + TN) * 8, "whole blocks a wave, whole pieces a thread");
  float* s = reinterpret_cast<float*>(smem);  // [TM + TN][PAD]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, kc = 4 * (tid & 7);
  // Thread t takes 4 k of every NT / 8th row from t / 8 on; rows past the end
  // repeat the last one (never stored), k past the end become zeros in LDS.
  float v[PIECES][4];
  auto fetch = [&](int k) {
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      const int r = (tid + NT * p) >> 3;
      const float* row = r < TM ? x + (size_t)min(f0 + r, M - 1) * K : w + (size_t)min(n0 + r - TM, N - 1) * K;
      if (VEC) {
        const floatx4 q = *reinterpret_cast<const floatx4_any*>(row + min(k, K - 4));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[p][e] = q[e];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[p][e] = row[min(k + e, K - 1)];
      }
    }
  };
  floatx4 acc[PER];
#pragma unroll
  for (int b = 0; b < PER; ++b) acc[b] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  fetch(kc);
  for (int k0 = 0; k0 < K; k0 += 32) {
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PIECES; ++p)
#pragma unroll
      for (int e = 0; e < 4; ++e) s[((tid + NT * p) >> 3) * PAD + kc + e] = k0 + kc + e < K ? v[p][e] : 0.0f;
    __syncthreads();
    fetch(k0 + 32 + kc);
#pragma unroll
    for (int ks = 0; ks < 32; ks += 4) {
      const int kk = ks + (lane >> 4);
#pragma unroll
      for (int b = 0; b < PER; ++b) {
        const int blk = wave + WAVES * b, bi = blk % (TM / 16), bj = blk / (TM / 16);
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(s[(16 * bi + (lane & 15)) * PAD + kk],
                                                      s[(TM + 16 * bj + (lane & 15)) * PAD + kk], acc[b], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int b = 0; b < PER; ++b) {
    const int blk = wave + WAVES * b, bi = blk % (TM / 16), bj = blk / (TM / 16);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      store_linear(acc[b][r], bias, out, f0 + 16 * bi + 4 * (lane >> 4) + r, n0 + 16 * bj + (lane & 15), M, N, relu);
  }
}

// 16-byte slot of chunk c of row r in a plane of rows of CH chunks (4 or 8).
template <int CH>
__device__ __forceinline__ int split_slot(int row, int chunk) {
  const int swz = CH == 8 ? row & 7 : ((row >> 1) & 3) ^ ((row >> 3) & 1);
  return (row * CH + (chunk ^ swz)) * 16;
}

template <int WN, int KS, int TI, int TJ, int KB, int D, bool VEC>
__global__ __launch_bounds__(64 * WN * KS) void f32_split_gemm_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const uint4* __restrict__ planes,
    const float* __restrict__ bias, float* __restrict__ out, int M, int N, int K, int relu) {
  constexpr int TM = 32 * TI, TN = 32 * TJ * WN, WAVES = WN * KS, NT = 64 * WAVES, KT = 32 * KB;
  constexpr int CH = KT / 8, PLANE = TM * KT * 2, BUF = 3 * PLANE, UA = TM * CH / NT, HS = 2 * KB / KS;
  static_assert(D % 2 == 0 && 128 % (D * KT) == 0, "two LDS buffers; planes padded to whole groups of D tiles");
  static_assert(UA >= 1 && UA * NT == TM * CH && HS * KS == 2 * KB, "whole units a thread, whole 16-k steps a wave");
  constexpr int kReduce = (KS - 1) * WN * TI * TJ * 4096;  // partial tiles of the other wave groups
  constexpr int kFallback = (TM + TN) * 33 * 4;
  constexpr int kMax = kReduce > kFallback ? kReduce : kFallback, kLds = 2 * BUF > kMax ? 2 * BUF : kMax;
  __shared__ __attribute__((aligned(16))) char smem[kLds];
  __shared__ int unsure_s;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, lk = lane >> 5;
  const int ks = wave / WN, wn = wave % WN;
  // Workgroups are dealt to the eight XCDs in turn: each XCD takes a run of
  // consecutive tiles, frames fastest, so that its L2 holds few weight rows.
  const int mt = (M + TM - 1) / TM, tiles = gridDim.x, xcd = blockIdx.x & 7, q8 = tiles >> 3, r8 = tiles & 7;
  const int tile = xcd * q8 + min(xcd, r8) + (blockIdx.x >> 3);
  const int f0 = (tile % mt) * TM, n0 = (tile / mt) * TN;
  auto split_tile = [&]() -> bool {
    // Frames past the end repeat the last one, row blocks past the end the
    // last block (neither is stored).
    const float* asrc[UA];
    int aat[UA];
#pragma unroll
    for (int u = 0; u < UA; ++u) {
      const int unit = tid + NT * u, row = unit / CH;
      asrc[u] = x + (size_t)min(f0 + row, M - 1) * K;
      aat[u] = split_slot<CH>(row, unit % CH);
    }
    const int k16 = split_k16(K), steps = (K + D * KT - 1) / (D * KT) * D, kc = 8 * (tid % CH);
    const uint4* bsrc[TJ];
#pragma unroll
    for (int j = 0; j < TJ; ++j)
      bsrc[j] = planes + ((size_t)min(n0 / 32 + TJ * wn + j, (N - 1) / 32) * k16 + ks * HS) * 192 + lane;
    struct Regs {
      float a[UA][8];
      uint4 b[TJ][HS][3];
    } r[D];
    auto fetch_a = [&](Regs& r, int t) {
      t = min(t, steps - 1);
#pragma unroll
      for (int u = 0; u < UA; ++u) load8<VEC>(asrc[u], KT * t + kc, K, r.a[u]);
    };
    auto fetch_b = [&](Regs& r, int t) {
      t = min(t, steps - 1);
#pragma unroll
      for (int j = 0; j < TJ; ++j)
#pragma unroll
        for (int h = 0; h < HS; ++h)
#pragma unroll
          for (int s = 0; s < 3; ++s) r.b[j][h][s] = bsrc[j][(size_t)(2 * KB * t + h) * 192 + 64 * s];
    };
    auto stage = [&](Regs& r, int buf) {
#pragma unroll
      for (int u = 0; u < UA; ++u) {
        uint4 p[3];
        split8(r.a[u], p);
#pragma unroll
        for (int s = 0; s < 3; ++s) *reinterpret_cast<uint4*>(smem + buf * BUF + s * PLANE + aat[u]) = p[s];
      }
    };
    // The large products a0 b0 and the five corrections have sums of their own:
    // the first is rounded once for 16 k, the others are small.
    floatx16 acc[TI][TJ], rest[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) acc[i][j] = rest[i][j] = floatx16{};
    struct Frags {
      bf16x8 a[TI][3];
    } g0, g1;
    auto read = [&](Frags& g, int buf, int h) {
      const char* base = smem + buf * BUF;
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int s = 0; s < 3; ++s)
          g.a[i][s] = *reinterpret_cast<const bf16x8*>(base + s * PLANE +
                                                       split_slot<CH>(32 * i + l32, 2 * (ks * HS + h) + lk));
    };
    auto multiply = [&](Frags& g, Regs& r, int h) {
      constexpr int pa[6] = {2, 0, 1, 0, 1, 0}, pb[6] = {0, 2, 1, 0, 0, 1};
#pragma unroll
      for (int p = 0; p < 6; ++p)
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int j = 0; j < TJ; ++j) {
            floatx16& sum = p == 3 ? acc[i][j] : rest[i][j];
            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(g.a[i][pa[p]], __builtin_bit_cast(bf16x8, r.b[j][h][pb[p]]), sum, 0,
                                                          0, 0);
          }
    };
    // The weights of tiles t + 1 .. t + D - 1 and the frames of tiles t + 2 .. t + D
    // are in registers or on their way while tile t is multiplied (four tiles
    // measured like two). Tiles past the end meet the weight planes' zeros.
    auto step = [&](Regs& cur, Regs& next, int t, int buf) {
      read(g0, buf, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < HS; ++h) {
        Frags& g = h & 1 ? g1 : g0;
        Frags& o = h & 1 ? g0 : g1;
        if (h + 1 < HS) read(o, buf, h + 1);
        __builtin_amdgcn_sched_barrier(0);
        if (h == 0) stage(next, buf ^ 1);
        if (h == HS - 1) fetch_a(next, t + 1 + D);
        multiply(g, cur, h);
        if (h == 0) {
#pragma unroll
          for (int i = 0; i < 6 * TI * TJ; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, (44 * UA + 6 * TI * TJ - 1) / (6 * TI * TJ), 0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      fetch_b(cur, t + D);
      lds_barrier();
    };
#pragma unroll
    for (int d = 0; d < D; ++d) {
      fetch_a(r[d], d);
      fetch_b(r[d], d);
    }
    stage(r[0], 0);
    fetch_a(r[0], D);
    if (tid == 0) unsure_s = 0;
    lds_barrier();
    for (int t = 0; t < steps; t += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) step(r[d], r[(d + 1) % D], t + d, d & 1);
    }
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] += rest[i][j][e];
    if (KS > 1) {
      // (The loop's last barrier is past every read of the staging buffers.)
      float* part = reinterpret_cast<float*>(smem) + (size_t)wn * TI * TJ * 1024 + lane;
      constexpr size_t kGroup = (size_t)WN * TI * TJ * 1024;
      if (ks > 0) {
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) part[(ks - 1) * kGroup + (i * TJ + j) * 1024 + r * 64] = acc[i][j][r];
      }
      lds_barrier();
      if (ks == 0) {
#pragma unroll
        for (int g = 0; g < KS - 1; ++g)
#pragma unroll
          for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j)
#pragma unroll
              for (int r = 0; r < 16; ++r) acc[i][j][r] += part[g * kGroup + (i * TJ + j) * 1024 + r * 64];
      }
    }
    // Magnitudes less one (zero wraps): the largest and the smallest.
    uint32_t most = 0u, least = 0xffffffffu;
    if (ks == 0) {
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const uint32_t m = (f2u(acc[i][j][e]) & 0x7fffffffu) - 1u;
            most = max(most, m);
            least = min(least, m);
          }
    }
    if (most >= 0x7f7fffffu || least < kSplitLow - 1u) unsure_s = 1;
    lds_barrier();
    if (unsure_s) {
      bool odd = least < kSplitLow - 1u;
      if (ks == 0) {
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) odd = odd || (f2u(acc[i][j][e]) & 0x7fffffffu) >= 0x7f800000u;
      }
      if (__syncthreads_or(odd)) return false;
      // Sums of zero (those of zero frames, as a padded batch has) are right unless
      // frames held values too small for the planes: magnitudes less one again, a
      // wave's TM / WAVES frames together. Half of 4000 x 2048 -> 512 zeros 63 us
      // (137 with one load at a time), of 1000 x 512 -> 512 10.6 (20).
      constexpr int FW = TM / WAVES, W = VEC ? 4 : 1;
      uint32_t tiny = 0xffffffffu;
#pragma unroll 1
      for (int k = W * lane; k < K; k += 64 * W) {
        float v[FW][W];
#pragma unroll
        for (int r = 0; r < FW; ++r) {
          const float* row = x + (size_t)min(f0 + FW * wave + r, M - 1) * K + k;
          if (VEC) {
            const floatx4 q = *reinterpret_cast<const floatx4_any*>(row);
#pragma unroll
            for (int e = 0; e < W; ++e) v[r][e] = q[e];
          } else {
            v[r][0] = *row;
          }
        }
#pragma unroll
        for (int r = 0; r < FW; ++r)
#pragma unroll
          for (int e = 0; e < W; ++e) tiny = min(tiny, (f2u(v[r][e]) & 0x7fffffffu) - 1u);
      }
      odd = tiny < kSplitTiny - 1u;
      if (__syncthreads_or(odd)) return false;
    }
    if (ks == 0) {
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const int n = n0 + 32 * (TJ * wn + j) + l32;
        if (n >= N) continue;
        const float b = bias ? bias[n] : 0.0f;
        float* o = out + (size_t)(f0 + 4 * lk) * N + n;
        const bool whole = f0 + TM <= M;
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int row = 32 * i + 8 * (r >> 2) + (r & 3);
            float v = acc[i][j][r] + b;
            if (relu) v = v < 0.0f ? 0.0f : v;  // (-0 and NaN pass, as the reference's `v < 0 ? 0 : v`)
            if (whole || f0 + 4 * lk + row < M) __builtin_nontemporal_store(v, o + (size_t)row * N);
          }
      }
    }
    return true;
  };
  if (!split_tile()) tile_f32<TM, TN, WAVES, VEC>(smem, x, w, bias, out, M, N, K, f0, n0, relu);
}

// ---- GEMM on fp32 MFMA: weights that the planes do not hold -----------------------
// out[f][n] = sum_k x[f][k] * w[n][k] (+ bias[n]) (ReLU), any M (frames), N,
// K with K % 4 == 0. Four waves in a 2 x 2 grid,
// each a (16 BI) x (16 BJ) tile of v_mfma_f32_16x16x4f32 blocks; workgroup
// tile (32 BI) x (32 BJ); K in tiles of GK staged in two LDS buffers as
// row-major [row][GK + 4] (16-byte loads and stores; the next tile's global
// loads sit in registers while the current one is multiplied, then go to
// the other buffer, one barrier per tile). Lane layout of 16x16x4: A[i][k]
// from lane i + 16k, B[k][j] from lane j + 16k, D[4q + r][j] in lane j + 16q
// (r < 4). In substep s of a K tile, lane group q multiplies k =
// (GK / 4) q + s, so each lane reads its GK / 4 values of a row as 16-byte
// LDS reads. One order per shape: the same bits whichever entry point runs it.
constexpr int kGK = 64;

template <int BI, int BJ, bool RELU>
__global__ __launch_bounds__(256) void f32_gemm_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                       const float* __restrict__ bias, float* __restrict__ out, int M,
                                                       int N, int K) {
  constexpr int TM = 32 * BI, TN = 32 * BJ;              // workgroup tile
  constexpr int ROW = kGK + 4, KQ = kGK / 4;              // LDS row (floats); k values per lane group
  constexpr int PER_ROW = kGK / 4, ROWS = 256 / PER_ROW;  // 16-byte loads per row; rows per pass
  constexpr int LA = TM / ROWS, LB = TN / ROWS;           // 16-byte loads per thread and operand
  static_assert(LA >= 1 && LB >= 1 && TM % ROWS == 0 && TN % ROWS == 0, "whole load passes");
  __shared__ __attribute__((aligned(16))) float a_s[2][TM * ROW];
  __shared__ __attribute__((aligned(16))) float b_s[2][TN * ROW];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int f0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  const int wm = (wave >> 1) * 16 * BI, wn = (wave & 1) * 16 * BJ;
  const int li = lane & 15, lq = lane >> 4;
  floatx4 acc[BI][BJ];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  // Global loads: thread t takes row t / PER_ROW (+ ROWS per further load),
  // the 16 bytes at k = 4 (t % PER_ROW) of the tile; rows past the edge and
  // k past K read as zero.
  const int lr = tid / PER_ROW, lc = 4 * (tid % PER_ROW);
  floatx4 ra[LA];
  float4 rb[LB];
  auto fetch = [&](int k0) {
    const int k = k0 + lc;
#pragma unroll
    for (int u = 0; u < LA; ++u) {
      const int f = f0 + lr + ROWS * u;
      ra[u] = (f < M && k < K) ? floatx4(*reinterpret_cast<const floatx4_any*>(x + (size_t)f * K + k)) : floatx4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < LB; ++u) {
      const int n = n0 + lr + ROWS * u;
      rb[u] = (n < N && k < K) ? *reinterpret_cast<const float4*>(w + (size_t)n * K + k) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int u = 0; u < LA; ++u) *reinterpret_cast<floatx4*>(&a_s[buf][(lr + ROWS * u) * ROW + lc]) = ra[u];
#pragma unroll
    for (int u = 0; u < LB; ++u) *reinterpret_cast<float4*>(&b_s[buf][(lr + ROWS * u) * ROW + lc]) = rb[u];
  };
  fetch(0);
  stage(0);
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < K; k0 += kGK) {
    const bool more = k0 + kGK < K;
    if (more) fetch(k0 + kGK);
#pragma unroll
    for (int h = 0; h < KQ / 4; ++h) {
      float4 av[BI], bv[BJ];
#pragma unroll
      for (int i = 0; i < BI; ++i)
        av[i] = *reinterpret_cast<const float4*>(&a_s[buf][(wm + 16 * i + li) * ROW + KQ * lq + 4 * h]);
#pragma unroll
      for (int j = 0; j < BJ; ++j)
        bv[j] = *reinterpret_cast<const float4*>(&b_s[buf][(wn + 16 * j + li) * ROW + KQ * lq + 4 * h]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < BI; ++i)
#pragma unroll
          for (int j = 0; j < BJ; ++j) {
            const float a = e == 0 ? av[i].x : e == 1 ? av[i].y : e == 2 ? av[i].z : av[i].w;
            const float b = e == 0 ? bv[j].x : e == 1 ? bv[j].y : e == 2 ? bv[j].z : bv[j].w;
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc[i][j], 0, 0, 0);
          }
    }
    if (more) {
      stage(buf ^ 1);
      __syncthreads();
      buf ^= 1;
    }
  }
#pragma unroll
  for (int j = 0; j < BJ; ++j) {
    const int n = n0 + wn + 16 * j + li;
    if (n >= N) continue;
    const float b = bias ? bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int f = f0 + wm + 16 * i + 4 * lq + r;
        if (f < M) {
          float v = acc[i][j][r] + b;
          if (RELU) v = v < 0.0f ? 0.0f : v;  // (-0 and NaN pass, as the reference's `v < 0 ? 0 : v`)
          out[(size_t)f * N + n] = v;
        }
      }
  }
}

// The same product for grids of at most one workgroup per CU: each of the
// four waves covers the whole 32 x 64 tile (2 x 4 blocks, eight
// accumulators in flight) over its quarter of every K tile (lane group q of
// wave w takes k = 16 w + 4 q .. + 3), and the four partial tiles are added
// in wave order in LDS at the end.
__global__ __launch_bounds__(256) void f32_gemm_wavek_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                             const float* __restrict__ bias, float* __restrict__ out,
                                                             int M, int N, int K, int relu) {
  constexpr int GK = 64, TM = 32, TN = 64, ROW = GK + 4;
  constexpr int PER_ROW = GK / 4, ROWS = 256 / PER_ROW, LA = TM / ROWS, LB = TN / ROWS;
  __shared__ __attribute__((aligned(16))) float a_s[2][TM * ROW];
  __shared__ __attribute__((aligned(16))) float b_s[2][TN * ROW];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int f0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  const int li = lane & 15, lq = lane >> 4;
  floatx4 acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  const int lr = tid / PER_ROW, lc = 4 * (tid % PER_ROW);
  floatx4 ra[LA];
  float4 rb[LB];
  auto fetch = [&](int k0) {
    const int k = k0 + lc;
#pragma unroll
    for (int u = 0; u < LA; ++u) {
      const int f = f0 + lr + ROWS * u;
      ra[u] = (f < M && k < K) ? floatx4(*reinterpret_cast<const floatx4_any*>(x + (size_t)f * K + k)) : floatx4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < LB; ++u) {
      const int n = n0 + lr + ROWS * u;
      rb[u] = (n < N && k < K) ? *reinterpret_cast<const float4*>(w + (size_t)n * K + k) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int u = 0; u < LA; ++u) *reinterpret_cast<floatx4*>(&a_s[buf][(lr + ROWS * u) * ROW + lc]) = ra[u];
#pragma unroll
    for (int u = 0; u < LB; ++u) *reinterpret_cast<float4*>(&b_s[buf][(lr + ROWS * u) * ROW + lc]) = rb[u];
  };
  fetch(0);
  stage(0);
  __syncthreads();
  int buf = 0;
  const int kl = 16 * wave + 4 * lq;
  for (int k0 = 0; k0 < K; k0 += GK) {
    const bool more = k0 + GK < K;
    if (more) fetch(k0 + GK);
    float4 av[2], bv[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) av[i] = *reinterpret_cast<const float4*>(&a_s[buf][(16 * i + li) * ROW + kl]);
#pragma unroll
    for (int j = 0; j < 4; ++j) bv[j] = *reinterpret_cast<const float4*>(&b_s[buf][(16 * j + li) * ROW + kl]);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float a = e == 0 ? av[i].x : e == 1 ? av[i].y : e == 2 ? av[i].z : av[i].w;
          const float b = e == 0 ? bv[j].x : e == 1 ? bv[j].y : e == 2 ? bv[j].z : bv[j].w;
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc[i][j], 0, 0, 0);
        }
    if (more) {
      stage(buf ^ 1);
      __syncthreads();
      buf ^= 1;
    }
  }
  // Partial tiles into LDS (the staging buffers, free once every wave is
  // past its last reads): part[w][f][n], then summed in wave order.
  __syncthreads();
  float* part = &a_s[0][0];
  static_assert(4 * TM * TN <= 2 * TM * ROW + 2 * TN * ROW, "partials fit the staging buffers");
  float* part_b = &b_s[0][0];
  auto slot = [&](int wv, int f, int n) -> float& {
    const int e = (wv * TM + f) * TN + n;
    return e < 2 * TM * ROW ? part[e] : part_b[e - 2 * TM * ROW];
  };
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) slot(wave, 16 * i + 4 * lq + r, 16 * j + li) = acc[i][j][r];
  __syncthreads();
  for (int e = tid; e < TM * TN; e += 256) {
    const int f = e / TN, n = e % TN;
    if (f0 + f >= M || n0 + n >= N) continue;
    float v = ((slot(0, f, n) + slot(1, f, n)) + slot(2, f, n)) + slot(3, f, n);
    v = v + (bias ? bias[n0 + n] : 0.0f);
    if (relu) v = v < 0.0f ? 0.0f : v;
    out[(size_t)(f0 + f) * N + n0 + n] = v;
  }
}

// Any K: 64 x 64 tiles, K in steps of 32 staged in LDS one
// float per thread and row, four waves of 2 x 2 v_mfma_f32_16x16x4f32 blocks.
constexpr int kGT = 64, kGA = 32, kGPad = kGA + 1;

__global__ __launch_bounds__(256) void f32_gemm_any_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                           const float* __restrict__ bias, float* __restrict__ out,
                                                           int M, int N, int K, int relu) {
  __shared__ float a_s[kGT][kGPad];  // frames x k
  __shared__ float b_s[kGT][kGPad];  // rows x k
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int f0 = blockIdx.y * kGT, n0 = blockIdx.x * kGT;
  const int fm = (wave >> 1) * 32, rn = (wave & 1) * 32;
  floatx4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  // Staging: thread t loads rows t / 32 + 8 s (s < 8), column t % 32.
  const int lr = tid >> 5, lc = tid & 31;
  for (int k0 = 0; k0 < K; k0 += kGA) {
    const int k = k0 + lc;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int r = lr + 8 * s;
      const int f = f0 + r, n = n0 + r;
      a_s[r][lc] = (f < M && k < K) ? x[(size_t)f * K + k] : 0.0f;
      b_s[r][lc] = (n < N && k < K) ? w[(size_t)n * K + k] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < kGA; ks += 4) {
      const int kk = ks + (lane >> 4), ii = lane & 15;
      const float a0 = a_s[fm + ii][kk], a1 = a_s[fm + 16 + ii][kk];
      const float b0 = b_s[rn + ii][kk], b1 = b_s[rn + 16 + ii][kk];
      acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b0, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b1, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b0, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b1, acc[1][1], 0, 0, 0);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = n0 + rn + 16 * j + (lane & 15);
      if (n >= N) continue;
      const float b = bias ? bias[n] : 0.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int f = f0 + fm + 16 * i + 4 * (lane >> 4) + r;
        if (f < M) {
          float v = acc[i][j][r] + b;
          if (relu) v = v < 0.0f ? 0.0f : v;
          out[(size_t)f * N + n] = v;
        }
      }
    }
}

// ---- GEMV (few frames, weight-bandwidth bound) ------------------------------
// Each wave takes RW consecutive weight rows at a time, in chunks of 1,024 k (256
// for rows of at most that: four frames of 3 -> 70000 46.5 -> 23.6 us)
// whose loads (E values a lane and row) are all in flight together, with the
// frames' values at the same k straight from the caches: a small launch is one
// round of loads, with no LDS and no barrier before it (the frames staged in LDS
// first, and 256 k a round: one frame of 1024 -> 3072 6.5 us, here 3.9, of 3072
// -> 1024 9.1 and 3.8, both at what a call costs the host; 1024 -> 151936 113 and
// 106, 5.9 TB/s). Then a wave reduction per row and frame. VEC: 16-byte loads (K
// % 4 == 0); frames may start at any float, with the same order of the sum.
template <int MF, int RW, bool VEC, int E>
__global__ __launch_bounds__(256) void f32_gemv_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                       const float* __restrict__ bias, float* __restrict__ out, int M,
                                                       int N, int K, int relu) {
  constexpr int kChunk = 64 * E;
  const int lane = threadIdx.x & 63, waves = gridDim.x * 4;
  // Value e of this lane: k0 + at(e); with `all`, the whole chunk lies in the row.
  auto load = [&](const float* row, int k0, bool all, float* v) {
    if (VEC) {
#pragma unroll
      for (int e = 0; e < E; e += 4) {
        const int k = k0 + 64 * e + 4 * lane;
        const floatx4 q = all || k < K ? floatx4(*reinterpret_cast<const floatx4_any*>(row + k)) : floatx4{0.f, 0.f, 0.f, 0.f};
        v[e] = q.x;
        v[e + 1] = q.y;
        v[e + 2] = q.z;
        v[e + 3] = q.w;
      }
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int k = k0 + 64 * e + lane;
        v[e] = all || k < K ? row[k] : 0.0f;
      }
    }
  };
  for (int n0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * RW; n0 < N; n0 += waves * RW) {
    float acc[RW][MF];
#pragma unroll
    for (int r = 0; r < RW; ++r)
#pragma unroll
      for (int f = 0; f < MF; ++f) acc[r][f] = 0.0f;
    // Rows past N re-read row N - 1 (never stored).
    const float* rows[RW];
#pragma unroll
    for (int r = 0; r < RW; ++r) rows[r] = w + (size_t)min(n0 + r, N - 1) * K;
    float v[RW][E];
    auto chunk = [&](int k0, bool all) {
#pragma unroll
      for (int f = 0; f < MF; ++f) {
        if (MF > 1 && f >= M) break;
        float u[E];
        load(x + (size_t)f * K, k0, all, u);
#pragma unroll
        for (int e = 0; e < E; ++e)
#pragma unroll
          for (int r = 0; r < RW; ++r) acc[r][f] = __builtin_fmaf(v[r][e], u[e], acc[r][f]);
      }
    };
    int k0 = 0;
    for (; k0 + kChunk <= K; k0 += kChunk) {
#pragma unroll
      for (int r = 0; r < RW; ++r) load(rows[r], k0, true, v[r]);
      chunk(k0, true);
    }
    if (k0 < K) {
#pragma unroll
      for (int r = 0; r < RW; ++r) load(rows[r], k0, false, v[r]);
      chunk(k0, false);
    }
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      const int n = n0 + r;
#pragma unroll
      for (int f = 0; f < MF; ++f) {
        if (MF > 1 && f >= M) break;
        float s = acc[r][f];
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
        if (lane == 0 && n < N) {
          float y = s + (bias ? bias[n] : 0.0f);
          if (relu) y = y < 0.0f ? 0.0f : y;
          out[(size_t)f * N + n] = y;
        }
      }
    }
  }
}

// ---- Non-causal multi-head attention ------------------------------------------
// One workgroup per (head, 16 query rows); keys in blocks of 32 staged in
// LDS with their values; online softmax (running maximum, rescaled sums),
// outputs in registers (thread t: rows 4 (t / 64) .. +3, channels t % 64,
// t % 64 + 64, ...).
constexpr int kAQ = 16, kAK = 32, kAMaxS = 256;

__global__ __launch_bounds__(256) void f32_attention_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                            const float* __restrict__ v, float* __restrict__ out,
                                                            int frames, int width, int S, float divisor) {
  __shared__ float q_s[kAQ][kAMaxS + 1];
  __shared__ float k_s[kAK][kAMaxS + 1];
  __shared__ float v_s[kAK][kAMaxS];
  __shared__ float p_s[kAQ][kAK + 1];
  __shared__ float scale_s[kAQ];
  const int tid = threadIdx.x, head = blockIdx.x, t0 = blockIdx.y * kAQ;
  const int hoff = head * S;
  for (int i = tid; i < kAQ * S; i += 256) {
    const int r = i / S, c = i - r * S;
    q_s[r][c] = t0 + r < frames ? q[(size_t)(t0 + r) * width + hoff + c] : 0.0f;
  }
  constexpr int kCh = kAMaxS / 64;  // channel slots per thread
  const int orow = 4 * (tid >> 6), oc = tid & 63;
  float o[4][kCh];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int j = 0; j < kCh; ++j) o[r][j] = 0.0f;
  // Per query row (threads 0..15 keep them): running maximum and sum.
  float run_max = -__builtin_inff(), run_sum = 0.0f;
  for (int s0 = 0; s0 < frames; s0 += kAK) {
    __syncthreads();
    for (int i = tid; i < kAK * S; i += 256) {
      const int r = i / S, c = i - r * S;
      const bool in = s0 + r < frames;
      k_s[r][c] = in ? k[(size_t)(s0 + r) * width + hoff + c] : 0.0f;
      v_s[r][c] = in ? v[(size_t)(s0 + r) * width + hoff + c] : 0.0f;
    }
    __syncthreads();
    // Scores: thread t -> (query row t / 16, keys t % 16 and t % 16 + 16).
    {
      const int qr = tid >> 4, kc = tid & 15;
      float d0 = 0.0f, d1 = 0.0f;
      for (int c = 0; c < S; ++c) {
        const float qv = q_s[qr][c];
        d0 = __builtin_fmaf(qv, k_s[kc][c], d0);
        d1 = __builtin_fmaf(qv, k_s[kc + 16][c], d1);
      }
      p_s[qr][kc] = s0 + kc < frames ? d0 / divisor : -__builtin_inff();
      p_s[qr][kc + 16] = s0 + kc + 16 < frames ? d1 / divisor : -__builtin_inff();
    }
    __syncthreads();
    // Softmax update per query row (16 threads).
    if (tid < kAQ) {
      float m = run_max;
      for (int j = 0; j < kAK; ++j) m = fmaxf(m, p_s[tid][j]);
      // The earlier blocks' sums rescaled to the new maximum (none before
      // the first block).
      const float scale = run_max == -__builtin_inff() ? 0.0f : expf(run_max - m);
      float sum = 0.0f;
      for (int j = 0; j < kAK; ++j) {
        const float e = p_s[tid][j] == -__builtin_inff() ? 0.0f : expf(p_s[tid][j] - m);
        p_s[tid][j] = e;
        sum += e;
      }
      run_sum = run_sum * scale + sum;
      scale_s[tid] = scale;
      run_max = m;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float sc = scale_s[orow + r];
#pragma unroll
      for (int j = 0; j < kCh; ++j) {
        const int c = oc + 64 * j;
        if (c < S) {
          float acc = o[r][j] * sc;
          for (int kk = 0; kk < kAK; ++kk) acc = __builtin_fmaf(p_s[orow + r][kk], v_s[kk][c], acc);
          o[r][j] = acc;
        }
      }
    }
  }
  __syncthreads();
  if (tid < kAQ) scale_s[tid] = 1.0f / run_sum;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int t = t0 + orow + r;
    if (t >= frames) continue;
    const float inv = scale_s[orow + r];
#pragma unroll
    for (int j = 0; j < kCh; ++j) {
      const int c = oc + 64 * j;
      if (c < S) out[(size_t)t * width + hoff + c] = o[r][j] * inv;
    }
  }
}

// ---- Non-causal multi-head attention on fp32 MFMA (head size HS, a multiple of 16) ----
// A workgroup's tile of 16 query rows of a head; wave w takes key blocks (16 keys)
// w, w + 4, ... and keeps its own running maximum, sum and outputs; the four
// partial results are merged in LDS at the end. Per key block the scores
// come transposed, S^T = K Q^T (16 keys x 16 queries, HS / 4 MFMAs with key
// rows and query rows both read as contiguous 16-byte pieces: in substep t
// lane group g multiplies channel g HS/4 + t), so that lane (query j, group
// g) holds the probabilities of keys 4g .. 4g + 3 for query j, which is
// exactly the A operand of P V when substep u takes key 4g + u.
//
// attention_tile_f32 does T such tiles, from query t0 on, with one read of the keys
// and values. AHEAD: the next block's are on their way while a block is multiplied,
// for a workgroup that has a CU to itself. A block's loads are without a branch
// (keys past the end repeat the last one): with one for each row the compiler
// waited for them all before the first product (333 frames of 4 x 128 18.8 ->
// 15.8 us, 500 of 8 x 64 15.9 -> 13.1; the same bits).
constexpr int attention_tile_bytes(int HS) { return (64 * HS + 128) * 4; }

template <int HS, int T, bool AHEAD>
__device__ __forceinline__ void attention_tile_f32(char* smem, const float* __restrict__ q, const float* __restrict__ k,
                                                   const float* __restrict__ v, float* __restrict__ out, int frames,
                                                   int width, float divisor, int head, int t0) {
  constexpr int CB = HS / 16, KQ = HS / 4;  // channel blocks; channels per lane group
  float(*o_s)[16][HS] = reinterpret_cast<float(*)[16][HS]>(smem);
  float(*m_s)[16] = reinterpret_cast<float(*)[16]>(smem + 64 * HS * 4);
  float(*l_s)[16] = m_s + 4;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, j = lane & 15, g = lane >> 4;
  const int hoff = head * HS;
  // This lane's query channels g KQ .. g KQ + KQ - 1 of query t0 + 16 i + j (zero past the end).
  float qv[T][KQ];
#pragma unroll
  for (int i = 0; i < T; ++i) {
    const bool in = t0 + 16 * i + j < frames;
    const float* src = q + (size_t)(t0 + 16 * i + j) * width + hoff + g * KQ;
#pragma unroll
    for (int c = 0; c < KQ; c += 4) {
      const float4 x4 = in ? *reinterpret_cast<const float4*>(src + c) : make_float4(0.f, 0.f, 0.f, 0.f);
      qv[i][c] = x4.x;
      qv[i][c + 1] = x4.y;
      qv[i][c + 2] = x4.z;
      qv[i][c + 3] = x4.w;
    }
  }
  floatx4 o[T][CB];
  float run_m[T], run_l[T];  // of query j
#pragma unroll
  for (int i = 0; i < T; ++i) {
#pragma unroll
    for (int c = 0; c < CB; ++c) o[i][c] = floatx4{0.f, 0.f, 0.f, 0.f};
    run_m[i] = -__builtin_inff();
    run_l[i] = 0.0f;
  }
  const int blocks = (frames + 15) / 16;
  // Keys past the end repeat the last one: their scores are not used, and their
  // values become zero in `outputs`.
  auto load_k = [&](float* b, int kb) {
    const float* src = k + (size_t)min(kb * 16 + j, frames - 1) * width + hoff + g * KQ;
#pragma unroll
    for (int c = 0; c < KQ; c += 4) {
      const float4 x4 = *reinterpret_cast<const float4*>(src + c);
      b[c] = x4.x;
      b[c + 1] = x4.y;
      b[c + 2] = x4.z;
      b[c + 3] = x4.w;
    }
  };
  // Values of keys 4g + u, channel 16c + j.
  auto load_v = [&](float (*b)[4], int kb) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float* src = v + (size_t)min(kb * 16 + 4 * g + u, frames - 1) * width + hoff + j;
#pragma unroll
      for (int c = 0; c < CB; ++c) b[c][u] = src[16 * c];
    }
  };
  // Scores S^T[key 4g + r][query j].
  auto products = [&](const float* b, floatx4* st) {
#pragma unroll
    for (int i = 0; i < T; ++i) st[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < KQ; ++t)
#pragma unroll
      for (int i = 0; i < T; ++i) st[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[t], qv[i][t], st[i], 0, 0, 0);
  };
  float p[T][4], alpha[T];
  auto softmax = [&](const floatx4* st, int kb) {
#pragma unroll
    for (int i = 0; i < T; ++i) {
      float sc[4], bm = -__builtin_inff();
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sc[r] = (kb * 16 + 4 * g + r < frames ? st[i][r] : -__builtin_inff()) / divisor;
        bm = fmaxf(bm, sc[r]);
      }
      bm = fmaxf(bm, __shfl_xor(bm, 16, 64));
      bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
      const float nm = fmaxf(run_m[i], bm);
      float bl = 0.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[i][r] = sc[r] == -__builtin_inff() ? 0.0f : expf(sc[r] - nm);
        bl += p[i][r];
      }
      bl += __shfl_xor(bl, 16, 64);
      bl += __shfl_xor(bl, 32, 64);
      alpha[i] = run_m[i] == -__builtin_inff() ? 0.0f : expf(run_m[i] - nm);
      run_l[i] = run_l[i] * alpha[i] + bl;
      run_m[i] = nm;
    }
  };
  auto outputs = [&](float (*b)[4], int kb) {
    if (kb == blocks - 1) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int c = 0; c < CB; ++c) b[c][u] = kb * 16 + 4 * g + u < frames ? b[c][u] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < T; ++i) {
      // Output rows are queries 4g + r: their rescale factors from lanes 4g + r.
      float ar[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) ar[r] = __shfl(alpha[i], 4 * g + r, 64);
#pragma unroll
      for (int c = 0; c < CB; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[i][c][r] *= ar[r];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int c = 0; c < CB; ++c) o[i][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[i][u], b[c][u], o[i][c], 0, 0, 0);
    }
  };
  const int last = blocks - 1;
  floatx4 st[T];
  float k0[KQ], v0[CB][4];
  load_k(k0, min(wave, last));
  if (AHEAD) {
    float k1[KQ], v1[CB][4];
    load_v(v0, min(wave, last));
    auto step = [&](float* kb0, float (*vb0)[4], float* kb1, float (*vb1)[4], int kb) {
      load_k(kb1, min(kb + 4, last));
      load_v(vb1, min(kb + 4, last));
      __builtin_amdgcn_sched_barrier(0);
      products(kb0, st);
      softmax(st, kb);
      outputs(vb0, kb);
    };
    for (int kb = wave; kb < blocks; kb += 8) {
      step(k0, v0, k1, v1, kb);
      if (kb + 4 < blocks) step(k1, v1, k0, v0, kb + 4);
    }
  } else {
    for (int kb = wave; kb < blocks; kb += 4) {
      products(k0, st);
      load_v(v0, kb);  // (in flight during the softmax)
      load_k(k0, min(kb + 4, last));
      softmax(st, kb);
      outputs(v0, kb);
    }
  }
  // Merge the four waves' partials: out = sum_w e^(m_w - M) O_w / sum_w e^(m_w - M) l_w.
#pragma unroll
  for (int i = 0; i < T; ++i) {
    if (T > 1) __syncthreads();
    if (g == 0) {
      m_s[wave][j] = run_m[i];
      l_s[wave][j] = run_l[i];
    }
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) o_s[wave][4 * g + r][16 * c + j] = o[i][c][r];
    __syncthreads();
    for (int e = tid; e < 16 * HS; e += 256) {
      const int row = e / HS, ch = e % HS, f = t0 + 16 * i + row;
      if (f >= frames) continue;
      float mx = -__builtin_inff();
#pragma unroll
      for (int w2 = 0; w2 < 4; ++w2) mx = fmaxf(mx, m_s[w2][row]);
      float num = 0.0f, den = 0.0f;
#pragma unroll
      for (int w2 = 0; w2 < 4; ++w2) {
        const float x = m_s[w2][row] == -__builtin_inff() ? 0.0f : expf(m_s[w2][row] - mx);
        num += x * o_s[w2][row][ch];
        den += x * l_s[w2][row];
      }
      out[(size_t)f * width + hoff + ch] = num / den;
    }
  }
}

template <int HS>
__global__ __launch_bounds__(256) void f32_attention_mfma_kernel(const float* __restrict__ q,
                                                                 const float* __restrict__ k,
                                                                 const float* __restrict__ v, float* __restrict__ out,
                                                                 int frames, int width, float divisor) {
  __shared__ __attribute__((aligned(16))) char smem[attention_tile_bytes(HS)];
  attention_tile_f32<HS, 1, false>(smem, q, k, v, out, frames, width, divisor, blockIdx.x, blockIdx.y * 16);
}

// ---- Non-causal multi-head attention on the bf16 matrix cores (head size 64, 96, 128) ----
// The products of f32_split_gemm_kernel: q, k, v and the probabilities as three
// bf16 planes each, six products, fp32 sums.
//
// attention_planes_kernel lays the planes out once, in the order the lanes of
// v_mfma_f32_32x32x16_bf16 hold them (fragments of [plane 3][lane 64] 16-byte
// pieces): q and k per 32 rows and 16 channels (lane l: row l % 32, channels
// 8 (l / 32) .. + 7), v per 16 keys and 32 channels (lane l: channel l % 32,
// keys 8 (i / 4) + 4 (l / 32) + i % 4, i < 8). attention_split_kernel, a
// workgroup per (head, 64 queries, share of the keys), runs two waves of 32
// queries over the even key blocks of 32 and two over the odd ones. Scores come
// transposed, S^T = K Q^T, so that lane l holds 16 of a block's scores of query
// l % 32 and lane l ^ 32 the others: the softmax needs one exchange a block.
// Exponentials of them are, as they lie, the B operand of O^T = V^T P^T in the
// key order above, and the outputs of a lane are its query's. The planes of q
// hold q log2(e) / sqrt(HS), so that scores are exponents as they are summed and
// the running maximum is one of them: the exponent of the largest is 0 (of a
// maximum that was scaled and rounded it would be the rounding error, past 128
// from 2^32 on). The running maximum moves (and the sums are rescaled) only when
// a score exceeds it by more than kSlack: exponentials up to 2^kSlack are as
// exact. The waves' sums are merged in LDS, those of the key shares by
// attention_merge_kernel.
//
// Bound by the MFMAs (16 key blocks a wave: 1.57 us a block of 3,072 MFMA
// cycles) and, for short inputs, by launches and first loads. One wave a SIMD
// (402 registers at 128: eight operand groups, 1 to 1.5 us of MFMAs, are on
// their way; four measured 176 us where eight take 169). Measured against
// attention_tile_f32 for all: 4096 frames of 4 x 128 569 -> 171 us, 1864 133 ->
// 57, 1000 42 -> 30, 1100 of 8 x 96 945 -> 45 (it ran on the VALU); error against
// 64 bits 7.2e-7 -> 4.1e-7 (4096), 5.0e-7 -> 1.7e-7 (1000).
//
// Values outside [2^-100, 2^60] in magnitude, but zero, set the head's word in
// `outside` (so do infinities and NaN); its queries run on fp32 MFMA, dealt over
// the shares. A workgroup then has the CU to itself, and an attention call takes, us,
// with all heads outside (as attention_tile_f32 in a launch of its own, and with
// four tiles in turn by share 0): 400 frames of 4 x 128 39.5 (20.8, 85), 576 32.5
// (25, 103), 1000 46.7 (40, 164), 1864 114 (133, 293), 4096 408 (569, 611); 640 of 8
// x 64 32 (25, 75), 1068 79 (54, 116), 2500 273 (198, 366). What is left is the planes'
// launch and one wave a SIMD. Scores of the next block beside the softmax of this
// one, or keys read 64 bytes a row and load, took the same times.
constexpr uint32_t kPlaneMost = 0x5d800000u;  // 2^60
constexpr float kSlack = 8.0f;
constexpr int kSplitQ = 64;  // queries a workgroup

struct SplitAttnArgs {
  const float *q, *k, *v;
  float* out;
  int frames, width, heads, shares;
  float divisor, scale;         // sqrt(head size); log2(e) / divisor
  uint4 *qp, *kp, *vp;          // planes [head][block 32][HS / 16][3][64]
  float* part;                  // [share][head][frames padded to 64][HS] sums (shares > 1)
  float2* part_ml;              // [share][head][frames padded to 64] maximum, denominator
  unsigned* outside;            // [heads]: `epoch` where the head's values do not fit the planes
  unsigned epoch;
};

template <int HS>
__global__ __launch_bounds__(256) void attention_planes_kernel(SplitAttnArgs a) {
  constexpr int C16 = HS / 16;
  const int blocks = (a.frames + 63) / 64 * 2, per_head = blocks * C16 * 64, total = a.heads * per_head;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int which = blockIdx.y;  // 0 q, 1 k, 2 v
  const int head = i / per_head, lane = i & 63, fragment = (i % per_head) >> 6;
  const float* src = (which == 0 ? a.q : which == 1 ? a.k : a.v) + head * HS;
  float v[8];
  if (which < 2) {
    const int row = fragment / C16 * 32 + (lane & 31), ch = fragment % C16 * 16 + 8 * (lane >> 5);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float4 x4 = row < a.frames ? *reinterpret_cast<const float4*>(src + (size_t)row * a.width + ch + 4 * h)
                                       : make_float4(0.f, 0.f, 0.f, 0.f);
      v[4 * h] = x4.x;
      v[4 * h + 1] = x4.y;
      v[4 * h + 2] = x4.z;
      v[4 * h + 3] = x4.w;
    }
  } else {
    // Fragments of a 32-key block: 16-key step (outer), 32-channel block.
    const int step = fragment / (HS / 32), ch = fragment % (HS / 32) * 32 + (lane & 31);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int key = 16 * step + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
      v[e] = key < a.frames ? src[(size_t)key * a.width + ch] : 0.0f;
    }
  }
  bool odd = false;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t m = f2u(v[e]) & 0x7fffffffu;
    odd = odd || m > kPlaneMost || m - 1u < kSplitTiny - 1u;
  }
  if (odd) a.outside[head] = a.epoch;
  uint4 p[3];
  if (which == 0) {
    float low[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float scaled = v[e] * a.scale;
      low[e] = __builtin_fmaf(v[e], a.scale, -scaled);
      v[e] = scaled;
    }
    split8(v, p, low);
  } else {
    split8(v, p);
  }
  uint4* dst = (which == 0 ? a.qp : which == 1 ? a.kp : a.vp) + ((size_t)head * (per_head >> 6) + fragment) * 192 + lane;
#pragma unroll
  for (int s = 0; s < 3; ++s) dst[64 * s] = p[s];
}

template <int HS>
__global__ __launch_bounds__(256, 1) void attention_split_kernel(SplitAttnArgs a) {
  constexpr int C16 = HS / 16, CB = HS / 32, G = 2 * C16, ROW = HS + 4;  // fragment groups a key block: C16 of k, C16 of v
  constexpr int AHEAD = G / 2;
  static_assert(G % AHEAD == 0, "a block's groups fill the ring a whole number of times");
  extern __shared__ __attribute__((aligned(16))) char attn_split_s[];
  float* o_s = reinterpret_cast<float*>(attn_split_s);  // [2][64][ROW]
  float2* ml_s = reinterpret_cast<float2*>(o_s + 2 * kSplitQ * ROW);  // [2][64]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, lk = lane >> 5;
  const int wq = wave & 1, wk = wave >> 1;
  // Workgroups are dealt to the XCDs in turn: each takes a run of tiles, the
  // queries of one head and share together, whose k and v its L2 then holds.
  const int tiles = gridDim.x, xcd = blockIdx.x & 7, q8 = tiles >> 3, r8 = tiles & 7, qtiles = (a.frames + 63) / 64;
  const int tile = xcd * q8 + min(xcd, r8) + (blockIdx.x >> 3);
  const int q0 = tile % qtiles * kSplitQ, share = tile / qtiles % a.shares, head = tile / qtiles / a.shares;
  const unsigned outside = a.outside[head];
  const int blocks64 = (a.frames + 63) / 64, blocks = (a.frames + 31) / 32;
  const size_t head_pieces = (size_t)blocks64 * 2 * C16 * 192;
  bf16x8 q[C16][3];
  {
    const uint4* src = a.qp + head * head_pieces + (size_t)(q0 / 32 + wq) * C16 * 192 + lane;
#pragma unroll
    for (int c = 0; c < C16; ++c)
#pragma unroll
      for (int s = 0; s < 3; ++s) q[c][s] = __builtin_bit_cast(bf16x8, src[c * 192 + 64 * s]);
  }
  const int first = blocks * share / a.shares + wk, last = blocks * (share + 1) / a.shares;
  const uint4* kp = a.kp + head * head_pieces + lane;
  const uint4* vp = a.vp + head * head_pieces + lane;
  floatx16 o[CB], small[CB];  // sums of the large products and of the corrections
#pragma unroll
  for (int c = 0; c < CB; ++c) o[c] = small[c] = floatx16{};
  float run_m = -__builtin_inff(), run_l = 0.0f;  // of this lane's query; the sum over this lane's keys
  bf16x8 ring[AHEAD][3];
  // Group g of block b: k's 16-channel steps, then v's (step, channel block) fragments.
  auto load = [&](int b, int g) {
    if (g >= G) {
      g -= G;
      b += 2;
    }
    b = min(b, blocks - 1);
    const uint4* src = (g < C16 ? kp : vp) + ((size_t)b * C16 + (g < C16 ? g : g - C16)) * 192;
#pragma unroll
    for (int s = 0; s < 3; ++s) ring[g % AHEAD][s] = __builtin_bit_cast(bf16x8, src[64 * s]);
  };
  if (first < last) {
#pragma unroll
    for (int g = 0; g < AHEAD; ++g) load(first, g);
  }
  // (The operands are on their way meanwhile.)
  if (outside == a.epoch) {
    // One share: all 64 queries with one read of the keys; else 32 or 16 a share.
    const auto queries = [&](auto tiles, int first) {
      if (first < kSplitQ && q0 + first < a.frames)
        attention_tile_f32<HS, tiles, true>(attn_split_s, a.q, a.k, a.v, a.out, a.frames, a.width, a.divisor, head, q0 + first);
    };
    if (a.shares == 1) queries(std::integral_constant<int, 4>{}, 0);
    else if (a.shares < 4) queries(std::integral_constant<int, 2>{}, 32 * share);
    else queries(std::integral_constant<int, 1>{}, 16 * share);
    return;
  }
  constexpr int pa[6] = {2, 0, 1, 0, 1, 0}, pb[6] = {0, 2, 1, 0, 0, 1};
  for (int b = first; b < last; b += 2) {
    floatx16 sc = floatx16{}, rest = floatx16{};
#pragma unroll
    for (int g = 0; g < C16; ++g) {
#pragma unroll
      for (int p = 0; p < 6; ++p) {
        floatx16& sum = p == 3 ? sc : rest;
        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[g % AHEAD][pa[p]], q[g][pb[p]], sum, 0, 0, 0);
      }
      load(b, g + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
    }
    float t[16], top = -__builtin_inff();
#pragma unroll
    for (int r = 0; r < 16; ++r) t[r] = sc[r] + rest[r];
    if (b == blocks - 1) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (b * 32 + 8 * (r >> 2) + 4 * lk + (r & 3) >= a.frames) t[r] = -__builtin_inff();
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) top = fmaxf(top, t[r]);
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    if (__any(top > run_m + kSlack)) {
      const float m = fmaxf(run_m, top), down = __builtin_amdgcn_exp2f(run_m - m);
      run_m = m;
      run_l *= down;
#pragma unroll
      for (int c = 0; c < CB; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          o[c][r] *= down;
          small[c][r] *= down;
        }
    }
    bf16x8 pr[2][3];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float e[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        e[i] = __builtin_amdgcn_exp2f(t[8 * h + i] - run_m);
        run_l += e[i];
      }
      uint4 w[3];
      split8(e, w);
#pragma unroll
      for (int s = 0; s < 3; ++s) pr[h][s] = __builtin_bit_cast(bf16x8, w[s]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = C16; g < G; ++g) {
      const int h = (g - C16) / CB, c = (g - C16) % CB;
#pragma unroll
      for (int p = 0; p < 6; ++p) {
        floatx16& sum = p == 3 ? o[c] : small[c];
        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[g % AHEAD][pa[p]], pr[h][pb[p]], sum, 0, 0, 0);
      }
      load(b, g + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  run_l += __shfl_xor(run_l, 32, 64);
  // Sums of both key halves to LDS: channel 32 c + 8 (r / 4) + 4 lk + r % 4 of query l32.
  {
    float* row = o_s + (size_t)(wk * kSplitQ + 32 * wq + l32) * ROW + 4 * lk;
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *reinterpret_cast<float4*>(row + 32 * c + 8 * r) =
            make_float4(o[c][4 * r] + small[c][4 * r], o[c][4 * r + 1] + small[c][4 * r + 1],
                        o[c][4 * r + 2] + small[c][4 * r + 2], o[c][4 * r + 3] + small[c][4 * r + 3]);
    if (lk == 0) ml_s[wk * kSplitQ + 32 * wq + l32] = make_float2(run_m, run_l);
  }
  lds_barrier();
  const int padded = blocks64 * 64;
  for (int e = tid; e < kSplitQ * HS / 4; e += 256) {
    const int row = e / (HS / 4), ch = e % (HS / 4) * 4, f = q0 + row;
    const float2 x = ml_s[row], y = ml_s[kSplitQ + row];
    const float m = fmaxf(x.x, y.x);
    const float fx = x.x == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(x.x - m);
    const float fy = y.x == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(y.x - m);
    const float l = fx * x.y + fy * y.y;
    const float4 u = *reinterpret_cast<const float4*>(o_s + (size_t)row * ROW + ch);
    const float4 v = *reinterpret_cast<const float4*>(o_s + (size_t)(kSplitQ + row) * ROW + ch);
    float4 s = make_float4(fx * u.x + fy * v.x, fx * u.y + fy * v.y, fx * u.z + fy * v.z, fx * u.w + fy * v.w);
    if (a.shares == 1) {
      if (f < a.frames) {
        float* o4 = a.out + (size_t)f * a.width + head * HS + ch;
        *reinterpret_cast<float4*>(o4) = make_float4(s.x / l, s.y / l, s.z / l, s.w / l);
      }
    } else {
      const size_t at = ((size_t)share * a.heads + head) * padded + f;
      *reinterpret_cast<float4*>(a.part + at * HS + ch) = s;
      if (ch == 0) a.part_ml[at] = make_float2(m, l);
    }
  }
}

// out = sum of the shares' sums / sum of their denominators, each at the common maximum.
template <int HS>
__global__ __launch_bounds__(256) void attention_merge_kernel(SplitAttnArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x, per = HS / 4;
  const int ch = i % per * 4, head = i / per % a.heads, f = i / per / a.heads;
  if (f >= a.frames || a.outside[head] == a.epoch) return;
  const size_t stride = (size_t)a.heads * ((a.frames + 63) / 64 * 64), at = stride / a.heads * head + f;
  float m = -__builtin_inff();
  for (int s = 0; s < a.shares; ++s) m = fmaxf(m, a.part_ml[s * stride + at].x);
  float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
  float l = 0.0f;
  for (int s = 0; s < a.shares; ++s) {
    const float2 ml = a.part_ml[s * stride + at];
    const float w = ml.x == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(ml.x - m);
    const float4 u = *reinterpret_cast<const float4*>(a.part + (s * stride + at) * HS + ch);
    l += w * ml.y;
    sum.x += w * u.x;
    sum.y += w * u.y;
    sum.z += w * u.z;
    sum.w += w * u.w;
  }
  float* o = a.out + (size_t)f * a.width + head * HS + ch;
  *reinterpret_cast<float4*>(o) = make_float4(sum.x / l, sum.y / l, sum.z / l, sum.w / l);
}

}  // namespace

bool f32_attention_supported(int frames, int width, int heads) {
  return frames >= 1 && frames <= 4096 && heads >= 1 && heads <= 65535 && width >= heads && width % heads == 0 &&
         width / heads <= kAMaxS;
}

// Weights of fewer columns have no planes: padded to 128 k they would take more
// than six times the values' memory.
constexpr int kSplitLeastK = 32;

// An FP32 weight's values, then the range check's word.
static size_t outside_offset(int64_t rows, int cols) { return ((size_t)rows * cols * 4 + 15) & ~(size_t)15; }

size_t f32_weight_bytes(int64_t rows, int cols) { return outside_offset(rows, cols) + 16; }

size_t f32_planes_bytes(int64_t rows, int cols) {
  return cols < kSplitLeastK ? 0 : (size_t)split_pieces(rows, cols) * 16;
}

const int* f32_weight_outside(const float* w, int64_t rows, int cols) {
  return reinterpret_cast<const int*>(reinterpret_cast<const char*>(w) + outside_offset(rows, cols));
}

hipError_t launch_f32_split(float* w, int64_t rows, int cols, void* planes, hipStream_t s) {
  int* outside = const_cast<int*>(f32_weight_outside(w, rows, cols));
  const hipError_t e = hipMemsetAsync(outside, 0, 16, s);
  if (e != hipSuccess) return e;
  f32_split_range_kernel<<<(int)std::min<int64_t>((rows + 3) / 4, 2048), 256, 0, s>>>(w, rows, cols, outside);
  const int64_t lanes = split_pieces(rows, cols) / 3;
  f32_split_planes_kernel<<<(int)std::min<int64_t>((lanes + 255) / 256, 4096), 256, 0, s>>>(w, rows, cols,
                                                                                          static_cast<uint4*>(planes));
  return hipGetLastError();
}

// The GEMM on fp32 MFMA.
static hipError_t launch_f32_gemm(const float* x, const float* w, const float* bias, float* out, int M, int N, int K,
                                  bool relu, hipStream_t s) {
  if (K % 4 != 0) {
    const dim3 grid((N + kGT - 1) / kGT, (M + kGT - 1) / kGT);
    f32_gemm_any_kernel<<<grid, 256, 0, s>>>(x, w, bias, out, M, N, K, relu);
    return hipGetLastError();
  }
  // The tile whose grid loads the CUs most evenly: rounds of 256
  // workgroups times the tile's area, the larger tile on a tie; a grid of at
  // most one 32 x 64 workgroup per CU splits K over its waves.
  const int big = ((M + 63) / 64) * ((N + 63) / 64), small = ((M + 31) / 32) * ((N + 63) / 64);
  const int64_t big_cost = (int64_t)((big + 255) / 256) * 2, small_cost = (small + 255) / 256;
  const dim3 grid((N + 63) / 64, (M + 31) / 32);
  if (big_cost <= small_cost)
    (relu ? f32_gemm_kernel<2, 2, true> : f32_gemm_kernel<2, 2, false>)<<<dim3((N + 63) / 64, (M + 63) / 64), 256, 0, s>>>(
        x, w, bias, out, M, N, K);
  else if (small <= 256 && K >= 256)
    f32_gemm_wavek_kernel<<<grid, 256, 0, s>>>(x, w, bias, out, M, N, K, relu);
  else
    (relu ? f32_gemm_kernel<1, 2, true> : f32_gemm_kernel<1, 2, false>)<<<grid, 256, 0, s>>>(x, w, bias, out, M, N, K);
  return hipGetLastError();
}

hipError_t launch_f32_linear(const float* x, const float* w, const void* weight_planes, const float* bias, float* out,
                             int M, int N, int K, bool relu, hipStream_t s) {
  if (M < 1 || N < 1 || K < 1) return hipErrorInvalidValue;
  // Up to four frames the GEMV is quicker at every size, from five on while its
  // waves (a row each) all run at once and a GEMM's K chain is longer. Measured
  // with five and eight frames, us (GEMV, GEMM): 1024 -> 3072 5.3 7.0, 8.4; 1024
  // -> 4096 6.6 8.9, 8.5; 2048 -> 5000 13.4 16.9, 13.6; 512 -> 3072 4.3 5.8, 6.1; 512 ->
  // 3500 6.1 8.1, 6.4; 192 -> 2048 3.8 4.8, 5.1; 128 -> 2048 3.9 4.9, 4.4; 64 -> 512
  // 3.7 4.7, 3.6.
  if (M <= 4 || (M <= 8 && (N <= 3072 ? K >= 192 || M == 5 : (int64_t)M * N <= (K >= 1024 ? 30720 : K >= 512 ? 20480 : 0)))) {
    // One row a wave; four (fewer reads of the frames' values) only where they
    // still leave the chip many rounds of waves. Measured, us (one row, four
    // rows): 1024 -> 3072, one frame 3.9 4.1; 1024 -> 151936, one 108 106, four
    // 178 145; 1024 -> 20000, eight 37.6 37.8 (GEMM 23.1); 1024 -> 2048, sixteen 9.5
    // 31 (GEMM 9.0).
#define FAH_GEMV(MF, RW)                                                                                        \
  do {                                                                                                          \
    const int groups = std::min((N + 4 * RW - 1) / (4 * RW), 2048);                                             \
    const auto kernel = K <= 256 ? (K % 4 ? f32_gemv_kernel<MF, RW, false, 4> : f32_gemv_kernel<MF, RW, true, 4>) \
                                 : (K % 4 ? f32_gemv_kernel<MF, RW, false, 16> : f32_gemv_kernel<MF, RW, true, 16>); \
    kernel<<<groups, 256, 0, s>>>(x, w, bias, out, M, N, K, relu);                                               \
  } while (0)
    const bool many = N >= 65536;
    if (M == 1) {
      if (many) FAH_GEMV(1, 4);
      else FAH_GEMV(1, 1);
    } else if (M <= 4) {
      if (many) FAH_GEMV(4, 4);
      else FAH_GEMV(4, 1);
    } else {
      FAH_GEMV(8, 1);
    }
#undef FAH_GEMV
    return hipGetLastError();
  }
  // With planes, fp32 MFMA all the same where the call is bound by a large
  // weight's bytes (planes are 1.5 times as many), or by the launch and the first
  // loads of a few K steps. Measured, us (planes, fp32): 16 frames of 1024 -> 50000
  // 60.6 49.1, of 1024 -> 20000 23.5 25.1, 20 of 256 -> 30000 13.3 9.2, 64 of 1024
  // -> 50000 64 87; 333 x 192 -> 1100 7.4 5.8, 1000 x 128 -> 512 6.0 4.9, 64 x 64 ->
  // 2048 5.6 3.8, 64 x 224 -> 1100 6.5 6.4, 9 x 192 -> 2048 4.8 5.4, 2000 x 192 -> 2048
  // 16.7 24.3. (Odd K has no such tile: 333 x 65 -> 512 6.3 10.2.)
  // The latter up to 256 tiles of 64 x 128, and up to 64 columns also where they leave
  // much of their last round idle (two a CU): of 64 -> 2048 1280 frames, 320 tiles, 9.8
  // 9.5, 1500, 384 tiles, 9.8 12.6, 2560, 640 tiles, 16.3 17.8; of 64 -> 3072 1500, 576
  // tiles, 16.6 13.9; 40 of 64 -> 50000 8.8 11.3.
  const int64_t wide = (int64_t)((M + 63) / 64) * ((N + 127) / 128);
  const bool tall = M <= 32 && N >= 28672;
  const bool narrow = wide <= 256 ? K <= 64 || (K <= 192 && M > 16) : K <= 64 && (wide <= 320 || (wide > 512 && wide <= 600));
  if (!weight_planes || (K % 4 == 0 && (tall || narrow)))
    return launch_f32_gemm(x, w, bias, out, M, N, K, relu, s);
  const uint4* planes = static_cast<const uint4*>(weight_planes);
  const auto tiles = [&](int tm, int tn) { return ((M + tm - 1) / tm) * ((N + tn - 1) / tn); };
  const auto run = [&](auto whole, auto any, int grid, int threads) {
    if (K % 4 == 0) whole<<<grid, threads, 0, s>>>(x, w, planes, bias, out, M, N, K, relu);
    else any<<<grid, threads, 0, s>>>(x, w, planes, bias, out, M, N, K, relu);
  };
#define FAH_SPLIT(WN, KS, TI, TJ, KB, D)                                                                     \
  run(f32_split_gemm_kernel<WN, KS, TI, TJ, KB, D, true>, f32_split_gemm_kernel<WN, KS, TI, TJ, KB, D, false>, \
      tiles(32 * TI, 32 * TJ * WN), 64 * WN * KS)
  // The largest tile that still loads the chip: 64 x 128 from 224 workgroups
  // on (with eight waves where they all run at once, four where several
  // workgroups of a CU follow each other), 32 x 64 from 128 on, else 32 x 32
  // with K split over four waves. Measured, us (8 waves, 4 waves, 32 x 64,
  // 32 x 32): 1000 x 512 -> 2048 19.2 19.7 23.7 25.0; 4000 x 2048 -> 512 52.7
  // 57.5 63.4 82.4; 4000 x 512 -> 2048 68.9 55.9 74.6 91.7; 1000 x 512 -> 1536
  // 17.2 17.5 16.3 20.5; 333 x 560 -> 1536 18.8 18.0 12.1 12.9; 300 x 1023 ->
  // 700 40.5 38.9 21.3 19.0; 20 x 512 -> 1024 14.4 14.2 8.2 7.1.
  if (wide > 256) FAH_SPLIT(4, 1, 2, 1, 1, 2);
  else if (wide >= 224) FAH_SPLIT(4, 2, 2, 1, 2, 2);
  else if (tiles(32, 64) >= 128) FAH_SPLIT(2, 2, 1, 1, 2, 2);
  else FAH_SPLIT(1, 4, 1, 1, 2, 2);
#undef FAH_SPLIT
  return hipGetLastError();
}

// Key shares of attention_split_kernel: as many as its workgroups (one a CU)
// leave room for, with four key blocks of 32 or more each. Measured with 1, 2,
// 3, 4 shares, us: 1000 frames of 4 heads of 128 (64 query tiles) 44 35 34 31;
// 1864 of 4 (120) 71 54 63 55; 1068 of 8 of 64 (136) 31 35 31 36; 4096 of 4
// (256) 169 177 181 185; 184 of 8 of 96 (24 tiles, 6 blocks) 12.9 14.8 14.6 15.4.
static int attention_shares(int frames, int heads) {
  const int tiles = (frames + 63) / 64 * heads, blocks = (frames + 31) / 32;
  return std::max(1, std::min(std::min(4, 256 / tiles), blocks / 4));
}

struct AttnLayout {
  size_t planes, part, part_ml, outside, bytes;
};
static AttnLayout attention_layout(int frames, int width, int heads) {
  const size_t padded = (size_t)(frames + 63) / 64 * 64, shares = attention_shares(frames, heads);
  AttnLayout l;
  l.planes = 4096;  // the heads' words first: they outlive a call
  l.part = l.planes + 3 * padded * width * 6;
  l.part_ml = l.part + (shares > 1 ? shares * padded * width * 4 : 0);
  l.bytes = l.part_ml + (shares > 1 ? shares * padded * heads * 8 : 0);
  return l;
}

size_t f32_attention_workspace(const float* q, const float* k, const float* out, int frames, int width, int heads) {
  const int S = width / heads;
  const bool aligned = (reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
  if (!aligned || heads > 1024 || (S != 64 && S != 96 && S != 128)) return 0;
  // Shorter ones are quicker without the extra launches (us, fp32 MFMA and
  // split: 250 frames of 4 x 128 14.5 16.2, 400 20.8 20.2, 576 25.6 23.1; 500
  // of 8 x 64 15.7 17.2, 1068 55.6 31.4). 96 has no fp32 MFMA kernel (184
  // frames of 8 x 96: 57 on the VALU, 13 here).
  if ((S == 128 && frames < 400) || (S == 64 && frames < 640)) return 0;
  return attention_layout(frames, width, heads).bytes;
}

template <int HS>
static hipError_t launch_split_attention(const SplitAttnArgs& a, hipStream_t s) {
  const int planes = a.heads * ((a.frames + 63) / 64 * 2) * (HS / 16) * 64, tiles = (a.frames + 63) / 64 * a.heads * a.shares;
  constexpr int lds = std::max((2 * kSplitQ * (HS + 4) + 4 * kSplitQ) * 4, attention_tile_bytes(HS));
  static const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void*>(attention_split_kernel<HS>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (raised != hipSuccess) return raised;
  attention_planes_kernel<HS><<<dim3((planes + 255) / 256, 3), 256, 0, s>>>(a);
  attention_split_kernel<HS><<<tiles, 256, lds, s>>>(a);
  if (a.shares > 1) attention_merge_kernel<HS><<<(a.frames * a.heads * (HS / 4) + 255) / 256, 256, 0, s>>>(a);
  return hipGetLastError();
}

hipError_t launch_f32_attention(const float* q, const float* k, const float* v, float* out, int frames, int width,
                                int heads, void* workspace, unsigned epoch, hipStream_t s) {
  if (!f32_attention_supported(frames, width, heads)) return hipErrorInvalidValue;
  const int S = width / heads;
  const float divisor = sqrtf((float)S);
  if (workspace) {
    const AttnLayout l = attention_layout(frames, width, heads);
    char* base = static_cast<char*>(workspace);
    SplitAttnArgs a{};
    a.q = q;
    a.k = k;
    a.v = v;
    a.out = out;
    a.frames = frames;
    a.width = width;
    a.heads = heads;
    a.shares = attention_shares(frames, heads);
    a.divisor = divisor;
    a.scale = (float)(1.4426950408889634 / std::sqrt((double)S));
    const size_t plane = (size_t)(frames + 63) / 64 * 64 * width * 6;
    a.qp = reinterpret_cast<uint4*>(base + l.planes);
    a.kp = reinterpret_cast<uint4*>(base + l.planes + plane);
    a.vp = reinterpret_cast<uint4*>(base + l.planes + 2 * plane);
    a.part = reinterpret_cast<float*>(base + l.part);
    a.part_ml = reinterpret_cast<float2*>(base + l.part_ml);
    a.outside = reinterpret_cast<unsigned*>(base);
    a.epoch = epoch;
    return S == 128 ? launch_split_attention<128>(a, s) : S == 96 ? launch_split_attention<96>(a, s) : launch_split_attention<64>(a, s);
  }
  const bool aligned = width % 4 == 0 && (reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k)) % 16 == 0;
  if (aligned && (S == 64 || S == 128)) {
    const dim3 grid(heads, (frames + 15) / 16);
    if (S == 128) f32_attention_mfma_kernel<128><<<grid, 256, 0, s>>>(q, k, v, out, frames, width, divisor);
    else f32_attention_mfma_kernel<64><<<grid, 256, 0, s>>>(q, k, v, out, frames, width, divisor);
    return hipGetLastError();
  }
  const dim3 grid(heads, (frames + kAQ - 1) / kAQ);
  f32_attention_kernel<<<grid, 256, 0, s>>>(q, k, v, out, frames, width, S, divisor);
  return hipGetLastError();
}

}  // namespace fah
