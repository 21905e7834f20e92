// fp32 GEMM on the gfx950 matrix cores.
//
// Replaces cublasSgemm / cublasSgemmStridedBatched behind ops::matmul and
// ops::bmm (reference src/ops/matmul.cpp:13-93).  Each operand is K-contiguous
// or MN-contiguous, which covers the four transpose cases.
//
// Main path, gemm_f32_split: every fp32 value is split, exactly, into three
// bf16 values on its way to LDS, and a product is six bf16 MFMAs into fp32
// accumulators: 2.5 PFLOP/s / 6 = 0.42 PFLOP/s where the fp32 MFMAs have
// 0.157.  Against 64-bit sums its error is 0.85 of theirs (see the kernel).
//
// Fallback, gemm_f32_mfma (rows that are not whole aligned float4s, offsets
// past 2 GB), whose tile also serves the split kernel's results that are not
// finite: v_mfma_f32_32x32x2_f32, tiles 128x128 (three blocks per CU) or
// 256x128 (two), 256 threads = 4 waves in 2x2, a stage of BK = 16 k = two
// slabs of 8: global -> registers -> LDS, double-buffered, pipelined inside
// one wave so the matrix core never waits on LDS (ordering fixed with
// sched_group_barrier).  The k index an MFMA step consumes is permuted so
// that lane group g = lane/32 owns k = 8*slab + 4*g + j for step j; A and B
// use the same permutation, so the contraction is unchanged.
//
// Tiles are ordered so that tiles sharing A rows land on the same XCD (block
// b runs on XCD b % 8) and, within it, in groups of 8 tile rows for L2 reuse.
// Small output grids are split along K into a workspace of partial products
// that a second kernel sums in a fixed order, so results stay bitwise
// reproducible.
#include <type_traits>

#include "common.h"
#include "mfma_sched.h"

using namespace ember;

namespace {

constexpr int kThreads = 256;
constexpr int kBK = 16;
constexpr int kGroupM = 8;
constexpr int kCUs = 256;

struct GemmArgs {
  const float* A;
  const float* B;
  float* C;
  int64_t M, N, K;
  int64_t lda, ldb, ldc;
  int64_t sA, sB, sC;
  int64_t kchunk;  // > 0: blockIdx.y is a K split of this many k (last one clipped)
  float alpha, beta;
  int tiles_m, tiles_n;
  // Optional extent read from device memory at run time: v = clamp(*dyn - dyn_base, 0, static extent);
  // dyn_dim 0: rows of C beyond v are not needed (whole tiles past v exit);
  // dyn_dim 1: K becomes v rounded up to 16 (operand rows up to there are read).
  const int64_t* dyn = nullptr;
  int64_t dyn_base = 0;
  int dyn_dim = 0;
  // Optional addend (single GEMMs only): C = alpha op(A) op(B) + beta D, with
  // D = C when null.  D may be C itself (ldd = ldc), never a shifted overlap.
  const float* D = nullptr;
  int64_t ldd = 0;
};

// The beta term's source for element (row, col) of the current C.
__device__ __forceinline__ const float* addend(const GemmArgs& a, const float* dst, int64_t row,
                                               int64_t col) {
  return a.D ? a.D + row * a.ldd + col : dst;
}

__device__ __forceinline__ int64_t dyn_extent(const GemmArgs& a, int64_t full) {
  return min(max(*a.dyn - a.dyn_base, int64_t{0}), full);
}

template <bool KC, int ROWS, int BK, int THREADS>
struct Stage {
  static constexpr int kStride = KC ? (BK + 4) : (ROWS + 8);
  static constexpr int kSize = KC ? ROWS * (BK + 4) : BK * (ROWS + 8);
  static constexpr int kChunks = ROWS * BK / 4;           // float4 chunks per tile
  static constexpr int kPerThread = kChunks / THREADS;    // loads per thread
  static_assert(kChunks % THREADS == 0, "tile not divisible among threads");

  f32x4 reg[kPerThread];

  // Global -> registers.  Operand rows [row0, row0+ROWS) x k [k0, k0+BK),
  // zero outside [0,R) x [0,K).
  template <bool VEC>
  __device__ __forceinline__ void load(const float* __restrict__ X, int64_t ld, int64_t R,
                                       int64_t K, int64_t row0, int64_t k0) {
#pragma unroll
    for (int p = 0; p < kPerThread; ++p) {
      const int c = threadIdx.x + p * THREADS;
      int64_t r, k;
      if (KC) {
        r = row0 + c / (BK / 4);
        k = k0 + 4 * (c % (BK / 4));
      } else {
        k = k0 + c / (ROWS / 4);
        r = row0 + 4 * (c % (ROWS / 4));
      }
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
      if (KC) {
        if (r < R) {
          const float* src = X + r * ld + k;
          if (VEC && k + 3 < K) {
            v = *reinterpret_cast<const f32x4*>(src);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (k + e < K) ? src[e] : 0.f;
          }
        }
      } else {
        if (k < K) {
          const float* src = X + k * ld + r;
          if (VEC && r + 3 < R) {
            v = *reinterpret_cast<const f32x4*>(src);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (r + e < R) ? src[e] : 0.f;
          }
        }
      }
      reg[p] = v;
    }
  }

  // Registers -> LDS in this operand's layout.
  __device__ __forceinline__ void store(float* __restrict__ lds) const {
#pragma unroll
    for (int p = 0; p < kPerThread; ++p) {
      const int c = threadIdx.x + p * THREADS;
      int off;
      if (KC) {
        off = (c / (BK / 4)) * kStride + 4 * (c % (BK / 4));
      } else {
        off = (c / (ROWS / 4)) * kStride + 4 * (c % (ROWS / 4));
      }
      *reinterpret_cast<f32x4*>(lds + off) = reg[p];
    }
  }

  // Fragment for MFMA steps j = 0..3 of k-slab `slab`, row `row` of the tile.
  __device__ __forceinline__ static f32x4 frag(const float* __restrict__ lds, int row, int slab,
                                               int g) {
    if (KC) {
      return *reinterpret_cast<const f32x4*>(lds + row * kStride + slab * 8 + 4 * g);
    } else {
      f32x4 v;
      const float* base = lds + (slab * 8 + 4 * g) * kStride + row;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = base[j * kStride];
      return v;
    }
  }
};

template <int BM, int BN>
__device__ __forceinline__ void tile_coords(const GemmArgs& a, int& tm, int& tn) {
  const int tiles = a.tiles_m * a.tiles_n;
  int t = blockIdx.x;
  if ((tiles & 7) == 0) t = (t & 7) * (tiles >> 3) + (t >> 3);
  if (a.dyn && a.dyn_dim == 0) {
    // Row tiles past a count read on the device are skipped.  Each XCD takes
    // a range of whole columns (every row tile of them), so each keeps the
    // same share of the work that remains whatever the count; with groups of
    // tile rows per XCD, the XCDs holding the first rows would do it all.
    tm = t % a.tiles_m;
    tn = t / a.tiles_m;
    return;
  }
  const int width = kGroupM * a.tiles_n;
  const int group = t / width;
  const int first = group * kGroupM;
  const int gsz = min(a.tiles_m - first, kGroupM);
  const int in = t - group * width;
  tm = first + in % gsz;
  tn = in / gsz;
}

// The LDS of one output tile on the fp32 MFMAs, and that tile (see the header):
// rows m0 ..., columns n0 ... of C, over K.
template <bool A_KC, bool B_KC, int BM, int BN, int THREADS>
constexpr int kFp32LdsFloats =
    2 * (Stage<A_KC, BM, kBK, THREADS>::kSize + Stage<B_KC, BN, kBK, THREADS>::kSize);

template <bool A_KC, bool B_KC, bool VEC, int BM, int BN, int THREADS>
__device__ __forceinline__ void fp32_tile(const GemmArgs& a, const float* __restrict__ A,
                                          const float* __restrict__ B, float* __restrict__ C,
                                          int64_t K, int64_t m0, int64_t n0, float* lds) {
  using SA = Stage<A_KC, BM, kBK, THREADS>;
  using SB = Stage<B_KC, BN, kBK, THREADS>;
  constexpr int kWM = THREADS / 128;                    // waves along M; two along N
  constexpr int FI = BM / (32 * kWM), FJ = BN / 64;     // 32x32 tiles per wave
  constexpr int NR = FI * (A_KC ? 1 : 4) + FJ * (B_KC ? 1 : 4);  // LDS reads per slab
  constexpr int NW = SA::kPerThread + SB::kPerThread;   // LDS stores per stage
  constexpr int NM = 4 * FI * FJ;                       // MFMAs per slab
  float* const lds_a = lds;                  // two stages each
  float* const lds_b = lds + 2 * SA::kSize;

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int g = lane >> 5, r = lane & 31;
  const int arow = wm * (BM / kWM) + r, brow = wn * (BN / 2) + r;

  f32x16 acc[FI][FJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  SA sa;
  SB sb;
  const int64_t nk = (K + kBK - 1) / kBK;
  if (nk > 0) {
    sa.template load<VEC>(A, a.lda, a.M, K, m0, 0);
    sb.template load<VEC>(B, a.ldb, a.N, K, n0, 0);
    sa.store(lds_a);
    sb.store(lds_b);
  }
  __syncthreads();

  f32x4 fa0[FI], fb0[FJ], fa1[FI], fb1[FJ];
#pragma unroll
  for (int i = 0; i < FI; ++i) fa0[i] = SA::frag(lds_a, arow + i * 32, 0, g);
#pragma unroll
  for (int j = 0; j < FJ; ++j) fb0[j] = SB::frag(lds_b, brow + j * 32, 0, g);

  for (int64_t kt = 0; kt < nk; ++kt) {
    const int cur = static_cast<int>(kt & 1);
    // Stage kt+1; the last iteration reloads its own stage into the idle
    // buffer, which nothing reads afterwards.
    const int64_t knext = (kt + 1 < nk ? kt + 1 : kt) * kBK;
    sa.template load<VEC>(A, a.lda, a.M, K, m0, knext);
    sb.template load<VEC>(B, a.ldb, a.N, K, n0, knext);
    const float* la = lds_a + cur * SA::kSize;
    const float* lb = lds_b + cur * SB::kSize;
    float* na = lds_a + (cur ^ 1) * SA::kSize;
    float* nb = lds_b + (cur ^ 1) * SB::kSize;

#pragma unroll
    for (int i = 0; i < FI; ++i) fa1[i] = SA::frag(la, arow + i * 32, 1, g);
#pragma unroll
    for (int j = 0; j < FJ; ++j) fb1[j] = SB::frag(lb, brow + j * 32, 1, g);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < FI; ++i)
#pragma unroll
        for (int j = 0; j < FJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa0[i][s], fb0[j][s], acc[i][j], 0, 0, 0);
    interleave<NR, NM, 0x100>();

    sa.store(na);
    sb.store(nb);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < FI; ++i)
#pragma unroll
        for (int j = 0; j < FJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa1[i][s], fb1[j][s], acc[i][j], 0, 0, 0);
    interleave<NW, NM / 2, 0x200>();
    __syncthreads();

#pragma unroll
    for (int i = 0; i < FI; ++i) fa0[i] = SA::frag(na, arow + i * 32, 0, g);
#pragma unroll
    for (int j = 0; j < FJ; ++j) fb0[j] = SB::frag(nb, brow + j * 32, 0, g);
#pragma unroll
    for (int s = 2; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < FI; ++i)
#pragma unroll
        for (int j = 0; j < FJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa1[i][s], fb1[j][s], acc[i][j], 0, 0, 0);
    interleave<NR, NM / 2, 0x100>();
  }

  // Accumulator layout of a 32x32 MFMA tile: lane (g, r), register e holds
  // row 8*(e/4) + 4*g + (e%4), column r.
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j) {
      const int64_t col = n0 + wn * (BN / 2) + j * 32 + r;
      if (col >= a.N) continue;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t row = m0 + wm * (BM / kWM) + i * 32 + 8 * (e >> 2) + 4 * g + (e & 3);
        if (row < a.M) {
          float* dst = C + row * a.ldc + col;
          const float v = a.alpha * acc[i][j][e];
          *dst = (a.beta != 0.f) ? v + a.beta * *addend(a, dst, row, col) : v;
        }
      }
    }
}

template <bool A_KC, bool B_KC, bool VEC, int BM, int BN, int OCC>
__global__ __launch_bounds__(kThreads, OCC) void gemm_f32_mfma(GemmArgs a) {
  __shared__ __attribute__((aligned(16))) float lds[kFp32LdsFloats<A_KC, B_KC, BM, BN, kThreads>];

  int tm, tn;
  tile_coords<BM, BN>(a, tm, tn);
  const int64_t bz = blockIdx.y;
  int64_t K = a.kchunk > 0 ? min(a.kchunk, a.K - bz * a.kchunk) : a.K;
  const int64_t m0 = static_cast<int64_t>(tm) * BM;
  const int64_t n0 = static_cast<int64_t>(tn) * BN;
  if (a.dyn) {  // uniform per block: the whole block leaves or none of it
    if (a.dyn_dim == 0) {
      if (m0 >= dyn_extent(a, a.M)) return;
    } else {
      K = min(K, (dyn_extent(a, K) + 15) / 16 * 16);
      if (K == 0 && a.beta == 1.f && !a.D) return;  // C stays as it is
    }
  }
  fp32_tile<A_KC, B_KC, VEC, BM, BN, kThreads>(a, a.A + bz * a.sA, a.B + bz * a.sB,
                                               a.C + bz * a.sC, K, m0, n0, lds);
}

// ------------------------------------------------- bf16 matrix cores, fp32 in
// Every fp32 value is the sum of three bf16 values exactly (8 + 8 + 8
// significand bits, each part rounded to nearest): x = x0 + x1 + x2.  A
// product is then taken as the six partial products
//   a0 b2 + a1 b1 + a2 b0 + a0 b1 + a1 b0 + a0 b0
// on v_mfma_f32_32x32x16_bf16, whose products are exact and whose sums are
// fp32; what is left out (a1 b2, a2 b1, a2 b2) is at most 2^-24 of the product
// (|a1| <= 2^-8, |a2| <= 2^-17 of a value) and 2^-27.5 of it in the root mean
// square.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned pack_bf16(float x, float y) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{x, y}, bf16x2));
}
__device__ __forceinline__ float bf16_lo(unsigned u) { return __builtin_bit_cast(float, u << 16); }
__device__ __forceinline__ float bf16_hi(unsigned u) {
  return __builtin_bit_cast(float, u & 0xffff0000u);
}

// Both operands are scaled by 2^24 first (B by the sign it is summed with, too):
// the last part of an unscaled value below 2^-110 would have no exponent left,
// and all three of one below 2^-134 would be zero.  Scaled, every part of every
// subnormal is a normal bf16 value.
constexpr float kScale = 0x1p24f, kUnscale = 0x1p-48f;

struct SplitWork {  // four k of one row on their way from fp32 to three parts
  float x[4];
  u32x2 part[3];
};

// One operand's tile: ROWS rows x 16 k of fp32, fetched into registers and
// stored to LDS as three bf16 planes of [2 k halves][ROWS slots][8 k].  An
// MFMA fragment (32 slots, one k half per lane group) is then one b128 read
// of 512 contiguous bytes per half; the halves lie 128 bytes apart modulo the
// 64 banks, so that the stores of four k per lane meet no bank twice.
//   K-contiguous: lane = (row, k quad), slot = row.
//   MN-contiguous: a wave takes one k quad of 64 P rows, P = 4 ROWS / THREADS;
//     a lane takes P consecutive rows of each of its four k, and row P l + i
//     goes to slot 32 P (l / 32) + 32 i + l % 32, so that a lane's rows land in
//     the P 32-slot tiles of one wave at the same place.
template <bool KC, int ROWS, int THREADS>
struct SplitTile {
  static constexpr int P = 4 * ROWS / THREADS;
  static constexpr int kHalf = ROWS * 16 + 128;   // bytes
  static constexpr int kPlane = 2 * kHalf;
  static constexpr int kBytes = 3 * kPlane;
  const char* base;      // the tile's first element at the current stage
  int64_t left;          // bytes from there to the operand's end
  int64_t step;          // bytes of a k
  int voff;              // this lane's first element, bytes from base
  int soff[KC ? P : 4];  // uniform offsets of the lane's loads
  int woff;              // where the lane's first four k go in LDS
  using Vec = std::conditional_t<KC || P == 4, f32x4, std::conditional_t<P == 2, f32x2, float>>;
  Vec reg[KC ? P : 4];   // K-contiguous: four k of a row; MN: P rows of a k

  __device__ __forceinline__ void init(const float* X, int64_t ld, int64_t R, int64_t K,
                                       int64_t row0, int wave, int lane) {
    step = KC ? 4 : 4 * ld;
    if constexpr (KC) {
      base = reinterpret_cast<const char*>(X + row0 * ld);
      left = ((R - row0 - 1) * ld + K) * 4;
      const int row = 16 * wave + (lane >> 2), quad = lane & 3;
      voff = static_cast<int>(row * ld * 4) + 16 * quad;
#pragma unroll
      for (int q = 0; q < P; ++q) soff[q] = static_cast<int>(q * (THREADS / 4) * ld * 4);
      woff = (quad >> 1) * kHalf + row * 16 + (quad & 1) * 8;
    } else {
      base = reinterpret_cast<const char*>(X + row0);
      left = ((K - 1) * ld + R - row0) * 4;
      const int quad = wave & 3, first = 64 * P * (wave >> 2);  // first row of the wave's
      voff = 4 * (first + P * lane);
#pragma unroll
      for (int j = 0; j < 4; ++j) soff[j] = static_cast<int>((4 * quad + j) * ld * 4);
      woff = (quad >> 1) * kHalf + (first + 32 * P * (lane >> 5) + (lane & 31)) * 16 + (quad & 1) * 8;
    }
  }

  static constexpr int kLoads = KC ? P : 4;
  // Load q of the current stage.  Past the operand's end the buffer resource
  // returns zeros, so no row or k is tested.
  __device__ __forceinline__ void load(int q) {
#if defined(__HIP_DEVICE_COMPILE__)
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(base), 0, static_cast<int>(min(max(left, int64_t{0}), int64_t{0x7fffffff})),
        0x00020000);
    const int at = voff + soff[q];
    if constexpr (sizeof(Vec) == 16)
      reg[q] = __builtin_bit_cast(Vec, __builtin_amdgcn_raw_buffer_load_b128(rs, at, 0, 0));
    else if constexpr (sizeof(Vec) == 8)
      reg[q] = __builtin_bit_cast(Vec, __builtin_amdgcn_raw_buffer_load_b64(rs, at, 0, 0));
    else
      reg[q] = __builtin_bit_cast(Vec, __builtin_amdgcn_raw_buffer_load_b32(rs, at, 0, 0));
#endif
  }
  // All loads of the current stage, of which `k` (four at a time) count.
  __device__ __forceinline__ void load_all(int k = 16) {
#pragma unroll
    for (int q = 0; q < kLoads; ++q) load(q);
    base += k * step;
    left -= k * step;
  }
  // Zeros for the k of the loaded stage that don't.
  __device__ __forceinline__ void mask(int k, int wave, int lane) {
    if (k <= 4 * (KC ? lane & 3 : wave & 3)) {
#pragma unroll
      for (int q = 0; q < kLoads; ++q) reg[q] = Vec{};
    }
  }
  // Element (k j of the lane's quad, row i of the lane's P).
  __device__ __forceinline__ float at(int j, int i) const {
    if constexpr (KC) return reg[i][j];
    else if constexpr (P == 1) return reg[j];
    else return reg[j][i];
  }
  // The split of row i's four k, in kSteps steps of at most four VALU
  // operations for the spaces between MFMAs; the last stores the parts.
  // `scale`: +-kScale.
  static constexpr int kSteps = 7;
  __device__ __forceinline__ void split_step(SplitWork& w, int i, int step, char* lds,
                                             float scale) const {
    if (step == 0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) w.x[j] = at(j, i) * scale;
    } else if (step == 1 || step == 3) {
      const int p = step / 3;
      w.part[p] = u32x2{pack_bf16(w.x[0], w.x[1]), pack_bf16(w.x[2], w.x[3])};
    } else if (step == 2 || step == 5) {
      const u32x2 h = w.part[step / 3];
      w.x[0] -= bf16_lo(h[0]);
      w.x[1] -= bf16_hi(h[0]);
      w.x[2] -= bf16_lo(h[1]);
      w.x[3] -= bf16_hi(h[1]);
    } else if (step == 6) {
      w.part[2] = u32x2{pack_bf16(w.x[0], w.x[1]), pack_bf16(w.x[2], w.x[3])};
#pragma unroll
      for (int p = 0; p < 3; ++p)
        *reinterpret_cast<u32x2*>(lds + woff + p * kPlane + i * (KC ? THREADS / 4 : 32) * 16) = w.part[p];
    }
  }
  __device__ __forceinline__ void store_all(char* lds, float scale) const {
#pragma unroll
    for (int i = 0; i < P; ++i) {
      SplitWork w;
#pragma unroll
      for (int t = 0; t < kSteps; ++t) split_step(w, i, t, lds, scale);
    }
  }
  // Part p of 32-slot tile t (from the wave's first), for lane offset `off`.
  __device__ __forceinline__ static bf16x8 frag(const char* lds, int off, int p, int t) {
    return __builtin_bit_cast(bf16x8,
                              *reinterpret_cast<const u32x4*>(lds + off + p * kPlane + t * 512));
  }
};

// Why: the fp32 MFMAs reach 151 TFLOP/s (0.96 of their peak) and bound every
// large product.  Here 32768x6144x2048 takes 3.7 ms in each layout against 5.5,
// 222 TFLOP/s: matrix cores 70-74% busy while power holds the clock near 1.8
// GHz (on zeros, which cost little power, the same launch takes 2.8 ms).
// Error against 64-bit sums in the 2-norm, normal data, K = 32 / 256 / 2048:
// 6.9e-8 / 2.4e-7 / 6.9e-7, where fp32 MFMAs give 1.0e-7 / 2.9e-7 / 8.1e-7; with
// the 512-thread tile's segments 6.9e-8 / 1.7e-7 / 2.4e-7 (K = 32768: 3.1e-7
// against 3.2e-6).  Only a sum of one or two terms that are not zero is further
// off: one term is rounded with 0.39 of a unit (rms) instead of 0.29.
//
// The bf16 MFMAs round their sums very slightly downwards (a mean of -1.3e-7
// of the mean magnitude at K = 2048, in proportion to the number of sums and
// their size), which sums over rows, columns or K splits would gather: with
// it, a value projection's weight gradient over 32768 tokens was 1.4 times as
// far from 64-bit sums as with fp32 MFMAs.  So the sum is held negated, B's
// sign flipped on the way to LDS, from 0.207 to 0.707 of K, which cancels the
// bias of sums that stay the same size along K or grow as sqrt(K), and all
// but 9% where they grow as K (nothing here depends on a row's or column's
// place).  Two things it cannot balance: terms that all lie in one half of K (a
// mean of 3e-8 at K = 2048, 6% of the spread) and a single pair of stages (K <=
// 32: 1e-8).  K splits start negated by the parity of the number's count of
// ones (0 1 1 0 1 0 0 1 ...); the products of a batch all start alike.  Turning
// 256 accumulators costs about one stage.
//
// What the split cannot give: an infinity or NaN has no three parts, nor has a
// value of 2^104 or more once scaled; such a result, or one past 2^80, is not
// finite, which is found here, and it is taken again in fp32.
//
// The 512-thread tile has the registers for a second set of sums and adds up K
// in segments of at most kSegK, an even number of them, with the same signs as
// K splits: as exact as that many splits (2048x1024x2048 in two chunks 4.85e-7
// -> 2.4e-7 in the 2-norm) without their planes.
constexpr int kSegK = 256;

// THREADS = 256: 4 waves in 2x2, wave tiles (BM/2)x(BN/2); 512: 8 waves in
// 4x2.  LDS is double buffered.  A 256x256 block has a CU to itself and one
// wave per SIMD, so the order of the wave's own instructions is what keeps the
// matrix core busy: it is written out MFMA by MFMA and pinned (sched_barrier),
// two to eight VALU operations of the split between two MFMAs of 32 cycles
// each.  Left to the compiler, the same work took 1.16 times as long.
template <bool A_KC, bool B_KC, int BM, int BN, int THREADS, int OCC>
__global__ __launch_bounds__(THREADS, OCC) void gemm_f32_split(GemmArgs a) {
  using TA = SplitTile<A_KC, BM, THREADS>;
  using TB = SplitTile<B_KC, BN, THREADS>;
  constexpr int kWM = THREADS / 128;                     // waves along M; two along N
  constexpr int FI = BM / (32 * kWM), FJ = BN / 64;      // 32x32 tiles per wave
  constexpr int kStage = TA::kBytes + TB::kBytes;
  constexpr bool kSegs = THREADS == 512;                 // K is summed in segments
  constexpr int64_t kSegPairs = kSegK / 32;
  __shared__ __attribute__((aligned(256))) char lds[2 * kStage];
  __shared__ int redo_flag;  // some wanted value of the block's is not finite
  if (threadIdx.x == 0) redo_flag = 0;

  int tm, tn;
  tile_coords<BM, BN>(a, tm, tn);
  const int64_t bz = blockIdx.y;
  const float* __restrict__ A = a.A + bz * a.sA;
  const float* __restrict__ B = a.B + bz * a.sB;
  float* __restrict__ C = a.C + bz * a.sC;
  int64_t K = a.kchunk > 0 ? min(a.kchunk, a.K - bz * a.kchunk) : a.K;
  const int64_t m0 = static_cast<int64_t>(tm) * BM;
  const int64_t n0 = static_cast<int64_t>(tn) * BN;
  if (a.dyn) {  // uniform per block: the whole block leaves or none of it
    if (a.dyn_dim == 0) {
      if (m0 >= dyn_extent(a, a.M)) return;
    } else {
      K = min(K, (dyn_extent(a, K) + 15) / 16 * 16);
      if (K == 0 && a.beta == 1.f && !a.D) return;  // C stays as it is
    }
  }

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int g = lane >> 5, r = lane & 31;

  f32x16 acc[FI][FJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  const int64_t nk = (K + 15) / 16;
  const int ra = g * TA::kHalf + (wm * (BM / kWM) + r) * 16;
  const int rb = TA::kBytes + g * TB::kHalf + (wn * (BN / 2) + r) * 16;
  const bool start = a.kchunk > 0 && (__builtin_popcountll(bz) & 1);  // negated
  if (nk > 0) {
    const int64_t pairs = (nk + 1) / 2;
    const int64_t turn[3] = {(pairs * 212) >> 10, (pairs * 724) >> 10, pairs};
    // kSegs: segments of `len` pairs, the first `more` of them one longer; one
    // for a short K split, whose neighbours start with the other sign.
    const unsigned segs =
        pairs > (a.kchunk > 0 ? kSegPairs : 1)
            ? 2 * static_cast<unsigned>((pairs + 2 * kSegPairs - 1) / (2 * kSegPairs))
            : 1;
    const unsigned len = static_cast<unsigned>(pairs) / segs;
    const unsigned more = static_cast<unsigned>(pairs) - len * segs;
    unsigned seg = 0;
    int64_t seg_end = len + (more > 0);
    const auto seg_neg = [&](unsigned i) { return start != ((__builtin_popcount(i) & 1) != 0); };
    float scale_b;  // of the values stored, which belong to pair `at`
    const auto sign_at = [&](int64_t at) {
      const bool neg = kSegs ? seg_neg(at < seg_end ? seg : seg + 1)
                             : start != (at >= turn[0] && at < turn[1]);
      scale_b = neg ? -kScale : kScale;
    };
    sign_at(0);
    TA ta;
    TB tb;
    ta.init(A, a.lda, a.M, K, m0, wave, lane);
    tb.init(B, a.ldb, a.N, K, n0, wave, lane);
    // A K that is not whole pairs of stages begins with what is missing, an
    // empty stage, a short one or both (a K-contiguous operand's K is whole
    // float4s), so that the loop has no k to leave out.  Where neither operand
    // is K-contiguous both end where memory says.
    const int rest = static_cast<int>(K - 16 * (nk - 1));
    const int first = !(A_KC || B_KC) ? 16 : nk & 1 ? 0 : rest;
    const int second = !(A_KC || B_KC) || !(nk & 1) ? 16 : rest;
    ta.load_all(first);
    tb.load_all(first);
    if (first < 16) {
      ta.mask(first, wave, lane);
      tb.mask(first, wave, lane);
    }
    ta.store_all(lds, kScale);
    tb.store_all(lds + TA::kBytes, scale_b);
    ta.load_all(second);
    tb.load_all(second);
    if (second < 16) {
      ta.mask(second, wave, lane);
      tb.mask(second, wave, lane);
    }
    wait_lgkm0();
    block_barrier();
    bf16x8 fa[2][3], fb[2][FJ][3];
#pragma unroll
    for (int p = 0; p < 3; ++p) fa[0][p] = TA::frag(lds, ra, p, 0);
#pragma unroll
    for (int j = 0; j < FJ; ++j)
#pragma unroll
      for (int p = 0; p < 3; ++p) fb[0][j][p] = TB::frag(lds, rb, p, j);

    // One stage: FI groups of 6 FJ MFMAs, one group per 32-row tile of A.
    // Between them, in this order: the split and store of the next stage's
    // fetched values, each followed by the fetch of the stage after it; a
    // barrier before the last group; the next stage's first fragments.
    auto stage = [&](auto odd) {
      constexpr int kOdd = decltype(odd)::value;
      constexpr int kGroup = 6 * FJ;
      // MFMA slots: the barrier's, those for the splits, fragment reads per
      // slot after the barrier.
      constexpr int kTurn = FI > 1 ? (FI - 1) * kGroup : 8;
      constexpr int kSlots = kTurn - (FI > 2 ? 8 : FI > 1 ? 2 : 1);
      constexpr int kReads = FI > 1 ? 1 : 3;
      constexpr int kQuads = TA::P + TB::P;
      constexpr int kWork = kQuads * TA::kSteps;
      const char* cur = lds + kOdd * kStage;
      char* nxt = lds + (1 - kOdd) * kStage;
      SplitWork w;
#pragma unroll
      for (int i = 0; i < FI; ++i) {
        constexpr int pa[6] = {0, 1, 2, 0, 1, 0}, pb[6] = {2, 1, 0, 1, 0, 0};  // smallest first
#pragma unroll
        for (int t = 0; t < 6; ++t)
#pragma unroll
          for (int j = 0; j < FJ; ++j) {
            const int in = t * FJ + j, m = i * kGroup + in;
            if (m == kTurn) {
              wait_lgkm0();
              block_barrier();
            }
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                fa[FI > 1 ? i & 1 : kOdd][pa[t]], fb[kOdd][j][pb[t]], acc[i][j], 0, 0, 0);
            if (i < FI - 1 && in < 3) fa[(i + 1) & 1][in] = TA::frag(cur, ra, in, i + 1);
            if (m >= kTurn) {
#pragma unroll
              for (int f = (m - kTurn) * kReads; f < (m - kTurn + 1) * kReads; ++f) {
                if (f < 3)
                  fa[FI > 1 ? 0 : 1 - kOdd][f] = TA::frag(nxt, ra, f, 0);
                else if (f < 3 + 3 * FJ)
                  fb[1 - kOdd][(f - 3) / 3][(f - 3) % 3] =
                      TB::frag(nxt, rb, (f - 3) % 3, (f - 3) / 3);
              }
            }
            if (m < kSlots) {
#pragma unroll
              for (int s = m * kWork / kSlots; s < (m + 1) * kWork / kSlots; ++s) {
                const int q = s / TA::kSteps, st = s % TA::kSteps;
                if (q < TA::P)
                  ta.split_step(w, q, st, nxt, kScale);
                else
                  tb.split_step(w, q - TA::P, st, nxt + TA::kBytes, scale_b);
                if (s == TA::P * TA::kSteps - 1) ta.load_all();
                if (s == kWork - 1) tb.load_all();
              }
            }
            __builtin_amdgcn_sched_barrier(0);
          }
      }
    };
    int64_t p = 0;
    const auto run_to = [&](int64_t end) {
      while (p < end) {
        stage(std::integral_constant<int, 0>{});
        sign_at(++p);
        stage(std::integral_constant<int, 1>{});
      }
    };
    if constexpr (kSegs) {
      f32x16 sum[FI][FJ];
#pragma unroll
      for (int i = 0; i < FI; ++i)
#pragma unroll
        for (int j = 0; j < FJ; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) sum[i][j][e] = 0.f;
      for (; seg < segs; ++seg) {
        run_to(seg_end);
        seg_end += len + (seg + 1 < more);
        const float sign = seg_neg(seg) ? -1.f : 1.f;
#pragma unroll
        for (int i = 0; i < FI; ++i)
#pragma unroll
          for (int j = 0; j < FJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              sum[i][j][e] = __builtin_fmaf(sign, acc[i][j][e], sum[i][j][e]);
              acc[i][j][e] = 0.f;
            }
      }
#pragma unroll
      for (int i = 0; i < FI; ++i)
#pragma unroll
        for (int j = 0; j < FJ; ++j) acc[i][j] = sum[i][j];
    } else {
#pragma unroll
      for (int part = 0; part < 3; ++part) {
        run_to(turn[part]);
        if (part < 2) {
#pragma unroll
          for (int i = 0; i < FI; ++i)
#pragma unroll
            for (int j = 0; j < FJ; ++j) acc[i][j] = -acc[i][j];
        }
      }
    }
  }

  // The lane's place in the output: register e of tile (i, j) is row slot
  // x = 8 (e / 4) + 4 g + e % 4 of MFMA tile i and column slot r of tile j.
  const int64_t rw0 = m0 + wm * (BM / kWM), cw0 = n0 + wn * (BN / 2);
  const bool mine = rw0 < a.M && cw0 < a.N;  // the wave has output
  const auto row_of = [&](int i, int e) {  // its uniform part; the lane's is lrow
    const int x = 8 * (e >> 2) + (e & 3);
    return A_KC || TA::P == 1 ? i * 32 + x : FI * x + i;
  };
  const auto col_of = [&](int j) { return B_KC || TB::P == 1 ? j * 32 + r : FJ * r + j; };
  const int lrow = A_KC || TA::P == 1 ? 4 * g : FI * 4 * g;
  const int rows_left = static_cast<int>(min(a.M - rw0, int64_t{BM}));
  const int cols_left = static_cast<int>(min(a.N - cw0, int64_t{BN}));

  // Rows that are wanted (up to the 16-row group of a device-side count: the
  // rest may come of memory that nobody filled).
  const int64_t rows_end =
      a.dyn && a.dyn_dim == 0 ? min((dyn_extent(a, a.M) + 15) / 16 * 16, a.M) : a.M;
  const int rows_wanted = static_cast<int>(min(rows_end - rw0, int64_t{BM}));
  // Whether a value that is wanted is not finite; ALL: every value is looked at.
  const auto not_finite = [&](auto all) {
    constexpr bool kAll = decltype(all)::value;
    float bad = 0.f;  // NaN once some value is not finite
#pragma unroll
    for (int i = 0; i < FI; ++i)
#pragma unroll
      for (int j = 0; j < FJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const bool wanted = kAll || (row_of(i, e) + lrow < rows_wanted && col_of(j) < cols_left);
          bad = __builtin_fmaf(wanted ? acc[i][j][e] : 0.f, 0.f, bad);
        }
    return __any(bad != bad);
  };
  bool redo = nk > 0 && mine && not_finite(std::true_type{});
  if (redo && (rows_wanted < BM / kWM || cols_left < BN / 2)) redo = not_finite(std::false_type{});
  // Whether any wave of the block has to.  C is needed as it was only where the
  // beta term may read it, so elsewhere the waves ask after their stores.
  const auto block_redo = [&]() {
    if (redo && lane == 0) redo_flag = 1;
    wait_lgkm0();
    block_barrier();
    return redo_flag != 0;
  };
  const bool ask_first = a.beta != 0.f;
  bool again = nk > 0 && ask_first && block_redo();

  const float back = start && !kSegs ? -kUnscale : kUnscale;
#if defined(__HIP_DEVICE_COMPILE__)
  // Stores (and the beta term's loads) through buffer resources based at this
  // wave's first output row of C (and of D): a row's byte offset splits into a
  // uniform part (in an SGPR) and the lane's part (computed once).
  const float* Dm = a.D ? a.D : C;
  const int64_t ldd = a.D ? a.ldd : a.ldc;
  const __amdgpu_buffer_rsrc_t rc =
      __builtin_amdgcn_make_buffer_rsrc(C + rw0 * a.ldc + cw0, 0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(Dm + rw0 * ldd + cw0), 0, 0x7fffffff, 0x00020000);
  const int lc = static_cast<int>(lrow * a.ldc * 4), ld = static_cast<int>(lrow * ldd * 4);
  // CHECKED: the wave tile reaches M.  BETA: the beta term is read, 16 values
  // before the first is used.  Where a lane has its FJ columns side by side (N
  // is then whole float4s) they go in one access, which may start at any float:
  // 4 bytes at a time, 16 apart, were what a short K took its time for
  // (8192x6144x32 TN 76 us, now 41).
  constexpr int V = B_KC || TB::P == 1 ? 1 : FJ;
  using Out = std::conditional_t<V == 4, u32x4, std::conditional_t<V == 2, u32x2, unsigned>>;
  static_assert(V == 1 || V == TB::P, "a lane's columns");
  auto store_all = [&](auto checked, auto with_beta) {
    constexpr bool kChecked = decltype(checked)::value, kBeta = decltype(with_beta)::value;
#pragma unroll
    for (int j = 0; j < FJ; j += V) {
      const int col = col_of(j);
      if (col >= cols_left) continue;
#pragma unroll
      for (int i = 0; i < FI; ++i)
#pragma unroll
        for (int e0 = 0; e0 < 16; e0 += 16 / V) {
          float d[16 / V][V];
#pragma unroll
          for (int e = 0; e < 16 / V; ++e) {
            const int ru = row_of(i, e0 + e);
            Out x{};
            if (kBeta && !(kChecked && ru + lrow >= rows_left)) {
              const int at = ld + 4 * col, row = static_cast<int>(ru * ldd * 4);
              if constexpr (V == 4) x = __builtin_amdgcn_raw_buffer_load_b128(rd, at, row, 0);
              else if constexpr (V == 2) x = __builtin_amdgcn_raw_buffer_load_b64(rd, at, row, 0);
              else x = __builtin_amdgcn_raw_buffer_load_b32(rd, at, row, 0);
            }
            __builtin_memcpy(d[e], &x, sizeof x);
          }
#pragma unroll
          for (int e = 0; e < 16 / V; ++e) {
            const int ru = row_of(i, e0 + e);
            if (kChecked && ru + lrow >= rows_left) continue;
            float out[V];
#pragma unroll
            for (int c = 0; c < V; ++c) {
              // + 0: a zero comes out positive
              const float v = a.alpha * __builtin_fmaf(back, acc[i][j + c][e0 + e], 0.f);
              out[c] = kBeta ? v + a.beta * d[e][c] : v;
            }
            Out x;
            __builtin_memcpy(&x, out, sizeof x);
            const int at = lc + 4 * col, row = static_cast<int>(ru * a.ldc * 4);
            if constexpr (V == 4) __builtin_amdgcn_raw_buffer_store_b128(x, rc, at, row, 0);
            else if constexpr (V == 2) __builtin_amdgcn_raw_buffer_store_b64(x, rc, at, row, 0);
            else __builtin_amdgcn_raw_buffer_store_b32(x, rc, at, row, 0);
          }
        }
    }
  };
  const bool full = rows_left >= BM / kWM;
  if (mine && !again) {
    if (a.beta != 0.f) {
      if (full) store_all(std::false_type{}, std::true_type{});
      else store_all(std::true_type{}, std::true_type{});
    } else {
      if (full) store_all(std::false_type{}, std::false_type{});
      else store_all(std::true_type{}, std::false_type{});
    }
  }
#endif
  if (nk > 0 && !ask_first) again = block_redo();
  if (__builtin_expect(again, 0)) {
    // The block's tile on the fp32 MFMAs, 32x64 per wave at a time (64x64 would
    // spill the registers of three blocks per CU).
    constexpr int kM = 32 * kWM;
    static_assert(kFp32LdsFloats<A_KC, B_KC, kM, 128, THREADS> * 4 <= 2 * kStage, "LDS");
    wait_vm_lgkm0<0>();  // this wave's stores are done before others write there
    for (int t = 0; t < (BM / kM) * (BN / 128); ++t) {
      const int64_t m = m0 + kM * (t / (BN / 128)), n = n0 + 128 * (t % (BN / 128));
      if (m >= a.M || n >= a.N) continue;
      __syncthreads();  // the tile before has read its LDS
      fp32_tile<A_KC, B_KC, true, kM, 128, THREADS>(a, A, B, C, K, m, n,
                                                    reinterpret_cast<float*>(lds));
    }
  }
}

// C = alpha * sum_{s<S} P[s] + beta * D (D = C when null), the split partials
// summed in order.  P is [S][M][N] dense; four columns per thread when the
// rows allow it.
//   S > 0: float4s, S planes known when compiled, so that all their loads are
//   in flight at once (in a loop, eight planes cost eight trips to memory:
//   256x576x576 in six chunks 12.1 us, now 11.5).
//   Splits past kMaxPlanes (a long K, as over a vocabulary: 1024x1024x32768
//   has 32) follow in a loop.
constexpr int kMaxPlanes = 16;
template <int S>
__global__ __launch_bounds__(kThreads) void splitk_reduce(const float* __restrict__ P, float* C,
                                                          int64_t M, int64_t N, int64_t ldc,
                                                          int splits, float alpha, float beta,
                                                          const int64_t* dyn, int64_t dyn_base,
                                                          const float* D, int64_t ldd) {
  const int64_t per = S > 0 ? 4 : 1;
  const int64_t cols = N / per;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= M * cols) return;
  // 32-bit where it fits: a 64-bit division is some hundred instructions.
  const int64_t m = M * cols < (int64_t{1} << 32)
                        ? static_cast<uint32_t>(i) / static_cast<uint32_t>(cols)
                        : i / cols;
  const int64_t n = (i - m * cols) * per;
  // Rows past the device-side count are not needed, except up to its 16-row
  // group: a later dyn_dim 1 product reads K rounded up to 16, and those rows
  // (products of zero-filled operand rows) must hold their zeros, as the
  // unsplit tiles store them.
  if (dyn && m >= min((max(*dyn - dyn_base, int64_t{0}) + 15) / 16 * 16, M)) return;
  const int64_t plane = M * N;
  if constexpr (S > 0) {
    f32x4* dst = reinterpret_cast<f32x4*>(C + m * ldc + n);
    const f32x4* src = D ? reinterpret_cast<const f32x4*>(D + m * ldd + n) : dst;
    const f32x4 old = beta != 0.f ? *src : f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 t[S];
#pragma unroll
    for (int k = 0; k < S; ++k) t[k] = *reinterpret_cast<const f32x4*>(P + k * plane + m * N + n);
    f32x4 s = t[0];
#pragma unroll
    for (int k = 1; k < S; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] += t[k][e];
    if constexpr (S == kMaxPlanes) {  // the planes past the first kMaxPlanes
#pragma unroll 8
      for (int k = S; k < splits; ++k) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(P + k * plane + m * N + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += x[e];
      }
    }
    f32x4 out;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = beta != 0.f ? alpha * s[e] + beta * old[e] : alpha * s[e];
    *dst = out;
  } else {
    float s = P[m * N + n];
    for (int k = 1; k < splits; ++k) s += P[k * plane + m * N + n];
    float* dst = C + m * ldc + n;
    const float* src = D ? D + m * ldd + n : dst;
    *dst = beta != 0.f ? alpha * s + beta * *src : alpha * s;
  }
}

template <int S>
void launch_reduce_n(unsigned blocks, const float* P, float* C, int64_t M, int64_t N, int64_t ldc,
                     int splits, float alpha, float beta, const int64_t* dyn, int64_t dyn_base,
                     const float* D, int64_t ldd, hipStream_t st) {
  splitk_reduce<S><<<blocks, kThreads, 0, st>>>(P, C, M, N, ldc, splits, alpha, beta, dyn,
                                                dyn_base, D, ldd);
}

// Skinny NT product for M <= 8 rows (decode: one token per sequence):
// C[M,N] = alpha * A[M,K] B[N,K]^T + beta * C.  The MFMA tiles would run
// 1/128 full and only N/128 workgroups wide; this kernel is bound by streaming
// B from HBM (4*N*K bytes) instead.  A workgroup owns kSkinnyRows consecutive
// rows of B; its 4 waves take one K quarter each, every lane streams float4s of
// those rows (1 KB per row per wave load) and dots them with the M rows of A
// (a few KB, served by L1/L2).  Partial sums are reduced across the wave by
// shuffles and across the 4 waves through LDS in wave order.
constexpr int kSkinnyRows = 4;
constexpr int kSkinnyMaxM = 8;

template <int MR>
__global__ __launch_bounds__(kThreads) void gemm_skinny_nt(const float* __restrict__ A,
                                                           int64_t lda,
                                                           const float* __restrict__ B,
                                                           int64_t ldb, float* C, int64_t ldc,
                                                           int M, int64_t N, int64_t K,
                                                           float alpha, float beta,
                                                           const float* D, int64_t ldd) {
  constexpr int NR = kSkinnyRows;
  __shared__ float red[kThreads / kWave][NR * MR];
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x / kWave;
  const int64_t n0 = static_cast<int64_t>(blockIdx.x) * NR;
  const int64_t K4 = K / 4;
  const int64_t quarter = (K4 + 3) / 4;
  const int64_t kb = w * quarter;
  const int64_t ke = kb + quarter < K4 ? kb + quarter : K4;
  const f32x4* brow[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int64_t n = n0 + r < N ? n0 + r : N - 1;  // rows past N re-read the last one
    brow[r] = reinterpret_cast<const f32x4*>(B + n * ldb);
  }
  float acc[NR][MR];
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[r][m] = 0.f;

  for (int64_t i = kb + lane; i < ke; i += 2 * kWave) {
    const int64_t i1 = i + kWave;
    const bool two = i1 < ke;
    f32x4 b0[NR], b1[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      b0[r] = brow[r][i];
      b1[r] = two ? brow[r][i1] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      if (m < M) {
        const f32x4* arow = reinterpret_cast<const f32x4*>(A + m * lda);
        const f32x4 x0 = arow[i];
        const f32x4 x1 = two ? arow[i1] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          acc[r][m] += b0[r].x * x0.x + b0[r].y * x0.y + b0[r].z * x0.z + b0[r].w * x0.w;
          acc[r][m] += b1[r].x * x1.x + b1[r].y * x1.y + b1[r].z * x1.z + b1[r].w * x1.w;
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      if (m < M) {
        const float s = wave_sum(acc[r][m]);
        if (lane == 0) red[w][r * MR + m] = s;
      }
    }
  __syncthreads();
  const int idx = threadIdx.x;
  if (idx < NR * MR) {
    const int r = idx / MR, m = idx % MR;
    const int64_t n = n0 + r;
    if (m < M && n < N) {
      float s = 0.f;
#pragma unroll
      for (int q = 0; q < kThreads / kWave; ++q) s += red[q][idx];
      float* c = C + m * ldc + n;
      const float* src = D ? D + m * ldd + n : c;
      *c = beta != 0.f ? alpha * s + beta * *src : alpha * s;
    }
  }
}

template <int MR>
int launch_skinny(const float* A, int64_t lda, const float* B, int64_t ldb, float* C,
                  int64_t ldc, int64_t M, int64_t N, int64_t K, float alpha, float beta,
                  const float* D, int64_t ldd, hipStream_t st) {
  const unsigned grid = static_cast<unsigned>((N + kSkinnyRows - 1) / kSkinnyRows);
  gemm_skinny_nt<MR><<<grid, kThreads, 0, st>>>(A, lda, B, ldb, C, ldc, static_cast<int>(M), N,
                                                 K, alpha, beta, D, ldd);
  return launch_status();
}

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The K splits a product can have, which size its workspace, and the plan of
// gemm_f32_mfma.
struct Plan {
  bool big;         // unsplit: 256x128 tiles (else 128x128)
  int64_t splits;   // 1 = no K split
  int64_t kchunk;   // k per split (multiple of kBK)
};

Plan make_plan(int64_t M, int64_t N, int64_t K, int64_t batch) {
  Plan p{false, 1, 0};
  const auto split = [&](int64_t s) {
    p.kchunk = cdiv(cdiv(K, s), kBK) * kBK;
    p.splits = cdiv(K, p.kchunk);
    return p;
  };
  const int64_t big_tiles = cdiv(M, 256) * cdiv(N, 128) * batch;
  if (big_tiles >= 4 * kCUs) {  // at least two full waves of 2 blocks per CU
    p.big = true;
    return p;
  }
  const int64_t tiles = cdiv(M, 128) * cdiv(N, 128) * batch;
  const int64_t target = 6 * kCUs;  // two waves of 3 blocks per CU
  // K chunks of at least 1024 from K = 2560 up (5000x960x2560 unsplit takes
  // 170 us, in three chunks 152; 4096x1024x3072 151 and 147 in two).  A grid
  // that would fill at most half the CUs (e.g. the projections of a short
  // prefill, M = 128) is latency-bound on its one pass over K: from K = 512,
  // up to eight chunks of at least 96, then chunks of 256 (256x576x576 in six
  // chunks 12.7 us, in two 18.4; 128x1024x1024 in eight 14.6, in four 18.3).
  const bool few = 2 * tiles <= kCUs;
  // From K = 4096, chunks of at least 1024 in a whole number of waves of
  // 256x128 tiles (two per CU), at least two.
  if (batch == 1 && K >= 4096) {
    int64_t s = cdiv(4 * kCUs, big_tiles);
    while (s < 16 && (big_tiles * s) % (2 * kCUs) != 0) ++s;
    if (s >= 2 && s <= K / 1024 && (big_tiles * s) % (2 * kCUs) == 0) return split(s);
  }
  if (batch == 1 && tiles < target && K >= (few ? 512 : 2560)) {
    const int64_t chunk = few ? std::min<int64_t>(256, std::max<int64_t>(96, K / 8)) : 1024;
    const int64_t s = std::min({int64_t{16}, cdiv(target, tiles), K / chunk});
    if (s >= 2) return split(s);
  }
  return p;
}

// Launch plan for gemm_f32_split: the tile shape and the K split of least
// predicted time.  The prediction counts what the busiest CU does, in
// microseconds: whole rounds of as many blocks as fit a CU, then what is
// left, a stage of 16 k costing `stage[n - 1]` while n blocks share the CU
// (`alone` when at most half the CUs have one, and clocks are high), and a
// round `ends` more for its first loads and its stores, which only other
// blocks on the same CU can cover.  A split adds its reduction: one launch
// and S + 1 planes of C through HBM.  The constants are fitted to times of
// 45 products (M, N 32 to 151936, K 64 to 8192, three layouts) on the tiles
// with 1 to 16 splits; choosing by them is on average 0.5% slower than the
// best of those, at worst 4%.  The 512-thread tile is for grids of one block
// per CU, where one wave per SIMD cannot issue fast enough (a stage alone
// takes 0.37-0.44 us instead of 0.53: when it was added 256x576x576 went 13.2
// -> 12.1 us, 2048x576x1536 33.1 -> 29.7, 509x3072x1024 31.7 -> 28.6,
// 1000x2048x2048 56.4 -> 52.4); with more blocks it is slower (4096x3072x1024
// 151 against 130 us).
struct SplitPlan {
  int tile;         // index into kTiles
  int64_t splits;   // 1 = no K split
  int64_t kchunk;   // k per split, whole pairs of stages
};
struct TileCost {
  int64_t bm, bn;
  int per_cu;
  double stage[3], alone, ends;
};
constexpr TileCost kTiles[4] = {{128, 128, 1, {0.61}, 0.44, 2.8},  // 512 threads
                                {128, 128, 3, {0.92, 1.17, 1.89}, 0.53, 4.56},
                                {256, 128, 2, {1.16, 2.19}, 0.78, 6.01},
                                {256, 256, 1, {1.92}, 1.38, 27.3}};

double predicted_us(const TileCost& t, int64_t M, int64_t N, int64_t K, int64_t batch,
                    int64_t splits) {
  const double stages = static_cast<double>(cdiv(K, 16));
  const int64_t blocks = cdiv(M, t.bm) * cdiv(N, t.bn) * batch * splits;
  const int64_t round = int64_t{t.per_cu} * kCUs;
  double us = static_cast<double>(blocks / round) * (t.stage[t.per_cu - 1] * stages + t.ends);
  const int64_t rest = blocks % round;
  if (rest > 0) {
    const int64_t n = cdiv(rest, kCUs);
    if (blocks == rest && 2 * rest <= kCUs)
      us += t.alone * stages + 3.0;
    else
      us += t.stage[n - 1] * stages + t.ends * static_cast<double>(n) / t.per_cu;
  }
  return us;
}

// `room`: the partial products that the workspace holds; `tiles`: the first
// of kTiles that may be used.
// From K = 4096 the split is all of `room`: shorter partial sums are also what
// keeps the error of long ones down (a weight gradient's terms vary along the
// tokens; 1024x2048x32768 in 8 chunks instead of 16 was 1.5 times further
// from 64-bit sums, and 4% faster).  Below that, a grid of few tiles is summed
// in segments of at most kMaxChain from K = 512, which the 512-thread tile does
// by itself and the others only by a split: 2048x1024x2048 unsplit was 1.66
// times further from 64-bit sums than in eight fp32 chunks of 256.
constexpr int64_t kMaxChain = 352;  // 0.85 sqrt(352 / 256) = 1.0 of such a chunk's error

SplitPlan make_split_plan(int64_t M, int64_t N, int64_t K, int64_t batch, int64_t room,
                          int tiles) {
  SplitPlan best{1, 1, 0};
  double least = 1e30;
  const bool short_chains =
      room > 1 && K >= 512 && K < 4096 && 2 * cdiv(M, 128) * cdiv(N, 128) <= kCUs;
  for (int t = 0; t < tiles; ++t)
    for (int64_t s = K >= 4096 ? room : 1; s <= room; ++s) {
      const int64_t chunk = s > 1 ? cdiv(cdiv(K, s), 32) * 32 : K;
      const int64_t n = s > 1 ? cdiv(K, chunk) : 1;  // at most s
      if (t == 0 && cdiv(M, 128) * cdiv(N, 128) * batch * n > kCUs) continue;  // one round only
      if (t > 0 && short_chains && chunk > kMaxChain) continue;
      double us = predicted_us(kTiles[t], M, N, chunk, batch, n);
      if (n > 1) us += 2.45 + static_cast<double>((n + 1) * M * N) * 4 / 5.21e6;
      if (us < least) {
        least = us;
        best = SplitPlan{t, n, n > 1 ? chunk : 0};
      }
    }
  return best;
}

template <bool A_KC, bool B_KC, int BM, int BN, int OCC>
int launch(const GemmArgs& a, int64_t ny, bool vec, hipStream_t st) {
  dim3 grid(static_cast<unsigned>(a.tiles_m) * a.tiles_n, static_cast<unsigned>(ny));
  if (vec)
    gemm_f32_mfma<A_KC, B_KC, true, BM, BN, OCC><<<grid, kThreads, 0, st>>>(a);
  else
    gemm_f32_mfma<A_KC, B_KC, false, BM, BN, OCC><<<grid, kThreads, 0, st>>>(a);
  return launch_status();
}

template <int BM, int BN, int OCC>
int launch_t(GemmArgs a, bool a_kc, bool b_kc, int64_t ny, bool vec, hipStream_t st) {
  a.tiles_m = static_cast<int>(cdiv(a.M, BM));
  a.tiles_n = static_cast<int>(cdiv(a.N, BN));
  if (a_kc && b_kc) return launch<true, true, BM, BN, OCC>(a, ny, vec, st);
  if (a_kc && !b_kc) return launch<true, false, BM, BN, OCC>(a, ny, vec, st);
  if (!a_kc && !b_kc) return launch<false, false, BM, BN, OCC>(a, ny, vec, st);
  return launch<false, true, BM, BN, OCC>(a, ny, vec, st);
}

template <bool A_KC, bool B_KC, int BM, int BN, int THREADS, int OCC>
int launch_split_t(GemmArgs a, int64_t ny, hipStream_t st) {
  a.tiles_m = static_cast<int>(cdiv(a.M, BM));
  a.tiles_n = static_cast<int>(cdiv(a.N, BN));
  dim3 grid(static_cast<unsigned>(a.tiles_m) * a.tiles_n, static_cast<unsigned>(ny));
  gemm_f32_split<A_KC, B_KC, BM, BN, THREADS, OCC><<<grid, THREADS, 0, st>>>(a);
  return launch_status();
}

template <int BM, int BN, int THREADS, int OCC>
int launch_split_tile(const GemmArgs& a, bool a_kc, bool b_kc, int64_t ny, hipStream_t st) {
  if (a_kc && b_kc) return launch_split_t<true, true, BM, BN, THREADS, OCC>(a, ny, st);
  if (a_kc && !b_kc) return launch_split_t<true, false, BM, BN, THREADS, OCC>(a, ny, st);
  if (!a_kc && !b_kc) return launch_split_t<false, false, BM, BN, THREADS, OCC>(a, ny, st);
  return launch_split_t<false, true, BM, BN, THREADS, OCC>(a, ny, st);
}

int launch_split(const GemmArgs& a, int tile, bool a_kc, bool b_kc, int64_t ny, hipStream_t st) {
  return tile == 0   ? launch_split_tile<128, 128, 512, 2>(a, a_kc, b_kc, ny, st)
         : tile == 1 ? launch_split_tile<128, 128, 256, 3>(a, a_kc, b_kc, ny, st)
         : tile == 2 ? launch_split_tile<256, 128, 256, 2>(a, a_kc, b_kc, ny, st)
                     : launch_split_tile<256, 256, 256, 1>(a, a_kc, b_kc, ny, st);
}

// How many of kTiles gemm_f32_split can use for these operands: none unless
// their rows are float4 rows that end on a whole float4; else those for which
// every byte offset inside a block's operand stage and output tile (the
// tile's rows of a K-contiguous operand and of C, 16 k of the other) stays
// below 2^31.
int split_tiles(const GemmArgs& a, bool a_kc, bool b_kc, bool vec) {
  if (!vec || (a_kc ? a.K : a.M) % 4 != 0 || (b_kc ? a.K : a.N) % 4 != 0) return 0;
  const auto fits = [&](int64_t rows) {
    const int64_t top = (int64_t{1} << 29) - 1024;  // floats
    return (a_kc ? rows - 1 : 16) * a.lda < top && (b_kc ? rows - 1 : 16) * a.ldb < top &&
           rows * std::max(a.ldc, a.D ? a.ldd : int64_t{0}) < top;
  };
  return fits(256) ? 4 : fits(128) ? 2 : 0;
}

int check_args(int transa, int transb, int64_t M, int64_t N, int64_t K, const float* A,
               int64_t lda, const float* B, int64_t ldb, const float* C, int64_t ldc,
               int64_t batch) {
  if (M < 0 || N < 0 || K < 0 || batch < 1) return EMBER_EINVAL;
  if (M == 0 || N == 0) return EMBER_OK;
  if (!C || (K > 0 && (!A || !B))) return EMBER_EINVAL;
  if (lda < (transa ? M : K) || ldb < (transb ? K : N) || ldc < N) return EMBER_EINVAL;
  if (cdiv(M, 128) * cdiv(N, 128) > 0x7fffffff || batch > 65535) return EMBER_EINVAL;
  return EMBER_OK;
}

}  // namespace

extern "C" size_t ember_gemm_f32_workspace_bytes(int64_t M, int64_t N, int64_t K,
                                                 int64_t batch) {
  if (M <= 0 || N <= 0 || K <= 0 || batch < 1) return 0;
  const Plan p = make_plan(M, N, K, batch);
  return p.splits > 1 ? static_cast<size_t>(p.splits * M * N) * sizeof(float) : 0;
}

namespace {

// One GEMM call; `dyn` (may be null) is the device-side extent of GemmArgs.
int gemm_run(int transa, int transb, int64_t M, int64_t N, int64_t K, float alpha,
             const float* A, int64_t lda, int64_t sA, const float* B, int64_t ldb, int64_t sB,
             float beta, float* C, int64_t ldc, int64_t sC, int64_t batch, void* workspace,
             size_t workspace_bytes, const int64_t* dyn, int64_t dyn_base, int dyn_dim,
             const float* D, int64_t ldd, hipStream_t st) {
  int rc = EMBER_OK;
  GemmArgs a{A, B, C, M, N, K, lda, ldb, ldc, sA, sB, sC, 0, alpha, beta, 0, 0};
  a.dyn = dyn;
  a.dyn_base = dyn_base;
  a.dyn_dim = dyn_dim;
  a.D = D;
  a.ldd = ldd;
  const bool vec = aligned16(A) && aligned16(B) && (lda % 4 == 0) && (ldb % 4 == 0) &&
                   (batch == 1 || (sA % 4 == 0 && sB % 4 == 0));
  const bool a_kc = !transa, b_kc = transb != 0;
  if (!dyn && batch == 1 && M <= kSkinnyMaxM && a_kc && b_kc && vec && K > 0 && K % 4 == 0 &&
      N <= int64_t{kSkinnyRows} * 0x7fffffff) {
    auto skinny = M == 1 ? launch_skinny<1>
                  : M == 2 ? launch_skinny<2>
                  : M <= 4 ? launch_skinny<4>
                           : launch_skinny<8>;
    return skinny(A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, D, ldd, st);
  }
  // Partial products need room for themselves, and a K known on the host.
  const Plan p = make_plan(M, N, K, batch);
  const bool room = p.splits > 1 && !(dyn && dyn_dim == 1) && workspace &&
                    workspace_bytes >= static_cast<size_t>(p.splits * M * N) * sizeof(float);
  const int tiles = split_tiles(a, a_kc, b_kc, vec);
  const bool fast = tiles > 0;
  SplitPlan sp{0, 1, 0};
  if (fast) sp = make_split_plan(M, N, K, batch, room ? p.splits : 1, tiles);
  const int64_t splits = fast ? sp.splits : room ? p.splits : 1;
  const int64_t kchunk = fast ? sp.kchunk : p.kchunk;
  if (splits > 1) {
    // Split s computes A[:, s*kchunk ...] B[s*kchunk ..., :] into plane s.
    GemmArgs pa = a;
    pa.C = static_cast<float*>(workspace);
    pa.ldc = N;
    pa.sA = a_kc ? kchunk : kchunk * lda;
    pa.sB = b_kc ? kchunk : kchunk * ldb;
    pa.sC = M * N;
    pa.kchunk = kchunk;
    pa.alpha = 1.f;
    pa.beta = 0.f;
    pa.D = nullptr;
    if ((rc = fast ? launch_split(pa, sp.tile, a_kc, b_kc, splits, st)
                   : launch_t<128, 128, 3>(pa, a_kc, b_kc, splits, vec, st)))
      return rc;
    const bool rvec = (N % 4 == 0) && (ldc % 4 == 0) && aligned16(C) &&
                      (!D || (ldd % 4 == 0 && aligned16(D)));
    const int64_t items = M * (rvec ? N / 4 : N);
    const unsigned blocks = static_cast<unsigned>(cdiv(items, kThreads));
    const int64_t* rdyn = dyn_dim == 0 ? dyn : nullptr;
    using Reduce = decltype(&launch_reduce_n<0>);
    constexpr Reduce kReduce[kMaxPlanes + 1] = {
        launch_reduce_n<0>,  launch_reduce_n<1>,  launch_reduce_n<2>,  launch_reduce_n<3>,
        launch_reduce_n<4>,  launch_reduce_n<5>,  launch_reduce_n<6>,  launch_reduce_n<7>,
        launch_reduce_n<8>,  launch_reduce_n<9>,  launch_reduce_n<10>, launch_reduce_n<11>,
        launch_reduce_n<12>, launch_reduce_n<13>, launch_reduce_n<14>, launch_reduce_n<15>,
        launch_reduce_n<16>};
    kReduce[rvec ? std::min<int64_t>(splits, kMaxPlanes) : 0](
        blocks, static_cast<const float*>(workspace), C, M, N, ldc, static_cast<int>(splits), alpha,
        beta, rdyn, dyn_base, D, ldd, st);
    return launch_status();
  }
  if (fast) return launch_split(a, sp.tile, a_kc, b_kc, batch, st);
  if (p.big) return launch_t<256, 128, 2>(a, a_kc, b_kc, batch, vec, st);
  return launch_t<128, 128, 3>(a, a_kc, b_kc, batch, vec, st);
}

}  // namespace

extern "C" int ember_gemm_f32_ws(int transa, int transb, int64_t M, int64_t N, int64_t K,
                                 float alpha, const float* A, int64_t lda, int64_t sA,
                                 const float* B, int64_t ldb, int64_t sB, float beta, float* C,
                                 int64_t ldc, int64_t sC, int64_t batch, void* workspace,
                                 size_t workspace_bytes, ember_stream_t s) {
  int rc = check_args(transa, transb, M, N, K, A, lda, B, ldb, C, ldc, batch);
  if (rc || M == 0 || N == 0) return rc;
  return gemm_run(transa, transb, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch,
                  workspace, workspace_bytes, nullptr, 0, 0, nullptr, 0, as_stream(s));
}

extern "C" int ember_gemm_f32_add(int transa, int transb, int64_t M, int64_t N, int64_t K,
                                  float alpha, const float* A, int64_t lda, const float* B,
                                  int64_t ldb, const float* D, int64_t ldd, float* C, int64_t ldc,
                                  void* workspace, size_t workspace_bytes, ember_stream_t s) {
  int rc = check_args(transa, transb, M, N, K, A, lda, B, ldb, C, ldc, 1);
  if (rc || M == 0 || N == 0) return rc;
  if (!D || ldd < N) return EMBER_EINVAL;
  if (D != C) {  // D is C itself or lies wholly apart from it
    const auto c0 = reinterpret_cast<uintptr_t>(C), d0 = reinterpret_cast<uintptr_t>(D);
    const uintptr_t c1 = c0 + static_cast<uintptr_t>((M - 1) * ldc + N) * sizeof(float);
    const uintptr_t d1 = d0 + static_cast<uintptr_t>((M - 1) * ldd + N) * sizeof(float);
    if (d0 < c1 && c0 < d1) return EMBER_EINVAL;
  } else if (ldd != ldc) {
    return EMBER_EINVAL;
  }
  return gemm_run(transa, transb, M, N, K, alpha, A, lda, 0, B, ldb, 0, 1.0f, C, ldc, 0, 1,
                  workspace, workspace_bytes, nullptr, 0, 0, D, ldd, as_stream(s));
}

extern "C" int ember_gemm_f32_dyn(int transa, int transb, int64_t M, int64_t N, int64_t K,
                                  float alpha, const float* A, int64_t lda, const float* B,
                                  int64_t ldb, float beta, float* C, int64_t ldc,
                                  const int64_t* count, int64_t base, int dim, void* workspace,
                                  size_t workspace_bytes, ember_stream_t s) {
  int rc = check_args(transa, transb, M, N, K, A, lda, B, ldb, C, ldc, 1);
  if (rc) return rc;
  if (!count || (dim != 0 && dim != 1) || base < 0) return EMBER_EINVAL;
  // 16-byte rows, and K in whole 16-k stages.
  const bool a_kc = !transa, b_kc = transb != 0;
  if (!aligned16(A) || !aligned16(B) || lda % 4 != 0 || ldb % 4 != 0 || K % 16 != 0 ||
      (!a_kc && M % 4 != 0) || (!b_kc && N % 4 != 0))
    return EMBER_EINVAL;
  if (M == 0 || N == 0) return EMBER_OK;
  return gemm_run(transa, transb, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 1,
                  workspace, workspace_bytes, count, base, dim, nullptr, 0, as_stream(s));
}

extern "C" int ember_gemm_f32(int transa, int transb, int64_t M, int64_t N, int64_t K,
                              float alpha, const float* A, int64_t lda, int64_t sA,
                              const float* B, int64_t ldb, int64_t sB, float beta, float* C,
                              int64_t ldc, int64_t sC, int64_t batch, ember_stream_t s) {
  return ember_gemm_f32_ws(transa, transb, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc,
                           sC, batch, nullptr, 0, s);
}
