// Batched fp32 GEMM on the CDNA4 matrix cores.
//
// C[b] = alpha * A[b] * B[b] + beta * C[b] for small and medium matrices, many
// per launch: the chunked score matrices S = A * N^T, their backward products
// dA = dS * N and dN = dS^T * A, and the `linear` operator.  The fp32 operands are split into three bf16 parts on their way
// into LDS and multiplied by six v_mfma_f32_16x16x32_bf16 per tile pair and 32 values of k (split_mfma.h: why, and what it
// does to the rounding).
//
// Bound by the matrix cores (96 cycles per 16 x 16 x 32 tile product).  Per depth-32 tile step a 256 x 128 workgroup of
// eight waves takes in 48 KiB of fp32 operands and issues 2 x 96 matrix instructions per SIMD (3072 cycles), beside which the
// split (44 vector instructions per eight values, one pass over the step's 12288 values: about 1060 cycles per SIMD) and the
// LDS traffic (72 KiB written, 192 KiB read: 1300 cycles) fit.  The step is double buffered: while the waves multiply tile
// t, they split tile t + 1, which is in registers, into the other buffer and issue the loads of tile t + 2.
//
// LDS layout: [part][k group g = 0..3][row], 16 bytes each = the eight values of k that a lane of lane group g feeds to one
// instruction (which k a slot stands for is free as long as both operands agree: slot j of group g is
// k = 4 g + (j & 3) + 16 (j >> 2), so that four lanes read 64 contiguous bytes of a row).  Row r of group g lies at place
// r ^ s(g), s = {0, 2, 12, 14}: the reads of a lane set {0-3, 12-15, 20-27} still touch 16 different places (a xor by such a
// value maps {4..11} to itself), and eight consecutive lanes that write two rows of four groups touch eight.
//
// HALF variants (config.half_precision: both operands hold float16 numbers): one fp16 part instead of three bf16 ones
// (exact), one v_mfma_f32_16x16x32_f16 per tile pair.  Sums stay fp32; the result is rounded to a float16 number when it is
// stored.
#include <type_traits>

#include "pbg_internal.h"
#include "mfma_tiles.h"
#include "split_mfma.h"

namespace pbg {
namespace {

constexpr int kStepK = 32;    // values of k per tile step
constexpr int kFoldSteps = 4;  // tile steps per partial sum (128 values of k)

__device__ __forceinline__ int group_swizzle(int g) { return (g & 1) * 2 + (g >> 1) * 12; }

// One operand's tile: ROWS rows (of A, or columns of B) by 32 values of k, by THREADS threads.  A unit is one row's eight
// values of one k group; a thread owns kUnits of them.
//   KMAJOR = false: element (r, k) at base[r * ld + k]   (k contiguous): four adjacent lanes own a row's four groups
//   KMAJOR = true : element (r, k) at base[k * ld + r]   (r contiguous): a wave owns one group of 64 * kUnits adjacent rows
// Rows past rmax are read from clamped addresses: they only feed entries of C that are never stored.
template <int ROWS, int THREADS, bool KMAJOR, bool HALF>
struct Operand {
  static constexpr int kUnits = ROWS * 4 / THREADS;
  static constexpr int kParts = HALF ? 1 : 3;
  float v[kUnits][8];
  const float* base;
  int ld, row[kUnits], rmax;
  bool vec;  // every vector load is aligned, and whole or absent

  static __device__ __forceinline__ int unit_group(int u) {
    // (of a k-major operand: the same for the wave, so that a row's address is a scalar and the lane's offset 32 bits)
    return KMAJOR ? __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3) : (threadIdx.x + u * THREADS) & 3;
  }
  static __device__ __forceinline__ int unit_row(int u) {
    if (KMAJOR) return (threadIdx.x >> 8) * (64 * kUnits) + (threadIdx.x & 63) * kUnits + u;
    return (threadIdx.x + u * THREADS) >> 2;
  }

  __device__ __forceinline__ void start(const float* base_, int ld_, int r0, int rmax_, int kmax, int aligned_to) {
    base = base_;
    ld = ld_;
    rmax = rmax_;
    vec = KMAJOR ? (kUnits == 1 || (aligned_to >= 2 && rmax % 2 == 0)) : aligned_to >= 4 && kmax % 4 == 0 && kmax > 0;
#pragma unroll
    for (int u = 0; u < kUnits; ++u) row[u] = min(r0 + unit_row(u), rmax - 1);
    if (KMAJOR && kUnits == 2 && vec) row[0] = min(r0 + unit_row(0), rmax - 2);
  }

  // Whole vectors of a step; of a k-major operand only the first call fetches (all units).  LAST: the step may reach past
  // kmax: those vectors are read from inside and zeroed.
  template <bool LAST>
  __device__ __forceinline__ void fetch_vec(int k0, int u, int kmax) {
    if constexpr (!KMAJOR) {
      const int k = k0 + 4 * unit_group(u);
      const float* p = base + (int64_t)row[u] * ld;
      float4 x = *reinterpret_cast<const float4*>(p + (LAST ? min(k, kmax - 4) : k));
      float4 y = *reinterpret_cast<const float4*>(p + (LAST ? min(k + 16, kmax - 4) : k + 16));
      if constexpr (LAST) {
        if (k >= kmax) x = make_float4(0.f, 0.f, 0.f, 0.f);
        if (k + 16 >= kmax) y = make_float4(0.f, 0.f, 0.f, 0.f);
      }
      v[u][0] = x.x; v[u][1] = x.y; v[u][2] = x.z; v[u][3] = x.w;
      v[u][4] = y.x; v[u][5] = y.y; v[u][6] = y.z; v[u][7] = y.w;
    } else if (u == 0) {
      const uint32_t at = 4u * (uint32_t)row[0];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int k = k0 + 4 * unit_group(0) + (j & 3) + 16 * (j >> 2);
        const char* q = reinterpret_cast<const char*>(base + (int64_t)(LAST ? min(k, kmax - 1) : k) * ld);
        if constexpr (kUnits == 2) {
          const float2 x = *reinterpret_cast<const float2*>(q + at);
          v[0][j] = x.x;
          v[1][j] = x.y;
        } else {
          v[0][j] = *reinterpret_cast<const float*>(q + at);
        }
        if constexpr (LAST) {
#pragma unroll
          for (int w = 0; w < kUnits; ++w) v[w][j] = k < kmax ? v[w][j] : 0.f;
        }
      }
    }
  }

  __device__ __forceinline__ void fetch(int k0, int kmax) {
    if (vec) {
      if (k0 + kStepK <= kmax) {
#pragma unroll
        for (int u = 0; u < kUnits; ++u) fetch_vec<false>(k0, u, kmax);
      } else {
#pragma unroll
        for (int u = 0; u < kUnits; ++u) fetch_vec<true>(k0, u, kmax);
      }
      return;
    }
    // unaligned rows, or k no multiple of 4 along them: value by value, zero past kmax
#pragma unroll
    for (int u = 0; u < kUnits; ++u)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int k = k0 + 4 * unit_group(u) + (j & 3) + 16 * (j >> 2);
        const int at = min(k, kmax - 1);
        const float x = KMAJOR ? base[(int64_t)at * ld + row[u]] : base[(int64_t)row[u] * ld + at];
        v[u][j] = k < kmax ? x : 0.f;
      }
  }

  __device__ __forceinline__ void stash(uint4* tile, int u) const {
    const int g = unit_group(u);
    // (a clamped row pair of a k-major operand keeps its own two places)
    uint4* dst = tile + g * ROWS + (unit_row(u) ^ group_swizzle(g));
    if constexpr (HALF) {
      const half8v h = pack_half8(v[u]);
      dst[0] = __builtin_bit_cast(uint4, h);
    } else {
      const Split8 s = split8(v[u]);
      dst[0] = s.h;
      dst[4 * ROWS] = s.m;
      dst[8 * ROWS] = s.l;
    }
  }
};

// WM x WN waves of TM x TN tiles of 16 x 16.
template <int WM, int WN, int TM, int TN, bool HALF>
struct GemmShape {
  static constexpr int kThreads = 64 * WM * WN;
  static constexpr int kRowsA = WM * TM * 16, kRowsB = WN * TN * 16;
  static constexpr int kParts = HALF ? 1 : 3;
  static constexpr int kStage = kParts * 4 * (kRowsA + kRowsB);  // 16-byte words per buffer
  static constexpr size_t kLds = 2 * sizeof(uint4) * kStage;
};

// BFIRST: GemmArgs.b_first
template <int WM, int WN, int TM, int TN, bool A_KMAJOR, bool B_KMAJOR, bool HALF, bool BFIRST>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_kernel(GemmArgs g, int tiles_m, int tiles_n, int a_align, int b_align) {
  using Shape = GemmShape<WM, WN, TM, TN, HALF>;
  constexpr int P = Shape::kParts;
  constexpr int RA = Shape::kRowsA, RB = Shape::kRowsB;
  extern __shared__ __attribute__((aligned(16))) uint4 gemm_lds[];

  // Workgroups are dealt round robin to the 8 dies, each with an L2 of its own: die x takes a contiguous stretch of tiles,
  // so that the tiles of one product (which share its operands) meet in one L2.
  const unsigned total = gridDim.x, die = blockIdx.x & 7, share = total >> 3, more = total & 7;
  const unsigned tile = die * share + (die < more ? die : more) + (blockIdx.x >> 3);
  const unsigned per = (unsigned)tiles_m * tiles_n;
  const unsigned batch = tile / per, in = tile - batch * per;
  const int m0 = (int)(in / tiles_n) * RA, n0 = (int)(in % tiles_n) * RB;

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm0 = (wave / WN) * (TM * 16);
  const int wn0 = (wave % WN) * (TN * 16);
  const int nk = (g.k + kStepK - 1) / kStepK;

  Operand<RA, Shape::kThreads, A_KMAJOR, HALF> oa;
  Operand<RB, Shape::kThreads, B_KMAJOR, HALF> ob;
  oa.start(g.a + (int64_t)batch * g.stride_a, g.lda, m0, g.m, g.k, a_align);
  ob.start(g.b + (int64_t)batch * g.stride_b + (g.b_index ? g.b_index[batch] * g.b_index_stride : 0), g.ldb, n0, g.n, g.k, b_align);

  // Blocked summation: `acc` collects kFoldSteps steps, then is folded into `tot`.  A single accumulator over k = 1000
  // rounds in proportion to the running sum at every step, coherently when the terms are alike (a power-law batch repeats
  // the same rows); two levels keep the error at that of a blocked CPU BLAS.
  float4v acc[TM][TN], tot[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      acc[i][j] = (float4v){0.f, 0.f, 0.f, 0.f};
      tot[i][j] = (float4v){0.f, 0.f, 0.f, 0.f};
    }

  auto stash = [&](uint4* buf, int u) {
    if (u < oa.kUnits) oa.stash(buf, u);
    else ob.stash(buf + P * 4 * RA, u - oa.kUnits);
  };
  constexpr int kUnits = decltype(oa)::kUnits + decltype(ob)::kUnits;
  const int lg = lane >> 4, lr = (lane & 15) ^ group_swizzle(lg);
  const int at_a = lg * RA + wm0 + lr, at_b = P * 4 * RA + lg * RB + wn0 + lr;

  if (nk > 0) {
    oa.fetch(0, g.k);
    ob.fetch(0, g.k);
#pragma unroll
    for (int u = 0; u < kUnits; ++u) stash(gemm_lds, u);
    if (nk > 1) {
      oa.fetch(kStepK, g.k);
      ob.fetch(kStepK, g.k);
    }
  }
  lds_barrier();

  // One step: products of tile kt; MORE: tile kt + 1 is split into the other buffer; FULL: tile kt + 2 is fetched, all of it
  // whole vectors inside the operands (then the step is one straight line, in which the scheduler spreads the split over
  // the matrix instructions).
  auto step = [&](int kt, auto more, auto full) {
    const uint4* cur = gemm_lds + (kt & 1) * Shape::kStage;
    uint4* next = gemm_lds + ((kt & 1) ^ 1) * Shape::kStage;
    uint4 fb[TN][P];
#pragma unroll
    for (int p = P - 1; p >= 0; --p)
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[j][p] = cur[at_b + p * 4 * RB + j * 16];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      uint4 fa[P];
#pragma unroll
      for (int p = 0; p < P; ++p) fa[p] = cur[at_a + p * 4 * RA + i * 16];
      if constexpr (HALF) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8v, fa[0]), __builtin_bit_cast(half8v, fb[j][0]), acc[i][j], 0, 0, 0);
      } else {
        // part pairs in ascending size; the tiles of a pair follow each other, so that no instruction waits for the last
        constexpr int first[6] = {0, 2, 1, 0, 1, 0}, second[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
        for (int q = 0; q < 6; ++q)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, fa[BFIRST ? second[q] : first[q]]),
                                                                __builtin_bit_cast(bf16x8, fb[j][BFIRST ? first[q] : second[q]]), acc[i][j], 0, 0, 0);
      }
      if constexpr (decltype(more)::value) {
#pragma unroll
        for (int u = i * kUnits / TM; u < (i + 1) * kUnits / TM; ++u) {
          stash(next, u);
          if constexpr (decltype(full)::value) {
            // (a k-major operand's loads fill all its units: they go out behind its last one)
            if (u < oa.kUnits) {
              if (!A_KMAJOR) oa.template fetch_vec<false>((kt + 2) * kStepK, u, g.k);
              else if (u == oa.kUnits - 1) oa.template fetch_vec<false>((kt + 2) * kStepK, 0, g.k);
            } else {
              if (!B_KMAJOR) ob.template fetch_vec<false>((kt + 2) * kStepK, u - oa.kUnits, g.k);
              else if (u == kUnits - 1) ob.template fetch_vec<false>((kt + 2) * kStepK, 0, g.k);
            }
          }
        }
      }
    }
    if constexpr (decltype(more)::value) {
#pragma unroll
      for (int q = 0; q < TM * TN * (HALF ? 1 : 6); ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a matrix instruction
        __builtin_amdgcn_sched_group_barrier(0x002, HALF ? 6 : 2, 0);  // vector instructions in its shadow
      }
    }
    if constexpr (decltype(more)::value && !decltype(full)::value) {
      if (kt + 2 < nk) {
        oa.fetch((kt + 2) * kStepK, g.k);
        ob.fetch((kt + 2) * kStepK, g.k);
      }
    }
    if ((kt & (kFoldSteps - 1)) == kFoldSteps - 1) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          tot[i][j] += acc[i][j];
          acc[i][j] = (float4v){0.f, 0.f, 0.f, 0.f};
        }
    }
    lds_barrier();
  };
  int kt = 0;
  const int straight = oa.vec && ob.vec ? g.k / kStepK - 2 : 0;
  for (; kt < straight; ++kt) step(kt, std::true_type{}, std::true_type{});
  for (; kt < nk - 1; ++kt) step(kt, std::true_type{}, std::false_type{});
  if (kt < nk) step(kt, std::false_type{}, std::false_type{});

  // D[i = 4 * (lane / 16) + r][j = lane % 16] lives in register r of the lane.
  float* __restrict__ c = g.c + (int64_t)batch * g.stride_c;
  if constexpr (!HALF) {
    // The split turns an infinite value (and one that rounds up to an infinite bf16 number) into NaN: a wave that finds one
    // in its part of the tile sums it again, entry by entry, without the split.
    float any = 0.f;  // NaN once an infinite or NaN value was added times 0
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) any = fmaf(0.f, tot[i][j][r] + acc[i][j][r], any);
    if (__any(any != 0.f)) {  // (NaN compares unequal)
      const int64_t step_a = A_KMAJOR ? g.lda : 1, row_a = A_KMAJOR ? 1 : g.lda;
      const int64_t step_b = B_KMAJOR ? g.ldb : 1, row_b = B_KMAJOR ? 1 : g.ldb;
#pragma unroll 1
      for (int e = 0; e < TM * TN * 4; ++e) {
        const int row = m0 + wm0 + (e / (4 * TN)) * 16 + 4 * (lane >> 4) + (e & 3);
        const int col = n0 + wn0 + (e / 4 % TN) * 16 + (lane & 15);
        if (row < g.m && col < g.n) {
          float* dst = c + (int64_t)row * g.ldc + col;
          const float* pa = oa.base + row * row_a;
          const float* pb = ob.base + col * row_b;
          float sum = 0.f, part = 0.f;
#pragma unroll 1
          for (int k = 0; k < g.k; ++k, pa += step_a, pb += step_b) {
            part = fmaf(*pa, *pb, part);
            if ((k + 1) % (kFoldSteps * kStepK) == 0) {
              sum += part;
              part = 0.f;
            }
          }
          const float v = g.alpha * (sum + part);
          *dst = g.beta != 0.f ? v + g.beta * *dst : v;
        }
      }
      return;
    }
  }
  auto store = [&](int i, int j, int r, auto&& finish) {
    const int col = n0 + wn0 + j * 16 + (lane & 15);
    const int row = m0 + wm0 + i * 16 + 4 * (lane >> 4) + r;
    if (row < g.m && col < g.n) {
      const float v = finish(g.alpha * (tot[i][j][r] + acc[i][j][r]));
      c[(int64_t)row * g.ldc + col] = HALF ? (float)(_Float16)v : v;
    }
  };
  if (g.beta == 0.f) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) store(i, j, r, [](float v) { return v; });
    return;
  }
  // What is there already is read a row of tiles ahead of its use, from clamped addresses: a read behind each store (which it
  // might alias) made 64 round trips of the epilogue, 25 us of a workgroup's 115 (80 products of 1000 x 1024 x 1100: 1.18 -> 1.03 ms;
  // float16 0.69 -> 0.51).
  float old[2][TN][4];
  auto read_old = [&](int i, float(&o)[TN][4]) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        o[j][r] = c[(int64_t)min(m0 + wm0 + i * 16 + 4 * (lane >> 4) + r, g.m - 1) * g.ldc + min(n0 + wn0 + j * 16 + (lane & 15), g.n - 1)];
  };
  read_old(0, old[0]);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    if (i + 1 < TM) read_old(i + 1, old[(i + 1) & 1]);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        // HALF: the product is a Half tensor of its own before autograd adds it to what is there
        // (two roundings: of the product, then of the sum)
        store(i, j, r, [&](float v) { return (HALF ? (float)(_Float16)v : v) + g.beta * old[i & 1][j][r]; });
  }
}

// Floats that every row start of an operand is aligned to (4, 2 or 1).
int row_alignment(const float* p, int ld, int64_t stride, int64_t more) {
  const uint64_t bits = ((uintptr_t)p >> 2) | (uint64_t)ld | (uint64_t)stride | (uint64_t)more;
  return bits % 4 == 0 ? 4 : bits % 2 == 0 ? 2 : 1;
}

template <int WM, int WN, int TM, int TN, bool AK, bool BK, bool HALF, bool BFIRST = false>
int launch_one(const GemmArgs& g, hipStream_t stream) {
  using Shape = GemmShape<WM, WN, TM, TN, HALF>;
  static LdsLimit limit;
  auto kernel = gemm_kernel<WM, WN, TM, TN, AK, BK, HALF, BFIRST>;
  const int rc = reserve_lds((const void*)kernel, &limit, Shape::kLds);
  if (rc != PBG_OK) return rc;
  const int64_t tm = ceil_div(g.m, Shape::kRowsA), tn = ceil_div(g.n, Shape::kRowsB);
  if (tm * tn * g.batch > 0x7fffffff) return fail(PBG_ERR_UNSUPPORTED, "gemm_f32: more than 2^31 - 1 tiles");
  hipLaunchKernelGGL(kernel, dim3((unsigned)(tm * tn * g.batch)), dim3(Shape::kThreads), Shape::kLds, stream, g, (int)tm, (int)tn,
                     row_alignment(g.a, g.lda, g.stride_a, 0), row_alignment(g.b, g.ldb, g.stride_b, g.b_index ? g.b_index_stride : 0));
  return check_launch("gemm_f32");
}

template <int WM, int WN, int TM, int TN, bool HALF>
int launch(const GemmArgs& g, hipStream_t stream) {
  if (!g.a_kmajor && !g.b_kmajor)
    return g.b_first && !HALF ? launch_one<WM, WN, TM, TN, false, false, HALF, !HALF>(g, stream)
                              : launch_one<WM, WN, TM, TN, false, false, HALF>(g, stream);
  if (!g.a_kmajor) return launch_one<WM, WN, TM, TN, false, true, HALF>(g, stream);
  if (!g.b_kmajor) return launch_one<WM, WN, TM, TN, true, false, HALF>(g, stream);
  return launch_one<WM, WN, TM, TN, true, true, HALF>(g, stream);
}

template <bool HALF>
int launch_sized(const GemmArgs& g, hipStream_t stream) {
  // The tile with the shortest schedule: workgroups on the busiest compute unit x tile area x what a unit of area costs on
  // that tile.  A larger tile stages fewer values per product and reads fewer LDS words per matrix instruction (measured on
  // 80 products of 1000 x 1100 x 1024: 64 x 64 tiles 1.43 ms, 128 x 128 1.23, 256 x 128 1.09; float16 0.74, 0.62, 0.49); a
  // smaller one pads less and fills the chip from fewer products (8 of those products: 0.130, 0.138, 0.150 ms).
  const int64_t cus = compute_units();
  auto cost = [&](int rows_a, int rows_b, int weight) {
    return ceil_div(ceil_div(g.m, rows_a) * ceil_div(g.n, rows_b) * g.batch, cus) * rows_a * rows_b * weight;
  };
  const int64_t small = cost(64, 64, HALF ? 150 : 130), square = cost(128, 128, HALF ? 127 : 112);
  const int64_t tall = cost(256, 128, 100), wide = cost(128, 256, 100);
  const int64_t big = tall < wide ? tall : wide;
  if (small <= square && small <= big) return launch<2, 2, 2, 2, HALF>(g, stream);
  if (square <= big) return launch<2, 4, 4, 2, HALF>(g, stream);
  return tall <= wide ? launch<4, 2, 4, 4, HALF>(g, stream) : launch<2, 4, 4, 4, HALF>(g, stream);
}

}  // namespace

int gemm_f32(const GemmArgs& g, hipStream_t stream) {
  if (g.batch <= 0 || g.m <= 0 || g.n <= 0) return PBG_OK;
  if (g.k < 0) return fail(PBG_ERR_INVALID, "gemm_f32: negative k");
  return g.half ? launch_sized<true>(g, stream) : launch_sized<false>(g, stream);
}

}  // namespace pbg

extern "C" int pbg_gemm_f32(const float* a, const float* b, float* c, int32_t batch, int32_t m, int32_t n, int32_t k,
                            int32_t lda, int32_t ldb, int32_t ldc, int64_t stride_a, int64_t stride_b,
                            int64_t stride_c, int32_t a_kmajor, int32_t b_kmajor, float alpha, float beta,
                            pbg_stream_t stream) {
  if (batch < 0 || m < 0 || n < 0 || k < 0) return pbg::fail(PBG_ERR_INVALID, "pbg_gemm_f32: negative size");
  if (batch == 0 || m == 0 || n == 0) return PBG_OK;
  if (!a || !b || !c) return pbg::fail(PBG_ERR_INVALID, "pbg_gemm_f32: null pointer");
  pbg::GemmArgs g{};
  g.a = a; g.b = b; g.c = c;
  g.stride_a = stride_a; g.stride_b = stride_b; g.stride_c = stride_c;
  g.lda = lda; g.ldb = ldb; g.ldc = ldc;
  g.m = m; g.n = n; g.k = k; g.batch = batch;
  g.a_kmajor = a_kmajor; g.b_kmajor = b_kmajor;
  g.alpha = alpha; g.beta = beta;
  return pbg::gemm_f32(g, (hipStream_t)stream);
}

extern "C" int pbg_gemm_f16(const float* a, const float* b, float* c, int32_t batch, int32_t m, int32_t n, int32_t k,
                            int32_t lda, int32_t ldb, int32_t ldc, int64_t stride_a, int64_t stride_b,
                            int64_t stride_c, int32_t a_kmajor, int32_t b_kmajor, float alpha, float beta,
                            pbg_stream_t stream) {
  if (batch < 0 || m < 0 || n < 0 || k < 0) return pbg::fail(PBG_ERR_INVALID, "pbg_gemm_f16: negative size");
  if (batch == 0 || m == 0 || n == 0) return PBG_OK;
  if (!a || !b || !c) return pbg::fail(PBG_ERR_INVALID, "pbg_gemm_f16: null pointer");
  pbg::GemmArgs g{};
  g.a = a; g.b = b; g.c = c;
  g.stride_a = stride_a; g.stride_b = stride_b; g.stride_c = stride_c;
  g.lda = lda; g.ldb = ldb; g.ldc = ldc;
  g.m = m; g.n = n; g.k = k; g.batch = batch;
  g.a_kmajor = a_kmajor; g.b_kmajor = b_kmajor;
  g.alpha = alpha; g.beta = beta;
  g.half = 1;
  return pbg::gemm_f32(g, (hipStream_t)stream);
}
