// k_gemm_kernel.h — the fp32 GEMM kernel template on gfx950 matrix cores (device code
// shared by the per-layout instantiation units k_gemm_{nn,nt,tn,q8}.hip; host
// planning and launch live in k_gemm.hip).
//
// Serves the reference's whole GEMM family (runtime/executor/gemm.cc:173-228:
// GemmNN + fused bias/act epilogue, GemmNT, GemmTN, GemmAccNN, the int8-B
// GemmNNQ8/NTQ8) and the attention contractions (attention.cc: QK^T, PV,
// dO V^T, P^T dO, dS K, dS^T Q), all as one kernel template:
//
//   C[z](m,n) = epilogue(alpha * sum_k A[z](m,k) B[z](k,n))
//
// with each operand either k-contiguous or row-contiguous in memory (so NT/TN
// read their operands in place, no transposes), a (b, h) batch decomposition
// with arbitrary element strides (attention heads live interleaved in
// [B*S, H*d] rows), and causal modes that skip whole tiles the causal mask
// zeroes.
//
// Mapping to CDNA4: a workgroup of 4 or 8 wavefronts (64 lanes) owns an
// MT_M x MT_N output tile; each wavefront owns a WM x WN sub-tile of 32x32
// blocks, 16 accumulators per lane each. Operand tiles (KT = 16 or 32 deep
// per config) are staged through LDS, double-buffered: the next stages'
// 16-byte global loads are in flight while the matrix cores consume the
// current one. The k loop carries no per-element address math: each lane's
// offsets from the stage origin are fixed at kernel entry (rows past the
// operand's end are clamped onto its last row: their products reach only
// outputs that are never stored), the origin advances by a uniform step, and
// only a final partial stage masks k.
//
// Products. The fp32 MFMA (v_mfma_f32_32x32x2_f32) peaks at 157 TFLOP/s and
// bounded every large GEMM here at 125-147; the bf16 MFMA runs 16x as many
// products. An fp32 value is exactly the sum of three bf16 values (24
// significand bits as 8 + 8 + 8, each part the round-to-nearest of what is
// left: Split4), so a product is nine bf16 products, each exact in fp32. The
// three smallest are at most 2^-26 of the whole, a quarter of the fp32
// product's own rounding, and are left out; the other six run as six
// v_mfma_f32_32x32x16_bf16 into one fp32 accumulator, smallest first. The
// accumulator is added to a second one and cleared every 64 k (kChunk), which
// keeps the rounding small. The bf16 MFMA's own additions lean to one side;
// half of the rows are computed negated, so that a sum over many rows of such
// results does not add the lean up (RowNegated below). Relative 2-norm error
// against 64 bits, fp32 MFMA | this: normal operands K = 16 7.4e-8 | 3.3e-8,
// K = 2048 8.1e-7 | 1.6e-7, K = 8192 1.62e-6 | 2.5e-7 (without the second
// accumulator 7.0e-7 at K = 2048); softmax gradients times a head of 8192
// classes 1.6e-6 | 2.3e-7; log-normal operands 6.6e-7 | 1.3e-7. An int8 operand
// is one bf16 part: three products.
// Measured: NT 8192x2048x5504 1330 -> 854 us, 8192x5504x2048 1334 -> 921 us,
// 200-216 TFLOP/s of fp32 products where 157 was the fp32 MFMA's peak. What
// bounds it now is power: the matrix cores are 70% busy at 1.78 GHz (2.4 with
// little to do), and a loop of bf16 MFMAs alone on random bits runs at the
// clock that makes 300.
//
// Range. fp32 operands are scaled by 2^24 (kOpScale, exact) before the split,
// and the sums by 2^-48 after it (2^-24 with an int8 operand): the smallest
// subnormal becomes 2^-125, so every part of every value is zero or a normal
// bf16 number, and what underflows among the products is below 2^-174 of the
// true scale, under a K-th of fp32's smallest subnormal for any K here.
// Unscaled, values under 2^-110 lost their low parts and those under 2^-134
// vanished, which a large other factor could lift to any size. Infinities and
// NaN, operands of 2^103 and more and sums of 2^80 and more do not survive the
// scaled split and show as non-finite accumulators: a wavefront that finds one
// in a 32x32 block computes that block again with the fp32 MFMA, straight
// from memory (Recompute below), so non-finites propagate as fp32 products do.
//
// k assignment: half-wavefront h supplies k = 16g + 8h + 0..7 of the group
// g of 16, for A and B alike. The split happens once per element and
// workgroup, between the global load and the LDS store; LDS holds the three
// parts as planes. A k-contiguous operand is kept as [o][k] rows and read
// with one 16-byte ds_read per part, fragment and lane; a row-contiguous one
// is kept as [k][o] rows and read with the transposing ds_read_b64_tr_b16.
//
// Workgroup order: the 8 XCDs (each with its own L2) receive workgroups
// round-robin, so the linear workgroup id is remapped to give each XCD a
// contiguous run of tiles, walked in groups of 8 tile-rows so the tiles
// resident on one XCD share A row-panels and B column-panels in its L2.
//
// Determinism: each output is owned by one lane of one workgroup and its k
// order is fixed by the tile loop; split-K writes per-slice partials that a
// second kernel sums in slice order. No atomics.
//
// Numerics: operands held to all 24 bits, fp32 accumulation in the matrix
// core (above). The reference accumulates in a different order (4-wide k
// groups / sequential), so GEMM outputs agree to within fp32 reordering
// error, not bit-for-bit.
#pragma once

#include "device_common.h"
#include "kernels.h"

#include <algorithm>
#include <type_traits>

namespace seeml_hip {
namespace gemm {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t uint32u __attribute__((aligned(1)));

constexpr int KG = 16;          // k covered by one MFMA
constexpr int kXcds = 8;
constexpr int kGroupRows = 8;   // tile-rows walked together (L2 panel sharing)
constexpr int kChunk = 64;      // k summed in the matrix core before a rounded fp32 addition
constexpr int kSplitAlign = 64; // split-K slice depth: a multiple of kChunk and every KT

// LDS layout of one part (plane) of an operand stage, in bf16 elements. A
// 16-byte fragment read serves 16 lanes a cycle (64 banks). [o][k] rows of
// KT with the 16-byte chunks of a row permuted by its row number, so that the
// 16 rows read at one logical chunk fall in 16 different bank quads, without
// padding. [k][o] rows padded to 64 bytes past a multiple of the banks: the
// four rows of a transposing read's 32 lanes fall in disjoint quarters.
// (Permuted by row pairs and padded by 32 bytes instead, every read took twice
// its cycles: 36% of the LDS cycles at 8192x2048x5504 were conflicts.)
template <int KT>
__device__ __forceinline__ constexpr int KcChunk(int o, int c) {
  return KT == 32 ? c ^ ((o >> 2) & 3) : c ^ ((o >> 3) & 1);
}
constexpr int RcStride(int mt) { return mt == 32 ? 32 : mt + 32; }
template <int MT, int KT, bool KC>
constexpr int PlaneElems() { return KC ? MT * KT : KT * RcStride(MT); }

// A wavefront-uniform pointer to global memory as one scalar value. Without
// this the compiler reassociates (base + per-lane offset) + stage step and
// keeps a 64-bit vector pointer per load in flight.
template <typename T>
using GlobalPtr = const __attribute__((address_space(1))) T*;
template <typename T>
__device__ __forceinline__ GlobalPtr<T> ScalarBase(const T* p) {
  GlobalPtr<T> q = (GlobalPtr<T>)p;
  asm("" : "+s"(q));
  return q;
}

// 2^24 x as three bf16 parts, 2^24 x = part 0 + part 1 + part 2 exactly for
// every |x| below 2^103. Packed: part i of (x0, x1) in p[i].
constexpr float kOpScale = 0x1p24f;
template <int PB>  // parts of B
constexpr float kUnscale = PB == 3 ? 0x1p-48f : 0x1p-24f;
__device__ __forceinline__ void Split2(float x0, float x1, uint32_t (&p)[3], float s0 = kOpScale,
                                       float s1 = kOpScale) {
  x0 *= s0;
  x1 *= s1;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const bf16x2 h = __builtin_convertvector((floatx2){x0, x1}, bf16x2);
    p[i] = __builtin_bit_cast(uint32_t, h);
    if (i < 2) {
      // What is left, exactly.
      x0 -= __builtin_bit_cast(float, p[i] << 16);
      x1 -= __builtin_bit_cast(float, p[i] & 0xFFFF0000u);
    }
  }
}

// A pair of int8 values, each one part, unscaled.
__device__ __forceinline__ uint32_t Exact2(float x0, float x1) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2){x0, x1}, bf16x2));
}

// Half of A's rows are negated on the way in, and their sums on the way out:
// the bf16 MFMA rounds towards minus infinity, a lean of up to 6e-8 of the
// outputs' size that a sum over many rows (a weight gradient's) would add up
// and that the two signs cancel. Which half costs no vector register in each
// layout: k-contiguous, every other 64 rows, one sign per wavefront on the way
// out and per vector on the way in; row-contiguous, the odd rows, one sign per
// element.
constexpr bool RowNegated(int64_t m) { return (m >> 6) & 1; }

// The parts of a lane's 8 consecutive k.
__device__ __forceinline__ void Split8(const float* x, bf16x8 (&f)[3], float scale) {
  uint32_t w[3][4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t p[3];
    Split2(x[2 * q], x[2 * q + 1], p, scale, scale);
#pragma unroll
    for (int part = 0; part < 3; ++part) w[part][q] = p[part];
  }
#pragma unroll
  for (int part = 0; part < 3; ++part)
    f[part] = __builtin_bit_cast(bf16x8, make_uint4(w[part][0], w[part][1], w[part][2], w[part][3]));
}

// One 16-deep step of a block of fragments into its accumulators: the six
// products of NA = NB = 3 parts, or the three of an exact (one-part) B,
// smallest first, each over all blocks so that consecutive MFMAs are
// independent. FOLD: the first step of a chunk (kChunk): the accumulators,
// holding the chunk before, are added to `sum`, unscaled (with the rows'
// sign), and start again from zero.
template <bool FOLD, bool A_KC, int BM, int BN, int PB>
__device__ __forceinline__ void MfmaStep(const bf16x8 (&fa)[BM][3], const bf16x8 (&fb)[BN][PB],
                                         floatx16 (&acc)[BM][BN], floatx16 (&sum)[BM][BN], float unscale) {
  constexpr int kProducts = PB == 3 ? 6 : 3;
  constexpr int ia[6] = {2, PB == 3 ? 0 : 1, PB == 3 ? 1 : 0, 1, 0, 0};
  constexpr int ib[6] = {0, PB == 3 ? 2 : 0, PB == 3 ? 1 : 0, 0, PB == 3 ? 1 : 0, 0};
  constexpr floatx16 kZero = {};
#pragma unroll
  for (int q = 0; q < kProducts; ++q)
#pragma unroll
    for (int i = 0; i < BM; ++i)
#pragma unroll
      for (int j = 0; j < BN; ++j) {
        if (FOLD && q == 0) {
#pragma unroll
          for (int v = 0; v < 16; ++v)
            sum[i][j][v] = __builtin_fmaf(acc[i][j][v], !A_KC && v & 1 ? -unscale : unscale, sum[i][j][v]);
        }
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            fa[i][ia[q]], fb[j][ib[q]], FOLD && q == 0 ? kZero : acc[i][j], 0, 0, 0);
      }
}

// The issue order of one stage: kFirst fragment reads, then after each of the
// kMfma MFMAs its share of the VALU operations that split kVecs vectors
// (kSplitOps each; 26 are the split, the rest room for addresses), LDS reads,
// an LDS write and, unless they are issued ahead of it all (kAhead), a global
// load. Left to itself the scheduler issues the MFMAs first and the split
// after them, so that a wavefront alone on its SIMD takes the sum of the two.
template <int kMfma, int kVecs, int kFirst, int kSplitOps, bool kAhead>
__device__ __forceinline__ void Interleave() {
  constexpr int kOps = (kSplitOps * kVecs + kMfma - 1) / kMfma;
  __builtin_amdgcn_sched_group_barrier(0x100, kFirst, 0);
#pragma unroll
  for (int q = 0; q < kMfma; ++q) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if constexpr (kAhead) __builtin_amdgcn_sched_group_barrier(0x100, (kFirst + 5) / 6, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, kOps, 0);
    if constexpr (!kAhead) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
    if constexpr (!kAhead) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
  }
}

// Whether any lane's accumulators hold a non-finite value. Uniform per
// wavefront.
__device__ __forceinline__ bool AnyNonFinite(const floatx16& acc) {
  float x = 0.0f;
#pragma unroll
  for (int v = 0; v < 16; ++v) x = __builtin_fmaf(acc[v], 0.0f, x);
  return __ballot(!(x == 0.0f)) != 0;
}

struct GemmKArgs {
  const void* A;
  const void* B;
  float* C;
  float* ws;
  int64_t M, N, K, lda, ldb, ldc;
  int64_t heads, batch;
  int64_t a_sb, a_sh, b_sb, b_sh, c_sb, c_sh;
  float alpha;
  int accumulate;
  const float* bias;
  int act;
  int causal;
  int splits;
  int64_t k_per_split;
  int tiles_m, tiles_n;
  const float* addend;  // fused AddEW (GemmDesc::addend): out = addend (+) c
  float* out;
  int addend_first;
  int write_c;
  float out_scale;  // GemmDesc::out_scaled: the AddEW consumes fl(out_scale * c)
  int out_scaled;
  int c_scaled;     // GemmDesc::c_gets_scaled: the C store is the scaled value
  int64_t ldo;      // row stride of addend and out
  // LoRA up-projection in the epilogue (GemmDesc::lora_t): with lora_t set,
  // out = c (+) fl(out_scale * u) where u = T B' over lora_r (T [M, lora_r]
  // row-major, B' [lora_r, N] row-major), the same MFMA k order as a tile
  // GEMM of u; addend unused. lora_y_first: c is the AddEW's first operand.
  const float* lora_t;
  const float* lora_b;
  int64_t lora_ldt, lora_ldb;
  int lora_r;
  int lora_y_first;
  // A Scale folded into the operand loads (GemmDesc::scale_stream, the
  // SCL instantiations): the scaled operand is read as fl(op_scale * x).
  float op_scale;
  // The AddBias (+ activation) after the fused AddEW (GemmDesc::post_bias,
  // the POST instantiations): h = o + pbias[n] to hout, act(h) to gout
  // (each when set), o to out only with write_out.
  const float* pbias;
  float* hout;
  float* gout;
  int pact;
  int write_out;
};

// The fused AddEW's sum o of value v and addend y, stored with what follows
// it (POST: the AddBias of bias value b, then the activation) at element
// offset `at` of the out / hout / gout arrays (one layout, row stride ldo).
template <bool POST>
__device__ __forceinline__ void FusedSum(const GemmKArgs& p, int64_t at, float y, float sv, float b) {
  const float o = p.addend_first ? y + sv : sv + y;
  if constexpr (!POST) {
    p.out[at] = o;
  } else {
    if (p.write_out) p.out[at] = o;
    const float h = o + b;
    if (p.hout) p.hout[at] = h;
    if (p.gout) p.gout[at] = dev_act(p.pact, h);
  }
}

// Tile configurations (the autotuner's arms).
struct CfgInfo {
  int mt_m, mt_n, kt, threads;
  const char* name;
};
inline constexpr CfgInfo kCfgs[] = {
    {128, 128, 16, 256, "128x128x16/w2x2"}, {128, 128, 16, 512, "128x128x16/w4x2"},
    {256, 128, 16, 512, "256x128x16/w4x2"}, {128, 256, 16, 512, "128x256x16/w2x4"},
    {128, 64, 32, 256, "128x64x32/w2x2"},   {64, 64, 32, 256, "64x64x32/w2x2"},
    {128, 32, 32, 256, "128x32x32/w4x1"},   {32, 128, 32, 256, "32x128x32/w1x4"},
    {64, 128, 32, 256, "64x128x32/w2x2"},   {128, 64, 32, 256, "128x64x32/w4x1"},
    {64, 64, 16, 256, "64x64x16/w2x2"},     {64, 128, 16, 256, "64x128x16/w2x2"},
};
// Wavefronts per SIMD to keep registers for: two of the large tiles'.
constexpr int MinWaves(int mt_m, int mt_n) { return mt_m * mt_n >= 128 * 128 ? 2 : 1; }
inline constexpr int kNumCfgs = sizeof(kCfgs) / sizeof(kCfgs[0]);
inline constexpr int kCfgDefault = 0, kCfgSmall = 5, kCfgSkinnyN = 6, kCfgSkinnyM = 7,
                     kCfgLarge = 2, kCfgWaves8 = 1, kCfgHalf = 9, kCfgSmallK16 = 10;

// One operand's MT x KT stage (outer index o = m for A / n for B), held in
// registers between its global loads and its LDS store, where it is split.
// KC = k-contiguous. Vector i of a thread is 4 elements along the contiguous
// direction.
//
// VEC (16-byte aligned rows, contiguous extent a multiple of 4): 16-byte
// loads at per-lane offsets fixed for the whole k loop; the stage origin is
// uniform. A final partial stage (k beyond the reduction's end) zeroes its
// out-of-range vectors, reading the row start instead.
// !VEC (any extent, stride and alignment; int8): the same vectors by loads
// that need only the element's own alignment. Row-contiguous, a vector that
// would pass the row's end is read back from the end and shifted into place
// at the LDS store (an extent below 4: element loads); k-contiguous, a final
// partial stage is read by elements. Out-of-range elements are zero.
//
// SC (VEC only): every loaded element in range is scaled, fl(sc * x), as a
// Scale instruction would have stored it; zeros past the reduction's end
// stay +0. A whole stage is scaled at its LDS store, where its loads are
// waited for anyway (scaled as loaded, each stage's loads would be waited
// for at once, a stage early: 2.5x slower on the rank-64 shapes); a final
// partial stage is scaled as loaded, under its in-range masks.
template <int MT, int KT, bool KC, typename T, int NT, bool VEC, bool IS_A, bool SC = false>
struct Stage {
  static constexpr bool kF32 = std::is_same<T, float>::value;
  static constexpr int kParts = kF32 ? 3 : 1;
  static constexpr int kPlane = PlaneElems<MT, KT, KC>();
  static constexpr int kElems = kParts * kPlane;  // LDS elements of a stage
  static constexpr int kVecs = MT * KT / 4;
  static constexpr int kPer = kVecs / NT;
  static_assert(kVecs % NT == 0, "stage shape");
  static_assert(!SC || VEC, "scaled loads need the vector form");
  // k-contiguous: rows between a thread's vectors (its first is below 64, or
  // below 128 with the step of 128), so that a vector's rows share a sign, and
  // whether the first one's sign depends on the tile or the wavefront.
  static constexpr int kRowStep = NT / (KT / 4);
  static constexpr bool kRowBase = IS_A && KC && (MT < 128 || kRowStep == 128);
  static_assert(!IS_A || !KC || kRowStep == 32 || kRowStep == 64 || kRowStep == 128, "one sign per vector");
  static_assert(!VEC || kF32, "int8 operands take the general form");
  float r[kPer][4];
  // Byte offset of vector i from the stage origin. VEC: the host checks that
  // it fits 32 bits, so a load is a uniform base plus a 32-bit offset.
  using Off = typename std::conditional<VEC, uint32_t, int64_t>::type;
  static constexpr int kSize = sizeof(T);
  Off off[kPer];
  int shift[kPer];    // !VEC, row-contiguous: places the vector was read back by
  int avail;          // !VEC, row-contiguous: elements of the row from the tile's start on
  bool few;           // !VEC, row-contiguous: rows of fewer than 4 elements
  uint32_t rs;        // kRowBase: the scale with the first vector's rows' sign, as bits
  float sc;           // SC: the factor
  bool pend;          // SC: loaded unscaled (a whole stage), scaled at the store

  __device__ __forceinline__ static void coords(int v, int& o, int& k) {
    if constexpr (KC) {
      o = v / (KT / 4);
      k = (v % (KT / 4)) * 4;
    } else {
      k = v / (MT / 4);
      o = (v % (MT / 4)) * 4;
    }
  }

  // o0: first row of the tile (a multiple of 4); oe: the operand's extent.
  __device__ __forceinline__ void init(int64_t ld, int64_t o0, int64_t oe) {
    if constexpr (kRowBase) {
      const int first = kRowStep == 128 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) * 64 : 0;
      rs = __builtin_bit_cast(uint32_t, kOpScale) | static_cast<uint32_t>(RowNegated(o0 + first)) << 31;
    }
    // >= 1: the tile starts in range.
    const int left = static_cast<int>(std::min<int64_t>(oe - o0, MT));
    if constexpr (!VEC && !KC) {
      avail = left;
      few = oe < 4;
    }
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      int o, k;
      coords(static_cast<int>(threadIdx.x) + i * NT, o, k);
      int oc = o;
      if constexpr (KC) {
        oc = std::min(o, left - 1);
      } else if constexpr (VEC) {
        oc = std::min(o, left - 4);
      } else {
        // Back to the row's last 4 elements: at least 0 from the row's start.
        oc = oe < 4 ? 0 : std::min(o, left - 4);
        shift[i] = o - oc;
      }
      off[i] = static_cast<Off>((KC ? oc * ld + k : k * ld + oc) * kSize);
    }
  }

  // Vector i, `back` bytes before its place.
  __device__ __forceinline__ void load_vec(int i, GlobalPtr<T> org, Off back = 0) {
    Off o = off[i] - back;
    // Bound to the stage's origin here: with the 32-bit offset's extension
    // hoisted out of the loop, every load took a 64-bit vector addition and
    // two offset registers (8-36 bytes of scratch on the largest tiles).
    if constexpr (VEC) asm("" : "+v"(o) : "s"(org));
    const GlobalPtr<char> src = (GlobalPtr<char>)org + o;
    if constexpr (kF32) {
      using V = typename std::conditional<VEC, floatx4, floatx4u>::type;
      const V q = *(GlobalPtr<V>)src;
      r[i][0] = q[0]; r[i][1] = q[1]; r[i][2] = q[2]; r[i][3] = q[3];
    } else {
      // The four bytes; made floats at the store, where they are waited for.
      r[i][0] = __builtin_bit_cast(float, *(GlobalPtr<uint32u>)src);
    }
  }
  __device__ __forceinline__ void put(int i, int e, T x, bool in) {
    if constexpr (kF32) {
      r[i][e] = in ? x : 0.0f;
    } else {
      const uint32_t b = in ? static_cast<uint8_t>(x) : 0u;
      const uint32_t w = e == 0 ? 0u : __builtin_bit_cast(uint32_t, r[i][0]);
      r[i][0] = __builtin_bit_cast(float, w | (b << (8 * e)));
    }
  }
  // Elements of vector i of a row of fewer than 4 (!VEC, row-contiguous).
  __device__ __forceinline__ void load_few(int i, GlobalPtr<T> org, bool in_k) {
    int o, k;
    coords(static_cast<int>(threadIdx.x) + i * NT, o, k);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = in_k && o + e < avail;
      put(i, e, org[in ? off[i] / kSize + o + e : 0], in);
    }
  }

  // A whole stage in range: one load per vector, no masks.
  __device__ __forceinline__ void load_full(GlobalPtr<T> org) {
    if constexpr (!VEC && !KC) {
      if (few) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) load_few(i, org, true);
        return;
      }
    }
#pragma unroll
    for (int i = 0; i < kPer; ++i) load_vec(i, org);
    if constexpr (SC) pend = true;
  }

  // A final partial stage, of 0 < kvalid < KT: k from kvalid on reads as zero.
  __device__ __forceinline__ void load_part(GlobalPtr<T> org, int64_t ld, int64_t kvalid) {
    if constexpr (SC) pend = false;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      int o, k;
      coords(static_cast<int>(threadIdx.x) + i * NT, o, k);
      if constexpr (!VEC && KC) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool in = k + e < kvalid;
          put(i, e, org[off[i] / kSize + (in ? e : -k)], in);
        }
      } else {
        const bool in = k < kvalid;  // VEC: a KC vector is wholly in or out (K % 4 == 0)
        if constexpr (!VEC && !KC) {
          if (few) {
            load_few(i, org, in);
            continue;
          }
        }
        load_vec(i, org, in ? 0 : static_cast<Off>((KC ? k : k * ld) * kSize));
        if constexpr (kF32) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (SC) r[i][e] = sc * r[i][e];
            r[i][e] = in ? r[i][e] : 0.0f;
          }
        } else {
          r[i][0] = in ? r[i][0] : 0.0f;
        }
      }
    }
  }

  // Splits the stage into its parts and stores them.
  __device__ __forceinline__ void store(__bf16* __restrict__ lds) const {
#pragma unroll
    for (int i = 0; i < kPer; ++i) store_vec(i, lds);
  }
  __device__ __forceinline__ void store_vec(int i, __bf16* __restrict__ lds) const {
    {
      int o, k;
      coords(static_cast<int>(threadIdx.x) + i * NT, o, k);
      __bf16* dst = KC ? lds + o * KT + KcChunk<KT>(o, k >> 3) * 8 + (k & 7)
                       : lds + k * RcStride(MT) + o;
      float q[4];
      if constexpr (kF32) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          q[e] = r[i][e];
          if constexpr (SC) if (pend) q[e] = sc * q[e];
        }
        if constexpr (!VEC && !KC) {
          if (avail < MT && !few) {  // this tile passes the row's end
            if (shift[i] & 1) { q[0] = q[1]; q[1] = q[2]; q[2] = q[3]; q[3] = 0.0f; }
            if (shift[i] & 2) { q[0] = q[2]; q[1] = q[3]; q[2] = q[3] = 0.0f; }
            if (shift[i] >= 4) q[0] = q[1] = q[2] = q[3] = 0.0f;
          }
        }
      } else {
        uint32_t w = __builtin_bit_cast(uint32_t, r[i][0]);
        if constexpr (!KC) {
          if (avail < MT && !few) w = shift[i] >= 4 ? 0u : w >> (8 * shift[i]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) q[e] = static_cast<float>(static_cast<int8_t>(w >> (8 * e)));
      }
      uint32_t lo[3], hi[3];
      if constexpr (kF32) {
        float s0 = kOpScale, s1 = IS_A && !KC ? -kOpScale : kOpScale;
        if constexpr (IS_A && KC) {
          if constexpr (kRowBase) {
            uint32_t bits = rs;
            asm("" : "+s"(bits));  // kept in a scalar register
            s0 = __builtin_bit_cast(float, bits);
          }
          s0 = s1 = RowNegated(i * kRowStep) ? -s0 : s0;
        }
        Split2(q[0], q[1], lo, s0, s1);
        Split2(q[2], q[3], hi, s0, s1);
      } else {
        lo[0] = Exact2(q[0], q[1]);
        hi[0] = Exact2(q[2], q[3]);
      }
#pragma unroll
      for (int part = 0; part < kParts; ++part)
        *reinterpret_cast<uint2*>(dst + part * kPlane) = make_uint2(lo[part], hi[part]);
    }
  }
};

__device__ __forceinline__ bf16x4 ReadTr(const __bf16* p) {
  typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)p);
}

// The parts of NB 32-wide fragments at o = w0 + 32i + r: k = 16g + 8h + 0..7.
template <int MT, int KT, bool KC, int NB, int P>
__device__ __forceinline__ void ReadFrags(const __bf16* __restrict__ lds, int w0, int g, int lane,
                                          bf16x8 (&f)[NB][P]) {
  constexpr int kPlane = PlaneElems<MT, KT, KC>();
  const int h = lane >> 5;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    if constexpr (KC) {
      const int o = w0 + 32 * i + (lane & 31);
      const __bf16* src = lds + o * KT + KcChunk<KT>(o, 2 * g + h) * 8;
#pragma unroll
      for (int part = 0; part < P; ++part)
        f[i][part] = *reinterpret_cast<const bf16x8*>(src + part * kPlane);
    } else {
      // A transposing read takes a [4 k][16 o] patch per 16 lanes, each lane
      // naming 4 o of one k, and returns 4 k of one o.
      const int k = KG * g + 8 * h + ((lane & 15) >> 2);
      const int o = w0 + 32 * i + (lane & 16) + 4 * (lane & 3);
#pragma unroll
      for (int part = 0; part < P; ++part) {
        const __bf16* src = lds + part * kPlane + k * RcStride(MT) + o;
        f[i][part] = __builtin_shufflevector(ReadTr(src), ReadTr(src + 4 * RcStride(MT)), 0, 1, 2, 3,
                                             4, 5, 6, 7);
      }
    }
  }
}

// Linear workgroup id -> logical id such that XCD x (= lin % 8) holds the
// contiguous logical range of its share. A bijection on [0, total).
// Workgroup counts fit 32 bits (a grid holds at most 2^32 - 1 workgroups),
// and 32-bit divisions are a few instructions where 64-bit ones are a long
// scalar routine run by every workgroup before its first load.
__device__ __forceinline__ uint32_t XcdLogical(uint32_t lin, uint32_t total) {
  const uint32_t per = total / kXcds, rem = total % kXcds;
  const uint32_t x = lin % kXcds, idx = lin / kXcds;
  return x < rem ? x * (per + 1) + idx : rem * (per + 1) + (x - rem) * per + idx;
}

// One workgroup's work item: logical id L (after the XCD remap) decomposes
// into (tile, split slice, batch z) over `nslices` slices. FUSED and LORA
// compile those epilogues in; each applies to a work item whose arguments
// ask for it (p.out / p.lora_t set), any other takes the plain write-back.
// SCL: a Scale folded into the loads of A (1) or B (2), factor p.op_scale.
// POST (with FUSED): the AddBias (+ activation) after the fused AddEW.
template <int MT_M, int MT_N, int KT, int WAVES_M, int WAVES_N, bool A_KC, bool B_KC, bool B_I8,
          bool VEC, bool FUSED, bool LORA, int SCL = 0, bool POST = false>
__device__ __forceinline__ void gemm_tile(const GemmKArgs& p, uint32_t L, uint32_t nslices) {
  static_assert(!POST || (FUSED && !LORA && !(MT_M == 256 && MT_N == 128)), "post-AddEW variants");
  using BT = typename std::conditional<B_I8, int8_t, float>::type;
  constexpr int NT = 64 * WAVES_M * WAVES_N;
  constexpr int WM = MT_M / WAVES_M, WN = MT_N / WAVES_N;
  constexpr int BM = WM / 32, BN = WN / 32;
  static_assert(WM % 32 == 0 && WN % 32 == 0 && KT % KG == 0 && kSplitAlign % KT == 0,
                "tile shape");
  constexpr bool kVecB = VEC && !B_I8;
  using StageA = Stage<MT_M, KT, A_KC, float, NT, VEC, true, SCL == 1>;
  using StageB = Stage<MT_N, KT, B_KC, BT, NT, kVecB, false, SCL == 2>;
  constexpr int TA = StageA::kElems, TB = StageB::kElems, PB = StageB::kParts;
  __shared__ __align__(16) __bf16 smem[2 * (TA + TB)];

  // What is one value per wavefront is kept in scalar registers (the
  // divisions below run on the vector ALU): operand bases then cost no
  // vector registers, and a load is a scalar base plus a 32-bit offset.
  auto uniform = [](auto v) { return __builtin_amdgcn_readfirstlane(static_cast<int>(v)); };
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
  const int h = lane >> 5, r = lane & 31;
  const int wm0 = (wave / WAVES_N) * WM, wn0 = (wave % WAVES_N) * WN;

  // Logical work item of this workgroup: (tile, split slice, batch z). The
  // small calls are bound by this entry, the first loads and the tail, so a
  // division or batch offset that is not needed is branched around, a stage
  // wholly in range takes one branch, and the tail's unscaling is the addition
  // (64x64x64: NN 5.13 -> 4.83 us, NT 5.12 -> 4.81, TN 5.14 -> 4.84;
  // 8x256x32: 5.0 -> 4.7).
  const uint32_t tiles = static_cast<uint32_t>(p.tiles_m) * static_cast<uint32_t>(p.tiles_n);
  uint32_t t_id = L, z = 0;
  int slice = 0;
  if (L >= tiles) {
    t_id = L % tiles;
    z = L / tiles;
    if (nslices > 1) {
      slice = uniform(z % nslices);
      z /= nslices;
    }
  }
  const uint32_t grp = p.tiles_m <= kGroupRows ? 0 : t_id / (kGroupRows * static_cast<uint32_t>(p.tiles_n));
  const uint32_t first = grp * kGroupRows;
  const uint32_t gm = std::min<uint32_t>(kGroupRows, static_cast<uint32_t>(p.tiles_m) - first);
  const uint32_t in_grp = t_id - grp * kGroupRows * static_cast<uint32_t>(p.tiles_n);
  const int64_t tm = uniform(first + in_grp % gm), tn = uniform(in_grp / gm);
  const int64_t m0 = tm * MT_M, n0 = tn * MT_N;
  const float* A = static_cast<const float*>(p.A);
  const BT* B = static_cast<const BT*>(p.B);
  float* C = p.C;
  if (z != 0) {
    const uint32_t heads = static_cast<uint32_t>(p.heads);
    const int64_t zb = uniform(z / heads), zh = uniform(z % heads);
    A += zb * p.a_sb + zh * p.a_sh;
    B += zb * p.b_sb + zh * p.b_sh;
    C += zb * p.c_sb + zh * p.c_sh;
  }

  // Causal lower-triangular output: a tile wholly above the diagonal is
  // exact zeros, with no reduction at all.
  if (p.causal == static_cast<int>(Causal::kLowerOut) && n0 > m0 + MT_M - 1) {
    for (int idx = threadIdx.x; idx < MT_M * MT_N; idx += NT) {
      const int64_t m = m0 + idx / MT_N, n = n0 + idx % MT_N;
      if (m < p.M && n < p.N) C[m * p.ldc + n] = 0.0f;
    }
    return;
  }

  int64_t kb = 0, ke = p.K;
  if (p.causal != static_cast<int>(Causal::kNone)) {
    if (p.causal == static_cast<int>(Causal::kKLeM)) ke = std::min<int64_t>(p.K, m0 + MT_M);
    if (p.causal == static_cast<int>(Causal::kKGeM)) kb = std::min<int64_t>(p.K, m0);
  }
  if (p.splits > 1) {
    kb = static_cast<int64_t>(slice) * p.k_per_split;
    ke = std::min<int64_t>(p.K, kb + p.k_per_split);
  }

  // The wavefront's 64 or 32 rows share a sign (WM divides wm0).
  const float unscale = A_KC && RowNegated(m0 + wm0) ? -kUnscale<PB> : kUnscale<PB>;
  floatx16 acc[BM][BN], sum[BM][BN];  // the current chunk's, and those before it
#pragma unroll
  for (int i = 0; i < BM; ++i)
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = sum[i][j][v] = 0.0f;

  // Two register sets: stage s is loaded into set s % 2 two iterations
  // before it is computed, stored to LDS buffer s % 2 one iteration before.
  StageA sa0, sa1;
  StageB sb0, sb1;

  auto a_buf = [&](int i) { return smem + i * TA; };
  auto b_buf = [&](int i) { return smem + 2 * TA + i * TB; };
  // One stage's contraction out of LDS. `fold`: the stage starts a chunk.
  constexpr int kPerChunk = kChunk / KT;  // stages
  auto compute = [&](const __bf16* __restrict__ as, const __bf16* __restrict__ bs, auto fold) {
#pragma unroll
    for (int g = 0; g < KT / KG; ++g) {
      bf16x8 fa[BM][3], fb[BN][PB];
      ReadFrags<MT_N, KT, B_KC, BN, PB>(bs, wn0, g, lane, fb);
      ReadFrags<MT_M, KT, A_KC, BM, 3>(as, wm0, g, lane, fa);
      if (decltype(fold)::value && g == 0) MfmaStep<true, A_KC>(fa, fb, acc, sum, unscale);
      else MfmaStep<false, A_KC>(fa, fb, acc, sum, unscale);
    }
  };
  auto compute_at = [&](int64_t s) {  // stage s from its buffer
    const int cur = static_cast<int>(s & 1);
    if (s % kPerChunk == 0) compute(a_buf(cur), b_buf(cur), std::true_type());
    else compute(a_buf(cur), b_buf(cur), std::false_type());
  };

  const int64_t span = ke > kb ? ke - kb : 0;
  const int64_t nfull = span / KT;
  const int64_t ntiles = (span + KT - 1) / KT;
  const int64_t a_step = A_KC ? KT : KT * p.lda;
  const int64_t b_step = B_KC ? KT : KT * p.ldb;
  const float* a_org = A + (A_KC ? m0 * p.lda + kb : kb * p.lda + m0);
  const BT* b_org = B + (B_KC ? n0 * p.ldb + kb : kb * p.ldb + n0);
  // Loads stage s < nfull (wholly in range) into a register set.
  auto load_full = [&](StageA& xa, StageB& xb, int64_t s) {
    xa.load_full(ScalarBase(a_org + s * a_step));
    xb.load_full(ScalarBase(b_org + s * b_step));
  };
  // Any stage: k beyond ke reads zero.
  auto load_any = [&](StageA& xa, StageB& xb, int64_t s) {
    if (s < nfull) {
      load_full(xa, xb, s);
    } else {
      xa.load_part(ScalarBase(a_org + s * a_step), p.lda, ke - kb - s * KT);
      xb.load_part(ScalarBase(b_org + s * b_step), p.ldb, ke - kb - s * KT);
    }
  };
  // kOneSet (the tiles of 64x64 wavefronts): their accumulators leave registers
  // for one stage set only. Each vector of stage t + 1 is split and stored
  // between the MFMAs of stage t, and its registers take stage t + 2's load at
  // once.
  constexpr bool kOneSet = BM * BN >= 4;
  // Interleave's room for the split. Beyond its 26 operations, more lets the
  // split run ahead of its share, which pays where fragments are read with one
  // LDS read each and on the 64x64-wavefront tiles; the transposing reads'
  // tiles wait longer for their first fragments with it (us at 24 | 40, at
  // 8192x2048x2048: NT 128x64 428 | 402, 256x128 362 | 335; NN 128x128 of four
  // wavefronts 432 | 404, 256x128 362 | 348; TN 256x128 344 | 363; 128x64 NN
  // 530 | 545, TN 532 | 562).
  // With int8 B it is 20 (2048x2048x2048 NN and NT 77.6 and 66.9 us at 24, 79.3
  // and 63.5 at 20; 8192x2048x2048 284 and 257, 282 and 243).
  // The NT 128x128 tile of four wavefronts takes 30: at 40 it reloads a spilled
  // register every chunk (2048x2048x2048 113 us at 40, 105 at 30).
  constexpr int kSplitOps = BM * BN == 1                                   ? 28
                            : !VEC                                         ? (PB == 1 ? 20 : 24)
                            : kOneSet && A_KC && B_KC && NT == 256         ? 30
                            : (kOneSet ? A_KC || NT == 256 : A_KC && B_KC) ? 40
                                                                           : 24;
  // Steady-state iteration on stage t (t + 2 < nfull): load stage t + 2 into
  // set `ld`, contract stage t, store stage t + 1 from set `st`. With VEC the
  // body is one basic block, scheduled as one interleave.
  auto steady = [&](StageA& lda_, StageB& ldb_, const StageA& sta, const StageB& stb,
                    int64_t t, int cur, auto fold) {
    load_full(lda_, ldb_, t + 2);
    // One block per wavefront: the loads go out first. Placed by the scheduler
    // they went out late in the stage, and the next one began by waiting for
    // them (us, as scheduled | loads first, NN, NT, TN: 1024x1024x2048 49, 44,
    // 50 | 38, 38, 42; 64x64x512 12.5, 12.8, 12.3 | 11.5, 11.4, 12.5;
    // 2048x1376x512 30.6, 27.8, 31.5 | 29.6, 27.8, 30.9).
    // (1000x770x1531 layer 116 -> 111.) An int8 operand leaves too few MFMAs.
    constexpr bool kAhead = BM * BN == 1 && PB == 3;
    if constexpr (kAhead) __builtin_amdgcn_sched_barrier(0);
    compute(a_buf(cur), b_buf(cur), fold);
    sta.store(a_buf(cur ^ 1));
    stb.store(b_buf(cur ^ 1));
    if constexpr (kAhead || BM * BN > 1)
      Interleave<(KT / KG) * BM * BN*(PB == 3 ? 6 : 3), StageA::kPer + StageB::kPer,
                 BM * 3 * (A_KC ? 1 : 2) + BN * PB * (B_KC ? 1 : 2), kSplitOps, kAhead>();
    __syncthreads();
  };

  constexpr int kLoraK = 8;  // a lane's k of the LoRA product: 8h + 0..7, rank <= 16
  // T's row and B's column entries of k = 8h + 0..7 (zero beyond the rank) of
  // block row i / block column j. Unconditional loads (the half beyond the
  // rank reads the other's and is zeroed), so that no branch splits the
  // loads in flight.
  auto load_lora_t = [&](int i, float* t) {
    const int64_t row = std::min<int64_t>(m0 + wm0 + 32 * i + r, p.M - 1);
    const bool in = 8 * h < p.lora_r;
    const float4* src = reinterpret_cast<const float4*>(p.lora_t + row * p.lora_ldt + (in ? 8 * h : 0));
    const float4 q0 = src[0], q1 = src[1];
    const float q[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
    for (int e = 0; e < kLoraK; ++e) t[e] = in ? q[e] : 0.0f;
  };
  auto load_lora_b = [&](int j, float* t) {
    const int64_t col = std::min<int64_t>(n0 + wn0 + 32 * j + r, p.N - 1);
    const bool in = 8 * h < p.lora_r;
#pragma unroll
    for (int e = 0; e < kLoraK; ++e) {
      const float x = p.lora_b[((in ? 8 * h : 0) + e) * p.lora_ldb + col];
      t[e] = in ? x : 0.0f;
    }
  };
  int64_t t = 0;
  if constexpr (kOneSet) {
    constexpr int kVA = StageA::kPer, kV = kVA + StageB::kPer;
    static_assert(KT == KG, "one fragment group per stage");
    if (ntiles > 0) {
      sa0.init(p.lda, m0, p.M);
      sb0.init(p.ldb, n0, p.N);
      if constexpr (SCL == 1) sa0.sc = p.op_scale;
      if constexpr (SCL == 2) sb0.sc = p.op_scale;
      load_any(sa0, sb0, 0);
      sa0.store(a_buf(0));
      sb0.store(b_buf(0));
      if (ntiles > 1) load_any(sa0, sb0, 1);
      __syncthreads();
      auto body = [&](int64_t s, int cur, auto fold) {  // stage s, s + 2 whole
        const GlobalPtr<float> a_next = ScalarBase(a_org + (s + 2) * a_step);
        const GlobalPtr<BT> b_next = ScalarBase(b_org + (s + 2) * b_step);
        bf16x8 fb[BN][PB];
        ReadFrags<MT_N, KT, B_KC, BN, PB>(b_buf(cur), wn0, 0, lane, fb);
#pragma unroll
        for (int i = 0; i < BM; ++i) {
          bf16x8 fa[1][3];
          ReadFrags<MT_M, KT, A_KC, 1, 3>(a_buf(cur), wm0 + 32 * i, 0, lane, fa);
          MfmaStep<decltype(fold)::value, A_KC>(fa, fb, reinterpret_cast<floatx16(&)[1][BN]>(acc[i]),
                                          reinterpret_cast<floatx16(&)[1][BN]>(sum[i]), unscale);
#pragma unroll
          for (int v = kV * i / BM; v < kV * (i + 1) / BM; ++v) {
            if (v < kVA) {
              sa0.store_vec(v, a_buf(cur ^ 1));
              sa0.load_vec(v, a_next);
            } else {
              sb0.store_vec(v - kVA, b_buf(cur ^ 1));
              sb0.load_vec(v - kVA, b_next);
            }
          }
        }
        Interleave<BM * BN*(PB == 3 ? 6 : 3), kV, 3 * (A_KC ? 1 : 2) + BN * PB * (B_KC ? 1 : 2), kSplitOps,
                   false>();
        __syncthreads();
      };
      for (; t + kPerChunk + 1 < nfull; t += kPerChunk) {  // a chunk
        body(t, 0, std::true_type());
#pragma unroll
        for (int u = 1; u < kPerChunk; ++u) body(t + u, u & 1, std::false_type());
      }
      for (; t < ntiles; ++t) {  // at most a chunk and two
        compute_at(t);
        if (t + 1 < ntiles) {
          const int nxt = static_cast<int>(t & 1) ^ 1;
          sa0.store(a_buf(nxt));
          sb0.store(b_buf(nxt));
          if (t + 2 < ntiles) load_any(sa0, sb0, t + 2);
          __syncthreads();
        }
      }
    }
  } else if (ntiles > 0) {
    sa0.init(p.lda, m0, p.M);
    sb0.init(p.ldb, n0, p.N);
    sa1.init(p.lda, m0, p.M);
    sb1.init(p.ldb, n0, p.N);
    if constexpr (SCL == 1) sa0.sc = sa1.sc = p.op_scale;
    if constexpr (SCL == 2) sb0.sc = sb1.sc = p.op_scale;
    load_any(sa0, sb0, 0);
    if (ntiles > 1) load_any(sa1, sb1, 1);
    sa0.store(a_buf(0));
    sb0.store(b_buf(0));
    __syncthreads();

    static_assert(kPerChunk % 2 == 0, "a chunk takes each register set alike often");
    for (; t + kPerChunk + 1 < nfull; t += kPerChunk) {  // a chunk
      steady(sa0, sb0, sa1, sb1, t, 0, std::true_type());
      steady(sa1, sb1, sa0, sb0, t + 1, 1, std::false_type());
#pragma unroll
      for (int u = 2; u < kPerChunk; u += 2) {
        steady(sa0, sb0, sa1, sb1, t + u, 0, std::false_type());
        steady(sa1, sb1, sa0, sb0, t + u + 1, 1, std::false_type());
      }
    }
    // The remaining stages (at most a chunk and two): masked loads where needed.
    for (; t < ntiles; ++t) {
      const int cur = static_cast<int>(t & 1);
      if (t + 2 < ntiles) {
        if (cur) load_any(sa1, sb1, t + 2);
        else load_any(sa0, sb0, t + 2);
      }
      compute_at(t);
      if (t + 1 < ntiles) {
        if (cur) {
          sa0.store(a_buf(0));
          sb0.store(b_buf(0));
        } else {
          sa1.store(a_buf(1));
          sb1.store(b_buf(1));
        }
        __syncthreads();
      }
    }
  }

#pragma unroll
  for (int i = 0; i < BM; ++i)
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        acc[i][j][v] = __builtin_fmaf(acc[i][j][v], !A_KC && v & 1 ? -unscale : unscale, sum[i][j][v]);

  // Recompute: a non-finite block's outputs by fp32 products, straight from
  // memory (k pairs 16g + j, 16g + 8 + j). Decided per 32x32 block of the
  // output, so that it does not depend on the tile config.
#pragma unroll
  for (int i = 0; i < BM; ++i)
#pragma unroll
    for (int j = 0; j < BN; ++j)
      if (__builtin_expect(AnyNonFinite(acc[i][j]), false)) {
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
        const int64_t m = std::min<int64_t>(m0 + wm0 + 32 * i + r, p.M - 1);
        const int64_t n = std::min<int64_t>(n0 + wn0 + 32 * j + r, p.N - 1);
#pragma unroll 1
        for (int64_t k0 = kb; k0 < ke; k0 += KG)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const bool in = k0 + 8 * h + e < ke;
            const int64_t k = in ? k0 + 8 * h + e : k0;
            float x = A[A_KC ? m * p.lda + k : k * p.lda + m];
            float y = static_cast<float>(B[B_KC ? n * p.ldb + k : k * p.ldb + n]);
            if constexpr (SCL == 1) x = p.op_scale * x;
            if constexpr (SCL == 2) y = p.op_scale * y;
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? x : 0.0f, in ? y : 0.0f, acc[i][j],
                                                             0, 0, 0);
          }
      }

  // A fused AddEW (GemmKArgs::out; FUSED instantiations, launched with one
  // slice and a plain epilogue). On a whole tile, each lane holds one base
  // pointer per array; element (i, j, v) sits a compile-time number of rows
  // and columns from it, so no per-element offsets stay live. The addends
  // are loaded first, all in flight together, then the sums are stored.
  // The value summed is the one the plain epilogue would store in C.
  if constexpr (LORA) if (p.lora_t) {
    // u = T B' block by block, one step of the k loop above (its products,
    // their order and its recomputation, so u has the bits of a tile GEMM).
    // Every fragment of the wavefront's blocks is loaded at once, before any
    // MFMA, so their latencies overlap; each block's outputs are stored right
    // after its MFMAs (stores from one base pointer per lane, with no
    // per-element bounds, measured 5% slower: the per-element form spreads
    // them between the next block's MFMAs).
    float tl[BM + BN][kLoraK];
#pragma unroll
    for (int i = 0; i < BM; ++i) load_lora_t(i, tl[i]);
#pragma unroll
    for (int j = 0; j < BN; ++j) load_lora_b(j, tl[BM + j]);
#pragma unroll
    for (int i = 0; i < BM; ++i)
#pragma unroll
      for (int j = 0; j < BN; ++j) {
        bf16x8 fa[1][3], fb[1][3];
        Split8(tl[i], fa[0], RowNegated(m0 + wm0) ? -kOpScale : kOpScale);
        Split8(tl[BM + j], fb[0], kOpScale);
        floatx16 ua[1][1] = {}, before[1][1] = {};
        MfmaStep<true, A_KC>(fa, fb, ua, before, unscale);
        floatx16& u = ua[0][0];
#pragma unroll
        for (int v = 0; v < 16; ++v) u[v] *= unscale;
        if (__builtin_expect(AnyNonFinite(u), false)) {
#pragma unroll
          for (int v = 0; v < 16; ++v) u[v] = 0.0f;
#pragma unroll
          for (int e = 0; e < kLoraK; ++e)
            u = __builtin_amdgcn_mfma_f32_32x32x2f32(tl[i][e], tl[BM + j][e], u, 0, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int64_t m = m0 + wm0 + 32 * i + 8 * (v >> 2) + 4 * h + (v & 3);
          const int64_t n = n0 + wn0 + 32 * j + r;
          if (m >= p.M || n >= p.N) continue;
          const float val = dev_act(p.act, p.alpha * acc[i][j][v]);
          const float sv = p.out_scaled ? p.out_scale * u[v] : u[v];
          p.out[m * p.ldo + n] = p.lora_y_first ? val + sv : sv + val;
        }
      }
    return;
  }
  if constexpr (FUSED) {
    if (p.out && p.splits == 1 && m0 + MT_M <= p.M && n0 + MT_N <= p.N &&
        (!POST || MT_M * p.ldo * 4 < (int64_t{1} << 30))) {
      const int64_t lm = m0 + wm0 + 4 * h, ln = n0 + wn0 + r;
      const float* ya = p.addend + lm * p.ldo + ln;
      float* oa = p.out + lm * p.ldo + ln;
      float* ca = C + lm * p.ldc + ln;
      float pb[BN];  // POST: the AddBias values of the lane's columns
#pragma unroll
      for (int j = 0; j < BN; ++j) pb[j] = POST ? p.pbias[ln + 32 * j] : 0.0f;
      const int64_t tile0 = m0 * p.ldo + n0;
      char* post_o = POST ? reinterpret_cast<char*>(p.out + tile0) : nullptr;
      char* post_h = POST && p.hout ? reinterpret_cast<char*>(p.hout + tile0) : nullptr;
      char* post_g = POST && p.gout ? reinterpret_cast<char*>(p.gout + tile0) : nullptr;
      const uint32_t post_lane = static_cast<uint32_t>(((lm - m0) * p.ldo + (ln - n0)) * 4);
      float yv[BM][BN][16];
#pragma unroll
      for (int i = 0; i < BM; ++i)
#pragma unroll
        for (int j = 0; j < BN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            yv[i][j][v] = ya[(32 * i + 8 * (v >> 2) + (v & 3)) * p.ldo + 32 * j];
#pragma unroll
      for (int i = 0; i < BM; ++i)
#pragma unroll
        for (int j = 0; j < BN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int64_t row = 32 * i + 8 * (v >> 2) + (v & 3);
            const float val = dev_act(p.act, p.alpha * acc[i][j][v]);
            const float sv = p.out_scaled ? p.out_scale * val : val;
            if (p.write_c) ca[row * p.ldc + 32 * j] = p.c_scaled ? sv : val;
            const float y = yv[i][j][v];
            if constexpr (POST) {
              // 32-bit byte offsets from the tile's wave-uniform origin (the
              // tile's span is checked to fit): three output arrays with no
              // 64-bit address per element.
              const uint32_t at = post_lane + static_cast<uint32_t>((row * p.ldo + 32 * j) * 4);
              const float o = p.addend_first ? y + sv : sv + y;
              if (p.write_out) *reinterpret_cast<float*>(post_o + at) = o;
              const float hv = o + pb[j];
              if (p.hout) *reinterpret_cast<float*>(post_h + at) = hv;
              if (p.gout) *reinterpret_cast<float*>(post_g + at) = dev_act(p.pact, hv);
            } else {
              oa[row * p.ldo + 32 * j] = p.addend_first ? y + sv : sv + y;
            }
          }
      return;
    }
  }

  // A whole tile with the plain epilogue (one slice, no accumulate, bias,
  // activation or causal zeroing): one base pointer per lane, every element
  // a compile-time number of rows and columns from it, no per-element bounds
  // or epilogue branches. Stores what the general write-back below stores.
  if constexpr (VEC) {
    if (!p.out && p.splits == 1 && !p.accumulate && !p.bias && p.act == 0 &&
        p.causal != static_cast<int>(Causal::kLowerOut) && m0 + MT_M <= p.M &&
        n0 + MT_N <= p.N) {
      float* ca = C + (m0 + wm0 + 4 * h) * p.ldc + n0 + wn0 + r;
#pragma unroll
      for (int i = 0; i < BM; ++i)
#pragma unroll
        for (int j = 0; j < BN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            ca[(32 * i + 8 * (v >> 2) + (v & 3)) * p.ldc + 32 * j] = p.alpha * acc[i][j][v];
      return;
    }
  }

  // Write-back. Lane (h, r) of the 32x32 block holds rows 8*(v/4) + 4*h + v%4
  // of column r in accumulator element v.
#pragma unroll
  for (int i = 0; i < BM; ++i)
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int64_t m = m0 + wm0 + 32 * i + 8 * (v >> 2) + 4 * h + (v & 3);
        const int64_t n = n0 + wn0 + 32 * j + r;
        if (m >= p.M || n >= p.N) continue;
        float val = acc[i][j][v];
        if (p.splits > 1) {
          p.ws[(static_cast<int64_t>(slice) * p.M + m) * p.N + n] = val;
          continue;
        }
        val = p.alpha * val;
        if (p.accumulate) val = C[m * p.ldc + n] + val;
        if (p.bias) val = val + p.bias[n];
        val = dev_act(p.act, val);
        if (p.causal == static_cast<int>(Causal::kLowerOut) && n > m) val = 0.0f;
        if (FUSED && p.out) {  // a partial tile
          const float sv = p.out_scaled ? p.out_scale * val : val;
          if (p.write_c) C[m * p.ldc + n] = p.c_scaled ? sv : val;
          const float y = p.addend[m * p.ldo + n];
          if constexpr (POST)
            FusedSum<true>(p, m * p.ldo + n, y, sv, p.pbias[n]);
          else
            p.out[m * p.ldo + n] = p.addend_first ? y + sv : sv + y;
        } else {
          C[m * p.ldc + n] = val;
        }
      }
}

template <int MT_M, int MT_N, int KT, int WAVES_M, int WAVES_N, bool A_KC, bool B_KC, bool B_I8,
          bool VEC, bool FUSED, bool LORA = false, int SCL = 0, bool POST = false>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N, MinWaves(MT_M, MT_N)) void gemm_mfma_kernel(GemmKArgs p) {
  const uint32_t tiles = static_cast<uint32_t>(p.tiles_m) * static_cast<uint32_t>(p.tiles_n);
  const uint32_t lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  const uint32_t L = XcdLogical(lin, tiles * gridDim.y * gridDim.z);
  gemm_tile<MT_M, MT_N, KT, WAVES_M, WAVES_N, A_KC, B_KC, B_I8, VEC, FUSED, LORA, SCL, POST>(
      p, L, gridDim.y);
}

// A GEMM group: up to kMaxGroup independent GEMMs of one tile config and
// operand layout in one launch (each unsplit and unbatched), member j
// owning logical work items [wg_end[j-1], wg_end[j]). The XCD remap runs
// over the whole launch, so each XCD walks a contiguous run of the members'
// tiles. Every output is computed by the same code, k order and epilogue as
// in the member's own launch: the same bits.
constexpr int kMaxGroup = kGemmGroupMax;
struct GemmGroupArgs {
  GemmKArgs m[kMaxGroup];
  uint32_t wg_end[kMaxGroup];
  uint32_t count;
};

template <int MT_M, int MT_N, int KT, int WAVES_M, int WAVES_N, bool A_KC, bool B_KC, bool LORA>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N, MinWaves(MT_M, MT_N)) void gemm_group_kernel(GemmGroupArgs g) {
  const uint32_t total = g.wg_end[g.count - 1];
  uint32_t L = XcdLogical(blockIdx.x, total);
  uint32_t j = 0;
  while (j + 1 < g.count && L >= g.wg_end[j]) ++j;
  if (j > 0) L -= g.wg_end[j - 1];
  gemm_tile<MT_M, MT_N, KT, WAVES_M, WAVES_N, A_KC, B_KC, false, true, true, LORA>(g.m[j], L, 1);
}

// The tile config the general form (!VEC: any extent, stride and alignment;
// int8) runs plan config `cfg` on: it exists for one large tile, whose 32x64 wavefronts leave it the
// registers, and the small one.
inline constexpr int GeneralCfg(int cfg) {
  return cfg <= 3 ? 1 : kCfgSmall;
}

// Launches config `cfg` of one operand-layout variant.
template <bool A_KC, bool B_KC, bool B_I8, bool VEC, bool FUSED = false>
void LaunchVariant(int cfg, dim3 grid, hipStream_t s, const GemmKArgs& a) {
  const dim3 block(kCfgs[cfg].threads);
#define SEEML_GEMM_CASE(I, MM, NN, KK, WM_, WN_)                                                \
  case I:                                                                                     \
    hipLaunchKernelGGL((gemm_mfma_kernel<MM, NN, KK, WM_, WN_, A_KC, B_KC, B_I8, VEC, FUSED>), grid, \
                       block, 0, s, a);                                                       \
    break;
  if constexpr (!VEC) {
    switch (GeneralCfg(cfg)) {
      SEEML_GEMM_CASE(1, 128, 128, 16, 4, 2)
      default:
      SEEML_GEMM_CASE(5, 64, 64, 32, 2, 2)
    }
  } else {
    switch (cfg) {
      SEEML_GEMM_CASE(0, 128, 128, 16, 2, 2)
      SEEML_GEMM_CASE(1, 128, 128, 16, 4, 2)
      SEEML_GEMM_CASE(2, 256, 128, 16, 4, 2)
      SEEML_GEMM_CASE(3, 128, 256, 16, 2, 4)
      SEEML_GEMM_CASE(4, 128, 64, 32, 2, 2)
      SEEML_GEMM_CASE(5, 64, 64, 32, 2, 2)
      SEEML_GEMM_CASE(6, 128, 32, 32, 4, 1)
      SEEML_GEMM_CASE(7, 32, 128, 32, 1, 4)
      SEEML_GEMM_CASE(8, 64, 128, 32, 2, 2)
      SEEML_GEMM_CASE(9, 128, 64, 32, 4, 1)
      SEEML_GEMM_CASE(10, 64, 64, 16, 2, 2)
        default:
      SEEML_GEMM_CASE(11, 64, 128, 16, 2, 2)
    }
  }
#undef SEEML_GEMM_CASE
}

// The LoRA-epilogue instantiations (GemmKArgs::lora_t): the tiles the base
// projection GEMMs run on (the large tiles of the d_model >= 2048 decoders
// and the 128x64 / 64x64 / 64x128 tiles of the small ones). Returns false
// for any other config.
template <bool A_KC, bool B_KC>
bool LaunchLoraVariant(int cfg, dim3 grid, hipStream_t s, const GemmKArgs& a) {
#define SEEML_LORA_CASE(I, MM, NN, KK, WM_, WN_)                                                       \
  case I:                                                                                            \
    hipLaunchKernelGGL((gemm_mfma_kernel<MM, NN, KK, WM_, WN_, A_KC, B_KC, false, true, true, true>), \
                       grid, dim3(kCfgs[I].threads), 0, s, a);                                       \
    return true;
  switch (cfg) {
    SEEML_LORA_CASE(0, 128, 128, 16, 2, 2)
    SEEML_LORA_CASE(2, 256, 128, 16, 4, 2)
    SEEML_LORA_CASE(4, 128, 64, 32, 2, 2)
    SEEML_LORA_CASE(5, 64, 64, 32, 2, 2)
    SEEML_LORA_CASE(8, 64, 128, 32, 2, 2)
    SEEML_LORA_CASE(9, 128, 64, 32, 4, 1)
    default:
      return false;
  }
#undef SEEML_LORA_CASE
}

// Tile configs with a group kernel (gemm_group_kernel): the configs the
// heuristic and the autotuner pick for the decoders' projection GEMMs.
inline constexpr bool GroupCfg(int cfg) { return cfg <= 5 || cfg == 8 || cfg == 9; }

// LORA: some member takes the LoRA epilogue (its registers cost the plain
// members occupancy, so groups without one use the kernel without it).
template <bool B_KC, bool LORA>
bool LaunchGroupVariant(int cfg, dim3 grid, hipStream_t s, const GemmGroupArgs& g) {
#define SEEML_GROUP_CASE(I, MM, NN, KK, WM_, WN_)                                                 \
  case I:                                                                                       \
    hipLaunchKernelGGL((gemm_group_kernel<MM, NN, KK, WM_, WN_, true, B_KC, LORA>), grid,         \
                       dim3(kCfgs[I].threads), 0, s, g);                                         \
    return true;
  switch (cfg) {
    SEEML_GROUP_CASE(0, 128, 128, 16, 2, 2)
    SEEML_GROUP_CASE(2, 256, 128, 16, 4, 2)
    SEEML_GROUP_CASE(4, 128, 64, 32, 2, 2)
    SEEML_GROUP_CASE(5, 64, 64, 32, 2, 2)
    SEEML_GROUP_CASE(8, 64, 128, 32, 2, 2)
    SEEML_GROUP_CASE(1, 128, 128, 16, 4, 2)
    SEEML_GROUP_CASE(3, 128, 256, 16, 2, 4)
    SEEML_GROUP_CASE(9, 128, 64, 32, 4, 1)
    default:
      return false;
  }
#undef SEEML_GROUP_CASE
}

// Tile configs with scaled-load instantiations (LaunchScaledVariant): the
// small tiles the rank-64 LoRA backward's dt = s du B^T (NT, A scaled) and
// dB = t^T (s du) (TN, B scaled) run on.
inline constexpr bool ScaledCfg(int cfg) { return cfg == 4 || cfg == 5 || (cfg >= 8 && cfg <= 11); }

template <bool A_KC, bool B_KC, int SCL>
bool LaunchScaledVariant(int cfg, dim3 grid, hipStream_t s, const GemmKArgs& a) {
#define SEEML_SCALED_CASE(I, MM, NN, KK, WM_, WN_)                                                     \
  case I:                                                                                            \
    hipLaunchKernelGGL((gemm_mfma_kernel<MM, NN, KK, WM_, WN_, A_KC, B_KC, false, true, false, false, \
                                         SCL>),                                                      \
                       grid, dim3(kCfgs[I].threads), 0, s, a);                                       \
    return true;
  switch (cfg) {
    SEEML_SCALED_CASE(4, 128, 64, 32, 2, 2)
    SEEML_SCALED_CASE(5, 64, 64, 32, 2, 2)
    SEEML_SCALED_CASE(8, 64, 128, 32, 2, 2)
    SEEML_SCALED_CASE(9, 128, 64, 32, 4, 1)
    SEEML_SCALED_CASE(10, 64, 64, 16, 2, 2)
    SEEML_SCALED_CASE(11, 64, 128, 16, 2, 2)
    default:
      return false;
  }
#undef SEEML_SCALED_CASE
}

// The post-AddEW instantiations (GemmKArgs::pbias): the fused AddEW's GEMM
// with an AddBias (+ activation) after it, on the small tile configs (the
// rank-64 LoRA up-projections u = t B feeding the biased MLP layers).
template <bool A_KC, bool B_KC>
bool LaunchPostVariant(int cfg, dim3 grid, hipStream_t s, const GemmKArgs& a) {
#define SEEML_POST_CASE(I, MM, NN, KK, WM_, WN_)                                                      \
  case I:                                                                                            \
    hipLaunchKernelGGL((gemm_mfma_kernel<MM, NN, KK, WM_, WN_, A_KC, B_KC, false, true, true, false, \
                                         0, true>),                                                  \
                       grid, dim3(kCfgs[I].threads), 0, s, a);                                       \
    return true;
  switch (cfg) {
    SEEML_POST_CASE(4, 128, 64, 32, 2, 2)
    SEEML_POST_CASE(5, 64, 64, 32, 2, 2)
    SEEML_POST_CASE(8, 64, 128, 32, 2, 2)
    SEEML_POST_CASE(9, 128, 64, 32, 4, 1)
    SEEML_POST_CASE(10, 64, 64, 16, 2, 2)
    SEEML_POST_CASE(11, 64, 128, 16, 2, 2)
    default:
      return false;
  }
#undef SEEML_POST_CASE
}

// Per-layout entry points, one instantiation unit each (built in parallel).
void LaunchNN(int cfg, bool vec, dim3 grid, hipStream_t s, const GemmKArgs& a);
void LaunchNT(int cfg, bool vec, dim3 grid, hipStream_t s, const GemmKArgs& a);
void LaunchTN(int cfg, bool vec, dim3 grid, hipStream_t s, const GemmKArgs& a);
void LaunchQ8(int cfg, bool b_kc, dim3 grid, hipStream_t s, const GemmKArgs& a);
// Group launches (A k-contiguous, B row- or k-contiguous); false for a
// config without a group kernel.
bool LaunchGroupNN(int cfg, dim3 grid, hipStream_t s, const GemmGroupArgs& g);
bool LaunchGroupNT(int cfg, dim3 grid, hipStream_t s, const GemmGroupArgs& g);
// Scaled-load launches: NT with A scaled, TN with B scaled; false for a
// config without the instantiation.
bool LaunchScaledNT(int cfg, dim3 grid, hipStream_t s, const GemmKArgs& a);
bool LaunchScaledTN(int cfg, dim3 grid, hipStream_t s, const GemmKArgs& a);
// Post-AddEW launches (NN); false for a config without the instantiation.
bool LaunchPostNN(int cfg, dim3 grid, hipStream_t s, const GemmKArgs& a);

}  // namespace gemm
}  // namespace seeml_hip
