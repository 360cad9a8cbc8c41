// k_gemm.hip — host side of the matrix-core GEMM engine (fp32): tile planning,
// split-K, launch-shape checks and the split-K reduction kernel. The kernel
// template itself is in k_gemm_kernel.h (design notes there), instantiated
// per operand layout in k_gemm_{nn,nt,tn,q8}.hip.
//
// Serves runtime/executor/gemm.cc:173-228 (GemmNN + fused bias/act
// epilogue, GemmNT, GemmTN, GemmAccNN, GemmNNQ8/NTQ8) and the attention
// contractions of attention.cc.
#include <atomic>
#include "k_gemm_kernel.h"

namespace seeml_hip {

using gemm::CfgInfo;
using gemm::GemmKArgs;
using gemm::kCfgs;
using gemm::kNumCfgs;

namespace {

constexpr int kThreads = 256;

// Sums split-K partials in slice order and applies the epilogue, a fused
// AddEW included (batch 1).
__global__ __launch_bounds__(kThreads) void splitk_reduce_kernel(GemmKArgs p) {
  const int64_t total = p.M * p.N;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads;
  for (int64_t idx = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; idx < total;
       idx += stride) {
    float val = p.ws[idx];
    for (int s = 1; s < p.splits; ++s) val += p.ws[static_cast<int64_t>(s) * total + idx];
    const int64_t m = idx / p.N, n = idx % p.N;
    val = p.alpha * val;
    if (p.accumulate) val = p.C[m * p.ldc + n] + val;
    if (p.bias) val = val + p.bias[n];
    val = dev_act(p.act, val);
    if (p.out) {
      const float sv = p.out_scaled ? p.out_scale * val : val;
      if (p.write_c) p.C[m * p.ldc + n] = p.c_scaled ? sv : val;
      const float y = p.addend[m * p.ldo + n];
      p.out[m * p.ldo + n] = p.addend_first ? y + sv : sv + y;
    } else {
      p.C[m * p.ldc + n] = val;
    }
  }
}

int64_t CeilDiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

bool VecOk(const void* base, int64_t ld, int64_t sb, int64_t sh, int64_t contiguous_extent) {
  return aligned16(base) && ld % 4 == 0 && sb % 4 == 0 && sh % 4 == 0 && contiguous_extent % 4 == 0;
}

}  // namespace

// Plan indices 0..kNumCfgs-1 are the MFMA tile configs; kNumCfgs selects the
// skinny (LoRA-shaped) kernels where the shape admits them.
int GemmSkinnyConfig() { return kNumCfgs; }
int GemmConfigCount() { return kNumCfgs + 1; }
const char* GemmConfigName(int cfg) {
  if (cfg == kNumCfgs) return "skinny";
  return cfg >= 0 && cfg < kNumCfgs ? kCfgs[cfg].name : "?";
}

// The heuristic takes the skinny kernels only for the shapes that stream a
// rank-wide operand through a reduction over the token rows (rowdot: N is
// the rank; colsum: a weight gradient), up to rank kSkinnyMaxRank. Wider
// ranks run on the tile kernels with split-K, which re-read the rank-wide
// operand far less (measured with the stream cold, rank 64: 8192x64x4096
// rowdot 110 -> 63 us, 64x4096x8192 colsum 85 -> 56 us; at rank 16 the two
// are within a few percent either way). A rank-K outer product (K <= 64)
// runs on the tile kernels: they time within 1% of the skinny outer kernel
// alone and their epilogue takes a following Scale + AddEW or a whole LoRA
// run. A forced skinny config still selects the outer kernel (tests).
constexpr int64_t kSkinnyMaxRank = 16;

namespace {
// The tile of a GEMM by how many workgroups each leaves for the chip's 256
// CUs. A larger tile reads its operands less often and splits them less per
// product, and loses more to a last round of the chip that it leaves partly
// idle, to the part of a tile beyond the output, and to the general write-back
// of partial tiles (5-6 us). Measured, one slice, us, NN:
//                 256x128 128x128 64x64 64x64x16              256x128 128x128 64x64 64x64x16
//   8192x2048x2048  355     404    --     --    2048x2752x64    18.9   20.4   15.5   13.7
//   2560x2560x512    44      48    57     56    744x5496x400    41.4   43.7   41.3   37.4
//   2048x2048x2048  139     110   122    122    2048x2752x512   48.2   52.7   48.9   48.2
//   2048x2752x2048  146     162   172    171    2948x1216x236   30.2   26.6   23.0   19.4
//   1024x1024x2048  137     102    42     48    744x5496x2048    145    153    146    144
//   60000x64x256     35      37    26     24    64x65536x512     105     60     38     41
// So: 256x128 from rounds filled to 7/8 on. 128x128 from nearly a workgroup per
// CU on, except below 7/8 of two per CU with partial tiles on a short reduction
// or just past a round. Else 64x64 (128x64 where 64x64 would pass two per CU).
// Outputs up to 64 wide or tall take 64x64. So do causal attention products,
// which skip per tile, below two 128x128 tiles per CU, unless they are tall and
// fill those tiles (one tile per CU, us, 128x128 | 64x64: 16x128x16x80 dQ 24 | 18,
// 2x2000x8x80 dQ 113 | 93; 2x1023x16x128 dQ 58 | 66).
// The 64x64 tile is 16 deep where a reduction of at most 128 has more of them
// than the three per CU that the LDS of the 32-deep one allows (3008x1984x64
// above; the deeper one has the LoRA and group kernels too), and 128x128 of
// eight wavefronts where short split-K slices make that many of filled ones
// (512x512x2048 in 16 slices 32 -> 26 us; 654x1177x6120 in 5 101 -> 122).
// Outputs up to 32 take the 32-wide tiles except with split-K at a workgroup
// per CU at most, where the 64x64 tile's stages are shorter (32x256x512 in two
// slices 12.0 -> 11.0 us; unsplit, its partial tiles pay the general write-back).
int TileFor(const GemmDesc& d, int splits) {
  constexpr int64_t kCus = 256, kMost = kCus * 7 / 8;
  auto tiles = [&](int64_t m, int64_t n) { return CeilDiv(d.M, m) * CeilDiv(d.N, n) * d.batch; };
  const int64_t small_groups = tiles(64, 64) * splits;
  if ((d.N <= 32) != (d.M <= 32) && !(splits > 1 && small_groups <= kCus))
    return d.N <= 32 ? gemm::kCfgSkinnyN : gemm::kCfgSkinnyM;
  const bool narrow = d.M <= 64 || d.N <= 64;
  const bool fills = CeilDiv(d.N, 128) * 128 * 7 <= d.N * 8 && CeilDiv(d.M, 128) * 128 * 7 <= d.M * 8;
  if (splits > 1 && fills && small_groups > 3 * kCus && d.K <= 256 * int64_t{splits}) return gemm::kCfgWaves8;
  const int small = d.K <= 128 && small_groups > 3 * kCus ? gemm::kCfgSmallK16 : gemm::kCfgSmall;
  if (narrow) return small;
  const int64_t large = tiles(256, 128), mid = tiles(128, 128);
  if (d.causal != Causal::kNone) {
    return mid >= 2 * kCus || (mid >= kMost && fills && d.M >= 4 * 128) ? gemm::kCfgDefault : small;
  }
  if (large * 8 >= CeilDiv(large, kCus) * kCus * 7) return gemm::kCfgLarge;
  if (mid >= kMost) {
    const bool partial = d.M % 128 != 0 || d.N % 128 != 0;
    const bool just_past = mid > kCus && mid < kCus * 5 / 4;
    return partial && mid < 2 * kMost && (d.K <= 512 || just_past) ? small : gemm::kCfgDefault;
  }
  if (tiles(128, 64) >= 2 * kMost) return gemm::kCfgHalf;
  return small;
}

// Split-K slices, part of a shape's summation order. The rank-wide outputs of
// the LoRA gradients (rowdot and colsum shapes, kind) have few tiles and a
// long reduction, and so have outputs of at most 64 tiles: enough slices to
// cover the chip twice with 64x64 or 128x128 tiles, each at least 128 deep.
// Elsewhere a slice costs a pass over the output and a launch (about 5 us),
// against about 0.55 us per 32 of depth that a lone workgroup takes: slices of
// 1024, no more than two 128x128 tiles' worth per CU (64x64 tiles' for outputs
// up to 64 wide or tall), where the output leaves CUs idle (600x1024x1024 takes
// 23 us in one slice, 600x1024x4096 82 us in one and 48 in four); two of at least 2048 up to
// two 64x64 tiles per CU (in one and two slices, us, NN: 1024x1024x8192 137 and
// 126, x4096 74 and 70, x2048 39 and 40; 1280x1024x8192 202 and 180); otherwise
// none. No shape takes more slices than 128-deep ones covering the chip twice.
int SplitsFor(const GemmDesc& d, SkinnyKind kind) {
  if (d.batch != 1 || d.causal != Causal::kNone || d.K < 256) return 1;
  const int64_t big = CeilDiv(d.M, 128) * CeilDiv(d.N, 128), mid = CeilDiv(d.M, 64) * CeilDiv(d.N, 64);
  const bool narrow = d.M <= 64 || d.N <= 64;
  const int64_t tiles = d.N <= 32 && d.M > 32   ? CeilDiv(d.M, 128)
                        : d.M <= 32 && d.N > 32 ? CeilDiv(d.N, 128)
                        : big >= 512 || (mid < 256 && !narrow) ? big : mid;
  if (tiles >= 512) return 1;
  int64_t most = d.K / 128;
  if (kind != SkinnyKind::kRowDot && kind != SkinnyKind::kColSum && mid > 64) most = mid < 256 ? d.K / 1024 : d.K / 2048;
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(CeilDiv(512, tiles), std::min<int64_t>(most, 64))));
}

// Whether the 16-byte form's 32-bit byte offsets reach the last row of a tile
// of config `cfg`: k-contiguous rows of 2^22 elements and more are too far
// apart for 256 of them (128, and row-contiguous ones, fit to 2^23).
bool TileOffsetsFit(const GemmDesc& d, int cfg) {
  constexpr int64_t kLong = int64_t{1} << 22;
  return !(d.a_kc && d.lda >= kLong && kCfgs[cfg].mt_m > 128) &&
         !(d.b_kc && d.ldb >= kLong && kCfgs[cfg].mt_n > 128);
}
}  // namespace

GemmPlan PlanGemmWith(const GemmDesc& d, int forced_cfg, int forced_splits) {
  GemmPlan plan;
  const SkinnyKind kind = SkinnyKindOf(d);
  const int64_t rank = kind == SkinnyKind::kRowDot ? d.N : std::min(d.M, d.N);
  const bool skinny = forced_cfg == kNumCfgs
                          ? kind != SkinnyKind::kNone
                          : forced_cfg < 0 && (kind == SkinnyKind::kRowDot || kind == SkinnyKind::kColSum) &&
                                rank <= kSkinnyMaxRank;
  if (skinny) {
    plan.cfg = kNumCfgs;
    plan.splits = 1;
    plan.ws_bytes = SkinnyWorkspace(d);
    return plan;
  }
  if (forced_splits >= 1)
    plan.splits = d.batch == 1 && d.causal == Causal::kNone ? forced_splits : 1;
  else
    plan.splits = SplitsFor(d, kind);
  plan.cfg = forced_cfg >= 0 && forced_cfg < kNumCfgs ? forced_cfg : TileFor(d, plan.splits);
  if (!TileOffsetsFit(d, plan.cfg)) plan.cfg = gemm::kCfgDefault;
  plan.ws_bytes = plan.splits > 1 ? static_cast<size_t>(plan.splits) * d.M * d.N * sizeof(float) : 0;
  return plan;
}

namespace {
// Compute units of the current device (cached per device; engines on
// several host threads may ask at once, and all store the same value).
int DeviceCUs() {
  static std::atomic<int> cus[16] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return 0;
  int n = cus[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess) {
      cus[dev].store(v, std::memory_order_relaxed);
      n = v;
    }
  }
  return n;
}
}  // namespace

GemmOrder GemmOrderOf(const GemmDesc& d) {
  const GemmPlan h = PlanGemmWith(d, -1, -1);
  GemmOrder o;
  o.skinny = h.cfg == kNumCfgs;
  o.splits = o.skinny ? 1 : h.splits;
  return o;
}

bool GemmPlanKeepsOrder(const GemmDesc& d, const GemmPlan& p) {
  const GemmOrder o = GemmOrderOf(d);
  if (o.skinny) return p.cfg == kNumCfgs;
  return p.cfg >= 0 && p.cfg < kNumCfgs && p.splits == o.splits && (p.n_split == 0 || p.splits == 1);
}

// The heuristic plan, and for large GEMMs whose 256x128 tiles leave much of a
// last round idle, the column split of at least two whole rounds with the
// remainder on 64x64 tiles (the autotuner's first arm).
GemmPlan PlanGemm(const GemmDesc& d) {
  const GemmPlan plan = PlanGemmWith(d, -1, -1);
  if (plan.cfg == kNumCfgs || plan.cfg == gemm::kCfgLarge || plan.splits != 1) return plan;
  const GemmPlan sp = PlanGemmSplit(d, 2, gemm::kCfgSmall);
  const int64_t cus = DeviceCUs();
  if (sp.n_split > 0 && cus > 0 && CeilDiv(d.M, 256) * (sp.n_split / 128) >= 2 * cus) return sp;
  return plan;
}


// Only the 256x128 tile, of which one workgroup's registers fill a CU, so
// a round of the chip is exactly one tile per CU.
GemmPlan PlanGemmSplit(const GemmDesc& d, int cfg, int tail_cfg, int64_t n_split) {
  GemmPlan plan = PlanGemmWith(d, cfg, 1);
  if (d.batch != 1 || d.causal != Causal::kNone || d.b_int8 || cfg < 0 || cfg >= kNumCfgs ||
      tail_cfg < 0 || tail_cfg >= kNumCfgs || plan.splits != 1 || !GemmVecForm(d))
    return plan;
  if (n_split <= 0) {
    if (plan.cfg != gemm::kCfgLarge) return plan;
    const CfgInfo& c = kCfgs[cfg];
    const int64_t cus = DeviceCUs();
    const int64_t tm = CeilDiv(d.M, c.mt_m), bands = CeilDiv(d.N, c.mt_n);
    if (cus <= 0 || (tm * bands) % cus == 0) return plan;
    int64_t b = bands - 1;
    while (b > 0 && (tm * b) % cus != 0) --b;
    if (b == 0) return plan;
    n_split = b * c.mt_n;
  }
  if (n_split >= d.N || n_split % 4 != 0) return plan;
  plan.tail_cfg = tail_cfg;
  plan.n_split = n_split;
  return plan;
}

bool GemmVecForm(const GemmDesc& d) {
  return !d.b_int8 && VecOk(d.A, d.lda, d.a_sb, d.a_sh, d.a_kc ? d.K : d.M) &&
         VecOk(d.B, d.ldb, d.b_sb, d.b_sh, d.b_kc ? d.K : d.N) &&
         d.lda < (int64_t{1} << 23) && d.ldb < (int64_t{1} << 23);
}

// Validates a tile-kernel launch of d under plan (one column range, no
// skinny kernels) and fills its kernel arguments, grid, config and load form.
Status CheckEpilogue(const GemmDesc& d, const GemmPlan& plan) {
  if (d.lora_t && (!d.out || d.addend || d.lora_r <= 0 || d.lora_r % 8 != 0 || d.lora_r > 16 || !d.lora_b ||
                   !aligned16(d.lora_t) || d.lora_ldt % 4 != 0 || plan.splits != 1 ||
                   !GemmLoraCfgOk(plan.cfg, d.b_kc) || !d.a_kc || d.b_int8 || d.batch != 1 ||
                   d.causal != Causal::kNone || d.accumulate || d.bias || !GemmVecForm(d)))
    return Status::Fail(kUnitEngine, "Gemm: unsupported LoRA epilogue");
  if (d.post_bias && !GemmPostOk(d, plan))
    return Status::Fail(kUnitEngine, "Gemm: unsupported AddBias after the fused AddEW");
  if (!d.post_bias && (d.post_h || d.post_g || !d.write_out))
    return Status::Fail(kUnitEngine, "Gemm: post-AddEW outputs without the AddBias");
  if (d.out && !d.lora_t && (!d.addend || d.batch != 1 || d.ldc != (d.ldo ? d.ldo : d.N) || d.causal != Causal::kNone ||
                d.accumulate || d.bias))
    return Status::Fail(kUnitEngine,
                        "Gemm: a fused AddEW needs batch 1, ldc == N and a plain epilogue "
                        "(no accumulate, bias or causal mode)");
  return Status::Ok();
}

Status PrepareKArgs(const GemmDesc& d, const GemmPlan& plan, const Ctx& ctx, GemmKArgs* out,
                    dim3* grid, int* cfg_out, bool* vec_out) {
  if (Status s = CheckEpilogue(d, plan); !s) return s;
  if (d.b_int8 && !d.a_kc)
    return Status::Fail(kUnitEngine, "Gemm: unsupported int8 operand layout");
  if (!d.a_kc && d.b_kc)
    return Status::Fail(kUnitEngine, "Gemm: unsupported operand layout (A row-major in m, B k-contiguous)");

  // 16-byte vector loads need 16-byte alignment of every batch base and a
  // contiguous extent that is a multiple of 4 (a float4 is then wholly in or
  // out of range); per-lane offsets within a tile must fit 32 bits. Other
  // GEMMs (int8 B, odd shapes) take the general form of the plan's tile.
  const bool vec = GemmVecForm(d);
  if (d.out_scaled && (!d.out || !vec))
    return Status::Fail(kUnitEngine, "Gemm: a fused Scale + AddEW needs the 16-byte-load kernels");
  if (d.out && !vec && d.ldo && d.ldo != d.N)
    return Status::Fail(kUnitEngine, "Gemm: a column view's fused AddEW needs the 16-byte-load kernels");
  if (d.out && !vec) return Status::Fail(kUnitEngine, "Gemm: a fused AddEW needs the 16-byte-load kernels");
  if (vec && !TileOffsetsFit(d, plan.cfg))
    return Status::Fail(kUnitEngine, "Gemm: row strides too long for this tile config");
  const int cfg = vec ? plan.cfg : gemm::GeneralCfg(plan.cfg);
  const CfgInfo& c = kCfgs[cfg];
  const int64_t tm = CeilDiv(d.M, c.mt_m), tn = CeilDiv(d.N, c.mt_n);
  // The kernel decomposes its linear workgroup id in 32 bits.
  if (tm * tn > 0x7FFFFFFF || d.batch > 65535 || plan.splits > 65535 ||
      tm * tn * c.threads > 0xFFFFFFFF || tm * tn * plan.splits * d.batch > 0xFFFFFFFF)
    return Status::Fail(kUnitEngine, "Gemm: grid exceeds launch limits");

  GemmKArgs& a = *out;
  a = GemmKArgs{};
  a.A = d.A;
  a.B = d.B;
  a.C = d.C;
  a.ws = static_cast<float*>(ctx.ws);
  a.M = d.M; a.N = d.N; a.K = d.K;
  a.lda = d.lda; a.ldb = d.ldb; a.ldc = d.ldc;
  a.heads = std::min(d.heads, d.batch);  // same (z / heads, z % heads) for z < batch; fits 32 bits
  a.batch = d.batch;
  a.a_sb = d.a_sb; a.a_sh = d.a_sh; a.b_sb = d.b_sb; a.b_sh = d.b_sh;
  a.c_sb = d.c_sb; a.c_sh = d.c_sh;
  a.alpha = d.alpha;
  a.accumulate = d.accumulate ? 1 : 0;
  a.bias = d.bias;
  a.act = d.act;
  a.causal = static_cast<int>(d.causal);
  a.splits = plan.splits;
  a.k_per_split = plan.splits > 1
                      ? CeilDiv(CeilDiv(d.K, plan.splits), gemm::kSplitAlign) * gemm::kSplitAlign
                      : d.K;
  a.tiles_m = static_cast<int>(tm);
  a.tiles_n = static_cast<int>(tn);
  a.addend = d.addend;
  a.out = d.out;
  a.addend_first = d.addend_first ? 1 : 0;
  a.write_c = d.write_c ? 1 : 0;
  a.out_scale = d.out_scale;
  a.out_scaled = d.out_scaled ? 1 : 0;
  a.c_scaled = d.c_gets_scaled ? 1 : 0;
  a.ldo = d.ldo ? d.ldo : d.N;
  a.lora_t = d.lora_t;
  a.lora_b = d.lora_b;
  a.lora_ldt = d.lora_ldt;
  a.lora_ldb = d.lora_ldb;
  a.lora_r = d.lora_r;
  a.lora_y_first = d.lora_y_first ? 1 : 0;
  a.op_scale = d.scale_stream ? d.stream_scale : 1.0f;
  a.pbias = d.post_bias;
  a.hout = d.post_h;
  a.gout = d.post_g;
  a.pact = d.post_act;
  a.write_out = d.write_out ? 1 : 0;

  *grid = dim3(static_cast<unsigned>(tm * tn), static_cast<unsigned>(plan.splits),
               static_cast<unsigned>(d.batch));
  *cfg_out = cfg;
  *vec_out = vec;
  return Status::Ok();
}

Status LaunchGemm(const GemmDesc& d, const GemmPlan& plan, const Ctx& ctx) {
  if (d.M <= 0 || d.N <= 0 || d.batch <= 0 || d.heads <= 0)
    return Status::Fail(kUnitEngine, "Gemm: empty shape");
  if (plan.n_split > 0) {
    if (plan.n_split >= d.N || plan.n_split % 4 != 0 || plan.splits != 1 || d.batch != 1 ||
        d.causal != Causal::kNone || d.b_int8 || plan.cfg < 0 || plan.cfg >= kNumCfgs ||
        plan.tail_cfg < 0 || plan.tail_cfg >= kNumCfgs)
      return Status::Fail(kUnitEngine, "Gemm: unsupported column split");
    // Two launches over column ranges of the same operands: C, B's columns,
    // bias and the fused AddEW's arrays are offset views with the full row
    // strides.
    const int64_t n1 = plan.n_split;
    GemmDesc left = d, right = d;
    left.N = n1;
    right.N = d.N - n1;
    const float* B = static_cast<const float*>(d.B);
    right.B = d.b_kc ? B + n1 * d.ldb : B + n1;
    right.C = d.C + n1;
    if (d.bias) right.bias = d.bias + n1;
    if (d.out) {
      left.ldo = right.ldo = d.ldo ? d.ldo : d.N;
      if (d.addend) right.addend = d.addend + n1;
      right.out = d.out + n1;
    }
    if (d.lora_t) right.lora_b = d.lora_b + n1;
    GemmPlan pl, pr;
    pl.cfg = plan.cfg;
    pr.cfg = plan.tail_cfg;
    if (Status s = LaunchGemm(left, pl, ctx); !s) return s;
    return LaunchGemm(right, pr, ctx);
  }
  if (d.scale_stream && plan.cfg != kNumCfgs && !GemmScaledOk(d, plan))
    return Status::Fail(kUnitEngine,
                        "Gemm: a scaled stream needs the skinny kernels or a scaled tile config");
  if (plan.cfg == kNumCfgs) {
    if (d.out) return Status::Fail(kUnitEngine, "Gemm: the skinny kernels take no fused AddEW");
    if (ctx.ws_bytes < SkinnyWorkspace(d))
      return Status::Fail(kUnitEngine, "Gemm: workspace too small for the skinny kernel");
    return LaunchSkinny(d, ctx);
  }
  if (plan.cfg < 0 || plan.cfg >= kNumCfgs) return Status::Fail(kUnitEngine, "Gemm: bad tile config");
  if (plan.splits > 1 && (d.batch != 1 || d.causal != Causal::kNone))
    return Status::Fail(kUnitEngine, "Gemm: split-K needs an unbatched, non-causal GEMM");
  if (plan.splits > 1 && ctx.ws_bytes < plan.ws_bytes)
    return Status::Fail(kUnitEngine, "Gemm: workspace too small for split-K");
  if (Status s = CheckEpilogue(d, plan); !s) return s;
  const bool vec_form = GemmVecForm(d);
  if (d.out && !d.lora_t && !vec_form && !d.out_scaled && !(d.ldo && d.ldo != d.N)) {
    // The general form has no fused epilogue: the GEMM stores C (always
    // safe: C's range is C's while the GEMM writes it), then the AddEW runs.
    GemmDesc plain = d;
    plain.addend = nullptr;
    plain.out = nullptr;
    if (Status s = LaunchGemm(plain, plan, ctx); !s) return s;
    return d.addend_first ? AddEW(d.addend, d.C, d.out, static_cast<size_t>(d.M * d.N), ctx)
                          : AddEW(d.C, d.addend, d.out, static_cast<size_t>(d.M * d.N), ctx);
  }
  GemmKArgs a;
  dim3 grid;
  int cfg = 0;
  bool vec = false;
  if (Status s = PrepareKArgs(d, plan, ctx, &a, &grid, &cfg, &vec); !s) return s;
  if (d.post_bias) {  // GemmPostOk: NN
    if (!gemm::LaunchPostNN(cfg, grid, ctx.stream, a))
      return Status::Fail(kUnitEngine, "Gemm: no post-AddEW kernel for this tile config");
  } else if (d.scale_stream) {  // GemmScaledOk: NT with A the stream, or TN with B
    const bool launched = d.a_kc ? gemm::LaunchScaledNT(cfg, grid, ctx.stream, a)
                                 : gemm::LaunchScaledTN(cfg, grid, ctx.stream, a);
    if (!launched) return Status::Fail(kUnitEngine, "Gemm: no scaled-load kernel for this tile config");
  } else if (d.b_int8) {
    gemm::LaunchQ8(cfg, d.b_kc, grid, ctx.stream, a);
  } else if (d.a_kc && !d.b_kc) {
    gemm::LaunchNN(cfg, vec, grid, ctx.stream, a);
  } else if (d.a_kc && d.b_kc) {
    gemm::LaunchNT(cfg, vec, grid, ctx.stream, a);
  } else {
    gemm::LaunchTN(cfg, vec, grid, ctx.stream, a);
  }
  if (Status s = LaunchStatus("Gemm"); !s) return s;
  if (plan.splits > 1) {
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3(grid_for(static_cast<size_t>(d.M * d.N), kThreads, 8192)),
                       dim3(kThreads), 0, ctx.stream, a);
    return LaunchStatus("Gemm(split-K reduce)");
  }
  return Status::Ok();
}

bool GemmScaledOk(const GemmDesc& d, const GemmPlan& plan) {
  if (plan.n_split != 0 || !gemm::ScaledCfg(plan.cfg) || !GemmVecForm(d) || d.out || d.lora_t ||
      d.b_int8 || d.batch != 1 || d.causal != Causal::kNone)
    return false;
  int64_t elems = 0;
  const void* stream = SkinnyStream(d, &elems);
  if (!stream) return false;
  if (d.a_kc && d.b_kc) return stream == d.A;
  if (!d.a_kc && !d.b_kc) return stream == d.B;
  return false;
}

bool GemmPostOk(const GemmDesc& d, const GemmPlan& plan) {
  return d.post_bias && d.out && d.addend && !d.lora_t && !d.scale_stream && d.a_kc && !d.b_kc &&
         !d.b_int8 && d.batch == 1 && d.causal == Causal::kNone && !d.accumulate && !d.bias &&
         d.act == 0 && plan.splits == 1 && plan.n_split == 0 && gemm::ScaledCfg(plan.cfg) &&
         GemmVecForm(d) && (d.post_act >= 0 && d.post_act <= 3);
}

bool GemmLoraCfgOk(int cfg, bool b_kc) {
  return cfg == 2 || cfg == 4 || cfg == 5 || cfg == 8 || cfg == 9 || (cfg == 0 && b_kc);
}

bool GemmGroupFits(const GemmDesc* ds, const GemmPlan* ps, int n) {
  if (n < 2 || n > gemm::kMaxGroup) return false;
  for (int j = 0; j < n; ++j) {
    const GemmDesc& d = ds[j];
    const GemmPlan& p = ps[j];
    if (p.cfg != ps[0].cfg || !gemm::GroupCfg(p.cfg) || p.splits != 1 || p.n_split != 0 ||
        d.batch != 1 || d.causal != Causal::kNone || d.b_int8 || !d.a_kc || d.b_kc != ds[0].b_kc ||
        d.scale_stream || d.post_bias || !GemmVecForm(d) || !CheckEpilogue(d, p))
      return false;
  }
  return true;
}

Status LaunchGemmGroup(const GemmDesc* ds, const GemmPlan* ps, int n, const Ctx& ctx) {
  if (!GemmGroupFits(ds, ps, n)) return Status::Fail(kUnitEngine, "Gemm group: members do not fit one launch");
  gemm::GemmGroupArgs g{};
  uint64_t total = 0;
  for (int j = 0; j < n; ++j) {
    dim3 grid;
    int cfg = 0;
    bool vec = false;
    if (Status s = PrepareKArgs(ds[j], ps[j], ctx, &g.m[j], &grid, &cfg, &vec); !s) return s;
    total += static_cast<uint64_t>(grid.x);
    if (total > 0x7FFFFFFF / static_cast<uint64_t>(kCfgs[cfg].threads))
      return Status::Fail(kUnitEngine, "Gemm group: grid exceeds launch limits");
    g.wg_end[j] = static_cast<uint32_t>(total);
  }
  g.count = static_cast<uint32_t>(n);
  const dim3 grid(static_cast<unsigned>(total));
  const bool ok = ds[0].b_kc ? gemm::LaunchGroupNT(ps[0].cfg, grid, ctx.stream, g)
                             : gemm::LaunchGroupNN(ps[0].cfg, grid, ctx.stream, g);
  if (!ok) return Status::Fail(kUnitEngine, "Gemm group: no group kernel for this tile config");
  return LaunchStatus("Gemm group");
}

GemmDesc GemmNNDesc(const float* A, const float* B, float* C, int64_t M, int64_t N, int64_t K) {
  GemmDesc d;
  d.A = A; d.B = B; d.C = C; d.M = M; d.N = N; d.K = K;
  d.lda = K; d.ldb = N; d.ldc = N;
  d.a_kc = true; d.b_kc = false;
  return d;
}

GemmDesc GemmNTDesc(const float* A, const float* B, float* C, int64_t M, int64_t N, int64_t K) {
  GemmDesc d;
  d.A = A; d.B = B; d.C = C; d.M = M; d.N = N; d.K = K;
  d.lda = K; d.ldb = K; d.ldc = N;
  d.a_kc = true; d.b_kc = true;
  return d;
}

GemmDesc GemmTNDesc(const float* A, const float* B, float* C, int64_t M, int64_t N, int64_t K) {
  GemmDesc d;
  d.A = A; d.B = B; d.C = C; d.M = M; d.N = N; d.K = K;
  d.lda = M; d.ldb = N; d.ldc = N;
  d.a_kc = false; d.b_kc = false;
  return d;
}

}  // namespace seeml_hip
