// Which tiles the prefill kernel (woq_gemm_w4.h) takes, whether workgroups share K, and its launches under bf16 compute.
#include <algorithm>
#include <cmath>

#include "woq_gemm_w4.h"

namespace woq {

// The kernel needs whole K steps of 128, activations already in the regime's dtype, and a group size
// whose boundaries never split a lane's 32 consecutive K values (8-bit weights: a K step, so groups of
// at least 128 or one scale per channel).  NF4 codes like the 4-bit integers.
bool gemm_w4_applies(const FpArgs& f, int wbits, int regime) {
  const int want = regime == kRegimeF16 ? WOQ_HIP_ACT_FP16 : WOQ_HIP_ACT_BF16;
  if ((wbits != 4 && wbits != 8) || f.x_dtype != want || ((uintptr_t)f.x & 15) != 0) return false;
  if (f.K % kTileK4 != 0 || f.K * 256 * 2 >= (int64_t)1 << 31) return false;
  if (f.G >= f.KT * (wbits == 4 ? kTileK4 : kTileK8)) return true;  // per-channel: one group
  return f.G >= (wbits == 4 ? 32 : 128) && (f.G & (f.G - 1)) == 0;
}

// ---- which tiles, and whether workgroups share K: the lowest of these estimates -----------------------------------------
// Microseconds of a K step of 128 by the weights' kind, measured at K = 4096 .. 14336 with one, two and (48 KiB of LDS) three
// 64 x 128 workgroups on a CU, one and two of 128 x 128, one of the others.  A workgroup alone on its CU has one wave a SIMD
// (eight waves: two), which issues a vector instruction every eight clocks only, two or three waves together one every four:
// that is why two tiles on a CU cost 1.6 times as much as one, and why sharing K pays until every CU has its three workgroups.
// The shared tiles cost about 0.25 and 0.5 us a megabyte besides (64 x 128, 128 x 256), written and read once: reduction terms.
// (INT4, M = 333, 11008 -> 4096: 72 us unsplit, 49-55 with 64 x 128 tiles in four, 46-50 with 128 x 256 in four; M = 128, 7168 ->
// 2048 25.7 with two, 17.8 with four; NF4, M = 77, 4096 -> 11008 40 -> 26.6; FP8, M = 1000, 7168 -> 4096 95 with 128 x 128 tiles, 77 with 128 x 256 in two).
struct StepTimes {
  double t42[3];   // 64 x 128
  double t2[2];    // 128 x 128 (0: not built)
  double t8, t8f;  // 128 x 256 on at most 192 CUs, on more (the clock drops)
  double t7, t163; // 128 x 448, 256 x 192 (0: not built)
};
constexpr StepTimes kSteps4 = {{0.74, 1.22, 1.66}, {1.05, 2.02}, 1.50, 1.68, 3.05, 2.75};
constexpr StepTimes kStepsNf4 = {{1.07, 1.50, 2.05}, {0, 0}, 1.85, 1.90, 0, 0};
constexpr StepTimes kSteps8 = {{0.73, 1.36, 0}, {1.25, 0}, 1.62, 1.80, 0, 0};
constexpr StepTimes kStepsFp8 = {{1.04, 1.82, 0}, {1.52, 0}, 1.95, 2.02, 0, 0};

struct TilePlan {
  int shape = 42, splits = 1;  // shape as launch_gemm_w4's argument
  double us = 1e30;
};
constexpr int kSplitMinSteps = 4;
constexpr int64_t kSplitScratchMax = 32 << 20;  // partial tiles of 256 workgroups of 128 x 256, the most that a plan has (64 x 128: 768, 24 MiB)
static int64_t split_bytes(int64_t M, int64_t N, int shape, int splits) {
  const int64_t bm = shape == 5 ? 128 : 64, bn = shape == 5 ? 256 : 128;
  return splits * ((M + bm - 1) / bm) * ((N + bn - 1) / bn) * bm * bn * (int64_t)sizeof(float);
}
// What a tile costs besides its K steps: the tables, the first requests, the stores (one 128 x 256 workgroup a CU: nothing hides them).
constexpr double kSlotUs8 = 6.0, kSlotUs42 = 5.0;
// scratch: bytes with which K may be shared between workgroups (split_k_prefill_rows, at least four steps each), 0: not; pair: gate and
// up as one problem of twice the columns, in the shapes whose waves have an even number of row-blocks
static TilePlan plan_tiles(int64_t M, int64_t N, int ksteps, const StepTimes& t, int64_t scratch, bool pair = false) {
  const int64_t np = (N + kTileN - 1) / kTileN * kTileN;
  auto wgs = [&](int bm, int bn) { return ((np + bn - 1) / bn) * ((M + bm - 1) / bm); };
  auto gens = [](int64_t w) { return (double)((w + 255) / 256); };
  TilePlan best;
  auto offer = [&](int shape, int splits, double us) {
    if (us < best.us) best.shape = shape, best.splits = splits, best.us = us;
  };
  scratch = std::min(scratch, kSplitScratchMax);
  const bool share = scratch > 0 && split_k_prefill_rows(M, np);
  const int most42 = t.t42[2] > 0 ? 3 : 2, most2 = t.t2[1] > 0 ? 2 : 1;
  for (int s = 1; s <= (share ? kPrefillSplitMax : 1); ++s) {
    const int kts = s == 1 ? ksteps : split_k_steps(ksteps, s);
    if (s > 1 && (kts < kSplitMinSteps || (s - 1) * kts >= ksteps)) break;
    const int64_t w42 = wgs(64, 128) * s, w8 = wgs(128, 256) * s;
    // (a short K must gain a microsecond: M = 116, 1280 -> 2973 ran 17.2 us shared by an estimate of 0.1 us less, 15.6 not)
    const double margin = (int64_t)ksteps * kTileK4 < kSplitKPrefillMinK ? 1.0 : 0.0;
    auto red = [&](int shape, double a, double b) { return s == 1 ? 0.0 : margin + a + b * (double)split_bytes(M, np, shape, s) * 1e-6; };
    const bool fits42 = s == 1 || split_bytes(M, np, 42, s) <= scratch, fits8 = s == 1 || split_bytes(M, np, 5, s) <= scratch;
    if (w42 <= 256 * most42 && fits42)
      offer(42, s, kts * t.t42[(w42 + 255) / 256 - 1] + red(42, 2.0 + 0.4 * s, 0.25));
    else if (s == 1)
      offer(42, 1, kts * t.t42[most42 - 1] * ((double)w42 / (256 * most42) + 0.25));
    if (s == 1 || (w8 <= 256 && fits8))
      offer(5, s, kts * gens(w8) * (w8 <= 192 ? t.t8 : t.t8f) + red(5, 2.0, 0.48));
  }
  const int64_t w2 = wgs(128, 128);
  if (t.t2[0] > 0 && !pair)
    offer(2, 1, ksteps * (w2 <= 256 ? t.t2[0] : most2 == 1 ? gens(w2) * t.t2[0] : t.t2[1] * (w2 <= 512 ? 1.0 : (double)w2 / 512 + 0.1)));
  if (t.t163 > 0 && !pair && wgs(256, 192) % 256 == 0) offer(163, 1, ksteps * gens(wgs(256, 192)) * t.t163);
  if (t.t7 > 0 && !pair) offer(7, 1, ksteps * gens(wgs(128, 448)) * t.t7);
  best.us += 0.125 * ksteps;  // launch, first requests, stores: 4 us at K = 4096, in proportion as in gemm_dense_cost's figures
  return best;
}
static const StepTimes& step_times(int wbits, int nf4, int fp8) { return wbits == 8 ? (fp8 ? kStepsFp8 : kSteps8) : nf4 ? kStepsNf4 : kSteps4; }

// K steps of a chain for an expert (whose own launch has scratch from kSplitKPrefillMinK on) of 64 (i - 1) < rows <= 64 i rows,
// i = 2 ..: as its own launch shares them with the scratch that woq_hip_linear_auto_split_k_workspace_bytes asks for (0: one chain).
static int chain_steps(int64_t K, int64_t N, int wbits, int row_tiles) {
  const int ksteps = (int)(K / kTileK4);
  const TilePlan p = plan_tiles(64 * row_tiles, N, ksteps, step_times(wbits, 0, 0), K >= kSplitKPrefillMinK ? kSplitScratchMax : 0);
  return p.splits > 1 ? split_k_steps(ksteps, p.splits) : 0;
}
// The largest [rows / 64, rounded up] that split_k_prefill_rows holds for.
static int chain_row_tiles(int64_t N) {
  return (int)std::max(kSplitKPrefillMaxRows / 64, kSplitKPrefillTiles / ((N + 127) / 128));
}
// Routed slots on 128 x 256 and 160 x 256 tiles: the K step of a slot of that many rows as a part of one of 128 (32 and 64 rows run their
// own bodies, of 128-row slots the others run that of 128; ten row tiles in chains keep the chain's sum in part in memory).
static double slot_weight(int64_t rows, int tile_rows, bool chained) {
  if (tile_rows == 128 && rows > 64) return 1.0;
  return (0.4 + 0.0047 * (double)((rows + 31) / 32 * 32)) * (chained && rows > 128 ? 1.12 : 1.0);
}
// Estimated microseconds of one grouped launch.  Slots of 160 are much alike (an expert's rows lie evenly in them), so they run in whole
// generations of the mean slot, the last of which ends with the tallest; of those of 128 the low ones fill what the tall ones
// leave.  (Without the tallest 160 rows were taken for experts of uneven sizes, where 128 are faster: of 159 layers of 8 to 64 experts with 60
// to 340 rows in the mean 15 by 1..12 %, now 2; 64 / 128 / 160 rows, us: 8 x 70..147 4352 -> 2816 148 / 123 / 138, 16 x 34..513 2048 -> 7168
// 473 / 411 / 433, 8 x 34..282 4096 -> 14336 751 / 654 / 694.)  From INT4 g128 / g64 / g32, us of a layer with 64, 128 and 160 rows a
// slot, experts x rows: 32 x 128 7168 -> 2048 606 / 537 / 494 and 3072 -> 1024 205 / 218 / 181, 16 x 100 4096 -> 2048 190 / 164 / 161, 8 x 256
// 7168 -> 2048 312 / 295 / 261, 16 x 250 5120 -> 1536 343 / 313 / 319, 8 x 128 4096 -> 1024 123 / 130 / 147 and 7168 -> 1024 158 / 177 / 189,
// 8 x 75 2048 -> 512 112 / 119 / 123, 8 x 100 5120 -> 2048 144 / 149 / 149, 8 x 450 1024 -> 2048 151 / 152 / 157.
static double grouped_us(const int64_t* counts, int64_t experts, int64_t K, int64_t N, int64_t N_own, int wbits, int tile_rows) {
  const StepTimes& t = step_times(wbits, 0, 0);
  const double steps = (double)((K + kTileK4 - 1) / kTileK4);
  int64_t slots = 0;
  double weight = 0, tallest = 0;
  for (int64_t e = 0; e < experts; ++e) {
    const int64_t n = counts[e];
    if (n <= 64) continue;
    const bool chained = tile_rows == 160 && (n + 63) / 64 <= chain_row_tiles(N_own) && chain_steps(K, N_own, wbits, (int)((n + 63) / 64));
    const int64_t own = (n + tile_rows - 1) / tile_rows;
    slots += own;
    if (tile_rows == 160) {
      const double each = slot_weight((n + own - 1) / own, 160, chained);
      weight += (double)own * each;
      tallest = std::max(tallest, each);
    } else
      weight += (double)(n / tile_rows) + (n % tile_rows ? slot_weight(n % tile_rows, 128, false) : 0.0);
  }
  if (tile_rows == 64) {
    const int most = t.t42[2] > 0 ? 3 : 2;
    const int64_t w = (N + 127) / 128 * slots;
    if (w <= 256 * most) return steps * t.t42[(w + 255) / 256 - 1] + kSlotUs42;
    return (steps * t.t42[most - 1] + kSlotUs42) * ((double)w / (256 * most) + 0.25);
  }
  const double cols = (double)((N + 255) / 256);
  const double mean = weight / (double)slots, w = cols * (tile_rows == 160 ? (double)slots : weight), gens = std::ceil(w / 256);
  const double us = steps * (w <= 192 ? t.t8 : t.t8f) * 1.05;
  return tile_rows == 160 ? us * (mean * gens + tallest - mean) + kSlotUs8 * gens : (us + kSlotUs8) * gens;
}
int gemm_w4_tile_rows(const int64_t* counts, int64_t experts, const int64_t* K, const int64_t* N, const int* wbits) {
  int best = 64;
  double us = 1e30;
  if (std::none_of(counts, counts + experts, [](int64_t n) { return n > 64; })) return best;
  for (int rows : {64, 128, 160}) {
    if (rows == 160 && (wbits[0] != 4 || wbits[1] != 4)) continue;
    const double here = grouped_us(counts, experts, K[0], N[0], N[0] / 2, wbits[0], rows) + grouped_us(counts, experts, K[1], N[1], N[1], wbits[1], rows);
    if (here < us) best = rows, us = here;
  }
  return best;
}
int gemm_w4_split_rows(int64_t K, int64_t N) {
  for (int i = chain_row_tiles(N); i >= 2; --i)
    if (chain_steps(K, N, 4, i) || chain_steps(K, N, 8, i)) return 64 * i;
  return 0;
}

// The slots of a routed layer (launch_gemm_w4_grouped) and the fp16 compute type have files of their own.
int gemm_w4_chain_steps(const FpArgs& f, int wbits, int row_tiles) { return row_tiles <= chain_row_tiles(f.N) ? chain_steps(f.K, f.N, wbits, row_tiles) : 0; }

// Estimated time of the automatic choice below with that scratch, in microseconds, for the comparison with the dense kernel
// (gemm_dense_cost).
double gemm_w4_cost(const FpArgs& f, int wbits, int64_t scratch_bytes) {
  return plan_tiles(f.M, f.N, (int)(f.KT / (wbits / 4)), step_times(wbits, f.nf4, f.fp8), scratch_bytes).us;
}

int64_t gemm_w4_scratch_bytes(int64_t M, int64_t N, int64_t ksteps, int wbits, int nf4, int fp8, bool pair, int64_t most) {
  if (most == 0) most = kSplitScratchMax;
  const TilePlan p = plan_tiles(M, pair ? 2 * N : N, (int)ksteps, step_times(wbits, nf4, fp8), most, pair);
  return p.splits > 1 ? std::min(most, split_bytes(M, (pair ? 2 * N : N) + 2 * kTileN - 1, p.shape, p.splits)) : 0;
}

// Gate and up of a gated MLP as one launch: it has twice the workgroups where one of them leaves the chip idle, and the gate's rows stay
// in registers, where two launches store them, read them and pass the post-op's epilogue twice (which costs a launch of its own 6 us,
// M = 1024, 4096 -> 14336: 105 us without, 166 with the silu, 221 with the product).  Two launches / the pair, us, g128: 1024 -> 512, M = 65
// 29.8 / 10.1, 4096 31.8 / 16.1; 2048 -> 5504, M = 128 37.5 / 15.6, 512 68 / 32, 4096 265 / 205; 4096 -> 14336, M = 128 69 / 45, 512 138 / 114,
// 2048 774 / 450, 4096 1000 / 854; 8192 -> 28672, M = 128 167 / 113, 4096 3370 / 3109.  Nowhere slower by more than 3 % up to 4096 rows
// (where the estimate keeps two launches the two are the same).  The lower bounds are not of speed -- 256 -> 512, M = 256 would be
// 22.6 / 6.8 --: smaller layers have the bits of the two launches.
constexpr int64_t kPairMinK = 1024, kPairMinN = 512;
bool gemm_w4_pair_applies(const FpArgs& f, int wbits, int regime) {
  if (wbits != 4 || regime != kRegimeBF16 || f.nf4 || !f.szb || !f.szb_b || f.M <= 64 || f.K < kPairMinK || f.N < kPairMinN) return false;
  if (!gemm_w4_applies(f, wbits, regime)) return false;
  const int ksteps = (int)f.KT;
  return plan_tiles(f.M, 2 * f.N, ksteps, kSteps4, kSplitScratchMax, true).us < 2 * plan_tiles(f.M, f.N, ksteps, kSteps4, kSplitScratchMax).us;
}
int launch_gemm_w4_pair(const FpArgs& f, hipStream_t st, const SplitKScratch* scratch) {
  int g_shift = 30;
  if (f.G < f.KT * kTileK4) {
    g_shift = 0;
    while (((int64_t)1 << g_shift) < f.G) ++g_shift;
  }
  const bool have = scratch && scratch->partial && scratch->counters;
  const TilePlan p = plan_tiles(f.M, 2 * f.N, (int)f.KT, kSteps4, have ? scratch->bytes : 0, true);
  return p.shape == 5 ? launch_shape<kRegimeBF16, G4Shape<8, 2, 8>, 4, false, false, true>(f, g_shift, st, p.splits, scratch)
                      : launch_shape<kRegimeBF16, G4Shape<4, 2>, 4, false, false, true>(f, g_shift, st, p.splits, scratch);
}

int launch_gemm_w4(const FpArgs& f, int wbits, int regime, hipStream_t st, int shape, int splits,
                   const SplitKScratch* scratch) {
  int g_shift = 30;
  if (f.G < f.KT * (wbits == 4 ? kTileK4 : kTileK8)) {
    g_shift = 0;
    while (((int64_t)1 << g_shift) < f.G) ++g_shift;
  }
  if (shape == 4) shape = 5;  // (four row-blocks a wave in the caller's terms: 128 x 256)
  if (f.nf4 && (shape != 0 || splits > 1)) return set_error("woq_gemm_w4_kernel: NF4 weights take the automatic shape only");
  if (wbits == 8 && shape != 0 && shape != 5 && shape != 2 && shape != 42)
    return set_error("woq_gemm_w4_kernel: 8-bit weights take the 128 x 256, 128 x 128 and 64 x 128 shapes");
  if (shape != 0 && shape != 42 && splits > 1) return set_error("woq_gemm_w4_kernel: K is split for the 64 x 128 shape only");
  if (shape == 0) {
    const bool have = scratch && scratch->partial && scratch->counters && splits == 0;
    const TilePlan p = plan_tiles(f.M, f.N, (int)(f.KT / (wbits / 4)), step_times(wbits, f.nf4, f.fp8), have ? scratch->bytes : 0);
    shape = p.shape;
    splits = p.splits;
  }
  if (splits == 0) splits = 1;
  if (wbits == 8) return launch_gemm_w4_8bit(f, regime, g_shift, st, shape, splits, scratch);
  return regime == kRegimeF16 ? launch_gemm_w4_f16(f, g_shift, st, shape, splits, scratch)
                              : launch_w4_4bit<kRegimeBF16>(f, g_shift, st, shape, splits, scratch);
}

}  // namespace woq
