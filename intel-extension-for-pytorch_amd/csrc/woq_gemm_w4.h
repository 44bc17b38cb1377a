// MFMA GEMM for 4-bit weights and large M (prefill): y[M, N] = x[M, K] * dequant(W)[N, K]^T.
//
// Reference counterpart: DequantGemmTPP (dequantize a [Kb x 32] weight block to a stack
// buffer, then libxsmm BRGEMM) driven by qlinear_woq_affine_impl
// (csrc/cpu/aten/utils/woq.h:1847-1944, 3104-3477).  There the block is re-dequantized for
// every M block of 64 rows; here a wave dequantizes a weight tile once per 128 rows.
//
//   * v_mfma_f32_16x16x32 with A = activations and B = weights, as in the decode kernel: the
//     dequantized registers of one packed dword ARE the B operand, so weights never touch LDS
//     in dequantized form and every weight is dequantized by exactly one wave;
//   * a workgroup is four waves (128 x 256 tiles: eight, see below), one per SIMD with the whole 512-entry register file; wave w owns NTW
//     weight row-blocks (16 columns each) for all 16 * MT rows of the workgroup, i.e. MT x NTW
//     accumulator tiles.  The shape built is 128 x 448 (MT 8, NTW 7: 224 accumulator registers;
//     14336 / 448 = 32 and 2048 / 128 = 16 give 512 workgroups = two full generations on 256 CUs).
//     One wave hides about two VALU instructions behind each MFMA (measured: 16.4 cycles per MFMA
//     with 0..2 independent VALU instructions in between, +4 cycles for each further one); a
//     dequantized dword costs 17 and feeds MT = 8 MFMAs, so the loop is VALU-issue-bound;
//   * per K step of 128 (one packed tile per row-block) the activations of the rows go from global
//     memory straight into LDS (global_load_lds_dwordx4, no staging registers), double buffered;
//     16-byte chunk p of row m is stored at chunk p ^ (m % 16), which makes the A-fragment reads
//     (16 rows, one chunk) conflict-free without padding.  The packed tiles take the same route
//     into a per-wave LDS stage two steps ahead and are read into registers during the last K
//     sub-step of the step before;
//   * the step is software pipelined over its 4 K sub-steps and NTW row-blocks: while the MT MFMAs
//     of one (sub-step, row-block) run, the VALU dequantizes the dword of the next one;
//   * 8-bit weights (WBITS 8; per-channel or groups of at least 128) run through the same loop: a K
//     step of 128 is then two packed tiles per row-block (a tile is 16 rows x 64 bytes), sub-step j
//     takes dwords 2 (j % 2), 2 (j % 2) + 1 of tile j / 2 -- the K offsets 64 (j / 2) + 16 c + 8 (j % 2)
//     of lane column c -- and the A fragment is read from the matching 16-byte chunk; 20 VALU
//     instructions per B operand (byte -> float, fma, pack) against 17;
//   * MERGED instances (4-bit weights, bf16 compute, when the caller passes the table): the scale and the
//     zero point of a (row, group) come as one dword, bf16 scale << 16 | fp16 (1024 + zero), and the two
//     nibble positions are read as the fp16 numbers 1024 + q and 64 + q, so that one scale serves both:
//     7 instead of 14 parameter requests and 21 instead of 56 vector instructions per K step and wave
//     (M = 2048, 4096 -> 14336: 198 against 202-206 us on the same boxes; same bits out);
//   * 128 x 256 tiles have eight waves of two row-blocks each (WAVES 8), two on a SIMD: one wave alone issues a vector
//     instruction every 8.2 clocks, two together one every 4.6 (MFMA with three vector instructions behind it: 30 clocks
//     alone, 21.4 each with two waves), and 2.5 vector instructions stand beside each MFMA here.  The A fragments of the next
//     sub-step are then read in all blocks of a sub-step instead of one (SPREAD: with every wave in the same block the LDS
//     stood still in the others).  Against four waves of four row-blocks, us: INT4 M = 512, 4096 -> 14336 62 / 56, NF4
//     M = 1000 172 / 126, FP8 M = 2048 329 / 273, INT8 M = 2048, 4096 -> 11008 199 / 180.  What bounds them now is LDS
//     reads (256 KiB a K step).  Four waves a workgroup with SPREAD were slower (128 x 448 by 5 %, 128 x 128 by 6 %); eight
//     waves of 128 x 512 91 us a generation but 448 workgroups where 128 x 448 makes 512 (M = 2048, N = 14336: 206 / 204).
#pragma once

#include <type_traits>

#include "woq_common.h"
#include "woq_internal.h"

namespace woq {

template <int MT_, int NTW_, int WAVES_ = 4>
struct G4Shape {
  static constexpr int MT = MT_;                        // 16-row accumulator tiles
  static constexpr int NTW = NTW_;                      // weight row-blocks (16 columns) per wave
  static constexpr int WAVES = WAVES_;                  // waves per workgroup
  static constexpr bool SPLITS = MT * NTW <= 8 || WAVES == 8;  // K may be shared by several workgroups
  static constexpr int BM = 16 * MT;                    // rows per workgroup
  static constexpr int BN = WAVES * NTW * kTileN;       // columns per workgroup
  static constexpr int XBYTES = BM * kTileK4 * 2;       // one activation buffer
  static constexpr int XLOADS = XBYTES / (WAVES * 1024);     // LDS loads per wave and buffer
  static constexpr int WSTAGE = WAVES * NTW * kTileBytes;    // one weight stage of 4-bit tiles (8-bit: two)
  static constexpr int SSTRIDE = NTW * kTileN + 4;      // fp32 row stride of the epilogue staging tile
  // Sets of A fragments.  Row-block during whose MFMAs those of the next K sub-step are read from LDS (FETCH_T in g4_tile).  One
  // block ahead of their first use needs a second set of MT fragment registers; with 16 row tiles
  // a block is long enough (256 cycles) to read them in the last block, each into the registers of
  // the fragment whose last MFMA has just been issued.
  static constexpr int XA_SETS = MT >= 16 || (MT > 8 && WAVES == 8) ? 1 : 2;
};

template <class S, int WBITS>
constexpr int g4_lds_bytes() {
  return 2 * S::XBYTES + 2 * S::WSTAGE * (WBITS / 4);
}

template <int REGIME>
__device__ __forceinline__ f4 g4_mfma(u4 a, u4 b, f4 c) {
  if constexpr (REGIME == kRegimeF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(bitcast<h8>(a), bitcast<h8>(b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(bitcast<b8>(a), bitcast<b8>(b), c, 0, 0, 0);
}

// (eight waves have 256 registers each: accumulators that need not be AGPRs leave the allocator free to place them)
template <int WAVES>
__device__ __forceinline__ void g4_opaque(f4& v) {
  if constexpr (WAVES == 8)
    asm volatile("" : "+v"(v));
  else
    asm volatile("" : "+a"(v));
}

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef const __attribute__((address_space(1))) void* global_ptr_t;

// gridDim.z > 1 (M x N that leaves CUs or their wave slots idle, see plan_tiles): workgroup z
// of a tile takes the K steps [z * kts, (z + 1) * kts), writes its accumulators to scratch memory as they
// lie in the registers, and the workgroup that arrives last at the tile's counter adds the partial
// tiles in z order (its own from the registers) and runs the epilogue.  Nobody waits; the order of
// the sum is fixed.  All scratch accesses are relaxed device-scope atomics, as in the decode kernel.
// Constants of one (row, group) from its merged dword: w = (1024 + q) * s + c = (64 + q) * s + c64, both
// exact in fp32 (an 11-bit integer times an 8-bit significand), so the fma result is the exact product
// (q - z) * s and the one rounding is the conversion to bf16, as with separate scale and zero point.
struct G4ConstsM {
  float s, c, c64;
  __device__ __forceinline__ void set(uint32_t pd) {
    s = bitcast<float>(pd & 0xFFFF0000u);
    const _Float16 h = bitcast<_Float16>((uint16_t)(pd & 0xFFFFu));
    c = -((float)h * s);
    c64 = __builtin_fmaf(960.0f, s, c);
  }
};
__device__ __forceinline__ u4 g4_dequant_m(uint32_t d, const G4Masks& k, uint32_t magic64, const G4ConstsM& q) {
  u4 r;
  const f2 f0 = g4_fma_pair((d & k.lo) | k.magic, q.s, q.c);
  const f2 f1 = g4_fma_pair((d & k.hi) | magic64, q.s, q.c64);
  r[0] = g4_cvt_pair(f0);
  const uint32_t d8 = d >> 8;
  const f2 f2_ = g4_fma_pair((d8 & k.lo) | k.magic, q.s, q.c);
  r[1] = g4_cvt_pair(f1);
  const f2 f3 = g4_fma_pair((d8 & k.hi) | magic64, q.s, q.c64);
  r[2] = g4_cvt_pair(f2_);
  r[3] = g4_cvt_pair(f3);
  return r;
}

// GROUPED (mixture of experts): the row tile of a workgroup is a slot of the routing tables -- at most G4_BM routed rows of
// one expert, whose tensors come from the group's pointer tables; a slot without an expert ends at once.
// 32 experts 7168 -> 2048 -> 7168, top-8, 512 tokens: 3738 us with three launches per expert (each on 32 to 192 workgroups),
// 640..670 us with one launch per linear (three of about 200 us, 64-row tiles), 543 with 128 x 256 tiles, merged parameter tables and
// gate and up in one launch, 496 with up to 160 rows a slot.
// PAIR: half of a wave's row-blocks are the gate projection's, half the up projection's, of the same columns: a lane has both values
// and stores silu(gate) * up, rounded as two launches round it.
// Where an expert's own launch would split K over workgroups (plan_tiles), the workgroup runs the same K steps in as many
// chains, one after the other, and adds them in the same order: the expert has the bits of its own launch.
// NF4: a dword's eight table values come from the 256-entry table of value pairs in LDS (nf4_dequant), built before the first
// request; four 8-byte reads, eight products and four conversions against 17 instructions for integers.
constexpr int kPrefillSplitMax = 4;  // workgroups that share the K steps of a tile
constexpr int kChainRowTiles = (int)(kSplitKPrefillTiles > kSplitKPrefillMaxRows / 64 ? kSplitKPrefillTiles : kSplitKPrefillMaxRows / 64);
struct G4Group {
  const MoeGroup* tables;
  int chains[kChainRowTiles + 1];  // CHAINS: [rows / 64, rounded up] K steps of a chain, 0: one chain
};
template <int REGIME, class S, int WBITS, bool FP8, bool MERGED = false, bool GROUPED = false, bool NF4 = false, bool CHAINS = false, bool PAIR = false>
__device__ __forceinline__ void g4_tile(const FpArgs& fa, const int g_shift, float* const sk_partial, int* const sk_counters, const int kts,
                                        const G4Group& grp) {
  static_assert(!NF4 || (WBITS == 4 && !FP8 && !MERGED && !GROUPED), "NF4 codes have a table and a scale");
  __shared__ f2 sNf4[NF4 ? kNf4LutEntries : 1];
  if constexpr (NF4) nf4_fill_lut(sNf4, (int)threadIdx.x, 64 * S::WAVES);  // (the barrier before the first use is the K loop's first)
  static_assert(GROUPED || !CHAINS, "an ungrouped launch splits K over workgroups");
  static_assert(!PAIR || S::NTW % 2 == 0, "pairs: as many row-blocks of each weight");
  constexpr int TPS = WBITS / 4;  // packed tiles per row-block and K step of 128
  // (ten row tiles on eight waves: one set of fragments only where a chain's sum needs the other's registers)
  constexpr int XA_SETS = S::WAVES == 8 && !CHAINS ? 2 : S::XA_SETS;
  constexpr bool SPREAD = S::WAVES == 8 && XA_SETS == 2;
  constexpr int FETCH_T = XA_SETS == 1 ? S::NTW - 1 : S::NTW - 2;
  constexpr int G4_MT = S::MT, G4_NTW = S::NTW, G4_BM = S::BM, G4_XBYTES = S::XBYTES, G4_XLOADS = S::XLOADS,
                G4_WSTAGE = S::WSTAGE * TPS, G4_SSTRIDE = S::SSTRIDE, G4_WAVES = S::WAVES;
  // two activation buffers, then two weight stages of WAVES x NTW tiles x 1 KiB
  extern __shared__ __align__(1024) uint8_t sX[];
  // (the epilogue's stage of one row tile of all waves lies in front of the weight stages)
  constexpr int kStageBytes = G4_WAVES * 16 * G4_SSTRIDE * (int)sizeof(float);
  constexpr int kXArea = 2 * G4_XBYTES > kStageBytes ? 2 * G4_XBYTES : (kStageBytes + 1023) & ~1023;
  uint8_t* const sW = sX + kXArea;

  int bx, by;  // this workgroup's tile, by XCD (xcd_tile)
  xcd_tile(bx, by);
  FpArgs fg;                        // GROUPED: this slot's problem
  const int64_t* xrow = nullptr;    // GROUPED: routed row of the slot -> row of x, or null: x has the routed rows
  int chain = kts;                  // CHAINS: K steps of a chain
  if constexpr (GROUPED) {
    const MoeGroup& g = *grp.tables;
    const int e = __builtin_amdgcn_readfirstlane(dq_uniform(g.slot_expert)[by]);
    if (e < 0) return;
    const int64_t row0 = __builtin_amdgcn_readfirstlane(dq_uniform(g.slot_row0)[by]);
    const int packed = __builtin_amdgcn_readfirstlane(dq_uniform(g.slot_rows)[by]);
    const int rows = packed & 0xFFFF, expert_rows = packed >> 16;  // (0: not known, one chain)
    if constexpr (CHAINS)
      if (expert_rows <= 64 * kChainRowTiles) {
        const int steps = grp.chains[(expert_rows + 63) / 64];
        chain = steps ? steps : kts;
      }
    fg = fa;
    fg.M = rows < G4_BM ? rows : G4_BM;
    fg.qweight = dq_uniform((const uint8_t*)dq_uniform(g.qweight)[e]);
    fg.scales = dq_uniform((const uint16_t*)dq_uniform(g.scales)[e]);
    fg.zeros = g.zeros ? dq_uniform(dq_uniform(g.zeros)[e]) : nullptr;
    fg.bias = g.bias ? dq_uniform(dq_uniform(g.bias)[e]) : nullptr;
    if constexpr (MERGED) fg.szb = dq_uniform(dq_uniform(g.szb)[e]);
    if constexpr (PAIR) {
      fg.qweight_b = dq_uniform((const uint8_t*)dq_uniform(g.qweight_b)[e]);
      fg.scales_b = dq_uniform((const uint16_t*)dq_uniform(g.scales_b)[e]);
      fg.zeros_b = g.zeros_b ? dq_uniform(dq_uniform(g.zeros_b)[e]) : nullptr;
      fg.bias_b = g.bias_b ? dq_uniform(dq_uniform(g.bias_b)[e]) : nullptr;
      if constexpr (MERGED) fg.szb_b = dq_uniform(dq_uniform(g.szb_b)[e]);
    }
    fg.out = (uint8_t*)fa.out + row0 * fa.N * 2;  // (16-bit rows)
    if (fa.other0) fg.other0 = (const uint8_t*)fa.other0 + row0 * fa.N * 2;
    if (g.x_row)
      xrow = dq_uniform(g.x_row) + row0;
    else
      fg.x = (const uint8_t*)fa.x + row0 * fa.K * 2;
    by = 0;
  }
  const FpArgs& f = GROUPED ? fg : fa;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4;
  const int M = (int)f.M, K = (int)f.K, NT = (int)f.NT, KG = (int)f.KG;
  const int KTW = (int)f.KT;   // packed tiles along K of a row-block
  // K steps of 128 of this workgroup: [kt_lo, KT); kts is even, so the buffer parity of a step is
  // that of its number whatever the split
  const int kt_lo = (int)blockIdx.z * kts;
  const int KT = KTW / TPS < kt_lo + kts ? KTW / TPS : kt_lo + kts;
  const int m0 = by * G4_BM;
  constexpr int G4_NTO = PAIR ? G4_NTW / 2 : G4_NTW;  // row-blocks of the output
  const int nt0 = (bx * G4_WAVES + wave) * G4_NTO;    // first row-block of this wave

  G4Masks km;
  asm volatile("s_mov_b32 %0, 0x000F000F" : "=s"(km.lo));
  asm volatile("s_mov_b32 %0, 0x00F000F0" : "=s"(km.hi));
  asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(km.magic));
  uint32_t magic64;  // fp16 64 twice: a nibble in place at bits 4..7 reads as 64 + q
  asm volatile("v_mov_b32 %0, 0x54005400" : "=v"(magic64));

  f4 acc[G4_MT][G4_NTW];
#pragma unroll
  for (int mt = 0; mt < G4_MT; ++mt)
#pragma unroll
    for (int t = 0; t < G4_NTW; ++t) acc[mt][t] = f4{0.f, 0.f, 0.f, 0.f};

  // ---- activations: load i of wave w fills LDS KiB number w * XLOADS + i of a buffer: rows
  // 4 (w * XLOADS + i) + lane / 16, physical chunk lane % 16 = logical chunk ^ (row % 16).  Rows
  // past M re-read row M - 1; their results are never stored.
  uint32_t xoff[G4_XLOADS];
#pragma unroll
  for (int i = 0; i < G4_XLOADS; ++i) {
    const int rowl = (wave * G4_XLOADS + i) * 4 + c;
    int rowc = m0 + rowl < M ? rowl : M - 1 - m0;
    if constexpr (GROUPED) {
      if (xrow) rowc = (int)xrow[rowc];  // (the host bounds rows of x * K * 2 below 2^31)
    }
    // (4-bit weights: the chunk 4 c + j of lane column c and sub-step j is kept at slot 4 j + c, so that the four
    // lane columns of a row read slots that differ in their low bits: chunks 8 apart share their banks)
    const int slot = r ^ (rowl & 15);
    const int chunk = WBITS == 4 ? ((slot & 3) << 2) | (slot >> 2) : slot;
    xoff[i] = (uint32_t)(rowc * K + chunk * 8) * 2u;
  }
  // All global addresses are a wave-uniform 64-bit base plus a 32-bit per-lane byte offset that
  // carries the K step, which keeps the bases in scalar registers.
  const uint8_t* xbase = (const uint8_t*)f.x + (int64_t)m0 * K * 2;
  auto load_x = [&](int kt, int buf) {
    const uint32_t ko = (uint32_t)kt * (kTileK4 * 2);
#pragma unroll
    for (int i = 0; i < G4_XLOADS; ++i)
      __builtin_amdgcn_global_load_lds((global_ptr_t)(xbase + (uint32_t)(xoff[i] + ko)),
                                       (lds_ptr_t)(sX + buf * G4_XBYTES + (wave * G4_XLOADS + i) * 1024), 16, 0,
                                       0);
  };
  // A fragment of row tile mt, sub-step j: row 16 mt + r, logical chunk 4 c + j (8-bit weights:
  // 8 (j / 2) + 2 c + j % 2, the K offsets of the lane column's bytes in tile j / 2)
  uint32_t rd[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int slot = WBITS == 4 ? j * 4 + c : 8 * (j / 2) + 2 * c + (j % 2);
    rd[j] = (uint32_t)(r * 256 + ((slot ^ r) << 4));
  }

  // ---- weights of one K tile: one dwordx4 + one (scale, zero) per row-block and lane.  Symmetric
  // weights carry no zero points: scale bytes are read (and ignored) instead of branching. ----
  constexpr bool kZeros = !NF4 && !FP8;
  const bool has_z = kZeros && f.zeros != nullptr;
  const uint8_t* wbase[G4_NTW];
  const uint8_t* sbase[G4_NTW];
  const uint8_t* zbase[G4_NTW];
  const uint8_t* mbase[G4_NTW];
#pragma unroll
  for (int t = 0; t < G4_NTW; ++t) {
    const bool second = t >= G4_NTO;  // PAIR: the up projection's row-blocks after the gate's
    const int nto = nt0 + (second ? t - G4_NTO : t);
    const int nt = nto < NT ? nto : NT - 1;
    wbase[t] = (second ? f.qweight_b : f.qweight) + (size_t)nt * KTW * kTileBytes;
    sbase[t] = (const uint8_t*)((second ? f.scales_b : f.scales) + (size_t)nt * KG * kTileN);
    zbase[t] = has_z ? (second ? f.zeros_b : f.zeros) + (size_t)nt * KG * kTileN : sbase[t];
    mbase[t] = (const uint8_t*)(second ? f.szb_b : f.szb) + (size_t)nt * KG * (kTileN * 4);
  }
  const uint32_t woff = (uint32_t)lane * 16u;
  auto load_q = [&](int kt, uint16_t (&s)[G4_NTW], uint8_t (&z)[G4_NTW]) {
    int g = (kt * kTileK4 + c * 32) >> g_shift;
    g = g < KG ? g : KG - 1;
    const uint32_t qoff = (uint32_t)(g * kTileN + r);
#pragma unroll
    for (int t = 0; t < G4_NTW; ++t) {
      s[t] = *(const uint16_t*)(sbase[t] + (uint32_t)(qoff * 2u));
      z[t] = 0;
      if constexpr (kZeros) {
        const uint8_t zb = *(zbase[t] + qoff);
        z[t] = has_z ? zb : (uint8_t)(WBITS == 4 ? 8 : 128);  // symmetric: the stored code of zero
      }
    }
  };
  auto load_m = [&](int kt, uint32_t (&p)[G4_NTW]) {
    int g = (kt * kTileK4 + c * 32) >> g_shift;
    g = g < KG ? g : KG - 1;
    const uint32_t qoff = (uint32_t)(g * kTileN + r) * 4u;
#pragma unroll
    for (int t = 0; t < G4_NTW; ++t) p[t] = *(const uint32_t*)(mbase[t] + qoff);
  };
  // The packed tiles of a K step travel global -> LDS -> registers: the LDS stage costs no
  // registers while the load is in flight, which lets the tiles be requested two steps ahead.
  // Each wave fills and reads only its own NTW KiB of a stage.
  uint8_t* const wmine = sW + wave * (G4_NTW * TPS * kTileBytes);
  auto dma_w = [&](int kt, int stage) {
    const uint32_t wo = (uint32_t)kt * (TPS * kTileBytes) + woff;
#pragma unroll
    for (int t = 0; t < G4_NTW; ++t)
#pragma unroll
      for (int u = 0; u < TPS; ++u)
        __builtin_amdgcn_global_load_lds((global_ptr_t)(wbase[t] + (uint32_t)(wo + u * kTileBytes)),
                                         (lds_ptr_t)(wmine + stage * G4_WSTAGE + (t * TPS + u) * kTileBytes), 16, 0,
                                         0);
  };
  auto read_w = [&](int stage, int t, int u) {
    return *(const u4*)(wmine + stage * G4_WSTAGE + (t * TPS + u) * kTileBytes + woff);
  };

  u4 wr[G4_NTW][TPS];
  uint16_t sr[G4_NTW];
  uint8_t zr[G4_NTW];
  G4Consts<REGIME> qc[WBITS == 4 ? G4_NTW : 1];
  G4ConstsM qm[G4_NTW];
  uint32_t mr[G4_NTW];
  float q8s[WBITS == 8 || NF4 ? G4_NTW : 1], q8c[WBITS == 8 ? G4_NTW : 1];  // 8-bit: scale, -(128 + z) * scale
  auto set_q = [&](int t, uint16_t sbits, float z) {
    if constexpr (MERGED) {
      qm[t].set(mr[t]);
    } else if constexpr (NF4) {
      q8s[t] = REGIME == kRegimeF16 ? f16_bits_to_f32(sbits) : bf16_bits_to_f32(sbits);
    } else if constexpr (WBITS == 4) {
      qc[t].set(sbits, z);
    } else {
      q8s[t] = REGIME == kRegimeF16 ? f16_bits_to_f32(sbits) : bf16_bits_to_f32(sbits);
      q8c[t] = -(z * q8s[t]);
    }
  };
  // B operand of row-block t, K sub-step j
  auto deq = [&](int t, int j) -> u4 {
    if constexpr (MERGED) {
      return g4_dequant_m(wr[t][0][j], km, magic64, qm[t]);
    } else if constexpr (NF4) {
      return nf4_dequant<REGIME>(wr[t][0][j], sNf4, q8s[t]);
    } else if constexpr (WBITS == 4) {
      return g4_dequant(wr[t][0][j], km, qc[t]);
    } else {
      const uint32_t d0 = wr[t][j / 2][2 * (j % 2)], d1 = wr[t][j / 2][2 * (j % 2) + 1];
      if constexpr (FP8 && REGIME == kRegimeF16)  // float8 e4m3fn bytes
        return bitcast<u4>(dequant8_f16_fp8(d0, d1, q8s[t]));
      else if constexpr (FP8)
        return bitcast<u4>(dequant8_bf16_fp8(d0, d1, q8s[t]));
      else if constexpr (REGIME == kRegimeF16)
        return bitcast<u4>(dequant8_f16_w8(d0, d1, q8s[t], q8c[t]));
      else
        return bitcast<u4>(dequant8_bf16_w8(d0, d1, q8s[t], q8c[t]));
    }
  };
  u4 bop[2];        // B operand in use / being dequantized
  u4 xa[XA_SETS][G4_MT];  // A fragments of the sub-step in use (/ of the next one)

  // s_waitcnt immediates (vmcnt in bits 3:0 and 15:14; expcnt 6:4 and lgkmcnt 11:8 left at maximum)
  constexpr int kVmcnt0 = 0x0F70, kLgkmcnt0 = 0xC07F;
  constexpr int kVmcntW = 0x0F70 | (G4_NTW * TPS);  // all but the last loads (one weight stage) have landed
  // everything older than one whole step of loads (2 NTW parameter loads -- one dword or no zero points: NTW --,
  // XLOADS + NTW * TPS LDS loads)
  constexpr int kStepLoads = ((MERGED || !kZeros ? 1 : 2) + TPS) * G4_NTW + G4_XLOADS;
  static_assert(kStepLoads < 64 && G4_NTW * TPS < 16, "s_waitcnt vmcnt is a 6-bit field");
  constexpr int kVmcntStep = 0x0F70 | (kStepLoads & 15) | ((kStepLoads >> 4) << 14);

  // With one set of fragment registers (16 row tiles) a wave reads the 16 fragments of the next sub-step in one block,
  // and four waves that do so at the same moment queue at the LDS: a ds_read_b128 issued next to vector work costs
  // 10 clocks alone and about 40 when the three other waves issue theirs with it.  The waves therefore meet at the
  // barrier in different blocks of the last sub-step -- wave w in block FETCH_T - w, the same moment for all -- and so
  // reach the fetching block one block apart, in every sub-step (M = 2048, 4096 -> 6144: 92 us against 99 us).
  constexpr int STAG_MAX = XA_SETS == 1 && G4_WAVES == 4 ? (FETCH_T < 3 ? FETCH_T : 3) : 0;
  auto wait_met = [](bool reads_too) {
    if (reads_too)
      __builtin_amdgcn_s_waitcnt(kVmcntW & kLgkmcnt0);
    else
      __builtin_amdgcn_s_waitcnt(kVmcntW);
  };
  const int bar_t = FETCH_T - (wave < STAG_MAX ? wave : STAG_MAX);
  load_x(kt_lo, 0);
  dma_w(kt_lo, 0);
  dma_w(KT > kt_lo + 1 ? kt_lo + 1 : kt_lo, 1);
  if constexpr (MERGED) load_m(kt_lo, mr); else load_q(kt_lo, sr, zr);
  __builtin_amdgcn_s_waitcnt(kVmcnt0);
  __syncthreads();
#pragma unroll
  for (int t = 0; t < G4_NTW; ++t) {
#pragma unroll
    for (int u = 0; u < TPS; ++u) wr[t][u] = read_w(0, t, u);
    set_q(t, sr[t], (float)zr[t]);
  }
  bop[0] = deq(0, 0);
#pragma unroll
  for (int mt = 0; mt < G4_MT; ++mt) xa[0][mt] = *(const u4*)(sX + mt * 4096 + rd[0]);

  // The accumulator tiles pass through an opaque statement on both sides of the K loop: without it
  // the optimizer splits each loop-carried vector into four scalars (the epilogue reads single
  // elements), and the tiles are then copied between registers in every iteration.
#pragma unroll
  for (int mt = 0; mt < G4_MT; ++mt)
#pragma unroll
    for (int t = 0; t < G4_NTW; ++t) g4_opaque<G4_WAVES>(acc[mt][t]);

  // (the requests of a chain's last steps are the next chain's first ones; -0 + x is x for every x)
  f4 total[CHAINS ? G4_MT : 1][CHAINS ? G4_NTW : 1];
  if constexpr (CHAINS) {
#pragma unroll
    for (int mt = 0; mt < G4_MT; ++mt)
#pragma unroll
      for (int t = 0; t < G4_NTW; ++t) total[mt][t] = f4{-0.f, -0.f, -0.f, -0.f};
  }
  for (int kt = kt_lo; kt < KT;) {  // (CHAINS: chain after chain, else once)
    const int kt_end = CHAINS && kt + chain < KT ? kt + chain : KT;
    for (; kt < kt_end; ++kt) {
      const uint8_t* xs = sX + (kt & 1) * G4_XBYTES;
      const uint8_t* xsn = sX + ((kt & 1) ^ 1) * G4_XBYTES;
      // ---- requests, in this order (s_waitcnt vmcnt counts from the youngest): parameters and
      // activations of step kt + 1, then (behind the first MFMA block) the weight tiles of step
      // kt + 2 into the stage that held step kt.  Past the end the last step is requested again. ----
      const int kt1 = kt + 1 < KT ? kt + 1 : KT - 1;
      const int kt2 = kt + 2 < KT ? kt + 2 : KT - 1;
      if constexpr (MERGED) load_m(kt1, mr); else load_q(kt1, sr, zr);
      load_x(kt1, (kt & 1) ^ 1);
      __builtin_amdgcn_sched_barrier(0);

      // 4 NTW blocks of MT MFMAs (one row-block t of one K sub-step j against the MT row tiles); the VALU
      // dequantizes the B operand of the next block meanwhile.  Block FETCH_T of a sub-step also
      // fetches the A fragments of the next sub-step; in the last sub-step these come from the other
      // buffer, so that block starts with the wait for this step's activations and the barrier.  Block t of the last sub-step reads the
      // tile of row-block t for the next step from LDS; its registers were last used one block before.
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int t = 0; t < G4_NTW; ++t) {
          const int cur = (j * G4_NTW + t) & 1;
          const bool last_t = t == G4_NTW - 1;
          const bool fetch_t = SPREAD || t == FETCH_T;
          const bool bar_here = SPREAD ? t == 0 : t == FETCH_T;
          if (j == 0 && t == 1) {
            // the LDS reads of the previous step's last blocks have returned: their stage is free
            __builtin_amdgcn_s_waitcnt(kLgkmcnt0);
            dma_w(kt2, kt & 1);
            __builtin_amdgcn_sched_barrier(0);
          }
          if (j == 3 && t == 0) __builtin_amdgcn_s_waitcnt(kVmcntStep);  // tiles of step kt + 1 are in LDS
          // Behind the barrier the other waves refill the buffer of this step.  In the first block the barrier stands before
          // the first use of the last sub-step's fragments: their reads must have returned (before a later block they have).
          // (What this wait costs: at most 2 %, M = 1000, 7168 -> 4096 FP8 72.0 -> 73.6 us; the other prompts 0 to 1 %.)
          if constexpr (STAG_MAX == 0) {
            if (bar_here && j == 3) {
              // Written as an instruction, not as the barrier builtin: before that one the compiler
              // waits for every outstanding load, the tiles requested for step kt + 2 included.
              wait_met(t == 0 || XA_SETS == 1);
              asm volatile("s_barrier" ::: "memory");
            }
          } else {
            // this wave's meeting block (see bar_t)
            if (j == 3 && t <= FETCH_T && t >= FETCH_T - STAG_MAX && bar_t == t) {
              wait_met(t == 0);
              __builtin_amdgcn_s_barrier();
            }
          }
          if (last_t && j == 3) {
#pragma unroll
            for (int u = 0; u < G4_NTW; ++u) set_q(u, sr[u], (float)zr[u]);
            bop[cur ^ 1] = deq(0, 0);
          } else if (last_t) {
            bop[cur ^ 1] = deq(0, j + 1);
          } else {
            bop[cur ^ 1] = deq(t + 1, j);
          }
#pragma unroll
          for (int mt = 0; mt < G4_MT; ++mt) {
            acc[mt][t] = g4_mfma<REGIME>(bop[cur], xa[(j & 1) % XA_SETS][mt], acc[mt][t]);
            if (SPREAD ? mt * G4_NTW / G4_MT == t : fetch_t)
              xa[((j & 1) ^ 1) % XA_SETS][mt] = j == 3 ? *(const u4*)(xsn + mt * 4096 + rd[0])
                                           : *(const u4*)(xs + mt * 4096 + rd[j + 1]);
          }
          if (j == 3) {
#pragma unroll
            for (int u = 0; u < TPS; ++u) wr[t][u] = read_w((kt & 1) ^ 1, t, u);
          }
#pragma unroll
          for (int mt = 0; mt < (NF4 && G4_WAVES == 8 ? 0 : G4_MT); ++mt) {  // (NF4 with eight waves: 126 us without, 132 with)
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (SPREAD ? mt < (t + 1) * G4_MT / G4_NTW - t * G4_MT / G4_NTW : fetch_t) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if constexpr (CHAINS) {
#pragma unroll
      for (int mt = 0; mt < G4_MT; ++mt)
#pragma unroll
        for (int t = 0; t < G4_NTW; ++t) {
#pragma unroll
          for (int e = 0; e < 4; ++e) total[mt][t][e] += acc[mt][t][e];
          acc[mt][t] = f4{0.f, 0.f, 0.f, 0.f};
        }
    }
  }
  if constexpr (CHAINS) {
#pragma unroll
    for (int mt = 0; mt < G4_MT; ++mt)
#pragma unroll
      for (int t = 0; t < G4_NTW; ++t) acc[mt][t] = total[mt][t];
  }

  // The requests past the last step are still writing LDS: drain them before the workgroup can end.
  __builtin_amdgcn_s_waitcnt(kVmcnt0);
#pragma unroll
  for (int mt = 0; mt < G4_MT; ++mt)
#pragma unroll
    for (int t = 0; t < G4_NTW; ++t) g4_opaque<G4_WAVES>(acc[mt][t]);

  // (built for the shapes that are launched with gridDim.z > 1)
  if constexpr (S::SPLITS && !GROUPED) if (gridDim.z > 1) {
    const int nsplit = (int)gridDim.z, z = (int)blockIdx.z;
    const int tiles = (int)(gridDim.x * gridDim.y), tile = (int)(blockIdx.y * gridDim.x + blockIdx.x);
    constexpr int kWaveFloats = G4_MT * G4_NTW * 256;
    // accumulator pair h of tile (mt, t): 64 lanes x 8 bytes side by side (an access of its four registers one by one, 16 bytes
    // apart in memory, moved a quarter as much per instruction)
    auto part = [&](int zz) { return (uint64_t*)(sk_partial + ((size_t)(zz * tiles + tile) * G4_WAVES + wave) * kWaveFloats) + lane; };
    auto at = [](int mt, int t, int h) { return ((mt * G4_NTW + t) * 2 + h) * 64; };
    uint64_t* const mine = part(z);
#pragma unroll
    for (int mt = 0; mt < G4_MT; ++mt)
#pragma unroll
      for (int t = 0; t < G4_NTW; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          __hip_atomic_store(mine + at(mt, t, h), bitcast<uint64_t>(f2{acc[mt][t][2 * h], acc[mt][t][2 * h + 1]}), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(kVmcnt0);  // this thread's stores have completed
    __syncthreads();
    __shared__ int s_last;
    if (tid == 0)
      s_last = __hip_atomic_fetch_add(sk_counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nsplit - 1;
    __syncthreads();
    if (!s_last) return;
    // the other workgroups' partial tiles, two row tiles of all of them in flight together; added in z order, this workgroup's
    // own from its registers in its turn
    auto sum = [&](auto count) {
      constexpr int N = decltype(count)::value;
      const uint64_t* src[N - 1];
#pragma unroll
      for (int k = 0; k < N - 1; ++k) src[k] = part(k + (k >= z ? 1 : 0));
#pragma unroll
      for (int mc = 0; mc < G4_MT; mc += 2) {
        uint64_t v[N - 1][2][G4_NTW][2];
#pragma unroll
        for (int k = 0; k < N - 1; ++k)
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int t = 0; t < G4_NTW; ++t)
#pragma unroll
              for (int h = 0; h < 2; ++h)
                v[k][i][t][h] = __hip_atomic_load(src[k] + at(mc + i, t, h), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int t = 0; t < G4_NTW; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const f2 own = {acc[mc + i][t][2 * h], acc[mc + i][t][2 * h + 1]};
              auto value = [&](int zz) {  // partial tile zz
                const f2 below = bitcast<f2>(v[zz < N - 1 ? zz : N - 2][i][t][h]), above = bitcast<f2>(v[zz > 0 ? zz - 1 : 0][i][t][h]);
                return zz < z ? below : zz > z ? above : own;
              };
              f2 total = value(0);
#pragma unroll
              for (int zz = 1; zz < N; ++zz) {
                const f2 p = value(zz);
                total[0] = total[0] + p[0];
                total[1] = total[1] + p[1];
              }
              acc[mc + i][t][2 * h] = total[0];
              acc[mc + i][t][2 * h + 1] = total[1];
            }
        __builtin_amdgcn_sched_barrier(0);  // (the next row tiles' loads stay behind: their registers are these)
      }
    };
    if (nsplit == 2)
      sum(std::integral_constant<int, 2>{});
    else if (nsplit == 3)
      sum(std::integral_constant<int, 3>{});
    else
      sum(std::integral_constant<int, 4>{});
    // the counter is back at zero for the next launch that uses it
    if (tid == 0) __hip_atomic_store(sk_counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  // ---- epilogue.  The weights are the first MFMA operand and the activations the second, so the
  // accumulator tile is D[n][m]: lane (r, c) holds row m = 16 mt + r and the four consecutive columns
  // n = 16 t + 4 c + e.  In the plain case (no post-op, output in the activation dtype) a lane rounds
  // its four values and stores them as 8 bytes straight from the registers: the four lane columns of a
  // row write 32 contiguous bytes, the NTW row-blocks of a wave follow each other in the row, and
  // nothing waits on LDS.  Post-ops go through a per-wave LDS tile (the activation buffers are idle
  // after the last barrier) so that the element-wise tail sees consecutive columns in consecutive lanes. ----
  const int64_t ncol0 = (int64_t)nt0 * kTileN;
  // (the output may be the other 16-bit type than the activations: fp16 rows converted from a bf16 tensor)
  const bool out_f16 = f.out_dtype == WOQ_HIP_ACT_FP16;
  const bool fast = f.fusion == WOQ_HIP_FUSE_NONE && (out_f16 || f.out_dtype == WOQ_HIP_ACT_BF16) && (f.N % 4) == 0 &&
                    (((uintptr_t)f.out & 7) | ((uintptr_t)f.bias & 15)) == 0;
  const bool hb = f.bias != nullptr;
  if constexpr (PAIR) {
    // a lane has the gate's and the up projection's values of the same four columns
    const bool hb2 = f.bias_b != nullptr, wide = (f.N % 4) == 0 && ((uintptr_t)f.out & 7) == 0;
#pragma unroll
    for (int t = 0; t < G4_NTO; ++t) {
      const int64_t n = ncol0 + t * kTileN + 4 * c;
      f4 b0 = f4{0.f, 0.f, 0.f, 0.f}, b1 = b0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (hb && n + e < f.N) b0[e] = f.bias[n + e];
        if (hb2 && n + e < f.N) b1[e] = f.bias_b[n + e];
      }
#pragma unroll
      for (int mt = 0; mt < G4_MT; ++mt) {
        const int m = m0 + mt * 16 + r;
        if (m >= M || n >= f.N) continue;
        uint16_t bits[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float y = pair_value<REGIME>(acc[mt][t][e], hb, b0[e], acc[mt][t + G4_NTO][e], hb2, b1[e], f.x_dtype);
          bits[e] = out_f16 ? f32_to_f16_bits(y) : f32_to_bf16_bits(y);
        }
        uint16_t* const at = (uint16_t*)f.out + (int64_t)m * f.N + n;
        if (wide) {
          *(u2*)at = u2{(uint32_t)bits[0] | ((uint32_t)bits[1] << 16), (uint32_t)bits[2] | ((uint32_t)bits[3] << 16)};
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < f.N) at[e] = bits[e];
        }
      }
    }
    return;
  }
  if (fast) {
    f4 bias4[G4_NTW];
#pragma unroll
    for (int t = 0; t < G4_NTW; ++t)
      bias4[t] = hb && ncol0 + t * kTileN + 4 * c < f.N ? *(const f4*)(f.bias + ncol0 + t * kTileN + 4 * c)
                                                        : f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mt = 0; mt < G4_MT; ++mt) {
      const int m = m0 + mt * 16 + r;
      if (m < M) {
        uint16_t* const row = (uint16_t*)f.out + (int64_t)m * f.N + ncol0 + 4 * c;
#pragma unroll
        for (int t = 0; t < G4_NTW; ++t) {
          const float y0 = finalize_acc<REGIME>(acc[mt][t][0], hb, bias4[t][0]);
          const float y1 = finalize_acc<REGIME>(acc[mt][t][1], hb, bias4[t][1]);
          const float y2 = finalize_acc<REGIME>(acc[mt][t][2], hb, bias4[t][2]);
          const float y3 = finalize_acc<REGIME>(acc[mt][t][3], hb, bias4[t][3]);
          u2 o;
          if (out_f16) {
            o[0] = (uint32_t)f32_to_f16_bits(y0) | ((uint32_t)f32_to_f16_bits(y1) << 16);
            o[1] = (uint32_t)f32_to_f16_bits(y2) | ((uint32_t)f32_to_f16_bits(y3) << 16);
          } else {
            o[0] = bitcast<uint32_t>(__builtin_convertvector(f2{y0, y1}, b2));
            o[1] = bitcast<uint32_t>(__builtin_convertvector(f2{y2, y3}, b2));
          }
          if (ncol0 + t * kTileN + 4 * c < f.N) *(u2*)(row + t * kTileN) = o;  // (N % 4 == 0: all four or none)
        }
      }
    }
    return;
  }
  // Post-ops in the activation type on rows of whole 8-byte pieces: ECH row tiles at a time through the wave's stage (inside
  // the activation buffers: the weight stages can still be written by the other waves' last requests), four columns a lane,
  // the operands of the next pair of pieces requested before the current pair is worked on.  One element a lane and
  // iteration, each waiting for its operand, took 20 us of a 88 us launch (M = 333, 11008 -> 4096 with a residual).
  constexpr int ECH = G4_MT % 8 == 0 && 8 * kStageBytes <= 2 * G4_XBYTES   ? 8
                      : G4_MT % 4 == 0 && 4 * kStageBytes <= 2 * G4_XBYTES ? 4
                      : 2 * kStageBytes <= 2 * G4_XBYTES                   ? 2
                                                                           : 1;
  const bool vec4 = f.fusion != WOQ_HIP_FUSE_NONE && f.out_dtype == f.x_dtype && (f.N % 4) == 0 &&
                    (((uintptr_t)f.out | (uintptr_t)f.other0 | (uintptr_t)f.other1) & 7) == 0 && ((uintptr_t)f.bias & 15) == 0;
  // (not for 128 x 448 tiles, whose K loop has no register to spare)
  if constexpr (G4_MT * G4_NTW <= 48) if (vec4) {
    float* const st4 = (float*)sX + wave * (ECH * 16 * G4_SSTRIDE);
    constexpr int ITS = ECH * G4_NTW;  // pieces of 64 lanes x 4 columns
#pragma unroll
    for (int mc = 0; mc < G4_MT; mc += ECH) {
#pragma unroll
      for (int i = 0; i < ECH; ++i)
#pragma unroll
        for (int t = 0; t < G4_NTW; ++t) *(f4*)(st4 + (16 * i + r) * G4_SSTRIDE + t * kTileN + 4 * c) = acc[mc + i][t];
      struct Piece {
        u2 a, b;
        int64_t at;  // element of the output, or -1
        int stage;
        f4 bias;
      };
      auto request = [&](int it) {
        Piece p;
        const int q = it * 64 + lane, row = q / (G4_NTW * 4), col = (q - row * (G4_NTW * 4)) * 4;
        const int m = m0 + mc * 16 + row;
        const int64_t n = ncol0 + col;
        p.stage = row * G4_SSTRIDE + col;
        p.at = it < ITS && m < M && n < f.N ? (int64_t)m * f.N + n : -1;
        p.a = p.b = u2{0u, 0u};
        p.bias = f4{0.f, 0.f, 0.f, 0.f};
        if (p.at >= 0) {
          if (f.other0) p.a = *(const u2*)((const uint16_t*)f.other0 + p.at);
          if (f.other1) p.b = *(const u2*)((const uint16_t*)f.other1 + p.at);
          if (hb) p.bias = *(const f4*)(f.bias + n);
        }
        return p;
      };
      auto finish = [&](const Piece& p) {
        if (p.at < 0) return;
        const f4 v = *(const f4*)(st4 + p.stage);
        u2 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float y = post_op(round_to_act(finalize_acc<REGIME>(v[e], hb, p.bias[e]), f.x_dtype), f.fusion, f.x_dtype,
                                  act_bits_to_f32((uint16_t)(p.a[e / 2] >> (16 * (e % 2))), f.x_dtype),
                                  act_bits_to_f32((uint16_t)(p.b[e / 2] >> (16 * (e % 2))), f.x_dtype));
          const uint32_t bits = out_f16 ? f32_to_f16_bits(y) : f32_to_bf16_bits(y);
          o[e / 2] = e % 2 ? o[e / 2] | (bits << 16) : bits;
        }
        *(u2*)((uint16_t*)f.out + p.at) = o;
      };
      Piece p0 = request(0), p1 = request(1);
#pragma unroll 1
      for (int it = 0; it < ITS; it += 2) {
        const Piece n0 = request(it + 2), n1 = request(it + 3);
        finish(p0);
        finish(p1);
        p0 = n0;
        p1 = n1;
      }
    }
    return;
  }
  float* stage = (float*)sX + wave * (16 * G4_SSTRIDE);
  Epilogue ep{f.bias, f.fusion, f.other0, f.other1, f.out, f.out_dtype, f.x_dtype, f.N};
#pragma unroll
  for (int mt = 0; mt < G4_MT; ++mt) {
#pragma unroll
    for (int t = 0; t < G4_NTW; ++t) *(f4*)(stage + r * G4_SSTRIDE + t * kTileN + 4 * c) = acc[mt][t];
#pragma unroll 1
    for (int it = 0; it < 16 * G4_NTW * kTileN / 64; ++it) {
      const int idx = it * 64 + lane;
      const int row = idx / (G4_NTW * kTileN), col = idx - row * (G4_NTW * kTileN);
      const int m = m0 + mt * 16 + row;
      const int64_t n = ncol0 + col;
      if (m < M && n < f.N) epilogue_store<REGIME>(ep, m, n, stage[row * G4_SSTRIDE + col]);
    }
  }
}

// GROUPED with 128-row slots: a slot of few rows runs the same columns with 32 or 64 rows' MFMAs and activations (every weight is
// dequantized as before; same bits).  Of 512 tokens on 32 experts, top-8, half of the experts have a second slot of about ten rows:
// gate + up 7168 -> 2048 350 -> 320 us, down 212 -> 175.
// With slots of up to 160 rows such an expert has one slot of ten row tiles in place of two, whose second still cost 0.7 of the first:
// 512 workgroups in two generations for 800 in more than three, gate + up 320 -> 286, down 175 -> 157.  Ten row tiles need the registers
// of the second set of fragments where K runs in chains (a chain's sum is kept beside the accumulators; some of it still goes to
// memory at a chain's end: 262 us without chains); with both sets and more of the sum in memory 316.
template <int REGIME, class S, int WBITS, bool FP8, bool MERGED = false, bool GROUPED = false, bool NF4 = false, bool CHAINS = false, bool PAIR = false>
__global__ __launch_bounds__(64 * S::WAVES) void woq_gemm_w4_kernel(const FpArgs fa, const int g_shift, float* const sk_partial,
                                                          int* const sk_counters, const int kts, const G4Group grp) {
  if constexpr (GROUPED && S::MT >= 8) {
    int bx, by;
    xcd_tile(bx, by);
    const int rows = __builtin_amdgcn_readfirstlane(dq_uniform(dq_uniform(grp.tables)->slot_rows)[by]) & 0xFFFF;
#define WOQ_SLOT(MT) return g4_tile<REGIME, G4Shape<MT, S::NTW, S::WAVES>, WBITS, FP8, MERGED, GROUPED, NF4, CHAINS, PAIR>(fa, g_shift, sk_partial, sk_counters, kts, grp)
    if (rows <= 32) WOQ_SLOT(2);
    if (rows <= 64) WOQ_SLOT(4);
    if constexpr (S::MT > 8) {
      if (rows <= 96) WOQ_SLOT(6);
      if (rows <= 128) WOQ_SLOT(8);
    }
#undef WOQ_SLOT
  }
  g4_tile<REGIME, S, WBITS, FP8, MERGED, GROUPED, NF4, CHAINS, PAIR>(fa, g_shift, sk_partial, sk_counters, kts, grp);
}

// Even, so that every split starts on buffer 0.
inline int split_k_steps(int ksteps, int splits) { return ((ksteps + splits - 1) / splits + 1) & ~1; }

template <int REGIME, class S, int WBITS = 4, bool FP8 = false, bool NF4 = false, bool PAIR = false>
int launch_shape(const FpArgs& f, int g_shift, hipStream_t st, int splits = 1,
                        const SplitKScratch* scratch = nullptr) {
  constexpr int kLds = g4_lds_bytes<S, WBITS>();
  static_assert(kLds <= 160 * 1024, "a workgroup's LDS");
  constexpr int kColumns = PAIR ? S::BN / 2 : S::BN;
  dim3 grid((unsigned)((f.NT * kTileN + kColumns - 1) / kColumns), (unsigned)((f.M + S::BM - 1) / S::BM),
            (unsigned)splits);
  const int ksteps = (int)(f.KT / (WBITS / 4));
  int kts = ksteps;
  if (splits > 1) {
    if (!S::SPLITS) return set_error("woq_gemm_w4_kernel: K is split for the 64 x 128 and 128 x 256 shapes only");
    kts = split_k_steps(ksteps, splits);
    const int64_t tiles = (int64_t)grid.x * grid.y;
    const int64_t need = (int64_t)splits * tiles * S::BM * S::BN * (int64_t)sizeof(float);
    if ((int64_t)(splits - 1) * kts >= ksteps)
      return set_error("woq_gemm_w4_kernel: %d K steps are too few for %d splits", ksteps, splits);
    if (!scratch || !scratch->partial || !scratch->counters || scratch->bytes < need || tiles > kSplitKCounters)
      return set_error("woq_gemm_w4_kernel: split K needs %lld bytes of workspace, the counter array and at most %d "
                       "tiles", (long long)need, kSplitKCounters);
  }
  if constexpr (REGIME == kRegimeBF16 && WBITS == 4 && !NF4) {
    if (f.szb) {  // scale and zero point of a (row, group) in one dword
      static const hipError_t lds_optin_m =
          hipFuncSetAttribute(reinterpret_cast<const void*>(&woq_gemm_w4_kernel<REGIME, S, WBITS, FP8, true, false, false, false, PAIR>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
      if (lds_optin_m != hipSuccess)
        return set_error("woq_gemm_w4_kernel: LDS opt-in failed: %s", hipGetErrorString(lds_optin_m));
      woq_gemm_w4_kernel<REGIME, S, WBITS, FP8, true, false, false, false, PAIR><<<grid, 64 * S::WAVES, kLds, st>>>(
          f, g_shift, splits > 1 ? scratch->partial : nullptr, splits > 1 ? scratch->counters : nullptr, kts, G4Group{});
      return check_launch("woq_gemm_w4_kernel");
    }
  }
  if constexpr (PAIR) {
    return set_error("woq_gemm_w4_kernel: a pair needs the merged parameter tables");
  } else {
    // more than 64 KiB of LDS per workgroup needs an opt-in (once per kernel and process)
    static const hipError_t lds_optin =
        hipFuncSetAttribute(reinterpret_cast<const void*>(&woq_gemm_w4_kernel<REGIME, S, WBITS, FP8, false, false, NF4>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (lds_optin != hipSuccess)
      return set_error("woq_gemm_w4_kernel: LDS opt-in failed: %s", hipGetErrorString(lds_optin));
    woq_gemm_w4_kernel<REGIME, S, WBITS, FP8, false, false, NF4><<<grid, 64 * S::WAVES, kLds, st>>>(
        f, g_shift, splits > 1 ? scratch->partial : nullptr, splits > 1 ? scratch->counters : nullptr, kts, G4Group{});
    return check_launch("woq_gemm_w4_kernel");
  }
}

// 4-bit weights in one of the shapes (launch_gemm_w4's argument).
// 256 rows x 192 columns (MT 16, NTW 3: 192 accumulator registers) dequantizes half as much per MFMA but measured no faster
// per output (95-120 us at K = 4096 against 103 for the 17 % larger 128 x 448 one): it is offered only where it tiles the
// problem into whole generations of 256 workgroups.  256 x 256 would need all 256 accumulator registers; the register
// allocator then copies accumulators through VGPRs and scratch, it measured slower and is not built.
template <int REGIME>
int launch_w4_4bit(const FpArgs& f, int g_shift, hipStream_t st, int shape, int splits, const SplitKScratch* scratch) {
  using S8 = G4Shape<8, 2, 8>;
  using S42 = G4Shape<4, 2>;
  if (f.nf4)
    return shape == 5 ? launch_shape<REGIME, S8, 4, false, true>(f, g_shift, st, splits, scratch)
                      : launch_shape<REGIME, S42, 4, false, true>(f, g_shift, st, splits, scratch);
  switch (shape) {
    case 42: return launch_shape<REGIME, S42>(f, g_shift, st, splits, scratch);
    case 5: return launch_shape<REGIME, S8>(f, g_shift, st, splits, scratch);
    case 163: return launch_shape<REGIME, G4Shape<16, 3>>(f, g_shift, st, splits, scratch);
    case 7: return launch_shape<REGIME, G4Shape<8, 7>>(f, g_shift, st, splits, scratch);
    default: return launch_shape<REGIME, G4Shape<8, 2>>(f, g_shift, st, splits, scratch);
  }
}

// in files of their own
int launch_gemm_w4_f16(const FpArgs& f, int g_shift, hipStream_t st, int shape, int splits, const SplitKScratch* scratch);
int launch_gemm_w4_8bit(const FpArgs& f, int regime, int g_shift, hipStream_t st, int shape, int splits, const SplitKScratch* scratch);
int gemm_w4_chain_steps(const FpArgs& f, int wbits, int row_tiles);  // K steps of a chain of an expert of that many row tiles of 64, 0: one chain

}  // namespace woq
