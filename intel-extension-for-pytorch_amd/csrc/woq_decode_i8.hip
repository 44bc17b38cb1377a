// lowp_mode INT8, up to four rows: the activations are quantized by the workgroups that multiply them.
//
// Reference counterpart: dynamic_quantize_per_block followed by the int8 GEMM
// (csrc/cpu/aten/utils/woq_dynamic_quant.h:1526-1750, csrc/cpu/aten/utils/woq.h:2172-2186).
//
// What bounds a decode step here is latency: the quantization of a row is a launch of 3 us (one read, one reduction, one write)
// before a launch of 5 us that streams the weight.  A row is a few KiB and comes from the L2, so every workgroup quantizes the
// rows for itself, into LDS, while its first weight tiles are on their way: the requests go out rows first, then the tiles of
// the wave's first rounds (kDepth: four, or two where a round has many registers), and only then does anything wait.
//   * split as in woq_decode_w4i8_kernel: a workgroup owns NTW weight row-blocks and all of K, wave w takes the K tiles w, w + W,
//     ...; the waves' fp32 sums are added in wave order.  Same bits as the two launches: the quantization is the same expressions
//     and every sum has the same order.
//   * rows are dealt to the waves in pieces of 512 elements (8 a lane), at most NP = 1 or 4 a wave: M x K up to 16384 with eight waves.
//   * LDS holds the quantized rows 16 bytes apart from whole multiples of 128 (the rows of an A fragment would share banks), and
//     their scales.
#include <type_traits>

#include "woq_common.h"
#include "woq_internal.h"
#include "woq_int8_common.h"

// the roundings of the epilogue (activation scale, bias) stay separate, as in the two launches' kernel (woq_gemm_w4i8.hip)
#pragma clang fp contract(off)

namespace woq {

struct DecodeI8Args {
  const uint16_t* x;
  int bf16;
  int M, K, NT, KT, KG, W;
  int pieces_per_row;
  int64_t N;
  const uint8_t* qweight;
  const float* scales;
  const uint8_t* zeros;
  int g_shift;           // round kt belongs to group kt >> g_shift
  int q_shift;           // PER_K, groups of at least 128: round kt belongs to activation block kt >> q_shift
  int block_lanes_log2;  // PER_K: lanes of an activation block
  int scale_cols;        // activation scales of a row
  int x_base;            // byte of LDS where the quantized rows (and the reduction) start
  Epilogue ep;
};

// Largest of 64 lanes' values, in every lane: row-wise by DPP, then over the four rows of sixteen lanes.
__device__ __forceinline__ float wave_max(float v) {
  auto step = [&](auto ctrl) {
    const int o = __builtin_amdgcn_update_dpp(0, bitcast<int>(v), decltype(ctrl)::value, 0xF, 0xF, true);
    v = fmaxf(v, bitcast<float>(o));
  };
  step(std::integral_constant<int, 0x128>{});  // row_ror 8, 4, 2, 1
  step(std::integral_constant<int, 0x124>{});
  step(std::integral_constant<int, 0x122>{});
  step(std::integral_constant<int, 0x121>{});
  const int b = bitcast<int>(v);
  return fmaxf(fmaxf(bitcast<float>(__builtin_amdgcn_readlane(b, 0)), bitcast<float>(__builtin_amdgcn_readlane(b, 16))),
               fmaxf(bitcast<float>(__builtin_amdgcn_readlane(b, 32)), bitcast<float>(__builtin_amdgcn_readlane(b, 48))));
}

// aq_quant(v, {s, 0}, symmetric) with the quotient from the reciprocal y = 1 / s, rounded to nearest: two steps of
// q + (v - q s) y make q the nearest float to v / s wherever it is not denormal (Markstein), and rint takes those to zero either
// way.  s between 2^-100 and 2^100: five instructions an element instead of a division's eleven and its mode switches.
__device__ __forceinline__ uint32_t quant_by_reciprocal(float v, float s, float y) {
  float q = v * y;
  q = __builtin_fmaf(__builtin_fmaf(-q, s, v), y, q);
  q = __builtin_fmaf(__builtin_fmaf(-q, s, v), y, q);
  float t = rintf(q);
  t = fminf(fmaxf(t, -128.0f), 127.0f);
  return (uint32_t)(uint8_t)(int8_t)(int)t;  // (a NaN clamps to -128, as there)
}

// GSUB, WBITS as in woq_decode_w4i8_kernel; NP: pieces of 512 row elements a wave quantizes.
template <bool PER_K, int NTW, int GSUB, int WBITS, int NP>
__global__ __launch_bounds__(512, 4) void woq_decode_i8_rows_kernel(const DecodeI8Args a) {
  static_assert(WBITS == 4 || GSUB == 1, "8-bit weights: one K block per round");
  constexpr int TPR = WBITS / 4;
  constexpr int kDepth = NTW * TPR * GSUB >= 4 ? 2 : 4;  // rounds of weight tiles in flight
  extern __shared__ __align__(1024) uint8_t smem[];
  float* const sscale = (float*)smem;         // [M][scale_cols]
  uint8_t* const sq = smem + a.x_base;        // [M][K + 16] quantized rows
  f4* const red = (f4*)sq;                    // [NTW][W][64], after the K loop
  __shared__ float spiece[32];                // largest absolute value of a piece
  const int W = a.W, M = a.M, K = a.K, KT = a.KT, KG = a.KG;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int r = lane & 15, c = lane >> 4;
  const int64_t nt0 = (int64_t)blockIdx.x * NTW;
  const int qstride = K + 16;

  // ---- requests: this wave's pieces of the rows, then the tiles of its first rounds ----
  const int pieces = M * a.pieces_per_row;
  u4 raw[NP];
  int prow[NP], pk[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int id = wave + W * i;
    prow[i] = id / a.pieces_per_row;
    pk[i] = (id - prow[i] * a.pieces_per_row) * 512 + lane * 8;
    raw[i] = u4{0u, 0u, 0u, 0u};
    if (id < pieces && pk[i] < K) raw[i] = *(const u4*)(a.x + (size_t)prow[i] * K + pk[i]);  // (K % 128 == 0: all eight or none)
  }
  __builtin_amdgcn_sched_barrier(0);

  const bool has_z = a.zeros != nullptr;
  const uint8_t* wbase[NTW];
  const float* sbase[NTW];
  const uint8_t* zbase[NTW];
#pragma unroll
  for (int t = 0; t < NTW; ++t) {
    wbase[t] = a.qweight + (size_t)(nt0 + t) * KT * TPR * kTileBytes;
    sbase[t] = a.scales + (size_t)(nt0 + t) * KG * kTileN;
    zbase[t] = has_z ? a.zeros + (size_t)(nt0 + t) * KG * kTileN : (const uint8_t*)sbase[t];
  }
  const int my_block = c / (4 / GSUB);
  struct Round {
    u4 w[NTW][TPR];
    float s[NTW][GSUB];
    uint8_t z[NTW];
  };
  Round ring[kDepth];
  // (past the end the last round is requested again: no branch around a load in flight)
  auto request = [&](int kt, Round& q) {
    kt = kt < KT ? kt : KT - 1;
    int g0 = GSUB == 1 ? (kt >> a.g_shift) : kt * GSUB;
    g0 = g0 < KG ? g0 : KG - 1;
    const uint32_t wo = (uint32_t)kt * (TPR * kTileBytes) + (uint32_t)lane * 16u;
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
#pragma unroll
      for (int u = 0; u < TPR; ++u) q.w[t][u] = __builtin_nontemporal_load((const u4*)(wbase[t] + (uint32_t)(wo + u * kTileBytes)));
#pragma unroll
      for (int g = 0; g < GSUB; ++g) q.s[t][g] = sbase[t][(uint32_t)((g0 + g) * kTileN + r)];
      q.z[t] = *(zbase[t] + (uint32_t)((g0 + (GSUB == 1 ? 0 : my_block)) * kTileN + r));
    }
  };
#pragma unroll
  for (int i = 0; i < kDepth; ++i) request(wave + W * i, ring[i]);
  __builtin_amdgcn_sched_barrier(0);

  // ---- quantize.  A group of NaNs has an infinite scale, as the extremes of nothing give it in act_quant_rows_kernel. ----
  float amax[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    amax[i] = -1.0f;
    const int id = wave + W * i;
    if (id >= pieces) continue;
    if (pk[i] < K) {
      float v[8];
      aq_unpack(raw[i], a.bf16 != 0, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) amax[i] = fmaxf(amax[i], fabsf(v[e]));
    }
    if constexpr (PER_K) {
      for (int s = 0; s < a.block_lanes_log2; ++s) amax[i] = fmaxf(amax[i], __shfl_xor(amax[i], 1 << s));
    } else {
      amax[i] = wave_max(amax[i]);
      if (lane == 0) spiece[id] = amax[i];
    }
  }
  // (the barriers are written as instructions: the weight requests stay in flight across them)
  if constexpr (!PER_K) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if (wave + W * i >= pieces) continue;
      amax[i] = wave_max(lane < a.pieces_per_row ? spiece[prow[i] * a.pieces_per_row + lane] : -1.0f);  // (at most 32 pieces)
    }
  }
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    if (wave + W * i >= pieces || pk[i] >= K) continue;
    const float top = amax[i] < 0.0f ? __builtin_inff() : amax[i];
    const AqParams p = aq_params(-top, top, true, nullptr);
    if constexpr (PER_K) {
      if ((lane & ((1 << a.block_lanes_log2) - 1)) == 0) sscale[prow[i] * a.scale_cols + (pk[i] >> (a.block_lanes_log2 + 3))] = p.s;
    } else {
      if (pk[i] == 0) sscale[prow[i]] = p.s;
    }
    float v[8];
    aq_unpack(raw[i], a.bf16 != 0, v);
    uint32_t o[8];
    if (p.s > 0x1p-100f && p.s < 0x1p+100f) {
      const float y = __fdiv_rn(1.0f, p.s);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = quant_by_reciprocal(v[e], p.s, y);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = aq_quant(v[e], p, true, false);
    }
    u2 out;
    if constexpr (WBITS == 4) {  // the order in which the nibbles of a dword come out
      out[0] = o[0] | (o[4] << 8) | (o[1] << 16) | (o[5] << 24);
      out[1] = o[2] | (o[6] << 8) | (o[3] << 16) | (o[7] << 24);
    } else {
      out[0] = o[0] | (o[1] << 8) | (o[2] << 16) | (o[3] << 24);
      out[1] = o[4] | (o[5] << 8) | (o[6] << 16) | (o[7] << 24);
    }
    *(u2*)(sq + prow[i] * qstride + pk[i]) = out;
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // ---- K loop ----
  f4 acc[NTW];
#pragma unroll
  for (int t = 0; t < NTW; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
  const uint8_t* const xrow = sq + (r < M ? r : M - 1) * qstride;  // (rows past M repeat the last one; never stored)
  int srow[4];  // first scale of the rows of this lane's accumulators
#pragma unroll
  for (int e = 0; e < 4; ++e) srow[e] = (4 * c + e < M ? 4 * c + e : M - 1) * a.scale_cols;
  auto multiply = [&](int kt, const Round& q) {
    i4 xa[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) xa[j] = *(const i4*)(xrow + kt * 128 + (WBITS == 4 ? 2 * c + j : 4 * j + c) * 16);
    f4 sa[PER_K ? GSUB : 1];
    if constexpr (PER_K) {
#pragma unroll
      for (int g = 0; g < GSUB; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) sa[g][e] = sscale[srow[e] + (GSUB == 1 ? kt >> a.q_shift : kt * GSUB + g)];
    }
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
      i4 bq0, bq1;
      if constexpr (WBITS == 8) {
        bq0 = bitcast<i4>(q.w[t][0] ^ u4{0x80808080u, 0x80808080u, 0x80808080u, 0x80808080u});
        bq1 = bitcast<i4>(q.w[t][TPR - 1] ^ u4{0x80808080u, 0x80808080u, 0x80808080u, 0x80808080u});
      } else {
        const uint32_t z4 = (has_z ? (uint32_t)q.z[t] : 8u) * 0x01010101u;
        bq0 = w8_decode16(q.w[t][0][0], q.w[t][0][1], z4);
        bq1 = w8_decode16(q.w[t][0][2], q.w[t][0][3], z4);
      }
#pragma unroll
      for (int g = 0; g < GSUB; ++g) {
        const bool mine = GSUB == 1 || my_block == g;
        i4 qc = __builtin_amdgcn_mfma_i32_16x16x64_i8(mine ? xa[0] : i4{0, 0, 0, 0}, bq0, i4{0, 0, 0, 0}, 0, 0, 0);
        qc = __builtin_amdgcn_mfma_i32_16x16x64_i8(mine ? xa[1] : i4{0, 0, 0, 0}, bq1, qc, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t][e] = w8_accumulate<PER_K>(qc[e], PER_K ? sa[g][e] : 0.0f, q.s[t][g], acc[t][e]);
      }
    }
  };
  int kt = wave;
  for (; kt + kDepth * W < KT; kt += kDepth * W) {
#pragma unroll
    for (int i = 0; i < kDepth; ++i) {
      const Round now = ring[i];
      request(kt + (kDepth + i) * W, ring[i]);
      multiply(kt + i * W, now);
    }
  }
#pragma unroll
  for (int i = 0; i < kDepth; ++i)
    if (kt + i * W < KT) multiply(kt + i * W, ring[i]);

  // ---- the waves' sums in wave order, then scale / bias / rounding / store ----
  __syncthreads();  // every wave is done with the rows: the region becomes `red`
#pragma unroll
  for (int t = 0; t < NTW; ++t) red[(t * W + wave) * 64 + lane] = acc[t];
  __syncthreads();
  const float* redf = (const float*)red;
  for (int idx = threadIdx.x; idx < NTW * 16 * M; idx += blockDim.x) {
    const int col = idx & 15, tm = idx >> 4;
    const int t = tm / M, m = tm - t * M;  // (M <= 4: the rows of lane column 0)
    const int64_t n = (nt0 + t) * kTileN + col;
    if (n >= a.N) continue;
    const int slot = col * 4 + m;
    float part[8];
#pragma unroll
    for (int w = 0; w < 8; ++w) part[w] = w < W ? redf[(t * W + w) * 256 + slot] : 0.0f;
    float s = part[0];
#pragma unroll
    for (int w = 1; w < 8; ++w) s = s + part[w];
    if (!PER_K) s = s * sscale[m];
    epilogue_store<kRegimeBF16>(a.ep, m, n, s);
  }
}

// Problems of woq_decode_w4i8_kernel (gemm_w4i8_applies) with one scale per row or (row, K block) -- a single row's statistics are
// the tensor's -- whose rows act_quant_rows_kernel would take, in at most four pieces a wave.  NF4 codes and asymmetric
// activations keep the two launches.
static int decode_i8_waves(const Int8Args& a) {
  const int64_t rounds = a.KT / (a.wbits / 4);
  return (int)(rounds < 8 ? rounds : 8);
}
// One row: any width (us with / without its quantization launch, kernels: 4096 -> 4096 5.7 / 8.8, -> 14336 8.9 / 11.3 among other
// passes, 14336 -> 4096 9.7 / 17.2).  More rows: up to 1024 rows x workgroups, since every workgroup pays for all of them and more
// than one of them a CU in turn (four rows 4096 -> 4096 8.8 / 11.1, -> 14336 13.2 / 11.4; three rows -> 11008, groups of 64, 12.9 / 11.9).
static int decode_i8_ntw(const Int8Args& a) {
  // two row-blocks a workgroup where single ones make more than three workgroups a CU, as in launch_gemm_w4i8
  return (a.wbits == 8 || a.group_size != 32) && a.NT >= 769 && a.NT % 2 == 0 ? 2 : 1;
}
bool decode_i8_rows_applies(const Int8Args& a, int64_t qbk, bool per_m, bool per_k, bool asym) {
  if (asym || a.nf4 || a.M > 4 || (a.M > 1 && !per_m)) return false;
  if (a.M > 1 && a.M * (a.NT / decode_i8_ntw(a)) > 1024) return false;
  if (!act_quant_rows_applies(a.x, a.x_dtype, a.K, a.workspace, a.K, qbk, per_m, per_k)) return false;
  return a.M * ((a.K + 511) / 512) <= 4 * decode_i8_waves(a);
}

int launch_decode_i8_rows(const Int8Args& a, int64_t qbk, bool per_k, hipStream_t st) {
  DecodeI8Args d;
  d.x = (const uint16_t*)a.x;
  d.bf16 = a.x_dtype == WOQ_HIP_ACT_BF16;
  d.M = (int)a.M; d.K = (int)a.K; d.NT = (int)a.NT; d.KG = (int)a.KG; d.N = a.N;
  d.KT = (int)(a.KT / (a.wbits / 4));
  d.W = decode_i8_waves(a);
  d.pieces_per_row = (int)((a.K + 511) / 512);
  d.qweight = a.qweight; d.scales = a.scales; d.zeros = a.zeros;
  d.g_shift = 30;
  if (a.group_size > 0)
    for (d.g_shift = 0; ((int64_t)128 << d.g_shift) < a.G;) ++d.g_shift;
  d.q_shift = d.block_lanes_log2 = 0;
  if (per_k) {
    while (((int64_t)128 << d.q_shift) < qbk) ++d.q_shift;
    while (((int64_t)8 << d.block_lanes_log2) < qbk) ++d.block_lanes_log2;
  }
  d.scale_cols = per_k ? (int)((a.K + qbk - 1) / qbk) : 1;
  d.x_base = (d.M * d.scale_cols * (int)sizeof(float) + 1023) & ~1023;
  d.ep = Epilogue{a.bias, a.fusion, a.other0, a.other1, a.out, a.out_dtype, a.x_dtype, a.N};
  const int gsub = a.wbits == 8 ? 1 : a.group_size == 32 ? 4 : a.group_size == 64 ? 2 : 1;
  const int ntw = decode_i8_ntw(a);
  const int rows = d.M * (d.K + 16), red = ntw * d.W * 64 * (int)sizeof(f4);
  const int smem = d.x_base + (rows > red ? rows : red);
  const unsigned grid = (unsigned)(a.NT / ntw);
  const bool one = d.M * d.pieces_per_row <= d.W;
#define WOQ_I8_ROWS(NTWV, GS, WB)                                                               \
  do {                                                                                          \
    if (per_k && one)                                                                           \
      woq_decode_i8_rows_kernel<true, NTWV, GS, WB, 1><<<grid, d.W * 64, smem, st>>>(d);        \
    else if (per_k)                                                                             \
      woq_decode_i8_rows_kernel<true, NTWV, GS, WB, 4><<<grid, d.W * 64, smem, st>>>(d);        \
    else if (one)                                                                               \
      woq_decode_i8_rows_kernel<false, NTWV, GS, WB, 1><<<grid, d.W * 64, smem, st>>>(d);       \
    else                                                                                        \
      woq_decode_i8_rows_kernel<false, NTWV, GS, WB, 4><<<grid, d.W * 64, smem, st>>>(d);       \
  } while (0)
  if (a.wbits == 8 && ntw == 2) WOQ_I8_ROWS(2, 1, 8);
  else if (a.wbits == 8) WOQ_I8_ROWS(1, 1, 8);
  else if (gsub == 4) WOQ_I8_ROWS(1, 4, 4);
  else if (gsub == 2 && ntw == 2) WOQ_I8_ROWS(2, 2, 4);
  else if (gsub == 2) WOQ_I8_ROWS(1, 2, 4);
  else if (ntw == 2) WOQ_I8_ROWS(2, 1, 4);
  else WOQ_I8_ROWS(1, 1, 4);
#undef WOQ_I8_ROWS
  return check_launch("woq_decode_w4i8_kernel");  // (a form of that kernel: reported as it)
}

}  // namespace woq
