// fp32 compute: lowp_mode NONE with fp32 activations (also what lowp_mode INT8 falls back to for
// fp32 activations).
//
// Reference counterpart: woq_gemm_fp32 -> qlinear_woq_affine_impl<float, float, float, float, float,
// float> (csrc/cpu/aten/kernels/WoqLinearKrnl.cpp:142-158): fp32 scales and zero points,
// w = (q - z) * s as a subtraction and a product in fp32 (csrc/cpu/aten/utils/woq.h:183-186,
// 703-708; NF4: table[q] * s), fp32 x fp32 products accumulated in fp32 on top of the fp32 bias,
// post-op and store in fp32.
//
// y[M, N] = x[M, K] * w[N, K]^T on v_mfma_f32_32x32x2_f32: workgroup tile 128 x 128, K step 32,
// 4 waves in a 2 x 2 grid, each owning 64 x 64 as 2 x 2 MFMA tiles (A = activations, B = weights:
// a lane's accumulator registers hold consecutive rows of its own output column); up to 64 rows
// (SMALL) the tile is 32 x 128 and a wave owns one 32 x 32 MFMA tile, a quarter of the MFMA work
// per K step.  Weights are dequantized once per workgroup and K step into LDS.  One MFMA consumes the K pair (2t, 2t + 1),
// lanes 0..31 the even element and lanes 32..63 the odd one; both LDS tiles keep the even elements
// of a row in floats 0..15 and the odd ones in floats 16..31, so that a lane reads the operands of
// four MFMAs with one 16-byte load.
#include <algorithm>

#include "woq_common.h"
#include "woq_internal.h"

namespace woq {

namespace {
constexpr int F_BM = 128, F_BN = 128, F_BK = 32;
constexpr int F_STRIDE = F_BK + 4;  // floats; keeps 16-byte alignment, spreads rows over the banks
}  // namespace

template <int WBITS, bool NF4, bool SMALL>
__global__ __launch_bounds__(256) void woq_fp32_kernel(const Fp32Args f) {
  static_assert(!NF4 || WBITS == 4, "NF4 codes are 4 bits wide");
  constexpr int TK = WBITS == 4 ? kTileK4 : kTileK8;
  constexpr int BM = SMALL ? 32 : F_BM;
  constexpr int XI = BM / 32;         // 16-byte activation pieces per thread and K step
  constexpr int TM = SMALL ? 1 : 2;   // MFMA tiles per wave along M and N
  constexpr int TN = SMALL ? 1 : 2;
  __shared__ __align__(16) float sA[BM * F_STRIDE];
  __shared__ __align__(16) float sB[F_BN * F_STRIDE];
  __shared__ float sTab[16];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int row0 = SMALL ? 0 : (wave >> 1) * 64;             // first row / column of this wave
  const int col0 = SMALL ? wave * 32 : (wave & 1) * 64;
  const int64_t m0 = (int64_t)blockIdx.y * BM;
  const int64_t n0 = (int64_t)blockIdx.x * F_BN;
  const int64_t nt0 = n0 / kTileN;
  const int64_t Kpad = f.KT * TK;
  const bool xvec = (f.K % 4) == 0;

  if (NF4) {
    if (tid < 16) sTab[tid] = kNf4Values[tid];
    __syncthreads();
  }

  f16v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  // weight slot of this thread: row-block ntl of the workgroup's eight, row r, and 16 of the 32 K
  // values of the step
  const int ntl = tid >> 5, r = tid & 15, hh = (tid >> 4) & 1;
  const int64_t nt = nt0 + ntl;
  const bool wvalid = nt < f.NT;

  // raw operands of one K step in registers: requested one step ahead, so that they travel
  // during the MFMAs of the step before
  f4 xa[XI];
  uint32_t d[4] = {0u, 0u, 0u, 0u};
  float s = 1.0f, z = 0.0f;
  auto request = [&](int64_t k0) {
    // ---- activations: BM rows x 32 floats, one 16-byte piece per thread and 32 rows ----
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int64_t m = m0 + (tid >> 3) + 32 * i;
      const int64_t k = k0 + (tid & 7) * 4;
      xa[i] = f4{0.f, 0.f, 0.f, 0.f};
      if (m < f.M) {
        if (xvec) {
          if (k < f.K) xa[i] = *(const f4*)(f.x + m * f.K + k);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (k + e < f.K) xa[i][e] = f.x[m * f.K + k + e];
        }
      }
    }
    // ---- weights: 16 values of one row with their scale and zero point ----
    if (wvalid) {
      const int64_t kt = k0 / TK;
      int64_t g = k0 / f.G;
      if (g >= f.KG) g = f.KG - 1;
      const int64_t qi = (nt * f.KG + g) * kTileN + r;
      s = f.scales[qi];
      z = f.zeros ? (float)f.zeros[qi] : (WBITS == 4 ? 8.0f : 128.0f);
      if (WBITS == 4) {
        const int c = (int)((k0 % TK) / 32);
        const uint32_t* p = (const uint32_t*)(f.qweight + ((nt * f.KT + kt) * 64 + (r + 16 * c)) * 16) + 2 * hh;
        d[0] = p[0];
        d[1] = p[1];
      } else {
        const int c = (int)((k0 % TK) / 16) + hh;
        const u4 v = *(const u4*)(f.qweight + ((nt * f.KT + kt) * 64 + (r + 16 * c)) * 16);
        d[0] = v[0]; d[1] = v[1]; d[2] = v[2]; d[3] = v[3];
      }
    }
  };

  if (Kpad > 0) request(0);
  for (int64_t k0 = 0; k0 < Kpad; k0 += F_BK) {
    // ---- dequantize to fp32 ----
    float w[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      float q;
      if (WBITS == 4)
        q = (float)((d[e >> 3] >> (4 * nibble_pos(e & 7))) & 0xFu);
      else
        q = (float)((d[e >> 2] >> (8 * (e & 3))) & 0xFFu);
      if (NF4)
        w[e] = wvalid ? __fmul_rn(sTab[(int)q], s) : 0.0f;
      else if (WBITS == 8 && f.fp8)  // float8 e4m3fn bytes: w = fp8(byte) * s (woq.h:728-741)
        w[e] = wvalid ? __fmul_rn(fp8_e4m3fn_to_f32((d[e >> 2] >> (8 * (e & 3))) & 0xFFu), s) : 0.0f;
      else
        w[e] = wvalid ? __fmul_rn(__fsub_rn(q, z), s) : 0.0f;
    }

    __syncthreads();  // the previous step's LDS reads are done
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      float* row = sA + ((tid >> 3) + 32 * i) * F_STRIDE;
      const int kl = (tid & 7) * 4;  // elements kl .. kl + 3: two even, two odd
      *(f2*)(row + (kl >> 1)) = f2{xa[i][0], xa[i][2]};
      *(f2*)(row + 16 + (kl >> 1)) = f2{xa[i][1], xa[i][3]};
    }
    {
      float* row = sB + (ntl * 16 + r) * F_STRIDE + hh * 8;  // elements 16 hh .. 16 hh + 15
      *(f4*)(row) = f4{w[0], w[2], w[4], w[6]};
      *(f4*)(row + 4) = f4{w[8], w[10], w[12], w[14]};
      *(f4*)(row + 16) = f4{w[1], w[3], w[5], w[7]};
      *(f4*)(row + 20) = f4{w[9], w[11], w[13], w[15]};
    }
    __syncthreads();
    if (k0 + F_BK < Kpad) request(k0 + F_BK);

    // ---- 16 K pairs: lane half h supplies element 2 t + h of pair t ----
    const int h = lane >> 5;
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      f4 af[TM], bf[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i)
        af[i] = *(const f4*)(sA + (row0 + i * 32 + (lane & 31)) * F_STRIDE + h * 16 + q4 * 4);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        bf[j] = *(const f4*)(sB + (col0 + j * 32 + (lane & 31)) * F_STRIDE + h * 16 + q4 * 4);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i][t], bf[j][t], acc[i][j], 0, 0, 0);
    }
  }

  // ---- epilogue: D[m][n], lane holds n = lane % 32, m = 8 * (e / 4) + 4 * (lane / 32) + e % 4 ----
  Epilogue ep{f.bias, f.fusion, f.other0, f.other1, f.out, WOQ_HIP_ACT_FP32, WOQ_HIP_ACT_FP32, f.N};
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int64_t n = n0 + col0 + j * 32 + (lane & 31);
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t m = m0 + row0 + i * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
        if (m < f.M && n < f.N) epilogue_store<kRegimeBF16>(ep, m, n, acc[i][j][e]);
      }
    }
}

// Few rows (decode), and prompts of any length where K is long (64 rows a workgroup): a workgroup owns NTW row-blocks of 16 output
// columns for all K, its W waves split K, and every operand goes from memory straight into the registers that feed the MFMA.  A packed weight tile already
// has the B layout of v_mfma_f32_16x16x4_f32: lane r + 16 c holds consecutive K values of row r, so MFMA number e of a
// tile takes each lane's value e, and the A operand of lane m + 16 c is x[m] at the same K, read as 16-byte pieces.
// Up to four rows (RT 0) the MFMA is v_mfma_f32_4x4x1_16b: its block l / 4 has the columns 4 (l / 4 % 4) .. + 3 and
// the K values of c = l / 16, so the four K quarters of a tile become four sums that are added with the waves'.
// A 16-row MFMA would spend three quarters of its time on absent rows (9 us of fp32 matrix work at 4096 -> 11008
// against 2.3 us).
// Bound: HBM and the launch up to four rows, the fp32 matrix pipes from 16 rows (16 rows, 4096 -> 11008: 9.2 us at 157 TFLOP/s).
// Against the tiles of 32 / 128 x 128 outputs above, whose workgroups (86 at N = 11008) go through K alone with two barriers
// every 32 values (us, INT8 per channel): 4096 -> 11008 M = 1 / 4 / 16 / 64 / 128 / 512 / 2048: 16.4 / 17.3 (16 waves: 16.5) / 25.5 / 64 / 123 / 446 /
// 1630 against 223 / 224 / 223 / 223 / 502 / 728 / 1868; 14336 -> 1024, M = 64 / 128 / 2048: 107 / 108 / 479 against 700 / 1761 / 1772.
// The tiles win where K is short (fp32_few_rows).  Error against 64 bits 2e-7 .. 8e-7 in the 2-norm (one chain over all of K:
// 1.1e-6 .. 2.2e-6).
enum { kFmtInt8, kFmtFp8, kFmtInt4, kFmtNf4 };

template <int RT, int NTW>
struct Fp32Decode {
  static constexpr int kRows = RT ? RT : 1;  // row tiles of a wave
  static constexpr int kWaves = RT <= 1 && NTW == 1 ? 16 : 8;  // narrow layers: more of K in flight per workgroup
  // (and up to four rows of a longer K, fp32_wide_workgroup; four row-blocks: the sums of 16 waves exceed 64 KiB of LDS)
  static constexpr int kMinWaves = RT <= 1 ? 4 : 2;              // per SIMD: 128 or 256 registers
};

template <int FMT, int RT, int NTW, int W = Fp32Decode<RT, NTW>::kWaves>
__global__ __launch_bounds__((W * 64), (Fp32Decode<RT, NTW>::kMinWaves))
void woq_fp32_decode_kernel(const Fp32Args f) {
  using S = Fp32Decode<RT, NTW>;
  constexpr int R = S::kRows;
  constexpr bool kBytes = FMT == kFmtInt8 || FMT == kFmtFp8;
  constexpr int TK = kBytes ? kTileK8 : kTileK4;
  constexpr int CH = TK / 4;        // K values of a lane in a tile, taken 16 at a time
  constexpr int SUB = CH / 16;
  constexpr bool kAheadX = RT <= 2;  // activations one step ahead; with three or four row tiles there are no registers for it
  __shared__ f4 red[W][NTW][64];
  __shared__ float tab[16];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4;
  const int64_t nt0 = (int64_t)blockIdx.x * NTW;
  const int64_t m0 = (int64_t)blockIdx.y * (RT ? 16 * RT : 4);
  const int KT = (int)f.KT;
  if (FMT == kFmtNf4) {
    if (tid < 16) tab[tid] = kNf4Values[tid];
    __syncthreads();
  }

  // absent rows and row-blocks repeat the last real one; their results are not stored
  const float* xrow[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int64_t m = m0 + 16 * i + (RT ? r : lane & 3);
    xrow[i] = f.x + (m < f.M ? m : f.M - 1) * f.K + c * CH;
  }
  int64_t nt[NTW];
#pragma unroll
  for (int j = 0; j < NTW; ++j) nt[j] = nt0 + j < f.NT ? nt0 + j : f.NT - 1;

  float s0[NTW], z0[NTW], s1[NTW], z1[NTW];
  u4 q0[NTW], q1[NTW];
  auto params = [&](int g, float* s, float* z) {
#pragma unroll
    for (int j = 0; j < NTW; ++j) {
      const int64_t qi = (nt[j] * f.KG + g) * kTileN + r;
      s[j] = f.scales[qi];
      if (FMT == kFmtInt8 || FMT == kFmtInt4) z[j] = f.zeros ? (float)f.zeros[qi] : (FMT == kFmtInt4 ? 8.0f : 128.0f);
    }
  };
  auto request_w = [&](int kt, u4* q, float* s, float* z) {
#pragma unroll
    for (int j = 0; j < NTW; ++j)
      q[j] = __builtin_nontemporal_load((const u4*)(f.qweight + ((nt[j] * f.KT + kt) * 64 + lane) * 16));
    if (f.KG > 1) {  // (a lane's K values of a tile lie in one group: groups are multiples of 32)
      const unsigned g = ((unsigned)kt * TK + c * CH) / (unsigned)f.G;
      params((int)(g < (unsigned)f.KG ? g : (unsigned)f.KG - 1), s, z);
    }
  };
  const bool xvec = (f.K % 4) == 0;
  auto request_x = [&](int kt, int sub, f4 (*x)[4]) {
    const int64_t k = (int64_t)kt * TK + sub * 16;
    if ((int64_t)(kt + 1) * TK <= f.K && xvec) {
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) x[i][q] = *(const f4*)(xrow[i] + k + 4 * q);
    } else {
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int e = 0; e < 4; ++e) x[i][q][e] = c * CH + k + 4 * q + e < f.K ? xrow[i][k + 4 * q + e] : 0.0f;
    }
  };

  f4 acc[NTW][R];
#pragma unroll
  for (int j = 0; j < NTW; ++j)
#pragma unroll
    for (int i = 0; i < R; ++i) acc[j][i] = f4{0.f, 0.f, 0.f, 0.f};

  f4 x0[R][4], x1[R][4];
  if (f.KG <= 1) params(0, s0, z0);
  if (wave < KT) {
    request_w(wave, q0, s0, z0);
    if (kAheadX) request_x(wave, 0, x0);
  }
  for (int kt = wave; kt < KT; kt += W) {
    const bool more = kt + W < KT;
    if (more) request_w(kt + W, q1, s1, z1);
#pragma unroll
    for (int sub = 0; sub < SUB; ++sub) {
      if (!kAheadX)
        request_x(kt, sub, x0);
      else if (sub + 1 < SUB)
        request_x(kt, sub + 1, x1);
      else if (more)
        request_x(kt + W, 0, x1);
#pragma unroll
      for (int j = 0; j < NTW; ++j) {
        float w[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const uint32_t q = kBytes ? (q0[j][e >> 2] >> (8 * (e & 3))) & 0xFFu
                                    : (q0[j][2 * sub + (e >> 3)] >> (4 * nibble_pos(e & 7))) & 0xFu;
          if (FMT == kFmtNf4)
            w[e] = __fmul_rn(tab[q], s0[j]);
          else if (FMT == kFmtFp8)
            w[e] = __fmul_rn(fp8_e4m3fn_to_f32(q), s0[j]);
          else
            w[e] = __fmul_rn(__fsub_rn((float)q, z0[j]), s0[j]);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e)
#pragma unroll
          for (int i = 0; i < R; ++i)
            acc[j][i] = RT ? __builtin_amdgcn_mfma_f32_16x16x4f32(x0[i][e >> 2][e & 3], w[e], acc[j][i], 0, 0, 0)
                           : __builtin_amdgcn_mfma_f32_4x4x1f32(x0[i][e >> 2][e & 3], w[e], acc[j][i], 0, 0, 0);
      }
      if (kAheadX)
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q) x0[i][q] = x1[i][q];
    }
#pragma unroll
    for (int j = 0; j < NTW; ++j) {
      q0[j] = q1[j];
      if (f.KG > 1) { s0[j] = s1[j]; z0[j] = z1[j]; }
    }
  }

  // ---- the waves' sums, in wave order (RT 0: and inside a wave the four K quarters) ----
  Epilogue ep{f.bias, f.fusion, f.other0, f.other1, f.out, WOQ_HIP_ACT_FP32, WOQ_HIP_ACT_FP32, f.N};
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (i) __syncthreads();
#pragma unroll
    for (int j = 0; j < NTW; ++j) red[wave][j][lane] = acc[j][i];
    __syncthreads();
    const int j = tid >> 6;  // (W >= NTW: one wave per row-block)
    if (j >= NTW || nt0 + j >= f.NT) continue;
    if (RT == 0) {
      const int e = lane & 3, col = lane >> 2;
      float sum = 0.0f;
#pragma unroll
      for (int w = 0; w < W; ++w)
#pragma unroll
        for (int q = 0; q < 4; ++q) sum += red[w][j][16 * q + col][e];
      const int64_t m = m0 + e, n = (nt0 + j) * kTileN + col;
      if (m < f.M && n < f.N) epilogue_store<kRegimeBF16>(ep, m, n, sum);
    } else {  // D[m][n]: lane holds n = lane % 16, m = 4 (lane / 16) + e
      f4 sum = red[0][j][lane];
#pragma unroll
      for (int w = 1; w < W; ++w) sum += red[w][j][lane];
      const int64_t n = (nt0 + j) * kTileN + r;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t m = m0 + 16 * i + 4 * c + e;
        if (m < f.M && n < f.N) epilogue_store<kRegimeBF16>(ep, m, n, sum[e]);
      }
    }
  }
}

// Row-blocks per workgroup: the shortest schedule, generations of 256 workgroups times a workgroup's length (its
// row-blocks and about half a one for the activations), ties to the larger count.
static int fp32_decode_ntw(int64_t NT, int64_t gy) {
  int best = 1;
  double best_cost = 1e300;
  for (int n = 1; n <= 4; ++n) {
    const int64_t wg = (NT + n - 1) / n * gy;
    const double cost = (double)((wg + 255) / 256) * (n + 0.5);
    if (cost <= best_cost) { best = n; best_cost = cost; }
  }
  return best;
}

// Up to four rows, two or three row-blocks a workgroup: sixteen waves where they have tiles.  Up to eight tiles half of sixteen waves
// only wait at the barrier (us, 8 / 16 waves: INT8 256 -> 8192, one row 3.3 / 3.6, INT4 1024 -> 8192 4.9 / 5.1, NF4 1024 -> 11008, four rows
// 6.6 / 6.8); one and two rows of 8-bit weights, whose tiles are half as long, gain from more on (INT8 768 -> 8192, one row 11 %
// slower with sixteen, two rows 5 %, 1024 -> 8192 7 % and even, four rows 2 % and 7 % faster).  Longer K: INT8 8192 -> 8192, one row 22.7 / 19.8,
// FP8 4096 -> 11008, four rows 23.0 / 20.2, INT4 1280 -> 8192 5..8 % faster (single lengths lose: INT4 2304 -> 11008, one row 10.4 / 10.8).
template <int FMT>
static bool fp32_wide_workgroup(const Fp32Args& f) {
  constexpr bool kBytes = FMT == kFmtInt8 || FMT == kFmtFp8;
  return f.KT > (kBytes && f.M <= 2 ? (f.M == 1 ? 16 : 12) : 8);
}

template <int FMT, int RT>
static void launch_fp32_decode_rows(const Fp32Args& f, unsigned gy, hipStream_t st) {
  const int ntw = fp32_decode_ntw(f.NT, gy);
  const dim3 grid((unsigned)((f.NT + ntw - 1) / ntw), gy);
  if constexpr (RT == 0) {
    if ((ntw == 2 || ntw == 3) && fp32_wide_workgroup<FMT>(f)) {
      if (ntw == 2)
        woq_fp32_decode_kernel<FMT, RT, 2, 16><<<grid, 1024, 0, st>>>(f);
      else
        woq_fp32_decode_kernel<FMT, RT, 3, 16><<<grid, 1024, 0, st>>>(f);
      return;
    }
  }
#define WOQ_FP32_DECODE(N) woq_fp32_decode_kernel<FMT, RT, N><<<grid, Fp32Decode<RT, N>::kWaves * 64, 0, st>>>(f)
  switch (ntw) {
    case 1: WOQ_FP32_DECODE(1); break;
    case 2: WOQ_FP32_DECODE(2); break;
    case 3: WOQ_FP32_DECODE(3); break;
    default: WOQ_FP32_DECODE(4);
  }
#undef WOQ_FP32_DECODE
}

template <int FMT>
static void launch_fp32_decode(const Fp32Args& f, hipStream_t st) {
  if (f.M <= 4) return launch_fp32_decode_rows<FMT, 0>(f, 1, st);
  const int64_t tiles = (f.M + 15) / 16, gy = (tiles + 3) / 4;
  switch ((tiles + gy - 1) / gy) {
    case 1: return launch_fp32_decode_rows<FMT, 1>(f, (unsigned)gy, st);
    case 2: return launch_fp32_decode_rows<FMT, 2>(f, (unsigned)gy, st);
    case 3: return launch_fp32_decode_rows<FMT, 3>(f, (unsigned)gy, st);
    default: return launch_fp32_decode_rows<FMT, 4>(f, (unsigned)gy, st);
  }
}

// The kernel for few rows or the tiles: the shorter of two estimates (us).
// Few rows: generations of 256 workgroups, each a fixed part and its MFMAs, 0.00103 us a K value and accumulator tile (eight
// waves), but at least one wave's way through one K tile (64 or, 4-bit, 128 K values); rows that are no multiple of 16 bytes are read value by value (1.75
// times).  Tiles: 8 + 0.115 K while they fit the chip once (SMALL: 5 + 0.05 K up to twice), 8 + 0.08 K per 256 of them beyond;
// 4-bit weights less.
// Measured few rows / tiles: K = 64, N = 16384, M = 64 12 / 9; K = 128, N = 65536, M = 32 / 64 / 128 25 / 46 / 88 against 15 / 22 / 46;
// N = 16384, M = 512: K = 256 98 / 71, 512 131 / 117, 1024 197 / 208, 2048 330 / 387; M = 4096: K = 1024 1512 / 1489, 2048 2604 / 2795;
// INT4 K = 256, M = 64 19 / 15, K = 1024, M = 512 209 / 195; 4090 -> 11000, M = 129 / 512 / 2048: 239 / 755 / 2757 against 464 / 720 / 2022; 512 -> 32,
// M = 8192 13 / 59; 4096 -> 11008, M = 8192 6385 / 6868.
static bool fp32_few_rows(const Fp32Args& f, int wbits) {
  // (its group index is 32 bits wide, its row blocks are a grid dimension)
  if (f.KT * kTileK4 >= (1ll << 31) || f.M > 64 * 65535) return false;
  if (f.M <= 4) return true;
  const double K = (double)f.K, thin = wbits == 4 ? 0.85 : 1.0;
  const int64_t tiles16 = (f.M + 15) / 16, gy = (tiles16 + 3) / 4, rt = (tiles16 + gy - 1) / gy;
  const int64_t ntw = fp32_decode_ntw(f.NT, gy);
  const double u = (double)(rt * ntw), gens = (double)(((f.NT + ntw - 1) / ntw * gy + 255) / 256);
  const double few = gens * (2.7 + 0.27 * u + u * std::max(wbits == 4 ? 0.6 : 0.26, 0.00103 * K) * (f.K % 4 ? 1.75 : 1.0));
  const int64_t columns = (f.NT * kTileN + F_BN - 1) / F_BN;
  double tiled;
  if (f.M <= 64) {
    const double wgs = (double)(columns * ((f.M + 31) / 32));
    tiled = (5.0 + 0.05 * thin * K) * std::max(1.0, wgs / 512.0);
  } else {
    const double wgs = (double)(columns * ((f.M + F_BM - 1) / F_BM));
    tiled = std::max(8.0 + 0.115 * thin * K, wgs / 256.0 * (8.0 + 0.08 * thin * K));
  }
  return few <= tiled;
}

int launch_fp32(const Fp32Args& f, int wbits, hipStream_t st) {
  if (f.G <= 0 || f.G % F_BK != 0) return set_error("woq_linear: fp32 compute needs groups that are multiples of 32");
  if (fp32_few_rows(f, wbits)) {
    if (wbits == 8)
      f.fp8 ? launch_fp32_decode<kFmtFp8>(f, st) : launch_fp32_decode<kFmtInt8>(f, st);
    else
      f.nf4 ? launch_fp32_decode<kFmtNf4>(f, st) : launch_fp32_decode<kFmtInt4>(f, st);
    return check_launch("woq_fp32_decode_kernel");
  }
  const bool small = f.M <= 64;
  const int bm = small ? 32 : F_BM;
  const dim3 grid((unsigned)((f.NT * kTileN + F_BN - 1) / F_BN), (unsigned)((f.M + bm - 1) / bm));
#define WOQ_FP32(WB, NF)                                          \
  (small ? woq_fp32_kernel<WB, NF, true><<<grid, 256, 0, st>>>(f) \
         : woq_fp32_kernel<WB, NF, false><<<grid, 256, 0, st>>>(f))
  if (wbits == 8)
    WOQ_FP32(8, false);
  else if (f.nf4)
    WOQ_FP32(4, true);
  else
    WOQ_FP32(4, false);
#undef WOQ_FP32
  return check_launch("woq_fp32_kernel");
}

}  // namespace woq
