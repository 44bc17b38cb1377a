// The prefill kernel over the slots of a routed layer.
#include "woq_gemm_w4.h"

namespace woq {

// Row tiles of the routed rows of all experts in one launch (woq_hip_moe_linear).
template <int REGIME, class S, int WBITS, bool MERGED, bool PAIR, bool CHAINS = true>
static int launch_grouped_shape(const FpArgs& f, int g_shift, const G4Group& g, int64_t slots, hipStream_t st) {
  constexpr int kLds = g4_lds_bytes<S, WBITS>();
  static_assert(kLds <= 160 * 1024, "a workgroup's LDS");
  const auto kernel = &woq_gemm_w4_kernel<REGIME, S, WBITS, false, MERGED, true, false, CHAINS, PAIR>;
  static const hipError_t lds_optin =
      hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  if (lds_optin != hipSuccess)
    return set_error("woq_gemm_w4_kernel: LDS opt-in failed: %s", hipGetErrorString(lds_optin));
  constexpr int kColumns = PAIR ? S::BN / 2 : S::BN;
  const dim3 grid((unsigned)((f.NT * kTileN + kColumns - 1) / kColumns), (unsigned)slots);
  kernel<<<grid, 64 * S::WAVES, kLds, st>>>(f, g_shift, nullptr, nullptr, (int)(f.KT / (WBITS / 4)), g);
  return check_launch("woq_gemm_w4_kernel (grouped)");
}

template <int REGIME, int WBITS, bool MERGED>
static int launch_grouped_type(const FpArgs& f, int g_shift, const G4Group& g, int64_t slots, int tile_rows, hipStream_t st) {
  using S8 = G4Shape<8, 2, 8>;
  using S42 = G4Shape<4, 2>;
  if constexpr (WBITS == 4)
    if (tile_rows == 160) {
      using S10 = G4Shape<10, 2, 8>;
      bool chains = false;
      for (int steps : g.chains) chains |= steps != 0;
      if (f.pair)
        return chains ? launch_grouped_shape<REGIME, S10, WBITS, MERGED, true, true>(f, g_shift, g, slots, st)
                      : launch_grouped_shape<REGIME, S10, WBITS, MERGED, true, false>(f, g_shift, g, slots, st);
      return chains ? launch_grouped_shape<REGIME, S10, WBITS, MERGED, false, true>(f, g_shift, g, slots, st)
                    : launch_grouped_shape<REGIME, S10, WBITS, MERGED, false, false>(f, g_shift, g, slots, st);
    }
  if (f.pair)
    return tile_rows == 128 ? launch_grouped_shape<REGIME, S8, WBITS, MERGED, true>(f, g_shift, g, slots, st)
                            : launch_grouped_shape<REGIME, S42, WBITS, MERGED, true>(f, g_shift, g, slots, st);
  return tile_rows == 128 ? launch_grouped_shape<REGIME, S8, WBITS, MERGED, false>(f, g_shift, g, slots, st)
                          : launch_grouped_shape<REGIME, S42, WBITS, MERGED, false>(f, g_shift, g, slots, st);
}

int launch_gemm_w4_grouped(const FpArgs& f, int wbits, int regime, const MoeGroup* grp, int64_t slots, int tile_rows,
                           hipStream_t st) {
  int g_shift = 30;
  if (f.G < f.KT * (wbits == 4 ? kTileK4 : kTileK8)) {
    g_shift = 0;
    while (((int64_t)1 << g_shift) < f.G) ++g_shift;
  }
  G4Group g{};
  g.tables = grp;
  for (int i = 2; i <= kChainRowTiles; ++i) g.chains[i] = gemm_w4_chain_steps(f, wbits, i);
  if (wbits == 8)
    return regime == kRegimeF16 ? launch_grouped_type<kRegimeF16, 8, false>(f, g_shift, g, slots, tile_rows, st)
                                : launch_grouped_type<kRegimeBF16, 8, false>(f, g_shift, g, slots, tile_rows, st);
  if (regime == kRegimeF16) return launch_grouped_type<kRegimeF16, 4, false>(f, g_shift, g, slots, tile_rows, st);
  return f.grp_szb ? launch_grouped_type<kRegimeBF16, 4, true>(f, g_shift, g, slots, tile_rows, st)
                   : launch_grouped_type<kRegimeBF16, 4, false>(f, g_shift, g, slots, tile_rows, st);
}

}  // namespace woq
