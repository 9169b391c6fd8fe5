// Launchers of the general-length column kernel for S samples per lane (gen_column).
// Each S is instantiated in a translation unit of its own: they compile side by side.
#pragma once
#include "generic.h"

#include <algorithm>

#include "generic_launch.h"

namespace ash {

template <int S, bool EVEN, int MODE, int NLK>
void launch_gcol_E(float2* spec, const Tables& T, const Geom& g, const DftMat& d, const ColDesc& cd, hipStream_t s) {
  const dim3 grid(gen_column_blocks(g.nX * g.nY)), block(64 * gcol_waves(S));
  const size_t lds = (size_t)GC_COLS * gcol_pitch(d, S) * sizeof(float);
  if constexpr (S > 4) {  // (a radix is taken past 256 samples)
    if (d.p > 1) {
      hipLaunchKernelGGL((k_gcolumn<S, EVEN, true, MODE, NLK>), grid, block, lds, s, spec, T, g, d, cd);
      return;
    }
  }
  hipLaunchKernelGGL((k_gcolumn<S, EVEN, false, MODE, NLK>), grid, block, lds, s, spec, T, g, d, cd);
}
template <int S, int MODE, int NLK>
void launch_gcol_SMN(float2* spec, const Tables& T, const Geom& g, const DftMat& d, const ColDesc& cd, hipStream_t s) {
  if (d.even) launch_gcol_E<S, true, MODE, NLK>(spec, T, g, d, cd, s);
  else launch_gcol_E<S, false, MODE, NLK>(spec, T, g, d, cd, s);
}
template <int S, int NLK>
void launch_graw(const Tables& T, const Geom& g, const ColDesc& cd, hipStream_t s) {
  const int blocks = std::min((g.nX * g.nY + GR_WPB - 1) / GR_WPB, 2048);
  hipLaunchKernelGGL((k_gcolumn_raw<S, NLK>), dim3(blocks), dim3(64 * GR_WPB), 0, s, T, g, cd);
}
template <int S>
void gen_column_S(float2* spec, const Tables& T, const Geom& g, const DftMat& d, const ColDesc& cd, hipStream_t s) {
  switch (cd.mode) {
    case COL_LOAD: launch_gcol_SMN<S, COL_LOAD, NL_NONE>(spec, T, g, d, cd, s); break;
    case COL_NL:  // (the march's updates; KT_MINMOD is an operator of its own)
      if (cd.nl == NL_KT) launch_gcol_SMN<S, COL_NL, NL_KT>(spec, T, g, d, cd, s);
      else if (cd.nl == NL_TVD) launch_gcol_SMN<S, COL_NL, NL_TVD>(spec, T, g, d, cd, s);
      else launch_gcol_SMN<S, COL_NL, NL_RUSANOV>(spec, T, g, d, cd, s);
      break;
    case COL_TAPER: launch_gcol_SMN<S, COL_TAPER, NL_NONE>(spec, T, g, d, cd, s); break;
    case COL_FINAL: launch_gcol_SMN<S, COL_FINAL, NL_NONE>(spec, T, g, d, cd, s); break;
    case COL_INJECT: launch_gcol_SMN<S, COL_INJECT, NL_NONE>(spec, T, g, d, cd, s); break;
    case COL_STORE: launch_gcol_SMN<S, COL_STORE, NL_NONE>(spec, T, g, d, cd, s); break;
    case COL_RAWNL:
      switch (cd.nl) {
        case NL_KT: launch_graw<S, NL_KT>(T, g, cd, s); break;
        case NL_KT_MINMOD: launch_graw<S, NL_KT_MINMOD>(T, g, cd, s); break;
        case NL_RUSANOV: launch_graw<S, NL_RUSANOV>(T, g, cd, s); break;
        case NL_TVD: launch_graw<S, NL_TVD>(T, g, cd, s); break;
        default: launch_graw<S, NL_NONE>(T, g, cd, s); break;
      }
      break;
    case COL_MAXABS: launch_gcol_SMN<S, COL_MAXABS, NL_NONE>(spec, T, g, d, cd, s); break;
    case COL_TOF: launch_gcol_SMN<S, COL_TOF, NL_NONE>(spec, T, g, d, cd, s); break;
    default: break;
  }
}

}  // namespace ash
