// Launchers of the general-size kernels (generic.h).
#include "generic.h"

#include <algorithm>

#include "generic_launch.h"

namespace ash {

namespace {

DftMat matrix_of(int n, int p) {
  DftMat d{};
  d.n = n;
  d.p = p;
  d.q = n / p;
  d.h = d.q / 2;
  d.even = d.q % 2 == 0;
  auto up = [](int v, int m) { return (v + m - 1) / m * m; };
  d.rows = d.even ? d.h / 2 + 1 : d.h + 1;
  d.R = up(d.rows, 16) / 16;
  d.Ke = up(d.even ? d.h / 2 + 1 : d.h + 1, 8);
  d.Kp = d.Ke + (d.even ? up((d.h + 1) / 2, 8) : 0);
  return d;
}

// Waves of a line block: four while they take at most three row tiles each, else
// eight (at most four tiles each at n = 1024).
int line_waves(const DftMat& d) { return d.p * d.R <= 12 ? 4 : 8; }
int line_tiles(const DftMat& d) { return (d.p * d.R + line_waves(d) - 1) / line_waves(d); }
size_t line_lds(const DftMat& d) { return (size_t)d.p * d.Kp * 16 * sizeof(float4); }

}  // namespace

DftMat dft_matrix_shape(int n, bool columns) {
  DftMat d = matrix_of(n, 1);
  if (n > (columns ? 256 : 128)) {
    // the radix that leaves the fewest products, if that is at most 0.6 of them (a small
    // gain is lost to the radix stage).  Shorter lines are bound by memory already;
    // shorter columns by the launch and the stages between the products: the KT pass at
    // 64x64x189 takes 15.5 us without a radix and 17.4 with one, at 128x128x300 56.6 and
    // 47.6, at 128x128x801 257 and 105, at 128x128x1995 1254 and 449.
    auto products = [](const DftMat& m) { return m.p * m.R * m.Kp; };
    DftMat best = d;
    for (int p : {3, 5, 7, 9}) {
      if (n % p) continue;
      const DftMat m = matrix_of(n, p);
      const bool fits = columns || (line_tiles(m) <= (m.even ? 3 : 4) && line_lds(m) <= 160 * 1024);
      if (products(m) < products(best) && fits) best = m;
    }
    if (10 * products(best) <= 6 * products(d)) d = best;
  }
  d.rs = columns ? d.Kp / 8 * 64 : 64;
  d.gs = columns ? 64 : d.R * 64;
  return d;
}
size_t dft_matrix_bytes(const DftMat& d) { return (size_t)d.R * (d.Kp / 8) * 64 * sizeof(float4); }
void dft_matrix_fill(const DftMat& d, float4* A, hipStream_t s) {
  const long tot = (long)d.R * (d.Kp / 8) * 64;
  const dim3 grid((unsigned)std::min<long>((tot + 255) / 256, 1024));
  if (d.even) hipLaunchKernelGGL(k_dft_matrix<true>, grid, dim3(256), 0, s, d, A);
  else hipLaunchKernelGGL(k_dft_matrix<false>, grid, dim3(256), 0, s, d, A);
}

namespace {

// CALL with T_ = the most row tiles of a wave, EVEN = the parity of the matrix length and
// RADIX = whether a radix stage precedes it
#define DISPATCH_CASE(key, t, even, radix, ...) \
  case key: { constexpr int T_ = t; constexpr bool EVEN = even, RADIX = radix; __VA_ARGS__; } break;
#define DISPATCH_TILES(d, ...)                                        \
  do {                                                                \
    switch (line_tiles(d) * 4 + (d).even * 2 + ((d).p > 1)) {         \
      DISPATCH_CASE(4, 1, false, false, __VA_ARGS__)                  \
      DISPATCH_CASE(5, 1, false, true, __VA_ARGS__)                   \
      DISPATCH_CASE(6, 1, true, false, __VA_ARGS__)                   \
      DISPATCH_CASE(7, 1, true, true, __VA_ARGS__)                    \
      DISPATCH_CASE(8, 2, false, false, __VA_ARGS__)                  \
      DISPATCH_CASE(9, 2, false, true, __VA_ARGS__)                   \
      DISPATCH_CASE(10, 2, true, false, __VA_ARGS__)                  \
      DISPATCH_CASE(11, 2, true, true, __VA_ARGS__)                   \
      DISPATCH_CASE(12, 3, false, false, __VA_ARGS__)                 \
      DISPATCH_CASE(13, 3, false, true, __VA_ARGS__)                  \
      DISPATCH_CASE(14, 3, true, false, __VA_ARGS__)                  \
      DISPATCH_CASE(15, 3, true, true, __VA_ARGS__)                   \
      DISPATCH_CASE(16, 4, false, false, __VA_ARGS__)                 \
      DISPATCH_CASE(17, 4, false, true, __VA_ARGS__)                  \
      default: break;                                                 \
    }                                                                 \
  } while (0)

}  // namespace

void gen_xfwd(float2* spec, const Geom& g, const DftMat& d, hipStream_t s) {
  const dim3 grid(g.nY * g.nfb), block(64 * line_waves(d));
  const size_t lds = line_lds(d);
  DISPATCH_TILES(d, hipLaunchKernelGGL((k_gx_fwd<EVEN, T_, RADIX>), grid, block, lds, s, spec, g, d));
}

void gen_xinv(int epi, float2* spec, const Tables& T, const Geom& g, const DftMat& d, const EpiDesc& e, hipStream_t s) {
  const dim3 grid(g.nY * g.nfb), block(64 * line_waves(d));
  const size_t lds = line_lds(d);
  if (epi == 2) DISPATCH_TILES(d, hipLaunchKernelGGL((k_gx_inv_sa<EVEN, T_, RADIX>), grid, block, lds, s, spec, T, g, d, e));
  else if (epi == 1) DISPATCH_TILES(d, hipLaunchKernelGGL((k_gx_inv<EVEN, T_, RADIX, 1>), grid, block, lds, s, spec, T, g, d, e));
  else DISPATCH_TILES(d, hipLaunchKernelGGL((k_gx_inv<EVEN, T_, RADIX, 0>), grid, block, lds, s, spec, T, g, d, e));
}

void gen_ypass(float2* spec, const Tables& T, const Geom& g, const DftMat& d, const OpDesc& op, hipStream_t s) {
  const dim3 grid(g.nX * g.nfb), block(64 * line_waves(d));
  const size_t lds = line_lds(d);
  if (d.p == 1 && d.R <= 2) {  // the operator from a table in LDS (see k_gy_pass)
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, block, lds + (size_t)d.n * 16 * sizeof(float2), s, spec, T, g, d, op);
    };
    if (op.precise) d.even ? launch(k_gy_pass<true, 1, false, true, true>) : launch(k_gy_pass<false, 1, false, true, true>);
    else d.even ? launch(k_gy_pass<true, 1, false, false, true>) : launch(k_gy_pass<false, 1, false, false, true>);
    return;
  }
  if (op.precise) DISPATCH_TILES(d, hipLaunchKernelGGL((k_gy_pass<EVEN, T_, RADIX, true>), grid, block, lds, s, spec, T, g, d, op));
  else DISPATCH_TILES(d, hipLaunchKernelGGL((k_gy_pass<EVEN, T_, RADIX, false>), grid, block, lds, s, spec, T, g, d, op));
}

void gen_ypower(const float2* spec, const Tables& T, const Geom& g, const DftMat& d, double2* part, hipStream_t s) {
  const dim3 grid(g.nX * g.nfb), block(64 * line_waves(d));
  const size_t lds = line_lds(d);
  DISPATCH_TILES(d, hipLaunchKernelGGL((k_gy_power<EVEN, T_, RADIX>), grid, block, lds, s, spec, T, g, d, part));
}

void gen_ysa(float2* spec, const Tables& T, const Geom& g, const ScreenDesc& sd, hipStream_t s) {
  const size_t lds = (size_t)ysa_rows(g.nY, sd.band, sd.phase != nullptr) * LF * sizeof(float2);
  hipLaunchKernelGGL(k_gy_sa, dim3(g.nX * g.nfb), dim3(256), lds, s, spec, T, g, sd);
}

int gen_column_blocks(int ncols) { return (ncols + GC_COLS - 1) / GC_COLS; }

void gen_column(float2* spec, const Tables& T, const Geom& g, const DftMat& d, const ColDesc& cd, hipStream_t s) {
  // S real samples per lane, 64 S >= nT
  if (g.nT <= 128) gen_column_S<2>(spec, T, g, d, cd, s);
  else if (g.nT <= 256) gen_column_S<4>(spec, T, g, d, cd, s);
  else if (g.nT <= 512) gen_column_S<8>(spec, T, g, d, cd, s);
  else if (g.nT <= 1024) gen_column_S<16>(spec, T, g, d, cd, s);
  else gen_column_S<32>(spec, T, g, d, cd, s);
}

}  // namespace ash
