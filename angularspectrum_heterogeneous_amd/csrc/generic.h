// General-size kernels: the same sweeps as kernels.h / column.h for grid sizes
// outside the FFT kernels' set (any line length 2..1024, any nT 4..2048), e.g.
// the odd and prime grids of the reference's validation scripts.
//
// The transforms are direct DFTs on the matrix cores (v_mfma_f32_16x16x4_f32:
// float32 operands and accumulation).  With e_j = x_j + x_{n-j} and
// o_j = x_j - x_{n-j} (0 <= j <= n/2) a length-n DFT is two real matrix products
//   C_k = sum_j cos(2 pi j k / n) e_j,   S_k = sum_j sin(2 pi j k / n) o_j,
//   X_k = C_k - i S_k,   X_{n-k} = C_k + i S_k,
// a quarter of the direct sum's products.  For even n = 2h the sums over even and
// odd j are kept apart: position h - k has the same terms with the signs
// (-1)^j and -(-1)^j, so the rows k <= h/2 give all four positions k, h - k,
// h + k and n - k, another half.  The matrices come from the full-length twiddle
// table exp(-2 pi i k / n) at (j k) mod n, so every entry is exact to one rounding,
// and lie in memory in the order in which the lanes load them (k_dft_matrix).
//
// A length n = p q with a small odd factor p runs a p-point DFT first (decimation in
// frequency): X_{p k + r} is the q-point DFT over s of W_n^{s r} sum_m x_{s + q m}
// W_p^{m r}, so the matrix is that of q and a p-th of the products remain.  The radix
// stage happens where the tile is folded into LDS; the inverse half of the y pass,
// whose input lies in the order p k + r, runs it last instead.  At 365 = 5 * 73 an x
// sweep takes 116 us instead of 211, the y pass 293 instead of 485.
//
// Per element of a complex line that is 2n flops (odd n) or n (even n): at
// 365x365x425 an x sweep does 20.7 GFLOP over 454 MB, so the matrix cores bound it
// above n of about 200 and memory below.  There, against the direct sums through LDS
// (a vector fma and two LDS reads per term): x sweep 2217 -> 211 us, y pass 5145 ->
// 485 us before the radix, KT column pass 5736 -> 613 us and 451 with it; at
// 193x193x1201, whose 1201 is prime, the KT column pass 17.7 -> 1.42 ms.
#pragma once
#include "column.h"

namespace ash {

constexpr int GEN_MAXL = 1024;  // general-size line kernels: 2 .. 1024

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Input position of matrix column r: natural order for odd n, the even positions
// and then (from column Ke on) the odd ones for even n.
template <bool EVEN>
__device__ __forceinline__ int hm_pos(const DftMat& d, int r) {
  if constexpr (EVEN) return r < d.Ke ? 2 * r : 2 * (r - d.Ke) + 1;
  else return r;
}
// and the column of input position j
template <bool EVEN>
__device__ __forceinline__ int hm_col(const DftMat& d, int j) {
  if constexpr (EVEN) return (j & 1) ? d.Ke + (j >> 1) : (j >> 1);
  else return j;
}

// Fills the matrix of one axis: entry (rt, g, lane) holds (cos, sin) at matrix row
// 16 rt + lane % 16 and columns 8 g + lane / 16 and 8 g + 4 + lane / 16, the A
// operands of two matrix-core products of four columns each; zero outside.  For lines
// the row tiles of a group lie side by side (a wave takes several row tiles through
// the groups together); for columns the groups of a row tile do (a wave takes one row
// tile at a time).  Each order is the faster one for its kernels: an x sweep at
// 365x365x425 takes 225 against 255 us, a column inverse there 323 against 408 us.
template <bool EVEN>
__global__ __launch_bounds__(256) void k_dft_matrix(DftMat d, float4* __restrict__ out) {
  const long tot = (long)d.R * (d.Kp / 8) * 64;
  for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < tot; e += (long)gridDim.x * 256) {
    const int lane = (int)(e % 64);
    const int rt = (int)(e / 64 % d.R), g = (int)(e / 64 / d.R);
    const int k = 16 * rt + (lane & 15);
    float v[4];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int j = hm_pos<EVEN>(d, 8 * g + 4 * q + (lane >> 4));
      float2 w = make_float2(0.f, 0.f);
      if (k < d.rows && j <= d.h) {
        const float4 t = d.tw[(int)(((long)j * k) % d.q) * d.p];
        w = make_float2(t.x, t.y);
      }
      v[2 * q] = w.x;
      v[2 * q + 1] = -w.y;
    }
    out[(long)rt * d.rs + (long)g * d.gs + lane] = make_float4(v[0], v[1], v[2], v[3]);
  }
}

// ---------------------------------------------------------------------------
// Lines (x and y sweeps).  A tile is all n positions of 16 consecutive f bins
// (128-byte segments), folded into LDS rows [column r][line] of (e.re, e.im,
// o.re, o.im): lane l's B operands of four matrix columns are one 16-byte read at
// 4 s + l/16 of line l%16, 1 KB in a row per wave.  Every matrix entry meets two
// operands (re and im), so the matrix stream from L2 stays at 16 B per CU-cycle of
// matrix-core time.
// ---------------------------------------------------------------------------
template <bool EVEN>
struct LineAcc {
  static constexpr int NP = EVEN ? 2 : 1;  // sums over even j and over odd j
  f32x4 c[NP][2], s[NP][2];                // [parity][re, im]
};

// The row tiles of a wave: [lo, lo + cnt) of n, counts that differ by at most one.  A
// line has p R of them, tile t = row tile t % R of residue t / R.
struct Tiles { int lo, cnt; };
__device__ __forceinline__ Tiles hm_tiles(int n, int wave, int W) {
  const int lo = wave * n / W;
  return {lo, (wave + 1) * n / W - lo};
}

// Walks ng matrix column groups through a ring of U register buffers: use(q) consumes
// buffer q, load(q, g) refills it with group g.  A refill is issued right after its
// buffer's use and consumed U - 1 groups later; the scheduling barriers keep it there
// (left to itself the compiler moves each load down to its use, and every group waits
// for L2: a column inverse at 193x193x1201 takes 559 against 867 us, 96 TFLOP/s).
template <int U, class Load, class Use>
__device__ __forceinline__ void hm_ring(int ng, Load load, Use use) {
#pragma unroll
  for (int q = 0; q < U; ++q) load(q, min(q, ng - 1));
  int g = 0;
  for (; g + 2 * U <= ng; g += U) {
#pragma unroll
    for (int q = 0; q < U; ++q) {
      use(q);
      load(q, g + U + q);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int q = 0; q < U; ++q)
    if (g + q < ng) {
      use(q);
      if (g + U + q < ng) load(q, g + U + q);
    }
#pragma unroll
  for (int q = 0; q < U - 1; ++q)
    if (g + U + q < ng) use(q);
}

// N row tiles from rt0 on together: the operands of a group serve all of them, 8 N
// products (256 N cycles of the SIMD's matrix core) per group.
template <bool EVEN, int N>
__device__ __forceinline__ void hm_line_n(const float4* eo, const DftMat& d, int rt0, int lane, LineAcc<EVEN>* a) {
  constexpr int U = N == 1 ? 4 : 2;
#pragma unroll
  for (int p = 0; p < LineAcc<EVEN>::NP; ++p) {
    const int gp = p == 0 ? 0 : d.Ke / 8, ng = (p == 0 ? d.Ke : d.Kp - d.Ke) / 8;
    const float4* ap = d.A + (long)gp * d.gs + rt0 * d.rs + lane;
    const float4* bp = eo + gp * 128 + lane;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int q = 0; q < 2; ++q) a[i].c[p][q] = a[i].s[p][q] = f32x4{0.f, 0.f, 0.f, 0.f};
    float4 w[U][N], b[U][2];
    hm_ring<U>(
        ng,
        [&](int q, int g) {
#pragma unroll
          for (int i = 0; i < N; ++i) w[q][i] = ap[g * d.gs + i * d.rs];
          b[q][0] = bp[g * 128];
          b[q][1] = bp[g * 128 + 64];
        },
        [&](int q) {
#pragma unroll
          for (int i = 0; i < N; ++i) {
            a[i].c[p][0] = mfma4(w[q][i].x, b[q][0].x, a[i].c[p][0]);
            a[i].c[p][1] = mfma4(w[q][i].x, b[q][0].y, a[i].c[p][1]);
            a[i].s[p][0] = mfma4(w[q][i].y, b[q][0].z, a[i].s[p][0]);
            a[i].s[p][1] = mfma4(w[q][i].y, b[q][0].w, a[i].s[p][1]);
          }
#pragma unroll
          for (int i = 0; i < N; ++i) {
            a[i].c[p][0] = mfma4(w[q][i].z, b[q][1].x, a[i].c[p][0]);
            a[i].c[p][1] = mfma4(w[q][i].z, b[q][1].y, a[i].c[p][1]);
            a[i].s[p][0] = mfma4(w[q][i].w, b[q][1].z, a[i].s[p][0]);
            a[i].s[p][1] = mfma4(w[q][i].w, b[q][1].w, a[i].s[p][1]);
          }
        });
  }
}
// The wave's tiles, T_ or T_ - 1 of them (T_ = ceil(p R / W)): together when they are
// rows of one matrix product (p = 1), else one after the other.
template <bool EVEN, int T_, bool RADIX>
__device__ __forceinline__ void hm_line(const float4* eo, const DftMat& d, const Tiles& t, int lane, LineAcc<EVEN> (&a)[T_]) {
  if constexpr (RADIX) {
#pragma unroll
    for (int i = 0; i < T_; ++i)
      if (i < t.cnt) {
        const int r = (t.lo + i) / d.R;
        hm_line_n<EVEN, 1>(eo + r * d.Kp * 16, d, t.lo + i - r * d.R, lane, a + i);
      }
  } else if (t.cnt == T_) hm_line_n<EVEN, T_>(eo, d, t.lo, lane, a);
  else if constexpr (T_ > 1) hm_line_n<EVEN, T_ - 1>(eo, d, t.lo, lane, a);
}

// The transform's values at output row k = 16 rt + 4 (lane / 16) + i of line
// lane % 16: P = C - i S belongs to position k of the forward transform and
// Q = C + i S to position n - k (the inverse swaps them); for even n also P2, Q2 of
// positions h - k and h + k.
template <bool EVEN>
__device__ __forceinline__ void hm_values(const LineAcc<EVEN>& a, int i, float2& P, float2& Q, float2& P2, float2& Q2) {
  float cr = a.c[0][0][i], ci = a.c[0][1][i], sr = a.s[0][0][i], si = a.s[0][1][i];
  if constexpr (EVEN) {
    const float cr1 = a.c[1][0][i], ci1 = a.c[1][1][i], sr1 = a.s[1][0][i], si1 = a.s[1][1][i];
    const float dcr = cr - cr1, dci = ci - ci1, dsr = sr1 - sr, dsi = si1 - si;
    P2 = make_float2(dcr + dsi, dci - dsr);
    Q2 = make_float2(dcr - dsi, dci + dsr);
    cr += cr1; ci += ci1; sr += sr1; si += si1;
  }
  P = make_float2(cr + si, ci - sr);
  Q = make_float2(cr - si, ci + sr);
}

// f(position, value) for every output of this lane in tile t: position(k, r) of output k
// of residue r
template <bool EVEN, bool INV, class Pos, class F>
__device__ __forceinline__ void hm_emit_at(const DftMat& d, const LineAcc<EVEN>& a, int t, int lane, Pos position, F f) {
  const int r = t / d.R, rt = t - r * d.R;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int k = 16 * rt + 4 * (lane >> 4) + i;
    float2 P, Q, P2, Q2;
    hm_values<EVEN>(a, i, P, Q, P2, Q2);
    if (k < d.rows) {
      f(position(k, r), INV ? Q : P);
      if (k > 0) f(position(d.q - k, r), INV ? P : Q);
      if constexpr (EVEN) {
        const int k2 = d.h - k;
        if (k2 != k) {
          f(position(k2, r), INV ? Q2 : P2);
          if (k > 0) f(position(d.h + k, r), INV ? P2 : Q2);
        }
      }
    }
  }
}
template <bool EVEN, bool INV, class F>
__device__ __forceinline__ void hm_emit(const DftMat& d, const LineAcc<EVEN>& a, int t, int lane, F f) {
  hm_emit_at<EVEN, INV>(d, a, t, lane, [&](int k, int r) { return d.p * k + r; }, f);
}

// cos and sin of 2 pi k / P, k = 1 .. P/2, as hi/lo pairs (fft_engine.h: constants
// rounded to float would bias every transform the same way).
template <int P> struct OddTrig;
template <> struct OddTrig<3> {
  static constexpr float ch[] = {-0.5f}, cl[] = {2.220446049250313e-16f};
  static constexpr float sh[] = {0.8660253882408142f}, sl[] = {1.5543625053737742e-08f};
};
template <> struct OddTrig<5> {
  static constexpr float ch[] = {0.30901700258255005f, -0.80901700258255f}, cl[] = {-8.207602597565256e-09f, 8.207602597565256e-09f};
  static constexpr float sh[] = {0.9510565400123596f, 0.5877852439880371f}, sl[] = {-2.3717205976936384e-08f, 8.304436249773062e-09f};
};
template <> struct OddTrig<7> {
  static constexpr float ch[] = {0.6234897971153259f, -0.22252093255519867f, -0.9009688496589661f}, cl[] = {4.743407444607328e-09f, -1.4011156679316628e-09f, -1.8243452970523322e-08f};
  static constexpr float sh[] = {0.7818315029144287f, 0.9749279022216797f, 0.4338837265968323f}, sl[] = {-2.0446398352191864e-08f, 9.960143820819667e-09f, 1.252072578949992e-08f};
};
template <> struct OddTrig<9> {
  static constexpr float ch[] = {0.7660444378852844f, 0.1736481785774231f, -0.5f, -0.9396926164627075f}, cl[] = {5.2336934786012534e-09f, -9.104926812497638e-10f, 2.220446049250313e-16f, -4.323200908373792e-09f};
  static constexpr float sh[] = {0.6427876353263855f, 0.9848077297210693f, 0.8660253882408142f, 0.3420201539993286f}, sl[] = {-2.5639845802061245e-08f, 2.3291137907222037e-08f, 1.5543625053737742e-08f, -1.0673659289750503e-08f};
};
// 1/n as a hi/lo pair (rounded to float it would scale every sample by the same error in
// every visit) and x times such a pair: the low product meets the high one before a
// rounding, for added to a rounded sum it would be lost
__device__ __forceinline__ float2 inverse_pair(int n) {
  const float hi = 1.f / (float)n;
  return make_float2(hi, fmaf(-hi, (float)n, 1.f) * hi);
}
__device__ __forceinline__ float by_pair(float x, float2 w) { return fmaf(x, w.x, x * w.y); }
// P-point DFT in registers, P odd: with a_m = x_m + x_{P-m}, b_m = x_m - x_{P-m},
// y_r = x_0 + sum cos(2 pi m r / P) a_m -+ i sum sin(2 pi m r / P) b_m, y_{P-r} its mirror.
template <int P, bool INV>
__device__ __forceinline__ void odd_dft(float2* x) {
  using C = OddTrig<P>;
  constexpr int H = P / 2;
  float2 a[H], b[H];
#pragma unroll
  for (int m = 1; m <= H; ++m) {
    a[m - 1] = cadd(x[m], x[P - m]);
    b[m - 1] = csub(x[m], x[P - m]);
  }
  const float2 x0 = x[0];
  float2 sum = x0;
#pragma unroll
  for (int m = 0; m < H; ++m) sum = cadd(sum, a[m]);
#pragma unroll
  for (int r = 1; r <= H; ++r) {
    float2 A = x0, B = make_float2(0.f, 0.f);
#pragma unroll
    for (int m = 1; m <= H; ++m) {
      const int j = (m * r) % P, jj = j > H ? P - j : j;
      if (jj == 0) {
        A = cadd(A, a[m - 1]);
      } else {
        const float2 c = make_float2(C::ch[jj - 1], C::cl[jj - 1]);
        const float2 s = j > H ? make_float2(-C::sh[jj - 1], -C::sl[jj - 1]) : make_float2(C::sh[jj - 1], C::sl[jj - 1]);
        A = make_float2(A.x + by_pair(a[m - 1].x, c), A.y + by_pair(a[m - 1].y, c));
        B = make_float2(B.x + by_pair(b[m - 1].x, s), B.y + by_pair(b[m - 1].y, s));
      }
    }
    const float2 u = make_float2(A.x + B.y, A.y - B.x), v = make_float2(A.x - B.y, A.y + B.x);
    x[r] = INV ? v : u;
    x[P - r] = INV ? u : v;
  }
  x[0] = sum;
}
// x times W_n^k (conjugated for the inverse), k < n, with the twiddle as a hi/lo pair: one
// rounded to float would scale the same element by the same error in every transform of
// a march, where the entries of the matrix average out over a sum.
template <bool INV>
__device__ __forceinline__ float2 cmul_tw(float2 x, float4 w) {
  if (INV) { w.y = -w.y; w.w = -w.w; }
  return make_float2(fmaf(x.x, w.x, fmaf(-x.y, w.y, fmaf(x.x, w.z, -x.y * w.w))),
                     fmaf(x.x, w.y, fmaf(x.y, w.x, fmaf(x.x, w.w, x.y * w.z))));
}
// x_r *= W_n^{s r}, r = 1 .. P-1; s r < n.  W_n^{(q-s) r} = W_p^r conj W_n^{s r}: the partner
// q - s enters its P-point DFT one place further on and takes the conjugate twiddles, so
// a folded pair reads one set (with two the line kernels hold 133 registers, three
// waves a SIMD).
template <int P, bool INV>
__device__ __forceinline__ void odd_twiddle(float2* x, const float4* tw, int s) {
#pragma unroll
  for (int r = 1; r < P; ++r) x[r] = cmul_tw<INV>(x[r], tw[s * r]);
}
template <int P, bool INV>
__device__ __forceinline__ void odd_twiddle_pair(float2* x, float2* partner, const float4* tw, int s) {
#pragma unroll
  for (int r = 1; r < P; ++r) {
    const float4 w = tw[s * r];
    x[r] = cmul_tw<INV>(x[r], w);
    partner[r] = cmul_tw<!INV>(partner[r], w);
  }
}

// Folds a line tile into LDS (rows [residue r][matrix column][line]); ld(position, line)
// reads one element.  All loads of a row (of four rows when p = 1) are issued before the
// first is used.
template <bool EVEN, bool INV, int P, class Ld>
__device__ __forceinline__ void hm_fold_p(float4* eo, const DftMat& d, int tid, int nthr, Ld ld) {
  const int line = tid & 15, step = nthr >> 4;
  for (int rr = tid >> 4; rr < d.Kp; rr += step) {
    const int j = hm_pos<EVEN>(d, rr);
    const bool pair = j > 0 && 2 * j != d.q;
    const int s0 = min(j, d.h), s1 = pair && j <= d.h ? d.q - j : s0;
    float2 a[P], b[P];
#pragma unroll
    for (int m = 0; m < P; ++m) {
      a[m] = ld(s0 + d.q * m, line);
      b[(m + 1) % P] = ld(s1 + d.q * m, line);
    }
    odd_dft<P, INV>(a);
    odd_dft<P, INV>(b);
    odd_twiddle_pair<P, INV>(a, b, d.tw, s0);
#pragma unroll
    for (int r = 0; r < P; ++r) {
      float4 v = make_float4(a[r].x, a[r].y, 0.f, 0.f);
      if (pair) v = make_float4(a[r].x + b[r].x, a[r].y + b[r].y, a[r].x - b[r].x, a[r].y - b[r].y);
      if (j > d.h) v = make_float4(0.f, 0.f, 0.f, 0.f);  // matrix padding
      eo[(r * d.Kp + rr) * 16 + line] = v;
    }
  }
}
// (`between` runs once, while the first rows' loads are in flight, when there is no radix)
struct HmNothing { __device__ void operator()() const {} };
template <bool EVEN, bool INV, bool RADIX, class Ld, class Fn = HmNothing>
__device__ __forceinline__ void hm_fold(float4* eo, const DftMat& d, int tid, int nthr, Ld ld, Fn between = Fn()) {
  if constexpr (RADIX) {
    switch (d.p) {
      case 3: hm_fold_p<EVEN, INV, 3>(eo, d, tid, nthr, ld); break;
      case 5: hm_fold_p<EVEN, INV, 5>(eo, d, tid, nthr, ld); break;
      case 7: hm_fold_p<EVEN, INV, 7>(eo, d, tid, nthr, ld); break;
      default: hm_fold_p<EVEN, INV, 9>(eo, d, tid, nthr, ld); break;
    }
    return;
  }
  const int line = tid & 15, step = nthr >> 4;
  float2 a[4], b[4];
  auto load = [&](int r0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int j = min(hm_pos<EVEN>(d, min(r0 + q * step, d.Kp - 1)), d.h);
      a[q] = ld(j, line);
      b[q] = ld(j == 0 ? 0 : d.n - j, line);
    }
  };
  load(tid >> 4);
  between();
  for (int r0 = tid >> 4; r0 < d.Kp; r0 += 4 * step) {
    if (r0 != tid >> 4) load(r0);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = r0 + q * step;
      if (r >= d.Kp) break;
      const int j = hm_pos<EVEN>(d, r);
      const bool pair = j > 0 && 2 * j != d.n;  // positions 0 and n/2 have no partner
      float4 v = make_float4(a[q].x, a[q].y, 0.f, 0.f);
      if (pair) v = make_float4(a[q].x + b[q].x, a[q].y + b[q].y, a[q].x - b[q].x, a[q].y - b[q].y);
      if (j > d.h) v = make_float4(0.f, 0.f, 0.f, 0.f);  // matrix padding
      eo[r * 16 + line] = v;
    }
  }
}

// The radix stage after the inverse q-point transforms z[r][s] (rows of 16 lines):
// x_{s + q m} = sum_r W_p^{-m r} W_n^{-s r} z_r[s]; st(position, line, value) stores.
template <int P, class St>
__device__ __forceinline__ void hm_combine_p(const float2* z, const DftMat& d, int tid, int nthr, St st) {
  const int line = tid & 15, step = nthr >> 4;
  for (int s = tid >> 4; s < d.q; s += step) {
    float2 x[P];
#pragma unroll
    for (int r = 0; r < P; ++r) x[r] = z[(r * d.q + s) * 16 + line];
    odd_twiddle<P, true>(x, d.tw, s);
    odd_dft<P, true>(x);
#pragma unroll
    for (int m = 0; m < P; ++m) st(s + d.q * m, line, x[m]);
  }
}
template <class St>
__device__ __forceinline__ void hm_combine(const float2* z, const DftMat& d, int tid, int nthr, St st) {
  switch (d.p) {
    case 3: hm_combine_p<3>(z, d, tid, nthr, st); break;
    case 5: hm_combine_p<5>(z, d, tid, nthr, st); break;
    case 7: hm_combine_p<7>(z, d, tid, nthr, st); break;
    default: hm_combine_p<9>(z, d, tid, nthr, st); break;
  }
}

// x-sweep, forward DFT along x.  Tile = (y, 16 f bins).  Padding lines past the last
// bin are zero and stay zero, so no load or store is guarded.
template <bool EVEN, int T_, bool RADIX>
__global__ __launch_bounds__(512) void k_gx_fwd(float2* __restrict__ spec, Geom g, DftMat d) {
  extern __shared__ float4 eo[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, W = blockDim.x >> 6;
  const int y = blockIdx.x / g.nfb, f0 = (blockIdx.x % g.nfb) * LF;
  const uint32_t sxb = (uint32_t)g.nY * g.MP * 8u;
  float2* base = spec + (long)y * g.MP + f0;
  hm_fold<EVEN, false, RADIX>(eo, d, tid, blockDim.x, [&](int pos, int line) { return gld(base, pos * sxb + line * 8u); });
  __syncthreads();
  const uint32_t lo = (lane & 15) * 8u;
  const Tiles t = hm_tiles(d.p * d.R, wave, W);
  LineAcc<EVEN> a[T_];
  hm_line<EVEN, T_, RADIX>(eo, d, t, lane, a);
#pragma unroll
  for (int i = 0; i < T_; ++i)
    if (i < t.cnt) hm_emit<EVEN, false>(d, a[i], t.lo + i, lane, [&](int pos, float2 v) { gst(base, pos * sxb + lo, v); });
}

// x-sweep, inverse DFT along x + the epilogues 0 and 1 of k_xfft_inv.
template <bool EVEN, int T_, bool RADIX, int EPI>
__global__ __launch_bounds__(512) void k_gx_inv(float2* __restrict__ spec, Tables T, Geom g, DftMat d, EpiDesc ep) {
  extern __shared__ float4 eo[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, W = blockDim.x >> 6;
  const int y = blockIdx.x / g.nfb, f0 = (blockIdx.x % g.nfb) * LF;
  const uint32_t sxb = (uint32_t)g.nY * g.MP * 8u;
  float2* base = spec + (long)y * g.MP + f0;
  hm_fold<EVEN, true, RADIX>(eo, d, tid, blockDim.x, [&](int pos, int line) { return gld(base, pos * sxb + line * 8u); });
  __syncthreads();
  const uint32_t lo = (lane & 15) * 8u;
  float ty = 1.f;
  const float* tx = nullptr;
  if constexpr (EPI == 1) {
    ty = ep.half ? T.tapy_h[y] : T.tapy_f[y];
    tx = ep.half ? T.tapx_h : T.tapx_f;
  }
  const Tiles t = hm_tiles(d.p * d.R, wave, W);
  LineAcc<EVEN> a[T_];
  hm_line<EVEN, T_, RADIX>(eo, d, t, lane, a);
#pragma unroll
  for (int i = 0; i < T_; ++i)
    if (i < t.cnt)
      hm_emit<EVEN, true>(d, a[i], t.lo + i, lane, [&](int pos, float2 v) {
        if constexpr (EPI == 1) v = cscale(v, tx[pos] * ty);
        gst(base, pos * sxb + lo, v);
      });
}

// x-sweep, inverse DFT along x + epilogue 2 of k_xfft_inv: scale, DC/Nyquist
// projection, frequency-weighted mask and the SA x stencil on the masked values,
// which pass through the tile's LDS (n * 16 float2 fit the folded tile) once every
// wave holds its T row tiles in registers.
template <bool EVEN, int T_, bool RADIX>
__global__ __launch_bounds__(512) void k_gx_inv_sa(float2* __restrict__ spec, Tables T, Geom g, DftMat d, EpiDesc ep) {
  extern __shared__ float4 eo[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, W = blockDim.x >> 6;
  const int y = blockIdx.x / g.nfb, f0 = (blockIdx.x % g.nfb) * LF;
  const uint32_t sxb = (uint32_t)g.nY * g.MP * 8u;
  float2* base = spec + (long)y * g.MP + f0;
  hm_fold<EVEN, true, RADIX>(eo, d, tid, blockDim.x, [&](int pos, int line) { return gld(base, pos * sxb + line * 8u); });
  __syncthreads();
  const Tiles t = hm_tiles(d.p * d.R, wave, W);
  LineAcc<EVEN> a[T_];
  hm_line<EVEN, T_, RADIX>(eo, d, t, lane, a);
  __syncthreads();
  float2* b = reinterpret_cast<float2*>(eo);
  const float lgy = T.lgy[y];
  {
    const int line = lane & 15, m = f0 + line;
    const float fe = T.fw_exp[m];
    const bool real = m == 0 || m == g.nyq;  // irfft/rfft round trip of the reference
#pragma unroll
    for (int i = 0; i < T_; ++i)
      if (i < t.cnt)
        hm_emit<EVEN, true>(d, a[i], t.lo + i, lane, [&](int pos, float2 v) {
          v = cscale(v, ep.scale);
          if (real) v.y = 0.f;
          if (ep.fw && m <= g.M) v = cscale(v, exp2f(fe * (T.lgx[pos] + lgy)));
          b[pos * 16 + line] = v;
        });
  }
  __syncthreads();
  const int n = d.n, line = tid & 15;
  const float cw = T.sa_cw[f0 + line];
  for (int k = tid >> 4; k < n; k += blockDim.x >> 4) {
    float2 v = b[k * 16 + line];
    if (ep.sa) {
      const float w = T.sa_wx[k];
      if (w != 0.f) {
        float2 dd;
        if (k == 0) dd = cscale(csub(b[16 + line], v), ep.invdx);
        else if (k == n - 1) dd = cscale(csub(v, b[(n - 2) * 16 + line]), ep.invdx);
        else dd = cscale(csub(b[(k + 1) * 16 + line], b[(k - 1) * 16 + line]), ep.inv2dx);
        const float2 cd = make_float2(cw * dd.y, -cw * dd.x);
        const float2 pin = k < n / 2 ? cscale(cadd(v, cd), 0.5f) : cscale(csub(v, cd), 0.5f);
        v = csub(v, cscale(pin, ep.sa_strength * w));
      }
    }
    gst(base, k * sxb + line * 8u, v);
  }
}

__device__ __forceinline__ LineConst line_const(const Tables& T, const OpDesc& op, int m) {
  const double kt = T.kt[m], ka = T.ka[m];
  LineConst lc;
  lc.kt2 = kt * kt;
  lc.ka2 = ka * ka;
  lc.ktd = kt;
  lc.kt = (float)kt;
  lc.ka = (float)ka;
  lc.ald = T.alpha[m] * op.dz_att;
  lc.asd = T.astar[m] * op.dz_att;
  lc.al = (float)lc.ald;
  lc.as = (float)lc.asd;
  lc.kept = kt > 0.0;
  return lc;
}

// y-pass: forward DFT along y, the visit operator, inverse DFT.  Tile = (x, 16 f
// bins).  A lane holds positions k and n - k (for even n also h - k and h + k) of its
// line, which is the pair the inverse transform folds: the operator and the fold
// happen in registers, and only the folded rows return to LDS.  The operator is
// evaluated at every position's own wavenumber (the grids are mirror images only up
// to rounding, and one ulp decides a mode at the evanescent cutoff).
//
// TABLE: all threads first evaluate the operator into LDS, while the line is on its way.
// For one or two row tiles (n up to 126 even, 63 odd), where two or three of the four
// waves have none and a lane evaluated 8 (odd n) or 16 positions one after the other:
// 51x51x101 8.7 -> 6.7 us, 128x96x801 51.5 -> 44.2.  With four tiles it gains nothing
// (120x101x301 25.1, 24.5 us), with three the LDS costs more (164 points: 61.9, 74.6).
template <bool EVEN, int T_, bool RADIX, bool PRECISE, bool TABLE = false>
__global__ __launch_bounds__(512) void k_gy_pass(float2* __restrict__ spec, Tables T, Geom g, DftMat d, OpDesc op) {
  static_assert(!TABLE || (T_ == 1 && !RADIX));
  extern __shared__ float4 eo[];
  float2* opt = reinterpret_cast<float2*>(eo + d.Kp * 16);  // TABLE: [position][line]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, W = blockDim.x >> 6;
  const int x = blockIdx.x / g.nfb, f0 = (blockIdx.x % g.nfb) * LF;
  const uint32_t syb = (uint32_t)g.MP * 8u;
  float2* base = spec + (long)x * g.nY * g.MP + f0;
  const int line = tid & 15, m = f0 + line;  // (blockDim.x is a multiple of 16)
  const double kx = T.kx[x];
  auto visit_at = [&](const LineConst& lc, int pos) {
    const double kk = kperp2(kx, T.ky[pos]);
    if constexpr (PRECISE) return visit_operator_fp64(op, kk, lc, m);
    else return visit_operator(op, kk, lc, m);
  };
  auto ld = [&](int pos, int l) { return gld(base, pos * syb + l * 8u); };
  if constexpr (TABLE) {
    hm_fold<EVEN, false, RADIX>(eo, d, tid, blockDim.x, ld, [&] {
      const LineConst lc = line_const(T, op, m);
      for (int pos = tid >> 4; pos < d.n; pos += blockDim.x >> 4) opt[pos * 16 + line] = visit_at(lc, pos);
    });
  } else {
    hm_fold<EVEN, false, RADIX>(eo, d, tid, blockDim.x, ld);
  }
  __syncthreads();
  const Tiles t = hm_tiles(d.p * d.R, wave, W);
  LineAcc<EVEN> a[T_];
  hm_line<EVEN, T_, RADIX>(eo, d, t, lane, a);
  __syncthreads();
  {
    LineConst lc;
    if constexpr (!TABLE) lc = line_const(T, op, m);
    auto apply = [&](int pos, float2 v) {
      float2 o;
      if constexpr (TABLE) o = opt[pos * 16 + line];
      else o = visit_at(lc, pos);
      return cmul_tw<false>(v, make_float4(o.x, o.y, d.norm_lo * o.x, d.norm_lo * o.y));
    };
    // folded row of output k of residue r from the values at k and q - k
    auto put = [&](int k, int r, float2 v, float2 vn, bool pair) {
      v = apply(d.p * k + r, v);
      float4 e = make_float4(v.x, v.y, 0.f, 0.f);
      if (pair) {
        vn = apply(d.p * (d.q - k) + r, vn);
        e = make_float4(v.x + vn.x, v.y + vn.y, v.x - vn.x, v.y - vn.y);
      }
      eo[(r * d.Kp + hm_col<EVEN>(d, k)) * 16 + line] = e;
    };
#pragma unroll
    for (int i = 0; i < T_; ++i) {
      if (i < t.cnt) {
        const int r = (t.lo + i) / d.R, rt = t.lo + i - r * d.R;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int k = 16 * rt + 4 * (lane >> 4) + q;
          float2 P, Q, P2, Q2;
          hm_values<EVEN>(a[i], q, P, Q, P2, Q2);
          if (k < d.rows) {
            put(k, r, P, Q, k > 0);
            if constexpr (EVEN) {
              if (d.h - k != k) put(d.h - k, r, P2, Q2, k > 0);
            }
          }
        }
      }
    }
  }
  __syncthreads();
  hm_line<EVEN, T_, RADIX>(eo, d, t, lane, a);
  if constexpr (!RADIX) {
    const uint32_t lo = (lane & 15) * 8u;
#pragma unroll
    for (int i = 0; i < T_; ++i)
      if (i < t.cnt) hm_emit<EVEN, true>(d, a[i], t.lo + i, lane, [&](int pos, float2 v) { gst(base, pos * syb + lo, v); });
    return;
  }
  __syncthreads();
  float2* z = reinterpret_cast<float2*>(eo);
#pragma unroll
  for (int i = 0; i < T_; ++i)
    if (i < t.cnt)
      hm_emit_at<EVEN, true>(d, a[i], t.lo + i, lane, [&](int k, int r) { return r * d.q + k; },
                             [&](int pos, float2 v) { z[pos * 16 + (lane & 15)] = v; });
  __syncthreads();
  hm_combine(z, d, tid, blockDim.x, [&](int pos, int line, float2 v) { gst(base, pos * syb + line * 8u, v); });
}

// Power-weighted obliquity sums of a (kx row, f block) tile (as k_ypower): forward
// DFT along y, then sum P k/k_z and sum P over propagating modes, a pair per block.
template <bool EVEN, int T_, bool RADIX>
__global__ __launch_bounds__(512) void k_gy_power(const float2* __restrict__ spec, Tables T, Geom g, DftMat d,
                                                  double2* __restrict__ part) {
  extern __shared__ float4 eo[];
  __shared__ double sred[2][8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, W = blockDim.x >> 6;
  const int x = blockIdx.x / g.nfb, f0 = (blockIdx.x % g.nfb) * LF;
  const uint32_t syb = (uint32_t)g.MP * 8u;
  const float2* base = spec + (long)x * g.nY * g.MP + f0;
  hm_fold<EVEN, false, RADIX>(eo, d, tid, blockDim.x, [&](int pos, int line) { return gld(base, pos * syb + line * 8u); });
  __syncthreads();
  const int m = f0 + (lane & 15);
  const double km = m <= g.M ? T.ka[m] : 0.0;  // ka[0] = 0: the DC bin weighs nothing
  const double kx = T.kx[x];
  double num = 0.0, den = 0.0;
  const Tiles t = hm_tiles(d.p * d.R, wave, W);
  LineAcc<EVEN> a[T_];
  hm_line<EVEN, T_, RADIX>(eo, d, t, lane, a);
#pragma unroll
  for (int i = 0; i < T_; ++i) {
    if (i >= t.cnt) break;
    hm_emit<EVEN, false>(d, a[i], t.lo + i, lane, [&](int pos, float2 v) {
      const double ky = T.ky[pos];
      const double kz2 = kz2_of(km, kperp2(kx, ky));
      if (km > 0.0 && kz2 > 0.0) obliquity_term(v, km, kz2, num, den);
    });
  }
  for (int o = 32; o > 0; o >>= 1) {
    num += __shfl_xor(num, o, 64);
    den += __shfl_xor(den, o, 64);
  }
  if (lane == 0) { sred[0][wave] = num; sred[1][wave] = den; }
  __syncthreads();
  if (tid == 0) {
    double s0 = 0.0, s1 = 0.0;
    for (int w = 0; w < W; ++w) { s0 += sred[0][w]; s1 += sred[1][w]; }
    part[blockIdx.x] = make_double2(s0, s1);
  }
}

// y-sweep without a transform (as k_ysa) for any nY: super-absorbing y pass,
// DC/Nyquist projection and an optional phase/amplitude screen.  Tile = (x, 16 f
// bins); the rows handled (all with a screen, else the two boundary bands) sit in
// LDS, ysa_rows * 128 bytes of it.
static __global__ __launch_bounds__(256) void k_gy_sa(float2* __restrict__ spec, Tables T, Geom g, ScreenDesc s) {
  extern __shared__ float2 sbuf[];
  const int L = g.nY;
  const int tid = threadIdx.x, l = tid & 15;
  const int x = blockIdx.x / g.nfb, f0 = (blockIdx.x % g.nfb) * LF;
  float2* base = spec + (long)x * g.nY * g.MP + f0;
  const int nrows = ysa_rows(L, s.band, s.phase != nullptr);
  const bool band = nrows < L;
  auto row_of = [&](int i) { return (band && i > s.band) ? L - nrows + i : i; };
#pragma unroll 4
  for (int i = tid >> 4; i < nrows; i += 16) sbuf[i * 16 + l] = base[(long)row_of(i) * g.MP + l];
  __syncthreads();
  const int m = f0 + l;
  const float cw = s.sa ? T.sa_cw[m] : 0.f;
  const float fs = (float)m / s.f0b;
  for (int i = tid >> 4; i < nrows; i += 16) {
    const int pos = row_of(i);
    float2 u = sbuf[i * 16 + l];
    if (s.sa) {
      const float w = T.sa_wy[pos];
      if (w != 0.f) {
        float2 d;
        if (pos == 0) d = cscale(csub(sbuf[(i + 1) * 16 + l], u), s.invdy);
        else if (pos == L - 1) d = cscale(csub(u, sbuf[(i - 1) * 16 + l]), s.invdy);
        else d = cscale(csub(sbuf[(i + 1) * 16 + l], sbuf[(i - 1) * 16 + l]), s.inv2dy);
        const float2 cd = make_float2(cw * d.y, -cw * d.x);
        const float2 pin = pos < L / 2 ? cscale(cadd(u, cd), 0.5f) : cscale(csub(u, cd), 0.5f);
        u = csub(u, cscale(pin, s.sa_strength * w));
      }
    }
    if (m == 0 || m == g.nyq) u.y = 0.f;
    if (s.phase) {
      const long idx = (long)x * g.nY + pos;
      const float th = s.phase[idx] * fs;
      float sn, cs;
      sincosf(th, &sn, &cs);
      u = cmul(u, make_float2(cs, -sn));
      if (s.amp) {
        const float amp = fminf(fmaxf(s.amp[idx], 1e-6f), 1.f);
        u = cscale(u, powf(amp, fs));
      }
      if (m == 0 || m == g.nyq) u.y = 0.f;
    }
    if (m <= g.M) base[(long)pos * g.MP + l] = u;
  }
}

// ---------------------------------------------------------------------------
// General-length t columns: one block takes 16 columns, the 16 output columns of
// a matrix-core product.  irfft and rfft are the real halves of the folded DFT:
//   inverse  C_t = sum_m a_m Re X_m cos, S_t = sum_m a_m Im X_m sin (a_0 = a_{nT/2}
//            = 1, else 2), u_t = (C_t - S_t) / nT, u_{nT-t} = (C_t + S_t) / nT;
//   forward  X_m = sum e_t cos - i sum o_t sin, e_t = u_t + u_{nT-t}, o_t = u_t - u_{nT-t}.
// Each column is a product column of its own: nothing of one reaches another.  A
// column keeps one LDS row in three forms: spectrum X[m] (float2), samples U[t] (float,
// skewed by one word per S samples so that lanes with S contiguous samples each fall
// in distinct banks) and folded samples E[t] = (e_t, o_t) (float2).  Each wave runs the
// real-space stage (column_realspace) on its 16 / W columns, lane ln with the S
// contiguous samples from S ln; the t taper is applied where the inverse writes U.
// The accumulators of a transform wait in registers for the barrier before the rows
// change form.  Semantics of the transforms (ASS:664, :685): the inverse ignores the
// imaginary parts of the DC bin and, for even nT, of the Nyquist bin; the forward
// writes them as zero.
// nT = p q with an odd radix p goes through the p residues r of the bin (or the p
// subsequences of the samples) as the lines do.  Residue 0 is the q-point transform of
// real samples, residues r and p - r are mirror images, so 1 <= r <= p/2 are complex
// q-point transforms and the others are not formed.  A row then holds the folded input
// as float2[Kp] of residue 0 and float4[Kp] of each other, and the inverse's output as
// q real and p/2 times q complex values before the radix stage.
// Per sample that is nT flops per transform (odd nT) or nT/2 (even), a p-th of it after a
// radix stage.  Without one the matrix cores bound the pass (96 TFLOP/s at nT = 1201);
// with one the vector work between the products does (at 365x365x425 the taper pass
// takes 363 us, 613 without the radix 5, of which the products are about 80).  The row
// pitch is an odd multiple of 8 floats: the 16 columns x 4 positions of an operand read
// fall in distinct banks.
// ---------------------------------------------------------------------------
constexpr int GC_COLS = 16;
constexpr int gcol_waves(int S) { return S == 2 ? 4 : 8; }
// row tiles per wave: nT <= 64 S has at most 2 S tiles (odd) or S + 1 (even)
constexpr int gcol_tiles(int S, bool even) {
  return ((even ? S + 1 : 2 * S) + gcol_waves(S) - 1) / gcol_waves(S);
}
// and with a radix stage (p > 1; p/2 + 1 residues of R tiles), over all lengths that take one
constexpr int gcol_radix_tiles(int S, bool even) {
  return S == 32 ? (even ? 3 : 6) : S == 16 ? (even ? 2 : 3) : (even ? 1 : 2);
}
// floats per row: nT/2 + 16 float2 (15 zeros stand under the matrix padding; with a radix
// p Kp float2 and the nT/2 + 1 bins) and nT + nT/S skewed samples
__host__ __device__ inline int gcol_pitch(const DftMat& d, int S) {
  const int x = d.p == 1 ? 2 * (d.n / 2 + 16) : 2 * d.p * d.Kp, b = 2 * (d.n / 2 + 1) + 2, u = d.n + d.n / S + 2;
  const int m = x > b ? x : b;
  return ((m > u ? m : u) + 7) / 16 * 16 + 8;
}

template <bool EVEN>
struct ColAcc {
  static constexpr int NP = EVEN ? 2 : 1;
  f32x4 c[NP], s[NP];
};

// One row tile of the column `in` (float2 rows, zero past position n/2).
template <bool EVEN>
__device__ __forceinline__ void hm_col_tile(const DftMat& d, int rt, int lane, const float2* in, ColAcc<EVEN>& a) {
  constexpr int ST = EVEN ? 2 : 1;  // positions of one parity
  constexpr int U = 4;
#pragma unroll
  for (int p = 0; p < ColAcc<EVEN>::NP; ++p) {
    const int gp = p == 0 ? 0 : d.Ke / 8, ng = (p == 0 ? d.Ke : d.Kp - d.Ke) / 8;
    const float4* ap = d.A + (long)rt * d.rs + gp * d.gs + lane;
    const float2* bp = in + p + ST * (lane >> 4);
    a.c[p] = a.s[p] = f32x4{0.f, 0.f, 0.f, 0.f};
    float4 w[U];
    float2 b[U][2];
    hm_ring<U>(
        ng,
        [&](int q, int g) {
          w[q] = ap[g * d.gs];
          b[q][0] = bp[g * 8 * ST];
          b[q][1] = bp[g * 8 * ST + 4 * ST];
        },
        [&](int q) {
          a.c[p] = mfma4(w[q].x, b[q][0].x, a.c[p]);
          a.s[p] = mfma4(w[q].y, b[q][0].y, a.s[p]);
          a.c[p] = mfma4(w[q].z, b[q][1].x, a.c[p]);
          a.s[p] = mfma4(w[q].w, b[q][1].y, a.s[p]);
        });
  }
}
template <bool EVEN, int TW>
__device__ __forceinline__ void hm_col(const DftMat& d, const Tiles& t, int lane, const float2* in, ColAcc<EVEN> (&a)[TW]) {
#pragma unroll
  for (int i = 0; i < TW; ++i)
    if (i < t.cnt) hm_col_tile<EVEN>(d, t.lo + i, lane, in, a[i]);
}

// f(position k <= n/2, C_k, S_k) for every output of this lane in one tile
template <bool EVEN, class F>
__device__ __forceinline__ void hm_col_emit(const DftMat& d, const ColAcc<EVEN>& a, int rt, int lane, F f) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int k = 16 * rt + 4 * (lane >> 4) + i;
    if (k >= d.rows) continue;
    if constexpr (EVEN) {
      f(k, a.c[0][i] + a.c[1][i], a.s[0][i] + a.s[1][i]);
      if (d.h - k != k) f(d.h - k, a.c[0][i] - a.c[1][i], a.s[1][i] - a.s[0][i]);
    } else {
      f(k, a.c[0][i], a.s[0][i]);
    }
  }
}

// --- radix stage of the columns (p = P) -----------------------------------------
// offset of residue r in the folded row and of its q values before the inverse's radix
// stage, in floats
__device__ __forceinline__ int ct_fold_off(const DftMat& d, int r) { return r == 0 ? 0 : (4 * r - 2) * d.Kp; }
__device__ __forceinline__ int ct_z_off(const DftMat& d, int r) { return r == 0 ? 0 : ((d.q + 1) & ~1) + (r - 1) * 2 * d.q; }

// Bin m (0 <= m < n) of a real column's spectrum: stored up to n/2, mirrored past it.
__device__ __forceinline__ float2 column_bin(const float2* sc, int m, const Geom& g, int sel, const float2* ref) {
  const int i = m <= g.M ? m : g.nT - m;
  float2 x = sc[i];
  const bool real = i == 0 || i == g.nyq;
  if (real) x.y = 0.f;
  x = tof_bin(sel, i, x, g.nyq, ref);
  if (real) x.y = 0.f;
  return m <= g.M ? x : cconj(x);
}

// Spectrum -> folded row, for the inverse.
template <bool EVEN, int P>
__device__ __forceinline__ void ct_fold_bins(float* row, const float2* sc, const DftMat& d, const Geom& g, int sel,
                                             const float2* ref, int lane) {
  for (int rr = lane; rr < d.Kp; rr += 64) {
    const int j = hm_pos<EVEN>(d, rr), jj = min(j, d.h);
    const bool pad = j > d.h, pair = !pad && j > 0 && 2 * j != d.q;
    float2 x[P / 2 + 1], y[P / 2 + 1];
    x[0] = column_bin(sc, P * jj, g, sel, ref);
#pragma unroll
    for (int r = 1; r <= P / 2; ++r) {
      x[r] = column_bin(sc, P * jj + r, g, sel, ref);
      y[r] = column_bin(sc, pair ? P * (d.q - jj) + r : r, g, sel, ref);
    }
    const float f = pad ? 0.f : (j == 0 || 2 * P * j == d.n) ? 1.f : 2.f;
    reinterpret_cast<float2*>(row)[rr] = pad ? make_float2(0.f, 0.f) : cscale(x[0], f);
#pragma unroll
    for (int r = 1; r <= P / 2; ++r) {
      float4 v = make_float4(x[r].x, x[r].y, 0.f, 0.f);
      if (pair) v = make_float4(x[r].x + y[r].x, x[r].y + y[r].y, x[r].x - y[r].x, x[r].y - y[r].y);
      if (pad) v = make_float4(0.f, 0.f, 0.f, 0.f);
      reinterpret_cast<float4*>(row + ct_fold_off(d, r))[rr] = v;
    }
  }
}

// The inverse's radix stage: x_{s + q m} = z_0[s] + 2 Re sum_{r <= P/2} W_P^{-m r} W_n^{-s r}
// z_r[s], scaled and tapered, from the row's z values to its skewed samples (the wave
// reads the row whole before it writes).
template <int S, int P>
__device__ __forceinline__ void ct_combine(float* row, const DftMat& d, float2 invN, const float* tt, int lane) {
  using C = OddTrig<P>;
  constexpr int H = P / 2, NI = (S + P - 1) / P;
  float v[NI][P];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int s = lane + 64 * i;
    if (s < d.q) {
      const float z0 = row[s];
      float2 y[H];
      float sum = 0.f;
#pragma unroll
      for (int r = 1; r <= H; ++r) {
        const float2 z = reinterpret_cast<const float2*>(row + ct_z_off(d, r))[s];
        y[r - 1] = cmul_tw<true>(z, d.tw[s * r]);
        sum += y[r - 1].x;
      }
      v[i][0] = fmaf(2.f, sum, z0);
#pragma unroll
      for (int m = 1; m <= H; ++m) {
        float A = 0.f, B = 0.f;
#pragma unroll
        for (int r = 1; r <= H; ++r) {
          const int j = (m * r) % P, jj = j > H ? P - j : j;
          if (jj == 0) {
            A += y[r - 1].x;
          } else {
            A += by_pair(y[r - 1].x, make_float2(C::ch[jj - 1], C::cl[jj - 1]));
            const float b = by_pair(y[r - 1].y, make_float2(C::sh[jj - 1], C::sl[jj - 1]));
            B += j > H ? -b : b;
          }
        }
        v[i][m] = fmaf(2.f, A - B, z0);
        v[i][P - m] = fmaf(2.f, A + B, z0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // one round's temporaries at a time
  }
  wave_sync();
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int s = lane + 64 * i;
    if (s < d.q) {
#pragma unroll
      for (int m = 0; m < P; ++m) {
        const int t = s + d.q * m;
        float x = by_pair(v[i][m], invN);
        if (tt) x *= tt[t];
        row[t + t / S] = x;
      }
    }
  }
}

// Samples -> folded row, for the forward transform: y_r[s] = W_n^{s r} sum_m u_{s + q m}
// W_P^{m r}, r <= P/2, folded over s and q - s; this is the sum over m.
template <int P>
__device__ __forceinline__ void ct_sample_dft(const float* u, float2* y) {
  using C = OddTrig<P>;
  constexpr int H = P / 2;
  float a[H], b[H], sum = u[0];
#pragma unroll
  for (int m = 1; m <= H; ++m) {
    a[m - 1] = u[m] + u[P - m];
    b[m - 1] = u[m] - u[P - m];
    sum += a[m - 1];
  }
  y[0] = make_float2(sum, 0.f);
#pragma unroll
  for (int r = 1; r <= H; ++r) {
    float A = u[0], B = 0.f;
#pragma unroll
    for (int m = 1; m <= H; ++m) {
      const int j = (m * r) % P, jj = j > H ? P - j : j;
      if (jj == 0) {
        A += a[m - 1];
      } else {
        A += by_pair(a[m - 1], make_float2(C::ch[jj - 1], C::cl[jj - 1]));
        const float w = by_pair(b[m - 1], make_float2(C::sh[jj - 1], C::sl[jj - 1]));
        B += j > H ? -w : w;
      }
    }
    y[r] = make_float2(A, -B);
  }
}
// rounds of 64 matrix columns of a q-point transform, q <= 64 S / P
constexpr int ct_rounds(int S, int P) {
  int most = 0;
  for (int q = 64 * S / P - 1; q <= 64 * S / P; ++q) {
    const int h = q / 2;
    const int kp = q % 2 ? (h + 8) / 8 * 8 : (h / 2 + 8) / 8 * 8 + ((h + 1) / 2 + 7) / 8 * 8;
    if (kp > most) most = kp;
  }
  return (most + 63) / 64;
}
template <int S, bool EVEN, int P>
__device__ __forceinline__ void ct_fold_samples(float* row, const DftMat& d, int lane) {
  constexpr int H = P / 2, NF = ct_rounds(S, P);
  float2 e0[NF];  // residue 0
  float4 v[NF][H];
#pragma unroll
  for (int i = 0; i < NF; ++i) {
    const int rr = lane + 64 * i;
    if (rr < d.Kp) {
      const int j = hm_pos<EVEN>(d, rr), jj = min(j, d.h);
      const bool pad = j > d.h, pair = !pad && j > 0 && 2 * j != d.q;
      const int s1 = pair ? d.q - jj : jj;
      float a[P], b[P];
#pragma unroll
      for (int m = 0; m < P; ++m) {
        const int t0 = jj + d.q * m, t1 = s1 + d.q * m;
        a[m] = row[t0 + t0 / S];
        b[(m + 1) % P] = row[t1 + t1 / S];
      }
      float2 x[H + 1], y[H + 1];
      ct_sample_dft<P>(a, x);
      ct_sample_dft<P>(b, y);
#pragma unroll
      for (int r = 1; r <= H; ++r) {
        const float4 w = d.tw[jj * r];
        x[r] = cmul_tw<false>(x[r], w);
        y[r] = cmul_tw<true>(y[r], w);
      }
      e0[i] = make_float2(pad ? 0.f : pair ? x[0].x + y[0].x : x[0].x, pair ? x[0].x - y[0].x : 0.f);
#pragma unroll
      for (int r = 1; r <= H; ++r) {
        float4 w = make_float4(x[r].x, x[r].y, 0.f, 0.f);
        if (pair) w = make_float4(x[r].x + y[r].x, x[r].y + y[r].y, x[r].x - y[r].x, x[r].y - y[r].y);
        if (pad) w = make_float4(0.f, 0.f, 0.f, 0.f);
        v[i][r - 1] = w;
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // one round's temporaries at a time
  }
  wave_sync();
#pragma unroll
  for (int i = 0; i < NF; ++i) {
    const int rr = lane + 64 * i;
    if (rr < d.Kp) {
      reinterpret_cast<float2*>(row)[rr] = e0[i];
#pragma unroll
      for (int r = 1; r <= H; ++r) reinterpret_cast<float4*>(row + ct_fold_off(d, r))[rr] = v[i][r - 1];
    }
  }
}

// One row tile of residue r of the folded column `row`.
template <bool EVEN>
__device__ __forceinline__ void ct_tile(const DftMat& d, int r, int rt, int lane, const float* row, LineAcc<EVEN>& a) {
  constexpr int U = 4;
#pragma unroll
  for (int p = 0; p < LineAcc<EVEN>::NP; ++p) {
    const int gp = p == 0 ? 0 : d.Ke / 8, ng = (p == 0 ? d.Ke : d.Kp - d.Ke) / 8;
    const float4* ap = d.A + (long)rt * d.rs + gp * d.gs + lane;
#pragma unroll
    for (int q = 0; q < 2; ++q) a.c[p][q] = a.s[p][q] = f32x4{0.f, 0.f, 0.f, 0.f};
    float4 w[U];
    if (r == 0) {
      const float2* bp = reinterpret_cast<const float2*>(row) + gp * 8 + (lane >> 4);
      float2 b[U][2];
      hm_ring<U>(
          ng,
          [&](int q, int g) {
            w[q] = ap[g * d.gs];
            b[q][0] = bp[g * 8];
            b[q][1] = bp[g * 8 + 4];
          },
          [&](int q) {
            a.c[p][0] = mfma4(w[q].x, b[q][0].x, a.c[p][0]);
            a.s[p][0] = mfma4(w[q].y, b[q][0].y, a.s[p][0]);
            a.c[p][0] = mfma4(w[q].z, b[q][1].x, a.c[p][0]);
            a.s[p][0] = mfma4(w[q].w, b[q][1].y, a.s[p][0]);
          });
    } else {
      const float4* bp = reinterpret_cast<const float4*>(row + ct_fold_off(d, r)) + gp * 8 + (lane >> 4);
      float4 b[U][2];
      hm_ring<U>(
          ng,
          [&](int q, int g) {
            w[q] = ap[g * d.gs];
            b[q][0] = bp[g * 8];
            b[q][1] = bp[g * 8 + 4];
          },
          [&](int q) {
            a.c[p][0] = mfma4(w[q].x, b[q][0].x, a.c[p][0]);
            a.c[p][1] = mfma4(w[q].x, b[q][0].y, a.c[p][1]);
            a.s[p][0] = mfma4(w[q].y, b[q][0].z, a.s[p][0]);
            a.s[p][1] = mfma4(w[q].y, b[q][0].w, a.s[p][1]);
            a.c[p][0] = mfma4(w[q].z, b[q][1].x, a.c[p][0]);
            a.c[p][1] = mfma4(w[q].z, b[q][1].y, a.c[p][1]);
            a.s[p][0] = mfma4(w[q].w, b[q][1].z, a.s[p][0]);
            a.s[p][1] = mfma4(w[q].w, b[q][1].w, a.s[p][1]);
          });
    }
  }
}

// CALL with P = d.p
#define CT_DISPATCH(d, CALL)                        \
  switch ((d).p) {                                  \
    case 3: { constexpr int P = 3; CALL; } break;   \
    case 5: { constexpr int P = 5; CALL; } break;   \
    case 7: { constexpr int P = 7; CALL; } break;   \
    default: { constexpr int P = 9; CALL; } break;  \
  }

// two blocks per CU and more for up to 1024 samples (four waves per SIMD); the FP64 tone
// burst and the longest rows take what they need
constexpr int gcol_waves_per_simd(int S, bool radix, int mode) { return radix && S <= 16 && mode != COL_INJECT && mode != COL_TOF ? 4 : 1; }

template <int S, bool EVEN, bool RADIX, int MODE, int NLK>
__global__ __launch_bounds__(64 * gcol_waves(S), gcol_waves_per_simd(S, RADIX, MODE)) void k_gcolumn(float2* __restrict__ spec, Tables T, Geom g, DftMat dm, ColDesc d) {
  constexpr int W = gcol_waves(S), TW = RADIX ? gcol_radix_tiles(S, EVEN) : gcol_tiles(S, EVEN), NC = GC_COLS / W;
  extern __shared__ float4 glds[];
  __shared__ float s_red[W];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int nT = g.nT, M = g.M, ncols = g.nX * g.nY;
  const Tiles tiles = hm_tiles(RADIX ? (dm.p / 2 + 1) * dm.R : dm.R, wave, W);
  const int pitch = gcol_pitch(dm, S);
  float* rows = reinterpret_cast<float*>(glds);
  auto skew = [](int t) { return t + t / S; };
  const int c0 = blockIdx.x * GC_COLS;
  const int t0 = lane * S;
  const float2 invN = inverse_pair(nT);
  constexpr bool spectral_in = MODE != COL_LOAD && MODE != COL_INJECT;
  constexpr bool rewrite = (MODE == COL_NL || MODE == COL_TAPER || MODE == COL_LOAD || MODE == COL_INJECT);
  constexpr bool FIN = MODE == COL_FINAL;
  constexpr bool tapered = (MODE == COL_NL || MODE == COL_TAPER || MODE == COL_MAXABS);
  const float* tt = tapered && d.taper ? (d.taper == 1 ? T.tapt_h : T.tapt_f) : nullptr;
  const LaneCol<S, 64, false, true> lc{lane, lane, t0, nT};
  const int row = (FIN || MODE == COL_TOF) ? *d.row : 0;
  const double Nn = d.nscale ? d.N * (d.nscale[0] / (d.nscale[1] + 1e-30)) : d.N;
  if (MODE == COL_NL && d.row && blockIdx.x == 0 && tid == 0) *d.row += 1;
  float wmax = 0.f;
  int nsub_global = 1;
  if constexpr (NLK != NL_NONE) {
    if (d.subcycle == SUBCYCLE_GLOBAL) {
      const float gm = __uint_as_float(*d.gmax);
      bool capped;
      nsub_global = substeps_for(Nn * (double)gm * d.dz / d.dT, (double)d.cfl_target, gm, &capped);
      if (capped && blockIdx.x == 0 && tid == 0 && d.subcap) atomicAdd(d.subcap, 1u);
    }
  }
  // inverse transform of the block's columns (bins modified by tof_bin(sel)) into U
  auto inverse = [&](int sel) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int col = wave * NC + i, c = c0 + col;
      if (c < ncols) {
        const float2* sc = spec + (long)c * g.MP;
        if constexpr (RADIX) {
          CT_DISPATCH(dm, (ct_fold_bins<EVEN, P>(rows + col * pitch, sc, dm, g, sel, d.tofref, lane)));
          continue;
        }
        float2* X = reinterpret_cast<float2*>(rows + col * pitch);
#pragma unroll 4
        for (int m = lane; m < M + 16; m += 64) {
          float2 x = sc[min(m, M)];
          const bool real = m == 0 || m == g.nyq;
          if (real) x.y = 0.f;
          x = tof_bin(sel, m, x, g.nyq, d.tofref);
          if (real) x.y = 0.f;
          const float f = m > M ? 0.f : real ? 1.f : 2.f;
          X[m] = m > M ? make_float2(0.f, 0.f) : cscale(x, f);
        }
      }
    }
    __syncthreads();
    float* uc = rows + (lane & 15) * pitch;
    if constexpr (RADIX) {
      LineAcc<EVEN> a[TW];
#pragma unroll
      for (int i = 0; i < TW; ++i)
        if (i < tiles.cnt) {
          const int r = (tiles.lo + i) / dm.R;
          ct_tile<EVEN>(dm, r, tiles.lo + i - r * dm.R, lane, uc, a[i]);
        }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < TW; ++i)
        if (i < tiles.cnt) {
          const int r = (tiles.lo + i) / dm.R;
          float* z = uc + ct_z_off(dm, r);
          hm_emit_at<EVEN, true>(dm, a[i], tiles.lo + i, lane, [](int k, int) { return k; }, [&](int k, float2 v) {
            if (r == 0) z[k] = v.x - v.y;
            else reinterpret_cast<float2*>(z)[k] = v;
          });
        }
      __syncthreads();
#pragma unroll 1
      for (int i = 0; i < NC; ++i)
        CT_DISPATCH(dm, (ct_combine<S, P>(rows + (wave * NC + i) * pitch, dm, invN, tapered ? tt : nullptr, lane)));
      wave_sync();  // (each wave reads on only its own columns)
      return;
    }
    ColAcc<EVEN> a[RADIX ? 1 : TW];
    if constexpr (!RADIX) hm_col<EVEN, TW>(dm, tiles, lane, reinterpret_cast<const float2*>(uc), a);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (RADIX ? 0 : TW); ++i)
      if (i < tiles.cnt)
        hm_col_emit<EVEN>(dm, a[i], tiles.lo + i, lane, [&](int t, float C, float Sn) {
          float v = by_pair(C - Sn, invN);
          if (tapered && tt) v *= tt[t];
          uc[skew(t)] = v;
          if (t > 0 && 2 * t != nT) {
            float w = by_pair(C + Sn, invN);
            if (tapered && tt) w *= tt[nT - t];
            uc[skew(nT - t)] = w;
          }
        });
    __syncthreads();
  };
  auto samples = [&](float (&u)[S], const float* uc) {
#pragma unroll
    for (int i = 0; i < S; ++i) u[i] = t0 + i < nT ? uc[lane * (S + 1) + i] : 0.f;
  };

  if constexpr (MODE == COL_TOF) {
    // the field (envelope: and its Hilbert transform) or its correlation with the reference
    float u[NC][S];
    inverse(d.tof_mode == TOF_ENVELOPE ? 0 : 2);
#pragma unroll
    for (int i = 0; i < NC; ++i) samples(u[i], rows + (wave * NC + i) * pitch);
    if (d.tof_mode == TOF_ENVELOPE) {
      __syncthreads();
      inverse(1);
    }
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int col = wave * NC + i, c = c0 + col;
      if (c >= ncols) continue;
      float uq[S];
      samples(uq, rows + col * pitch);
      wave_sync();
      const bool nz = spectrum_nonzero<64>(spec + (long)c * g.MP, M, lane);
      column_tof<S, 64, false, true>(u[i], uq, lc, rows + col * pitch, d, c, true, ncols, row, nz);
    }
    return;
  } else {
    if constexpr (spectral_in) inverse(0);
    if constexpr (MODE == COL_INJECT) {
      bool any = false;
      for (int c = c0; c < min(c0 + GC_COLS, ncols); ++c) any = any || column_has_source(d, c);
      if (!any) return;
    }
#pragma unroll 1
    for (int i = 0; i < NC; ++i) {
      const int col = wave * NC + i, c = c0 + col;
      if (c >= ncols) break;
      float* uc = rows + col * pitch;
      if constexpr (MODE == COL_LOAD) {
        const float* src = d.rin + (long)c * nT;
        float mx = 0.f;
        double e2 = 0.0;
#pragma unroll
        for (int q = 0; q < S; ++q) {
          const int t = lane + 64 * q;
          const float v = t < nT ? src[t] : 0.f;
          mx = fmaxf(mx, fabsf(v));
          e2 += (double)v * (double)v;
          if (t < nT) uc[skew(t)] = v;
        }
        for (int o = 32; o > 0; o >>= 1) e2 += __shfl_xor(e2, o, 64);
        if (lane == 0 && d.ibefore) d.ibefore[c] = e2;
        wmax = fmaxf(wmax, mx);
        wave_sync();
      } else if constexpr (MODE == COL_INJECT) {
        const bool src = column_has_source(d, c);
#pragma unroll 1
        for (int t = lane; t < nT; t += 64) uc[skew(t)] = src ? source_sample(d, c, nT, t) : 0.f;
        wave_sync();
      } else if constexpr (MODE == COL_STORE) {
        float* dst = d.rout + (long)c * nT;
        for (int t = lane; t < nT; t += 64) dst[t] = uc[skew(t)];
      } else if constexpr (MODE == COL_MAXABS) {
        for (int t = lane; t < nT; t += 64) wmax = fmaxf(wmax, fabsf(uc[skew(t)]));
      } else if constexpr (MODE != COL_TAPER) {
        float u[S];
        samples(u, uc);
        if constexpr (MODE == COL_NL) {
          ColDesc dr = d;  // (the taper is in U already)
          dr.taper = 0;
          column_realspace<S, 64, false, true, MODE, NLK>(u, lc, dr, T, c, true, ncols, row, Nn, nsub_global, wmax);
        } else {
          column_realspace<S, 64, false, true, MODE, NLK>(u, lc, d, T, c, true, ncols, row, Nn, nsub_global, wmax);
        }
        if constexpr (rewrite) {
          wave_sync();
#pragma unroll
          for (int q = 0; q < S; ++q)
            if (t0 + q < nT) uc[lane * (S + 1) + q] = u[q];
          wave_sync();
        }
      }
      if constexpr (rewrite && RADIX) {
        CT_DISPATCH(dm, (ct_fold_samples<S, EVEN, P>(uc, dm, lane)));
      } else if constexpr (rewrite) {
        // U -> E (the row is read whole before it is written)
        constexpr int NF = S / 2 + 1;  // positions 0 .. M + 15 <= 32 S + 15, 64 per round
        float2 e[NF];
#pragma unroll
        for (int q = 0; q < NF; ++q) {
          const int t = lane + 64 * q;
          e[q] = make_float2(0.f, 0.f);
          if (t <= M) {
            const float v = uc[skew(t)];
            const bool pair = t > 0 && 2 * t != nT;
            const float w = pair ? uc[skew(nT - t)] : 0.f;
            e[q] = make_float2(v + w, pair ? v - w : 0.f);
          }
        }
        wave_sync();
        float2* E = reinterpret_cast<float2*>(uc);
#pragma unroll
        for (int q = 0; q < NF; ++q)
          if (lane + 64 * q < M + 16) E[lane + 64 * q] = e[q];
      }
    }
    if constexpr (rewrite) {
      __syncthreads();
      float* ec = rows + (lane & 15) * pitch;
      float2* xc = reinterpret_cast<float2*>(ec);
      if constexpr (RADIX) {
        LineAcc<EVEN> a[TW];
#pragma unroll
        for (int i = 0; i < TW; ++i)
          if (i < tiles.cnt) {
            const int r = (tiles.lo + i) / dm.R;
            ct_tile<EVEN>(dm, r, tiles.lo + i - r * dm.R, lane, ec, a[i]);
          }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < TW; ++i)
          if (i < tiles.cnt)
            hm_emit<EVEN, false>(dm, a[i], tiles.lo + i, lane, [&](int m, float2 v) {
              // (past nT/2: the mirrored bin, of another residue; residue 0 forms it itself)
              if (m == 0 || m == g.nyq) v.y = 0.f;
              if (m <= M) xc[m] = v;
              else if (tiles.lo + i >= dm.R) xc[nT - m] = cconj(v);
            });
      } else {
        ColAcc<EVEN> a[TW];
        hm_col<EVEN, TW>(dm, tiles, lane, xc, a);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < TW; ++i)
          if (i < tiles.cnt)
            hm_col_emit<EVEN>(dm, a[i], tiles.lo + i, lane, [&](int m, float C, float Sn) {
              xc[m] = make_float2(C, (m == 0 || m == g.nyq) ? 0.f : -Sn);
            });
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < NC; ++i) {
        const int col = wave * NC + i, c = c0 + col;
        if (c < ncols) {
          float2* sc = spec + (long)c * g.MP;
          const float2* X = reinterpret_cast<const float2*>(rows + col * pitch);
          if (MODE == COL_INJECT && !column_has_source(d, c)) continue;
          for (int m = lane; m <= M; m += 64) sc[m] = MODE == COL_INJECT ? cadd(sc[m], X[m]) : X[m];
        }
      }
    }
    if constexpr (FIN || MODE == COL_LOAD || MODE == COL_MAXABS) {
      if (MODE != COL_MAXABS && !d.stats) return;
      for (int o = 32; o > 0; o >>= 1) wmax = fmaxf(wmax, __shfl_xor(wmax, o, 64));
      if (lane == 0) s_red[wave] = wmax;
      __syncthreads();
      if (tid == 0) {
        float m = s_red[0];
        for (int k = 1; k < W; ++k) m = fmaxf(m, s_red[k]);
        if constexpr (MODE == COL_MAXABS) {
          d.partial[blockIdx.x] = __float_as_uint(m);
        } else {
          unsigned* slot = FIN ? d.stats + row + 1 : d.stats;
          if (!FIN || row < d.max_rows) atomicMax(slot, __float_as_uint(m));
        }
      }
    }
  }
}

// Nonlinear update of real columns of any length (COL_RAWNL, no transform): one wave
// per column, lane ln holds the S contiguous samples from S ln.  Columns pass through
// LDS, so that memory sees whole rows (128x96x801: 72 -> 17-25 us, KT 55).
constexpr int GR_WPB = 4;
template <int S, int NLK>
__global__ __launch_bounds__(64 * GR_WPB) void k_gcolumn_raw(Tables T, Geom g, ColDesc d) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nT = g.nT, ncols = g.nX * g.nY, t0 = lane * S;
  const LaneCol<S, 64, false, true> lc{lane, lane, t0, nT};
  __shared__ float rows[GR_WPB][64 * (S + 1)];  // sample t at t + t/S: a lane's samples start in its own bank
  float* row = rows[wave];
  const double Nn = d.nscale ? d.N * (d.nscale[0] / (d.nscale[1] + 1e-30)) : d.N;
  float wmax = 0.f;
  int nsub_global = 1;
  if constexpr (NLK != NL_NONE) {
    if (d.subcycle == SUBCYCLE_GLOBAL) {
      const float gm = __uint_as_float(*d.gmax);
      bool capped;
      nsub_global = substeps_for(Nn * (double)gm * d.dz / d.dT, (double)d.cfl_target, gm, &capped);
      if (capped && blockIdx.x == 0 && threadIdx.x == 0 && d.subcap) atomicAdd(d.subcap, 1u);
    }
  }
  for (int c = blockIdx.x * GR_WPB + wave; c < ncols; c += gridDim.x * GR_WPB) {
    if (d.cflag && d.cflag[c] == 0) continue;
    const float* src = d.rin + (long)c * nT;
    float u[S];
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int t = lane + 64 * i;
      u[i] = t < nT ? src[t] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < S; ++i) row[lane + 64 * i + (lane + 64 * i) / S] = u[i];
    wave_sync();
#pragma unroll
    for (int i = 0; i < S; ++i) u[i] = row[t0 + i + lane];
    column_realspace<S, 64, false, true, COL_RAWNL, NLK>(u, lc, d, T, c, true, ncols, 0, Nn, nsub_global, wmax);
    float* dst = d.rout + (long)c * nT;
#pragma unroll
    for (int i = 0; i < S; ++i) row[t0 + i + lane] = u[i];
    wave_sync();
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int t = lane + 64 * i;
      if (t < nT) dst[t] = row[t + t / S];
    }
    wave_sync();
  }
}

}  // namespace ash
