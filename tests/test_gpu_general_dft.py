"""The matrix-core DFTs of the general-size kernels at the sizes where their tiling
can go wrong: the smallest lengths, one position around every 16-row tile and 8-column
group, even lengths whose quarter is on and off a tile edge, the last length of every
tiles-per-wave and samples-per-lane class, lengths that take a radix stage first, and
the longest lines and columns.

Against the FP64 oracle, rel-L2.  A length-n line sums n/2 float32 products per output,
relative rounding error at most 6e-8 sqrt(n/2) in the root mean square; an operator
runs at most four line and two column transforms, so the sum in quadrature over the
longest shape here (1000 + 1023 lines, 2047 samples) stays below 6e-8 sqrt(2 * 511 +
2 * 511 + 1024) = 3.4e-6.  The bound is the general kernels' 5e-6.
"""
import numpy as np
import pytest

from oracle import asm_oracle as O
from tests.conftest import rel_l2
from tests.test_gpu_ops import _dev, _field, _params, _plan

pytestmark = pytest.mark.gpu

SHAPES = [(2, 3, 4), (3, 2, 5), (15, 16, 7), (17, 31, 15), (32, 33, 31), (30, 34, 32), (62, 63, 33), (66, 65, 62),
          (5, 6, 127), (6, 5, 128), (5, 4, 129), (4, 5, 255), (5, 6, 258), (6, 5, 511), (4, 3, 513), (3, 4, 1022),
          (4, 3, 1025), (3, 4, 1536), (5, 4, 2047), (126, 127, 9), (130, 129, 8), (254, 255, 6), (258, 257, 5),
          (382, 385, 4), (511, 514, 4), (1000, 3, 16), (3, 1023, 17), (1024, 5, 8), (6, 1022, 8), (1023, 2, 6),
          # lines that take a radix 3, 5, 7 or 9 first, odd and even quotients
          (129, 132, 5), (135, 130, 6), (133, 140, 5), (252, 245, 4), (365, 366, 4), (385, 147, 5), (990, 7, 6),
          (7, 1001, 5), (1008, 4, 6),
          # y passes that take the operator from a table: one and two row tiles, and the
          # first length past them
          (5, 60, 9), (3, 62, 6), (3, 64, 5), (7, 124, 18), (5, 126, 6), (4, 61, 33),
          # y passes with a power-of-two or 3 2^k line: one x row a block up to 768 pairs, else two
          (46, 64, 1024), (48, 64, 1024), (2, 384, 256), (2, 192, 512), (6, 128, 256),
          # and columns (with 16 columns to a block, some blocks partly filled)
          (5, 4, 129), (4, 5, 130), (3, 7, 133), (5, 5, 135), (6, 5, 189), (7, 5, 252), (5, 7, 300), (4, 5, 301),
          (5, 9, 425), (4, 4, 510), (3, 5, 513), (5, 4, 801), (4, 5, 1010), (3, 6, 1022), (5, 4, 1035), (4, 5, 1200),
          (3, 7, 1995), (4, 4, 2043), (5, 4, 2044), (4, 5, 2045), (3, 4, 2046)]


@pytest.mark.parametrize("shape", SHAPES)
def test_general_transforms_match_oracle(shape):
    p = _params(shape, useFreqWeightedBoundary=True, useSuperAbsorbing=True)
    nX, nY, nT = shape
    dz = 3.08e-4
    u = _field(shape)
    u64 = u.astype(np.float64)
    plan = _plan(shape, p, dz)
    x = _dev(u)
    got = {"attenuation": plan.attenuation_step(x, 0.5), "propagator": plan.angular_spectrum_step(x, True),
           "freq_weighted": plan.freq_weighted_boundary_step(x), "super_absorbing": plan.super_absorbing_step(x)}
    _, afh, _, _, _ = O.precalculate_ad_pow2(p.alpha0, nX, nY, nT, p.dX, p.dY, dz, p.dT, p.c0, p.f0,
                                             p.attenPow, split_step=True, n_bins=nT // 2 + 1)
    _, HHh = O.precalculate_mas(nX, nY, nT, p.dX, p.dY, dz, p.dT, p.c0, split_step=True,
                                adaptive_filtering=True, want_full=True)
    _, ablh = O.precalculate_abl(nX, nY, nT, p.boundaryFactor, True, p.boundaryProfile)
    af = O.precalculate_abl_freq(nX, nY, nT, p.dT, p.c0, p.f0, p.boundaryFactor, p.boundaryProfile)
    wx = O.make_boundary_weights(nX, O.boundary_width(nX, p.boundaryFactor)).astype(np.float64)
    wy = O.make_boundary_weights(nY, O.boundary_width(nY, p.boundaryFactor)).astype(np.float64)
    ref = {"attenuation": O.attenuation_step(u64, afh), "propagator": O.angular_spectrum_step(u64, HHh, ablh),
           "freq_weighted": O.freq_weighted_boundary_step(u64, af),
           "super_absorbing": O.super_absorbing_step(u64, wx, wy, p.dX, p.dY, p.dT, p.c0, p.superAbsorbingStrength)}
    for name in got:
        g, r = got[name].cpu().numpy(), ref[name]
        assert np.isfinite(g).all(), name
        # (tiny grids can be absorbed whole: compare against the input's norm then)
        e = np.linalg.norm(g - r) / max(np.linalg.norm(r), 1e-3 * np.linalg.norm(u64))
        print(shape, name, f"{e:.2e}", flush=True)
        assert e < 5e-6, (name, e)
    plan.close()


def test_general_columns_do_not_mix():
    """Sixteen columns share a block: zeros in a column stay exact zeros, and a column of
    NaN leaves its neighbours as they are."""
    shape = (5, 7, 301)
    p = _params(shape)
    plan = _plan(shape, p, 3.08e-4)
    u = _field(shape)
    u[2, 3] = 0.0
    phase = np.zeros(shape[:2], dtype=np.float32)
    want = plan.apply_phase_screen(_dev(u), _dev(phase)).cpu().numpy()
    assert not want[2, 3].any()
    v = u.copy()
    v[1, 2] = np.nan
    got = plan.apply_phase_screen(_dev(v), _dev(phase)).cpu().numpy()
    assert np.isnan(got[1, 2]).all()
    keep = np.ones(shape[:2], dtype=bool)
    keep[1, 2] = False
    assert np.array_equal(got[keep], want[keep])
    assert rel_l2(want, u) < 2e-6


@pytest.mark.parametrize("nT", [7, 63, 65, 129, 257, 300, 513, 801, 1025, 2047])
def test_raw_columns_move_through_lds_whole(nT):
    """The nonlinear step of real columns around every samples-per-lane class: against the
    oracle (the operator tests' 1e-6: a few float32 operations a sample), in place, and the
    peak of the field to the last bit."""
    from angularspectrum_heterogeneous_amd import _lib
    shape = (5, 27, nT)  # 135 columns: three blocks of the peak, the last partly filled
    p = _params(shape)
    N, dz = p.beta / (2 * p.c0 ** 3 * p.rho0), 3.08e-4
    plan = _plan(shape, p, dz)
    u = _field(shape, p0=3e6)
    got = plan.nonlinear_step(_dev(u), _lib.NL_RUSANOV, dz)
    assert rel_l2(got.cpu().numpy(), O.rusanov_flux_standard(u.astype(np.float64), N, dz, p.dT)) < 1e-6
    x = _dev(u)
    plan.nonlinear_step(x, _lib.NL_RUSANOV, dz, out=x)
    assert np.array_equal(x.cpu().numpy(), got.cpu().numpy())
    assert plan.max_abs(_dev(u)) == float(np.abs(u).max())
