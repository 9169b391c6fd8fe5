"""Source injection: the spectra of a step's source slices are added to the columns that
carry one (COL_INJECT), on FFT columns (one, two and four per wave) and general-length
ones, with sparse masks that leave waves, halves of waves and whole blocks without a
source, dense slices, and both at once.

A source crossed in the last step adds to the field after everything else, so the solve
with it equals the solve without it plus the dense source.  The sum is formed on the
spectrum: two transforms of log2(nT) float32 passes each (a direct sum of nT/2 terms for
general lengths) round it by at most 6e-8 sqrt(2 * 512) = 2e-6 relative to the norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(64, 64, 256), (64, 33, 512), (20, 64, 1024), (9, 7, 2048), (51, 33, 101), (10, 13, 300), (7, 5, 1201)]


def _setup(shape, kind, rng):
    from angularspectrum_heterogeneous_amd.sources import SourceSlice
    from angularspectrum_heterogeneous_amd.workloads import axes, gaussian_beam, params_kwargs
    nX, nY, nT = shape
    dX, dT = 3.08e-4, 4e-8
    field = gaussian_beam(nX, nY, nT, dX, dT)
    kw = params_kwargs(dX=dX, dY=dX, dT=dT, propDist=2 * dX, dZmin=dX)
    mask = rng.random((nX, nY)) < 0.1
    mask[: nX // 2] = False
    mask[-1, -1] = True
    sparse = SourceSlice(mask, rng.uniform(-1e-6, 1e-6, (nX, nY)) * mask, axes(nT, dT), 1e6, 3e5, 3, 2)
    dense = (1e5 * rng.standard_normal(shape)).astype(np.float32)
    planes = {"sparse": [sparse], "dense": [dense], "both": [dense, sparse]}[kind]
    return field, kw, [(1.5 * dX, p) for p in planes]


@pytest.mark.parametrize("kind", ["sparse", "dense", "both"])
@pytest.mark.parametrize("shape", SHAPES)
def test_injection_adds_the_source(shape, kind):
    from angularspectrum_heterogeneous_amd.solver import SolverParams, angular_spectrum_solve
    rng = np.random.default_rng(sum(shape))
    field, kw, planes = _setup(shape, kind, rng)
    base = angular_spectrum_solve(field, SolverParams(**kw), verbose=False)
    got = angular_spectrum_solve(field, SolverParams(**kw, sourcePlanes=planes), verbose=False)
    want = base[0].astype(np.float64) + sum(np.asarray(p, dtype=np.float64) for _, p in planes)
    e = np.linalg.norm(got[0] - want) / np.linalg.norm(want)
    print(shape, kind, f"{e:.2e}", flush=True)
    assert e < 2e-6
    # the maps of the last step see the field with the source
    np.testing.assert_array_equal(got[1][:, :, -1], got[0].min(2))
    np.testing.assert_array_equal(got[2][:, :, -1], got[0].max(2))
    if kind == "sparse":
        # columns without a source are the other solve's, bit for bit
        bare = ~planes[0][1].mask
        np.testing.assert_array_equal(got[0][bare], base[0][bare])
