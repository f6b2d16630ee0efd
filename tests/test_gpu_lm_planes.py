"""l-major <-> m-major planes at the edges of the 32 x 32 conversion tiles:
state and composition round trips are copies, so they are exact; the order is
pinned by an analysis of a synthesised single harmonic."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmax,mmax,nr", [(1, 0, 9), (31, 31, 8), (32, 32, 9), (33, 30, 10), (64, 63, 8), (95, 40, 9)])
def test_state_round_trip_is_exact(lmax, mmax, nr):
    import gdhip

    print("case: lm planes lmax=%d mmax=%d nr=%d" % (lmax, mmax, nr), flush=True)
    nlat, nlon = lmax + 2 + lmax % 2, 192
    s = gdhip.CNAB2Step(lmax, nlat, nlon, nr, mmax=mmax)
    rng = np.random.default_rng(lmax)
    re, im = rng.standard_normal(s.shape), rng.standard_normal(s.shape)
    s.set_state(re, im)
    a, b = s.get_state()
    assert np.array_equal(a, re) and np.array_equal(b, im)
    s.enable_composition()
    s.set_composition(re[0] + 1j * im[0])
    assert np.array_equal(s.get_composition(), re[0] + 1j * im[0])


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-5)])
def test_modes_keep_their_place(prec, tol):
    """Each coefficient of a truncated field comes back in its own l-major place."""
    import gdhip

    lmax, mmax, nr = 37, 33, 3
    cfg = gdhip.create_shtnskit_config(lmax, mmax, nlat=40, nlon=72, precision=prec)
    spec, back = (gdhip.SHTnsSpectralField(cfg, nr) for _ in range(2))
    phys = gdhip.SHTnsPhysicalField(cfg, nr)
    spec.data_real[...] = 1.0 + np.arange(cfg.nlm) + 0.25 * np.arange(nr)[:, None]
    spec.data_imag[...] = (cfg.m_values > 0) * (0.5 + np.arange(cfg.nlm))
    gdhip.shtnskit_spectral_to_physical(spec, phys)
    gdhip.shtnskit_physical_to_spectral(phys, back)
    # rounding of 38 x 40 term sums relative to the largest coefficient
    assert np.abs(back.complex() - spec.complex()).max() < tol * np.abs(spec.complex()).max()
