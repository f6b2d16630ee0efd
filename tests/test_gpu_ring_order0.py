"""Order 0 of a real ring is real: the boundary ring passes ignore whatever the
imaginary parts of order 0 hold (NaN, infinity, a value beyond the FP32 range),
and a grid value that is not finite leaves the imaginary part of order 0 at 0,
at every kind of ring length (compiled plans of two and three stages, even and
odd, dealiased and up to the Nyquist limit, and the runtime plan).  What is
ignored cannot change a bit, so results are compared exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (nlon, mmax)
CASES = [(36, 11), (48, 15), (54, 26), (81, 20), (96, 31), (162, 40), (243, 40), (384, 40), (512, 40), (768, 40), (864, 40)]


@pytest.mark.parametrize("prec", ["fp64", "fp32", "bf16x3"])
@pytest.mark.parametrize("nlon,mmax", CASES)
def test_order0_imaginary_parts_are_ignored(nlon, mmax, prec):
    import gdhip

    nr, lmax = 4, mmax + 2
    print("case: order 0 nlon=%d mmax=%d %s" % (nlon, mmax, prec), flush=True)
    cfg = gdhip.create_shtnskit_config(lmax, mmax, nlat=lmax + 4 + lmax % 2, nlon=nlon, precision=prec)
    rng = np.random.default_rng(nlon)
    re, im = rng.standard_normal((2, nr, cfg.nlm))
    zero = cfg.m_values == 0
    im[:, zero] = 0.0
    grids = []
    for junk in (0.0, np.nan, np.inf, 1e300):
        z = im.copy()
        z[:, zero] = junk
        g = gdhip.SHTnsPhysicalField(cfg, nr)
        gdhip.shtnskit_spectral_to_physical(gdhip.SHTnsSpectralField(cfg, nr, re, z), g)
        grids.append(g.data)
    assert np.isfinite(grids[0]).all()
    for g in grids[1:]:
        assert np.array_equal(g, grids[0])


@pytest.mark.parametrize("prec", ["fp64", "fp32", "bf16x3"])
@pytest.mark.parametrize("nlon,mmax", CASES)
def test_order0_poloidal_part_needs_no_v_phi(nlon, mmax, prec):
    """At order 0 the poloidal coefficients come from v_theta alone: (i m / sin)
    v_phi is 0 there, also where v_phi holds an infinity."""
    import gdhip

    nr, lmax = 3, mmax + 2
    print("case: order 0 v_phi nlon=%d mmax=%d %s" % (nlon, mmax, prec), flush=True)
    cfg = gdhip.create_shtnskit_config(lmax, mmax, nlat=lmax + 4 + lmax % 2, nlon=nlon, precision=prec)
    vt, vp = np.random.default_rng(nlon).standard_normal((2, nr, nlon, cfg.nlat))
    zero = cfg.m_values == 0
    pols = []
    for junk in (False, True):
        y = vp.copy()
        if junk:
            y[1, 3, cfg.nlat - 2] = np.inf
        F = [gdhip.SHTnsSpectralField(cfg, nr) for _ in range(2)]
        comps = [None] + [gdhip.SHTnsPhysicalField(cfg, nr, data=d) for d in (vt, y)]
        gdhip.shtnskit_vector_analysis(gdhip.SHTnsVectorField(cfg, nr, comps), F[0], F[1])
        pols.append(F[1].complex()[:, zero])
    assert np.isfinite(pols[0]).all()
    assert np.array_equal(pols[1], pols[0])
