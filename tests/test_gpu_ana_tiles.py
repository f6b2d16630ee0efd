"""The analysis' Legendre contraction at the edges of its node tiles (nlat/2 at
and around 32, 48, 64, 96, 128, 192 and beyond, where node chunks add), row
tiles (parity groups of 16 and 17 degrees, empty odd groups at m = lmax) and
level tiles, against numpy projections on the plan's FP64 tables (pinned
elsewhere).

Tolerances, relative to the largest value: sums over up to 400 nodes of terms
of random sign, a few hundred rounding units of the operands: 1e-13 in FP64,
2e-5 in FP32, 2e-4 for the BF16x3 contraction (its products carry 2^-16)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (nlat/2, lmax, mmax, nr)
CASES = [(12, 20, 20, 1), (17, 30, 30, 7), (31, 31, 31, 8), (32, 32, 32, 9), (33, 32, 20, 16), (47, 33, 33, 17),
         (48, 63, 21, 15), (49, 64, 10, 2), (63, 31, 5, 33), (64, 40, 12, 3), (65, 40, 12, 3), (95, 65, 8, 9),
         (96, 31, 31, 8), (97, 33, 7, 17), (127, 32, 6, 5), (128, 40, 6, 16), (129, 40, 6, 9), (191, 34, 6, 3),
         (192, 40, 5, 17), (193, 33, 5, 9), (400, 20, 4, 2)]


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp32", 2e-5), ("bf16x3", 2e-4)])
@pytest.mark.parametrize("nlat2,lmax,mmax,nr", CASES)
def test_ana_tiles(nlat2, lmax, mmax, nr, prec, tol):
    import gdhip

    nlat, nlon = 2 * nlat2, 96 if mmax <= 32 else 144
    print("case: ana nlat2=%d lmax=%d mmax=%d nr=%d %s" % (nlat2, lmax, mmax, nr, prec), flush=True)
    cfg = gdhip.create_shtnskit_config(lmax, mmax, nlat=nlat, nlon=nlon, precision=prec)
    P, dP = cfg.plm_tables()
    m, l = cfg.m_values, cfg.l_values
    Q = m[:, None] * P / np.sin(cfg.theta_grid)
    x, y = np.random.default_rng(nlat2).standard_normal((2, nr, nlon, nlat))
    w = 2 * np.pi * cfg.gauss_weights / nlon
    X, Y = (np.fft.rfft(f, axis=1)[:, :mmax + 1] * w for f in (x, y))

    def project(G, tab):
        return np.stack([G[:, mk] @ tab[i] for i, mk in enumerate(m)], axis=-1)

    def G(f):
        return gdhip.SHTnsPhysicalField(cfg, nr, data=np.ascontiguousarray(f))

    def check(field, ref, what):
        ref.imag[:, m == 0] = 0.0
        e = np.abs(field.complex() - ref).max() / np.abs(ref).max()
        assert e < tol, "%s: %.2e" % (what, e)

    F = [gdhip.SHTnsSpectralField(cfg, nr) for _ in range(3)]
    gdhip.shtnskit_physical_to_spectral(G(x), F[0])
    check(F[0], project(X, P), "scalar")
    gdhip.shtnskit_vector_analysis(gdhip.SHTnsVectorField(cfg, nr, [None, G(x), G(y)]), F[1], F[2])
    inv = np.where(l > 0, 1.0 / np.maximum(l * (l + 1), 1), 0.0)
    check(F[2], inv * (project(X, dP) - 1j * project(Y, Q)), "poloidal")
    check(F[1], inv * (-1j * project(X, Q) - project(Y, dP)), "toroidal")
