"""Boundary transforms over the compiled ring lengths and lengths without a
compiled plan, at the edges of the ring groups (node counts not a multiple of
the group, one group, orders up to the Nyquist limit), against numpy FFTs and
the FP64 Legendre tables of the plan (pinned elsewhere).

Tolerances, relative to the largest value: sums of about 50 Legendre terms and
log2(n) FFT stages, a few hundred rounding units: 1e-13 in FP64, 2e-5 in FP32."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = [36, 48, 54, 64, 72, 81, 96, 108, 128, 144, 162, 192, 216, 243, 256, 288, 324, 384, 432, 486, 512, 576,
           648, 729, 768, 864]


def _close(a, b, tol, what):
    e = np.abs(a - b).max() / np.abs(b).max()
    assert e < tol, "%s: %.2e" % (what, e)


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp32", 2e-5)])
@pytest.mark.parametrize("nlon", LENGTHS)
def test_ring_lengths(nlon, prec, tol):
    import gdhip

    mmax = min((nlon - 1) // 2, 40)
    lmax, nr = mmax + 3, 3
    nlat = {0: lmax + 5, 1: lmax + 11}[nlon % 2]
    nlat += nlat % 2
    print("case: ring nlon=%d nlat=%d mmax=%d %s" % (nlon, nlat, mmax, prec), flush=True)
    cfg = gdhip.create_shtnskit_config(lmax, mmax, nlat=nlat, nlon=nlon, precision=prec)
    P, dP = cfg.plm_tables()
    m, l = cfg.m_values, cfg.l_values
    s = np.sin(cfg.theta_grid)
    Q = m[:, None] * P / s
    rng = np.random.default_rng(nlon)

    def spec():
        z = rng.standard_normal((nr, cfg.nlm)) + 1j * rng.standard_normal((nr, cfg.nlm)) * (m > 0)
        z[:, 0] = 0.0
        return z

    def rings(coef):  # Fourier sums (nr, nlat, mmax + 1) -> grid (nr, nlon, nlat)
        return np.fft.irfft(coef, n=nlon, axis=-1, norm="forward").transpose(0, 2, 1)

    def fourier(a, tab):
        out = np.zeros((nr, nlat, nlon // 2 + 1), complex)
        for k in range(mmax + 1):
            out[:, :, k] = a[:, m == k] @ tab[m == k]
        return out

    def project(f, tab):
        G = np.fft.rfft(f, axis=1)[:, :mmax + 1] * (2 * np.pi * cfg.gauss_weights / nlon)
        return np.stack([G[:, mk] @ tab[i] for i, mk in enumerate(m)], axis=-1)

    def F(z=None):
        f = gdhip.SHTnsSpectralField(cfg, nr)
        if z is not None:
            f.data_real[...], f.data_imag[...] = z.real, z.imag
        return f

    def G(x=None):
        return gdhip.SHTnsPhysicalField(cfg, nr, data=None if x is None else np.ascontiguousarray(x))

    a, t = spec(), spec()
    g = G()
    gdhip.shtnskit_spectral_to_physical(F(a), g)
    _close(g.data, rings(fourier(a, P)), tol, "scalar synthesis")
    vec = gdhip.SHTnsVectorField(cfg, nr)
    gdhip.shtnskit_vector_synthesis(F(t), F(a), vec)
    _close(vec.theta_component.data, rings(fourier(a, dP) + 1j * fourier(t, Q)), tol, "v_theta")
    _close(vec.phi_component.data, rings(1j * fourier(a, Q) - fourier(t, dP)), tol, "v_phi")
    x, y = rng.standard_normal((2, nr, nlon, nlat))
    b = F()
    gdhip.shtnskit_physical_to_spectral(G(x), b)
    ref = project(x, P)
    ref.imag[:, m == 0] = 0.0
    _close(b.complex(), ref, tol, "scalar analysis")
    tor, pol = F(), F()
    gdhip.shtnskit_vector_analysis(gdhip.SHTnsVectorField(cfg, nr, [None, G(x), G(y)]), tor, pol)
    inv = np.where(l > 0, 1.0 / np.maximum(l * (l + 1), 1), 0.0)
    S = inv * (project(x, dP) - 1j * project(y, Q))
    T = inv * (-1j * project(x, Q) - project(y, dP))
    for z in (S, T):
        z.imag[:, m == 0] = 0.0
    _close(pol.complex(), S, tol, "poloidal analysis")
    _close(tor.complex(), T, tol, "toroidal analysis")
