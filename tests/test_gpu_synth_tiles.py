"""The synthesis' Legendre contraction with the spectral columns in registers at
the edges of its degree groups (parities of 16, 17, 32, 64, 65 and 128 degrees,
the last order's single one; 129, which the LDS form takes), node tiles (one
node, 16, 17) and level tiles (1, 8, 9, 16, 17), against numpy sums on the
plan's FP64 tables (pinned elsewhere).

Tolerances, relative to the largest value: sums over up to 258 degrees of terms
of random sign, a few hundred rounding units of the operands: 1e-13 in FP64,
2e-5 in FP32, 2e-4 for the BF16x3 contraction (its products carry 2^-16)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (lmax, mmax, nlat/2, nr)
CASES = [(1, 1, 2, 1), (2, 2, 17, 3), (30, 30, 16, 8), (31, 31, 17, 9), (32, 32, 33, 16), (33, 20, 18, 17), (63, 31, 33, 1),
         (64, 12, 47, 2), (95, 10, 49, 7), (127, 6, 65, 9), (128, 6, 70, 3), (254, 3, 129, 2), (255, 4, 128, 5),
         (256, 3, 130, 2)]


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp32", 2e-5), ("bf16x3", 2e-4)])
@pytest.mark.parametrize("lmax,mmax,nlat2,nr", CASES)
def test_synth_tiles(lmax, mmax, nlat2, nr, prec, tol):
    import gdhip

    nlat, nlon = 2 * nlat2, 96
    print("case: synth lmax=%d mmax=%d nlat2=%d nr=%d %s" % (lmax, mmax, nlat2, nr, prec), flush=True)
    cfg = gdhip.create_shtnskit_config(lmax, mmax, nlat=nlat, nlon=nlon, precision=prec)
    P, dP = cfg.plm_tables()
    m = cfg.m_values
    Q = m[:, None] * P / np.sin(cfg.theta_grid)
    rng = np.random.default_rng(lmax)

    def field():
        f = gdhip.SHTnsSpectralField(cfg, nr)
        z = rng.standard_normal((nr, cfg.nlm)) + 1j * rng.standard_normal((nr, cfg.nlm)) * (m > 0)
        z[:, 0] = 0.0
        f.data_real[...], f.data_imag[...] = z.real, z.imag
        return f, z

    def grid(a, tab):
        out = np.zeros((nr, nlat, nlon // 2 + 1), complex)
        for k in range(mmax + 1):
            out[:, :, k] = a[:, m == k] @ tab[m == k]
        return out

    def check(data, coef, what):
        ref = np.fft.irfft(coef, n=nlon, axis=-1, norm="forward").transpose(0, 2, 1)
        e = np.abs(data - ref).max() / np.abs(ref).max()
        assert e < tol, "%s: %.2e" % (what, e)

    (fs, s), (ft, t) = field(), field()
    g = gdhip.SHTnsPhysicalField(cfg, nr)
    gdhip.shtnskit_spectral_to_physical(fs, g)
    check(g.data, grid(s, P), "scalar")
    vec = gdhip.SHTnsVectorField(cfg, nr)
    gdhip.shtnskit_vector_synthesis(ft, fs, vec)
    check(vec.theta_component.data, grid(s, dP) + 1j * grid(t, Q), "v_theta")
    check(vec.phi_component.data, 1j * grid(s, Q) - grid(t, dP), "v_phi")
