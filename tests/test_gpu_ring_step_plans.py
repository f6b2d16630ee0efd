"""The step's nonlinear terms and the transposed ones over ring lengths with
and without a compiled plan, with orders up to the Nyquist limit, against the
FP64 oracle: tangential and full (with composition: test_gpu_ring_step_composition.py).

Tolerances, relative to each field's largest value: those of the step's own
parity tests, 1e-10 in FP64 and 1e-4 in FP32 (products of fields whose curls
amplify rounding); the adjoint's dot product 1e-12 of its terms' scale."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (nlon, lmax): every compiled length, two without a plan, and undealiased grids
CASES = [(36, 11), (48, 15), (54, 17), (64, 20), (72, 23), (81, 26), (96, 25), (108, 24), (128, 24), (144, 24),
         (162, 24), (192, 24), (216, 24), (243, 24), (256, 24), (288, 24), (324, 24), (384, 24), (432, 24), (486, 24),
         (512, 24), (576, 24), (648, 24), (729, 24), (768, 24), (864, 24), (54, 26), (96, 47), (128, 63)]


def _relf(a, b):
    return [np.abs(a[k] - b[k]).max() / max(np.abs(b[k]).max(), 1e-300) for k in range(len(b))]


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-10), ("fp32", 1e-4)])
@pytest.mark.parametrize("nlon,lmax", CASES)
def test_nonlinear_over_ring_lengths(oracle, nlon, lmax, prec, tol):
    import gdhip

    nlat, nr = lmax + 5 + (lmax + 5) % 2, 9
    st = oracle.seeded_state(nlon, lmax, lmax, nr, amp=1e-3)
    full_fits = nlon <= 512  # the 15-field pass refuses longer rings
    for full in (False, True) if full_fits else (False,):
        print("case: step ring nlon=%d lmax=%d %s full=%d" % (nlon, lmax, prec, full), flush=True)
        g = gdhip.CNAB2Step(lmax, nlat, nlon, nr, precision=prec, radials=full, full_products=full)
        g.set_state_complex(st)
        err = _relf(g.nonlinear(), oracle.Model(lmax, nlat, nlon, nr, radials=full).nonlinear(st))
        g.close()
        print("nl rel err", err)
        assert max(err) < tol


@pytest.mark.parametrize("nlon,lmax", [(54, 17), (54, 26), (108, 24), (192, 24), (256, 24), (864, 24)])
def test_adjoint_over_ring_lengths(oracle, nlon, lmax):
    import gdhip

    print("case: adjoint ring nlon=%d lmax=%d" % (nlon, lmax), flush=True)
    nlat, nr = lmax + 5 + (lmax + 5) % 2, 9
    g = gdhip.CNAB2Step(lmax, nlat, nlon, nr, precision="fp64")
    rng = np.random.default_rng(nlon)
    x = oracle.seeded_state(nlon, lmax, lmax, nr, amp=1.0, zero_boundaries=False)
    v, mu = (rng.standard_normal(g.shape) + 1j * rng.standard_normal(g.shape) for _ in range(2))
    vals = []
    for s in (1, -1):
        g.set_state_complex(x + s * v)
        vals.append(g.nonlinear())
    jv = 0.5 * (vals[0] - vals[1])
    g.set_state_complex(x)
    lam = gdhip.nonlinear_adjoint(g, mu)
    g.close()
    lhs, rhs = (float(np.sum(a.real * b.real + a.imag * b.imag)) for a, b in ((mu, jv), (lam, v)))
    assert abs(lhs - rhs) <= 1e-12 * np.abs(mu).sum() * np.abs(jv).max()
