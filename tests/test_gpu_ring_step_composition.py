"""-u.grad C, the composition's product of the step's ring pass, against the FP64
oracle's -u.grad T with T := C (the same operator) at ring lengths of the
compiled register plans of two and three stages, odd ones, grids with orders up
to the Nyquist limit, and node counts with and without a multiple of 8 (which
decide the blocks' order), beside the five fields' nonlinear terms.

Tolerances as in the step's own parity tests, relative to the largest value:
1e-10 in FP64, 1e-4 in FP32."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (nlon, lmax, nlat)
CASES = [(54, 17, 28), (54, 26, 32), (64, 20, 32), (72, 23, 48), (81, 26, 40), (108, 24, 30), (128, 63, 64), (162, 24, 48),
         (243, 24, 30), (256, 24, 32), (324, 24, 30), (432, 24, 32), (512, 24, 48), (648, 24, 30), (768, 24, 32)]


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-10), ("fp32", 1e-4)])
@pytest.mark.parametrize("nlon,lmax,nlat", CASES)
def test_composition_product(oracle, nlon, lmax, nlat, prec, tol):
    import gdhip

    nr = 9
    print("case: step composition nlon=%d lmax=%d nlat=%d %s" % (nlon, lmax, nlat, prec), flush=True)
    st = oracle.seeded_state(nlon, lmax, lmax, nr, amp=1e-3)
    C = oracle.seeded_state(nlon + 1, lmax, lmax, nr, nfields=1, amp=1e-3, zero_boundaries=False)[0]
    g = gdhip.CNAB2Step(lmax, nlat, nlon, nr, precision=prec)
    g.enable_composition(2.0)
    g.set_state_complex(st)
    g.set_composition(C)
    g.run(1)
    model = oracle.Model(lmax, nlat, nlon, nr)
    ref5 = model.nonlinear(st)
    sC = st.copy()
    sC[4] = C
    ref, nl, nl5 = model.nonlinear(sC)[4], g.get_composition_history(), g.get_history()
    g.close()
    err = [np.abs(a - b).max() / max(np.abs(b).max(), 1e-300) for a, b in [(nl, ref)] + list(zip(nl5, ref5))]
    print("nl rel err", err)
    assert max(err) < tol


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-10), ("fp32", 1e-4)])
@pytest.mark.parametrize("nlon,lmax,nlat", [(72, 23, 48), (81, 26, 32), (216, 24, 32), (288, 24, 48), (384, 24, 32), (512, 24, 32)])
def test_full_products_in_launch_order(oracle, nlon, lmax, nlat, prec, tol):
    import gdhip

    nr = 9
    print("case: step full nlon=%d lmax=%d nlat=%d %s" % (nlon, lmax, nlat, prec), flush=True)
    st = oracle.seeded_state(nlon, lmax, lmax, nr, amp=1e-3)
    g = gdhip.CNAB2Step(lmax, nlat, nlon, nr, precision=prec, radials=True, full_products=True)
    g.set_state_complex(st)
    nl = g.nonlinear()
    g.close()
    ref = oracle.Model(lmax, nlat, nlon, nr, radials=True).nonlinear(st)
    err = [np.abs(a - b).max() / max(np.abs(b).max(), 1e-300) for a, b in zip(nl, ref)]
    print("nl rel err", err)
    assert max(err) < tol
