"""The analysis where the nodes take several chunks (the second one of 96 nodes or
of 192, at both edges), and in the step's record order (nodes strided), whose
node-to-lane mapping differs from that of the stand-alone transforms: node tiles
of 128 and 192, the FP32 sum in two halves, and chunks that add.

The stand-alone cases are checked as in test_gpu_ana_tiles.  The step's are
checked as whole nonlinear terms against the FP64 oracle, with the tolerances of
the step's own parity tests relative to each field's largest value: 1e-10 in FP64
and 1e-4 in FP32 (products of fields whose curls amplify rounding)."""
import numpy as np
import pytest

import test_gpu_ana_tiles as tiles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp32", 2e-5), ("bf16x3", 2e-4)])
@pytest.mark.parametrize("nlat2,lmax,mmax,nr", [(288, 33, 6, 9), (289, 20, 5, 17), (384, 33, 4, 3)])
def test_ana_chunks(nlat2, lmax, mmax, nr, prec, tol):
    tiles.test_ana_tiles(nlat2, lmax, mmax, nr, prec, tol)


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-10), ("fp32", 1e-4)])
@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("nlat2", [97, 128, 130, 192, 193, 289])
def test_step_nonlinear_over_node_tiles(oracle, nlat2, full, prec, tol):
    import gdhip

    lmax, nlon, nr = 20, 64, 9
    print("case: step nodes nlat2=%d full=%d %s" % (nlat2, full, prec), flush=True)
    st = oracle.seeded_state(nlat2, lmax, lmax, nr, amp=1e-3)
    g = gdhip.CNAB2Step(lmax, 2 * nlat2, nlon, nr, precision=prec, radials=full, full_products=full)
    g.set_state_complex(st)
    nl = g.nonlinear()
    g.close()
    ref = oracle.Model(lmax, 2 * nlat2, nlon, nr, radials=full).nonlinear(st)
    err = [np.abs(nl[k] - ref[k]).max() / max(np.abs(ref[k]).max(), 1e-300) for k in range(len(ref))]
    print("nl rel err", err)
    assert max(err) < tol
