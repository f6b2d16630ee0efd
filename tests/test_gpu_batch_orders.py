"""Fused batches of shells whose grids are not dealiased (orders up to the
Nyquist limit), alone and beside dealiased shells of the same ring length, at
ring lengths of every batched form: each shell gets the bits of its own run,
and its synthesis is part of the fused launches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (nlon, nlat, lmax, lmax of a dealiased shell of that ring): a length without
# a compiled plan, two- and three-stage register plans, a short length's plan
RINGS = [(36, 24, 17, 11), (72, 40, 35, 23), (128, 72, 63, 41), (243, 104, 100, 56), (96, 48, 47, 31)]


@pytest.mark.parametrize("prec", ["fp64", "fp32", "bf16x3"])
@pytest.mark.parametrize("nlon,nlat,lmax,lmax_deal", RINGS)
def test_batch_of_undealiased_shells(nlon, nlat, lmax, lmax_deal, prec):
    import gdhip

    print("case: batch orders nlon=%d lmax=%d %s" % (nlon, lmax, prec), flush=True)
    groups = []
    for _ in range(2):
        groups.append([])
        for k, (L, nr) in enumerate([(lmax, 9), (lmax_deal, 17), (lmax, 13)]):
            s = gdhip.CNAB2Step(L, nlat, nlon, nr, precision=prec)
            s.set_state_complex(gdhip.seeded_state(40 + k, L, nr, amp=1e-3))
            groups[-1].append(s)
    alone, batched = groups
    for s in alone:
        s.run(4, graph=True)
    batch = gdhip.StepBatch(batched)
    batch.run(4)
    batch.synchronize()
    for a, b in zip(alone, batched):
        sa, sb = a.get_state_complex(), b.get_state_complex()
        assert np.isfinite(sb).all() and np.array_equal(sa, sb)
    batch.close()
    # the shells that are not dealiased take part in the fused launches: a
    # synthesis launch takes microseconds, an empty sequence between two events
    # a fraction of one
    only = gdhip.StepBatch([batched[0], batched[2]])
    only.tune(reps=100)
    print("fused synthesis ms", only.tune_ms)
    assert only.tune_ms[1] > 1e-3
    only.close()
