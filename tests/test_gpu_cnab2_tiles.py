"""The l-major rhs / solve kernels at the edges of their column tiles: band
widths 1 and 7, truncated orders (mmax < lmax), a partly filled last tile, and
column lengths that take 64, 32 and 16 columns a block, each mode against the
oracle, device arrays, in place and out of place.

Tolerances: the rhs is a (2bw+1)-term FP64 sum (errors of a few ulp of its
largest term); the no-pivot banded solve's error grows with cond(S_l), about
1e3 at these steps, over 2n rows: 1e-11 of the field's largest value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("lmax,mmax,nr,bw", [(1, 0, 9, 1), (20, 7, 17, 2), (33, 33, 16, 7), (40, 31, 97, 3),
                                             (9, 9, 150, 3), (5, 3, 230, 4)])
@pytest.mark.parametrize("bc", [False, True])
def test_cnab2_tiles_match_oracle(oracle, lmax, mmax, nr, bw, bc):
    import torch

    import gdhip
    from gdhip._arrays import prepare
    from gdhip._lib import check, lib

    print("case: cnab2 tiles lmax=%d mmax=%d nr=%d bw=%d bc=%s" % (lmax, mmax, nr, bw, bc), flush=True)
    dt, nu = 1e-5, 1.0
    cfg = gdhip.create_shtnskit_config(lmax, mmax, nlat=2 * ((lmax + 2) // 2) + 2, nlon=96)
    dom = gdhip.create_radial_domain(nr, 0.35)
    M = gdhip.create_shtns_timestepping_matrices(cfg, dom, nu, dt, bw=bw, bc_rows=bc)
    st = oracle.seeded_state(4, lmax, mmax, nr, nfields=3, amp=1e-3)
    u, nl, nlp = st[0], st[1] * 100, st[2] * 100
    lo = cfg.l_values.astype(np.int32)
    L, S, LU = M._fetch()
    rhs_ref = oracle.cnab2_rhs(lo, L, dt, 0.5, u, nl, nlp, bc_rows=bc)
    sol_ref = oracle.cnab2_solve(lo, LU, rhs_ref)

    def F(z):
        return gdhip.SHTnsSpectralField(cfg, nr, *[torch.from_numpy(np.ascontiguousarray(p)).cuda()
                                                   for p in (z.real, z.imag)])

    def host(f):
        return f.data_real.cpu().numpy() + 1j * f.data_imag.cpu().numpy()

    fu, fn, fp, rhs, sol = F(u), F(nl), F(nlp), F(u * 0), F(u * 0)
    gdhip.build_rhs_cnab2(rhs, fu, fn, fp, dt, M)
    gdhip.solve_implicit_step(sol, rhs, M)
    assert _rel(host(rhs), rhs_ref) < 1e-13
    assert _rel(host(sol), sol_ref) < 1e-11
    inp = F(u)
    gdhip.build_rhs_cnab2(inp, inp, fn, fp, dt, M)  # the rhs over u
    assert np.array_equal(host(inp), host(rhs))
    gdhip.solve_implicit_step(inp, inp, M)
    assert np.array_equal(host(inp), host(sol))
    ctx, flags, p = prepare(fu.data_real, fu.data_imag, fn.data_real, fn.data_imag, fp.data_real, fp.data_imag)
    check(lib().gd_cnab2_rhs_solve(M._h, lmax, mmax, nr, *p, flags))
    assert _rel(host(fu), sol_ref) < 1e-11
