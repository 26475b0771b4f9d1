"""The kernels that share one site's work among several waves on small
lattices, and the general ones above their limits, against the C oracle."""
import numpy as np
import pytest

import susy_amd
import surrogate_ref as sr
from oracle_lib import Oracle, random_links, random_tf, rel_err

pytestmark = pytest.mark.gpu


def pair(ncol, dims, **kw):
    args = dict(dims=dims, iseed=5, kappa_u1=1.0, bmass=1.0, G=0.2, fmass=0.3, **kw)
    return Oracle(ncol, **args), susy_amd.Lattice(ncol, **args)


# The smallest lattices, halves that are no multiple of the 64 sites of a
# block, odd extents (no even-odd halves of one size), and both sides of the
# limits: U(2) pre-pass in the kernel up to 1296 sites, five waves up to 32768
# (U(2), and U(3) FP32), 4096 (U(4) FP64) and 3072 (U(3) FP64, U(4) FP32); above,
# blocks of 64, 128 and 256 sites, by what divides the lattice among 8 XCDs.
# Bounds: a result sums some 20 NCOL products of order one, so rounding is
# about 1e-15 (FP64) and 6e-7 (FP32) of the largest element.
@pytest.mark.parametrize("ncol,dims", [
    (2, (2, 2, 2, 2)), (2, (3, 5, 2, 7)), (2, (6, 6, 6, 6)), (2, (6, 6, 6, 7)),
    (2, (16, 16, 16, 8)), (2, (16, 15, 18, 8)),
    (3, (1, 2, 3, 5)), (3, (8, 8, 8, 6)), (3, (8, 8, 7, 7)), (3, (16, 16, 16, 8)),
    (3, (16, 15, 18, 8)),
    (4, (2, 2, 2, 2)), (4, (3, 3, 5, 2)), (4, (8, 8, 8, 6)), (4, (8, 8, 7, 7)),
    (4, (8, 8, 8, 8)), (4, (8, 8, 7, 10)), (4, (8, 8, 12, 8)), (4, (8, 8, 7, 14)),
])
def test_operator_across_limits(ncol, dims):
    print("operator", ncol, dims, flush=True)
    O, lat = pair(ncol, dims)
    lk = random_links(O.link_shape(), 3, 0.2)
    O.set_links(lk)
    lat.set_links(lk)
    src = random_tf(O.tf_shape(), 9)
    h = lat.tf_alloc(2)
    lat.tf_upload(h, src)
    want = {s: O.fermion_op(src, s) for s in (1, -1)}
    dsq = O.fermion_op(want[1], -1) + 0.3 ** 2 * src
    for form, tol in ((susy_amd.FORM_FP64, 1e-13), (susy_amd.FORM_FP32, 1e-5)):
        for sign in (1, -1):
            lat.fermion_op(h, h + 1, sign, form)
            assert rel_err(lat.tf_download(h + 1), want[sign]) < tol, (form, sign)
        lat.dsq(h, h + 1, form)
        assert rel_err(lat.tf_download(h + 1), dsq) < tol, form
    lat.close()


# The surrogate's kernels work on 16 and 64 sites a block: site counts below
# one block, on its edge and with a remainder, for every group the matrices of
# which are held in registers.  Bounds as for the other surrogate tests:
# float32 sums of some 700 terms, features rounded to float32 once.
@pytest.mark.parametrize("ncol,dims", [(2, (1, 2, 1, 4)), (2, (2, 2, 2, 8)), (3, (3, 3, 2, 5)),
                                       (4, (4, 4, 4, 1)), (4, (3, 5, 2, 3)), (5, (2, 3, 2, 3))])
def test_surrogate_site_blocks(ncol, dims):
    print("surrogate", ncol, dims, flush=True)
    lat = susy_amd.Lattice(ncol, dims=dims, G=0.05)
    U = random_links(lat.link_shape(), 3, 0.3)
    lat.set_links(U)
    lat.sg_init(seed=5, scale=2.0)
    th = sr.unpack(lat.sg_get_params())
    th["b1"] = np.random.default_rng(6).standard_normal(sr.NCH) * 0.2
    th["b2"] = np.random.default_rng(7).standard_normal(sr.NCH) * 0.2
    lat.sg_set_params(sr.pack(th))
    th, geo = sr.weights_used(sr.unpack(lat.sg_get_params())), sr.Geometry(dims)
    assert rel_err(lat.sg_features(), sr.features(geo, U)) < 1e-6
    S_ref, F_ref = sr.action_and_force(geo, th, U)
    S, F = lat.sg_eval()
    assert abs(S / S_ref - 1) < 1e-5
    assert rel_err(F, F_ref) < 1e-5
    Ft = random_links(lat.link_shape(), 9, 0.5) - np.eye(ncol)
    loss, g = lat.sg_loss_grad(U, Ft)
    loss_ref, g_ref = sr.force_loss_grad(geo, th, U, Ft)
    assert abs(loss / loss_ref - 1) < 1e-5
    assert rel_err(g, sr.pack(g_ref).astype(np.float64)) < 1e-4
    lat.close()


# The iteration's scalar steps, from few partials up to 8192, the last number
# that the blocks of FP64 sum themselves (test_solver_routes: both sides).  The first 12
# iterations follow the oracle to rounding (later ones amplify it: on the U(3)
# lattice |r|^2 of any two roundings differs by 1e-5 after 40 and by a tenth
# after 46); at the end every system's true residual is below the bound, with
# the FP32 form's margin as in its other tests.
@pytest.mark.parametrize("ncol,dims", [(2, (2, 2, 2, 2)), (3, (3, 3, 2, 5)), (2, (16, 16, 16, 8)),
                                       (2, (16, 15, 18, 8))])
def test_solver_scalar_steps(ncol, dims):
    print("solver", ncol, dims, flush=True)
    O, lat = pair(ncol, dims)
    lk = random_links(O.link_shape(), 3, 0.2)
    O.set_links(lk)
    lat.set_links(lk)
    src = random_tf(O.tf_shape(), 9)
    shifts = [0.5, 2.0, 9.0]
    h = lat.tf_alloc(5)
    lat.tf_upload(h, src)
    it, sz = lat.congrad_multi(h, h + 1, shifts, 12, 1e-10)
    it_o, sz_o, psi = O.congrad_multi(src, shifts, 12, 1e-10)
    assert it == it_o == 12
    assert abs(sz / sz_o - 1) < 1e-6
    for j in range(3):
        assert rel_err(lat.tf_download(h + 1 + j), psi[j]) < 1e-10, j
    n2 = np.vdot(src, src).real
    for form, margin in ((susy_amd.FORM_FP64, 1.01), (susy_amd.FORM_FP32, 4)):
        assert lat.congrad_multi(h, h + 1, shifts, 500, 1e-10, form)[0] < 500
        for j in range(3):
            lat.dsq(h + 1 + j, h + 4)
            r = src - lat.tf_download(h + 4) - shifts[j] * lat.tf_download(h + 1 + j)
            assert np.vdot(r, r).real <= margin * 1e-10 * n2, (form, j)
    lat.close()


# The force's four waves a link share its terms by direction: sites below and
# beyond a block, with and without the determinant terms, over two poles and
# every site order.  Sums of some 70 products, relative to the whole force:
# 1e-12 leaves three digits over their rounding.
@pytest.mark.parametrize("ncol,dims", [(2, (2, 2, 2, 2)), (2, (6, 6, 6, 7)), (3, (1, 2, 3, 5)),
                                       (3, (4, 5, 4, 6)), (4, (3, 3, 5, 2)), (4, (4, 4, 4, 10))])
@pytest.mark.parametrize("G", [0.0, 0.2])
def test_force_waves(ncol, dims, G):
    print("force", ncol, dims, G, flush=True)
    args = dict(dims=dims, iseed=5, kappa_u1=1.0, bmass=1.0, G=G)
    O, lat = Oracle(ncol, **args), susy_amd.Lattice(ncol, **args)
    lk = random_links(O.link_shape(), 3, 0.2)
    O.set_links(lk)
    lat.set_links(lk)
    h = lat.tf_alloc(2)
    sol = np.stack([random_tf(O.tf_shape(), 9), random_tf(O.tf_shape(), 10)])
    for j in range(2):
        lat.tf_upload(h + j, sol[j])
    O.set_mom(np.zeros(O.link_shape(), complex))
    O.fermion_force(0.1, sol, [0.7, -0.3])
    want = O.get_mom()
    for order in (0, 1, 2):
        lat.set_site_order(order)
        lat.set_mom(np.zeros(O.link_shape(), complex))
        lat.fermion_force(0.1, h, [0.7, -0.3])
        assert rel_err(lat.get_mom(), want) < 1e-12, order
    lat.close()


# U(5): the operator's ordinary kernel takes its determinant scalars one after
# the other in both precisions, and the force's waves make two columns each,
# in rounds of three and two rows.  Site counts below one block, beyond it
# with a remainder in each half, and over several XCDs; inputs and bounds are
# those of the tests above.
@pytest.mark.parametrize("dims", [(3, 3, 5, 2), (4, 4, 5, 2), (4, 6, 5, 6)])
def test_operator_u5_blocks(dims):
    test_operator_across_limits(5, dims)


@pytest.mark.parametrize("dims", [(3, 3, 5, 2), (4, 4, 5, 2), (4, 6, 5, 6)])
@pytest.mark.parametrize("G", [0.0, 0.2])
def test_force_u5_blocks(dims, G):
    test_force_waves(5, dims, G)


def partials(dims, chunk):
    """blocks of the operator, one partial of <p, A p> each, in chunks of
    `chunk` sites of both halves of the site order, shared by 8 XCDs"""
    vol = int(np.prod(dims))
    chunks = -(-(vol - vol // 2) // chunk)
    return 8 * -(-chunks // 8) * 2 * 16


# The two ways of an iteration's scalar steps at their limits, 8192 partials in
# FP64 and 6144 in FP32: every block sums them (four launches) or one block does
# (six).  All these lattices work in chunks of 64 sites.  Both forms follow the
# oracle's first 12 iterations: FP64 as in test_solver_scalar_steps; in FP32 every
# iteration adds its roundings of some 6e-7 to vectors that the shifted operator
# (condition below 1e3 on these links) amplifies by less than 100 in all.  At
# the end the true residuals are below the bound, with that test's margins.
@pytest.mark.parametrize("dims,four64,four32", [((16, 16, 16, 6), True, True),
                                                ((12, 12, 12, 16), True, False),
                                                ((12, 12, 12, 24), False, False)])
def test_solver_routes(dims, four64, four32):
    print("solver routes", dims, flush=True)
    n = partials(dims, 64)
    assert (n <= 8192, n <= 6144) == (four64, four32)
    O, lat = pair(2, dims)
    lk = random_links(O.link_shape(), 3, 0.2)
    O.set_links(lk)
    lat.set_links(lk)
    src = random_tf(O.tf_shape(), 9)
    shifts = [0.5, 2.0, 9.0]
    h = lat.tf_alloc(5)
    lat.tf_upload(h, src)
    it_o, sz_o, psi = O.congrad_multi(src, shifts, 12, 1e-10)
    n2 = np.vdot(src, src).real
    for form, sz_tol, tol, margin in ((susy_amd.FORM_FP64, 1e-6, 1e-10, 1.01),
                                      (susy_amd.FORM_FP32, 1e-3, 1e-4, 4)):
        it, sz = lat.congrad_multi(h, h + 1, shifts, 12, 1e-10, form)
        assert it == it_o == 12
        assert abs(sz / sz_o - 1) < sz_tol, form
        for j in range(3):
            assert rel_err(lat.tf_download(h + 1 + j), psi[j]) < tol, (form, j)
        assert lat.congrad_multi(h, h + 1, shifts, 500, 1e-10, form)[0] < 500
        for j in range(3):
            lat.dsq(h + 1 + j, h + 4)
            r = src - lat.tf_download(h + 4) - shifts[j] * lat.tf_download(h + 1 + j)
            assert np.vdot(r, r).real <= margin * 1e-10 * n2, (form, j)
    lat.close()


# Limits that test_operator_across_limits does not reach: U(2) in FP32 takes
# the ordinary kernel between 3072 and 6144 sites, the five waves on both sides of
# that range; the pre-pass has a thread per site and trace up to 65536 sites
# and a thread per site above.
@pytest.mark.parametrize("dims", [(8, 8, 8, 6), (8, 8, 7, 7), (8, 8, 10, 8), (8, 8, 8, 12),
                                  (16, 16, 16, 16), (16, 16, 16, 17)])
def test_operator_more_limits(dims):
    test_operator_across_limits(2, dims)
