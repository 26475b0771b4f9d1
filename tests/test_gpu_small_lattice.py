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
# (U(2), and U(3) FP32), 3072 (FP64) and 6144 (U(4) FP32).
# Bounds: a result sums some 20 NCOL products of order one, so rounding is
# about 1e-15 (FP64) and 6e-7 (FP32) of the largest element.
@pytest.mark.parametrize("ncol,dims", [
    (2, (2, 2, 2, 2)), (2, (3, 5, 2, 7)), (2, (6, 6, 6, 6)), (2, (6, 6, 6, 7)),
    (2, (16, 16, 16, 8)), (2, (16, 15, 18, 8)),
    (3, (1, 2, 3, 5)), (3, (8, 8, 8, 6)), (3, (8, 8, 7, 7)), (3, (16, 16, 16, 8)),
    (3, (16, 15, 18, 8)),
    (4, (2, 2, 2, 2)), (4, (3, 3, 5, 2)), (4, (8, 8, 8, 6)), (4, (8, 8, 7, 7)),
    (4, (8, 8, 12, 8)), (4, (8, 8, 7, 14)),
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
