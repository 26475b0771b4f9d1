"""Performance cases: the calls that RHMC programs on this library spend their
time in, over the lattices and gauge groups the library is configured for.

Kinds of case (`kind`):
  op    one application of the fermion operator D (sign +1) or D^dagger
        (sign -1) to a field in device memory (susy_fermion_op_noalloc).
  kick  one fermion kick of the integrator at fixed links: the multi-shift
        solve over the poles `first` .. 14 of the rational action and the
        force of those poles, which updates the momenta.  `form` is the
        solver's precision form.  first = 0 is the outer level; first = 9 is
        the middle level of the pole-split integrator.
  traj  a whole trajectory (heatbath, molecular dynamics, Metropolis test).

The FP32 form solves to FP32 accuracy, so its momenta and links are handed
back as single-precision complex numbers; the FP64 form's as double.
"""
import ctypes
import math
import os

import numpy as np
import torch

import susy_amd
from susy_amd.start_config import SMALL_DIMS, START_FILE, tile

E = ((1, 0, 0, 0), (0, 1, 0, 0), (0, 0, 1, 0), (0, 0, 0, 1), (-1, -1, -1, -1))
EPS = 0.025            # kick size: the outer step of the plain integrator, halved
COUPLINGS = dict(PBC=-1, Norder=15, kappa_u1=0.0, fmass=0.0, G=0.05, error_per_site=1e-5)


def _case(name, kind, ncol, dims, **kw):
    return dict({"name": name, "kind": kind, "ncol": ncol, "nx": dims[0], "ny": dims[1],
                 "nz": dims[2], "nt": dims[3]}, **kw)


def listed():
    return [
        # the operator alone: the regression lattices of the smallest runs
        # (latency), a ragged lattice, the mid-sized one and production
        _case("op_u2_4x4", "op", 2, (4, 4, 4, 4), sign=1),
        _case("op_dag_u3_8x16", "op", 3, (8, 8, 8, 16), sign=-1),
        _case("op_dag_u4_6x10", "op", 4, (6, 6, 6, 10), sign=-1),
        _case("op_u4_16x32", "op", 4, (16, 16, 16, 32), sign=1),
        # outer kicks, plain FP64: the small U(2) chain, the U(3) solver
        # configuration, U(4) at the thermalised small production lattice
        _case("kick_fp64_u2_4x4", "kick", 2, (4, 4, 4, 4), form="fp64", first=0, iters=38),
        _case("kick_fp64_u3_8x16", "kick", 3, (8, 8, 8, 16), form="fp64", first=0, iters=220),
        _case("kick_fp64_u4_8x16", "kick", 4, (8, 8, 8, 16), form="fp64", first=0, iters=1350),
        # mixed precision: outer kicks at the mixed-precision workload's size
        # and at the small production lattice, the middle level's kick at the
        # production lattice
        _case("kick_fp32_u4_8x16", "kick", 4, (8, 8, 8, 16), form="fp32", first=0, iters=1500),
        _case("kick_fp32_u4_12x24", "kick", 4, (12, 12, 12, 24), form="fp32", first=0, iters=400),
        _case("kick_fp32_u4_16x32", "kick", 4, (16, 16, 16, 32), form="fp32", first=9, iters=103),
        # whole trajectories: the plain chain of the regression lattice and
        # the production form (FP32 + learned force + pole split) in small
        _case("traj_fp64_u2_4x4", "traj", 2, (4, 4, 4, 4), form="fp64", nstep=5, iters=620),
        _case("traj_split_u4_4x8", "traj", 4, (4, 4, 4, 8), form="split", nstep=2, iters=3700),
    ]


def draw(rng):
    while True:
        kind = rng.choice(["op", "op", "kick", "kick", "kick", "traj"])
        ncol = rng.choice([2, 3, 4])
        if kind == "traj":
            top, n = 512, rng.choice([2, 3, 4])
            dims = [rng.choice([2, 3, 4, 5, 6]) for _ in range(3)] + [rng.choice([4, 6, 7, 8])]
        else:
            top, n = (131072, 0) if kind == "op" else (32768 if ncol == 4 else 16384, 0)
            hi = math.log(16.4 if kind == "op" else 12.4)
            dims = [int(round(math.exp(rng.uniform(math.log(3), hi)))) for _ in range(3)]
            dims.append(int(round(math.exp(rng.uniform(math.log(4), math.log(32))))))
        vol = dims[0] * dims[1] * dims[2] * dims[3]
        if vol % 2 == 0 and 128 <= vol <= top:
            break
    c = _case("", kind, ncol, dims)
    del c["name"]
    if kind == "op":
        c["sign"] = rng.choice([1, -1])
    elif kind == "kick":
        c["form"] = rng.choice(["fp64", "fp32"])
        c["first"] = rng.choice([0, 0, 9])
        c["iters"] = 40 if c["first"] else 100
    else:
        c["form"], c["nstep"], c["iters"] = ("fp64", n, 130 * n) if ncol == 2 else \
            ("split", n, 1800 * n)
    return c


# ---------------------------------------------------------------------
# Inputs

def _dims(case):
    return case["nx"], case["ny"], case["nz"], case["nt"]


def _params(case):
    prod = case["ncol"] == 4
    return dict(COUPLINGS, dims=_dims(case), Nroot=2 if prod else 1, lam=2.0 if prod else 1.0,
                bmass=0.4 if prod else 0.5, niter=5000, traj_length=0.25 if prod else 1.0,
                nstep=case.get("nstep", 5), nstep_gauge=10)


def _normal(gen, *shape):
    """complex Gaussian numbers of unit variance"""
    r = torch.randn(*shape, 2, generator=gen, device="cuda", dtype=torch.float64)
    return torch.view_as_complex(r) * math.sqrt(0.5)


_therm = {}


def _therm_links(dims):
    """the committed thermalised U(4) links, tiled (read once per process)"""
    if dims not in _therm:
        small = susy_amd.Lattice(4, dims=SMALL_DIMS)
        small.load_config(START_FILE)
        links = small.get_links()
        small.close()
        _therm[dims] = tile(links, SMALL_DIMS, [b // s for b, s in zip(dims, SMALL_DIMS)])
    return torch.from_numpy(_therm[dims]).cuda()


def _links(case, gen):
    """thermalised links, a short drift away, where the lattice is a multiple
    of the thermalised one; unit links with fluctuations elsewhere"""
    ncol, dims = case["ncol"], _dims(case)
    vol = math.prod(dims)
    noise = _normal(gen, vol, 5, ncol, ncol)
    if ncol == 4 and case["kind"] != "op" and not any(b % s for b, s in zip(dims, SMALL_DIMS)):
        return _therm_links(dims) + 0.01 * noise
    return torch.eye(ncol, device="cuda", dtype=torch.complex128) + 0.1 * noise


def _inputs(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    ncol, vol = case["ncol"], math.prod(_dims(case))
    links = _links(case, gen)
    field = _normal(gen, vol, 16, ncol, ncol) if case["kind"] != "traj" else None
    mom = _normal(gen, vol, 5, ncol, ncol) if case["kind"] == "kick" else None
    return links, field, mom


def _theta(ncol):
    """parameters of the learned force: the production ones (U(4)) or those of
    the U(2) workload"""
    root = os.path.dirname(os.path.abspath(susy_amd.__file__))
    return np.load(os.path.join(root, "configs", "surrogate_u4_split_theta.npy"))


def prepare(case, seed):
    ncol = case["ncol"]
    links, field, mom = _inputs(case, seed)
    lat = susy_amd.Lattice(ncol, iseed=1000 + seed, **_params(case))
    lat.set_links(links.cpu().numpy())
    state = {"case": case, "lat": lat}
    if case["kind"] == "op":
        # Twist_Fermion fields in the library's layout: planes of V numbers
        state["src"] = field.reshape(lat.V, -1).t().contiguous().reshape(16, ncol, ncol, lat.V)
        state["dst"] = torch.zeros_like(state["src"])
        state["args"] = (lat.h, ctypes.c_void_p(state["src"].data_ptr()),
                         ctypes.c_void_p(state["dst"].data_ptr()), case["sign"])
        torch.cuda.synchronize()
    elif case["kind"] == "kick":
        lat.set_mom(mom.cpu().numpy())
        coef = lat.rhmc()
        state["shifts"], state["amps"] = coef[16 + case["first"]:31], coef[1 + case["first"]:16]
        state["src"] = lat.tf_alloc(1)
        state["sol"] = lat.tf_alloc(15 - case["first"])
        lat.tf_upload(state["src"], field.cpu().numpy())
    elif case["form"] == "split":
        lat.sg_init(1)
        lat.sg_set_params(_theta(ncol))
        lat.set_split(9, 2)
    return state


# ---------------------------------------------------------------------
# One pass

def run(state):
    case, lat = state["case"], state["lat"]
    if case["kind"] == "op":
        lat._check(lat.L.susy_fermion_op_noalloc(*state["args"]))
        return state["dst"]
    if case["kind"] == "kick":
        fp32 = case["form"] == "fp32"
        lat.congrad_multi(state["src"], state["sol"], state["shifts"], 5000, 1e-10,
                          susy_amd.FORM_FP32 if fp32 else susy_amd.FORM_FP64)
        norm = lat.fermion_force(EPS, state["sol"], state["amps"])
        mom = lat.get_mom()
        return {"mom": mom.astype(np.complex64), "norm": np.float32(norm)} if fp32 else \
            {"mom": mom, "norm": norm}
    split = case["form"] == "split"
    stats = lat.update(susy_amd.FORM_FP32 | susy_amd.FORM_SURROGATE | susy_amd.FORM_SPLIT
                       if split else susy_amd.FORM_FP64)
    # the action's parts at the start and the end, and the new links and momenta
    out = {"actions": stats[11:23].copy(), "links": lat.get_links(), "mom": lat.get_mom()}
    if split:
        out = {"actions": out["actions"].astype(np.float32),
               "links": out["links"].astype(np.complex64),
               "mom": out["mom"].astype(np.complex64)}
    return out


def work(case):
    n, vol = case["ncol"], math.prod(_dims(case))
    size = 16 if case["kind"] == "op" or case["form"] == "fp64" else 8
    mat, prod = n * n * size * vol, 8 * n ** 3 * vol
    if case["kind"] == "op":
        # source, destination and links once; 160 matrix products per site
        return {"bytes": 37 * mat, "flops": 160 * prod}
    # per iteration: D and D^dagger (two operators' products; p, D p and the
    # links read, D p and A p written), the updates of r and p; `iters` is
    # the iteration count met on these inputs
    return {"bytes": case["iters"] * (11 * 16 + 2 * 5) * mat, "flops": case["iters"] * 320 * prod}


# ---------------------------------------------------------------------
# The same in 64 bits, in plain torch

class _Exact:
    """Fields over the lattice, [t][z][y][x][...], for one set of links
    [5][t][z][y][x][N][N]."""

    def __init__(self, case, links):
        self.dims, self.n = _dims(case), case["ncol"]
        self.shape = self.dims[::-1]
        nx, ny, nz, nt = self.dims
        t, z, y, x = np.meshgrid(np.arange(nt), np.arange(nz), np.arange(ny), np.arange(nx),
                                 indexing="ij")
        lex = (x + nx * (y + ny * (z + nz * t))).ravel()
        odd = ((x + y + z + t) & 1).ravel() == 1
        self.site = torch.from_numpy(np.where(odd, (lex + lex.size) // 2, lex // 2)).cuda()
        self.t = torch.arange(nt, device="cuda").reshape(nt, 1, 1, 1, 1, 1)
        self.G = _params(case)["G"]
        self.set(self.field(links))

    def field(self, a):
        """(V, k, N, N) in site order -> [k][t][z][y][x][N][N]"""
        a = a[self.site].reshape(*self.shape, a.shape[1], self.n, self.n)
        return a.permute(4, 0, 1, 2, 3, 5, 6).contiguous()

    def sites(self, f):
        """the inverse of field()"""
        k = f.shape[0]
        f = f.permute(1, 2, 3, 4, 0, 5, 6).reshape(-1, k, self.n, self.n)
        out = torch.empty_like(f)
        out[self.site] = f
        return out

    def set(self, U):
        self.U = U
        self.inv, det = [], []
        for a in range(5):
            w, d = self._inverse(U[a])
            self.inv.append(w)
            det.append(d)
        self.pd = {}
        for a in range(5):
            for b in range(5):
                if a != b:
                    self.pd[a, b] = (det[a].conj() * det[b] * self.sh(det[b], E[a]).conj() *
                                     self.sh(det[a], E[b]))

    def _inverse(self, m):
        """inverse and determinant by elimination (links are near unitary: no
        pivoting); the determinant keeps two trailing unit axes"""
        n = self.n
        aug = torch.cat([m, torch.eye(n, device="cuda", dtype=m.dtype).expand_as(m)], -1)
        rows, det = [aug[..., i, :] for i in range(n)], 1
        for k in range(n):
            piv = rows[k][..., k:k + 1]
            det = det * piv
            rows[k] = rows[k] / piv
            rows = [r if i == k else r - r[..., k:k + 1] * rows[k] for i, r in enumerate(rows)]
        return torch.stack(rows, -2)[..., n:], det.unsqueeze(-1)

    def sh(self, f, d):
        """f at x + d"""
        return torch.roll(f, [-d[3], -d[2], -d[1], -d[0]], [0, 1, 2, 3])

    def fe(self, f, d):
        """a fermion field at x + d: antiperiodic in t"""
        tt = self.t + d[3]
        sign = torch.where((tt < 0) | (tt >= self.shape[0]), -1.0, 1.0).double()
        return self.sh(f, d) * sign

    def D(self, v):
        U, mm = self.U, torch.matmul

        def H(m):
            return m.mH

        def neg(d):
            return tuple(-i for i in d)

        def add(*ds):
            return tuple(sum(i) for i in zip(*ds))

        def tr(m):
            return m.diagonal(dim1=-2, dim2=-1).sum(-1)[..., None, None]

        eta, psi = v[0], v[1:6]
        chi, p = {}, 6
        for a in range(5):
            for b in range(a + 1, 5):
                chi[a, b], chi[b, a] = v[p], -v[p]
                p += 1
        one = torch.eye(self.n, device="cuda", dtype=v.dtype)
        out = []
        acc = 0
        for a in range(5):
            m = neg(E[a])
            acc = acc + 0.5 * (mm(psi[a], H(U[a])) - mm(H(self.sh(U[a], m)), self.fe(psi[a], m)))
        T = [tr(mm(self.inv[a], psi[a])) for a in range(5)]
        te = tr(eta)
        for (a, b), pd in self.pd.items():
            acc = acc + 0.5 * self.G * pd * (T[b] + self.fe(T[a], E[b])) * one
        out.append(acc)
        for b in range(5):
            acc = 0.5 * (mm(self.fe(eta, E[b]), H(U[b])) - mm(H(U[b]), eta))
            s = 0
            for a in range(5):
                if a == b:
                    continue
                m = neg(E[a])
                acc = acc + mm(self.sh(U[a], E[b]), chi[a, b]) - \
                    mm(self.fe(chi[a, b], m), self.sh(U[a], m))
                s = s + te * self.pd[a, b] + self.fe(te * self.pd[b, a], m)
            out.append(acc - 0.5 * self.G * s * self.inv[b])
        for a in range(5):
            for b in range(a + 1, 5):
                acc = mm(U[a], self.fe(psi[b], E[a])) - mm(psi[b], self.sh(U[a], E[b])) - \
                    mm(U[b], self.fe(psi[a], E[b])) + mm(psi[a], self.sh(U[b], E[a]))
                ab = add(E[a], E[b])
                for c in range(5):
                    if c in (a, b):
                        continue
                    d, e = [k for k in range(5) if k not in (a, b, c)]
                    perm = (a, b, c, d, e)
                    s = (-1) ** sum(perm[i] > perm[j] for i in range(5) for j in range(i + 1, 5))
                    acc = acc + s * (
                        mm(self.fe(chi[d, e], add(ab, E[c])), H(self.sh(U[c], ab))) -
                        mm(H(self.sh(U[c], neg(E[c]))), self.fe(chi[d, e], ab)))
                out.append(acc)
        return torch.stack(out)

    def Ddag(self, v):
        return -self.D(v.mH.contiguous()).mH

    def solve(self, src, shifts, stop=1e-26, most=2000):
        """(D^dag D + shift_j)^-1 src, multi-shift conjugate gradient"""
        k, s0 = len(shifts), shifts[0]
        x = [torch.zeros_like(src) for _ in range(k)]
        ps = [src.clone() for _ in range(k)]
        r, z, zold = src.clone(), [1.0] * k, [1.0] * k
        alpha, beta, live = 0.0, 1.0, list(range(k))
        rr = first = float(src.abs().square().sum())
        for _ in range(most):
            Ap = self.Ddag(self.D(ps[0])) + s0 * ps[0]
            new_beta = rr / float((ps[0].conj() * Ap).real.sum())
            znew = [1.0] * k
            for j in live[1:]:
                ds = shifts[j] - s0
                znew[j] = z[j] * zold[j] * beta / (
                    new_beta * alpha * (zold[j] - z[j]) + zold[j] * beta * (1 + ds * new_beta))
            r = r - new_beta * Ap
            rr_new = float(r.abs().square().sum())
            new_alpha = rr_new / rr
            for j in live:
                x[j] += new_beta * (znew[j] / z[j]) * ps[j]
                ps[j] = znew[j] * r + new_alpha * (znew[j] / z[j]) ** 2 * ps[j]
            zold, z = z, znew
            alpha, beta, rr = new_alpha, new_beta, rr_new
            live = [j for j in live if j == 0 or z[j] ** 2 * rr > stop * first]
            if rr <= stop * first:
                break
        return x

    def force(self, sols, amps):
        """dS/dUbar of sum_j amp_j <src, (D^dag D + shift_j)^-1 src>"""
        U0 = self.U
        pairs = [(x, self.D(x)) for x in sols]
        F = torch.zeros_like(U0)
        for (x, px), amp in zip(pairs, amps):
            U = U0.clone().requires_grad_(True)
            self.set(U)
            S = -2.0 * amp * (px.conj() * self.D(x)).real.sum()
            F += torch.autograd.grad(S, U)[0] / 2
        self.set(U0)
        return F


def exact(case, seed):
    vol, ncol = math.prod(_dims(case)), case["ncol"]
    if case["kind"] == "traj" or (case["kind"] == "kick" and vol * ncol ** 3 > 230000):
        return None                      # minutes of solves in plain torch
    if case["kind"] == "kick" and not any(b % s for b, s in zip(_dims(case), SMALL_DIMS)) \
            and ncol == 4:
        return None                      # over a thousand iterations
    links, field, mom = _inputs(case, seed)
    X = _Exact(case, links)
    v = X.field(field)
    if case["kind"] == "op":
        got = X.sites(X.D(v) if case["sign"] == 1 else X.Ddag(v))
        return got.reshape(vol, -1).t().contiguous().reshape(16, ncol, ncol, vol)
    lat = susy_amd.Lattice(ncol, **dict(_params(case), dims=(2, 2, 2, 2)))
    coef = lat.rhmc()                    # the rational approximation's table
    lat.close()
    sols = X.solve(v, [float(s) for s in coef[16 + case["first"]:31]])
    F = X.force(sols, coef[1 + case["first"]:16])
    new = X.sites(X.field(mom) - EPS * F).cpu().numpy()
    return {"mom": new, "norm": EPS * float(F.abs().square().sum()) ** 0.5 / vol}
