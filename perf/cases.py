"""The performance cases: what programs on this library spend their time in, call by call.

A program that computes light scattering by a particle makes the particle's
operator (GpuMatVec), applies it some hundreds of times inside a Krylov solve,
and evaluates incident fields, cross sections and Jones matrices around it.
Sizes are those of the library's tests and benchmark (the 280-dipole sphere,
the sphere 40 dipoles across on an 80^3 grid, the ellipsoid 64 x 48 x 32 with a
block of orientations, the sphere 128 across on 256^3) and generic ones; every
operator runs on the grid that the default rule picks for its box.

A case's "kind" says which call it is:
  apply   op.apply / op.apply_batch on device vectors (one matrix-vector
          product, or one for each right-hand side of a block)
  setup   a new particle: the operator from its dipole list, and its first product
  solve   one block of incident fields to polarisations (host arrays in and out,
          or device-resident)
  jones   Jones matrices of a solved particle on a grid of scattering angles
  fields  the incident fields of a block of orientations, and the cross
          sections of its solutions
"""
import functools
import math
from types import SimpleNamespace

import numpy as np
import torch

import dda_amd as D
from dda_amd import problem as P

GRID_UNIT = 5e-7

# kind, shape, box, nmat (materials), m (first refractive index), |m| kd, prec, nrhs,
# conj; for solves the method, mode, tolerance and whether the arrays are the
# host's; for jones the angle grid
_DEFAULTS = dict(nmat=1, m_re=1.5, m_im=0.1, mkd=0.5, prec=64, nrhs=1, conj=False)


def _case(name, kind, shape, bx, by, bz, **more):
    return {**_DEFAULTS, "name": name, "kind": kind, "shape": shape, "bx": bx, "by": by, "bz": bz, **more}


def listed():
    return [
        # the smallest: a sphere 8 across (16^3 grid), where the latency of a product counts
        _case("apply sphere 8", "apply", "ellipsoid", 8, 8, 8),
        # an ordinary single particle, sphere 40 across (80^3 grid), double precision
        _case("apply sphere 40", "apply", "ellipsoid", 40, 40, 40),
        # an ordinary ragged particle of two materials in single precision, the adjoint product of CGNR
        _case("apply ragged 47x35x59", "apply", "ellipsoid", 47, 35, 59, prec=32, nmat=2, conj=True),
        # sphere 128 across (256^3 grid), double precision: the product of a plain FP64 solve
        _case("apply sphere 128", "apply", "ellipsoid", 128, 128, 128),
        # the same in single precision, both polarisations as one block: the product of a mixed solve
        _case("block sphere 128 x2", "apply", "ellipsoid", 128, 128, 128, prec=32, nrhs=2),
        # 64 orientations of a small particle, both polarisations: the block of an orientation average
        _case("block ellipsoid 64 x128", "apply", "ellipsoid", 64, 48, 32, prec=32, nrhs=128, m_re=1.33, m_im=0.01,
              mkd=0.6),
        # the largest: a sphere 256 across (8.8 million dipoles, 512^3 grid)
        _case("apply sphere 256", "apply", "ellipsoid", 256, 256, 256, prec=32),
        # a stream of different particles: every one needs its operator and interaction tensor
        _case("setup ellipsoid 96", "setup", "ellipsoid", 96, 72, 60),
        # a whole solve through the host-array interface, double precision QMR-CS
        _case("solve sphere 40 qmr", "solve", "ellipsoid", 40, 40, 40, method="qmr", mode="fp64", eps=1e-10, host=True),
        # a whole mixed-precision block solve on device-resident fields
        _case("solve ellipsoid 64 x32", "solve", "ellipsoid", 64, 48, 32, nrhs=32, m_re=1.33, m_im=0.01, mkd=0.6,
              method="bicgstab", mode="mixed", eps=1e-10, host=False),
        # the scattering grid of the sphere 40 across, both polarisations (2 x 6 degree steps)
        _case("jones sphere 40", "jones", "ellipsoid", 40, 40, 40, nrhs=2, ntheta=91, nphi=61),
        # what surrounds the orientation block's solve
        _case("fields ellipsoid 64 x128", "fields", "ellipsoid", 64, 48, 32, nrhs=128, m_re=1.33, m_im=0.01, mkd=0.6),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: extents and block sizes spread over their logarithms, any shape."""
    kind = rng.choice(["apply"] * 6 + ["setup", "solve", "jones", "fields"])
    shape = rng.choice(["ellipsoid", "ellipsoid", "box", "cylinder"])
    big = {"apply": 200, "setup": 96, "solve": 40, "jones": 64, "fields": 96}[kind]
    n = _log(rng, 8, big)
    dims = [n] + [max(3, int(round(n * rng.uniform(0.4, 1.0)))) for _ in range(2)]
    if kind == "apply" and rng.random() < 0.15:  # a rod or fibre, long in one axis
        dims = [_log(rng, 100, 512)] + [rng.randint(6, 40) for _ in range(2)]
    rng.shuffle(dims)
    c = {**_DEFAULTS, "kind": kind, "shape": shape, "bx": dims[0], "by": dims[1], "bz": dims[2],
         "m_re": round(rng.uniform(1.2, 1.6), 3), "m_im": round(rng.uniform(0.01, 0.2), 3),
         "mkd": round(rng.uniform(0.3, 0.6), 3)}
    cells = dims[0] * dims[1] * dims[2]
    if kind == "apply":
        c.update(prec=rng.choice([32, 64]), nmat=rng.choice([1, 1, 2]), conj=rng.random() < 0.25)
        most = max(1, min(128, 8_000_000 // cells))
        c["nrhs"] = rng.choice([1, min(2, most), _log(rng, 1, most)])
    elif kind == "setup":
        c.update(prec=rng.choice([32, 64]))
    elif kind == "solve":
        c.update(m_re=round(rng.uniform(1.2, 1.5), 3), nrhs=_log(rng, 1, 16), eps=1e-10, host=rng.random() < 0.5,
                 method=rng.choice(["qmr", "bicgstab"]), mode=rng.choice(["fp64", "mixed"]))
    elif kind == "jones":
        c.update(nrhs=2, ntheta=rng.randint(31, 181), nphi=rng.randint(1, 61))
    else:
        c.update(nrhs=_log(rng, 1, max(2, min(128, 16_000_000 // cells))))
    return c


# ---------------------------------------------------------------------------------------------
# The particle of a case
# ---------------------------------------------------------------------------------------------

def _mask(c):
    """[z, y, x] truth values: the cell-centre rule per axis."""
    h = [(np.arange(c[b]) + 0.5 - c[b] / 2) / (c[b] / 2) for b in ("bx", "by", "bz")]
    x, y, z = h[0][None, None, :] ** 2, h[1][None, :, None] ** 2, h[2][:, None, None] ** 2
    if c["shape"] == "box":
        return np.ones((c["bz"], c["by"], c["bx"]), bool)
    if c["shape"] == "cylinder":  # axis along x
        return np.broadcast_to(y + z <= 1.0, (c["bz"], c["by"], c["bx"]))
    return x + y + z <= 1.0


@functools.lru_cache(maxsize=1)
def _particle(shape, bx, by, bz, nmat, m_re, m_im, mkd):
    """Geometry and parameters: the particle's dipole list is data that a program reads once."""
    c = dict(shape=shape, bx=bx, by=by, bz=bz)
    zyx = np.argwhere(_mask(c))
    m = complex(m_re, m_im)
    mats = [m, 1.3 * m][:nmat]
    mat = (zyx[:, 0] > bz // 3).astype(np.uint8) if nmat > 1 else None
    g = P.DipoleGeometry(zyx[:, ::-1], mat, mats, GRID_UNIT)
    return P.DDAParams(g, 2 * math.pi * GRID_UNIT * abs(m) / mkd)


def _params(c):
    return _particle(c["shape"], c["bx"], c["by"], c["bz"], c["nmat"], c["m_re"], c["m_im"], c["mkd"])


@functools.lru_cache(maxsize=1)
def _ctx():
    return D.Context(0)


def _orientations(c, seed):
    """(props, pols) [nrhs, 3]: seeded directions, both polarisations of each in turn."""
    dirs = P.directions((c["nrhs"] + 1) // 2, seed)
    out = [(p, q) for d in dirs for p, p1, p2 in [P.beam_pols(d)] for q in (p1, p2)][:c["nrhs"]]
    return np.array([p for p, _ in out]), np.array([q for _, q in out])


def _couple(c, params, props, pols):
    both = [P.couple_constants(params, p, q) for p, q in zip(props, pols)]
    return np.array([a for a, _ in both]), np.array([s for _, s in both])


def _vectors(c, params, n, seed, prec):
    """n seeded dipole vectors on the GPU, components uniform in [-1, 1), zero padding."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    real = torch.float64 if prec == 64 else torch.float32
    v = torch.rand((n, 3, params.vec_stride, 2), generator=gen, device="cuda", dtype=real) * 2 - 1
    v[:, :, params.nv:] = 0
    return torch.view_as_complex(v).reshape(-1)


def _operator(c, params):
    g = params.geometry
    return D.GpuMatVec(_ctx(), g.pos, g.mat, g.box, g.grid_unit, params.wave_num, precision=c["prec"],
                       grid=params.grid, nmat=len(g.materials))


def prepare(case, seed):
    c, params = case, _params(case)
    s = SimpleNamespace(case=c, params=params, seed=seed)
    s.props, s.pols = _orientations(c, seed)
    s.cc, s.cs = _couple(c, params, s.props, s.pols)
    k, n = c["nrhs"], params.vec_size
    if c["kind"] != "setup":
        s.op = _operator(c, params)
        s.op.set_couple_constants_batch(s.cs)
    if c["kind"] in ("apply", "setup"):
        s.x = _vectors(c, params, k, seed, c["prec"])
        s.y = torch.empty_like(s.x)
    elif c["kind"] == "solve":
        s.solver = D.SOLVER_CLASSES[c["method"]](s.op, mode=c["mode"])
        s.einc = np.array([P.einc_plane(params, p, q) for p, q in zip(s.props, s.pols)])
        if not c["host"]:
            s.einc = torch.from_numpy(s.einc.reshape(-1)).cuda()
            s.pol = torch.empty_like(s.einc)
    elif c["kind"] == "jones":
        s.pol = _vectors(c, params, k, seed, 64)
        s.frame = P.beam_pols(s.props[0])
    else:
        s.pol = _vectors(c, params, k, seed, 64)
        s.einc = torch.empty_like(s.pol)
    return s


def _at(t):
    """A torch tensor as the device vector that an entry point takes."""
    return SimpleNamespace(ptr=t.data_ptr())


def run(s):
    c, k = s.case, s.case["nrhs"]
    if c["kind"] == "apply":
        s.op.apply_batch(s.x.data_ptr(), s.y.data_ptr(), k, conj=c["conj"])
        return s.y
    if c["kind"] == "setup":
        op = _operator(c, s.params)
        op.set_couple_constants(s.cs[0])
        op.apply(s.x.data_ptr(), s.y.data_ptr())
        op.close()
        return s.y
    if c["kind"] == "solve":
        if c["host"]:
            return s.solver.get_pol_vecs(s.einc, c["eps"])[0]
        s.solver.solve_device(_at(s.einc), _at(s.pol), k, c["eps"])
        return s.pol
    if c["kind"] == "jones":
        prop, pol1, pol2 = s.frame
        step = [math.pi / max(1, c["ntheta"] - 1), 2 * math.pi / c["nphi"]]
        return D.jones(s.op, _at(s.pol), 0, prop, pol1, pol2, c["ntheta"], 0.0, step[0], c["nphi"], 0.0, step[1])
    D.incident_plane(s.op, s.props, s.pols, out=_at(s.einc))
    cext, cabs = D.cross_sections(s.op, _at(s.pol), _at(s.einc), k, s.cc)
    return {"einc": s.einc, "cext": cext, "cabs": cabs}


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------------

def _fft_flops(n):
    return 5.0 * n * math.log2(n)


def _product(params, c, esz, k):
    """(bytes, flops) of k products with one tensor: vectors in and out, the eighth of the transformed
    tensor that its symmetry leaves, the index arrays; transforms of the occupied rows, planes and columns."""
    (gx, gy, gz), (bx, by, bz) = params.grid, params.geometry.box
    octant = 6 * (gx // 2 + 1) * (gy // 2 + 1) * (gz // 2 + 1) * esz
    flops = k * 3 * 2 * (by * bz * _fft_flops(gx) + bz * gx * _fft_flops(gy) + gx * gy * _fft_flops(gz))
    flops += k * gx * gy * gz * 9 * 8
    return octant + k * 2 * 3 * params.nv * esz + 4 * params.nv, flops


def work(case):
    c, params = case, _params(case)
    esz = c["prec"] // 4
    nv, k = params.nv, c["nrhs"]
    if c["kind"] == "apply":
        b, f = _product(params, c, esz, k)
    elif c["kind"] == "setup":
        b, f = _product(params, c, esz, 1)
        gx, gy, gz = params.grid
        # an eighth of the tensor suffices: six components, each axis in turn
        b += 6 * (gx // 2 + 1) * (gy // 2 + 1) * (gz // 2 + 1) * esz + 13 * nv
        f += 6 / 4 * (gy * gz * _fft_flops(gx) + gx * gz * _fft_flops(gy) + gx * gy * _fft_flops(gz))
    elif c["kind"] == "solve":
        # thirty products at the least, in the precision that the iteration runs in
        b, f = _product(params, c, 8 if c["mode"] == "mixed" else 16, k)
        b, f = 30 * b, 30 * f
    elif c["kind"] == "jones":
        q = 2 * c["ntheta"] * c["nphi"]
        b, f = 2 * 3 * nv * 16 + 4 * nv + q * 64, q * nv * 24.0
    else:
        b, f = k * 3 * nv * 16 * 2 + 4 * nv, k * nv * 60.0
    return {"bytes": float(b), "flops": float(f)}


# ---------------------------------------------------------------------------------------------
# The same in 64 bits, in plain torch
# ---------------------------------------------------------------------------------------------

_COMPONENTS = [(0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)]


class _Exact:
    """A = I - sqrt(a) G sqrt(a) by torch's own transforms, complex double."""

    def __init__(self, c, params):
        self.params, self.c = params, c
        gx, gy, gz = params.grid
        self.grid = (gz, gy, gx)
        p = torch.from_numpy(params.geometry.pos.astype(np.int64)).cuda()
        self.at = (p[:, 2] * gy + p[:, 1]) * gx + p[:, 0]
        self.mat = torch.from_numpy(params.geometry.mat.astype(np.int64)).cuda()
        self.keep = [self.tensor(a) for a in range(6)] if gx * gy * gz <= 1 << 24 else None

    def tensor(self, comp):
        gz, gy, gx = self.grid
        off = []
        for ax, n in enumerate((gx, gy, gz)):
            i = torch.arange(n, device="cuda", dtype=torch.float64)
            i = torch.where(i <= n // 2, i, i - n)
            shape = [1, 1, 1]
            shape[2 - ax] = n
            off.append(i.reshape(shape))
        bx, by, bz = self.params.geometry.box
        r = torch.sqrt(off[0] ** 2 + off[1] ** 2 + off[2] ** 2)
        inside = (off[0].abs() < bx) & (off[1].abs() < by) & (off[2].abs() < bz) & (r > 0)
        r = torch.where(inside, r, torch.ones_like(r))
        mu, nu = _COMPONENTS[comp]
        kr = self.params.kd * r
        q = off[mu] * off[nu] / (r * r)
        re, im = (3 - kr * kr) * q, -3 * kr * q
        if mu == nu:
            re, im = re + kr * kr - 1, im + kr
        g = torch.complex(re, im) * torch.polar(torch.where(inside, 1 / r ** 3, torch.zeros_like(r)), kr)
        return torch.fft.fftn(g)

    def product(self, x, s):
        """x, s: [3, nv] (vector, sqrt of the polarisabilities in grid units)."""
        gz, gy, gx = self.grid
        spec = []
        for a in range(3):
            w = torch.zeros(gz * gy * gx, dtype=torch.complex128, device="cuda")
            w[self.at] = x[a] * s[a]
            spec.append(torch.fft.fftn(w.reshape(self.grid)))
        out = [0, 0, 0]
        for comp, (mu, nu) in enumerate(_COMPONENTS):
            t = self.keep[comp] if self.keep else self.tensor(comp)
            out[mu] = out[mu] + t * spec[nu]
            if mu != nu:
                out[nu] = out[nu] + t * spec[mu]
        del spec
        return torch.stack([x[a] - s[a] * torch.fft.ifftn(out[a]).reshape(-1)[self.at] for a in range(3)])

    def roots(self, cs):
        s = torch.from_numpy(np.ascontiguousarray(cs)).cuda() * GRID_UNIT ** -1.5
        return s[self.mat].T.contiguous()

    def solve(self, b, s):
        """BiCGStab, restarted on the residual until it is 1e-13 of the right-hand side."""
        x = torch.zeros_like(b)
        for _ in range(6):
            r0 = b - self.product(x, s)
            goal = float(torch.linalg.vector_norm(r0))
            if goal <= 1e-13 * float(torch.linalg.vector_norm(b)):
                break
            r, p, d, rho = r0.clone(), r0.clone(), torch.zeros_like(b), torch.vdot(r0.reshape(-1), r0.reshape(-1))
            for _ in range(400):
                v = self.product(p, s)
                alpha = rho / torch.vdot(r0.reshape(-1), v.reshape(-1))
                t = r - alpha * v
                w = self.product(t, s)
                omega = torch.vdot(w.reshape(-1), t.reshape(-1)) / torch.vdot(w.reshape(-1), w.reshape(-1))
                d = d + alpha * p + omega * t
                r = t - omega * w
                if float(torch.linalg.vector_norm(r)) <= 1e-6 * goal:
                    break
                new = torch.vdot(r0.reshape(-1), r.reshape(-1))
                p = r + (new / rho * alpha / omega) * (p - omega * v)
                rho = new
            x = x + d
        return x


def _padded(params, v):
    out = torch.zeros((3, params.vec_stride), dtype=torch.complex128, device="cuda")
    out[:, :params.nv] = v
    return out.reshape(-1)


def _phases(params, q):
    """exp(i k q . r) at the dipoles, r in grid units from the box's centre."""
    at = params.geometry.pos - (np.array(params.geometry.box) - 1) / 2
    t = params.kd * (torch.from_numpy(at).cuda() @ torch.from_numpy(np.ascontiguousarray(q, np.float64)).cuda().T)
    return torch.polar(torch.ones_like(t), t)


def exact(case, seed):
    c, params = case, _params(case)
    props, pols = _orientations(c, seed)
    cc, cs = _couple(c, params, props, pols)
    k, nv = c["nrhs"], params.nv
    if c["kind"] in ("apply", "setup"):
        x = _vectors(c, params, k, seed, c["prec"]).to(torch.complex128).reshape(k, 3, -1)[:, :, :nv]
        e, out = _Exact(c, params), []
        for r in range(k):
            v = x[r].conj() if c["conj"] else x[r]
            y = e.product(v.contiguous(), e.roots(cs[r]))
            out.append(_padded(params, y.conj() if c["conj"] else y))
        return torch.cat(out)
    if c["kind"] == "solve":
        e, out = _Exact(c, params), []
        for r in range(k):
            s = e.roots(cs[r])
            b = s * torch.from_numpy(P.einc_plane(params, props[r], pols[r])).cuda().reshape(3, -1)[:, :nv]
            out.append(_padded(params, s * e.solve(b, s) * GRID_UNIT ** 3))
        out = torch.cat(out)
        return out.reshape(k, -1).cpu().numpy() if c["host"] else out
    p = _vectors(c, params, k, seed, 64).reshape(k, 3, -1)[:, :, :nv]
    wave = params.wave_num
    if c["kind"] == "fields":
        cext, cabs, einc = [], [], []
        mat = torch.from_numpy(params.geometry.mat.astype(np.int64)).cuda()
        for r in range(k):
            e = _phases(params, props[r:r + 1])[:, 0][None, :] * torch.from_numpy(pols[r]).cuda()[:, None]
            w = torch.from_numpy(-np.imag(1 / cc[r]) - 2 / 3 * wave ** 3).cuda()[mat].T
            einc.append(_padded(params, e))
            cext.append(float((p[r] * e.conj()).imag.sum()) * 4 * math.pi * wave)
            cabs.append(float((w * p[r].abs() ** 2).sum()) * 4 * math.pi * wave)
        return {"einc": torch.cat(einc), "cext": np.array(cext), "cabs": np.array(cabs)}
    # Jones matrices: field components perpendicular and parallel to the scattering plane of both solutions
    prop, pol1, pol2 = P.beam_pols(props[0])
    nt, nf = c["ntheta"], c["nphi"]
    th = np.repeat(np.arange(nt) * (math.pi / max(1, nt - 1)), nf)[:, None]
    ph = np.tile(np.arange(nf) * (2 * math.pi / nf), nt)[:, None]
    lie = np.cos(ph) * pol2 + np.sin(ph) * pol1
    dirs, perp, par = (np.cos(th) * prop + np.sin(th) * lie, np.sin(ph) * pol2 - np.cos(ph) * pol1,
                       -np.sin(th) * prop + np.cos(th) * lie)
    field = []
    for q in np.array_split(np.arange(nt * nf), max(1, nt * nf * nv // 100_000_000)):
        f = _phases(params, dirs[q]).conj()
        field.append(1j * wave ** 2 * (p.reshape(6, nv) @ f).reshape(2, 3, -1))
    field = torch.cat(field, 2).transpose(1, 2).cpu().numpy()
    e = np.array([[(field[r] * perp).sum(1), (field[r] * par).sum(1)] for r in range(2)])  # [solution][perp, par]
    cp, sp = np.cos(ph[:, 0]), np.sin(ph[:, 0])
    out = [cp * e[1, 1] + sp * e[0, 1], sp * e[1, 1] - cp * e[0, 1], cp * e[1, 0] + sp * e[0, 0],
           sp * e[1, 0] - cp * e[0, 0]]
    return np.stack(out, axis=1).reshape(-1, 2, 2)
