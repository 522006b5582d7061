"""The work that programs have this framework do, as a list of measurable cases.

A case is a dict of plain values.  `listed()` gives the standing ones, `draw(rng)` one
more of the same ranges, `prepare(case, seed)` what a program holds before the call,
`run(state)` one pass through the public entry points, `exact(case, seed)` the same
results in 64 bits from plain torch, and `work(case)` the bytes and operations that the
pass cannot do without.

Kinds:
  energy  one energy_and_gradient(F, dF) on device-resident fields
  step    the fast minimiser's evaluation: FP32 iterate of the scaled variables, FP32
          gradient, products of the new gradient with stored vectors
  solve   a minimisation of a fixed number of evaluations from the cold start
  vext    the external potential of a solute, Lennard-Jones and Poisson electrostatics
  host    energy_and_gradient on host arrays, as a host program's plug-in calls it

The results of FP32 evaluations are returned in FP32, the precision that they carry; those
of FP64 evaluations in FP64.
"""
from __future__ import annotations

import ctypes as C
import functools
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mdft-dev_general_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

from mdft import ck as _ck  # noqa: E402
from mdft import gpu as _gpu  # noqa: E402
from mdft import minimize as _minimize  # noqa: E402
from mdft import warmstart as _warmstart  # noqa: E402
from mdft.constants import QFACT, kT_of, spce  # noqa: E402
from mdft.workloads import Solute  # noqa: E402

MRSO = 2            # molecular symmetry order of water
N0 = 0.0333         # bulk density of the workloads, 1/A^3
KT = kT_of(298.0)   # kJ/mol
DQ, NQ = 0.05, 1024  # c(k) table: step (1/A) and rows
EPS64, EPS32 = float(np.finfo(np.float64).eps), float(np.finfo(np.float32).eps)
MAXEVAL = 10        # evaluations of a `solve` pass
RCUT = 10.0         # Lennard-Jones cutoff, A


# ---------------------------------------------------------------------------- the cases

def _case(name, kind, n, spacing, mmax, precision="fp64", **more):
    return {"name": name, "kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "spacing": spacing, "mmax": mmax,
            "precision": precision, **more}


def listed():
    return [
        # the smallest call of a program that couples many small systems, or of a unit test:
        # a dozen short launches and one read-back
        _case("call_16_m1", "energy", (16, 16, 16), 0.5, 1),
        # the neutral sphere of the first workload (24 A, 48^3, mmax 1): the lowest useful order
        _case("lj_sphere_48_m1", "energy", (48, 48, 48), 0.5, 1),
        # the ion of the second workload (32 A, 96^3, mmax 3) in the reference's precision
        _case("na_ion_96_m3", "energy", (96, 96, 96), 1.0 / 3.0, 3),
        # the 20-atom solute (40 A, 128^3, mmax 5) in the reference's precision: one step of
        # the plain minimisation, and the confirming evaluation of the fast one
        _case("solute20_128_m5", "energy", (128, 128, 128), 0.3125, 5),
        # one evaluation of the warm start's training set (24 A, 64^3, mmax 3) in FP32
        _case("warmstart_64_m3_fp32", "energy", (64, 64, 64), 0.375, 3, "fp32"),
        # an odd box with an odd number of points, as a user's box and spacing give
        _case("odd_box_45_75_81_m2", "energy", (45, 75, 81), 0.4, 2),
        # the headline's unit of work: the fast minimiser's evaluation of the 20-atom solute
        _case("minimiser_128_m5", "step", (128, 128, 128), 0.3125, 5, "fp32"),
        # the same in a flat box whose sides are no powers of two, at an even order
        _case("minimiser_75_90_100_m4", "step", (100, 90, 75), 0.35, 4, "fp32"),
        # a whole fast solve, cut after ten evaluations: cold start, directions, line search
        _case("solve_64_m3", "solve", (64, 64, 64), 0.375, 3, "fp32", fast=True),
        # the external potential of a 20-atom solute, computed once per solute
        _case("vext_solute20_96_m3", "vext", (96, 96, 96), 1.0 / 3.0, 3, natom=20),
        # the same around a globule: many atoms, of which each point sees few within the cutoff
        _case("vext_globule_64_m3", "vext", (64, 64, 64), 0.6, 3, natom=1000),
        # the evaluation called from a host program with its own arrays (the plug-in's form)
        _case("host_48_m3", "host", (48, 48, 48), 0.5, 3),
    ]


# sides that factor into 2, 3 and 5, as the transforms need
_SIDES = [16, 18, 20, 24, 25, 27, 30, 32, 36, 40, 45, 48, 50, 54, 60, 64, 72, 75, 80, 81, 90, 96, 100, 108, 120, 125, 128]


def _orientations(mmax):
    return (mmax + 1) * (2 * mmax + 1) * (2 * (mmax // MRSO) + 1)


def draw(rng):
    kind = rng.choice(["energy", "energy", "energy", "step", "step", "solve", "vext", "host"])
    # field elements (points times orientations) allowed: what keeps a pass below the largest listed one
    most = {"energy": 128 ** 3 * 330, "step": 128 ** 3 * 330, "solve": 64 ** 3 * 84, "vext": 64 ** 3 * 84,
            "host": 48 ** 3 * 84}[kind]
    while True:
        mmax = rng.randint(1, 5)
        side = math.exp(rng.uniform(math.log(16), math.log(128)))
        near = [s for s in _SIDES if side / 1.5 <= s <= side * 1.5]
        n = [rng.choice(near) for _ in range(3)]
        if n[0] * n[1] * n[2] * _orientations(mmax) <= most:
            break
    precision = {"step": "fp32", "vext": "fp64", "host": "fp64"}.get(kind) or rng.choice(["fp64", "fp32"])
    more = {}
    if kind == "vext":
        more["natom"] = round(math.exp(rng.uniform(0.0, math.log(1000))))
    if kind == "solve":
        more["fast"] = precision == "fp32"
    c = _case("", kind, n, round(rng.uniform(0.3125, 0.5), 4), mmax, precision, **more)
    del c["name"]
    return c


# ---------------------------------------------------------------------------- inputs

def _sizes(case):
    n = (case["nx"], case["ny"], case["nz"])
    return n, tuple(v * case["spacing"] for v in n), n[0] * n[1] * n[2], _orientations(case["mmax"])


@functools.lru_cache(maxsize=None)
def _table(mmax):
    """c(k) of the solvent: a file that a program reads once."""
    return _ck.synthetic_ck(mmax, NQ, DQ, seed=1000 + mmax, n0=N0, mrso=MRSO)


def _quadrature(mmax):
    """theta, phi, psi of each orientation, its weight, and the theta weights (which sum to 1)."""
    x, w = np.polynomial.legendre.leggauss(mmax + 1)
    x, w = x[::-1], w[::-1] / 2.0
    nphi, npsi = 2 * mmax + 1, 2 * (mmax // MRSO) + 1
    th, ph, ps = np.meshgrid(np.arccos(x), 2 * np.pi * np.arange(nphi) / nphi,
                             2 * np.pi / MRSO * np.arange(npsi) / npsi, indexing="ij")
    weight = np.broadcast_to(w[:, None, None], th.shape) * 8 * np.pi ** 2 / (nphi * npsi * MRSO)
    return th.ravel(), ph.ravel(), ps.ravel(), weight.ravel(), w


def _solute(case, seed):
    """Atoms in a ball at the centre of the box: positions, charges (neutral), sigma, epsilon."""
    rng = np.random.default_rng(seed)
    length = np.array(_sizes(case)[1])
    natom = case.get("natom", max(1, min(12, int(length.min() / 8.0) ** 2)))
    radius = min(0.25 * length.min(), 2.0 * natom ** (1.0 / 3.0))
    d = rng.normal(size=(natom, 3))
    xyz = length / 2 + d / np.linalg.norm(d, axis=1)[:, None] * radius * rng.uniform(size=(natom, 1)) ** (1.0 / 3.0)
    q = rng.normal(0.0, 0.4, natom)
    return Solute(xyz, q - q.mean() if natom > 1 else np.array([1.0]), rng.uniform(2.5, 4.0, natom),
                  rng.uniform(0.2, 1.0, natom))


def _points(n, length):
    """Grid points [N, 3], x fastest, on the GPU."""
    ax = [torch.arange(n[k], dtype=torch.float64, device="cuda") * (length[k] / n[k]) for k in range(3)]
    z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    return torch.stack([x.reshape(-1), y.reshape(-1), z.reshape(-1)], dim=1)


def _fields(case, seed):
    """vext [N, no] (kJ/mol) with cores, a polar shell and a dependence on every angle, and a
    density near exp(-vext / kT), as a minimisation meets it: xi [N, no]."""
    n, length, N, no = _sizes(case)
    sol = _solute(case, seed)
    pts = _points(n, length)
    box = torch.tensor(length, dtype=torch.float64, device="cuda")
    basis_r = torch.zeros(N, 6, dtype=torch.float64, device="cuda")
    for a in range(len(sol.q)):
        d = pts - torch.tensor(sol.xyz[a], device="cuda")
        d -= box * torch.round(d / box)
        r2 = (d * d).sum(1).clamp_min(1e-3)
        s6 = (sol.sig[a] ** 2 / r2) ** 3
        basis_r[:, 0] += 4 * 0.8 * math.sqrt(sol.eps[a]) * (s6 * s6 - s6)
        soft = (r2 + 2.0).rsqrt()
        basis_r[:, 1:4] += (60.0 * sol.q[a]) * d * (soft ** 3)[:, None]
        basis_r[:, 4] += 4.0 * sol.q[a] * soft ** 2
        basis_r[:, 5] -= 3.0 * sol.q[a] * soft ** 3
    th, ph, ps, _, _ = _quadrature(case["mmax"])
    angle = np.stack([np.ones(no), np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th),
                      np.sin(th) ** 2 * np.cos(2 * ps), np.cos(th) * np.sin(2 * ps + ph)])
    vext = torch.matmul(basis_r, torch.tensor(angle, device="cuda")).clamp_max_(QFACT / 2)
    del basis_r, pts
    g = torch.Generator(device="cuda").manual_seed(seed)
    xi = torch.randn(N, no, dtype=torch.float64, device="cuda", generator=g).mul_(0.05).add_(1.0)
    for r in range(0, N, 1 << 18):
        v = vext[r:r + (1 << 18)]
        xi[r:r + (1 << 18)] *= torch.exp((v / KT).clamp(-3.0, 50.0) * -0.5)
    return vext, xi


def _scale(mmax):
    """s(io) of the scaled variables u = s xi: the square root of the weight over its mean."""
    w = _quadrature(mmax)[3]
    return torch.tensor(np.sqrt(w / w.mean()), device="cuda")


def _step_inputs(case, seed):
    vext, xi = _fields(case, seed)
    u = xi.mul_(_scale(case["mmax"])).float()
    del xi
    g = torch.Generator(device="cuda").manual_seed(seed + 1)
    vecs = [torch.randn(u.shape, dtype=torch.float32, device="cuda", generator=g) for _ in range(2)]
    return vext, u, vecs


# ---------------------------------------------------------------------------- the passes

class _Field(_gpu.DeviceBuffer):
    """A torch tensor as one of the engine's device fields."""

    def __init__(self, engine, tensor):
        self.engine, self.tensor = engine, tensor
        self.nbytes = tensor.numel() * tensor.element_size()
        self.ptr = C.c_void_p(tensor.data_ptr())

    def free(self):
        self.ptr = None


def _engine(case):
    n, length, _, _ = _sizes(case)
    return _gpu.Engine(n, length, case["mmax"], MRSO, KT, N0, case["precision"])


def prepare(case, seed):
    kind = case["kind"]
    eng = _engine(case)
    s = {"case": case, "engine": eng}
    if kind == "vext":
        s["solute"], s["solvent"] = _solute(case, seed), spce(N0)
        _, _, N, no = _sizes(case)
        s["vext"] = torch.empty(N, no, dtype=torch.float64, device="cuda")
        return s
    eng.set_ck(_table(case["mmax"]))
    if kind == "step":
        vext, u, vecs = _step_inputs(case, seed)
        s["xi"], s["df"], s["vecs"] = u, torch.empty_like(u), vecs
    else:
        vext, xi = _fields(case, seed)
        if kind == "host":
            s["xi"] = xi.reshape(-1).cpu().numpy()
        elif kind == "solve":
            s["xi"], s["g"] = xi, torch.empty_like(xi)
        else:
            s["xi"] = xi
            s["df"] = torch.empty(xi.shape, dtype=torch.float32 if case["precision"] == "fp32" else torch.float64,
                                  device="cuda")
    torch.cuda.synchronize()  # the engine has a stream of its own
    eng.set_vext(_Field(eng, vext))
    return s


def _parts(case, parts):
    return parts.astype(np.float32) if case["precision"] == "fp32" else parts


def run(state):
    case, eng = state["case"], state["engine"]
    kind = case["kind"]
    if kind == "vext":
        eng.compute_vext(state["solute"], state["solvent"], rcut=RCUT, electrostatics="poisson")
        eng._check(eng.lib.mdft_get_vext(eng._h, state["vext"].data_ptr(), _gpu.DEVICE_PTRS))
        return state["vext"]
    if kind == "host":
        parts, df = eng.energy_and_gradient(state["xi"])
        return {"F": parts, "dF": df}
    if kind == "solve":
        xi, g = _Field(eng, state["xi"]), _Field(eng, state["g"])
        _warmstart.cold_start(eng, xi)
        fast = case["fast"]
        r = _minimize.minimize(eng, xi, g=g, m=1, gtol=0.0, maxeval=MAXEVAL, fnoise=1e-6 if fast else 1e-7,
                               fp32_vectors=fast, fp32_iterate=fast, scaled=fast, step0="newton" if fast else 0.0,
                               ftol=1e-3, ftol_absolute=True)
        xi, F = state["xi"], np.array([r.F])
        return {"F": _parts(case, F), "xi": xi.float() if fast else xi}
    parts = np.zeros(3)
    pp = parts.ctypes.data_as(C.POINTER(C.c_double))
    if kind == "step":
        flags = _gpu.DEVICE_PTRS | _gpu.DF_FP32 | _gpu.SCALED_VARS | _gpu.XI_FP32
        df, dots = state["df"], np.zeros(3)
        vecs = (C.c_void_p * 3)(state["vecs"][0].data_ptr(), state["vecs"][1].data_ptr(), df.data_ptr())
        eng._check(eng.lib.mdft_energy_and_gradient_dots(eng._h, state["xi"].data_ptr(), pp, df.data_ptr(), flags, 3,
                                                         vecs, dots.ctypes.data_as(C.POINTER(C.c_double))))
        return {"F": _parts(case, parts), "dF": df, "products": dots.astype(np.float32)}
    flags = _gpu.DEVICE_PTRS | (_gpu.DF_FP32 if case["precision"] == "fp32" else 0)
    eng._check(eng.lib.mdft_energy_and_gradient(eng._h, state["xi"].data_ptr(), pp, state["df"].data_ptr(), flags))
    return {"F": _parts(case, parts), "dF": state["df"]}


# ---------------------------------------------------------------------------- bytes and operations

def work(case):
    n, _, N, no = _sizes(case)
    L = case["mmax"]
    H1, nth, nphi, npsi = L // MRSO + 1, L + 1, 2 * L + 1, 2 * (L // MRSO) + 1
    nmu = [m // MRSO + 1 for m in range(L + 1)]
    np_ = sum((2 * m + 1) * nmu[m] for m in range(L + 1))
    npc = sum((m // MRSO + 1) * (2 * (k // MRSO) + 1) for m in range(L + 1) for khi in range(-m, m + 1)
              for k in range(abs(khi), L + 1))
    fft = 5.0 * N * math.log2(N)  # one complex field
    # both angular transforms (a sum over psi, one over phi, one over theta each) and the local terms
    flops = N * (2 * (4 * no * H1 + 8 * nth * nphi * nphi * H1 + 4 * np_ * nth) + 40 * no)
    flops += 2 * np_ * fft
    # both rotations of every wave vector and the contraction with c
    flops += N * (2 * 8 * sum((2 * m + 1) ** 2 * nmu[m] for m in range(L + 1)) + 8 * npc)
    b = {"energy": 24 if case["precision"] == "fp64" else 20, "host": 24, "step": 24, "vext": 8}.get(case["kind"], 0)
    if case["kind"] == "vext":
        sphere = min(1.0, 4.0 / 3.0 * math.pi * RCUT ** 3 / (N * case["spacing"] ** 3))
        flops = N * no * (20.0 * case["natom"] * sphere) + no * fft / 2
    if case["kind"] == "solve":  # each evaluation, and each iteration's pass over the vectors
        x = 4 if case["fast"] else 8
        flops, b = MAXEVAL * flops, MAXEVAL * (4 * x + 4 * x)
    return {"bytes": float(N * no * b), "flops": float(flops)}


# ---------------------------------------------------------------------------- the results in 64 bits

def _wigner(m, a, b, theta):
    """d^m_{a b}(theta) by the explicit sum; theta a torch tensor (FP64)."""
    f = math.factorial
    c, s = torch.cos(theta / 2), torch.sin(theta / 2)
    out = torch.zeros_like(theta)
    for k in range(max(0, b - a), min(m + b, m - a) + 1):
        coef = (-1.0) ** (a - b + k) / (f(m + b - k) * f(k) * f(a - b + k) * f(m - a - k))
        out += coef * c ** (2 * m + b - a - 2 * k) * s ** (a - b + 2 * k)
    return out * math.sqrt(f(m + a) * f(m - a) * f(m + b) * f(m - b))


def _projections(L):
    return [(m, mup, mu2) for m in range(L + 1) for mup in range(-m, m + 1) for mu2 in range(m // MRSO + 1)]


def _transforms(L):
    """Dense forms of the two angular transforms: to projections [no, np], and back [np, no]
    (the values are the real part of conj(projections) times the latter)."""
    th, ph, ps, _, wt = _quadrature(L)
    nphi, npsi = 2 * L + 1, 2 * (L // MRSO) + 1
    weight = np.repeat(wt, nphi * npsi) / (nphi * npsi)
    theta = torch.tensor(th)
    fwd, back = [], []
    for m, mup, mu2 in _projections(L):
        d = _wigner(m, mup, MRSO * mu2, theta).numpy() * math.sqrt(2 * m + 1)
        wave = np.exp(1j * (mup * ph + MRSO * mu2 * ps))
        fwd.append(d * weight * wave)
        back.append(d * wave * (1.0 if mu2 == 0 else 2.0))
    return (torch.tensor(np.stack(fwd, axis=1), device="cuda"), torch.tensor(np.stack(back), device="cuda"))


def _dft3(x, sign):
    """Unnormalised transform of x [nz, ny, nx, k] over its first three axes."""
    for _ in range(3):
        n = x.shape[2]
        j = torch.arange(n, device="cuda")
        arg = (torch.outer(j, j) % n).double() * (sign * 2 * math.pi / n)
        x = torch.tensordot(torch.polar(torch.ones_like(arg), arg), x, dims=([1], [2]))
        # [nz, ny, nx] -> [kx, nz, ny] -> [ky, kx, nz] -> [kz, ky, kx]
    return x


def _waves(n, length):
    """Wave vectors of one axis, +pi/d on the Nyquist index."""
    m = np.arange(n)
    return 2 * np.pi / length * np.where(m <= n // 2, m, m - n)


def _single(z):
    """A default-kind complex value of the reference: rounded to single precision."""
    return z.float().double()


def _chop(re, im, eps):
    """The reference's chop: a component below eps becomes 0 and the other single precision."""
    small = re.abs() < eps
    re, im = torch.where(small, 0.0, re), torch.where(small, _single(im), im)
    small = im.abs() < eps
    return torch.complex(torch.where(small, _single(re), re), torch.where(small, 0.0, im))


def _ornstein_zernike(p, case):
    """The q-space step on the projections p [N, np]: each (q, -q) pair is rotated to the frame
    of q, contracted with c(|q|) and rotated back.  In place."""
    n, length, N, _ = _sizes(case)
    L = case["mmax"]
    where = {k: i for i, k in enumerate(_projections(L))}
    t = _table(L)
    cols = {(int(t.m[i]), int(t.n[i]), int(t.mu[i]) // MRSO, int(t.nu[i]) // MRSO, int(t.khi[i])): i
            for i in range(len(t.m))}
    table = torch.tensor(t.c, device="cuda")
    iz, iy, ix = np.meshgrid(*[np.arange(v) for v in reversed(n)], indexing="ij")
    mz, my, mx = (-iz) % n[2], (-iy) % n[1], (-ix) % n[0]
    g, gm = ((iz * n[1] + iy) * n[0] + ix).ravel(), ((mz * n[1] + my) * n[0] + mx).ravel()
    plane = n[0] * n[1]
    first = (iz.ravel() < mz.ravel()) | ((iz.ravel() == mz.ravel()) & (g % plane <= gm % plane))
    nyq = ((ix == n[0] // 2) | (iy == n[1] // 2) | (iz == n[2] // 2)).ravel()[first]
    q = np.stack([_waves(n[0], length[0])[ix.ravel()], _waves(n[1], length[1])[iy.ravel()],
                  _waves(n[2], length[2])[iz.ravel()]], axis=1)[first]
    g, gm = g[first], gm[first]
    for r in range(0, len(g), 1 << 16):
        a, b = (torch.tensor(v[r:r + (1 << 16)], device="cuda") for v in (g, gm))
        qv = torch.tensor(q[r:r + (1 << 16)], device="cuda")
        own = a == b
        own_nyq = own & torch.tensor(nyq[r:r + (1 << 16)], device="cuda")
        size, flat = qv.norm(dim=1), torch.hypot(qv[:, 0], qv[:, 1])
        theta = torch.atan2(flat, qv[:, 2])
        phi = torch.where(flat > 0, torch.atan2(qv[:, 1], qv[:, 0]),
                          torch.where(qv[:, 2] < 0, math.pi, 0.0).to(qv))
        eff = size / DQ
        iq = eff.floor().long()
        al = (eff - iq)[:, None]
        xa, xb = p[a], p[b]
        rot, va, vb = {}, {}, {}
        for m in range(L + 1):
            mup = range(-m, m + 1)
            d = torch.stack([torch.stack([_wigner(m, i, k, theta) for k in mup], -1) for i in mup], -2)
            e = torch.stack([i * phi for i in mup], -1)[:, :, None]
            rot[m] = R = _chop(d * torch.cos(e), -d * torch.sin(e), EPS32)
            for mu2 in range(m // MRSO + 1):
                at = [where[(m, i, mu2)] for i in mup]
                ya = (xa[:, at, None] * R).sum(1)
                yb = (xb[:, at, None] * R.flip(2)).sum(1) * (-1.0) ** m
                for khi in mup:
                    va[(m, khi, mu2)], vb[(m, khi, mu2)] = ya[:, khi + m], yb[:, khi + m]
        ga, gb = {}, {}
        for khi in range(-L, L + 1):
            order = range(abs(khi), L + 1)
            pair = [(k, nu2) for k in order for nu2 in range(-(k // MRSO), k // MRSO + 1)]
            wa = torch.stack([va[(k, khi, -nu2)] if nu2 < 0 else vb[(k, khi, nu2)].conj() for k, nu2 in pair], -1)
            wb = torch.stack([vb[(k, khi, -nu2)] if nu2 < 0 else va[(k, khi, nu2)].conj() for k, nu2 in pair], -1)
            sign = torch.tensor([(-1.0) ** abs(khi + MRSO * nu2) if nu2 < 0 else (-1.0) ** k for k, nu2 in pair],
                                dtype=torch.float64, device="cuda")
            for m in order:
                for mu2 in range(m // MRSO + 1):
                    c = table[:, [cols[(m, k, mu2, nu2, khi)] for k, nu2 in pair]].conj() * sign
                    c = al * c[iq + 1] + (1 - al) * c[iq]
                    for w, gam in ((wa, ga), (wb, gb)):
                        s = (c * w).sum(1)
                        gam[(m, khi, mu2)] = _chop(s.real, s.imag, EPS64)
        outa, outb = torch.empty_like(xa), torch.empty_like(xb)
        for m in range(L + 1):
            Rc = rot[m].conj()
            for mu2 in range(m // MRSO + 1):
                ya = torch.stack([ga[(m, k, mu2)] for k in range(-m, m + 1)], -1)[:, None, :]
                yb = torch.stack([gb[(m, k, mu2)] for k in range(-m, m + 1)], -1)[:, None, :]
                at = [where[(m, i, mu2)] for i in range(-m, m + 1)]
                outa[:, at] = (ya * Rc).sum(2)
                outb[:, at] = (yb * Rc.flip(2)).sum(2) * (-1.0) ** m
        outb = torch.where(own_nyq[:, None], outb.conj(), outb)
        p[a] = outa
        p[b] = outb  # of a pair q == -q the second store stays


def _exact_energy(case, vext, xi):
    """F parts (FP64) and, per block of points, dF: the ideal, external and excess terms."""
    n, length, N, no = _sizes(case)
    L = case["mmax"]
    rho0 = N0 / (8 * math.pi ** 2 / MRSO)
    dv = case["spacing"] ** 3
    w = torch.tensor(_quadrature(L)[3], device="cuda")
    fwd, back = _transforms(L)
    np_ = fwd.shape[1]
    p = torch.empty(N, np_, dtype=torch.complex128, device="cuda")
    step = 1 << 17
    for r in range(0, N, step):
        o = (xi[r:r + step] ** 2 - 1) * rho0
        p[r:r + step] = torch.complex(o @ fwd.real, o @ fwd.imag)
    shape = (n[2], n[1], n[0], -1)
    for k in range(0, np_, 16):
        p[:, k:k + 16] = _dft3(p[:, k:k + 16].reshape(shape), +1).reshape(N, -1)
    _ornstein_zernike(p, case)
    for k in range(0, np_, 16):
        p[:, k:k + 16] = _dft3(p[:, k:k + 16].reshape(shape), -1).reshape(N, -1) / N
    pre = -KT * 8 * math.pi ** 2 / MRSO / N0
    parts = torch.zeros(3, dtype=torch.float64, device="cuda")
    df = torch.empty(N, no, dtype=torch.float64, device="cuda")
    for r in range(0, N, step):
        x, ve, y = xi[r:r + step], vext[r:r + step], p[r:r + step]
        vexc = (y.real @ back.real + y.imag @ back.imag) * pre * w
        rho = x * x * rho0
        some = rho > EPS64
        lg = torch.log(torch.where(some, x * x, 1.0))
        rho_in = torch.where(some, rho, 0.0)
        parts[0] += KT * dv * (w * (rho_in * lg - rho_in + rho0)).sum()
        parts[1] += dv * (w * rho_in * ve).sum()
        parts[2] += 0.5 * dv * ((rho - rho0) * vexc).sum()
        df[r:r + step] = 2 * rho0 * x * (torch.where(some, w * (KT * lg + ve), 0.0) + vexc)
    return parts, df


def _exact_vext(case, seed):
    n, length, N, no = _sizes(case)
    sol, water = _solute(case, seed), spce(N0)
    th, ph, ps, _, _ = _quadrature(case["mmax"])
    ct, st, cp, sp, cs, ss = np.cos(th), np.sin(th), np.cos(ph), np.sin(ph), np.cos(ps), np.sin(ps)
    rot = np.array([[ct * cp * cs - sp * ss, -ct * cp * ss - sp * cs, st * cp],
                    [ct * sp * cs + cp * ss, -ct * sp * ss + cp * cs, st * sp], [-st * cs, st * ss, ct]])
    off = [torch.tensor(np.einsum("abo,b->oa", rot, np.array(s.r)), device="cuda") for s in water.sites]
    pts = _points(n, length)
    box = torch.tensor(length, dtype=torch.float64, device="cuda")
    out = torch.zeros(N, no, dtype=torch.float64, device="cuda")
    for s, site in enumerate(water.sites):
        if not site.eps > 0:
            continue
        here = {}  # orientations that put the site at the same place
        for o, at in enumerate(off[s].cpu().numpy()):
            here.setdefault(tuple(at), []).append(o)
        for at, which in here.items():
            pos = pts + torch.tensor(at, device="cuda")
            lj = torch.zeros(N, dtype=torch.float64, device="cuda")
            for a in range(len(sol.q)):
                d = pos - torch.tensor(sol.xyz[a], device="cuda")
                d -= box * torch.round(d / box)
                r2 = (d * d).sum(1).clamp_min(1e-12)
                sr6 = ((0.5 * (site.sig + sol.sig[a])) ** 2 / r2) ** 3
                lj += torch.where(r2 < RCUT ** 2, 4 * math.sqrt(site.eps * sol.eps[a]) * (sr6 * sr6 - sr6), 0.0)
            out[:, which] += lj[:, None]
    # cloud-in-cell charges, V(k) = 4 pi rho(k) / k^2, times the smeared charges of each orientation
    rho = torch.zeros(n[2], n[1], n[0], 1, dtype=torch.complex128, device="cuda")
    for x, q in zip(sol.xyz, sol.q):
        node = [math.floor(x[k] % length[k] / (length[k] / n[k])) % n[k] for k in range(3)]
        frac = [abs(x[k] / (length[k] / n[k]) - math.floor(x[k] / (length[k] / n[k]))) for k in range(3)]
        for corner in range(8):
            up = [corner >> k & 1 for k in range(3)]
            i = [(node[k] + up[k]) % n[k] for k in range(3)]
            rho[i[2], i[1], i[0]] += q * math.prod(frac[k] if up[k] else 1 - frac[k] for k in range(3))
    rho /= case["spacing"] ** 3
    half = n[0] // 2 + 1
    m = [np.arange(v) for v in n]
    m = [np.where(v < k // 2, v, v - k) for v, k in zip(m, n)]
    kp = torch.meshgrid(*[torch.tensor(2 * np.pi * m[k] / length[k], device="cuda") for k in (2, 1, 0)], indexing="ij")
    k2 = sum(v * v for v in kp)
    V = _dft3(rho, -1)[..., 0] * torch.where(k2 > EPS64, 4 * math.pi / k2.clamp_min(EPS64), 0.0)
    kv = torch.meshgrid(*[torch.tensor(_waves(n[k], length[k]), device="cuda") for k in (2, 1, 0)], indexing="ij")
    weight = torch.full((n[0],), 2.0, dtype=torch.float64, device="cuda")
    weight[0] = 1.0
    if n[0] % 2 == 0:
        weight[half - 1] = 1.0
    weight[half:] = 0.0
    V = V * torch.exp(-0.25 * sum(v * v for v in kv) / 2) * weight
    for o in range(0, no, 12):
        z = torch.zeros(n[2], n[1], n[0], min(12, no - o), dtype=torch.complex128, device="cuda")
        for s, site in enumerate(water.sites):
            at = off[s][o:o + 12]
            arg = kv[0][..., None] * at[:, 2] + kv[1][..., None] * at[:, 1] + kv[2][..., None] * at[:, 0]
            z += site.q * torch.polar(torch.ones_like(arg), arg)  # conj(sigma)
        z = _dft3(z * V[..., None], +1)
        out[:, o:o + 12] += QFACT / N * z.real.reshape(N, -1)
    return out.clamp_max_(QFACT / 2)


def exact(case, seed):
    kind = case["kind"]
    if kind == "solve":
        return None  # the iterates depend on every rounding before them
    if kind == "vext":
        return _exact_vext(case, seed)
    if kind != "step":
        vext, xi = _fields(case, seed)
        parts, df = _exact_energy(case, vext, xi)
        return {"F": parts, "dF": df.reshape(-1) if kind == "host" else df}
    vext, u, vecs = _step_inputs(case, seed)
    s = _scale(case["mmax"])
    parts, df = _exact_energy(case, vext, u.double() / s)
    df /= s
    dots = [sum((df[r:r + (1 << 17)] * v[r:r + (1 << 17)].double()).sum() for r in range(0, len(df), 1 << 17))
            for v in (*vecs, df)]
    return {"F": parts, "dF": df, "products": torch.stack(dots)}
