"""GPU test of the FP64 final pass's logarithm: with c(k) = 0 and vext = 0 the gradient is
w 2 rho0 xi kT ln(xi^2), compared with the logarithm in extended precision of the rounded xi^2.

Tolerance: at most 0.57 units in the last place from the logarithm, 1/2 from each of the five
products with it and the one behind: 4 eps of each value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def values(rng, n):
    """xi^2 next to 1, at and around the edges of the table's 1/256 intervals of [1/2, 1), over many
    binades (above the threshold of the vanishing density), and of ordinary size."""
    edge = 0.5 + (2 * np.arange(128) + 1) / 512.0
    parts = [1.0 + rng.uniform(-1, 1, 200) * 2.0 ** -rng.integers(1, 52, 200),
             np.concatenate([e * (1.0 + s * 2.0 ** -50) for e in (edge, 2 * edge) for s in (-8, -1, 0, 1, 8)]),
             2.0 ** rng.uniform(-38, 120, 400), rng.uniform(0.0, 4.0, 800) + 1e-9]
    y = np.concatenate(parts)
    y = np.concatenate([y, [1.0, 0.5, 2.0, 0.25, 1.0 - 2.0 ** -53, 1.0 + 2.0 ** -52]])
    return np.sqrt(np.resize(y, n))


@pytest.mark.parametrize("mmax", [0, 1, 3, 5])
def test_logarithm(mmax):
    from mdft import ck
    from mdft.gpu import Engine
    kT = 2.4777
    table = ck.synthetic_ck(mmax, 256, 0.1, seed=3, n0=0.0333)
    table.c[:] = 0.0
    n = (16, 12, 15) if mmax < 3 else (4, 5, 6)
    eng = Engine(n, [0.5 * v for v in n], mmax, 2, kT, 0.0333, "fp64")
    eng.set_ck(table)
    eng.set_vext(np.zeros(eng.N * eng.no))
    xi = values(np.random.default_rng(mmax), eng.N * eng.no)
    _, df = eng.energy_and_gradient(xi)
    w = np.tile(eng.quadrature()[2], eng.N)
    rho0 = 0.0333 / (8.0 * np.pi ** 2 / 2)
    lg = np.log((xi * xi).astype(np.longdouble))
    ref = w * 2.0 * rho0 * xi * kT * lg
    eng.close()
    assert np.all(np.abs(df - ref) <= 4.0 * np.finfo(np.float64).eps * np.abs(ref))
