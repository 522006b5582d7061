"""GPU test of the two forms of the q-space rotations, against the oracle: grids of which all pairs,
some and hardly any have rotation matrices with chopped entries (planes of special phi, the cone
around the polar axis), with full and partial tiles of either form, alone or as the last of an interval.

Tolerances: rotations and contraction are sums of at most 4 (mmax + 1)^2 products of FP64, 1e-13 of the
largest, and a chop too many or too few changes an entry by 6e-8 of its size: 1e-10 of the field's largest
modulus, and of energies and gradients, finds it.  In FP32
1e-5, the precision's parity bar."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one axis along z (theta = 0 only), along x (theta = pi/2), all planes special, a long polar axis (small
# angles), unequal lengths, an even cube
GRIDS = (((1, 1, 12), (3.0, 3.0, 6.0)), ((12, 1, 1), (6.0, 3.0, 3.0)), ((2, 2, 2), (3.0, 3.0, 3.0)),
         ((5, 3, 40), (24.0, 20.0, 4.0)), ((9, 10, 8), (4.1, 5.3, 3.7)), ((12, 12, 12), (6.0, 6.0, 6.0)))


@pytest.mark.parametrize("precision,mmax", [("fp64", m) for m in range(2, 7)] + [("fp32", m) for m in range(1, 6)])
def test_rotation_forms(precision, mmax):
    from mdft import ck
    from mdft.gpu import Engine
    from oracle import oracle as O
    bar = 1e-10 if precision == "fp64" else 1e-5
    table = ck.synthetic_ck(mmax, 1024, 0.05, seed=5 + mmax, n0=0.0333)
    for n, length in GRIDS:
        print(f"[qspace] {precision} mmax={mmax} {n}", flush=True)
        eng = Engine(n, length, mmax, 2, 2.4777, 0.0333, precision)
        ora = O.Oracle(n, length, mmax, 2, 2.4777, 0.0333)
        for e in (eng, ora):
            e.set_ck(table)
        rng = np.random.default_rng(sum(n))
        xi = 1.0 + 0.3 * rng.uniform(-1, 1, eng.N * eng.no)
        vext = rng.uniform(-2.0, 5.0, eng.N * eng.no)
        eng.set_vext(vext)
        ref = ora.excess_stage(xi, 3)
        got = eng.excess_stage(xi, 3)
        assert np.abs(got - ref).max() <= bar * np.abs(ref).max(), n
        parts, df = eng.energy_and_gradient(xi)
        pref, dref = ora.energy_and_gradient(xi, vext)
        assert np.abs(parts - pref).max() <= bar * np.abs(pref).max(), (n, parts, pref)
        assert np.abs(df - dref).max() <= bar * np.abs(dref).max(), n
        eng.close()


@pytest.mark.parametrize("mmax", [3, 4, 5, 6])
def test_small_entries_are_chopped(mmax):
    """Directions 1e-14 off the plane theta = pi/2: entries of the rotation that vanish there are up to 5e-14, which the
    chop sets to 0.  Kept, they change the field by some 1e-14 of it.  Rounding: the square root of the at most
    4 (mmax + 1)^2 products per sum, eps each, once for the rotations and once for the contraction; of the largest
    modulus among the directions off the special planes."""
    from mdft import ck
    from mdft.gpu import Engine
    from oracle import oracle as O
    n, length = (25, 30, 12), (3.0, 4.1, 3.0e14)
    table = ck.synthetic_ck(mmax, 1024, 0.05, seed=5 + mmax, n0=0.0333)
    eng = Engine(n, length, mmax, 2, 2.4777, 0.0333, "fp64")
    ora = O.Oracle(n, length, mmax, 2, 2.4777, 0.0333)
    for e in (eng, ora):
        e.set_ck(table)
    xi = 1.0 + 0.3 * np.random.default_rng(mmax).uniform(-1, 1, eng.N * eng.no)
    eng.set_vext(np.zeros(xi.size))
    ref = ora.excess_stage(xi, 3)
    got = eng.excess_stage(xi, 3)
    eng.close()
    ref, got = (v.reshape(12, 30, 25, -1)[1:, [y for y in range(30) if y % 15], 1:] for v in (ref, got))
    err = np.abs(got - ref).max() / np.abs(ref).max()
    print(f"[qspace] mmax={mmax} {err:.2e}", flush=True)
    assert err <= 4.0 * (mmax + 1) * np.finfo(np.float64).eps


# more than 4096 pairs, below which FP64 keeps one form for all: a plane along z and one across (all directions
# special; of theta = pi/2 only), a long polar axis, unequal lengths, an even box
LARGE_GRIDS = (((1, 90, 96), (3.0, 31.0, 35.0)), ((96, 90, 1), (35.0, 31.0, 3.0)), ((6, 5, 300), (24.0, 20.0, 24.0)),
               ((18, 20, 25), (4.1, 5.3, 3.7)), ((24, 20, 18), (12.0, 10.0, 9.0)))


@pytest.mark.parametrize("mmax", range(3, 7))
def test_rotation_forms_of_large_grids(mmax):
    from mdft import ck
    from mdft.gpu import Engine
    from oracle import oracle as O
    table = ck.synthetic_ck(mmax, 1024, 0.05, seed=5 + mmax, n0=0.0333)
    for n, length in LARGE_GRIDS:
        print(f"[qspace] mmax={mmax} {n}", flush=True)
        eng = Engine(n, length, mmax, 2, 2.4777, 0.0333, "fp64")
        ora = O.Oracle(n, length, mmax, 2, 2.4777, 0.0333)
        for e in (eng, ora):
            e.set_ck(table)
        rng = np.random.default_rng(sum(n))
        xi = 1.0 + 0.3 * rng.uniform(-1, 1, eng.N * eng.no)
        vext = rng.uniform(-2.0, 5.0, eng.N * eng.no)
        eng.set_vext(vext)
        ref = ora.excess_stage(xi, 3)
        got = eng.excess_stage(xi, 3)
        assert np.abs(got - ref).max() <= 1e-10 * np.abs(ref).max(), n
        parts, df = eng.energy_and_gradient(xi)
        pref, dref = ora.energy_and_gradient(xi, vext)
        assert np.abs(parts - pref).max() <= 1e-10 * np.abs(pref).max(), (n, parts, pref)
        assert np.abs(df - dref).max() <= 1e-10 * np.abs(dref).max(), n
        eng.close()
