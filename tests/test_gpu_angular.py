"""GPU test of the angular kernels at the edges of their tiles: numbers of points just below,
at and above a workgroup's, for every order, against the oracle.

Tolerances: the projections are sums over the no orientations, exact to about sqrt(no) eps
of their 2-norm (the FP32 kernel rounds its terms first): 4 sqrt(no) eps.  Energies and
gradients: the engine's parity bars, 1e-10 in FP64 and 1e-5 in FP32."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 1, 15, 16, 18, 30, 32, 36, 64, 75, 125, 128, 135, 256, 270 points
GRIDS = ((1, 1, 1), (5, 3, 1), (4, 2, 2), (3, 3, 2), (5, 2, 3), (4, 8, 1), (3, 3, 4), (4, 4, 4), (5, 5, 3), (5, 5, 5),
         (16, 4, 2), (5, 9, 3), (16, 16, 1), (9, 5, 6))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("mmax", range(6))
def test_tiles_of_points(precision, mmax):
    from mdft import ck
    from mdft.gpu import Engine
    from oracle import oracle as O
    eps = np.finfo(np.float64 if precision == "fp64" else np.float32).eps
    bar = 1e-10 if precision == "fp64" else 1e-5
    table = ck.synthetic_ck(mmax, 512, 0.05, seed=11, n0=0.0333)
    for n in GRIDS:
        length = [0.5 * v for v in n]
        print(f"[angular] {precision} mmax={mmax} {n}", flush=True)
        eng = Engine(n, length, mmax, 2, 2.4777, 0.0333, precision)
        ora = O.Oracle(n, length, mmax, 2, 2.4777, 0.0333)
        for e in (eng, ora):
            e.set_ck(table)
        rng = np.random.default_rng(sum(n))
        xi = 1.0 + 0.3 * rng.uniform(-1, 1, eng.N * eng.no)
        vext = rng.uniform(-2.0, 5.0, eng.N * eng.no)
        eng.set_vext(vext)
        ref = ora.excess_stage(xi, 1).reshape(eng.N, -1)
        got = eng.excess_stage(xi, 1)
        assert np.linalg.norm(got - ref) <= 4.0 * np.sqrt(eng.no) * eps * np.linalg.norm(ref), n
        parts, df = eng.energy_and_gradient(xi)
        pref, dref = ora.energy_and_gradient(xi, vext)
        # (F_id and F_ext are sums of terms of both signs: relative to the largest part)
        assert np.abs(parts - pref).max() <= bar * np.abs(pref).max(), (n, parts, pref)
        assert np.abs(df - dref).max() <= bar * np.abs(dref).max(), n
        eng.close()


@pytest.mark.parametrize("mmax", range(6))
def test_fast_step_on_partial_tiles(mmax):
    """The fast minimiser's evaluation (FP32 iterate of the scaled variables, FP32 gradient, products
    of the gradient) where the last tile is not full, against the oracle.  The products are FP64
    sums over the gradient as stored: exact to about sqrt(n) eps of their terms' 2-norm."""
    import ctypes as C
    from mdft import ck
    from mdft.gpu import DEVICE_PTRS, DF_FP32, SCALED_VARS, XI_FP32, DeviceBuffer, Engine
    from oracle import oracle as O
    table = ck.synthetic_ck(mmax, 512, 0.05, seed=11, n0=0.0333)
    dp = C.POINTER(C.c_double)
    for n in GRIDS:
        length = [0.5 * v for v in n]
        print(f"[angular] step mmax={mmax} {n}", flush=True)
        eng = Engine(n, length, mmax, 2, 2.4777, 0.0333, "fp32")
        ora = O.Oracle(n, length, mmax, 2, 2.4777, 0.0333)
        for e in (eng, ora):
            e.set_ck(table)
        rng = np.random.default_rng(sum(n))
        vext = rng.uniform(-2.0, 5.0, eng.N * eng.no)
        eng.set_vext(vext)
        w = eng.quadrature()[2]
        s = np.tile(np.sqrt(w / w.mean()), eng.N)
        u = (s * (1.0 + 0.3 * rng.uniform(-1, 1, eng.N * eng.no))).astype(np.float32)
        vecs = [rng.standard_normal(u.size).astype(np.float32) for _ in range(2)]
        du, dg, *dv = (DeviceBuffer(eng, 4 * u.size) for _ in range(4))
        for b, v in ((du, u), (dv[0], vecs[0]), (dv[1], vecs[1])):
            b.upload(v)
        parts, dots = np.zeros(3), np.zeros(3)
        ptrs = (C.c_void_p * 3)(dv[0].ptr, dg.ptr, dv[1].ptr)
        eng._check(eng.lib.mdft_energy_and_gradient_dots(eng._h, du.ptr, parts.ctypes.data_as(dp), dg.ptr,
                                                         DEVICE_PTRS | DF_FP32 | SCALED_VARS | XI_FP32, 3, ptrs,
                                                         dots.ctypes.data_as(dp)))
        df = dg.download(np.float32).astype(np.float64)
        pref, dref = ora.energy_and_gradient(u.astype(np.float64) / s, vext)
        dref = dref / s
        assert np.abs(parts - pref).max() <= 1e-5 * np.abs(pref).max(), (n, parts, pref)
        assert np.abs(df - dref).max() <= 1e-5 * np.abs(dref).max(), n
        for got, v in zip(dots, (vecs[0].astype(np.float64), df, vecs[1].astype(np.float64))):
            assert abs(got - df @ v) <= 1e-15 * np.sqrt(df.size) * (np.abs(df) @ np.abs(v)), (n, got, df @ v)
        eng.close()


# more points than 2048 workgroups take in one tile each, and a last tile that is not full
LARGE = {0: (80, 81, 90), 1: (75, 75, 54), 2: (40, 45, 45), 3: (36, 45, 45), 4: (25, 32, 30), 5: (25, 27, 25)}


@pytest.mark.parametrize("mmax", range(6))
def test_fast_step_of_several_tiles_per_workgroup(mmax):
    """The same evaluation where a workgroup takes a second and later tile, the short last one among them: sums, tables
    and prefetched values that carry over.  The bars are those above; the energies' FP32 terms are summed in FP64
    over the tiles, so they hold for any number of points."""
    import ctypes as C
    from mdft import ck
    from mdft.gpu import DEVICE_PTRS, DF_FP32, SCALED_VARS, XI_FP32, DeviceBuffer, Engine
    from oracle import oracle as O
    n = LARGE[mmax]
    print(f"[angular] step mmax={mmax} {n}", flush=True)
    table = ck.synthetic_ck(mmax, 512, 0.05, seed=11, n0=0.0333)
    dp = C.POINTER(C.c_double)
    length = [0.5 * v for v in n]
    eng = Engine(n, length, mmax, 2, 2.4777, 0.0333, "fp32")
    ora = O.Oracle(n, length, mmax, 2, 2.4777, 0.0333)
    for e in (eng, ora):
        e.set_ck(table)
    rng = np.random.default_rng(mmax)
    vext = rng.uniform(-2.0, 5.0, eng.N * eng.no)
    eng.set_vext(vext)
    w = eng.quadrature()[2]
    s = np.tile(np.sqrt(w / w.mean()), eng.N)
    u = (s * (1.0 + 0.3 * rng.uniform(-1, 1, eng.N * eng.no))).astype(np.float32)
    vecs = [rng.standard_normal(u.size).astype(np.float32) for _ in range(2)]
    pref, dref = ora.energy_and_gradient(u.astype(np.float64) / s, vext)
    dref = dref / s
    du, dg, *dv = (DeviceBuffer(eng, 4 * u.size) for _ in range(4))
    for b, v in ((du, u), (dv[0], vecs[0]), (dv[1], vecs[1])):
        b.upload(v)
    ptrs = (C.c_void_p * 3)(dv[0].ptr, dg.ptr, dv[1].ptr)
    first = None
    for _ in range(2):
        parts, dots = np.zeros(3), np.zeros(3)
        eng._check(eng.lib.mdft_energy_and_gradient_dots(eng._h, du.ptr, parts.ctypes.data_as(dp), dg.ptr,
                                                         DEVICE_PTRS | DF_FP32 | SCALED_VARS | XI_FP32, 3, ptrs,
                                                         dots.ctypes.data_as(dp)))
        df = dg.download(np.float32).astype(np.float64)
        assert np.abs(parts - pref).max() <= 1e-5 * np.abs(pref).max(), (parts, pref)
        assert np.abs(df - dref).max() <= 1e-5 * np.abs(dref).max()
        for got, v in zip(dots, (vecs[0].astype(np.float64), df, vecs[1].astype(np.float64))):
            assert abs(got - df @ v) <= 1e-15 * np.sqrt(df.size) * (np.abs(df) @ np.abs(v)), (got, df @ v)
        if first is None:
            first = parts, dots, df
    assert all(np.array_equal(a, b) for a, b in zip(first, (parts, dots, df)))
    eng.close()
