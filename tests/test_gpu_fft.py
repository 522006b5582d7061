"""GPU test of the batched FFT: the projection field after the forward transforms
(mdft_excess_stage 2) against numpy's FFT of the field before them (stage 1), for line
lengths with every radix, on each axis, with few and with many columns.

Tolerance: an FFT of N points is exact to about eps log2 N of the result's 2-norm; five
times that is allowed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = (16, 18, 20, 24, 25, 27, 30, 32, 36, 40, 45, 48, 50, 54, 60, 64, 72, 75, 80, 81, 90, 96, 100, 108, 120, 125,
           128, 144, 150, 160, 180, 192, 200, 240, 256, 1, 6, 15, 135, 250)


@pytest.mark.parametrize("precision,mmax", [("fp64", 0), ("fp64", 1), ("fp64", 2), ("fp64", 5), ("fp32", 1),
                                            ("fp32", 2), ("fp32", 4)])
def test_forward_transform_of_every_length(precision, mmax):
    from mdft import ck
    from mdft.gpu import Engine
    eps = np.finfo(np.float64 if precision == "fp64" else np.float32).eps
    table = ck.synthetic_ck(mmax, 1024, 0.05, seed=3, n0=0.0333)
    for i, n in enumerate(LENGTHS):
        other = [(5, 3), (4, 9), (2, 2)][i % 3]
        for axis in range(3):
            shape = list(other)
            shape.insert(axis, n)
            print(f"[fft] {precision} mmax={mmax} {shape}", flush=True)
            eng = Engine(shape, [0.5 * v for v in shape], mmax, 2, 2.4777, 0.0333, precision)
            eng.set_ck(table)
            eng.set_vext(np.zeros(eng.N * eng.no))
            xi = 1.0 + 0.3 * np.random.default_rng(n + axis).uniform(-1, 1, eng.N * eng.no)
            p = eng.excess_stage(xi, 1).reshape(shape[2], shape[1], shape[0], -1)
            got = eng.excess_stage(xi, 2).reshape(p.shape)
            ref = np.fft.ifftn(p, axes=(0, 1, 2)) * eng.N
            err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
            assert err <= 5.0 * eps * max(1.0, np.log2(eng.N)), (shape, err)
            eng.close()


@pytest.mark.parametrize("precision,mmax,shape", [
    ("fp64", 0, (2, 640, 3)), ("fp64", 1, (3, 2, 648)), ("fp64", 1, (2, 1250, 5)), ("fp64", 1, (1250, 3, 2)),
    ("fp64", 1, (3, 1, 1215)), ("fp32", 1, (2, 3, 1280)), ("fp32", 2, (3, 750, 2)), ("fp32", 2, (2500, 2, 1)),
    ("fp32", 2, (1, 2, 2500)), ("fp32", 2, (2, 2430, 3))])
def test_long_axes_of_few_projections(precision, mmax, shape):
    """Lines whose full batch of columns is more than the LDS holds: the forward transform against numpy's, and
    the evaluation, whose transforms are of fewer numbers per point, against the oracle at the engine's parity bars."""
    from mdft import ck
    from mdft.gpu import Engine
    from oracle import oracle as O
    eps = np.finfo(np.float64 if precision == "fp64" else np.float32).eps
    bar = 1e-10 if precision == "fp64" else 1e-5
    print(f"[fft] {precision} mmax={mmax} {shape}", flush=True)
    table = ck.synthetic_ck(mmax, 1024, 0.05, seed=3, n0=0.0333)
    length = [0.5 * v for v in shape]
    eng = Engine(shape, length, mmax, 2, 2.4777, 0.0333, precision)
    ora = O.Oracle(shape, length, mmax, 2, 2.4777, 0.0333)
    for e in (eng, ora):
        e.set_ck(table)
    rng = np.random.default_rng(sum(shape))
    xi = 1.0 + 0.3 * rng.uniform(-1, 1, eng.N * eng.no)
    vext = rng.uniform(-2.0, 5.0, eng.N * eng.no)
    eng.set_vext(vext)
    p = eng.excess_stage(xi, 1).reshape(shape[2], shape[1], shape[0], -1)
    got = eng.excess_stage(xi, 2).reshape(p.shape)
    ref = np.fft.ifftn(p, axes=(0, 1, 2)) * eng.N
    assert np.linalg.norm(got - ref) <= 5.0 * eps * np.log2(eng.N) * np.linalg.norm(ref)
    parts, df = eng.energy_and_gradient(xi)
    pref, dref = ora.energy_and_gradient(xi, vext)
    eng.close()
    assert np.abs(parts - pref).max() <= bar * np.abs(pref).max()
    assert np.abs(df - dref).max() <= bar * np.abs(dref).max()


@pytest.mark.parametrize("precision,mmax,shape", [("fp64", 1, (2, 1280, 2)), ("fp64", 3, (2, 2, 648)), ("fp32", 3, (2, 1280, 2))])
def test_longer_axes_are_refused(precision, mmax, shape):
    from mdft import ck
    from mdft.gpu import Engine, MdftError
    print(f"[fft] refused: {precision} mmax={mmax} {shape}", flush=True)
    eng = Engine(shape, [0.5 * v for v in shape], mmax, 2, 2.4777, 0.0333, precision)
    eng.set_ck(ck.synthetic_ck(mmax, 1024, 0.05, seed=3, n0=0.0333))
    eng.set_vext(np.zeros(eng.N * eng.no))
    with pytest.raises(MdftError):
        eng.energy_and_gradient(np.ones(eng.N * eng.no))
    eng.close()
