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
