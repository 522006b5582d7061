"""GPU tests of calls that meet a full device: what the library then does without, and that it goes on after an
error.  Each runs in a process of its own, in which hipMalloc refuses what the test asks it to."""
import os
import subprocess
import sys
import textwrap

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SHIM = os.path.join(ROOT, "tests", "mock_hip", "_build", "liballoc_limit.so")

HEAD = f"""
import ctypes as C, sys
sys.path[:0] = [{ROOT!r}, {os.path.join(ROOT, "mdft-dev_general_amd")!r}]
limit = C.CDLL({SHIM!r}, mode=C.RTLD_GLOBAL)   # before the library
limit.limit_room.argtypes = limit.limit_size.argtypes = [C.c_size_t]
FULL = C.c_size_t(-1).value
import numpy as np
from mdft import ck, workloads
from mdft.constants import Site, Solvent
from mdft.gpu import DeviceBuffer, Engine, MdftError
from oracle import oracle as O
ENOMEM = -2
"""


def run(body, *args):
    if not os.path.exists(SHIM):
        subprocess.check_call(["make", "-C", os.path.dirname(os.path.dirname(SHIM))])
    r = subprocess.run([sys.executable, "-c", HEAD + textwrap.dedent(body), *map(str, args)], capture_output=True,
                       text=True, timeout=110)
    print(r.stdout[-3000:], r.stderr[-3000:], flush=True)
    assert r.returncode == 0 and "held" in r.stdout


@pytest.mark.parametrize("off_axis", [0, 1])
def test_vext_without_room_for_the_places(off_axis):
    """Sites on the molecule's axis are summed once per place, in a table of 9 MB here, where that and the Poisson
    fields (12 MB) fit; without it each orientation is summed, which gives the same to the rounding of sums of a few
    hundred terms and of the transforms (1e-9 of the largest value)."""
    run("""
    n, mmax = (24, 20, 18), 5
    length = [0.6 * v for v in n]
    sites = [(0.4, 2.6, 0.3, (0.0, 0.0, -0.6)), (-0.4, 3.0, 0.5, (0.0, 0.0, 0.7))]
    if int(sys.argv[1]):
        sites.append((0.2, 2.1, 0.1, (0.1, -0.7, 0.5)))
    solv = Solvent("test", 2, 0.0333, [Site(*s) for s in sites])
    rng = np.random.default_rng(1)
    q = rng.normal(0, 0.4, 12)
    sol = workloads.Solute(rng.uniform(0, 1, (12, 3)) * length, q, rng.uniform(2.0, 3.5, 12), rng.uniform(0.2, 0.9, 12))
    def engine():
        return Engine(n, length, mmax, 2, 2.4777, 0.0333, "fp64")
    ref = {}
    eng = engine()
    for kind in ("poisson", "none"):
        eng.compute_vext(sol, solv, rcut=7.0, electrostatics=kind)
        ref[kind] = eng.get_vext()
    eng.close()
    eng = engine()
    for kind, room in (("none", 6 << 20), ("poisson", 15 << 20)):
        eng.close()   # (and the blocks that it keeps)
        eng = engine()
        print(kind, "table refused" if kind == "none" else "fields refused beside the table", flush=True)
        before = limit.limit_failures()
        limit.limit_room(room)
        eng.compute_vext(sol, solv, rcut=7.0, electrostatics=kind)
        limit.limit_room(FULL)
        assert limit.limit_failures() > before
        got = eng.get_vext()
        clip = ref[kind].max()
        below = (ref[kind] < clip) | (got < clip)
        assert np.abs(got - ref[kind])[below].max() <= 1e-9 * max(1.0, np.abs(ref[kind][ref[kind] < clip]).max())
    eng.close()
    eng = engine()
    limit.limit_room(5 << 20)
    try:
        eng.compute_vext(sol, solv, rcut=7.0)
        raise SystemExit("a potential without room for its fields")
    except MdftError as e:
        assert e.code == ENOMEM, e
    limit.limit_room(FULL)
    eng.compute_vext(sol, solv, rcut=7.0)
    assert np.array_equal(eng.get_vext(), ref["poisson"])
    eng.close()
    print("held")
    """, off_axis)


def test_calls_after_a_refused_scratch_allocation():
    """A larger call whose scratch memory is refused, then the smaller one that ran before: the same results."""
    run("""
    n, mmax, N = (6, 5, 4), 2, 120
    eng = Engine(n, [0.5 * v for v in n], mmax, 2, 2.4777, 0.0333, "fp64")
    eng.set_ck(ck.synthetic_ck(mmax, 512, 0.05, seed=1, n0=0.0333))
    rng = np.random.default_rng(0)
    eng.set_vext(rng.uniform(-2.0, 5.0, N * eng.no))
    xi = 1.0 + 0.2 * rng.uniform(-1, 1, N * eng.no)
    parts, df = eng.energy_and_gradient(xi)
    npts = 5000
    p, f = DeviceBuffer(eng, 16 * npts * eng.np_), DeviceBuffer(eng, 8 * npts * eng.no)
    p.upload(rng.standard_normal(2 * npts * eng.np_))
    print("projections to angles", flush=True)
    before = limit.limit_failures()
    limit.limit_size(24 * ((npts + 3) // 4))
    try:
        eng._check(eng.lib.mdft_proj2angl(eng._h, p.ptr, npts, f.ptr))
        raise SystemExit("a transform without its scratch memory")
    except MdftError as e:
        assert e.code == ENOMEM and limit.limit_failures() > before, e
    limit.limit_size(0)
    again = eng.energy_and_gradient(xi)
    assert np.array_equal(again[0], parts) and np.array_equal(again[1], df)

    from mdft.warmstart import WarmStartNet
    net = WarmStartNet((5, 8, 2), (1, 3), (1, 1), seed=5)
    def buffers(n):
        N = n[0] * n[1] * n[2]
        b = DeviceBuffer(eng, 20 * N), DeviceBuffer(eng, 8 * N)
        for v in b:
            v.upload(rng.standard_normal(v.nbytes // 4).astype(np.float32))
        return b
    small, big = (4, 4, 4), (16, 16, 16)   # weight gradients in 1 and 4 slices of 2 8 27 + 2 sums
    sx, st = buffers(small)
    bx, bt = buffers(big)
    loss, grads = net.loss_grad(small, sx, st), net.get_grads()
    print("training step", flush=True)
    before = limit.limit_failures()
    limit.limit_size(4 * 4 * 434)
    try:
        net.loss_grad(big, bx, bt)
        raise SystemExit("a gradient without its scratch memory")
    except RuntimeError:
        assert limit.limit_failures() > before
    limit.limit_size(0)
    assert net.loss_grad(small, sx, st) == loss and np.array_equal(net.get_grads(), grads)
    net.close()
    eng.close()
    print("held")
    """)


@pytest.mark.parametrize("precision,mmax", [("fp64", 1), ("fp64", 3), ("fp32", 4)])
def test_no_evaluation_after_a_table_that_did_not_fit(precision, mmax):
    """set_ck that fails half way leaves no table: an evaluation then says so instead of using what is left of two."""
    run("""
    precision, mmax = sys.argv[1], int(sys.argv[2])
    n, N = (6, 5, 4), 120
    eng = Engine(n, [0.5 * v for v in n], mmax, 2, 2.4777, 0.0333, precision)
    one, two = (ck.synthetic_ck(mmax, 1024, dq, seed=1, n0=0.0333) for dq in (0.05, 0.04))
    eng.set_ck(one)
    rng = np.random.default_rng(0)
    eng.set_vext(rng.uniform(-2.0, 5.0, N * eng.no))
    xi = 1.0 + 0.2 * rng.uniform(-1, 1, N * eng.no)
    parts, df = eng.energy_and_gradient(xi)
    eng.set_ck(two)
    # of the second table, and of its fragments for the matrix cores (per block khi 2 columns by 4 rows)
    frags = sum((sum(2 * (m // 2) + 1 for m in range(abs(k), mmax + 1)) + 1) // 2 *
                ((sum(m // 2 + 1 for m in range(abs(k), mmax + 1)) + 3) // 4) for k in range(-mmax, mmax + 1))
    sizes = 16 * eng.npc * eng.nq, (8 if precision == "fp64" else 4) * 64 * frags * (eng.nq - 1)
    for size in sizes:
        eng.close()
        eng = Engine(n, [0.5 * v for v in n], mmax, 2, 2.4777, 0.0333, precision)
        eng.set_vext(np.zeros(N * eng.no))
        eng.set_ck(one)
        print("refusing", size, flush=True)
        before = limit.limit_failures()
        limit.limit_size(size)
        try:
            eng.set_ck(two)
            raise SystemExit("a table without room")
        except MdftError as e:
            assert e.code == ENOMEM and limit.limit_failures() > before, e
        limit.limit_size(0)
        try:
            eng.energy_and_gradient(xi)
            raise SystemExit("an evaluation without a table")
        except MdftError as e:
            print(e, flush=True)
            assert "c(k)" in str(e)
    eng.set_ck(one)
    eng.energy_and_gradient(xi)
    eng.close()
    print("held")
    """, precision, mmax)


@pytest.mark.parametrize("mmax", [3, 4, 5, 6])
def test_classes_of_pairs_without_memory(mmax):
    """Without memory for the classes of the q-space pairs all of them keep the entry by entry rotations, which are
    right for any: field, energies and gradient against the oracle at the bars of the two forms (1e-10)."""
    run("""
    mmax = int(sys.argv[1])
    n, length = (18, 20, 25), (4.1, 5.3, 3.7)   # (in a smaller box all pairs keep that form anyway)
    table = ck.synthetic_ck(mmax, 1024, 0.05, seed=5 + mmax, n0=0.0333)
    eng = Engine(n, length, mmax, 2, 2.4777, 0.0333, "fp64")
    ora = O.Oracle(n, length, mmax, 2, 2.4777, 0.0333)
    rng = np.random.default_rng(3)
    xi = 1.0 + 0.3 * rng.uniform(-1, 1, eng.N * eng.no)
    vext = rng.uniform(-2.0, 5.0, eng.N * eng.no)
    eng.set_vext(vext)
    # pairs: the half space of q, and of each plane that is its own image the half plane
    pairs = sum(1 for z in range(n[2] // 2 + 1) for y in range(n[1]) for x in range(n[0])
                if (n[2] - z) % n[2] != z or ((n[1] - y) % n[1], (n[0] - x) % n[0]) >= (y, x))
    limit.limit_size(8 * pairs)
    for e in (eng, ora):
        e.set_ck(table)
    assert limit.limit_failures() > 0
    limit.limit_size(0)
    ref = ora.excess_stage(xi, 3)
    assert np.abs(eng.excess_stage(xi, 3) - ref).max() <= 1e-10 * np.abs(ref).max()
    parts, df = eng.energy_and_gradient(xi)
    pref, dref = ora.energy_and_gradient(xi, vext)
    assert np.abs(parts - pref).max() <= 1e-10 * np.abs(pref).max()
    assert np.abs(df - dref).max() <= 1e-10 * np.abs(dref).max()
    eng.set_ck(table)   # and with memory again
    again, da = eng.energy_and_gradient(xi)
    assert np.abs(again - pref).max() <= 1e-10 * np.abs(pref).max()
    assert np.abs(da - dref).max() <= 1e-10 * np.abs(dref).max()
    eng.close()
    print("held")
    """, mmax)
