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
