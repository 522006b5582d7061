"""CPU test of the kept device blocks (csrc/devmem.hip) over a mock of HIP's memory calls: which block an
allocation gets, the bound, who gets it back, and that no thread's allocation waits for another's free."""
import ctypes as C
import os
import subprocess
import threading

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "mdft-dev_general_amd", "csrc")
GIB = 1 << 30
OUT_OF_MEMORY = 2


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("devmem") / "libdevmem_mock.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-w", "-x", "c++",
                           os.path.join(CSRC, "devmem.hip"), os.path.join(ROOT, "tests", "mock_hip", "devmem_mock.cpp"),
                           "-o", so, "-lpthread"])
    return so


class Mem:
    def __init__(self, so):
        self.lib = C.CDLL(so)
        self.lib.t_malloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.lib.t_free.argtypes = [C.c_void_p, C.c_int]
        self.lib.mock_device.argtypes = [C.c_int, C.c_size_t]
        self.lib.mock_used.restype = C.c_size_t
        self.lib.mock_holds.argtypes = [C.c_void_p]

    def alloc(self, n):
        p = C.c_void_p()
        rc = self.lib.t_malloc(C.byref(p), n)
        return p.value if rc == 0 else -rc

    def free(self, p, synced=0):
        assert self.lib.t_free(p, synced) == 0


@pytest.fixture
def mem(built):
    m = Mem(built)
    m.lib.mock_gate(1)
    m.lib.mock_device(0, 64 * GIB)
    m.lib.t_context(0, 1)
    yield m
    m.lib.mock_gate(1)
    m.lib.mock_device(0, 64 * GIB)
    m.lib.t_context(0, -1)
    assert m.lib.mock_used() == 0


@pytest.mark.parametrize("synced", [0, 1])
def test_a_freed_block_goes_to_the_next_allocation_of_its_size(mem, synced):
    a = mem.alloc(1000)
    mem.free(a, synced)
    b = mem.alloc(1001)
    assert b != a
    c = mem.alloc(1000)
    d = mem.alloc(1000)
    assert c == a and d not in (a, b)
    for p in (b, c, d):
        mem.free(p)


def test_at_most_two_gib_are_kept_the_oldest_given_back_first(mem):
    blocks = [mem.alloc(GIB // 2 + k) for k in range(6)]
    for p in blocks:
        mem.free(p)
    assert [mem.lib.mock_holds(p) for p in blocks] == [0, 0, 0, 1, 1, 1]
    big = mem.alloc(2 * GIB + 1)
    mem.free(big)
    assert not mem.lib.mock_holds(big)
    assert mem.lib.mock_used() == sum(GIB // 2 + k for k in (3, 4, 5))


def test_an_allocation_that_fails_gets_the_kept_memory(mem):
    mem.lib.mock_device(0, GIB)
    a = mem.alloc(GIB // 2)
    mem.free(a)
    b = mem.alloc(GIB)
    assert b > 4095 and not mem.lib.mock_holds(a)
    assert mem.alloc(8) == -OUT_OF_MEMORY
    assert mem.lib.hipGetLastError() == 0  # not left for the next launch's check
    mem.free(b)
    c = mem.alloc(8)
    mem.free(c)


def test_nothing_is_kept_without_a_context_or_for_another_device(mem):
    mem.lib.mock_device(1, 64 * GIB)
    a = mem.alloc(100)
    mem.free(a)  # no context there
    assert not mem.lib.mock_holds(a)
    b = mem.alloc(100)
    mem.lib.t_context(1, 1)
    mem.lib.mock_device(0, 64 * GIB)
    mem.free(b)  # from a thread whose device is another
    assert not mem.lib.mock_holds(b)
    c = mem.alloc(100)
    mem.free(c)
    mem.lib.mock_device(1, 64 * GIB)
    d = mem.alloc(100)
    assert d != c
    mem.free(d)
    mem.lib.t_context(1, -1)
    assert not mem.lib.mock_holds(d) and mem.lib.mock_holds(c)


@pytest.mark.parametrize("what", ["free that is kept", "free beyond the bound", "failed allocation", "last context"])
def test_no_allocation_waits_while_another_thread_waits_for_the_device(mem, what):
    if what == "free that is kept":
        p = mem.alloc(64)
        wait = lambda: mem.free(p)
    elif what == "free beyond the bound":
        old = mem.alloc(2 * GIB)
        mem.free(old)
        p = mem.alloc(64)
        wait = lambda: mem.free(p, 1)  # gives the old block back
    elif what == "failed allocation":
        p = mem.alloc(64 * GIB - 8192)
        q = mem.alloc(7000)
        mem.free(q)
        wait = lambda: mem.free(mem.alloc(8000), 1)
    else:
        mem.lib.mock_device(1, 64 * GIB)
        mem.lib.t_context(1, 1)
        p = mem.alloc(64)
        mem.free(p)
        wait = lambda: mem.lib.t_context(1, -1)
    mem.lib.mock_gate(0)
    one = threading.Thread(target=wait)
    one.start()
    assert mem.lib.mock_await_waiter()
    got = []
    two = threading.Thread(target=lambda: got.append(mem.alloc(32)))
    two.start()
    two.join(5.0)
    done = not two.is_alive()
    mem.lib.mock_gate(1)
    one.join()
    two.join()
    assert done
    mem.free(got[0], 1)
    if what == "failed allocation":
        mem.free(p)
    if what == "last context":
        mem.lib.t_context(1, -1)
