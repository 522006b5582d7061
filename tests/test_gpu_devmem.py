"""GPU test of the device allocations that the library keeps for reuse: contents, sizes, an
owner that outlives its block's first user, contexts in two threads, and that the last
context gives the memory back."""
import threading

import numpy as np
import pytest
import torch  # before the library: it brings the HIP runtime that both use

pytestmark = pytest.mark.gpu


def _engine():
    from mdft.gpu import Engine
    return Engine((8, 6, 4), (4.0, 3.0, 2.0), 1, 2, 2.4777, 0.0333, "fp64")


@pytest.mark.parametrize("nbytes", [8, 4096, (1 << 20) + 8, 1 << 28])
def test_freed_blocks_are_reused_whole(nbytes):
    from mdft.gpu import DeviceBuffer
    eng = _engine()
    x = np.random.default_rng(nbytes).standard_normal(nbytes // 8)
    a = DeviceBuffer(eng, nbytes)
    a.upload(x)
    a.free()
    b, c = DeviceBuffer(eng, nbytes), DeviceBuffer(eng, nbytes)
    assert b.ptr.value != c.ptr.value
    b.upload(x)
    c.upload(-x)
    assert np.array_equal(b.download(), x) and np.array_equal(c.download(), -x)
    for v in (b, c):
        v.free()
    eng.close()


def test_contexts_in_two_threads_share_the_kept_blocks():
    from mdft.gpu import DeviceBuffer
    bad = []

    def work(seed):
        eng = _engine()
        rng = np.random.default_rng(seed)
        for k in range(200):
            x = rng.standard_normal(1000 + 500 * (k % 3))
            v = DeviceBuffer(eng, x.nbytes)
            v.upload(x)
            if not np.array_equal(v.download(), x):
                bad.append((seed, k))
            v.free()
        eng.close()

    threads = [threading.Thread(target=work, args=(s,)) for s in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_the_last_context_gives_the_memory_back():
    from mdft.gpu import DeviceBuffer
    one = _engine()
    free0 = torch.cuda.mem_get_info()[0]
    two = _engine()
    for _ in range(2):
        v = [DeviceBuffer(two, 1 << 29) for _ in range(6)]   # 3 GiB, of which at most 2 stay
        for b in v:
            b.free()
    assert torch.cuda.mem_get_info()[0] >= free0 - (2 << 30) - (64 << 20)
    two.close()
    one.close()
    assert torch.cuda.mem_get_info()[0] >= free0 - (64 << 20)


def test_a_freed_block_is_the_next_of_its_size():
    from mdft.gpu import DeviceBuffer
    eng = _engine()
    a = DeviceBuffer(eng, 123456)
    at = a.ptr.value
    a.free()
    b, c = DeviceBuffer(eng, 123464), DeviceBuffer(eng, 123456)
    assert b.ptr.value != at and c.ptr.value == at
    for v in (b, c):
        v.free()
    free0 = torch.cuda.mem_get_info()[0]
    v = [DeviceBuffer(eng, 1 << 29) for _ in range(6)]
    for x in v:
        x.free()
    assert torch.cuda.mem_get_info()[0] <= free0 - (1 << 30)   # some of them are still held
    eng.close()
