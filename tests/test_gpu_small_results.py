"""Results on their way to the host: by a kernel into page-locked memory up to 16 KiB of whole words, by a copy otherwise."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from dynet_amd import Device, DevTensor, DyhipError
from dynet_amd.device import PinnedArray
from tests.util import f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1, 4, 12])  # bytes
@pytest.mark.parametrize("nbytes", [1, 4, 6, 252, 256, 260, 1024, 4092, 16380, 16384, 16388, 20001])  # 64 threads, 1024; copies
def test_every_byte_comes_back_and_none_beside_it(dev, nbytes, offset):
    x = np.random.default_rng(nbytes).integers(0, 256, 20480).astype(np.uint8)
    whole = dev.empty(x.size // 4, np.uint32)
    whole.set(x.view(np.uint32))
    src = DevTensor(dev, whole.ptr + offset, (nbytes,), np.uint8)
    assert np.array_equal(src.numpy(), x[offset:offset + nbytes])


def test_results_of_several_threads_and_queues(dev):
    """Each thread reads its own tensor over and over, two of them through a queue of their own."""
    xs = [f32(np.full(1 + 1000 * k, k + 0.5)) for k in range(4)]
    ts = [dev.tensor(x) for x in xs]
    dev.sync()
    forks = [dev.fork(), dev.fork()]
    wrong = []

    def read(k):
        t = ts[k] if k < 2 else DevTensor(forks[k - 2], ts[k].ptr, ts[k].shape, np.float32)
        for _ in range(200):
            if not np.array_equal(t.numpy(), xs[k]):
                wrong.append(k)

    threads = [threading.Thread(target=read, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for f in forks:
        f.close()
    assert not wrong


@pytest.mark.parametrize("n", [1, 256, 300, 4096])
def test_each_result_is_that_of_the_kernel_before(dev, n):
    x = dev.empty(n)
    for k in range(600):  # past the launches that are waited for through the runtime
        dev.constant(x, k + 0.25)
        assert np.all(x.numpy() == k + 0.25)


def test_a_source_outside_the_gpus_memory_is_copied(dev):
    staging = PinnedArray((8,))
    staging.array[:] = np.arange(8)
    assert np.array_equal(DevTensor(dev, staging.ptr, (8,), np.float32).numpy(), np.arange(8, dtype=np.float32))
    staging.close()


def test_a_wait_that_gave_up_behind_another_threads_wait_is_reported():
    """A thread waits for a queue with work in it while this one launches a product whose waits give up at once: the other
    thread's read of the counter comes before that product, the next wait has to look again."""
    d = Device(0, mem_mb=(1024, 64, 64, 64))
    try:
        M, N, K = 4352, 4096, 512  # cut tiles, finished inside the kernel
        l, r, y, busy = d.empty((K, M)), d.empty((N, K)), d.empty((N, M)), d.empty(1 << 27)
        for t in (l, r):
            d.constant(t, 1.0)
        for _ in range(3):
            d.gemm_nn(M, N, K, l, r, 0.0, y)  # the wait below looks at the counter
            for _ in range(300):  # of 512 MB each: 20 ms and more
                d.constant(busy, 1.0)
            errors = []

            def wait():
                try:
                    d.sync()
                except DyhipError as e:
                    errors.append(e)

            other = threading.Thread(target=wait)
            other.start()
            time.sleep(0.005)  # it waits now
            d.set_gemm_handoff(0, False)
            d.gemm_nn(M, N, K, l, r, 0.0, y)
            d.set_gemm_handoff()
            other.join()
            wait()
            assert len(errors) == 1 and "gave up" in str(errors[0])
            d.sync()  # reported once
        d.gemm_nn(M, N, K, l, r, 0.0, y)
        assert np.all(y.numpy() == K)
    finally:
        d.close()


def test_an_error_that_another_call_left_behind_is_not_the_copys(dev):
    """A program's own failed HIP call leaves its error with the runtime; reading results and waiting have nothing to do with it."""
    hip = C.CDLL("libamdhip64.so.7")  # the runtime that the library is linked with: already loaded
    x = dev.tensor(f32([1.0, 2.0]))
    M, N, K = 4352, 4096, 512  # its waits are counted: the next wait reads the counter
    l, r, y = dev.empty((K, M)), dev.empty((N, K)), dev.empty((N, M))
    dev.constant(l, 1.0)
    dev.constant(r, 1.0)
    dev.sync()
    assert hip.hipSetDevice(4096) != 0
    assert np.array_equal(x.numpy(), [1.0, 2.0])
    hip.hipGetLastError()
    dev.gemm_nn(M, N, K, l, r, 0.0, y)
    assert hip.hipSetDevice(4096) != 0
    dev.sync()
    hip.hipGetLastError()
    assert np.all(y.numpy() == K)
