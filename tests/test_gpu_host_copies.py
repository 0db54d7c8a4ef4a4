"""Blocking reads through the pinned staging buffers: bytes come back as they were
written, for sizes of one chunk, of several without threads, of
fewer and of more chunks than there are buffers, and ends that are not whole
chunks (19 N^3 values never are)."""
import numpy as np
import pytest

from lbmcl_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, precision, storage", [
    (4, "f32", "fp16"), (8, "f64", "native"), (16, "f32", "native"), (16, "f64", "native"), (32, "f32", "native"),
    (32, "f64", "native"), (64, "f32", "fp16"), (64, "f32", "native"), (64, "f64", "native"), (128, "f32", "native")])
def test_written_state_reads_back(n, precision, storage):
    with capi.Context(n, stride=n, precision=precision, storage=storage, profile=False) as g:
        g.initialize()
        rng = np.random.default_rng(n)
        words = [rng.integers(0, 256, 19 * n ** 3 * g.sdtype(0).itemsize, dtype=np.uint8) for _ in range(2)]
        for b in (0, 1):
            g.write_state(b, words[b].view(g.sdtype))
        for b in (0, 1):
            assert np.array_equal(g.read_state(b).view(np.uint8), words[b])
        for b in (1, 0):  # the buffers in another order, right after each other
            assert np.array_equal(g.read_state(b).view(np.uint8), words[b])


def test_reads_wait_for_the_work_before_them():
    """A read sees the iterations enqueued before it, and a force set after them
    does not reach back."""
    n = 128
    with capi.Context(n, stride=64, profile=False) as g:
        g.initialize()
        g.compute_range(1, 200)
        g.compute(201, update_macro=True)
        rho, u = g.read_rho(), g.read_u()
        g.finish()
        assert np.array_equal(rho, g.read_rho(), equal_nan=True) and np.array_equal(u, g.read_u(), equal_nan=True)
        g.set_force(np.full(3 * n ** 3, 1e-5, np.float32))
        g.compute_range(202, 20)
        g.set_force(None)
        g.compute(222, update_macro=True)
        assert not np.array_equal(rho, g.read_rho(), equal_nan=True)


def test_reads_of_two_threads_and_after_a_trim():
    """One read has the pinned buffers, another thread's does without them; a trim
    in between changes nothing."""
    import threading
    want, got = {}, {}

    def run(i, out, trim):
        with capi.Context(64, stride=64, velocity=0.04 + 0.01 * i, profile=False) as g:
            g.initialize()
            g.compute_range(1, 20)
            out[i] = [g.read_state(k % 2) for k in range(4)]
            if trim:
                capi.trim()
            out[i] += [g.read_state(k % 2) for k in range(4)]

    for i in range(3):
        run(i, want, False)
    threads = [threading.Thread(target=run, args=(i, got, True)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(3):
        assert len(got[i]) == 8
        for a, b in zip(want[i], got[i]):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
