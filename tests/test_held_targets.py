"""Pinned targets that a kernel writes by itself are released only once its writes are over.

The pool is the library's own on the stand-in runtime, the kernels HostKernels', and the events a gate: while it is
shut, the GPU has not come to the save's event yet."""
import threading
from unittest.mock import patch

import pytest

torch = pytest.importorskip("torch")

from kvsnap_amd import dataplane
from kvsnap_amd.pool import CudaPool, PinnedCapacityError
from tests.test_copy_few_host import CUDA_CHECKS, FewKernels, caches
from tests.test_dataplane_host import plane_over
from tests.test_pool import fake_pool_path      # noqa: F401 (a fixture)

WAIT = 20


class Gate:
    """Events that complete once the gate is open (or fail)."""

    def __init__(self):
        self.reached, self.open, self.failing = threading.Event(), threading.Event(), False
        gate = self

        class Event:
            def record(self, stream=None):
                pass

            def synchronize(self):
                gate.reached.set()
                assert gate.open.wait(WAIT)
                if gate.failing:
                    raise RuntimeError("event synchronize: unknown error")

            def query(self):
                return gate.open.is_set()

        self.Event = Event


@pytest.fixture(params=["staged", "direct", "direct-general"])
def saving(request, fake_pool_path, monkeypatch):       # noqa: F811
    """(plane, its gate, a target of two records, a thread that saves into it)."""
    kernels = FewKernels()
    if request.param == "direct-general":
        monkeypatch.setattr(dataplane, "FEW_BLOCKS", 0)
    with patch.multiple(dataplane, kernel_library=lambda library=None: kernels, **CUDA_CHECKS):
        plane = plane_over(caches("token", 9), 4, save_mode=request.param.split("-")[0])
        gate = Gate()
        plane.torch.cuda.Event = gate.Event
        plane.pool = CudaPool(2 * plane.block_bytes, 0, library=fake_pool_path)
        target = plane.pool.reserve(2 * plane.block_bytes)
        failed = []

        def save():
            try:
                plane.save_gather([3, 5], [(target, 0), (target, plane.block_bytes)], 7)
            except BaseException as exc:
                failed.append(exc)

        saver = threading.Thread(target=save)
        saver.start()
        assert gate.reached.wait(WAIT)      # queued, and waited for with the pool free again
        yield plane, gate, target, saver, failed
        gate.failing = False
        gate.open.set()
        saver.join(WAIT)
        plane.pool.close()


def test_a_close_meanwhile_waits_for_the_kernel(saving):
    plane, gate, target, saver, _ = saving
    assert not target.ready()
    closer = threading.Thread(target=target.close)
    closer.start()
    closer.join(0.2)
    assert closer.is_alive() and not target.closed
    gate.open.set()
    closer.join(WAIT)
    saver.join(WAIT)
    assert target.closed
    plane.pool.reserve(2 * plane.block_bytes).close()


def test_a_pool_close_meanwhile_waits_for_the_kernel(saving):
    plane, gate, target, saver, _ = saving
    closer = threading.Thread(target=plane.pool.close)
    closer.start()
    closer.join(0.2)
    assert closer.is_alive() and plane.pool.handle is not None
    gate.open.set()
    closer.join(WAIT)
    saver.join(WAIT)
    assert target.closed


def test_writes_that_cannot_be_proven_over_keep_the_target_reserved(saving):
    plane, gate, target, saver, failed = saving
    gate.failing = True
    gate.open.set()
    saver.join(WAIT)
    assert len(failed) == 1
    with pytest.raises(RuntimeError):
        target.close()
    assert not target.closed
    with pytest.raises(PinnedCapacityError):
        plane.pool.reserve(1)
    gate.failing = False
    target.close()
    plane.pool.reserve(2 * plane.block_bytes).close()
