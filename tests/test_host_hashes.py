"""Records hashed on host threads: the native function against hashlib and the oracle, which saves take it, and what
waits for it (not the save)."""
import ctypes as C
import hashlib
import os
import threading
from unittest.mock import MagicMock, patch

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from kvsnap_amd import dataplane, native
from kvsnap_amd.blobs import BlobDirectory
from kvsnap_amd.host_tier import HostTier
from kvsnap_amd.pool import CopyFailed, CudaPool
from tests.test_copy_few_host import CUDA_CHECKS, FewKernels, caches
from tests.test_dataplane_host import CpuCuda, plane_over, slabs
from tests.test_pool import fake_pool_path      # noqa: F401 (a fixture)

LIBRARY = native.kernel_library()
needs_sha = pytest.mark.skipif(not LIBRARY.kvsnap_hash_records_available(), reason="no SHA instructions here")


@needs_sha
@pytest.mark.parametrize("threads", [1, 2, 8])
@pytest.mark.parametrize("n", [1, 2, 3, 17])
def test_digests_and_crcs_at_the_padding_s_edges(oracle_lib, threads, n):
    for size in (0, 1, 7, 55, 56, 63, 64, 65, 119, 120, 127, 128, 4099, 70000):
        data = np.random.default_rng(size).integers(0, 256, (n, size + 3), dtype=np.uint8)
        at = (C.c_uint64 * n)(*[data.ctypes.data + i * (size + 3) + 1 for i in range(n)])       # any alignment
        sha, crc = np.zeros((n + 1, 32), dtype=np.uint8), np.zeros(n + 1, dtype=np.uint32)
        assert LIBRARY.kvsnap_hash_records(at, size, n, sha.ctypes.data, crc.ctypes.data, threads) == 0
        for i in range(n):
            record = data[i, 1:1 + size]
            assert bytes(sha[i]) == hashlib.sha256(record.tobytes()).digest(), (size, i)
            assert crc[i] == oracle_lib.crc32c(record), (size, i)
        assert not sha[n].any() and not crc[n]


def test_bad_arguments_are_refused():
    out = np.zeros(64, dtype=np.uint8).ctypes.data
    at = (C.c_uint64 * 1)(out)
    for n, threads, size, records in ((-1, 1, 8, at), (1, 0, 8, at), (1, 257, 8, at), (1, 1, 8, None),
                                      (1, 1, (1 << 40) + 1, at)):
        assert LIBRARY.kvsnap_hash_records(records, size, n, out, out, threads) == -1
    assert LIBRARY.kvsnap_hash_records(None, 8, 0, None, None, 1) == 0


@needs_sha
def test_calls_at_the_same_time_share_their_helping_threads():
    """Four callers that ask for four threads each: themselves, and three helpers between them."""
    data = np.random.default_rng(1).integers(0, 256, (16, 1 << 21), dtype=np.uint8)
    at = (C.c_uint64 * 16)(*[row.ctypes.data for row in data])
    want = [hashlib.sha256(row.tobytes()).digest() for row in data]
    before, wrong = len(os.listdir("/proc/self/task")), []

    def caller():
        for _ in range(6):
            sha, crc = np.zeros((16, 32), dtype=np.uint8), np.zeros(16, dtype=np.uint32)
            assert LIBRARY.kvsnap_hash_records(at, 1 << 21, 16, sha.ctypes.data, crc.ctypes.data, 4) == 0
            wrong.extend(i for i in range(16) if bytes(sha[i]) != want[i])

    callers = [threading.Thread(target=caller) for _ in range(4)]
    for thread in callers:
        thread.start()
    most = 0
    while any(thread.is_alive() for thread in callers):
        most = max(most, len(os.listdir("/proc/self/task")) - before)
    # Sixteen without the sharing; threads on their way out are still listed for a moment.
    assert not wrong and 4 < most <= 4 + 3 + 3


class HashingKernels(FewKernels):
    def __init__(self):
        super().__init__()
        self.parts = []

    def kvsnap_hash_records_available(self):
        return 1

    def kvsnap_hash_records(self, records, size, n, sha, crc, threads):
        self.parts.append(n)
        return LIBRARY.kvsnap_hash_records(records, size, n, sha, crc, threads)


@pytest.fixture
def kernels(monkeypatch):
    found = HashingKernels()
    monkeypatch.setattr(dataplane.os, "sched_getaffinity", lambda pid: set(range(64)))
    monkeypatch.setattr(dataplane, "HASH_THREADS", 2)
    with patch.multiple(dataplane, kernel_library=lambda library=None: found, **CUDA_CHECKS):
        yield found


@needs_sha
@pytest.mark.parametrize("few_bytes", [0, 1 << 20], ids=["in-parts", "one-launch"])
@pytest.mark.parametrize("mode", ["staged", "direct"])
@pytest.mark.parametrize("shared", [True, False], ids=["one-allocation", "allocation-each"])
@pytest.mark.parametrize("chunk", [1, 3, 1 << 20])
@pytest.mark.parametrize("tokens", [1, 39, 44])
def test_the_digests_of_a_save_of_few_records(kernels, oracle_lib, monkeypatch, few_bytes, mode, shared, tokens, chunk):
    monkeypatch.setattr(dataplane, "FEW_BYTES", few_bytes)
    monkeypatch.setattr(CpuCuda.Event, "query", lambda self: False)     # parts that have landed are taken together
    plane = plane_over(caches("token", 14), 4, save_mode=mode)
    ids = [7, 2, 5, 0, 8, 13, 1, 9, 4, 11, 3][:-(-tokens // 4)]
    targets, plain, digests = slabs(plane, len(ids), shared=shared), slabs(plane, len(ids), shared=shared), []
    count = plane.save_gather(ids, targets, tokens, digests=digests, chunk_bytes=chunk * plane.block_bytes)
    plane.save_gather(ids, plain, tokens)
    # A hashed staged save copies each run of back-to-back targets whole, a direct one launches once a chunk.
    assert count == (-(-len(ids) // chunk) if mode == "direct" else 1 if shared else len(ids))
    records = [a.at(offset, plane.block_bytes) for a, offset in targets]
    assert records == [a.at(offset, plane.block_bytes) for a, offset in plain]
    assert len(digests) == 1
    assert digests[0].result() == [(hashlib.sha256(r).hexdigest(), oracle_lib.crc32c(np.frombuffer(r, np.uint8)))
                                   for r in records]
    if few_bytes and chunk >= len(ids):
        assert kernels.parts == [len(ids)]
    else:
        assert kernels.parts == [b - a for low in range(0, len(ids), chunk)
                                 for a, b in dataplane._parts(low, min(low + chunk, len(ids)), 4)]


def test_parts():
    """Each twice the one before, and a last one that takes a rest of less than half of it along."""
    sizes = lambda n, part: [b - a for a, b in dataplane._parts(0, n, part)]
    assert sizes(128, 16) == [16, 32, 80] and sizes(64, 16) == [16, 32, 16] and sizes(32, 16) == [16, 16]
    assert sizes(23, 16) == [23] and sizes(24, 16) == [16, 8] and sizes(1, 16) == [1] and sizes(0, 16) == []
    assert sizes(7, 1) == [1, 2, 4] and dataplane._parts(5, 12, 4) == [(5, 9), (9, 12)]


def expected(records):
    import oracle
    return [(hashlib.sha256(r).hexdigest(), oracle.crc32c(r)) for r in records]


class Held:
    """A plane on the library's own pool whose host hashes wait for ``open``."""

    def __init__(self, kernels, pool_path, mode):
        self.open, self.begun, self.fail = threading.Event(), threading.Event(), False
        real = kernels.kvsnap_hash_records

        def hashing(*arguments):
            self.begun.set()
            assert self.open.wait(5)
            return -1 if self.fail else real(*arguments)

        kernels.kvsnap_hash_records = hashing
        self.plane = plane_over(caches("token", 14), 4, save_mode=mode)
        self.size = self.plane.block_bytes
        self.plane.pool = CudaPool(12 * self.size, 0, library=pool_path)

    def hashing(self):
        """The plane's hashing thread is at work; a save in one launch is hashed by who needs it done."""
        return self.one_launch or self.begun.wait(5)

    def save(self, ids=(3, 1, 4, 11, 5, 9)):
        staged, digests = self.plane.pool.reserve(len(ids) * self.size), []
        targets = [(staged, i * self.size) for i in range(len(ids))]
        self.plane.save_gather(list(ids), targets, 4 * len(ids), digests=digests)
        return staged, targets, digests[0], [C.string_at(staged.pointer + at, self.size) for _, at in targets]


@pytest.fixture(params=[("staged", 0), ("staged", 1 << 20), ("direct", 0)], ids=["parts", "one-launch", "direct"])
def held(request, kernels, monkeypatch, fake_pool_path):       # noqa: F811
    monkeypatch.setattr(dataplane, "FEW_BYTES", request.param[1])
    found = Held(kernels, fake_pool_path, request.param[0])
    found.one_launch = request.param[1] > 0
    yield found
    found.open.set()
    found.plane.close()


def after(held, call):
    """``call`` in a thread of its own: it must wait until the hashes go on."""
    thread = threading.Thread(target=call)
    thread.start()
    thread.join(0.2)
    assert thread.is_alive()
    held.open.set()
    thread.join(20)
    assert not thread.is_alive()


@needs_sha
def test_a_save_returns_when_its_records_have_landed(held):
    staged, _, digests, records = held.save()
    assert held.hashing() and not digests.ready() and staged.ready()
    staged.wait()                                            # its copies; the pool is free meanwhile
    held.plane.pool.reserve(held.size).close()
    after(held, digests.result)
    assert digests.ready() and digests.result() == expected(records)


@needs_sha
def test_closing_a_target_waits_until_its_records_are_read(held):
    staged, _, digests, records = held.save()
    assert held.hashing()
    after(held, staged.close)
    assert staged.closed and digests.result() == expected(records)


@needs_sha
@pytest.mark.parametrize("write", ["save", "write", "zero", "copy"])
def test_writing_a_target_waits_until_its_records_are_read(held, write):
    staged, targets, digests, records = held.save()
    other = held.plane.pool.reserve(held.size)
    assert held.hashing()
    buffer = C.create_string_buffer(held.size)
    # Elsewhere nothing waits.
    held.plane.save_gather([2], [(other, 0)], 4)
    after(held, {"save": lambda: held.plane.save_gather([2], targets[3:4], 4),
                 "write": lambda: staged.write(bytes(6 * held.size)),
                 "zero": lambda: staged.zero(held.size + 3, 5),
                 "copy": lambda: staged.copy(C.addressof(buffer), held.size, held.size, to_host=True)}[write])
    staged.wait()
    assert digests.result() == expected(records)
    assert [C.string_at(staged.pointer + at, held.size) for _, at in targets] != records


@needs_sha
def test_a_hash_that_fails_is_raised_by_result(held):
    held.fail = True
    held.open.set()
    staged, _, digests, _ = held.save()
    for _ in range(2):
        with pytest.raises(RuntimeError):
            digests.result()
    staged.close()


@needs_sha
def test_a_plane_closed_meanwhile_finishes_its_hashes(held):
    staged, _, digests, records = held.save()
    assert held.hashing()
    after(held, held.plane.close)
    assert staged.closed and digests.result() == expected(records)


@needs_sha
def test_without_a_thread_result_does_the_work(held, monkeypatch):
    monkeypatch.setattr(dataplane, "HostHashes", MagicMock(side_effect=RuntimeError("can't start new thread")))
    held.open.set()
    staged, _, digests, records = held.save()
    assert digests.result() == expected(records)


@needs_sha
@pytest.mark.parametrize("tier", ["host", "blobs"])
@pytest.mark.parametrize("fail", [False, True])
def test_the_blocks_are_free_before_the_hashes(held, tmp_path, tier, fail):
    """``fenced`` is set when the records have landed; a hash that fails is not an unproven copy."""
    fenced, found = threading.Event(), []
    held.fail = fail

    def save():
        try:
            if tier == "host":
                found.append(HostTier(held.plane, 1 << 20).save([3, 1, 4], 12, fenced=fenced))
            else:
                found.append(BlobDirectory(tmp_path).save(held.plane, [3, 1, 4], 12, fenced=fenced))
        except Exception as exc:
            found.append(exc)

    saver = threading.Thread(target=save)
    saver.start()
    assert held.begun.wait(5) and fenced.wait(2) and saver.is_alive()
    held.open.set()
    saver.join(20)
    if fail:
        assert type(found[0]) is RuntimeError and not isinstance(found[0], CopyFailed)
    else:
        assert [len(segment["blob_id"]) for segment in found[0]["segments"]] == [64] * 3


def test_the_rule(kernels, monkeypatch):
    plane = plane_over(caches("token", 14), 4)
    threads = lambda n: plane._hash_threads(kernels, n)
    assert threads(1) == threads(32) == 2 and threads(33) == 0
    monkeypatch.setattr(dataplane.os, "sched_getaffinity", lambda pid: {3})
    assert threads(16) == 1 and threads(17) == 0
    monkeypatch.setattr(dataplane.os, "sched_getaffinity", lambda pid: set(range(512)))
    monkeypatch.setattr(dataplane, "HASH_THREADS", 400)
    assert threads(1) == 256
    monkeypatch.setattr(dataplane, "HASH_THREADS", 0)
    assert threads(1) == 0
    monkeypatch.setattr(dataplane, "HASH_THREADS", 2)
    plane.timer = object()
    assert threads(1) == 2                  # a timer times what runs
    plane.timer = None
    kernels.kvsnap_hash_records_available = lambda: 0
    assert threads(1) == 0
