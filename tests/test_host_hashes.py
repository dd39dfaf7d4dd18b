"""Records hashed on host threads: the native function against hashlib and the oracle, and which saves take it."""
import ctypes as C
import hashlib
import os
import threading
from unittest.mock import patch

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from kvsnap_amd import dataplane, native
from tests.test_copy_few_host import CUDA_CHECKS, FewKernels, caches
from tests.test_dataplane_host import plane_over, slabs

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
def test_a_save_of_few_records_has_their_digests_when_it_returns(kernels, oracle_lib, monkeypatch, few_bytes, mode,
                                                                 shared, tokens, chunk):
    monkeypatch.setattr(dataplane, "FEW_BYTES", few_bytes)
    plane = plane_over(caches("token", 14), 4, save_mode=mode)
    ids = [7, 2, 5, 0, 8, 13, 1, 9, 4, 11, 3][:-(-tokens // 4)]
    targets, plain, digests = slabs(plane, len(ids), shared=shared), slabs(plane, len(ids), shared=shared), []
    count = plane.save_gather(ids, targets, tokens, digests=digests, chunk_bytes=chunk * plane.block_bytes)
    plane.save_gather(ids, plain, tokens)
    # A hashed staged save copies each run of back-to-back targets whole, a direct one launches once a chunk.
    assert count == (-(-len(ids) // chunk) if mode == "direct" else 1 if shared else len(ids))
    records = [a.at(offset, plane.block_bytes) for a, offset in targets]
    assert records == [a.at(offset, plane.block_bytes) for a, offset in plain]
    assert len(digests) == 1 and digests[0].ready()
    assert digests[0].result() == [(hashlib.sha256(r).hexdigest(), oracle_lib.crc32c(np.frombuffer(r, np.uint8)))
                                   for r in records]
    assert sum(kernels.parts) == len(ids) and max(kernels.parts) <= (4 if not few_bytes else len(ids))


@needs_sha
def test_a_target_closed_meanwhile_fails_the_save_and_gives_no_digests(kernels, monkeypatch):
    monkeypatch.setattr(dataplane, "FEW_BYTES", 0)
    plane = plane_over(caches("token", 14), 4)
    targets, digests = slabs(plane, 9, shared=False), []
    real = kernels.kvsnap_hash_records

    def closing(*arguments):
        targets[5][0].closed = True
        return real(*arguments)

    kernels.kvsnap_hash_records = closing
    with pytest.raises(RuntimeError):
        plane.save_gather(list(range(9)), targets, 36, digests=digests)
    assert not digests and kernels.parts == [4]


def test_the_rule(kernels, monkeypatch):
    plane = plane_over(caches("token", 14), 4)
    threads = lambda n: plane._hash_threads(kernels, n)
    assert threads(1) == threads(32) == 2 and threads(33) == 0
    monkeypatch.setattr(dataplane.os, "sched_getaffinity", lambda pid: {3})
    assert threads(16) == 1 and threads(17) == 0
    monkeypatch.setattr(dataplane, "HASH_THREADS", 0)
    assert threads(1) == 0
    monkeypatch.setattr(dataplane, "HASH_THREADS", 2)
    plane.timer = object()
    assert threads(1) == 0
    plane.timer = None
    kernels.kvsnap_hash_records_available = lambda: 0
    assert threads(1) == 0
