"""Hashed saves of few records on the GPU plane: digests equal to the oracle's, taken on the host."""
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest
import torch

from kvsnap_amd import dataplane, synth
from kvsnap_amd.native import kernel_library

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["staged", "direct"])
@pytest.mark.parametrize("layout", ["vllm", "kv_split"])
@pytest.mark.parametrize("n", [1, 2, 20, 65])
def test_digests_equal_the_oracle(hip_library, oracle_lib, mode, layout, n):
    caches, backing = synth.make_caches(4, 80, layout=layout)
    plane = dataplane.TorchBlockDataPlane(caches, 16, 64 << 20, save_mode=mode)
    try:
        plane.warm_up()
        keep = synth.fill(plane, n)
        torch.cuda.synchronize()
        hosted = plane._hash_threads(kernel_library(), n)
        staged, digests, size = plane.pool.reserve(n * plane.block_bytes), [], plane.block_bytes
        plane.save_gather(list(range(3, 3 + n)), [(staged, i * size) for i in range(n)], n * 16 - 5, digests=digests)
        assert hosted == 0 or isinstance(digests[0]._event, dataplane.HostHashJob)
        crcs, shas = oracle_lib.digest_records(staged.pointer, size, size, n, threads=4)
        assert digests[0].result() == [(bytes(h).hex(), int(c)) for h, c in zip(shas, crcs)]
        record = np.frombuffer(staged.read_range((n - 1) * size, size), dtype=np.uint8)
        expected = record.copy()
        oracle_lib.zero_tail(expected, plane.layers, 11)
        assert np.array_equal(record, expected)
        staged.close()
        del keep
    finally:
        plane.close()


def test_a_process_that_ends_with_its_hashes_in_flight_exits_cleanly(hip_library, tmp_path):
    """The hashing thread reads the pinned arena: it is done before the runtime goes away, plane closed or not."""
    script = tmp_path / "end_while_hashing.py"
    script.write_text("""
import torch
from kvsnap_amd import synth
from kvsnap_amd.dataplane import TorchBlockDataPlane
caches, backing = synth.make_caches(36, 80, layout="kv_split")
plane = TorchBlockDataPlane(caches, 16, 256 << 20)
plane.warm_up()
backing.zero_()
torch.cuda.synchronize()
staged = plane.pool.reserve(64 * plane.block_bytes)
digests = []
plane.save_gather(list(range(64)), [(staged, i * plane.block_bytes) for i in range(64)], 64 * 16, digests=digests)
print("saved", flush=True)
""")
    env = dict(os.environ, PYTHONPATH=str(Path(__file__).resolve().parents[1]), KVSNAP_HASH_THREADS="8")
    done = subprocess.run([sys.executable, str(script)], capture_output=True, text=True, timeout=120, env=env)
    assert done.returncode == 0 and "saved" in done.stdout, (done.returncode, done.stderr[-2000:])
