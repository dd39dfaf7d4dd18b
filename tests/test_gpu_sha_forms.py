"""The SHA-256 kernel's quad form (eight lanes a record, 24 records a workgroup) and the rule that picks it.

Quad workgroups up to 64 (1536 records), the two-lane form (64 records a workgroup) above: record counts at the
edges of a round wave (8), a workgroup and the rule; messages of 1 to 14 blocks, so that launches end on every
block of a step and before the second step; chains cut into ranges whose launches change form between them."""
import ctypes as C
import hashlib

import numpy as np
import pytest
import torch

from kvsnap_amd.dataplane import _check, kernel_library

pytestmark = pytest.mark.gpu


def records(n, size, pitch, shift, seed):
    host = np.random.default_rng(seed).integers(0, 256, n * pitch + shift, dtype=np.uint8)
    want = [hashlib.sha256(host[shift + r * pitch: shift + r * pitch + size].tobytes()).digest() for r in range(n)]
    return torch.from_numpy(host).cuda(), want


def digests(out, n):
    return [bytes(row) for row in out[:n].cpu().numpy()]


@pytest.mark.parametrize("n", [1, 7, 8, 9, 23, 24, 25, 49, 1536, 1537])
@pytest.mark.parametrize("size, shift", [(0, 0), (55, 0), (56, 0), (64, 16), (200, 0), (448, 3), (512, 0), (840, 0)])
def test_record_counts_and_block_counts_at_the_edges(hip_library, n, size, shift):
    lib, stream = kernel_library(), torch.cuda.current_stream().cuda_stream
    pitch = -(-max(size, 16) // 16) * 16
    data, want = records(n, size, pitch, shift, n * 1000 + size)
    out = torch.zeros((n, 32), dtype=torch.uint8, device="cuda")
    _check(lib, lib.kvsnap_sha256_records(data.data_ptr() + shift, size, pitch, n, out.data_ptr(), stream))
    assert digests(out, n) == want


@pytest.mark.parametrize("cut", [1, 2, 3, 4, 5, 8, 9])
def test_chains_whose_launches_change_form_keep_their_digests(hip_library, cut):
    """25 records of 14 blocks in ranges of ``cut``: alone (quad) and beside 1537 records (two-lane) by turns."""
    lib, stream = kernel_library(), torch.cuda.current_stream().cuda_stream
    sets = [(25, 840, *records(25, 840, 848, 0, cut)), (1537, 840, *records(1537, 840, 848, 0, 50 + cut))]
    nblocks = int(lib.kvsnap_sha256_blocks(840))
    states = [torch.zeros((n, 8), dtype=torch.int32, device="cuda") for n, *_ in sets]
    outs = [torch.zeros((n, 32), dtype=torch.uint8, device="cuda") for n, *_ in sets]
    at, launch = [0, 0], 0
    while min(at) < nblocks:
        take = [i for i in (0, 1) if at[i] < nblocks and (i == 0 or launch % 2)]
        take = take or [1]
        table = [(C.c_uint64 * len(take))() for _ in range(7)]
        counts = (C.c_int64 * len(take))()
        for k, i in enumerate(take):
            end = min(at[i] + cut, nblocks)
            n, size, data, _ = sets[i]
            for column, value in zip(table, (data.data_ptr(), size, 848, at[i], end, states[i].data_ptr(),
                                             outs[i].data_ptr())):
                column[k] = value
            counts[k] = n
            at[i] = end
        _check(lib, lib.kvsnap_sha256_ranges(len(take), *table[:3], counts, *table[3:], stream))
        launch += 1
    for (n, _, _, want), out in zip(sets, outs):
        assert digests(out, n) == want
