"""kvsnap_copy_few against torch's copies of the same bytes: spans of one and several passes of a wave, 8-byte
aligned ones, every fill of the last block, 1 to 128 blocks, records in pinned and in device memory."""
import ctypes as C

import pytest
import torch

from kvsnap_amd import synth
from kvsnap_amd.dataplane import TorchBlockDataPlane, _check, kernel_library

pytestmark = pytest.mark.gpu


def tables(bases, pitch, sizes):
    offsets = [sum(sizes[:i]) for i in range(len(sizes))]
    columns = (offsets, bases, [pitch] * len(sizes), [size // 8 for size in sizes])
    return [torch.tensor(column, dtype=torch.int64, device="cuda") for column in columns]


@pytest.mark.parametrize("n", [1, 2, 127, 128])
@pytest.mark.parametrize("tokens, slot, spans, shift", [(16, 256, 5, 0), (4, 8, 3, 0), (16, 24, 2, 8),
                                                        (16, 2048, 3, 0), (3, 40, 7, 8), (16, 2056, 2, 0)])
def test_saves_and_restores_equal_torch(hip_library, n, tokens, slot, spans, shift):
    lib, stream = kernel_library(), torch.cuda.current_stream().cuda_stream
    span, blocks = tokens * slot, 140
    pitch = span + 8 * (shift != 0)
    generator = torch.Generator(device="cuda").manual_seed(n + slot)
    cache = torch.randint(0, 256, (spans, blocks * pitch + shift), dtype=torch.uint8, device="cuda",
                          generator=generator)
    views = [cache[s, shift:].view(blocks, pitch)[:, :span] for s in range(spans)]
    span_tables = tables([v.data_ptr() for v in views], pitch, [span] * spans)
    args = [t.data_ptr() for t in span_tables]
    ids = torch.randperm(blocks, generator=torch.Generator().manual_seed(n))[:n].tolist()
    size = span * spans
    for pinned in (True, False):
        record = torch.zeros((n, size + 8), dtype=torch.uint8, **({"pin_memory": True} if pinned
                                                                   else {"device": "cuda"}))
        addresses = (C.c_uint64 * n)(*[record.data_ptr() + i * (size + 8) for i in range(n)])
        block_ids = (C.c_int64 * n)(*ids)
        for filled in sorted({0, 1, tokens - 1}):
            record.fill_(0xA5)
            _check(lib, lib.kvsnap_copy_few(1, addresses, block_ids, n, *args, spans, span, filled,
                                            tokens if filled else 0, 12, stream))
            torch.cuda.synchronize()
            want = torch.stack([torch.cat([v[b] for v in views]) for b in ids]).cpu()
            if filled:
                want[-1].view(spans, span)[:, filled * slot:] = 0
            assert torch.equal(record[:, :size].cpu(), want)
            assert (record[:, size:] == 0xA5).all()
        record.copy_(torch.randint(0, 256, record.shape, dtype=torch.uint8))
        other = torch.randint(0, 256, cache.shape, dtype=torch.uint8, device="cuda", generator=generator)
        want = other.clone()
        into = [other[s, shift:].view(blocks, pitch)[:, :span] for s in range(spans)]
        device_record = record.cuda()
        for s in range(spans):
            want[s, shift:].view(blocks, pitch)[ids, :span] = device_record[:, s * span:(s + 1) * span]
        span_tables[1].copy_(torch.tensor([v.data_ptr() for v in into], dtype=torch.int64))
        _check(lib, lib.kvsnap_copy_few(0, addresses, block_ids, n, *args, spans, span, 0, 0, 12, stream))
        assert torch.equal(other, want)
        span_tables[1].copy_(torch.tensor([v.data_ptr() for v in views], dtype=torch.int64))


def test_bad_counts_are_refused(hip_library):
    lib = kernel_library()
    t = torch.zeros(4, dtype=torch.int64, device="cuda").data_ptr()
    one, ids = (C.c_uint64 * 129)(), (C.c_int64 * 129)()
    for n, spans, filled, tokens in ((129, 1, 0, 0), (-1, 1, 0, 0), (1, 1, 5, 4), (1, 1, 1, 0), (1, -1, 0, 0)):
        assert lib.kvsnap_copy_few(1, one, ids, n, t, t, t, t, spans, 8, filled, tokens, 12, 0) == -1


def test_records_behind_an_odd_sized_reservation_round_trip(hip_library):
    """Off the kernels' 8-byte boundaries a staged save and a copy-engine restore go the general way."""
    caches, backing = synth.make_caches(4, 20, layout="vllm")
    plane = TorchBlockDataPlane(caches, 16, 4 << 20, save_mode="staged", restore_mode="dma")
    try:
        odd = plane.pool.reserve(3)
        staged, size = plane.pool.reserve(2 * plane.block_bytes), plane.block_bytes
        assert staged.pointer % 8
        targets = [(staged, 0), (staged, size)]
        plane.save_gather([3, 9], targets, 32)
        plane.load_scatter([12, 1], targets)
        for tensor in caches.values():
            bits = tensor.view(torch.int16)
            assert torch.equal(bits[[12, 1]], bits[[3, 9]])
        staged.close()
        odd.close()
    finally:
        plane.close()
