"""Which calls go through kvsnap_copy_few, and that each leaves what the general path leaves (CPU kernels)."""
import ctypes as C
from contextlib import nullcontext
from unittest.mock import patch

import pytest

torch = pytest.importorskip("torch")

from kvsnap_amd import dataplane
from tests.test_dataplane_host import HostKernels, cache_bits, host_tables, plane_over, slabs

CUDA_CHECKS = dict(_int64_device_tensors=host_tables, _int32_device_output=lambda t, device, count: None,
                   _current_stream_handle=lambda device: 0)


class GeneralKernels(HostKernels):
    """HostKernels with the unhashed direct save's gather."""

    def kvsnap_gather_to_records(self, dests, blocks, n, offsets, bases, pitches, words, n_spans, hint, programs,
                                 stream):
        self.launches.append(("gather_to", n))
        for dest, block in zip(self._int64(dests, n), self._int64(blocks, n)):
            for offset, base, pitch, count in self._spans(offsets, bases, pitches, words, n_spans):
                C.memmove(dest + offset, base + block * pitch, 8 * count)
        return 0


class FewKernels(GeneralKernels):
    """HostKernels with kvsnap_copy_few, its lists read from host memory as the library reads them."""

    def kvsnap_copy_few(self, save, records, blocks, n, offsets, bases, pitches, words, n_spans, hint, filled,
                        tokens, programs, stream):
        self.launches.append(("few_save" if save else "few_restore", n))
        assert n <= 128 and (filled < tokens if tokens else not filled)
        for i in range(n):
            for offset, base, pitch, count in self._spans(offsets, bases, pitches, words, n_spans):
                record, cache, length = records[i] + offset, base + blocks[i] * pitch, 8 * count
                if not save:
                    C.memmove(cache, record, length)
                    continue
                keep = length // tokens * filled if tokens and i == n - 1 else length
                assert keep % 8 == 0
                C.memmove(record, cache, keep)
                C.memset(record + keep, 0, length - keep)
        return 0


@pytest.fixture(params=[True, False], ids=["few", "general"])
def kernels(request):
    found = FewKernels() if request.param else GeneralKernels()
    with patch.multiple(dataplane, kernel_library=lambda library=None: found, **CUDA_CHECKS):
        yield found


def caches(layout, blocks, heads=2, width=8, tokens=4, layers=3, seed=0):
    generator = torch.Generator().manual_seed(seed)
    shape = {"token": (layers, blocks, tokens, heads, width), "head": (layers, blocks, heads, tokens, width),
             "split": (layers, 2, blocks, tokens, heads, width)}[layout]
    storage = torch.randint(-2**15, 2**15, shape, dtype=torch.int16, generator=generator).view(torch.bfloat16)
    return {f"layer.{i}": storage[i].permute(0, 2, 1, 3) if layout == "token" else storage[i]
            for i in range(layers)}


def records_of(plane, ids, tokens, **options):
    targets = slabs(plane, len(ids), shared=True)
    targets[0][0].fill(0, b"\xa5" * (len(ids) * plane.block_bytes))
    count = plane.save_gather(ids, targets, tokens, **options)
    return count, targets[0][0].at(0, len(ids) * plane.block_bytes), targets


@pytest.mark.parametrize("mode", ["staged", "direct"])
@pytest.mark.parametrize("layout, heads, width", [("token", 2, 8), ("split", 1, 4), ("split", 3, 10), ("head", 2, 8),
                                                  ("token", 1, 2)])
@pytest.mark.parametrize("tokens", [1, 3, 4, 18, 20])
def test_saves_equal_the_general_path(kernels, mode, layout, heads, width, tokens):
    held = caches(layout, 9, heads, width)
    plane = plane_over(held, 4, save_mode=mode)
    ids = [7, 2, 5, 0, 8][:-(-tokens // 4)]
    count, got, _ = records_of(plane, ids, tokens)
    few = isinstance(kernels, FewKernels)
    # A head-major block's tail, or a token slot of fewer than 8 bytes, is not the front of each span.
    takes = few and (tokens % 4 == 0 or (layout != "head" and heads * width * 2 % 8 == 0))
    assert (("few_save", len(ids)) in kernels.launches) == takes
    assert count == 1
    with patch.multiple(dataplane, kernel_library=lambda library=None: GeneralKernels(), **CUDA_CHECKS):
        assert got == records_of(plane_over(held, 4, save_mode=mode), ids, tokens)[1]


@pytest.mark.parametrize("mode", ["kernel", "dma"])
def test_restores_equal_the_general_path(kernels, mode):
    source, target = caches("token", 9, seed=1), caches("token", 9, seed=2)
    plane = plane_over(source, 4)
    _, _, targets = records_of(plane, [3, 1, 6], 12)
    progress = []
    into = plane_over(target, 4, restore_mode=mode, device_staging_bytes=0)
    into._place_stream = lambda: None
    kernels.launches.clear()
    before = cache_bits(target)
    assert into.load_scatter([8, 0, 4], targets, progress=progress) == 1
    assert [left for _, left in progress] == [3 * plane.block_bytes, 0]
    assert (kernels.launches == [("few_restore", 3)]) == isinstance(kernels, FewKernels)
    for name, bits in cache_bits(target).items():
        want = before[name].clone()
        want[[8, 0, 4]] = cache_bits(source)[name][[3, 1, 6]]
        assert torch.equal(bits, want)


def test_the_rule(monkeypatch):
    """At most 128 blocks, one chunk; FEW_BYTES for staged saves and dma restores."""
    found = FewKernels()
    with patch.multiple(dataplane, kernel_library=lambda library=None: found, **CUDA_CHECKS):
        held = caches("token", 140)
        size = plane_over(held, 4).block_bytes

        def few(save, n, mode, **options):
            plane = plane_over(held, 4, **({"save_mode": mode} if save else {"restore_mode": mode,
                                                                               "device_staging_bytes": 0}))
            plane._place_stream = lambda: None
            targets = slabs(plane, n, shared=True)
            found.launches.clear()
            if save:
                plane.save_gather(list(range(n)), targets, 4 * n, **options)
            else:
                plane.load_scatter(list(range(n)), targets, **options)
            return any(name.startswith("few") for name, _ in found.launches)

        for save, capped, free in ((True, "staged", "direct"), (False, "dma", "kernel")):
            monkeypatch.setattr(dataplane, "FEW_BYTES", 3 * size)
            assert few(save, 3, capped) and not few(save, 4, capped)
            assert few(save, 4, free) and few(save, 128, free) and not few(save, 129, free)
            assert few(save, 3, capped, chunk_bytes=3 * size) and not few(save, 3, capped, chunk_bytes=size)


def test_closed_sources_and_outside_targets_are_refused_before_the_launch(kernels):
    plane = plane_over(caches("token", 9), 4)
    targets = slabs(plane, 2, shared=True)
    with pytest.raises(ValueError):
        plane.save_gather([1, 2], [targets[0], (targets[0][0], 1 + plane.block_bytes)], 8)
    with pytest.raises(ValueError):
        plane.load_scatter([1, 2], [targets[0], (targets[0][0], -1)])
    targets[0][0].closed = True
    for call in (lambda: plane.save_gather([1, 2], targets, 8), lambda: plane.load_scatter([1, 2], targets)):
        with pytest.raises(RuntimeError):
            call()
    assert not any(name.startswith(("few", "gather", "restore")) for name, _ in kernels.launches)


@pytest.mark.parametrize("save, mode", [(True, "staged"), (True, "direct"), (False, "dma"), (False, "kernel")])
@pytest.mark.parametrize("shift", [0, 8, 1, 4])
def test_records_off_the_word_boundaries_go_the_general_way(save, mode, shift):
    """A reservation behind one of an odd size starts off an 8-byte boundary."""
    found = FewKernels()
    with patch.multiple(dataplane, kernel_library=lambda library=None: found, **CUDA_CHECKS):
        held = caches("token", 9)
        plane = plane_over(held, 4, **({"save_mode": mode} if save else {"restore_mode": mode,
                                                                           "device_staging_bytes": 0}))
        plane._place_stream = lambda: None
        size = plane.block_bytes
        slab = plane.pool.reserve(2 * size + shift)
        assert slab.pointer % 16 == 0
        targets = [(slab, shift), (slab, shift + size)]
        if save:
            plane.save_gather([2, 7], targets, 7)
            assert slab.at(shift, size) == records_of(plane, [2], 4)[1]
        else:
            slab.fill(shift, records_of(plane, [2, 7], 8)[1])
            found.launches.clear()
            plane.load_scatter([4, 1], targets)
            assert all(torch.equal(bits[[4, 1]], bits[[2, 7]]) for bits in cache_bits(held).values())
    assert any(name.startswith("few") for name, _ in found.launches[:1]) == (shift % 8 == 0)


@pytest.mark.parametrize("save", [True, False])
def test_the_launch_is_made_with_the_plane_s_device_current(save, monkeypatch):
    """The calling thread may have another device current."""
    found, current, seen = FewKernels(), [], []
    real = found.kvsnap_copy_few

    class Current:
        def __init__(self, device):
            self.device = device

        def __enter__(self):
            current.append(self.device)

        def __exit__(self, *exc):
            current.pop()

    def launch(*arguments):
        seen.append(list(current))
        return real(*arguments)

    monkeypatch.setattr(found, "kvsnap_copy_few", launch)
    with patch.multiple(dataplane, kernel_library=lambda library=None: found, **CUDA_CHECKS):
        plane = plane_over(caches("token", 9), 4)
        plane.torch.cuda.device = Current
        targets = slabs(plane, 2, shared=True)
        if save:
            plane.save_gather([2, 7], targets, 8)
        else:
            plane.load_scatter([2, 7], targets)
    assert seen == [[0]]


@pytest.mark.parametrize("save, name", [(True, "gather_to"), (False, "restore")])
def test_a_timer_times_the_launch_and_does_not_change_it(save, name):
    class Timer:
        spans = []

        def wants(self, wanted):
            return True

        def span(self, wanted, stream):
            self.spans.append(wanted)
            return nullcontext()

    found = FewKernels()
    with patch.multiple(dataplane, kernel_library=lambda library=None: found, **CUDA_CHECKS):
        plane = plane_over(caches("token", 9), 4)
        plane.timer = Timer()
        targets = slabs(plane, 2, shared=True)
        if save:
            plane.save_gather([2, 7], targets, 8)
        else:
            plane.load_scatter([2, 7], targets)
    assert found.launches == [("few_save" if save else "few_restore", 2)] and Timer.spans == [name]
