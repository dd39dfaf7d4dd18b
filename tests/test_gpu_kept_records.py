"""The gather's two stores (records kept in the memory-side cache, or streamed past it) at the line between them,
and the scatter that reads them back."""
import pytest
import torch

from kvsnap_amd.dataplane import gather_blocks, scatter_blocks

pytestmark = pytest.mark.gpu

SPANS, SPAN = 64, 16 << 10          # 1 MiB records


@pytest.mark.parametrize("n", [1, 767, 768, 769])
def test_gather_then_scatter_around_768_mib_of_records(hip_library, n):
    generator = torch.Generator(device="cuda").manual_seed(n)
    cache = torch.randint(0, 256, (SPANS, n + 3, SPAN), dtype=torch.uint8, device="cuda", generator=generator)
    other = torch.zeros_like(cache)
    order = torch.randperm(n + 3, device="cuda", generator=generator)
    ids, into = order[:n].contiguous(), order.flip(0)[:n].contiguous()

    def tables(storage):
        columns = ([s * SPAN for s in range(SPANS)], [storage[s].data_ptr() for s in range(SPANS)], [SPAN] * SPANS,
                   [SPAN // 8] * SPANS)
        return [torch.tensor(column, dtype=torch.int64, device="cuda") for column in columns]

    records = torch.empty((n, SPANS * SPAN), dtype=torch.uint8, device="cuda")
    gather_blocks(ids, *tables(cache), records.data_ptr(), SPANS * SPAN, min_span_bytes=SPAN)
    scatter_blocks(records.data_ptr(), SPANS * SPAN, into, *tables(other), min_span_bytes=SPAN)
    for s in range(SPANS):
        picked = cache[s].index_select(0, ids)
        assert torch.equal(records[:, s * SPAN:(s + 1) * SPAN], picked)
        assert torch.equal(other[s].index_select(0, into), picked)
    assert not other[:, order.flip(0)[n:]].any()
