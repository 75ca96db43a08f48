"""GPU: the order in which a prefill grid takes its row blocks (whole spans) does
not reach the output: every sequence of a batch gives the bits it gives alone,
over numbers of (sequence, KV head) segments that take the orders apart (one,
two, four, other numbers, a multiple of eight), with ragged widths.
"""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,gqa,queries", [(256, 3, 130), (64, 4, 200)])
@pytest.mark.parametrize("batch,hk", [(1, 1), (1, 2), (2, 1), (2, 2), (4, 1), (3, 1), (5, 2), (4, 2)])
def test_row_blocks_in_any_order_give_the_same_bits(batch, hk, dim, gqa, queries):
    from pkv import ops

    gen = torch.Generator(device="cuda").manual_seed(7 * batch + hk)
    fmt = ops.PageFormat(hk, dim, 16, 8, 64)
    widths = torch.tensor([max(1, queries - 37 * b) for b in range(batch)], dtype=torch.int32, device="cuda")
    lens = widths + torch.tensor([90 * b for b in range(batch)], dtype=torch.int32, device="cuda")
    top = int(lens.max())
    per = -(-top // 16)
    table = torch.randperm(batch * per, generator=gen, device="cuda").to(torch.int32).view(batch, per)
    pool = ops.allocate_pool(fmt, batch * per)
    k, v = (torch.randn((batch, hk, top, dim), generator=gen, device="cuda").to(fmt.dtype) for _ in range(2))
    ops.append_quantize(fmt, pool, k, v, table, torch.zeros_like(lens), lens)
    q = torch.randn((batch, hk * gqa, queries, dim), generator=gen, device="cuda").to(fmt.dtype)
    small = torch.empty(256, dtype=torch.uint8, device="cuda")  # room for no partials: whole spans

    def call(rows):
        return ops.paged_attention(fmt, pool, q[rows], table[rows], lens[rows], scale=dim ** -0.5,
                                   widths=widths[rows], workspace=small)

    together = call(slice(None))
    for b in range(batch):
        assert torch.equal(together[b], call(slice(b, b + 1))[0])
        assert not together[b, :, int(widths[b]):].any() and together[b, :, 0].any()
