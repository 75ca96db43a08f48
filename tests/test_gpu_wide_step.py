"""GPU: single-token steps that the prefill kernel serves (more than 32 query
heads per KV head), through ``append_paged_attention`` and ``paged_attention``.

Their spans are cut into pieces, whose partials live in a workspace: the
result's bits must not depend on which calls ran before.
"""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _case(heads, seed=0, lens=(3000, 1501), dim=64):
    from pkv import ops

    gen = torch.Generator(device="cuda").manual_seed(heads + seed)
    fmt = ops.PageFormat(1, dim, 16, 8, 64)
    lens = torch.tensor(lens, dtype=torch.int32, device="cuda")
    batch, per = lens.numel(), -(-int(lens.max()) // 16)
    table = torch.randperm(batch * per, generator=gen, device="cuda").to(torch.int32).view(batch, per)
    pool = ops.allocate_pool(fmt, batch * per)
    k, v = (torch.randn((batch, 1, int(lens.max()), dim), generator=gen, device="cuda").to(fmt.dtype)
            for _ in range(2))
    ops.append_quantize(fmt, pool, k, v, table, torch.zeros_like(lens), lens - 1)
    new = [torch.randn((batch, 1, 1, dim), generator=gen, device="cuda").to(fmt.dtype) for _ in range(2)]
    q = torch.randn((batch, heads, 1, dim), generator=gen, device="cuda").to(fmt.dtype)
    fused = lambda: ops.append_paged_attention(fmt, pool, *new, q, table, lens, scale=dim ** -0.5)
    attend = lambda: ops.paged_attention(fmt, pool, q, table, lens, scale=dim ** -0.5)
    fused()  # the new token is in its page for both
    return fused, attend


def _forget():
    from pkv import ops

    ops._PLANS.clear()
    ops._WORKSPACES.clear()


@pytest.mark.parametrize("heads", [40, 71])
def test_bits_do_not_depend_on_the_order_of_calls(heads):
    fused, attend = _case(heads)
    _forget()
    first = attend(), fused()
    _forget()
    again = fused(), attend()
    assert torch.equal(first[0], again[1]) and torch.equal(first[1], again[0])
