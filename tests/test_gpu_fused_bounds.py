"""GPU: the fused single-token step where a sequence's length runs past its
block table (``pkv_append_paged_attention`` against the two separate calls).

The new token of such a sequence has no page: ``append_quantize`` drops it, and
the step must leave every page as it does -- the middle sequence of the batch
must not write through the next one's table row, the last one must not read
past the table.  Outputs (over the tokens that have pages) within two steps of
the element plus 2^-8 of the row's largest element: each form rounds its
probabilities to 16 bits against its own running maximum.
"""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

CASES = [
    # (heads, kv_heads, dim, bits, group, page, dtype): the append's forms
    (8, 2, 64, 16, 32, 16, "bfloat16"),     # float pages, four column slots
    (16, 2, 128, 16, 32, 32, "float16"),    # float pages, two slots (grouped)
    (32, 8, 128, 8, 64, 16, "bfloat16"),    # quantized pages, four slots
    (16, 2, 128, 4, 64, 16, "bfloat16"),    # quantized pages, two slots (grouped)
    (6, 2, 256, 8, 128, 64, "bfloat16"),    # head_dim 256
]


@pytest.mark.parametrize("waves", [0, 3, 37])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x) for x in c))
def test_token_past_the_block_table_is_dropped(case, waves):
    from pkv import ops

    heads, hk, dim, bits, group, page, dtype = case
    gen = torch.Generator(device="cuda").manual_seed(dim + bits)
    fmt = ops.PageFormat(hk, dim, page, bits, group, getattr(torch, dtype))
    per = 4
    cap = per * page
    lens = torch.tensor([20, cap + 1, 33, cap + 1], dtype=torch.int32, device="cuda")
    batch = lens.numel()
    table = torch.randperm(batch * per, generator=gen, device="cuda").to(torch.int32).view(batch, per)
    pool = ops.allocate_pool(fmt, batch * per)
    k, v = (torch.randn((batch, hk, cap, dim), generator=gen, device="cuda").to(fmt.dtype) for _ in range(2))
    ops.append_quantize(fmt, pool, k, v, table, torch.zeros_like(lens), lens - 1)
    new = [torch.randn((batch, hk, 1, dim), generator=gen, device="cuda").to(fmt.dtype) for _ in range(2)]
    q = torch.randn((batch, heads, 1, dim), generator=gen, device="cuda").to(fmt.dtype)

    apart, fused = pool.clone(), pool.clone()
    ops.append_quantize(fmt, apart, *new, table, lens - 1)
    want = ops.paged_attention(fmt, apart, q, table, lens, scale=dim ** -0.5, waves=waves).float()
    got = ops.append_paged_attention(fmt, fused, *new, q, table, lens, scale=dim ** -0.5, waves=waves).float()
    assert torch.equal(fused, apart)
    full = table[1].long()  # nothing of the sequences without a page for the token has changed
    assert torch.equal(fused[full], pool[full]) and not torch.equal(fused, pool)
    step = 2.0 ** -7 if dtype == "bfloat16" else 2.0 ** -10
    bound = want.abs() * step + want.abs().amax(-1, keepdim=True) * 2.0 ** -8 + 1e-6
    assert torch.isfinite(got).all() and bool(((got - want).abs() <= bound).all())
