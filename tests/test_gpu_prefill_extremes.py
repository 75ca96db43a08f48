"""GPU: infinities and NaN in float pages under prefill spans cut into pieces:
tokens that score -inf weigh nothing wherever the pieces end (a piece may hold
no other token), and a NaN reaches the queries that see it and no other.
"""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("dead", [(128, 512), (0, 384), (1000, 1400)])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_cut_spans_with_tokens_that_are_not_finite(dtype, dead, value):
    from pkv import ops

    gen = torch.Generator(device="cuda").manual_seed(5)
    fmt = ops.PageFormat(2, 64, 16, 16, 32, getattr(torch, dtype))
    n, nq = 1500, 100
    per = -(-n // 16)
    table = torch.randperm(per, generator=gen, device="cuda").to(torch.int32).view(1, per)
    pool = ops.allocate_pool(fmt, per)
    k, v = (torch.randn((1, 2, n, 64), generator=gen, device="cuda") for _ in range(2))
    q = torch.randn((1, 8, nq, 64), generator=gen, device="cuda")
    k[..., 0] = 0.0
    q[..., 0] = -1.0
    nan = value != value
    # -inf scores for a stretch of tokens; a NaN in one of the chunk's own
    k[:, :, n - 50 if nan else dead[0]:n - 49 if nan else dead[1], 0] = value
    k, v, q = (x.to(fmt.dtype) for x in (k, v, q))
    lens = torch.tensor([n], dtype=torch.int32, device="cuda")
    ops.append_quantize(fmt, pool, k, v, table, torch.zeros_like(lens))
    small = torch.empty(256, dtype=torch.uint8, device="cuda")
    whole = ops.paged_attention(fmt, pool, q, table, lens, scale=0.125, workspace=small).float()
    cut = ops.paged_attention(fmt, pool, q, table, lens, scale=0.125).float()
    if nan:
        sees = torch.arange(nq, device="cuda") >= nq - 50
        assert torch.isnan(cut[:, :, sees]).all() and torch.isnan(whole[:, :, sees]).all()
        cut, whole = cut[:, :, ~sees], whole[:, :, ~sees]
    assert torch.isfinite(cut).all() and torch.isfinite(whole).all()
    step = 2.0 ** -7 if dtype == "bfloat16" else 2.0 ** -10
    bound = whole.abs() * step + whole.abs().amax(-1, keepdim=True) * 2.0 ** -8 + 1e-6
    assert bool(((cut - whole).abs() <= bound).all())
    at = torch.arange(nq, device="cuda") + n - nq
    s = torch.bmm(q[0].double().view(2, -1, 64), k[0].double().transpose(1, 2).contiguous()) * 0.125
    s.masked_fill_(torch.arange(n, device="cuda")[None] > at.repeat(4)[:, None], float("-inf"))
    want = torch.bmm(torch.softmax(s, -1), v[0].double()).view(8, nq, 64)
    if nan:
        want = want[:, ~sees]
    err = (cut[0].double() - want).abs()
    assert float(err.max()) <= 2e-2 and float(err.mean()) <= 2e-3
