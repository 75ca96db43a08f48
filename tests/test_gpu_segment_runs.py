"""GPU: decode calls with the library's own choice of runs -- one run per
(sequence, KV head) segment for short block tables, grouped runs for few
segments -- against the same call with explicit waves (equal shares of the
tiles, merged), and the fused append on float pages.

Outputs within two bf16 (f16) steps of the element plus 2^-8 of the row's
largest element: each form rounds its probabilities to 16 bits against its own
running maximum.  Pages are the same bytes.
"""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

CASES = [
    # (heads, kv_heads, dim, bits, group, page, dtype, queries, lengths)
    (8, 2, 64, 16, 32, 16, "bfloat16", 1, (128, 256, 384, 512)),
    (32, 8, 128, 8, 64, 16, "bfloat16", 1, (1, 700, 16, 1009)),
    (8, 1, 128, 4, 64, 32, "bfloat16", 1, (33, 5, 64)),          # two column slots
    (16, 2, 256, 8, 128, 64, "float16", 1, (300, 511)),          # one slot
    (4, 4, 100, 4, 32, 16, "bfloat16", 1, (17, 900, 250, 3)),
    (12, 1, 64, 8, 32, 16, "bfloat16", 1, (65, 1000)),           # 12 rows
    (32, 8, 128, 8, 64, 16, "bfloat16", 5, (5, 600, 1024)),      # two row blocks
    (14, 2, 128, 16, 32, 16, "float16", 2, (9, 77, 400)),
    (8, 2, 128, 8, 64, 16, "bfloat16", 1, (5000, 3)),            # few segments, long
    (4, 1, 128, 16, 32, 16, "bfloat16", 1, (9000,)),
    (4, 1, 256, 4, 64, 128, "float16", 1, (20000,)),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x) for x in c[:8]))
def test_own_runs_match_explicit_waves(case):
    from pkv import ops

    heads, hk, dim, bits, group, page, dtype, nq, lengths = case
    gen = torch.Generator(device="cuda").manual_seed(dim + nq)
    fmt = ops.PageFormat(hk, dim, page, bits, group, getattr(torch, dtype))
    lens = np.array(lengths, np.int32)
    batch, per = len(lens), -(-int(lens.max()) // page)
    table = torch.randperm(batch * per, generator=gen, device="cuda").to(torch.int32).view(batch, per)
    # stale bytes past every sequence's end
    pool = torch.randint(0, 256, (batch * per, fmt.page_bytes), generator=gen, dtype=torch.uint8,
                         device="cuda")
    k, v = (torch.randn((batch, hk, int(lens.max()), dim), generator=gen, device="cuda").to(fmt.dtype)
            for _ in range(2))
    q = torch.randn((batch, heads, nq, dim), generator=gen, device="cuda").to(fmt.dtype)
    zeros = torch.zeros(batch, dtype=torch.int32)
    ops.append_quantize(fmt, pool, k, v, table, zeros, (lens - 1).tolist())
    lens_d = torch.from_numpy(lens).cuda()
    new = [torch.stack([x[b, :, lens[b] - 1:lens[b]] for b in range(batch)]) for x in (k, v)]
    widths = torch.from_numpy(np.minimum(lens, nq).astype(np.int32)) if nq > 1 else None
    args = dict(scale=dim ** -0.5)

    steps = 2.0 ** -7 if dtype == "bfloat16" else 2.0 ** -10

    def close(a, b):
        a, b = a.float(), b.float()
        assert torch.isfinite(a).all() and torch.isfinite(b).all()
        bound = b.abs() * steps + b.abs().amax(-1, keepdim=True) * 2.0 ** -8 + 1e-6
        assert bool(((a - b).abs() <= bound).all()), float(((a - b).abs() - bound).max())

    apart = pool.clone()
    ops.append_quantize(fmt, apart, *new, table, (lens - 1).tolist())
    own = ops.paged_attention(fmt, apart, q, table, lens_d, widths=widths, **args)
    for waves in (37, 1024):
        close(own, ops.paged_attention(fmt, apart, q, table, lens_d, widths=widths, waves=waves, **args))
    if nq == 1:  # the same step with the append in the call
        for waves in (0, 37):
            fused = pool.clone()
            out = ops.append_paged_attention(fmt, fused, *new, q, table, lens_d, waves=waves, **args)
            assert torch.equal(fused, apart)
            close(out, own)
