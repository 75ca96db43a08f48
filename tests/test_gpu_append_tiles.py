"""GPU: an append of several tokens per sequence (one wave per page tile) writes
the bytes that appending them one at a time (one wave per token) writes.

The one-token append is pinned bit for bit against the quantizer oracle by the
parity suite; here every layout, ragged widths, begun and ended tiles, rows
that are not 16-byte aligned, unmapped pages and values past the f16 range
(infinite scales, infinities, NaN) give the same pool either way.
"""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

CASES = [
    # (bits, dim, group, page, dtype, tokens, values)
    (8, 128, 64, 16, "bfloat16", 37, "normal"),
    (8, 128, 128, 32, "float16", 9, "normal"),
    (8, 64, 32, 16, "bfloat16", 65, "normal"),
    (8, 256, 32, 64, "bfloat16", 33, "normal"),
    (4, 128, 64, 16, "bfloat16", 48, "normal"),
    (4, 64, 64, 128, "float16", 19, "normal"),
    (4, 256, 128, 16, "bfloat16", 31, "normal"),
    (16, 64, 32, 16, "float16", 40, "normal"),
    (16, 128, 32, 32, "bfloat16", 50, "normal"),
    (16, 256, 32, 16, "bfloat16", 17, "normal"),
    # rows of odd length, and rows that start off a 16-byte address
    (8, 37, 32, 16, "bfloat16", 34, "normal"),
    (4, 100, 32, 16, "float16", 18, "normal"),
    (16, 37, 32, 16, "bfloat16", 21, "normal"),
    (8, 128, 64, 16, "bfloat16", 20, "offset"),
    # scales past the f16 range, infinities, NaN, constant rows, signed zeros
    (8, 128, 64, 16, "bfloat16", 33, "wild"),
    (4, 128, 32, 16, "bfloat16", 33, "wild"),
]


def _values(shape, dtype, kind, rng):
    x = rng.standard_normal(shape).astype(np.float32)
    if kind == "wild":
        rows = x.reshape(-1, shape[-1])
        pick = rng.integers(0, 8, len(rows))
        rows[pick == 0] *= 1e9          # bias and scale past the f16 range
        rows[pick == 1] *= 3e6          # large finite scales
        rows[pick == 2, 5] = np.inf
        rows[pick == 3, 6] = -np.inf
        rows[pick == 4, 7] = np.nan
        rows[pick == 5] = 0.25
        rows[pick == 6] = np.where(rows[pick == 6] > 0, 0.0, -0.0)
    t = torch.from_numpy(x).to("cuda", getattr(torch, dtype))
    if kind == "offset":
        flat = torch.empty(t.numel() + 3, dtype=t.dtype, device="cuda")
        flat[3:] = t.reshape(-1)
        t = flat[3:].view(shape)
    return t


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x) for x in c))
def test_several_tokens_append_as_one_at_a_time(case):
    from pkv import ops

    bits, dim, group, page, dtype, tokens, kind = case
    rng = np.random.default_rng(tokens)
    batch, heads = 5, 3
    fmt = ops.PageFormat(heads, dim, page, bits, group, getattr(torch, dtype))
    # starts at every place in a tile; widths 0 (nothing), 1, ragged and full
    starts = np.array([0, 15, 16, 7, 33], np.int32)
    widths = np.array([tokens, 0, 1, max(1, tokens // 2), tokens], np.int32)
    per = -(-(int(starts.max()) + tokens) // page)
    table = rng.permutation(batch * per).astype(np.int32).reshape(batch, per)
    table[4, -1] = -1  # an unmapped page takes nothing
    table_d = torch.from_numpy(table).cuda()
    k, v = (_values((batch, heads, tokens, dim), dtype, kind, rng) for _ in range(2))
    pools = [torch.full((batch * per, fmt.page_bytes), 0xA5, dtype=torch.uint8, device="cuda")
             for _ in range(2)]
    lens = torch.full((batch,), -1, dtype=torch.int32, device="cuda")
    ops.append_quantize(fmt, pools[0], k, v, table_d, torch.from_numpy(starts),
                        torch.from_numpy(widths), new_lens=lens)
    for t in range(tokens):
        ops.append_quantize(fmt, pools[1], k[:, :, t:t + 1], v[:, :, t:t + 1], table_d,
                            torch.from_numpy(starts + t), torch.from_numpy((widths > t).astype(np.int32)))
    assert torch.equal(pools[0], pools[1])
    assert lens.cpu().tolist() == (starts + widths).tolist()
