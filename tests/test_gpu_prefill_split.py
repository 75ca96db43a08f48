"""GPU: prefill spans cut into pieces (f32 partials, merged with the decode parts'
in one launch) against the same call with a workspace that holds no partials,
and against the oracle.

A workspace of the decode parts' size alone runs the call as it is without the
split, so the same inputs through both give the reference: outputs within two
bf16 steps of the element plus 2^-8 of the row's largest element (each form
rounds its probabilities to 16 bits against its own running maximum), the
rows past a sequence's width exactly zero in both.
"""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

CASES = [
    # (batch, heads, kv_heads, dim, bits, group, page, dtype, queries, cached, widths)
    (1, 32, 8, 128, 8, 64, 16, "bfloat16", 500, (1300,), (500,)),      # S = 4, one segment per XCD
    (1, 8, 2, 128, 4, 64, 32, "bfloat16", 200, (700,), None),          # segments not a multiple of 8
    (3, 12, 3, 64, 8, 32, 16, "float16", 77, (0, 500, 1100), (77, 1, 40)),
    (2, 4, 1, 256, 8, 128, 64, "bfloat16", 130, (400, 900), (130, 64)),
    (2, 8, 8, 128, 16, 32, 16, "bfloat16", 90, (300, 800), (90, 90)),
    (4, 8, 1, 100, 4, 32, 16, "bfloat16", 150, (0, 0, 20, 3000), (150, 2, 5, 150)),
    (6, 8, 2, 128, 8, 64, 16, "bfloat16", 300, (90, 500, 40, 1, 700, 0), (1, 300, 4, 1, 2, 130)),  # mixed
    (2, 4, 1, 128, 16, 32, 16, "float16", 64, (0, 5), (64, 33)),       # spans too short to cut
    (1, 4, 1, 64, 8, 64, 128, "bfloat16", 2000, (2100,), (1777,)),
    (2, 8, 2, 128, 8, 64, 16, "bfloat16", 100, (10, 30), (3, 2)),      # no wide sequence in a wide call
]


def _run(case, positions=False):
    from pkv import ops

    batch, heads, hk, dim, bits, group, page, dtype, nq, cached, widths = case
    gen = torch.Generator(device="cuda").manual_seed(dim + nq)
    fmt = ops.PageFormat(hk, dim, page, bits, group, getattr(torch, dtype))
    w = np.array(widths or (nq,) * batch, np.int32)
    lens = np.array(cached, np.int32) + w
    per = -(-int(lens.max()) // page)
    table = torch.randperm(batch * per, generator=gen, device="cuda").to(torch.int32).view(batch, per)
    pool = ops.allocate_pool(fmt, batch * per)
    kv = [torch.randn((batch, hk, int(lens.max()), dim), generator=gen, device="cuda").to(fmt.dtype)
          for _ in range(2)]
    ops.append_quantize(fmt, pool, *kv, table, torch.zeros(batch, dtype=torch.int32), lens.tolist())
    q = torch.randn((batch, heads, nq, dim), generator=gen, device="cuda").to(fmt.dtype)
    if widths:  # padding rows may hold anything
        for b in range(batch):
            q[b, :, int(w[b]):] = float("nan")
    args = dict(scale=dim ** -0.5, widths=torch.from_numpy(w) if widths else None)
    if positions:
        args["q_pos"] = torch.from_numpy((lens - w)[:, None] + np.arange(nq)[None]).to(torch.int32)
    need = ops.workspace_bytes(fmt, heads, nq, 64)
    small = torch.empty(max(256, need), dtype=torch.uint8, device="cuda")
    whole = ops.paged_attention(fmt, pool, q, table, lens.tolist(), waves=64, workspace=small, **args)
    cut = ops.paged_attention(fmt, pool, q, table, lens.tolist(), **args)
    again = ops.paged_attention(fmt, pool, q, table, lens.tolist(), **args)
    return w, whole, cut, again, (fmt, pool, table, lens, q, kv)


@pytest.mark.parametrize("positions", [False, True], ids=["lens", "q_pos"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x) for x in c[:9]))
def test_cut_spans_match_whole_spans(case, positions):
    w, whole, cut, again, _ = _run(case, positions)
    assert torch.equal(cut.view(torch.int16), again.view(torch.int16))
    for b, n in enumerate(w):
        assert not cut[b, :, int(n):].any() and not whole[b, :, int(n):].any()
    a, b = cut.float(), whole.float()
    assert torch.isfinite(a).all()
    steps = 2.0 ** -7 if case[7] == "bfloat16" else 2.0 ** -10
    bound = b.abs() * steps + b.abs().amax(-1, keepdim=True) * 2.0 ** -8 + 1e-6
    assert bool(((a - b).abs() <= bound).all()), float(((a - b).abs() - bound).max())


@pytest.mark.parametrize("case", [CASES[0], CASES[1], CASES[6]], ids=lambda c: "-".join(str(x) for x in c[:9]))
def test_cut_spans_match_float64(case):
    """Against float64 attention over the pages' own values (exported)."""
    from pkv import ops

    batch, heads, hk, dim, bits, group, page, dtype, nq, cached, widths = case
    w, _, cut, _, (fmt, pool, table, lens, q, _) = _run(case)
    for b in range(batch):
        n, length = int(w[b]), int(lens[b])
        ids = table[b, :-(-length // page)].contiguous()
        t = ops.gather_pages(fmt, pool, ids)
        k, v = (ops.dequantize_rows(t[3 * i:3 * i + 3], bits, dim, group).double().transpose(0, 1)
                .reshape(hk, -1, dim)[:, :length] for i in range(2))
        s = torch.bmm(q[b, :, :n].double().reshape(hk, -1, dim), k.transpose(1, 2).contiguous()) * dim ** -0.5
        at = (torch.arange(n, device="cuda") + length - n).repeat(heads // hk)
        s.masked_fill_(torch.arange(length, device="cuda")[None] > at[:, None], float("-inf"))
        want = torch.bmm(torch.softmax(s, -1), v.contiguous()).view(heads, n, dim)
        err = (cut[b, :, :n].double() - want).abs()
        assert float(err.max()) <= 2e-2 and float(err.mean()) <= 2e-3


def test_workspace_of_a_batch_covers_the_smaller_one():
    from pkv import _native as nat
    from pkv import ops

    lib = nat.load()
    for bits, dim, group in ((8, 128, 64), (4, 256, 64), (16, 64, 32)):
        lay = ops.PageFormat(2, dim, 16, bits, group).c_layout
        for nq in (1, 5, 64, 500):
            for batch in (1, 3, 64):
                assert lib.pkv_attention_batch_workspace_bytes(lay, 8, nq, batch, 100) >= \
                    lib.pkv_attention_workspace_bytes(lay, 8, nq, 100)
        assert lib.pkv_attention_batch_workspace_bytes(lay, 8, 64, 0, 100) < 0
