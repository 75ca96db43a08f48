"""GPU: the page export by tiles gives the bytes of the general export kernel, and
page copies of several workgroups per page copy every byte.

Outputs off a 16-byte address take the general kernel (pinned to the oracle by
the parity suite's append -> gather cases), so the same pages into such tensors
are the reference; ids outside the pool leave their rows as they are.
"""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

LAYOUTS = [
    # (bits, dim, group, page, dtype, heads)
    (8, 128, 64, 16, "bfloat16", 3),
    (8, 64, 32, 32, "float16", 1),
    (8, 256, 128, 64, "bfloat16", 2),
    (8, 37, 32, 16, "bfloat16", 2),
    (8, 80, 32, 128, "bfloat16", 2),
    (4, 128, 64, 16, "bfloat16", 3),
    (4, 64, 64, 32, "bfloat16", 2),
    (4, 256, 32, 16, "float16", 1),
    (4, 100, 128, 16, "bfloat16", 2),
    (16, 64, 32, 16, "float16", 3),
    (16, 128, 32, 32, "bfloat16", 2),
    (16, 256, 32, 16, "bfloat16", 1),
    (16, 72, 32, 16, "bfloat16", 2),
]


def _pool(case, pages):
    from pkv import ops

    bits, dim, group, page, dtype, heads = case
    fmt = ops.PageFormat(heads, dim, page, bits, group, getattr(torch, dtype))
    gen = torch.Generator(device="cuda").manual_seed(dim + bits)
    return fmt, torch.randint(0, 256, (pages, fmt.page_bytes), generator=gen, dtype=torch.uint8,
                              device="cuda")


@pytest.mark.parametrize("case", LAYOUTS, ids=lambda c: "-".join(str(x) for x in c))
def test_export_by_tiles_matches_the_general_kernel(case):
    from pkv import _native as nat
    from pkv import ops

    fmt, pool = _pool(case, 9)
    ids = torch.tensor([4, 0, 8, 3, 7], dtype=torch.int32, device="cuda")
    got = ops.gather_pages(fmt, pool, ids)
    # the same tensors, each 2 bytes past an aligned address
    flat = [torch.zeros(t.numel() * t.element_size() + 2, dtype=torch.uint8, device="cuda") for t in got]
    args = [t.data_ptr() + 2 for t in flat]
    if not fmt.quantized:
        args = [args[0], None, None, args[1], None, None]
    nat.check(nat.load().pkv_gather_pages(nat.stream_handle(pool.device), fmt.c_layout, nat.ptr(pool),
                                          pool.shape[0], nat.ptr(ids), ids.numel(), *args), "gather")
    for t, f in zip(got, flat):
        assert torch.equal(t.reshape(-1).view(torch.uint8), f[2:])


def test_export_skips_ids_outside_the_pool():
    from pkv import _native as nat
    from pkv import ops

    fmt, pool = _pool(LAYOUTS[0], 5)
    whole = ops.gather_pages(fmt, pool, torch.tensor([2, 2, 2], dtype=torch.int32))
    ids = torch.tensor([-1, 2, 5], dtype=torch.int32, device="cuda")
    outs = [torch.full_like(t, 7) for t in whole]
    nat.check(nat.load().pkv_gather_pages(nat.stream_handle(pool.device), fmt.c_layout, nat.ptr(pool),
                                          pool.shape[0], nat.ptr(ids), 3, *[nat.ptr(t) for t in outs]), "gather")
    for t, w in zip(outs, whole):
        assert torch.equal(t[1].view(torch.uint8), w[1].view(torch.uint8))  # (random bits hold NaN)
        assert bool((t[0] == 7).all()) and bool((t[2] == 7).all())


@pytest.mark.parametrize("case", [LAYOUTS[2], LAYOUTS[4], LAYOUTS[6]], ids=lambda c: "-".join(str(x) for x in c))
def test_page_copies_copy_every_byte(case):
    from pkv import ops

    fmt, pool = _pool(case, 8)
    want = pool.clone()
    for s, d in ((1, 6), (0, 7)):
        want[d] = want[s]
    ops.copy_pages(fmt, pool, [1, 9, 0, 3], [6, 2, 7, -1])
    assert torch.equal(pool, want)
