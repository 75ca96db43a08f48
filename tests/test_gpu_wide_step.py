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


@pytest.mark.parametrize("heads", [40, 71])
def test_bits_do_not_depend_on_the_shared_workspace(heads):
    from pkv import ops

    fused, _ = _case(heads)
    _forget()
    first = fused()
    ops.attention_workspace(torch.device("cuda", 0), 64 << 20)
    assert torch.equal(first, fused())


@pytest.mark.parametrize("heads", [40, 71])
def test_two_streams(heads):
    """Steps on two streams at once give the bits they give alone, with a shared
    workspace large enough for either's partials."""
    from pkv import ops

    steps = [_case(heads, seed, (6000, 2000 + seed))[0] for seed in (0, 1)]
    ops.attention_workspace(torch.device("cuda", 0), 64 << 20)
    want = [step() for step in steps]
    streams = [torch.cuda.Stream() for _ in steps]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    got = [[], []]
    for _ in range(30):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i].append(steps[i]())
    torch.cuda.synchronize()
    for outs, w in zip(got, want):
        assert all(torch.equal(out, w) for out in outs)


def test_captured_step_equals_the_eager_one():
    from pkv.device_arena import DevicePageArena, DeviceRunner
    from pkv.layer import AttentionStack, ModelSpec
    from pkv.ops import PageFormat

    spec = ModelSpec(hidden=128, query_heads=40, kv_heads=1, head_dim=64, num_layers=2, dtype="bfloat16")
    model = AttentionStack(spec, device="cuda", seed=3)
    arena = DevicePageArena(PageFormat(1, 64, 16, 8, 64), 400, num_layers=2, max_slots=2, max_tokens=3000)
    runner = DeviceRunner(model, arena)
    slots = [arena.open_slot() for _ in range(2)]
    gen = torch.Generator(device="cuda").manual_seed(1)
    draw = lambda n: torch.randn((2, n, 128), generator=gen, device="cuda").to(torch.bfloat16)
    runner.execute(slots, draw(2400), [2400, 1100])
    step = runner.capture_decode(slots, draw(1))
    for _ in range(3):
        before = list(arena.lengths)
        step.hidden.copy_(draw(1))
        step.replay()
        out = step.out.clone()
        arena.truncate(slots, before)
        eager = runner.execute(slots, step.hidden)
        assert torch.equal(out, eager)


def test_without_room_for_partials_the_call_runs_whole_spans(monkeypatch):
    """The partials' memory refused (a full device): the wide call and the wide
    step take the small workspace and give whole spans' bits."""
    from pkv import ops

    gen = torch.Generator(device="cuda").manual_seed(2)
    fmt = ops.PageFormat(2, 64, 16, 8, 64)
    n, nq = 2000, 70
    per = -(-n // 16)
    table = torch.randperm(2 * per, generator=gen, device="cuda").to(torch.int32).view(2, per)
    pool = ops.allocate_pool(fmt, 2 * per)
    lens = torch.tensor([n, 1200], dtype=torch.int32, device="cuda")
    widths = torch.tensor([nq, 1], dtype=torch.int32, device="cuda")
    k, v = (torch.randn((2, 2, n, 64), generator=gen, device="cuda").to(fmt.dtype) for _ in range(2))
    ops.append_quantize(fmt, pool, k, v, table, torch.zeros_like(lens), lens)
    q = torch.randn((2, 8, nq, 64), generator=gen, device="cuda").to(fmt.dtype)
    waves = ops.split_waves(fmt, 8, nq, 2, q.device)
    small = torch.empty(ops.workspace_bytes(fmt, 8, nq, waves), dtype=torch.uint8, device="cuda")
    call = lambda **kw: ops.paged_attention(fmt, pool, q, table, lens, scale=0.125, widths=widths, **kw)
    whole = call(waves=waves, workspace=small)
    step, _ = _case(40)
    empty, refused, limit = torch.empty, [], [small.numel()]

    def full(*args, **kw):
        if kw.get("dtype") is torch.uint8 and args[0] > limit[0]:
            refused.append(args[0])
            raise torch.OutOfMemoryError
        return empty(*args, **kw)

    cut = step()
    monkeypatch.setattr(torch, "empty", full)
    assert torch.equal(call(), whole) and len(refused) == 1
    limit[0] = 256
    out = step()
    monkeypatch.undo()
    assert len(refused) == 2 and torch.isfinite(out).all()
    bound = cut.float().abs() * 2.0 ** -7 + cut.float().abs().amax(-1, keepdim=True) * 2.0 ** -8 + 1e-6
    assert bool(((out.float() - cut.float()).abs() <= bound).all())
