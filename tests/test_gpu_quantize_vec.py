"""GPU: the row quantizer's and dequantizer's vector kernels give the bytes of the
general kernels.

Rows that do not start at a 16-byte address take the general kernels (pinned to
the quantizer oracle by the parity suite), so the same values at an odd offset
are the reference here: remainders of a workgroup, padded rows, every group
size, and rows with infinities, NaN and ranges past f16.
"""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _rows(rows, dim, dtype, wild):
    rng = np.random.default_rng(rows * 1000 + dim)
    x = rng.standard_normal((rows, dim)).astype(np.float32)
    x[::5] *= 300.0
    x[3::7] = 0.25
    if wild:
        x[1::6] *= 1e9
        x[2::6, 0] = np.inf
        x[4::6, dim // 2] = -np.inf
        x[5::6, -1] = np.nan
    return torch.from_numpy(x).to("cuda", getattr(torch, dtype))


def _general(values, bits, group):
    """The same rows one element off alignment, through the C ABI."""
    from pkv import _native as nat
    from pkv import ops

    rows, dim = values.shape
    off = torch.empty(values.numel() + 1, dtype=values.dtype, device="cuda")
    off[1:] = values.reshape(-1)
    got = ops.quantize_rows(off[1:].view(rows, dim), bits, group)
    flat = torch.empty(rows * dim + 1, dtype=torch.float32, device="cuda")
    out = flat[1:]  # 4 bytes off a 16-byte address
    nat.check(nat.load().pkv_dequantize_rows(
        nat.stream_handle(values.device), *[nat.ptr(t) for t in got], rows, dim, bits, group,
        nat.ptr(out)), "dequantize")
    return got, out.view(rows, dim)


@pytest.mark.parametrize("wild", [False, True], ids=["finite", "wild"])
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows,dim,group", [
    (1, 8, 32), (3, 128, 32), (129, 128, 64), (65, 128, 128), (37, 96, 64), (130, 80, 32),
    (11, 264, 128), (5, 4096, 64), (33, 100, 32),
])
def test_vector_rows_match_the_general_kernels(rows, dim, group, bits, dtype, wild):
    from pkv import ops

    values = _rows(rows, dim, dtype, wild)
    got = ops.quantize_rows(values, bits, group)
    want, floats = _general(values, bits, group)
    for g, w in zip(got, want):
        assert torch.equal(g.view(torch.uint8), w.view(torch.uint8))
    back = ops.dequantize_rows(got, bits, dim, group)
    assert torch.equal(back.view(torch.int32), floats.view(torch.int32))
