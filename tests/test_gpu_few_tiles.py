"""GPU: grouped decode runs over few tiles (fewer runs, each with an iteration of
every wave) against the same call with explicit waves, with the checks of
``test_gpu_segment_runs``: lengths past the whole-segment form, one to a few
(sequence, KV head) segments, runs that end inside a segment and on its edge.
"""

from __future__ import annotations

import pytest

runs = pytest.importorskip("test_gpu_segment_runs")
pytestmark = pytest.mark.gpu

CASES = [
    # (heads, kv_heads, dim, bits, group, page, dtype, queries, lengths)
    (8, 1, 128, 4, 64, 32, "bfloat16", 1, (4000,)),           # 8 rows: grouped by default, fused
    (8, 1, 128, 4, 64, 32, "bfloat16", 1, (2500, 1300)),
    (4, 1, 128, 8, 64, 16, "bfloat16", 1, (3000,)),           # 4 rows: grouped for few segments
    (4, 1, 128, 8, 64, 16, "bfloat16", 1, (2048, 1024)),
    (8, 2, 64, 16, 32, 16, "bfloat16", 1, (1500, 1499, 1)),
    (12, 1, 128, 8, 64, 16, "bfloat16", 1, (700,)),           # 12 rows, one column slot
    (16, 2, 256, 8, 128, 64, "float16", 1, (1111,)),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x) for x in c[:8]) + f"-{c[8][0]}")
def test_few_tiles_match_explicit_waves(case):
    runs.test_own_runs_match_explicit_waves(case)
