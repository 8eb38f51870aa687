"""GPU parity of the varlen softmax where few workgroups make it narrow.

A grid of fewer than 256 (128) workgroups narrows a workgroup's column lanes
to half a cache line (a quarter, an eighth); each width here also has a
sequence longer than the rows a workgroup holds, and empty and one-row ones.
Bounds as in ``test_gpu_softmax``.
"""

import pytest
import torch

from test_gpu_softmax import _run

pytestmark = pytest.mark.gpu

# five sequences, so 5 * ceil(columns / lanes) workgroups at a width (empty ones count)
LENGTHS = [700, 0, 9000, 1, 0]


@pytest.mark.parametrize("dtype,features", [
    (torch.float32, 4),      # one vector: 1 lane
    (torch.bfloat16, 64),    # 8 vectors: 1 lane (40 workgroups)
    (torch.float16, 520),    # 65 vectors: 2 lanes (165)
    (torch.float32, 600),    # 150 vectors: 4 lanes (190)
    (torch.bfloat16, 2048),  # 256 vectors: 4 lanes stay at 320 -> 8 lanes would be 160
    (torch.float32, 3),      # scalar columns: 1 lane
    (torch.float16, 301),    # scalar columns: 8 lanes (190) -> 4
])
def test_narrow_softmax(dtype, features):
    _run(LENGTHS, (features,), dtype, seed=features)


@pytest.mark.parametrize("features", [8, 32, 40, 512])
def test_many_short_sequences(features):
    """300 sequences of at most 40 rows: no narrowing, up to 64 column lanes."""
    _run([(7 * i) % 41 for i in range(300)], (features,), torch.bfloat16, seed=features + 1)
