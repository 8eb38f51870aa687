"""GPU parity of the norms on short rows, at the edges of their layouts.

A row is held by 4 to 64 lanes with one to three 16-byte vectors each, and in
the backward past 128 vectors by teams of three, four or eight waves; these
widths are the last of one layout and the first of the next, with few rows
(one partial step) and with enough for several steps of a full grid and a
ragged last one.  Bounds as in ``test_gpu_norms``.
"""

import pytest
import torch

from test_gpu_add_rmsnorm import test_add_rmsnorm_fwd_bwd as _add_case
from test_gpu_norms import test_layernorm_fwd_bwd as _ln_case
from test_gpu_norms import test_rmsnorm_fwd_bwd as _rms_case

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16]
VECTORS = [3, 4, 5, 8, 9, 16, 17, 32, 33, 48, 49, 64, 65, 96, 97, 128, 129, 192, 193, 256, 257]


def _shape(i, vectors, many):
    dtype = DTYPES[i % 3]
    dim = vectors * (4 if dtype == torch.float32 else 8)
    # 8,203 rows: two steps of 512 blocks at one row per wave, and the forward's grouped loads
    return dtype, ((8203 if vectors <= 64 else 4203) if many else 35, dim)


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("i,vectors", list(enumerate(VECTORS)))
def test_short_rows(i, vectors, many):
    _rms_case(*_shape(i, vectors, many), with_w=vectors != 33)
    _ln_case(*_shape(i + 1, vectors, many), params="wb" if vectors != 48 else "b")
    _add_case(*_shape(i + 2, vectors, many), with_w=vectors != 64, with_dh=True)
