"""GPU parity of the norms on short rows, at the edges of their layouts.

A row is held by 4 to 64 lanes with one to three 16-byte vectors each, and in
the backward past 128 vectors by teams of three, four or eight waves; these
widths are the last of one layout and the first of the next, with few rows
(one partial step) and with enough for several steps of a full grid and a
ragged last one.  Widths that are not whole vectors, and buffers that are not
aligned to one, take the same layouts with element-aligned vectors.  Bounds as
in ``test_gpu_norms``.
"""

import pytest
import torch

import test_gpu_add_rmsnorm
import test_gpu_norms
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


# widths that are not whole 16-byte vectors: one element more than a layout's
# last whole vector, one fewer than the next, and the widest rows of either pass
ODD_VECTORS = [1, 2, 4, 9, 17, 33, 49, 65, 97, 129, 193, 257, 513, 1000]


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("i,vectors", list(enumerate(ODD_VECTORS)))
def test_odd_widths(i, vectors, many):
    def odd(j, extra):
        dtype, (rows, dim) = _shape(j, vectors, many and vectors <= 257)
        vec = 4 if dtype == torch.float32 else 8
        return dtype, (rows, dim + (1 if extra else vec - 1))

    _rms_case(*odd(i, True), with_w=vectors != 33)
    _ln_case(*odd(i + 1, False), params="wb" if vectors != 49 else "b")
    _add_case(*odd(i + 2, vectors % 2 == 0), with_w=vectors != 65, with_dh=True)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dim", [64, 768, 1536, 4096, 1001])
def test_unaligned_buffers(monkeypatch, dtype, dim):
    """Rows, parameters and gradients that start one element past a 16-byte boundary."""
    def off_by_one(shape, *args, **kw):
        t = aligned(shape, *args, **kw)
        return torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(shape)

    aligned = test_gpu_norms.randn
    monkeypatch.setattr(test_gpu_norms, "randn", off_by_one)
    monkeypatch.setattr(test_gpu_add_rmsnorm, "randn", off_by_one)
    for rows in (37, 4203):
        _rms_case(dtype, (rows, dim), with_w=True)
        _ln_case(dtype, (rows, dim), params="wb")
        _add_case(dtype, (rows, dim), with_w=True, with_dh=True)
