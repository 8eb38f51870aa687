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


@pytest.mark.parametrize("dtype,dim,off", [
    (torch.float32, 5, 0), (torch.float32, 301, 0), (torch.float32, 768, 1), (torch.float32, 1001, 0),
    (torch.float32, 2999, 0), (torch.float16, 130, 0), (torch.float16, 770, 0), (torch.float16, 4095, 0)])
def test_layernorm_xhat_far_from_zero(dtype, dim, off):
    """The weight gradient sum(dy * x-hat) of rows 1,000 standard deviations from
    zero, given their statistics: x - 1,000 is a multiple of 1/2 and dy +-1, so
    x-hat = (x - mean) * rstd has the rounding of two operations, and the sum at
    most 2^-24 per addition (as many as rows) of the sum of magnitudes.  The
    rounding of mean * rstd, left in x-hat, is up to 2^-14."""
    from scree_amd.kernels.hip import norms

    rows = 35
    g = torch.Generator().manual_seed(dim + rows)
    x = (1000 + 0.5 * torch.randint(-2, 3, (rows, dim), generator=g)).to(dtype)
    dy = (2 * torch.randint(0, 2, (rows, dim), generator=g) - 1).to(dtype)
    x, dy = (torch.cat([torch.zeros(off, dtype=dtype), t.reshape(-1)]).cuda()[off:].view(rows, dim) for t in (x, dy))
    mean = torch.full((rows,), 1000.0, device="cuda")
    rstd = (0.5 + 1.5 * torch.rand(rows, generator=g)).cuda()  # mean * rstd is not a float
    w = torch.ones(dim, dtype=dtype, device="cuda")
    _, dw, db = norms.layernorm_bwd(dy, x, w, mean, rstd, True, True, p_like=w.float())
    terms = dy.double() * (x.double() - 1000) * rstd.double()[:, None]
    bound = (rows + 2) * 2.0 ** -24 * terms.abs().sum(0)
    err = (dw.double() - terms.sum(0)).abs()
    print(f"case: LayerNorm x-hat {dtype} {rows} x {dim} + {off}: {float((err / bound).max()):.3f} of the bound", flush=True)
    assert (err <= bound).all()
    assert torch.equal(db.double(), dy.double().sum(0))


@pytest.mark.parametrize("dtype,dim", [(torch.float32, 5), (torch.float32, 301), (torch.bfloat16, 128),
                                       (torch.float16, 770), (torch.bfloat16, 1536), (torch.bfloat16, 4095)])
def test_non_finite_rows_stay_alone(dtype, dim):
    """A NaN as a row's last element (repeated by an odd width's last vector) and
    an infinity as another's first: those rows as the formulas give them, every
    other row bit for bit as without them, and NaN in the parameter gradients."""
    from scree_amd.kernels.hip import norms

    print(f"case: non-finite rows {dtype} x {dim}", flush=True)
    rows, randn = 37, test_gpu_norms.randn
    x, r, dy = (randn((rows, dim), dtype, 7 + i) for i in range(3))
    w, b = (randn((dim,), dtype, 10 + i) for i in range(2))
    bad = x.clone()
    bad[3, -1], bad[20, 0] = float("nan"), float("inf")
    others = torch.tensor([i not in (3, 20) for i in range(rows)], device="cuda")

    def steps(x):
        y, rs = norms.rmsnorm_fwd(x, w, 1e-6, True)
        yield (y, *norms.rmsnorm_bwd(dy, x, w, rs, True, dw_like=w))
        y, mu, rs = norms.layernorm_fwd(x, w, b, 1e-5, True)
        yield (y, *norms.layernorm_bwd(dy, x, w, mu, rs, True, True, p_like=w)[:2])
        h, y, rs = norms.add_rmsnorm_fwd(x, r, w, 1e-6, True)
        yield (y, *norms.add_rmsnorm_bwd(dy, r, h, w, rs, True, dw_like=w))

    for i, ((y, dx, dw), (y0, dx0, _)) in enumerate(zip(steps(bad), steps(x))):
        for a, a0 in ((y, y0), (dx, dx0)):
            assert torch.isfinite(a0).all()
            assert torch.equal(a[others], a0[others])
            assert a[3].isnan().all()
        assert dw.isnan().all()
        if i == 1:  # LayerNorm: the mean is infinite
            assert y[20].isnan().all()
        else:       # RMSNorm: rstd is 0
            assert y[20, 0].isnan() and not y[20, 1:].any()
