"""GPU parity of the fp32 matrix-instruction attention at the sizes where its
forms can go wrong: sequence lengths around the 32-row tile and the 128-row
item, with 4, 2 and 1 waves sharing a row tile in each pass (the launchers
choose by the number of row tiles, for dK/dV as if its launch were the smaller
by the query heads per K/V head), in both mask modes, with and without grouped
K/V heads.  Bounds as in ``test_gpu_attention_fp32``.
"""

import pytest
import torch

from parity import cu_of, np64, randn, say
from test_gpu_attention_fp32 import TOL, run_fp32_case

pytestmark = pytest.mark.gpu

TILE_LENGTHS = [1, 31, 32, 33, 64, 65, 96, 127, 128, 129, 160, 2]
MANY_LENGTHS = TILE_LENGTHS + [(7 * i) % 30 + 1 for i in range(48)]


def shares(lengths, dim, heads, kv_heads):
    """Waves per row tile of the forward and dQ, and of dK/dV (the launchers'
    rule restated, so that each case knows which kernels it runs)."""
    def share(blocks):
        tiles = 4 * blocks
        if tiles < (1024 if dim >= 64 else 2048):
            return 4
        return 2 if tiles < (3072 if dim >= 128 else 5120) else 1

    tmax = -(-sum(lengths) // 128) + len(lengths)
    return share(tmax * heads), share(tmax * kv_heads // (heads // kv_heads))


@pytest.mark.parametrize("heads,waves", [(8, 4), (32, 2), (84, 1)])  # 608, 2,432 and 6,384 row tiles
@pytest.mark.parametrize("dim", [16, 32, 64, 128])
@pytest.mark.parametrize("causal", [True, False])
def test_fp32_waves_per_row_tile(dim, heads, waves, causal):
    assert shares(TILE_LENGTHS, dim, heads, heads) == (waves, waves)
    run_fp32_case(TILE_LENGTHS, heads, dim, causal, seed=900 + dim)


@pytest.mark.parametrize("dim,heads,waves", [
    (16, 4, (4, 4)), (16, 12, (2, 4)), (16, 32, (1, 2)), (16, 72, (1, 1)),
    (32, 4, (4, 4)), (32, 12, (2, 4)), (32, 32, (1, 2)), (32, 72, (1, 1)),
    (64, 2, (4, 4)), (64, 12, (2, 4)), (64, 16, (2, 2)), (64, 72, (1, 1)),
    (128, 2, (4, 4)), (128, 8, (2, 4)), (128, 16, (1, 2)), (128, 44, (1, 1))])
@pytest.mark.parametrize("causal", [True, False])
def test_fp32_waves_per_row_tile_grouped(dim, heads, waves, causal):
    """Two query heads per K/V head: each dK/dV form steps to the next head of a group."""
    assert shares(MANY_LENGTHS, dim, heads, heads // 2) == waves
    run_fp32_case(MANY_LENGTHS, heads, dim, causal, seed=950 + dim, kv_heads=heads // 2)


@pytest.mark.parametrize("dim", [16, 64, 128])
def test_fp32_single_token_any_row_stride(dim):
    """One token whose row stride says nothing (0, as a size-1 axis may have):
    the same output and gradients as from a contiguous tensor."""
    import scree_amd
    from scree_amd.kernels import varlen_attention

    say(f"case: fp32 one token, row stride 0, D={dim}")
    _, cu = cu_of([1])
    heads = 4
    base = [randn((1, heads, dim), torch.float32, 40 + i) for i in range(4)]

    def run(ts):
        qa, ka, va = (t.detach().requires_grad_(True) for t in ts[:3])
        out = varlen_attention(*(scree_amd.Array(values=t, offsets=cu) for t in (qa, ka, va)),
                               causal=True).values
        out.backward(ts[3])
        return [out.detach(), qa.grad, ka.grad, va.grad]

    got = run([t.as_strided((1, heads, dim), (0, dim, 1)) for t in base])
    want = run(base)
    torch.cuda.synchronize()
    assert torch.equal(got[0], base[2])  # the only key's value
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def _c_abi_step(q, k, v, do, cu, causal, scale):
    """Forward and backward through the C entry points, which take any scale."""
    from scree_amd.kernels.hip import _ffi
    from scree_amd.kernels.hip import attention as A

    lib, (n, heads, dim) = _ffi.lib(), q.shape
    o, dq, dk, dv = (torch.empty_like(t) for t in (q, q, k, v))
    lse = torch.empty((n, heads), device=q.device)
    delta = torch.empty_like(lse)
    ws = A.attention_schedule(cu, n, dim, causal)

    def call(fn, ts, strided):
        strides = _ffi.int64_array(sum((t.stride()[:2] for t in strided), ()))
        _ffi.check(fn(*map(_ffi.ptr, ts), _ffi.ptr(cu), cu.numel() - 1, n, heads, k.shape[1], dim,
                      strides, scale, int(causal), _ffi.DTYPE_F32, _ffi.ptr(ws), ws.numel(),
                      _ffi.stream_of(q)))

    call(lib.scree_attn_fwd_gqa, (q, k, v, o, lse), (q, k, v, o))
    call(lib.scree_attn_bwd_gqa, (do, q, k, v, o, lse, dq, dk, dv, delta), (do, q, k, v, o, dq, dk, dv))
    torch.cuda.synchronize()
    return o, lse, dq, dk, dv


@pytest.mark.parametrize("heads", [4, 84, 216])
@pytest.mark.parametrize("dim", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("causal", [True, False])
def test_fp32_scale_of_zero_or_less(dim, heads, causal):
    """A negative scale is the positive one on -q, and a scale of 0 any scale on
    q = 0 with no gradient to q and k: the same products in the same order, so
    the results are equal bit for bit.  (A mask of -inf on the scores would turn
    into +inf or NaN here.)"""
    lengths = [1, 33, 70, 129]
    say(f"case: fp32 scale <= 0, H={heads} D={dim} causal={causal}")
    _, cu = cu_of(lengths)
    n, scale = sum(lengths), dim ** -0.5
    q, do = (randn((n, heads, dim), torch.float32, 60 + i) for i in range(2))
    k, v = (randn((n, heads // 2, dim), torch.float32, 62 + i) for i in range(2))
    o, lse, dq, dk, dv = _c_abi_step(-q, k, v, do, cu, causal, scale)
    for got, want in zip(_c_abi_step(q, k, v, do, cu, causal, -scale), (o, lse, -dq, dk, dv)):
        assert torch.isfinite(want).all() and torch.equal(got, want)
    o, lse, _, _, dv = _c_abi_step(torch.zeros_like(q), k, v, do, cu, causal, scale)
    zero = torch.zeros_like
    for got, want in zip(_c_abi_step(q, k, v, do, cu, causal, 0.0), (o, lse, zero(q), zero(k), dv)):
        assert torch.isfinite(want).all() and torch.equal(got, want)


@pytest.mark.parametrize("heads", [4, 84, 216])
@pytest.mark.parametrize("dim", [16, 64, 256])
@pytest.mark.parametrize("causal", [True, False])
def test_fp32_scores_keep_every_bit(dim, heads, causal):
    """Whole-number q and k and a scale that is a power of two: the scores are
    exact, so adding 512 to 2,048 (by head_dim) to all of them leaves the output
    as it is, to the rounding of the weights (an ulp of the exponential, and up
    to 24 * 2^-24 in the exponent of one that counts) and of the sums.  Scores
    rounded in units of log2(e) would be off by up to 2^-13 there."""
    lengths = [1, 33, 70, 129]
    say(f"case: fp32 exact scores, H={heads} D={dim} causal={causal}")
    _, cu = cu_of(lengths)
    n, scale = sum(lengths), dim ** -0.5
    q, k = ((2 * randn((n, heads, dim), torch.float32, 80 + i)).round().clamp(-3, 3) for i in range(2))
    v, do = (randn((n, heads, dim), torch.float32, 82 + i) for i in range(2))
    k[..., 0] = 8.0
    outs = []
    for shift in (0.0, 1024.0):
        q[..., 0] = shift
        outs.append(_c_abi_step(q, k, v, do, cu, causal, scale)[0])
    worst = float((outs[1] - outs[0]).abs().max())
    say(f"  largest difference {worst:.2e}")
    assert worst <= 2.0 ** -20 * float(v.abs().max())


@pytest.mark.parametrize("heads", [4, 32])
@pytest.mark.parametrize("dim", [16, 32, 64, 128, 256])
def test_fp32_one_key_has_no_score_gradient(dim, heads):
    """Sequences of one token with a score of 0: the only weight is 1 and the
    output the value, so dP and Delta are the same products, summed in the same
    order in both backward passes, and dQ (with q = 0) and dK (with k = 0) are 0.
    96 sequences, 4 query heads per K/V head: dQ with 4 waves per row tile at 4
    heads and one at 32, dK/dV with 4."""
    n = 96
    say(f"case: fp32 one key, H={heads} D={dim}")
    _, cu = cu_of([1] * n)
    q, do = (randn((n, heads, dim), torch.float32, 90 + i) for i in range(2))
    k, v = (randn((n, heads // 4, dim), torch.float32, 92 + i) for i in range(2))
    o, _, dq, _, _ = _c_abi_step(torch.zeros_like(q), k, v, do, cu, True, dim ** -0.5)
    assert torch.equal(o, v.repeat_interleave(4, dim=1))
    assert not dq.any()
    _, _, _, dk, _ = _c_abi_step(q, torch.zeros_like(k), v, do, cu, True, dim ** -0.5)
    assert not dk.any()


def _fwd64(q, k, v, lengths, causal, scale):
    """Masked softmax attention in fp64 by torch, non-finite scores included."""
    outs, a = [], 0
    for n in lengths:
        qq, kk, vv = (t[a:a + n].double().cpu().transpose(0, 1) for t in (q, k, v))
        a += n
        s = qq @ kk.transpose(1, 2) * scale
        if causal:
            s = s.masked_fill(~torch.ones(n, n, dtype=torch.bool).tril(), float("-inf"))
        outs.append((torch.softmax(s, -1) @ vv).transpose(0, 1))
    return torch.cat(outs).numpy()


@pytest.mark.parametrize("heads", [2, 84, 200])  # 4, 2 and 1 waves per row tile
@pytest.mark.parametrize("dim", [16, 32, 64, 128])
@pytest.mark.parametrize("causal", [True, False])
def test_fp32_non_finite_scores(dim, heads, causal):
    """A first tile of keys with scores of -inf (no weight, and NaN for the rows
    that see nothing else) and a NaN key (NaN for the rows that see it): as in the
    plain formula, and nothing changes in the other sequences, gradients included."""
    import numpy as np

    lengths = [70, 129, 33, 90]
    say(f"case: fp32 non-finite scores, H={heads} D={dim} causal={causal}")
    _, cu = cu_of(lengths)
    n, scale = sum(lengths), dim ** -0.5
    q, k, v, do = (randn((n, heads, dim), torch.float32, 20 + i) for i in range(4))
    q[..., 0] = 1.0
    clean = _c_abi_step(q, k, v, do, cu, causal, scale)
    bad = k.clone()
    bad[70:102, :, 0] = float("-inf")  # the second sequence's first 32 keys
    bad[199 + 40] = float("nan")       # past the third: key 7 of the last sequence
    got = _c_abi_step(q, bad, v, do, cu, causal, scale)
    want = _fwd64(q, bad, v, lengths, causal, scale)
    o = np64(got[0])
    assert np.array_equal(np.isnan(o), np.isnan(want))
    assert np.nanmax(np.abs(o - want)) <= TOL + 2.0 ** -24 * np.nanmax(np.abs(want))
    assert np.isnan(want[70:102]).all() if causal else not np.isnan(want[70:199]).any()
    for a, b in zip(got, clean):
        assert torch.isfinite(b).all()
        assert torch.equal(a[:70], b[:70]) and torch.equal(a[199:232], b[199:232])
    if causal:  # the rows before the NaN key
        assert torch.equal(got[0][232:239], clean[0][232:239])
