"""GPU parity of the fp32 matrix-instruction attention at the sizes where its
forms can go wrong: sequence lengths around the 32-row tile and the 128-row
item, with 4, 2 and 1 waves sharing a row tile (the launchers choose by the
number of row tiles: 4 below 2,048, or 1,024 from head_dim 64 up; 2 below
5,120, or 3,072 at head_dim 128), in both mask modes, with and without grouped
K/V heads.  Bounds as in ``test_gpu_attention_fp32``.
"""

import pytest
import torch

from parity import cu_of, randn, say
from test_gpu_attention_fp32 import run_fp32_case

pytestmark = pytest.mark.gpu

# 19 row blocks per head (ceil(868 / 128) + 12), 76 row tiles
TILE_LENGTHS = [1, 31, 32, 33, 64, 65, 96, 127, 128, 129, 160, 2]


@pytest.mark.parametrize("heads", [8, 32, 84])  # 608, 2,432 and 6,384 row tiles: 4, 2, 1 waves
@pytest.mark.parametrize("dim", [16, 32, 64, 128])
@pytest.mark.parametrize("causal", [True, False])
def test_fp32_waves_per_row_tile(dim, heads, causal):
    # grouped K/V heads below 64 columns; without them the dK/dV pass takes the same form
    run_fp32_case(TILE_LENGTHS, heads, dim, causal, seed=900 + dim,
                  kv_heads=heads // 2 if dim < 64 else heads)


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


@pytest.mark.parametrize("heads", [4, 84])
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


@pytest.mark.parametrize("heads", [4, 84])
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
