"""The matrix-core kernels for fp32 inputs and for bf16 / fp16 head dimensions
other than 32, 64 and 128 (up to 256, rows of whole 16-byte units): at the
edges of their tiles (16 and 32 query rows, 16- and 32-column chunks, 64-column
groups of y, 256-key steps, several splits), with a key that takes nearly all
of a row's attention and with values that share a large mean, where the
expanded distance cancels and is taken directly, against the score evaluated in
float64.

Bars: without p rounding every score within rtol 1e-4 of the float64 one (the
logits carry ~4 * 2^-24 of sum_d |q_d k_d| / sqrt(D) <= ~20 here, which enters
the score twice: ~1e-5, and a mean of 100 in the values 100 * 2^-24 per
element of a distance of ~1: ~1e-5), with the other fp32 tests' absolute floor.
At a key of p = 1 - delta the distance is (1 - p) |v|: a few 2^-24 / delta."""

import pytest
import torch

from oracle import dropkv_ref as R

pytestmark = pytest.mark.gpu


def _inputs(dtype, B, Hq, Hkv, D, Lq, Lk, seed, v_mean=0.0):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, Hq, Lq, D, generator=g).to(dtype)
    k = torch.randn(B, Hkv, Lk, D, generator=g).to(dtype)
    v = (torch.randn(B, Hkv, Lk, D, generator=g) + v_mean).to(dtype)
    return q, k, v


def _check(got, ref, rtol):
    got, ref = got.double().cpu(), ref.double()
    atol = 1e-6 * ref.abs().amax(dim=-1, keepdim=True).clamp_min(1e-30)
    err = (got - ref).abs() - (atol + rtol * ref.abs())
    assert torch.isfinite(got).all() and (err <= 0).all(), f"worst excess {err.max().item():.3e}"


@pytest.mark.parametrize("dtype,Hq,Hkv,D,Lk,W", [
    (torch.float32, 2, 2, 64, 256, 16),     # 16 rows: one row block; one step
    (torch.float32, 2, 2, 64, 257, 17),     # 17 rows: two row blocks; a second split of one key
    (torch.float32, 8, 2, 32, 255, 8),      # 32 rows
    (torch.float32, 7, 1, 128, 1000, 5),    # 35 rows: two chunks, the second of three rows
    (torch.float32, 4, 2, 36, 777, 3),      # 36 columns: a partial chunk, one group of y
    (torch.float32, 2, 1, 256, 700, 1),     # window 1, four groups of y
    (torch.float32, 4, 4, 4, 64, 64),       # four columns; every key in the window
    (torch.bfloat16, 4, 2, 8, 300, 8),      # eight columns
    (torch.float16, 16, 2, 72, 513, 9),     # 72 rows, 72 columns
    (torch.bfloat16, 2, 2, 136, 511, 16),   # three groups of y, a partial chunk
    (torch.float16, 8, 4, 200, 1025, 8),
    (torch.bfloat16, 32, 2, 256, 2100, 16),  # 256 rows: eight chunks
])
@pytest.mark.parametrize("splits", [0, 1])
def test_scores_vs_float64(gpu, dtype, Hq, Hkv, D, Lk, W, splits):
    from dropkv_amd import ops
    q, k, v = _inputs(dtype, 2, Hq, Hkv, D, W + 3 if Lk > W + 3 else W, Lk, seed=D + Lk)
    ref = R.dropkv_scores_fp64(q, k, v, W)
    got = ops.scores(q.to(gpu), k.to(gpu), v.to(gpu), W, p_round=False, splits=splits)
    _check(got, ref, 1e-4)
    again = ops.scores(q.to(gpu), k.to(gpu), v.to(gpu), W, p_round=False, splits=splits)
    assert torch.equal(got, again)


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 96), (torch.float16, 256), (torch.float32, 64)])
def test_rounded_p(gpu, dtype, D):
    """p rounded to the input type (the identity for fp32): scores off by more
    than 1e-4 only where a p rounds the other way, on few keys and by at most
    the rounding step of p (2^-8 / 2^-11) twice over, W g rows sharing it."""
    from dropkv_amd import ops
    q, k, v = _inputs(dtype, 1, 8, 2, D, 8, 3000, seed=D)
    ref = R.dropkv_scores_fp64(q, k, v, 8, p_round=dtype)
    got = ops.scores(q.to(gpu), k.to(gpu), v.to(gpu), 8, p_round=True).double().cpu()
    rel = (got - ref).abs() / ref.abs().clamp_min(1e-30)
    assert rel.max() < 2e-2 and (rel > 1e-4).double().mean() < 2e-2


@pytest.mark.parametrize("dtype,D", [(torch.float32, 128), (torch.bfloat16, 192)])
def test_dominant_key_and_common_mean(gpu, dtype, D):
    from dropkv_amd import ops
    W, Lk = 8, 1200
    q, k, v = _inputs(dtype, 1, 4, 2, D, W, Lk, seed=3)
    # one key along the queries' common direction: p within 1e-4 .. 1e-1 of 1
    q = (q * 0.05 + 1.0).to(dtype)
    k[:, 0, 700] = 1.3 * (torch.tensor(float(Lk)).log() / D ** 0.5).to(dtype) + 0.4
    ref = R.dropkv_scores_fp64(q, k, v, W)
    got = ops.scores(q.to(gpu), k.to(gpu), v.to(gpu), W, p_round=False)
    p = torch.softmax((q[:, :2].double() @ k[:, :1].double().transpose(-1, -2)) / D ** 0.5, -1)
    assert p.max() > 0.9  # the case is what it says
    _check(got, ref, 1e-3)
    q, k, v = _inputs(dtype, 1, 4, 2, D, W, Lk, seed=4, v_mean=100.0)
    ref = R.dropkv_scores_fp64(q, k, v, W)
    _check(ops.scores(q.to(gpu), k.to(gpu), v.to(gpu), W, p_round=False), ref, 1e-4)
