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
    (torch.float32, 2, 2, 64, 257, 17),     # 17 rows: two row blocks; a second step of one key
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


def test_many_splits_fp32(gpu):
    """More than 32 key splits: the merge's second batch of partials."""
    from dropkv_amd import ops
    q, k, v = _inputs(torch.float32, 1, 2, 1, 64, 8, 17500, seed=11)
    ref = R.dropkv_scores_fp64(q, k, v, 8)
    for p_round in (False, True):  # (rounding to fp32 is the identity)
        _check(ops.scores(q.to(gpu), k.to(gpu), v.to(gpu), 8, p_round=p_round), ref, 1e-4)


def test_many_splits_rounded_p(gpu):
    """70 key splits: each workgroup combines the statistics of more splits than
    it reads up front.  Against the float64 score with p rounded: off by more
    than 1e-4 only where a p rounds the other way (as test_rounded_p)."""
    from dropkv_amd import ops
    q, k, v = _inputs(torch.bfloat16, 1, 4, 1, 96, 8, 20000, seed=12)
    got = ops.scores(q.to(gpu), k.to(gpu), v.to(gpu), 8, p_round=False, splits=78)
    _check(got, R.dropkv_scores_fp64(q, k, v, 8), 1e-4)
    ref = R.dropkv_scores_fp64(q, k, v, 8, p_round=torch.bfloat16)
    got = ops.scores(q.to(gpu), k.to(gpu), v.to(gpu), 8, p_round=True, splits=78).double().cpu()
    rel = (got - ref).abs() / ref.abs().clamp_min(1e-30)
    assert rel.max() < 2e-2 and (rel > 1e-4).double().mean() < 2e-2


@pytest.mark.parametrize("Lk", [4200, 4097])
def test_several_tiles_a_wave_and_row_groups(gpu, Lk):
    """More than 1024 workgroups of 64 keys: a wave takes several 16-key tiles,
    and with 72 rows of 256 columns the rows are staged in groups, each key's
    sum carried from one to the next."""
    from dropkv_amd import ops
    q, k, v = _inputs(torch.bfloat16, 1, 48, 16, 256, 24, Lk, seed=13)
    args = q.to(gpu), k.to(gpu), v.to(gpu), 24
    _check(ops.scores(*args, p_round=False), R.dropkv_scores_fp64(q, k, v, 24), 1e-4)
    # p and y rounded (y's operands in 16 bits: groups of 64 rows), as the other
    # tests of that path
    got, ref = ops.scores(*args, y_round=True).cpu(), R.fallback_scores(q, k, v, 24)
    torch.testing.assert_close(got, ref, rtol=2e-2, atol=1e-3)
    rel = (got.double() - ref.double()).abs() / ref.double().abs().clamp_min(1e-30)
    assert (rel > 1e-3).double().mean().item() < 1e-2


@pytest.mark.parametrize("dtype,D", [(torch.float32, 64), (torch.bfloat16, 96), (torch.float16, 256)])
@pytest.mark.parametrize("p_round", [False, True])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("key", [5, 700 - 8, 699])
def test_value_that_is_not_finite(gpu, dtype, D, p_round, value, key):
    """The last query row sees every key, so an infinite or NaN value in any row
    of V leaves no finite score in its head, whichever of the other rows see it
    (0 * inf is NaN in p @ V, as in torch); other heads are not touched."""
    from dropkv_amd import ops
    q, k, v = _inputs(dtype, 1, 6, 3, D, 8, 700, seed=14)
    clean = ops.scores(q.to(gpu), k.to(gpu), v.to(gpu), 8, p_round=p_round).cpu()
    v[0, 1, key, 3] = value
    got = ops.scores(q.to(gpu), k.to(gpu), v.to(gpu), 8, p_round=p_round).cpu()
    ref = R.dropkv_scores_reference(q, k, v, 8, match_pytorch_precision=p_round)
    assert not torch.isfinite(ref[0, 1]).any() and not torch.isfinite(got[0, 1]).any()
    assert torch.equal(got[:, ::2], clean[:, ::2]) and torch.isfinite(clean).all()


@pytest.mark.parametrize("dtype,D", [(torch.float32, 64), (torch.bfloat16, 96)])
@pytest.mark.parametrize("lo,hi", [(0, 1), (0, 256), (250, 700), (0, 1192), (1193, 1199)])
def test_keys_of_minus_infinity(gpu, dtype, D, lo, hi):
    """Keys whose logits are -inf have p = 0 and a score of 0; whole steps and
    splits of them leave the other keys' scores alone."""
    from dropkv_amd import ops
    q, k, v = _inputs(dtype, 1, 4, 2, D, 8, 1200, seed=15)
    q[..., 0] = 1.0
    k[:, :, lo:hi, 0] = float("-inf")
    ref = R.dropkv_scores_fp64(q, k, v, 8)
    assert torch.isfinite(ref).all() and (ref[:, :, lo:hi] == 0).all()
    got = ops.scores(q.to(gpu), k.to(gpu), v.to(gpu), 8, p_round=False)
    # (few keys left: p up to 1 - delta, whose score is off by 2^-24 / delta)
    _check(got, ref, 1e-3)
    assert (got[:, :, lo:hi] == 0).all()
