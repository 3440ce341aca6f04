"""Layer-calls of rows of up to 512 keys, whose selection one pass-2 workgroup
does alone (solo_tail): bit for bit the scores, kept indices and rows of the
separate selection kernels (``set_tail_select(False)``), and the oracle's rule on
the same scores.  Sizes at the edges of the tiles and of the rule, windows that
cover the row, rows kept whole, a pooling window wider than the row, and ties:
V = 0 leaves every unprotected key a candidate (more than are ranked at once)."""

import pytest
import torch

from oracle import dropkv_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Lk", [1, 2, 31, 33, 255, 256, 257, 511, 512, 513])
@pytest.mark.parametrize("D,dtype,g,W,ks", [(64, torch.bfloat16, 4, 8, 11), (128, torch.float16, 8, 8, 5),
                                            (32, torch.bfloat16, 1, 1, 129)])
@pytest.mark.parametrize("zero_v", [False, True])
def test_solo_rows(gpu, Lk, D, dtype, g, W, ks, zero_v):
    from dropkv_amd import ops
    W = min(W, Lk)
    gen = torch.Generator().manual_seed(Lk + D)
    q = torch.randn(2, 3 * g, Lk, D, generator=gen).to(dtype).to(gpu)
    k, v = (torch.randn(2, 3, Lk, D, generator=gen).to(dtype).to(gpu) for _ in range(2))
    if zero_v:
        v.zero_()
    for keep in sorted({max(1, W), max(1, Lk // 10), max(1, Lk // 2), Lk}):
        for pw in {0, W}:
            out = []
            for tail in (True, False):
                ops.set_tail_select(tail)
                try:
                    plan = ops.EvictPlan(q, k, W, ks, keep, protect_window=pw, keep_scores=True)
                    out.append([x.clone() for x in plan(q, k, v)] + [plan.scores.clone()])
                finally:
                    ops.set_tail_select(True)
            for a, b in zip(*out):
                assert torch.equal(a, b), (keep, pw)
            idx, ko, vo, scores = (x.cpu() for x in out[0])
            assert torch.equal(idx, R.topk_sorted(R.pool_protect(scores.clone(), ks, pw), keep)), (keep, pw)
            rk, rv = R.gather_compressed(k.cpu(), v.cpu(), idx)
            assert torch.equal(ko, rk) and torch.equal(vo, rv)


@pytest.mark.parametrize("B,Hkv,splits", [(1, 2, 1), (33, 4, 0)])  # one split asked for; 132 rows, one workgroup each
@pytest.mark.parametrize("Lk", [513, 2047, 2048, 2049, 4095, 4096, 4097])
@pytest.mark.parametrize("zero_v", [False, True])
def test_long_rows_in_one_split(gpu, B, Hkv, splits, Lk, zero_v):
    """Rows of up to 4096 keys held by one workgroup are selected alone too:
    several rounds of the ordered emit (2048 keys each) and more candidates than
    are ranked at once.  Bit for bit the separate kernels, and the oracle's rule."""
    from dropkv_amd import ops
    W, ks, D = 8, 63, 64
    gen = torch.Generator().manual_seed(Lk)
    q = torch.randn(B, 2 * Hkv, W, D, generator=gen).bfloat16().to(gpu)
    k, v = (torch.randn(B, Hkv, Lk, D, generator=gen).bfloat16().to(gpu) for _ in range(2))
    if zero_v:
        v[:, :, Lk // 3:] = 0
    for keep in (W, Lk // 10, Lk // 2 + 1, Lk - 1, Lk):
        out = []
        for tail in (True, False):
            ops.set_tail_select(tail)
            try:
                plan = ops.EvictPlan(q, k, W, ks, keep, keep_scores=True, splits=splits)
                out.append([x.clone() for x in plan(q, k, v)] + [plan.scores.clone()])
            finally:
                ops.set_tail_select(True)
        for a, b in zip(*out):
            assert torch.equal(a, b), keep
        idx, ko, vo, scores = (x.cpu() for x in out[0])
        assert torch.equal(idx, R.topk_sorted(R.pool_protect(scores.clone(), ks, W), keep)), keep
        rk, rv = R.gather_compressed(k.cpu(), v.cpu(), idx)
        assert torch.equal(ko, rk) and torch.equal(vo, rv)
