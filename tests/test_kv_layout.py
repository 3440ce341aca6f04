"""K/V layouts of the layer-call (``ops.evict``, ``EvictPlan``,
``dropkv_evict_strided``): rows that lie apart are read in place, everything
the kernels cannot address is copied first, and the result is that of the
contiguous copy, bit for bit.

The CPU tests walk the routing rule over the forms it can meet (no kernel
runs); the GPU test compares each form with its contiguous copy."""

import ctypes

import pytest
import torch

from dropkv_amd import _lib, ops

# form -> builder of K or V [B, H, L, D] from a seeded generator
B, H, L = 2, 4, 300


def _proj(g, D, dtype, width=None, at=0, rows=L):
    """[B, rows, width] projection; heads at columns at .. at + H*D."""
    width = H * D if width is None else width
    x = torch.randn(B, rows, width, generator=g).to(dtype)
    return x[:, :, at:at + H * D].view(B, rows, H, D) if width != H * D else x.view(B, rows, H, D)


FORMS = {
    "per head": lambda g, D, t: torch.randn(B, H, L, D, generator=g).to(t),
    "projection": lambda g, D, t: _proj(g, D, t).transpose(1, 2),
    "fused projection": lambda g, D, t: torch.randn(B, L, 3 * H, D, generator=g).to(t)[:, :, H:2 * H].transpose(1, 2),
    "buffer rows": lambda g, D, t: torch.randn(B, H, L + 37, D, generator=g).to(t)[:, :, 5:5 + L],
    "padded rows": lambda g, D, t: torch.randn(B, H, L, D + 16, generator=g).to(t)[..., :D],
    "one head, expanded": lambda g, D, t: torch.randn(B, 1, L, D, generator=g).to(t).expand(B, H, L, D),
    "one row, expanded": lambda g, D, t: torch.randn(B, H, 1, D, generator=g).to(t).expand(B, H, L, D),
    "columns apart": lambda g, D, t: torch.randn(B, H, L, 2 * D, generator=g).to(t)[..., ::2],
    "transposed rows": lambda g, D, t: torch.randn(B, H, D, L, generator=g).to(t).transpose(2, 3),
    "odd row stride": lambda g, D, t: torch.randn(B, H, L, D + 1, generator=g).to(t)[..., :D],
}
IN_PLACE = ("per head", "projection", "fused projection", "buffer rows", "padded rows", "one head, expanded")


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (80, torch.float16), (33, torch.bfloat16),
                                     (64, torch.float32)])
def test_route(form, D, dtype):
    """Read in place only with whole 16-byte rows that do not overlap; the
    strides reproduce the tensor from its storage either way."""
    t = FORMS[form](torch.Generator().manual_seed(1), D, dtype)
    u, (sb, sh, sl) = ops._evict_kv(t)
    want = form in IN_PLACE and (t.is_contiguous() or D % 8 == 0)
    assert (u.data_ptr() == t.data_ptr()) == want
    assert torch.equal(torch.as_strided(u, t.shape, (sb, sh, sl, 1), u.storage_offset()), t)
    assert u.data_ptr() % 16 == 0 and sl >= D
    if not t.is_contiguous():
        assert u.is_contiguous() or (sb | sh | sl | D) * t.element_size() % 16 == 0


def test_route_misaligned_and_far_rows():
    flat = torch.randn(B * L * H * 64 + 8).to(torch.bfloat16)
    t = flat[1:1 + B * L * H * 64].view(B, L, H, 64).transpose(1, 2)  # 2 bytes past a 16-byte unit
    u, strides = ops._evict_kv(t)
    assert u.is_contiguous() and torch.equal(u, t) and strides == (H * L * 64, L * 64, 64)
    d = flat[1:1 + B * H * L * 64].view(B, H, L, 64)
    u, _ = ops._evict_kv(d)
    assert u.data_ptr() % 16 == 0 and torch.equal(u, d)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_route_far_rows(dtype):
    """Rows in place up to the distance that 32-bit offsets reach (2 GiB over the
    head's rows and 1024 more), copied from one 16-byte unit beyond (views with
    no memory behind them)."""
    es, rows = dtype.itemsize, 4096
    limit = (1 << 31) // es // (rows + 1024) // (16 // es) * (16 // es)
    for sl, in_place in ((limit, True), (limit + 16 // es, False), (1 << 20, False)):
        far = torch.empty(1, 1, 1, 64, dtype=dtype, device="meta").as_strided((1, 2, rows, 64), (128, 64, sl, 1))
        u, strides = ops._evict_kv(far)
        assert strides == ((128, 64, sl) if in_place else (2 * rows * 64, rows * 64, 64))
        assert u.stride() == (far.stride() if in_place else (2 * rows * 64, rows * 64, 64, 1))


@pytest.mark.parametrize("over,msg", [
    (dict(k_sl=63), "16-byte"),
    (dict(v_sh=-64), "16-byte"),
    (dict(k_sl=0), "overlap"),
    (dict(v_sl=32), "overlap"),
    (dict(k_sl=1 << 26), "too far"),
    (dict(D=33, k_sl=40, v_sl=40), "whole 16-byte"),
])
def test_c_entry_refuses_what_the_kernels_cannot_read(over, msg):
    lib = _lib.load()
    fake = ctypes.c_void_p(1 << 20)  # never dereferenced: the checks fail first
    a = dict(D=64, k_sb=8192, k_sh=64, k_sl=512, v_sb=8192, v_sh=64, v_sl=512)
    a.update(over)
    rc = lib.dropkv_evict_strided(fake, 0, 0, 0, 1, fake, a["k_sb"], a["k_sh"], a["k_sl"], fake, a["v_sb"], a["v_sh"],
                                  a["v_sl"], 1, 1, 8, 8, 64, 100, a["D"], 8, 1e-6, 1, 0, 0, 11, 8, 10, None, fake,
                                  fake, fake, 10, fake, 1 << 30, None)
    assert rc == 2 and msg in lib.dropkv_last_error().decode()


@pytest.mark.gpu
@pytest.mark.parametrize("D,dtype,Hq,W", [
    (64, torch.bfloat16, 8, 8),     # one row-chunk
    (128, torch.float16, 16, 16),   # two
    (128, torch.bfloat16, 32, 16),  # four: the wide kernels
    (32, torch.bfloat16, 4, 8),
    (80, torch.bfloat16, 8, 8),     # the kernels for other head dimensions
    (64, torch.float32, 8, 8),
])
def test_layouts_equal_their_contiguous_copy(gpu, D, dtype, Hq, W):
    q = torch.randn(B, Hq, 64, D, generator=torch.Generator().manual_seed(0)).to(dtype).to(gpu)
    names = list(FORMS)
    for i, kf in enumerate(names):
        vf = names[(i + 1) % len(names)] if i % 2 else kf  # K and V alike, and not
        g = torch.Generator().manual_seed(i)
        src = [FORMS[f](g, D, dtype) for f in (kf, vf)]
        # the same views on the GPU: storage copied whole, strides kept
        k, v = (torch.as_strided(torch.as_strided(t, (t.untyped_storage().nbytes() // t.element_size(),), (1,), 0)
                                 .to(gpu), t.shape, t.stride(), t.storage_offset()) for t in src)
        got = ops.evict(q, k, v, W, 11, 60)
        ref = ops.evict(q, k.contiguous(), v.contiguous(), W, 11, 60)
        plan = ops.EvictPlan(q, k, W, 11, 60)(q, k, v)
        for x, y, z in zip(got, ref, plan):
            assert torch.equal(x, y) and torch.equal(z, y), (kf, vf)
