"""GPU: the int8 products of a few hundred rows (64- and 128-row tiles) at the edges of their tiles, plain and with the producer as
their last step."""
import numpy as np
import pytest
import torch

from oracle import pyoracle as orc
from tscale_amd import AttentionContext, capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = AttentionContext(0, max_seqs=1, max_heads=1)
    yield c
    c.close()


dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("m,n,k", [(129, 1, 64), (191, 130, 192), (193, 127, 128), (257, 129, 1088), (700, 4097, 64), (1100, 4100, 320), (2050, 2000, 64)])
def test_products_at_tile_edges(ctx, m, n, k):
    """Rows, columns and K that do not fill a tile or a stage; all result forms, nothing outside the block written."""
    rng = np.random.default_rng(m + n + k)
    a, w = (rng.integers(-127, 128, s).astype(np.int8) for s in ((m, k), (n, k)))
    want = orc.matmul_i8(a, w)
    da, dw = dev(a.view(np.uint8)), dev(w.view(np.uint8))
    buf = torch.full((m + 1, n + 3), -7, dtype=torch.int32, device="cuda")
    ctx.matmul_i8(da, dw, out=buf[:m, :n])
    f = ctx.matmul_i8(da, dw, mode=capi.MM_F32, scale=0.25)
    state = rng.standard_normal((m, n)).astype(np.float32)
    added = ctx.matmul_i8(da, dw, mode=capi.MM_ADD_SCALED, scale=0.003, out=dev(state))
    torch.cuda.synchronize()
    assert np.array_equal(buf[:m, :n].cpu().numpy(), want) and (buf[m:] == -7).all() and (buf[:, n:] == -7).all()
    assert np.array_equal(f.cpu().numpy(), want.astype(np.float32) * np.float32(0.25))
    assert np.array_equal(added.cpu().numpy(), orc.matmul_i8(a, w, mode=2, scale=0.003, out=state))


@pytest.mark.parametrize("m,n,k", [(1, 313001, 64), (16, 104170, 192), (17, 31300, 640), (31, 19999, 1088), (32, 12003, 2048), (5, 6600, 3072)])
def test_products_of_a_large_matrix_under_few_rows(ctx, m, n, k):
    """Blocks of rows cut by the waves' shares, a last block that is not full, K that ends in half a stage; all result forms."""
    test_products_at_tile_edges(ctx, m, n, k)


@pytest.mark.parametrize("m,heads,d,k", [(40, 2, 128, 64), (129, 3, 64, 192), (190, 5, 128, 320), (1030, 33, 64, 128), (1300, 17, 128, 64)])
@pytest.mark.parametrize("variant", ["rope", "resid", "relu"])
def test_products_with_the_producer_at_tile_edges(ctx, m, heads, d, k, variant):
    """Bytes, scales and the updated state are those of the product followed by the producer's own launch."""
    rng = np.random.default_rng(m + heads + k)
    n = heads * d
    a, w = (dev(rng.integers(-127, 128, s).astype(np.int8).view(np.uint8)) for s in ((m, k), (n, k)))
    a[3] = 0                                       # a row of zeros: scale and bytes 0
    state = rng.standard_normal((m, n)).astype(np.float32)
    pos = dev(rng.integers(-1, 70, m).astype(np.int32))
    outs = []
    for fused in (True, False):
        kw = {"rope": dict(pos=pos, rope=dev(orc.fill_rope(d, 64)), scale_mult=0.4,
                           rope_heads=max(1, heads - 1), scale_heads=(heads // 2, 1)),
              "resid": dict(resid=dev(state), resid_scale=0.01), "relu": dict(relu=True, row_major_scale=True)}[variant]
        if fused:
            q, s = ctx.matmul_normalize(a, w, heads, capi.I8, **kw)
        else:
            q, s = ctx.rope_normalize_rows(ctx.matmul_i8(a, w), heads, capi.I8, **kw)
        outs.append((q, s, kw.get("resid")))
    torch.cuda.synchronize()
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    if variant == "resid":
        assert torch.equal(outs[0][2], outs[1][2])


@pytest.mark.parametrize("m,n,k,split", [(32, 2048, 8192, True), (33, 513, 6144, True), (64, 768, 3072, True), (128, 132, 4096, True),
                                         (8, 256, 1024, False), (32, 2048, 2048, False), (129, 256, 4096, False)])
@pytest.mark.parametrize("mode", [capi.MM_I32, capi.MM_F32, capi.MM_ADD_SCALED])
def test_product_through_a_lent_workspace(ctx, m, n, k, split, mode):
    """Long products of few rows go through the workspace in parts, short ones and many rows do not touch it; the result is the
    same with and without."""
    g = torch.Generator(device="cuda").manual_seed(m * n)
    a = torch.randint(-127, 128, (m, k), device="cuda", generator=g, dtype=torch.int32).to(torch.int8).view(torch.uint8)
    w = torch.randint(-127, 128, (n, k), device="cuda", generator=g, dtype=torch.int32).to(torch.int8).view(torch.uint8)
    room = torch.full((16 * m * n,), 0x7fedcba9, dtype=torch.int32, device="cuda")
    state = torch.randn((m, n), device="cuda", generator=g) if mode == capi.MM_ADD_SCALED else None
    outs = [ctx.matmul_i8(a, w, mode=mode, scale=1e-3, out=None if state is None else state.clone(), workspace=ws) for ws in (None, room)]
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    assert bool((room != 0x7fedcba9).any()) == split
