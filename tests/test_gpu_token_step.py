"""GPU: the layer's token step as one library call (tsattn_layer_token) against the chain of calls it stands for, and the
few-row product and the small normalisation it is made of at the edges of their tiles."""
import numpy as np
import pytest
import torch

from oracle import pyoracle as orc
from tscale_amd import AttentionContext, KVCache, attention, capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = AttentionContext(0, max_seqs=128, max_heads=16, max_head_dim=128)
    yield c
    c.close()


def int8(g, *shape):
    return (torch.randn(shape, device="cuda", generator=g) * 32).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)


@pytest.mark.parametrize("B,H,d,dim,relu,max_len", [
    (1, 12, 64, 768, 64, 1400),       # splits of the cache; K in three groups per part
    (3, 2, 128, 256, 128, 40), (16, 3, 64, 384, 128, 90), (17, 3, 64, 384, 64, 90), (33, 2, 128, 128, 128, 20), (128, 1, 64, 128, 64, 12)])
def test_token_step_equals_the_chain(ctx, monkeypatch, B, H, d, dim, relu, max_len):
    """Three layers (window 1, short window with a slope, all keys), two tokens: the cache bytes, scales and lengths of both
    are equal, states and outputs equal up to int8 roundings of k * value that the order of the attention's sums flips."""
    g = torch.Generator(device="cuda").manual_seed(B * 1000 + d)
    qsum = H * d
    layers = [{"proj": int8(g, 4 * qsum, dim), "combiner": int8(g, dim, 4 * qsum), "expand": int8(g, H * relu, dim), "contract": int8(g, dim, H * relu),
               "qv_scale": 0.02, "combiner_scale": 0.03, "contract_scale": 0.025, "width": w, "slope": sl} for w, sl in ((1, 0.0), (5, 0.5), (max_len, 0.0))]
    k0, v0 = int8(g, 3, B, H, max_len, d), int8(g, 3, B, H, max_len, d)
    lens = torch.randint(0, max_len + 1, (B,), device="cuda", generator=g, dtype=torch.int32)
    lens[0] = max_len - 2                                            # some are full before the second token, some empty
    state0 = torch.randn((B, dim), device="cuda", generator=g)
    rope = ctx.fill_rope_table(d, max_len + 8)

    def steps(chain):
        with monkeypatch.context() as m:
            if chain:
                m.setattr(attention, "_layer_token", lambda *a: None)
            caches = []
            for i in range(3):
                c = KVCache(ctx, capi.I8, B, H, max_len, d)
                c.k.copy_(k0[i]); c.v.copy_(v0[i]); c.k_scale.fill_(0.01); c.v_scale.fill_(attention.VEC_SCALE); c.cache_len.copy_(lens)
                caches.append(c)
            state, keep, outs = state0.clone(), {}, []
            for step in range(2):
                pending = None
                for layer, c in zip(layers, caches):
                    val, pending = attention.add_lookup_product(ctx, layer, c, lens + step, rope, state, scratch=keep, pending=pending, defer=True)
                    outs.append(val.clone())
                outs.append(attention.flush_state(ctx, pending, state))
            torch.cuda.synchronize()
            return caches, state, outs

    got_c, got_s, got_o = steps(False)
    want_c, want_s, want_o = steps(True)
    for c, w in zip(got_c, want_c):
        assert torch.equal(c.cache_len, w.cache_len) and torch.equal(c.v_scale, w.v_scale)
        assert (c.k != w.k).float().mean() < 1e-3 and (c.v != w.v).float().mean() < 1e-3
    rms = want_s.square().mean().sqrt()
    assert (got_s - want_s).abs().max() / rms < 2e-2
    assert (got_o[0] - want_o[0]).abs().max() < 2e-5


@pytest.mark.parametrize("m", [1, 15, 16, 17, 32, 33, 64, 65, 128])
@pytest.mark.parametrize("n,k", [(1, 64), (15, 192), (17, 8192), (130, 576), (33001, 128)])
def test_few_row_product_at_tile_edges(ctx, m, n, k):
    rng = np.random.default_rng(m * 31 + n + k)
    a = rng.integers(-127, 128, (m, k)).astype(np.int8)
    w = rng.integers(-127, 128, (n, k)).astype(np.int8)
    want = orc.matmul_i8(a, w)
    da, dw = torch.from_numpy(a.view(np.uint8)).cuda(), torch.from_numpy(w.view(np.uint8)).cuda()
    planes = ctx.matmul_i8(da, dw, mode=capi.MM_I32_PLANES)
    f = ctx.matmul_i8(da, dw, mode=capi.MM_F32, scale=0.5)
    torch.cuda.synchronize()
    assert np.array_equal(planes.sum(dim=0, dtype=torch.int32).cpu().numpy(), want)
    assert np.array_equal(f.cpu().numpy(), want.astype(np.float32) * np.float32(0.5))


@pytest.mark.parametrize("rows,heads,d,dtype", [(1, 1, 64, capi.I8), (5, 7, 64, capi.E4M3), (33, 3, 128, capi.I8), (64, 64, 128, capi.I8), (4097, 1, 64, capi.I8),
                                                (3, 5, 384, capi.I8), (2, 3, 512, capi.I8)])
def test_normalisation_of_few_pairs(ctx, rows, heads, d, dtype):
    """Several planes, a group of zeros, rows that do not fill a wave; 4096 pairs are the last of the small launches."""
    g = torch.Generator(device="cuda").manual_seed(rows * 7 + d)
    planes = torch.randint(-30000, 30000, (5, rows, heads * d), device="cuda", generator=g, dtype=torch.int32)
    planes[:, 0, :d] = 0
    kw, okw = {}, {}
    if d <= 128:
        pos, rope = np.arange(rows, dtype=np.int32) % 50, orc.fill_rope(d, 50)
        okw = dict(pos=pos, rope=rope)
        kw = dict(pos=torch.from_numpy(pos).cuda(), rope=torch.from_numpy(rope).cuda())
    got, scale = ctx.rope_normalize_rows(planes, heads, dtype, **kw)
    x = planes.sum(dim=0, dtype=torch.int32).cpu().numpy().astype(np.float32)
    want, want_scale = orc.rope_normalize_rows(dtype, x, heads, **okw)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), want.view(np.uint8)) and np.array_equal(scale.cpu().numpy(), want_scale)
