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
    (1, 12, 64, 768, 64, 1400),       # K in three groups per part
    (1, 12, 64, 768, 64, 4000),       # splits of the cache
    (32, 16, 128, 2048, 128, 70),     # normalisations in launches of their own
    # sixteen waves with the front: one step of two rows per lane group, several steps, several splits (test_decode_steps.cpp holds the list)
    (3, 2, 64, 128, 64, 200), (3, 2, 128, 256, 128, 100), (3, 2, 64, 128, 64, 700), (3, 2, 128, 256, 128, 400), (13, 12, 64, 768, 64, 1025),
    (3, 2, 64, 128, 64, 4500), (3, 2, 128, 256, 128, 2300),
    (3, 2, 128, 256, 128, 40), (16, 3, 64, 384, 128, 90), (17, 3, 64, 384, 64, 90), (33, 2, 128, 128, 128, 20), (128, 1, 64, 128, 64, 12)])
def test_token_step_equals_the_chain(ctx, monkeypatch, B, H, d, dim, relu, max_len):
    """Three layers (window 1, short window with a slope, all keys), two tokens: after every layer the caches (bytes, scales,
    lengths), the attention's output, the product left for the next layer and the state are the chain's, bit for bit: the
    launches make the same float operations in the same order."""
    g = torch.Generator(device="cuda").manual_seed(B * 1000 + d)
    qsum = H * d
    layers = [{"proj": int8(g, 4 * qsum, dim), "combiner": int8(g, dim, 4 * qsum), "expand": int8(g, H * relu, dim), "contract": int8(g, dim, H * relu),
               "qv_scale": 0.02, "combiner_scale": 0.03, "contract_scale": 0.025, "width": w, "slope": sl} for w, sl in ((1, 0.0), (5, 0.5), (max_len, 0.0))]
    k0, v0 = int8(g, 3, B, H, max_len, d), int8(g, 3, B, H, max_len, d)
    lens = torch.randint(0, max_len + 1, (B,), device="cuda", generator=g, dtype=torch.int32)
    lens[0] = max_len - 2                                            # some are full before the second token, some empty
    state0 = torch.randn((B, dim), device="cuda", generator=g)
    rope = ctx.fill_rope_table(d, max_len + 8)

    fused = []
    layer_token = attention._layer_token

    def steps(chain):
        with monkeypatch.context() as m:
            m.setattr(attention, "_layer_token", (lambda *a: None) if chain else (lambda *a: fused.append(layer_token(*a)) or fused[-1]))
            caches = []
            for i in range(3):
                c = KVCache(ctx, capi.I8, B, H, max_len, d)
                c.k.copy_(k0[i]); c.v.copy_(v0[i]); c.k_scale.fill_(0.01); c.v_scale.fill_(attention.VEC_SCALE); c.cache_len.copy_(lens)
                caches.append(c)
            state, keep, seen = state0.clone(), {}, []
            for step in range(2):
                pending = None
                for i, (layer, c) in enumerate(zip(layers, caches)):
                    val, pending = attention.add_lookup_product(ctx, layer, c, lens + step, rope, state, scratch=keep, pending=pending, defer=True)
                    now = {"k": c.k, "v": c.v, "k_scale": c.k_scale, "v_scale": c.v_scale, "cache_len": c.cache_len, "output": val,
                           "product": pending[0].sum(dim=0, dtype=torch.int32), "state": state}
                    seen += [((step, i, name), x.clone()) for name, x in now.items()]
                    assert pending[1] == attention._product_scale(layer["contract_scale"], H * relu)
                seen += [((step, "norm"), attention.flush_state(ctx, pending, state).clone()), ((step, "state"), state.clone())]
            torch.cuda.synchronize()
            return seen

    got, want = steps(False), steps(True)
    assert len(fused) == 6 and all(f is not None for f in fused)
    for (what, x), (_, y) in zip(got, want):
        assert torch.equal(x, y), what
    assert not torch.equal(want[0][1], k0[0])   # (the step has written a row of keys)


def one_layer(g, H, d, dim, width):
    return {"proj": int8(g, 4 * H * d, dim), "combiner": int8(g, dim, 4 * H * d), "expand": int8(g, H * d, dim), "contract": int8(g, dim, H * d),
            "qv_scale": 0.02, "combiner_scale": 0.03, "contract_scale": 0.025, "width": width, "slope": 0.5}


@pytest.mark.parametrize("d,max_len", [(64, 60), (64, 140), (128, 60), (128, 70)])   # short and long steps
def test_cache_tokens_sixteen_megabytes_apart(ctx, monkeypatch, d, max_len):
    """A cache whose tokens are 2^24 bytes apart: the general kernel with the front, bit for bit the chain (which appends in the general
    kernel without one); the same layer on a near cache adds up in another order."""
    g = torch.Generator(device="cuda").manual_seed(d + max_len)
    H, dim, apart = 2, 128 * (d // 64), 1 << 24
    layer = one_layer(g, H, d, dim, max_len)
    k0, v0 = int8(g, 1, H, max_len, d), int8(g, 1, H, max_len, d)
    state0 = torch.randn((1, dim), device="cuda", generator=g)
    rope, pos = ctx.fill_rope_table(d, max_len), torch.tensor([max_len - 2], dtype=torch.int32, device="cuda")
    far = [torch.zeros(max_len * apart, dtype=torch.uint8, device="cuda").as_strided((1, H, max_len, d), (max_len * apart, d, apart, 1)) for _ in range(2)]

    def step(chain, planes):
        c = KVCache(ctx, capi.I8, 1, H, max_len, d)
        if planes is not None:
            c.k, c.v = planes
        c.k.copy_(k0); c.v.copy_(v0); c.k_scale.fill_(0.01); c.v_scale.fill_(attention.VEC_SCALE); c.cache_len.fill_(max_len - 2)
        state = state0.clone()
        with monkeypatch.context() as m:
            if chain:
                m.setattr(attention, "_layer_token", lambda *a: None)
            val, pending = attention.add_lookup_product(ctx, layer, c, pos, rope, state, scratch={}, defer=True)
        out = [val, pending[0].sum(dim=0, dtype=torch.int32), state, c.k, c.v, c.k_scale, c.cache_len]
        return [x.clone() if x.stride(-1) == 1 else x for x in out[:3]] + [x.contiguous().clone() for x in out[3:]]

    got, want, near = step(False, far), step(True, far), step(False, None)
    torch.cuda.synchronize()
    for x, y in zip(got, want):
        assert torch.equal(x, y)
    for x, y in zip(got[3:], near[3:]):
        assert torch.equal(x, y)
    # single-precision sums of at most 140 terms of order 1 in another order
    assert (got[0] - near[0]).abs().max().item() < 1e-4


def test_state_rows_too_far_apart_for_32_bit_offsets(ctx):
    """Two rows of the state more than 2^31 bytes apart: the normalisations become launches of their own, with the same bits."""
    g = torch.Generator(device="cuda").manual_seed(5)
    B, H, d, dim, max_len = 2, 2, 64, 128, 20
    layers = [one_layer(g, H, d, dim, w) for w in (max_len, 3)]
    k0, v0 = int8(g, 2, B, H, max_len, d), int8(g, 2, B, H, max_len, d)
    state0 = torch.randn((B, dim), device="cuda", generator=g)
    rope, pos = ctx.fill_rope_table(d, max_len), torch.tensor([7, 3], dtype=torch.int32, device="cuda")
    pitch = (1 << 29) + 4
    far = torch.empty(pitch + dim, dtype=torch.float32, device="cuda").as_strided((B, dim), (pitch, 1))

    def steps(state):
        state.copy_(state0)
        seen, pending, keep = [], None, {}
        for i, layer in enumerate(layers):
            c = KVCache(ctx, capi.I8, B, H, max_len, d)
            c.k.copy_(k0[i]); c.v.copy_(v0[i]); c.k_scale.fill_(0.01); c.v_scale.fill_(attention.VEC_SCALE); c.cache_len.copy_(pos)
            val, pending = attention.add_lookup_product(ctx, layer, c, pos, rope, state, scratch=keep, pending=pending, defer=True)
            seen += [val.clone(), pending[0].sum(dim=0, dtype=torch.int32), state.clone(), c.k, c.v, c.k_scale, c.cache_len]
        return seen + [attention.flush_state(ctx, pending, state), state.clone()]

    got, want = steps(far), steps(torch.empty((B, dim), dtype=torch.float32, device="cuda"))
    torch.cuda.synchronize()
    for x, y in zip(got, want):
        assert torch.equal(x, y)


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
