"""GPU: decode with sixteen waves per workgroup at the edges of its steps, and with cache tokens too far apart for 24-bit offsets."""
import numpy as np
import pytest
import torch

from oracle import pyoracle as orc
from tests.test_gpu_decode import gpu_cache, make_cache
from tscale_amd import AttentionContext, capi

pytestmark = pytest.mark.gpu

# Single-precision sums of some thousand terms of order 1 (2^-24 each, and 1e-6 of a weight for the exponential): below 1e-5; the four-wave
# kernel is held to the same 1e-4 where the whole path is checked.
TOLERANCE = 1e-4


@pytest.fixture(scope="module")
def ctx():
    c = AttentionContext(0, max_seqs=4, max_heads=4, max_head_dim=128, max_splits=8)
    yield c
    c.close()


def queries(seed, dtype, B, H, d, bf16):
    """8-bit queries and scales [B, H] for the oracle, and what the call is given: these, or the bf16 values they come from."""
    x = torch.from_numpy(np.random.default_rng(seed).standard_normal((B, H * d)).astype(np.float32)).to(torch.bfloat16 if bf16 else torch.float32)
    q, qs = orc.quantize_rows(dtype, x.to(torch.float32).numpy(), H)
    qs = np.ascontiguousarray(qs.T)
    return (q, qs, x.cuda(), None) if bf16 else (q, qs, torch.from_numpy(q).cuda(), torch.from_numpy(qs).cuda())


# steps of 512 and 1024 rows (width 64), 256 and 512 (width 128): one row past a step of four waves, a step of sixteen less and plus one,
# several; the number of rows that decides is the room in the cache, and the sequences behind it are shorter
@pytest.mark.parametrize("d,room", [(64, 513), (64, 1023), (64, 1025), (64, 2100), (128, 257), (128, 511), (128, 513), (128, 1100)])
@pytest.mark.parametrize("dtype", [capi.I8, capi.E4M3])
@pytest.mark.parametrize("splits", [1, 2])
def test_sixteen_waves(ctx, d, room, dtype, splits, bf16=False):
    B, H = 4, 3
    lens = [room, 0, 1, room // 2 + 3]
    k, v, ks, vs = make_cache(room + d, dtype, B, H, room, d, lens)
    q, qs, dq, dqs = queries(room, dtype, B, H, d, bf16)
    want = orc.decode(dtype, q, qs, k, v, ks, vs, np.array(lens, np.int32), room, 0.01)
    cache = gpu_cache(ctx, dtype, k, v, ks, vs, lens)
    out = ctx.compute_val_lookup_decode(cache, dq, dqs, room, 0.01, n_splits=splits)
    torch.cuda.synchronize()
    out = out.cpu().numpy()
    for b, n in enumerate(lens):
        assert (np.abs(out[b] - want[b]).max() < TOLERANCE) if n else not out[b].any(), b


# one step of two rows per lane group: 512 and 256 rows, which e4m3 takes from 129 and 65 rows (a quarter of the four waves' step) to 256 and 128
@pytest.mark.parametrize("d,room", [(64, 129), (64, 255), (64, 256), (128, 65), (128, 127), (128, 128)])
@pytest.mark.parametrize("bf16", [False, True])
def test_sixteen_waves_in_one_short_step(ctx, d, room, bf16):
    test_sixteen_waves(ctx, d, room, capi.E4M3, 1, bf16)


@pytest.mark.parametrize("d,L", [(64, 60), (64, 140), (128, 60), (128, 70)])   # short and long steps
@pytest.mark.parametrize("dtype", [capi.I8, capi.E4M3])
@pytest.mark.parametrize("bf16", [False, True])
def test_distant_tokens_in_short_and_long_steps(ctx, d, L, dtype, bf16):
    test_tokens_sixteen_megabytes_apart(ctx, d, L, dtype, bf16)


@pytest.mark.parametrize("d", [64, 128])
def test_tokens_sixteen_megabytes_apart(ctx, d, L=5, dtype=capi.I8, bf16=False):
    """The rows of a head 2^24 bytes apart: offsets of 64 bits."""
    B, H, apart = 1, 2, 1 << 24
    k, v, ks, vs = make_cache(d, dtype, B, H, L, d, [L])
    q, qs, dq, dqs = queries(d, dtype, B, H, d, bf16)
    want = orc.decode(dtype, q, qs, k, v, ks, vs, np.array([L], np.int32), L, 0.0)
    cache = gpu_cache(ctx, dtype, k, v, ks, vs, [L])
    for name in ("k", "v"):
        far = torch.zeros(L * apart, dtype=torch.uint8, device="cuda").as_strided((B, H, L, d), (L * apart, d, apart, 1))
        far.copy_(getattr(cache, name))
        setattr(cache, name, far)
    out = ctx.compute_val_lookup_decode(cache, dq, dqs, L, 0.0)
    torch.cuda.synchronize()
    assert np.abs(out.cpu().numpy() - want).max() < TOLERANCE
