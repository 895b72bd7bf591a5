"""GPU: the embedding sum, the final softmax with the greedy choice (ComputePrediction, gpt/train/cpu_infer.cpp:552-582) and
the sampled choice (SampleFromDistr, :585-599) through the C ABI against the oracle."""
import math

import numpy as np
import pytest
import torch

from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from tscale_amd import AttentionContext
    c = AttentionContext(0, max_seqs=1, max_heads=16, max_head_dim=128)
    yield c
    c.close()


dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()


def test_embed_rows_bit_exact(ctx):
    rng = np.random.default_rng(5)
    embed = rng.integers(-127, 128, (300, 256)).astype(np.int8)
    labels = rng.integers(-2, 302, (41, 3)).astype(np.int32)      # some empty slots on both sides
    want = orc.embed_rows(labels, embed, 0.0173)
    got = ctx.embed_rows(dev(labels), dev(embed.view(np.uint8)), 0.0173)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), want)
    one = ctx.embed_rows(dev(labels[:, 0].copy()), dev(embed.view(np.uint8)), 0.0173).cpu().numpy()
    assert np.array_equal(one, orc.embed_rows(labels[:, :1], embed, 0.0173))


@pytest.mark.parametrize("n_rows,n,planes", [(32, 50257, 1), (3, 1000, 4), (1, 7, 1)])
def test_softmax_rows_and_greedy_choice(ctx, n_rows, n, planes):
    rng = np.random.default_rng(n)
    parts = (rng.standard_normal((planes, n_rows, n)) * 3000).astype(np.int32)
    vec = parts.sum(axis=0).astype(np.int32)
    bias = rng.standard_normal(n).astype(np.float32)
    scale = 2e-3
    # the reference's own arithmetic (polynomial exp2, eight running sums); a single running float sum over 50k terms,
    # the oracle's other mode, is itself 1e-4 off
    want, want_arg = orc.softmax_rows(vec, scale, bias, exp2_mode=1)
    src = dev(parts if planes > 1 else vec)
    prob, arg = ctx.softmax_rows(src, scale, dev(bias))
    torch.cuda.synchronize()
    got = prob.cpu().numpy()
    assert np.array_equal(arg.cpu().numpy(), want_arg)
    big = want > 1e-30
    assert np.abs(got[big] / want[big] - 1).max() < 1e-4 and np.abs(got - want).max() < 5e-5
    assert np.abs(got.sum(axis=1) - 1).max() < 1e-4
    # the choice alone, without the probabilities and without a bias
    _, arg2 = ctx.softmax_rows(src, scale, None, want_prob=False)
    assert np.array_equal(arg2.cpu().numpy(), orc.softmax_rows(vec, scale, None)[1])


def test_softmax_rows_ties_and_negative_rows(ctx):
    tie = np.zeros((2, 600), dtype=np.int32)
    tie[0, [77, 300, 599]] = 9
    tie[1] = -40000
    prob, arg = ctx.softmax_rows(dev(tie), 1e-3)
    assert arg.cpu().numpy().tolist() == [77, 0]
    want, _ = orc.softmax_rows(tie, 1e-3)
    assert np.abs(prob.cpu().numpy() - want).max() < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("n_rows,n,temperature", [(8, 50257, 1.0), (32, 1000, 0.7), (3, 77, 2.5)])
def test_sample_rows_matches_the_oracle(ctx, n_rows, n, temperature):
    """SampleFromDistr on the device against the oracle, with the caller's random words and with the counter-based
    generator.  Scores are compared through the choice: a different index is accepted only where the oracle's own
    scores of the two indices are within rounding of each other (logf and log differ in the last bit between libm
    and the device)."""
    rng = np.random.default_rng(n)
    w = (rng.standard_normal((n_rows, n)) * 3).astype(np.float32)
    prob = np.exp(w - w.max(axis=1, keepdims=True)); prob = (prob / prob.sum(axis=1, keepdims=True)).astype(np.float32)
    prob[0, 5] = 0.0                                                     # never chosen
    words = rng.integers(0, 2**32, (n_rows, n), dtype=np.uint64).astype(np.uint32)
    dprob = torch.from_numpy(prob).cuda()
    for rnd, seed, offset in ((words, 0, 0), (None, 1313, 12345)):
        want = orc.sample_rows(prob, temperature, rnd=rnd, seed=seed, offset=offset)
        drnd = None if rnd is None else torch.from_numpy(rnd.view(np.int32)).cuda()
        got = ctx.sample_rows(dprob, temperature, rnd=drnd, seed=seed, offset=offset).cpu().numpy()
        for i in np.nonzero(got != want)[0]:
            r = rnd[i] if rnd is not None else np.array([orc.mix32(seed, offset + i * n + k) for k in range(n)], dtype=np.uint32)
            u = (r.astype(np.float64) + 0.5) / 2.0**32
            with np.errstate(divide="ignore"):
                score = np.log(prob[i].astype(np.float64)) / temperature - np.log(-np.log(u))
            assert abs(score[got[i]] - score[want[i]]) < 1e-5 * max(1.0, abs(score[want[i]])), (i, got[i], want[i])
        assert got[0] != 5


@pytest.mark.gpu
def test_sample_rows_argument_checks(ctx):
    from tscale_amd import capi
    prob = torch.full((2, 10), 0.1, dtype=torch.float32, device="cuda")
    with pytest.raises(capi.TsattnError):
        ctx.sample_rows(prob, 0.0)
    with pytest.raises(capi.TsattnError):
        ctx.sample_rows(prob, -1.0)


@pytest.mark.parametrize("n_rows,n", [(1, 4096), (3, 4097), (2, 8193), (32, 50257), (513, 4099), (1030, 4101), (1, 1100000), (4097, 3)])
def test_softmax_and_choices_at_chunk_edges(ctx, n_rows, n):
    """The library's forms -- records in lent scratch, records in the probabilities' place or choices exchanged between chunks,
    one workgroup per row over its own input -- against each other and float64, with ties over chunk boundaries."""
    from tscale_amd import capi
    g = torch.Generator(device="cuda").manual_seed(n)
    src = (torch.randn((n_rows, n), device="cuda", generator=g) * 3000).to(torch.int32)
    top = int(src.max()) + 5
    for at in (n - 1, n // 2, (n // 2 + 4096) % n):
        src[::2, at] = top
    bias = -torch.randn(n, device="cuda", generator=g).abs() * (src.amax(0) < top)   # (ties stay ties, and the largest)
    w = src.double() * float(np.float32(1e-3)) + bias.double()
    want = torch.softmax(w * math.log(2.0), 1)
    # the reference's exponent of 2 takes w = vec * scale + bias in float: three roundings of up to 2^-24 |w|, the subtraction's, and
    # the exponential's one; then sums of n terms
    rel = (4 * float(w.abs().max()) * 2.0 ** -24 * math.log(2.0) + 1e-5)
    p1, a1 = ctx.softmax_rows(src, 1e-3, bias)
    _, a2 = ctx.softmax_rows(src, 1e-3, bias, want_prob=False)
    stream = torch.cuda.current_stream().cuda_stream
    def flat(prob, vec, argmax):
        capi.check(ctx.lib.tsattn_softmax_rows(ctx._h, n_rows, n, vec.data_ptr(), 1, 0, n, 1e-3, bias.data_ptr(), prob, n, argmax.data_ptr(), stream))
    p3, a3, a4, a5 = torch.empty_like(p1), torch.empty_like(a1), torch.empty_like(a1), torch.empty_like(a1)
    flat(p3.data_ptr(), src, a3)
    flat(None, src, a4)
    over = src.clone()
    flat(over.data_ptr(), over, a5)
    for p in (p1, p3, over.view(torch.float32)):
        assert ((p.double() - want).abs() <= rel * want + 1e-30).all()
        assert (p.double().sum(1) - 1).abs().max() < 1e-5
    first = (src.double() * float(np.float32(1e-3)) + bias.double()).argmax(1)
    for a in (a1, a2, a3, a4, a5):
        assert torch.equal(a, a1)
    assert (w.gather(1, a1.long()[:, None]) - w.gather(1, first[:, None])).abs().max() < 1e-5   # (float logits may tie)
    assert (a1[::2].long() == min(n - 1, n // 2, (n // 2 + 4096) % n)).all()
    # the sampled choice, with and without scratch
    c1 = ctx.sample_rows(p1, 0.9, seed=5, offset=17)
    c2 = torch.empty_like(c1)
    capi.check(ctx.lib.tsattn_sample_rows(ctx._h, n_rows, n, p1.data_ptr(), n, 0.9, None, 0, 5, 17, c2.data_ptr(), stream))
    torch.cuda.synchronize()
    assert torch.equal(c1, c2)


def test_softmax_and_sampling_overlap_on_streams(ctx):
    """One handle, four streams: nothing of a call stands in the handle, so what the calls return does not depend on others."""
    g = torch.Generator(device="cuda").manual_seed(3)
    src = [(torch.randn((5 + i, 20011), device="cuda", generator=g) * 3000).to(torch.int32) for i in range(4)]
    def calls(x, seed):
        prob, best = ctx.softmax_rows(x, 2e-3)
        return prob, best, ctx.softmax_rows(x, 2e-3, want_prob=False)[1], ctx.sample_rows(prob, 0.8, seed=seed)
    want = [calls(x, i) for i, x in enumerate(src)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in src]
    got = []
    for r in range(20):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got.append((i, calls(src[i], i)))
    torch.cuda.synchronize()
    for i, outs in got:
        assert all(torch.equal(a, b) for a, b in zip(outs, want[i]))

def test_masked_and_infinite_logits(ctx):
    """-inf masks a value out; +inf is the greedy choice (its row has no distribution); both in one row of several chunks and of one."""
    for n in (1000, 20000):
        src = torch.zeros((1, n), dtype=torch.int32, device="cuda")
        src[0, 7], src[0, n - 2] = 3000, 9000
        bias = torch.zeros(n, device="cuda")
        bias[n - 2], bias[3:6] = -math.inf, -math.inf
        prob, best = ctx.softmax_rows(src, 1e-3, bias)
        w = src.double() * float(np.float32(1e-3)) + bias.double()
        assert best.item() == 7 and (prob.double() - torch.softmax(w * math.log(2.0), 1)).abs().max() < 1e-6
        assert (prob[0, 3:6] == 0).all() and prob[0, n - 2] == 0
        assert ctx.sample_rows(prob, 1e-3, seed=1).item() == 7
        bias[n // 2] = math.inf
        for want_prob in (True, False):
            assert ctx.softmax_rows(src, 1e-3, bias, want_prob=want_prob)[1].item() == n // 2


@pytest.mark.parametrize("temperature", [0.05, 0.3])
def test_sample_rows_at_low_temperatures(ctx, temperature):
    """Where log(prob) / temperature is large, the single-precision score that picks the candidates has its largest error: all
    probabilities within a few rounding steps of each other, so that only exact scores tell the winner."""
    rng = np.random.default_rng(11)
    n_rows, n = 6, 9001
    prob = (np.float32(1e-4) * (1 + rng.integers(0, 8, (n_rows, n)) * np.float32(2.0 ** -22))).astype(np.float32)
    prob[3:] = (np.exp(rng.standard_normal((3, n)) * 0.01) / n).astype(np.float32)
    got = ctx.sample_rows(dev(prob), temperature, seed=21, offset=3).cpu().numpy()
    want = orc.sample_rows(prob, temperature, seed=21, offset=3)
    for i in np.nonzero(got != want)[0]: # (the two logf differ in their last bit: 2^-23 of log(prob) / temperature, both ways)
        def score(k):
            u = (float(orc.mix32(21, 3 + i * n + int(k))) + 0.5) / 2.0**32
            return math.log(float(prob[i, k])) / temperature - math.log(-math.log(u))
        assert abs(score(got[i]) - score(want[i])) <= 4 * 2.0 ** -23 * abs(math.log(float(prob[i, got[i]])) / temperature), (i, got[i], want[i])


def test_softmax_and_sampling_replay(ctx):
    """Recorded once, replayed on other inputs with eager work between the replays: the eager results every time."""
    g = torch.Generator(device="cuda").manual_seed(8)
    src = torch.zeros((7, 20011), dtype=torch.int32, device="cuda")
    calls = lambda: (lambda p: (*p, ctx.softmax_rows(src, 2e-3, want_prob=False)[1], ctx.sample_rows(p[0], 0.8, seed=4)))(ctx.softmax_rows(src, 2e-3))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        calls()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        recorded = calls()
    for _ in range(4):
        src.copy_((torch.randn(src.shape, device="cuda", generator=g) * 3000).to(torch.int32))
        want = calls()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(recorded, want))
