"""The offline fp32 attention on the bf16 matrix cores, where it can go wrong:
query blocks and key tiles that end inside a tile, one tile to many turns of
the position ring, contexts that start inside a block, items of different
lengths, and values that are not finite.

The products left out are below 2^-30 of the whole one, and the sums are fp32:
the error in the 2-norm is that of the projections and the attention at a few
roundings of random sign each, 2^-19 at most (measured 2^-21).
"""
import numpy as np
import pytest
import torch

import relpos_oracle as O
import relpos_mhsa as M
import workloads as W
from _util import oracle_params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    M.library()
    yield
    torch.cuda.synchronize()


def make(d, h, T, seed):
    rng = np.random.default_rng(seed)
    w = W.make_layer_weights(rng, d, h, True, False)
    layer = M.RelPositionMultiHeadAttention(d, h, True)
    layer.load_weights(W.prefixed(w, "l"), "l")
    layer.set_dtype(O.F32)
    return rng, layer, oracle_params(w, d, h), O.RelPositionalEncoding(d, 5000, True).get_encoding(T)


def forward(layer, x, pos, ctx, lengths, T):
    before = M.debug_attention_forms()
    got = layer.forward(torch.from_numpy(x).cuda(), torch.from_numpy(pos).float().cuda().contiguous(), ctx,
                        M.key_padding_mask(lengths, T)).cpu().numpy().astype(np.float64)
    after = M.debug_attention_forms()
    assert {k for k in after if after[k] > before[k]} == {"generic"}
    return got


@pytest.mark.parametrize("d,h,B,T,ctx", [
    (512, 8, 16, 17, None), (512, 8, 16, 64, None), (256, 2, 64, 33, None), (256, 2, 32, 65, ((5, 40), "regular")),
    (512, 8, 4, 225, ((30, 0), "regular")), (1024, 8, 3, 353, None), (1024, 8, 3, 353, ((70, 13), "chunked_limited")),
    (256, 2, 16, 200, ((100, -1), "regular"))])
def test_forward_against_oracle(d, h, B, T, ctx):
    rng, layer, p, pos = make(d, h, T, d + B + T)
    x = rng.standard_normal((B, T, d)).astype(np.float32)
    lengths = [T] + [max(1, T - 1 - 37 * i % T) for i in range(1, B)]
    got = forward(layer, x, pos, M.AttentionContext.new(*ctx) if ctx else None, lengths, T)
    for b in sorted({0, 1, B - 1}):
        ref = O.mhsa_forward(p, x[b:b + 1], pos, O.AttentionContext.new(*ctx) if ctx else None,
                             O.key_padding_mask([lengths[b]], T), O.F32)
        rows = np.isfinite(ref).all(axis=-1)
        err = np.linalg.norm(got[b:b + 1][rows] - ref[rows]) / np.linalg.norm(ref[rows])
        assert rows.any() and err < 2.0 ** -19, (b, err)


@pytest.mark.parametrize("d,h", [(512, 8), (256, 2)])
def test_scores_of_one_product(d, h):
    """Scores that one product makes up (around 250 and 180), two keys a query:
    the output is one key's probability, and its logit the difference of the
    two scores. Each is rounded as an fp32 product (2^-24 and, for the parts'
    own sum, 2^-27) and once more when it is scaled; the probability's
    roundings weigh up to 10 times as much in the logit, under 100 2^-24 in
    all. The values have large second and third parts, of which the own key's
    and the other's third differ in sign; roundings are spread evenly, so half
    of the errors are below half their bound."""
    B, T, dk = 128 // h, 64, d // h
    rng = np.random.default_rng(d)
    w = {"l.%s.weight" % n: np.zeros((d, d), dtype=np.float32)
         for n in ("linear_q", "linear_k", "linear_v", "linear_out", "linear_pos")}
    for i in range(h):
        for c, n in enumerate(("linear_q", "linear_k", "linear_v")):
            w["l.%s.weight" % n][i * dk, 3 * i + c] = 1
        w["l.linear_out.weight"][i, i * dk] = 1
    w["l.pos_bias_u"] = w["l.pos_bias_v"] = np.zeros((h, dk), dtype=np.float32)
    layer = M.RelPositionMultiHeadAttention(d, h, False)
    layer.load_weights(w, "l")
    layer.set_dtype(O.F32)
    x = np.zeros((B, T, d), dtype=np.float32)
    ulp = 2.0 ** -23
    steps = lambda: rng.integers(1, 40, (B, T, h)) * ulp  # noqa: E731
    q = (16 * (1 + 255 * 2.0 ** -15 + 2.0 ** -16 - steps())).astype(np.float32)
    k = (128 * (1 + 255 * 2.0 ** -15 + 2.0 ** -16 - steps())).astype(np.float32)
    k[:, 1::2] = (128 * (1 + 2.0 ** -15 - 2.0 ** -16 + steps())[:, 1::2]).astype(np.float32)
    even = (np.arange(T) % 2 == 0).astype(np.float32)
    for i in range(h):
        x[:, :, 3 * i], x[:, :, 3 * i + 1], x[:, :, 3 * i + 2] = q[..., i], k[..., i], even
    pos = O.RelPositionalEncoding(d, 5000, True).get_encoding(T)
    before = M.debug_attention_forms()["generic"]
    got = layer.forward(torch.from_numpy(x).cuda(), torch.from_numpy(pos).float().cuda().contiguous(),
                        M.AttentionContext.new((1, 0), "regular"), None).cpu().numpy().astype(np.float64)
    assert M.debug_attention_forms()["generic"] == before + 1
    q, k = q.astype(np.float64)[:, 1:], k.astype(np.float64)
    s = np.stack([q * k[:, :-1], q * k[:, 1:]]) / np.sqrt(dk)  # of the key before, of its own
    p = got[:, 1:, :h]
    first = (even[:-1] == 1)[None, :, None]
    diff = np.where(first, s[0] - s[1], s[1] - s[0])
    use = (p > 0.1) & (p < 0.9)
    err = np.abs(np.log(p[use] / (1 - p[use])) - diff[use])
    bound = (2 + 2.0 ** -3) * 2.0 ** -24 * s.sum(axis=0)[use] + 100 * 2.0 ** -24
    assert use.sum() > 1000 and (err <= bound).all(), f"{np.max(err / bound):.3g} of the bound"
    assert np.median(err / bound) <= 0.5, f"half are above {np.median(err / bound):.3g} of the bound"


def test_values_that_are_not_finite():
    """A frame of infinities behind an item's end hides from its queries, and
    the other items do not see it."""
    d, h, B, T = 512, 8, 16, 100
    rng, layer, p, pos = make(d, h, T, 5)
    x = rng.standard_normal((B, T, d)).astype(np.float32)
    lengths = [70] * B
    clean = forward(layer, x, pos, None, lengths, T)
    x[3, 75] = np.inf
    got = forward(layer, x, pos, None, lengths, T)
    keep = np.arange(B) != 3
    assert np.array_equal(got[keep], clean[keep])
    err = np.linalg.norm(got[3, :70] - clean[3, :70]) / np.linalg.norm(clean[3, :70])
    assert err < 2.0 ** -19, err


@pytest.mark.parametrize("d,h,B,T,ctx", [(512, 8, 16, 100, None), (1024, 8, 4, 225, None),
                                         (512, 8, 4, 225, ((40, 7), "regular")), (256, 2, 32, 130, ((20, 20), "regular"))])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_frames_that_are_not_finite(d, h, B, T, ctx, value):
    """Frames of NaNs or infinities at both ends, in the middle and in the
    padding: a query that sees one, or is one and sees any, is NaN, as its
    scores are, and every other query is what it is without them."""
    rng, layer, p, pos = make(d, h, T, d + B)
    x = rng.standard_normal((B, T, d)).astype(np.float32)
    lengths = [T, T - 60, T, T - 33] + [T - 5] * (B - 4)
    context = M.AttentionContext.new(*ctx) if ctx else None
    clean = forward(layer, x, pos, context, lengths, T)
    x[0, T - 1, 3], x[1, T - 60:], x[2, 70], x[3, T - 20] = value, value, value, value
    got = forward(layer, x, pos, context, lengths, T)
    for b in range(min(B, 5)):
        i, j = np.arange(T)[:, None], np.arange(T)[None]
        seen = (j < lengths[b]) & ((j >= i - ctx[0][0]) & (j <= i + ctx[0][1]) if ctx else True)
        bad = ~np.isfinite(x[b]).all(axis=1)
        hit = (seen & bad[None]).any(axis=1) | (bad & seen.any(axis=1))
        assert np.isnan(got[b][hit]).all(), b
        ok = seen.any(axis=1) & ~hit
        if ok.any():
            err = np.linalg.norm(got[b][ok] - clean[b][ok]) / np.linalg.norm(clean[b][ok])
            assert err < 2.0 ** -19, (b, err)


def test_time_of_frames_that_are_not_finite():
    """A launch with NaNs in the padding, or an infinity that every query of an
    item sees, takes no more than 4 times an ordinary one (measured 1.2 and
    1.7; 9 to 15 times where every such query walked its keys one by one)."""
    B, T = 4, 375
    rng, layer, p, pos = make(1024, 8, T, 3)
    x = torch.randn((B, T, 1024), generator=torch.Generator("cuda").manual_seed(3), device="cuda")
    pos = torch.from_numpy(pos).float().cuda().contiguous()
    keys = M.key_padding_mask([T] + [T // 2] * (B - 1), T)

    def best(x):
        times = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(5):
                layer.forward(x, pos, None, keys)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    plain = best(x)
    padded, infinite = x.clone(), x.clone()
    padded[1:, T // 2:] = float("nan")
    infinite[1, 3] = float("inf")
    assert best(padded) < 4 * plain
    assert best(infinite) < 4 * plain


def test_tiny_values():
    """Values too small for three bf16 parts (under 2^-110), in all heads of an
    item and in one head of another, keep the relative error of ordinary ones;
    items beside them are what they are without. Outputs get the size of a
    head's values through a linear_out that scales by 2^20."""
    d, h, B, T = 512, 8, 16, 100
    rng = np.random.default_rng(1)
    w = W.make_layer_weights(rng, d, h, False, False)
    w["linear_v.weight"][:64] *= np.float32(2.0 ** -116)
    w["linear_out.weight"] = np.eye(d, dtype=np.float32) * np.float32(2.0 ** 20)
    layer = M.RelPositionMultiHeadAttention(d, h, False)
    layer.load_weights(W.prefixed(w, "l"), "l")
    layer.set_dtype(O.F32)
    p, pos = oracle_params(w, d, h), O.RelPositionalEncoding(d, 5000, True).get_encoding(T)
    x = rng.standard_normal((B, T, d)).astype(np.float32)
    x[2] *= np.float32(2.0 ** -118)
    got = forward(layer, x, pos, None, [T] * B, T)
    for b in (0, 2, 3):
        ref = O.mhsa_forward(p, x[b:b + 1], pos, None, None, O.F32)
        for lo, hi in ((0, 64), (64, d)):
            if b == 2 and lo == 0:
                continue  # (2^-234: zeros)
            err = np.linalg.norm(got[b:b + 1, :, lo:hi] - ref[..., lo:hi]) / np.linalg.norm(ref[..., lo:hi])
            assert err < 2.0 ** -19, (b, lo, err)


# long inputs (the ring of position blocks turns several times) and short ones
@pytest.mark.parametrize("d,h,B,T,form", [(512, 8, 8, 230, "generic"), (256, 2, 32, 161, "generic"),
                                          (1024, 8, 4, 353, "generic"), (512, 8, 2, 129, "generic_key_split"),
                                          (256, 2, 1, 97, "generic_key_split")])
def test_position_scores_of_the_kernel_that_runs(d, h, B, T, form):
    """The position scores that the debug entry gives are those of the kernel
    that a forward of this shape runs, and match the rel_shift of (q + v) P^T
    over the kernel's own q and P: products of d_k terms in fp32, rounded d_k
    times at most, once when a sum's halves meet and once when scaled."""
    rng, layer, p, pos = make(d, h, T, d + T)
    x = torch.from_numpy(rng.standard_normal((B, T, d)).astype(np.float32)).cuda()
    pos = torch.from_numpy(pos).float().cuda().contiguous()
    before = M.debug_attention_forms()
    got, q, P = layer.debug_position_scores(x, pos, with_inputs=True)
    after = M.debug_attention_forms()
    assert {k for k in after if after[k] > before[k]} == {form}
    dk = d // h
    q = q.cpu().numpy().astype(np.float64).reshape(B, T, h, dk).transpose(0, 2, 1, 3)
    P = P.cpu().numpy().astype(np.float64).reshape(2 * T - 1, h, dk).transpose(1, 2, 0)
    qv = (q.astype(np.float32) + np.float32(p.pos_bias_v).reshape(1, h, 1, dk)).astype(np.float64)
    scale = O.f32_scale(dk)
    ref = scale * O.rel_shift(np.matmul(qv, P[None]))[..., :T]
    mag = scale * O.rel_shift(np.matmul(np.abs(qv), np.abs(P[None])))[..., :T]
    assert (np.abs(got.cpu().numpy() - ref) <= (dk + 2) * 2.0 ** -24 * mag).all()
