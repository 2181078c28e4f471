"""The fp32 projections on the bf16 matrix cores, where they can go wrong:
remainders of their row tiles, one to many 64-column stages, every split of
the contraction, each weight kind, and values that are not finite.

The kernels write an fp32 value as the exact sum of three bf16 values and
leave out products below 2^-30 of the whole one, so their results carry the
error of fp32 sums: K 2^-24 |A| |W|^T per element at most (K roundings), and
in the 2-norm that of K / 16 roundings of random sign.
"""
import numpy as np
import pytest
import torch

import relpos_oracle as O
import relpos_mhsa as M
import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    M.library()
    yield
    torch.cuda.synchronize()


def make_ff(rng, d, f, kind):
    """(module, [W1, W2] in float64 as the kernels hold them)"""
    w, dense = {}, []
    for name, o, i in (("linear1", f, d), ("linear2", d, f)):
        if kind == "u8":
            codes = rng.integers(0, 256, size=(o, i))
            sc = np.exp2(rng.uniform(-9, -7, size=(o, i // 64))).astype(np.float16)
            bi = rng.uniform(-0.3, 0.1, size=(o, i // 64)).astype(np.float16)
            w["f.%s.weight" % name], w["f.%s.scales" % name], w["f.%s.biases" % name] = W.pack_u8(codes), sc, bi
            dense.append(O.dequantize(W.pack_u8(codes), sc, bi, 8, 64, O.F32).astype(np.float64))
        else:
            m = (rng.standard_normal((o, i)) / np.sqrt(i)).astype(np.float32)
            w["f.%s.weight" % name] = m
            dense.append((O.bf16_round(m) if kind == "bf16" else m).astype(np.float64))
    m = M.FeedForward(d, f, False)
    m.load_weights(w, "f")
    m.set_dtype(O.BF16 if kind == "bf16" else O.F32)
    return m, dense


def check(got, x, w, what):
    ref, mag = x @ w.T, np.abs(x) @ np.abs(w).T
    k = x.shape[1]
    err = np.abs(got.astype(np.float64) - ref)
    assert (err <= k * 2.0 ** -24 * mag).all(), what
    rel = np.linalg.norm(err) / np.linalg.norm(ref)
    assert rel <= 2.0 ** -22 * max(1.0, np.sqrt(k / 1024)), f"{what}: {rel:.2e}"


# 64-wide K is one stage; 513 and 1025 rows of 4096 columns are past the line
# of the large tiles; the K-parallel kernel takes the few-row short-K ones
@pytest.mark.parametrize("kind", ["f32", "bf16", "u8"])
@pytest.mark.parametrize("d,f,rows", [(64, 4096, 129), (128, 4096, 97), (192, 4096, 513), (192, 4096, 1025),
                                      (1024, 1024, 351), (512, 4096, 577)])
def test_linear1_tiles(d, f, rows, kind):
    rng = np.random.default_rng(d + f + rows)
    m, dense = make_ff(rng, d, f, kind)
    x = rng.standard_normal((rows, d)).astype(np.float32)
    got = m.debug_linear(0, torch.from_numpy(x).cuda()).cpu().numpy()
    check(got, x.astype(np.float64), dense[0], f"linear1 {kind} {rows}x{f}x{d}")


# K = 1088 .. 4096: one, two, four and eight splits, uneven ones among them
@pytest.mark.parametrize("kind", ["f32", "bf16", "u8"])
@pytest.mark.parametrize("d,f,rows", [(64, 1088, 1), (128, 2048, 31), (64, 4096, 33), (1024, 4096, 14),
                                      (1024, 4032, 225), (1024, 2048, 700), (1024, 4096, 1537)])
def test_linear2_splits(d, f, rows, kind):
    rng = np.random.default_rng(7 * d + f + rows)
    m, dense = make_ff(rng, d, f, kind)
    x = rng.standard_normal((rows, f)).astype(np.float32)
    got = m.debug_linear(1, torch.from_numpy(x).cuda()).cpu().numpy()
    check(got, x.astype(np.float64), dense[1], f"linear2 {kind} {rows}x{d}x{f}")


@pytest.mark.parametrize("kind", ["f32", "bf16", "u8"])
@pytest.mark.parametrize("which,rows", [(0, 300), (1, 40)])
def test_sums_of_few_terms(which, rows, kind):
    """A product that is a sum by itself is rounded as one fp32 product: half a
    unit in the last place, 2^-24, and 2^-27 for the small parts' own sum (they
    are 2^-6 of it, rounded 7 times) and what is left out. Two terms are
    rounded twice more where they meet."""
    rng = np.random.default_rng(rows)
    m, dense = make_ff(rng, 256, 4096, kind)
    k = 4096 if which else 256
    for terms, bound in ((1, 2.0 ** -24 + 2.0 ** -27), (2, 3 * 2.0 ** -24 + 2.0 ** -27)):
        x = np.zeros((rows, k), dtype=np.float32)
        for r in range(rows):
            x[r, rng.choice(k, terms, replace=False)] = rng.standard_normal(terms)
        got = m.debug_linear(which, torch.from_numpy(x).cuda()).cpu().numpy().astype(np.float64)
        x = x.astype(np.float64)
        over = np.abs(got - x @ dense[which].T) - bound * (np.abs(x) @ np.abs(dense[which]).T)
        assert (over <= 0).all(), f"{terms} terms: {over.max():.3g}"


def test_rows_past_two_gib():
    """131,137 rows of 4096: the activations' last rows lie past 2^31 bytes,
    and give bit for bit what the same rows give among 33,000."""
    rng = np.random.default_rng(3)
    m, _ = make_ff(rng, 64, 4096, "f32")
    few = torch.randn((33000, 4096), generator=torch.Generator("cuda").manual_seed(3), device="cuda")
    x = torch.zeros((131137, 4096), device="cuda")
    x[-33000:] = few
    got = m.debug_linear(1, x)
    assert torch.equal(got[-33000:], m.debug_linear(1, few))
    assert not got[:-33000].any()


@pytest.mark.parametrize("kind", ["f32", "bf16", "u8"])
@pytest.mark.parametrize("which,rows", [(0, 130), (1, 40)])
def test_values_that_are_not_finite(which, rows, kind):
    """Infinities, NaN and values that round to a bf16 infinity give what fp32
    sums give, in their rows alone (one split and several)."""
    rng = np.random.default_rng(rows)
    m, dense = make_ff(rng, 128, 2048, kind)
    k = 2048 if which else 128
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x[3, 5], x[7, 9], x[11, 70], x[13, 1], x[13, 2] = np.inf, -np.inf, np.nan, np.inf, -np.inf
    x[17, 100] = np.float32(3.4e38)
    got = m.debug_linear(which, torch.from_numpy(x).cuda()).cpu().numpy()
    with np.errstate(all="ignore"):
        ref = x.astype(np.float64) @ dense[which].T
        r32 = ref.astype(np.float32)
    special = [3, 7, 11, 13, 17]
    np.testing.assert_array_equal(np.isnan(got), np.isnan(r32))
    np.testing.assert_array_equal(np.where(np.isinf(r32), r32, 0), np.where(np.isinf(got), got, 0))
    row = r32[17]
    np.testing.assert_allclose(got[17][np.isfinite(row)], row[np.isfinite(row)], rtol=k * 2.0 ** -23)
    rest = [r for r in range(rows) if r not in special]
    check(got[rest], x[rest].astype(np.float64), dense[which], f"rows beside them, {kind}")


@pytest.mark.parametrize("kind", ["f32", "bf16", "u8"])
@pytest.mark.parametrize("which,rows", [(0, 321), (1, 45)])
def test_rows_of_infinities_and_nans(which, rows, kind):
    """Whole rows and columns that are not finite, a NaN whose leading bits are
    an infinity's, infinities that meet weights of zero, overflows of finite
    rows, and a weight that is not finite: what plain fp32 sums give."""
    rng = np.random.default_rng(5 + rows)
    m, dense = make_ff(rng, 128, 2048, kind)
    if kind != "u8":
        w = {"f.linear%d.weight" % (i + 1): d.astype(np.float32) for i, d in enumerate(dense)}
        w["f.linear%d.weight" % (which + 1)][3, :32] = 0
        w["f.linear%d.weight" % (which + 1)][5, 7] = -np.inf
        m.load_weights(w, "f")
        dense = [w["f.linear1.weight"].astype(np.float64), w["f.linear2.weight"].astype(np.float64)]
    k = 2048 if which else 128
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x[rows - 1, 40] = x[4, 0] = np.inf
    x[5], x[6], x[7], x[8, ::2] = np.inf, -np.inf, np.nan, -np.inf
    x[9, 100] = np.uint32(0x7F800001).view(np.float32)  # (a NaN with no bit in its leading half)
    x[10] = 0
    x[11, 2] = np.float32(3e38)
    got = m.debug_linear(which, torch.from_numpy(x).cuda()).cpu().numpy()
    with np.errstate(all="ignore"):
        ref = x.astype(np.float64) @ dense[which].T
        r32 = ref.astype(np.float32)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(r32))
    np.testing.assert_array_equal(np.where(np.isinf(r32), r32, 0), np.where(np.isinf(got), got, 0))
    rest = np.setdiff1d(np.arange(rows), [4, 5, 6, 7, 8, 9, 11, rows - 1])
    cols = np.isfinite(dense[which]).all(axis=1)
    check(got[rest][:, cols], x[rest].astype(np.float64), dense[which][cols], f"rows beside them, {kind}")


@pytest.mark.parametrize("kind", ["f32", "u8"])
def test_time_of_rows_that_are_not_finite(kind):
    """Rows with NaNs or infinities cost a reading of the row (1.3 times a
    launch where every row has one), not a recomputation of its sums (11 to 18
    times)."""
    rng = np.random.default_rng(2)
    m, _ = make_ff(rng, 1024, 4096, kind)
    x = torch.randn((1500, 1024), generator=torch.Generator("cuda").manual_seed(2), device="cuda")

    def best(x):
        times = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(5):
                m.forward(x)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    plain = best(x)
    for value in (float("nan"), float("inf")):
        y = x.clone()
        y[:, 3] = value
        assert best(y) < 4 * plain, value


@pytest.mark.parametrize("scale", [1e-20, 1e-3, 1e4, 1e18])
def test_scaled_inputs(scale):
    """The parts keep 24 bits over the fp32 range, not around 1 alone."""
    rng = np.random.default_rng(5)
    m, dense = make_ff(rng, 256, 4096, "f32")
    x = (rng.standard_normal((160, 256)) * scale * np.exp2(rng.uniform(-12, 12, size=(160, 256)))).astype(np.float32)
    got = m.debug_linear(0, torch.from_numpy(x).cuda()).cpu().numpy()
    check(got, x.astype(np.float64), dense[0], f"scale {scale}")


@pytest.mark.parametrize("kind", ["f32", "bf16", "u8"])
@pytest.mark.parametrize("which,rows", [(0, 160), (1, 40)])
def test_tiny_values(which, rows, kind):
    """Rows whose values are too small for three bf16 parts (under 2^-110),
    beside ordinary and zero rows, and an ordinary row of some tiny values.
    Products below the smallest normal number, 2^-126, lose up to 2^-150."""
    rng = np.random.default_rng(11)
    m, dense = make_ff(rng, 256, 4096, kind)
    k = 4096 if which else 256
    x = rng.standard_normal((rows, k)).astype(np.float32)
    for r, scale in ((1, -112), (2, -116), (5, -119), (6, -122)):
        x[r] *= np.float32(2.0 ** scale)
    x[9, ::2] *= np.float32(2.0 ** -118)
    x[12] = 0
    got = m.debug_linear(which, torch.from_numpy(x).cuda()).cpu().numpy().astype(np.float64)
    x = x.astype(np.float64)
    ref, mag = x @ dense[which].T, np.abs(x) @ np.abs(dense[which]).T
    assert (np.abs(got - ref) <= k * (2.0 ** -24 * mag + 2.0 ** -149)).all()
    for r in (1, 2, 5):
        rel = np.linalg.norm(got[r] - ref[r]) / np.linalg.norm(ref[r])
        assert rel <= 2.0 ** -20, f"row {r}: {rel:.2e}"
    assert not got[12].any()


# one utterance's Q/K/V and position projections in one launch, with 1 to 3
# row tiles each; the result is that of the two apart
@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("d,h,T", [(256, 4, 17), (512, 8, 33), (512, 8, 65)])
def test_paired_projections(d, h, T, quant):
    rng = np.random.default_rng(d + T)
    w = W.make_layer_weights(rng, d, h, not quant, quant, centred=quant)
    layer = M.RelPositionMultiHeadAttention(d, h, not quant)
    layer.load_weights(W.prefixed(w, "l"), "l")
    layer.set_dtype(O.F32)
    x = torch.from_numpy(rng.standard_normal((1, T, d)).astype(np.float32)).cuda()
    pos = torch.from_numpy(O.RelPositionalEncoding(d, 5000, True).get_encoding(T)).float().cuda().contiguous()
    q, P = layer.debug_position_scores(x, pos, with_inputs=True)[1:]
    assert torch.equal(q, layer.debug_linear("linear_q", x))
    assert torch.equal(P.reshape(-1, d), layer.debug_linear("linear_pos", pos).reshape(-1, d))
