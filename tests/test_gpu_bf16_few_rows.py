"""The bf16 projections of few output tiles: remainders of the row tiles, waves
without a stage, uneven stages, each tile form on both sides of its line, V^T
of an utterance that ends inside an attention tile, and the order of their
sums, which is that of the large tiles or, for a handful of tiles, of runs of
256 columns.

A result is the bf16 rounding of an fp32 sum: 2^-8 of the value (half a unit
in the last place at most) and K 2^-24 |A| |W|^T for the sum's roundings.
"""
import numpy as np
import pytest
import torch

import relpos_oracle as O
import relpos_mhsa as M
import workloads as W
from _util import bf16_abs_excess, oracle_params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    M.library()
    yield
    torch.cuda.synchronize()


def linear(rng, o, i, quant):
    """(checkpoint entries of one linear, its weight in float64 as the kernel holds it)"""
    if not quant:
        m = (rng.standard_normal((o, i)) / np.sqrt(i)).astype(np.float32)
        return {"weight": m}, O.bf16_round(m).astype(np.float64)
    codes = rng.integers(0, 256, size=(o, i))
    sc = np.exp2(rng.uniform(-9, -7, size=(o, i // 64))).astype(np.float16)
    bi = rng.uniform(-0.3, 0.1, size=(o, i // 64)).astype(np.float16)
    w = W.pack_u8(codes)
    return ({"weight": w, "scales": sc, "biases": bi},
            O.dequantize(w, sc, bi, 8, 64, O.BF16).astype(np.float64))


# (d, f, rows): linear1 is f x d, linear2 d x f. 1 stage to 64 of them, and
# 256 tiles of 32 x 32, 64 x 32 and 64 x 64 or just more
@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("d,f,rows", [(64, 64, 1), (64, 576, 33), (192, 1088, 31), (512, 2048, 65), (1024, 4096, 32),
                                      (1024, 4096, 64), (1024, 4096, 65), (1024, 4096, 129), (1024, 4096, 203),
                                      (1024, 4096, 257), (1024, 4096, 513), (1024, 4096, 705)])
def test_linears(d, f, rows, quant):
    rng = np.random.default_rng(d + f + rows)
    w, dense = {}, []
    for name, o, i in (("linear1", f, d), ("linear2", d, f)):
        part, m = linear(rng, o, i, quant)
        w.update({"f.%s.%s" % (name, k): v for k, v in part.items()})
        dense.append(m)
    ff = M.FeedForward(d, f, False)
    ff.load_weights(w, "f")
    ff.set_dtype(O.BF16)
    for i, k in enumerate((d, f)):
        x = O.bf16_round(rng.standard_normal((rows, k)).astype(np.float32))
        got = ff.debug_linear(i, torch.from_numpy(x).cuda().bfloat16()).float().cpu().numpy().astype(np.float64)
        x = x.astype(np.float64)
        ref, mag = x @ dense[i].T, np.abs(x) @ np.abs(dense[i]).T
        assert (np.abs(got - ref) <= 2.0 ** -8 * np.abs(ref) + 1.01 * k * 2.0 ** -24 * mag).all(), f"linear{i + 1}"


# K of 1 to 64 stages (phases of four or two, ends inside one), and every tile
# form: 32 x 32 up to 256 rows of 1024 columns, 64 x 32 up to 512 (u8, and
# dense past K = 1024), 64 x 64 (u8; dense ones take the tile kernel)
@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("k,rows", [(64, 40), (128, 33), (192, 1), (256, 64), (320, 31), (384, 257), (448, 65), (512, 500),
                                    (576, 129), (704, 400), (1024, 203), (1024, 700), (1344, 300), (2240, 97),
                                    (4096, 203), (4096, 400), (4096, 641)])
def test_rows_alone_and_in_a_batch(k, rows, quant):
    """Rows give the same results bit for bit alone and among enough others
    for the large tiles."""
    rng = np.random.default_rng(k + rows)
    part, _ = linear(rng, 1024, k, quant)
    ff = M.FeedForward(k, 1024, False)
    w = {"f.linear1.%s" % n: v for n, v in part.items()}
    w.update({"f.linear2.%s" % n: v for n, v in linear(rng, k, 1024, quant)[0].items()})
    ff.load_weights(w, "f")
    ff.set_dtype(O.BF16)
    x = torch.from_numpy(rng.standard_normal((1600, k)).astype(np.float32)).cuda().bfloat16()
    assert torch.equal(ff.debug_linear(0, x[:rows].contiguous()), ff.debug_linear(0, x)[:rows])


# 8 runs are one round of the waves, 9 and 17 two and three
@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("f,rows", [(768, 1), (2048, 33), (2304, 64), (4352, 31)])
def test_runs_of_the_contraction(f, rows, quant):
    """Fewer than 16 tiles: 2^24 in the first run and -2^24 in the last leave
    what the runs between add up to, 1 + 1 from two steps of one run, which a
    single chain would lose one by one."""
    d = 64
    m, x = np.zeros((d, f), dtype=np.float32), np.zeros((rows, f), dtype=np.float32)
    for k, a, b in ((0, 4096, 4096), (256, 1, 1), (320, 1, 1), (f - 1, 4096, -4096)):
        m[:, k], x[:, k] = a, b
    w = {"f.linear1.weight": np.zeros((f, d), dtype=np.float32), "f.linear2.weight": m}
    if quant:
        sc = np.ones((d, f // 64), dtype=np.float16)
        sc[:, 0] = sc[:, -1] = 4096
        w.update({"f.linear2.weight": W.pack_u8((m != 0).astype(np.int64)), "f.linear2.scales": sc,
                  "f.linear2.biases": np.zeros_like(sc)})
    ff = M.FeedForward(d, f, False)
    ff.load_weights(w, "f", M.QuantizationConfig() if quant else None)
    ff.set_dtype(O.BF16)
    got = ff.debug_linear(1, torch.from_numpy(x).cuda().bfloat16()).float().cpu().numpy()
    assert (got == 2.0).all(), np.unique(got)


# Q/K/V with V^T and the position rows, in one launch or apart
@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("d,h,B,T", [(256, 2, 1, 1), (256, 4, 1, 33), (256, 2, 3, 31), (512, 8, 2, 97),
                                     (1024, 8, 1, 125), (1024, 8, 1, 203)])
def test_attention_layer(d, h, B, T, quant):
    rng = np.random.default_rng(d + B + T)
    w = W.make_layer_weights(rng, d, h, True, quant)
    a = np.sqrt(3.0 / d)  # (quantised weights of the usual size: +-a)
    for n in [k[:-7] for k in w if k.endswith(".scales")]:
        w[n + ".scales"] = np.full((d, d // 64), 2 * a / 255, dtype=np.float16)
        w[n + ".biases"] = np.full((d, d // 64), -a, dtype=np.float16)
    x = rng.standard_normal((B, T, d)).astype(np.float32)
    pos = O.RelPositionalEncoding(d, 5000, True).get_encoding(T)
    lengths = [T] + [max(1, T // 2)] * (B - 1)
    layer = M.RelPositionMultiHeadAttention(d, h, True)
    layer.load_weights(W.prefixed(w, "l"), "l")
    layer.set_dtype(O.BF16)
    got = layer.forward(torch.from_numpy(x).cuda().bfloat16(), torch.from_numpy(pos).cuda().bfloat16().contiguous(),
                        None, M.key_padding_mask(lengths, T)).float().cpu().numpy().astype(np.float64)
    ref = O.mhsa_forward(oracle_params(w, d, h), O.bf16_round(x), O.bf16_round(pos), None,
                         O.key_padding_mask(lengths, T), O.BF16)
    rows = np.isfinite(ref).all(axis=-1)
    assert np.isfinite(got).all() and rows.sum() >= T
    assert bf16_abs_excess(got[rows], ref[rows], 2e-2)[0] <= 1.0
