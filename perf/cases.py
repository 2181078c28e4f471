"""The work a program has this library do, as cases that can be timed and checked.

The sizes are those of the 0.6B model (d_model 1024, 8 heads, FeedForward 4096)
and of the large one (d_model 512, 8 heads, FeedForward 2048), conv kernel 9,
at the encoder's 12.5 frames a second. Each case goes through the public
classes of relpos_mhsa.py; `kind` names the call:

  attention   RelPositionMultiHeadAttention.forward
  sublayers   stack_sublayer_forward_ over `layers` attention sublayers
  ff          FeedForward.forward
  conv        ConvolutionModule.forward
  blocks      encoder_forward over `layers` ConformerBlocks
  attn_step   StreamState.step: one chunk per session against the cache ring
  block_steps StreamingEncoder.step_: one chunk per session through `layers` blocks

`u8`: the projections hold affine 8-bit weights in groups of 64, quantised
from weights of the usual size as the checkpoints are. `dtype`: the modules'
dtype (streamed activations are f32 in either). `padded`: the items of the
batch end at different frames.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "mlx-nemo-rs_amd"))

import relpos_mhsa as M  # noqa: E402

NORMS = ("norm_feed_forward1", "norm_self_att", "norm_conv", "norm_feed_forward2", "norm_out")
CHUNKS = 8  # chunks a streaming state has in hand; passes take them in turn


def _case(name, kind, d, batch, frames, dtype, **more):
    c = {"name": name, "kind": kind, "d_model": d, "batch": batch, "frames": frames, "dtype": dtype, "layers": 1,
         "u8": False, "padded": False, "window": 0, "causal": False, "norm": "batch_norm", "kernel": 9, "cache": 0}
    c.update(more)
    return c


def listed():
    return [
        # one utterance of 10 s through an attention layer of the large model in the default dtype
        _case("attention_f32_single", "attention", 512, 1, 125, "float32"),
        # a server's batch of utterances of up to 30 s, padded to the longest
        _case("attention_bf16_batch", "attention", 1024, 8, 375, "bfloat16", padded=True),
        # recordings of 10 minutes under limited-context attention
        _case("attention_bf16_window", "attention", 1024, 2, 7500, "bfloat16", window=128),
        # two-minute recordings through every attention sublayer of a quantised encoder (a whole call)
        _case("sublayers_u8_long", "sublayers", 1024, 4, 1500, "bfloat16", layers=24, u8=True, padded=True),
        # the batch of 30 s through the block's convolution module
        _case("conv_bf16_batch", "conv", 1024, 8, 375, "bfloat16", padded=True),
        # one utterance of an odd length through a quantised FeedForward: a command-line transcription
        _case("ff_u8_single", "ff", 1024, 1, 203, "bfloat16", u8=True),
        # the batch of 30 s through one whole block: the offline encoder's unit of work
        _case("block_bf16_batch", "blocks", 1024, 8, 375, "bfloat16", padded=True),
        # one utterance of 10 s through one whole block of a quantised checkpoint
        _case("block_u8_single", "blocks", 1024, 1, 125, "bfloat16", u8=True),
        # a batch through two blocks of a streaming model run offline: its causal convolutions make a
        # bf16 model's activations f32 (a whole call)
        _case("blocks_causal_bf16", "blocks", 1024, 4, 375, "bfloat16", layers=2, causal=True, norm="layer_norm",
              padded=True),
        # 16 live sessions, 14-frame chunks, through one attention layer
        _case("attn_step_f32_sessions", "attn_step", 1024, 16, 14, "float32", cache=70),
        # 16 live sessions through a block of the f32 model, in all parts
        _case("block_step_f32_sessions", "block_steps", 1024, 16, 14, "float32", cache=70, causal=True,
              norm="layer_norm"),
        # one live session (a microphone) through a block of a quantised bf16 model: latency
        _case("block_step_u8_single", "block_steps", 1024, 1, 14, "bfloat16", cache=70, causal=True,
              norm="layer_norm", u8=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attention", "attention", "sublayers", "ff", "conv", "blocks", "attn_step", "block_steps"])
    d = rng.choice([512, 1024])
    c = _case("", kind, d, 1, 1, rng.choice(["float32", "bfloat16"]))
    del c["name"]
    c["u8"] = rng.random() < 0.4 and kind != "conv"
    if kind in ("attn_step", "block_steps"):
        c.update(batch=_log(rng, 1, 48), frames=rng.choice([2, 7, 14]), cache=70)
        if kind == "block_steps":
            c.update(causal=True, norm=rng.choice(["batch_norm", "layer_norm"]))
    elif kind == "attention" and rng.random() < 0.3:
        c.update(batch=rng.randint(1, 2), frames=_log(rng, 600, 7500), window=rng.choice([64, 128]),
                 dtype="bfloat16")
    else:
        c.update(frames=_log(rng, 17, 1500), padded=rng.random() < 0.5)
        c["batch"] = _log(rng, 1, max(1, min(16, 4500 // c["frames"])))
        if kind == "sublayers":
            c["layers"] = rng.randint(2, 4)
        if kind in ("conv", "blocks"):
            c.update(causal=rng.random() < 0.3, norm=rng.choice(["batch_norm", "layer_norm"]))
            c["kernel"] = rng.choice([9, 31])
    c["padded"] = c["padded"] and c["batch"] > 1
    return c


# ---------------------------------------------------------------------------
# parameters
# ---------------------------------------------------------------------------

class _Maker:
    """Parameters and inputs from one seed. Tensors are made on the GPU and
    handed to load_weights as host arrays under their checkpoint names."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed) & 0x7FFFFFFF)

    def normal(self, *shape, scale=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32) * scale

    def uniform(self, lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(*shape, generator=self.g, device="cuda", dtype=torch.float32)

    def ints(self, lo, hi, n):
        """n whole numbers of [lo, hi]."""
        return [int(v) for v in torch.randint(lo, hi + 1, (n,), generator=self.g, device="cuda").tolist()]

    def linear(self, w, name, out, inp, u8, bias=True):
        a = math.sqrt(6.0 / (out + inp))
        m = self.uniform(-a, a, out, inp)
        if u8:
            # affine 8-bit in groups of 64 along the input: w ~ scale * code + bias
            q = m.view(out, inp // 64, 64)
            lo, hi = q.amin(-1), q.amax(-1)
            s, b = ((hi - lo) / 255).half(), lo.half()
            codes = ((q - b.float()[..., None]) / s.float()[..., None]).round().clamp(0, 255).to(torch.uint8)
            w[name + ".weight"] = codes.view(out, inp).cpu().numpy().view(np.uint32)
            w[name + ".scales"], w[name + ".biases"] = s.cpu().numpy(), b.cpu().numpy()
        else:
            w[name + ".weight"] = m.cpu().numpy()
        if bias:
            b = self.normal(out, scale=0.05)
            w[name + ".bias"] = (b.half() if u8 else b).cpu().numpy()

    def attention(self, w, p, d, heads, u8):
        for n in ("linear_q", "linear_k", "linear_v", "linear_out"):
            self.linear(w, "%s.%s" % (p, n), d, d, u8)
        self.linear(w, p + ".linear_pos", d, d, u8, bias=False)
        for n in ("pos_bias_u", "pos_bias_v"):
            w["%s.%s" % (p, n)] = self.normal(heads, d // heads, scale=0.2).cpu().numpy()

    def ff(self, w, p, d, u8):
        self.linear(w, p + ".linear1", 4 * d, d, u8)
        self.linear(w, p + ".linear2", d, 4 * d, u8)

    def conv(self, w, p, d, k, norm, u8):
        self.linear(w, p + ".pointwise_conv1", 2 * d, d, u8)
        self.linear(w, p + ".pointwise_conv2", d, d, u8)
        w[p + ".depthwise_conv.weight"] = self.normal(d, k, 1, scale=k ** -0.5).cpu().numpy()
        w[p + ".depthwise_conv.bias"] = self.normal(d, scale=0.05).cpu().numpy()
        w[p + ".batch_norm.weight"] = self.uniform(0.5, 1.5, d).cpu().numpy()
        w[p + ".batch_norm.bias"] = self.normal(d, scale=0.1).cpu().numpy()
        if norm == "batch_norm":
            w[p + ".batch_norm.running_mean"] = self.normal(d, scale=0.1).cpu().numpy()
            w[p + ".batch_norm.running_var"] = self.uniform(0.5, 2.0, d).cpu().numpy()

    def block(self, w, p, c):
        d = c["d_model"]
        self.ff(w, p + ".feed_forward1", d, c["u8"])
        self.attention(w, p + ".self_attn", d, 8, c["u8"])
        self.conv(w, p + ".conv", d, c["kernel"], c["norm"], c["u8"])
        self.ff(w, p + ".feed_forward2", d, c["u8"])
        for n in NORMS:
            w["%s.%s.weight" % (p, n)] = self.uniform(0.8, 1.2, d).cpu().numpy()
            w["%s.%s.bias" % (p, n)] = self.normal(d, scale=0.05).cpu().numpy()


def _make(case, seed):
    """(one weight map per layer, inputs) of a case, from the seed alone."""
    mk, d, kind = _Maker(seed), case["d_model"], case["kind"]
    maps = []
    for _ in range(case["layers"]):
        w = {}
        if kind in ("attention", "sublayers", "attn_step"):
            mk.attention(w, "m", d, 8, case["u8"])
            if kind == "sublayers":
                w["norm.weight"] = mk.uniform(0.8, 1.2, d).cpu().numpy()
                w["norm.bias"] = mk.normal(d, scale=0.05).cpu().numpy()
        elif kind == "ff":
            mk.ff(w, "m", d, case["u8"])
        elif kind == "conv":
            mk.conv(w, "m", d, case["kernel"], case["norm"], case["u8"])
        else:
            mk.block(w, "m", case)
        maps.append(w)
    b, t, cache = case["batch"], case["frames"], case["cache"]
    x = {}
    if kind in ("attn_step", "block_steps"):
        x["chunks"] = [mk.normal(b, t, d) for _ in range(CHUNKS)]
        x["fills"] = mk.ints(0, cache, b)
        x["cache"] = mk.normal(case["layers"], b, cache, d)
        for i, f in enumerate(x["fills"]):  # what was never filled is zeros
            x["cache"][:, i, : cache - f] = 0.0
        x["time"] = mk.normal(case["layers"], b, d, case["kernel"] - 1, scale=0.5)
    else:
        x["x"] = mk.normal(b, t, d).to(_dtype(case))
        x["lengths"] = [t] + mk.ints((t + 1) // 2, t, b - 1) if case["padded"] else None
    return maps, x


def _dtype(case):
    return getattr(torch, case["dtype"])


def _positions(case):
    """The position table of a case's attention in the modules' dtype (a centred band under a window)."""
    n = case["window"] + 1 if case["window"] else case["cache"] + case["frames"]
    return M.RelPositionalEncoding(case["d_model"], 5000, True).get_encoding(n).cuda().to(_dtype(case)).contiguous()


def _windowed(case):
    return M.AttentionContext.new((case["window"], case["window"]), "regular") if case["window"] else None


class _State:
    pass


def prepare(case, seed):
    maps, x = _make(case, seed)
    d, kind, dt = case["d_model"], case["kind"], _dtype(case)
    s = _State()
    s.kind = kind
    quant = M.QuantizationConfig() if case["u8"] else None
    mods = []
    for w in maps:
        if kind in ("attention", "sublayers", "attn_step"):
            m = M.RelPositionMultiHeadAttention(d, 8, True)
        elif kind == "ff":
            m = M.FeedForward(d, 4 * d, True)
        elif kind == "conv":
            m = M.ConvolutionModule(d, case["kernel"], case["norm"], case["causal"], True)
        else:
            m = M.ConformerBlock(d, 8, 4 * d, case["kernel"], case["norm"], case["causal"], True)
        m.load_weights(w, "m", quant)
        m.set_dtype(dt)
        mods.append(m)
    s.mods = mods
    if kind not in ("ff", "conv"):
        s.pos = _positions(case)
    s.context, s.lengths = _windowed(case), x.get("lengths")
    s.keys = M.key_padding_mask(s.lengths, case["frames"]) if s.lengths else None
    if kind == "attn_step":
        s.chunks, s.at = x["chunks"], 0
        s.stream = mods[0].stream(case["batch"], case["cache"], case["frames"])
        s.stream.load_cache(x["cache"][0], x["fills"])
        s.mask = M.StreamingMask((case["cache"], case["frames"] - 1), "chunked_limited")
    elif kind == "block_steps":
        s.chunks, s.at = x["chunks"], 0
        s.stream = M.StreamingEncoder(mods, case["batch"], case["cache"], case["frames"])
        s.stream.load_cache(x["cache"], x["time"], x["fills"])
        s.mask = M.StreamingMask((case["cache"], case["frames"] - 1), "chunked_limited")
    else:
        s.x = x["x"]
        if kind == "sublayers":
            s.gamma = np.stack([w["norm.weight"] for w in maps])
            s.beta = np.stack([w["norm.bias"] for w in maps])
    return s


def run(state):
    s, kind = state, state.kind
    if kind == "attention":
        return s.mods[0].forward(s.x, s.pos, s.context, s.keys)
    if kind == "sublayers":
        # in place on the residual stream, which a program gets new from the layers before
        return M.stack_sublayer_forward_(s.mods, s.x.clone(), s.pos, s.context, s.keys, s.gamma, s.beta)
    if kind == "ff":
        return s.mods[0].forward(s.x)
    if kind == "conv":
        return s.mods[0].forward(s.x, s.lengths)
    if kind == "blocks":
        return M.encoder_forward(s.mods, s.x, s.pos, s.context, s.lengths)
    chunk = s.chunks[s.at % CHUNKS]
    s.at += 1
    if kind == "attn_step":
        return s.stream.step(chunk, s.pos, s.mask)
    return s.stream.step_(chunk, s.pos, s.mask)  # (in place: norm_out keeps the chunk's values in range)


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------

def work(case):
    """Every input and parameter read once and every output written once;
    2 operations per multiply-add of the projections, the visible (query,
    key) pairs and the depthwise conv."""
    d, b, t, n, kind = case["d_model"], case["batch"], case["frames"], case["layers"], case["kind"]
    rows, streaming = b * t, kind in ("attn_step", "block_steps")
    act = 4 if streaming or case["dtype"] == "float32" else 2
    out = 4 if case["causal"] else act
    per = 1.125 if case["u8"] else 4 if case["dtype"] == "float32" else 2  # bytes of a weight
    keys = case["cache"] + t
    if streaming:
        pairs, table = rows * keys * 0.75, 0  # (sessions' caches are filled to all degrees; the table is memoised)
    else:
        seen = min(t, 2 * case["window"] + 1) if case["window"] else t
        pairs, table = rows * seen * (0.8 if case["padded"] else 1.0), 2 * seen - 1
    attn_w, ff_w, conv_w = (5 if table else 4) * d * d, 8 * d * d, 3 * d * d
    attn = 2.0 * (4 * rows + table) * d * d + 6.0 * d * pairs
    ff, conv = 16.0 * rows * d * d, 2.0 * rows * d * (3 * d + case["kernel"])
    io = rows * d * (act + out)
    # the cached keys and values that a step reads and its chunk's that it writes
    cache = 4.0 * (2 * b * keys * d + 3 * rows * d) if streaming else 0.0
    time = 2 * 4.0 * b * d * (case["kernel"] - 1) if streaming else 0.0
    table_b = table * d * (4 if case["dtype"] == "float32" else 2)
    if kind in ("attention", "sublayers", "attn_step"):
        return {"bytes": n * (attn_w * per + cache) + table_b + io, "flops": n * attn}
    if kind == "ff":
        return {"bytes": ff_w * per + io, "flops": ff}
    if kind == "conv":
        return {"bytes": conv_w * per + io, "flops": conv}
    return {"bytes": n * ((attn_w + 2 * ff_w + conv_w) * per + cache + time) + table_b + io,
            "flops": n * (attn + 2 * ff + conv)}


def tolerance(case):
    kind, f32 = case["kind"], case["dtype"] == "float32"
    if f32:
        # f32 sums in another order: measured 2e-7 to 5e-7 from the 64-bit value
        return {"rel": 2e-6}
    if kind in ("attn_step", "block_steps"):
        # f32 throughout but for the position rows, which are stored in bf16 and may round the other way
        return {"rel": 5e-4}
    # bf16 stored after every operation, 2 to 5 roundings of 2^-9 each in a layer
    return {"rel": {"attention": 1e-2, "ff": 1e-2, "conv": 1e-2, "sublayers": 2e-2, "blocks": 1e-2}[kind]}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------

class _Exact:
    """The modules over parameters that hold their cast values, every
    operation in 64 bits without a rounding between."""

    def __init__(self, w, case):
        self.w, self.case, self.bf = w, case, case["dtype"] == "bfloat16"

    def cast(self, a):
        t = torch.from_numpy(np.ascontiguousarray(a)).cuda().float()
        return (t.bfloat16() if self.bf else t).double()

    def linear(self, name, x):
        w = self.w
        if name + ".scales" in w:
            codes = torch.from_numpy(w[name + ".weight"].view(np.uint8)).cuda().double()
            s, b = self.cast(w[name + ".scales"]), self.cast(w[name + ".biases"])
            m = (codes.view(codes.shape[0], -1, 64) * s[..., None] + b[..., None]).view(codes.shape)
        else:
            m = self.cast(w[name + ".weight"])
        y = x @ m.t()
        return y + self.cast(w[name + ".bias"]) if name + ".bias" in w else y

    def norm(self, x, g, b):
        mu = x.mean(-1, keepdim=True)
        var = ((x - mu) ** 2).mean(-1, keepdim=True)
        return (x - mu) / torch.sqrt(var + 1e-5) * self.cast(self.w[g]) + self.cast(self.w[b])

    def ff(self, p, x):
        h = self.linear(p + ".linear1", x)
        return self.linear(p + ".linear2", h * torch.sigmoid(h))

    def attention(self, p, xq, xkv, pos, offset, lo, hi, window, stored=False):
        """Queries xq at frames offset + i over keys xkv; item b sees keys [lo[b], hi[b])."""
        d = xq.shape[-1]
        dk = d // 8
        heads = lambda y: y.view(y.shape[0], y.shape[1], 8, dk).transpose(1, 2).contiguous()  # noqa: E731
        q, k, v = (heads(self.linear(p + n, a)) for n, a in ((".linear_q", xq), (".linear_k", xkv),
                                                             (".linear_v", xkv)))
        pp = self.linear(p + ".linear_pos", pos.double())
        if stored:  # the position rows are a bf16 array also where the activations are f32
            pp = pp.bfloat16().double()
        pp = pp.view(-1, 8, dk).transpose(0, 1).contiguous()  # [H, rows, dk]
        centre = (pp.shape[1] - 1) // 2
        u, vb = self.cast(self.w[p + ".pos_bias_u"])[None, :, None], self.cast(self.w[p + ".pos_bias_v"])[None, :, None]
        out = torch.zeros_like(q)
        n_q, n_k = q.shape[2], k.shape[2]
        lo, hi = (torch.tensor(a, device="cuda").view(-1, 1, 1, 1) for a in (lo, hi))
        for i0 in range(0, n_q, 512):
            i1 = min(i0 + 512, n_q)
            j0 = max(0, offset + i0 - window) if window else 0
            j1 = min(n_k, offset + i1 + window) if window else n_k
            i = torch.arange(offset + i0, offset + i1, device="cuda")[:, None]
            j = torch.arange(j0, j1, device="cuda")[None]
            far = (j - i + centre).clamp(0, pp.shape[1] - 1)
            band = torch.matmul(q[:, :, i0:i1] + vb, pp.transpose(1, 2).contiguous()[None])
            bd = torch.gather(band, 3, far.expand(q.shape[0], 8, i1 - i0, j1 - j0))
            s = torch.matmul(q[:, :, i0:i1] + u, k[:, :, j0:j1].transpose(2, 3).contiguous())
            s = (s + bd) / math.sqrt(dk)
            seen = (j >= lo) & (j < hi)
            if window:
                seen = seen & ((j - i).abs() <= window)
            s = s.masked_fill(~seen, -math.inf)
            # (a query that sees no key gives zeros)
            out[:, :, i0:i1] = torch.matmul(torch.softmax(s, -1).nan_to_num(0.0), v[:, :, j0:j1])
        return self.linear(p + ".linear_out", out.transpose(1, 2).reshape(xq.shape))

    def conv(self, p, x, lengths, past=None):
        """(output, the last kernel - 1 frames); `past` [B, D, K - 1]: the frames before."""
        a, g = self.linear(p + ".pointwise_conv1", x).chunk(2, -1)
        u = a * torch.sigmoid(g)
        if lengths is not None:
            t = torch.arange(u.shape[1], device="cuda")[None, :, None]
            u = u * (t < torch.tensor(lengths, device="cuda")[:, None, None])
        k = self.case["kernel"]
        left = k - 1 if self.case["causal"] else (k - 1) // 2
        u = u.transpose(1, 2)
        u = torch.cat([past.double(), u], 2) if past is not None else torch.nn.functional.pad(u, (left, k - 1 - left))
        dw = self.cast(self.w[p + ".depthwise_conv.weight"])[:, :, 0]
        t = u.shape[2] - k + 1
        y = sum(u[:, :, i:i + t] * dw[:, i, None] for i in range(k))
        y = (y + self.cast(self.w[p + ".depthwise_conv.bias"])[:, None]).transpose(1, 2)
        if self.case["norm"] == "batch_norm":
            n = p + ".batch_norm."
            y = (y - self.cast(self.w[n + "running_mean"])) / torch.sqrt(self.cast(self.w[n + "running_var"]) + 1e-5)
            y = y * self.cast(self.w[n + "weight"]) + self.cast(self.w[n + "bias"])
        else:
            y = self.norm(y, p + ".batch_norm.weight", p + ".batch_norm.bias")
        return self.linear(p + ".pointwise_conv2", y * torch.sigmoid(y))

    def block(self, x, attend, lengths, past=None):
        nrm = lambda i, y: self.norm(y, "m.%s.weight" % NORMS[i], "m.%s.bias" % NORMS[i])  # noqa: E731
        x = x + 0.5 * self.ff("m.feed_forward1", nrm(0, x))
        x = x + attend(nrm(1, x))
        x = x + self.conv("m.conv", nrm(2, x), lengths, past)
        x = x + 0.5 * self.ff("m.feed_forward2", nrm(3, x))
        return nrm(4, x)


def exact(case, seed):
    maps, x = _make(case, seed)
    kind, b, t, cache = case["kind"], case["batch"], case["frames"], case["cache"]
    layers = [_Exact(w, case) for w in maps]
    pos = _positions(case)[0] if kind not in ("ff", "conv") else None
    streaming = kind in ("attn_step", "block_steps")
    y = x["chunks"][0].double() if streaming else x["x"].double()
    lengths = x.get("lengths")
    lo = [cache - f for f in x["fills"]] if streaming else [0] * b
    hi = [cache + t] * b if streaming else lengths or [t] * b
    for i, m in enumerate(layers):
        p = "m" if kind in ("attention", "sublayers", "attn_step") else "m.self_attn"

        def attend(h):
            # (a streaming chunk of `frames` sees the whole cache's chunks and itself)
            keys = torch.cat([x["cache"][i].double(), h], 1) if streaming else h
            f32_rows = m.bf and (streaming or case["causal"] and i > 0)
            return m.attention(p, h, keys, pos, cache, lo, hi, case["window"], stored=f32_rows)

        if kind in ("attention", "attn_step"):
            y = attend(y)
        elif kind == "sublayers":
            y = y + attend(m.norm(y, "norm.weight", "norm.bias"))
        elif kind == "ff":
            y = m.ff("m", y)
        elif kind == "conv":
            y = m.conv("m", y, lengths)
        else:
            y = m.block(y, attend, lengths, x["time"][i] if streaming else None)
    return y
