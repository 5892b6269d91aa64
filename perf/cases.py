"""The passes that this framework's performance is measured on.

Each case is one pass as a user's training or serving program makes it: a group of layers forward and backward (or
forward alone, for serving) through the operator-level entry points, on inputs that are already on the GPU.  The sizes
are those of the repository's own workloads - the MNIST convnet, ResNet-50's bottleneck blocks and stem, the 21 x 1
speech stack, the recurrent layers and the linear layers of a speech model - with other batch sizes, lengths and widths
around them, odd ones among them.

    listed()             the fixed cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what the program has in hand before the call
    run(state)           one pass -> its outputs
    work(case)           bytes and operations that the pass cannot do without
    tolerance(case)      how far two correct implementations may be apart
"""
import math

import torch

from flashlight_amd import ops

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SIZEOF = {"f32": 4, "bf16": 2, "f16": 2}
RNN_MODES = {"relu": ops.RNN_RELU, "tanh": ops.RNN_TANH, "lstm": ops.RNN_LSTM, "gru": ops.RNN_GRU}
RNN_GATES = {"relu": 1, "tanh": 1, "lstm": 4, "gru": 3}
BN_AXES = [2]           # batch norm over the channels of [W, H, C, N]
BN_MOMENTUM, BN_EPSILON = 0.1, 1e-5


def listed():
    return [
        # The smallest work: a step (with its SGD update) of the MNIST convnet, about twenty small calls.
        {"name": "mnist_b64", "kind": "mnist", "batch": 64},
        # Bottleneck blocks of ResNet-50 in training: the first stage's large planes in fp32 ...
        {"name": "block_f32_56_b32", "kind": "block", "dtype": "f32", "batch": 32, "plane": 56, "mid": 64, "stride": 1},
        # ... the third stage (six of the sixteen blocks) in bf16 at the batch of the whole-step benchmark ...
        {"name": "block_bf16_14_b64", "kind": "block", "dtype": "bf16", "batch": 64, "plane": 14, "mid": 256, "stride": 1},
        # ... and the strided entry into the last stage, with its projection shortcut and a ragged last batch, in f16.
        {"name": "block_f16_7_s2_b33", "kind": "block", "dtype": "f16", "batch": 33, "plane": 7, "mid": 512, "stride": 2},
        # The stem: 7x7 stride 2 over the image, batch norm, ReLU and max pool over the largest planes of the network.
        {"name": "stem_bf16_224_b64", "kind": "stem", "dtype": "bf16", "batch": 64, "image": 224},
        # Serving one image: a block forward with running statistics, where latency and launches count.
        {"name": "infer_f16_28_b1", "kind": "infer", "dtype": "f16", "batch": 1, "plane": 28, "mid": 128},
        # The speech stack (21 x 1 windows, 80 -> 250 -> 250 -> 250 channels) in training, as benchmarked ...
        {"name": "speech_f32_t1500_b16", "kind": "speech", "dtype": "f32", "batch": 16, "frames": 1500, "channels": 250},
        # ... and a short last batch of utterances of an odd length in bf16.
        {"name": "speech_bf16_t1111_b7", "kind": "speech", "dtype": "bf16", "batch": 7, "frames": 1111, "channels": 250},
        # Recurrent layers of an acoustic model in training: stacked bidirectional LSTM (the largest work listed) ...
        {"name": "lstm_train_512x2_bi", "kind": "rnn", "mode": "lstm", "train": True, "input": 512, "hidden": 512,
         "layers": 2, "bidirectional": True, "frames": 200, "batch": 32},
        # ... and one wide GRU layer at a batch of 64.
        {"name": "gru_train_1024", "kind": "rnn", "mode": "gru", "train": True, "input": 1024, "hidden": 1024,
         "layers": 1, "bidirectional": False, "frames": 100, "batch": 64},
        # Streaming recognition: a chunk of a few frames of a few streams through an LSTM with carried state.
        {"name": "lstm_stream_320x3", "kind": "rnn", "mode": "lstm", "train": False, "input": 80, "hidden": 320,
         "layers": 3, "bidirectional": False, "frames": 25, "batch": 5},
        # The end of an acoustic model: linear, ReLU, layer norm, classifier over word pieces, log-softmax and cross
        # entropy, forward and backward.
        {"name": "tail_bf16_4000", "kind": "tail", "dtype": "bf16", "frames": 4000, "width": 2000, "classes": 9998},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_rnn(rng):
    while True:
        c = {"kind": "rnn", "mode": rng.choice(["lstm", "lstm", "gru", "gru", "tanh", "relu"]),
             "train": rng.random() < 0.7, "input": rng.choice([40, 80, 129, 256, 512, 1024]),
             "hidden": rng.choice([128, 200, 256, 320, 384, 512, 640, 768, 1024]), "layers": rng.choice([1, 1, 2, 3]),
             "bidirectional": rng.random() < 0.5, "frames": _log_int(rng, 8, 300), "batch": _log_int(rng, 1, 64)}
        steps = c["frames"] * c["layers"] * (3 if c["train"] else 1)
        if work(c)["flops"] <= 4e11 and steps <= 1200:
            return c


def draw(rng):
    kind = rng.choice(["mnist", "block", "block", "block", "stem", "infer", "speech", "speech", "rnn", "rnn", "rnn", "tail"])
    if kind == "mnist":
        return {"kind": kind, "batch": _log_int(rng, 1, 512)}
    if kind == "rnn":
        return _draw_rnn(rng)
    dtype = rng.choice(["f32", "bf16", "bf16", "f16"])
    stage = rng.randrange(4)
    image = rng.choice([192, 224, 224, 256])
    if kind == "block":
        return {"kind": kind, "dtype": dtype, "batch": _log_int(rng, 4, 64), "plane": (image >> 2) >> stage,
                "mid": 64 << stage, "stride": rng.choice([1, 1, 2]) if stage else 1}
    if kind == "infer":
        return {"kind": kind, "dtype": dtype, "batch": _log_int(rng, 1, 16), "plane": (image >> 2) >> stage, "mid": 64 << stage}
    if kind == "stem":
        return {"kind": kind, "dtype": dtype, "batch": _log_int(rng, 4, 64), "image": image}
    if kind == "speech":
        return {"kind": kind, "dtype": dtype, "batch": _log_int(rng, 1, 24), "frames": _log_int(rng, 200, 1800),
                "channels": rng.choice([128, 200, 250, 250, 256, 320])}
    return {"kind": kind, "dtype": dtype, "frames": _log_int(rng, 64, 6000), "width": rng.choice([256, 512, 768, 1024, 1200, 2000]),
            "classes": rng.choice([29, 128, 1000, 4001, 9998])}


# ---- inputs ---------------------------------------------------------------------------
class _Maker:
    """Seeded inputs on the GPU with the distributions of the layers' neighbours."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def randn(self, *shape, dtype=torch.float32, scale=1.0, shift=0.0):
        t = torch.randn(*shape, generator=self.g, device="cuda")
        return t.mul_(scale).add_(shift).to(dtype)

    def uniform(self, *shape, bound):
        return torch.empty(*shape, device="cuda").uniform_(-bound, bound, generator=self.g)

    def activations(self, *shape, dtype):
        """What comes out of a batch norm and a ReLU."""
        return torch.randn(*shape, generator=self.g, device="cuda").clamp_(min=0).to(dtype)

    def labels(self, n, classes):
        return torch.randint(0, classes, (n,), generator=self.g, device="cuda", dtype=torch.int32)

    def conv(self, k, c, kh, kw):
        """Kaiming-normal master weights."""
        return self.randn(k, c, kh, kw, scale=math.sqrt(2.0 / (c * kh * kw)))

    def norm(self, c):
        """Scale, shift and running statistics of a batch norm."""
        return {"gamma": self.randn(c, scale=0.1, shift=1.0), "beta": torch.zeros(c, device="cuda"),
                "mean": self.randn(c, scale=0.1), "var": self.randn(c, scale=0.05, shift=1.0).abs_()}


def prepare(case, seed):
    return {"mnist": _prepare_mnist, "block": _prepare_block, "infer": _prepare_infer, "stem": _prepare_stem,
            "speech": _prepare_speech, "rnn": _prepare_rnn, "tail": _prepare_tail}[case["kind"]](case, _Maker(seed))


def run(state):
    return state["run"](state)


# ---- the MNIST convnet: one training step ------------------------------------------------
def _prepare_mnist(case, m):
    b = case["batch"]
    shapes = [(32, 1, 5, 5), (32,), (64, 32, 5, 5), (64,), (3136, 1024), (1024,), (1024, 10), (10,)]
    fan = [25, 25, 800, 800, 3136, 3136, 1024, 1024]
    params = [m.uniform(*s, bound=1.0 / math.sqrt(f)) for s, f in zip(shapes, fan)]
    return {"run": _run_mnist, "x": m.randn(b, 1, 28, 28), "labels": m.labels(b, 10), "params": params,
            "velocity": [torch.zeros_like(p) for p in params], "one": torch.ones(1, device="cuda")}


def _run_mnist(s):
    x, (w1, b1, w2, b2, w3, b3, w4, b4) = s["x"], s["params"]
    conv, pool = {"px": 2, "py": 2}, (2, 2, 2, 2, 0, 0)
    a1 = ops.conv2d(x, w1, b1, **conv)
    r1 = ops.relu(a1)
    p1, m1 = ops.pool2d(r1, *pool)
    a2 = ops.conv2d(p1, w2, b2, **conv)
    r2 = ops.relu(a2)
    p2, m2 = ops.pool2d(r2, *pool)
    f = p2.reshape(p2.shape[0], -1)
    a3 = ops.linear(f, w3, b3)
    r3 = ops.relu(a3)
    a4 = ops.linear(r3, w4, b4)
    logp = ops.log_softmax(a4)
    loss, stats = ops.categorical_cross_entropy(logp, s["labels"])

    d = ops.categorical_cross_entropy_backward(s["one"], logp.shape, logp.dtype, s["labels"], stats)
    d = ops.log_softmax_backward(d, logp)
    d, dw4, db4 = ops.linear_backward(d, r3, w4)
    d = ops.relu_backward(d, a3)
    d, dw3, db3 = ops.linear_backward(d, f, w3)
    d = ops.pool2d_backward(d.reshape(p2.shape), r2.shape, m2, *pool)
    d = ops.relu_backward(d, a2)
    dw2, db2 = ops.conv2d_backward_filter_bias(d, p1, w2.shape, True, **conv)
    d = ops.conv2d_backward_data(d, p1.shape, w2, **conv)
    d = ops.pool2d_backward(d, r1.shape, m1, *pool)
    d = ops.relu_backward(d, a1)
    dw1, db1 = ops.conv2d_backward_filter_bias(d, x, w1.shape, True, **conv)
    grads = [dw1, db1, dw2, db2, dw3, db3, dw4, db4]
    ops.sgd_step(s["params"], grads, s["velocity"], lr=1e-3, momentum=0.9, weight_decay=1e-4)
    return {"loss": loss, "logp": logp, "grads": grads, "params": s["params"], "velocity": s["velocity"]}


# ---- convolution + batch norm + ReLU, as the network modules put them together ----------
# A training pass is the forward pass of one micro-batch and the backward pass of another, as a program that
# accumulates gradients or runs its stages as a pipeline has them in flight: the backward pass starts from what that
# other micro-batch's forward pass kept, which is in hand before the call.  (Were it the same micro-batch, the last bit
# of a convolution would now and then decide the sign of a ReLU's input, and a gradient come or go with it.)
def _forward(x, w, bn, geo, residual=None, relu=True):
    a, _ = ops.conv2d(x, w, None, keep_gathered=True, **geo)
    return _norm(a, bn, residual, relu)[0]


def _norm(a, bn, residual=None, relu=True):
    """Batch norm, residual and ReLU -> (output, what the backward pass needs of them).  The mask form needs planes of a
    multiple of 4 elements."""
    masked = relu and a.shape[2] * a.shape[3] % 4 == 0
    y, sm, si, *mask = ops.batchnorm_relu(a, bn["gamma"], bn["beta"], bn["mean"], bn["var"], BN_AXES, BN_MOMENTUM, BN_EPSILON,
                                          residual=residual, relu=relu, want_mask=masked)
    return y, {"a": a, "y": None if masked or not relu else y, "sm": sm, "si": si, "mask": mask[0] if mask else None, "relu": relu}


def _kept(m, x, w, bn, geo, residual=False, relu=True):
    """What the forward pass of one layer kept for its backward pass: -> (the layer's output, that).  The convolution's
    result is drawn (no value near zero, where rounding decides a ReLU), the rest follows from it."""
    oh = (x.shape[2] + 2 * geo.get("py", 0) - w.shape[2]) // geo.get("sy", 1) + 1
    ow = (x.shape[3] + 2 * geo.get("px", 0) - w.shape[3]) // geo.get("sx", 1) + 1
    a = torch.randn(x.shape[0], w.shape[0], oh, ow, generator=m.g, device="cuda")
    a = a.add_(torch.sign(a), alpha=0.1)
    r = a.clamp(min=0).mul_(0.5).to(x.dtype) if residual else None
    y, kept = _norm(a.to(x.dtype), dict(bn, mean=None, var=None), r, relu)
    gathered = ops.conv2d(x, w, None, keep_gathered=True, **geo)[1]
    return y, dict(kept, x=x, gathered=gathered)


def _backward(dy, k, w, bn, geo, want_dx=True, want_residual=False, addend=None):
    """-> (dx or None, gradient of the residual or None, [dw, dgamma, dbeta])"""
    dr = None
    if k["relu"]:
        da, dg, db, dr = ops.batchnorm_relu_backward(dy, k["a"], k["y"], bn["gamma"], k["sm"], k["si"], BN_AXES,
                                                     want_residual_grad=want_residual, mask=k["mask"])
    else:
        da, dg, db = ops.batchnorm_backward(dy, k["a"], bn["gamma"], k["sm"], k["si"], BN_AXES)
    dw, _ = ops.conv2d_backward_filter_bias(da, k["x"], w.shape, False, gathered=k["gathered"], **geo)
    dx = ops.conv2d_backward_data(da, k["x"].shape, w, addend=addend, **geo) if want_dx else None
    return dx, dr, [dw, dg, db]


def _cast(weights, dtype):
    """The step's copy of the fp32 master weights in the storage type."""
    return weights if dtype == torch.float32 else ops.astype_many(weights, dtype)


def _block_shapes(case):
    mid, stride = case["mid"], case.get("stride", 1)
    out = 4 * mid
    cin = 2 * mid if stride == 2 else out
    shapes = [(mid, cin, 1, 1), (mid, mid, 3, 3), (out, mid, 1, 1)]
    if stride == 2:
        shapes.append((out, cin, 1, 1))
    return shapes, case["plane"] * stride, stride


def _prepare_block(case, m):
    dt, b = DTYPES[case["dtype"]], case["batch"]
    shapes, plane, st = _block_shapes(case)
    three, proj = {"sx": st, "sy": st, "px": 1, "py": 1}, {"sx": st, "sy": st}
    s = {"run": _run_block, "dtype": dt, "geo": [{}, three, {}, proj], "weights": [m.conv(*c) for c in shapes],
         "bn": [m.norm(c[0]) for c in shapes], "x": m.activations(b, shapes[0][1], plane, plane, dtype=dt),
         "dy": m.randn(b, 4 * case["mid"], case["plane"], case["plane"], dtype=dt)}
    h = x = m.activations(b, shapes[0][1], plane, plane, dtype=dt)
    w, s["kept"] = _cast(s["weights"], dt), []
    for i in range(len(w)):
        h, kept = _kept(m, x if i in (0, 3) else h, w[i], s["bn"][i], s["geo"][i], residual=i == 2, relu=i != 3)
        s["kept"].append(kept)
    return s


def _run_block(s):
    x, bn, geo, kept = s["x"], s["bn"], s["geo"], s["kept"]
    w = _cast(s["weights"], s["dtype"])
    projected = len(w) == 4
    shortcut = _forward(x, w[3], bn[3], geo[3], relu=False) if projected else x
    h = _forward(x, w[0], bn[0], geo[0])
    h = _forward(h, w[1], bn[1], geo[1])
    y = _forward(h, w[2], bn[2], geo[2], residual=shortcut)

    d, dr, g3 = _backward(s["dy"], kept[2], w[2], bn[2], geo[2], want_residual=True)
    d, _, g2 = _backward(d, kept[1], w[1], bn[1], geo[1])
    grads = g2 + g3
    if projected:
        dr, _, g4 = _backward(dr, kept[3], w[3], bn[3], geo[3])
        grads = grads + g4
    dx, _, g1 = _backward(d, kept[0], w[0], bn[0], geo[0], addend=dr)
    return {"y": y, "dx": dx, "grads": g1 + grads, "running": [t for n in bn for t in (n["mean"], n["var"])]}


def _prepare_infer(case, m):
    dt = DTYPES[case["dtype"]]
    shapes, plane, _ = _block_shapes(case)
    return {"run": _run_infer, "x": m.activations(case["batch"], shapes[0][1], plane, plane, dtype=dt),
            "weights": [m.conv(*s).to(dt) for s in shapes], "bn": [m.norm(s[0]) for s in shapes]}


def _run_infer(s):
    x = h = s["x"]
    for i, (w, bn) in enumerate(zip(s["weights"], s["bn"])):
        p = w.shape[2] // 2
        h = ops.conv2d(h, w, None, px=p, py=p)
        h, _, _ = ops.batchnorm(h, bn["gamma"], bn["beta"], bn["mean"], bn["var"], BN_AXES, False, BN_MOMENTUM, BN_EPSILON)
        if i + 1 == len(s["weights"]):
            h = torch.add(h, x)
        h = ops.relu(h)
    return h


# ---- the stem: convolution over the image, batch norm, ReLU, max pool ---------------------
def _prepare_stem(case, m):
    dt, b, im = DTYPES[case["dtype"]], case["batch"], case["image"]
    s = {"run": _run_stem, "dtype": dt, "geo": {"sx": 2, "sy": 2, "px": 3, "py": 3}, "pool": (3, 3, 2, 2, 1, 1),
         "x": m.randn(b, 3, im, im, dtype=dt), "weights": m.conv(64, 3, 7, 7), "bn": m.norm(64),
         "dy": m.randn(b, 64, im // 4, im // 4, dtype=dt)}
    h, s["kept"] = _kept(m, m.randn(b, 3, im, im, dtype=dt), s["weights"].to(dt), s["bn"], s["geo"])
    s["argmax"], s["shape"] = ops.pool2d(h, *s["pool"])[1], h.shape
    return s


def _run_stem(s):
    w, bn, geo, pool = _cast([s["weights"]], s["dtype"])[0], s["bn"], s["geo"], s["pool"]
    h = _forward(s["x"], w, bn, geo)
    y, argmax = ops.pool2d(h, *pool)
    d = ops.pool2d_backward(s["dy"], s["shape"], s["argmax"], *pool)
    _, _, grads = _backward(d, s["kept"], w, bn, geo, want_dx=False)      # a training step needs no gradient of the image
    return {"y": y, "argmax": argmax, "grads": grads, "running": [bn["mean"], bn["var"]]}


# ---- the speech stack ------------------------------------------------------------------------
def _speech_layers(case):
    """(weight shape, stride, input frames, output frames) of the three layers."""
    c, t, layers = case["channels"], case["frames"], []
    for cin, stride in ((80, 1), (c, 1), (c, 2)):
        pad = ops.derive_padding(t, 21, stride, -1)
        to = (t + 2 * pad - 21) // stride + 1
        layers.append(((c, cin, 1, 21), stride, pad, t, to))
        t = to
    return layers


def _prepare_speech(case, m):
    dt, b, layers = DTYPES[case["dtype"]], case["batch"], _speech_layers(case)
    s = {"run": _run_speech, "dtype": dt, "x": m.randn(b, 80, 1, case["frames"], dtype=dt),
         "weights": [m.conv(*l[0]) for l in layers], "bn": [m.norm(l[0][0]) for l in layers],
         "geo": [{"sx": l[1], "sy": 1, "px": l[2], "py": 0} for l in layers],
         "dy": m.randn(b, case["channels"], 1, layers[-1][4], dtype=dt), "kept": []}
    h, w = m.randn(b, 80, 1, case["frames"], dtype=dt), _cast(s["weights"], dt)
    for i in range(3):
        h, kept = _kept(m, h, w[i], s["bn"][i], s["geo"][i])
        s["kept"].append(kept)
    return s


def _run_speech(s):
    w, bn, geo = _cast(s["weights"], s["dtype"]), s["bn"], s["geo"]
    h = s["x"]
    for i in range(3):
        h = _forward(h, w[i], bn[i], geo[i])
    d, grads = s["dy"], []
    for i in (2, 1, 0):
        d, _, g = _backward(d, s["kept"][i], w[i], bn[i], geo[i], want_dx=i > 0)   # the features are the network's input
        grads = g + grads
    return {"y": h, "grads": grads, "running": [t for n in bn for t in (n["mean"], n["var"])]}


# ---- recurrent layers -------------------------------------------------------------------------
def _rnn_args(case):
    return case["hidden"], case["layers"], RNN_MODES[case["mode"]], case["bidirectional"]


def _prepare_rnn(case, m):
    t, b, h = case["frames"], case["batch"], case["hidden"]
    dirs = 2 if case["bidirectional"] else 1
    s = {"args": _rnn_args(case), "x": m.randn(t, b, case["input"]), "hx": None, "cx": None,
         "w": m.uniform(ops.rnn_param_count(case["input"], *_rnn_args(case)), bound=1.0 / math.sqrt(h))}
    if case["train"]:
        s.update(run=_run_rnn_train, dy=m.randn(t, b, dirs * h))
    else:
        shape = (case["layers"] * dirs, b, h)
        s.update(run=_run_rnn_infer, hx=m.uniform(*shape, bound=0.9), cx=m.randn(*shape) if case["mode"] == "lstm" else None)
    return s


def _run_rnn_train(s):
    y, hy, cy, reserve = ops.rnn(s["x"], None, None, s["w"], *s["args"])
    dx, dhx, dcx, dw = ops.rnn_backward(s["x"], s["w"], reserve, *s["args"], grad_output=s["dy"])
    return {"y": y, "hy": hy, "cy": cy, "dx": dx, "dhx": dhx, "dcx": dcx, "dw": dw}


def _run_rnn_infer(s):
    y, hy, cy, _ = ops.rnn(s["x"], s["hx"], s["cx"], s["w"], *s["args"])
    return {"y": y, "hy": hy, "cy": cy}


# ---- linear, ReLU, layer norm, classifier, loss ---------------------------------------------------
def _prepare_tail(case, m):
    dt, n, d, c = DTYPES[case["dtype"]], case["frames"], case["width"], case["classes"]
    return {"run": _run_tail, "dtype": dt, "x": m.randn(n, d, dtype=dt), "labels": m.labels(n, c),
            "one": torch.full((1,), 2.0 ** 14 if dt == torch.float16 else 1.0, device="cuda"),     # f16 trains with a loss scale
            "weights": [m.uniform(d, d, bound=1.0 / math.sqrt(d)), m.uniform(d, c, bound=1.0 / math.sqrt(d))],
            "bias": [m.uniform(d, bound=1.0 / math.sqrt(d)), m.uniform(c, bound=1.0 / math.sqrt(d))],
            "gamma": m.randn(d, scale=0.1, shift=1.0), "beta": m.randn(d, scale=0.1)}


def _run_tail(s):
    x, (b1, b2) = s["x"], s["bias"]
    w1, w2 = s["weights"] if s["dtype"] == torch.float32 else ops.astype_many(s["weights"], s["dtype"])
    a = ops.linear(x, w1, b1)
    r = ops.relu(a)
    h, ctx = ops.layer_norm(r, (0,), 1e-5, s["gamma"], s["beta"])
    z = ops.linear(h, w2, b2)
    logp = ops.log_softmax(z)
    loss, stats = ops.categorical_cross_entropy(logp, s["labels"])

    d = ops.categorical_cross_entropy_backward(s["one"], logp.shape, logp.dtype, s["labels"], stats)
    d = ops.log_softmax_backward(d, logp)
    d, dw2, db2 = ops.linear_backward(d, h, w2)
    d, dgamma, dbeta = ops.layer_norm_backward(d, ctx, s["gamma"])
    d = ops.relu_backward(d, a)
    dx, dw1, db1 = ops.linear_backward(d, x, w1)
    return {"loss": loss, "logp": logp, "dx": dx, "grads": [dw1, db1, dgamma, dbeta, dw2, db2]}


# ---- what a pass cannot do without ---------------------------------------------------------------
def work(case):
    """Operations: the products of the pass, twice the multiply-adds.  Bytes: inputs read and outputs written once, and
    in training what the forward pass keeps for the backward pass (each layer's input and its output before the
    normalisation) written once and read once."""
    kind = case["kind"]
    size = SIZEOF[case.get("dtype", "f32")]
    if kind == "mnist":
        b = case["batch"]
        params = 32 * 25 + 32 + 64 * 800 + 64 + 3136 * 1024 + 1024 + 10240 + 10
        macs = b * (784 * 32 * 25 * 2 + 196 * 64 * 800 * 3 + 3136 * 1024 * 3 + 10240 * 3)
        kept = b * (784 * 32 + 196 * 32 + 196 * 64 + 49 * 64 + 1024 + 10)
        return {"bytes": 4 * (784 * b + 2 * kept + 5 * params), "flops": 2 * macs}
    if kind in ("block", "infer"):
        shapes, plane, stride = _block_shapes(case)
        b, out = case["batch"], case["plane"] ** 2
        planes = [plane * plane, out, out, out]
        weights = sum(k * c * kh * kw for k, c, kh, kw in shapes)
        macs = b * sum(p * k * c * kh * kw for p, (k, c, kh, kw) in zip(planes, shapes))
        x, y = b * plane * plane * shapes[0][1], b * out * 4 * case["mid"]
        if kind == "infer":
            return {"bytes": size * (x + y + weights), "flops": 2 * macs}
        kept = b * sum(p * s[0] for p, s in zip(planes, shapes)) + b * (planes[0] + out) * case["mid"]
        return {"bytes": size * (2 * x + 2 * y + 2 * kept) + 8 * weights, "flops": 6 * macs}
    if kind == "stem":
        b, im = case["batch"], case["image"]
        x, a, y = b * 3 * im * im, b * 64 * (im // 2) ** 2, b * 64 * (im // 4) ** 2
        return {"bytes": size * (x + 2 * a + 2 * y) + y, "flops": 2 * 2 * a * 147}
    if kind == "speech":
        b, layers = case["batch"], _speech_layers(case)
        macs = [b * to * s[0] * s[1] * 21 for s, _, _, _, to in layers]
        weights = sum(s[0] * s[1] * 21 for s, _, _, _, _ in layers)
        kept = b * sum(s[0] * to for s, _, _, _, to in layers) * 2
        x, y = b * 80 * case["frames"], b * case["channels"] * layers[-1][4]
        return {"bytes": size * (x + 2 * y + 2 * kept) + 8 * weights, "flops": 2 * (3 * sum(macs) - macs[0])}
    if kind == "rnn":
        t, b, h, g = case["frames"], case["batch"], case["hidden"], RNN_GATES[case["mode"]]
        dirs = 2 if case["bidirectional"] else 1
        params = macs = kept = 0
        for l in range(case["layers"]):
            cin = case["input"] if l == 0 else dirs * h
            params += dirs * g * h * (cin + h + 2)
            macs += dirs * g * h * (cin + h) * t * b
            kept += dirs * t * b * h * (g + 1 + (case["mode"] == "lstm"))
        x, y = t * b * case["input"], t * b * dirs * h
        if not case["train"]:
            return {"bytes": 4 * (x + y + params), "flops": 2 * macs}
        return {"bytes": 4 * (2 * x + 2 * y + 2 * params + 2 * kept), "flops": 6 * macs}
    n, d, c = case["frames"], case["width"], case["classes"]
    weights = d * d + d * c
    return {"bytes": size * (2 * n * d + 2 * 3 * n * d + 2 * n * c + weights) + 4 * weights + 4 * n, "flops": 6 * n * weights}


def tolerance(case):
    """About four times what a pass differs by when its sums run in another order (other kernels: fp32 storage, up to
    2.8e-6 in the 2-norm and 2.1e-5 at most) or from the same pass in fp32 storage (bf16: 3e-3 to 1e-2 and 0.1; f16: 4e-4 to
    7e-4 and 7e-3).  Of the stem's max-pool indices 2.7e-3 (bf16), 3.3e-4 (f16) and none (f32) were others.  The MNIST step
    goes forward and backward on one batch: from a few hundred images on, a ReLU's or a pool's choice falls differently
    here and there (5.6e-4 and 5.4e-3 in the first layer's gradient)."""
    if case["kind"] == "mnist":
        return {"rel": 2.2e-3, "max": 2e-2}
    dtype = case.get("dtype", "f32")
    t = {"f32": {"rel": 1.2e-5, "max": 1e-4}, "bf16": {"rel": 2e-2, "max": 0.4}, "f16": {"rel": 2.8e-3, "max": 2.8e-2}}[dtype]
    if case["kind"] == "stem":
        t["differ"] = {"f32": 1e-5, "bf16": 1e-2, "f16": 1.4e-3}[dtype]
    return t
