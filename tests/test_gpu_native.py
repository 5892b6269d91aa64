"""The operators that ops.py reaches through the native module against the same calls through the code behind it: the same results,
and the same errors for what either refuses, over the forms of arguments that they take."""
import pytest
import torch

from flashlight_amd import capi, ops

pytestmark = pytest.mark.gpu


class _Declines:
    """A native module that leaves everything to the code behind it."""

    def __getattr__(self, name):
        return lambda *a: None


def _flat(v):
    if isinstance(v, (tuple, list)):
        return [t for x in v for t in _flat(x)]
    return [v]


def _call(f):
    try:
        return _flat(f()), None
    except Exception as e:      # noqa: BLE001 - compared below
        return None, (type(e), str(e))


def _both(f, declines=False):
    """f through the native module (whose answer is None for what it leaves) and through the code behind it."""
    seen = []

    class Counts:
        def __getattr__(self, name):
            g = getattr(capi.native(), name)

            def call(*a):
                seen.append(True)               # (an error of its own is an answer)
                r = g(*a)
                seen[-1] = r is not None
                return r
            return call
    before = ops._native
    try:
        ops._native = Counts()
        got, err = _call(f)
        ops._native = _Declines()
        want, err2 = _call(f)
    finally:
        ops._native = before
    assert err == err2
    if err is None:
        assert len(got) == len(want)
        for a, b in zip(got, want):
            if b is None or not torch.is_tensor(b):
                assert a is None and b is None or a == b
                continue
            assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and a.device == b.device
            assert not a.requires_grad and torch.equal(a, b)
    assert seen and any(seen) != declines, seen


def _refused(*fs):
    """Calls that either way refuses on the host, before a kernel could read or write past an operand's end."""
    for f in fs:
        _both(f, declines=True)
        with pytest.raises(ValueError):
            f()


def _r(*shape, dtype=torch.float32):
    g = torch.Generator(device="cuda").manual_seed(sum(shape) + len(shape))
    return torch.randn(*shape, generator=g, device="cuda").to(dtype)


DTYPES = [torch.float32, torch.bfloat16, torch.float16]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("xs,ws,geo", [
    ((3, 16, 14, 14), (24, 16, 3, 3), dict(px=1, py=1)),
    ((2, 32, 28, 28), (64, 32, 3, 3), dict(px=1, py=1, sx=2, sy=2)),
    ((3, 64, 9, 11), (40, 64, 1, 1), {}),
    ((2, 12, 10, 13), (8, 6, 3, 5), dict(px=2, py=1, sx=1, sy=2, dx=1, dy=1, groups=2)),
])
def test_convolutions(dtype, xs, ws, geo):
    x, w, b = _r(*xs, dtype=dtype), _r(*ws, dtype=dtype), _r(ws[0])
    y = ops.conv2d(x, w, None, **geo)
    g, add = _r(*y.shape, dtype=dtype), _r(*xs, dtype=dtype)
    for bias in (None, b, b[:0], b.reshape(1, -1)):
        _both(lambda: ops.conv2d(x, w, bias, **geo))
    _both(lambda: ops.conv2d(x, torch.nn.Parameter(w, requires_grad=True), None, keep_gathered=True, **geo))
    _both(lambda: ops.conv2d(x, w, b.to(torch.float16), **geo), declines=True)
    _both(lambda: ops.conv2d_backward_data(g, x.shape, w, **geo))
    _both(lambda: ops.conv2d_backward_data(g, tuple(xs), w, addend=add, **geo))
    _both(lambda: ops.conv2d_backward_data(g, list(xs), w, **geo), declines=True)
    kept = ops.conv2d(x, w, None, keep_gathered=True, **geo)[1]
    _both(lambda: ops.conv2d_backward_filter_bias(g, x, w.shape, False, gathered=kept, **geo))
    _both(lambda: ops.conv2d_backward_filter_bias(g, x, tuple(ws), True, **geo))


def test_convolutions_that_are_refused():
    x, w = _r(2, 16, 8, 8), _r(8, 16, 3, 3)
    for f in (lambda: ops.conv2d(x.cpu(), w, None), lambda: ops.conv2d(x, w.cpu(), None), lambda: ops.conv2d(x[:, :, ::2], w, None),
              lambda: ops.conv2d(x, w.half(), None), lambda: ops.conv2d(x[0], w, None), lambda: ops.conv2d(x, w, _r(9)),
              lambda: ops.conv2d(x, w, None, groups=2), lambda: ops.conv2d(x, w, None, sx=0), lambda: ops.conv2d(x, _r(8, 16, 9, 9), None),
              lambda: ops.conv2d(x.double(), w.double(), None), lambda: ops.conv2d(None, w, None), lambda: ops.conv2d(x, w, None, sx=1.5),
              lambda: ops.conv2d(x[:0], w, None),
              lambda: ops.conv2d_backward_data(_r(2, 8, 5, 6), x.shape, w), lambda: ops.conv2d_backward_data(_r(2, 8, 6, 6), x.shape, w, addend=x.half()),
              lambda: ops.conv2d_backward_filter_bias(_r(2, 8, 6, 6), x, w.shape, False, gathered=torch.empty(5, dtype=torch.uint8, device="cuda")),
              lambda: ops.relu(x.cpu()), lambda: ops.relu(x.t() if x.dim() == 2 else x.transpose(0, 1)), lambda: ops.relu(x.int()),
              lambda: ops.relu_backward(x, x[:1]), lambda: ops.pool2d(x, 9, 9, 1, 1, 0, 0), lambda: ops.linear(_r(3, 5), _r(4, 6)),
              lambda: ops.linear_backward(_r(3, 7), _r(3, 4), _r(4, 6)), lambda: ops.batchnorm(x, _r(3), None, _r(16), _r(16), [2], False, 0.1, 1e-5),
              lambda: ops.batchnorm(x, None, None, None, _r(16), [2], False, 0.1, 1e-5),
              lambda: ops.batchnorm_relu(x, None, None, None, None, [0, 2], 0.1, 1e-5), lambda: ops.batchnorm_relu(x, None, None, None, None, [4], 0.1, 1e-5),
              lambda: ops.batchnorm_relu(x, None, None, None, None, [2], 0.1, 1e-5, residual=x[:1])):
        _both(f, declines=True)


def test_convolutions_of_operands_that_are_refused():
    """Operands of two types, and a gathered input that is not the forward call's bytes."""
    geo, xs, ws = dict(sx=2, sy=2), (3, 128, 28, 28), (128, 128, 1, 1)
    x, w = _r(*xs, dtype=torch.bfloat16), _r(*ws, dtype=torch.bfloat16)
    y, kept = ops.conv2d(x, w, None, keep_gathered=True, **geo)
    assert kept is not None and kept.dtype == torch.uint8
    n, g, dw, db = kept.numel(), _r(*y.shape, dtype=torch.bfloat16), torch.empty(ws, device="cuda"), torch.empty(128, device="cuda")
    _both(lambda: ops.conv2d_backward_filter_bias(g, x, ws, True, gathered=kept, **geo))
    data, grads = ops.conv2d_backward_data, ops.conv2d_backward_filter_bias
    _refused(lambda: data(g, xs, w.float(), **geo), lambda: data(g.float(), xs, w, **geo), lambda: data(g, xs, w.half(), **geo),
             lambda: data(g, xs, w.to(torch.uint8), **geo), lambda: data(g.half(), xs, w, addend=x.half(), **geo),
             lambda: grads(g.float(), x, ws, True, **geo), lambda: grads(g, x.float(), ws, True, **geo), lambda: grads(g.half(), x, ws, False, **geo),
             lambda: grads(g, x, ws, True, gathered=torch.zeros(n, dtype=torch.bool, device="cuda"), **geo),
             lambda: grads(g, x, ws, True, gathered=torch.zeros(n, device="cuda"), **geo),
             lambda: grads(g, x, ws, True, gathered=torch.zeros(2 * n, dtype=torch.uint8, device="cuda")[::2], **geo),
             lambda: grads(g, x, ws, True, gathered=kept.cpu(), **geo))
    static = ops.conv2d_backward_filter_bias_static
    for f in (lambda: static(g.float(), x, dw, db, **geo), lambda: static(g, x, dw, db[:127], **geo), lambda: static(g, x, dw.half(), db, **geo),
              lambda: static(g, x, dw.transpose(0, 1), db, **geo)):
        with pytest.raises(ValueError):
            f()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape,axes", [((3, 8, 14, 14), [2]), ((2, 5, 7, 9), (2,)), ((4, 3, 2, 5), [0, 1, 2]), ((6, 10), [0]), ((3, 4, 5), [1, 2])])
def test_batch_norm(dtype, shape, axes):
    x = _r(*shape, dtype=dtype)
    c = 1
    for a in axes:
        c *= shape[len(shape) - 1 - a]
    w, b, m, v = _r(c), _r(c), _r(c), _r(c).abs() + 0.5
    _both(lambda: ops.batchnorm(x, w, b, m, v, axes, False, 0.1, 1e-5))
    _both(lambda: ops.batchnorm(x, None, b[:0], m, v, axes, False, 0, 1))
    _both(lambda: ops.batchnorm(x, w.double().float().half(), b, m, v, axes, False, 0.1, 1e-5), declines=True)
    res, g = _r(*shape, dtype=dtype), _r(*shape, dtype=dtype)

    def train(**k):
        rm, rv = m.clone(), v.clone()
        return ops.batchnorm_relu(x, w, b, rm, rv, axes, 0.1, 1e-5, **k), rm, rv
    inner = x.numel() // c if axes[0] else 1
    _both(lambda: train())
    _both(lambda: train(residual=res, relu=False))
    masked = axes == [2] and shape[-1] * shape[-2] % 4 == 0
    if masked:
        _both(lambda: train(residual=res, want_mask=True))
    elif inner % 4:
        _both(lambda: train(want_mask=True), declines=True)
    _, sm, si = ops.batchnorm(x, w, b, None, None, axes, True, 0.1, 1e-5)
    _both(lambda: ops.batchnorm_backward(g, x, w, sm, si, axes))
    if axes[0] == 0:                            # (one feature per element of a row: not fused with the ReLU, refused above)
        return
    y, sm, si = ops.batchnorm_relu(x, w, b, None, None, axes, 0.1, 1e-5)
    _both(lambda: ops.batchnorm_relu_backward(g, x, y, w, sm, si, axes, want_residual_grad=True))
    _both(lambda: ops.batchnorm_relu_backward(g, x, None, w, sm, si, axes), declines=True)
    if masked:
        mask = ops.batchnorm_relu(x, w, b, None, None, axes, 0.1, 1e-5, want_mask=True)[3]
        _both(lambda: ops.batchnorm_relu_backward(g, x, None, w, sm, si, axes, mask=mask))
        _both(lambda: ops.batchnorm_relu_backward(g, x, None, w, sm, si, axes, mask=mask[1:]), declines=True)


@pytest.mark.parametrize("want_mask", [False, True])
def test_running_statistics_that_are_refused(want_mask):
    """They are updated in place, one of them per feature."""
    x, m, v = _r(2, 16, 8, 8), _r(16), _r(16).abs()
    call = lambda m, v: lambda: ops.batchnorm_relu(x, None, None, m, v, [2], 0.1, 1e-5, want_mask=want_mask)
    _refused(call(m[:15], v), call(m, v[:1]), call(_r(17), v), call(m, _r(32)), call(m.half(), v), call(m, v.double()), call(None, v[:8]))

    def taken(*k):
        t = [None if s is None else s.clone() for s in k]
        return ops.batchnorm_relu(x, None, None, *t, [2], 0.1, 1e-5, want_mask=want_mask), t
    _both(lambda: taken(m, v))
    _both(lambda: taken(m.reshape(1, 16, 1, 1), v.reshape(4, 4)))
    _both(lambda: taken(None, None))
    _both(lambda: taken(m[:0], v[:0]))


def test_other_operands_that_are_refused():
    """Gradients, saved statistics, payloads and SGD's lists of another type, or fewer than the kernels read."""
    x, g, w = _r(2, 16, 8, 8), _r(2, 16, 8, 8), _r(16)
    y, sm, si, mask = ops.batchnorm_relu(x, w, None, None, None, [2], 0.1, 1e-5, want_mask=True)
    for bad in (sm[:15], sm.half(), sm.double(), sm.cpu(), torch.empty(32, device="cuda")[::2], None):
        for a, b in ((bad, si), (sm, bad)):
            _refused(lambda: ops.batchnorm_backward(g, x, w, a, b, [2]), lambda: ops.batchnorm_relu_backward(g, x, y, w, a, b, [2]),
                     lambda: ops.batchnorm_relu_backward(g, x, None, w, a, b, [2], mask=mask))
    p, am = ops.pool2d(x, 2, 2, 2, 2, 0, 0)
    back = lambda g, am, mode=0: lambda: ops.pool2d_backward(g, x.shape, am, 2, 2, 2, 2, 0, 0, mode)
    _refused(back(p[:1], am), back(p, am[:, 1:].contiguous()), back(p, am.int()), back(p, am.bool()), back(p, None), back(p[:1], None, 1))
    _both(back(p.reshape(32, 4, 4), am), declines=True)
    _both(back(p, None, 2))
    lp = ops.log_softmax(x)
    _refused(lambda: ops.log_softmax_backward(g.half(), lp), lambda: ops.log_softmax_backward(g[:1], lp), lambda: ops.log_softmax_backward(g, lp.half()))
    _both(lambda: ops.log_softmax_backward(g.reshape(-1, 8), lp), declines=True)
    a, b = [_r(3, 5), _r(7)], lambda *f: [h(t) for h, t in zip(f, (_r(3, 5), _r(7)))]
    own, short, half = (lambda t: t.clone()), (lambda t: t.flatten()[1:].clone()), (lambda t: t.half())
    for bad in (b(own, short), b(half, half), b(own, half), b(own)):
        _refused(lambda: ops.sgd_step(a, bad, b(own, own), 0.1, 0.9), lambda: ops.sgd_step(a, b(own, own), bad, 0.1, 0.9),
                 lambda: ops.sgd_step(a, bad, None, 0.1))
    _refused(lambda: ops.sgd_step(b(own, half), b(own, half), b(own, half), 0.1, 0.9))


@pytest.mark.parametrize("dtype", DTYPES)
def test_the_others(dtype):
    x, g = _r(4, 6, 9, 12, dtype=dtype), _r(4, 6, 9, 12, dtype=dtype)
    _both(lambda: ops.relu(x))
    _both(lambda: ops.relu(x[:0]))
    _both(lambda: ops.relu_backward(g, x))
    for mode in (0, ops.PoolingMode.MAX, ops.PoolingMode.AVG_INCLUDE_PADDING, 2):
        _both(lambda: ops.pool2d(x, 3, 3, 2, 2, 1, 1, mode))
        y, am = ops.pool2d(x, 3, 3, 2, 2, 1, 1, mode)
        _both(lambda: ops.pool2d(x, 2, 3, 1, 2, 0, 1, mode, train=False))
        _both(lambda: ops.pool2d_backward(y, x.shape, am, 3, 3, 2, 2, 1, 1, mode))
    _both(lambda: ops.pool2d(x[0], 3, 3, 2, 2, 1, 1), declines=True)
    for frames in (1, 33):
        a, w, b = _r(frames, 40, dtype=dtype), _r(40, 24, dtype=dtype), _r(24)
        _both(lambda: ops.linear(a, w, b))
        _both(lambda: ops.linear(a.reshape(1, frames, 40), w))
        _both(lambda: ops.linear_backward(_r(frames, 24, dtype=dtype), a, w))
        _both(lambda: ops.linear_backward(_r(frames, 24, dtype=dtype), a, w, want_bias=False))
        lp = ops.log_softmax(a)
        _both(lambda: ops.log_softmax(a))
        _both(lambda: ops.log_softmax_backward(_r(frames, 40, dtype=dtype), lp))
    many = [_r(3, 5), _r(7), _r(2, 2, 2)]
    for to in DTYPES:
        _both(lambda: ops.astype_many(many, to))
    _both(lambda: ops.astype_many(tuple(many), dtype), declines=True)

    def sgd(**k):
        p, v = [t.clone().to(dtype) for t in many], [torch.ones_like(t).to(dtype) for t in many]
        ops.sgd_step(p, [t.to(dtype) * 2 for t in many], v, lr=0.1, momentum=0.9, **k)
        return p, v
    _both(lambda: sgd())
    _both(lambda: sgd(weight_decay=1e-2, nesterov=True))


def test_other_streams_threads_and_wrapped_tensors():
    x, w = _r(8, 32, 28, 28), _r(64, 32, 3, 3)
    want = ops.conv2d(x, w, None, px=1, py=1)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        big = torch.empty(64 << 20, device="cuda").normal_()
        x2 = x * 1
        y = ops.conv2d(x2, w, None, px=1, py=1)       # on this stream, behind both
    s.synchronize()
    assert torch.equal(y, want) and big.numel()
    import threading
    outs = [None] * 4

    def work(k):
        for _ in range(50):
            outs[k] = ops.conv2d(x, w, None, px=1, py=1)
        torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(torch.equal(o, want) for o in outs)
    # a tensor without memory of its own (inside vmap) is refused as before
    with pytest.raises(Exception):
        torch.vmap(ops.relu)(x)
