"""GPU parity of rnn / rnnBackward through the C ABI against oracle/flref.c (which is
pinned against PyTorch's RNN / LSTM / GRU in tests/test_oracle_rnn.py): all four modes,
stacked, bidirectional, with and without initial states and output gradients."""
import ctypes as C

import numpy as np
import pytest
import torch

from flashlight_amd import capi, ops
from gpu_util import dev, host
from oracle import flref
from refmath import rel_l2

pytestmark = pytest.mark.gpu
MODES = [flref.RNN_RELU, flref.RNN_TANH, flref.RNN_LSTM, flref.RNN_GRU]


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("I,H,L,bidir,T,B,states", [
    (2, 2, 2, True, 3, 2, False),          # AutogradRnnTest.cpp:24-31
    (5, 7, 1, False, 6, 3, True),
    (4, 3, 3, True, 5, 2, True),
    (6, 4, 2, False, 1, 4, False),         # one step
    (40, 64, 2, True, 20, 8, True),        # sizes that reach the matrix-core products
    (80, 96, 1, False, 33, 5, False),
    # hidden sizes that are multiples of 16 with at most 64 batch columns take the fused
    # step kernels: one, two and four batch tiles, fewer contraction chunks than waves,
    # a single batch column; 65 columns and the sizes above take the two-kernel steps
    (24, 16, 1, True, 4, 17, True),
    (10, 48, 2, True, 5, 33, True),
    (12, 128, 1, False, 7, 64, False),
    (9, 160, 2, True, 6, 1, True),
    (12, 32, 1, True, 4, 65, True),
    (5, 7, 2, False, 3, 1, True),          # stacked, layer activations of 21 floats (no 16-byte multiple)
    (3, 5, 3, True, 3, 1, False),
])
def test_rnn_forward_backward(mode, I, H, L, bidir, T, B, states):
    rng = np.random.default_rng(1000 * mode + I + H + L + T)
    D = 2 if bidir else 1
    d = flref.rnn_desc(I, H, L, bidir, mode, T, B)
    n = flref.rnn_param_count(d)
    assert ops.rnn_param_count(I, H, L, mode, bidir) == n
    w = (rng.standard_normal(n) / np.sqrt(H)).astype(np.float32)
    x = rng.standard_normal((T, B, I)).astype(np.float32)
    hx = rng.standard_normal((L * D, B, H)).astype(np.float32) if states else None
    cx = rng.standard_normal((L * D, B, H)).astype(np.float32) if states and mode == flref.RNN_LSTM else None
    dy = rng.standard_normal((T, B, D * H)).astype(np.float32)
    dhy = rng.standard_normal((L * D, B, H)).astype(np.float32)
    dcy = rng.standard_normal((L * D, B, H)).astype(np.float32) if mode == flref.RNN_LSTM else None
    ry, rhy, rcy = flref.rnn_fwd(d, x, w, hx, cx)
    rdx, rdhx, rdcx, rdw = flref.rnn_bwd(d, x, w, hx, cx, dy, dhy, dcy)

    o = lambda a: None if a is None else dev(a)
    y, hy, cy, reserve = ops.rnn(dev(x), o(hx), o(cx), dev(w), H, L, mode, bidir)
    assert rel_l2(host(y), ry) <= 1e-4 and rel_l2(host(hy), rhy) <= 1e-4
    if mode == flref.RNN_LSTM:
        assert rel_l2(host(cy), rcy) <= 1e-4
    else:
        assert cy is None
    dx, dhx, dcx, dw = ops.rnn_backward(dev(x), dev(w), reserve, H, L, mode, bidir, dev(dy), dev(dhy), o(dcy))
    assert rel_l2(host(dx), rdx) <= 2e-4
    assert rel_l2(host(dhx), rdhx) <= 2e-4
    assert rel_l2(host(dw), rdw) <= 2e-4
    if mode == flref.RNN_LSTM:
        assert rel_l2(host(dcx), rdcx) <= 2e-4


def test_relu_layers_keep_the_sums_of_the_fp32_instruction():
    """The input products of ReLU layers, on whose choices the same step's gradients hang: the bits of the fp32 instruction in every layer,
    also where the other modes' run in three bf16 parts."""
    I, H, L, T, B = 512, 512, 2, 200, 64
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn(T, B, I, generator=g, device="cuda")
    for mode, same in ((flref.RNN_RELU, True), (flref.RNN_TANH, False)):
        w = torch.randn(ops.rnn_param_count(I, H, L, mode, False), generator=g, device="cuda") / H ** 0.5
        y = ops.rnn(x, None, None, w, H, L, mode, False)[0]
        capi.set_option("MATMUL_FP32_CORES", "1")
        try:
            want = ops.rnn(x, None, None, w, H, L, mode, False)[0]
        finally:
            capi.set_option("MATMUL_FP32_CORES", None)
        assert torch.equal(y, want) == same


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("I,H,L,T,B", [
    (40, 32, 2, 64, 16),        # 1024 rows: the bias sums of both directions in one launch, as the weight gradients, in slices
    (129, 48, 1, 41, 25),       # 1025 rows: not the bias sums; rows of no whole pieces
    (33, 16, 1, 3, 2),          # fewer rows than a stage
    (520, 64, 1, 43, 24),       # more input gradients than are added in a launch of their own
    (6, 20, 2, 30, 40),         # (40 columns: the second layer's input)
])
def test_both_directions_share_their_products(mode, I, H, L, T, B):
    test_rnn_forward_backward(mode, I, H, L, True, T, B, True)


@pytest.mark.parametrize("option,value", [("MATMUL_VALU", "1"), ("MATMUL_PLANES", "0"), ("MATMUL_PLANES", "7")])
def test_both_directions_keep_to_the_kernels_that_are_asked_for(option, value):
    """The projections of two directions under a switch that chooses between the products' kernels: a direction's outputs have the bits of a layer of
    that direction alone, which makes its projections by itself."""
    I, H, T, B, G = 40, 64, 10, 16, 4
    g = torch.Generator(device="cuda").manual_seed(8)
    x = torch.randn(T, B, I, generator=g, device="cuda")
    w = torch.randn(ops.rnn_param_count(I, H, 1, ops.RNN_LSTM, True), generator=g, device="cuda") / H ** 0.5
    mats, biases = G * H * (I + H), 2 * G * H
    try:
        capi.set_option("RNN_SEQUENCES", "never")
        capi.set_option(option, value)
        y = ops.rnn(x, None, None, w, H, 1, ops.RNN_LSTM, True)[0]
        for k in (0, 1):
            one = torch.cat([w[k * mats:(k + 1) * mats], w[2 * mats + k * biases:2 * mats + (k + 1) * biases]])
            z = ops.rnn(x.flip(0).contiguous() if k else x, None, None, one, H, 1, ops.RNN_LSTM, False)[0]
            assert torch.equal(y[:, :, k * H:(k + 1) * H], z.flip(0) if k else z)
    finally:
        capi.set_option(option, None)
        capi.set_option("RNN_SEQUENCES", None)


@pytest.mark.parametrize("mode,I,H,L,bidir,T,B,states", [
    # whole sequences in one launch: hidden sizes that are multiples of 4 up to 1024.  4, 8 and 16 units per workgroup,
    # a last workgroup with units to spare, a last contraction chunk with columns to spare, more waves than chunks
    (flref.RNN_LSTM, 7, 20, 1, True, 5, 70, True),         # 5 column groups per direction
    (flref.RNN_LSTM, 9, 500, 1, False, 4, 18, True),       # 4 units; 31 chunks + 4 columns
    (flref.RNN_GRU, 130, 516, 1, True, 3, 20, True),       # 8 units (the last workgroup has 4), misaligned input width
    (flref.RNN_LSTM, 8, 1024, 1, True, 2, 17, True),       # 16 units, the most registers
    (flref.RNN_GRU, 8, 1000, 1, False, 3, 66, True),       # 5 clusters of 63 workgroups: two launches
    (flref.RNN_TANH, 8, 1020, 2, False, 3, 5, False),
    (flref.RNN_RELU, 8, 4, 2, True, 7, 16, True),          # one workgroup per cluster
    (flref.RNN_LSTM, 8, 64, 1, False, 1, 1, True),         # one step, one column
    (flref.RNN_GRU, 6, 1028, 1, False, 2, 3, True),        # too wide: a launch per step
])
def test_whole_sequence_launches(mode, I, H, L, bidir, T, B, states):
    before = capi.lib().flhip_rnn_sequence_launches()
    capi.set_option("RNN_SEQUENCES", "always")       # (also where the sequence is too short to gain by them)
    try:
        test_rnn_forward_backward(mode, I, H, L, bidir, T, B, states)
    finally:
        capi.set_option("RNN_SEQUENCES", None)
    launches = capi.lib().flhip_rnn_sequence_launches() - before
    clusters = (2 if bidir else 1) * -(-B // 16)
    assert launches >= 2 * L if H <= 1024 else launches == 0
    if (H, clusters) == (1000, 5):      # 63 workgroups each: four to the first launch, forward and backward
        assert launches == 4


@pytest.mark.parametrize("mode,I,H,L,bidir,T,B,states", [
    # where the exchange of a sequence launch lies: in place of the first direction's gate gradients, in idle buffers (the topmost layer
    # has one more), behind everything
    (flref.RNN_LSTM, 9, 20, 3, True, 6, 18, True),         # whole chunks: shared, and idle buffers
    (flref.RNN_LSTM, 70, 16, 1, False, 9, 33, True),
    (flref.RNN_TANH, 5, 20, 2, True, 6, 18, True),         # a last chunk of 4: both directions in idle buffers
    (flref.RNN_RELU, 3, 12, 2, False, 9, 5, True),         # chunks larger than the state
    (flref.RNN_GRU, 12, 48, 1, False, 7, 17, True),        # one layer, the topmost
    (flref.RNN_GRU, 12, 48, 3, False, 7, 17, True),        # lower layers: behind everything
    (flref.RNN_GRU, 200, 32, 2, True, 5, 40, True),        # a wide input
    (flref.RNN_GRU, 6, 20, 3, True, 6, 9, True),
])
def test_whole_sequence_launches_in_what_the_pass_leaves_idle(mode, I, H, L, bidir, T, B, states):
    test_whole_sequence_launches(mode, I, H, L, bidir, T, B, states)


def test_whole_sequences_without_room_for_their_exchange():
    """A workspace of the size without sequence launches is accepted, and the steps run instead."""
    I, H, L, T, B = 12, 48, 3, 40, 17
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn(T, B, I, generator=g, device="cuda")
    w = torch.randn(ops.rnn_param_count(I, H, L, ops.RNN_GRU, False), generator=g, device="cuda") / H ** 0.5
    dy = torch.randn(T, B, H, generator=g, device="cuda")
    y, _, _, reserve = ops.rnn(x, None, None, w, H, L, ops.RNN_GRU, False)
    want = ops.rnn_backward(x, w, reserve, H, L, ops.RNN_GRU, False, dy)
    d = capi.RnnDesc(I, H, L, 0, ops.RNN_GRU, T, B, capi.F32)
    full = capi.lib().flhip_rnn_workspace_bytes(C.byref(d))
    capi.set_option("RNN_SEQUENCES", "never")
    try:
        least = capi.lib().flhip_rnn_workspace_bytes(C.byref(d))
    finally:
        capi.set_option("RNN_SEQUENCES", None)
    assert least < full
    count, P = capi.lib().flhip_rnn_sequence_launches, lambda t: C.c_void_p(t.data_ptr())
    before = count()
    ws, dx, dw = torch.empty(least, dtype=torch.uint8, device="cuda"), torch.empty_like(x), torch.empty_like(w)
    capi.check(capi.lib().flhip_rnn_bwd(C.byref(d), P(x), P(w), P(dy), None, None, P(reserve), reserve.numel() * reserve.element_size(), P(dx), None,
                                        None, P(dw), P(ws), least, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert count() == before and rel_l2(host(dx), host(want[0])) <= 1e-5 and rel_l2(host(dw), host(want[3])) <= 1e-5


@pytest.mark.parametrize("mode,I,H,L,T,B,states,launches", [
    # stacked layers in one launch: 4, 8 and 16 units per workgroup, two to four layers, last workgroups, chunks and column groups with some to spare
    (flref.RNN_LSTM, 7, 20, 2, 6, 5, True, 1),
    (flref.RNN_LSTM, 9, 320, 3, 5, 5, True, 1),            # 4 units
    (flref.RNN_LSTM, 33, 516, 2, 4, 3, True, 1),           # 8 units, the last workgroup has 4; odd input width
    (flref.RNN_LSTM, 8, 1024, 2, 3, 16, False, 1),         # the most registers
    (flref.RNN_LSTM, 8, 256, 4, 3, 64, True, 1),           # 16 units, four layers of four column groups
    (flref.RNN_LSTM, 8, 1024, 2, 3, 17, False, 2),         # two column groups: more clusters than compute units, a launch per layer
    (flref.RNN_LSTM, 8, 512, 4, 2, 40, False, 4),
    (flref.RNN_GRU, 12, 48, 3, 7, 17, True, 1),
    (flref.RNN_GRU, 5, 256, 2, 4, 50, True, 1),
    (flref.RNN_GRU, 6, 384, 2, 3, 70, True, 1),            # 16 units, 5 column groups
    (flref.RNN_TANH, 8, 1020, 2, 3, 5, False, 1),
    (flref.RNN_LSTM, 3, 16, 4, 8, 1, True, 1),             # one column
    (flref.RNN_TANH, 3, 4, 4, 1, 1, True, 4),              # no room for the exchanges in what the pass leaves idle
    (flref.RNN_RELU, 8, 64, 2, 6, 16, True, 2),            # a launch per layer
    (flref.RNN_TANH, 8, 16, 5, 3, 4, True, 5),             # five layers: a launch per layer
])
def test_stacked_layers_in_one_launch(mode, I, H, L, T, B, states, launches):
    count = capi.lib().flhip_rnn_sequence_launches
    try:
        capi.set_option("RNN_SEQUENCES", "stacked")
        test_rnn_forward_backward(mode, I, H, L, False, T, B, states)
        x = torch.randn(T, B, I, device="cuda")
        w = torch.randn(ops.rnn_param_count(I, H, L, mode, False), device="cuda") / H ** 0.5
        hx = torch.rand(L, B, H, device="cuda")
        if mode == flref.RNN_GRU:
            hx[0, 0, 0] = float("inf")      # (an infinite state that a product with zero would lose)
        cx = torch.randn(L, B, H, device="cuda") if mode == flref.RNN_LSTM else None
        before = count()
        got = [t for t in ops.rnn(x, hx, cx, w, H, L, mode, False) if t is not None]
        assert count() - before == launches
        capi.set_option("RNN_SEQUENCES", "always")
        want = [t for t in ops.rnn(x, hx, cx, w, H, L, mode, False) if t is not None]
    finally:
        capi.set_option("RNN_SEQUENCES", None)
    for a, b in zip(got, want):             # outputs, last states and all that is kept for the backward pass: the same sums in another order
        a, b = host(a.view(torch.float32)), host(b.view(torch.float32))
        assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isinf(a), np.isinf(b))
        ok = np.isfinite(b)
        assert rel_l2(a[ok], b[ok]) <= 1e-5


@pytest.mark.parametrize("mode,I,H,L,T,B", [
    (flref.RNN_LSTM, 9, 320, 3, 5, 5), (flref.RNN_LSTM, 33, 516, 2, 4, 3), (flref.RNN_LSTM, 8, 256, 4, 1, 64), (flref.RNN_LSTM, 8, 1024, 2, 3, 16),
    (flref.RNN_GRU, 6, 384, 2, 3, 70), (flref.RNN_GRU, 12, 48, 3, 7, 17), (flref.RNN_TANH, 8, 1020, 2, 3, 5), (flref.RNN_LSTM, 3, 16, 2, 9, 1)])
def test_stacked_layers_captured_and_eager(mode, I, H, L, T, B):
    """A launch for each diagonal of layers and steps in a graph, one launch for all without: the same bits, in what the forward pass keeps too, in every replay."""
    count = capi.lib().flhip_rnn_sequence_launches
    gen = torch.Generator(device="cuda").manual_seed(H + T)
    x, dy = torch.empty(T, B, I, device="cuda"), torch.randn(T, B, H, generator=gen, device="cuda")
    w = torch.randn(ops.rnn_param_count(I, H, L, mode, False), generator=gen, device="cuda") / H ** 0.5
    hx = torch.rand(L, B, H, generator=gen, device="cuda")
    cx = torch.randn(L, B, H, generator=gen, device="cuda") if mode == flref.RNN_LSTM else None
    run = lambda: ops.rnn(x, hx, cx, w, H, L, mode, False)
    keep = lambda out: [t.clone() for t in out[:3] if t is not None] + [t for t in ops.rnn_backward(x, w, out[3], H, L, mode, False, dy) if t is not None]
    x.zero_()
    run()
    torch.cuda.synchronize()
    before = count()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        static = run()
    assert count() == before
    for _ in range(3):
        x.copy_(torch.randn(T, B, I, generator=gen, device="cuda"))
        before = count()
        want = keep(run())
        assert count() > before
        for t in static:
            if t is not None:
                t.zero_()
        graph.replay()
        for a, b in zip(keep(static), want):
            assert torch.equal(a, b) and bool(b.isfinite().all())


def test_a_wait_of_stacked_layers_that_gives_up_ends_in_not_a_number():
    T, B, I, H, L = 5, 20, 8, 64, 3
    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(T, B, I, device="cuda", generator=gen)
    for mode in (ops.RNN_TANH, ops.RNN_LSTM, ops.RNN_GRU):
        w = torch.randn(ops.rnn_param_count(I, H, L, mode, False), device="cuda", generator=gen) / H ** 0.5
        try:
            capi.set_option("RNN_SEQUENCES", "stacked")
            want = ops.rnn(x, None, None, w, H, L, mode, False)[:2]
            capi.set_option("RNN_WAIT", "-1")
            y, hy, cy, _ = ops.rnn(x, None, None, w, H, L, mode, False)
            assert all(bool(torch.isnan(t).all()) for t in (y, hy, cy) if t is not None)
            capi.set_option("RNN_WAIT", None)
            got = ops.rnn(x, None, None, w, H, L, mode, False)[:2]
            assert all(torch.equal(a, b) for a, b in zip(got, want))
        finally:
            capi.set_option("RNN_WAIT", None)
            capi.set_option("RNN_SEQUENCES", None)


@pytest.mark.parametrize("mode,I,H,L,bidir,T,B,states", [
    (flref.RNN_LSTM, 12, 48, 3, True, 4, 20, True),        # the step kernels follow on the projections already made
    (flref.RNN_GRU, 12, 512, 2, False, 3, 33, True),
    (flref.RNN_RELU, 8, 64, 2, True, 5, 16, False),
    (flref.RNN_TANH, 8, 16, 2, True, 1, 1, True),
    (flref.RNN_LSTM, 7, 20, 2, True, 4, 9, True),          # a hidden size off 16, more than 64 columns: the two-kernel steps
    (flref.RNN_GRU, 9, 500, 2, False, 3, 18, True),
    (flref.RNN_LSTM, 5, 32, 2, True, 3, 70, True),
    (flref.RNN_RELU, 8, 4, 2, False, 4, 5, False),
])
def test_refused_sequence_launches(mode, I, H, L, bidir, T, B, states):
    """What runs where the runtime refuses a cooperative launch, after the initial states and the input projections have been
    put in place for it: forward alone, backward alone, and both."""
    before = capi.lib().flhip_rnn_sequence_launches()
    try:
        capi.set_option("RNN_SEQUENCES", "refused")
        test_rnn_forward_backward(mode, I, H, L, bidir, T, B, states)
        assert capi.lib().flhip_rnn_sequence_launches() == before
        x = torch.randn(T, B, I, device="cuda")
        w = torch.randn(ops.rnn_param_count(I, H, L, mode, bidir), device="cuda") / H ** 0.5
        dy = torch.randn(T, B, (2 if bidir else 1) * H, device="cuda")
        run = {}
        for fwd in ("refused", "always"):
            for bwd in ("refused", "always"):
                capi.set_option("RNN_SEQUENCES", fwd)
                y, hy, cy, reserve = ops.rnn(x, None, None, w, H, L, mode, bidir)
                capi.set_option("RNN_SEQUENCES", bwd)
                run[fwd, bwd] = [t for t in (y, hy, cy) + tuple(ops.rnn_backward(x, w, reserve, H, L, mode, bidir, dy)) if t is not None]
        for got in run.values():
            for a, b in zip(got, run["always", "always"]):
                # the same sums in another order, through a few steps
                assert rel_l2(host(a), host(b)) <= 1e-5
                if H % 16 == 0 and B <= 64:
                    assert torch.equal(a, b)
    finally:
        capi.set_option("RNN_SEQUENCES", None)


@pytest.mark.parametrize("mode,I,H,L,T,B", [
    (flref.RNN_LSTM, 9, 320, 3, 5, 5),           # 4 units per workgroup; the step kernels follow
    (flref.RNN_GRU, 12, 48, 3, 7, 17),
    (flref.RNN_TANH, 8, 64, 2, 6, 16),
    (flref.RNN_LSTM, 7, 20, 2, 6, 5),            # a hidden size off 16, more than 64 columns: the two-kernel steps
    (flref.RNN_GRU, 6, 128, 2, 6, 70),
])
def test_refused_launch_of_stacked_layers(mode, I, H, L, T, B):
    """What runs where the runtime refuses the one launch of all layers, after their initial states and exchanges and the lowest layer's
    projections have been put in place for it."""
    g = torch.Generator(device="cuda").manual_seed(mode + H)
    x = torch.randn(T, B, I, generator=g, device="cuda")
    w = torch.randn(ops.rnn_param_count(I, H, L, mode, False), generator=g, device="cuda") / H ** 0.5
    hx = torch.rand(L, B, H, generator=g, device="cuda")
    cx = torch.randn(L, B, H, generator=g, device="cuda") if mode == flref.RNN_LSTM else None
    count, P = capi.lib().flhip_rnn_sequence_launches, lambda t: None if t is None else C.c_void_p(t.data_ptr())
    before = count()
    try:
        capi.set_option("RNN_SEQUENCES", "never")
        want = ops.rnn(x, hx, cx, w, H, L, mode, False)
        capi.set_option("RNN_SEQUENCES", "refused")
        d = capi.RnnDesc(I, H, L, 0, mode, T, B, capi.F32)
        n = capi.lib().flhip_rnn_workspace_bytes(C.byref(d))
        ws = torch.zeros(n, dtype=torch.uint8, device="cuda")
        got = [torch.zeros_like(t) if t is not None else None for t in want]
        y, hy, cy, reserve = got
        capi.check(capi.lib().flhip_rnn_fwd(C.byref(d), P(x), P(hx), P(cx), P(w), P(y), P(hy), P(cy), P(reserve), reserve.numel() * reserve.element_size(),
                                            P(ws), n, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    finally:
        capi.set_option("RNN_SEQUENCES", None)
    assert count() == before
    # elements not yet written (-1) of the exchanges of all layers, T rows each; one layer's own leaves T - 1
    assert int((ws[: n // 4 * 4].view(torch.int32) == -1).sum()) > T * B * ((H + 15) // 16 * 16)
    for a, b in zip(got[:3], want[:3]):
        if b is None:
            continue
        assert rel_l2(host(a), host(b)) <= 1e-5      # the same sums in another order
        if H % 16 == 0 and B <= 64:
            assert torch.equal(a, b)


@pytest.mark.parametrize("H,B,bidir,T,fwd,bwd", [
    (64, 16, False, 7, 0, 0), (64, 16, False, 8, 1, 1), (64, 32, True, 5, 0, 0), (64, 32, True, 6, 1, 1),
    (64, 33, False, 4, 0, 0), (64, 33, False, 5, 1, 1),
    (512, 16, True, 5, 0, 0), (512, 16, True, 6, 1, 1), (1024, 20, True, 2, 0, 0), (1024, 20, True, 3, 1, 1),     # against a launch per step
    (64, 65, False, 2, 0, 0), (64, 65, False, 3, 1, 1), (20, 4, True, 1, 0, 0), (20, 4, True, 2, 1, 1),
    (512, 512, False, 4, 0, 0), (512, 512, False, 8, 0, 4),                    # four launches: backward alone
])
def test_where_sequence_launches_pay(H, B, bidir, T, fwd, bwd):
    """Launches of the two passes on both sides of the lines between the kernels, and what they give against each other."""
    gen = torch.Generator(device="cuda").manual_seed(H + B + T)
    x = torch.randn(T, B, 16, device="cuda", generator=gen)
    w = torch.randn(ops.rnn_param_count(16, H, 1, ops.RNN_LSTM, bidir), device="cuda", generator=gen) / H ** 0.5
    dy = torch.randn(T, B, (2 if bidir else 1) * H, device="cuda", generator=gen)
    count = capi.lib().flhip_rnn_sequence_launches

    def run():
        n = [count()]
        y, hy, cy, reserve = ops.rnn(x, None, None, w, H, 1, ops.RNN_LSTM, bidir)
        n.append(count())
        out = (y, hy, cy) + tuple(ops.rnn_backward(x, w, reserve, H, 1, ops.RNN_LSTM, bidir, dy))
        return out, n[1] - n[0], count() - n[1]
    got, nf, nb = run()
    assert (nf, nb) == (fwd, bwd)
    try:
        capi.set_option("RNN_SEQUENCES", "never" if fwd or bwd else "always")
        want, nf, nb = run()
    finally:
        capi.set_option("RNN_SEQUENCES", None)
    assert (nf > 0) == (fwd == bwd == 0)
    for a, b in zip(got, want):
        assert rel_l2(host(a), host(b)) <= 1e-5          # the same sums in another order


@pytest.mark.parametrize("mode", MODES)
def test_not_a_number_states_end(mode):
    """A state of any NaN, the pattern that marks an element as not yet written among them, gives NaN results."""
    T, B, I, H = 5, 3, 4, 32
    x = torch.ones(T, B, I, device="cuda")
    w = torch.full((ops.rnn_param_count(I, H, 1, mode, False),), 0.1, device="cuda")
    hx = torch.full((1, B, H), -1, dtype=torch.int32, device="cuda").view(torch.float32)
    y, hy, cy, reserve = ops.rnn(x, hx, None, w, H, 1, mode, False)
    dy = torch.full((T, B, H), -1, dtype=torch.int32, device="cuda").view(torch.float32)
    dx, _, _, dw = ops.rnn_backward(x, w, reserve, H, 1, mode, False, dy)
    assert mode == ops.RNN_RELU or bool(torch.isnan(y).all())      # (NaN > 0 is false: ReLU gives 0)
    assert bool(torch.isnan(dw).any()) and dx.shape == x.shape


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("L,bidir", [(1, False), (2, True)])
def test_a_wait_that_gives_up_ends_in_not_a_number(mode, L, bidir):
    """The first workgroup of every cluster stops waiting at once (the others run as ever, and all end): every output that
    depends on what it did not wait for is NaN, in ReLU layers too and in the layers above; the next call is as ever."""
    T, B, I, H, D = 5, 20, 8, 64, 2 if bidir else 1
    gen = torch.Generator(device="cuda").manual_seed(mode)
    x = torch.randn(T, B, I, device="cuda", generator=gen)
    w = torch.randn(ops.rnn_param_count(I, H, L, mode, bidir), device="cuda", generator=gen) / H ** 0.5
    dy = torch.randn(T, B, D * H, device="cuda", generator=gen)
    nan = lambda t: bool(torch.isnan(t).all())
    fine = lambda t: bool(torch.isfinite(t).all())

    def forward():
        return ops.rnn(x, None, None, w, H, L, mode, bidir)
    try:
        capi.set_option("RNN_SEQUENCES", "always")
        y0, hy0, _, reserve = forward()
        d0 = ops.rnn_backward(x, w, reserve, H, L, mode, bidir, dy)
        capi.set_option("RNN_WAIT", "-1")
        y, hy, cy, _ = forward()
        assert nan(hy) and (cy is None or nan(cy))
        if L == 1:                                  # the first step of the other workgroups needs nobody else
            units = torch.isnan(y[0]).all(0)
            assert 0 < int(units.sum()) < H and bool(units[0]) and fine(y[0][:, ~units]) and nan(y[1:])
        else:
            assert nan(y)
        dx, dhx, dcx, dw = ops.rnn_backward(x, w, reserve, H, L, mode, bidir, dy)
        assert nan(dhx) and nan(dw) and (dcx is None or nan(dcx))
        assert nan(dx[:-1]) if L == 1 else nan(dx)
        capi.set_option("RNN_WAIT", None)
        y, hy, _, reserve = forward()
        d = ops.rnn_backward(x, w, reserve, H, L, mode, bidir, dy)
        assert torch.equal(y, y0) and torch.equal(hy, hy0) and torch.equal(d[0], d0[0]) and torch.equal(d[3], d0[3])
    finally:
        capi.set_option("RNN_WAIT", None)
        capi.set_option("RNN_SEQUENCES", None)


def test_two_streams_at_once():
    """Sequences issued on two streams without waiting for each other give what they give alone."""
    T, B, I, H = 30, 32, 64, 512
    gen = torch.Generator(device="cuda").manual_seed(4)
    w = torch.randn(ops.rnn_param_count(I, H, 1, ops.RNN_LSTM, True), device="cuda", generator=gen) / H ** 0.5
    xs = [torch.randn(T, B, I, device="cuda", generator=gen) for _ in range(2)]
    dy = torch.randn(T, B, 2 * H, device="cuda", generator=gen)

    def run(x):
        y, hy, cy, reserve = ops.rnn(x, None, None, w, H, 1, ops.RNN_LSTM, True)
        return (y,) + tuple(t for t in ops.rnn_backward(x, w, reserve, H, 1, ops.RNN_LSTM, True, dy) if t is not None)

    alone = [run(x) for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in xs]
    got = [[], []]
    for _ in range(3):
        for i, st in enumerate(streams):
            with torch.cuda.stream(st):
                got[i].append(run(xs[i]))
    torch.cuda.synchronize()
    for i in range(2):
        for res in got[i]:
            assert all(torch.equal(a, b) for a, b in zip(res, alone[i]))


def _random_configs(n, seed):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(n):
        out.append((int(rng.integers(0, 4)), int(rng.integers(1, 70)),
                    int(rng.choice([16, 32, 48, 64, 80, 96, 128, 20, 7])), int(rng.integers(1, 4)),
                    bool(rng.integers(0, 2)), int(rng.integers(1, 9)),
                    int(rng.choice([1, 2, 5, 16, 17, 31, 32, 33, 48, 64, 65, 70])), bool(rng.integers(0, 2))))
    return out


@pytest.mark.parametrize("mode,I,H,L,bidir,T,B,states", _random_configs(30, 11))
def test_random_configurations(mode, I, H, L, bidir, T, B, states):
    """Seeded random sizes around the conditions of the fused step kernels (hidden sizes that
    are / are not multiples of 16, batches around the 16-column tiles and the limit of 64)."""
    test_rnn_forward_backward(mode, I, H, L, bidir, T, B, states)


@pytest.mark.parametrize("mode", [flref.RNN_LSTM, flref.RNN_GRU])
def test_missing_output_gradients_are_zero(mode):
    # only y was differentiated: the closure hands empty dhy / dcy (Functions.cpp:1677-1699)
    rng = np.random.default_rng(7)
    I, H, L, T, B = 6, 5, 2, 4, 3
    d = flref.rnn_desc(I, H, L, True, mode, T, B)
    w = (rng.standard_normal(flref.rnn_param_count(d)) * 0.4).astype(np.float32)
    x = rng.standard_normal((T, B, I)).astype(np.float32)
    dy = rng.standard_normal((T, B, 2 * H)).astype(np.float32)
    rdx, rdhx, rdcx, rdw = flref.rnn_bwd(d, x, w, None, None, dy, None, None)
    y, hy, cy, reserve = ops.rnn(dev(x), None, None, dev(w), H, L, mode, True)
    dx, dhx, dcx, dw = ops.rnn_backward(dev(x), dev(w), reserve, H, L, mode, True, dev(dy))
    assert rel_l2(host(dx), rdx) <= 2e-4 and rel_l2(host(dw), rdw) <= 2e-4 and rel_l2(host(dhx), rdhx) <= 2e-4
    # and only the final state differentiated
    dhy = rng.standard_normal((2 * L, B, H)).astype(np.float32)
    rdx, _, _, rdw = flref.rnn_bwd(d, x, w, None, None, None, dhy, None)
    dx, _, _, dw = ops.rnn_backward(dev(x), dev(w), reserve, H, L, mode, True, None, dev(dhy))
    assert rel_l2(host(dx), rdx) <= 2e-4 and rel_l2(host(dw), rdw) <= 2e-4


def test_rnn_errors():
    x = dev(np.zeros((3, 2, 4), np.float32))
    w = dev(np.zeros(ops.rnn_param_count(4, 5, 1, ops.RNN_TANH, False), np.float32))
    with pytest.raises(ValueError):
        ops.rnn(x, None, None, w[:-1], 5, 1, ops.RNN_TANH, False)          # parameter count
    with pytest.raises(ValueError):
        ops.rnn(x, dev(np.zeros((1, 2, 6), np.float32)), None, w, 5, 1, ops.RNN_TANH, False)   # state dims
    with pytest.raises(ValueError):
        ops.rnn(x, None, dev(np.zeros((1, 2, 5), np.float32)), w, 5, 1, ops.RNN_TANH, False)   # cell state without LSTM
    with pytest.raises(ValueError):
        ops.rnn(x, None, None, w, 5, 1, ops.RNN_TANH, False, dropout=1.5)   # not a probability
    y, hy, cy, reserve = ops.rnn(x, None, None, w, 5, 1, ops.RNN_TANH, False)
    with pytest.raises(ValueError):
        ops.rnn_backward(x, w, None, 5, 1, ops.RNN_TANH, False, y)           # no payload


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("I,H,L,bidir,T,B,p", [
    (4, 3, 3, True, 5, 2, 0.5),            # the two-kernel steps
    (10, 48, 2, True, 5, 33, 0.3),         # the fused step kernels
    (40, 64, 3, False, 12, 8, 0.2),
    (5, 7, 2, False, 3, 1, 0.7),
])
def test_rnn_dropout_between_layers(mode, I, H, L, bidir, T, B, p):
    """Dropout on the output sequence of every layer but the last (backend/cudnn/RNN.cpp:83-90):
    same mask (a function of the seed) and scale as the CPU checker, forward and backward;
    another seed gives another result, one layer ignores the setting."""
    rng = np.random.default_rng(2000 * mode + I + H + L + T)
    D = 2 if bidir else 1
    seed = 0xC0FFEE1234567
    d = flref.rnn_desc(I, H, L, bidir, mode, T, B, dropout=p, seed=seed)
    w = (rng.standard_normal(flref.rnn_param_count(d)) / np.sqrt(H)).astype(np.float32)
    x = rng.standard_normal((T, B, I)).astype(np.float32)
    hx = rng.standard_normal((L * D, B, H)).astype(np.float32)
    cx = rng.standard_normal((L * D, B, H)).astype(np.float32) if mode == flref.RNN_LSTM else None
    dy = rng.standard_normal((T, B, D * H)).astype(np.float32)
    dhy = rng.standard_normal((L * D, B, H)).astype(np.float32)
    dcy = rng.standard_normal((L * D, B, H)).astype(np.float32) if mode == flref.RNN_LSTM else None
    ry, rhy, rcy = flref.rnn_fwd(d, x, w, hx, cx)
    rdx, rdhx, rdcx, rdw = flref.rnn_bwd(d, x, w, hx, cx, dy, dhy, dcy)

    o = lambda a: None if a is None else dev(a)
    y, hy, cy, reserve = ops.rnn(dev(x), o(hx), o(cx), dev(w), H, L, mode, bidir, dropout=p, seed=seed)
    assert rel_l2(host(y), ry) <= 1e-4 and rel_l2(host(hy), rhy) <= 1e-4
    if mode == flref.RNN_LSTM:
        assert rel_l2(host(cy), rcy) <= 1e-4
    dx, dhx, dcx, dw = ops.rnn_backward(dev(x), dev(w), reserve, H, L, mode, bidir, dev(dy), dev(dhy), o(dcy),
                                        dropout=p, seed=seed)
    assert rel_l2(host(dx), rdx) <= 2e-4
    assert rel_l2(host(dhx), rdhx) <= 2e-4
    assert rel_l2(host(dw), rdw) <= 2e-4
    if mode == flref.RNN_LSTM:
        assert rel_l2(host(dcx), rdcx) <= 2e-4
    y2 = ops.rnn(dev(x), o(hx), o(cx), dev(w), H, L, mode, bidir, dropout=p, seed=seed + 1)[0]
    assert rel_l2(host(y2), ry) > 1e-3
    y3 = ops.rnn(dev(x), o(hx), o(cx), dev(w), H, L, mode, bidir, dropout=p, seed=seed)[0]
    assert torch.equal(y3, y)


def test_rnn_dropout_needs_more_than_one_layer_and_a_valid_probability():
    x = dev(np.zeros((3, 2, 4), np.float32))
    w = dev(np.zeros(ops.rnn_param_count(4, 5, 1, flref.RNN_GRU, False), np.float32))
    a = ops.rnn(x, None, None, w, 5, 1, flref.RNN_GRU, False)[0]
    b = ops.rnn(x, None, None, w, 5, 1, flref.RNN_GRU, False, dropout=0.9, seed=3)[0]
    assert torch.equal(a, b)
    with pytest.raises(ValueError):
        ops.rnn(x, None, None, w, 5, 1, flref.RNN_GRU, False, dropout=1.0)
