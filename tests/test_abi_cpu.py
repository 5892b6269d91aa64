"""CPU-side checks of the C ABI: the library loads, exports every symbol the
header declares, and the argument checks that need no GPU behave as documented."""
import ctypes as C
import os
import re

import pytest

from flashlight_amd import capi
from flashlight_amd.ops import bn_view, derive_padding

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_header_symbols_are_exported_and_bound():
    text = open(os.path.join(ROOT, "include", "flhip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    declared = set(re.findall(r"\b(flhip_[a-z0-9_]+)\s*\(", text))
    assert declared, "no declarations parsed"
    lib = capi.lib()
    for name in declared:
        assert hasattr(lib, name), name
    assert declared == set(capi.SYMBOLS)


@pytest.mark.parametrize("I,H,L,bidir,mode,T,B", [(512, 512, 2, 1, 2, 200, 32), (1024, 1024, 2, 1, 2, 1000, 64), (320, 512, 1, 0, 1, 400, 64),
                                                  (1024, 1024, 1, 0, 3, 100, 64)])
def test_sequence_launches_take_no_workspace_of_their_own(I, H, L, bidir, mode, T, B):
    """What the backward pass of a recurrent layer holds: the gate gradients twice per direction, the gradients of the output and (two
    buffers) of the widest input, for every step; beyond that at most twice 16 partial products of the largest weights' gradient and 1 MiB."""
    d = capi.RnnDesc(I, H, L, bidir, mode, T, B, capi.F32)
    D, G = 1 + bidir, {1: 1, 2: 4, 3: 3}[mode]
    widest = max(I, D * H)
    held = T * B * (2 * D * G * H + D * H + 2 * widest)
    assert 4 * held <= capi.lib().flhip_rnn_workspace_bytes(C.byref(d)) <= 4 * (held + 2 * 16 * G * H * widest) + (1 << 20)


@pytest.mark.parametrize("C_,W,K,kw,left", [(320, 60, 32, 9, False), (320, 200, 320, 9, False), (320, 1500, 640, 9, True), (256, 60, 32, 9, True),
                                            (320, 200, 320, 21, False), (320, 1500, 320, 21, True), (260, 1500, 320, 9, True)])
def test_one_row_layers_that_leave_their_rows(C_, W, K, kw, left):
    """fp32 layers of one-row windows leave their channels-last rows to the filter gradient, those of more than 256 channels where both passes have the
    tiles and products for the kernels that use them; no room is asked for otherwise."""
    d = capi.ConvDesc(1, C_, 1, W, K, 1, kw, 1, 1, 0, kw // 2, 1, 1, 1, capi.F32)
    rows = capi.lib().flhip_conv2d_gathered_bytes(C.byref(d))
    assert (rows > 0) == left
    assert rows <= capi.lib().flhip_conv2d_workspace_bytes(C.byref(d), capi.CONV_FWD)


def test_layer_geometry_is_kept_by_value():
    """Whatever can be an index is taken as one: arrays of one element, which have no hash, and tensors, whose hash is their identity."""
    import numpy as np
    import torch
    from flashlight_amd import ops
    plan = lambda s, x=(2, 3, 9, 9): ops._conv_plan(x, (4, 3, 3, 3), s, 1, 1, 1, 1, 1, 1, capi.F32)[2]
    stride = torch.tensor(1)
    assert plan(2) == plan(np.array(2)) == plan(np.int64(2)) == (2, 4, 9, 5) and plan(stride) == plan(True) == (2, 4, 9, 9)
    stride.fill_(2)
    assert plan(stride) == plan(2, tuple(np.array([2, 3, 9, 9]))) == plan(2, tuple(torch.tensor([2, 3, 9, 9]))) == (2, 4, 9, 5)
    with pytest.raises(TypeError):
        plan(2.0)
    with pytest.raises(ValueError):
        plan(1, (2, 5, 9, 9))


def test_version_and_arch():
    text = open(os.path.join(ROOT, "include", "flhip.h")).read()
    declared = int(re.search(r"#define\s+FLHIP_VERSION\s+(\d+)", text).group(1))
    assert capi.lib().flhip_version() == declared >= 200
    assert capi.lib().flhip_arch() == b"gfx950"


def test_convert_many_launch_split():
    """How flhip_convert_many cuts a list of tensors into launches: 64 tensors or 2^31 - 1
    pieces of 2048 elements per launch, whichever comes first; empty tensors take no slot."""
    lib = capi.lib()

    def plan(sizes):
        n = (C.c_size_t * len(sizes))(*sizes)
        where = (C.c_int32 * len(sizes))()
        launches = lib.flhip_convert_many_launches(n, len(sizes), where)
        return launches, list(where)

    assert plan([]) == (0, [])
    assert plan([0, 0]) == (0, [-1, -1])
    assert plan([5] * 64) == (1, [0] * 64)
    assert plan([5] * 65) == (2, [0] * 64 + [1])
    assert plan([5, 0] * 65)[0] == 2
    big = (1 << 40) - 1                       # 2^29 pieces
    launches, where = plan([big] * 9)         # three fit under 2^31 - 1, the fourth does not
    assert launches == 3 and where == [0, 0, 0, 1, 1, 1, 2, 2, 2]
    # exactly the grid limit fits, one more piece does not
    limit = (1 << 31) - 1
    rest = limit - 3 * (1 << 29)
    assert plan([big] * 3 + [rest * 2048])[0] == 1
    assert plan([big] * 3 + [rest * 2048 + 1])[0] == 2
    assert plan([1 << 40])[0] == -1           # refused, like the call itself


def test_layernorm_row_limits():
    """Rows that the row kernels take: up to 16 KiB, and no more of them than their int row counters can step past."""
    applies = capi.lib().flhip_layernorm_applies
    assert applies(4096, 1, capi.F32) and not applies(4097, 1, capi.F32)
    assert applies(8192, 1, capi.BF16) and not applies(8193, 1, capi.F16)
    assert applies(2, 1 << 30, capi.BF16) and not applies(2, (1 << 30) + 1, capi.BF16)
    assert not applies(2, (1 << 31) - 1, capi.BF16)
    assert applies(1, 1 << 14, capi.F32) and not applies(1, (1 << 14) + 1, capi.F32)
    assert not applies(0, 4, capi.F32) and not applies(4, 0, capi.F32) and not applies(4, 4, 17)


def test_layernorm_backward_slices():
    """Partial sums of the backward pass (and one more row of them): a workgroup to each of few long rows."""
    ws = capi.lib().flhip_layernorm_bwd_workspace_bytes
    for n, rows, slices in ((6590, 5, 5), (2000, 4000, 512), (1025, 30, 30), (1024, 30, 7), (29, 3, 1)):
        assert ws(n, rows, capi.F16) == (slices + 1) * 2 * n * 4, (n, rows)


def test_thin_products_cut_only_long_contractions():
    """Workspace for the slices of A * B with few columns: only where a second launch pays for itself."""
    ws = capi.lib().flhip_matmul_slices_bytes
    for m, n, k in ((512, 64, 704), (512, 8, 704), (3996, 45, 352)):                              # the last: two rounds of workgroups
        assert ws(m, n, k - 4, 0, 0, capi.F32) == 0 and ws(m, n, k, 0, 0, capi.F32) > 0
    assert ws(512, 64, 512, 1, 0, capi.F32) > 0                                                   # A^T * B: always the faster one


@pytest.mark.parametrize("n,c,k,plane,thin", [(1, 256, 64, 7, True), (1, 256, 64, 4, False), (1, 2048, 512, 7, True), (1, 128, 512, 4, False),
                                              (1, 512, 1024, 7, True), (1, 512, 1024, 4, False), (24, 2048, 1000, 1, True),
                                              (25, 2048, 1000, 1, False), (1, 1024, 2048, 4, False)])
def test_1x1_windows_with_few_tiles(n, c, k, plane, thin):
    """Which fp32 forward passes of 1x1 windows take the kernels for few tiles (they copy the weights to the workspace)."""
    d = capi.ConvDesc(n, c, plane, plane, k, 1, 1, 1, 1, 0, 0, 1, 1, 1, capi.F32)
    assert (capi.lib().flhip_conv2d_workspace_bytes(C.byref(d), capi.CONV_FWD) > 0) == thin


@pytest.mark.parametrize("n,c,t,k,kw,stride,dtype,parts", [
    (31, 16, 193, 64, 7, 1, capi.BF16, 31), (4, 64, 1017, 40, 15, 2, capi.F16, 32), (9, 64, 603, 100, 9, 1, capi.BF16, 72),
    (17, 97, 400, 193, 6, 1, capi.F16, 272), (17, 80, 985, 384, 8, 2, capi.BF16, 306), (7, 250, 1111, 250, 21, 1, capi.BF16, 224),
    (16, 128, 1500, 128, 21, 1, capi.BF16, 256), (7, 80, 200, 250, 21, 1, capi.F32, 336)])
def test_one_row_filter_gradient_partial_tiles(n, c, t, k, kw, stride, dtype, parts):
    """How many partial tiles (one per workgroup) the filter gradient of one-row windows leaves in its workspace, behind the
    channels-last rows: as many as their own cost is worth, in 16-bit storage more than the 256 compute units only for long
    ranges and few taps."""
    d = capi.ConvDesc(n, c, 1, t, k, 1, kw, 1, stride, 0, kw // 2, 1, 1, 1, dtype)
    cs = min(v for v in (32, 64, 96, 128, 256) if c <= v)
    rows = (n * t * cs * (4 if dtype == capi.F32 else 2) + 255) // 256 * 256
    tile = (kw + 4) // 4 * 4 * 2048 * 4
    assert capi.lib().flhip_conv2d_workspace_bytes(C.byref(d), capi.CONV_BWD_FILTER) == rows + parts * tile


def test_conv_out_dims_and_errors():
    lib = capi.lib()
    oh, ow = C.c_int32(), C.c_int32()
    d = capi.ConvDesc(32, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1, 1, 1, 1, capi.F32)
    assert lib.flhip_conv2d_out_dims(C.byref(d), C.byref(oh), C.byref(ow)) == capi.OK
    assert (oh.value, ow.value) == (56, 56)
    d = capi.ConvDesc(64, 3, 224, 224, 64, 7, 7, 2, 2, 3, 3, 1, 1, 1, capi.F32)
    assert lib.flhip_conv2d_out_dims(C.byref(d), C.byref(oh), C.byref(ow)) == capi.OK
    assert (oh.value, ow.value) == (112, 112)
    bad = capi.ConvDesc(1, 3, 8, 8, 4, 3, 3, 1, 1, 0, 0, 1, 1, 2, capi.F32)   # groups !| C
    assert lib.flhip_conv2d_out_dims(C.byref(bad), C.byref(oh), C.byref(ow)) == capi.INVALID_ARGUMENT
    with pytest.raises(ValueError):
        capi.check(capi.INVALID_ARGUMENT)
    assert b"groups" in lib.flhip_last_error()
    bad = capi.ConvDesc(1, 3, 2, 2, 4, 5, 5, 1, 1, 0, 0, 1, 1, 1, capi.F32)   # kernel > input
    assert lib.flhip_conv2d_out_dims(C.byref(bad), C.byref(oh), C.byref(ow)) == capi.INVALID_ARGUMENT


def test_pool_out_dims_and_errors():
    lib = capi.lib()
    oh, ow = C.c_int32(), C.c_int32()
    d = capi.PoolDesc(32, 64, 112, 112, 3, 3, 2, 2, 1, 1, 0, capi.F32)
    assert lib.flhip_pool2d_out_dims(C.byref(d), C.byref(oh), C.byref(ow)) == capi.OK
    assert (oh.value, ow.value) == (56, 56)
    bad = capi.PoolDesc(1, 1, 8, 8, 2, 2, 2, 2, 2, 2, 0, capi.F32)            # pad >= window
    assert lib.flhip_pool2d_out_dims(C.byref(bad), C.byref(oh), C.byref(ow)) == capi.INVALID_ARGUMENT
    bad = capi.PoolDesc(1, 1, 8, 8, 2, 2, 2, 2, 0, 0, 7, capi.F32)            # unknown mode
    assert lib.flhip_pool2d_out_dims(C.byref(bad), C.byref(oh), C.byref(ow)) == capi.INVALID_ARGUMENT


def test_null_arguments_are_rejected_before_any_launch():
    lib = capi.lib()
    d = capi.PoolDesc(1, 1, 8, 8, 2, 2, 2, 2, 0, 0, 0, capi.F32)
    assert lib.flhip_pool2d_fwd(C.byref(d), None, None, None, None) == capi.INVALID_ARGUMENT
    # max-pool backward without the forward argmax: the reference throws
    # std::invalid_argument (onednn/Pool2D.cpp:190-193)
    assert lib.flhip_pool2d_bwd(C.byref(d), C.c_void_p(16), None, C.c_void_p(16), None) == capi.INVALID_ARGUMENT
    b = capi.BnDesc(4, 3, 10, capi.F32)
    assert lib.flhip_bn_workspace_bytes(C.byref(b)) > 0
    assert lib.flhip_bn_bwd(C.byref(b), C.c_void_p(16), C.c_void_p(16), None, None, None,
                            C.c_void_p(16), None, None, None, 0, None) == capi.INVALID_ARGUMENT
    assert lib.flhip_copy_bytes(C.c_void_p(16), C.c_void_p(32), 24, None) == capi.INVALID_ARGUMENT


def test_bn_view_and_same_padding():
    assert bn_view((8, 3, 13, 13), [2]) == (8, 3, 169)
    assert bn_view((8, 4, 13, 13), [0, 1, 2]) == (8, 676, 1)
    with pytest.raises(ValueError):
        bn_view((8, 4, 13, 13), [0, 2])
    # fl::derivePadding (flashlight/fl/nn/Utils.cpp:87-100)
    assert derive_padding(56, 3, 1, -1) == 1
    assert derive_padding(224, 7, 2, -1) == 3
    assert derive_padding(56, 1, 2, -1) == 0
    assert derive_padding(1500, 21, 1, -1) == 10
    assert derive_padding(1500, 21, 2, -1) == 10
    assert derive_padding(28, 5, 1, -1) == 2
    assert derive_padding(112, 3, 2, -1) == 1
    assert derive_padding(9, 3, 1, 4) == 4


def test_plan_lists():
    """The kernel families of the backward passes have names; the forward pass has no plans."""
    lib = capi.lib()
    for pas in (capi.CONV_BWD_DATA, capi.CONV_BWD_FILTER):
        n = lib.flhip_conv2d_plan_count(pas)
        assert n >= 2
        names = [lib.flhip_conv2d_plan_name(pas, i) for i in range(n)]
        assert all(names) and len(set(names)) == n
        assert lib.flhip_conv2d_plan_name(pas, n) is None and lib.flhip_conv2d_plan_name(pas, -1) is None
    assert lib.flhip_conv2d_plan_count(capi.CONV_FWD) == 0
