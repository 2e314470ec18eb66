"""The int8 convolution's window kernel at the edges of its tiles: rows shorter
than a fill group, column segments with a ragged last one, stride-1 1x1 layers
and 1x1 planes as one row of pixels, one-row kernels with a stride, channel counts that are no
multiple of 4, 16 or 32, and every split of a workgroup into channel blocks and
reduction parts.  Integer sums and separately rounded fp32 steps: bit for bit
against the oracle, and the same from the gather kernel."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import nhip  # noqa: E402
from test_gpu_int8 import _gpu, dev, host, oracle, run  # noqa: E402,F401

pytestmark = pytest.mark.gpu

CASES = [
    # (n, c, h, w, k, kernel, stride, dil, pad, term, act)
    (2, 5, 6, 3, 33, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 101, 1),      # rows of 3 pixels
    (1, 7, 5, 1, 1, (3, 1), (1, 1), (1, 1), (1, 1, 0, 0), 1, 0),         # rows of 1 pixel, one channel
    (2, 3, 9, 150, 32, (3, 3), (2, 2), (1, 1), (1, 1, 1, 1), 101, 0),    # 75 columns, three input channels
    (1, 18, 5, 261, 40, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 102, 1),   # column segments, last one ragged
    (1, 18, 5, 261, 40, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 2, 1),
    (3, 34, 19, 17, 65, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), 101, 1),   # 1x1: 323 pixels as one row
    (1, 64, 1, 2, 96, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), 1, 1),       # 1x1: two pixels
    # 1x1 planes: the images as one row of pixels, 16-channel groups with a remainder
    (133, 50, 1, 1, 70, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), 1, 1),
    (37, 64, 1, 1, 33, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), 101, 0),
    (1, 9, 1, 1, 5, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), 102, 1),
    (2, 48, 13, 11, 70, (1, 1), (2, 2), (1, 1), (0, 0, 0, 0), 101, 0),   # 1x1 with a stride: every second row
    (1, 20, 9, 9, 32, (1, 3), (3, 1), (1, 1), (2, 2, 1, 1), 1, 0),       # one-row kernel, padded rows
    (1, 16, 12, 40, 24, (5, 5), (2, 2), (2, 2), (4, 4, 4, 4), 101, 1),   # dilated, padding wider than a group
    (1, 600, 14, 12, 32, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 101, 0),  # deep: few pixels per window
    (2, 109, 20, 19, 40, (5, 5), (2, 2), (1, 1), (2, 2, 2, 2), 101, 1),  # seven chunks of channels per pixel, unpadded
    (1, 1500, 9, 30, 32, (5, 5), (2, 2), (1, 1), (2, 2, 2, 2), 1, 0),    # no window fits: the gather kernel
]
CFGS = ["", "1,32,1,1", "1,32,1,8", "2,16,2,2", "1,16,4,1", "3,32,1,4"]


def _layer(case, int8_in):
    n, c, h, w, k, ker, st, dl, pad, term, act = case
    rng = np.random.default_rng(sum(case[:5]) + term)
    x = (rng.integers(-128, 128, (n, c, h, w)).astype(np.int8) if int8_in
         else rng.uniform(-2.5, 2.5, (n, c, h, w)).astype(np.float32))
    wt = rng.integers(-127, 128, (k, c) + ker).astype(np.int8)
    scale = rng.uniform(20, 200, k).astype(np.float32)
    b = rng.normal(0, 0.3, k).astype(np.float32)
    # an output scale that uses the int8 range
    spread = 73.0 * 73.0 * np.sqrt(c * ker[0] * ker[1]) / (scale.mean() * 60.0)
    return nhip.conv_desc(c, k, ker, st, dl, pad, act=act, int8_scale_term=term), x, wt, b, scale, 60.0, 60.0 / spread


def _fits(cfg, case):
    """Whether the layer has the rows and columns of a split (a column segment is whole rows or sixteens)."""
    n, c, h, w, k, ker, st, dl, pad, _, _ = case
    oh = (h + pad[0] + pad[1] - dl[0] * (ker[0] - 1) - 1) // st[0] + 1
    ow = (w + pad[2] + pad[3] - dl[1] * (ker[1] - 1) - 1) // st[1] + 1
    if ker == (1, 1) and st == (1, 1):  # the image, or 1x1 planes' images, as one row
        oh, ow = 1, (n if h * w == 1 else h * w)
    r, cw = (int(v) for v in cfg.split(",")[:2])
    return r <= oh and cw <= ow and (cw == ow or cw % 16 == 0)


def _timed(layer):
    nhip.timer_start("conv_int8_win")
    got = run(*layer)
    return got, nhip.timer_stop()[0]


@pytest.mark.parametrize("int8_in", [True, False], ids=["i8", "f32"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])) + f"-t{c[9]}")
def test_window_kernel_bit_exact(case, int8_in, nhip_env):
    layer = _layer(case, int8_in)
    exp = oracle(*layer)
    window = case is not CASES[-1]
    for cfg in CFGS:
        if cfg and not _fits(cfg, case):
            continue
        nhip_env.setenv("NHIP_INT8_WIN_CFG", cfg)
        got, launches = _timed(layer)
        np.testing.assert_array_equal(got, exp, err_msg=f"split {cfg or 'chosen'}")
        assert launches == (1 if window else 0)
    nhip_env.setenv("NHIP_INT8_FOOTPRINT", "0")
    got, launches = _timed(layer)
    np.testing.assert_array_equal(got, exp, err_msg="gather kernel")
    assert launches == 0


@pytest.mark.parametrize("n,k,int8_in,window", [(13, 1, False, True), (14, 1, False, False), (21, 33, True, True),
                                               (22, 33, True, False), (53, 1, True, True)])
def test_sixteen_columns_leave_to_the_gather_kernel(n, k, int8_in, window):
    """640 channels leave room for 16 columns, 80 tiles an image: either side of the workgroups from which the gather
    kernel takes the layer; int8 with one channel block never leaves."""
    layer = _layer((n, 640, 16, 80, k, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 101, 1), int8_in)
    got, launches = _timed(layer)
    assert launches == (1 if window else 0)
    np.testing.assert_array_equal(got, oracle(*layer))


@pytest.mark.parametrize("int8_in", [True, False], ids=["i8", "f32"])
def test_unaligned_input_and_output(int8_in):
    """Tensors at odd element offsets: the kernel's wide loads and stores take any element alignment."""
    d, x, wt, b, scale, is_, os_ = _layer(CASES[5], int8_in)
    exp = oracle(d, x, wt, b, scale, is_, os_)
    conv = nhip.Conv2dInt8(d, wt, b, scale, is_, os_)
    xd = dev(x)
    flat = torch.empty(xd.numel() + 1, dtype=xd.dtype, device="cuda")
    src = flat[1:].view(xd.shape)
    src.copy_(xd)
    out = torch.empty(exp.size + 1, dtype=torch.int8, device="cuda")[1:].view(exp.shape)
    out.fill_(77)
    conv.forward(src, out=out)
    np.testing.assert_array_equal(host(out), exp)
