"""GPU parity of the int8 depthwise kernel that forms 4 x 4 outputs per thread
(3x3 and 5x5, stride 1 and 2) against the CPU oracle, bit for bit, at the
edges of its groups: extents off the group of four, bands of rows, several
planes per workgroup, windows past every side of the image."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import nhip  # noqa: E402
from oracle import refcpu  # noqa: E402

pytestmark = pytest.mark.gpu

CASES = [
    # (n, c, h, w, kernel, stride, pad(t,b,l,r), offset of the input in elements)
    (1, 1, 1, 1, 3, 1, (1, 1, 1, 1), 0),
    (2, 5, 7, 7, 5, 1, (2, 2, 2, 2), 0),        # several planes per workgroup
    (3, 300, 7, 9, 3, 1, (1, 1, 1, 1), 1),      # misaligned input, three planes per workgroup
    (1, 3, 112, 51, 3, 1, (1, 1, 1, 1), 0),     # bands of rows, odd width
    (1, 4, 75, 130, 5, 2, (2, 2, 2, 2), 3),     # bands, stride 2
    (2, 260, 13, 14, 3, 2, (0, 1, 1, 0), 0),
    (1, 2, 3, 2, 5, 1, (4, 2, 12, 9), 0),       # windows wholly outside the image
    (1, 2, 40, 1500, 3, 1, (1, 1, 0, 2), 2),    # a plane above the staging size
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:6])))
@pytest.mark.parametrize("in_i8,term,act", [(True, 101, 1), (False, 101, 0), (True, 1, 1), (False, 1, 0)])
def test_dw_int8_runs_bit_exact(case, in_i8, term, act):
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    nhip.init(0)
    n, c, h, w, ker, s, pad, off = case
    rng = np.random.default_rng([n, c, h, w, ker, s, int(in_i8), term])
    count = n * c * h * w
    flat = (rng.integers(-128, 128, count + off).astype(np.int8) if in_i8
            else rng.uniform(-1.5, 1.5, count + off).astype(np.float32))
    wq = rng.integers(-128, 128, (c, 1, ker, ker)).astype(np.int8)
    ws = rng.uniform(20, 200, c).astype(np.float32)
    b = rng.normal(0, 0.3, c).astype(np.float32)
    d = nhip.conv_desc(c, c, (ker, ker), (s, s), pad=pad, act=act, int8_scale_term=term, group=c)
    conv = nhip.DwConv2dInt8(d, wq, b, ws, 60.0, 25.0)
    x = torch.from_numpy(flat).cuda()[off:].view(n, c, h, w)
    nhip.timer_start("dwconv_int8_runs")
    got = conv.forward(x).cpu().numpy()
    assert nhip.timer_stop()[0] == 1
    g = refcpu.geom(n, c, h, w, c, (ker, ker), (s, s), (1, 1), pad)
    exp = refcpu.dwconv2d_int8(g, flat[off:].reshape(n, c, h, w), wq, b, ws, 60.0, 25.0, term, act)
    assert got.dtype == exp.dtype
    np.testing.assert_array_equal(got, exp)
