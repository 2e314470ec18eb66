"""fp32 depthwise on column runs from LDS: bit-exact against the oracle at the
edges of its runs, bands and plane groups."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import nhip  # noqa: E402
from oracle import refcpu  # noqa: E402

pytestmark = pytest.mark.gpu

CASES = [
    # (n, c, h, w, kernel, stride, pad(t,b,l,r), offset of the input in elements)
    (1, 1, 1, 1, 5, 1, (2, 2, 2, 2), 0),
    (2, 5, 7, 7, 3, 1, (1, 1, 1, 1), 1),         # one run a column, several planes a workgroup
    (2, 300, 9, 6, 5, 1, (2, 2, 2, 2), 0),       # two runs, two planes a workgroup
    (1, 3, 61, 75, 3, 1, (1, 1, 1, 1), 2),       # bands
    (1, 4, 75, 130, 5, 2, (2, 2, 2, 2), 3),      # bands, stride 2
    (1, 2, 130, 113, 5, 1, (0, 4, 1, 3), 0),     # a plane above the staging size
    (2, 9, 4, 3, 5, 2, (4, 2, 6, 5), 0),         # windows wholly outside the image
    (1, 2, 16, 900, 3, 1, (1, 1, 1, 1), 1),      # wide rows: bands of one run
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:6])))
@pytest.mark.parametrize("act", [0, 1])
def test_dw_runs_bit_exact(case, act, nhip_env):
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    nhip.init(0)
    nhip_env.setenv("NHIP_DW_RUNS", "2")
    n, c, h, w, ker, s, pad, off = case
    rng = np.random.default_rng([n, c, h, w, ker, s])
    flat = rng.standard_normal(n * c * h * w + off).astype(np.float32)
    flat[off] = np.inf
    wt = rng.standard_normal((c, 1, ker, ker)).astype(np.float32)
    b = rng.standard_normal(c).astype(np.float32)
    d = nhip.conv_desc(c, c, (ker, ker), (s, s), pad=pad, act=act, group=c)
    nhip.timer_start("dw_f32_runs")
    got = nhip.DwConv2dF32(d, wt, b).forward(torch.from_numpy(flat).cuda()[off:].view(n, c, h, w)).cpu().numpy()
    assert nhip.timer_stop()[0] == 1
    with np.errstate(all="ignore"):
        exp = refcpu.dwconv2d_f32(refcpu.geom(n, c, h, w, c, (ker, ker), (s, s), (1, 1), pad),
                                  flat[off:].reshape(n, c, h, w), wt, b)
        exp = refcpu.relu_f32(exp) if act else exp
    np.testing.assert_array_equal(got, exp)


@pytest.mark.parametrize("n,c,h,w", [(3, 200, 1040, 1040), (2, 300, 1037, 1041)])
def test_wide_rows_past_32_bit_offsets(n, c, h, w):
    """Rows that the column runs cannot stage in a tensor past 2 GiB: whole images at a time on the window kernel,
    bit for bit what it gives on one image's half of the channels."""
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    nhip.init(0)
    rng = np.random.default_rng([n, c, w])
    wt, b = rng.standard_normal((c, 1, 3, 3)).astype(np.float32), rng.standard_normal(c).astype(np.float32)

    def plan(lo, hi):
        return nhip.DwConv2dF32(nhip.conv_desc(hi - lo, hi - lo, act=1, group=hi - lo), wt[lo:hi], b[lo:hi])

    x = torch.randn((n, c, h, w), device="cuda")
    assert x.numel() * 4 >= 2 ** 31
    nhip.timer_start("dw3x3s")
    got = plan(0, c).forward(x)
    assert nhip.timer_stop()[0] == 2
    for i in range(n):
        for lo, hi in ((0, c // 2), (c // 2, c)):
            assert torch.equal(got[i:i + 1, lo:hi], plan(lo, hi).forward(x[i:i + 1, lo:hi].contiguous()))
