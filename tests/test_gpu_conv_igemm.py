"""fp32 convolutions with short reductions on the fp32 implicit GEMM, against
64-bit sums: the edges of its 64 x 64 tiles and of its stages of 16, pixels
across images, planes that are no multiple of four; and which kernel a launch
takes on either side of each line of the rule.

Bound: a chain of n fp32 products and sums, n + 2 roundings of 2^-24 of
sum |x w|, and the epilogue's of the result."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import nhip  # noqa: E402
from oracle import refcpu  # noqa: E402
from test_gpu_conv_split import data, sums64  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    nhip.init(0)


def run(case, x, wt, b, res, kernel="conv_igemm"):
    n, c, h, w, k, ker, st, dl, pad, _, act = case
    plan = nhip.Conv2dF32(nhip.conv_desc(c, k, ker, st, dl, pad, act=act), wt, b)
    nhip.timer_start(kernel)
    got = plan.forward(torch.from_numpy(x).cuda(), residual=None if res is None else torch.from_numpy(res).cuda())
    return got.cpu().numpy(), nhip.timer_stop()[0]


CASES = [
    # (n, c, h, w, k, kernel, stride, dilation, pad(t,b,l,r), residual, act)
    (1, 1, 1, 1, 1, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), False, 0),       # one pixel, one channel
    (1, 1, 9, 7, 64, (1, 3), (1, 1), (1, 1), (0, 0, 1, 1), True, 1),       # 63 pixels, a whole tile of channels
    (3, 3, 15, 13, 65, (3, 3), (2, 2), (1, 1), (1, 1, 1, 1), True, 4),     # two stages; pixels across images
    (5, 1, 8, 8, 33, (4, 4), (1, 1), (1, 1), (2, 1, 2, 1), True, 0),       # one whole stage, whole vectors
    (1, 2, 20, 31, 40, (5, 5), (1, 2), (2, 1), (3, 4, 0, 1), False, 1),    # 50 products, dilation
    (2, 4, 11, 12, 130, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), True, 0),    # three stages
    (3, 9, 40, 34, 130, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), True, 1),    # 81 products, six stages
    (2, 10, 39, 39, 200, (1, 11), (1, 1), (1, 1), (0, 0, 5, 5), False, 0),  # 110 products, seven stages
    (3, 16, 23, 21, 48, (1, 1), (2, 2), (1, 1), (0, 0, 0, 0), True, 1),    # 1x1 with a stride: whole octets
    (2, 48, 60, 99, 240, (1, 1), (2, 1), (1, 1), (0, 0, 0, 0), False, 1),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])) + "k" + "x".join(map(str, c[5])))
def test_short_reductions_against_64_bits(case):
    x, wt, b, res = data(case, [CASES.index(case), 8])
    got, launches = run(case, x, wt, b, res)
    assert launches == 1
    s, m = sums64(case, x, wt)
    exp = s + b.astype(np.float64)[None, :, None, None] + (0 if res is None else res.astype(np.float64))
    if case[-1] == 1:
        exp = np.maximum(exp, 0)
    if case[-1] == 4:
        exp = 1 / (1 + np.exp(-exp))
    bound = m * 2.0 ** -24 * (wt[0].size + 2) + 2.0 ** -22 * (np.abs(exp) + 4)
    assert np.all(np.abs(got - exp) <= bound)


def test_non_finite_values():
    case = CASES[2][:-2] + (False, 0)
    x, wt, b, _ = data(case, 78)
    x.reshape(-1)[[5, 130, 400, 777]] = [np.inf, -np.inf, np.nan, 3.4e38]
    wt.reshape(-1)[::7] = 0.0  # 0 * inf
    got, launches = run(case, x, wt, b, None)
    assert launches == 1
    n, c, h, w, k, ker, st, dl, pad, _, _ = case
    with np.errstate(all="ignore"):
        exp = refcpu.conv2d_f32(refcpu.geom(n, c, h, w, k, ker, st, dl, pad), x, wt, b)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(exp))
    np.testing.assert_array_equal(got[np.isinf(exp)], exp[np.isinf(exp)])
    fin = np.isfinite(exp)
    np.testing.assert_allclose(got[fin], exp[fin], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("n,c,h,w,k,ker,st,kernel", [
    (1, 3, 64, 64, 32, 3, 2, "conv_igemm"),      # a small stem
    (32, 3, 96, 96, 32, 3, 2, "conv_smallk"),    # four blocks per CU
    (32, 3, 96, 96, 33, 3, 2, "conv_igemm"),     # 33 channels: not on the one-block kernel
    (2, 3, 80, 83, 64, 5, 2, "conv_split"),      # 75 products by the table, 53 tiles
    (2, 3, 160, 162, 64, 5, 2, "conv_igemm"),    # 203 tiles
    (2, 3, 160, 162, 32, 5, 2, "conv_split"),    # few output channels
    (1, 12, 50, 50, 64, 1, 2, "conv_split"),     # one octet and a half, 10 tiles
    (2, 12, 150, 150, 64, 1, 2, "conv_igemm"),   # 176 tiles
    (1, 12, 50, 50, 48, 1, 2, "conv_igemm"),     # up to 48 channels
    (2, 24, 150, 150, 64, 1, 2, "conv_igemm"),   # 24 products, 176 tiles
    (2, 72, 150, 150, 64, 1, 2, "conv_split"),   # 72 products: from three tiles per two CUs
])
def test_which_kernel(n, c, h, w, k, ker, st, kernel):
    case = (n, c, h, w, k, (ker, ker), (st, st), (1, 1), (ker // 2,) * 4, False, 0)
    x, wt, b, _ = data(case, 3)
    got, launches = run(case, x, wt, b, None, kernel)
    assert launches == 1
    ref = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(wt).double(),
                                     torch.from_numpy(b).double(), stride=st, padding=ker // 2).numpy()
    assert np.linalg.norm(got - ref) <= 1e-6 * np.linalg.norm(ref)
