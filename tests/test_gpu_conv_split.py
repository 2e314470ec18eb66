"""fp32 Convolution on the split-operand implicit GEMM (every fp32 value as
three bf16 pieces) against the CPU oracle and against 64-bit sums: the edges
of its blocks (32 channels, 32 pixels, 8 and 16 input channels, ragged
reductions), each of its work splits, and non-finite values.

Bound against 64 bits: a sum of n products whose pieces drop terms below
2^-23 |x w| (a second piece is at most 2^-8 of the number, a third 2^-16: two
products of 2^-24) and whose accumulators round once per 16 products (unit
2^-24): 2^-23 + 2^-24 (n / 16 + 6 + parts) of sum |x w|, far above what is seen
and far below the fp32 chain's n 2^-24 for the long reductions here."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import nhip  # noqa: E402
from oracle import refcpu  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    nhip.init(0)


CASES = [
    # (n, c, h, w, k, kernel, stride, dilation, pad(t,b,l,r), residual, act)
    (1, 1, 1, 1, 1, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), False, 0),
    (2, 3, 19, 23, 33, (7, 7), (2, 2), (1, 1), (3, 3, 3, 3), True, 1),     # table order, pixels across images
    (3, 16, 9, 7, 65, (3, 3), (2, 2), (1, 1), (1, 1, 1, 1), False, 1),     # whole 16-channel steps
    (1, 21, 12, 10, 31, (3, 3), (1, 2), (2, 1), (2, 2, 1, 0), True, 0),    # ragged octet, dilation
    (2, 24, 8, 8, 64, (5, 5), (2, 2), (1, 1), (2, 2, 2, 2), True, 4),      # whole octets, sigmoid
    (1, 9, 11, 13, 5, (2, 3), (1, 1), (1, 1), (0, 1, 2, 0), False, 0),     # channels padded by more than a third
    (1, 600, 4, 5, 40, (1, 1), (2, 2), (1, 1), (0, 0, 0, 0), True, 1),
    (1, 130, 6, 6, 20, (5, 5), (3, 3), (1, 1), (2, 2, 2, 2), False, 0),    # reduction in several launches' parts
    (5, 48, 21, 21, 130, (3, 3), (2, 2), (1, 1), (1, 1, 1, 1), True, 1),
]
CFGS = [None, "1,1,4,1", "1,2,3,2", "1,4,1,1", "2,1,8,3", "2,4,2,1", "1,1,16,5"]


def run(case, x, wt, b, res):
    n, c, h, w, k, ker, st, dl, pad, _, act = case
    d = nhip.conv_desc(c, k, ker, st, dl, pad, bias=True, act=act, algorithm=nhip.ALGO_IMPLICIT_GEMM)
    plan = nhip.Conv2dF32(d, wt, b)
    nhip.timer_start("conv_split_f32")
    got = plan.forward(torch.from_numpy(x).cuda(), residual=None if res is None else torch.from_numpy(res).cuda())
    launches = nhip.timer_stop()[0]
    return got.cpu().numpy(), launches


def data(case, seed):
    n, c, h, w, k, ker, st, dl, pad, with_res, _ = case
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    wt = (rng.standard_normal((k, c) + ker) * 0.3).astype(np.float32)
    oh = (h + pad[0] + pad[1] - dl[0] * (ker[0] - 1) - 1) // st[0] + 1
    ow = (w + pad[2] + pad[3] - dl[1] * (ker[1] - 1) - 1) // st[1] + 1
    res = rng.standard_normal((n, k, oh, ow)).astype(np.float32) if with_res else None
    return x, wt, rng.standard_normal(k).astype(np.float32), res


def sums64(case, x, wt):
    """(sum x w, sum |x w|) per output, in 64 bits."""
    n, c, h, w, k, ker, st, dl, pad, _, _ = case
    x = np.pad(x.astype(np.float64), ((0, 0), (0, 0), pad[:2], pad[2:]))
    oh = (x.shape[2] - dl[0] * (ker[0] - 1) - 1) // st[0] + 1
    ow = (x.shape[3] - dl[1] * (ker[1] - 1) - 1) // st[1] + 1
    s, m = np.zeros((n, k, oh, ow)), np.zeros((n, k, oh, ow))
    for i in range(ker[0]):
        for j in range(ker[1]):
            win = x[:, :, i * dl[0]:i * dl[0] + (oh - 1) * st[0] + 1:st[0],
                    j * dl[1]:j * dl[1] + (ow - 1) * st[1] + 1:st[1]]
            s += np.einsum("kc,nchw->nkhw", wt[:, :, i, j].astype(np.float64), win)
            m += np.einsum("kc,nchw->nkhw", np.abs(wt[:, :, i, j]).astype(np.float64), np.abs(win))
    return s, m


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])) + f"k{c[5][0]}s{c[6][0]}")
@pytest.mark.parametrize("cfg", CFGS)
def test_conv_split_against_64_bits(case, cfg, nhip_env):
    for name in ("NHIP_POINTWISE", "NHIP_CONV_KQ", "NHIP_GEMM_DMA", "NHIP_CONV_SMALLK"):
        nhip_env.setenv(name, "0")
    if cfg:
        nhip_env.setenv("NHIP_SPLIT_CFG", cfg)
    x, wt, b, res = data(case, [CASES.index(case), 5])
    got, launches = run(case, x, wt, b, res)
    assert launches == 1
    s, m = sums64(case, x, wt)
    exp = s + b.astype(np.float64)[None, :, None, None] + (0 if res is None else res.astype(np.float64))
    act = case[-1]
    if act == 1:
        exp = np.maximum(exp, 0)
    if act == 4:
        exp = 1 / (1 + np.exp(-exp))
    terms = wt[0].size
    bound = m * (2.0 ** -23 + 2.0 ** -24 * (terms / 16 + 6 + 16)) + 2.0 ** -22 * (np.abs(exp) + 4)
    assert np.all(np.abs(got - exp) <= bound)


@pytest.mark.parametrize("case", [CASES[1], CASES[2], CASES[3], CASES[7]], ids=lambda c: "x".join(map(str, c[:5])))
def test_conv_split_non_finite_values(case, nhip_env):
    """Infinities, NaN and values beyond bf16's range of rounding give what a
    plain fp32 sum gives, and touch no other output."""
    nhip_env.setenv("NHIP_CONV_KQ", "0")
    case = case[:-2] + (False, 0)
    x, wt, b, _ = data(case, 77)
    flat = x.reshape(-1)
    at = np.random.default_rng(1).choice(flat.size, 4, replace=False)
    flat[at] = [np.inf, -np.inf, np.nan, 3.4e38]
    wt.reshape(-1)[::7] = 0.0  # 0 * inf
    got, _ = run(case, x, wt, b, None)
    n, c, h, w, k, ker, st, dl, pad, _, _ = case
    with np.errstate(all="ignore"):
        exp = refcpu.conv2d_f32(refcpu.geom(n, c, h, w, k, ker, st, dl, pad), x, wt, b)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(exp))
    np.testing.assert_array_equal(got[np.isinf(exp)], exp[np.isinf(exp)])
    fin = np.isfinite(exp)
    np.testing.assert_allclose(got[fin], exp[fin], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("k", [33, 48, 64])
@pytest.mark.parametrize("n,c,h,w,ker", [(2, 3, 17, 23, 3), (3, 2, 9, 8, 4), (1, 1, 40, 31, 5)])
def test_short_reduction_two_channel_blocks(n, c, h, w, ker, k, nhip_env):
    """The short-reduction kernel's second block of 32 output channels: 33 to
    64 channels, ragged pixel blocks, residual."""
    nhip_env.setenv("NHIP_CONV_SMALLK", "2")
    case = (n, c, h, w, k, (ker, ker), (2, 2), (1, 1), (1, 1, 1, 1), True, 1)
    x, wt, b, res = data(case, [n, c, k])
    d = nhip.conv_desc(c, k, (ker, ker), (2, 2), act=1, algorithm=nhip.ALGO_IMPLICIT_GEMM)
    nhip.timer_start("conv_smallk")
    got = nhip.Conv2dF32(d, wt, b).forward(torch.from_numpy(x).cuda(), residual=torch.from_numpy(res).cuda())
    assert nhip.timer_stop()[0] == 1
    s, m = sums64(case, x, wt)
    exp = np.maximum(s + b[None, :, None, None].astype(np.float64) + res, 0)
    bound = m * 2.0 ** -24 * (wt[0].size + 2) + 2.0 ** -22 * (np.abs(exp) + 4)  # an fp32 chain of the products
    assert np.all(np.abs(got.cpu().numpy() - exp) <= bound)


# 3x3 stride-1 layers whose algorithm the library chooses: (n, c, h, w, k, taken by
# the split kernel).  17 input channels: padding them to eight adds over a third, so
# the reduction runs by the table of taps.
AUTO_CASES = [(2, 16, 9, 7, 40, True), (1, 17, 11, 13, 33, True), (3, 17, 8, 8, 16, True), (2, 18, 10, 6, 16, True),
              (1, 20, 12, 12, 48, True), (1, 33, 7, 9, 35, True), (1, 200, 6, 5, 130, True)]


def auto_layer(n, c, h, w, k, seed):
    rng = np.random.default_rng([n, c, h, w, k, seed])
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    wt = (rng.standard_normal((k, c, 3, 3)) * 0.3).astype(np.float32)
    b, res = rng.standard_normal(k).astype(np.float32), rng.standard_normal((n, k, h, w)).astype(np.float32)
    return x, wt, b, res, nhip.Conv2dF32(nhip.conv_desc(c, k, act=1), wt, b)


@pytest.mark.parametrize("n,c,h,w,k,taken", AUTO_CASES)
def test_chosen_algorithm_against_64_bits(n, c, h, w, k, taken):
    x, wt, b, res, plan = auto_layer(n, c, h, w, k, 3)
    nhip.timer_start("conv_split_f32")
    got = plan.forward(torch.from_numpy(x).cuda(), residual=torch.from_numpy(res).cuda()).cpu().numpy()
    assert nhip.timer_stop()[0] == (1 if taken else 0)
    s, m = sums64((n, c, h, w, k, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), True, 1), x, wt)
    exp = np.maximum(s + b.astype(np.float64)[None, :, None, None] + res, 0)
    bound = m * (2.0 ** -23 + 2.0 ** -24 * (wt[0].size / 16 + 6 + 16)) + 2.0 ** -22 * (np.abs(exp) + 4)
    assert np.all(np.abs(got - exp) <= bound)


# either side of each line of the rule that leaves the Winograd kernels (GFLOP of the direct convolution)
AUTO_LINES = [(1, 32, 137, 140, 72, True), (1, 32, 139, 140, 72, False),      # 0.795, 0.807
              (1, 176, 78, 79, 64, True), (1, 176, 79, 79, 64, False),        # 1.249, 1.265: 176 or more input channels
              (1, 168, 70, 72, 64, False),                                    # 0.975, fewer
              (1, 64, 134, 134, 48, True), (1, 64, 135, 135, 48, False),      # 0.993, 1.008: at most 48 output channels
              (1, 64, 120, 120, 56, False)]                                   # 0.929, more


@pytest.mark.parametrize("n,c,h,w,k,taken", AUTO_LINES)
def test_where_the_chosen_algorithm_leaves_winograd(n, c, h, w, k, taken):
    x, wt, b, res, plan = auto_layer(n, c, h, w, k, 4)
    nhip.timer_start("conv_split_f32")
    got = plan.forward(torch.from_numpy(x).cuda(), residual=torch.from_numpy(res).cuda()).cpu().double()
    assert nhip.timer_stop()[0] == (1 if taken else 0)
    ref = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(wt).double(),
                                     torch.from_numpy(b).double(), padding=1)
    ref = (ref + torch.from_numpy(res).double()).clamp_min(0)
    # normwise: the sums above, or Winograd F(4,3), whose transforms lose about four bits
    assert ((got - ref).norm() / ref.norm()).item() < (1e-6 if taken else 6e-6)


@pytest.mark.parametrize("c", [17, 24])
def test_chosen_algorithm_non_finite_values(c):
    n, h, w, k = 2, 9, 8, 40
    x, wt, b, _, _ = auto_layer(n, c, h, w, k, 5)
    plan = nhip.Conv2dF32(nhip.conv_desc(c, k), wt, b)
    x.reshape(-1)[[3, 200, 555, 1100]] = [np.inf, -np.inf, np.nan, 3.4e38]
    nhip.timer_start("conv_split_f32")
    got = plan.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    assert nhip.timer_stop()[0] == 1
    with np.errstate(all="ignore"):
        exp = refcpu.conv2d_f32(refcpu.geom(n, c, h, w, k, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)), x, wt, b)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(exp))
    np.testing.assert_array_equal(got[np.isinf(exp)], exp[np.isinf(exp)])
    fin = np.isfinite(exp)
    np.testing.assert_allclose(got[fin], exp[fin], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("c", [1, 5, 6, 7, 8, 9])
def test_fewer_channels_than_an_octet(c, nhip_env):
    """One image of 6 channels: eight channel planes are more than the whole tensor."""
    nhip_env.setenv("NHIP_CONV_SMALLK", "0")
    case = (1, c, 37, 41, 34, (5, 5), (2, 2), (1, 1), (2, 2, 2, 2), False, 0)
    x, wt, b, _ = data(case, [c, 9])
    got, launches = run(case, x, wt, b, None)
    assert launches == 1
    s, m = sums64(case, x, wt)
    bound = m * (2.0 ** -23 + 2.0 ** -24 * (wt[0].size / 16 + 6 + 16)) + 2.0 ** -22 * (np.abs(s) + 4)
    assert np.all(np.abs(got - (s + b.astype(np.float64)[None, :, None, None])) <= bound)


def test_remainder_of_sub_batches_has_its_workspace():
    """A batch past 2 GiB runs in sub-batches of whole images: 2674 of these and
    one more, which alone splits its reduction over the launch."""
    c, k, hw, n = 1024, 64, 14, 2675
    rng = np.random.default_rng(31)
    wt = (rng.standard_normal((k, c, 1, 1)) * 0.05).astype(np.float32)
    plan = nhip.Conv2dF32(nhip.conv_desc(c, k, (1, 1), pad=(0, 0, 0, 0)), wt, rng.standard_normal(k).astype(np.float32))
    assert plan.workspace_size(1, hw, hw) > 0
    x = torch.randn((n, c, hw, hw), device="cuda")
    got = plan.forward(x)
    assert torch.equal(got[-1:], plan.forward(x[-1:].clone()))
    assert torch.equal(got[:2], plan.forward(x[:2674])[:2])


@pytest.mark.parametrize("cfg", [None, "1,1,1,1", "2,1,2,1"])
def test_sums_of_one_product(cfg, nhip_env):
    """One product per sum, without the pieces' dropped terms: rounded once, as a fused multiply-add rounds it."""
    for name in ("NHIP_POINTWISE", "NHIP_CONV_KQ", "NHIP_GEMM_DMA", "NHIP_CONV_SMALLK"):
        nhip_env.setenv(name, "0")
    if cfg:
        nhip_env.setenv("NHIP_SPLIT_CFG", cfg)
    case = (2, 1, 33, 31, 70, (1, 1), (2, 2), (1, 1), (0, 0, 0, 0), False, 0)
    x, wt, b, _ = data(case, 41)
    got, launches = run(case, x, wt, b * 0, None)
    assert launches == 1
    s, _ = sums64(case, x, wt)
    np.testing.assert_array_equal(got, s.astype(np.float32))


@pytest.mark.parametrize("n,large,c,k,hw,ker", [(8, 32, 1024, 64, 14, 1), (1, 4, 128, 32, 52, 3)])
def test_workspace_of_a_larger_batch(n, large, c, k, hw, ker):
    """A launch whose parts do not fit the workspace that the largest batch needs runs in one part."""
    rng = np.random.default_rng(32)
    wt, b = (rng.standard_normal((k, c, ker, ker)) * 0.05).astype(np.float32), rng.standard_normal(k).astype(np.float32)
    plan = nhip.Conv2dF32(nhip.conv_desc(c, k, (ker, ker), pad=(ker // 2,) * 4), wt, b)
    x = torch.randn((n, c, hw, hw), device="cuda")
    need = plan.workspace_size(n, hw, hw)
    assert need > 0
    ref = torch.nn.functional.conv2d(x.cpu().double(), torch.from_numpy(wt).double(), torch.from_numpy(b).double(),
                                     padding=ker // 2)
    for size in {0, need - 1, min(need, plan.workspace_size(large, hw, hw))}:
        nhip.timer_start("conv_split_f32")
        got = plan.forward(x, workspace=torch.empty(size, dtype=torch.uint8, device="cuda"))
        assert nhip.timer_stop()[0] == 1
        assert ((got.cpu().double() - ref).norm() / ref.norm()).item() < 1e-6


@pytest.mark.parametrize("cfg", [None, "1,1,1,1", "2,2,2,1", "1,2,3,2"])
@pytest.mark.parametrize("case", [CASES[0], CASES[1], CASES[2], CASES[3]], ids=lambda c: "x".join(map(str, c[:5])))
def test_products_near_overflow(case, cfg, nhip_env):
    """x w is finite where the product of their rounded bf16 pieces is not: one product per sum, just below the
    largest fp32 number."""
    for name in ("NHIP_POINTWISE", "NHIP_CONV_KQ", "NHIP_GEMM_DMA", "NHIP_CONV_SMALLK"):
        nhip_env.setenv(name, "0")
    if cfg:
        nhip_env.setenv("NHIP_SPLIT_CFG", cfg)
    case = case[:-2] + (False, 0)
    x, wt, b, _ = data(case, 5)
    rng = np.random.default_rng(6)
    x[:] = 0
    x.reshape(-1)[x.size // 2] = -1.8428e19
    wt[:] = rng.uniform(1.8426e19, 1.8428e19, wt.shape) * rng.choice([-1, 1], wt.shape)
    got, launches = run(case, x, wt, b * 0, None)
    assert launches == 1
    s, _ = sums64(case, x, wt)
    assert np.abs(s).max() > 3.39e38 and np.abs(s).max() < 3.4028e38
    np.testing.assert_allclose(got, s, rtol=2.0 ** -22)


@pytest.mark.parametrize("case", [CASES[0], CASES[1], CASES[2], CASES[3], CASES[7]], ids=lambda c: "x".join(map(str, c[:5])))
@pytest.mark.parametrize("what", ["x", "one x", "w", "rows", "both"])
def test_operands_that_bf16_pieces_do_not_hold(case, what, nhip_env):
    """Numbers whose lower pieces would fall under bf16's smallest subnormal (2^-133): inputs down to fp32's, one
    such input among zeros, weights of all rows or of some, and products near the subnormal numbers.  A chain of
    fp32 sums: n + 2 roundings of 2^-24 of sum |x w|, or of 2^-149 where the sums are subnormal."""
    for name in ("NHIP_POINTWISE", "NHIP_CONV_KQ", "NHIP_GEMM_DMA", "NHIP_CONV_SMALLK"):
        nhip_env.setenv(name, "0")
    case = case[:-2] + (False, 0)
    x, wt, b, _ = data(case, 15)
    scales = [1e-33, 1e-36, 3e-38, 1e-41]
    for scale in scales if what != "rows" else [1]:
        xs, ws = x, wt
        if what == "x":
            xs = x * np.float32(scale)
        if what == "one x":
            xs = np.zeros_like(x)
            xs.reshape(-1)[x.size // 2] = scale * 1.2345678
        if what == "w":
            ws = wt * np.float32(scale)
        if what == "both":
            xs, ws = x * np.float32(scale * 1e10), wt * np.float32(3e-9)
        if what == "rows":
            ws = wt.copy()
            for i in range(ws.shape[0]):
                ws[i] *= np.float32([1, 1e-37, 0, 1e-41, 1e30][i % 5])
                if i % 2:
                    ws[i].reshape(-1)[::3] *= np.float32(1e-20)
        xs, ws = xs.astype(np.float32), ws.astype(np.float32)
        got, launches = run(case, xs, ws, b * 0, None)
        assert launches == 1
        s, m = sums64(case, xs, ws)
        terms = wt[0].size
        assert np.all(np.abs(got - s) <= m * 2.0 ** -24 * (terms + 2) + 2.0 ** -149 * (terms + 2)), scale
