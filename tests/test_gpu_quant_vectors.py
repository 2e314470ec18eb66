"""The vectorised Quantize / Requantize / Dequantize kernels against the
oracle, bit for bit: planes that end inside a group of four elements, planes
smaller than a group, element counts off four, buffers aligned only to their
elements, one scale and one per channel."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import nhip  # noqa: E402
from oracle import refcpu  # noqa: E402

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1, 1), (3, 7, 1, 1), (2, 5, 1, 3), (2, 3, 2, 1), (3, 16, 7, 7), (2, 9, 13, 5), (1, 40, 64, 80), (5, 33, 31, 29),
          # on the vector kernels (3072 elements per CU): each kind of plane, counts off four, the first count taken and the last not
          (1, 1101, 51, 15), (3, 262145, 1, 1), (1, 400003, 1, 2), (11, 9973, 1, 9), (3, 1033, 15, 17), (1, 3072, 1, 256), (1, 786431, 1, 1)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("off", [0, 1])
def test_quant_vectors_bit_exact(shape, per_channel, off):
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    nhip.init(0)
    n, c = shape[:2]
    count = int(np.prod(shape))
    rng = np.random.default_rng([*shape, int(per_channel), off])
    k = c if per_channel else 1
    isc, osc = rng.uniform(1e-4, 3e-3, k).astype(np.float32), rng.uniform(0.5, 4.0, k).astype(np.float32)
    bias = (rng.standard_normal(k) * 3).astype(np.float32)
    xi = rng.integers(-400000, 400000, count + off).astype(np.int32)
    xi[off:off + 3] = [2 ** 31 - 1, -2 ** 31, 0][:count]
    xf = rng.uniform(-90, 90, count + off).astype(np.float32)
    xf[off:off + 2] = [np.nan, -np.inf][:count]
    di, df = torch.from_numpy(xi).cuda()[off:].view(shape), torch.from_numpy(xf).cuda()[off:].view(shape)
    got = [nhip.quantize(df, osc), nhip.requantize(di, isc, osc, bias, nhip.ACT_RELU),
           nhip.requantize(di, isc, osc), nhip.dequantize(di, isc, bias), nhip.dequantize(di, isc)]
    hi, hf = xi[off:].reshape(shape), xf[off:].reshape(shape)
    for i in range(n):
        exp = [refcpu.quantize_f32_i8(hf[i], osc, shape[2] * shape[3]), refcpu.requantize_i32_i8(hi[i], isc, osc, bias, 1),
               refcpu.requantize_i32_i8(hi[i], isc, osc, None, 0), refcpu.dequantize_i32_f32(hi[i], isc, bias),
               refcpu.dequantize_i32_f32(hi[i], isc, None)]
        for g, e in zip(got, exp):
            np.testing.assert_array_equal(g[i].cpu().numpy(), e)
