"""Products on the bf16 matrix cores (operands split into three bf16 parts), value-checked where the kernel can go wrong:
the smallest k, k beside a multiple of every tile depth, outputs beside the tiles, every tile of the planner, ranges of k,
and operands the parts cannot represent, which are multiplied again on the FP32 matrix cores.  Tolerance: 1e-5 * sqrt(k)
of the largest |a|.|b| dot product, as for every other product; the summation error of k FP32 terms stays below it."""
import math

import numpy as np
import pytest

from adhip import ir as IR
from parity import RED_RTOL, assert_close

pytestmark = pytest.mark.gpu


def _product(hip_device, layout, a, b):
    (m, k), n = a.shape, b.shape[1]
    cmds = []
    if layout[0] == "k":
        cmds.append(IR.CreateMat(a.reshape(-1), [m, k], "a"))
    else:
        cmds += [IR.CreateMat(np.ascontiguousarray(a.T).reshape(-1), [k, m], "at"), IR.Permute(a="at", p=[1, 0], res="a")]
    if layout[1] == "n":
        cmds.append(IR.CreateMat(b.reshape(-1), [k, n], "b"))
    else:
        cmds += [IR.CreateMat(np.ascontiguousarray(b.T).reshape(-1), [n, k], "bt"), IR.Permute(a="bt", p=[1, 0], res="b")]
    cmds += [IR.DotProduct(a="a", b="b", res="c"), IR.EX()]
    hip_device.execute(IR.IRProcedure("main", cmds), {"c"})
    got = hip_device.get_tensor("c")
    assert got.dim == [m, n]
    return np.asarray(got.data, dtype=np.float32).reshape(m, n)


@pytest.mark.parametrize("layout", ["kn", "kk", "mn", "mk"])
@pytest.mark.parametrize("shape", [(96, 100, 31), (96, 100, 32), (65, 63, 65), (129, 64, 63), (64, 64, 64), (1, 9000, 47), (9000, 1, 33),
                                   (128, 128, 2048), (100, 130, 1500), (700, 800, 1100), (1500, 1400, 300), (2300, 2100, 520),
                                   (4100, 3900, 48), (4097, 4095, 33)])
def test_split_products(layout, shape, hip_device):
    m, n, k = shape
    print(f"[case] split product {m}x{n}x{k} layout {layout}", flush=True)
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    got = _product(hip_device, layout, a, b)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    assert_close(got.reshape(-1), (a64 @ b64).reshape(-1), RED_RTOL * math.sqrt(k), f"c ({layout})", scale=float((np.abs(a64) @ np.abs(b64)).max()))


@pytest.mark.parametrize("layout", ["kn", "mk"])
@pytest.mark.parametrize("shape", [(130, 70, 77), (300, 200, 1100), (1500, 1400, 300)])
def test_operands_that_the_parts_cannot_represent(layout, shape, hip_device):
    """Infinities, NaN, values that round to infinity in bf16 and sums of 2^-110: what comes out is what the FP32
    matrix cores give, and the rest of the product is as before."""
    m, n, k = shape
    print(f"[case] unrepresentable operands {m}x{n}x{k} layout {layout}", flush=True)
    rng = np.random.default_rng(k)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    b[k // 2] = np.abs(b[k // 2]) + 0.5
    a[3, k // 2] = np.inf
    a[5, k // 2] = -np.inf
    a[7, 1] = np.nan
    a[9] = 0.0
    a[9, k - 1] = np.finfo(np.float32).max      # finite, but beyond bf16's largest value
    b[k - 1] *= 0.25                            # ... and times this still finite
    a[11] *= np.float32(2.0 ** -118)
    got = _product(hip_device, layout, a, b)
    assert np.all(got[3] == np.inf) and np.all(got[5] == -np.inf) and np.all(np.isnan(got[7]))
    with np.errstate(over="ignore"):
        assert np.array_equal(got[9], a[9, k - 1] * b[k - 1])
    rows = [r for r in range(m) if r not in (3, 5, 7, 9, 11)]
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    assert_close(got[rows].reshape(-1), (a64[rows] @ b64).reshape(-1), RED_RTOL * math.sqrt(k), "c", scale=float((np.abs(a64[rows]) @ np.abs(b64)).max()))
    assert_close(got[11] * 2.0 ** 118, (a64[11] @ b64) * 2.0 ** 118, RED_RTOL * math.sqrt(k), "tiny row",
                 scale=float((np.abs(a64[11]) @ np.abs(b64)).max() * 2.0 ** 118))
