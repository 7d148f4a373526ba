"""Products on the bf16 matrix cores (operands split into three bf16 parts), value-checked where the kernel can go wrong:
the smallest k, k beside a multiple of every tile depth, outputs beside the tiles, ranges of k, operands of every magnitude,
and what does not come out finite, which is multiplied again on the FP32 matrix cores.  Tolerance: 1e-5 * sqrt(k) of the
largest |a|.|b| dot product, as for every other product: it sees a wrong element, not a lost part of one, for which there
is test_product_bits.py, on every tile of the planner."""
import math
import time

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


@pytest.mark.parametrize("shape,layout", [((130, 70, 77), "kn"), ((300, 200, 256), "mk"), ((300, 200, 1100), "kk"), ((2000, 1900, 1030), "mn")])
@pytest.mark.parametrize("ea,eb", [(-118, 60), (-122, 90), (-126, 100), (-130, 110), (-140, 115), (-140, 90), (90, -122), (-62, -64)])
def test_operands_at_the_bottom_of_the_range(shape, layout, ea, eb, hip_device):
    """Operands down into FP32's subnormals beside large ones: the result is an ordinary number, and as precise as any
    other.  Bound: an operand is held to the bit it has, so the error is that of the sum alone, for which 2^-24 sqrt(k)
    of the root mean square is what k roundings of partial sums no larger than the result add up to; where the result
    is itself subnormal, half of its last bit (one for each of the few ranges that k is cut into) comes on top."""
    m, n, k = shape
    print(f"[case] small operands {m}x{n}x{k} layout {layout} 2^{ea} x 2^{eb}", flush=True)
    rng = np.random.default_rng(m + 1000 + ea)
    a = rng.standard_normal((m, k), dtype=np.float32) * np.float32(2.0 ** ea)
    b = rng.standard_normal((k, n), dtype=np.float32) * np.float32(2.0 ** eb)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    want = (a64 @ b64).reshape(-1)
    got = _product(hip_device, layout, a, b).reshape(-1).astype(np.float64)
    rms = math.sqrt(float(np.mean(want ** 2)))
    err = math.sqrt(float(np.mean((got - want) ** 2)))
    assert err <= 2.0 ** -24 * math.sqrt(k) * rms + 4 * 2.0 ** -149, (err / rms, rms)


def _time(hip_device, a, b):
    (m, k), n = a.shape, b.shape[1]
    cmds = [IR.CreateMat(a.reshape(-1), [m, k], "a"), IR.CreateMat(b.reshape(-1), [k, n], "b"), IR.DotProduct(a="a", b="b", res="c"), IR.EX()]
    prog = hip_device.compile(IR.IRProcedure("main", cmds), {"c"})
    prog.upload()
    best = math.inf
    for _ in range(5):
        t0 = time.perf_counter()
        for _ in range(20):
            prog.enqueue()
        prog.sync()
        best = min(best, time.perf_counter() - t0)
    prog.close()
    return best


@pytest.mark.parametrize("shape,times", [((4096, 4096, 1024), 4.5), ((4096, 1024, 4096), 6.0)])
def test_tiny_results_cost_nothing_and_infinities_little(shape, times, hip_device):
    """Rows of results around 2^-105 in every tile take the time of any others.  Where a result is not finite, a
    wavefront multiplies again on the FP32 matrix cores, which run at half of the rate and, straight from memory, at
    half of that: with the first attempt 3.3 times on the 256x256 tile, 4.7 where half of the wavefronts have no part in it."""
    m, n, k = shape
    print(f"[case] time of tiny and infinite results {m}x{n}x{k}", flush=True)
    rng = np.random.default_rng(k)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    plain = _time(hip_device, a, b)
    tiny = a.copy()
    tiny[5::32] *= np.float32(2.0 ** -110)
    infinite = a.copy()
    infinite[5::32, 7] = np.inf
    assert _time(hip_device, tiny, b) < 1.25 * plain
    assert _time(hip_device, infinite, b) < times * plain
