"""Products below the matrix-core tiles, value-checked beside the points where the number of lanes per result changes (k = 4,
8, ... 256), in one block and in many, alone, with an element-wise epilogue and as a grouped launch, and with operands that
have no unit stride.  Tolerance: 1e-5 * sqrt(k) of the largest |a|.|b| dot product, which the sum of k FP32 terms stays below."""
import math
import re

import numpy as np
import pytest

from adhip import ir as IR
from adhip.device import lower_describe
from parity import RED_RTOL, assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (2, 3, 4), (3, 2, 5), (16, 16, 16), (16, 16, 17), (7, 9, 64), (64, 48, 65), (5, 5, 257),
                                   (1, 1, 5000), (300, 290, 3), (33, 31, 200)])
@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("epilogue", [False, True])
def test_small_products(m, n, k, strided, epilogue, hip_device):
    print(f"[case] small product {m}x{n}x{k} strided {strided} epilogue {epilogue}", flush=True)
    rng = np.random.default_rng(m + 5 * n + 11 * k)
    s = 2 if strided else 1
    an, bn = rng.standard_normal((m, k, s), dtype=np.float32), rng.standard_normal((k, n, s), dtype=np.float32)
    cmds = [IR.CreateMat(an.reshape(-1), [m, k, s], "a3"), IR.CreateMat(bn.reshape(-1), [k, n, s], "b3"),
            IR.Index(a="a3", index=0, dim=2, res="a"), IR.Index(a="b3", index=0, dim=2, res="b"), IR.DotProduct(a="a", b="b", res="c")]
    a64, b64 = an[:, :, 0].astype(np.float64), bn[:, :, 0].astype(np.float64)
    want = a64 @ b64
    if epilogue:
        wn = rng.standard_normal((m, n), dtype=np.float32)
        cmds += [IR.CreateMat(wn.reshape(-1), [m, n], "w"), IR.ElwMultiply(a="c", b="w", res="y")]
        want = want * wn
    keep = "y" if epilogue else "c"
    hip_device.execute(IR.IRProcedure("main", cmds + [IR.EX()]), {keep})
    got = hip_device.get_tensor(keep)
    assert got.dim == [m, n]
    scale = float((np.abs(a64) @ np.abs(b64)).max()) * (float(np.abs(wn).max()) if epilogue else 1.0)
    assert_close(got.data, want.reshape(-1), RED_RTOL * math.sqrt(k), keep, scale=scale)


@pytest.mark.parametrize("count,m,n,k", [(2, 16, 16, 8), (3, 64, 8, 33), (17, 20, 30, 5), (16, 8, 64, 64)])
def test_small_products_grouped(count, m, n, k, hip_device):
    print(f"[case] {count} small products {m}x{n}x{k}", flush=True)
    rng = np.random.default_rng(count + m)
    a, b = rng.standard_normal((count, m, k), dtype=np.float32), rng.standard_normal((count, k, n), dtype=np.float32)
    cmds = []
    for i in range(count):
        cmds += [IR.CreateMat(a[i].reshape(-1), [m, k], f"a{i}"), IR.CreateMat(b[i].reshape(-1), [k, n], f"b{i}"), IR.DotProduct(a=f"a{i}", b=f"b{i}", res=f"c{i}")]
    proc = IR.IRProcedure("main", cmds + [IR.EX()])
    keep = {f"c{i}" for i in range(count)}
    assert re.search(r"launch dots_\w+ \[dot_naive\] kernel=adhip_dot_small_grouped", lower_describe(proc, keep))
    hip_device.execute(proc, keep)
    for i in range(count):
        want = a[i].astype(np.float64) @ b[i].astype(np.float64)
        assert_close(hip_device.get_tensor(f"c{i}").data, want.reshape(-1), RED_RTOL * math.sqrt(k), f"c{i}", scale=float((np.abs(a[i]) @ np.abs(b[i])).max()))
