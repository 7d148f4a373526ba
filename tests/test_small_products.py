"""How small products are spread over blocks and lanes, from the plan; and their values beside the points where that changes.
Tolerance of the values: 1e-5 * sqrt(k) of the largest |a|.|b| dot product, as for every other product."""
import math
import re

import numpy as np
import pytest

from adhip import ir as IR
from adhip.device import lower_describe
from parity import RED_RTOL, assert_close


def _program(m, n, k, strided=False, seed=0, b_along_k=False):
    rng = np.random.default_rng(seed)
    s = 2 if strided else 1
    a, b = rng.standard_normal((m, k, s), dtype=np.float32), rng.standard_normal((k, n, s), dtype=np.float32)
    cmds = [IR.CreateMat(a.reshape(-1), [m, k, s], "a3"), IR.CreateMat(b.reshape(-1), [k, n, s], "b3"),
            IR.Index(a="a3", index=0, dim=2, res="a"), IR.Index(a="b3", index=0, dim=2, res="b"), IR.DotProduct(a="a", b="b", res="c"), IR.EX()]
    if b_along_k:
        cmds[1] = IR.CreateMat(np.ascontiguousarray(b.transpose(1, 0, 2)).reshape(-1), [n, k, s], "b3")
        cmds[3:4] = [IR.Index(a="b3", index=0, dim=2, res="bt"), IR.Permute(a="bt", p=[1, 0], res="b")]
    return IR.IRProcedure("main", cmds), a[:, :, 0].astype(np.float64), b[:, :, 0].astype(np.float64)


def _blocks(m, n, k, strided=False, b_along_k=False):
    text = lower_describe(_program(m, n, k, strided, b_along_k=b_along_k)[0], {"c"})
    return int(re.search(r"launch dot_c_\w+ \[dot_naive\] kernel=\w+ grid=\((\d+),1,1\) block=256", text).group(1))


@pytest.mark.parametrize("m,n,k", [(128, 128, 1), (256, 64, 1), (64, 64, 1), (64, 64, 4), (64, 32, 8), (16, 16, 64), (32, 32, 16),
                                   (8, 8, 256), (4, 4, 1024), (60, 60, 60)])
def test_no_block_walks_over_results(m, n, k):
    """A block has 256 lanes; results (at least one lane each) beyond them belong to other blocks, also where k is short:
    the weight gradient of a perceptron at batch 1 to 4.  With more lanes to a result there are more blocks."""
    assert _blocks(m, n, k) * 256 >= m * n * min(max(1, (k + 7) // 8), 64)


@pytest.mark.parametrize("m,n,k,blocks", [(16, 16, 16, 1), (16, 16, 17, 8), (8, 16, 32, 1), (8, 16, 33, 8), (5, 5, 128, 1), (5, 5, 129, 7), (2, 2, 1024, 1)])
def test_up_to_256_results_stay_in_one_block_while_it_has_the_lanes(m, n, k, blocks):
    assert _blocks(m, n, k) == blocks


@pytest.mark.parametrize("m,n,k,lanes", [(255, 255, 1000, 2), (200, 200, 4096, 4), (300, 300, 300, 2), (314, 313, 70, 2), (314, 314, 70, 1), (700, 700, 50, 1),
                                         (64, 64, 5000, 32), (1, 1000, 3000, 64)])
def test_large_products_without_unit_strides_do_not_overfill_the_chip(m, n, k, lanes):
    """Three wavefronts per SIMD (196608 lanes) are the most that lanes are added for, but for operands that both lie
    along k, up to 65536 results."""
    assert _blocks(m, n, k, strided=True) == (m * n * lanes + 255) // 256
    assert _blocks(m, n, k, strided=True, b_along_k=True) == (m * n * (64 if m * n < 65536 else lanes) + 255) // 256


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(128, 128, 1), (16, 16, 16), (16, 16, 17), (15, 17, 16), (8, 16, 32), (8, 16, 33), (5, 5, 128), (5, 5, 129),
                                   (2, 2, 1024), (2, 2, 1025), (257, 1, 16), (255, 255, 300), (314, 313, 70), (314, 314, 70)])
@pytest.mark.parametrize("strided,b_along_k", [(False, False), (True, False), (True, True)])
def test_values_where_the_lanes_change(m, n, k, strided, b_along_k, hip_device):
    print(f"[case] small product {m}x{n}x{k} strided {strided} b along k {b_along_k}", flush=True)
    proc, a, b = _program(m, n, k, strided, seed=m + n + k, b_along_k=b_along_k)
    hip_device.execute(proc, {"c"})
    assert_close(hip_device.get_tensor("c").data, (a @ b).reshape(-1), RED_RTOL * math.sqrt(k), "c", scale=float((np.abs(a) @ np.abs(b)).max()))
