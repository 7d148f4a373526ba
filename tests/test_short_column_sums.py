"""Column sums over up to 128 rows take one launch, longer ones chunks and a second one."""
import re

import numpy as np
import pytest

from adhip import ir as IR
from adhip.device import lower_describe

SHAPES = [(33, 256), (64, 64), (65, 1000), (127, 258), (128, 4100), (129, 64), (200, 28)]


def _program(rows, cols, x, op):
    cmds = [IR.CreateMat(x.reshape(-1), [rows, cols], "x"), IR.Permute(a="x", p=[1, 0], res="xt"), op(a="xt", res="c"), IR.EX()]
    return IR.IRProcedure("main", cmds), {"c"}


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_launches(rows, cols):
    proc, keep = _program(rows, cols, np.zeros((rows, cols), np.float32), IR.Sum)
    blocks = re.findall(r"launch \S+ \[reduce_col\] \S+ grid=\((\d+),(\d+),1\) block=(\d+)", lower_describe(proc, keep))
    assert (len(blocks) == 1) == (rows <= 128), blocks
    if rows <= 128:
        assert blocks[0][1:] == ("1", "256"), blocks


@pytest.mark.gpu
@pytest.mark.parametrize("op", [IR.Sum, IR.Max])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_values(rows, cols, op, hip_device):
    """A sum of n values in any order is off by at most (n - 1) 2^-24 of the sum of magnitudes; a maximum by nothing."""
    print(f"[case] short column reduction {rows}x{cols}", flush=True)
    x = np.random.default_rng(rows * cols).standard_normal((rows, cols), dtype=np.float32)
    proc, keep = _program(rows, cols, x, op)
    hip_device.execute(proc, keep)
    got = np.asarray(hip_device.get_tensor("c").data, np.float64)
    if op is IR.Max:
        assert np.array_equal(got, x.max(0).astype(np.float64))
    else:
        x64 = x.astype(np.float64)
        assert np.all(np.abs(got - x64.sum(0)) <= rows * 2.0 ** -24 * np.abs(x64).sum(0))
