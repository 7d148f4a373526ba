"""A row sum and a column sum over one operand that nothing else passes over: one pass for both."""
import re

import numpy as np
import pytest

from adhip import ir as IR
from adhip.device import lower_describe


def _program(rows, cols, x, col_first=False, own=False, other=None):
    """r = (x * x).sum(1), c = x.sum(0) (or, with `other`, of x + other) and the total of r; `own`: the column sums of y = x x."""
    cmds = [IR.CreateMat(x.reshape(-1), [rows, cols], "x"), IR.ElwMultiply(a="x", b="x", res="q")]
    src = "q" if own else "x"
    if other is not None:
        cmds += [IR.CreateMat(other.reshape(-1), [rows, cols], "o"), IR.ElwAdd(a="x", b="o", res="xo")]
        src = "xo"
    row, col = [IR.Sum(a="q", res="r")], [IR.Permute(a=src, p=[1, 0], res="xt"), IR.Sum(a="xt", res="c")]
    cmds += col + row if col_first else row + col
    cmds += [IR.View(a="r", target_dim=[1, rows], res="rv"), IR.Sum(a="rv", res="t"), IR.EX()]
    return IR.IRProcedure("main", cmds), {"r", "c", "t"}


def _passes(text, rows, cols):
    return re.findall(r"launch \S+ \[(elw_colsum|reduce_row|reduce_col)\] \S+ grid=\S+ block=\d+ bytes=(\d+)", text)


@pytest.mark.parametrize("rows,cols", [(1024, 1024), (4100, 256), (16, 65536)])
@pytest.mark.parametrize("col_first", [False, True])
@pytest.mark.parametrize("own", [False, True])
def test_one_pass_reads_the_operand(rows, cols, col_first, own):
    proc, keep = _program(rows, cols, np.zeros((rows, cols), np.float32), col_first, own)
    big = [kind for kind, b in _passes(lower_describe(proc, keep), rows, cols) if int(b) >= 4 * rows * cols]
    assert big == ["elw_colsum"]


def test_small_or_different_operands_keep_their_own():
    for rows, cols, other in ((512, 512, None), (1024, 1022, None), (1024, 1024, np.zeros((1024, 1024), np.float32))):
        proc, keep = _program(rows, cols, np.zeros((rows, cols), np.float32), other=other)
        assert "elw_colsum" not in lower_describe(proc, keep), (rows, cols)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(1024, 1024), (4100, 256), (1031, 1020), (16, 65536), (65537, 260), (9000, 516)])
@pytest.mark.parametrize("col_first,own", [(False, False), (True, True)])
def test_values(rows, cols, col_first, own, hip_device):
    """A value goes through as many additions as stand between it and the result: four in a lane, six across the wavefront or
    sixteen across the block, one per 256-column run or per 64th of the row tiles, and for the total a 1024th of the rows: fewer
    than 40 + (rows + cols) / 256, each rounded by at most 2^-24 of a partial sum that is no larger than the sum of magnitudes."""
    print(f"[case] paired sums {rows}x{cols}", flush=True)
    rng = np.random.default_rng(rows + cols)
    x = rng.standard_normal((rows, cols), dtype=np.float32)
    proc, keep = _program(rows, cols, x, col_first, own)
    x64 = x.astype(np.float64)
    want = {"r": (x64 * x64).sum(1), "c": (x64 * x64 if own else x64).sum(0), "t": np.array([(x64 * x64).sum()])}
    terms = {"r": x64 * x64, "c": (x64 * x64 if own else x64).T, "t": (x64 * x64).reshape(1, -1)}
    for _ in range(3):
        hip_device.execute(proc, keep)
        for k in keep:
            got = np.asarray(hip_device.get_tensor(k).data, np.float64)
            size = 2.0 ** -24 * (40 + (rows + cols) / 256) * np.abs(terms[k]).sum(1)
            assert np.all(np.abs(got - want[k]) <= size), (k, np.max(np.abs(got - want[k]) / size))
