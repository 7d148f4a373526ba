"""Groups that run the same generated kernel on other buffers share its launches: how many fit one."""
import re

import numpy as np
import pytest

from adhip import ir as IR
from adhip.device import lower_describe
from oracle.interp import OracleDevice
from test_library_cpu import _compile_check


def _column_sums(count, rows, cols):
    cmds, keep = [], set()
    for i in range(count):
        cmds += [IR.CreateMat(np.zeros(rows * cols, np.float32), [rows, cols], f"x{i}"), IR.Permute(a=f"x{i}", p=[1, 0], res=f"t{i}"), IR.Sum(a=f"t{i}", res=f"s{i}")]
        keep.add(f"s{i}")
    return IR.IRProcedure("main", cmds + [IR.EX()]), keep


def _wide_passes(count, operands, n, rng=None):
    """y<i> = a<i>0 + a<i>1 * a<i>1 + ... of operands of their own, in `count` groups."""
    cmds, keep = [], set()
    for i in range(count):
        for q in range(operands):
            v = rng.standard_normal(n).astype(np.float32) if rng else np.zeros(n, np.float32)
            cmds.append(IR.CreateMat(v, [n], f"a{i}_{q}"))
        total = f"a{i}_0"
        for q in range(1, operands):
            cmds += [IR.ElwMultiply(a=f"a{i}_{q}", b=f"a{i}_{q}", res=f"p{i}_{q}"), IR.ElwAdd(a=total, b=f"p{i}_{q}", res=f"y{i}_{q}")]
            total = f"y{i}_{q}"
        keep.add(total)
    return IR.IRProcedure("main", cmds + [IR.EX()]), keep



@pytest.mark.parametrize("rows,cols", [(2048, 4096), (16384, 256), (300, 1024)])
def test_chunked_column_sums_share_both_their_launches(rows, cols):
    """However many chunks of rows a sum has."""
    text = lower_describe(*_column_sums(3, rows, cols))
    assert [int(n) for n in re.findall(r"launch \S+_x(\d+) \[reduce_col\]", text)] == [3, 3] and len(re.findall("launch ", text)) == 2, text


@pytest.mark.parametrize("count,operands,instances", [(16, 5, [2]), (16, 12, [2, 2]), (9, 20, [4, 4]), (24, 24, [3] * 8)])
def test_a_shared_launch_takes_at_most_96_pointers(count, operands, instances):
    """(A pass stores up to several results; how many is not what this test is about.)"""
    proc, keep = _wide_passes(count, operands, 1 << 18)
    text = lower_describe(proc, keep)
    launches = re.findall(r"^\s*launch (\S+) .*args:(.*)$", text, re.M)
    assert [int(n) for n in re.findall(r"^\s*launch \S+_x(\d+) ", text, re.M)] == instances, text
    assert all(len(args.split()) <= 96 for _, args in launches), text
    rc, msg = _compile_check(proc, keep)
    assert rc == 0, msg


@pytest.mark.gpu
@pytest.mark.parametrize("count,operands", [(16, 12), (9, 20)])
def test_values_of_wide_passes(count, operands, hip_device):
    """Sums and products in the same order as the oracle's, one rounding each: the same bits."""
    print(f"[case] {count} passes of {operands} operands", flush=True)
    proc, keep = _wide_passes(count, operands, 5000, np.random.default_rng(count))
    hip_device.execute(proc, keep)
    dev = OracleDevice()
    dev.execute(proc, keep)
    for k in sorted(keep):
        assert np.array_equal(np.asarray(hip_device.get_tensor(k).data, np.float32), np.asarray(dev.get_tensor(k).data, np.float32)), k


@pytest.mark.gpu
def test_values_of_chunked_column_sums(hip_device):
    """Whole numbers: exact."""
    print("[case] three chunked column sums", flush=True)
    rows, cols, cmds, keep = 2048, 512, [], set()
    rng = np.random.default_rng(2)
    x = [rng.integers(-8, 9, (rows, cols)).astype(np.float32) for _ in range(3)]
    for i in range(3):
        cmds += [IR.CreateMat(x[i].reshape(-1), [rows, cols], f"x{i}"), IR.Permute(a=f"x{i}", p=[1, 0], res=f"t{i}"), IR.Sum(a=f"t{i}", res=f"s{i}")]
        keep.add(f"s{i}")
    proc = IR.IRProcedure("main", cmds + [IR.EX()])
    assert "_x3 [reduce_col]" in lower_describe(proc, keep)
    hip_device.execute(proc, keep)
    for i in range(3):
        assert np.array_equal(np.asarray(hip_device.get_tensor(f"s{i}").data), x[i].sum(0))
