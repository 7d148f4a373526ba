"""Launches that run as one have the LDS of all of them: what exceeds a CU's 160 KB is left apart, and every such program compiles."""
import re

import numpy as np
import pytest

from adhip import ir as IR
from adhip.device import lower_describe
from test_library_cpu import _compile_check


def _sums_and_product(sums, first_rows, cols, product):
    """`sums` column sums of one block each, no two of one shape, and beside them, if asked for, a product of 64x64 tiles."""
    cmds, keep = [], set()
    for i in range(sums):
        rows = first_rows + i
        cmds += [IR.CreateMat(np.ones(rows * cols, np.float32), [rows, cols], f"x{i}"), IR.Permute(a=f"x{i}", p=[1, 0], res=f"t{i}"), IR.Sum(a=f"t{i}", res=f"s{i}")]
        keep.add(f"s{i}")
    if product:
        m, n, k = product
        cmds += [IR.CreateMat(np.ones(m * k, np.float32), [m, k], "a"), IR.CreateMat(np.ones(k * n, np.float32), [k, n], "b"), IR.DotProduct(a="a", b="b", res="c")]
        keep.add("c")
    return IR.IRProcedure("main", cmds + [IR.EX()]), keep


PROGRAMS = {
    "30 sums of 10.. rows, a product": (30, 10, 64, (1024, 768, 512)),
    "26 sums of 33.. rows, a product": (26, 33, 64, (1000, 784, 500)),
    "30 sums of 70.. rows, a product": (30, 70, 64, (1024, 768, 512)),
    "80 sums": (80, 2, 64, None),   # as many as the arguments of one launch: 80 KB
    "80 sums, a small product": (80, 2, 64, (64, 64, 64)),
}


@pytest.mark.parametrize("name", PROGRAMS)
def test_programs_of_many_single_blocks_compile(name):
    proc, keep = _sums_and_product(*PROGRAMS[name])
    rc, msg = _compile_check(proc, keep)
    assert rc == 0, msg
    assert "lowered" not in msg, msg   # at the first attempt


def test_a_few_single_blocks_still_share_a_launch_with_a_product():
    text = lower_describe(*_sums_and_product(4, 10, 64, (1024, 768, 512)))
    assert re.search(r"shared\d+_2x, one launch", text) and "[merged]" in text, text


@pytest.mark.gpu
@pytest.mark.parametrize("name", PROGRAMS)
def test_values(name, hip_device):
    """Whole numbers: exact."""
    print(f"[case] {name}", flush=True)
    sums, first_rows, cols, product = PROGRAMS[name]
    proc, keep = _sums_and_product(sums, first_rows, cols, product)
    hip_device.execute(proc, keep)
    for i in range(sums):
        assert np.array_equal(np.asarray(hip_device.get_tensor(f"s{i}").data), np.full(cols, first_rows + i, np.float32))
    if product:
        assert np.array_equal(np.asarray(hip_device.get_tensor("c").data), np.full(product[0] * product[1], product[2], np.float32))
