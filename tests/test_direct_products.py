"""The kernel without a staging buffer addresses a step by 32-bit byte offsets unless an operand's lines are long: which of
the two a product gets, read from the generated source (no tensor of these sizes is ever touched)."""
import math
import re

import numpy as np
import pytest

from adhip import ir as IR
from adhip.device import lower_describe
from parity import RED_RTOL, assert_close
from test_library_cpu import _compile_check


def _program(m, n, k, layout, long_a, long_b, products, values=None):
    """c = a b; a long operand is the front of every line of a wider matrix."""
    def operand(name, rows, cols, along_cols, long):
        outer, inner = (rows, cols) if along_cols else (cols, rows)
        lines = np.zeros((outer, long // inner if long else 1, inner), np.float32)
        if values:
            lines[:, 0] = values[name] if along_cols else values[name].T
        cmds, src = [IR.CreateMat(lines.reshape(-1), list(lines.shape), name + "m")], name + "f"
        cmds.append(IR.Index(a=name + "m", index=0, dim=1, res=src))
        if not along_cols:
            cmds.append(IR.Permute(a=src, p=[1, 0], res=name + "t"))
            src = name + "t"
        return cmds, src

    cmds, keep = [], set()
    for i in range(products):
        ca, a = operand(f"a{i}", m, k, layout[0] == "k", long_a)
        cb, b = operand(f"b{i}", k, n, layout[1] == "n", long_b)
        cmds += ca + cb + [IR.DotProduct(a=a, b=b, res=f"c{i}")]
        keep.add(f"c{i}")
    return IR.IRProcedure("main", cmds + [IR.EX()]), keep


@pytest.mark.parametrize("m,n,k,kernel", [
    (544, 1017, 64, "64_rim_pair"), (544, 1017, 65, "64x64_rim_direct"), (544, 1017, 127, "64x64_rim_direct"), (544, 1017, 128, "64_rim_pair"),
    (544, 1017, 448, "64_rim_pair"), (544, 1017, 449, "64x64_rim_direct"),
    (300, 300, 64, "32x32_rim_direct"), (600, 600, 64, "64_rim_pair"), (1000, 500, 128, "32x64_rim_direct"),
    (320, 256, 3264, "64_splitk"), (128, 128, 3264, "32x32_splitk_direct")])
def test_where_staging_is_the_faster(m, n, k, kernel):
    """Sizes beside the lines between the kernels with and without a staging buffer."""
    text = lower_describe(*_program(m, n, k, "kn", 0, 0, 1))
    assert re.findall(r"kernel=adhip_gemm_kn_(\w+)", text) == [kernel], text


LONG, MIDDLE = 36_000_000, 1 << 21


@pytest.mark.parametrize("products", [1, 2])
@pytest.mark.parametrize("m,n,k,layout,long_a,long_b,offset", [
    (31, 3, 4096, "kn", LONG, 0, "unsigned long long"),   # fewer than four columns: 30 lines of A are 2^32 bytes on
    (31, 5, 4096, "kn", LONG, 0, "unsigned long long"),
    (3, 31, 4096, "mk", 0, LONG, "unsigned long long"),   # the same with the operands' roles exchanged
    (3, 1400, 64, "mn", LONG, 0, "unsigned long long"),   # ... and along the lines that k counts
    (1400, 3, 64, "mn", 0, LONG, "unsigned long long"),
    (31, 3, 4096, "kn", MIDDLE, 0, "unsigned"),
    (31, 3, 4096, "kn", 0, 0, "unsigned"),
])
def test_offsets_are_as_wide_as_the_lines(m, n, k, layout, long_a, long_b, offset, products, tmp_path, monkeypatch):
    monkeypatch.setenv("ADHIP_DUMP_CODE_DIR", str(tmp_path))
    monkeypatch.setenv("ADHIP_SHARE_INDEPENDENT", "0")
    proc, keep = _program(m, n, k, layout, long_a, long_b, products)
    rc, msg = _compile_check(proc, keep)
    assert rc == 0, msg
    sources = [p.read_text() for p in tmp_path.glob("adhip_gemm_*.hip")]
    assert len(sources) == 1 and f"#define GROUPED {int(products > 1)}\n" in sources[0]
    assert f"#define OFFSET {offset}\n" in sources[0], [line for line in sources[0].splitlines() if "define OFFSET" in line]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,layout,long_a,long_b", [(31, 3, 4096, "kn", 1 << 22, 0), (3, 31, 4096, "mk", 0, 1 << 22), (3, 1400, 64, "mn", (1 << 22) + 2, 0),
                                                        (1400, 3, 67, "kn", 0, (1 << 22) + 2), (45, 60, 131, "kk", 0, 131 << 15)])
def test_long_lines(m, n, k, layout, long_a, long_b, hip_device):
    """With 64-bit offsets the same values; tolerance as for every other product."""
    print(f"[case] product {m}x{n}x{k} layout {layout} lines {long_a} {long_b}", flush=True)
    rng = np.random.default_rng(m + n + k)
    values = {"a0": rng.standard_normal((m, k), dtype=np.float32), "b0": rng.standard_normal((k, n), dtype=np.float32)}
    proc, keep = _program(m, n, k, layout, long_a, long_b, 1, values)
    hip_device.execute(proc, keep)
    a, b = values["a0"].astype(np.float64), values["b0"].astype(np.float64)
    assert_close(hip_device.get_tensor("c0").data, (a @ b).reshape(-1), RED_RTOL * math.sqrt(k), "c", scale=float((np.abs(a) @ np.abs(b)).max()))
