"""Column sums that ride on an element-wise pass which stands behind one of their readers, or which shares with them an
operand repeated along the rows: descent steps on the squares of an element-wise function of three matrices and a bias."""
import re

import numpy as np
import pytest

from adhip import autodiff, nn
from adhip.device import Device, lower_describe
from oracle.interp import OracleDevice
from parity import RED_RTOL, assert_close


def _descent(dev, rows, cols):
    autodiff.set_device(dev)
    autodiff.eager_dep_opt()
    rng = np.random.default_rng(rows + cols)

    def uniform(*dim):
        return autodiff.tensor(rng.uniform(-1, 1, size=dim).astype(np.float32), list(dim))

    a, b, bias = uniform(rows, cols), uniform(rows, cols), uniform(cols)
    y = (a * b + bias).sigmoid() + a.sin()
    loss = (y * y).sum(0).sum(0)
    loss.forward()
    loss.backward()
    nn.SGD([a, b], 0.01).step()
    nn.SGD([bias], 0.01 / rows).step()
    outs = {"loss": loss.val(), "a": a.val(), "b": b.val(), "bias": bias.val()}
    for v in outs.values():
        v.keep()
    return outs


def test_both_column_sums_ride_on_the_pass_that_updates():
    from adhip.core import STATE
    from adhip import ir as IR
    outs = _descent(Device(), 256, 512)
    STATE.irb.add_cmd(IR.EX())
    text = lower_describe(STATE.irb.proc, {v.id for v in outs.values()})
    kinds = re.findall(r"launch \S+ \[(\w+)\]", text)
    assert kinds.count("elw_colsum") == 1 and "reduce_col" not in kinds, text


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(256, 256), (300, 1028), (1024, 512), (17, 4100)])
def test_descent_matches_the_oracle(rows, cols, hip_device):
    print(f"[case] descent {rows}x{cols}", flush=True)
    got = {}
    for name, dev in (("hip", hip_device), ("oracle", OracleDevice())):
        outs = _descent(dev, rows, cols)
        autodiff.execute()
        got[name] = {k: np.asarray(v.get().data, dtype=np.float64) for k, v in outs.items()}
    for k, want in got["oracle"].items():
        assert_close(got["hip"][k], want, RED_RTOL, k, scale=float(max(np.abs(want).max(), 1.0)))
