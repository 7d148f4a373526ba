"""Attention on the bf16 matrix cores: every width of heads it takes compiles without spilled registers, and values at the edges
of its tiles of 32 keys, its eight key groups and its blocks of 64 rows, and where its parts cannot represent an operand."""
import math
import re

import numpy as np
import pytest

from adhip import autodiff, nn
from adhip.core import ValueData
from adhip.device import Device, lower_describe
from parity import RED_RTOL, assert_close

WIDTHS = [(d, dv) for d in (32, 64, 96, 128) for dv in (32, 64, 128)]


class Capture(Device):
    def execute(self, proc, deps):
        self.proc, self.deps = proc, list(deps)

    def get_tensor(self, id):
        return ValueData.none()


def _program(dev, q, k, v, scale_dim):
    autodiff.set_device(dev)
    t = [autodiff.tensor(x.reshape(-1), list(x.shape)) for x in (q, k, v)]
    o = nn.Attention(t[0], t[1], t[2], scale_dim)
    o.forward()
    o.val().keep()
    autodiff.execute()
    return o


def _zeros(sq, sk, d, dv):
    return [np.zeros(s, np.float32) for s in ((sq, d), (sk, d), (sk, dv))]


@pytest.mark.parametrize("d,dv", WIDTHS)
def test_every_width_compiles_without_spills(d, dv):
    from test_library_cpu import _compile_check
    dev = Capture()
    _program(dev, *_zeros(100, 400, d, dv), 64)
    text = lower_describe(dev.proc, dev.deps)
    assert f"kernel=adhip_attention_d{d}_v{dv}_k" in text and "_parts " in text and "[attention_split]" in text, text
    rc, msg = _compile_check(dev.proc, dev.deps)
    assert rc == 0 and "lowered" not in msg, msg


@pytest.mark.parametrize("sq,sk,d,dv", [(64, 31, 64, 64), (64, 64, 48, 48), (64, 64, 64, 48), (64, 64, 160, 128),
                                                        (64, 400, 48, 48), (64, 400, 64, 48), (64, 400, 160, 128),
                                        (2048, 255, 64, 64), (64, 32, 32, 32), (300, 300, 32, 64), (2048, 320, 32, 32), (64, 320, 64, 128),
                                        (63, 256, 64, 64), (1, 256, 64, 32)])
def test_what_it_does_not_take_stays_on_the_fp32_ones(sq, sk, d, dv):
    dev = Capture()
    _program(dev, *_zeros(sq, sk, d, dv), 64)
    text = lower_describe(dev.proc, dev.deps)
    assert "[attention]" in text and "_parts" not in text, text


@pytest.mark.parametrize("sq,sk,d,dv", [(64, 256, 64, 64), (1, 257, 64, 64), (1, 256, 128, 32), (1, 256, 96, 128), (64, 321, 64, 128), (1, 321, 32, 32)])
def test_what_it_takes(sq, sk, d, dv, monkeypatch):
    dev = Capture()
    _program(dev, *_zeros(sq, sk, d, dv), 64)
    assert "_parts" in lower_describe(dev.proc, dev.deps)
    monkeypatch.setenv("ADHIP_ATTENTION_PARTS", "0")
    assert "_parts" not in lower_describe(dev.proc, dev.deps)
    _program(dev, *_zeros(sq, 32, d, dv), 64)
    monkeypatch.setenv("ADHIP_ATTENTION_PARTS", "32")
    assert "_parts" in lower_describe(dev.proc, dev.deps)


def test_a_program_that_fits_the_static_scratch_area_without_parts_still_fits():
    """Keys and values in parts take six bytes a number: 2500 x 64 of eight heads 15 MB, beside 24 MB without them."""
    from adhip import workloads as W
    for seq, parts in ((512, True), (2500, False)):
        dev = Capture()
        W.attention_forward(dev, seq, 512, 8).run()
        text = lower_describe(dev.proc, dev.deps)
        assert ("_parts" in text) == parts, text


def _exact(q, k, v, scale_dim):
    s = q.astype(np.float64) @ k.astype(np.float64).T / math.sqrt(scale_dim)
    e = np.exp(s - s.max(1, keepdims=True))
    return (e / e.sum(1, keepdims=True)) @ v.astype(np.float64)


@pytest.mark.gpu
@pytest.mark.parametrize("d,dv", WIDTHS)
@pytest.mark.parametrize("sq,sk", [(64, 32), (1, 33), (65, 63), (130, 255), (63, 257), (200, 520)])
def test_values(sq, sk, d, dv, hip_device):
    print(f"[case] attention in parts {sq}x{sk} d {d} dv {dv}", flush=True)
    rng = np.random.default_rng(sq + 3 * sk + 7 * d + dv)
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((sq, d), (sk, d), (sk, dv)))
    got = _program(hip_device, q, k, v, 16).val().get()
    # a score is a sum of d products of size 1, over 4: its error, 2^-24 sqrt(d) sqrt(d) / 4 at most, is the probability's relative one
    assert_close(got.data, _exact(q, k, v, 16).reshape(-1), RED_RTOL * math.sqrt(max(sk, d)), "o")


def _heads_in_one_matrix(dev, q, w, heads, d, dv):
    """Every head's query, keys and values are columns of wider matrices, keys and values of one."""
    autodiff.set_device(dev)
    Q, KV = (autodiff.tensor(x.reshape(-1), list(x.shape)) for x in (q, w))
    out = []
    for h in range(heads):
        k0, v0 = 4 + h * d, 4 + heads * d + h * dv
        out.append(nn.Attention(Q.r(range(h * d, (h + 1) * d), 1), KV.r(range(k0, k0 + d), 1), KV.r(range(v0, v0 + dv), 1), 16))
        out[-1].forward()
        out[-1].val().keep()
    autodiff.execute()
    return out


@pytest.mark.parametrize("d,dv", [(64, 32), (128, 128)])
def test_strided_operands_are_read_where_they_are(d, dv):
    dev, heads, sk = Capture(), 3, 400
    width = heads * (d + dv) + 8
    _heads_in_one_matrix(dev, np.zeros((65, heads * d), np.float32), np.zeros((sk, width), np.float32), heads, d, dv)
    text = lower_describe(dev.proc, dev.deps)
    assert text.count("[attention_split]") == 1 and "[copy]" not in text and "[elw]" not in text, text
    assert re.search(rf"\.parts#\d+ {sk} {width} {width}\n", text) and f" 65 {sk} {heads * d} {width} {width} " in text, text


@pytest.mark.gpu
@pytest.mark.parametrize("d,dv", WIDTHS)
@pytest.mark.parametrize("sq,sk", [(65, 385), (130, 512)])
def test_strided_operands(sq, sk, d, dv, hip_device):
    """The columns that belong to no head are NaN."""
    heads = 3
    print(f"[case] attention in parts {sq}x{sk} d {d} dv {dv}, {heads} heads in one matrix", flush=True)
    rng = np.random.default_rng(sq + 3 * sk + 7 * d + dv)
    q, w = rng.standard_normal((sq, heads * d)).astype(np.float32), rng.standard_normal((sk, heads * (d + dv) + 8)).astype(np.float32)
    w[:, :4] = w[:, -4:] = np.nan
    for h, o in enumerate(_heads_in_one_matrix(hip_device, q, w, heads, d, dv)):
        k0, v0 = 4 + h * d, 4 + heads * d + h * dv
        want = _exact(q[:, h * d:(h + 1) * d], w[:, k0:k0 + d], w[:, v0:v0 + dv], 16)
        assert_close(o.val().get().data, want.reshape(-1), RED_RTOL * math.sqrt(max(sk, d)), f"o{h}")   # (as above)


@pytest.mark.gpu
@pytest.mark.parametrize("d,dv", WIDTHS)
@pytest.mark.parametrize("sq,sk", [(64, 32), (1, 33), (65, 63), (130, 255), (63, 257)])
def test_values_in_parts_where_the_other_kernel_is_faster(sq, sk, d, dv, hip_device, monkeypatch):
    monkeypatch.setenv("ADHIP_ATTENTION_PARTS", "32")
    test_values(sq, sk, d, dv, hip_device)


@pytest.mark.gpu
def test_operands_that_the_parts_cannot_represent(hip_device):
    """A value beyond bf16's largest number and an infinite one: their blocks of 64 rows are what the FP32 matrix cores make of
    them, the others are as before."""
    print("[case] attention in parts, unrepresentable operands", flush=True)
    rng = np.random.default_rng(5)
    sq, sk, d, dv = 190, 140, 64, 64
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((sq, d), (sk, d), (sk, dv)))
    v[7, 3] = np.finfo(np.float32).max
    v[9, 5] = np.inf
    got = np.asarray(_program(hip_device, q, k, v, 16).val().get().data, np.float64).reshape(sq, dv)
    want = _exact(q, k, v, 16)
    assert np.all(got[:, 5] == np.inf)
    cols = [c for c in range(dv) if c != 5]
    np.testing.assert_allclose(got[:, cols], want[:, cols], rtol=2e-4, atol=2e-4)
    q[70] = np.nan
    v[9, 5] = v[7, 3] = 1.0
    got = np.asarray(_program(hip_device, q, k, v, 16).val().get().data, np.float64).reshape(sq, dv)
    assert np.all(np.isnan(got[70]))
    rows = [r for r in range(sq) if r != 70]
    np.testing.assert_allclose(got[rows], _exact(q, k, v, 16)[rows], rtol=0, atol=2e-5)


@pytest.mark.gpu
def test_operands_that_the_parts_cannot_represent_in_parts(hip_device, monkeypatch):
    monkeypatch.setenv("ADHIP_ATTENTION_PARTS", "32")
    test_operands_that_the_parts_cannot_represent(hip_device)
