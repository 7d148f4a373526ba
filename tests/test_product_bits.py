"""That products are held to FP32's 24 bits, on every tile of the planner in every operand layout (the kernel is asserted).

Exact programs, whose results FP32 holds without rounding, so that no part of an operand can be missing, twice there or in
another's place: a matrix of 24-bit values times a selection (one power of two per column, or per row of the left operand),
and rows with one 12-bit value times a matrix of 12-bit values.  The first needs the products of the left operand's three
parts with the right one's first, the second the same the other way round, the third the product of the second parts.

And the error of sums: with each of the six products of parts the sum is rounded twice per 8 k, 1.5 k roundings of partial sums
that grow with the square root, each off by 2^-24 / sqrt(3) of them at the root mean square: 2^-25 sqrt(k) of the result's.
Products of which one term is left out are off by more than that (test_a_missing_term_is_seen, on the CPU)."""
import math
import re

import numpy as np
import pytest

from adhip import ir as IR
from adhip.device import lower_describe

TILES = [  # m, n, k, kernel
    (4096, 4096, 64, "256"), (3990, 4011, 277, "256_rim"), (2048, 4096, 96, "128"), (4100, 3900, 48, "128_rim"),
    (2048, 2048, 512, "128_pair"), (2100, 2000, 530, "128_rim_pair"), (1024, 1024, 2048, "128_splitk"), (1000, 1100, 2050, "128_rim_splitk"),
    (2048, 2048, 128, "128x64"), (2100, 2100, 260, "128x64_rim"), (1024, 2048, 64, "64"), (1500, 1100, 40, "64_rim"), (128, 128, 128, "32x32_direct"),
    (65, 63, 65, "32x32_rim_direct"), (64, 64, 2048, "32x32_splitk_direct"), (100, 130, 1500, "32x32_rim_splitk_direct"),
    (640, 1344, 256, "64_pair"), (544, 1017, 129, "64_rim_pair"), (1000, 900, 448, "64_rim_pair"), (576, 1024, 64, "64_pair"), (320, 256, 3264, "64_splitk"),
    (157, 506, 2807, "64_rim_splitk"),
    # k below 32: the FP32 matrix cores
    (4096, 4096, 16, "256_f32"), (3072, 3072, 16, "128_f32"), (2900, 3000, 16, "128_rim_f32"), (4096, 4096, 31, "128_rim_f32"), (2048, 2048, 16, "128x64_f32"),
    (2100, 2100, 7, "128x64_rim_f32"), (128, 128, 16, "64_f32"), (96, 100, 31, "64_rim_f32")]


def _values(rng, bits, *shape):
    """Values of exactly `bits` significant bits, between 1 and 2 in magnitude."""
    v = rng.integers(1 << (bits - 1), 1 << bits, size=shape) | 1
    return (v * 2.0 ** (1 - bits) * rng.choice([-1.0, 1.0], size=shape)).astype(np.float32)


def _exact_programs(m, n, k, rng):
    """(left, right, result) for each of the three kinds."""
    pos, power = (np.arange(n) * 7 + 3) % k, (2.0 ** rng.integers(-3, 4, size=n) * rng.choice([-1.0, 1.0], size=n)).astype(np.float32)
    a, b = _values(rng, 24, m, k), np.zeros((k, n), dtype=np.float32)
    b[pos, np.arange(n)] = power
    yield a, b, a[:, pos] * power
    pos, power = (np.arange(m) * 5 + 1) % k, (2.0 ** rng.integers(-3, 4, size=m) * rng.choice([-1.0, 1.0], size=m)).astype(np.float32)
    a, b = np.zeros((m, k), dtype=np.float32), _values(rng, 24, k, n)
    a[np.arange(m), pos] = power
    yield a, b, b[pos] * power[:, None]
    one, b = _values(rng, 12, m), _values(rng, 12, k, n)
    a = np.zeros((m, k), dtype=np.float32)
    a[np.arange(m), pos] = one
    yield a, b, b[pos] * one[:, None]


def _bound(k):
    return 2.0 ** -25 * math.sqrt(k)


# ---- on the CPU: what these programs see


def _parts(x):
    out = []
    for _ in range(3):
        u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
        p = ((u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000).astype(np.uint32).view(np.float32)
        out.append(p.astype(np.float64))
        x = (x - p).astype(np.float32)
    return out


TERMS = [(2, 0), (0, 2), (1, 1), (1, 0), (0, 1), (0, 0)]


def _sum_of_terms(a, b, missing=None):
    pa, pb = _parts(a), _parts(b)
    return sum(pa[i] @ pb[j] for i, j in TERMS if (i, j) != missing)


def test_the_six_terms_are_exact_here():
    for a, b, want in _exact_programs(40, 50, 64, np.random.default_rng(0)):
        assert np.array_equal(_sum_of_terms(a, b).astype(np.float32), want)
        assert np.array_equal(a.astype(np.float64) @ b.astype(np.float64), want)   # FP32 holds the result


@pytest.mark.parametrize("missing", TERMS)
def test_a_missing_term_is_seen(missing):
    rng = np.random.default_rng(1)
    assert any(not np.array_equal(_sum_of_terms(a, b, missing).astype(np.float32), want) for a, b, want in _exact_programs(40, 50, 64, rng))
    for k in (64, 277, 1024, 2050):
        a, b = rng.standard_normal((60, k), dtype=np.float32), rng.standard_normal((k, 70), dtype=np.float32)
        exact = a.astype(np.float64) @ b.astype(np.float64)
        off = np.sqrt(np.mean((_sum_of_terms(a, b, missing) - exact) ** 2) / np.mean(exact ** 2))
        all_six = np.sqrt(np.mean((_sum_of_terms(a, b) - exact) ** 2) / np.mean(exact ** 2))
        assert off > _bound(k) > 2.0 * all_six, (k, off, _bound(k), all_six)


# ---- on the GPU


def _run(hip_device, layout, a, b, kernel, w=None):
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
    cmds.append(IR.DotProduct(a="a", b="b", res="c"))
    if w is not None:
        cmds += [IR.CreateMat(w.reshape(-1), [m, n], "w"), IR.ElwAddEq(s="w", o="c")]
    proc, keep = IR.IRProcedure("main", cmds + [IR.EX()]), "c" if w is None else "w"
    assert re.findall(r"launch dot_\w+ \[dot_mfma\] kernel=(\w+)", lower_describe(proc, {keep})) == [f"adhip_gemm_{layout}_{kernel}"]
    hip_device.execute(proc, {keep})
    got = hip_device.get_tensor(keep)
    assert got.dim == [m, n]
    return np.asarray(got.data, dtype=np.float32).reshape(m, n)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["kn", "kk", "mn", "mk"])
@pytest.mark.parametrize("tile", TILES, ids=lambda t: f"{t[3]}-{t[0]}x{t[1]}x{t[2]}")
def test_exact_products(tile, layout, hip_device):
    m, n, k, kernel = tile
    print(f"[case] exact products {m}x{n}x{k} layout {layout}", flush=True)
    for i, (a, b, want) in enumerate(_exact_programs(m, n, k, np.random.default_rng(m + n + k))):
        got = _run(hip_device, layout, a, b, kernel)
        assert np.array_equal(got, want), (i, np.argwhere(got != want)[:5], np.count_nonzero(got != want))


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["kn", "kk", "mn", "mk"])
@pytest.mark.parametrize("tile", [t for t in TILES if t[3] in ("256_rim", "128_rim_pair", "32x32_rim_direct", "128_rim_f32")], ids=lambda t: f"{t[3]}-{t[0]}x{t[1]}x{t[2]}")
def test_exact_products_added_in_place(tile, layout, hip_device):
    """w += a b on the accumulators: one FP32 addition to an exact product."""
    m, n, k, kernel = tile
    print(f"[case] exact products added in place {m}x{n}x{k} layout {layout}", flush=True)
    rng = np.random.default_rng(m + n + k + 1)
    for a, b, want in _exact_programs(m, n, k, rng):
        w = rng.standard_normal((m, n), dtype=np.float32)
        assert np.array_equal(_run(hip_device, layout, a, b, kernel + "_e0", w), w + want)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["kn", "mk"])
@pytest.mark.parametrize("tile", [t for t in TILES if t[2] >= 64], ids=lambda t: f"{t[3]}-{t[0]}x{t[1]}x{t[2]}")
def test_error_of_sums(tile, layout, hip_device):
    m, n, k, kernel = tile
    print(f"[case] error of sums {m}x{n}x{k} layout {layout}", flush=True)
    rng = np.random.default_rng(m + 2 * n + 3 * k)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    exact = a.astype(np.float64) @ b.astype(np.float64)
    err = math.sqrt(float(np.mean((_run(hip_device, layout, a, b, kernel) - exact) ** 2) / np.mean(exact ** 2)))
    assert err <= _bound(k), (err, _bound(k))


@pytest.mark.gpu
@pytest.mark.parametrize("count,m,n,k,kernel", [(16, 2048, 512, 16, "kn_256_f32"), (5, 500, 500, 64, "kn_64_rim"), (5, 500, 64, 500, "kn_32x32_rim_direct"),
                                                (8, 2048, 128, 1024, "kn_64"), (8, 2048, 128, 2048, "kn_128_splitk"), (4, 1000, 132, 2050, "kn_128_rim_splitk"), (8, 2000, 132, 2050, "kn_128_rim_pair"), (6, 1536, 1536, 96, "kn_256"),
                                                (7, 1500, 1500, 50, "kn_256_rim"), (16, 100, 100, 31, "kn_64_rim_f32")])
def test_exact_products_grouped(count, m, n, k, kernel, hip_device):
    print(f"[case] {count} exact products {m}x{n}x{k}", flush=True)
    rng = np.random.default_rng(count + m + n + k)
    cmds, wants = [], []
    for i in range(count):
        a, b, want = list(_exact_programs(m, n, k, rng))[i % 3]
        cmds += [IR.CreateMat(a.reshape(-1), [m, k], f"a{i}"), IR.CreateMat(b.reshape(-1), [k, n], f"b{i}"), IR.DotProduct(a=f"a{i}", b=f"b{i}", res=f"c{i}")]
        wants.append(want)
    proc, keep = IR.IRProcedure("main", cmds + [IR.EX()]), {f"c{i}" for i in range(count)}
    assert re.findall(r"launch dots_\w+ \[dot_mfma\] kernel=(\w+)", lower_describe(proc, keep)) == [f"adhip_gemm_{kernel}_grouped"]
    hip_device.execute(proc, keep)
    for i, want in enumerate(wants):
        assert np.array_equal(np.asarray(hip_device.get_tensor(f"c{i}").data).reshape(m, n), want), i
