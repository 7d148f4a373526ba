"""Small outputs on the kernel without a staging buffer (64x64, 64x32, 32x64 and 32x32 tiles, k shared between eight
wavefronts in steps of 32): bit for bit on exact programs, at sizes beside its tiles, its steps and its wavefronts' turns."""
import numpy as np
import pytest

from test_product_bits import _bound, _exact_programs, _run

pytestmark = pytest.mark.gpu

SHAPES = [  # m, n, k, kernel
    (64, 64, 64, "32x32_direct"),           # two steps for eight wavefronts
    (96, 128, 256, "32x32_direct"),         # ... a step each
    (33, 95, 288, "32x32_rim_direct"),      # ... a ninth step; tiles moved back inside the product
    (40, 31, 257, "32x32_rim_direct"),      # fewer columns than a tile, k one beyond a step
    (3, 1000, 95, "32x32_rim_direct"),      # fewer rows than a tile, k one short of a step
    (1000, 5, 79, "32x32_rim_direct"),
    (999, 500, 289, "32x64_rim_direct"),
    (500, 999, 97, "32x64_rim_direct"),
    (1024, 768, 512, "64x64_direct"),
    (1001, 777, 543, "64x64_rim_direct"),
    (4200, 90, 65, "64x32_rim_direct"),     # 32x64 would be more than 256 blocks
    (64, 128, 1900, "32x32_rim_splitk_direct"),  # ranges of k, the last one shorter
]


@pytest.mark.parametrize("layout", ["kn", "kk", "mn", "mk"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
def test_exact_direct_products(shape, layout, hip_device):
    m, n, k, kernel = shape
    print(f"[case] exact direct product {m}x{n}x{k} layout {layout}", flush=True)
    for i, (a, b, want) in enumerate(_exact_programs(m, n, k, np.random.default_rng(m + n + k))):
        got = _run(hip_device, layout, a, b, kernel)
        assert np.array_equal(got, want), (i, np.argwhere(got != want)[:5], np.count_nonzero(got != want))


@pytest.mark.parametrize("layout", ["kn", "kk", "mn", "mk"])
@pytest.mark.parametrize("m,n,k,splits", [(33, 95, 288, 1), (40, 31, 257, 1), (31, 40, 257, 1), (3, 1000, 95, 1), (1000, 5, 79, 1), (130, 190, 1000, 3)])
@pytest.mark.parametrize("tile", ["64,64", "64,32", "32,64", "32,32"])
def test_exact_direct_products_on_every_tile(tile, m, n, k, splits, layout, hip_device, monkeypatch):
    """Also on the tiles that the planner does not take for a shape."""
    print(f"[case] exact direct product {m}x{n}x{k} layout {layout} tile {tile}", flush=True)
    monkeypatch.setenv("ADHIP_DOT_PLAN", f"{tile},{splits},8")
    kernel = tile.replace(",", "x") + "_rim" + ("_splitk" if splits > 1 else "") + "_direct"
    for i, (a, b, want) in enumerate(_exact_programs(m, n, k, np.random.default_rng(m + n + k))):
        got = _run(hip_device, layout, a, b, kernel)
        assert np.array_equal(got, want), (i, np.argwhere(got != want)[:5], np.count_nonzero(got != want))


@pytest.mark.parametrize("shape", [s for s in SHAPES if s[2] >= 256], ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
def test_error_of_direct_sums(shape, hip_device):
    """Eight sums of an eighth of k each: less than the bound for one sum over k (see test_product_bits.py)."""
    m, n, k, kernel = shape
    print(f"[case] error of a direct product {m}x{n}x{k}", flush=True)
    rng = np.random.default_rng(m + 2 * n + 3 * k)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    exact = a.astype(np.float64) @ b.astype(np.float64)
    err = float(np.sqrt(np.mean((_run(hip_device, "kn", a, b, kernel) - exact) ** 2) / np.mean(exact ** 2)))
    assert err <= _bound(k), (err, _bound(k))
