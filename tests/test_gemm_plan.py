"""The launch plan of the f16 GEMMs (csrc/gemm_plan.hpp) on the host: which tile a product takes,
that the GPU tests' shapes reach every tile, and that a split stays inside its workspace."""
import pytest

from gemm_plans import plans
import test_gpu_gemm_tiles as tiles

TILES, FIRST_SPLIT = 7, 4


@pytest.fixture(autouse=True)
def _compiler():
    if plans([]) is None:
        pytest.skip("no host C++ compiler")


@pytest.mark.parametrize("M,K,n", [(2047, 1536, 4096), (1900, 1536, 4096), (4000, 1536, 2048), (3000, 1536, 2560),
                                   (2047, 256, 1536), (1500, 256, 1536), (700, 1536, 8960)])
def test_products_just_over_a_round_share_the_cus(M, K, n):
    """One round of more than 256 and at most 512 tiles, two a CU: with one tile a CU these took two
    rounds, or a larger tile's long fill, and 4 to 11 % longer."""
    p = plans([(0, M, K, (n,))])[0]
    assert p["shared"] and 256 >= p["tiles"] // 2 >= 64 and p["tiles"] <= 512, p


def test_short_split_products_take_short_tiles():
    """200 tokens in 64-token tiles: two 128-token ones are 56 tokens of padding and took 15.3 us
    where these take 10.1 (K 2048) and 17.5 against 13.6 (K 4096)."""
    for p in plans([(1, 200, 2048, (1536,)), (1, 200, 4096, (1536,)), (1, 200, 6144, (1536,))]):
        assert p["bm"] == 64 and p["splits"] > 1, p


def test_gpu_shapes_reach_every_tile():
    """The plan's constants decide which tile a shape of test_gpu_gemm_tiles.py runs on."""
    plain = plans([(0, *s) for s in tiles.SHAPES])
    assert {p["cfg"] for p in plain} == set(range(TILES))
    geglu = plans([(0, M, K, (2 * n,)) for M, K, n in tiles.GEGLU_SHAPES])
    assert {p["cfg"] for p in geglu} == set(range(TILES))
    split = plans([(1, *s) for s in tiles.SPLIT_SHAPES])
    assert all(p["splits"] > 1 for p in split) and {p["cfg"] for p in split} == set(range(FIRST_SPLIT, TILES))
    # a ragged last tile of each height and width among them
    for c in range(TILES):
        mine = [(s, p) for s, p in zip(tiles.SHAPES, plain) if p["cfg"] == c]
        assert any(s[0] % p["bm"] for s, p in mine)
        assert mine[0][1]["bn"] == 128 or any(n % p["bn"] for s, p in mine for n in s[2])


def test_splits_fit_the_workspace():
    """Tickets and partials of whatever the plan takes lie inside g4a_gemm16_ws_bytes, for every
    product that may split."""
    shapes = [(1, M, K, ns) for M in (1, 2, 63, 64, 65, 127, 128, 129, 191, 200, 257, 300, 511, 640, 1000, 1024, 1281, 2047, 2560)
              for K in (64, 256, 320, 512, 576, 1024, 1536, 2048, 4096, 6144, 12288, 16384, 65536)
              for ns in ((128,), (256,), (384, 128), (1536,), (2048, 256, 256), (2560,), (4096, 512, 512), (8960,), (16256,))]
    for s, p in zip(shapes, plans(shapes)):
        if p["splits"] > 1:
            part = p["tiles"] * p["splits"] * p["bm"] * p["bn"] * 4
            assert 2048 + part <= p["ws_bytes"] and p["tiles"] * 4 <= 2048 and p["splits"] <= s[2] // 64, (s, p)
