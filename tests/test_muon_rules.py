"""The rules that pick a Muon batch's padding and GEMM tile edges, and the FLOPs counted from them."""
import pytest

from morph_amd import _lib, muon


def pad(rows, cols, count, steps=5):
    return _lib.lib().morph_muon_pad_multiple(rows, cols, count, steps)


def edge(m, n, k, batch, flags=0, epilogue=0):
    return _lib.lib().morph_gemm_tile_edge(m, n, k, batch, flags, epilogue)


@pytest.mark.parametrize("rows,cols,count", [(3072, 6144, 42), (6144, 3072, 1), (768, 2048, 4), (768, 2048, 36),
                                             (192, 448, 12), (700, 330, 1), (330, 700, 64), (900, 450, 8),
                                             (512, 768, 70)])
def test_executed_flops_are_those_of_the_tiles(rows, cols, count):
    """Every tile of every product, counted one by one: the upper triangle of A and B'."""
    m, n = min(rows, cols), max(rows, cols)
    flops = 0
    for c in [64] * (count // 64) + [count % 64] * (count % 64 > 0):
        u = pad(rows, cols, c)
        mp, np_ = -(-m // u) * u, -(-n // u) * u
        for k, epilogue in ((np_, 0), (mp, 1)):
            e = edge(mp, mp, k, c, _lib.GEMM_SYMMETRIC, epilogue)
            flops += c * sum(2 * e * e * k for i in range(mp // e) for j in range(i, mp // e))
        flops += c * 2 * mp * np_ * mp
    assert muon.ns_executed_flops(rows, cols, count, 5) == 5 * flops
    assert muon.ns_executed_flops(rows, cols, count, 0) == 0


def test_executed_flops_of_one_workgroup_chains():
    # 200 x 96: X [96, 224], A [96, 96]: six 32 x 32 tiles, two for each of three waves
    assert pad(200, 96, 1) == 0
    assert muon.ns_executed_flops(200, 96, 1, 5) == 2 * 5 * (6 * 1024 * (224 + 96) + 96 * 96 * 224)
    # 128 x 480: ten tiles on six waves, which compute twelve
    assert muon.ns_executed_flops(128, 480, 64, 1) == 64 * 2 * (12 * 1024 * (480 + 128) + 128 * 128 * 480)
    assert pad(200, 96, 1, 0) > 0  # no iterations: the general passes


def test_the_256_edge_has_three_stages_of_k_at_least():
    """By its costs: the 128 edge alone runs launches of one or two stages (K of 64 or 128)."""
    short = {edge(m, n, k, b, f, e) for m in range(256, 2049, 256) for n in range(256, 4097, 256)
             for k in (64, 128) for b in (1, 2, 3, 5, 8, 13, 21, 34, 48, 64, 100, 1000)
             for f, e in ((0, 0), (0, 1), (0, 2), (_lib.GEMM_SYMMETRIC, 0), (_lib.GEMM_SYMMETRIC, 1))
             if f == 0 or m == n}
    assert short == {64, 128}
    assert edge(256, 1024, 192, 53) == 256


def test_bad_arguments():
    assert pad(0, 8, 1) < 0 and pad(8, 8, 65) < 0 and pad(8, 8, 1, -1) < 0
    assert edge(64, 64, 32, 1) < 0 and edge(96, 64, 64, 1) < 0 and edge(64, 64, 64, 0) < 0
    assert edge(64, 64, 64, 1, 4) < 0 and edge(64, 64, 64, 1, 0, 3) < 0
