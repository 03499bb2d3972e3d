"""Which kernel a call's shape is given, at the lines where it changes (csrc/*_launch.h), on the host alone and for the 256 compute
units that the lines were measured on.  The results that either side of a line computes are the GPU tests' matter."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
UNITS = 256
TEAM, LONE = 4, 1  # waves that share sixteen tokens


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    library = tmp_path_factory.mktemp("rules") / "librules.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", str(ROOT / "tests/launch_rules.cpp"), "-o", str(library)],
                   check=True)
    return C.CDLL(str(library))


def teams(rules, waves, depth, passes=0, count=1, flying=1):
    out = (C.c_int * 4)()
    rules.w16_teams(passes, waves, count, depth, flying, UNITS, out)
    return dict(zip(("teams", "blocks", "waves", "rows"), out))


@pytest.mark.parametrize("depth", [1, 4, 8])
@pytest.mark.parametrize("waves,roles", [(4, TEAM), (256, TEAM), (1024, TEAM), (1025, LONE), (3072, LONE), (8192, LONE)])
def test_width16_passes_of_their_own(rules, depth, waves, roles):
    """Beyond four teams a unit both passes go to lone waves, like a step's."""
    for passes in (0, 1, 2):
        chosen = teams(rules, waves, depth, passes)
        assert chosen["waves"] == roles
        assert chosen["teams"] * chosen["blocks"] >= waves > chosen["teams"] * (chosen["blocks"] - 1)
        assert not (passes and chosen["rows"])  # the backward pass is another launch


@pytest.mark.parametrize("waves,evaluated,with_gradient", [(1025, 5, 5), (2048, 8, 8), (2049, 5, 5), (2560, 5, 5), (2561, 6, 4), (3072, 6, 4), (3073, 7, 7),
                                                           (4096, 8, 8), (4097, 6, 6), (4608, 6, 6), (8192, 8, 8), (8193, 7, 7), (65536, 8, 8)])
def test_width16_lone_waves_are_shared_out_evenly(rules, waves, evaluated, with_gradient):
    """Every unit has as many blocks, of eight lone waves at most, and every block as many waves."""
    for passes, share in ((0, with_gradient), (1, evaluated), (2, with_gradient)):
        chosen = teams(rules, waves, 8, passes=passes)
        assert chosen["teams"] == share
        per_unit = -(-chosen["blocks"] // UNITS)
        assert (share - 1) * per_unit * UNITS < waves <= share * per_unit * UNITS


@pytest.mark.parametrize("depth", [4, 8])
@pytest.mark.parametrize("flying,last", [(2, 224), (3, 179), (4, 149)])
def test_width16_batches_in_flight_fit_side_by_side(rules, depth, flying, last):
    """A unit has room for one block of teams: on streams of their own, `flying` batches' blocks are no more than the units - an eighth more
    with the rows in LDS - unless blocks of four teams, the largest, already are.  Beyond `last` blocks of four teams' tokens, lone waves."""
    for blocks in range(1, last + 40):
        chosen = teams(rules, 4 * blocks, depth, flying=flying)
        assert chosen["waves"] == (TEAM if blocks <= last else LONE), blocks
        if blocks <= last:
            places = UNITS * 9 // 8 if chosen["rows"] else UNITS
            assert chosen["blocks"] * flying <= places or (chosen["teams"] == 4 and not chosen["rows"]), (blocks, chosen)
        assert chosen["teams"] * chosen["blocks"] >= 4 * blocks > chosen["teams"] * (chosen["blocks"] - 1)


@pytest.mark.parametrize("depth,K,blocks,steps,shared", [
    (8, 1, 1, 1, True), (4, 1, 4000, 64, True),                           # one batch: its launch is all there is
    (8, 2, 1, 2, True), (8, 2, 128, 2, True), (8, 2, 160, 2, False),      # depth 8, two in flight
    (8, 3, 1, 3, True), (8, 3, 40, 3, True), (8, 3, 1, 6, True), (8, 3, 96, 4, False),
    (8, 4, 1, 1, False), (8, 4, 1, 3, True), (8, 4, 1, 5, True), (8, 4, 40, 4, True), (8, 4, 96, 4, False), (8, 4, 128, 4, False),
    (8, 16, 16, 16, True), (8, 8, 200, 8, False),
    (4, 2, 1, 1, False), (4, 2, 1, 3, True), (4, 2, 96, 2, True), (4, 4, 128, 4, True), (4, 4, 160, 2, False), (4, 8, 160, 2, False),
    (4, 4, 200, 4, False), (4, 8, 200, 8, False),
])
def test_width16_shared_launches(rules, depth, K, blocks, steps, shared):
    """The better one of the two as they were measured, where they differ by 5 % or more (csrc/width16_launch.h)."""
    assert bool(rules.w16_shares_launches(depth, K, min(K, 4), blocks, steps, UNITS)) is shared


PLAIN, GELU, GELU_BACKWARD, GELU_ONLY = 0, 2, 3, 5  # epilogues


@pytest.mark.parametrize("M,N,K,forward,gelu,backward,gelu_backward", [
    # test_gpu_gemm.py
    (16384, 1024, 256, 0, 0, 0, 0), (16384, 1024, 512, 0, 256, 128, 128), (8192, 2048, 1024, 256, 256, 128, 128),
    (16384, 3072, 1024, 256, 0, 256, 256), (16384, 1024, 4096, 256, 256, 256, 256),
    # test_gpu_gemm_columns.py
    (10240, 1024, 1152, 256, 256, 192, 192), (4096, 3584, 896, 256, 256, 0, 0), (12288, 768, 896, 192, 0, 0, 0),
    (10240, 640, 768, 128, 128, 0, 0), (16384, 1024, 640, 0, 256, 128, 0), (16640, 1280, 1024, 128, 128, 128, 0),
    (8320, 896, 896, 128, 128, 128, 128), (12416, 768, 768, 192, 0, 192, 0), (10368, 1024, 1152, 256, 256, 192, 192),
    (4224, 3072, 768, 256, 0, 0, 0),
])
def test_columns_of_256_row_tiles(rules, M, N, K, forward, gelu, backward, gelu_backward):
    """What the shapes of the kernel's tests are given; 0: 128-row blocks."""
    def columns(N, K, mode):
        return rules.gemm_columns_of_256(M, N, K, mode, UNITS)

    assert (columns(N, K, PLAIN), columns(N, K, GELU)) == (forward, gelu)
    assert columns(N, K, GELU_ONLY) == gelu
    assert (columns(K, N, PLAIN), columns(K, N, GELU_BACKWARD)) == (backward, gelu_backward)


@pytest.mark.parametrize("M,N,K", [(3584, 1920, 1024), (10240, 768, 1024), (4224, 1536, 1280), (2176, 3072, 1024), (4352, 3456, 2816), (13312, 1152, 3840)])
def test_gelu_backward_where_two_blocks_of_128_columns_fit_every_unit(rules, M, N, K):
    """22 to 29 % slower on 256-row tiles of 192 columns, which fill half of a round or of the second one (M x N outputs)."""
    assert rules.gemm_columns_of_256(M, N, K, GELU_BACKWARD, UNITS) == 0
    assert rules.gemm_columns_of_256(4096, 2304, 2304, GELU_BACKWARD, UNITS) == 192  # 216 tiles: 10 % faster


def test_columns_of_256_row_tiles_in_several_rounds(rules):
    """The shapes of test_gpu_gemm_columns_rounds.py: more tiles than units, and half a tile of rows at the end."""
    import test_gpu_gemm_columns_rounds as shapes
    for mode, listed in ((PLAIN, shapes.PLAIN), (GELU, shapes.GELU), (GELU_ONLY, shapes.GELU), (GELU_BACKWARD, shapes.GELU_BACKWARD)):
        for M, N, K, columns in listed:
            if mode == GELU_BACKWARD:
                N, K = K, N
            assert rules.gemm_columns_of_256(M, N, K, mode, UNITS) == columns
            assert M % 256 == 128 and (M + 255) // 256 * (N // columns) > UNITS
    assert rules.gemm_columns_of_256(10240, 640, 768, GELU_ONLY, UNITS) == 128
    assert rules.gemm_columns_of_256(4096, 4096, 1024, GELU_ONLY, UNITS) == 256  # test_gpu_evaluate.py
