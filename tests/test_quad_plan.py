"""CPU: the launch plans of the four-wave GEMM (gemm_quad.hip), from the built library itself
(qd_gemm_quad_plan: the decision the launchers take), and that the GPU tests run what they pick."""

import ctypes as C

import pytest

from test_gpu_quad import INSTANCES, ROWS, SHAPES

ROOM = 1 << 40
EPI = {"qkv": (0,), "o": (1,), "gu": (2,), "down": (1,)}
KINDS = {0: "plain", 1: "plain", 2: "swiglu"}


@pytest.fixture(scope="module")
def plan():
    from qdecode import _lib

    def f(M, N, K, epi, room=ROOM):
        out = (C.c_int64 * 6)()
        if _lib.LIB.qd_gemm_quad_plan(M, N, K, epi, room, out) != 1:
            return None
        mt, nt, nbuf, splits, ks_per, outs = out
        return {"key": ("split" if splits > 1 else KINDS[epi], mt, nt), "nbuf": nbuf, "splits": splits,
                "ks_per": ks_per, "outs": outs}
    return f


def test_instances_are_what_their_shapes_launch(plan):
    for key, (M, N, K) in INSTANCES.items():
        for epi in (2,) if key[0] == "swiglu" else (0, 1):
            assert plan(M, N, K, epi)["key"] == key


@pytest.mark.parametrize("name", list(SHAPES))
def test_gpu_tests_cover_the_projections(plan, name):
    """Every tile shape of every row count from 33 to 64 and 257 to 16384, with and without room for
    split partials, is an instance that runs; the unsplit ones from 257 rows run at the projection's
    own size too."""
    N, K = SHAPES[name]
    for epi in EPI[name]:
        own = {plan(M, N, K, epi)["key"] for M in ROWS}
        for M in [*range(33, 65), *range(257, 16385)]:
            for room in (ROOM, 0):
                key = plan(M, N, K, epi, room)["key"]
                assert key in INSTANCES, (M, room)
                if M >= 1024 or (M > 256 and room and key[0] != "split"):
                    assert key in own, (M, key)


def test_plans_cover_their_product(plan):
    """K splits without an empty one, blocks no wider than the tile and whole groups of eight columns,
    stage buffers within the LDS."""
    for M in (33, 50, 64, 257, 500, 777, 1023, 1024, 2500, 9000):
        for N in (128, 256, 640, 2560, 6144, 9728, 30720):
            for K in (128, 640, 2560, 9728):
                for epi in (0, 1, 2):
                    for room in (0, 3 * M * N, ROOM):
                        p = plan(M, N, K, epi, room)
                        if p is None:            # the LDS-staged kernel's
                            assert M <= 64 and N <= 2048 and K % 512 == 0
                            continue
                        kind, mt, nt = p["key"]
                        S, ks = p["splits"], p["ks_per"]
                        assert (S - 1) * ks < K // 64 <= S * ks
                        assert S == 1 or (epi != 2 and S * M * N <= room)
                        assert 0 < p["outs"] <= (16 if epi == 2 else 32) * nt and p["outs"] % 8 == 0
                        assert (p["nbuf"] * 32 * (mt + nt) * 8 + (16 if p["nbuf"] == 2 else 0)) * 16 <= 160 * 1024
