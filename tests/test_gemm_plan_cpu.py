"""The prefill GEMM's launch plan, as qh_gemm_plan gives it on the host."""
import ctypes
import random

import pytest

from qwen35_amd import abi

from _util import gemm_plan as plan

CUS = 256
PROJ = {"in_proj": (2560, (8192, 4096, 32, 32)), "qkv": (2560, (8192, 1024, 1024)),
        "o": (4096, (2560,)), "gate_up": (2560, (9216, 9216)), "down": (9216, (2560,))}


def busiest_xcd(p, M, N, cus=CUS):
    """Work items per CU of the busiest XCD, item by item as the kernels hand them out."""
    tiles_m = -(-M // p["bm"])
    tiles_n = sum(-(-n // p["nstep"]) for n in N)
    count = [0] * 8
    if p["tile"] < 0:      # XCD x: N tiles x, x + 8, ... with all their row tiles and slices
        for tn in range(tiles_n):
            count[tn % 8] += tiles_m * p["S"]
    elif p["S"] == 8:      # one slice of every tile
        count = [tiles_m * tiles_n] * 8
    else:                  # the x-th eighth
        items = tiles_m * tiles_n * p["S"]
        per = -(-items // 8)
        for x in range(8):
            count[x] = max(0, min(items - x * per, per))
    return -(-max(count) // (cus // 8))


def shapes():
    r = random.Random(3)
    for M in (2, 16, 24, 64, 96, 128, 257, 288, 320, 400, 512, 576, 640, 928, 1024, 1345, 1536, 1600, 2048, 3201, 3264,
              3700, 4096):
        for K, N in PROJ.values():
            yield M, K, N, None
    for _ in range(300):
        K = 128 * r.randint(1, 130)
        yield r.randint(2, 4096), K, tuple(r.randint(1, 9000) for _ in range(r.randint(1, 4))), r.choice([0, None])


def test_plan_counts_the_busiest_xcd():
    for M, K, N, ws in shapes():
        for kb in (K // 128, 1):
            p = plan(M, K, N, ws, kb)
            assert p["load"] == busiest_xcd(p, M, N), (M, K, N, kb, p)
            if p["S"] > 1:
                ldp = sum(-(-n // p["nstep"]) for n in N) * p["nstep"]
                assert ws != 0 and p["S"] * M * ldp * 4 <= int(abi.load().qh_gemm_workspace_size(M, K))


# Rows at which two or three rounds of 64 x 128 ring tiles on the busiest XCD take 10 - 19 % longer than
# the 128 x 192 or 64 x 64 ring tiles, and up to 47 % longer than the best tile shape.
@pytest.mark.parametrize("name,rows", [("down", (1345, 1408, 1536, 1600, 3201, 3232, 3264)),
                                       ("o", (1345, 1536, 1600, 3201, 3264)), ("in_proj", (257, 288, 320))])
def test_plan_ring_rounds(name, rows):
    K, N = PROJ[name]
    for M in rows:
        p = plan(M, K, N)
        assert (p["tile"], p["bn"]) != (-1, 128), (M, p)


# Rows where a ring plan with K slices is the fastest measured.
@pytest.mark.parametrize("name,rows", [("down", (257, 288, 320, 577, 640)), ("o", (144, 160, 257, 288, 577, 640))])
def test_plan_ring_split(name, rows):
    K, N = PROJ[name]
    for M in rows:
        p = plan(M, K, N)
        assert p["tile"] == -1 and p["S"] > 1, (M, p)


def test_plan_rejects():
    lib, out = abi.load(), (ctypes.c_int * 7)()
    n = (ctypes.c_int * 1)(64)
    for M, K, nseg, np, op in ((0, 128, 1, n, out), (2, 100, 1, n, out), (2, 128, 0, n, out), (2, 128, 5, n, out),
                               (2, 128, 1, None, out), (2, 128, 1, n, None)):
        assert lib.qh_gemm_plan(M, K, nseg, np and ctypes.cast(np, ctypes.c_void_p), 1, CUS, 0,
                                op and ctypes.cast(op, ctypes.c_void_p)) == -1
