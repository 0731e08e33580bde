"""The tile and K split that each 16-bit product runs on (host only): what the
card holds, choices that were measured, and that the GPU tests' shapes reach
every kernel that can be chosen."""
import ctypes

import pytest

import test_gpu_gemm_pipe as P

DENSE, ROWS, KS, ROWS_KEY = 0, 1, 2, 3
# tiles of gemm_tile.h's kPipeTiles; three of them also split K.  A row-group key
# product can also run the 64x64 ring tile.
TILES = ((256, 256), (256, 192), (256, 128), (128, 192), (128, 128), (128, 128), (128, 64), (64, 64))
SPLIT = (4, 6, 7)
RING = len(TILES)


@pytest.fixture(scope="module")
def plan():
    from rwkv_mlx_amd import _lib
    if not _lib.LIB_PATH.exists():
        pytest.skip("not built")
    f = _lib.lib()["_ZN7rwkvmoe9gemm_planEiiiiiiPiS0_"]  # rwkvmoe::gemm_plan (internal.h)

    def run(mode, m, n, k, groups=1):
        """(tile, K split, work items that the card holds at once)"""
        cfg, ks = ctypes.c_int(-1), ctypes.c_int(-1)
        held = f(mode, m, n, n, k, groups, ctypes.byref(cfg), ctypes.byref(ks))
        assert held > 0
        return cfg.value, ks.value, held
    return run


def test_a_split_runs_in_one_round(plan):
    split = 0
    for n in (64, 192, 512, 768, 1024, 2048, 5120, 8192):
        for k in (256, 768, 2048, 4096, 8704):
            for m in (65, 90, 128, 200, 333, 512, 777, 1300):
                cfg, ks, held = plan(DENSE, m, n, k)
                bm, bn = TILES[cfg]
                assert n % bn == 0 and held == 256 * (2 if cfg in (5, 7) else 1)
                if ks > 1:
                    split += 1
                    assert cfg in SPLIT and -(-m // bm) * (n // bn) * ks <= held and k // 64 // ks >= 4
    assert split > 20


@pytest.mark.parametrize("m,n,k,most", [
    # value products of 65 to 512 tokens; the fastest of the timed tiles and splits took `most` work items or more,
    # unsplit ones 14-40% longer (260 x 768 x 3072 fp16: 10.6 us on 64x64 in 4 or 5 parts, 14.3 unsplit)
    (80, 512, 2048, 128), (260, 768, 3072, 192), (333, 1024, 3584, 192), (420, 1024, 3584, 192),
    (200, 2048, 8192, 192), (333, 2048, 8192, 192)])
def test_middle_batches_split(plan, m, n, k, most):
    cfg, ks, _ = plan(DENSE, m, n, k)
    bm, bn = TILES[cfg]
    assert ks > 1 and -(-m // bm) * (n // bn) * ks >= most


def test_gpu_shapes_reach_every_kernel(plan):
    value, key, rows_key, rows_value, kgroups = (set() for _ in range(5))
    form = lambda p: (p[0], p[1] > 1)
    for N, C, F in P.SHAPES + P.INSTANCES:
        value.add(form(plan(DENSE, N, C, F)))
        key.add(form(plan(DENSE, N, F, C)))
    for N, C, F, E, k, _ in P.ROW_GROUPS:
        rows_key.add(plan(ROWS_KEY, N * k, F, C, E)[0])
        rows_value.add(plan(ROWS, N * k, C, F, E)[0])
    for N, C, F, E, k in P.K_GROUPS:
        avg = max(1, (N * k + 128 * E + 127) // 128 * 128 // E // 64) * 64
        kgroups |= {plan(KS, F, C, avg, E)[0], plan(KS, C, F, avg, E)[0]}
    every = set(range(len(TILES)))
    assert value == key == {(c, False) for c in every} | {(c, True) for c in SPLIT}
    assert rows_key == every | {RING} and rows_value == kgroups == every
