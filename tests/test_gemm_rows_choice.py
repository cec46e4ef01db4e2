"""Which products the kernel that multiplies a batch of rows straight from the int8 weights takes: host arithmetic of the library,
no GPU call."""
import os
import random
import subprocess
import sys

import pytest

from deepj_amd import HipNative

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("k,n", [(768, 50257), (1500, 8001), (2048, 4001), (4096, 16385), (256, 256), (768, 768)])
@pytest.mark.parametrize("norm", [False, True])
def test_long_batches_stay_on_the_larger_tiles(k, n, norm):
    """Past the rows it was measured at: at 1500 rows and more against a weight that the fp16 GEMM refuses it takes up to 1.7
    times k_gemm_q8's time."""
    assert HipNative.q8GemmRowsTile(300, 4096, 16385, norm)[0]
    for m in (769, 1024, 1500, 2048, 4096):
        for alloc_free in (False, True):
            assert HipNative.q8GemmRowsTile(m, k, n, norm, alloc_free=alloc_free) == (0, 0, 1)


def test_every_choice_is_one_the_kernel_has():
    rng = random.Random(5)
    seen = set()
    for _ in range(20000):
        m, k, n = (int(round(2 ** rng.uniform(a, b))) for a, b in ((1, 9.6), (3, 14), (1, 16)))
        norm, prepared, alloc_free = (rng.random() < 0.5 for _ in range(3))
        rows, cols, shares = HipNative.q8GemmRowsTile(m, k, n, norm, prepared, alloc_free)
        seen.add((rows, cols, shares))
        if not rows:
            continue
        assert rows in (32, 64) and cols in (32, 64, 96) and shares in (1, 2, 4)
        if shares > 1:                                   # columns in pairs; a chunk of 128 k for each of a share's wavefronts' turns
            assert n % 2 == 0 and not alloc_free and -(-k // 128) >= 2 * shares
        if not alloc_free:                               # never where the fp16 GEMM is taken
            assert not (HipNative.q8GemmTilePrepared if prepared else HipNative.q8GemmTile)(m, k, n)[0]
    assert len(seen) == 12                               # eleven and none


def test_a_product_whose_rows_are_ready_is_taken_in_more_cases():
    """Right behind the product that leaves its rows ready it runs there wherever it does by itself without a normalisation."""
    rng, more = random.Random(6), 0
    for _ in range(5000):
        m, k, n = (int(round(2 ** rng.uniform(a, b))) for a, b in ((1, 10), (3, 14), (3, 14)))
        for prepared in (False, True):
            alone, behind = HipNative.q8GemmRowsTile(m, k, n, prepared=prepared), HipNative.q8GemmRowsTileBehind(m, k, n, prepared)
            assert behind[0] or not alone[0], (m, k, n, prepared)
            more += behind[0] > 0 and not alone[0]
    assert more > 100 and HipNative.q8GemmRowsTileBehind(0, 64, 64) == (0, 0, 1)
    assert HipNative.q8GemmRowsTile(64, 11008, 4096) == (0, 0, 1) and HipNative.q8GemmRowsTileBehind(64, 11008, 4096) == (32, 64, 2)


def test_the_switch_that_keeps_every_gemm_on_k_gemm_q8():
    shapes = [(30, 2048, 6144), (64, 4096, 22016), (200, 2048, 11264), (512, 2048, 6144), (200, 768, 2304)]
    program = f"""
from deepj_amd import HipNative as H
for m, k, n in {shapes}:
    for norm in (False, True):
        for alloc_free in (False, True):
            assert H.q8GemmRowsTile(m, k, n, norm, alloc_free=alloc_free) == (0, 0, 1), (m, k, n)
    assert H.q8GemmPath(m, k, n) == H.q8GemmTilePrepared(m, k, n)[0] == 0, (m, k, n)
"""
    subprocess.run([sys.executable, "-c", program], check=True, timeout=120, cwd=ROOT, env=dict(os.environ, DEEPJ_HIP_GEMM_F16="0"))
    for m, k, n in shapes:
        assert HipNative.q8GemmRowsTile(m, k, n, norm=True)[0] or HipNative.q8GemmPath(m, k, n)
