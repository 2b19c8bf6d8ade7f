"""The dense kernels' tile plan (host code): the shapes of the GPU tile tests take the
configurations and splits that those tests are there for, and a plan keeps to its scratch."""

import pytest

from tests.gpu_util import nt_plan
from tests.test_gpu_gemm_tiles import K_MAJOR, QLORA, TILES


def test_tile_tests_reach_every_configuration():
    for m, n, k, split, *plan in TILES:
        assert nt_plan(m, n, k, split=split) == tuple(plan), (m, n, k)
    for m, n, k, a, b, *plan in K_MAJOR:
        assert nt_plan(m, n, k, a + 2 * b) == tuple(plan), (m, n, k)
    for t, n, k, forward, backward in QLORA:
        assert (nt_plan(t, n, k), nt_plan(t, k, n)) == (forward, backward), (t, n, k)
    tiles = {(c, s > 1) for *_, c, s in TILES}
    every = {(c, False) for c in range(1, 9)} | {(c, True) for c in range(1, 8)}
    assert every <= tiles
    assert {(c, s > 1) for *_, c, s in K_MAJOR} == {(1, True), (3, False), (3, True), (4, False),
                                                   (8, False), (8, True)}
    wide = {(c, False) for c in range(2, 9)} | {(2, True), (3, True), (5, True)}
    for side in (3, 4):
        assert wide <= {(row[side][0], row[side][1] > 1) for row in QLORA}


@pytest.mark.parametrize("m,n,k", [(990, 1536, 8960), (300, 3584, 18944), (523, 1536, 151936)])
def test_plan_without_scratch_is_unsplit(m, n, k):
    assert nt_plan(m, n, k)[1] > 1
    assert nt_plan(m, n, k, split=False)[1] == 1
