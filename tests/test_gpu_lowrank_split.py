"""Few HGRAVS01 pairs (several workgroups per pair): the same bits as the
right factor's and then the left factor's GEMV through a mid buffer, at
ragged rows, ranks of one to many rounds of right tiles, and pair counts on
both sides of the rule."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from tests import hk_testutil as U

pytestmark = pytest.mark.gpu
SHAPES = [(1, 32, 32, 1), (17, 32, 1024, 1), (2048, 160, 768, 1), (1000, 384, 2048, 2), (300, 288, 4096, 3),
          (4100, 64, 96, 2), (64, 2016, 160, 2), (40, 96, 256, 256), (40, 96, 256, 257), (1040, 32, 64, 512),
          (1040, 32, 64, 513)]


@pytest.fixture(scope="module")
def ctx():
    from hawking_amd.runtime import Context
    return Context(0)


@pytest.mark.parametrize("rows,rank,cols,n", SHAPES)
def test_few_pairs_match_two_launches(ctx, oracle, rows, rank, cols, n):
    from hawking_amd.organs import OrganSet, SyntheticOrgan, gemv_lowrank_set
    print("[gpu-case] lowrank split", rows, rank, cols, n, flush=True)
    sys.stdout.flush()
    tag = SHAPES.index((rows, rank, cols, n)) << 12
    key = lambda k: oracle.stream_key(U.SEED, (0x10E << 40) + tag + k)
    m = min(n, 5)
    lefts = [SyntheticOrgan(ctx, 5, rows, rank, key(2 * i), 0, group=64, sigma=0.05) for i in range(m)]
    rights = [SyntheticOrgan(ctx, 5, rank, cols, key(2 * i + 1), 0, group=64) for i in range(m)]
    ls, rs = OrganSet(ctx, [lefts[i % m] for i in range(n)]), OrganSet(ctx, [rights[i % m] for i in range(n)])
    xs = np.random.default_rng(tag).standard_normal((n, cols)).astype(np.float32)
    x, ys = ctx.to_device(xs), (rows + 3) // 4 * 4
    y1, y2 = ctx.to_device(np.full((n, ys), 3.0, np.float32)), ctx.to_device(np.full((n, ys), 3.0, np.float32))
    m1, m2 = ctx.empty((n, rank)), ctx.empty((n, rank))
    gemv_lowrank_set(ctx, ls, rs, x, cols, y1, ys, mid=m1, mid_stride=rank)
    rs.gemv(x, cols, m2, rank)
    ls.gemv(m2, rank, y2, ys)
    a = y1.download()
    assert np.array_equal(m1.download(), m2.download())
    assert np.array_equal(a, y2.download())
    assert np.all(a[:, rows:] == 3.0)
    gemv_lowrank_set(ctx, ls, rs, x, cols, y2, ys)  # mid is optional
    assert np.array_equal(a, y2.download())
    for i in {0, n - 1}:
        w = lefts[i % m].decode().astype(np.float64) @ (rights[i % m].decode().astype(np.float64) @
                                                        xs[i].astype(np.float64))
        assert oracle.relative_l2(a[i, :rows], w) < 2e-5
