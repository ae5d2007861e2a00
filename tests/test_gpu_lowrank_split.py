"""Few HGRAVS01 pairs (several workgroups per pair): the same bits as the
right factor's and then the left factor's GEMV through a mid buffer, at
ragged rows, ranks of one to many rounds of right tiles, inputs on both sides
of the widest that fit its LDS (3,072 and 4,096 columns at rank 288), and pair
counts on both sides of the rule."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from tests import hk_testutil as U

pytestmark = pytest.mark.gpu
SHAPES = [(1, 32, 32, 1), (17, 32, 1024, 1), (2048, 160, 768, 1), (1000, 384, 2048, 2), (300, 288, 3072, 3),
          (300, 288, 4096, 3),
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


OVERLAPS = [(2048, 160, 768, 1), (300, 64, 1024, 3), (64, 2016, 160, 2)]


@pytest.mark.parametrize("rows,rank,cols,n", OVERLAPS)
def test_few_pairs_in_place(ctx, oracle, rows, rank, cols, n):
    """A pair's y or mid over its x, and mid inside y: the bits of separate
    buffers (a pair in one workgroup has read what it overwrites)."""
    from hawking_amd.organs import HgravS01LowRank, OrganSet, SyntheticOrgan, gemv_lowrank_set
    print("[gpu-case] lowrank in place", rows, rank, cols, n, flush=True)
    sys.stdout.flush()
    key = lambda k: oracle.stream_key(U.SEED, (0x10F << 40) + rows * 16 + k)
    lefts = [SyntheticOrgan(ctx, 5, rows, rank, key(2 * i), 0, group=64, sigma=0.05) for i in range(n)]
    rights = [SyntheticOrgan(ctx, 5, rank, cols, key(2 * i + 1), 0, group=64) for i in range(n)]
    ls, rs = OrganSet(ctx, lefts), OrganSet(ctx, rights)
    xs = np.random.default_rng(rows).standard_normal((n, cols)).astype(np.float32)
    y, st = ctx.empty((n, rows)), 4096

    def call(x, x_stride, mid, mid_stride, out, out_stride):
        ctx.call("hk_gemv_lowrank_set", ls.h, rs.h, x, x_stride, mid, mid_stride, out, out_stride, ctx.stream)

    gemv_lowrank_set(ctx, ls, rs, ctx.to_device(xs), cols, y, rows)
    want = y.download()
    rec = np.zeros((n, st), np.float32)
    rec[:, :cols] = xs
    for at in (0, 4, cols // 8 * 4):  # y, then mid, from x's start and from inside it
        b = ctx.to_device(rec)
        call(b.ptr, st, None, 0, b.offset(at), st)
        assert np.array_equal(b.download()[:, at:at + rows], want), ("y over x", at)
        b = ctx.to_device(rec)
        call(b.ptr, st, b.offset(at), st, y.ptr, rows)
        assert np.array_equal(y.download(), want), ("mid over x", at)
    if rank <= rows:
        x = ctx.to_device(xs)
        call(x.ptr, cols, y.ptr, rows, y.ptr, rows)
        assert np.array_equal(y.download(), want), "mid in y"
    # x and y side by side in a record do not overlap
    b = ctx.to_device(rec)
    call(b.ptr, st, None, 0, b.offset(cols), st)
    assert np.array_equal(b.download()[:, cols:cols + rows], want)
    if rows <= cols:
        x = ctx.to_device(xs[0])
        HgravS01LowRank(lefts[0], rights[0]).matvec_device(x, x)
        assert np.array_equal(x.download()[:rows], want[0])
