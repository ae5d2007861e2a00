"""Small GEMV launches (row tiles' steps split over a workgroup's waves) at
the edges of their rule: one and two steps, steps that do not divide over the
waves, tile counts on both sides of each change of shape, ragged rows, and the
residual in the same launch."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from tests import hk_testutil as U

pytestmark = pytest.mark.gpu
KIND = {"q4": U.HK_Q4, "bin": U.HK_BIN, "mixed": U.HK_MIXED, "q8": 4, "u3": 5, "rice": 6}
UNIT = {"q4": 32, "bin": 128, "mixed": 64, "q8": 16, "u3": 32, "rice": 128}


@pytest.fixture(scope="module")
def ctx():
    from hawking_amd.runtime import Context
    return Context(0)


def _organ(ctx, oracle, kind, rows, cols, tag):
    from hawking_amd.organs import SyntheticOrgan
    group = {"q4": 32, "q8": 64, "u3": 64}.get(kind, 128)
    return SyntheticOrgan(ctx, KIND[kind], rows, cols, oracle.stream_key(U.SEED, (0x59 << 40) + 2 * tag),
                          oracle.stream_key(U.SEED, (0x59 << 40) + 2 * tag + 1), group=group)


def _check_rows(o, kind, x, y, rows):
    """|y - y64| per row within the engine's bound: each x to 2^-24 of its
    unit's max, one f32 rounding per unit and a few for the sums (a
    residual's products and adds: one more rounding per column at most)."""
    w = np.concatenate([o.decode(r0, n) for r0, n in rows]).astype(np.float64)
    got = np.concatenate([y[r0:r0 + n] for r0, n in rows]).astype(np.float64)
    x64, cols = x.astype(np.float64), x.size
    terms = cols // UNIT[kind] + 20 + (2 * int(0.1 * cols) if kind == "rice" else 0)
    bound = 2.0 ** -23 * np.abs(x64).max() * np.abs(w).sum(1) + terms * 2.0 ** -24 * (np.abs(w) @ np.abs(x64))
    assert np.all(np.abs(got - w @ x64) <= bound), kind


SHAPES = [("q4", 1, 32), ("q4", 17, 2048), ("q4", 100, 7168), ("q4", 33, 5248), ("q8", 1, 7168), ("q8", 40, 64),
          ("q8", 15, 1088), ("bin", 16, 512), ("bin", 17, 640), ("bin", 500, 1536), ("bin", 100, 2560),
          ("bin", 70, 7168), ("mixed", 33, 512), ("mixed", 33, 1152), ("mixed", 100, 7168), ("u3", 16, 32),
          ("u3", 50, 160), ("u3", 160, 768), ("u3", 20, 6144), ("rice", 8, 128), ("rice", 300, 1024),
          ("rice", 50, 1536), ("rice", 33, 7168)]


@pytest.mark.parametrize("kind,rows,cols", SHAPES, ids=[f"{k}-{r}x{c}" for k, r, c in SHAPES])
def test_small_launches_within_bound(ctx, oracle, kind, rows, cols):
    from hawking_amd.organs import OrganSet
    print("[gpu-case] split gemv", kind, rows, cols, flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(rows * 7 + cols)
    n, ys = 3, (rows + 3) // 4 * 4
    orgs = [_organ(ctx, oracle, kind, rows, cols, 16 * SHAPES.index((kind, rows, cols)) + i) for i in range(n)]
    xs = rng.standard_normal((n, cols)).astype(np.float32)
    xs[1, ::3] = 0.0
    xs[2, 5] *= 1e4
    y = ctx.to_device(np.full((n, ys), 7.0, np.float32))
    OrganSet(ctx, orgs).gemv(ctx.to_device(xs), cols, y, ys)
    got = y.download()
    assert np.all(got[:, rows:] == 7.0)  # nothing past the organ's rows
    for i in range(n):
        _check_rows(orgs[i], kind, xs[i], got[i], [(0, rows)])
        assert np.array_equal(got[i, :rows], orgs[i].matvec(xs[i]))


# ragged organs whose row tiles sit on both sides of each change of shape (the
# long rows: the shapes of Q4 and q8 organs of more than 16 steps)
TILES = [(k, t, 1024) for k in ("q4", "q8", "bin", "mixed", "rice") for t in (256, 257, 513, 1025, 2049, 4097)]
TILES += [("q4", t, 2176) for t in (1024, 1025, 1280, 1281, 2048, 2049, 4096, 4097)]
TILES += [(k, t, c) for k, c in (("q8", 2112), ("q4", 6176)) for t in (512, 513, 768, 769, 1024, 1025, 1280, 1281)]
TILES += [("q8", t, 4224) for t in (1025, 1536, 1537, 2048)] + [(k, t, 512) for k in ("q4", "q8") for t in (512, 513)]
TILES += [(k, t, c) for k, c in (("q8", 1088), ("mixed", 1024)) for t in (4096, 16383, 16384)]


@pytest.mark.parametrize("kind,tiles,cols", TILES, ids=[f"{k}-{t}x{c}" for k, t, c in TILES])
def test_tile_count_edges(ctx, oracle, kind, tiles, cols):
    rows = 16 * tiles - 3
    print("[gpu-case] split gemv tiles", kind, tiles, cols, flush=True)
    sys.stdout.flush()
    o = _organ(ctx, oracle, kind, rows, cols, 0x1000 + TILES.index((kind, tiles, cols)))
    x = np.random.default_rng(tiles).standard_normal(cols).astype(np.float32)
    _check_rows(o, kind, x, o.matvec(x), [(0, 48), (rows // 2, 64), (rows - 48, 48)])


STREAMED = [("bin", 64, 1536), ("mixed", 64, 1152), ("u3", 64, 800), ("q4", 64, 2048), ("q4", 64, 5248), ("q8", 64, 1088),
            ("q8", 64, 4160)]


@pytest.mark.parametrize("kind,rows,cols", STREAMED, ids=[f"{k}-{r}x{c}" for k, r, c in STREAMED])
def test_split_sums_are_the_streamed_sums(ctx, oracle, kind, rows, cols):
    """An organ alone and in a set of the streamed launch shapes (16,384 row
    tiles) gives the same bits: its terms keep their step order."""
    from hawking_amd.organs import OrganSet
    n = 16384 // (rows // 16)
    print("[gpu-case] split = streamed", kind, rows, cols, flush=True)
    sys.stdout.flush()
    base = [_organ(ctx, oracle, kind, rows, cols, 0x2000 + i) for i in range(8)]
    s = OrganSet(ctx, [base[i % 8] for i in range(n)])
    xs = np.random.default_rng(3).standard_normal((n, cols)).astype(np.float32)
    y = ctx.empty((n, rows))
    s.gemv(ctx.to_device(xs), cols, y, rows)
    got = y.download()
    for i in (0, 5, n // 2 + 3, n - 1):
        assert np.array_equal(got[i], base[i % 8].matvec(xs[i])), i


SETS = [(k, c) for k in KIND for c in (1024, 4224)]


@pytest.mark.parametrize("kind,cols", SETS, ids=[f"{k}-{c}" for k, c in SETS])
def test_bits_do_not_depend_on_the_set(ctx, oracle, kind, cols):
    """An organ's result is the same bits in sets on both sides of every change
    of the launch shape (32 row tiles an organ: 160 to 6,400 tiles)."""
    from hawking_amd.organs import OrganSet
    print("[gpu-case] split gemv, sets", kind, cols, flush=True)
    sys.stdout.flush()
    base = [_organ(ctx, oracle, kind, 509, cols, 0x4000 + i) for i in range(3)]
    xs = np.random.default_rng(cols).standard_normal((200, cols)).astype(np.float32)
    x = ctx.to_device(xs)
    alone = {i: base[i % 3].matvec(xs[i]) for i in (0, 1, 4, 9, 19, 32, 63, 99, 199)}
    for n in (2, 5, 10, 20, 33, 64, 100, 200):
        y = ctx.to_device(np.full((n, 512), 7.0, np.float32))
        OrganSet(ctx, [base[i % 3] for i in range(n)]).gemv(x, cols, y, 512)
        got = y.download()
        assert np.all(got[:, 509:] == 7.0)
        for i in alone:
            assert i >= n or np.array_equal(got[i, :509], alone[i]), (n, i)


@pytest.mark.parametrize("kind,unit", [("q4", 128), ("q8", 64)])
def test_long_rows_round_like_short_ones(ctx, oracle, kind, unit):
    """Error against 64 bits of rows of S = 7168 / unit steps.  A row of four
    steps shows what its terms round (e0); adding the blocks up adds, with a
    roundoff of 0.41 2^-24 of each partial sum and random signs, that times the
    square root of 5 + S / 32 (one chain of S steps: of S / 2, 2.1e-7 for Q4 and
    2.3e-7 for q8, beyond the bound).  8 % for the sample."""
    from hawking_amd.organs import OrganSet
    print("[gpu-case] split gemv, long rows in 64 bits", kind, flush=True)
    sys.stdout.flush()

    def error(cols, n):
        o = _organ(ctx, oracle, kind, 2048, cols, 0x5000)
        xs = np.random.default_rng(cols).standard_normal((n, cols)).astype(np.float32)
        y = ctx.to_device(np.zeros((n, 2048), np.float32))
        OrganSet(ctx, [o] * n).gemv(ctx.to_device(xs), cols, y, 2048)
        want = xs.astype(np.float64) @ o.decode().astype(np.float64).T
        return np.linalg.norm(y.download() - want) / np.linalg.norm(want)

    e0, S = error(4 * unit, 16), 7168 // unit
    for n in (2, 5, 12):
        assert error(7168, n) <= 1.08 * np.hypot(e0, 0.41 * 2.0 ** -24 * np.sqrt(5 + S / 32)), n


ONE = [(k, 300, 1024) for k in KIND] + [("rice", 8, 128), ("rice", 65536, 128), ("bin", 40, 512)]


@pytest.mark.parametrize("kind,rows,cols", ONE, ids=[f"{k}-{r}x{c}" for k, r, c in ONE])
def test_set_of_one_organ(ctx, oracle, kind, rows, cols):
    """A set of one organ (its views only in the set's device tables) is the
    organ's own call to the bit."""
    from hawking_amd.organs import OrganSet
    print("[gpu-case] split gemv, set of one", kind, rows, cols, flush=True)
    sys.stdout.flush()
    o = _organ(ctx, oracle, kind, rows, cols, 0x3000 + ONE.index((kind, rows, cols)))
    x = np.random.default_rng(rows).standard_normal(cols).astype(np.float32)
    y = ctx.to_device(np.full((1, rows + 4), 7.0, np.float32))
    OrganSet(ctx, [o]).gemv(ctx.to_device(x), cols, y, (rows + 4) // 4 * 4)
    got = y.download()[0]
    assert np.array_equal(got[:rows], o.matvec(x)) and np.all(got[rows:] == 7.0)
    edge = min(48, rows)
    _check_rows(o, kind, x, got, [(0, edge), (rows - edge, edge)])
