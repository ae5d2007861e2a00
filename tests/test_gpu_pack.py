"""The device packers at the edges of their lane groups, bit for bit against
the oracle: one group, partial last waves, ragged 3-bit tails, weights that
are not 16-byte aligned, and binary groups whose magnitudes span so much that
the f64 sum of |w| depends on its order."""
from __future__ import annotations

import ctypes as C
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from hawking_amd.runtime import Context
    return Context(0)


def _weights(n, seed):
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal(n) * 0.02).astype(np.float32)
    w[::7] = -0.0
    # every other 128-group spans 2^-60 .. 2^6, so partial sums round
    wide = np.ldexp(rng.standard_normal(n), rng.integers(-60, 7, n)).astype(np.float32)
    g = np.arange(n) // 128 % 2 == 1
    w[g] = wide[g]
    w[-min(n, 5):] = np.float32(1e-42)  # subnormals
    return w


def _device(ctx, w, shift):
    """w on the device, `shift` floats past a 16-byte boundary."""
    buf = ctx.to_device(np.concatenate([np.zeros(shift, np.float32), w]))
    return buf, buf.offset(shift)


@pytest.mark.parametrize("groups,shift", [(1, 0), (1, 1), (3, 2), (33, 0), (130, 3), (2049, 0)])
def test_packers_bit_exact_at_group_edges(ctx, oracle, groups, shift):
    print("[gpu-case] packers", groups, shift, flush=True)
    sys.stdout.flush()

    def run(fn, w, scales, code_bytes, *shape):
        buf, p = _device(ctx, w, shift)
        s, c = ctx.empty(scales, np.uint16), ctx.empty(code_bytes, np.uint8)
        ctx.call(fn, p, *shape, s.ptr, c.ptr, ctx.stream)
        return s.download(), c.download()

    w = _weights(groups * 128, 100 + groups)
    cases = [("hk_pack_bin", 128, 16, (groups, 128), oracle.bin_pack(w.reshape(groups, 128))),
             ("hk_pack_q8", 64, 64, (groups, 128), oracle.uniform_pack(w, groups, 128, 8, 64)),
             ("hk_pack_q2", 64, 16, (w.size,), oracle.q2_pack(w))]
    if shift == 0:  # the Q4 packer takes 16-byte aligned weights only
        cases += [("hk_pack_q4", G, G // 2, (groups, 128, G), oracle.q4_pack(w.reshape(groups, 128), G))
                  for G in (32, 64, 128)]
    for fn, G, per, shape, (rs, rc) in cases:
        s, c = run(fn, w, w.size // G, w.size // G * per, *shape)
        assert np.array_equal(s, rs), (fn, shape)
        assert np.array_equal(c, np.asarray(rc).reshape(-1)), (fn, shape)
    for count in (w.size, w.size - 1, w.size - 61, max(1, w.size - 127)):
        g3 = (count + 63) // 64
        s, c = run("hk_pack_u3", w[:count].copy(), g3, g3 * 24, C.c_size_t(count))
        rs, rc = oracle.uniform_pack(w[:count], 1, count, 3, 64)
        assert np.array_equal(s, rs) and np.array_equal(c, rc), ("hk_pack_u3", count)


PACKERS = [("hk_pack_q4", 32, 16), ("hk_pack_bin", 128, 16), ("hk_pack_q8", 64, 64), ("hk_pack_q2", 64, 16),
           ("hk_pack_u3", 64, 24)]


@pytest.mark.parametrize("fn,group,per", PACKERS)
def test_packers_flag_nonfinite_and_clear(ctx, oracle, fn, group, per):
    """A NaN or infinity anywhere (first, last and inside), and a scale past
    f16 where the format refuses one, is HK_E_NONFINITE; the next call on the
    same context is clean and packs the same bytes."""
    from hawking_amd._lib import HK_E_NONFINITE, HawkingError
    print("[gpu-case] packers non-finite", fn, flush=True)
    sys.stdout.flush()
    rows, cols = 33, 384
    n = rows * cols
    shape = {"hk_pack_q4": (rows, cols, group), "hk_pack_q2": (C.c_size_t(n),),
             "hk_pack_u3": (C.c_size_t(n),)}.get(fn, (rows, cols))
    w = (np.random.default_rng(5).standard_normal(n) * 0.02).astype(np.float32)
    s, c = ctx.empty(n // group, np.uint16), ctx.empty(n // group * per, np.uint8)

    def pack(v):
        ctx.call(fn, ctx.to_device(v).ptr, *shape, s.ptr, c.ptr, ctx.stream)
        return s.download(), c.download()

    want = pack(w)
    bad = [(i, v) for i in (0, 777, n - 1) for v in (np.nan, np.inf, -np.inf)]
    if fn not in ("hk_pack_bin", "hk_pack_q2"):  # (those two store an infinite scale)
        bad.append((n // 2, np.float32(3e38)))
    for i, v in bad:
        b = w.copy()
        b[i] = v
        with pytest.raises(HawkingError) as e:
            pack(b)
        assert e.value.code == HK_E_NONFINITE, (i, v)
        got = pack(w)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), (i, v)
