"""The fused terminal head over the lm_head kinds it takes (q8, Q4, binary)
and one it must leave to the separate launches (a binary lm_head with a
residual), at small and ragged vocabularies and its widest hidden size."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from tests import hk_testutil as U

pytestmark = pytest.mark.gpu
KIND = {"q4": U.HK_Q4, "bin": U.HK_BIN, "q8": 4, "rice": 6}


@pytest.fixture(scope="module")
def ctx():
    from hawking_amd.runtime import Context
    return Context(0)


def _organ(ctx, oracle, kind, rows, cols):
    from hawking_amd.organs import SyntheticOrgan
    return SyntheticOrgan(ctx, KIND[kind], rows, cols, oracle.stream_key(U.SEED, (0x4EAD << 32) + rows * 8 + cols),
                          0, group={"q4": 32, "q8": 64}.get(kind, 128))


CASES = [(k, v, h, c) for k in sorted(KIND)
         for v, h, c in ((1, 128, 0), (15, 640, 3), (257, 8192, 1), (4101, 1024, 100), (70000, 512, 331))]
CASES.append(("q8", 140001, 2048, 7))  # weights larger than the Infinity Cache
# row tiles on both sides of each change of the waves a tile
CASES += [(k, v, h, 5) for k, h in (("q8", 2048), ("q4", 4096)) for v in (12288, 12289)]
CASES += [(k, v, h, 5) for k, h in (("q8", 1024), ("q4", 2048)) for v in (8192, 8193, 32768, 32769)]


@pytest.mark.parametrize("kind,vocab,hidden,cut", CASES)
def test_head_kinds(ctx, oracle, kind, vocab, hidden, cut):
    from hawking_amd.head import TerminalHead
    print("[gpu-case] head", kind, vocab, hidden, flush=True)
    sys.stdout.flush()
    lm = _organ(ctx, oracle, kind, vocab, hidden)
    rng = np.random.default_rng(vocab + hidden)
    h = rng.standard_normal(hidden).astype(np.float32)
    nw = (rng.standard_normal(hidden) * 0.02).astype(np.float32)
    head = TerminalHead(ctx, nw, lm, vocab - cut)
    for _ in range(2):  # the second call finds the key cleared
        tok = head.greedy(h)
        logits, xn = head.logits.download(), head.xn.download()
        assert tok == oracle.argmax_greedy(logits, vocab - cut)
    # the logits are the lm_head's own GEMV of xn, to the bit
    assert np.array_equal(logits, lm.matvec(xn))
    # each xn to a few roundings, the logits to the engine's bound on it
    assert np.all(np.abs(xn - oracle.rmsnorm_1p(h, nw, 1e-6)) <= 2e-6 * np.abs(xn) + 1e-30)
    w, x64 = lm.decode(0, min(vocab, 300)).astype(np.float64), xn.astype(np.float64)
    terms = hidden // 16 + 20 + (2 * int(0.1 * hidden) if kind == "rice" else 0)
    bound = 2.0 ** -23 * np.abs(x64).max() * np.abs(w).sum(1) + terms * 2.0 ** -24 * (np.abs(w) @ np.abs(x64))
    assert np.all(np.abs(logits[:300] - w @ x64) <= bound)
    assert head.pick.download().tolist() == [0, 0]


@pytest.mark.parametrize("kind", ["q4", "bin"])
def test_head_kinds_flag_nonfinite(ctx, oracle, kind):
    from hawking_amd._lib import HawkingError
    from hawking_amd.head import TerminalHead
    print("[gpu-case] head non-finite", kind, flush=True)
    sys.stdout.flush()
    head = TerminalHead(ctx, np.zeros(512, np.float32), _organ(ctx, oracle, kind, 300, 512))
    h = np.ones(512, np.float32)
    for value in (np.inf, np.nan):
        bad = h.copy()
        bad[511] = value
        with pytest.raises(HawkingError):
            head.greedy(bad)
        assert int(head.token.download()[0]) == -1
    assert head.greedy(h) == oracle.argmax_greedy(head.logits.download())


@pytest.mark.parametrize("kind", sorted(KIND))
def test_head_in_place(ctx, oracle, kind):
    """xn over hidden and the logits over hidden: hidden has been read when
    either is written."""
    from hawking_amd.head import TerminalHead
    print("[gpu-case] head in place", kind, flush=True)
    sys.stdout.flush()
    lm = _organ(ctx, oracle, kind, 70000, 2048)
    rng = np.random.default_rng(11)
    h, nw = rng.standard_normal(2048).astype(np.float32), (rng.standard_normal(2048) * 0.02).astype(np.float32)
    head = TerminalHead(ctx, nw, lm)
    want = head.greedy(h)
    want_xn = head.xn.download()
    for case in ("xn", "logits"):
        head = TerminalHead(ctx, nw, lm)
        if case == "xn":
            head.xn.upload(h)
            head.greedy_device(head.xn)
        else:
            head.logits.upload(np.concatenate([h, np.zeros(70000 - 2048, np.float32)]))
            head.greedy_device(head.logits)
        assert ctx.device_status() == 0
        xn, logits = head.xn.download(), head.logits.download()
        assert np.all(np.abs(xn - want_xn) <= 2e-6 * np.abs(want_xn)), case
        assert np.array_equal(logits, lm.matvec(xn)), case
        assert int(head.token.download()[0]) == oracle.argmax_greedy(logits) == want, case


@pytest.mark.parametrize("kind,hidden", [(k, h) for k in sorted(KIND) for h in (640, 8192)])
def test_head_norm_weight_alignment(ctx, oracle, kind, hidden):
    """The norm weight at any 4-byte address gives the same bits."""
    from hawking_amd.head import TerminalHead
    print("[gpu-case] head norm weight alignment", kind, hidden, flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(hidden)
    h, nw = rng.standard_normal(hidden).astype(np.float32), (rng.standard_normal(hidden) * 0.02).astype(np.float32)
    head = TerminalHead(ctx, nw, _organ(ctx, oracle, kind, 300, hidden))
    want = head.greedy(h)
    xn, logits = head.xn.download(), head.logits.download()
    hd = ctx.to_device(h)
    for shift in (1, 2, 3):
        w = ctx.to_device(np.concatenate([np.full(shift, 9.0, np.float32), nw, np.full(4, 9.0, np.float32)]))
        ctx.call("hk_terminal_greedy", hd.ptr, w.offset(shift), head.eps, head.lm_head.h, 300, head.xn.ptr,
                 head.logits.ptr, head.pick.ptr, head.token.ptr, ctx.stream)
        assert ctx.device_status() == 0 and int(head.token.download()[0]) == want, shift
        assert np.array_equal(head.xn.download(), xn) and np.array_equal(head.logits.download(), logits), shift
