"""The batched block's launch shapes: gate/up with one or two workgroups a CU,
routed and shared intermediates
of different sizes.  A token's output must be the same bits in every batch it
runs in, and within tolerance of the oracle."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from tests import hk_testutil as U

pytestmark = pytest.mark.gpu
# hidden, inter, shared_inter, experts, top_k, tokens: the last batch of each
# row takes the wide shapes, its one-token batches the small ones
SHAPES = [(256, 128, 384, 16, 4, 64),     # shared wider than routed
          (1024, 768, 128, 32, 8, 40),    # routed wider, more than 256 gate/up items
          (4480, 256, 0, 64, 3, 24),      # the largest hidden with two workgroups a CU, no shared expert
          (4608, 256, 256, 64, 3, 24),    # one step past it
          (8192, 128, 256, 16, 2, 5)]     # the widest hidden: two images a group


@pytest.fixture(scope="module")
def ctx():
    from hawking_amd.runtime import Context
    return Context(0)


@pytest.mark.parametrize("H,I,SI,E,K,T", SHAPES)
def test_batch_shapes(ctx, oracle, H, I, SI, E, K, T):
    from hawking_amd.moe import MoeModel, MoeShape
    print("[gpu-case] batch shape", H, I, SI, E, K, T, flush=True)
    sys.stdout.flush()
    shape = MoeShape(n_layers=1, hidden=H, inter=I, shared_inter=SI, n_experts=E, top_k=K, expert_kind=U.HK_Q4,
                     expert_group=32, shared_gate=False, router=1, routed_scaling_factor=2.5)
    m = MoeModel(ctx, shape)
    m.fill_synthetic(U.SEED)
    xb = U.to_bf16_bits(np.random.default_rng(H + T).standard_normal((T, H)).astype(np.float32)).reshape(T, H)
    y, ids, w = m.routed_moe(0, xb)
    assert ctx.device_status() == 0
    for t in (0, T // 2, T - 1):
        y1, ids1, w1 = m.routed_moe(0, xb[t:t + 1])
        assert np.array_equal(ids1[0], ids[t]) and np.array_equal(w1[0], w[t])
        assert np.array_equal(y1[0], y[t]), f"token {t} depends on the batch"
    y2, _, _ = m.routed_moe(0, xb[:T // 2 + 1])
    assert np.array_equal(y2, y[:T // 2 + 1])
    x = U.bf16_to_f32(xb[0])
    M, *_ = U.oracle_noaux(oracle, U.SEED, shape, 0, x)
    out, rids, *_ = M.forward(x)
    _, router, _ = U.dense(oracle, U.SEED, shape, 0)
    if U.noaux_margin_ok(oracle.gemv_f32(router, x), U.router_bias(oracle, U.SEED, shape, 0), 1, 1, K):
        assert ids[0].tolist() == rids.tolist()
        assert oracle.relative_l2(y[0], out) < 2e-5


def _f64_token(oracle, shape, x, ids, w):
    """The block of one token in 64 bits over its routed ids and weights."""
    def dec(e, p):
        o = U.oracle_organ(oracle, U.SEED, shape, 0, e, p)
        return oracle.q4_decode(o.scales, o.codes, o.rows, o.cols, o.group).astype(np.float64).reshape(o.rows, o.cols)

    y = np.zeros(shape.hidden)
    for e, we in list(zip(ids.tolist(), w.astype(np.float64).tolist())) + [(shape.n_experts, 1.0)]:
        g, u = dec(e, 0) @ x, dec(e, 1) @ x
        y += we * (dec(e, 2) @ (g / (1.0 + np.exp(-g)) * u))
    return y


def test_batch_shapes_tiny_activations(ctx, oracle):
    """Activations near 2^-112 keep their precision in every batch: the images
    carry an exponent each, so a token's bits do not depend on the batch and
    its error against 64 bits is what ordinary activations show (four f32
    stages of 2-3e-7 each)."""
    from hawking_amd.moe import MoeModel, MoeShape
    print("[gpu-case] batch tiny activations", flush=True)
    H, T = 1024, 40
    shape = MoeShape(n_layers=1, hidden=H, inter=768, shared_inter=128, n_experts=32, top_k=8, expert_kind=U.HK_Q4,
                     expert_group=32, shared_gate=False, router=1, routed_scaling_factor=2.5)
    m = MoeModel(ctx, shape)
    m.fill_synthetic(U.SEED)
    x = np.random.default_rng(7).standard_normal((T, H)).astype(np.float32) * np.float32(2.0 ** -56)
    xb = U.to_bf16_bits(x).reshape(T, H)
    y, ids, w = m.routed_moe(0, xb)
    assert ctx.device_status() == 0
    for t in (0, T - 1):
        want = _f64_token(oracle, shape, U.bf16_to_f32(xb[t]).astype(np.float64), ids[t], w[t])
        assert np.linalg.norm(y[t] - want) <= 1.5e-6 * np.linalg.norm(want), t
        y1, ids1, _ = m.routed_moe(0, xb[t:t + 1])
        assert np.array_equal(ids1[0], ids[t]) and np.array_equal(y1[0], y[t]), f"token {t} depends on the batch"
