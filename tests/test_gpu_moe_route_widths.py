"""The decode route kernels over hidden sizes on both sides of each of their
instantiations (registers for 1,024, 2,048, 4,096 and 8,192 columns, and for
2,048, 4,096 and 8,192 in the mixed-1p5 layer): route ids exact under the
router margin rule, weights within 1e-6 of FP64, outputs within 2e-5 rel-L2
of the oracle (the tolerances of the layer tests these follow)."""
import numpy as np
import pytest

from tests import hk_testutil as U
from tests.test_gpu_moe15 import build_layer, router_weights_f64

pytestmark = pytest.mark.gpu
TOL = 2e-5


@pytest.fixture(scope="module")
def ctx():
    from hawking_amd.runtime import Context
    return Context(0)


def _inputs(oracle, H, tag):
    return [oracle.normal(oracle.stream_key(U.SEED, tag + t), H, 1.0) for t in range(3)]


@pytest.mark.parametrize("H", [128, 1024, 1152, 2176, 4096, 4224, 8192])
def test_route_widths(ctx, oracle, H):
    from hawking_amd.moe import MoeModel, MoeShape
    print("[gpu-case] route width", H, flush=True)
    shape = MoeShape(n_layers=1, hidden=H, inter=128, shared_inter=128, n_experts=18, top_k=4,
                     expert_kind=U.HK_Q4, expert_group=32, shared_gate=True)
    m = MoeModel(ctx, shape)
    m.fill_synthetic(U.SEED + H)
    ctx.device_status()
    checked = 0
    for h in _inputs(oracle, H, 0x3170):
        out, ids, w = m.moe_suffix(0, h)
        L, rout, rids, rw, logits = U.oracle_layer(oracle, U.SEED + H, shape, 0, h)
        assert oracle.relative_l2(out, L.forward_f64(h, ids)) < TOL
        if not U.router_margin_ok(logits, shape.top_k):
            continue
        checked += 1
        assert ids.tolist() == rids.tolist()
        assert np.max(np.abs(w - router_weights_f64(L, h, ids))) <= 1e-6
        assert oracle.relative_l2(out, rout) < TOL
    assert checked >= 1
    assert ctx.device_status() == 0


@pytest.mark.parametrize("H", [2176, 4096, 4224])
def test_mixed15_route_widths(ctx, oracle, H):
    print("[gpu-case] mixed15 route width", H, flush=True)
    layer, ref = build_layer(ctx, oracle, H, 128, 128, 6, 3, 32, tag=0x17)
    ctx.device_status()
    checked = 0
    for h in _inputs(oracle, H, 0x3171):
        out, ids, w = layer.moe_suffix(h)
        rout, rids, rw, _, logits = ref.forward(h)
        assert oracle.relative_l2(out, ref.forward_f64(h, ids)) < TOL
        if not U.router_margin_ok(logits, 3):
            continue
        checked += 1
        assert ids.tolist() == rids.tolist()
        assert np.all(np.abs(w - router_weights_f64(ref, h, ids)) <= 1e-6)
    assert checked >= 1
    assert ctx.device_status() == 0
    layer.free()
