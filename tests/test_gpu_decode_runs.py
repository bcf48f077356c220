"""The batch builds of the run-wise gate/up kernels (moe_decode_gu_gb, moe_decode_gu_xgb: two groups per CU) at the
edges of their range: calls of 896 items per CU, the fewest that take them (on 256 CUs), and of 882, which keep
the one-group builds; runs that end inside a slot and span two tokens, the widest hidden size and top-16, TQ2_T
and other types. The products and sums are those of
the one-token builds, so a batch equals its tokens run one at a time up to the rounding of a fused
multiply-add: fp32 throughout, two orders of at most K = 4096 products, sqrt(K) 2^-24 = 4e-6."""
import numpy as np
import pytest

from gyrodx import synth
from gyrodx.engine import PATH_DECODE, Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,F,U,type_id,n", [
    (2560, 640, 10, 144, 2), (2560, 640, 10, 144, 7), (2560, 640, 10, 148, 3), (2560, 640, 10, 149, 8),
    (4096, 1024, 16, 144, 3), (4096, 384, 7, 151, 5), (256, 1024, 16, 144, 8), (1536, 768, 11, 145, 4),
    (256, 1024, 16, 144, 7), (256, 896, 16, 148, 8), (2304, 128, 14, 144, 7), (2304, 128, 14, 148, 7),
])
def test_batch_runs(oracle_mod, E, F, U, type_id, n):
    layer = synth.make_layer(5400 + E + F + n, E=E, F=F, n_expert=24, n_used=U, type_id=type_id)
    x = synth.make_tokens(5500 + n, n, E)
    print(f"batch runs E={E} F={F} top-{U} type {type_id} n={n}", flush=True)
    eng = Engine(max_tok=8)
    try:
        eng.add_layer(layer)
        out = eng.forward(0, x, PATH_DECODE)
        ids, _ = eng.last_routes(n)
        one = np.concatenate([eng.forward(0, x[t:t + 1], PATH_DECODE) for t in range(n)])
    finally:
        eng.close()
    ref, trace = oracle_mod.OracleLayer(layer).forward(x, trace=True)
    np.testing.assert_array_equal(ids, trace["route_ids"][:n])
    assert oracle_mod.rel_rms(ref, out) <= 4e-6 and oracle_mod.rel_rms(one, out) <= 4e-6
