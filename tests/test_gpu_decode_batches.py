"""The batch decode kernels over their whole range: every batch size (on 256 CUs 2, 0, 4, 0, 2, 4, 4 blocks per lane
for 2 to 8 tokens at hidden 2048; 0, 0, 2, 0, 0, 4, 4 at 1024), with and without sign vectors and in a residual
stack. The kernels form the same products and sums in the same order as the one-token kernels,
so a batch equals its tokens run one at a time bit for bit."""
import numpy as np
import pytest

from gyrodx import synth
from gyrodx.engine import PATH_DECODE, Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,n", [(E, n) for E in (1024, 2048) for n in range(2, 9)])
@pytest.mark.parametrize("signs", [True, False])
def test_batch_equals_single_tokens(oracle_mod, E, n, signs):
    L = synth.make_layer(400 + n, E=E, F=512, n_expert=40)
    if not signs:
        L.gate_signs = L.down_signs = None
    x = synth.make_tokens(401, n, E)
    eng = Engine(max_tok=8)
    try:
        eng.add_layer(L)
        print(f"decode batch: E {E} n {n} signs {signs}", flush=True)
        out = eng.forward(0, x, PATH_DECODE)
        ids, w = eng.last_routes(n)
        one = np.concatenate([eng.forward(0, x[t:t + 1], PATH_DECODE) for t in range(n)])
        stack = eng.forward_stack([0, 0], x, PATH_DECODE)
        stack1 = np.concatenate([eng.forward_stack([0, 0], x[t:t + 1], PATH_DECODE) for t in range(n)])
    finally:
        eng.close()
    ref, trace = oracle_mod.OracleLayer(L).forward(x, trace=True)
    np.testing.assert_array_equal(ids, trace["route_ids"][:n])
    np.testing.assert_allclose(w, trace["route_w"][:n], rtol=1e-5)
    assert oracle_mod.rel_rms(ref, out) < 2e-6
    np.testing.assert_array_equal(out.view(np.uint32), one.view(np.uint32))
    np.testing.assert_array_equal(stack.view(np.uint32), stack1.view(np.uint32))
