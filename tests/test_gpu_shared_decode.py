"""The decode path's own shared-expert kernels (moe_router_s, moe_decode_shared_down) at the edges of
their range, against the CPU oracle through the C ABI: the narrowest shared expert (one 64-column run,
most lanes past the last column), widths that end inside a load and inside a run of four loads, the
largest hidden width, each row format, 1 to 8 tokens.

Bar: decode keeps everything in fp32, so against the oracle's fp32 the difference is that of two
summation orders, at most about sqrt(K) 2^-24 relative for K = 4096 products: 4e-6, stated as 5e-6."""
import pytest

from gyrodx import synth
from gyrodx.engine import PATH_DECODE, Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,F,U,SF,sh_type,n", [
    (1280, 256, 4, 64, 8, 1), (1280, 256, 4, 64, 30, 8), (1280, 256, 4, 64, 0, 5),
    (2560, 640, 10, 1088, 0, 2), (2560, 640, 10, 2112, 30, 3), (1024, 512, 8, 4160, 8, 2),
    (4096, 256, 2, 320, 8, 8), (4096, 256, 2, 320, 0, 7), (4096, 256, 2, 192, 30, 1),
])
def test_shared_decode_edges(oracle_mod, E, F, U, SF, sh_type, n):
    layer = synth.make_layer(5000 + E + SF + sh_type, E=E, F=F, n_expert=16, n_used=U, SF=SF, sh_type=sh_type)
    x = synth.make_tokens(5100 + n, n, E)
    ref = oracle_mod.OracleLayer(layer).forward(x)
    print(f"shared decode E={E} F={F} SF={SF} format {sh_type} n={n}", flush=True)
    eng = Engine(max_tok=8)
    try:
        eng.add_layer(layer)
        r = oracle_mod.rel_rms(ref, eng.forward(0, x, PATH_DECODE))
        print(f"rel_rms {r:.2e}", flush=True)
        assert r <= 5e-6
    finally:
        eng.close()
