"""The shared expert's down rows inside the routed down kernel (moe_decode_down_gs, _xgs) at the edges of what
they take: the widest rows (1024 columns: every lane's load used), widths that end inside a lane's first and second
load, 1, 4, 10, 16 and 20 output rows a group and 22 and 24, the most that the builds with three shared rows a wave
are given; both row formats, TQ2_T and other types, alone and with a stack's residual; and one width past the range, which keeps the launch of its own.

Bar: fp32 throughout, so two summation orders of at most K = 4096 products: sqrt(K) 2^-24 = 4e-6, stated
as 5e-6 (a two-layer stack: 1e-5)."""
import pytest

from gyrodx import synth
from gyrodx.engine import PATH_DECODE, PATH_GENERIC, Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,F,U,type_id,SF,sh_type,n", [
    (2560, 640, 10, 144, 1024, 8, 2), (2560, 640, 10, 144, 1024, 30, 1), (2560, 640, 10, 148, 640, 8, 3),
    (2560, 640, 10, 151, 576, 30, 8), (256, 128, 1, 144, 64, 8, 1), (256, 256, 3, 147, 512, 30, 4),
    (4096, 256, 2, 144, 960, 30, 2), (4096, 256, 2, 149, 1024, 8, 5), (2560, 640, 10, 144, 1088, 8, 2),
    (2816, 384, 4, 144, 704, 8, 2), (2304, 384, 3, 144, 1024, 30, 5), (2304, 256, 6, 148, 576, 8, 5),
    (1536, 384, 6, 150, 1024, 30, 8),
])
def test_shared_folded(oracle_mod, E, F, U, type_id, SF, sh_type, n):
    layer = synth.make_layer(5200 + E + SF + sh_type, E=E, F=F, n_expert=16, n_used=U, type_id=type_id, SF=SF,
                             sh_type=sh_type)
    x = synth.make_tokens(5300 + n, n, E)
    print(f"shared folded E={E} F={F} type {type_id} SF={SF} format {sh_type} n={n}", flush=True)
    eng = Engine(max_tok=8)
    try:
        eng.add_layer(layer)
        r = oracle_mod.rel_rms(oracle_mod.OracleLayer(layer).forward(x), eng.forward(0, x, PATH_DECODE))
        s = oracle_mod.rel_rms(eng.forward_stack([0, 0], x, PATH_GENERIC), eng.forward_stack([0, 0], x, PATH_DECODE))
        print(f"rel_rms {r:.2e}, stack {s:.2e}", flush=True)
        assert r <= 5e-6 and s <= 1e-5
    finally:
        eng.close()
