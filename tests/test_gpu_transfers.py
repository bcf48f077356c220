"""Host transfers in parts (set_tokens, read_outputs, gm_forward) at the sizes where their plan changes:
one part below the threaded copy's threshold and the parts at it, a part of one slot, several slots, one thread's
and the helpers' uploads, and a dozen parts and more, whose staging slots come round while copies are still queued. Rows that
went through the engine in one transfer each way must equal, bit for bit, the same rows sent eight at a
time (32 KB, a single part)."""
import numpy as np
import pytest

from gyrodx import synth
from gyrodx.engine import PATH_DECODE, PATH_PREFILL, Engine

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    eng = Engine(max_tok=640)
    eng.add_layer(synth.make_layer(5300, E=1024, F=256, n_expert=16, n_used=2))
    yield eng
    eng.close()


# 4 KB a token. Downloads: one part copied by the caller up to 992 KB, two parts of 512 KB with the helpers at 1 MB, three,
# 4 MB, 12 MB in 2 MB slots, 24 MB in 13 parts. Uploads: one part up to 1 MB, two up to 2 MB, three up to 6 MB (the last
# that the caller copies), whole slots with the helpers from there on.
@pytest.mark.parametrize("n", [88, 96, 128, 136, 248, 256, 264, 512, 520, 1032, 1536, 1544, 3080, 6200])
def test_tokens_and_outputs_in_parts(engine, n):
    print(f"transfers: {n} tokens", flush=True)
    x = synth.make_tokens(5301 + n, n, 1024)
    engine.set_tokens(x)
    engine.run(PATH_DECODE, 8, n // 8, [0])
    got = engine.read_outputs(n)
    ref = np.concatenate([engine.forward(0, x[i:i + 8], PATH_DECODE) for i in range(0, n, 8)])
    np.testing.assert_array_equal(got.view(np.uint32), ref.view(np.uint32))


def test_forward_in_parts_is_repeatable(engine):
    """gm_forward with a multi-part input and output and the flag words in the first part."""
    x = synth.make_tokens(5400, 640, 1024)
    engine.set_tokens(x)
    engine.run(PATH_PREFILL, 640, 1, [0])
    ref = engine.read_outputs(640)
    for _ in range(3):
        np.testing.assert_array_equal(engine.forward(0, x, PATH_PREFILL).view(np.uint32), ref.view(np.uint32))


def test_empty_read_is_refused(engine):
    engine.set_tokens(synth.make_tokens(5500, 8, 1024))
    with pytest.raises(RuntimeError):
        engine.read_outputs(0)
