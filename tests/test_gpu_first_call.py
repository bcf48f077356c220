"""The first call of an engine under HIP graph capture, for every batch size: the kernels of the decode path are
loaded with the layer, so gm_forward_decode_noalloc loads nothing itself (a load is not allowed while a stream is
captured). The replayed graph equals gm_forward bit for bit."""
import numpy as np
import pytest
import torch

from gyrodx import synth
from gyrodx.engine import PATH_DECODE, Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [
    dict(E=2048, F=512, n_used=8), dict(E=2048, F=512, n_used=8, mixed_types=True, SF=512), dict(E=2560, F=640, n_used=10, SF=640, sh_type=8),
    dict(E=2560, F=640, n_used=10, type_id=148), dict(E=1024, F=1024, n_used=16, SF=1088, sh_type=0),
], ids=["tq2", "mixed_shared", "coder_q8_shared", "coder_148", "wide_shared"])
def test_capture_before_any_call(kw):
    layer = synth.make_layer(61, n_expert=32, **kw)
    x = synth.make_tokens(62, 8, layer.E)
    xd, od = torch.from_numpy(x).cuda(), torch.zeros((9, 8, layer.E), device="cuda")
    eng = Engine(max_tok=8)
    try:
        li = eng.add_layer(layer)
        print(f"capture of the first call: {kw}", flush=True)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for n in range(1, 9):
                eng.forward_decode_noalloc(li, xd.data_ptr(), n, od[n].data_ptr(), torch.cuda.current_stream().cuda_stream)
        for _ in range(3):
            od.zero_()
            graph.replay()
            torch.cuda.synchronize()
            out = od.cpu().numpy()
            for n in range(1, 9):
                ref = eng.forward(li, x[:n], PATH_DECODE)
                np.testing.assert_array_equal(out[n, :n].view(np.uint32), ref.view(np.uint32))
        del graph
    finally:
        eng.close()
