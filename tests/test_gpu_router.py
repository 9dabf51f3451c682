"""Router logits above 32 tokens (f32 MFMA chains): partial sums and the A8 of x at the edges of both tile sizes."""
import numpy as np
import pytest

import oracle
from llmoe import Layer, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E", [(33, 256), (64, 64), (65, 192), (256, 128), (257, 64), (319, 256), (321, 192)])
def test_router_tiles_bit_exact(gpu, T, E):
    import torch
    print(f"[router tiles] T={T} E={E}", flush=True)
    L = synth.make_layer(40 + E, E=E, mix=2, experts=[0])
    x = synth.make_x(T, T, outlier_frac=0.01)
    x[T - 1] *= np.float32(1e-38)      # products below the normal range: the chains keep subnormals
    G = Layer(L["blob"], L["gu_off"], L["d_off"], L["bits"], L["bias"], L["Wr"], n_experts=E, pool=E, max_tokens=T)
    G.forward(torch.from_numpy(x).to(gpu))
    part = G.read("logits_part", (8, T, E), np.float32)
    lg = part[0].copy()
    for c in range(1, 8):
        lg = (lg + part[c]).astype(np.float32)
    assert np.array_equal(lg.view(np.uint32), oracle.router_logits(x, L["Wr"]).view(np.uint32))
    q, s, sm = oracle.quant_a8(x)
    assert np.array_equal(G.read("xq", (T, 2048), np.int8), q)
    assert np.array_equal(G.read("xs", (T, 16), np.float32).view(np.uint32), s.view(np.uint32))
    assert np.array_equal(G.read("xsum", (T, 16), np.int32), sm)
    G.close()
