"""The routing selection (bit descents over ballots) against the CPU oracle: ties everywhere, pools from K to E - 1,
every top-K, infinities, and expert counts that do not fill the four keys per lane."""
import numpy as np
import pytest

import oracle
from llmoe import Layer, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,K,C,T,levels", [
    (256, 8, 256, 32, 3),      # three distinct scores: nearly all comparisons tie
    (256, 8, 48, 32, 3),
    (256, 8, 8, 32, 0),        # the pool is exactly the top-K
    (256, 1, 255, 7, 0),
    (192, 6, 191, 33, 2),      # several blocks, the last one of one token
    (64, 8, 9, 70, 4),
    (128, 3, 64, 1, 1),        # every score equal; one token (its pool is not computed)
    (256, 8, 100, 64, -1),     # infinite and huge logits
])
def test_selection_matches_oracle(gpu, E, K, C, T, levels):
    import torch
    print(f"[select] E={E} K={K} C={C} T={T} levels={levels}", flush=True)
    rng = np.random.default_rng(E + 10 * K + C + T)
    L = synth.make_layer(9, E=E, mix=2, experts=[0], zero_bias=levels > 0)
    lg = rng.standard_normal((T, E)).astype(np.float32)
    if levels > 0:
        lg = rng.integers(0, levels, (T, E)).astype(np.float32)
    if levels < 0:
        pick = rng.random((T, E))
        lg[pick < 0.1] = np.inf
        lg[pick > 0.9] = -np.inf
        lg[(pick > 0.45) & (pick < 0.55)] = -1e30
    G = Layer(L["blob"], L["gu_off"], L["d_off"], L["bits"], L["bias"], L["Wr"], n_experts=E, top_k=K, pool=C,
              max_tokens=T)
    ref_k, ref_w = oracle.route(lg, L["bias"], K=K, C=C)
    for _ in range(2):   # (the routing state is left clear for the next call)
        G.route(T, logits=torch.from_numpy(lg).to(gpu))
        torch.cuda.synchronize()
        assert np.array_equal(G.read("topk", (T, K), np.int32), ref_k)
        assert np.array_equal(G.read("topw", (T, K), np.float32).view(np.uint32), ref_w.view(np.uint32))
    G.close()
