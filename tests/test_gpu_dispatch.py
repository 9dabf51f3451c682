"""Externally routed steps (llmoe_dispatch + llmoe_experts): from one token to several blocks with a ragged last one, K = 8
and 6. The work lists and their split are the step's own, also right after a forward that left split lists in the same
words; the routing is copied when the call's work runs, so the caller's arrays are free to be overwritten behind it on the
same stream. Everything against the CPU oracle bit for bit."""
import numpy as np
import pytest

import oracle
from llmoe import Layer, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [8, 6])
@pytest.mark.parametrize("T,block", [(1, 32), (17, 32), (32, 32), (33, 32), (77, 32), (13, 8)])
def test_dispatch_after_split_forward(gpu, T, block, K):
    import torch
    print(f"[dispatch] T={T} block={block} K={K}", flush=True)
    L = synth.make_layer(70, mix="mixed", shared=True)
    G = Layer(L["blob"], L["gu_off"], L["d_off"], L["bits"], L["bias"], L["Wr"], top_k=K, block=block, has_shared=True,
              max_tokens=80)
    G.forward(torch.from_numpy(synth.make_x(71, 1)).to(gpu))
    assert tuple(G.read("n_items", (6,), np.int32)[4:] >> 24) == (2, 2)   # (the stale state that must not survive)

    rng = np.random.default_rng(T + K)
    topk = np.stack([rng.choice(256, K, replace=False) for _ in range(T)]).astype(np.int32)
    topw = rng.uniform(0.05, 0.6, (T, K)).astype(np.float32)
    xq, xs, xsum = oracle.quant_a8(synth.make_x(72 + T, T))
    dk, dw = torch.from_numpy(topk).to(gpu), torch.from_numpy(topw).to(gpu)
    G.dispatch(dk, dw)
    dk.zero_()
    dw.fill_(9.0)
    out = G.experts(*(torch.from_numpy(a).to(gpu) for a in (xq, xs, xsum)))
    torch.cuda.synchronize()
    assert np.array_equal(G.read("topk", (T, K), np.int32), topk)
    assert np.array_equal(G.read("topw", (T, K), np.float32).view(np.uint32), topw.view(np.uint32))
    n = G.read("n_items", (6,), np.int32)
    assert np.array_equal(n[4:] & 0xFFFFFF, n[:2]), "unit counts"
    r = oracle.Layer(L, K=K).experts(xq, xs, xsum, topk, topw)
    S = T * (K + 1)
    assert np.array_equal(G.read("slot_token", (S,), np.int32), r["slot_token"])
    assert np.array_equal(G.read("tok_slots", (T, K + 1), np.int32), r["tok_slots"])
    assert np.array_equal(G.read("Z", (S, 512), np.uint16), r["Z"]), "gate_up"
    assert np.array_equal(G.read("Y", (S, 2048), np.float32).view(np.uint32), r["Y"].view(np.uint32)), "down"
    assert np.array_equal(out.cpu().numpy().view(np.uint32), r["out"].view(np.uint32))
    G.close()
