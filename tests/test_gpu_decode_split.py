"""Decode units split finer (fewer strips per wave) when a step has few units: every width, both sides of each bound,
one and two items per expert, against the CPU oracle bit for bit."""
import numpy as np
import pytest

import oracle
from llmoe import Layer, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,mix,shared,pool,split", [
    (1, 2, False, 256, (2, 2)),          # the smallest lists
    (1, 3, True, 256, (2, 2)),
    (1, 8, True, 256, (2, 2)),           # 8-bit gate_up has one strip per wave at every split; down one at the finest
    (2, 4, False, 256, (2, 2)),
    (5, "mixed", True, 256, (2, 1)),     # down between the bounds
    (20, 2, True, 16, (2, 2)),           # a pool of 16: items of 16 slots, two per busy expert
    (17, 3, True, 40, (2, 0)),           # two shared items; 3-bit gate_up units halved (their most), down unsplit
    (32, "mixed", True, 256, (0, 0)),    # about 160 experts: no split
    (8, 2, False, 256, (1, 1)),          # gate_up between the bounds: halved, not quartered
    (32, "mixed", True, 48, (1, 1)),
    (4, 3, False, 256, (2, 1)),
    (2, 8, False, 256, (2, 1)),
    (4, 8, True, 256, (2, 0)),           # the finest gate_up beside unsplit down units
])
def test_split_units_match_oracle(gpu, T, mix, shared, pool, split):
    import torch
    print(f"[decode split] T={T} mix={mix} shared={shared} pool={pool}", flush=True)
    L = synth.make_layer(300 + T, mix=mix, shared=shared, experts=None if mix == "mixed" else [0, 1, 2])
    G = Layer(L["blob"], L["gu_off"], L["d_off"], L["bits"], L["bias"], L["Wr"], pool=pool, has_shared=shared,
              max_tokens=32)
    x = synth.make_x(400 + T, T)
    out = G.forward(torch.from_numpy(x).to(gpu))
    torch.cuda.synchronize()
    r = oracle.Layer(L).forward(x, C=pool)
    assert np.array_equal(G.read("topk", (T, 8), np.int32), r["topk"])
    S = T * 8 + (T if shared else 0)
    assert np.array_equal(G.read("Z", (S, 512), np.uint16), r["Z"]), "gate_up"
    assert np.array_equal(G.read("Y", (S, 2048), np.float32).view(np.uint32), r["Y"].view(np.uint32)), "down"
    assert np.array_equal(out.cpu().numpy().view(np.uint32), r["out"].view(np.uint32))
    n = G.read("n_items", (6,), np.int32)
    assert tuple(n[4:] >> 24) == split, f"units {n[0]} / {n[1]} split {n[4:] >> 24}"
    G.close()
