"""Tiled dense projections whose workgroups hold several (chunk, row block) tasks: more tasks than workgroups, an even and
an uneven share, runs that start inside a chunk and cross into the next, a last chunk of one token. Every workgroup's share
is a closed form evaluated in the kernel, so a wrong term would skip rows or (accumulating) add them twice: outputs against
the CPU oracle bit for bit, store and accumulate."""
import sys
from pathlib import Path

import numpy as np
import pytest

import oracle
from llmoe import Dense, synth

sys.path.insert(0, str(Path(__file__).resolve().parent / "golden"))
import gen  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,bits,R,tasks", [
    (1025, 8, 3072, 17 * 24),    # the last of 17 chunks is one token
    (2049, 3, 2048, 33 * 8),
    (1024, 4, 4096, 16 * 16),    # as many tasks as CUs
    (2048, 2, 4096, 32 * 16),    # twice as many
    (700, 8, 3584, 11 * 28),     # 28 row blocks: a chunk's end falls inside the shares
])
def test_dense_shares_bit_exact(gpu, T, bits, R, tasks):
    import torch
    print(f"[dense shares] T={T} bits={bits} R={R}", flush=True)
    waves, strips = 8, 1 if bits == 8 else 2
    assert -(-T // 64) * (R // (16 * waves * strips)) == tasks
    assert tasks >= torch.cuda.get_device_properties(gpu).multi_processor_count
    blob = oracle.pack_i8(*gen.matrix(5000 + bits, R, 2048, bits), bits)
    xq, xs, xsum = oracle.quant_a8(synth.make_x(5100 + T, T))
    D = Dense(blob, R, bits, max_tokens=T)
    dx = [torch.from_numpy(a).to(gpu) for a in (xq, xs, xsum)]
    y0 = np.random.default_rng(T).standard_normal((T, R)).astype(np.float32)
    y = D.forward(*dx)
    acc = torch.from_numpy(y0).to(gpu)
    D.forward(*dx, out=acc, accumulate=True)
    torch.cuda.synchronize()
    ref = oracle.dense(blob, R, 2048, bits, xq, xs, xsum)
    assert np.array_equal(y.cpu().numpy().view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(acc.cpu().numpy().view(np.uint32), (y0 + ref).view(np.uint32))
    D.close()
