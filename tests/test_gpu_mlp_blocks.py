"""The warm-start network's kernels at the edges of their row blocks, against the numpy restatement
with the same bfloat16 rounding points (oracle/learned_oracle.py): one row, ragged rows of a 16-row
block, the first batch in 32-row blocks, one, two and three hidden layers of widths that give the
waves one, two and four column tiles, an output wider than a tile, one wide layer among narrow ones up
to the widest that the row blocks take (4864 between 128 inputs and 64 outputs), where two buffers of the
widest layer would exceed a workgroup's LDS from 2560 on, and networks too wide for the row blocks (one
GEMM per layer)."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import learned_oracle as lo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,features,outputs,hidden", [
    (1, 50, 14, (64,)),
    (17, 64, 70, (256, 128)),
    (100, 311, 35, (512, 512, 512)),
    (4097, 200, 20, (192, 128)),
    (33, 70, 9, (2496,)),
    (4097, 70, 9, (2560,)),
    (33, 311, 35, (2560, 512)),
    (65, 311, 35, (512, 3072)),
    (20, 311, 35, (4096,)),
    (33, 70, 9, (4864,)),
    (33, 70, 9, (4928,)),
    (33, 70, 9, (5120,)),
])
def test_mlp_row_blocks_match_oracle(gpu_device, rows, features, outputs, hidden):
    import torch

    from sap_warp_amd import _native as nat
    from sap_warp_amd.learned import Mlp

    rng = np.random.default_rng(rows)
    m = Mlp(features, outputs, hidden=hidden, seed=3, out_scale=1.0)
    o = lo.Mlp(list(m.dims), features, outputs)
    Ws, bs = lo.unflat(o, m.read().astype(np.float64))
    for l, b in enumerate(bs):
        b[:] = rng.standard_normal(b.shape) * 0.1
        if l == len(bs) - 1:
            b[outputs:] = 0.0
    flat = np.concatenate([np.concatenate([w.ravel(), b]) for w, b in zip(Ws, bs)]).astype(np.float32)
    m.write_params(flat)
    o.W, o.b = lo.unflat(o, flat.astype(np.float64))
    norm = (rng.standard_normal(features), 0.5 + rng.random(features), rng.standard_normal(outputs),
            0.5 + rng.random(outputs))
    m.set_normalization(*norm)
    o.x_mean, o.x_std, o.y_mean, o.y_std = [a.astype(np.float32).astype(np.float64) for a in norm]
    x = rng.standard_normal((rows, features)).astype(np.float32)
    t = rng.standard_normal((rows, outputs)).astype(np.float32)
    xd, td = torch.as_tensor(x, device="cuda:0"), torch.as_tensor(t, device="cuda:0")
    y = torch.full((rows + 1, outputs), 7.0, dtype=torch.float32, device="cuda:0")
    m.forward(xd, y, batch=rows)
    ref = o.predict(x.astype(np.float64))
    # a bfloat16 rounding of an activation that falls the other way moves the output by 2^-9 of one term
    assert np.max(np.abs(y[:rows].cpu().numpy() - ref)) / max(1.0, np.max(np.abs(ref))) < 2e-3
    assert bool((y[rows] == 7.0).all())
    loss = torch.zeros(1, dtype=torch.float32, device="cuda:0")
    m.gradients(xd, td, loss)
    l_ref, gW, gb = o.loss_and_grads(x.astype(np.float64), t.astype(np.float64))
    assert abs(float(loss.item()) - l_ref) <= 1e-3 * l_ref
    g = m.read(nat.MLP_GRADS)
    for got, want in zip(lo.unflat(o, g.astype(np.float64)), (gW, gb)):
        for a, b in zip(got, want):
            assert np.linalg.norm(a - b) <= 1e-2 * max(np.linalg.norm(b), 1e-12)
    m.adam(1e-3)
    opt, p = lo.Adam(lr=1e-3), [flat.astype(np.float64).copy()]
    opt.step(p, [g.astype(np.float64)])
    np.testing.assert_allclose(m.read(), p[0], rtol=1e-5, atol=1e-7)
    # the updated bfloat16 weights are the ones the next forward pass reads
    m.forward(xd, y, batch=rows)
    o.W, o.b = lo.unflat(o, m.read().astype(np.float64))
    ref = o.predict(x.astype(np.float64))
    assert np.max(np.abs(y[:rows].cpu().numpy() - ref)) / max(1.0, np.max(np.abs(ref))) < 2e-3
    # an output that overlaps its input: every row is still computed from the input as it was
    want = y[:rows].clone()
    over = torch.zeros(rows * max(features, outputs), dtype=torch.float32, device="cuda:0")
    over[:rows * features].copy_(xd.reshape(-1))
    m.forward(over[:rows * features].view(rows, features), over[:rows * outputs].view(rows, outputs))
    assert bool((over[:rows * outputs].view(rows, outputs) == want).all())


def test_captured_overlapping_forward(gpu_device):
    """A forward pass onto its own input, captured on a reserved workspace (nothing is allocated then):
    every replay gives what the pass gives eagerly, also with eager passes between them."""
    import torch

    from sap_warp_amd.learned import Mlp

    rows, features, outputs = 70, 64, 20
    m = Mlp(features, outputs, hidden=(128, 192), seed=5, out_scale=1.0)
    m.reserve(rows)
    buf = torch.zeros(rows * features, dtype=torch.float32, device="cuda:0")
    x, y = buf.view(rows, features), buf[:rows * outputs].view(rows, outputs)
    want = torch.empty((rows, outputs), dtype=torch.float32, device="cuda:0")
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            m.forward(x, y)
        gen = torch.Generator(device="cuda:0").manual_seed(2)
        for _ in range(4):
            rand = torch.randn((rows, features), generator=gen, device="cuda:0")
            m.forward(rand, want)
            buf.copy_(rand.reshape(-1))
            g.replay()
            stream.synchronize()
            assert torch.equal(y, want)
