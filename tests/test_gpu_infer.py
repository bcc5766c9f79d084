"""The one-launch inference kernel: the same bits whatever the rows per
workgroup, and the layer-by-layer arithmetic (bf16 operands and activations,
wider sums) of the network, over widths, depths, ragged row counts and outputs."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _net(ns, width, depth, nb, seed=1, max_batch=256):
    from abc_inference_transcription_amd.surrogate import Surrogate
    return Surrogate(ns, n_bins=nb, width=width, depth=depth, max_batch=max_batch, seed=seed)


def _reference(torch, s, x, width, depth, ns):
    """float64 sums of bf16 operands, activations rounded to bf16 per layer."""
    p = torch.tensor(s.get_params())
    r = lambda a: a.to(torch.bfloat16).double()
    in_pad, out_pad = -(-s.n_in // 64) * 64, -(-2 * ns // 128) * 128
    h, at = r(x.cpu()), 0
    h = torch.nn.functional.pad(h, (0, in_pad - s.n_in))
    for l in range(depth + 1):
        i, o = (in_pad if l == 0 else width), (out_pad if l == depth else width)
        W, b = r(p[at:at + i * o].view(o, i)), p[at + i * o:at + i * o + o].double()
        at += i * o + o
        z = h @ W.t() + b
        h = r((z * torch.sigmoid(z)).float()) if l < depth else z
    return h[:, :2 * ns]


# 16, 32 and 64 rows per workgroup with remainders; outputs that are and are
# not multiples of 4, of one and of several 32-feature steps per wave
@pytest.mark.parametrize("n,ns,width,depth,nb", [
    (1, 90, 512, 4, 5), (15, 3, 128, 1, 1), (17, 65, 256, 2, 8), (33, 300, 384, 3, 2),
    (4097, 90, 512, 4, 5), (8200, 7, 128, 2, 5), (16385, 45, 256, 1, 5), (16450, 90, 384, 2, 5)])
def test_inference_matches_layer_arithmetic(n, ns, width, depth, nb):
    import torch
    s = _net(ns, width, depth, nb)
    x = torch.randn(n, s.n_in, generator=torch.Generator().manual_seed(n)).to(s.dev)
    print(f"\n[infer] n={n} ns={ns} width={width} depth={depth}", flush=True)
    y = s.predict(x).cpu()
    rows = torch.arange(0, n, max(1, n // 300))
    want = _reference(torch, s, x[rows.to(s.dev)], width, depth, ns)
    # FP32 sums of 512 terms are off by about 1e-6 of them; an activation near a
    # bf16 rounding boundary may round the other way (2^-8 of it, among hundreds)
    err = (y[rows].double() - want).norm(dim=1) / want.norm(dim=1)
    assert float(err.max()) < 4e-3
    small = s.predict(x[:min(n, 40)].contiguous()).cpu()       # 16 rows per workgroup
    assert torch.equal(small, y[:small.shape[0]])
    tail = s.predict(x[n - min(n, 9):].contiguous()).cpu()
    assert torch.equal(tail, y[n - tail.shape[0]:])
    s.close()


def test_large_activations_and_unaligned_outputs():
    """Pre-activations far below zero (subnormal and zero sigmoids) and an output
    buffer aligned to four bytes only."""
    import torch
    s = _net(90, 256, 2, 5)
    p = s.get_params()
    s.set_params(p * 40.0)
    x = 20.0 * torch.randn(513, s.n_in, generator=torch.Generator().manual_seed(2)).to(s.dev)
    y = s.predict(x)
    want = _reference(torch, s, x, 256, 2, 90)
    err = (y.cpu().double() - want).norm(dim=1) / want.norm(dim=1)
    assert torch.isfinite(y).all() and float(err.max()) < 4e-3
    buf = torch.zeros(513 * 180 + 1, device=s.dev)
    torch.cuda.synchronize()
    assert s.L.abc_mlp_forward_dev(s.h, 513, C.c_void_p(x.data_ptr()),
                                   C.c_void_p(buf.data_ptr() + 4)) == 0
    assert s.L.abc_mlp_synchronize(s.h) == 0
    assert torch.equal(buf[1:].view(513, 180), y)
    s.close()


def test_training_refreshes_the_inference_weights():
    import torch
    s = _net(12, 256, 2, 5)
    g = torch.Generator().manual_seed(3)
    x = torch.randn(256, s.n_in, generator=g).to(s.dev)
    t = torch.randn(256, 12, generator=g).to(s.dev)
    a = s.predict(x)
    s.train(x, t, 3, batch=256)
    b = s.predict(x)
    want = _reference(torch, s, x, 256, 2, 12)
    assert not torch.equal(a, b)
    assert float(((b.cpu().double() - want).norm(dim=1) / want.norm(dim=1)).max()) < 4e-3
    s.close()
