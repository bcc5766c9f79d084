"""Networks of many outputs: their output layer is shared by workgroups where the
rows alone would leave CUs idle; the same bits as the layer-by-layer path."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _net(ns, width, depth):
    from abc_inference_transcription_amd.surrogate import Surrogate
    return Surrogate(ns, width=width, depth=depth, max_batch=512, seed=1)


def test_many_outputs_of_few_rows():
    """100 rows, one layer of 512: 256 outputs 24 us, 2,048 outputs 44 us by one
    workgroup per row tile and 23 shared."""
    import torch
    best = {}
    for ns in (128, 1024):
        s = _net(ns, 512, 1)
        x = torch.randn(100, s.n_in, device=s.dev)
        s.predict(x)
        best[ns] = np.inf
        for _ in range(60):
            torch.cuda.synchronize()
            t = time.perf_counter()
            s.predict(x)
            best[ns] = min(best[ns], 1e6 * (time.perf_counter() - t))
        s.close()
    print(f"\n[wide outputs] us: {best}", flush=True)
    assert best[1024] < 1.4 * best[128]


# one to eight shares of the outputs, the last one short, and rows from one to
# several tiles per CU; the wider network of zeros goes layer by layer
@pytest.mark.parametrize("ns,width,depth", [(129, 128, 1), (300, 256, 2), (1024, 512, 1)])
@pytest.mark.parametrize("n", [1, 33, 700, 2100, 4097, 17000])
def test_shared_outputs_equal_layer_by_layer(ns, width, depth, n):
    import torch
    a, b = _net(ns, width, depth), _net(ns, 640, depth)
    g = torch.Generator().manual_seed(n)
    ip, op = -(-a.n_in // 64) * 64, -(-2 * ns // 128) * 128
    flat, out, at = torch.tensor(a.get_params()), [], 0
    for l in range(depth + 1):
        i, o = (ip if l == 0 else width), (op if l == depth else width)
        ib, ob = (ip if l == 0 else 640), (op if l == depth else 640)
        W, c = flat[at:at + i * o].view(o, i), 0.3 * torch.randn(o, generator=g)
        flat[at + i * o:at + i * o + o] = c
        at += i * o + o
        Wb, cb = torch.zeros(ob, ib), torch.zeros(ob)
        Wb[:o, :i], cb[:o] = W, c
        out += [Wb.reshape(-1), cb]
    a.set_params(flat.numpy())
    b.set_params(torch.cat(out).numpy())
    x = torch.randn(n, a.n_in, generator=g).to(a.dev)
    print(f"\n[wide outputs] n={n} width={width} ns={ns}", flush=True)
    ya = a.predict(x)
    assert torch.isfinite(ya).all() and torch.equal(ya, b.predict(x))
    a.close()
    b.close()
