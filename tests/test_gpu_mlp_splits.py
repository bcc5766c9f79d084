"""The weight and bias gradients' split sums: batches whose last chunk is short
or empty, layers that are not split at all, and Adam's step from the same sums."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.mark.parametrize("n,width,depth,ns", [
    (1, 128, 1, 3),        # one chunk of 128
    (129, 128, 2, 7),      # K = 256: not split
    (700, 256, 1, 65),     # K = 768
    (1100, 512, 2, 90),    # K = 1,152
    (4100, 128, 2, 5),     # 16 chunks of 384: five of them empty
    (64, 2048, 2, 4)])     # a layer of 512 tiles: its gradient is one sum
def test_split_sums(n, width, depth, ns):
    import torch

    import mlp_ref as M
    from abc_inference_transcription_amd.surrogate import Surrogate
    s = Surrogate(ns, width=width, depth=depth, max_batch=n, seed=n)
    rng = np.random.default_rng(n)
    x = rng.normal(0, 0.7, (n, s.n_in)).astype(f32)
    t = rng.normal(0, 1, (n, ns)).astype(f32)
    xd, td = torch.tensor(x, device="cuda"), torch.tensor(t, device="cuda")
    loss, g = s.grad(xd, td)
    w0 = s.get_params()
    loss_ref, g_ref = M.loss_and_grad(w0.astype(np.float64), x.astype(np.float64),
                                      t.astype(np.float64), s.n_in, width, depth, ns)
    # the bounds that the network's other gradient tests state for bf16 operands
    assert abs(loss - loss_ref) < 2e-2 * abs(loss_ref)
    layers, _, _, _ = M.layout(s.n_in, width, depth, ns)
    print(f"\n[mlp] n={n} width={width} depth={depth} loss {loss:.5g} {loss_ref:.5g}", flush=True)
    for (i, o, wo, bo) in layers:
        for a, b in ((g[wo:wo + i * o], g_ref[wo:wo + i * o]), (g[bo:bo + o], g_ref[bo:bo + o])):
            nrm = np.linalg.norm(b)
            assert np.linalg.norm(a - b) < 6e-2 * nrm, (wo, np.linalg.norm(a - b) / nrm)

    # Adam from m = v = 0 on that gradient: the same sums in the same order, then
    # a few roundings of 32 bits of the update and one of the weight
    lr, b1, b2, eps = 1e-3, 0.9, 0.999, 1e-8
    lb = torch.full((2,), 7.0, device="cuda")
    torch.cuda.synchronize()
    s._chk(s.L.abc_mlp_train_step_dev(s.h, n, C.c_void_p(xd.data_ptr()), C.c_void_p(td.data_ptr()),
                                      lr, b1, b2, eps, 0.0, C.c_void_p(lb[1:].data_ptr())), "step")
    s._chk(s.L.abc_mlp_synchronize(s.h), "sync")
    w1 = s.get_params()
    assert lb[0].item() == 7.0 and abs(lb[1].item() - loss) <= 1e-5 * abs(loss)
    m = (f32(1) - f32(b1)) * g
    v = (f32(1) - f32(b2)) * g * g
    c1, c2 = f32(1) - f32(b1), f32(1) - f32(b2)
    want = w0.astype(np.float64) - lr * (m / c1).astype(np.float64) / (np.sqrt(v / c2) + f32(eps))
    big = np.abs(g) > 1e-12
    assert np.all(np.abs(w1 - want)[big] <= 1e-5 * lr + 1.3e-7 * np.abs(w0)[big])
    assert np.all(np.abs(w1 - w0)[~big] <= 1e-3 * lr + 1.3e-7 * np.abs(w0)[~big])
    s.close()
