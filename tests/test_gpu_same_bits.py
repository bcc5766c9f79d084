"""Two ways to the same numbers: the one-launch inference and the layer-by-layer
path, the screen's short expression and the one it stands for."""
import ctypes as C

import numpy as np
import pytest

from abc_inference_transcription_amd.design import config_design

pytestmark = pytest.mark.gpu


def _net(ns, width, depth, seed=1, max_batch=512):
    from abc_inference_transcription_amd.surrogate import Surrogate
    return Surrogate(ns, width=width, depth=depth, max_batch=max_batch, seed=seed)


def _layers(s, width, depth):
    """(in, out) of every layer, padded as the flat parameters are."""
    ip, op = -(-s.n_in // 64) * 64, -(-2 * s.n_stats // 128) * 128
    return [(ip if l == 0 else width, op if l == depth else width) for l in range(depth + 1)]


# a network of width 640 is computed layer by layer; with the narrow network's
# weights and zeros its extra units are silu(0) = 0 and end every sum with zeros
@pytest.mark.parametrize("width,depth,ns", [(128, 1, 3), (256, 2, 90), (384, 3, 64), (512, 4, 90)])
@pytest.mark.parametrize("n", [1, 77, 1000, 5000, 17000])
def test_one_launch_equals_layer_by_layer(width, depth, ns, n):
    import torch
    a, b = _net(ns, width, depth), _net(ns, 640, depth)
    g = torch.Generator().manual_seed(n)
    flat = torch.tensor(a.get_params()) * 1.5
    la, lb, out, at = _layers(a, width, depth), _layers(b, 640, depth), [], 0
    for (i, o), (ib, ob) in zip(la, lb):
        W, c = flat[at:at + i * o].view(o, i), 0.3 * torch.randn(o, generator=g)
        flat[at + i * o:at + i * o + o] = c
        at += i * o + o
        Wb, cb = torch.zeros(ob, ib), torch.zeros(ob)
        Wb[:o, :i], cb[:o] = W, c
        out += [Wb.reshape(-1), cb]
    a.set_params(flat.numpy())
    b.set_params(torch.cat(out).numpy())
    x = (2.0 * torch.randn(n, a.n_in, generator=g)).to(a.dev)
    ya, yb = a.predict(x), b.predict(x)
    print(f"\n[same bits] n={n} width={width} depth={depth}", flush=True)
    assert torch.isfinite(ya).all() and ya.abs().max() > 0.1
    assert torch.equal(ya, yb)
    a.close()
    b.close()


def _in_range(y, mean, sd):
    """Which predictions (n x K) have all moments well inside the ranges of the
    screen's short expression."""
    K = len(mean)
    gx, gw = np.polynomial.hermite_e.hermegauss(7)
    gw = gw / gw.sum()
    s = np.exp(0.5 * np.clip(y[:, K:], -12.0, 12.0))
    v = np.sinh(mean[:, None] + sd[:, None] * (y[:, :K, None] + s[:, :, None] * gx))
    e = (v * gw).sum(-1)
    d = v - e[:, :, None]
    c2, c3, c4 = ((d ** q * gw).sum(-1) for q in (2, 3, 4))
    ok = (np.abs(e) > 2.0**-19) & (np.abs(e) < 2.0**29) & (c2 > 2.0**-37) & (c2 < 2.0**29)
    ok &= (np.abs(c3) > 2.0**-79) & (np.abs(c3) < 2.0**44) & (c4 > 2.0**-99) & (c4 < 2.0**59)
    return ok.all(1)


@pytest.mark.parametrize("G", [37, 700])
def test_short_variance_equals_the_expression(engine_factory, G):
    """Particles scored beside one out of the short expression's range (their
    workgroup then takes the expression as it stands) and beside ones inside it;
    genes beyond its range among the others."""
    import torch
    eng = engine_factory(config_design(cells=100))
    K, n = 90, 800
    rng = np.random.default_rng(G)
    data = np.asfortranarray(rng.lognormal(0.5, 1.0, (G, K)))
    data[3, 7] = 1e12
    se = np.asfortranarray(data * rng.uniform(0.05, 0.3, (G, K)))
    s = _net(K, 256, 2)
    s.mean = torch.tensor(rng.uniform(0.3, 1.5, K), dtype=torch.float32, device=s.dev)
    s.sd = torch.tensor(rng.uniform(0.3, 1.0, K), dtype=torch.float32, device=s.dev)
    x = torch.randn(n, s.n_in, generator=torch.Generator().manual_seed(2)).to(s.dev)
    odd = x.clone()
    odd[7::8] *= 2000.0                  # the last particle of every workgroup
    y, yo = (s.predict(a).double().cpu().numpy() for a in (x, odd))
    mean, sd = s.mean.double().cpu().numpy(), s.sd.double().cpu().numpy()
    inside = _in_range(y, mean, sd).reshape(-1, 8).all(1)
    with np.errstate(over="ignore", invalid="ignore"):
        outside = ~_in_range(yo, mean, sd).reshape(-1, 8)[:, 7]
    use = np.repeat(inside & outside, 8)
    use[7::8] = False
    assert use.sum() > 500
    parts = np.array([45, 45], np.int32)
    p = lambda a: C.c_void_p(a.ctypes.data)
    eng._chk(eng.L.abc_accept_begin(eng.ctx, K, G, p(data), p(se), p(parts), 2, 10.0, 0, 4.8, 0,
                                    0.02), "begin")
    both = [s.scores(eng, v) for v in (x, odd)]
    torch.cuda.synchronize()             # the engine has a stream of its own
    a, b = (t.cpu().numpy()[use] for t in both)
    print(f"\n[same bits] {use.sum()} particles, {G} genes", flush=True)
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert np.isfinite(a).all() and len(np.unique(a[:, 1])) > 100
    for z in (0.5, 2.0, 4.0):
        a, b = (s.screen(eng, v, z=z)[0].cpu().numpy()[use] for v in (x, odd))
        assert np.array_equal(a, b)
    s.close()
