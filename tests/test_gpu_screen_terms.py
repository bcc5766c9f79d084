"""The surrogate's screen: scores and pass flags of every particle against the
same formula in NumPy, at the edges of a workgroup's particles (8) and genes
(two of 256 lanes), on both of its paths: moments and data inside the range of
the short form of the variance term, and outside it (tiny or huge moments, a
huge datum, a datum that is not finite, a threshold at the clamp)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
CLAMP = 1e6
GX = np.array([-3.7504397177257425, -2.366759410734541, -1.1544053947399682, 0.0,
               1.1544053947399682, 2.366759410734541, 3.7504397177257425])
GW = np.array([0.000548268855972217, 0.03075712396758652, 0.2401231786050127, 0.45714285714285724,
               0.2401231786050127, 0.03075712396758652, 0.000548268855972217])
f32 = np.float32


@pytest.fixture(scope="module")
def eng(engine_factory):
    from abc_inference_transcription_amd.design import reference_design
    return engine_factory(reference_design(cells=55))


def _reference(y, mean, sd, data, W, thr):
    """margins (n x G) with a bound of their error.  The moments may differ by
    one unit of their 24 bits (6e-8); sums of up to 90 terms add 90 * 6e-8 of
    their magnitude: 1e-5 of the magnitudes covers both."""
    n, K = y.shape[0], y.shape[1] // 2
    mu, lv = y[:, :K].astype(np.float64), np.clip(y[:, K:].astype(np.float64), -12, 12)
    sv = np.sinh(mean[None, :, None] + sd[None, :, None] * (mu[..., None] +
                                                            np.exp(0.5 * lv)[..., None] * GX))
    m1 = (GW * sv).sum(-1)
    e = sv - m1[..., None]
    v2, v3, v4 = (GW * e**2).sum(-1), (GW * e**3).sum(-1), (GW * e**4).sum(-1)
    d = data[None, :, :]                                  # 1 x G x K
    dl, w = d - m1[:, None, :], W[None, :, :]
    a, c3, c4, ae = v2[:, None, :], np.abs(v3)[:, None, :], v4[:, None, :], np.abs(m1)[:, None, :]
    em = (w * (dl**2 + a)).sum(-1)
    ev = (w**2 * np.maximum(4 * dl**2 * a - 4 * dl * v3[:, None, :] + c4 - a**2, 0)).sum(-1)
    dem = 1e-5 * (w * (dl**2 + 2 * np.abs(dl) * (ae + np.abs(d)) + a)).sum(-1)
    dev = 1e-5 * (w**2 * (4 * dl**2 * a + 8 * np.abs(dl) * (ae + np.abs(d)) * a +
                          4 * (np.abs(dl) + ae + np.abs(d)) * c3 + c4 + a**2)).sum(-1)
    # the kernel's 32-bit sums may overflow to infinity: sd infinite, margin 0
    m, x2, x3, x4 = (q[:, None, :].astype(f32) for q in (m1, v2, v3, v4))
    dl32, w32 = d.astype(f32) - m, w.astype(f32)
    ev32 = np.zeros(em.shape, f32)
    for k in range(K):
        q = dl32[..., k]
        ev32 += (w32[..., k] * w32[..., k]) * np.maximum(
            f32(4) * q * q * x2[..., k] - f32(4) * q * x3[..., k] + x4[..., k] -
            x2[..., k] * x2[..., k], f32(0))
    s = np.where(np.isinf(ev32), np.inf, np.sqrt(ev))
    u = (thr[None, :] - em) / s
    du = (dem + 1e-6 * np.abs(thr)[None, :] + np.abs(u) * dev / (2 * s)) / s + 1e-5 * np.abs(u)
    return u, du


@pytest.mark.parametrize("n,G,K,kind", [
    (1, 1, 3, "plain"), (7, 255, 90, "plain"), (8, 256, 5, "plain"), (9, 257, 90, "plain"),
    (17, 511, 2, "plain"), (16, 513, 45, "plain"), (9, 300, 7, "zero mean"),
    (20, 257, 7, "huge moments"), (12, 520, 6, "genes")])
def test_screen_terms(eng, n, G, K, kind):
    import torch
    from scipy.special import ndtr
    from abc_inference_transcription_amd import _lib
    from abc_inference_transcription_amd.screened_abc import _end
    from abc_inference_transcription_amd.surrogate import Surrogate
    rng = np.random.default_rng(1000 * n + G)
    sur = Surrogate(K, n_bins=5, width=128, depth=1, max_batch=64, seed=3)
    mean, sd = rng.uniform(0.3, 2.0, K), rng.uniform(0.1, 0.6, K)
    if kind == "zero mean":
        mean[:] = 0.0
        p = sur.get_params()
        p[:] = 0.0           # every prediction is 0 with variance 1
        sur.set_params(p)
    if kind == "huge moments":
        mean[0], sd[0] = 22.0, 0.5   # E s about 2e9
    sur.mean = torch.tensor(mean, dtype=torch.float32, device="cuda")
    sur.sd = torch.tensor(sd, dtype=torch.float32, device="cuda")
    mean, sd = sur.mean.cpu().double().numpy(), sur.sd.cpu().double().numpy()
    x = torch.randn(n, sur.n_in, device="cuda")
    data = np.asfortranarray(np.sinh(rng.uniform(0.0, 2.5, (G, K))))
    se = np.asfortranarray(np.abs(data) * rng.uniform(0.1, 0.5, (G, K)))
    thr = rng.uniform(0.5, 60.0, G)
    if kind == "huge moments":
        data[:, 0], se[:, 0] = 2e9, 1e9
    if kind == "genes":
        data[5, 2], se[5, 2] = 2.0**31, 2.0**30     # lanes of both halves, one in each
        data[300, 1], se[300, 1] = -2.0**33, 2.0**31
        data[7, 0] = np.nan
        thr[11], thr[256 + 40] = CLAMP, 2 * CLAMP
        thr[5], thr[300] = 1e5, 1e5
    vp = lambda a: a.ctypes.data_as(C.c_void_p)
    parts = np.array([K], np.int32)
    eng._chk(eng.L.abc_accept_begin(eng.ctx, K, G, vp(data), vp(se), vp(parts), 1, CLAMP, 0, 2 * CLAMP,
                                    0, 0.0), "begin")
    eng._chk(eng.L.abc_accept_set_thresholds(eng.ctx, vp(thr)), "thresholds")
    y = sur.predict(x).cpu().numpy()
    sc = sur.scores(eng, x)
    torch.cuda.synchronize()  # the engine has a stream of its own
    sc = sc.cpu().numpy().astype(np.float64)
    flags = {z: sur.screen(eng, x, z=z)[0].cpu().numpy().astype(bool) for z in (0.5, 4.0)}
    _end(eng, G, 16)
    sur.close()

    W = (1.0 / (K * (se**2 + 0.01 * data**2))).astype(f32).astype(np.float64)
    keep = np.isfinite(data).all(1) & (thr < CLAMP)
    u, du = _reference(y, mean, sd, data.astype(f32).astype(np.float64)[keep], W[keep], thr[keep])
    clamped = int((thr >= CLAMP).sum())
    print(f"\n[screen] {kind} n={n} G={G} K={K} margin {u.max():.3g}", flush=True)
    want = ndtr(u).sum(1) + clamped
    assert np.all(np.abs(sc[:, 0] - want) <= np.minimum(0.4 * du, 1.0).sum(1) + 2e-6 * G + 1e-6)
    if clamped:
        assert np.all(np.isinf(sc[:, 1])) and all(f.all() for f in flags.values())
        return
    best = u.max(1)
    assert np.all(np.abs(sc[:, 1] - best) <= du.max(1) + 1e-6)
    for z, f in flags.items():
        sure = np.abs(u + z) > du + 1e-5
        assert np.all(f[(sure & (u > -z)).any(1)])
        assert not np.any(f[(sure & (u < -z)).all(1)])

