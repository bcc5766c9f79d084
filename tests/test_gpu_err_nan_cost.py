"""Statistics and data that are not numbers (a ratio or a correlation of cells
without a count) are ordinary inputs of the error kernels: the same bits as the
oracle's and about the time of finite ones."""
import ctypes as C

import numpy as np
import pytest

from abc_inference_transcription_amd.design import reference_design

pytestmark = pytest.mark.gpu
PARTS = np.array([5, 5, 5, 5, 11, 11, 11], np.int32)


@pytest.fixture(scope="module")
def eng(engine_factory):
    return engine_factory(reference_design(cells=55))


def _ms(eng, torch, particles, genes, value, n=9973, G=3419):
    """Milliseconds of abc_errors_dev, the best of several calls, with one
    statistic of that share of the particles and of the genes set to value."""
    p = lambda t: C.c_void_p(t.data_ptr())
    g = torch.Generator(device="cuda").manual_seed(1)
    u = lambda *s: torch.rand(*s, generator=g, dtype=torch.float64, device="cuda")
    x, d = 3.0 * u(53, n), 0.1 + u(53, G)
    se, err = 0.2 * d, torch.zeros(G, n, dtype=torch.float64, device="cuda")
    x[3, u(n) < particles] = value
    d[5, u(G) < genes] = value
    torch.cuda.synchronize()
    best = np.inf
    for _ in range(6):
        eng._chk(eng.L.abc_errors_dev(eng.ctx, n, 53, p(x), G, p(d), p(se),
                                      PARTS.ctypes.data_as(C.c_void_p), len(PARTS), 10.0, p(err)),
                 "errors")
        best = min(best, float(eng.last_timing()[3]))
    return best


# formed again one pair a lane, these took 5 (particles) and 4.5 (genes) times
# as long as finite ones, twice a kernel that divides throughout
@pytest.mark.parametrize("particles,genes", [(1.0, 0.0), (0.0, 0.05), (0.3, 0.5)])
def test_nan_costs_what_numbers_cost(eng, particles, genes):
    import torch
    plain, nan = _ms(eng, torch, 0.0, 0.0, 0.0), _ms(eng, torch, particles, genes, float("nan"))
    print(f"\n[nan cost] finite {plain:.3f} ms, NaN {nan:.3f} ms", flush=True)
    assert nan < 1.6 * plain


@pytest.mark.parametrize("mode", [0, 1])
def test_nan_everywhere_bit_exact(oracle, eng, mode):
    """NaN in data, errors of either sign and statistics: the error matrix and
    the lists (NaN errors are never accepted)."""
    rng = np.random.default_rng(3)
    n, G, K = 700, 1100, 9
    parts = np.array([4, 5], np.int32)
    stats, data, se = (rng.lognormal(0.0, 0.5, s) for s in ((n, K), (G, K), (G, K)))
    for a in (stats, data, se):
        rows = rng.choice(len(a), len(a) // 3, replace=False)
        a[rows, rng.integers(0, K, len(rows))] = rng.choice([np.nan, -np.nan], len(rows))
    stats[5, 2] = np.inf
    stats[5, 3] = np.nan
    want = oracle.errors(stats, data, se, parts)
    got = eng.errors(stats, data, se, parts=parts)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~np.isnan(got)], want[~np.isnan(want)])
    eps = float(np.nanquantile(want, 0.05))
    lists = eng.accept(stats, data, se, parts=parts, mode=mode, eps=eps, k=40)
    for g in range(G):
        o = np.argsort(want[:, g], kind="stable")
        o = o[~np.isnan(want[o, g])]
        o = o[:40] if mode else o[want[o, g] <= eps]
        assert np.array_equal(lists[g][0], o + 1) and np.array_equal(lists[g][1], want[o, g]), g
