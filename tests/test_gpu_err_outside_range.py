"""Operands outside the range of the error kernels' division by known
denominators (infinite, tiny, huge): the oracle's bits whatever share of a
tile's particles and genes has them, and no more time than dividing takes."""
import ctypes as C

import numpy as np
import pytest

from abc_inference_transcription_amd.design import reference_design

pytestmark = pytest.mark.gpu
PARTS = np.array([5, 5, 5, 5, 11, 11, 11], np.int32)
ODD = np.array([np.inf, -np.inf, 1e-300, 1e300, 1e61, 1e-40, np.nan])


@pytest.fixture(scope="module")
def eng(engine_factory):
    return engine_factory(reference_design(cells=55))


def _ms(eng, torch, particles, genes, value, n=9973, G=3419):
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


# a kernel that divides throughout takes 2.7 times the time of finite operands;
# pairs formed again one particle at a time took 5 and 4.5 times
@pytest.mark.parametrize("particles,genes,value", [
    (1.0, 0.0, np.inf), (0.0, 0.05, np.inf), (0.0, 1.0, np.inf), (0.0, 0.05, 1e70)])
def test_odd_operands_cost_at_most_a_division(eng, particles, genes, value):
    import torch
    plain, odd = _ms(eng, torch, 0.0, 0.0, 0.0), _ms(eng, torch, particles, genes, value)
    print(f"\n[outside range] plain {plain:.3f} ms, with {value} {odd:.3f} ms", flush=True)
    assert odd < 3.2 * plain


# shares of 1/64 to all of the particles and genes; the last tile of 64 genes
# full or of one gene, its particles a remainder
@pytest.mark.parametrize("n,G", [(1111, 1025), (1100, 1024), (300, 700)])
@pytest.mark.parametrize("particles,genes", [(0.02, 0.02), (0.15, 0.3), (0.5, 0.0), (1.0, 0.1),
                                             (0.1, 1.0), (1.0, 1.0)])
def test_any_share_bit_exact(oracle, eng, n, G, particles, genes):
    rng = np.random.default_rng(n + G)
    K, parts = 12, np.array([5, 0, 7], np.int32)
    stats, data, se = (rng.lognormal(0.0, 1.0, s) for s in ((n, K), (G, K), (G, K)))
    for a, share in ((stats, particles), (data, genes)):
        rows = np.nonzero(rng.random(len(a)) < share)[0]
        a[rows, rng.integers(0, K, len(rows))] = rng.choice(ODD, len(rows))
    data[G - 1, 3] = 1e-200              # the gene that the last tile's idle lanes repeat
    want = oracle.errors(stats, data, se, parts, clamp=1e290)
    got = eng.errors(stats, data, se, parts=parts, clamp=1e290)
    num = ~np.isnan(want)
    assert np.array_equal(np.isnan(got), ~num) and np.array_equal(got[num], want[num])
    # the first block of a top-k session is the same kernel's
    want = oracle.errors(stats, data, se, parts, clamp=30.0)
    lists = eng.accept(stats, data, se, parts=parts, clamp=30.0, mode=1, k=25)
    for g in range(0, G, 7):
        o = np.argsort(want[:, g], kind="stable")
        o = o[~np.isnan(want[o, g])][:25]
        assert np.array_equal(lists[g][0], o + 1) and np.array_equal(lists[g][1], want[o, g]), g
