"""The tiled error kernel (known-divisor division, overlapping last tiles,
pairs formed again where operands leave its range) against the CPU oracle, bit
for bit, at the edges of its tiles and dispatch."""
import numpy as np
import pytest

from abc_inference_transcription_amd.design import reference_design

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng(engine_factory):
    return engine_factory(reference_design(cells=55))


def _same(a, b):
    return np.array_equal(np.isnan(a), np.isnan(b)) and \
        np.array_equal(np.nan_to_num(a, nan=-1.0).view(np.uint64),
                       np.nan_to_num(b, nan=-1.0).view(np.uint64))


# particles x genes: one lane per pair; 16-particle tiles with 4-particle waves
# (remainders 0, 1, 3); 64-particle tiles (remainders); one gene past a tile
@pytest.mark.parametrize("n,G,parts", [
    (3, 40, [5, 5, 3]), (64, 3200, [1]), (65, 3200, [5, 5, 5, 5, 11, 11, 11]),
    (67, 3201, [16]), (1024, 1024, [17]), (1025, 1025, [45, 45]), (1039, 1087, [0, 7, 0, 9, 0]),
    (4100, 64, [5, 5, 5, 5, 11, 11, 11]), (257, 4097, [100, 28])])
def test_error_tiles_bit_exact(oracle, eng, n, G, parts):
    rng = np.random.default_rng(n + G)
    K = sum(parts)
    stats = rng.lognormal(0.0, 2.0, (n, K)) * rng.choice([0.0, 1.0], (n, K), p=[0.1, 0.9])
    data = rng.lognormal(0.0, 2.0, (G, K)) * rng.choice([0.0, 1.0], (G, K), p=[0.1, 0.9])
    se = data * rng.uniform(0.0, 0.3, (G, K))
    print(f"\n[err tiles] n={n} G={G} K={K}", flush=True)
    got = eng.errors(stats, data, se, parts=parts, clamp=1e300)
    assert _same(got, oracle.errors(stats, data, se, np.array(parts, np.int32), clamp=1e300))


@pytest.mark.parametrize("n,G", [(70, 3200), (1100, 1030)])
def test_error_tiles_extreme_operands(oracle, eng, n, G):
    """NaN, infinite, tiny and huge statistics, data and errors: particles and
    genes outside the fast division's range keep the reference's bits."""
    rng = np.random.default_rng(5)
    K, parts = 20, [5, 5, 10]
    odd = np.array([np.nan, np.inf, -np.inf, 1e-300, 5e-324, 1e300, -1e-40, 1e61, 0.0, 1.7e308])
    a = [rng.lognormal(0.0, 1.0, s) for s in ((n, K), (G, K), (G, K))]
    for x in a:
        rows = rng.choice(len(x), 60, replace=False)
        x[rows, rng.integers(0, K, 60)] = rng.choice(odd, 60)
    got = eng.errors(*a, parts=parts, clamp=10.0)
    assert _same(got, oracle.errors(*a, np.array(parts, np.int32), clamp=10.0))
