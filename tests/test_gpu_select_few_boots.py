"""Model probabilities with fewer resamples than a workgroup has waves: the
waves share a resample's labels."""
import time

import numpy as np
import pytest

from abc_inference_transcription_amd.design import reference_design

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng(engine_factory):
    return engine_factory(reference_design(cells=55))


def test_one_resample_uses_every_wave(eng):
    """8 million labels: 1 resample took the 7 ms of 4 with a wave each."""
    c = np.array([[4_000_000, 4_000_000]], np.int64)

    def ms(n_boot):
        best = np.inf
        for _ in range(5):
            t = time.perf_counter()
            eng.model_probs(c, n_boot=n_boot)
            best = min(best, time.perf_counter() - t)
        return 1e3 * best

    one, four = ms(1), ms(4)
    print(f"\n[few boots] 1 resample {one:.2f} ms, 4 resamples {four:.2f} ms", flush=True)
    assert one < 0.6 * four


# labels around whole rounds of one, two and four waves (128, 256, 512 draws),
# odd numbers among them; the last workgroup's resamples one, two and three
@pytest.mark.parametrize("n_boot", [1, 2, 3, 4, 8, 9, 10, 11])
@pytest.mark.parametrize("M", [2, 3, 8])
def test_shared_resamples_bit_exact(oracle, eng, n_boot, M):
    rng = np.random.default_rng(M)
    total = np.array([2, 3, 127, 128, 129, 255, 256, 257, 511, 512, 513, 514, 639, 641, 5001])
    c = np.array([rng.multinomial(t, rng.dirichlet(np.ones(M))) for t in total], np.int64)
    got = eng.model_probs(c, seed=4, n_boot=n_boot, alpha=0.8)
    want = oracle.model_probs(c, seed=4, n_boot=n_boot, alpha=0.8)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
