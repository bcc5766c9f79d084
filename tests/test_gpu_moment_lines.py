"""The moment model's split between teams and single lanes: no step in a call's
time where one more particle is asked for, and the same bits on both sides of the
lines of the rule (every particle in teams, some of them, other item counts)."""
import time

import numpy as np
import pytest

from abc_inference_transcription_amd.design import REF_CHASE, REF_PULSE, reference_design

pytestmark = pytest.mark.gpu
AGES = [2.0, 6.0, 10.0, 14.0, 18.0]


@pytest.fixture(scope="module")
def eng(engine_factory):
    return engine_factory(reference_design(cells=55))


@pytest.mark.parametrize("model", [3, 4])
def test_one_more_particle(eng, model):
    """4,096 and 4,097 particles: 48 and 56 ms (model 3), 42 and 54 ms (model 4)
    with a line between them."""
    from abc_inference_transcription_amd.engine import MomentCfg
    cfg = MomentCfg(AGES, REF_PULSE, REF_CHASE, is_chase=[0] * 6 + [1] * 5, cycle=20.0)
    th = eng.sample_prior(model, 4097, seed=0, first=0)
    calls = {n: np.asfortranarray(th[:n]) for n in (4096, 4097)}
    best = dict.fromkeys(calls, np.inf)
    for _ in range(5):
        for n, x in calls.items():
            t = time.perf_counter()
            eng.recover(model, x, cfg)
            best[n] = min(best[n], 1e3 * (time.perf_counter() - t))
    print(f"\n[moment lines] model {model}: {best}", flush=True)
    assert best[4097] < 1.12 * best[4096]


# (condition, age) items, and particles on both sides of the rule's lines on 256
# CUs: cycle maps of 10 columns at 13,056 (waves of one lane a particle 2,040,
# 2,050), trajectories at 4,736 with 55 items (4,070, 4,125), 261,888 with one
@pytest.mark.parametrize("model,n,conds,ages", [
    (1, 4736, 11, 5), (3, 4737, 11, 5), (5, 4800, 11, 5), (2, 13056, 2, 2), (4, 13057, 2, 2),
    (1, 65537, 1, 1), (2, 40, 11, 5)])
def test_same_bits_across_the_lines(eng, model, n, conds, ages):
    from abc_inference_transcription_amd.engine import MomentCfg
    cfg = MomentCfg(AGES[:ages], REF_PULSE[:conds], REF_CHASE[:conds], cycle=20.0, rtol=1e-7)
    th = eng.sample_prior(model, n, seed=5, first=0)
    print(f"\n[moment lines] model {model} n={n} items={conds * ages}", flush=True)
    whole, steps = eng.recover(model, th, cfg, steps=True)
    rows = np.random.default_rng(n).choice(n, min(n, 300), replace=False)
    rows = np.append(rows, [0, n - 1])
    # a call of so few is all teams
    part, st = eng.recover(model, np.asfortranarray(th[rows]), cfg, steps=True)
    same = lambda a, b: np.array_equal(np.ascontiguousarray(a).view(np.uint64),
                                       np.ascontiguousarray(b).view(np.uint64))
    assert same(whole[rows], part) and np.array_equal(steps[rows], st)
