"""The bound of the fixed-epsilon rule's device list: a batch that passes it by
itself, a tight session after a loose one on the same context, and the memory
that a large session leaves behind."""
import ctypes as C
import time

import numpy as np
import pytest

from abc_inference_transcription_amd.design import reference_design

pytestmark = pytest.mark.gpu
PARTS = np.array([3, 2], np.int32)
p = lambda a: C.c_void_p(a.ctypes.data)


def _inputs(n, G, seed):
    rng = np.random.default_rng(seed)
    data = np.asfortranarray(rng.lognormal(0.0, 0.2, (G, 5)))
    return np.asfortranarray(rng.lognormal(0.0, 0.2, (n, 5))), data, np.asfortranarray(0.1 * data)


def _begin(eng, data, se, eps):
    eng._chk(eng.L.abc_accept_begin(eng.ctx, 5, len(data), p(data), p(se), p(PARTS), 2, 10.0, 0,
                                    eps, 0, 0.02), "begin")


def _add(eng, x, first=0):
    eng._chk(eng.L.abc_accept_add(eng.ctx, len(x), p(x), first), "add")


def _end(eng, G, cap):
    counts, idx, err = np.zeros(G, np.int64), np.zeros(cap, np.int64), np.zeros(cap)
    eng._chk(eng.L.abc_accept_end(eng.ctx, p(counts), p(idx), p(err), cap, None), "end")
    return counts, idx, err


def test_one_batch_beyond_the_list(oracle, engine_factory):
    """2^26 + 2.9 million pairs in one batch, after a small one and before
    another: lists of every batch, whole and in order."""
    eng = engine_factory(reference_design(cells=55))
    n, G = 2000, 35000
    x, data, se = _inputs(n, G, 1)
    more = [_inputs(40, 1, 2)[0], _inputs(30, 1, 3)[0]]
    _begin(eng, data, se, 10.0)
    for b, first in ((more[0], 0), (x, 40), (more[1], 40 + n)):
        print(f"\n[bounds] batch of {len(b)}", flush=True)
        _add(eng, b, first)
    rows = np.vstack([more[0], x, more[1]])
    counts, idx, err = _end(eng, G, len(rows) * G)
    assert np.all(counts == len(rows))
    idx, err = idx.reshape(G, -1), err.reshape(G, -1)
    for g in (0, 1, 17777, G - 1):
        e = oracle.errors(rows, data[g:g + 1], se[g:g + 1], PARTS)[:, 0]
        o = np.argsort(e, kind="stable")
        assert np.array_equal(idx[g], o + 1) and np.array_equal(err[g], e[o]), g


def test_memory_of_a_large_session_is_given_back(engine_factory):
    """60 million pairs: the lists took 4.4 GB of device memory until the context
    was destroyed, besides the 2 GB of candidates."""
    import torch
    n, G = 2000, 30000
    x, data, se = _inputs(n, G, 4)
    free = torch.cuda.mem_get_info()[0]
    eng = engine_factory(reference_design(cells=55))
    _begin(eng, data, se, 10.0)
    _add(eng, x)
    counts = _end(eng, G, n * G)[0]
    assert np.all(counts == n)
    held = free - torch.cuda.mem_get_info()[0]
    print(f"\n[bounds] held after the session: {held / 2**30:.2f} GiB", flush=True)
    assert held < 3 << 30


def test_tight_session_after_a_loose_one(engine_factory):
    """The first session's 60 million candidates set the capacity of later
    batches, not where their accepted pairs are kept."""
    x, data, se = _inputs(2000, 30000, 5)
    eps = 0.25

    def tight(eng):
        best, out = np.inf, None
        for _ in range(8):
            _begin(eng, data, se, eps)
            t = time.perf_counter()
            for a in range(0, 2000, 250):
                _add(eng, np.asfortranarray(x[a:a + 250]), a)
            out = _end(eng, len(data), 20_000_000)
            best = min(best, time.perf_counter() - t)
        return best, out

    fresh_t, fresh = tight(engine_factory(reference_design(cells=55)))
    eng = engine_factory(reference_design(cells=55))
    _begin(eng, data, se, 10.0)
    _add(eng, x)
    after_t, after = tight(eng)
    total = int(fresh[0].sum())
    print(f"\n[bounds] {total} pairs: fresh {1e3 * fresh_t:.1f} ms, after a loose session "
          f"{1e3 * after_t:.1f} ms", flush=True)
    for a, b in zip(fresh, after):
        assert np.array_equal(a, b)
    assert after_t < 2.0 * fresh_t
