"""Pools of device blocks on the device: release on request, alignments of several contexts made and
dropped at once, and alignments that outlive their context.  (The pools' own rules: test_pool.py.)"""
import ctypes as C
import threading

import numpy as np
import pytest

import rscape_amd as R
from rscape_amd import synth

pytestmark = pytest.mark.gpu


def free_bytes():
    hip = C.CDLL("libamdhip64.so")
    f, t = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


def scores(c, ax, w):
    m = c.msa(ax, w)
    ext = m.calculate("GTp", counts=R.COUNTS_INT8 if w is None else R.COUNTS_W8)
    cov = m.get_cov()[0]
    m.close()
    return cov, ext


def test_trim_gives_memory_back():
    """An alignment's records (72 MB at 1500 columns) stay with the context when it is closed and go
    back to the device with trim; the next alignment scores as before."""
    c = R.Context(0)
    ax = synth.random_msa(40, 1500, np.random.default_rng(1), gap=0.1)
    first, _ = scores(c, ax, None)
    kept = free_bytes()
    c.trim()
    assert free_bytes() - kept >= 32 * 1500 * 1500
    assert np.array_equal(scores(c, ax, None)[0], first)
    c.close()


def test_contexts_in_threads():
    """Three contexts, each with a thread that makes, scores and drops alignments of several sizes, one of
    them kept beside the others and trimmed under: the scores are those of one thread alone."""
    rng = np.random.default_rng(2)
    jobs = []
    for k, (N, L) in enumerate(((60, 41), (300, 97), (513, 64), (7, 200), (61, 42))):
        jobs.append((synth.random_msa(N, L, rng, gap=0.1), rng.uniform(0.2, 2.0, N) if k % 2 else None))
    c = R.Context(0)
    ref = [scores(c, *j) for j in jobs]
    c.close()
    bad = []

    def work(t):
        try:
            c = R.Context(0)
            keep = c.msa(*jobs[t])
            for i in range(12):
                k = (i * (t + 2)) % len(jobs)
                cov, ext = scores(c, *jobs[k])
                if not (np.array_equal(cov, ref[k][0]) and ext == ref[k][1]):
                    bad.append((t, i, k))
                if i % 5 == 4:
                    c.trim()
            keep.calculate("GTp", counts=R.COUNTS_INT8 if jobs[t][1] is None else R.COUNTS_W8)
            if not np.array_equal(keep.get_cov()[0], ref[t][0]):
                bad.append((t, "kept"))
            keep.close()
            c.close()
        except Exception as e:                                   # pytest does not see another thread's
            bad.append((t, repr(e)))

    th = [threading.Thread(target=work, args=(t,)) for t in range(3)]
    for x in th:
        x.start()
    for x in th:
        x.join()
    assert not bad, bad


def test_alignment_outlives_its_context():
    """An alignment dropped after its context, and one used by another context and dropped after both."""
    ax = synth.random_msa(50, 90, np.random.default_rng(3), gap=0.1)
    a, b = R.Context(0), R.Context(0)
    ref, ext = scores(b, ax, None)
    m, n = a.msa(ax), a.msa(ax)
    m.calculate("GTp")
    n.ctx = b
    a.close()
    assert n.calculate("GTp") == ext and np.array_equal(n.get_cov()[0], ref)
    m.close()
    assert np.array_equal(scores(b, ax, None)[0], ref)
    b.close()
    n.close()
