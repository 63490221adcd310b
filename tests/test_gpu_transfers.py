"""Host arrays of every size class of the staged copies (below the staging limit, within the ring of
pinned slots, past its end, with partial last pieces) reach the device and come back unchanged, from
one thread and from several at once, and together in one call (DeviceSolver.assemble).
"""
from __future__ import annotations

import ctypes as C
import threading

import numpy as np
import pytest

import cfd_amd
from cfd_amd import _lib as L
from cfd_amd import LduPattern, Method, SolveControl, cases

pytestmark = pytest.mark.gpu

MIB = 1 << 17  # doubles in a MiB


def _diagonal(n):
    i = np.arange(n, dtype=np.int32)
    none = np.zeros(0, np.int32)
    return cfd_amd.DeviceSolver(LduPattern(n, 0, n, np.arange(n + 1, dtype=np.int32), i, i, none, none))


def _round_trip(dev, seed):
    x = np.random.default_rng(seed).standard_normal(dev.n)
    dev.set_x(x)
    assert np.array_equal(dev.get_x(), x)


@pytest.mark.parametrize("n", [1, 3 * MIB - 1, 3 * MIB, 4 * MIB + 1, 16 * MIB - 1, 16 * MIB + 1, 32 * MIB,
                               32 * MIB + 1, 70 * MIB + 77])
def test_round_trip(n):
    with _diagonal(n) as dev:
        for seed in range(3):
            _round_trip(dev, seed)


def test_round_trips_from_several_threads():
    devs = [_diagonal(n) for n in (5 * MIB, 18 * MIB + 3, 7 * MIB + 1, 16 * MIB)]
    failed = []

    def work(k):
        try:
            for seed in range(4):
                _round_trip(devs[k], 10 * k + seed)
        except BaseException as e:
            failed.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(devs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for d in devs:
        d.close()
    assert not failed


def _mapped_mib():
    with open("/proc/self/status") as f:
        return next(int(line.split()[1]) for line in f if line.startswith("VmSize:")) / 1024


def test_staging_memory_is_bounded_and_given_back():
    """More callers at once than staging areas are kept: all results whole, and the areas go with the
    cached memory (a copy needs 32 MiB of pinned memory; 8 callers' areas are kept)."""
    devs = [_diagonal(4 * MIB + 11 * k) for k in range(12)]
    xs = [np.random.default_rng(k).standard_normal(d.n) for k, d in enumerate(devs)]
    for d, x in zip(devs, xs):
        d.set_x(x)
    gate = threading.Barrier(len(devs))
    same = [False] * len(devs)

    def work(k):
        ok = True
        for _ in range(10):
            gate.wait()
            ok = np.array_equal(devs[k].get_x(), xs[k]) and ok
        same[k] = ok

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(devs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(same)
    before = _mapped_mib()
    slabs = C.c_size_t()
    L.call("cfdg_release_cached_memory", C.byref(slabs), None)
    freed = before - _mapped_mib() - slabs.value / 2 ** 20  # device memory is mapped, too
    assert 32 <= freed <= 8 * 32 + 16
    for seed in range(2):  # and anew
        _round_trip(devs[0], seed)
    for d in devs:
        d.close()


@pytest.mark.parametrize("shape", [(40, 40, 40), (75, 70, 66)])  # 3.5 and 19 MiB of coefficients
def test_coefficients_of_a_host_call(shape):
    s = cases.momentum_system(cases.box_mesh(*shape, jitter=0.2, seed=8), 1.0, 9)
    pat = cases.csr_pattern(s.n, s.owner, s.neighbour)
    x = np.zeros(s.n)
    with cfd_amd.DeviceSolver(pat) as dev:
        st = dev.solve(s.diag, s.upper, s.lower, s.source, x, Method.BiCgStab, False,
                       SolveControl(1e-10 * float(np.linalg.norm(s.source)), 300))
        assert st.converged
    r = s.source - cases.ldu_to_csr(pat, s.diag, s.upper, s.lower).to_scipy() @ x
    assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(s.source)
