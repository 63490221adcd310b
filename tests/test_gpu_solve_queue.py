"""The queueing of iterations (one, two or four to a graph launch, as many as the reported
residuals let the host expect): a solve ends at the same iteration with the same residual and
solution, bit for bit, launched kernel by kernel (a system's first solve) and replayed from graphs,
at every iteration limit around the sizes of the graphs, without a tolerance to reach, from a
converged start and with a right-hand side that is not a number.
"""
from __future__ import annotations

import numpy as np
import pytest

import cfd_amd
from cfd_amd import AmgHierarchy, AmgSettings, Method, Precision, SolveControl, cases

pytestmark = pytest.mark.gpu

RUNS = {"cg": (Method.Cg, False, Precision.FP64), "bicgstab": (Method.BiCgStab, False, Precision.FP64),
        "amg": (Method.Cg, True, Precision.FP64), "mixed": (Method.Cg, True, Precision.MIXED_FP32)}


def _system(shape=(15, 13, 11)):
    s = cases.pressure_system(cases.box_mesh(*shape, jitter=0.2, seed=5), rhs_seed=6)
    pat = cases.csr_pattern(s.n, s.owner, s.neighbour)
    dev = cfd_amd.DeviceSolver(pat)
    dev.assemble(s.diag, s.upper, s.lower)
    dev.set_amg(AmgHierarchy(cases.ldu_to_csr(pat, s.diag, s.upper, s.lower), AmgSettings(strength_decay=0.5)).view())
    dev.set_rhs(s.source)
    return s, dev


def _solve(dev, run, control):
    dev.set_x(None)
    st = dev.solve_resident(*RUNS[run], control)
    return st.iterations, st.converged, st.residual, st.true_residual, dev.get_x().tobytes()


@pytest.mark.parametrize("run", list(RUNS))
def test_every_limit_ends_alike_in_direct_and_graph_launches(run):
    s, dev = _system()
    tol = 1e-9 * float(np.linalg.norm(s.source))
    with dev:
        full = _solve(dev, run, SolveControl(tol, 400))
        assert full[1] and full == _solve(dev, run, SolveControl(tol, 400))
        for limit in list(range(10)) + [full[0] - 1, full[0], full[0] + 1]:
            with _system()[1] as fresh:  # its first solve launches kernel by kernel
                direct = _solve(fresh, run, SolveControl(tol, limit))
            assert _solve(dev, run, SolveControl(tol, limit)) == direct
            assert direct[0] == min(limit, full[0])
            assert direct[1] == (limit >= full[0])
        assert _solve(dev, run, SolveControl(0.0, 23))[0] == 23  # no tolerance to reach


@pytest.mark.parametrize("run", list(RUNS))
def test_converged_start_and_nan(run):
    s, dev = _system()
    tol = 1e-7 * float(np.linalg.norm(s.source))
    with dev:
        for _ in range(3):
            dev.set_x(None)
            assert dev.solve_resident(*RUNS[run], SolveControl(0.01 * tol, 400)).converged
            st = dev.solve_resident(*RUNS[run], SolveControl(tol, 400))  # from the solution
            assert st.converged and st.iterations == 0
        b = s.source.copy()
        b[3] = np.nan
        dev.set_rhs(b)
        for _ in range(2):
            dev.set_x(None)
            st = dev.solve_resident(*RUNS[run], SolveControl(tol, 9))
            assert not st.converged
