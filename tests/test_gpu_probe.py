"""Kernel timing counts the launches that did work: one an iteration, and for the level-0 sweep the cycle
after which the iteration limit was found exceeded; none more when a solve converges or breaks down."""
from __future__ import annotations

import numpy as np
import pytest

import cfd_amd
from cfd_amd import AmgHierarchy, AmgSettings, Method, Precision, SolveControl, cases

pytestmark = pytest.mark.gpu

SWEEP, SPMV = 1, 2


@pytest.mark.parametrize("prec", [Precision.FP64, Precision.MIXED_FP32])
def test_launches_counted(prec):
    s = cases.pressure_system(cases.box_mesh(15, 13, 11, jitter=0.2, seed=5), rhs_seed=6)
    pat = cases.csr_pattern(s.n, s.owner, s.neighbour)
    view = AmgHierarchy(cases.ldu_to_csr(pat, s.diag, s.upper, s.lower), AmgSettings(strength_decay=0.5)).view()
    tol = 1e-9 * float(np.linalg.norm(s.source))
    with cfd_amd.DeviceSolver(pat) as dev:
        dev.set_amg(view)
        dev.set_rhs(s.source)

        def launches(kind, limit):
            dev.set_x(None)
            dev.probe(kind)
            st = dev.solve_resident(Method.Cg, True, prec, SolveControl(tol, limit))
            _, n, _ = dev.probe_read(prec)
            dev.probe(0)
            return st, n

        dev.assemble(s.diag, s.upper, s.lower)
        for limit in (0, 3, 300):
            for kind in (SWEEP, SPMV):
                st, n = launches(kind, limit)
                assert st.converged == (limit == 300)
                assert n == st.iterations + (kind == SWEEP and not st.converged)
        dev.assemble(0.0 * s.diag, 0.0 * s.upper, 0.0 * s.lower)  # p.Ap = 0 in the first iteration
        for kind in (SWEEP, SPMV):
            st, n = launches(kind, 300)
            assert (st.iterations, st.converged, n) == (1, False, 1)
