"""Dense tails of the orders that only a kept hierarchy takes (513 to 768 rows): the mixed solve with
the tail needs no more iterations than without it (+1 for rounding), and both end within the
tolerance-implied distance of the FP64 solution; the one-shot solve, whose hierarchy serves one
solve, is unchanged by it.
"""
from __future__ import annotations

import numpy as np
import pytest

import cfd_amd
from cfd_amd import AmgHierarchy, AmgSettings, Method, Precision, SolveControl, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(16, 16, 16), (20, 17, 13), (48, 44, 40), (48, 48, 48)])
def test_kept_tail(monkeypatch, shape):
    s = cases.pressure_system(cases.box_mesh(*shape, jitter=0.2, seed=5), rhs_seed=6)
    pat = cases.csr_pattern(s.n, s.owner, s.neighbour)
    h = AmgHierarchy(cases.ldu_to_csr(pat, s.diag, s.upper, s.lower), AmgSettings(strength_decay=0.5))
    assert any(512 < n <= 768 for n in h.level_sizes()[1:-1]), h.level_sizes()
    control = SolveControl(1e-9 * float(np.linalg.norm(s.source)), 300)

    def solve(prec):
        with cfd_amd.DeviceSolver(pat) as dev:
            dev.assemble(s.diag, s.upper, s.lower)
            dev.set_amg(h.view())
            dev.set_rhs(s.source)
            st = dev.solve_resident(Method.Cg, True, prec, control)
            assert st.converged
            return st.iterations, dev.get_x()

    _, x64 = solve(Precision.FP64)
    with_tail, xt = solve(Precision.MIXED_FP32)
    once = np.zeros(s.n)
    one_shot = cfd_amd.solve_amg_cg(h.view(), s.source, once, control, precision=Precision.MIXED_FP32).iterations
    monkeypatch.setenv("CFDG_DENSE_TAIL", "0")
    without, xf = solve(Precision.MIXED_FP32)
    assert with_tail <= without + 1 and one_shot <= without + 1
    # |x - x64| <= |A^-1| (|r| + |r64|), and the solution is at least as smooth as the right-hand side:
    # 25 tolerances in the norm (six at most were measured)
    for x in (xt, xf, once):
        assert np.linalg.norm(x - x64) <= 25e-9 * np.linalg.norm(x64)
