"""Dense tails end at 512 rows where their inverse would hold more than a tenth of the finest operator's
entries, also in a hierarchy given to set_amg: a level of 513 to 768 rows is smoothed, so that the mixed
solve is, bit for bit, the one without dense tails, and agrees with the FP64 solution.
"""
from __future__ import annotations

import numpy as np
import pytest

import cfd_amd
from cfd_amd import AmgHierarchy, AmgSettings, Method, Precision, SolveControl, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(16, 16, 16), (20, 17, 13)])
def test_level_above_the_tail_order(monkeypatch, shape):
    s = cases.pressure_system(cases.box_mesh(*shape, jitter=0.2, seed=5), rhs_seed=6)
    pat = cases.csr_pattern(s.n, s.owner, s.neighbour)
    h = AmgHierarchy(cases.ldu_to_csr(pat, s.diag, s.upper, s.lower), AmgSettings(strength_decay=0.5))
    assert h.level_sizes()[1:-1] and all(512 < n <= 768 for n in h.level_sizes()[1:-1]), h.level_sizes()
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
    its, x = solve(Precision.MIXED_FP32)
    monkeypatch.setenv("CFDG_DENSE_TAIL", "0")
    its_off, x_off = solve(Precision.MIXED_FP32)
    assert its == its_off and np.array_equal(x, x_off)
    # |x - x64| <= |A^-1| (|r| + |r64|), and the solution is at least as smooth as the right-hand side:
    # 25 tolerances in the norm (six at most were measured)
    assert np.linalg.norm(x - x64) <= 25e-9 * np.linalg.norm(x64)
