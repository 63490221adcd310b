"""FP32 level-0 kernels with two rows a lane against one (CFDG_NO_PAIR_SWEEPS): mixed FP32 and BF16
solves, alone and in a batch, with the stencil and the per-slot column layouts, are bit-identical. The
prolongation pairs slices at every size (the small members leave a block's last pair incomplete or
empty); the post-sweep pairs the chunks of a row group, of which there are several above 262,144 rows.
"""
from __future__ import annotations

import numpy as np
import pytest

import cfd_amd
from cfd_amd import AmgHierarchy, AmgSettings, Method, Precision, SolveControl, cases

pytestmark = pytest.mark.gpu


def _system(shape, seed):
    mesh = cases.box_mesh(*shape, jitter=0.2, seed=seed)
    s = cases.pressure_system(mesh, rhs_seed=seed)
    pat = cases.csr_pattern(s.n, s.owner, s.neighbour)
    view = AmgHierarchy(cases.ldu_to_csr(pat, s.diag, s.upper, s.lower), AmgSettings(strength_decay=0.5)).view()
    return s, pat, view


def _build(s, pat, view):
    dev = cfd_amd.DeviceSolver(pat)
    dev.assemble(s.diag, s.upper, s.lower)
    dev.set_amg(view)
    dev.set_rhs(s.source)
    return dev


SHAPES = [(20, 20, 20), (9, 13, 40), (17, 11, 23)]  # 125, 74 and 68 slices of 64 rows


@pytest.mark.parametrize("stencil", [True, False])
@pytest.mark.parametrize("prec", [Precision.MIXED_FP32, Precision.MIXED_BF16])
def test_pair_sweeps_bitwise_alone_and_batched(monkeypatch, stencil, prec):
    if stencil:
        monkeypatch.delenv("CFDG_NO_STENCIL", raising=False)
    else:
        monkeypatch.setenv("CFDG_NO_STENCIL", "1")
    systems = [_system(shape, 60 + i) for i, shape in enumerate(SHAPES)]
    results = {}
    for pair in (True, False):
        if pair:
            monkeypatch.delenv("CFDG_NO_PAIR_SWEEPS", raising=False)
        else:
            monkeypatch.setenv("CFDG_NO_PAIR_SWEEPS", "1")
        devs = [_build(*t) for t in systems]
        try:
            ctls = [SolveControl(1e-9 * np.linalg.norm(t[0].source), 300) for t in systems]
            alone = []
            for d, c in zip(devs, ctls):
                d.set_x(None)
                st = d.solve_resident(Method.Cg, True, prec, c)
                assert st.converged
                alone.append((st.iterations, st.residual, d.get_x()))
            with cfd_amd.Batch(devs, Method.Cg, True, prec) as batch:
                for d in devs:
                    d.set_x(None)
                stats = batch.solve(ctls)
                batched = [(st.iterations, st.residual, d.get_x()) for st, d in zip(stats, devs)]
            results[pair] = (alone, batched)
        finally:
            for d in devs:
                d.close()
    for which in (0, 1):
        for a, b in zip(results[True][which], results[False][which]):
            assert a[0] == b[0] and a[1] == b[1]
            assert np.array_equal(a[2], b[2])


@pytest.mark.parametrize("lanes,csr", [(2, 0), (4, 1), (1, 1)])
def test_pair_prolongation_with_other_transfer_layouts(monkeypatch, lanes, csr):
    """P_0 laid out with several lanes per row or as CSR (forced by a layout rule) takes the
    paired prolongation's general path; solves stay bit-identical to the one-slice kernels."""
    import json
    from pathlib import Path

    from cfd_amd import autotune

    rule = {"min_rows": 1000, "max_rows": 20000, "min_mean": 3.0, "max_mean": 6.0, "lanes": lanes, "csr": csr}
    autotune.apply({"layout_rules": [rule]})
    try:
        systems = [_system(shape, 70 + i) for i, shape in enumerate(SHAPES[1:])]
        results = {}
        for pair in (True, False):
            if pair:
                monkeypatch.delenv("CFDG_NO_PAIR_SWEEPS", raising=False)
            else:
                monkeypatch.setenv("CFDG_NO_PAIR_SWEEPS", "1")
            devs = [_build(*t) for t in systems]
            try:
                ctls = [SolveControl(1e-9 * np.linalg.norm(t[0].source), 300) for t in systems]
                out = []
                for d, c in zip(devs, ctls):
                    d.set_x(None)
                    st = d.solve_resident(Method.Cg, True, Precision.MIXED_FP32, c)
                    assert st.converged
                    out.append((st.iterations, d.get_x()))
                with cfd_amd.Batch(devs, Method.Cg, True, Precision.MIXED_FP32) as batch:
                    for d in devs:
                        d.set_x(None)
                    stats = batch.solve(ctls)
                    out += [(st.iterations, d.get_x()) for st, d in zip(stats, devs)]
                results[pair] = out
            finally:
                for d in devs:
                    d.close()
        for a, b in zip(results[True], results[False]):
            assert a[0] == b[0]
            assert np.array_equal(a[1], b[1])
    finally:
        path = Path(cfd_amd.__file__).resolve().parent / "tuning.json"
        autotune.apply(json.loads(path.read_text()) if path.exists() else {"layout_rules": []})


# Two chunks a row group, three, and two with column offsets that need 32 bits; the last slice and the
# last chunk are incomplete.
LARGE = [(67, 65, 63), (83, 81, 79), (190, 190, 8)]
LAYOUTS = {"symmetric": (), "stencil": ("CFDG_NO_SYM",), "explicit": ("CFDG_NO_SYM", "CFDG_NO_STENCIL")}


@pytest.fixture(scope="module")
def large_systems():
    out = []
    for i, shape in enumerate(LARGE):
        s = cases.pressure_system(cases.box_mesh(*shape, jitter=0.2, seed=80 + i), rhs_seed=80 + i)
        pat = cases.csr_pattern(s.n, s.owner, s.neighbour)
        a = cases.ldu_to_csr(pat, s.diag, s.upper, s.lower)
        out.append((s, pat, AmgHierarchy(a, AmgSettings(strength_decay=0.5), device=True).view()))
    return out


def _results(systems, runs):
    devs = [_build(*t) for t in systems]
    try:
        ctls = [SolveControl(1e-8 * np.linalg.norm(t[0].source), 20) for t in systems]
        out = {}
        for run in runs:
            res = []
            for d, c in zip(devs, ctls):
                d.set_x(None)
                st = d.solve_resident(*run, c)
                res.append((st.iterations, st.residual, st.true_residual, d.get_x()))
            with cfd_amd.Batch(devs, *run) as batch:
                batch.zero_x()
                for d, st in zip(devs, batch.solve(ctls)):
                    res.append((st.iterations, st.residual, st.true_residual, d.get_x()))
            out[run] = res
        return out
    finally:
        for d in devs:
            d.close()


def _same(a, b):
    for run in a:
        for x, y in zip(a[run], b[run]):
            assert x[:3] == y[:3] and np.array_equal(x[3], y[3]), run


def test_pairs_of_chunks(monkeypatch, large_systems):
    """Groups of two and three chunks: one row a lane and two give the same bits in every layout, and the
    layouts of one matrix give the same bits as each other (BF16 rows have one layout)."""
    cycles = [(Method.Cg, True, Precision.MIXED_FP32), (Method.Cg, True, Precision.MIXED_BF16)]
    krylov = [(Method.Cg, True, Precision.FP64), (Method.Cg, False, Precision.FP64), (Method.BiCgStab, False, Precision.FP64)]
    first = None
    for layout, switches in LAYOUTS.items():
        with monkeypatch.context() as env:
            for name in switches:
                env.setenv(name, "1")
            here = _results(large_systems, cycles + krylov)
            env.setenv("CFDG_NO_PAIR_SWEEPS", "1")
            _same(_results(large_systems, cycles), here)
        first = first or here
        _same(here, first)
