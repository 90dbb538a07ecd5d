"""What changes between two solves on one context and one state vector - Krylov
tolerances, the iteration limit, the source term - reaches the second solve,
which replays the graphs captured during the first: it gives what a context
of its own gives, bit for bit (every sum of the solver has a fixed order)."""
import numpy as np
import pytest

from cases import cfg0_problem

pytestmark = pytest.mark.gpu


def _context(P):
    from tdycore_amd.mpfao import MPFAO
    return MPFAO(P["mesh"], P["face_bc"], P["K"], P["porosity"], P["Sr"], **P["kw"])


def _solve(g, U, P, driver, opts, source=None):
    """One step from U0 in the buffer U: (state, iteration counts)."""
    import torch
    g.SetSourceSink(source)
    U.copy_(torch.tensor(P["U0"], device="cuda"))
    run = g.run_ts_be if driver == "ts" else g.run_snes_steps
    st = run(U, 3600.0, 1, opts)
    return U.cpu().numpy(), (st["newton_its"], st["linear_its"])


@pytest.mark.parametrize("driver,fp32,coarse", [("snes", 0, 0), ("snes", 1, 1), ("ts", 0, 1), ("ts", 1, 0)])
def test_tolerances_of_each_solve(driver, fp32, coarse):
    print(f"[case] tolerances driver={driver} fp32={fp32} coarse={coarse}", flush=True)
    import torch
    P = cfg0_problem(n=10)
    g = _context(P)
    U = torch.empty(P["mesh"].nc, dtype=torch.float64, device="cuda")
    counts = []
    for tol in (dict(ksp_rtol=1e-2), dict(ksp_rtol=1e-9), dict(ksp_rtol=1e-9, ksp_atol=1e-6), dict(ksp_rtol=1e-2)):
        kw = dict(snes_rtol=1e-8, pc_block=64, krylov_fp32=fp32, pc_coarse=coarse, ksp_restart=8, **tol)
        got, its = _solve(g, U, P, driver, g.solver_options(**kw))
        h = _context(P)
        ref, its_ref = _solve(h, torch.empty_like(U), P, driver, h.solver_options(**kw))
        h.close()
        assert its == its_ref, (tol, its, its_ref)
        assert np.array_equal(got, ref), tol
        counts.append(its[1])
    assert counts[1] > 1.5 * counts[0] and counts[3] == counts[0]
    g.close()


@pytest.mark.parametrize("fp32", [0, 1])
def test_iteration_limit_of_each_solve(fp32):
    """A limit below what the solve needs fails it, also after solves without one."""
    print(f"[case] iteration limit fp32={fp32}", flush=True)
    import torch
    from tdycore_amd import _lib
    P = cfg0_problem(n=10)
    g = _context(P)
    U = torch.empty(P["mesh"].nc, dtype=torch.float64, device="cuda")
    kw = dict(snes_rtol=1e-8, ksp_rtol=1e-9, pc_block=64, krylov_fp32=fp32, ksp_restart=8)
    first = _solve(g, U, P, "snes", g.solver_options(**kw))
    with pytest.raises(_lib.TdyHipError) as e:
        _solve(g, U, P, "snes", g.solver_options(ksp_max_it=3, **kw))
    assert e.value.code == _lib.ERR_NOCONV
    again = _solve(g, U, P, "snes", g.solver_options(**kw))
    assert first[1] == again[1] and np.array_equal(first[0], again[0])
    g.close()


@pytest.mark.parametrize("driver,fp32", [("snes", 0), ("ts", 1)])
def test_source_of_each_solve(driver, fp32):
    """A source set after a first solve, changed and cleared."""
    print(f"[case] source driver={driver} fp32={fp32}", flush=True)
    import torch
    P = cfg0_problem(n=8)
    g = _context(P)
    nc = P["mesh"].nc
    U = torch.empty(nc, dtype=torch.float64, device="cuda")
    o = g.solver_options(snes_rtol=1e-8, ksp_rtol=1e-8, pc_block=64, krylov_fp32=fp32, ksp_restart=8)
    # about 1e-5 of the largest cell's residual scale, rho phi V / dt
    q = 1e-5 * np.random.default_rng(3).random(nc) * (1.0 if driver == "ts" else float(P["mesh"].cell_vol.max()))
    states = []
    for src in (None, q, 2.0 * q, None):
        got, its = _solve(g, U, P, driver, o, src)
        h = _context(P)
        ref, its_ref = _solve(h, torch.empty_like(U), P, driver, o, src)
        h.close()
        assert its == its_ref and np.array_equal(got, ref)
        states.append(got)
    assert not np.array_equal(states[0], states[1]) and not np.array_equal(states[1], states[2])
    assert np.array_equal(states[0], states[3])
    g.close()


def test_tolerance_of_a_batch_after_a_solve():
    """The lockstep batch's solves follow their own options too."""
    print("[case] batch after a solve", flush=True)
    import torch
    from tdycore_amd.batch import FusedBatch
    P = cfg0_problem(n=10)

    def batch(g, U, opts):
        U.copy_(torch.tensor(P["U0"], device="cuda"))
        torch.cuda.synchronize()
        b = FusedBatch()
        b.add(g, U, opts, 3600.0, 1.0, 3600.0, 3600.0)
        done = []
        while len(b):
            done += b.round()
        b.close()
        torch.cuda.synchronize()
        return U.cpu().numpy(), done[0][1], done[0][2]["linear_its"]

    kw = dict(snes_rtol=1e-8, pc_block=64, ksp_restart=8)
    g, h = _context(P), _context(P)
    U = torch.empty(P["mesh"].nc, dtype=torch.float64, device="cuda")
    first = batch(g, U, g.solver_options(ksp_rtol=1e-2, **kw))
    got = batch(g, U, g.solver_options(ksp_rtol=1e-9, **kw))
    ref = batch(h, torch.empty_like(U), h.solver_options(ksp_rtol=1e-9, **kw))
    assert first[1] == got[1] == ref[1] == 0
    assert got[2] == ref[2] > first[2] and np.array_equal(got[0], ref[0])
    g.close()
    h.close()
