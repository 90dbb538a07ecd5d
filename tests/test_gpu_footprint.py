"""The serving footprint bounds what a context holds, term by term: also
where no two preconditioner blocks share their index tables."""
import numpy as np
import pytest

from tdycore_amd import serving, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,width", [((40, 40, 20), 64), ((40, 40, 20), 256), ((31, 24, 17), 512)])
def test_footprint_of_blocks_of_any_shape(n, width):
    import torch
    from tdycore_amd.mpfao import MPFAO
    print(f"[case] footprint {n} width {width}", flush=True)
    P = workloads.ensemble_box_problem(*n, 5, 0.6)
    m = P["mesh"]
    # runs of consecutive cells, half to all of the width long
    cuts = np.cumsum(np.random.default_rng(0).integers(width // 2, width + 1, size=2 * m.nc // width + 2))
    part = np.searchsorted(cuts, np.arange(m.nc), side="right")
    g = MPFAO(m, P["face_bc"], P["K"], P["porosity"], P["Sr"], **P["kw"])
    g.set_pc_partition(part)
    U = torch.tensor(P["U0"], device="cuda", dtype=torch.float64)
    g.run_snes_steps(U, 3600.0, 1, g.solver_options(pc_block=width, pc_coarse=1))
    held = g.device_bytes()
    g.close()
    rows = len(np.unique(part)) * width
    bound = serving.footprint_bytes(m.nc, m.nf, m.nv, m.nbnd, rows, width=width)
    print(f"  held {held}, bound {bound}", flush=True)
    assert held <= bound - (3 << 20)  # without its constant
