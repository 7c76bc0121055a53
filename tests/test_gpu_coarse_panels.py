"""The block-form coarse solve with a velocity block of more than 512 unknowns (panel LU and
substitution with the factors read from memory), at the edges of its range: 512 unknowns
(still the one-workgroup LU), 567 and 640, 729 and 1000 (the 5^3 grids), 1008 with 504 pressures.
Against the FP64 form's LU of the whole reduced system, which matches the oracle's
dgetrf/dgetrs; both solve the same system in FP64, 1e-10 as for the smaller blocks.  Twice, the second
time with other values in the same buffers."""
import numpy as np
import pytest

from conftest import params, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box,faces,m", [((4, 4, 4), 21, 512), ((4, 5, 5), 63, 567), ((4, 4, 5), 21, 640),
                                         ((5, 5, 5), 63, 729), ((5, 5, 5), 21, 1000), ((6, 3, 7), 21, 1008)])
def test_panel_block_coarse_solve(box, faces, m):
    from to_merge_master_parmoon_amd import _abi, problem
    from to_merge_master_parmoon_amd.multigrid import build_hierarchy
    prob = problem.Problem(cx=box[0], cy=box[1], cz=box[2], n_levels=2, nu=0.05, conv_kind=_abi.CONV_FOURIER,
                           rhs_kind=_abi.RHS_FOURIER, dirichlet_faces=faces, perturb=0.1)
    assert prob.descs[0].n_active == m
    prm = dict(internal_project_pressure=1 if faces == 63 else 0)
    out = []
    f = np.random.default_rng(530).standard_normal(prob.n_dof(0))
    for precision in (0, 1, 2):
        mg = build_hierarchy(prob, params(precision=precision, **prm))
        out.append(mg.solve_exact(f))
        # a second operator in the same buffers, the reference's LU again beside the block form
        keep = [v.copy() for v in prob.arrays(0)["a"]]
        for v in prob.arrays(0)["a"]:
            v *= 1.25
        mg.update_values(0, prob.descs[0])
        mg.refactor()
        out[-1] = np.concatenate([out[-1], mg.solve_exact(f)])
        for v, k in zip(prob.arrays(0)["a"], keep):
            v[:] = k
        mg.close()
    n = len(f)
    for x in out[1:]:
        assert rel(x[:n], out[0][:n]) <= 1e-10 and rel(x[n:], out[0][n:]) <= 1e-10
    assert rel(out[0][n:], out[0][:n]) > 1e-3
