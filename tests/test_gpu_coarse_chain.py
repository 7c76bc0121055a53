"""The triangular sweeps of the FP64 coarse solve (one workgroup per 64 unknowns, each value
published with the launch's generation) at the edges of a block: 6 unknowns, 448 = 7 blocks, 196
and 702 with 4 and 62 in the last one.  Against the oracle's SolveExact, 1e-10 as for the other
coarse solves; four right-hand sides in turn, so that no generation takes another's values."""
import numpy as np
import pytest

from conftest import params, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box,faces,n", [((1, 1, 1), 63, 6), ((2, 2, 1), 1, 196), ((4, 2, 2), 21, 448),
                                         ((3, 3, 2), 1, 702)])
def test_chain_at_block_edges(box, faces, n):
    import pmg_oracle
    from to_merge_master_parmoon_amd import _abi, problem
    from to_merge_master_parmoon_amd.multigrid import build_hierarchy
    prob = problem.Problem(cx=box[0], cy=box[1], cz=box[2], n_levels=2, nu=0.05, conv_kind=_abi.CONV_FOURIER,
                           rhs_kind=_abi.RHS_FOURIER, dirichlet_faces=faces, perturb=0.1)
    pin = faces == 63
    assert 3 * prob.descs[0].n_active + prob.descs[0].n_pdof - pin == n
    prm = dict(internal_project_pressure=int(pin))
    mg = build_hierarchy(prob, params(precision=0, **prm))
    orc = pmg_oracle.Oracle(params(**prm), prob.descs, refactor=0)
    for seed in range(4):
        f = np.random.default_rng(540 + seed).standard_normal(prob.n_dof(0))
        want, info = orc.solve_exact(f)
        assert info == 0
        assert rel(mg.solve_exact(f), want) <= 1e-10
    mg.close()
    orc.close()
