"""New values that change the form of the velocity rows: with the shared block only one of the nine
row-blocked copies is refreshed, so a level that turns to nine blocks has to bring the others up to
date, and a level that turns back reads none of them.  Defect, sweep and V-cycle against the oracle
after each change; FP64 1e-13 (V-cycle 1e-12), FP32 patch data 2e-5 as for one sweep elsewhere."""
import numpy as np
import pytest

from conftest import params, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,bound", [(0, 1e-13), (1, 2e-5)])
def test_form_changes_with_new_values(precision, bound):
    import pmg_oracle
    from to_merge_master_parmoon_amd import problem
    from to_merge_master_parmoon_amd.multigrid import build_hierarchy
    prob = problem.oseen3d(8)
    mg = build_hierarchy(prob, params(precision=precision))
    keep = [[b.copy() for b in prob.arrays(lvl)["a"]] for lvl in range(prob.n_levels)]
    rng = np.random.default_rng(31)
    for coupled in (False, True, False, True):
        for lvl in range(prob.n_levels):
            arr, d = prob.arrays(lvl), prob.descs[lvl]
            ne = int(arr["a_rowptr"][d.n_active])
            for b in range(9):
                arr["a"][b][:] = keep[lvl][b]
                if coupled:
                    w = 1.1 if b == 4 else 1.0 if b in (0, 8) else 0.03 * (1 if b in (1, 2, 5) else -1)
                    arr["a"][b][:ne] = w * keep[lvl][0][:ne]
            mg.update_values(lvl, d)
        mg.refactor()
        assert all(mg.shared_block(lvl) != coupled for lvl in range(prob.n_levels))
        orc = pmg_oracle.Oracle(params(), prob.descs, refactor=0)
        lvl = prob.n_levels - 1
        u, f = rng.standard_normal(prob.n_dof(lvl)), rng.standard_normal(prob.n_dof(lvl))
        assert rel(mg.matvec(lvl, u), orc.matvec(lvl, u)) <= 1e-13
        x = u.copy()
        assert orc.cell_vanka(lvl, x, f, 2) == 0
        assert rel(mg.cell_vanka(lvl, u.copy(), f, 2), x) <= bound
        z, st = orc.vcycle(f)
        assert st == 0 and rel(mg.cycle(f), z) <= max(10 * bound, 1e-12)
        orc.close()
    mg.close()
