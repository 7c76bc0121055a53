"""Coarse systems whose velocity block cannot be inverted by itself, in the range where the block
form took the place of the dense LU (513 to 1024 velocity unknowns per component): one velocity
dof without (or almost without) coupling to any other, held by the pressure alone, so that the
whole system is regular.  The mixed forms then factor the whole system as the FP64 form does, with
the same kernels: solve_exact within 1e-13 of it, alone and, by the iterations and the solution of
FGMRES (the tolerance of the solve, 1e-10, times 100), in a batch beside an ordinary problem."""
import numpy as np
import pytest

from conftest import params, rel

pytestmark = pytest.mark.gpu


def _problem(scale, faces=63, box=(5, 5, 5)):
    from to_merge_master_parmoon_amd import _abi, problem
    prob = problem.Problem(cx=box[0], cy=box[1], cz=box[2], n_levels=2, nu=0.05, conv_kind=_abi.CONV_FOURIER,
                           rhs_kind=_abi.RHS_FOURIER, dirichlet_faces=faces, perturb=0.1)
    if scale is not None:
        a = prob.arrays(0)
        rp, kc = a["a_rowptr"], a["a_kcol"]
        row = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
        r = prob.descs[0].n_active // 2
        for v in a["a"]:
            v[(row == r) | (kc == r)] *= scale
    return prob


@pytest.mark.parametrize("faces", [63, 21])
@pytest.mark.parametrize("scale", [0.0, 1e-14])
@pytest.mark.parametrize("precision", [1, 2])
def test_whole_system_factored(faces, scale, precision):
    from to_merge_master_parmoon_amd.multigrid import build_hierarchy
    prob = _problem(scale, faces)
    assert 512 < prob.descs[0].n_active <= 1024
    prm = dict(internal_project_pressure=int(faces == 63))
    f = np.random.default_rng(560).standard_normal(prob.n_dof(0))
    out = []
    for p in (0, precision):
        mg = build_hierarchy(prob, params(precision=p, **prm))
        assert mg.shared_block(0)
        if p:
            mg.refactor()   # set up again before the first solve
            mg.synchronize()
        out.append(mg.solve_exact(f))
        mg.refactor()
        out.append(mg.solve_exact(f))
        mg.close()
    assert rel(out[2], out[0]) <= 1e-13 and rel(out[3], out[0]) <= 1e-13


def test_batch_beside_an_ordinary_problem():
    from to_merge_master_parmoon_amd.multigrid import NSEBatch, build_hierarchy
    probs = [_problem(None), _problem(0.0), _problem(None, box=(3, 3, 3))]
    kw = dict(precision=2, sc_gmres_restart=30, sc_lin_red_factor_saddle=1e-10, sc_lin_res_norm_min_saddle=0.0,
              sc_lin_maxit_saddle=100)
    batch = NSEBatch(probs, params(**kw))
    batch.setup()
    rhs = [p.rhs(-1).copy() for p in probs]
    sols = [np.zeros_like(r) for r in rhs]
    its, _, st = batch.fgmres(sols, rhs)
    batch.close()
    assert st == [0, 0, 0]
    for p, r, x, it in zip(probs, rhs, sols, its):
        mg = build_hierarchy(p, params(**kw))
        y = np.zeros_like(r)
        it1, _, st1 = mg.fgmres(y, r)
        mg.close()
        assert st1 == 0 and abs(it - it1) <= 1
        n = p.descs[-1].n_udof
        for v in (x, y):
            v[3 * n::4] -= v[3 * n::4].mean()
        assert rel(x, y) <= 1e-8
