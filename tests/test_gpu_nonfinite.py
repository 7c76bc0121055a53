"""Values that overflow, and where they spread to.

The local and coarse solves in FP64 have the same finite and non-finite unknowns as the oracle's
dgetrs, which leaves an unknown that is finished alone: right-hand sides of about 1e306 let some
of the unknowns of a patch (of a block of 64 of the coarse system) overflow, after the pressures
and some velocities have come out finite.  In the FP32 color step an infinite velocity reaches the
rows that are coupled to it and no others: in a patch where it stands in one row, the product with
the stored inverse is infinite, not the NaN of two infinities or of zero times infinity."""
import numpy as np
import pytest

from conftest import params

pytestmark = pytest.mark.gpu


def _problem(box, faces, levels=2):
    from to_merge_master_parmoon_amd import _abi, problem
    return problem.Problem(cx=box[0], cy=box[1], cz=box[2], n_levels=levels, nu=0.1, conv_kind=_abi.CONV_FOURIER,
                           rhs_kind=_abi.RHS_FOURIER, dirichlet_faces=faces, perturb=0.1)


@pytest.mark.parametrize("noalloc", [False, True])
def test_finished_unknowns_of_a_patch_stay(noalloc):
    import ctypes as C
    import pmg_oracle
    from to_merge_master_parmoon_amd.multigrid import DeviceVector, build_hierarchy
    prob = _problem((1, 1, 1), 1)
    prm = dict(internal_project_pressure=0)
    f = 10.0 ** 306.5 * np.random.default_rng(7).standard_normal(prob.n_dof(1))
    orc = pmg_oracle.Oracle(params(**prm), prob.descs, refactor=0)
    x = np.zeros_like(f)
    assert orc.cell_vanka(1, x, f, 1) == 0
    orc.close()
    p = np.isfinite(x[3 * prob.descs[1].n_udof:])
    assert 0 < p.sum() < len(p)   # the first cell's pressures come out, later ones do not
    mg = build_hierarchy(prob, params(precision=0, **prm))
    if noalloc:   # residual and local solve in two launches
        du, df = DeviceVector(mg, len(f), np.zeros_like(f)), DeviceVector(mg, len(f), f)
        assert mg._lib.pmg_vanka_smooth_noalloc(mg._ctx, 1, du.ptr, df.ptr, 1) == 0
        y = du.download()
    else:
        y = mg.cell_vanka(1, np.zeros_like(f), f, 1)
    mg.close()
    assert np.array_equal(np.isfinite(y), np.isfinite(x))


@pytest.mark.parametrize("box,faces,e", [((1, 1, 1), 1, 306.5), ((1, 1, 3), 21, 306.5), ((3, 2, 2), 63, 307.0)])
def test_finished_unknowns_of_a_coarse_block_stay(box, faces, e):
    import pmg_oracle
    from to_merge_master_parmoon_amd.multigrid import build_hierarchy
    prob = _problem(box, faces)
    prm = dict(internal_project_pressure=int(faces == 63))
    f = 10.0 ** e * np.random.default_rng(8).standard_normal(prob.n_dof(0))
    orc = pmg_oracle.Oracle(params(**prm), prob.descs, refactor=0)
    x, info = orc.solve_exact(f)
    assert info == 0
    orc.close()
    # the unknowns of the reduced system (the oracle keeps the Dirichlet rows and the fixed pressure)
    n, na = prob.descs[0].n_udof, prob.descs[0].n_active
    free = np.concatenate([np.arange(na), n + np.arange(na), 2 * n + np.arange(na), np.arange(3 * n + (faces == 63), len(x))])
    assert 0 < np.isfinite(x[free]).sum() < len(free)
    mg = build_hierarchy(prob, params(precision=0, **prm))
    y = mg.solve_exact(f)
    mg.close()
    assert np.array_equal(np.isfinite(y[free]), np.isfinite(x[free]))


@pytest.mark.parametrize("precision", [1, 2])
def test_uncoupled_rows_stay(precision):
    from to_merge_master_parmoon_amd.multigrid import build_hierarchy, color_cells
    prob = _problem((4, 4, 4), 63)
    d, a = prob.descs[1], prob.arrays(1)
    rp, kc, bp, bc = a["a_rowptr"], a["a_kcol"], a["b_rowptr"], a["b_kcol"]
    ug, pg = a["u_global"].reshape(-1, 27), a["p_global"].reshape(-1, 4)
    _, ptr, order = color_cells(d.n_cells, a["u_global"], d.n_udof)
    # cells of the first color whose lowest dof stands in one row only, an active vertex row of
    # another number of entries than 16 k (the lanes past its end read no entry)
    cells = []
    for c in order[:ptr[1]]:
        rows = [kc[rp[r]:rp[r + 1]] for r in ug[c]]
        g = min(r.min() for r in rows)
        inside = [r for r, cols in zip(ug[c], rows) if g in cols]
        if g < d.n_active and len(inside) == 1 and inside[0] < d.n_active and (rp[inside[0] + 1] - rp[inside[0]]) % 16 \
                and not any(g in bc[bp[i]:bp[i + 1]] for i in pg[c]):
            cells.append((c, g))
    assert cells
    mg = build_hierarchy(prob, params(precision=precision))
    c, g = cells[0]
    u = np.zeros(mg.n_dof[1])
    u[g] = np.inf
    y = mg.cell_vanka(1, u, np.zeros_like(u), 1)
    mg.close()
    assert np.isinf(y[3 * d.n_udof + pg[c]]).all()
