"""One launch per color (csrc/k_patch.hip): FP64, FP32 and BF16 sweeps against the oracle's FP64 sweep
where the launch can go wrong: boxes one coarse cell wide, colors of 1 to 4 cells, dofs with
one update, levels whose cells are no multiple of the XCDs', and rows longer than a hexahedral
grid's: edge rows of 105 entries take the general record shape, vertex rows of more than 128
the two-launch form.  Bounds: FP64 1e-13 (the sums of a residual in another order), FP32 rounding
of the local inverses 2e-5, and BF16's 2e-2."""
import ctypes as C

import numpy as np
import pytest

from conftest import params, rel

pytestmark = pytest.mark.gpu


def _longer_rows(prob, level, extra, rng):
    """The level with extra = (edge, vertex) more entries in the active rows of edge and vertex
    dofs, at other dofs of several cells in the two rings around them (small values, the same
    in A11 .. A33)."""
    from to_merge_master_parmoon_amd import _abi
    d, a = prob.descs[level], prob.arrays(level)
    rp, kc = a["a_rowptr"], a["a_kcol"]
    shared = np.bincount(a["u_global"].reshape(-1), minlength=d.n_udof) > 1
    rows, vals = [], []
    for r in range(d.n_udof):
        cols, v = kc[rp[r]:rp[r + 1]], a["a"][0][rp[r]:rp[r + 1]]
        if r < d.n_active and len(cols) >= 75:
            ring = np.unique(np.concatenate([kc[rp[c]:rp[c + 1]] for c in cols if shared[c]]))
            more = np.setdiff1d(ring[shared[ring]], cols)[:extra[len(cols) > 75]]
            w = 1e-3 * np.abs(v).max() * rng.standard_normal(len(more))
            cols, v = np.concatenate([cols, more]), np.concatenate([v, w])
            order = np.argsort(cols)
            cols, v = cols[order], v[order]
        rows.append(cols)
        vals.append(v)
    out = _abi.PmgLevelDesc()
    C.memmove(C.byref(out), C.byref(d), C.sizeof(d))
    ptr = np.concatenate([[0], np.cumsum([len(c) for c in rows])]).astype(np.int32)
    col, val, zero = np.concatenate(rows).astype(np.int32), np.concatenate(vals), np.zeros(ptr[-1])
    out.a_rowptr, out.a_kcol = ptr.ctypes.data_as(_abi.c_int_p), col.ctypes.data_as(_abi.c_int_p)
    out.a_nnz = int(ptr[-1])
    for b in range(9):
        out.a[b] = (val if b in (0, 4, 8) else zero).ctypes.data_as(_abi.c_double_p)
    return out, (ptr, col, val, zero), sorted(set(np.diff(ptr)))


@pytest.mark.parametrize("box,faces,extra", [((1, 1, 1), 1, None), ((1, 1, 3), 21, None), ((3, 2, 2), 63, None),
                                             ((5, 3, 1), 21, None), ((3, 3, 3), 63, (30, 3)), ((3, 3, 3), 21, (0, 3)),
                                             ((3, 3, 3), 63, (5, 40))])
@pytest.mark.parametrize("precision,bound", [(0, 1e-13), (1, 2e-5), (2, 2e-2)])
def test_color_step_matches_oracle(box, faces, extra, precision, bound):
    import pmg_oracle
    from to_merge_master_parmoon_amd import _abi, problem
    from to_merge_master_parmoon_amd.multigrid import NSEMultiGrid
    prob = problem.Problem(cx=box[0], cy=box[1], cz=box[2], n_levels=2, nu=0.1, conv_kind=_abi.CONV_FOURIER,
                           rhs_kind=_abi.RHS_FOURIER, dirichlet_faces=faces, perturb=0.1)
    descs, keep = list(prob.descs), None
    rng = np.random.default_rng(5)
    if extra:
        descs[1], keep, lengths = _longer_rows(prob, 1, extra, rng)
        assert lengths[-2:] == [75 + extra[0], 125 + extra[1]]
    prm = dict(internal_project_pressure=1 if faces == 63 else 0)
    u = rng.standard_normal(prob.n_dof(1))
    f = rng.standard_normal(prob.n_dof(1))
    orc = pmg_oracle.Oracle(params(**prm), descs, refactor=0)
    x = u.copy()
    assert orc.cell_vanka(1, x, f, 2) == 0
    orc.close()
    mg = NSEMultiGrid(params(precision=precision, **prm))
    for d in descs:
        mg.add_level(d)
    mg.setup()
    assert mg.shared_block(1)
    y = mg.cell_vanka(1, u.copy(), f, 2)
    mg.close()
    assert rel(y, x) <= bound
