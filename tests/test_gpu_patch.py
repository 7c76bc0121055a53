"""One launch per color (csrc/k_patch.hip): FP64, FP32 and BF16 sweeps against the oracle's FP64 sweep
where the launch can go wrong: boxes one coarse cell wide, colors of 1 to 4 cells, dofs with
one update, colors of 512 cells and more, whose patches go to the XCDs in eighths, with 3 cells
moved to a color of their own so that the eighths differ, and rows longer than a hexahedral
grid's: edge rows of 105 entries take the general record shape, vertex rows of more than 128
the two-launch form.  Levels of up to 2048 patches a color store the full inverse, larger ones
the block form.  Bounds: FP64 1e-13 (the sums of a residual in another order), FP32 rounding
of the local inverses 2e-5, and BF16's 2e-2."""
import ctypes as C
import functools

import numpy as np
import pytest

from conftest import params, rel

pytestmark = pytest.mark.gpu


def _longer_rows(prob, level, extra, rng, below=1 << 30):
    """The level with extra = (edge, vertex) more entries in the active rows of edge and vertex
    dofs (numbers below `below`), at other dofs of several cells: an edge row's in the halos of all
    its cells, so that no patch reads more dofs than before, a vertex row's in the two rings around it
    (small values, the same in A11 .. A33)."""
    from to_merge_master_parmoon_amd import _abi
    d, a = prob.descs[level], prob.arrays(level)
    rp, kc = a["a_rowptr"], a["a_kcol"]
    shared = np.bincount(a["u_global"].reshape(-1), minlength=d.n_udof) > 1
    cells = np.split(np.argsort(a["u_global"].reshape(-1), kind="stable") // 27,
                     np.cumsum(np.bincount(a["u_global"].reshape(-1), minlength=d.n_udof))[:-1])
    ug, halo = a["u_global"].reshape(-1, 27), {}

    def common_halo(r):
        for c in cells[r]:
            if c not in halo:
                halo[c] = np.unique(np.concatenate([kc[rp[q]:rp[q + 1]] for q in ug[c]]))
        return functools.reduce(np.intersect1d, [halo[c] for c in cells[r]])

    rows, vals = [], []
    for r in range(d.n_udof):
        cols, v = kc[rp[r]:rp[r + 1]], a["a"][0][rp[r]:rp[r + 1]]
        if r < min(d.n_active, below) and len(cols) >= 75:
            ring = common_halo(r) if len(cols) == 75 else \
                np.unique(np.concatenate([kc[rp[c]:rp[c + 1]] for c in cols if shared[c]]))
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
    mg.set_profiling(True)
    y = mg.cell_vanka(1, u.copy(), f, 2)
    # one launch per color, or (vertex rows of more than 128 entries) two
    assert (mg.timers()["vanka_solve"]["calls"] > 0) == (extra is not None and 125 + extra[1] > 128)
    mg.close()
    assert rel(y, x) <= bound


def _split_color(prob, desc):
    """The level with 3 cells of its first color in a color of their own; the color sizes."""
    from to_merge_master_parmoon_amd import _abi
    from to_merge_master_parmoon_amd.multigrid import color_cells
    n, ptr, order = color_cells(desc.n_cells, prob.arrays(prob.n_levels - 1)["u_global"], desc.n_udof)
    order = np.concatenate([order[3:], order[:3]]).astype(np.int32)
    ptr = np.concatenate([[0], ptr[1:] - 3, [desc.n_cells]]).astype(np.int32)
    out = _abi.PmgLevelDesc()
    C.memmove(C.byref(out), C.byref(desc), C.sizeof(desc))
    out.n_colors, out.ptr_colors = n + 1, ptr.ctypes.data_as(_abi.c_int_p)
    out.cell_reorder = order.ctypes.data_as(_abi.c_int_p)
    return out, (ptr, order), np.diff(ptr)


# 16 x 16 x 20 cells (640 a color, full inverse); 24 x 32 x 24 (2304, block form) with the grid's
# record shape and the general one
@pytest.mark.parametrize("box,levels,extra,precisions", [((4, 4, 5), 3, None, (0, 1, 2)),
                                                         ((3, 4, 3), 4, None, (1, 2)),
                                                         ((3, 4, 3), 4, (30, 3), (1, 2))])
def test_large_colors_match_oracle(box, levels, extra, precisions):
    import pmg_oracle
    from to_merge_master_parmoon_amd import _abi, problem
    from to_merge_master_parmoon_amd.multigrid import NSEMultiGrid
    prob = problem.Problem(cx=box[0], cy=box[1], cz=box[2], n_levels=levels, nu=0.1, conv_kind=_abi.CONV_FOURIER,
                           rhs_kind=_abi.RHS_FOURIER, dirichlet_faces=63, perturb=0.1)
    descs, top, keep = list(prob.descs), levels - 1, None
    rng = np.random.default_rng(12)
    if extra:
        descs[top], keep, lengths = _longer_rows(prob, top, extra, rng, below=4000)
        assert 75 + extra[0] in lengths and lengths[-1] <= 128
    descs[top], keep_colors, sizes = _split_color(prob, descs[top])
    assert sizes[0] % 8 and sizes.max() >= 512 and (levels == 3 or sizes.max() > 2048)
    u = rng.standard_normal(prob.n_dof(top))
    f = rng.standard_normal(prob.n_dof(top))
    orc = pmg_oracle.Oracle(params(), descs, refactor=0)
    x = u.copy()
    assert orc.cell_vanka(top, x, f, 1) == 0
    orc.close()
    for precision in precisions:
        mg = NSEMultiGrid(params(precision=precision))
        for d in descs:
            mg.add_level(d)
        mg.setup()
        assert mg.shared_block(top)
        mg.set_profiling(True)
        y = mg.cell_vanka(top, u.copy(), f, 1)
        assert mg.timers()["vanka_solve"]["calls"] == 0   # one launch per color
        mg.close()
        assert rel(y, x) <= (1e-13, 2e-5, 2e-2)[precision]


@pytest.mark.parametrize("precision", [0, 2])
def test_large_color_of_a_compacted_batch(precision):
    """A batch whose smaller problem ends first goes on with lists of the other's patches, 512 a
    color: each problem's iterations and solution as alone (1e-10 of the solve times 100)."""
    from to_merge_master_parmoon_amd import problem
    from to_merge_master_parmoon_amd.multigrid import NSEBatch, build_hierarchy
    probs = [problem.oseen3d(16, nu=0.01), problem.oseen3d(8, nu=1.0)]
    batch = NSEBatch(probs, params(precision=precision))
    batch.setup()
    rhs = [p.rhs(-1).copy() for p in probs]
    sols = [np.zeros_like(r) for r in rhs]
    its, _, st = batch.fgmres(sols, rhs)
    batch.close()
    assert st == [0, 0] and its[1] < its[0]
    for p, r, x, it in zip(probs, rhs, sols, its):
        mg = build_hierarchy(p, params(precision=precision))
        y = np.zeros_like(r)
        it1, _, st1 = mg.fgmres(y, r)
        mg.close()
        n = 3 * p.descs[-1].n_udof
        for v in (x, y):
            v[n::4] -= v[n::4].mean()
        assert st1 == 0 and abs(it - it1) <= 1 and rel(x, y) <= 1e-8
