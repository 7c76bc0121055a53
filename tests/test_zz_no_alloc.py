"""pmg_vanka_smooth_noalloc (no reference counterpart: the FP64 colored Vanka sweeps of
pmg_vanka_smooth for callers that cannot allocate, with their scratch in a file-scope
device array) against pmg_vanka_smooth, through the C ABI on device vectors.

pmg_vanka_smooth takes one launch per color and the other the residual and the local solve in two,
with the same arithmetic, so their results are compared bit for bit, on two calls in a row with the second on a smaller level (the array
keeps the first call's contents), with the global relaxation on (its copy of u lives in
the array too) and off; a level whose scratch exceeds the array is refused with
PMG_ERR_UNSUPPORTED, as is a mixed-precision context.
"""
import ctypes as C

import numpy as np
import pytest

from conftest import params

pytestmark = pytest.mark.gpu


def _smooth_both(mg, lvl, u0, f, sweeps):
    from to_merge_master_parmoon_amd.multigrid import DeviceVector
    n = mg.n_dof[lvl]
    ua, ub, fd = DeviceVector(mg, n, u0), DeviceVector(mg, n, u0), DeviceVector(mg, n, f)
    mg._check(mg._lib.pmg_vanka_smooth(mg._ctx, lvl, ua.ptr, fd.ptr, sweeps, 1), "vanka")
    mg._check(mg._lib.pmg_vanka_smooth_noalloc(mg._ctx, lvl, ub.ptr, fd.ptr, sweeps), "vanka noalloc")
    a, b = ua.download(), ub.download()
    for v in (ua, ub, fd):
        v.free()
    return a, b


@pytest.mark.parametrize("alpha", [1.0, 0.9])
def test_noalloc_smoother_matches_smoother(oseen16, alpha):
    from to_merge_master_parmoon_amd.multigrid import build_hierarchy
    mg = build_hierarchy(oseen16, params(sc_smooth_damp_factor_saddle=alpha, sc_smooth_damp_factor_coarse_saddle=0.8))
    for call, (lvl, sweeps) in enumerate([(2, 2), (1, 1)]):   # second call: the smaller level
        n = mg.n_dof[lvl]
        rng = np.random.default_rng(600 + call)
        u0, f = rng.standard_normal(n), rng.standard_normal(n)
        a, b = _smooth_both(mg, lvl, u0, f, sweeps)
        print(f"alpha {alpha} call {call} level {lvl}: max |diff| {np.max(np.abs(a - b)):.3e}", flush=True)
        assert not np.array_equal(a, u0)
        assert np.array_equal(a, b)
    mg.close()


def test_noalloc_refuses_oversized_and_mixed():
    from to_merge_master_parmoon_amd import problem
    from to_merge_master_parmoon_amd.multigrid import DeviceVector, build_hierarchy
    P = problem.oseen3d(32)
    # 32^3 with the relaxation copy: 4096 x 96 + 954947 doubles > 8 MiB
    mg = build_hierarchy(P, params(sc_smooth_damp_factor_saddle=0.9))
    n = mg.n_dof[3]
    u, f = DeviceVector(mg, n, np.zeros(n)), DeviceVector(mg, n, np.ones(n))
    st = mg._lib.pmg_vanka_smooth_noalloc(mg._ctx, 3, u.ptr, f.ptr, 1)
    assert st == 10, mg._lib.pmg_last_error_string(mg._ctx)
    assert b"static scratch" in mg._lib.pmg_last_error_string(mg._ctx)
    # without the relaxation the same level fits (4096 x 96 doubles)
    mg.set_params(sc_smooth_damp_factor_saddle=1.0)
    mg.setup()
    assert mg._lib.pmg_vanka_smooth_noalloc(mg._ctx, 3, u.ptr, f.ptr, 1) == 0
    u.free(); f.free()
    mg.close()
    mm = build_hierarchy(problem.oseen3d(8), params(precision=1))
    n = mm.n_dof[1]
    u, f = DeviceVector(mm, n, np.zeros(n)), DeviceVector(mm, n, np.ones(n))
    assert mm._lib.pmg_vanka_smooth_noalloc(mm._ctx, 1, u.ptr, f.ptr, 1) == 10
    u.free(); f.free()
    mm.close()


def test_noalloc_nodal_sweep_matches(oseen16):
    """Nodal Vanka (smoother 4) relaxes on every sweep: its copy of u is always taken from
    the array; two calls in a row, the second on the smaller level."""
    from to_merge_master_parmoon_amd.multigrid import build_hierarchy
    mg = build_hierarchy(oseen16, params(sc_smoother_saddle=4, sc_smooth_damp_factor_saddle=1.0))
    for call, lvl in enumerate([2, 1]):
        n = mg.n_dof[lvl]
        rng = np.random.default_rng(620 + call)
        u0, f = rng.standard_normal(n), rng.standard_normal(n)
        a, b = _smooth_both(mg, lvl, u0, f, 2)
        assert not np.array_equal(a, u0)
        assert np.array_equal(a, b)
    mg.close()
