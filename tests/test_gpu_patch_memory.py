"""What the one-launch color step and the interleaved operator input keep on the device, and when.

A level whose form cannot take them holds neither (FP64 with nine velocity blocks or shared_block
off, refinement steps; the copy below 150,000 velocity dofs), and a level that turns to a form
that can gets its records at the next set-up: then no separate local solve is launched any more
and the results are those of a context that had the form from the start, bit for bit."""
import numpy as np
import pytest

from conftest import params

pytestmark = pytest.mark.gpu


def _free():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _used(prob, **kw):
    from to_merge_master_parmoon_amd.multigrid import build_hierarchy
    before = _free()
    mg = build_hierarchy(prob, params(**kw))
    used = before - _free()
    mg.close()
    return used


def _local_solves(mg, u, f):
    """the sweep's result and its launches of a local solve of its own"""
    mg.set_profiling(True)
    mg.reset_timers()
    y = mg.cell_vanka(mg.n_levels - 1, u.copy(), f, 2)
    calls = mg.timers()["vanka_solve"]["calls"]
    mg.set_profiling(False)
    return y, calls


@pytest.mark.parametrize("with_step,without", [(dict(precision=0), dict(precision=0, shared_block=0)),
                                               (dict(precision=2), dict(precision=2, bf16_refine_steps=1))])
def test_no_records_where_no_launch_reads_them(oseen16, with_step, without):
    # the first launch of a kernel can allocate memory that stays (its scratch)
    _used(oseen16, **with_step)
    _used(oseen16, **without)
    # 4096 + 512 cells of at least 2 KB, less what one context allocates more than another in units
    # of 2 MB; the refinement steps store 85 x 85 floats per cell (padded to 7232)
    records = 2048 * (4096 + 512)
    kref = 4 * 7232 * (4096 + 512) if "bf16_refine_steps" in without else 0
    assert _used(oseen16, **without) - kref <= _used(oseen16, **with_step) - records // 2


def test_no_copy_below_its_size():
    from to_merge_master_parmoon_amd import problem
    from to_merge_master_parmoon_amd.multigrid import DeviceVector, NSEMultiGrid
    prob = problem.oseen3d(24, 3)
    assert 50_000 < prob.descs[-1].n_udof < 150_000
    mg = NSEMultiGrid(params(precision=0))
    for d in prob.descs:
        mg.add_level(d)
    n, lvl = mg.n_dof[-1], mg.n_levels - 1
    x, y = DeviceVector(mg, n, np.ones(n)), DeviceVector(mg, n)
    before = _free()
    assert mg._lib.pmg_matvec(mg._ctx, lvl, x.ptr, y.ptr, 1) == 0
    assert _free() == before
    mg.close()


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_records_come_with_the_form(precision):
    from to_merge_master_parmoon_amd import problem
    from to_merge_master_parmoon_amd.multigrid import build_hierarchy
    prob = problem.oseen3d(8)
    rng = np.random.default_rng(41)
    n = prob.n_dof(prob.n_levels - 1)
    u, f = rng.standard_normal(n), rng.standard_normal(n)
    mg = build_hierarchy(prob, params(precision=precision))
    want, calls = _local_solves(mg, u, f)
    z = mg.cycle(f)
    mg.close()
    assert calls == 0
    if precision == 0:   # nine blocks first, the shared one with new values
        keep = [[b.copy() for b in prob.arrays(lvl)["a"]] for lvl in range(prob.n_levels)]
        for lvl in range(prob.n_levels):
            ne = int(prob.arrays(lvl)["a_rowptr"][prob.descs[lvl].n_active])
            prob.arrays(lvl)["a"][4][:ne] *= 1.1
        mg = build_hierarchy(prob, params(precision=0))
    else:
        mg = build_hierarchy(prob, params(precision=precision, bf16_refine_steps=1))
    assert _local_solves(mg, u, f)[1] > 0
    mg.cycle(f)
    mg.cycle(f)   # (a captured cycle holds the two launches)
    if precision == 0:
        for lvl in range(prob.n_levels):
            for b, v in enumerate(keep[lvl]):
                prob.arrays(lvl)["a"][b][:] = v
            mg.update_values(lvl, prob.descs[lvl])
    else:
        mg.set_params(bf16_refine_steps=0)
    mg.refactor()
    got, calls = _local_solves(mg, u, f)
    assert calls == 0 and np.array_equal(got, want)
    for _ in range(3):
        assert np.array_equal(mg.cycle(f), z)
    mg.close()
