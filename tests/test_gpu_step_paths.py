"""The forms hx_update takes by size and setting, at the sizes where each can go wrong, against the oracle: the time
step from minima combined by one workgroup or by several, face fluxes folded into the Local at small row sizes with
the viscous jumps reconciled by a launch of their own, the folded update with the admissibility fix on (including a
stage 0 that needs a fix), and the per-case time step over meshes of unequal cases. Bars are the parity ones: relative
L2 <= 1e-12, time steps to 1e-13, counts equal; a batch equals its cases alone bit for bit."""
import ctypes

import numpy as np
import pytest

from hexed_amd import abi, configs
from hexed_amd.device import Context, Device_mesh

from helpers import o_call, say, update_folds
from test_admissibility import UNSTABLE, is_admissible, unstable_case
from test_gpu_batch import run_batch_vs_single
from test_gpu_parity import build, compare_mesh, ids

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def run_updates(host, dev, opts, steps, fields=("state", "faces"), ldg=True):
    s = host.struct()
    st_o, st_d = abi.hx_update_status(), abi.hx_update_status()
    for it in range(steps):
        o_call("oracle_update", ctypes.byref(s), ctypes.byref(opts), ctypes.byref(st_o))
        dev.update(opts, st_d)
        assert abs(st_d.time_step - st_o.time_step) <= 1e-13 * st_o.time_step
        assert (st_d.iteration, st_d.fix_admis_iters) == (st_o.iteration, st_o.fix_admis_iters)
        compare_mesh(f"update {it}", host, dev, fields=fields, ldg=ldg)
    return st_o


# one minimum per 4 elements: one alone, a few, and just below, at and just above the 4096 that one workgroup combines
@pytest.mark.parametrize("local", [False, True], ids=["global", "local"])
@pytest.mark.parametrize("n", [1, 17, 127, 128, 129])
def test_time_step_minima(ctx, n, local):
    say(f"[gpu] time step from the minima of {n}x{n} elements, local time {local}")
    host = build((2, 8, False, n), seed=n)
    dev = Device_mesh(ctx, host.copy())
    run_updates(host, dev, abi.update_options(max_safety=0.5, local_time=local), 3, fields=("state",))
    dev.close()


# (n_dim, row_size, deformed, elements per axis): element counts that leave the last tile part full
FOLD = [(1, 2, False, 7), (1, 3, True, 5), (2, 2, False, 9), (2, 2, True, 5), (2, 3, True, 7), (3, 2, True, 3),
        (3, 3, False, 5), (3, 3, True, 3), (3, 4, False, 3), (3, 5, True, 3)]


@pytest.mark.parametrize("cfg", FOLD, ids=ids)
@pytest.mark.parametrize("ns", [False, True], ids=["euler", "ns"])
def test_default_folding(ctx, cfg, ns):
    say(f"[gpu] default folding {'ns' if ns else 'euler'} {ids(cfg)}")
    host = build(cfg, with_av=ns, seed=cfg[1])
    dev = Device_mesh(ctx, host.copy())
    kw = dict(visc=abi.constant(2e-3), cond=abi.constant(3e-3)) if ns else {}
    run_updates(host, dev, abi.update_options(max_safety=0.3, **kw), 2, ldg=not (ns and update_folds(host)))
    dev.close()


@pytest.mark.parametrize("fold", [-1, 0, 1])
@pytest.mark.parametrize("case", UNSTABLE, ids=lambda c: "nd%d_rs%d_safety%g" % (c[0], c[1], c[4]))
def test_fix_after_folded_stage(ctx, case, fold):
    """Unstable steps with the fix on: the face states, the ones a fix between the stages works on included."""
    nd, rs, n, mach, safety, pfac = case
    say(f"[gpu] fix after a folded stage {case} fold {fold}")
    host = unstable_case(nd, rs, n, mach, pfac)
    dev = Device_mesh(ctx, host.copy())
    dev.set_face_fold(fold)
    st = run_updates(host, dev, abi.update_options(max_safety=safety, fix_admis=True), 4)
    assert st.fix_admis_iters > 0 and dev.is_admissible() and is_admissible(host)[0]
    dev.close()


@pytest.mark.parametrize("cfg", [(2, 4, False, 6), (3, 3, True, 3), (3, 6, True, 2)], ids=ids)
def test_navier_stokes_with_fix_on(ctx, cfg):
    say(f"[gpu] navier-stokes with the fix on {ids(cfg)}")
    host = build(cfg, with_av=True, seed=5)
    dev = Device_mesh(ctx, host.copy())
    opts = abi.update_options(max_safety=0.3, visc=abi.constant(2e-3), cond=abi.constant(3e-3), fix_admis=True)
    run_updates(host, dev, opts, 2, ldg=not update_folds(host))
    dev.close()


# elements per axis of each case: one alone, equal, unequal, one several workgroups reduce beside one of one element
@pytest.mark.parametrize("sizes", [[3], [2, 2, 2], [1, 7, 2, 1], [6, 1], [1] * 17], ids=str)
def test_case_time_steps(ctx, sizes):
    say(f"[gpu] per-case time steps {sizes}")
    cases = [configs.euler_box(n, 6, mach=0.3 + 0.02 * k, seed=k, deformed=k % 2 == 1, jitter=0.1 * (k % 2))
             for k, n in enumerate(sizes)]
    run_batch_vs_single(ctx, cases, abi.update_options(max_safety=0.5), abi.HX_FP64)
