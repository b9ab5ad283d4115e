"""The forms hx_update takes by size and setting, at the sizes where each can go wrong, against the oracle: the time
step from minima combined by one workgroup or by several, face fluxes folded into the Local at small row sizes with
the viscous jumps reconciled by a launch of their own, the folded update with the admissibility fix on (including a
stage 0 that needs a fix, on boxes and on trees), and the per-case time step over meshes of unequal cases. Bars are the
parity ones: relative L2 <= 1e-12, time steps to 1e-13, counts equal; a batch equals its cases alone bit for bit."""
import ctypes
import math

import numpy as np
import pytest

from hexed_amd import abi, configs
from hexed_amd.device import Context, Device_mesh

from helpers import freestream, init_faces, o_call, say, set_vertices, smooth_state, update_folds
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


# one minimum per 4 elements: one alone, a few, just below and at the 4096 that one workgroup combines, and above, where
# several workgroups do: a few minima more than one round of theirs, and more than two rounds
MINIMA = [1, 17, 127, 128, 129, 182]
CHEBY = 1 / (1 - math.cos(math.pi / 2))  # the Chebyshev step of a single stage (math.cpp:104-107)


@pytest.mark.parametrize("n", MINIMA)
def test_time_step_minima(ctx, n):
    say(f"[gpu] time step from the minima of {n}x{n} elements")
    host = build((2, 8, False, n), seed=n)
    dev = Device_mesh(ctx, host.copy())
    run_updates(host, dev, abi.update_options(max_safety=0.5), 3, fields=("state",))
    dev.close()


@pytest.mark.parametrize("n", [17, 129, 182])
def test_time_step_minima_limited_and_enqueued(ctx, n):
    """A maximum below Max_dt, and updates whose time step and status stay on the device (replays of a graph), another mesh's
    updates on the same context between them: as the synchronous ones, bit for bit."""
    say(f"[gpu] limited and enqueued time steps, {n}x{n} elements")
    host = build((2, 8, False, n), seed=n)
    sync, queued, other = (Device_mesh(ctx, host.copy()) for _ in range(3))
    free = abi.update_options(max_safety=0.5)
    st = sync.update(free)
    queued.update(free)
    limit = .25 * st.time_step
    limited = abi.update_options(max_safety=0.5, max_time_step=limit)
    flow = 0.
    for opts, start in ((limited, abi.hx_update_status()), (free, None)):
        queued.update_async(opts, 2, start)
        other.update(abi.update_options(max_safety=0.4))
        got = queued.status_sync()
        for _ in range(2):
            sync.update(opts, st)
            flow += st.time_step
        assert (st.time_step == limit * CHEBY) == (opts is limited)
        assert (got.time_step, got.flow_time) == (st.time_step, flow)
    assert got.iteration == 4
    a, b = (d.download("state", 0, out=np.zeros_like(host.state[0])) for d in (sync, queued))
    assert np.array_equal(a, b)
    for d in (sync, queued, other):
        d.close()


def test_local_time_step(ctx):
    """Local time stepping takes min(1, max_time_step) times the Chebyshev step, and no reduction."""
    say("[gpu] local time stepping")
    host = build((2, 8, False, 17), seed=17)
    dev = Device_mesh(ctx, host.copy())
    run_updates(host, dev, abi.update_options(max_safety=0.5, local_time=True), 3, fields=("state",))
    assert dev.update(abi.update_options(max_safety=0.5, local_time=True, max_time_step=.5)).time_step == .5 * CHEBY
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


def unstable_tree(nd, rs, base, levels, frac, seed):
    """Low pressure with large perturbations on a tree: a step of max_safety 2 leaves elements, their faces and fine
    faces of hanging faces inadmissible after stage 0."""
    m = configs.tree_mesh(base=base, rs=rs, levels=levels, frac=frac, seed=seed, nd=nd,
                          bc=(abi.HX_BC_FREESTREAM, freestream(nd)))
    m.av = [np.zeros((k, 2, m.nq)) for k in m.n_elem]
    smooth_state(m, amp=0.2, seed=seed)
    st = m.state[0]
    ke = 0.5 * (st[:, :nd] ** 2).sum(1) / st[:, nd]
    st[:, nd + 1] = ke + (st[:, nd + 1] - ke) * 0.05
    init_faces(m)
    set_vertices(m)
    return m


@pytest.mark.parametrize("fold", [-1, 0, 1])
@pytest.mark.parametrize("case", [(2, 3, 3, 2, .4, 1), (2, 4, 3, 2, .4, 1), (3, 4, 2, 1, .5, 2), (3, 6, 2, 1, .4, 2)],
                         ids=lambda c: "nd%d_rs%d" % c[:2])
def test_fix_after_stage_on_tree(ctx, case, fold):
    """The fix fires inside updates on meshes with hanging faces (after stage 0 in each case's first update)."""
    say(f"[gpu] fix inside an update on a tree {case} fold {fold}")
    host = unstable_tree(*case)
    dev = Device_mesh(ctx, host.copy())
    dev.set_face_fold(fold)
    st = run_updates(host, dev, abi.update_options(max_safety=2., fix_admis=True), 3, fields=("state", "faces", "av"))
    assert st.fix_admis_iters >= 9 and dev.is_admissible() and is_admissible(host)[0]
    dev.close()


@pytest.mark.parametrize("fold", [-1, 0])
def test_fix_of_fine_faces_alone(ctx, fold):
    """A stage 0 that leaves fine faces of a hanging face inadmissible and everything else admissible: energy dips
    between the nodes of a coarse element whose velocity carries it below zero there."""
    say(f"[gpu] fix of fine faces alone fold {fold}")
    nd, rs = 2, 6
    host = configs.tree_mesh(base=2, rs=rs, levels=1, frac=.4, seed=0, nd=nd,
                             bc=(abi.HX_BC_FREESTREAM, freestream(nd, mach=.1)))
    host.av = [np.zeros((k, 2, host.nq)) for k in host.n_elem]
    smooth_state(host, mach=.1, amp=.02, seed=0)
    e, f = (int(x[0]) for x in np.where(host.face_slot[0] == host.ref_slot[0, 0]))
    st = host.state[0][e]
    prof = np.where(np.arange(rs) < 2, .18, 1.)
    st[nd + 1] *= (prof[:, None] if f // 2 == 1 else prof[None, :]).repeat(rs, 1 if f // 2 == 1 else 0).ravel()
    st[:nd] = .8 * np.random.default_rng(63).uniform(-1, 1, (nd, host.nq)) * np.sqrt(2 * st[nd] * st[nd + 1]) / nd
    init_faces(host)
    set_vertices(host)
    # the oracle's stage 0 alone: which of the arrays the check reads it leaves inadmissible
    alone = host.copy()
    s, ko, dt = alone.struct(), abi.hx_kernel_options(0., 0, 0, 0), ctypes.c_double()
    o_call("oracle_max_dt_euler", ctypes.byref(s), ctypes.byref(ko), .8, .8, 0, ctypes.byref(dt))
    ko.dt = dt.value
    o_call("oracle_apply_state_bcs", ctypes.byref(s))
    o_call("oracle_compute_euler", ctypes.byref(s), ctypes.byref(ko))
    faces = alone.faces[:, nd * host.nfq:(nd + 2) * host.nfq]
    fine = alone.ref_slot[:, 1:]
    assert (alone.state[0][:, nd:] > 0).all() and (faces[np.unique(alone.face_slot[0])] > 0).all()
    assert (faces[fine[fine >= 0]] < 0).any()
    dev = Device_mesh(ctx, host.copy())
    dev.set_face_fold(fold)
    st = run_updates(host, dev, abi.update_options(max_safety=.8, fix_admis=True), 2, fields=("state", "faces", "av"))
    assert st.fix_admis_iters == 1
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
