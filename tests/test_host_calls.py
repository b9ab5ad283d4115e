"""The host code around the kernels on a HIP runtime without a device (tests/cpp/fake_hip.cpp): which calls an entry point
makes, in which order, and on an error. Each script runs in a process of its own, since the runtime is chosen when the
library is loaded; kernels do not run there, so no results are compared."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, sys
sys.path[:0] = [{root!r}, {here!r}]
fake = ctypes.CDLL({lib!r}, ctypes.RTLD_GLOBAL)
fake.fake_log.restype = ctypes.c_char_p
import numpy as np
from hexed_amd import abi, configs, mesh
from hexed_amd.device import Context, Device_group, Device_mesh
def calls():
    out = fake.fake_log().decode().splitlines()
    fake.fake_clear()
    return out
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("fake") / "libamdhip64.so.7")
    subprocess.run(["g++", "-O1", "-std=c++20", "-Wall", "-fPIC", "-shared", "-Wl,-soname,libamdhip64.so.7", "-o", lib,
                    os.path.join(HERE, "cpp", "fake_hip.cpp")], check=True)

    def script(text):
        code = PRELUDE.format(root=os.path.dirname(HERE), here=HERE, lib=lib) + text
        r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, f"status {r.returncode}\n{r.stdout}\n{r.stderr}"
    return script


def test_no_alloc_contexts_have_their_own_time_step(run):
    """The stage kernels of hx_update_no_alloc read the time step after the call has returned, so a second context of the
    GPU, on a stream of its own, must not form its time step in the same place."""
    run("""
seen = []
for c in [Context(0), Context(0)]:
    dev = Device_mesh(c, configs.euler_box(2, 4, seed=1))
    st = abi.hx_update_status()
    calls()
    dev.lib.hx_update_no_alloc(dev.ptr, ctypes.byref(abi.update_options()), ctypes.byref(st))
    at = {x for x in calls() if x.startswith("time step ")}
    assert len(at) == 1 and at != {"time step (nil)"}, at
    seen += at
assert seen[0] != seen[1], seen
""")


def test_no_alloc_minima_have_one_writer(run):
    """The minima in the array that all contexts of a GPU share: a context leaves none there while another one's work with
    the array is unfinished, and uses none that another has written since."""
    run("""
def minima(dev):
    calls()
    dev.lib.hx_update_no_alloc(dev.ptr, ctypes.byref(abi.update_options()), ctypes.byref(abi.hx_update_status()))
    log = calls()
    return [x for x in log if x.startswith("minima")], any("k_max_dt" in x for x in log)
a, b = Context(0), Context(0)
da, db = (Device_mesh(c, configs.euler_box(2, 4, seed=1)) for c in (a, b))
kept = minima(da)[0]
assert kept[0] == "minima (nil)" and kept[1] != "minima (nil)", kept
fake.fake_busy(1)  # a's stages are running
assert minima(db) == (["minima (nil)"] * 2, True)
fake.fake_busy(1)  # its own unfinished work is no obstacle
assert minima(da)[0] == kept
assert minima(db) == (kept, True)
fake.fake_busy(1)
assert minima(da) == (["minima (nil)"] * 2, True)
b.close()
assert minima(da) == (kept, True)
""")


def test_calc_jacobian_errors_wait_for_the_uploads(run):
    """The uploads of hx_calc_jacobian read the caller's arrays: whichever later call fails, it returns only after the
    stream has passed them."""
    run("""
m = mesh.box(3, 3, 2, deformed=True, jitter=0.1, seed=1, bc=(abi.HX_BC_COPY, [0.] * 5))
m.node_adj = np.zeros((m.n_elem[1], 6, m.nfq))
dev = Device_mesh(Context(0), m)
vd = m.vertex_data()
jacobian = lambda: dev.lib.hx_calc_jacobian(dev.ptr, ctypes.byref(vd))
assert jacobian() == abi.HX_OK
failed = 0
for kind in (0, 1):
    for after in range(100):
        calls()
        fake.fake_fail(kind, after)
        status = jacobian()
        fake.fake_fail(kind, -1)
        log = calls()
        copies = [k for k, x in enumerate(log) if x.startswith("copy")]
        assert not copies or "wait" in log[copies[-1]:], (kind, after, log)
        if status == abi.HX_OK:
            break
        failed += 1
assert failed >= 8, failed
""")


@pytest.mark.parametrize("row_sizes", [[4], [5], [6], [4, 6]], ids=str)
def test_group_of_some_row_sizes(run, row_sizes):
    """A fused group that has no mesh of some of the row sizes its kernels are built for."""
    run(f"""
ctx, devs = Context(0), []
for rs in {row_sizes}:
    m = configs.euler_box(2, rs, seed=1)
    devs.append(Device_mesh(ctx, m))
    devs[-1].set_cases(1, [np.zeros(m.n_elem[0], np.int32), None])
g = Device_group(ctx, devs)
assert g.fused
g.update(abi.update_options())
assert sum("k_fused_local_euler" in x for x in calls()) == 2
""")


def test_group_cases_registered_anew(run):
    """More cases on a member of a live group than the group was created with: their time steps have room."""
    run("""
ctx = Context(0)
m = mesh.concat([configs.euler_box(1, 4, seed=k) for k in range(20)])
dev = Device_mesh(ctx, m)
dev.set_cases(1, [np.zeros(20, np.int32), None])
g = Device_group(ctx, [dev])
opts = abi.update_options()
g.update(opts)
for n in (20, 1, 10):
    dev.set_cases(n, [(np.arange(20) * n // 20).astype(np.int32), None])
    dev.lib.hx_mesh_mark_changed(dev.ptr)
    g.update(opts, (abi.hx_update_status * n)())
""")


def test_failed_group_leaves_its_meshes_free(run):
    """A group whose creation fails does not count among its meshes' groups."""
    run("""
ctx = Context(0)
m = configs.euler_box(2, 4, seed=1)
dev = Device_mesh(ctx, m)
dev.set_cases(1, [np.zeros(m.n_elem[0], np.int32), None])
fake.fake_fail(0, 0)  # the upload of the member tables
try:
    Device_group(ctx, [dev])
    raise SystemExit("the group was created")
except RuntimeError:
    pass
fake.fake_fail(0, -1)
dev.close()
""")


UPDATE_WITH_FIX = """
m = configs.euler_box(2, 4, seed=1)
dev = Device_mesh(Context(0), m)
opts, st = abi.update_options(local_time=True, fix_admis=True), abi.hx_update_status()
calls()
"""


def test_update_checks_admissibility_once_before_a_fix(run):
    """The verdict that makes an update call the fix is the fix's first: one check per iteration and one per stage."""
    run(UPDATE_WITH_FIX + """
fake.fake_verdict(0, 1)
dev.update(opts, st)
assert st.fix_admis_iters == 1
log = calls()
assert sum("k_admissibleI" in x for x in log) == 3, log
""")


def test_update_that_ends_not_finite_leaves_its_faces(run):
    """A folded stage 0 extrapolates into the second face buffer; an update that its check ends leaves the faces in the
    first, where a download reads them."""
    run(UPDATE_WITH_FIX + """
fake.fake_verdict(1, 1)
assert dev.lib.hx_update(dev.ptr, ctypes.byref(opts), ctypes.byref(st)) == abi.HX_ERR_NOT_FINITE
log = calls()
check = [k for k, x in enumerate(log) if "k_admissibleI" in x][-1]
assert any("k_faces_to_primary" in x for x in log[check:]), log
""")


def test_cases_that_could_not_be_registered_are_refused(run):
    """A registration that runs out of memory leaves no cases: neither the old ones, some of whose tables are gone, nor a part
    of the new ones."""
    run("""
ctx = Context(0)
m = mesh.concat([configs.euler_box(1, 4, seed=k) for k in range(8)])
dev = Device_mesh(ctx, m)
one, eight = np.zeros(8, np.int32), np.arange(8, dtype=np.int32)
dev.set_cases(1, [one, None])
g = Device_group(ctx, [dev])
opts, st = abi.update_options(), (abi.hx_update_status * 8)()
failed = 0
for after in range(100):
    dev.set_cases(1, [one, None])
    dev.lib.hx_mesh_mark_changed(dev.ptr)
    fake.fake_fail(2, after)
    status = dev.lib.hx_mesh_set_cases(dev.ptr, 8, abi.iptr(eight), None)
    fake.fake_fail(2, -1)
    if status == abi.HX_OK:
        break
    calls()
    assert dev.lib.hx_update_cases(dev.ptr, ctypes.byref(opts), st) == abi.HX_ERR_INVALID, after
    assert dev.lib.hx_group_update(g.ptr, ctypes.byref(opts), st) == abi.HX_ERR_INVALID, after
    assert not any(x.startswith("launch") for x in calls())
    failed += 1
assert failed >= 4, failed
dev.set_cases(8, [eight, None])
g.update(opts, st)
""")
