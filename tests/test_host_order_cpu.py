"""The order in which the host side queues its work, on the CPU: the library on a HIP runtime that notes
the calls instead of running kernels (hip_host_shim.cpp), each case in a process of its own."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, re, sys
shim = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
shim.shim_log.restype = ctypes.c_char_p
sys.path.insert(0, sys.argv[2])
import numpy as np
from conftest import load_package
pkg = load_package()
def log():
    return [l.split() for l in shim.shim_log().decode().splitlines()]
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("shim") / "hip_host_shim.so")
    subprocess.run(["g++", "-std=c++20", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "hip_host_shim.cpp")],
                   check=True)
    return so


def run(shim, code, *args):
    r = subprocess.run([sys.executable, "-c", PRELUDE + code, shim, HERE, *map(str, args)], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


UPLOADS = """
refused, V = sys.argv[3] == "refused", int(sys.argv[4])
faces = np.arange(30, dtype=np.int32).reshape(-1, 3)
if refused:  # the stages' size
    shim.shim_refuse_pinned(ctypes.c_size_t(12 * V))
ctx = pkg.CollisionContext(10, V)
ctx.set_topology(faces, V)
dev = np.zeros((V, 3), np.float32)
for k in range(8):
    if k == 5:  # a device copy in between, into the buffer of the last upload
        ctx.update_vertices(dev.ctypes.data, pkg.MEM_DEVICE)
    else:
        ctx.update_vertices(np.full((V, 3), k, np.float32))
    ctx.step(pkg.BVH_REFIT if k else pkg.BVH_BUILD, pkg.FRONT_KEEP if k else pkg.FRONT_GENERATE)
text = log()
main = next(l[-1] for l in text if l[0] == "launch")
# walk the log: what of the context's stream each copy onto another stream is known to follow
launched, recorded, waited, read_at, uploads = 0, {}, {}, {}, 0
current = None
for l in text:
    if l[0] == "launch" and l[-1] == main:
        launched += 1
        if current:
            read_at[current] = launched  # the step's kernels read the current buffer
    elif l[0] == "record":
        recorded[l[1]] = (l[-1], launched)
    elif l[0] == "wait":
        st, at = recorded[l[1]]
        if st == main:
            waited[l[-1]] = max(waited.get(l[-1], 0), at)
    elif l[0] == "copy" and launched >= 0 and l[1] in BUFFERS(text):
        if l[-1] != main:
            assert waited.get(l[-1], 0) >= read_at.get(l[1], 0), (l, waited, read_at)
            uploads += 1
        current = l[1]
assert uploads == (0 if not refused and V < 87382 else 7), uploads
"""


@pytest.mark.parametrize("V", [30, 87381, 87382])
@pytest.mark.parametrize("pinned", ["there", "refused"])
def test_uploads_follow_the_steps_that_read_their_buffer(shim, pinned, V):
    """Host vertices up to 1 MB go through a pinned stage on the context's stream, larger ones and those
    whose stage cannot be had on the copy stream: there every upload has waited for the kernels of the
    last step that read its buffer."""
    run(shim, """
def BUFFERS(text):  # the two vertex buffers: the targets of the eight updates
    seen = [l[1] for l in text if l[0] == "copy"]
    return {x for x in seen if seen.count(x) >= 3}
""" + UPLOADS, pinned, V)


def test_counters_are_cleared_once_a_step(shim):
    """A refit clears the step's counters for the KEEP or REORDER that follows it: cleared twice, what the
    last KEEP's records left open would be lost on the way."""
    run(shim, """
ctx = pkg.CollisionContext(100, 300)
ctx.set_topology(np.arange(300, dtype=np.int32).reshape(-1, 3), 300)
v = np.zeros((300, 3), np.float32)
for k, (bvh, front, resets) in enumerate([(pkg.BVH_BUILD, pkg.FRONT_GENERATE, 1), (pkg.BVH_REFIT, pkg.FRONT_KEEP, 0),
                                          (pkg.BVH_REFIT, pkg.FRONT_REORDER, 0), (pkg.BVH_NONE, pkg.FRONT_REORDER, 1),
                                          (pkg.BVH_NONE, pkg.FRONT_KEEP, 1)]):
    shim.shim_clear()
    ctx.update_vertices(v)
    ctx.step(bvh, front)
    assert sum("k_reset_step" in l[1] for l in log()) == resets, (k, log())
""")


@pytest.mark.parametrize("T", [200000, 1 << 20])
def test_a_set_keep_shape_holds_for_every_keep_kernel(shim, T):
    """autotune_set's grid, unroll and workgroup size reach the kernel that tests the grid records and the
    one that tests the boxes instead (scenes of 2^20 triangles and more launch both)."""
    run(shim, """
T = int(sys.argv[3])
ctx = pkg.CollisionContext(T, 3, int_front_cap=4096, ext_front_cap=4096, pair_cap=4096)
ctx.set_topology(np.tile(np.array([[0, 1, 2]], np.int32), (T, 1)), 3)
ctx.update_vertices(np.zeros((3, 3), np.float32))
ctx.step(pkg.BVH_BUILD, pkg.FRONT_GENERATE)
ctx.step(pkg.BVH_REFIT, pkg.FRONT_KEEP)
for grid, unroll, block in [(777, 4, 512), (64, 1, 128), (3000, 2, 256)]:
    pkg.autotune_set(pkg.TUNE_KEEP, T, grid, unroll, block)
    shim.shim_clear()
    ctx.step(pkg.BVH_REFIT, pkg.FRONT_KEEP)
    keeps = [l for l in log() if l[0] == "launch" and "6k_keepI" in l[1]]
    assert len(keeps) == (2 if T >= 1 << 20 else 1)
    for l in keeps:
        assert "k_keepILi%dELi%dE" % (unroll, block // 64) in l[1] and l[3] == str(grid) and l[5] == str(block), keeps
""", T)


def test_refits_write_the_records_that_keep_reads(shim):
    """The 16-byte records are written by refits of scenes of 2^20 triangles and more, not by those of a
    smaller scene in a large context nor of an inter-object front's second object."""
    run(shim, """
T = 1 << 20
caps = dict(int_front_cap=4096, ext_front_cap=4096, pair_cap=4096)
v = np.zeros((3, 3), np.float32)
faces = np.tile(np.array([[0, 1, 2]], np.int32), (T, 1))
ctx = pkg.CollisionContext(T, 3, **caps)
def refits(step):  # the pointers that the two refit kernels have
    shim.shim_clear()
    step()
    kernels = [int(l[7]) for l in log() if l[0] == "launch" and "k_refit" in l[1]]
    assert len(kernels) == 2 and kernels[0] == kernels[1]
    return kernels[0]
ctx.set_topology(faces, 3)
ctx.update_vertices(v)
full = refits(lambda: ctx.step(pkg.BVH_BUILD, pkg.FRONT_GENERATE))
for n, records in [(T, True), (T - 1, False), (5000, False), (T, True)]:
    ctx.set_topology(faces[:n], 3)
    ctx.update_vertices(v)
    want = full if records else full - 2  # without the internal nodes' and the leaves' records
    assert refits(lambda: ctx.step(pkg.BVH_BUILD, pkg.FRONT_GENERATE)) == want
    assert refits(lambda: ctx.step(pkg.BVH_REFIT, pkg.FRONT_KEEP)) == want
inter = pkg.InterFront(ctx, T, 3, **caps)
inter.set_topology(faces, 3)
inter.update_vertices(v)
for op in (pkg.BVH_BUILD, pkg.BVH_REFIT):
    assert refits(lambda: inter.step(op, pkg.FRONT_KEEP)) == full - 2
""")


@pytest.mark.parametrize("Vd,Vr", [(87382, 30), (30, 87382), (90000, 90000)])
def test_uploads_follow_the_inter_steps_that_read_their_buffer(shim, Vd, Vr):
    """An inter-object step reads both objects' vertices (its narrow phase): the next upload into either
    one's buffer on the copy stream waits for it, not only for the queried context's own step."""
    run(shim, """
Vd, Vr = int(sys.argv[3]), int(sys.argv[4])
faces = np.arange(30, dtype=np.int32).reshape(-1, 3)
ctx = pkg.CollisionContext(10, Vd)
ctx.set_topology(faces, Vd)
inter = pkg.InterFront(ctx, 10, Vr, int_front_cap=4096, ext_front_cap=4096, pair_cap=4096)
inter.set_topology(faces, Vr)
large = {"d": Vd > 87381, "r": Vr > 87381}
read = {}
checked = 0
for k in range(6):
    for who, obj, V in (("d", ctx, Vd), ("r", inter, Vr)):
        shim.shim_clear()
        obj.update_vertices(np.zeros((V, 3), np.float32))
        if large[who] and k >= 2:  # waited for an event recorded after the inter step before last
            waits = [l for l in log() if l[0] == "wait"]
            assert len(waits) == 1 and waits[0][1] in read[k - 2], (k, who, waits, read)
            checked += 1
    shim.shim_clear()
    ctx.step(pkg.BVH_REFIT if k else pkg.BVH_BUILD, pkg.FRONT_KEEP if k else pkg.FRONT_GENERATE)
    inter.step(pkg.BVH_REFIT if k else pkg.BVH_BUILD, pkg.FRONT_KEEP if k else pkg.FRONT_GENERATE)
    text = log()
    last = max(i for i, l in enumerate(text) if l[0] == "launch")
    read[k] = {l[1] for l in text[last:] if l[0] == "record"}  # events recorded after its last kernel
assert checked == 4 * sum(large.values())
""", Vd, Vr)
