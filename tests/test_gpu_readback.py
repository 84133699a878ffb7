"""Read-outs and host uploads at the edges of their paths: no step yet, a new topology, capacities given
by the caller, the sizes where the pinned buffers end."""
import numpy as np
import pytest
import torch  # before the library: both then use the HIP runtime that torch brings

from conftest import load_package

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pkg():
    return load_package()


def _device_buffer(pairs):
    return torch.full((pairs, 2), -1, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("first", ["host", "device", "stats", "digest"])
@pytest.mark.parametrize("read", [False, True])
@pytest.mark.parametrize("front", ["FRONT_PURE_BVH_CD", "FRONT_GENERATE", "FRONT_KEEP"])
def test_new_topology_starts_without_pairs(pkg, oracle, front, read, first):
    """After set_topology every read-out reports no pairs until the next step, whether or not the old
    mesh's were read and whichever read-out asks first; the next step's pairs are the new mesh's."""
    print(f"[gpu] read-outs after a new topology: {front}, old pairs read {read}, {first} first", flush=True)
    big, small = pkg.Scene.preset("cloth256", n=40), pkg.Scene.preset("spheres", subdiv=1, spacing=1.9)
    ctx = pkg.CollisionContext(big.num_tris, big.num_verts)
    buf = _device_buffer(64)

    def check(kind):
        if kind == "host":
            assert [len(ctx.pairs(f)) for f in (False, True)] == [0, 0]
        elif kind == "device":
            assert [ctx.pairs_to_device(buf.data_ptr(), 64, f) for f in (False, True)] == [0, 0]
            assert (buf == -1).all()
        elif kind == "stats":
            s = ctx.stats()
            assert (s["bp_pairs"], s["np_pairs"], s["implicit_pairs"], s["int_front"], s["ext_front"]) == (0,) * 5
        else:
            assert ctx.digest(False) == ctx.digest(True) == (0, 0)

    for filtered in (False, True):
        assert len(ctx.pairs(filtered)) == 0  # nor are there any before the first step
    ctx.set_topology(big.faces(), big.num_verts)
    for k, op in enumerate([pkg.FRONT_GENERATE, getattr(pkg, front)]):
        ctx.update_vertices(big.frame(200 + k))
        ctx.step(pkg.BVH_REFIT if k else pkg.BVH_BUILD, op)
    if read:
        assert len(ctx.pairs(False)) > big.num_tris
    ctx.set_topology(small.faces(), small.num_verts)
    for kind in [first] + [k for k in ("host", "device", "stats", "digest") if k != first]:
        check(kind)
    ctx.update_vertices(small.frame(0))
    ctx.step(pkg.BVH_BUILD, pkg.FRONT_GENERATE)
    for filtered in (False, True):
        np.testing.assert_array_equal(oracle.pair_set(ctx.pairs(filtered)), oracle.pair_set(
            oracle.bruteforce_pairs(small.faces(), small.frame(0), filtered)))
    ctx.close()


@pytest.mark.parametrize("cap", [1, (1 << 32) - 1, 1 << 32, 1 << 40, (1 << 40) + 256, (1 << 63) - 1])
def test_device_read_out_takes_any_capacity(pkg, oracle, cap):
    """The caller's capacity says how many pairs its buffer takes, not how many there are: every frame's
    count and pairs are the frame's own whatever it is (the buffer here holds them all)."""
    print(f"[gpu] device read-out with capacity {cap}", flush=True)
    sc = pkg.Scene.preset("cloth256", n=40)
    ctx = pkg.CollisionContext(sc.num_tris, sc.num_verts)
    ctx.set_topology(sc.faces(), sc.num_verts)
    for k, fr in enumerate((0, 290)):
        v = sc.frame(fr)
        ctx.update_vertices(v)
        ctx.step(pkg.BVH_BUILD, pkg.FRONT_GENERATE)
        want = oracle.pair_set(oracle.bruteforce_pairs(sc.faces(), v, False))
        buf = _device_buffer(len(want) + 64)
        assert ctx.pairs_to_device(buf.data_ptr(), cap, filtered=False) == len(want)
        got = buf.cpu().numpy()
        if cap >= len(want):
            np.testing.assert_array_equal(oracle.pair_set(got[: len(want)]), want)
        assert (got[min(cap, len(want)):] == -1).all() and (got[: min(cap, len(want))] >= 0).all()
    ctx.close()


def _groups(sizes):
    """Groups of equal triangles far from one another: every pair within a group is a hit."""
    t = np.array([[0, 0, 0], [1, 0, 0.2], [0, 1, 0.1]], np.float32)
    at = np.repeat(np.arange(len(sizes)), sizes)
    v = t[None] + np.stack([3.0 * (at % 32), 3.0 * (at // 32), 0.0 * at], 1)[:, None]
    return np.arange(3 * len(at), dtype=np.int32).reshape(-1, 3), v.reshape(-1, 3).astype(np.float32), at


@pytest.mark.parametrize("count", [0, 1, 65535, 65536, 65537, 130816])
def test_host_read_out_at_the_pinned_limit(pkg, oracle, count):
    """Host read-outs of up to 65,536 pairs go through a pinned buffer, larger ones do not: the pairs around
    the limit, read twice and in pieces of a smaller capacity, and a small read-out after a large one."""
    print(f"[gpu] host read-out of {count} pairs", flush=True)
    big = {0: 1, 1: 2, 130816: 512}.get(count, 362)
    sizes = [big] + [2] * (count - big * (big - 1) // 2) + [1]
    faces, v, at = _groups(sizes)
    first = np.concatenate([[0], np.cumsum(sizes)])
    want = np.concatenate([[(first[g] + i, first[g] + j) for i in range(m) for j in range(i + 1, m)] or
                           np.zeros((0, 2)) for g, m in enumerate(sizes)]).astype(np.int32).reshape(-1, 2)
    assert len(want) == count
    ctx = pkg.CollisionContext(len(faces), len(v))
    ctx.set_topology(faces, len(v))
    ctx.update_vertices(v)
    for op in (pkg.FRONT_PURE_BVH_CD, pkg.FRONT_GENERATE, pkg.FRONT_KEEP):
        ctx.step(pkg.BVH_BUILD if op == pkg.FRONT_PURE_BVH_CD else pkg.BVH_NONE, op)
        for filtered in (False, True, False):
            np.testing.assert_array_equal(oracle.pair_set(ctx.pairs(filtered)), oracle.pair_set(want))
    few = np.full((7, 2), -1, np.int32)  # room for fewer than there are
    import ctypes
    n = ctypes.c_int64()
    assert pkg.lib().bvhcd_get_pairs(ctx._h, few.ctypes.data, 5, ctypes.byref(n), pkg.MEM_HOST, 1) == pkg.OK
    assert n.value == count and (few[min(count, 5):] == -1).all() and (few[:min(count, 5)] >= 0).all()
    ctx.close()


@pytest.mark.parametrize("a,b", [((255,), (257,)), ((256,), (256,)), ((256, 1), (256, 1)), ((3,), (5,)), ((1,), (0, 1))])
def test_inter_host_read_out_at_the_pinned_limit(pkg, a, b):
    """The same for an inter-object front: 65,535, 65,536 and 65,537 pairs, a few, and none."""
    print(f"[gpu] inter read-out {a} {b}", flush=True)
    (fa, va, ga), (fb, vb, gb) = _groups(a), _groups(b)
    want = np.array([(i, j) for i in range(len(fa)) for j in np.flatnonzero(gb == ga[i])], np.int32).reshape(-1, 2)
    ctx = pkg.CollisionContext(max(len(fa), 2), 3 * len(fa) + 3)
    ctx.set_topology(fa, len(va))
    ctx.update_vertices(va)
    ctx.step(pkg.BVH_BUILD, pkg.FRONT_GENERATE)
    inter = pkg.InterFront(ctx, len(fb), len(vb), int_front_cap=1 << 18, ext_front_cap=1 << 18, pair_cap=1 << 18)
    inter.set_topology(fb, len(vb))
    inter.update_vertices(vb)
    for k, op in enumerate((pkg.FRONT_GENERATE, pkg.FRONT_KEEP)):
        inter.step(pkg.BVH_REFIT if k else pkg.BVH_BUILD, op)
        for filtered in (False, True, False):
            got = inter.pairs(filtered)
            np.testing.assert_array_equal(got[np.lexsort((got[:, 1], got[:, 0]))], want)
    inter.close()
    ctx.close()


def test_uploads_across_the_stage_limit(pkg, oracle):
    """Host vertices go through a pinned stage up to 87,381 of them and on the copy stream beyond: scenes on
    both sides of the limit in one context, one after another, every frame's array overwritten right
    after its upload, steps queued without a read-out between. Every scene's last pairs are brute force's."""
    print("[gpu] uploads across the stage limit", flush=True)
    small, large = pkg.Scene.preset("cloth256", n=60), pkg.Scene.preset("cloth256", n=296)
    assert small.num_verts <= 87381 < large.num_verts
    ctx = pkg.CollisionContext(large.num_tris, large.num_verts)
    for sc in (small, large, small, small, large):
        ctx.set_topology(sc.faces(), sc.num_verts)
        buf = np.empty((sc.num_verts, 3), np.float32)
        for k in range(9):
            buf[:] = sc.frame(200 + 8 * k)
            ctx.update_vertices(buf)
            buf[:] = np.nan
            ctx.step(pkg.BVH_REFIT if k else pkg.BVH_BUILD, pkg.FRONT_KEEP if k else pkg.FRONT_GENERATE)
        want = oracle.pair_set(oracle.bruteforce_pairs(sc.faces(), sc.frame(264), True))
        np.testing.assert_array_equal(oracle.pair_set(ctx.pairs(True)), want)
    ctx.close()
