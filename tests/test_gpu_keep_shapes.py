"""KEEP's launch shapes on scenes of 2^20 triangles and more, where it tests 16-byte grid records first."""
import numpy as np
import pytest

from conftest import load_package

pytestmark = pytest.mark.gpu

SHAPES = [(16384, 1, 128), (300, 1, 256), (4096, 1, 512), (16384, 2, 128), (1536, 2, 256), (777, 2, 512),
          (64, 4, 128), (3001, 4, 256), (8192, 4, 512), (8, 4, 512)]


@pytest.fixture(scope="module")
def pkg():
    return load_package()


@pytest.mark.parametrize("preset,n,skip_adjacent", [("cloth1024", 726, False), ("cloth1024", 726, True),
                                                    ("layers4", 370, False)])
def test_keep_launch_shapes_on_grid_records(pkg, preset, n, skip_adjacent):
    """Every unroll and workgroup size, on a folded cloth (the records decide nearly every entry) and on
    sheets of one grid on one another (they leave many open, the boxes are tested instead): the pairs of
    a pure traversal in another context."""
    sc = pkg.Scene.preset(preset, n=n)
    print(f"[gpu] keep shapes on grid records: {preset} {sc.num_tris} skip {skip_adjacent}", flush=True)
    assert sc.num_tris >= 1 << 20
    ctx, ref = (pkg.CollisionContext(sc.num_tris, sc.num_verts, narrow_phase=False, skip_adjacent=skip_adjacent)
                for _ in range(2))
    frames = [sc.frame(sc.frames - 6 + k) for k in range(4)]
    want = []
    ref.set_topology(sc.faces(), sc.num_verts)
    for v in frames:
        ref.update_vertices(v)
        ref.step(pkg.BVH_BUILD, pkg.FRONT_PURE_BVH_CD)
        want.append(ref.digest(False))
    assert len(set(want)) == len(want) and want[0][1] > 0
    ref.close()
    ctx.set_topology(sc.faces(), sc.num_verts)
    ctx.update_vertices(frames[0])
    ctx.step(pkg.BVH_BUILD, pkg.FRONT_GENERATE)
    try:
        for k, shape in enumerate(SHAPES):
            pkg.autotune_set(pkg.TUNE_KEEP, sc.num_tris, *shape)
            for at in (1 + k % 3, 0):  # away from where the front was made, and back
                ctx.update_vertices(frames[at])
                ctx.step(pkg.BVH_REFIT, pkg.FRONT_KEEP)
                assert ctx.digest(False) == want[at], (shape, at)
    finally:
        pkg.autotune_set(pkg.TUNE_KEEP, sc.num_tris, 16384, 2, 128)  # the size's default
        ctx.close()


@pytest.mark.parametrize("jitter", [0.0, 0.02])
def test_keep_default_shapes_of_large_scenes(pkg, jitter):
    """More than 2^22 triangles, where the records and the boxes have shapes of their own: sheets of one grid
    on one another (the boxes), and every vertex displaced by 2 % of an edge (the records)."""
    sc = pkg.Scene.preset("layers4", n=726)
    print(f"[gpu] keep default shapes: {sc.num_tris}, jitter {jitter}", flush=True)
    assert sc.num_tris > 1 << 22
    move = np.random.default_rng(1).standard_normal((sc.num_verts, 3)).astype(np.float32) * np.float32(jitter / 725)
    ctx = pkg.CollisionContext(sc.num_tris, sc.num_verts, narrow_phase=False)
    ctx.set_topology(sc.faces(), sc.num_verts)
    got = []
    frames = [sc.frame(sc.frames - 4 + k) + move for k in range(4)]
    for k, v in enumerate(frames):
        ctx.update_vertices(v)
        ctx.step(pkg.BVH_REFIT if k else pkg.BVH_BUILD, pkg.FRONT_KEEP if k else pkg.FRONT_GENERATE)
        got.append(ctx.digest(False))
    for v, d in zip(frames, got):
        ctx.update_vertices(v)
        ctx.step(pkg.BVH_BUILD, pkg.FRONT_PURE_BVH_CD)
        assert ctx.digest(False) == d and d[1] > sc.num_tris
    ctx.close()


def test_keep_counts_every_entry_once(pkg):
    """Node tests of a KEEP: an entry that the grid records leave open counts once, like any other. On
    coinciding sheets the first KEEP tests the records and the second the boxes at once, on the same
    front and vertices: both report the same number."""
    sc = pkg.Scene.preset("layers4", n=370)
    print(f"[gpu] keep node tests, {sc.num_tris}", flush=True)
    ctx = pkg.CollisionContext(sc.num_tris, sc.num_verts, narrow_phase=False)
    ctx.set_topology(sc.faces(), sc.num_verts)
    ctx.update_vertices(sc.frame(sc.frames - 2))
    ctx.step(pkg.BVH_BUILD, pkg.FRONT_GENERATE)
    ctx.update_vertices(sc.frame(sc.frames - 1))
    tests = []
    for op in (pkg.BVH_REFIT, pkg.BVH_NONE, pkg.BVH_NONE):
        ctx.step(op, pkg.FRONT_KEEP)
        s = ctx.stats()
        tests.append(s["node_visits"])
    assert tests[0] == tests[1] == tests[2]
    assert tests[0] >= s["int_front"] + s["ext_front"] - s["implicit_pairs"] > sc.num_tris
    ctx.close()


def test_keep_of_moved_boxes_descends(pkg):
    """Boxes given by the caller, moved since the front was made: KEEP's records and descents find what a
    pure traversal of the same boxes finds, on a cloth that folds on and one that falls back open."""
    sc = pkg.Scene.preset("cloth1024", n=726)
    print(f"[gpu] keep of moved boxes, {sc.num_tris}", flush=True)
    faces = sc.faces()
    ctx, ref = (pkg.CollisionContext(sc.num_tris, sc.num_verts, narrow_phase=False) for _ in range(2))
    for c in (ctx, ref):
        c.set_topology(faces, sc.num_verts)
    seen = set()
    for k, fr in enumerate([-12, -8, -1, -12]):
        v = sc.frame(sc.frames + fr)[faces]
        boxes = np.concatenate([v.min(1), v.max(1)], 1)
        for c, op in ((ctx, pkg.FRONT_KEEP if k else pkg.FRONT_GENERATE), (ref, pkg.FRONT_PURE_BVH_CD)):
            c.update_boxes(boxes)
            c.step(pkg.BVH_REFIT if k else pkg.BVH_BUILD, op)
        s = ctx.stats()
        assert ctx.digest(False) == ref.digest(False) and s["implicit_pairs"] == 0, fr
        if k in (1, 2):
            assert s["node_visits"] > s["int_front"] + s["ext_front"], fr  # it did descend
        seen.add(ctx.digest(False))
    assert len(seen) == 3
    ctx.close()
    ref.close()
