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
