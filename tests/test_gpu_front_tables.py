"""Fronts ordered by tabled digit passes: taken by capacity (more than 2^25 entries), with the entries'
number on the device, so that any number of them goes through it."""
import numpy as np
import pytest

from conftest import load_package

pytestmark = pytest.mark.gpu

CAP = (1 << 25) + 64


@pytest.fixture(scope="module")
def pkg():
    return load_package()


def _rows(a):
    return a[np.lexsort((a[:, 1], a[:, 0]))]


def _spot(copies, others):
    """`copies` of one triangle (each pair of them an external entry) and `others` far from them."""
    rng = np.random.default_rng(0)
    a = np.repeat(rng.random((1, 3, 3)), copies, 0)
    b = 30 + 10 * rng.random((others, 1, 3)) + 0.3 * rng.random((others, 3, 3))
    v = np.concatenate([a, b]).reshape(-1, 3).astype(np.float32)
    return np.arange(len(v), dtype=np.int32).reshape(-1, 3), v


@pytest.mark.parametrize("scheduler", ["SCHED_PLAIN", "SCHED_LEARNED_NO_NET"])
@pytest.mark.parametrize("copies,others,entries", [(1, 0, (0, 0)), (2, 0, (0, 1)), (91, 0, (0, 4095)),
                                                   (91, 2, (91, 4096)), (91, 4, (93, 4097)), (300, 4000, None)])
def test_front_orders_of_large_capacities(pkg, oracle, copies, others, entries, scheduler):
    """No entry, one, a tile of 4096 less one, full and plus one, and many tiles, in node order (plain
    schedule) and in query order: fronts and pairs equal the oracle's after GENERATE and two UPDATEs."""
    print(f"[gpu] tabled front order: {copies} + {others}, {scheduler}", flush=True)
    faces, v = _spot(copies, others)
    T = len(faces)
    ctx = pkg.CollisionContext(T, 3 * T, int_front_cap=CAP, ext_front_cap=CAP, pair_cap=1 << 20,
                               scheduler=getattr(pkg, scheduler))
    ctx.set_topology(faces, 3 * T)
    orc = oracle.OracleContext(faces, 3 * T)
    moved = (v + np.random.default_rng(1).normal(0, 0.4, v.shape)).astype(np.float32)
    for k, (xyz, op) in enumerate([(v, (0, 1)), (moved, (1, 2)), (v, (1, 2))]):
        for c in (ctx, orc):
            c.update_vertices(xyz)
            c.step(*op)
        for w in (0, 1):
            got, want = ctx.export_front(w), orc.front(w)
            if k == 0 and entries is not None:
                assert len(want) == entries[w]
            key = got[:, 1] if scheduler == "SCHED_PLAIN" else got[:, 0]
            assert (np.diff(key) >= 0).all(), (k, w)
            np.testing.assert_array_equal(_rows(got), _rows(np.asarray(want).reshape(-1, 2)), err_msg=f"{k} {w}")
        np.testing.assert_array_equal(oracle.pair_set(ctx.pairs(False)), oracle.pair_set(orc.pairs(False)))
    ctx.close()
