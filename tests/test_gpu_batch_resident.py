"""The resident form of the lockstep batch (2D): instances of one patch, of
several, nodes with more neighbours in their patch than the kernels' 8 and 12
rows hold (the second takes the launch-per-iteration form), constraints of one
component, loads on constrained nodes; against a dense FP64 solve.  A relative
residual of TOL leaves a relative error of at most cond(K) TOL."""
import threading

import numpy as np
import pytest
from scipy.spatial import Delaunay

import cudafemproject_amd as F
from cudafemproject_amd.problem import BatchInstance, load_batch, plate_batch
from helpers import dense_K

pytestmark = pytest.mark.gpu

TOL = 1e-11


def instance(nodes, elems, rng, nr, code=3):
    x = nodes[:, 0]
    fixed = np.flatnonzero(x <= x.min() + 0.3 * (x.max() - x.min())).astype(np.int32)
    codes = np.full(len(fixed), code, np.int32)
    codes[::2] = 3  # (no rigid motion is left)
    f = rng.standard_normal((len(nodes), nr, 2))
    return BatchInstance(nodes=nodes, elems=elems.astype(np.int32), E=float(rng.uniform(1e7, 3e7)),
                         nu=float(rng.uniform(0.2, 0.35)), constr_node=fixed, constr_code=codes, f=f)


def fan(degree):
    """A node with `degree` neighbours, a second ring around them."""
    a = 2 * np.pi * np.arange(degree) / degree
    ring = np.stack([np.cos(a), np.sin(a)], 1)
    nodes = np.concatenate([[[0.0, 0.0]], ring, 2.0 * ring])
    i, j = np.arange(degree), (np.arange(degree) + 1) % degree
    elems = np.concatenate([np.stack([np.zeros(degree, int), 1 + i, 1 + j], 1),
                            np.stack([1 + i, 1 + degree + i, 1 + degree + j], 1),
                            np.stack([1 + i, 1 + degree + j, 1 + j], 1)])
    return nodes, elems


def scattered(n, rng):
    """Delaunay triangles of a jittered grid (node degrees up to about 9)."""
    g = np.stack(np.meshgrid(np.arange(n), np.arange(n), indexing="ij"), -1).reshape(-1, 2).astype(float)
    nodes = g + rng.uniform(-0.3, 0.3, g.shape)
    t = Delaunay(nodes).simplices
    e = nodes[t]
    d1, d2 = e[:, 1] - e[:, 0], e[:, 2] - e[:, 0]
    det = d1[:, 0] * d2[:, 1] - d1[:, 1] * d2[:, 0]
    return nodes, t[np.abs(det) > 0.05]  # (no slivers on the hull)


def used(nodes, elems):
    ids = np.unique(elems)
    new = np.full(len(nodes), -1)
    new[ids] = np.arange(len(ids))
    return nodes[ids], new[elems]


def check(ctx, insts, precision=F.FP64):
    load_batch(ctx, insts)
    us, st, _ = ctx.batch_solve([b.f for b in insts], precision=precision, tol=TOL)
    us2, st2, _ = ctx.batch_solve([b.f for b in insts], precision=precision, tol=TOL)
    assert np.all(st["status"] == 0) and np.all(st["rel_res"] <= TOL)
    assert np.array_equal(st, st2)
    for b, u, u2 in zip(insts, us, us2):
        K = dense_K(b.problem())
        assert np.array_equal(u, u2)
        for r in range(b.f.shape[1]):
            x = np.linalg.solve(K, b.f[:, r].ravel())
            assert np.linalg.norm(u[:, r].ravel() - x) <= np.linalg.cond(K) * TOL * np.linalg.norm(x)


@pytest.mark.parametrize("degrees", [(6,), (8, 3), (9, 6), (12, 8), (13, 5), (40, 6)])
def test_neighbour_counts(ctx, degrees):
    rng = np.random.default_rng(sum(degrees))
    check(ctx, [instance(*fan(d), rng, 4) for d in degrees])


@pytest.mark.parametrize("nr,code", [(1, 3), (2, 1), (3, 2), (4, 3)])
def test_scattered_meshes(ctx, nr, code):
    """One to several patches an instance, nodes in no order."""
    rng = np.random.default_rng(10 * nr + code)
    insts = []
    for n in (3, 16, 17, 24):
        nodes, elems = used(*scattered(n, rng))
        p = rng.permutation(len(nodes))
        q = np.empty_like(p)
        q[p] = np.arange(len(p))
        insts.append(instance(nodes[p], q[elems], rng, nr, code))
    check(ctx, insts, F.MIXED if nr == 2 else F.FP64)


def test_more_workgroups_than_the_device_holds(ctx):
    """Instances wait for their turn: the same bits as one at a time."""
    insts = plate_batch(90, seed=3, nx_range=(60, 80), ny_range=(30, 40))
    load_batch(ctx, insts)
    us, st, _ = ctx.batch_solve([b.f for b in insts], precision=F.FP64, tol=1e-9)
    assert np.all(st["status"] == 0)
    for i in (0, 41, 89):
        load_batch(ctx, insts[i:i + 1])
        u1, s1, _ = ctx.batch_solve([insts[i].f], precision=F.FP64, tol=1e-9)
        assert np.array_equal(us[i], u1[0]) and np.array_equal(st[i], s1[0])


def test_two_batches_at_once():
    """Two contexts in two threads share the device."""
    insts = plate_batch(40, seed=4, nx_range=(30, 60), ny_range=(20, 40))
    want, got = {}, {}

    def work(k, out):
        with F.Context(0) as c:
            load_batch(c, insts[20 * k:20 * k + 20])
            for _ in range(3):
                out[k] = c.batch_solve([b.f for b in insts[20 * k:20 * k + 20]], tol=1e-9)[0]

    for k in (0, 1):
        work(k, want)
    ts = [threading.Thread(target=work, args=(k, got)) for k in (0, 1)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for k in (0, 1):
        for a, b in zip(want[k], got[k]):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("degree,fixed,resident", [(8, False, 1), (9, False, 1), (12, False, 1),
                                                   (13, False, 0), (13, True, 1), (40, True, 1)])
def test_form_by_neighbour_count(degree, fixed, resident):
    """The rows are chosen before the launch: no launch runs in vain, and none
    on rows that lack a neighbour (a constrained node's hold none)."""
    nodes, elems = fan(degree)
    rng = np.random.default_rng(degree)
    b = instance(nodes, elems, rng, 2)
    con = np.union1d(b.constr_node, [0]) if fixed else np.setdiff1d(b.constr_node, [0])
    b.constr_node = con.astype(np.int32)
    b.constr_code = np.full(len(con), 3, np.int32)
    with F.Context(0) as c:
        check(c, [b, instance(*fan(5), rng, 2)])
        assert c.resident_info() == (2 * resident, 0)


def test_patience_with_queued_peers():
    """Instances of more than half the device each: the second one's first
    workgroups wait for the rest of it until the first one ends, here some ten
    times the bound of a wait (2 ms).  Nobody gives up, and the bits are those
    with the usual bound."""
    insts = plate_batch(3, seed=5, nx_range=(255, 260), ny_range=(255, 260))
    rhs = [b.f[:, :1] for b in insts]
    with F.Context(0) as c:
        load_batch(c, insts)
        us, st, ms = c.batch_solve(rhs, precision=F.FP64, tol=1e-8)
        print(f"[patience] {ms:.1f} ms, {st['iterations'].ravel()} iterations", flush=True)
        assert np.all(st["status"] == 0) and c.resident_info() == (1, 0)
        assert ms > 40.0  # (three instances in turn: each waits some 10 ms)
        c.set_resident(F.RESIDENT_TEST_SHORT_WAITS)
        us2, st2, _ = c.batch_solve(rhs, precision=F.FP64, tol=1e-8)
        assert c.resident_info() == (2, 0)
        assert np.array_equal(st, st2) and all(np.array_equal(a, b) for a, b in zip(us, us2))


@pytest.mark.parametrize("nr,n,count", [(1, 258, 3), (4, 175, 4), (2, 120, 9)])
def test_large_instances_take_turns(nr, n, count):
    """More patches than the device holds, in instances of up to two thirds of
    it: every launch completes (in fresh contexts: the hardware starts a launch's
    workgroups differently from one to the next), with the same bits."""
    insts = plate_batch(count, seed=7, nx_range=(n - 3, n + 3), ny_range=(n - 3, n + 3))
    rhs = [b.f[:, :nr] for b in insts]
    first = None
    for k in range(3):
        print(f"[turns] {nr} {n} {count} context {k}", flush=True)
        with F.Context(0) as c:
            load_batch(c, insts)
            for _ in range(2):
                us, st, _ = c.batch_solve(rhs, precision=F.FP64, tol=1e-6)
                assert np.all(st["status"] == 0)
                first = us if first is None else first
                assert all(np.array_equal(a, b) for a, b in zip(us, first))
            assert c.resident_info() == (2, 0)
