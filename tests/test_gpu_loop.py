"""The resident iteration loop against the launch-per-pass loop (CVO_NO_GRAPH=1)
of the same library, which the other tests pin to the oracle.

Both evaluate the same pairs with the same float operations; only the order of
the FP64 sums differs (relative 1e-16 a sum), so over a dozen iterations the
stored pairs are equal and the float poses agree to a few units in the last
place (2e-6 absolute at entries of order one, metres up to ten)."""
import os
import threading

import numpy as np
import pytest

from conftest import params_from_yaml
from rkhs_ba_amd import CvoGPU, synth

pytestmark = pytest.mark.gpu

ITERS = 12


def pair(n, m, seed=0, classes=0, feats=5, geo=False):
    src, tgt, T = synth.planes_spheres_pair(seed, max(n, 64), max(m, 64))
    out = []
    for c, k in ((src, n), (tgt, m)):
        rng = np.random.default_rng([seed, k])
        sem = None
        if classes:
            sem = rng.random((c.n, classes)).astype(np.float32)
            sem /= sem.sum(1, keepdims=True)
        g = rng.random((c.n, 2)).astype(np.float32) + 0.1 if geo else None
        f = c.feat[:, :feats] if feats <= 5 else np.concatenate([c.feat, c.feat[:, :feats - 5]], 1)
        out.append(synth.Cloud(c.xyz, np.ascontiguousarray(f), sem, g).subset(np.arange(k)))
    return out[0], out[1]


def run(cvo, src, tgt, adaptive=False):
    cvo.set_trace(ITERS)
    if adaptive:
        ret, T, _, it = cvo.align_adaptive(src, tgt, np.eye(4))
    else:
        ret, T, _, it, _ = cvo.align(src, tgt, np.eye(4))
    return ret, T, it, cvo.get_trace()


def both(p, src, tgt, adaptive=False, pose="fp64", tuning=None, env=None, ran="completed"):
    """ran: what cvo_get_loop_counts says of the first of the two runs."""
    cvo = CvoGPU(params=p)
    try:
        cvo.set_pose_arithmetic(pose)
        if tuning:
            cvo.set_tuning(**tuning)
        print("resident", src.n, tgt.n, flush=True)
        for k, v in (env or {}).items():
            os.environ[k] = v
        try:
            a = run(cvo, src, tgt, adaptive)
        finally:
            for k in env or {}:
                del os.environ[k]
        counts = {k: int(k == ran) for k in ("completed", "abandoned", "declined")}
        assert cvo.loop_counts() == counts
        print("per pass", src.n, tgt.n, flush=True)
        os.environ["CVO_NO_GRAPH"] = "1"
        try:
            b = run(cvo, src, tgt, adaptive)
        finally:
            del os.environ["CVO_NO_GRAPH"]
        assert cvo.loop_counts() == counts
    finally:
        cvo.close()
    assert a[0] == b[0] and a[2] == b[2]
    np.testing.assert_allclose(a[1], b[1], rtol=0, atol=2e-6)
    assert [(r.nnz, r.max_row, r.num_neighbors) for r in a[3]] == [(r.nnz, r.max_row, r.num_neighbors) for r in b[3]]
    assert [r.ell for r in a[3]] == pytest.approx([r.ell for r in b[3]], rel=1e-6)
    return a


def params(**kw):
    p = params_from_yaml("planes_spheres_5k.yaml")
    p.MAX_ITER = ITERS
    for k, v in kw.items():
        setattr(p, k, v)
    return p


# one row; below, at and above a chunk of 8 rows, a block of 16, the 32 blocks
# that exchange in one level, a lane-count step, and a tile of every block
@pytest.mark.parametrize("n,m", [(1, 40), (7, 64), (8, 64), (9, 64), (17, 64), (511, 700), (513, 300), (1040, 900),
                                 (4097, 3001), (8200, 8200), (20011, 20011)])
def test_sizes(n, m):
    src, tgt = pair(n, m)
    both(params(), src, tgt)


@pytest.mark.parametrize("n,kw,adaptive", [(131072, {}, False), (32768, dict(is_using_kdtree=1), False),
                                           (16384, {}, True)])
def test_most_rows(n, kw, adaptive):
    src, tgt = pair(n + 1, 700)
    both(params(MAX_ITER=2, **kw), src.subset(np.arange(n)), tgt, adaptive)
    both(params(MAX_ITER=2, **kw), src, tgt, adaptive, ran="declined")
    if adaptive:  # the self problem of the target has rows too
        both(params(MAX_ITER=2), tgt, src.subset(np.arange(n)), adaptive)
        both(params(MAX_ITER=2), tgt, src, adaptive, ran="declined")


def test_launches_follow_one_another():
    # 600 iterations in three launches: the state goes through memory, the words
    # of the exchanges stay
    src, tgt = pair(1501, 1303)
    p = params(MAX_ITER=600)
    cvo = CvoGPU(params=p)
    try:
        cvo.set_trace(600)
        print("launches one after another", flush=True)
        a = cvo.align(src, tgt, np.eye(4)), [(r.nnz, r.max_row, r.num_neighbors, r.ell) for r in cvo.get_trace()]
        b = cvo.align(src, tgt, np.eye(4)), [(r.nnz, r.max_row, r.num_neighbors, r.ell) for r in cvo.get_trace()]
        assert cvo.loop_counts() == dict(completed=2, abandoned=0, declined=0)
        assert a[0][3] > 256
        # fewer iterations than a launch: the same first ones
        p.MAX_ITER = 250
        cvo.write_params(p)
        c = cvo.align(src, tgt, np.eye(4)), [(r.nnz, r.max_row, r.num_neighbors, r.ell) for r in cvo.get_trace()]
    finally:
        cvo.close()
    np.testing.assert_array_equal(a[0][1], b[0][1])
    assert a[1] == b[1] and a[1][:249] == c[1][:249]


@pytest.mark.parametrize("lanes", [4, 8])
def test_lanes_of_more_rows_than_a_round(lanes):
    src, tgt = pair(20011, 20011)
    both(params(), src, tgt, tuning=dict(lanes_per_row=lanes, cell_scale=0.7))


@pytest.mark.parametrize("kw,cloud,opts", [
    (dict(nearest_neighbors_max=6), {}, {}),                                   # rows over the cap
    (dict(is_using_semantics=1, s_ell=0.5, s_sigma=1.0), dict(classes=19), {}),
    (dict(is_using_semantics=1, s_ell=0.5, s_sigma=1.0, nearest_neighbors_max=9), dict(classes=7, feats=3), {}),
    (dict(is_using_intensity=0, is_using_geometric_type=1), dict(geo=True), {}),
    (dict(is_using_kdtree=2), {}, {}),
    (dict(is_using_kdtree=1), {}, dict(tuning=dict(lanes_per_row=8))),
    (dict(is_using_kdtree=1), dict(classes=19), dict(tuning=dict(lanes_per_row=16, lanes_small_ell=4, split_ell=0.3))),
    ({}, {}, dict(pose="reference")),
    ({}, {}, dict(tuning=dict(lanes_per_row=4, cell_scale=0.5, xcd_remap=0))),
    ({}, dict(feats=8), dict(adaptive=True)),
    (dict(nearest_neighbors_max=8), {}, dict(adaptive=True)),                  # capped self problems too
])
def test_options(kw, cloud, opts):
    src, tgt = pair(1501, 1303, **cloud)
    both(params(**kw), src, tgt, **opts)


def test_a_wait_that_runs_out_falls_back():
    # no wait at all: the first word that is not there yet ends the launch, and
    # the registration is done by the launch-per-pass loop from the saved state
    src, tgt = pair(1501, 1303)
    both(params(), src, tgt, env={"CVO_LOOP_WAIT_MS": "0"}, ran="abandoned")


def test_a_context_pauses_after_an_abandoned_launch():
    # the launch itself ends at once (no wait); each later one that is abandoned
    # doubles the pause, one that completes ends it
    src, tgt = pair(513, 300)
    cvo = CvoGPU(params=params())
    try:
        def align(times, wait=None):
            before = cvo.loop_counts()
            if wait is not None:
                os.environ["CVO_LOOP_WAIT_MS"] = wait
            try:
                Ts = [cvo.align(src, tgt, np.eye(4))[1] for _ in range(times)]
            finally:
                os.environ.pop("CVO_LOOP_WAIT_MS", None)
            for T in Ts:
                np.testing.assert_allclose(T, want, rtol=0, atol=2e-6)
            return [v - before[k] for k, v in cvo.loop_counts().items()]

        want = cvo.align(src, tgt, np.eye(4))[1]
        print("pause after an abandoned launch", flush=True)
        assert align(1, "0") == [0, 1, 0]
        assert align(32, "0") == [0, 0, 32]
        assert align(1, "0") == [0, 1, 0]
        assert align(64) == [0, 0, 64]
        assert align(3) == [3, 0, 0]
        assert align(1, "0") == [0, 1, 0]
        assert align(33) == [1, 0, 32]
    finally:
        cvo.close()


def test_threads_share_the_compute_units():
    # four registrations at once, each wanting every compute unit
    src, tgt = pair(4500, 4500)
    want = both(params(), src, tgt)
    got, counts = [None] * 4, [None] * 4

    def work(i):
        cvo = CvoGPU(params=params())
        try:
            got[i] = [cvo.align(src, tgt, np.eye(4))[1] for _ in range(3)]
            counts[i] = cvo.loop_counts()
        finally:
            cvo.close()

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert all(sum(c.values()) == 3 for c in counts), counts
    # each has its share of the units, so nearly all run resident
    assert sum(c["completed"] for c in counts) >= 9, counts
    for g in got:
        for T in g:
            np.testing.assert_allclose(T, want[1], rtol=0, atol=2e-6)


def test_calls_beside_a_window_that_captures():
    # every window captures its outer iteration; a registration by passes captures
    # too, and both read back at their end
    src, tgt = pair(2000, 2000)
    clouds, _, inits = synth.window_frames(1, n_frames=3, n_min=800, n_max=900)
    pb = params_from_yaml("ba_window.yaml")
    pb.multiframe_max_iters = 1
    pb.multiframe_min_nonzeros = 1
    errors = []

    def guarded(work):
        def run():
            try:
                work()
            except Exception as e:  # noqa: BLE001
                errors.append(e)
        return threading.Thread(target=run)

    def windows():
        cvo = CvoGPU(params=pb)
        try:
            for _ in range(60):
                cvo.align_multiframe(clouds, inits, [1, 0, 0], [(0, 1), (1, 2)])
        finally:
            cvo.close()

    def registrations():
        cvo = CvoGPU(params=params())
        try:
            cvo.set_trace(ITERS)
            for _ in range(60):
                cvo.align(src, tgt, np.eye(4))
        finally:
            cvo.close()

    print("windows beside registrations", flush=True)
    ts = [guarded(windows), guarded(registrations), guarded(windows), guarded(registrations)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
