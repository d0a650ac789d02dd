"""GPU multi-frame IRLS bundle adjustment (cvo_align_multiframe) against the
oracle's restatement of CvoBatchIRLS::solve (src/cvo/IRLS.cpp:148-367) with the
same (r, J) and Levenberg-Marquardt schedule.

Tolerances: after one outer iteration the poses agree to 1e-9 (same pair sets
bit for bit, FP64 sums in another order); after ten outer iterations to 1e-6;
the reference's own contract for converged poses is 1e-4 rad / 1e-4 m."""
import os
import sys

import numpy as np
import pytest

from conftest import CONFIGS, params_from_yaml
from rkhs_ba_amd import CvoError, CvoGPU, synth

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def ba_gpu():
    c = CvoGPU(os.path.join(CONFIGS, "ba_window.yaml"))
    yield c
    c.close()


def window(seed=0, n_frames=4, n_min=1500, n_max=2500):
    return synth.window_frames(seed, n_frames=n_frames, n_min=n_min, n_max=n_max)


def all_edges(n):
    return [(i, j) for i in range(n) for j in range(i + 1, n)]


def rel_errors(P, gts):
    out = []
    for f in range(1, len(P)):
        Ta = np.linalg.inv(P[0]) @ P[f]
        Tb = np.linalg.inv(gts[0]) @ gts[f]
        E = np.linalg.inv(Tb) @ Ta
        out.append((np.degrees(np.arccos(np.clip((np.trace(E[:3, :3]) - 1) / 2, -1, 1))), np.linalg.norm(E[:3, 3])))
    return np.array(out)


def run_both(ba_gpu, oracle, p, clouds, inits, hold, edges):
    ba_gpu.write_params(p)
    say(f"gpu BA frames={len(clouds)} edges={len(edges)} max_iters={p.multiframe_max_iters}")
    g = ba_gpu.align_multiframe(clouds, inits, hold, edges)
    say(f"oracle BA (gpu took {g['seconds']:.3f} s, {g['iters']} iterations)")
    P, it, _ = oracle.align_multiframe(p, clouds, inits, hold, edges, threads=8)
    return g, P, it


def test_one_outer_iteration_matches_oracle(ba_gpu, oracle):
    p = params_from_yaml("ba_window.yaml")
    p.multiframe_max_iters = 1
    clouds, gts, inits = window()
    g, P, it = run_both(ba_gpu, oracle, p, clouds, inits, [1, 0, 0, 0], all_edges(4))
    assert g["iters"] == it == 1
    assert np.abs(g["poses"][:, :3, :4] - inits[:, :3, :4]).max() > 1e-6   # the solve moved the poses
    np.testing.assert_allclose(g["poses"][:, :3, :4], P[:, :3, :4], rtol=0, atol=1e-9)
    np.testing.assert_array_equal(g["poses"][0], inits[0])


def test_ten_outer_iterations_match_oracle(ba_gpu, oracle):
    p = params_from_yaml("ba_window.yaml")
    p.multiframe_max_iters = 10
    clouds, gts, inits = window(seed=3, n_frames=5)
    g, P, it = run_both(ba_gpu, oracle, p, clouds, inits, [1, 0, 0, 0, 0], all_edges(5))
    assert g["iters"] == it
    np.testing.assert_allclose(g["poses"][:, :3, :4], P[:, :3, :4], rtol=0, atol=1e-6)
    e0, e1 = rel_errors(inits, gts), rel_errors(g["poses"], gts)
    assert e1[:, 0].max() < e0[:, 0].max()
    assert len(g["per_iter_seconds"]) >= g["iters"]


def test_partial_edge_graph_and_decay(ba_gpu, oracle):
    # a chain of edges, two constant frames, a faster lengthscale schedule
    p = params_from_yaml("ba_window.yaml")
    p.multiframe_max_iters = 6
    p.multiframe_iter_per_ell = 1
    clouds, gts, inits = window(seed=5, n_frames=5)
    edges = [(0, 1), (1, 2), (2, 3), (3, 4), (4, 1)]
    g, P, it = run_both(ba_gpu, oracle, p, clouds, inits, [1, 0, 0, 1, 0], edges)
    assert g["iters"] == it
    np.testing.assert_allclose(g["poses"][:, :3, :4], P[:, :3, :4], rtol=0, atol=1e-6)
    np.testing.assert_array_equal(g["poses"][3], inits[3])


def test_deterministic_and_direct_launch(ba_gpu):
    p = params_from_yaml("ba_window.yaml")
    p.multiframe_max_iters = 3
    ba_gpu.write_params(p)
    clouds, gts, inits = window(seed=7)
    say("BA determinism: graph x2")
    a = ba_gpu.align_multiframe(clouds, inits, [1, 0, 0, 0], all_edges(4))
    b = ba_gpu.align_multiframe(clouds, inits, [1, 0, 0, 0], all_edges(4))
    np.testing.assert_array_equal(a["poses"], b["poses"])
    say("BA determinism: direct launches")
    os.environ["CVO_NO_GRAPH"] = "1"
    try:
        c = ba_gpu.align_multiframe(clouds, inits, [1, 0, 0, 0], all_edges(4))
    finally:
        del os.environ["CVO_NO_GRAPH"]
    np.testing.assert_array_equal(a["poses"], c["poses"])
    say("BA determinism: profiled launches")
    ba_gpu.set_profiling(True)
    try:
        ba_gpu.reset_kernel_stats()
        d = ba_gpu.align_multiframe(clouds, inits, [1, 0, 0, 0], all_edges(4))
        st = ba_gpu.kernel_stats()
    finally:
        ba_gpu.set_profiling(False)
    np.testing.assert_array_equal(a["poses"], d["poses"])
    assert st["launches"]["assoc"] == d["iters"]
    assert st["launches"]["ba_pair"] > 0


def test_edge_cases(ba_gpu):
    p = params_from_yaml("ba_window.yaml")
    p.multiframe_max_iters = 3
    ba_gpu.write_params(p)
    clouds, gts, inits = window(n_frames=3)
    say("BA no edges")
    r = ba_gpu.align_multiframe(clouds, inits, [0, 0, 0], np.zeros((0, 2), np.int32))
    assert r["iters"] == 0
    np.testing.assert_array_equal(r["poses"][:, :3, :4], inits[:, :3, :4])
    say("BA all constant")
    r = ba_gpu.align_multiframe(clouds, inits, [1, 1, 1], [(0, 1), (1, 2)])
    assert r["iters"] == 3
    np.testing.assert_array_equal(r["poses"][:, :3, :4], inits[:, :3, :4])
    say("BA invalid arguments")
    with pytest.raises(CvoError):
        ba_gpu.align_multiframe(clouds, inits, [1, 0, 0], [(0, 0)])
    with pytest.raises(CvoError):
        ba_gpu.align_multiframe(clouds, inits, [1, 0, 0], [(0, 3)])
    many = [clouds[0]] * 22
    with pytest.raises(CvoError):
        ba_gpu.align_multiframe(many, np.tile(np.eye(4), (22, 1, 1)), None, [(0, 1)])


def test_align_frames_updates_pose_vec_in_place(ba_gpu, oracle):
    from rkhs_ba_amd import CvoFrame
    p = params_from_yaml("ba_window.yaml")
    p.multiframe_max_iters = 2
    ba_gpu.write_params(p)
    clouds, gts, inits = window(seed=9, n_frames=3)
    frames = [CvoFrame(c, T) for c, T in zip(clouds, inits)]
    edges = [(frames[0], frames[1]), (frames[1], frames[2]), (frames[0], frames[2])]
    say("BA align_frames")
    secs = ba_gpu.align_frames(frames, [True, False, False], edges)
    assert secs > 0
    P, it, _ = oracle.align_multiframe(p, clouds, inits, [1, 0, 0], [(0, 1), (1, 2), (0, 2)])
    for f, T in zip(frames, P):
        np.testing.assert_allclose(f.pose_vec.reshape(3, 4), T[:3, :4], rtol=0, atol=1e-8)


@pytest.mark.parametrize("sizes,shift", [((1, 64, 700), 0.0), ((63, 65, 513), 0.0), ((511, 512, 1025), 0.0),
                                         ((1500, 1300, 1700), 100.0)])
def test_moments_match_oracle(ba_gpu, oracle, sizes, shift):
    """The solve's polynomials in the poses where a frame is one row, a wave's
    rows and one more, a moment block's rows and one more, and far from the
    world's origin.  The oracle sums over the pairs at every candidate; both are
    FP64, so 1e-9 as above, and 1e-8 at 100 m (the pair offsets, 0.1 m, lose
    three digits more in its world coordinates)."""
    p = params_from_yaml("ba_window.yaml")
    p.multiframe_max_iters = 2
    p.multiframe_min_nonzeros = 1
    clouds, gts, inits = window(seed=11, n_frames=3, n_min=2000)
    clouds = [c.subset(np.arange(n)) for c, n in zip(clouds, sizes)]
    inits = inits.copy()
    inits[:, :3, 3] += shift
    g, P, it = run_both(ba_gpu, oracle, p, clouds, inits, [1, 0, 0], [(0, 1), (1, 2), (2, 0)])
    assert g["iters"] == it
    np.testing.assert_allclose(g["poses"][:, :3, :4], P[:, :3, :4], rtol=0, atol=1e-8 if shift else 1e-9)


@pytest.mark.parametrize("far", [200.0, 4000.0, 3e4, 1e5, 1e6])
def test_moments_of_clouds_with_a_stray_return_match_oracle(ba_gpu, oracle, far):
    """One point of each cloud far from the rest moves the middle of its bounding
    box by half as much, and no pair: the moments are taken about the paired
    points.  1e-9 as above."""
    p = params_from_yaml("ba_window.yaml")
    p.multiframe_max_iters = 2
    p.multiframe_min_nonzeros = 1
    clouds, gts, inits = window(seed=11, n_frames=3)
    away = [(far, 0.3 * far, 0.0), (-0.6 * far, far, 1.0), (0.2 * far, -far, -2.0)]
    clouds = [synth.Cloud(np.concatenate([c.xyz, np.float32([a])]), *(None if x is None else np.concatenate([x, x[:1]])
                          for x in (c.feat, c.sem))) for c, a in zip(clouds, away)]
    g, P, it = run_both(ba_gpu, oracle, p, clouds, inits, [1, 0, 0], [(0, 1), (1, 2), (2, 0)])
    assert g["iters"] == it
    say(f"stray at {far}: {np.abs(g['poses'][:, :3, :4] - P[:, :3, :4]).max():.3e}")
    np.testing.assert_allclose(g["poses"][:, :3, :4], P[:, :3, :4], rtol=0, atol=1e-9)


def test_ragged_window_within_a_workspace_limit():
    """One long frame among short ones: the moments' partials are those of each
    edge's own blocks, and under a limit that does not hold them the blocks walk
    more rows, down to one an edge.  Same pairs, FP64 sums in another order: 1e-9."""
    p = params_from_yaml("ba_window.yaml")
    p.multiframe_max_iters = 2
    p.multiframe_min_nonzeros = 1
    p.multiframe_num_neighbors = 64
    sizes = [20000] + [400] * 7
    clouds, gts, inits = window(seed=11, n_frames=8, n_min=20000, n_max=20000)
    clouds = [c.subset(np.arange(n)) for c, n in zip(clouds, sizes)]
    edges, hold = all_edges(8), [1] + [0] * 7

    def run(limit):
        c = CvoGPU(params=p)
        try:
            c.set_workspace_limit(limit)
            say(f"ragged window, limit {limit}")
            r = c.align_multiframe(clouds, inits, hold, edges)
            return r["poses"], c.workspace_bytes()
        finally:
            c.close()

    want, used = run(0)
    # 7 edges of 20000 rows and 21 of 400: 301 blocks of 512 rows, 670 doubles each
    partials = 5 * 8 * 670 * 301 // 4
    for short in (0, partials // 3, partials // 4 * 3, partials):
        got, held = run(used - short)
        assert held <= used - partials + 4096  # given back
        np.testing.assert_allclose(got[:, :3, :4], want[:, :3, :4], rtol=0, atol=1e-9)
    with pytest.raises(CvoError):
        run(used // 2)


@pytest.mark.parametrize("free", [1, 2, 10, 11, 20])
def test_solve_sizes_match_oracle(ba_gpu, oracle, free):
    """The normal equations of 6 dof (less than a factorisation block) to 120
    (the most; two rows a lane, 74 edges: more than a wave lists at once).  Two
    outer iterations as above: 1e-9."""
    p = params_from_yaml("ba_window.yaml")
    p.multiframe_max_iters = 2
    p.multiframe_min_nonzeros = 1
    n = free + 1
    clouds, gts, inits = window(seed=5, n_frames=n, n_min=600, n_max=700)
    edges = [(i, j) for i in range(n) for j in range(i + 1, min(n, i + 5))]
    g, P, it = run_both(ba_gpu, oracle, p, clouds, inits, [1] + [0] * free, edges)
    assert g["iters"] == it
    np.testing.assert_allclose(g["poses"][:, :3, :4], P[:, :3, :4], rtol=0, atol=1e-9)
