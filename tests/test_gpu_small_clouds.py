"""Small clouds are sorted by one block in LDS (up to 2048 points at one grid
level, up to 8192 at three or more), larger ones by the general passes: the same
cloud padded past the limit with points out of every kernel's reach takes the
general path and must give the same association, pairs and values bit for bit."""
import numpy as np
import pytest

from conftest import params_from_yaml
from rkhs_ba_amd import synth
from rkhs_ba_amd.pointcloud import CvoPointCloud

pytestmark = pytest.mark.gpu

LIMIT = 8192


def cloud(c, idx, total=None, far=0.0):
    """Points idx of c, the first repeated far away up to total."""
    geo = np.random.default_rng(5).uniform(0.05, 1.0, size=(c.n, 2)).astype(np.float32)
    xyz, feat, sem, geo = c.xyz[idx], c.feat[idx], c.sem[idx], geo[idx]
    pad = 0 if total is None else total - len(idx)
    if pad > 0:
        xyz = np.concatenate([xyz, np.repeat(xyz[:1] + np.float32(far), pad, 0)])
        feat, sem, geo = (np.concatenate([a, np.repeat(a[:1], pad, 0)]) for a in (feat, sem, geo))
    return CvoPointCloud.from_arrays(xyz, feat, sem, geo)


@pytest.mark.parametrize("n", [1, 2, 3, 255, 1024, 1025, 2049, 8191, 8192])
@pytest.mark.parametrize("crowded", [False, True])
def test_small_path_equals_general(cvo_gpu, n, crowded):
    p = params_from_yaml("street_60k.yaml")
    p.is_using_geometric_type = 1
    cvo_gpu.write_params(p)
    src, tgt, T = synth.street_pair(4, n=9000)
    idx = np.arange(n) % 40 if crowded else np.arange(n)  # crowded: repeated points, full cells and capped rows
    print(f"small clouds n={n} crowded={crowded}", flush=True)
    a = cvo_gpu.compute_association_gpu(cloud(src, idx), cloud(tgt, idx), T, 0.3)
    b = cvo_gpu.compute_association_gpu(cloud(src, idx, LIMIT + 1, 300.0), cloud(tgt, idx, LIMIT + 1, -300.0), T, 0.3)
    np.testing.assert_array_equal(a.row_ptr, b.row_ptr[: n + 1])
    assert b.row_ptr[-1] == b.row_ptr[n]
    np.testing.assert_array_equal(a.col, b.col)
    np.testing.assert_array_equal(a.val, b.val)
    assert n < 255 or len(a.col) > 0


@pytest.mark.parametrize("n", [2047, 2048, 2049, 4097, 8192, 8193])
@pytest.mark.parametrize("ell", [0.5, 0.22, 0.05])
def test_levels_of_a_registration_equal_general(cvo_gpu, n, ell):
    """A registration's grid has a level for every lengthscale between ell_min and
    ell_init: its first association, at the coarsest, a middle and the finest."""
    p = params_from_yaml("planes_spheres_5k.yaml")
    p.ell_init, p.ell_min = ell, (0.5 if ell < 0.5 else 0.05)
    p.MAX_ITER, p.is_exporting_association = 1, 1
    cvo_gpu.write_params(p)
    src, tgt, T = synth.planes_spheres_pair(4, n, n)

    def padded(c, far):
        pad = LIMIT + 2 - c.n
        xyz = np.concatenate([c.xyz, np.repeat(c.xyz[:1] + np.float32(far), pad, 0)])
        return synth.Cloud(xyz, np.concatenate([c.feat, np.repeat(c.feat[:1], pad, 0)]))

    print(f"levels n={n} ell={ell}", flush=True)
    a = cvo_gpu.align(src, tgt, T, association=True)[4]
    b = cvo_gpu.align(padded(src, 100.0), padded(tgt, -100.0), T, association=True)[4]
    np.testing.assert_array_equal(a.row_ptr, b.row_ptr[: n + 1])
    assert b.row_ptr[-1] == b.row_ptr[n]
    np.testing.assert_array_equal(a.col, b.col)
    np.testing.assert_array_equal(a.val, b.val)
    assert len(a.col) > 0
