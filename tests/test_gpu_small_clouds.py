"""Small clouds are sorted by one block in LDS, larger ones by the general
passes: the same cloud padded past the limit with points out of every kernel's
reach takes the general path and must give the same association, pairs and
values bit for bit."""
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
