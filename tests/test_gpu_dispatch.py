"""The kernels behind each rule of the launch code, at the sizes where the rules change: how
walks are split along their axis, which radii have which kernels, remainders of tiles.  All
against the CPU oracle; the stages are bit-exact, so there is no tolerance."""
import numpy as np
import pytest

import oracle
from hdog import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hd():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from hdog import HDoG
    h = HDoG(0)
    yield h
    h.close()


def noise(shape, seed):
    return np.random.default_rng(seed).integers(0, 4000, shape, dtype=np.uint16)


# lines shorter than a window, one segment, several with a short last one; partial tiles
@pytest.mark.parametrize("shape", [(1, 43, 130), (61, 64, 129), (53, 22, 64), (127, 35, 200)])
def test_split_walks_bitexact(hd, shape):
    img = noise(shape, 3)
    got = hd.Normalize3DFilter(img, 100, 10, 10)
    np.testing.assert_array_equal(got.cpu().numpy(), oracle.normalize3d(img, 100, 10, 10))
    s = (2.0, 1.6, 3.2, 2.56)
    hd.initGaussian3DKernel(*s, truncate=4.0)
    dog = hd.DoG3DFilter(got)
    ref, _ = oracle.dog3d(got.cpu().numpy(), *s, truncate=4.0, gamma=1.0)
    np.testing.assert_array_equal(dog.cpu().numpy(), ref)


# Hessian tiles per records-only work-group: one to four, with a short last walk
@pytest.mark.parametrize("shape", [(70, 40, 70), (33, 640, 700), (49, 1500, 1600)])
def test_records_walks_give_the_materialized_regions(hd, shape):
    import torch
    vol = synth.make_volume("c0", shape=shape, n_blobs=shape[0] * shape[1] * shape[2] // 20000,
                            seed=11)
    img = torch.from_numpy(vol).to(hd.device)
    p = hd.make_params(shape, 10, 10, 0, 2.0, 2.0, 3.2, 3.2, 4.0)
    hd.run_device(img, p)
    a = hd.download_regions()
    hd.run_device(img, p, hd.alloc_intermediates(shape))
    b = hd.download_regions()
    for k in ("label", "count", "size16", "isum", "imax", "centroid", "norm"):
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)


# a mask's bytes are read in fours from any address, its labels written in quads or words:
# every remainder of the width, fewer than four voxels, a mask that starts at an odd byte
@pytest.mark.parametrize("shape", [(1, 1, 1), (1, 1, 3), (2, 1, 2), (5, 9, 61), (5, 9, 62),
                                   (17, 10, 63), (17, 9, 64), (3, 8, 129)])
@pytest.mark.parametrize("skip", [0, 1, 3])
def test_labels_of_any_mask_address(hd, shape, skip):
    import torch
    n = int(np.prod(shape))
    mask = (np.random.default_rng(n).random(n) < 0.4).astype(np.uint8) * 255
    store = torch.zeros(n + 8, dtype=torch.uint8, device=hd.device)
    store[skip:skip + n] = torch.from_numpy(mask).to(hd.device)
    pd = store[skip:skip + n].view(shape)
    store[skip + n:] = 1  # what follows the mask is not read as part of it
    np.testing.assert_array_equal(hd.CCL(pd).cpu().numpy(), oracle.ccl3d(mask.reshape(shape)))
