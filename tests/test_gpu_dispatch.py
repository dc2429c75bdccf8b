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
    blobs = synth.blob_table(shape, shape[0] * shape[1] * shape[2] // 20000, 11)
    img = hd.synth_volume(shape, blobs, 11, 200.0, 200.0, 20.0)
    p = hd.make_params(shape, 10, 10, 0, 2.0, 2.0, 3.2, 3.2, 4.0)
    hd.run_device(img, p)
    a = hd.download_regions()
    hd.run_device(img, p, hd.alloc_intermediates(shape))
    b = hd.download_regions()
    for k in ("label", "count", "size16", "isum", "imax", "centroid", "norm"):
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)


# given labels: tiles of one region, of a region per voxel (more than a tile's table holds),
# of none, regions across tiles, ragged edges; with and without the raw stack, max and sum
@pytest.mark.parametrize("shape,kind", [((17, 9, 65), "solid"), ((16, 8, 64), "points"),
                                        ((33, 41, 130), "random"), ((20, 16, 64), "empty")])
@pytest.mark.parametrize("ave", [False, True])
def test_features_of_given_labels(hd, shape, kind, ave):
    rng = np.random.default_rng(7)
    pd = np.zeros(shape, np.uint8)
    if kind == "solid":
        pd[:] = 1
    elif kind == "points":
        pd[::2, ::2, ::2] = 1
    elif kind == "random":
        pd[:] = rng.random(shape) < 0.07
    hess = (rng.standard_normal((6,) + shape) * 0.01).astype(np.float32)
    norm = rng.standard_normal(shape).astype(np.float32)
    img = noise(shape, 8)
    labels = hd.CCL(pd)
    np.testing.assert_array_equal(labels.cpu().numpy(), oracle.ccl3d(pd))
    o = oracle.regions(labels.cpu().numpy(), hess, norm, img, ave)
    g = hd.RegionalFeatures(labels, hess, norm, img, ave)
    for k in ("label", "count", "size16", "isum", "imax"):
        np.testing.assert_array_equal(g[k][1:], o[k][1:], err_msg=k)
    np.testing.assert_array_equal(g["centroid"][1:], o["centroid"][1:])
    # sums: FP64 in another order, rounded once to FP32
    n = o["count"][1:, None].astype(np.float64)
    mag = np.abs(hess).max() * n
    assert np.all(np.abs(g["hsum"][1:].astype(np.float64) - o["hsum"][1:]) <=
                  1.2e-7 * np.abs(o["hsum"][1:]) + 1e-12 * mag)
    d = np.abs(g["norm"][1:].astype(np.float64) - o["norm"][1:])
    assert np.all(d <= (1.2e-7 * np.abs(o["norm"][1:]) + 1e-12 * n[:, 0] * np.abs(norm).max()
                        if ave else 0.0))
    bare = hd.RegionalFeatures(labels, hess, norm, None, ave)
    np.testing.assert_array_equal(bare["count"], g["count"])
    assert not bare["isum"].any() and not bare["imax"].any()


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


# Gaussian radii without a compile-time kernel: fewer taps than outputs per step, windows wider
# than the volume, the largest radius, a small radius that exceeds the large one along z; and
# NaN and infinities, which reach exactly the outputs whose windows hold them
@pytest.mark.parametrize("shape,s,trunc", [((9, 17, 70), (0.2, 0.2, 0.4, 0.3), 2.0),
                                           ((11, 23, 65), (1.0, 0.4, 1.4, 0.9), 2.0),
                                           ((20, 61, 129), (2.2, 1.1, 3.6, 1.8), 4.0),
                                           ((33, 70, 64), (1.4, 2.6, 2.3, 1.5), 3.0),
                                           ((7, 200, 90), (5.0, 1.0, 10.0, 3.3), 4.0),
                                           ((90, 5, 3), (1.5, 9.9, 8.2, 9.0), 4.0)])
@pytest.mark.parametrize("finite", [True, False])
def test_dog_of_any_radii(hd, shape, s, trunc, finite):
    rng = np.random.default_rng(21)
    norm = (rng.standard_normal(shape) * 0.3).astype(np.float32)
    if not finite:
        for v in (np.nan, np.inf, -np.inf):
            norm[tuple(int(rng.integers(n)) for n in shape)] = v
    hd.initGaussian3DKernel(*s, truncate=trunc)
    ref, _ = oracle.dog3d(norm, *s, truncate=trunc, gamma=1.0)
    np.testing.assert_array_equal(hd.DoG3DFilter(norm).cpu().numpy(), ref)


# normalization radii: windows shorter than a group of outputs, those with walks of their own,
# the walks of any radius on both sides of their column and LDS limits, larger ones; ragged
# strips, planes narrower and lower than a window; E and D with the same values
@pytest.mark.parametrize("rxy,rz", [(1, 2), (2, 4), (3, 7), (4, 1), (7, 3), (9, 9), (10, 6),
                                    (16, 11), (17, 5), (24, 24), (25, 10), (11, 25)])
@pytest.mark.parametrize("shape", [(3, 7, 5), (34, 41, 70), (9, 75, 193)])
def test_normalize_of_any_radii(hd, shape, rxy, rz):
    img = np.random.default_rng(rxy).integers(0, 65536, shape, dtype=np.uint16)
    want, e, d = oracle.normalize3d(img, 20000, rxy, rz, return_ed=True)
    np.testing.assert_array_equal(hd.Normalize3DFilter(img, 20000, rxy, rz).cpu().numpy(), want)
    n, ge, gd = hd.Normalize3DFilterWithBounds(img, 20000, rxy, rz)
    np.testing.assert_array_equal(n.cpu().numpy(), want)
    np.testing.assert_array_equal(ge.cpu().numpy(), e)
    np.testing.assert_array_equal(gd.cpu().numpy(), d)


# region numbers and counts across blocks, groups and chunks of the root counts, and a stack
# with more regions than the arrays of the call before hold, then one with fewer
def test_region_numbering_over_growing_and_shrinking_lists(hd):
    from hdog import HDoG
    fresh = HDoG(0)
    try:
        for shape, step in (((3, 40, 70), 3), ((40, 300, 1500), 2), ((5, 64, 64), 4)):
            pd = np.zeros(shape, np.uint8)
            pd[::step, ::step, 1::step] = 1
            # (steps of two keep neighbours apart, also where rows wrap)
            labels = fresh.CCL(pd)
            hess = np.zeros((6,) + shape, np.float32)
            g = fresh.RegionalFeatures(labels, hess, np.ones(shape, np.float32), None)
            at = np.flatnonzero(pd)
            lab = labels.cpu().numpy().ravel()
            roots = at[lab[at] == at]
            np.testing.assert_array_equal(g["label"][1:], roots.astype(np.uint32))
            np.testing.assert_array_equal(g["count"][1:], np.unique(lab[at], return_counts=True)[1])
    finally:
        fresh.close()


# region lists into page-locked memory (one kernel), pageable memory (short ones staged, long
# ones copied) and a mix of both: the same arrays, nothing written past the count
@pytest.mark.parametrize("shape,step", [((6, 40, 70), 4), ((40, 300, 1200), 3)])
def test_region_lists_in_any_host_memory(hd, shape, step):
    import torch
    from hdog import _capi as C
    pd = np.zeros(shape, np.uint8)
    pd[::step, ::step, 1::step] = 1
    rng = np.random.default_rng(31)
    g = hd.RegionalFeatures(hd.CCL(pd), rng.standard_normal((6,) + shape).astype(np.float32),
                            rng.standard_normal(shape).astype(np.float32), noise(shape, 1))
    n = len(g["label"])
    fields = (("label", torch.int32, "label"), ("size", torch.int16, "size16"),
              ("voxels", torch.int64, "count"), ("centroid_x", torch.float32, "cx"),
              ("structureness", torch.float32, "structureness"),
              ("intensity_sum", torch.int64, "isum"), ("intensity_max", torch.int16, "imax"))
    for kind in ("locked", "mixed", "odd"):
        reg = C.Regions()
        reg.capacity = n + 5
        held = []
        for k, (field, dt, _) in enumerate(fields):
            pin = kind != "mixed" or k % 2 == 0
            size = torch.empty(0, dtype=dt).element_size()
            skip = 1 if kind == "odd" else 0  # elements past the start: every alignment
            a = torch.full((n + 5 + skip,), 7, dtype=dt, pin_memory=pin)
            held.append(a[skip:])
            setattr(reg, field, a.data_ptr() + skip * size)
        hd._check(C.hdog_regions_download(hd._h, hd._stream(), C.ctypes.byref(reg)))
        assert reg.count == n
        for a, (_, _, key) in zip(held, fields):
            np.testing.assert_array_equal(a[:n].numpy().view(g[key].dtype), g[key], err_msg=key)
            assert (a[n:] == 7).all()


# region sums of noise with narrow Gaussians: more regions per work-group than its table holds
# (512 slots below sxy^2 sz = 3.2, 256 above), maximum and sum, against the materialized path
@pytest.mark.parametrize("sigmas", [(0.9, 0.7, 1.5, 1.2), (1.6, 1.25, 2.6, 2.0)])
@pytest.mark.parametrize("ave", [False, True])
def test_region_sums_beyond_the_table(hd, sigmas, ave):
    shape = (35, 70, 150)
    img = hd._dev(noise(shape, 12), __import__("torch").uint16)
    p = hd.make_params(shape, 3, 3, 0, *sigmas, truncate=3.0, is_ave_mode=ave)
    bufs = hd.alloc_intermediates(shape)
    hd.run_device(img, p, bufs)
    want = hd.RegionalFeatures(bufs["labels"], bufs["hess"], bufs["norm"], img, ave)
    hd.run_device(img, p)
    got = hd.download_regions()
    for k in ("label", "count", "isum", "imax", "centroid"):
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)
    # FP64 sums in another order, rounded once to FP32
    n = want["count"][:, None].astype(np.float64)
    big = max(float(bufs["hess"].abs().max()), float(bufs["norm"].abs().max()))
    for k in ("hsum", "norm"):
        a, b = (x[k].astype(np.float64).reshape(len(n), -1) for x in (got, want))
        assert np.all(np.abs(a - b) <= 1.2e-7 * np.abs(b) + 1e-12 * n * big), k


# soft response, gradient of the Hessian step for a given mask: tiles and strips with
# remainders, volumes smaller than a difference's reach, all voxels (the first one too), some,
# and one tile's corner only.  FP32 volumes and weights behind FP64 products of three
# elements: some 1e-5 of the largest gradient; the bound is that of the other gradient tests
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 2, 5), (17, 9, 65), (16, 8, 120), (33, 13, 190)])
@pytest.mark.parametrize("kind", ["all", "some", "corner"])
def test_soft_gradient_of_given_masks(hd, shape, kind):
    import types

    import soft_reference as ref
    import torch
    from hdog import soft
    s1, s2, tau = [1.6, 2.0, 2.0], [2.56, 3.2, 3.2], 0.05
    rad1, rad2 = soft.radii(s1), soft.radii(s2)
    rng = np.random.default_rng(shape[2])
    v = torch.from_numpy(rng.standard_normal(shape).astype(np.float32))
    t = torch.from_numpy((rng.random(shape) < 0.1).astype(np.uint8))
    m = {"all": np.ones(shape), "some": rng.random(shape) < 0.2, "corner": np.zeros(shape)}[kind]
    if kind == "corner":
        m[min(15, shape[0] - 1):18, min(7, shape[1] - 1):9, min(63, shape[2] - 1):66] = 1
    m = torch.from_numpy(m.astype(np.uint8))
    vd, td = v.to(hd.device), t.to(hd.device)
    dog = soft.run_forward(hd, vd, td, s1, s2, tau, rad1, rad2)[2]
    ctx = types.SimpleNamespace(saved_tensors=(vd, dog, m.to(hd.device), td), hd=hd, s1=s1[::-1],
                                s2=s2[::-1], r1=list(rad1)[::-1], r2=list(rad2)[::-1], gamma=1.0,
                                tau=tau, count=int(m.sum()), dev_sigma=torch.device("cpu"))
    gv, _, _, gtau = soft._SoftFn.backward(ctx, 1.0)[:4]
    v64 = v.double().requires_grad_()
    t64 = torch.tensor(tau, dtype=torch.float64, requires_grad=True)
    ref.forward(v64, torch.tensor(s1, dtype=torch.float64), torch.tensor(s2, dtype=torch.float64),
                t64, t, rad1, rad2, mask=m.bool())[0].backward()
    err = float((gv.cpu().double() - v64.grad).abs().max())
    assert err <= 2e-3 * float(v64.grad.abs().max())
    assert abs(float(gtau) - float(t64.grad)) <= 2e-3 * abs(float(t64.grad)) + 1e-6


# soft response, sigma gradients through each pair of passes: one compiled radius pair along x
# and y, two, none, more weights than lanes along z.  Bound of the other gradient tests, on the
# scale of the largest (FP32 volumes of unit size: some 1e-6 of it)
@pytest.mark.parametrize("s1,s2", [([1.6, 2.0, 2.0], [2.56, 3.2, 3.2]),
                                   ([2.0, 1.6, 2.0], [3.2, 2.56, 3.2]),
                                   ([1.1, 2.3, 0.9], [1.9, 3.1, 1.7]),
                                   ([8.0, 1.0, 1.2], [9.0, 1.6, 1.5])])
def test_soft_sigma_gradients_of_any_radii(hd, s1, s2):
    import soft_reference as ref
    import torch
    from hdog import soft
    shape = (19, 21, 70)
    rad1, rad2 = soft.radii(s1), soft.radii(s2)
    rng = np.random.default_rng(5)
    v = torch.from_numpy(rng.standard_normal(shape).astype(np.float32))
    t = torch.from_numpy((rng.random(shape) < 0.1).astype(np.uint8))
    a, b = (torch.tensor(s, dtype=torch.float64, requires_grad=True) for s in (s1, s2))
    tau = torch.tensor(0.05, dtype=torch.float64)
    vd, td = v.to(hd.device), t.to(hd.device)
    mask = soft.run_forward(hd, vd, td, s1, s2, 0.05, rad1, rad2)[3].cpu()
    soft.soft_loss(hd, vd, td, a, b, tau, rad1, rad2).backward()
    got = torch.cat([a.grad, b.grad])
    a2, b2 = (torch.tensor(s, dtype=torch.float64, requires_grad=True) for s in (s1, s2))
    ref.forward(v.double(), a2, b2, tau, t, rad1, rad2, mask=mask.bool())[0].backward()
    want = torch.cat([a2.grad, b2.grad])
    assert int(mask.sum()) > 100
    assert float((got - want).abs().max()) <= 2e-3 * float(want.abs().max())


def soft_normalize_by_hand(v, m, rxy, rz):
    """Windows of (value, lowest linear index) extremes, NaN skipped (none: +-inf, all ones),
    FP32 box sums in window order; x, then y, then z."""
    shape, N = v.shape, v.size
    mn, mx = (np.where(np.isnan(v), np.float32(f), v) for f in (np.inf, -np.inf))
    own = np.where(np.isnan(v), 0xFFFFFFFF, np.arange(N).reshape(shape)).astype(np.uint32)
    jn, jx = own.copy(), own.copy()
    for axis, r in ((2, rxy), (1, rxy), (0, rz)):
        taps = [np.clip(np.arange(shape[axis]) + t, 0, shape[axis] - 1) for t in range(-r, r + 1)]
        for f, j, best in ((mn, jn, np.less), (mx, jx, np.greater)):
            g, h = f.copy(), j.copy()
            for t in taps:
                a, k = np.take(f, t, axis), np.take(j, t, axis)
                take = best(a, g) | ((a == g) & (k < h))
                g, h = np.where(take, a, g), np.where(take, k, h)
            f[...], j[...] = g, h
    e, d = mn.copy(), mx.copy()
    for axis, r in ((2, rxy), (1, rxy), (0, rz)):
        k = np.float32(1) / np.float32(2 * r + 1)
        for f in (e, d):
            s = np.zeros_like(f)
            for t in range(-r, r + 1):
                s += np.take(f, np.clip(np.arange(shape[axis]) + t, 0, shape[axis] - 1), axis)
            f[...] = s * k
    n = np.where(v >= np.float32(m), (v - e) / (d - e), np.float32(0))
    return n, np.stack([e, d], -1), np.stack([jn, jx])


# soft normalization forward: windows shorter than a group of outputs, longer, the longest with
# a walk, beyond; lines shorter than the window, strips and segments with remainders; ties,
# signed zeros, infinities and windows of NaN only
@pytest.mark.parametrize("rxy,rz", [(1, 1), (2, 3), (3, 2), (4, 5), (10, 10), (23, 23), (24, 2),
                                    (5, 24)])
@pytest.mark.parametrize("kind", ["noise", "ties", "special"])
def test_soft_normalization_bitexact(hd, rxy, rz, kind):
    import torch
    from hdog import _capi as C
    shape = (37, 43, 133) if kind != "special" else (5, 9, 70)
    rng = np.random.default_rng(rxy)
    v = rng.standard_normal(shape).astype(np.float32)
    if kind == "ties":
        v = np.round(v)  # -0 and +0 among them
    if kind == "special":
        v[:, :, 0:30] = np.nan
        v[:, 3:, 40:60] = np.inf
        v[2:, :, 65:] = -np.inf
    D, H, W = shape
    vd = torch.from_numpy(v).to(hd.device)
    n = torch.empty_like(vd)
    ed = torch.empty(shape + (2,), dtype=torch.float32, device=hd.device)
    arg = torch.empty((2,) + shape, dtype=torch.int32, device=hd.device)
    p = C.ctypes.c_void_p
    hd._check(C.hdog_soft_normalize_forward(hd._h, hd._stream(), p(vd.data_ptr()), p(n.data_ptr()),
                                            p(ed.data_ptr()), p(arg.data_ptr()), -0.25, W, H, D,
                                            rxy, rz))
    with np.errstate(all="ignore"):
        wn, wed, warg = soft_normalize_by_hand(v, -0.25, rxy, rz)
    np.testing.assert_array_equal(arg.cpu().numpy().view(np.uint32), warg)
    np.testing.assert_array_equal(ed.cpu().numpy(), wed)
    np.testing.assert_array_equal(n.cpu().numpy(), wn)


# its adjoint at the same radii, against FP64 sums over the same indices: few extremes per
# patch, plateaus where every window has its own, NaN windows without one.  Bound: three FP32
# window sums of up to 47 terms and some hundred terms per target, of 6e-8 each, on the sum of
# the terms' magnitudes
@pytest.mark.parametrize("rxy,rz", [(1, 1), (2, 3), (3, 2), (4, 5), (10, 10), (23, 23), (24, 2)])
@pytest.mark.parametrize("shape,kind", [((37, 43, 133), "noise"), ((5, 70, 64), "plateau"),
                                        ((2, 3, 65), "noise"), ((9, 8, 70), "nan")])
def test_soft_normalization_adjoint(hd, rxy, rz, shape, kind):
    import torch
    from hdog import _capi as C
    rng = np.random.default_rng(rz)
    v = rng.standard_normal(shape).astype(np.float32)
    if kind == "plateau":
        v = np.maximum(v - 2.5, 0).astype(np.float32)
    D, H, W = shape
    N = v.size
    gn = rng.standard_normal(shape).astype(np.float32)
    e = rng.standard_normal(shape).astype(np.float32)
    ed = np.stack([e, e + 1 + rng.random(shape).astype(np.float32)], -1)
    vin = v.copy()
    if kind == "nan":
        vin[:, :, :50] = np.nan
    with np.errstate(all="ignore"):
        arg = soft_normalize_by_hand(vin, 0.0, rxy, rz)[2]
    dev = [torch.from_numpy(np.ascontiguousarray(a)).to(hd.device)
           for a in (v, ed, arg.view(np.int32), gn)]
    gv = torch.empty_like(dev[0])
    p = [C.ctypes.c_void_p(a.data_ptr()) for a in dev + [gv]]
    hd._check(C.hdog_soft_normalize_backward(hd._h, hd._stream(), *p, -0.25, W, H, D, rxy, rz))
    E, Dl, v64 = ed[..., 0].astype(np.float64), ed[..., 1].astype(np.float64), v.astype(np.float64)
    g = np.where(v >= np.float32(-0.25), gn, 0).astype(np.float64)
    want = g / (Dl - E)
    size = np.abs(want)
    for part, j in ((g * (v64 - Dl) / (Dl - E) ** 2, arg[0]), (-g * (v64 - E) / (Dl - E) ** 2, arg[1])):
        for out, x in ((want, part), (size, np.abs(part))):
            for axis, r in ((0, rz), (1, rxy), (2, rxy)):
                L = shape[axis]
                M = np.zeros((L, L))  # M[p, c]: taps of the window of c that land on p
                for t in range(-r, r + 1):
                    np.add.at(M, (np.clip(np.arange(L) + t, 0, L - 1), np.arange(L)), 1.0 / (2 * r + 1))
                x = np.moveaxis(np.tensordot(M, x, (1, axis)), 0, axis)
            ok = j.ravel() != 0xFFFFFFFF
            out += np.bincount(j.ravel()[ok].astype(np.int64), x.ravel()[ok], N).reshape(shape)
    assert np.all(np.abs(gv.cpu().numpy() - want) <= 4e-5 * size)


# fused y / z min/max: windows longer than the volume, just as long, ending and starting blocks
# of 21 slices on either side of the volume's end, several z segments with short ones
@pytest.mark.parametrize("depth", [2, 10, 11, 12, 21, 22, 31, 32, 33, 43, 74])
def test_minmax_zy_of_any_depth(hd, depth):
    img = noise((depth, 37, 70), depth)
    got = hd.Normalize3DFilter(img, 100, 10, 10)
    np.testing.assert_array_equal(got.cpu().numpy(), oracle.normalize3d(img, 100, 10, 10))


# one-pass y / z min/max of other radii: every group of four radii along y and each within
# one, both ends along z, just beyond them (two passes); tiles and segments with remainders
@pytest.mark.parametrize("shape", [(2, 5, 65), (43, 37, 70)])
@pytest.mark.parametrize("rxy,rz", [(4, 4), (4, 12), (5, 5), (6, 7), (7, 4), (8, 12), (9, 8), (13, 6),
                                    (14, 4), (15, 9), (16, 12), (17, 4), (8, 13), (3, 4), (4, 3)])
def test_minmax_zy_of_other_radii(hd, shape, rxy, rz):
    img = noise(shape, rxy + rz)
    got = hd.Normalize3DFilter(img, 100, rxy, rz)
    np.testing.assert_array_equal(got.cpu().numpy(), oracle.normalize3d(img, 100, rxy, rz))


# either side of the sizes where the row walkers take over from the walks of any radius
@pytest.mark.parametrize("shape", [(384, 24, 20), (385, 24, 20), (64, 448, 20), (64, 449, 20)])
def test_row_walkers_by_size(hd, shape):
    img = noise(shape, 2)
    got = hd.Normalize3DFilter(img, 100, 10, 10)
    np.testing.assert_array_equal(got.cpu().numpy(), oracle.normalize3d(img, 100, 10, 10))
    s = (2.0, 1.6, 3.2, 2.56)
    hd.initGaussian3DKernel(*s, truncate=4.0)
    dog = hd.DoG3DFilter(got)
    ref, _ = oracle.dog3d(got.cpu().numpy(), *s, truncate=4.0, gamma=1.0)
    np.testing.assert_array_equal(dog.cpu().numpy(), ref)


# widths whose rows and planes start anywhere in a cache line, on lines, and beyond one group of
# lanes; lines along z run over a whole plane's columns
@pytest.mark.parametrize("shape", [(5, 3, 21), (26, 11, 61), (23, 16, 80), (22, 30, 132)])
@pytest.mark.parametrize("rxy,rz", [(10, 10), (8, 4), (3, 2), (4, 25)])
def test_lines_along_z_of_any_width(hd, shape, rxy, rz):
    img = noise(shape, rz)
    got = hd.Normalize3DFilter(img, 100, rxy, rz)
    np.testing.assert_array_equal(got.cpu().numpy(), oracle.normalize3d(img, 100, rxy, rz))
    s = (2.0, 1.6, 3.2, 2.56) if rxy == 10 else (1.3, 2.3, 2.1, 3.7)
    hd.initGaussian3DKernel(*s, truncate=4.0)
    dog = hd.DoG3DFilter(got)
    ref, _ = oracle.dog3d(got.cpu().numpy(), *s, truncate=4.0, gamma=1.0)
    np.testing.assert_array_equal(dog.cpu().numpy(), ref)


# either side of the size where the z walk of radius 10 takes over: 2048 slices of 64 x 32 tiles
# and one more, and a plane of more tiles than that
@pytest.mark.parametrize("shape", [(1024, 33, 20), (683, 65, 20), (2, 33, 65), (3, 2160, 700)])
def test_minmax_zy_by_size(hd, shape):
    img = noise(shape, 4)
    got = hd.Normalize3DFilter(img, 100, 10, 10)
    np.testing.assert_array_equal(got.cpu().numpy(), oracle.normalize3d(img, 100, 10, 10))


# the z walk of radius 10 itself at the depths of test_minmax_zy_of_any_depth (1100 tiles: from
# two slices on)
@pytest.mark.parametrize("depth", [2, 10, 11, 12, 21, 22, 31, 32, 33, 43, 74])
def test_minmax_zy_walk_of_any_depth(hd, depth):
    img = noise((depth, 35200, 3), depth)
    got = hd.Normalize3DFilter(img, 100, 10, 10)
    np.testing.assert_array_equal(got.cpu().numpy(), oracle.normalize3d(img, 100, 10, 10))


# the row walkers and the z walk themselves, beyond the sizes that the walks of any radius take:
# odd columns, one and several segments with short last ones
@pytest.mark.parametrize("shape", [(400, 83, 130), (389, 201, 61), (130, 301, 401), (770, 43, 65)])
@pytest.mark.parametrize("sigmas,truncate", [((2.0, 1.6, 3.2, 2.56), 4.0), ((4.0, 1.8, 6.0, 2.7), 2.0)])
def test_row_walkers_bitexact(hd, shape, sigmas, truncate):
    img = noise(shape, 8)
    got = hd.Normalize3DFilter(img, 100, 10, 10)
    np.testing.assert_array_equal(got.cpu().numpy(), oracle.normalize3d(img, 100, 10, 10))
    hd.initGaussian3DKernel(*sigmas, truncate=truncate)
    dog = hd.DoG3DFilter(got)
    ref, _ = oracle.dog3d(got.cpu().numpy(), *sigmas, truncate=truncate, gamma=1.0)
    np.testing.assert_array_equal(dog.cpu().numpy(), ref)


# soft response with the row walker's weights of their own along y (more than 28 k rows)
def test_soft_sigma_gradients_by_the_row_walker(hd):
    import soft_reference as ref
    import torch
    from hdog import soft
    shape, s1, s2 = (40, 241, 190), [1.6, 2.0, 2.0], [2.56, 3.2, 3.2]
    rad1, rad2 = soft.radii(s1), soft.radii(s2)
    rng = np.random.default_rng(6)
    v = torch.from_numpy(rng.standard_normal(shape).astype(np.float32))
    t = torch.from_numpy((rng.random(shape) < 0.1).astype(np.uint8))
    a, b = (torch.tensor(s, dtype=torch.float64, requires_grad=True) for s in (s1, s2))
    tau = torch.tensor(0.05, dtype=torch.float64)
    vd, td = v.to(hd.device).requires_grad_(), t.to(hd.device)
    # (the loss's own mask: sigmas given as lists would be rounded to FP32 on the way)
    mask = soft.run_forward(hd, vd.detach(), td, a, b, 0.05, rad1, rad2)[3].cpu()
    soft.soft_loss(hd, vd, td, a, b, tau, rad1, rad2).backward()
    v64 = v.double().requires_grad_()
    a2, b2 = (torch.tensor(s, dtype=torch.float64, requires_grad=True) for s in (s1, s2))
    ref.forward(v64, a2, b2, tau, t, rad1, rad2, mask=mask.bool())[0].backward()
    got, want = torch.cat([a.grad, b.grad]), torch.cat([a2.grad, b2.grad])
    assert float((got - want).abs().max()) <= 2e-3 * float(want.abs().max())
    err = (vd.grad.cpu().double() - v64.grad).abs().max()
    assert float(err) <= 2e-3 * float(v64.grad.abs().max())


# records of the differentiable form, a slot per voxel: planes, rows, few columns, tiles cut
# along every axis (whose upper and lower neighbours' blocks then differ in size), and enough
# work-groups for four rows per wave.  FP32 volumes of unit size and chains of some fifty
# roundings (6e-8 each) on either side of a product of three elements: 1e-4 of the largest
# gradient
@pytest.mark.parametrize("shape", [(1, 200, 500), (2, 200, 500), (3, 2, 700), (35, 61, 3),
                                   (18, 43, 131), (3, 1030, 1100)])
def test_soft_gradient_by_blocks_of_any_shape(hd, shape):
    import types

    import soft_reference as ref
    import torch
    from hdog import soft
    s1, s2, tau = [1.6, 2.0, 2.0], [2.56, 3.2, 3.2], 0.05
    rad1, rad2 = soft.radii(s1), soft.radii(s2)
    g = torch.Generator().manual_seed(shape[2])
    v = torch.randn(shape, generator=g)
    t = (torch.rand(shape, generator=g) < 0.1).to(torch.uint8)
    m = (torch.rand(shape, generator=g) < 0.2).to(torch.uint8)
    vd, td = v.to(hd.device), t.to(hd.device)
    dog = soft.run_forward(hd, vd, td, s1, s2, tau, rad1, rad2)[2]
    ctx = types.SimpleNamespace(saved_tensors=(vd, dog, m.to(hd.device), td), hd=hd, s1=s1[::-1],
                                s2=s2[::-1], r1=list(rad1)[::-1], r2=list(rad2)[::-1], gamma=1.0,
                                tau=tau, count=int(m.sum()), dev_sigma=torch.device("cpu"))
    gv, _, _, gtau = soft._SoftFn.backward(ctx, 1.0)[:4]
    v64 = v.double().requires_grad_()
    t64 = torch.tensor(tau, dtype=torch.float64, requires_grad=True)
    ref.forward(v64, torch.tensor(s1, dtype=torch.float64), torch.tensor(s2, dtype=torch.float64),
                t64, t, rad1, rad2, mask=m.bool())[0].backward()
    err = float((gv.cpu().double() - v64.grad).abs().max())
    most = float(v64.grad.abs().max())  # 0 for a plane, whose differences along z are
    print(shape, "error", err, "largest gradient", most, flush=True)
    assert err <= 1e-4 * most
    assert abs(float(gtau) - float(t64.grad)) <= 1e-4 * abs(float(t64.grad)) + 1e-6


def test_soft_mask_and_loss_by_blocks_of_any_shape(hd):
    # the forward pass: the mask is the Hessian stage's of the same DoG volume, the count its
    # number of voxels, and the loss the FP64 one of its elements
    import torch
    from hdog import soft
    s1, s2, tau = [1.6, 2.0, 2.0], [2.56, 3.2, 3.2], 1e-3
    for shape in [(2, 200, 500), (3, 2, 700), (35, 61, 3), (18, 43, 131), (3, 1030, 1100)]:
        g = torch.Generator().manual_seed(shape[1])
        v = torch.randn(shape, generator=g).to(hd.device)
        t = (torch.rand(shape, generator=g) < 0.1).to(torch.uint8).to(hd.device)
        loss, count, dog, mask = soft.run_forward(hd, v, t, s1, s2, tau, soft.radii(s1),
                                                  soft.radii(s2))
        hess, pd = hd.HessianPositiveDefiniteWithElement(dog)
        assert torch.equal(mask.view(torch.uint8), pd.view(torch.uint8)), shape
        on = pd.view(torch.uint8).bool()
        assert count == int(on.sum()) > 0
        xx, xy, xz, yy, yz, zz = (hess[k][on].double() for k in range(6))
        u = -(xx * yy * zz + 2 * xy * yz * xz - xx * yz * yz - yy * xz * xz - zz * xy * xy) / tau
        want = float((torch.nn.functional.softplus(u) - t[on].bool() * u).sum() / count)
        assert abs(float(loss) - want) <= 1e-9 * abs(want), shape


def records_equal_given_labels(hd, img, p, bufs, ave):
    """The regions of the records-only pass, against those of the materialized volumes' labels
    (a fold of its own).  Sums: FP64 in another order, rounded once to FP32."""
    want = hd.RegionalFeatures(bufs["labels"], bufs["hess"], bufs["norm"], img, ave)
    hd.run_device(img, p)
    got = hd.download_regions()
    assert len(want["label"]) > 1000
    for k in ("label", "count", "isum", "imax", "centroid"):
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)
    n = want["count"][:, None].astype(np.float64)
    big = max(float(bufs["hess"].abs().max()), float(bufs["norm"].abs().max()))
    for k in ("hsum", "norm"):
        a, b = (x[k].astype(np.float64).reshape(len(n), -1) for x in (got, want))
        assert np.all(np.abs(a - b) <= 1.2e-7 * np.abs(b) + 1e-12 * n * big), k


# one group of waves for a work-group's tiles (above 1024 work-groups) and four, with either
# table size
@pytest.mark.parametrize("shape", [(3, 1040, 1040), (3, 1040, 960)])
@pytest.mark.parametrize("sigmas", [(0.9, 0.7, 1.5, 1.2), (1.6, 1.25, 2.6, 2.0)])
@pytest.mark.parametrize("ave", [False, True])
def test_region_sums_by_work_groups(hd, shape, sigmas, ave):
    img = hd._dev(noise(shape, 12), __import__("torch").uint16)
    p = hd.make_params(shape, 3, 3, 0, *sigmas, truncate=3.0, is_ave_mode=ave)
    bufs = hd.alloc_intermediates(shape)
    hd.run_device(img, p, bufs)
    records_equal_given_labels(hd, img, p, bufs, ave)


# records of walks over one to four Hessian tiles, two rows per wave and four: all six elements
@pytest.mark.parametrize("shape", [(70, 40, 70), (33, 640, 700), (49, 1500, 1600)])
def test_records_walks_give_the_elements(hd, shape):
    blobs = synth.blob_table(shape, shape[0] * shape[1] * shape[2] // 20000, 11)
    img = hd.synth_volume(shape, blobs, 11, 200.0, 200.0, 20.0)
    p = hd.make_params(shape, 10, 10, 0, 1.2, 1.0, 2.0, 1.6, 3.0)
    bufs = hd.alloc_intermediates(shape)
    hd.run_device(img, p, bufs)
    records_equal_given_labels(hd, img, p, bufs, False)


# 16-bit storage at radii without kernels of their own: the normalized stack is the FP32 one
# rounded; the DoG of that stack, formed in FP32, equals the oracle's where it stays FP32, and
# is at most a unit in the last place from it where it is rounded to 16 bits (the product with
# the scale may be rounded on the way or not)
@pytest.mark.parametrize("form,dtype,digits", [("fp16", "float16", 10), ("bf16", "bfloat16", 7),
                                               ("fp16_dog32", "float16", 0),
                                               ("bf16_dog32", "bfloat16", 0)])
@pytest.mark.parametrize("rxy,rz,s", [(8, 4, (2.2, 1.1, 3.6, 1.8)), (3, 2, (0.3, 0.2, 0.6, 0.5)),
                                      (9, 25, (8.1, 1.3, 9.6, 2.1))])
def test_16_bit_storage_at_any_radii(hd, form, dtype, digits, rxy, rz, s):
    import torch
    dtype = getattr(torch, dtype)
    for shape in ((34, 41, 70), (9, 75, 193)):
        img = hd._dev(noise(shape, 5), torch.uint16)
        norm = hd.Normalize3DFilter(img, 100, rxy, rz)
        p = hd.make_params(shape, rxy, rz, 100, *s, truncate=4.0, precision=form)
        bufs = hd.alloc_intermediates(shape, form)
        hd.run_device(img, p, bufs)
        assert torch.equal(bufs["norm"], norm.to(dtype))
        want = torch.from_numpy(oracle.dog3d(bufs["norm"].float().cpu().numpy(), *s, truncate=4.0,
                                             gamma=1.0)[0])
        got = bufs["dog"].cpu()
        if not digits:
            assert got.dtype == torch.float32 and torch.equal(got, want)
        else:
            assert got.dtype == dtype
            want = want.to(dtype).double()
            least = 2.0 ** -24 if dtype == torch.float16 else 0.0
            assert bool(((got.double() - want).abs() <= want.abs() * 2.0 ** -digits + least).all())


# lines of at most eight slices, held in registers, and one more; windows within the line, at its
# ends, past both, longer than a walk takes; E and D; values that a tap outside the line, or one
# too many at its end, would change
@pytest.mark.parametrize("depth", [1, 2, 3, 7, 8, 9])
@pytest.mark.parametrize("rxy,rz", [(3, 1), (8, 5), (10, 10), (16, 2), (4, 24), (25, 3), (2, 30)])
def test_normalize_of_few_slices(hd, depth, rxy, rz):
    for shape in ((depth, 9, 257), (depth, 37, 6)):
        img = noise(shape, 100 * depth + rz)
        img[:, 2:4, 3:5] = 65535
        want, e, d = oracle.normalize3d(img, 300, rxy, rz, return_ed=True)
        got, ge, gd = hd.Normalize3DFilterWithBounds(img, 300, rxy, rz)
        for a, b, name in ((got, want, "norm"), (ge, e, "E"), (gd, d, "D")):
            np.testing.assert_array_equal(a.cpu().numpy(), b, err_msg=name)


@pytest.mark.parametrize("depth", [1, 2, 5, 8, 9])
@pytest.mark.parametrize("s,trunc", [((1.3, 0.3, 2.1, 0.5), 2.0), ((2.2, 1.1, 3.6, 1.8), 4.0),
                                     ((1.0, 7.9, 1.5, 9.9), 4.0)])
@pytest.mark.parametrize("finite", [True, False])
def test_dog_of_few_slices(hd, depth, s, trunc, finite):
    for shape in ((depth, 9, 257), (depth, 37, 6)):
        rng = np.random.default_rng(depth)
        norm = (rng.standard_normal(shape) * 0.3).astype(np.float32)
        if not finite:
            for v in (np.nan, np.inf, -np.inf):
                norm[tuple(int(rng.integers(n)) for n in shape)] = v
        hd.initGaussian3DKernel(*s, truncate=trunc)
        ref, _ = oracle.dog3d(norm, *s, truncate=trunc, gamma=1.0)
        np.testing.assert_array_equal(hd.DoG3DFilter(norm).cpu().numpy(), ref)


# soft normalization of a few slices: windows past both ends of a line, ties among the voxels that
# they repeat; either side of the depth that has passes of its own
@pytest.mark.parametrize("depth", [1, 2, 8, 9])
@pytest.mark.parametrize("rxy,rz", [(3, 2), (8, 5), (4, 23)])
def test_soft_normalization_of_few_slices(hd, depth, rxy, rz):
    import torch
    from hdog import _capi as C
    for shape in ((depth, 13, 133), (depth, 37, 6)):
        v = np.round(np.random.default_rng(rz).standard_normal(shape) * 2).astype(np.float32)
        D, H, W = shape
        vd = torch.from_numpy(v).to(hd.device)
        n = torch.empty_like(vd)
        ed = torch.empty(shape + (2,), dtype=torch.float32, device=hd.device)
        arg = torch.empty((2,) + shape, dtype=torch.int32, device=hd.device)
        p = C.ctypes.c_void_p
        hd._check(C.hdog_soft_normalize_forward(hd._h, hd._stream(), p(vd.data_ptr()),
                                                p(n.data_ptr()), p(ed.data_ptr()),
                                                p(arg.data_ptr()), -0.25, W, H, D, rxy, rz))
        with np.errstate(all="ignore"):
            wn, wed, warg = soft_normalize_by_hand(v, -0.25, rxy, rz)
        np.testing.assert_array_equal(arg.cpu().numpy().view(np.uint32), warg)
        np.testing.assert_array_equal(ed.cpu().numpy(), wed)
        np.testing.assert_array_equal(n.cpu().numpy(), wn)


# planes of few rows: either side of the row count where the walk along x and y begins (2 H = 3 r)
@pytest.mark.parametrize("shape,r", [((6, 11, 200), 8), ((6, 12, 200), 8), ((5, 35, 130), 24),
                                     ((5, 36, 130), 24), ((400, 1, 70), 3), ((7, 4, 300), 3)])
def test_normalize_of_few_rows(hd, shape, r):
    img = noise(shape, r)
    got, ge, gd = hd.Normalize3DFilterWithBounds(img, 300, r, 4)
    want, e, d = oracle.normalize3d(img, 300, r, 4, return_ed=True)
    for a, b, name in ((got, want, "norm"), (ge, e, "E"), (gd, d, "D")):
        np.testing.assert_array_equal(a.cpu().numpy(), b, err_msg=name)


# Gaussians longer than the plane has rows, whose taps past it are left out but for one
@pytest.mark.parametrize("rows", [1, 3, 8, 31, 32, 33])
@pytest.mark.parametrize("finite", [True, False])
def test_dog_of_few_rows(hd, rows, finite):
    rng = np.random.default_rng(rows)
    norm = (rng.standard_normal((11, rows, 130)) * 0.3).astype(np.float32)
    if not finite:
        for v in (np.nan, np.inf, -np.inf):
            norm[tuple(int(rng.integers(n)) for n in norm.shape)] = v
    for s in ((7.9, 1.1, 9.9, 1.8), (2.0, 2.0, 3.2, 3.2)):
        hd.initGaussian3DKernel(*s, truncate=4.0)
        ref, _ = oracle.dog3d(norm, *s, truncate=4.0, gamma=1.0)
        np.testing.assert_array_equal(hd.DoG3DFilter(norm).cpu().numpy(), ref)
