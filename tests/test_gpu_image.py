"""Image calls (``rasterize`` / ``rasterize_views``, eager) against the op they
no longer go through: the same pixels from tight rectangles and 16-pixel tiles,
gradients equal up to the order of their sums."""

from __future__ import annotations

import math

import pytest
import torch

from gaussian_splats_hip import scenes
from gaussian_splats_hip.kernels.rasterize.image import image_tile
from gaussian_splats_hip.kernels.rasterize.interface import rasterize_outputs
from gaussian_splats_hip.kernels.rasterize.views import camera_tensors, rasterize_views_outputs
from gaussian_splats_hip.splats import GaussianSplat, rasterize, rasterize_views
from gaussian_splats_hip.splats.camera import host_extrinsics

pytestmark = pytest.mark.gpu

PARAMS = ("mean", "rotation", "scale", "opacity", "color")


def _needles(n, size):
    """Gaussians from 2 to ~e^7 times longer than wide, in every direction
    (conditions of the 2-D covariance up to ~1e6, on both sides of the line
    above which the reference's extent is kept)."""
    scene = scenes.edge_case_scene(n=n, sh_degree=1, image_size=size, seed=5)
    g = torch.Generator().manual_seed(9)
    scene.scale[:, 1:] = scene.scale[:, :1] - 7 * torch.rand(n, 1, generator=g)
    scene.scale[: n // 4, 0] += 3
    return scene


def _op(scene, params, cam, tile, mode):
    r, t = host_extrinsics(cam)
    (fx, fy), (cx, cy), (w, h) = cam.focal_length, cam.principal_point, cam.image_size
    return rasterize_outputs(*params, r, t, float(fx), float(fy), float(cx), float(cy), w, h, tile,
                             0.999, scene.near, scene.far, mode, 0.95)[0]


def _same_gradients(a, b):
    """Two sums of the same float32 terms in other orders: two runs of one path
    (atomic adds) differ by up to 1e-5 of a gradient's norm; one entry missing
    at one tile would show as 1e-3 or more in scenes of this size."""
    for name, x, y in zip(PARAMS, a, b):
        assert (x - y).norm() <= 1e-4 * y.norm(), name


@pytest.mark.parametrize("mode", ["gaussian", "ellipsoid"])
@pytest.mark.parametrize("tile", [4, 8, 16, 32])
@pytest.mark.parametrize("kind,size", [("edge", (96, 80)), ("edge", (17, 1)), ("needle", (333, 207)),
                                       ("cloud", (1111, 1043)), ("cloud", (1100, 1030)),
                                       ("small", (1111, 1043)), ("wide", (4097, 17))])
def test_image_equals_op(kind, size, tile, mode, device):
    if kind == "needle":
        scene = _needles(3000, size)
    elif kind == "cloud":  # above 4096 tiles of 16 pixels: whole tiles per wave
        scene = scenes.edge_case_scene(n=20000, sh_degree=0, image_size=size, seed=6)
    elif kind == "small":  # lists of a small scene, shared by 2 x 2 tiles
        scene = scenes.edge_case_scene(n=2000, image_size=size, seed=7)
    elif kind == "wide":  # above 4096 pixels: tiles of 32
        scene = scenes.edge_case_scene(n=3000, image_size=size, seed=7)
        scene.mean[:, 1] *= 0.01
    else:
        scene = scenes.edge_case_scene(n=1000, image_size=size)
    scene = scene.to(device)
    cam = scene.cameras[0]
    splats = GaussianSplat.from_tensors(*scene.params())
    leaves = [p.detach().clone().requires_grad_(True) for p in scene.params()]
    image = rasterize(splats, cam, tile, near=scene.near, far=scene.far, rendering_mode=mode)
    if kind in ("small", "wide") and mode == "gaussian":
        lists = image.grad_fn.saved_tensors[8].shape[0]
        assert lists == {"small": 35 * 33, "wide": 129}[kind]
    expected = _op(scene, leaves, cam, tile, mode)
    if mode == "ellipsoid":
        # A pixel within rounding of the ellipse's edge may lie outside the
        # reference's rectangle for one tile size and inside for another.
        same = (image == expected).all(-1).float().mean()
        assert same > 0.9995
        with pytest.raises(AssertionError):
            image.sum().backward()
        return
    with torch.no_grad():
        assert torch.equal(image, rasterize(splats, cam, tile, near=scene.near, far=scene.far))
    if kind == "needle" and tile != 16:
        # The walk's own overlap test evaluates a needle's form at the edges of
        # a tile's rectangle, whose rounding depends on the tile: an entry of
        # alpha at the cut, 1/255, may be skipped with one tile size and blended
        # with another, in the op as here.  (Colours are below 2.)
        differs = (image != expected).any(-1)
        assert differs.float().mean() < 1e-3
        assert (image - expected).abs().max() < 4 / 255
        expected = _op(scene, leaves, cam, 16, mode)
    assert torch.equal(image, expected)
    weight = torch.linspace(-1, 1, image.numel(), device=device).reshape(image.shape)
    (image * weight).sum().backward()
    (expected * weight).sum().backward()
    grads = [getattr(splats, n).grad for n in PARAMS]
    if kind != "needle":
        _same_gradients(grads, [p.grad for p in leaves])
        return
    # A needle's chain back through its covariance amplifies the rounding of
    # the sums over pixels by the condition number: two runs of the op itself
    # differ by up to 3e-4 of the means' norm, as their atomic adds fall.  The
    # differences are held to 8 times the largest of those between the op's four
    # tile sizes (four orders of the sums, six pairs; in 24 runs no difference
    # was above 1.8 times it.  A single pair, of tiles of 4 and 32 pixels, can
    # agree by chance to a ninth of another pair's difference).
    orders = []
    for other in (4, 8, 16, 32):
        again = [p.detach().clone().requires_grad_(True) for p in scene.params()]
        (_op(scene, again, cam, other, mode) * weight).sum().backward()
        orders.append([p.grad for p in again])
    for i, (name, x, y) in enumerate(zip(PARAMS, grads, (p.grad for p in leaves))):
        spread = max((orders[a][i] - orders[b][i]).norm() for a in range(4) for b in range(a))
        assert (x - y).norm() <= 8 * spread + 1e-6 * y.norm(), name


@pytest.mark.parametrize("n,focal", [(60_000, 1600.0), (120_000, 2400.0)])
def test_image_long_lists(n, focal, device):
    """Lists above 8192 entries: four waves per tile and a backward in segments
    (at the longer focal length on more than 4096 tiles with work), against the
    op's checkpointed walk; a second backward through one graph re-zeroes its
    accumulator."""
    scene = scenes.config4(n=n, focal=focal)
    scene = scene.to(device)
    cam = scene.cameras[0]
    splats = GaussianSplat.from_tensors(*scene.params())
    leaves = [p.detach().clone().requires_grad_(True) for p in scene.params()]
    image = rasterize(splats, cam, 16)
    ranges, walk_records = (image.grad_fn.saved_tensors[i] for i in (8, -1))
    lengths = ranges[:, 1] - ranges[:, 0]
    assert lengths.max() > 8192 and walk_records is not None
    assert (4 * (lengths > 0).sum() >= 4096) == (focal == 2400.0)
    expected = _op(scene, leaves, cam, 16, "gaussian")
    # The op's checkpoints cut a pixel's colour into partial sums at list
    # positions: up to 64 roundings of a sum below 4.
    assert (image - expected).abs().max() < 64 * 4 * 2.0 ** -24
    with torch.no_grad():
        assert (image - rasterize(splats, cam, 16)).abs().max() < 64 * 4 * 2.0 ** -24
    loss = (image - scene.target).square().mean()
    first = torch.autograd.grad(loss, [getattr(splats, n) for n in PARAMS], retain_graph=True)
    second = torch.autograd.grad(loss, [getattr(splats, n) for n in PARAMS])
    want = torch.autograd.grad((expected - scene.target).square().mean(), leaves)
    _same_gradients(first, want)
    _same_gradients(second, want)


@pytest.mark.parametrize("size,n", [(48, 4000), (24, 700), (24, 65), (24, 129), (736, 2500)])
def test_image_walk_segments(size, n, device):
    """Faint Gaussians that each cover the image: every pixel walks the whole
    list, through the fixed cuts of its walk records, and some pixels saturate on
    the way."""
    g = torch.Generator().manual_seed(n)
    scene = scenes.edge_case_scene(n=n, sh_degree=1, image_size=(size, size), seed=3)
    scene.mean[:, :2] = torch.randn(n, 2, generator=g) * 0.3
    scene.mean[:, 2] = -(torch.rand(n, generator=g) + 3)
    scene.scale[:] = torch.rand(n, 3, generator=g) * 0.5 + 0.5
    scene.opacity[:] = torch.randn(n, 1, generator=g) * 0.3 - 5
    scene.opacity[n // 2::97] = 1.0
    scene.mean[n // 2::97, :2] = torch.tensor([1.0, 0.5])
    scene.scale[n // 2::97] = -1.0
    scene = scene.to(device)
    cam = scene.cameras[0]
    splats = GaussianSplat.from_tensors(*scene.params())
    leaves = [p.detach().clone().requires_grad_(True) for p in scene.params()]
    image = rasterize(splats, cam, near=scene.near, far=scene.far)
    expected = _op(scene, leaves, cam, 16, "gaussian")
    assert torch.equal(image, expected)
    weight = torch.linspace(-1, 1, image.numel(), device=device).reshape(image.shape)
    loss = (image * weight).sum()
    first = torch.autograd.grad(loss, [getattr(splats, p) for p in PARAMS], retain_graph=True)
    second = torch.autograd.grad(loss, [getattr(splats, p) for p in PARAMS])
    (expected * weight).sum().backward()
    _same_gradients(first, [p.grad for p in leaves])
    _same_gradients(second, [p.grad for p in leaves])


def _points(n, size, spread, background=0):
    """Faint Gaussians of half a pixel in ``spread`` pixels around the middle: each
    pixel takes few entries of its tile's long list.  Ten wide opaque ones lie
    across them halfway into the list, a little below the middle, so the tiles'
    quarters walk to different depths.  ``background``: of the Gaussians, those
    that lie all over the image instead, faint too."""
    scene = scenes.edge_case_scene(n=n, sh_degree=1, image_size=size, seed=8)
    m = n - background
    mean, scale = scene.mean[m:].clone(), scene.scale[m:].clone()
    g = torch.Generator().manual_seed(n)
    pixel = 5 / (0.75 * size[0])
    scene.mean[:, :2] = torch.randn(n, 2, generator=g) * spread * pixel
    scene.mean[:, 2] = -(torch.rand(n, generator=g) * 0.1 + 5)
    scene.scale[:] = math.log(0.5 * pixel) + torch.tensor([-0.5, 0.5, 0.0])
    scene.opacity[:] = torch.randn(n, 1, generator=g) * 0.3 - 4.5
    scene.mean[m:], scene.scale[m:] = mean, scale
    scene.mean[-10:] = torch.tensor([0.0, -2 * pixel, -5.05])
    scene.rotation[-10:] = torch.tensor([1.0, 0.0, 0.0, 0.0])
    scene.scale[-10:] = torch.log(torch.tensor([60.0, 6.0, 1.0]) * pixel)
    scene.opacity[-10:] = 6.0
    return scene


@pytest.mark.parametrize("size,n,spread,background,shared", [
    ((24, 24), 24_000, 2.0, 0, False), ((40, 24), 90_000, 3.0, 0, False),
    ((1111, 1043), 70_000, 8.0, 4000, True), ((4096, 1712), 20_000, 8.0, 0, False),
    ((4096, 2816), 20_000, 8.0, 0, True)])
def test_image_long_walks(size, n, spread, background, shared, device):
    """Walks that drop records and double their spacing, in images of 11, 7 and 3
    records per tile, with a list per tile and with lists shared by 2 x 2."""
    scene = _points(n, size, spread, background).to(device)
    cam = scene.cameras[0]
    splats = GaussianSplat.from_tensors(*scene.params())
    leaves = [p.detach().clone().requires_grad_(True) for p in scene.params()]
    image = rasterize(splats, cam, near=scene.near, far=scene.far)
    walk_records = image.grad_fn.saved_tensors[-1]
    tiles = -(-size[0] // 16) * -(-size[1] // 16)
    records = {True: 11, False: 7 if tiles < 42_130 else 3}[tiles < 26_810]
    padded = walk_records.numel() // (records * 4096 + 32)
    assert walk_records.numel() == padded * (records * 4096 + 32) and padded >= tiles
    assert (image.grad_fn.saved_tensors[8].shape[0] < tiles) == shared
    keys = walk_records[padded * records * 4096:].view(torch.int32).reshape(padded, 4, 2)
    expected = _op(scene, leaves, cam, 16, "gaussian")
    if background:  # the op's checkpoints cut a pixel's colour into partial sums (see below)
        assert (image - expected).abs().max() < 64 * 4 * 2.0 ** -24
    else:
        assert torch.equal(image, expected)
    # Without a symmetry that the wide Gaussians' rotation gradients, odd moments
    # over their pixels, would cancel by.
    weight = torch.randn(image.shape, device=device, generator=torch.Generator(device).manual_seed(n))
    (image * weight).sum().backward()
    (expected * weight).sum().backward()
    _same_gradients([getattr(splats, n).grad for n in PARAMS], [p.grad for p in leaves])
    # The spacing has doubled, and not equally often in a tile's quarters.
    doubled = keys[..., 1]
    assert doubled.max() >= 1 and (doubled.amax(1) != doubled.amin(1)).any()


def test_views_image_equals_op(device):
    scene = scenes.config5(seed=2, n=4000, views=5, size=90, focal=110).to(device)
    splats = GaussianSplat.from_tensors(*scene.params())
    leaves = [p.detach().clone().requires_grad_(True) for p in scene.params()]
    images = rasterize_views(splats, scene.cameras, tile_size=8)
    r, t, k, w, h = camera_tensors(scene.cameras)
    expected = rasterize_views_outputs(*leaves, r, t, k, w, h, 8, 0.999, 0.2, 100.0, "gaussian",
                                       0.95)[0]
    assert torch.equal(images, expected)
    (images - scene.target).abs().mean().backward()
    (expected - scene.target).abs().mean().backward()
    _same_gradients([getattr(splats, n).grad for n in PARAMS], [p.grad for p in leaves])


@pytest.mark.parametrize("size,n", [((96, 80), 1000), ((1111, 1043), 30_000), ((4097, 17), 3000)])
@pytest.mark.parametrize("path", ["image", "op4", "op16"])
def test_gradient_that_is_not_finite(path, size, n, device):
    """An infinite gradient at one pixel reaches the Gaussians that the pixel took
    and no others, whose gradients are those without it."""
    scene = scenes.edge_case_scene(n=n, image_size=size, seed=7)
    scene.mean[:, 1] *= size[1] / size[0]
    scene.color[:, 0] += 3  # no channel clamped at 0, which has no gradient
    scene = scene.to(device)
    cam = scene.cameras[0]
    if path == "image":
        splats = GaussianSplat.from_tensors(*scene.params())
        params = [getattr(splats, p) for p in PARAMS]
        image = rasterize(splats, cam, near=scene.near, far=scene.far)
    else:
        params = [p.detach().clone().requires_grad_(True) for p in scene.params()]
        image = _op(scene, params, cam, int(path[2:]), "gaussian")

    def gradients(weight):
        return torch.autograd.grad(image, params, weight, retain_graph=True)

    weight = torch.randn(image.shape, device=device, generator=torch.Generator(device).manual_seed(2))
    y, x = size[1] // 2, size[0] // 2
    weight[y, x] = 0
    want = gradients(weight)
    alone = torch.zeros_like(weight)
    alone[y, x] = 1
    took = gradients(alone)[4].flatten(1).any(1)
    assert 0 < took.sum() < n
    weight[y, x] = torch.tensor([float("inf"), 1.0, -1.0])
    got = gradients(weight)
    assert not got[4][took].isfinite().all()
    _same_gradients([g[~took] for g in got], [w[~took] for w in want])


def test_image_is_no_view(device):
    """One camera's image is a tensor of its own, as the op's output is: it can
    be detached in place, and its gradient reaches the backward as it is."""
    scene = scenes.edge_case_scene(n=200, image_size=(48, 32)).to(device)
    cam = scene.cameras[0]
    splats = GaussianSplat.from_tensors(*scene.params())
    image = rasterize(splats, cam, near=scene.near, far=scene.far)
    assert image.shape == (32, 48, 3) and not image._is_view()
    assert image.grad_fn.name() == "_RenderImageBackward"
    image.detach_()
    with torch.no_grad():
        image = rasterize(splats, cam, near=scene.near, far=scene.far)
    assert image.shape == (32, 48, 3) and not image._is_view()
    image.detach_()
    assert rasterize_views(splats, [cam]).shape == (1, 32, 48, 3)


def test_views_of_32_pixel_tiles(device):
    """A mosaic above 256 tiles of 16 pixels per axis: tiles of 32, each walked
    whole by one wave (the wide image's, above, in quarters)."""
    scene = scenes.config5(seed=2, n=2000, views=36, size=704, focal=880).to(device)
    splats = GaussianSplat.from_tensors(*scene.params())
    leaves = [p.detach().clone().requires_grad_(True) for p in scene.params()]
    images = rasterize_views(splats, scene.cameras)
    ranges, order = (images.grad_fn.saved_tensors[i] for i in (8, -2))
    assert ranges.shape[0] == (6 * 22) ** 2 and not (order[order >= 0] & 0x7F).any()
    r, t, k, w, h = camera_tensors(scene.cameras)
    expected = rasterize_views_outputs(*leaves, r, t, k, w, h, 32, 0.999, 0.2, 100.0, "gaussian",
                                       0.95)[0]
    assert torch.equal(images, expected)
    weight = torch.linspace(-1, 1, images[0].numel(), device=device).reshape(images[0].shape)
    (images * weight).mean().backward()
    (expected * weight).mean().backward()
    _same_gradients([getattr(splats, n).grad for n in PARAMS], [p.grad for p in leaves])


def test_no_gaussians_and_nothing_visible(device):
    scene = scenes.edge_case_scene(n=40, image_size=(50, 30)).to(device)
    cam = scene.cameras[0]
    for params in (tuple(p[:0] for p in scene.params()),
                   (scene.mean * torch.tensor([1.0, 1.0, -1.0], device=device), *scene.params()[1:])):
        splats = GaussianSplat.from_tensors(*params)
        image = rasterize(splats, cam, near=scene.near, far=scene.far)
        assert image.shape == (30, 50, 3) and not image.any()
        image.sum().backward()
        assert all(not getattr(splats, n).grad.any() for n in PARAMS)


def test_saved_tensor_hooks(device):
    """The forward's tensors go through saved-tensor hooks (here to the host
    and back) like any autograd function's."""
    scene = scenes.edge_case_scene(n=500, image_size=(64, 48)).to(device)
    cam = scene.cameras[0]
    grads = []
    for hooked in (False, True):
        splats = GaussianSplat.from_tensors(*(p.clone() for p in scene.params()))
        if hooked:
            with torch.autograd.graph.save_on_cpu():
                image = rasterize(splats, cam, near=scene.near, far=scene.far)
        else:
            image = rasterize(splats, cam, near=scene.near, far=scene.far)
        image.square().sum().backward()
        grads.append([getattr(splats, n).grad for n in PARAMS])
    _same_gradients(*grads)


def test_backward_frees_the_walk(device):
    """A backward that does not retain the graph frees what the forward kept for
    it (here 54 MB of walk records), also while the image is held."""
    scene = scenes.edge_case_scene(n=500, image_size=(640, 480)).to(device)
    splats = GaussianSplat.from_tensors(*scene.params())
    held = []
    for _ in range(2):  # the first call also makes the gradients
        image = None
        before = torch.cuda.memory_allocated()
        image = rasterize(splats, scene.cameras[0], near=scene.near, far=scene.far)
        kept = torch.cuda.memory_allocated() - before
        image.sum().backward()
        held.append(torch.cuda.memory_allocated() - before)
    assert kept > 50 << 20
    assert held[1] <= image.numel() * 4 + (1 << 20)


def test_image_far_away(device):
    """Small Gaussians on few tiles of a large image: a list per tile after all,
    in a frame and in a step, and the stages' times of both attempts under the
    usual names."""
    from gaussian_splats_hip.kernels.rasterize.image import far_away
    from gaussian_splats_hip.timing import record_timings

    assert far_away(211_177, 1_185_219, 56, 1_000_000)
    assert not far_away(94_490, 1_337_256, 162, 1_000_000)  # not an eighth in one list
    assert not far_away(577_233, 41_233_268, 968, 2_000_000)  # larger than a list tile
    assert not far_away(211_177, 1_185_219, 1024, 1_000_000)  # many tiles
    assert not far_away(8192, 24_000, 4, 20_000)  # short lists
    scene = _points(30_000, (1111, 1043), 20.0).to(device)
    cam = scene.cameras[0]
    splats = GaussianSplat.from_tensors(*scene.params())
    leaves = [p.detach().clone().requires_grad_(True) for p in scene.params()]
    with record_timings(device) as times:
        image = rasterize(splats, cam, near=scene.near, far=scene.far)
    assert set(times["default"]) == {"Project", "Bin", "Emit", "Sort", "Composite"}
    ranges = image.grad_fn.saved_tensors[8]
    assert ranges.shape[0] == 70 * 66
    expected = _op(scene, leaves, cam, 16, "gaussian")
    assert torch.equal(image, expected)
    with torch.no_grad():
        assert torch.equal(image, rasterize(splats, cam, near=scene.near, far=scene.far))
    weight = torch.randn(image.shape, device=device, generator=torch.Generator(device).manual_seed(1))
    (image * weight).sum().backward()
    (expected * weight).sum().backward()
    _same_gradients([getattr(splats, n).grad for n in PARAMS], [p.grad for p in leaves])


@pytest.mark.parametrize("n", [40_000, 14_000])
def test_image_one_long_list(n, device):
    """One list above 8192 entries among many short ones (faint Gaussians in
    front of the others) on more than 4096 tiles, its length known to the host
    (bucketing) or not (small scenes): four waves per tile and walk records."""
    scene = scenes.edge_case_scene(n=n, sh_degree=0, image_size=(1111, 1043), seed=6)
    g = torch.Generator().manual_seed(4)
    m = n - 10_000
    scene.mean[m:] = torch.tensor([0.05, 0.03, -0.8]) + torch.randn(10_000, 3, generator=g) * 0.002
    scene.scale[m:], scene.opacity[m:] = -6.0, -5.3
    scene = scene.to(device)
    splats = GaussianSplat.from_tensors(*scene.params())
    leaves = [p.detach().clone().requires_grad_(True) for p in scene.params()]
    image = rasterize(splats, scene.cameras[0], near=scene.near, far=scene.far)
    ranges, walk_records = (image.grad_fn.saved_tensors[i] for i in (8, -1))
    assert (ranges[:, 1] - ranges[:, 0]).max() > 8192 and walk_records is not None
    expected = _op(scene, leaves, scene.cameras[0], 16, "gaussian")
    # The op's checkpoints cut a pixel's colour into partial sums (see below).
    assert (image - expected).abs().max() < 64 * 4 * 2.0 ** -24
    weight = torch.linspace(-1, 1, image.numel(), device=device).reshape(image.shape)
    (image * weight).sum().backward()
    (expected * weight).sum().backward()
    _same_gradients([getattr(splats, n).grad for n in PARAMS], [p.grad for p in leaves])


def test_plan_without_checkpoints(device):
    """A whole-tile forward without a checkpoint buffer leaves keys of a plan
    without segments, also for lists above 8192 entries."""
    from gaussian_splats_hip.kernels.rasterize import _native as nat

    w, h = 1111, 1043
    scene = _points(60_000, (w, h), 8.0, 4000).to(device)
    splats = GaussianSplat.from_tensors(*scene.params())
    image = rasterize(splats, scene.cameras[0], near=scene.near, far=scene.far)
    records, _, ids, ranges = image.grad_fn.saved_tensors[5:9]
    assert (ranges[:, 1] - ranges[:, 0]).max() > 8192
    view = nat.make_view(1.0, 1.0, 0.0, 0.0, w, h, 16, opacity_threshold=0.999, list_shift=1)
    out = [torch.empty((h, w, 3), device=device), torch.empty((h, w), device=device)]
    ncon = torch.empty((h, w), dtype=torch.int32, device=device)
    keys = nat.workspace(nat.library().gs_tile_order_workspace_bytes(4 * ranges.shape[0]), device)
    lib, ptr, stream = nat.library(), nat.ptr, nat.stream(device)
    nat.check(lib.gs_composite(
        ptr(records), records.shape[0], ptr(ids), ids.numel(), ptr(ranges), None, view,
        *map(ptr, out), ptr(ncon), None, 0, None, 0, ptr(keys), keys.numel(), stream), "composite")
    order = torch.empty(lib.gs_tile_order_items(view, 1), dtype=torch.int32, device=device)
    nat.check(lib.gs_tile_order(ptr(ranges), ptr(ncon), view, ptr(order), ptr(keys), keys.numel(),
                                1, stream), "tile_order")
    assert torch.equal(out[0], image)
    tiles = order[order >= 0]
    assert len(tiles) == 4 * ranges.shape[0] and not (tiles & 0x7F).any()


def test_image_tile_rule():
    assert image_tile(4, 1920, 1080, 10) == 16
    assert image_tile(32, 4096, 4096, 10) == 16
    assert image_tile(4, 4097, 16, 10) == 32
    assert image_tile(4, 8193, 16, 10) is None
    assert image_tile(64, 640, 480, 10) is None
    assert image_tile(8, 800, 800, 10, views=16) == 16
    assert image_tile(8, 1000, 1000, 10, views=25) == 32
    assert image_tile(16, 640, 480, 1 << 26) is None


@pytest.mark.parametrize("n,tw,th", [(1, 1, 1), (63, 5, 3), (64, 4, 1), (65, 3, 7), (1000, 256, 2),
                                     (1025, 17, 256), (5000, 30, 41), (24576, 26, 26),
                                     (255, 3, 2), (256, 3, 2), (257, 3, 2), (12288, 9, 11),
                                     (12289, 9, 11)])
def test_small_lists_equal_bucketing(n, tw, th, device):
    """gs_small_lists against the row/column bucketing: the same lists (ties
    by index, Gaussians without a rectangle nowhere), and the clear buffer."""
    from gaussian_splats_hip.kernels.rasterize import _native as nat
    from gaussian_splats_hip.kernels.rasterize.image import small_lists
    from gaussian_splats_hip.kernels.rasterize.intersections import bin_tiles

    g = torch.Generator().manual_seed(n + tw)
    x0, y0 = torch.randint(tw, (n,), generator=g), torch.randint(th, (n,), generator=g)
    w = (torch.rand(n, generator=g).pow(3) * (tw - x0)).long() + 1
    h = (torch.rand(n, generator=g).pow(3) * (th - y0)).long() + 1
    rects = x0 | (w - 1) << 8 | y0 << 16 | (h - 1) << 24
    # Few distinct depths, so ties are common.
    keys = torch.randint(1 << 30, (max(1, n // 3),), generator=g)[
        torch.randint(max(1, n // 3), (n,), generator=g)]
    culled = torch.rand(n, generator=g) < 0.2
    rects[culled], keys[culled] = 0xFFFFFFFF, 0xFFFFFFFF

    def int32(t):
        return torch.where(t >= 1 << 31, t - (1 << 32), t).to(torch.int32).to(device)

    rects, keys = int32(rects), int32(keys)
    nbytes = nat.library().gs_small_lists_bytes(n, tw, th)
    assert nbytes
    clear = torch.full((n, 9), 7.0, device=device)
    ids, ranges = small_lists(keys, rects, tw, th, nbytes, clear)
    assert not clear.any()
    starts = torch.arange(tw * th, device=device) * n
    assert torch.equal(ranges[:, 0], starts)
    want_ids, want = bin_tiles(keys.clone(), None, None, tw, th, tile_rects=rects)
    lengths = want[:, 1] - want[:, 0]
    assert torch.equal(ranges[:, 1] - starts, lengths)
    tile = torch.repeat_interleave(torch.arange(tw * th, device=device), lengths)
    at = torch.arange(len(want_ids), device=device) - want[tile, 0] + starts[tile]
    assert torch.equal(ids[at], want_ids)


def test_small_lists_limits(device):
    from gaussian_splats_hip.kernels.rasterize import _native as nat

    size = nat.library().gs_small_lists_bytes
    assert size(24576, 26, 26) and not size(24577, 1, 1) and not size(0, 4, 4)
    assert size(256, 256, 256) and not size(257, 256, 256) and not size(10, 257, 1)
