"""Rendering calls that return only the image.

``rasterize`` and ``rasterize_views`` return images; the op behind them
(``torch.ops.gaussian_splats_hip.rasterize``) also returns the reference's
projected Gaussians and sorted tile lists for the caller's tile size
(src/gaussian_splats/kernels/rasterize/interface.py:17-244).  An eager call of
the two functions does not go through the op: nothing but the pixels leaves it,
so it is free in what it lists and in which tiles:

* each Gaussian is listed for the tiles it can change (``gs_project_image``),
  about half of the reference's rectangle;
* the tiles are those the kernels do best at (``image_tile``), whatever tile
  size the caller names;
* the projection writes the compositing records alone, and both compositing
  directions read them.

A pixel's entries that blend are the same, in the same order, so images are
those of the op (``tests/test_gpu_image.py``); gradients differ in the order of
their sums.  An infinite colour is the exception: the forward walk adds it times
0 to the pixels of a tile that do not take it, and the tile is one of 16 pixels
here, so NaN reaches further around such a Gaussian than with the op's smaller
tiles.  (Selects in the walk cost it 0.5 to 10%.  A gradient that is not finite
reaches only the Gaussians its pixel took.)  Traced calls (``torch.compile``) use
the registered op.
"""

from __future__ import annotations

from ctypes import addressof

import torch

from . import _native as nat
from .intersections import MAX_BUCKET_GAUSSIANS, MAX_BUCKET_TILES, bin_tiles, depth_key_range


def mosaic_columns(views: int, tiles_w: int, tiles_h: int) -> int:
    """Views per mosaic row: the most nearly square layout whose tile grid fits
    ``MAX_BUCKET_TILES`` per axis (row/column bucketing), else the most nearly
    square one."""
    if views <= 1:
        return 1
    best, best_key = 1, None
    for cols in range(1, views + 1):
        rows = -(-views // cols)
        w, h = cols * tiles_w, rows * tiles_h
        fits = w <= MAX_BUCKET_TILES and h <= MAX_BUCKET_TILES
        # Fitting layouts first, then the squarest, then the fewest empty slots.
        key = (not fits, max(w, h), rows * cols - views)
        if best_key is None or key < best_key:
            best, best_key = cols, key
    return best


#: The compositing calls split each tile over four waves below this many tiles
#: with work (kCompositeSplitTiles); lists above this length count as long
#: (kCheckpointMinList, from which the op's whole-tile walks record checkpoints).
SPLIT_TILES, LONG_LIST = 4096, 8192

#: Tile sizes the op takes; any other goes to it, which refuses it.
OP_TILES = (4, 8, 16, 32)


def image_tile(asked: int, width: int, height: int, n: int, views: int = 1) -> int | None:
    """Tile size of an image call for which the caller ``asked`` one the op
    takes, or None when the op itself has to run: it refuses the size, or
    row/column bucketing takes neither grid (the op's other binning then runs,
    with the caller's tile size).  16 pixels: smaller tiles leave lanes of the
    compositing waves idle and list a Gaussian many times over (200k Gaussians
    at 1080p, forward and backward: 3.65 ms with the default tile size 4, 0.52 ms
    with 16); 32 where the grid of 16-pixel tiles is larger than bucketing
    takes."""
    if asked not in OP_TILES or width <= 0 or height <= 0 or views * n >= MAX_BUCKET_GAUSSIANS:
        return None
    for tile in (16, 32):
        tw, th = nat.tiles(width, height, tile)
        cols = mosaic_columns(views, tw, th)
        if cols * tw <= MAX_BUCKET_TILES and -(-views // cols) * th <= MAX_BUCKET_TILES:
            return tile
    return None


def far_away(longest: int, entries: int, lists: int, n: int) -> bool:
    """Whether ``lists`` shared lists of a single view of ``n`` Gaussians are to be
    made again, one per tile: Gaussians smaller than a list tile (``entries`` below
    two each) on few tiles, the ``longest`` list with more than an eighth of them,
    as a scene seen from far away.  Each tile walks up to four times its own
    entries there, and nothing was saved in placing them.  1M of them far away at
    1080p, a frame 1392 us with shared lists, 786 with lists made again (620 before
    lists were shared), a step 2910 and 1376 (1735); 200k a step 1693 and 1099
    (1450)."""
    return (lists * 4 < SPLIT_TILES and longest > LONG_LIST and 8 * longest > n
            and entries < 2 * n)


class ImageRequest:
    """Everything but the Gaussians of an image call on ``n`` of them: the
    ``cameras`` (``camera_floats`` of ``views`` of them), the views and the
    scalars.  ``stacked``: the images keep their view axis (``rasterize_views``);
    one camera's image without it is written as such, since a select of the stack
    would make the caller's image a view and its gradient a filled and copied
    stack (1080p, a step: 16 us of GPU time and three launches).

    The lists are those of ``tiles`` = (width, height) list tiles, laid out by
    ``list_view``; the compositing tiles by ``view``.  ``small``: the bytes of a
    small scene's lists' workspace, or 0.

    In a single view of many tiles 2 x 2 compositing tiles share a list (the
    views' ``list_shift``).  A walk ends where its pixels are opaque, mostly long before
    the list does (1M Gaussians at 1080p: after 126 of 1535 entries), so most
    entries are placed and never read; half of the rows and columns are about
    half of the entries to place, while a tile tests about twice the entries it
    walks.  1M at 1080p: 642 -> 613 us a step, 4M in a small cube: 2432 -> 1961,
    200k at 1080p: 525 -> 513.  With fewer tiles the walks, not the placing, set
    the time (800k at 800 x 600: +5%, 300k in a small cube at 800 x 800: +86%),
    and 16 views of 2500 tiles, which walk a quarter of their lists, gained
    nothing."""

    __slots__ = ("arguments", "floats", "view", "list_view", "views", "shape", "tiles", "near",
                 "far", "gaussian", "small")

    def __init__(self, n, cameras, views, width, height, tile, threshold, near, far,
                 rendering_mode, confidence, stacked, share=True):
        self.arguments = (n, cameras, views, width, height, tile, threshold, near, far,
                          rendering_mode, confidence, stacked)
        self.views, self.floats = views, cameras
        self.shape = (views, height, width, 3) if stacked else (height, width, 3)
        tw, th = nat.tiles(width, height, tile)
        shift = int(share and tile == 16 and self.views == 1 and tw * th >= SPLIT_TILES)
        tw, th = nat.tiles(width, height, tile << shift)
        cols = mosaic_columns(self.views, tw, th)
        self.tiles = (cols * tw, -(-self.views // cols) * th)
        self.small = nat.library().gs_small_lists_bytes(n * self.views, *self.tiles)
        self.near, self.far = near, far
        self.gaussian = rendering_mode == "gaussian"

        def view(tile, shift):
            return nat.make_view(
                1.0, 1.0, 0.0, 0.0, width, height, tile, near, far, rendering_mode, confidence,
                opacity_threshold=threshold, views=self.views, mosaic_cols=cols, list_shift=shift,
            )

        self.view = view(tile, shift)
        self.list_view = view(tile << shift, 0) if shift else self.view

    def unshared(self) -> ImageRequest:
        """The same request with a list per tile."""
        return ImageRequest(*self.arguments, share=False)

    def cameras(self):
        """The three arrays of ``floats``: rotations, translations, intrinsics."""
        base = addressof(self.floats)
        return base, base + 36 * self.views, base + 48 * self.views


class _Walk:
    """What the forward keeps for its backward beside the saved tensors, which
    hold everything of size but the accumulator (the backward takes that), so
    that a backward which does not retain the graph frees it."""

    __slots__ = ("view", "accumulator")


def small_lists(depth_keys, tile_rects, tiles_w, tiles_h, nbytes, clear=None):
    """Tile lists of a small scene (gs_small_lists; ``nbytes`` its workspace):
    ``(gaussian_ids, ranges)`` with n slots per tile, so no total is read back
    and the call does not wait.  ``clear``: an optional [N, C] tensor to zero."""
    n, device = tile_rects.shape[0], tile_rects.device
    ids = torch.empty(n * tiles_w * tiles_h, dtype=torch.int32, device=device)
    ranges = torch.empty((tiles_w * tiles_h, 2), dtype=torch.int64, device=device)
    ws = nat.workspace(nbytes, device)
    nat.check(
        nat.library().gs_small_lists(
            nat.ptr(depth_keys), nat.ptr(tile_rects), n, tiles_w, tiles_h, nat.ptr(ranges),
            nat.ptr(ids), ids.numel(), nat.ptr(ws), ws.numel(), nat.ptr(clear),
            clear.shape[1] if clear is not None else 0, nat.stream(device),
        ),
        "small_lists",
    )
    return ids, ranges


def forward_image(params, request: ImageRequest, keep: bool, timer=None, again=False):
    """Projects, bins and composites; returns ``(image, saved, walk)``, the last
    two None unless ``keep`` (a backward will follow).  ``again``: the call's
    timer has been started."""
    mark = timer or (lambda name: None)
    device = nat.require_gpu(*params)
    mean, rotation, scale, opacity, color = (nat.prepare(t) for t in params)
    if color.shape[1] > 16:
        raise NotImplementedError(
            f"SH degrees above 3 are not implemented. Got {color.shape[1]} coefficients."
        )
    lib, stream, ptr = nat.library(), nat.stream(device), nat.ptr
    n, views = mean.shape[0], request.views
    vn = views * n
    view = nat.GsView.from_buffer_copy(request.view)  # active_, split_tiles are set below
    width, height = view.image_width, view.image_height
    tiles_w, tiles_h = request.tiles

    records = torch.empty((vn, 12), dtype=torch.float32, device=device)
    depth_keys = torch.empty(vn, dtype=torch.int32, device=device)
    tile_rects = torch.empty(vn, dtype=torch.int32, device=device)
    if not again:
        mark("start")
    nat.check(
        nat.launch("project", lambda: lib.gs_project_image(
            ptr(mean), ptr(rotation), ptr(scale), ptr(opacity), ptr(color), n, color.shape[1],
            *request.cameras(), request.list_view, ptr(records), ptr(depth_keys),
            ptr(tile_rects), stream,
        )),
        "project_image",
    )
    mark("project")
    backward = keep and request.gaussian
    # The backward's [V N, 9] gradient accumulator, zeroed beside the depth sort.
    accumulator = (torch.empty((vn, 9), dtype=torch.float32, device=device) if backward else None)
    if request.small:
        ids, ranges = small_lists(depth_keys, tile_rects, tiles_w, tiles_h, request.small,
                                  accumulator)
        # Unknown to the host; a list may hold them all.  An image alone is not
        # split for that (14k Gaussians at 1111 x 1043: 109 us, 117 split; with a
        # backward 324 and 308, and 5043 and 1656 where a list does hold 10k).
        longest, known = n if backward else 0, False
        mark("bin")
        mark("emit")
    else:
        ids, ranges = bin_tiles(
            depth_keys, None, None, tiles_w, tiles_h, timer=mark, tile_rects=tile_rects,
            clear=accumulator, key_range=depth_key_range(request.near, request.far),
        )
        longest, known = nat.longest_list(ranges), True
    mark("sort")
    subs = 1 << (2 * view.list_shift)  # compositing tiles per list
    lists = nat.active_tiles(ranges)
    if view.list_shift and far_away(longest, ids.numel(), lists, n):
        del records, depth_keys, tile_rects, accumulator, ids, ranges
        return forward_image(params, request.unshared(), keep, timer, again=True)
    view.active_tiles = lists * subs
    # With a long list the longest walk may set the time of a launch: its tiles
    # are split over four waves however many have work.  Whether it does is not
    # known before the walk.  1M Gaussians at 1080p with a dense spot, a step with
    # a wave per tile and with four: 652 and 743 us where the spot's pixels
    # saturate after some hundred entries, 10.9 and 4.5 ms where they do not; 80k
    # in a small cube on 4704 tiles 963 and 804.
    view.split_tiles = (2 if known else 1) if longest > LONG_LIST else 0
    num_tiles, total = tiles_w * tiles_h * subs, ids.numel()
    image = torch.empty(request.shape, dtype=torch.float32, device=device)
    if not backward:
        nat.check(
            nat.launch("composite", lambda: lib.gs_composite_image(
                ptr(records), vn, ptr(ids), total, ptr(ranges), view, ptr(image), stream,
            )),
            "composite_image",
        )
        mark("composite")
        return image, None, None
    final_transmittance = torch.empty((views, height, width), dtype=torch.float32, device=device)
    n_contributors = torch.empty((views, height, width), dtype=torch.int32, device=device)
    hits = nat.hit_mask_buffer(view, total, device)
    order = walk_records = None
    walk_bytes = lib.gs_composite_walk_bytes(view)
    if walk_bytes:
        # Every tile split: the walk's state at some positions, for a backward in
        # segments (no plan: the segments are dealt in tile order).
        walk_records = nat.workspace(walk_bytes, device)
        nat.check(
            nat.launch("composite", lambda: lib.gs_composite_walk(
                ptr(records), vn, ptr(ids), total, ptr(ranges), view, ptr(image),
                ptr(final_transmittance), ptr(n_contributors), ptr(hits), nat.buffer_bytes(hits),
                ptr(walk_records), walk_bytes, stream,
            )),
            "composite_walk",
        )
        mark("composite")
    else:
        keys = nat.workspace(lib.gs_tile_order_workspace_bytes(num_tiles), device)
        nat.check(
            nat.launch("composite", lambda: lib.gs_composite(
                ptr(records), vn, ptr(ids), total, ptr(ranges), None, view, ptr(image),
                ptr(final_transmittance), ptr(n_contributors), None, 0, ptr(hits),
                nat.buffer_bytes(hits), ptr(keys), keys.numel(), stream,
            )),
            "composite",
        )
        mark("composite")
        # The backward's dispatch plan, behind the forward on the stream.
        order = torch.empty(lib.gs_tile_order_items(view, 1), dtype=torch.int32, device=device)
        nat.check(
            lib.gs_tile_order(ptr(ranges), ptr(n_contributors), view, ptr(order), ptr(keys),
                              keys.numel(), 1, stream),
            "tile_order",
        )
    walk = _Walk()
    walk.view, walk.accumulator = view, accumulator
    saved = (records, tile_rects, ids, ranges, final_transmittance, n_contributors, hits, order,
             walk_records)
    return image, saved, walk


def _aligned(t: torch.Tensor | None) -> torch.Tensor | None:
    if t is None or (t.is_contiguous() and t.data_ptr() % 16 == 0):
        return t
    return t.clone(memory_format=torch.contiguous_format)


def backward_image(params, saved, walk: _Walk, request: ImageRequest, grad_image):
    """Gradients of the five parameter tensors for the image gradient."""
    params = tuple(_aligned(t) for t in params)
    mean, color = params[0], params[4]
    (records, tile_rects, ids, ranges, final_transmittance, n_contributors, hits, order,
     walk_records) = (_aligned(t) for t in saved)
    n, device = mean.shape[0], mean.device
    if grad_image is None:
        return tuple(torch.zeros_like(t) for t in params)
    grad_image = _aligned(grad_image.float())
    accumulator, walk.accumulator = walk.accumulator, None
    if accumulator is None:  # a second backward through the same graph
        accumulator = torch.zeros((records.shape[0], 9), dtype=torch.float32, device=device)
    grads = tuple(torch.empty_like(t) for t in params)
    if n == 0:
        return grads
    lib, stream, ptr = nat.library(), nat.stream(device), nat.ptr
    nat.check(
        nat.launch("composite_bwd", lambda: lib.gs_composite_bwd_image(
            ptr(records), records.shape[0], ptr(ids), ptr(ranges), ptr(grad_image),
            ptr(final_transmittance), ptr(n_contributors), ptr(order), walk.view,
            ptr(accumulator), ids.numel(), ptr(hits), nat.buffer_bytes(hits), ptr(walk_records),
            nat.buffer_bytes(walk_records), stream,
        )),
        "composite_bwd_image",
    )
    nat.check(
        nat.launch("project_bwd", lambda: lib.gs_project_bwd_image(
            *(ptr(t) for t in params), n, color.shape[1], *request.cameras(), walk.view,
            ptr(tile_rects), ptr(accumulator), *(ptr(g) for g in grads), stream,
        )),
        "project_bwd_image",
    )
    return grads


class _RenderImage(torch.autograd.Function):
    @staticmethod
    def forward(ctx, mean, rotation, scale, opacity, color, request, timer):
        params = (mean, rotation, scale, opacity, color)
        image, saved, walk = forward_image(params, request, True, timer)
        ctx.set_materialize_grads(False)
        ctx.request, ctx.walk = request, walk
        if saved is not None:
            ctx.save_for_backward(*params, *saved)
        return image

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, grad_image):
        if ctx.walk is None:
            raise AssertionError(
                "Backward gradients are only supported for Gaussian rendering."
            )
        saved = ctx.saved_tensors
        grads = backward_image(saved[:5], saved[5:], ctx.walk, ctx.request, grad_image)
        return (*grads, None, None)


def render_image(params, request: ImageRequest, timer=None) -> torch.Tensor:
    """The image or stack of images (``request.shape``) of ``request``'s cameras,
    differentiable with respect to the five parameter tensors in Gaussian mode."""
    if torch.is_grad_enabled() and any(t.requires_grad for t in params):
        return _RenderImage.apply(*params, request, timer)
    return forward_image(params, request, False, timer)[0]
