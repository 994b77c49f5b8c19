"""Reconstruction algorithms: ``fp``, ``bp``, ``fbp``, ``fdk``, ``sirt``.

Drop-in for ``kernelkit/algo.py`` of the reference (:18-368).  Host inputs
are copied to the device; results come back as host numpy arrays unless the
caller passes device outputs (``out``) or asks for them (``return_gpu``).

``fdk`` fuses pre-weight + row filter into one kernel that writes straight
into the backprojector's texture.  ``sirt`` runs four launches per
iteration: a plain forward projection of ``x`` into a projection buffer,
one coalesced pass writing ``R * (A x - y)`` into the backprojection
texture, the backprojection whose epilogue applies
``x <- clip(mask * (x - C * A^T r))``, and the rebuild of the forward
projector's texture of ``x``.
"""
from __future__ import annotations

from typing import Any, Callable, Sequence

import numpy as np

from kernelkit import _native, device
from kernelkit.geom.proj import Beam, ProjectionGeometry
from kernelkit.geom.vol import VolumeGeometry
from kernelkit.kernel import (BaseKernel, ProjectionTexture, as_device_array,
                              default_device, is_device_array, reads_planes)
from kernelkit.kernels.cone_bp import VoxelDrivenConeBP
from kernelkit.operator import XrayTransform
from kernelkit.processing import filter_into, filter_rows_into
from kernelkit.projector import BackProjector, ForwardProjector


def _to_host(t, out=None):
    return device.to_host(t, out)


def fp(volume: Any, projection_geometry, volume_geometry: VolumeGeometry,
       out=None):
    """Forward projection (``algo.py:18-49``).

    Returns a host array unless ``out`` is a device tensor (then it is
    filled and returned).
    """
    op = XrayTransform(projection_geometry, volume_geometry)
    vol = as_device_array(volume)
    dev_out = out if is_device_array(out) else None
    result = op(vol, out=dev_out)
    if dev_out is not None:
        return dev_out
    return _to_host(result, out if isinstance(out, np.ndarray) else None)


def bp(projections: Any, projection_geometry, volume_geometry: VolumeGeometry,
       filter: Any = None, preproc_fn: Callable = None,
       kernel: BaseKernel = None, out=None,
       projection_axes: Sequence[int] = (0, 1, 2), **kwargs):
    """Backprojection with optional FDK filtering (``algo.py:52-126``).

    ``preproc_fn(projections, projection_geometry)`` runs on the device
    tensor first; with ``filter`` the projections are pre-weighted and
    row-filtered (fused, into the backprojector's texture).  Returns a host
    array unless ``out`` is a device tensor.
    """
    projection_axes = tuple(projection_axes)
    proj = as_device_array(projections)
    if is_device_array(out):
        out_dev = as_device_array(out)
    else:
        default_device()
        out_dev = device.empty(tuple(int(s) for s in volume_geometry.shape),
                               like=proj)
    if preproc_fn is not None:
        if is_device_array(projections):   # the caller's memory: copy first
            proj = proj.clone()
        preproc_fn(proj, projection_geometry)
    kwargs.pop("beam", None)
    kwargs.update(projection_axes=projection_axes)
    K = VoxelDrivenConeBP(**kwargs) if kernel is None else kernel
    ptor = BackProjector(K, texture_type="layered")
    ptor.projection_geometry = projection_geometry
    ptor.volume_geometry = volume_geometry
    if filter is not None:
        if projection_axes != (0, 1, 2):
            raise NotImplementedError()
        tex = ProjectionTexture(*proj.shape, like=proj)
        if reads_planes(K):
            filtered = device.empty(tuple(proj.shape), like=proj)
            filter_rows_into(proj, filtered, geoms=list(projection_geometry),
                             filter=filter)
            tex.update(filtered, planes=True)
        else:
            tex.zero()
            filter_into(proj, tex, geoms=list(projection_geometry),
                        filter=filter)
        ptor._textures = tex
    else:
        ptor.projections = proj
    ptor.volume = out_dev
    # non-additive, as the reference's ``ptor()`` (its volume is zero-filled
    # first, ``projector.py:586-587``)
    ptor(additive=False)
    if is_device_array(out):
        return _to_host(out_dev)
    return _to_host(out_dev, out if isinstance(out, np.ndarray) else None)


def fbp(projections: Any, projection_geometry, volume_geometry,
        filter: Any = "ramlak", **bp_kwargs):
    """Parallel-beam FBP: not implemented, as in the reference
    (``algo.py:129-166``)."""
    raise NotImplementedError(
        "FBP is not implemented yet. Use a conebeam geometry with the `bp` "
        "function, or file an issue.")


def fdk(projections: Any, projection_geometry: Any,
        volume_geometry: VolumeGeometry, filter: Any = "ramlak",
        **bp_kwargs):
    """Feldkamp-Davis-Kress (``algo.py:169-223``): pre-weight, row filter,
    adjoint-scaled voxel-driven backprojection (no extra FDK normalisation,
    as in the reference)."""
    for p in projection_geometry:
        if p.beam != Beam.CONE:
            raise NotImplementedError(
                "Only cone beam geometry is supported at the moment.")
    if "kernel" not in bp_kwargs:
        bp_kwargs.update(kernel=VoxelDrivenConeBP())
    return bp(projections, projection_geometry, volume_geometry,
              filter=filter, **bp_kwargs)


def _check_mask_shape(mask, shape) -> None:
    """Raise ``ValueError`` unless ``mask`` broadcasts to the volume shape.

    The reference multiplies ``x *= mask`` (``algo.py:356-357``), so any
    mask that broadcasts against the volume is accepted; the update kernel
    reads it through strides (0 along broadcast axes).  Checked on the
    shape alone, before any device work.
    """
    mshape = tuple(int(s) for s in np.shape(mask))
    try:
        full = np.broadcast_shapes(mshape, tuple(shape))
    except ValueError:
        full = None
    if full != tuple(shape):
        raise ValueError(f"mask of shape {mshape} does not broadcast to the "
                         f"volume shape {tuple(shape)}")


class _SirtState:
    """Device buffers and launch arguments of one SIRT problem."""

    def __init__(self, projections, projection_geometry, volume_geometry,
                 mask, min_constraint, max_constraint):
        if mask is not None:
            _check_mask_shape(mask, tuple(int(s) for s in
                                          volume_geometry.shape))
        self.pg = list(projection_geometry)
        self.vg = volume_geometry
        n = len(self.pg)
        rows = int(self.pg[0].detector.rows)
        cols = int(self.pg[0].detector.cols)
        self.n, self.rows, self.cols = n, rows, cols
        default_device()            # raises without a HIP device
        if isinstance(projections, (list, tuple)):
            y = device.stack([as_device_array(p) for p in projections])
        else:
            y = as_device_array(projections)
        if tuple(y.shape) != (n, rows, cols):
            raise ValueError(f"projections of shape {tuple(y.shape)} do not "
                             f"match the geometry ({n}, {rows}, {cols})")
        self.y = y
        shape = tuple(int(s) for s in volume_geometry.shape)
        self.shape = shape
        self.fptor = ForwardProjector()
        self.fptor.projection_geometry = self.pg
        self.fptor.volume_geometry = volume_geometry
        self.bptor = BackProjector(texture_type="pitch2d")
        self.bptor.projection_geometry = self.pg
        self.bptor.volume_geometry = volume_geometry
        # every buffer is of the measurements' kind (torch or not)
        self.x = device.zeros(shape, like=y)
        # C = 1/BP(1), R = 1/FP(1) with inf -> 0 (algo.py:320-333)
        C = device.zeros(shape, like=y)
        self.bptor.projections = device.full((n, rows, cols), 1.0, like=y)
        self.bptor.volume = C
        self.bptor()
        R = device.empty((n, rows, cols), like=y)
        self.fptor.volume = device.full(shape, 1.0, like=y)
        self.fptor.projections = R
        self.fptor()
        lib = _native.lib()
        st = _native.stream_ptr()
        _native.check(lib.kk_recip_or_zero(_native._vp(C.data_ptr()),
                                           C.numel(), st))
        _native.check(lib.kk_recip_or_zero(_native._vp(R.data_ptr()),
                                           R.numel(), st))
        self.C, self.R = C, R
        # textures: x for the FP, residual for the BP (halo stays zero; every
        # element of planes is written by each residual pass)
        self.fptor.volume = self.x
        self.xtex = self.fptor._texture
        self.rtex = self.bptor._textures
        self.planes = self.rtex.planes is not None
        if not self.planes:
            self.rtex.zero()
        self.res = self.rtex.values()
        # a broadcast view: stride 0 along the mask's broadcast axes
        self.mask = (None if mask is None else device.broadcast_to(
            as_device_array(mask), shape))
        self.lo = 0.0 if min_constraint is None else float(min_constraint)
        self.hi = 0.0 if max_constraint is None else float(max_constraint)
        self.clip_lo = 0 if min_constraint is None else 1
        self.clip_hi = 0 if max_constraint is None else 1
        self.scale = float(volume_geometry.voxel_volume())
        # forward-projection buffer of the residual step
        self.p = device.empty((n, rows, cols), like=y)

    def iterate(self):
        lib = _native.lib()
        st = _native.stream_ptr()
        fk, bk = self.fptor.kernel, self.bptor.kernel
        # residual (FP(x) - y) * R into the BP texture: a plain forward
        # projection into a buffer, then one coalesced pass (cheaper on
        # MI355X than the forward kernel's residual epilogue, which reads
        # y and R one detector row per lane)
        fk._launch(self.xtex, self.p, self.rows, self.cols, False, None)
        rtex = _native._vp(self.rtex.hold_planes() if self.planes
                           else self.rtex.ptr)
        residual = (lib.kk_residual_to_bp_planes if self.planes
                    else lib.kk_residual_to_bp_texture)
        _native.check(residual(
            _native._vp(self.p.data_ptr()), _native.i64(self.p.stride()),
            _native._vp(self.y.data_ptr()), _native.i64(self.y.stride()),
            _native._vp(self.R.data_ptr()), _native.i64(self.R.stride()),
            self.n, self.rows, self.cols, rtex, st))
        mask_ptr = None if self.mask is None else _native._vp(
            self.mask.data_ptr())
        mask_st = None if self.mask is None else _native.i64(
            self.mask.stride())
        # x only; its forward-projection frames are rebuilt afterwards by
        # the texture kernel (coalesced), which on MI355X costs ~1.2 ms at
        # 512^3 against ~7.8 ms for the update epilogue's scattered
        # frame stores
        args = (bk._plan.ptr, rtex, self.n, self.rows, self.cols,
                _native._vp(self.x.data_ptr()), _native.i32(self.shape),
                _native.i64(self.x.stride()), _native._vp(self.C.data_ptr()),
                _native.i64(self.C.stride()), mask_ptr, mask_st, self.lo,
                self.hi, self.clip_lo, self.clip_hi)
        if self.planes:
            _native.check(lib.kk_sirt_bp_update_planes(*args, self.scale, st))
        else:
            _native.check(lib.kk_sirt_bp_update(*args, None, 0, self.scale,
                                                st))
        self.xtex.update(self.x, planes=fk.reads_planes)

    def capture(self):
        """Record one iteration in a HIP graph (the library's own stream
        capture, :class:`kernelkit._native.Graph`): its four launches replay
        as one.  Nothing is allocated or cleared inside the iteration (every
        launch writes all it reads next), so the graph holds kernel nodes
        only."""
        self.graph = _native.Graph.capture(self.iterate)
        return self.graph

    def step(self):
        """One iteration: a graph replay once captured, else eager."""
        g = getattr(self, "graph", None)
        if g is None:
            self.iterate()
        else:
            g.replay()


def sirt(projections: Any, projection_geometry: Any,
         volume_geometry: VolumeGeometry, iters: int = 100,
         verbose: bool = True, mask: Any = None,
         min_constraint: float = None, max_constraint: float = None,
         return_gpu: bool = False, callback: callable = None,
         residual_every: int = 10, graph: bool = False):
    """Simultaneous Iterative Reconstruction Technique (``algo.py:226-368``).

    ``x <- clip(mask * (x - C * A^T (R * (A x - y))))`` from ``x = 0`` with
    ``C = 1/A^T 1`` and ``R = 1/A 1``.  ``callback(i, x, residual)`` gets
    device tensors.  The residual norm is only computed (a device-to-host
    sync) every ``residual_every`` iterations when ``verbose``.
    ``graph=True`` (not in the reference) records one iteration in a HIP
    graph and replays it, one launch per iteration instead of four.
    """
    if len(projections) != len(projection_geometry):
        raise ValueError("Number of projections does not match number of "
                         "geometries.")
    if mask is not None:
        _check_mask_shape(mask, tuple(int(s) for s in volume_geometry.shape))
    state = _SirtState(projections, projection_geometry, volume_geometry,
                       mask, min_constraint, max_constraint)
    if graph and iters > 0:
        state.capture()
    bar = range(iters)
    if verbose:
        from tqdm import tqdm
        bar = tqdm(bar, desc="SIRT")
    res_norm = ""
    for i in bar:
        state.step()
        if verbose and residual_every is not None:
            if i % residual_every == 0:
                res_norm = str(float(np.linalg.norm(
                    device.to_host(state.res))))
            bar.set_description(f"SIRT: {res_norm}")
        if callback is not None:
            callback(i, state.x, state.res)
    if return_gpu:
        return state.x
    return _to_host(state.x)
