"""torch.autograd binding of the projective smoothing path.

``projected_image(pos, w, h, camera)`` renders the exact-mode quartic image of
particles at world positions ``pos`` (n, 3) with weights ``w`` and smoothing
lengths ``h`` through the C ABI (project_particles, grid build, gather,
retrieve), and its backward calls ilc_psg_backward, then carries the
projected-frame position gradient back to world coordinates through the
projection's FP32 matrix (projective_smoothing_reconstruction.cpp:175-205).
Particles that the depth mask removes get dL/dw = 0.  The reference renders
only; this binding exists so that gradients can be checked against finite
differences.
"""
from __future__ import annotations

import atexit
import collections
import math
import threading

import torch

from .backend import (ProjectiveSmoothingGrid, camera_pixel_points, camera_projection,
                      project_particles)


# Handles that a forward pass may take over instead of creating its own.  A
# handle's device buffers are about fifteen allocations, and freeing them waits
# for the device: a forward and backward of 20k particles on 96^2 pixels takes
# 0.70 ms with a handle of its own, 0.47 with one taken over.  Handles of up to
# _POOL_ROWS particles, pixels and grid cells are kept (at most some 60 MB each; a
# larger pass takes longer than the allocations), _POOL_SIZE per device over all
# configurations, the newest (two alternate while the image of the pass before
# is alive).  They are not torch's memory: release_handles() gives it back.
_POOL_ROWS = 1 << 18
_POOL_SIZE = 4
_pool = collections.defaultdict(collections.deque)   # device: (target, kernel), handle, event
_pool_lock = threading.RLock()   # a lease may end inside the collector, on any thread


def release_handles():
    """Destroys the handles that no pass holds (their memory goes back)."""
    with _pool_lock:
        held = list(_pool.values())
        _pool.clear()
    del held


atexit.register(release_handles)


class _Lease:
    """A handle for one forward pass and its backward passes.  It belongs to the
    lease alone; when the lease ends, the handle goes to the pool together with
    an event behind its last work, which its next holder's stream waits for."""

    def __init__(self, device, target, kernel, rows):
        self.device, self.config = device, (target, kernel)
        self.event = None        # None: not to be pooled
        self.small = rows <= _POOL_ROWS
        self.psg = None
        if self.small:
            with _pool_lock:
                free = _pool[device]
                for k in range(len(free) - 1, -1, -1):   # the newest
                    if free[k][0] == self.config:
                        _, self.psg, event = free[k]
                        del free[k]
                        break
            if self.psg is not None:
                torch.cuda.current_stream(device).wait_event(event)
        if self.psg is None:
            self.psg = ProjectiveSmoothingGrid(device, target, mode="exact", kernel=kernel)

    def used(self):
        """Marks the end of the work enqueued so far on the current stream."""
        stream = torch.cuda.current_stream(self.device)
        with torch.cuda.device(self.device):
            if not self.small or torch.cuda.is_current_stream_capturing():
                # a captured graph keeps reading the handle's buffers
                self.small, self.event = False, None
                return
        event = torch.cuda.Event()
        if self.event is not None:
            stream.wait_event(self.event)   # passes on several streams
        event.record(stream)
        self.event = event

    def failed(self):
        """The handle is destroyed with the lease."""
        self.small, self.event = False, None

    def __del__(self):
        if getattr(self, "event", None) is None or _pool_lock is None:
            return
        self.psg._keep = []   # the next holder sets its own points
        oldest = None
        with _pool_lock:
            free = _pool[self.device]
            free.append((self.config, self.psg, self.event))
            if len(free) > _POOL_SIZE:
                oldest = free.popleft()
        del oldest   # destroyed outside the lock


class ProjectedImage(torch.autograd.Function):
    @staticmethod
    def forward(ctx, pos, w, h, camera, kernel, scale, target_particles_per_cell):
        dev = pos.device
        p4 = torch.cat([pos.detach().float(), w.detach().float().reshape(-1, 1)], 1).contiguous()
        proj = project_particles(camera, p4, dev.index)
        # depth mask: project unit weights and see which become 0
        ones = torch.cat([pos.detach().float(), torch.ones_like(p4[:, :1])], 1).contiguous()
        kept = project_particles(camera, ones, dev.index)[:, 3] != 0
        pts = camera_pixel_points(camera, dev.index)
        lease = _Lease(dev.index, int(target_particles_per_cell), kernel,
                       max(proj.shape[0], pts.shape[0]))
        psg = lease.psg
        psg.init_backend(proj.shape[0])
        psg.setup_projected_particles(proj, h.detach().float())
        psg.setup_evaluation_points(pts, layout_nx=int(camera["nx"]))
        psg.run()
        img = psg.retrieve_results(float(scale))
        if math.prod(psg.grid_info()["num_cells"]) > _POOL_ROWS:
            lease.failed()
        lease.used()
        ctx.lease, ctx.scale, ctx.kept = lease, float(scale), kept
        ctx.keep_pts = pts
        minv, _ = camera_projection(camera)
        ctx.jac = torch.from_numpy(minv[:2].copy()).to(dev)   # d(x', y') / d(x, y, z)
        ctx.dtypes = (pos.dtype, w.dtype, h.dtype)
        return img.reshape(int(camera.get("ny", camera["nx"])), int(camera["nx"]))

    @staticmethod
    def backward(ctx, grad_img):
        lease = ctx.lease
        try:
            gw, gh, gx, gy = lease.psg.backward(grad_img.contiguous().reshape(-1), ctx.scale)
        except Exception:
            lease.failed()
            raise
        lease.used()
        gw = torch.where(ctx.kept, gw, torch.zeros_like(gw))
        gpos = gx[:, None] * ctx.jac[0][None, :] + gy[:, None] * ctx.jac[1][None, :]
        tp, tw, th = ctx.dtypes
        return gpos.to(tp), gw.to(tw), gh.to(th), None, None, None, None


def projected_image(pos, w, h, camera, kernel="quartic", scale=1.0,
                    target_particles_per_cell=1000):
    """Image (ny, nx) = scale * sum_j w_j W(|x_pixel - x'_j|, h_j), differentiable
    in pos, w and h."""
    return ProjectedImage.apply(pos, w, h, camera, kernel, scale, target_particles_per_cell)
