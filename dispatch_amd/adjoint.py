"""Differentiable formal solution: the emergent intensity of a set of rays (and the
mean intensity J) as a torch.autograd.Function of the opacity and source cubes.

Forward: each ray is swept patch by patch, as DISPATCH sweeps a column of patches
(`patch` planes each, 23 by default): one m3drt_sc_sweep per patch whose upstream
ghost plane is the previous patch's last plane (chi, S) with the intensity that
patch left on its exit plane (set_upstream_boundary / set_downstream_boundary,
SRC/rt_patch_mod.f90:3270-3300, 3471-3511).  The exit planes of the patches are the
checkpoints: one (nf, ny, nx) plane per patch boundary and ray, kept for the
backward pass.  The patch sweeps give the single-launch sweep's results bit for bit
(the ghost plane carries exactly the values the upwind plane holds).

Backward: per ray whose exit plane (or J) carries a cotangent, the patches are
taken in reverse sweep order: the patch's intensity is recomputed from its
checkpoint into one patch-sized scratch, and m3drt_sc_adjoint runs the patch in
reverse, accumulating the cotangents of its chi and S; the cotangent it returns
for its ghost plane is that of the previous patch's exit plane (I) and last plane
(chi, S), and is handed on.  Nothing larger than a patch is recomputed.

Where memory allows, a gradient will be taken and J is not asked for, the forward also
keeps a ray's whole intensity cube (RaySet.keep), and the recomputation (12 of the 48 B a
point and ray moves) falls away.  The checkpoints are written all the same, the patches
are the same either way, and so is every sum's order: a cube is only a shortcut, what is
kept changes the time and not a bit of the gradient, and cubes are given back wherever an
allocation here fails or a later solution finds the memory short.
The reference has no adjoint; its forward is rt_patch_t%short_char2
(SRC/rt_solvers_mod.f90:224-507) with integrate_intensity
(SRC/rt_patch_mod.f90:3399-3431).

chi500 (the tau500 step scale) and the directions are held fixed.
"""
from __future__ import annotations

import itertools
import threading
import weakref
from dataclasses import dataclass

import numpy as np
import torch

from . import m3drt


@dataclass
class RaySet:
    """The directions of one formal solution over a box in the native layout
    (nz, nf, ny, nx): unit vectors (nray, 3), J weights (nray), chi500 (nz, ny, nx),
    chi500 at each ray's upwind points (list of (nz, ny, nx)), the ghost planes'
    chi500 below the bottom and above the top, the cell sizes; `patch` planes per
    patch of the checkpointed sweep; `keep`, how many rays of a solution keep their
    intensity cubes from the forward to the backward pass at most: a number (0: none, the
    least memory), or "auto", as many as half of the memory holds that the backward
    pass and the caller's leave (_kept_cubes).  The results are the same."""
    ctx: "m3drt.Context"
    vec: np.ndarray
    wj: np.ndarray
    ds: tuple
    chi500: torch.Tensor
    chi500_up: list
    g500_bot: torch.Tensor
    g500_top: torch.Tensor
    patch: int = 23
    keep: "int | str" = "auto"

    def __post_init__(self):
        if self.keep != "auto" and not (isinstance(self.keep, int) and self.keep >= 0):
            raise ValueError("RaySet.keep is a number of rays or 'auto'")

    def up(self, r):
        return self.vec[r][2] > 0

    def sweep(self, r, chi, S, ghosts, **out):
        """The whole column in one launch."""
        v = self.vec[r]
        up = self.up(r)
        gc, gs, gi = ghosts[0] if up else ghosts[1]
        self.ctx.sc_sweep(chi, S, gc, gs, gi, self.chi500, self.chi500_up[r], self.g500_bot if up else self.g500_top,
                          dir=1 if up else -1, ds=self.ds, vec=v, wj=float(self.wj[r]), **out)

    # ---------------------------------------------------------------- patches
    def patches(self, r, nz):
        """(z0, z1) of every patch in sweep order."""
        b = [(z0, min(nz, z0 + self.patch)) for z0 in range(0, nz, self.patch)]
        return b if self.up(r) else b[::-1]

    def _ghost_of(self, r, k, bounds, chi, S, ghosts, ckpt):
        """The upstream ghost (chi, S, I) and its chi500 of patch k (sweep order)."""
        up = self.up(r)
        if k == 0:
            return (ghosts[0] if up else ghosts[1]), (self.g500_bot if up else self.g500_top)
        z0, z1 = bounds[k - 1]
        zl = z1 - 1 if up else z0          # the previous patch's last plane in sweep order
        return (chi[zl], S[zl], ckpt[k - 1]), self.chi500[zl]

    def sweep_patch(self, r, k, bounds, chi, S, ghosts, ckpt, J=None, **out):
        """Patch k (sweep order) of ray r: J (a whole cube) accumulates over the
        patch's planes; the other outputs (exit_I, I_out) are the patch's own."""
        (gc, gs, gi), g500 = self._ghost_of(r, k, bounds, chi, S, ghosts, ckpt)
        z0, z1 = bounds[k]
        if J is not None:
            out["J"] = J[z0:z1]
        self.ctx.sc_sweep(chi[z0:z1], S[z0:z1], gc, gs, gi, self.chi500[z0:z1], self.chi500_up[r][z0:z1], g500,
                          dir=1 if self.up(r) else -1, ds=self.ds, vec=self.vec[r], wj=float(self.wj[r]), **out)

    def sweep_checkpointed(self, r, chi, S, ghosts, ckpt, exit_I, J=None, cube=None):
        """The ray patch by patch: ckpt (npatch - 1, nf, ny, nx) receives the exit
        plane of every patch but the last, whose exit plane goes to exit_I; cube, if
        given, every cell's intensity."""
        bounds = self.patches(r, chi.shape[0])
        for k, (z0, z1) in enumerate(bounds):
            ex = ckpt[k] if k + 1 < len(bounds) else exit_I
            out = {} if cube is None else {"I_out": cube[z0:z1]}
            self.sweep_patch(r, k, bounds, chi, S, ghosts, ckpt, exit_I=ex, J=J, **out)

    def adjoint_checkpointed(self, r, chi, S, ghosts, ckpt, scratch, gbars, chibar, Sbar, Jbar=None,
                             exit_bar=None, work=None, cube=None):
        """The reverse of sweep_checkpointed: patch by patch from the exit, each
        patch's intensity read from cube, or recomputed from its checkpoint into scratch
        (>= patch planes).  gbars: the true ghost planes' cotangents (accumulated); work: three
        (nf, ny, nx) planes for the patch-boundary cotangents."""
        bounds = self.patches(r, chi.shape[0])
        up = self.up(r)
        gcb, *gib = work
        carry = exit_bar
        for k in range(len(bounds) - 1, -1, -1):
            z0, z1 = bounds[k]
            if cube is not None:
                I = cube[z0:z1]
            else:
                I = scratch[:z1 - z0]
                self.sweep_patch(r, k, bounds, chi, S, ghosts, ckpt, I_out=I)
            (gc, gs, gi), g500 = self._ghost_of(r, k, bounds, chi, S, ghosts, ckpt)
            if k == 0:
                tb = gbars[0] if up else gbars[1]
                ghost_bars = dict(ghost_chibar=tb[0], ghost_Sbar=tb[1], ghost_Ibar=tb[2])
            else:
                # the previous patch's last plane: S's cotangent added in place, chi's
                # product rounded before it is added, I's in the plane not read now
                pz0, pz1 = bounds[k - 1]
                zl = pz1 - 1 if up else pz0
                below = gib[k % 2]
                gcb.zero_()
                below.zero_()
                ghost_bars = dict(ghost_chibar=gcb, ghost_Sbar=Sbar[zl], ghost_Ibar=below)
            self.ctx.sc_adjoint(chi[z0:z1], S[z0:z1], gc, gs, gi, self.chi500[z0:z1], self.chi500_up[r][z0:z1],
                                g500, I, dir=1 if up else -1, ds=self.ds, vec=self.vec[r], wj=float(self.wj[r]),
                                chibar=chibar[z0:z1], Sbar=Sbar[z0:z1],
                                Jbar=None if Jbar is None else Jbar[z0:z1], exit_bar=carry, **ghost_bars)
            if k > 0:
                chibar[zl] += gcb
                carry = below


class _Cubes:
    """The intensity cubes that one solution keeps for its backward pass, by ray.  Any
    thread may take them away: a cube already popped by its backward pass stays alive
    there, and the memory of one dropped goes back to the stream it came from."""

    def __init__(self):
        self.by_ray = {}
        with _lock:
            _live[next(_order)] = self

    def add(self, r, like):
        """Ray r's cube, None where there is no room for it."""
        try:
            cube = torch.empty_like(like)
        except torch.OutOfMemoryError:
            return None
        with _lock:
            self.by_ray[r] = cube
        return cube

    def pop(self, r):
        with _lock:
            return self.by_ray.pop(r, None)

    def held(self, device):
        return sum(t.numel() * t.element_size() for t in self.by_ray.values() if t.device == device)


_lock = threading.RLock()
_order = itertools.count()
_live = weakref.WeakValueDictionary()       # every solution's _Cubes, oldest first


def _give_back(device, most=0):
    """Drops cubes, the oldest solution's first, until at most `most` bytes are kept on
    the device: (the bytes still kept, whether any went)."""
    with _lock:
        live = [c for _, c in sorted(_live.items())]
        held = [c.held(device) for c in live]
        total, gone = sum(held), False
        for c, n in zip(live, held):
            if n and total > most:
                c.by_ray.clear()
                total, gone = total - n, True
    return total, gone


def _alloc(device, make):
    """make(), once more without the kept cubes if it finds no memory."""
    try:
        return make()
    except torch.OutOfMemoryError:
        if not _give_back(device)[1]:
            raise
    return make()


def _kept_cubes(chi, nray):
    """How many of nray rays keep their intensity cube: all solutions' cubes together at
    most half of the memory (the driver's free and the caching allocator's) that
    would be left with no cube kept, after what the backward pass takes (the cotangents
    of chi and S, a patch and planes: three cubes) and as much again as this process
    holds otherwise, for the backward pass of the caller's own graph.  Earlier solutions
    give theirs back where that has become less than they keep, so that a graph of many
    solutions ends with the memory that the checkpoints alone take."""
    cube = max(1, chi.numel() * chi.element_size())
    held = _give_back(chi.device, most=1 << 62)[0]
    used = torch.cuda.memory_allocated(chi.device) - held
    free = torch.cuda.mem_get_info(chi.device)[0] + torch.cuda.memory_reserved(chi.device) - used
    most = max(0, (free - 3 * cube - used) // 2)
    held = _give_back(chi.device, most)[0]
    return max(0, min(nray, (most - held) // cube))


class _FormalSolution(torch.autograd.Function):
    @staticmethod
    def forward(fctx, rs, want_J, rays, grad, chi, S, gc_up, gs_up, gi_up, gc_dn, gs_dn, gi_dn):
        ghosts = ((gc_up, gs_up, gi_up), (gc_dn, gs_dn, gi_dn))
        nz, nf, ny, nx = chi.shape
        new = lambda shape: _alloc(chi.device, lambda: torch.empty(shape, dtype=chi.dtype, device=chi.device))
        exits = new((len(rs.vec), nf, ny, nx)).zero_()
        J = new(chi.shape).zero_() if want_J else None
        npatch = (nz + rs.patch - 1) // rs.patch
        ckpt = {r: new((max(npatch - 1, 1), nf, ny, nx)) for r in rays}
        cubes, keep = None, 0
        if grad and not want_J:
            keep = _kept_cubes(chi, len(rays)) if rs.keep == "auto" else min(rs.keep, len(rays))
            cubes = _Cubes()
        for r in rays:
            cube = None
            if keep > 0:
                cube = cubes.add(r, chi)
                keep = keep - 1 if cube is not None else 0
            rs.sweep_checkpointed(r, chi, S, ghosts, ckpt[r], exits[r], J=J, cube=cube)
        fctx.rs, fctx.rays, fctx.ckpt, fctx.cubes = rs, rays, ckpt, cubes
        fctx.save_for_backward(chi, S, gc_up, gs_up, gi_up, gc_dn, gs_dn, gi_dn)
        if want_J:
            return exits, J
        none = torch.zeros((), dtype=chi.dtype, device=chi.device)
        fctx.mark_non_differentiable(none)
        return exits, none

    @staticmethod
    def backward(fctx, exit_bar, J_bar):
        rs, rays, ckpt, cubes = fctx.rs, fctx.rays, fctx.ckpt, fctx.cubes
        chi, S, gc_up, gs_up, gi_up, gc_dn, gs_dn, gi_dn = fctx.saved_tensors
        ghosts = ((gc_up, gs_up, gi_up), (gc_dn, gs_dn, gi_dn))
        if J_bar is not None and J_bar.dim() == 0:
            J_bar = None
        if J_bar is not None:
            J_bar = J_bar.contiguous()
        zeros = lambda like: _alloc(chi.device, lambda: torch.zeros_like(like))
        chibar, Sbar = zeros(chi), zeros(S)
        gbars = tuple(tuple(zeros(t) for t in g) for g in ghosts)
        if exit_bar is not None:
            exit_bar = exit_bar.contiguous()
            live = (exit_bar.flatten(1).abs().amax(dim=1) > 0).cpu().numpy()
        else:
            live = np.zeros(len(rs.vec), bool)
        scratch = work = None
        for r in rays:
            cube = None if cubes is None else cubes.pop(r)      # freed once its ray is done
            if not live[r] and J_bar is None:
                continue
            if scratch is None and cube is None:
                shape = (min(rs.patch, chi.shape[0]),) + tuple(chi.shape[1:])
                scratch = _alloc(chi.device, lambda: torch.empty(shape, dtype=chi.dtype, device=chi.device))
            if work is None:
                work = tuple(zeros(gc_up) for _ in range(3))
            rs.adjoint_checkpointed(r, chi, S, ghosts, ckpt[r], scratch, gbars, chibar, Sbar, Jbar=J_bar,
                                    exit_bar=exit_bar[r] if live[r] else None, work=work, cube=cube)
        fctx.ckpt = fctx.cubes = None
        (gcb_u, gsb_u, gib_u), (gcb_d, gsb_d, gib_d) = gbars
        return None, None, None, None, chibar, Sbar, gcb_u, gsb_u, gib_u, gcb_d, gsb_d, gib_d


def formal_solution(rs: RaySet, chi, S, ghost_up, ghost_down, want_J=False, rays=None):
    """Exit planes of every ray, (nray, nf, ny, nx) (the emergent intensity for the
    upward rays), and J when want_J; differentiable in chi, S and the ghost planes.
    chi, S: FP32 native cubes (nz, nf, ny, nx); ghost_up / ghost_down: (chi, S, I)
    planes (nf, ny, nx) below the bottom and above the top.  rays: the indices of
    the rays to sweep (default all; the others' exit planes stay zero and they add
    nothing to J)."""
    rays = list(range(len(rs.vec))) if rays is None else [int(r) for r in rays]
    grad = torch.is_grad_enabled() and any(t.requires_grad for t in (chi, S, *ghost_up, *ghost_down))
    exits, J = _FormalSolution.apply(rs, want_J, rays, grad, chi, S, *ghost_up, *ghost_down)
    return (exits, J) if want_J else exits
