"""m3drt_sc_sweep_noalloc, the sweep entry point that allocates nothing (its
scratch is the library's fixed device array), against m3drt_sc_sweep on the same
inputs through the C ABI: the same kernels, so the same bits, on two calls in a
row (the second smaller), around the context's own scratch, under HIP graph
capture, and a size beyond the fixed array refused before any launch."""
import numpy as np
import pytest
import torch

from dispatch_amd import m3drt, synth

pytestmark = pytest.mark.gpu


def _problem(nx, ny, nz, nf, seed):
    box = synth.make_box(nx=nx, ny=ny, nz=nz, nf=nf, seed=seed)
    chi, S = synth.build_cubes(box, torch.float32)
    ghost = synth.ghost_planes(box, chi, torch.float32)
    rays, w = synth.gauss_rays(6)
    return box, chi, S, ghost, rays, w


def _solve(ctx, prob, rays_sel, noalloc, J=None, exits=None):
    box, chi, S, ghost, rays, w = prob
    if J is None:
        J = torch.zeros_like(chi)
    outs = []
    for r in rays_sel:
        v = rays[r]
        up = v[2] > 0
        gchi, gS, gI = ghost["up" if up else "down"]
        ex = torch.zeros_like(gchi) if exits is None else exits[r]
        ctx.sc_sweep(chi, S, gchi, gS, gI, box.chi500, synth.chi500_upwind(box, v),
                     box.g500_bot if up else box.g500_top, dir=1 if up else -1, ds=box.ds, vec=v,
                     wj=float(w[r]), J=J, exit_I=ex, noalloc=noalloc)
        outs.append(ex)
    return J, outs


RAYS = [0, 5, 13, 20]


def test_noalloc_matches_the_allocating_sweep_twice(ctx):
    # the second call is smaller: the fixed array keeps the first call's contents
    for shape, seed in (((120, 120, 46, 16), 5), ((60, 36, 20, 8), 6)):
        prob = _problem(*shape, seed)
        Ja, ea = _solve(ctx, prob, RAYS, noalloc=False)
        Jb, eb = _solve(ctx, prob, RAYS, noalloc=True)
        torch.cuda.synchronize()
        assert torch.equal(Ja, Jb)
        for a, b in zip(ea, eb):
            assert torch.equal(a, b)
        assert float(Ja.abs().max()) > 0


def test_noalloc_leaves_the_context_scratch_alone(ctx):
    prob = _problem(48, 48, 30, 8, 7)
    Ja, _ = _solve(ctx, prob, RAYS, noalloc=False)
    Jb, _ = _solve(ctx, prob, [RAYS[0]], noalloc=True)
    Jb, _ = _solve(ctx, prob, RAYS[1:], noalloc=False, J=Jb)   # the context's scratch again
    torch.cuda.synchronize()
    assert torch.equal(Ja, Jb)


def test_noalloc_under_graph_capture(ctx):
    prob = _problem(60, 60, 24, 8, 8)
    box, chi, S, ghost, rays, w = prob
    Jref, _ = _solve(ctx, prob, RAYS, noalloc=False)
    torch.cuda.synchronize()
    cus = {r: synth.chi500_upwind(box, rays[r]) for r in RAYS}
    J = torch.zeros_like(chi)
    ex = {r: torch.zeros_like(ghost["up"][0]) for r in RAYS}
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        with torch.cuda.graph(g, stream=s):
            J.zero_()
            for r in RAYS:
                v = rays[r]
                up = v[2] > 0
                gchi, gS, gI = ghost["up" if up else "down"]
                ctx.sc_sweep(chi, S, gchi, gS, gI, box.chi500, cus[r], box.g500_bot if up else box.g500_top,
                             dir=1 if up else -1, ds=box.ds, vec=v, wj=float(w[r]), J=J, exit_I=ex[r],
                             noalloc=True)
    torch.cuda.synchronize()
    for rep in range(3):
        J.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(J, Jref), rep
        # eager work between the replays, on the same fixed array
        _solve(ctx, _problem(36, 36, 12, 4, 9 + rep), RAYS[:1], noalloc=True)
        torch.cuda.synchronize()


def test_noalloc_refuses_beyond_its_fixed_size(ctx):
    # 8 bytes per cell of nx*ny*(nz+1): 120*120*301*8 = 34.7 MB > 32 MiB
    box = synth.make_box(nx=120, ny=120, nz=300, nf=1, seed=10)
    chi, S = synth.build_cubes(box, torch.float32)
    ghost = synth.ghost_planes(box, chi, torch.float32)
    v = synth.gauss_rays(6)[0][0]
    J = torch.zeros_like(chi)
    with pytest.raises(m3drt.M3drtError, match="fixed"):
        ctx.sc_sweep(chi, S, *ghost["up"], box.chi500, synth.chi500_upwind(box, v), box.g500_bot, dir=1,
                     ds=box.ds, vec=v, wj=1.0, J=J, noalloc=True)
    torch.cuda.synchronize()
    assert float(J.abs().max()) == 0.0          # nothing ran
    # the allocating entry point takes the same call
    ctx.sc_sweep(chi, S, *ghost["up"], box.chi500, synth.chi500_upwind(box, v), box.g500_bot, dir=1,
                 ds=box.ds, vec=v, wj=1.0, J=J)
    torch.cuda.synchronize()
    assert float(J.abs().max()) > 0.0


def _slab(nx, ny, nz, nf, dtype, seed=1):
    """A slab in the reference layout (nz, ny, nx, nf) and its directions' geometry."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: (torch.rand(s, generator=g, device="cuda") + 0.5)
    cube = lambda k: (r(nz, ny, nx, nf) * k).to(dtype)
    plane = lambda k: (r(ny, nx, nf) * k).to(dtype)
    args = (cube(1e-7), cube(1.0), plane(1e-7), plane(1.0), plane(1.0), r(nz, ny, nx) * 1e-7, r(nz, ny, nx) * 1e-7,
            r(ny, nx) * 1e-7)
    return args, dict(dir=1, ds=(50e5, 50e5, 10e5), vec=(0.3, -0.4, 0.866), layout="reference", wj=0.25)


@pytest.mark.parametrize("nf,nx,ny,nz,dtype", [(250, 120, 120, 3, torch.float32), (300, 120, 120, 3, torch.float32),
                                               (1024, 120, 120, 2, torch.float32), (170, 120, 120, 3, torch.float64),
                                               (40, 120, 120, 230, torch.float32), (97, 101, 67, 250, torch.float32)])
def test_frequencies_in_runs_have_the_same_bits(ctx, nf, nx, ny, nz, dtype):
    """Slabs with the frequencies at unit stride whose two intensity planes fit the fixed
    array, in two to eight runs of frequencies, with run lengths that do not divide nf:
    the allocating sweep's bits, and no error left behind by a call that succeeds."""
    args, geo = _slab(nx, ny, nz, nf, dtype)
    with pytest.raises(m3drt.M3drtError):
        ctx.sc_sweep(*args, **dict(geo, dir=0), exit_I=torch.zeros_like(args[4]))
    left = m3drt.last_error()
    out = []
    for noalloc in (False, True):
        J, ex = torch.full_like(args[0], 0.125), torch.zeros_like(args[4])
        ctx.sc_sweep(*args, J=J, exit_I=ex, noalloc=noalloc, **geo)
        torch.cuda.synchronize()
        assert m3drt.last_error() == left
        out.append((J, ex))
    assert float(out[0][1].abs().max()) > 0
    for a, b in zip(*out):
        assert torch.equal(a, b)


def test_capture_with_little_scratch_has_the_same_bits():
    """A fresh context whose scratch holds the planes of a few frequencies only, captured:
    the capture takes them in runs, and its replays give the eager call's bits."""
    args, geo = _slab(60, 60, 5, 200, torch.float32)
    ctx = m3drt.Context(0)
    try:
        few = [t[..., :16].contiguous() for t in args[:5]]
        ctx.sc_sweep(*few, *args[5:], J=torch.zeros_like(few[0]), **geo)      # 1 MiB of scratch
        J = torch.zeros_like(args[0])
        s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            with torch.cuda.graph(g, stream=s):
                J.zero_()
                ctx.sc_sweep(*args, J=J, **geo)
        torch.cuda.synchronize()
        ref = torch.zeros_like(J)
        ctx.sc_sweep(*args, J=ref, **geo)                                     # the scratch grows
        torch.cuda.synchronize()
        assert float(ref.abs().max()) > 0
        for rep in range(3):
            J.fill_(float("nan"))
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(J, ref), rep
            ctx.sc_sweep(*args, J=torch.zeros_like(J), **geo)
            torch.cuda.synchronize()
    finally:
        ctx.close()


@pytest.mark.parametrize("nz", [1, 2])
@pytest.mark.parametrize("noalloc", [False, True])
def test_exit_plane_over_the_ghost_plane(ctx, nz, noalloc):
    """exit_I laid over ghost_I, as a column of slabs hands its planes on: the values of a
    call with a plane of its own, with one plane (where other workgroups could read what
    has been written) and with more."""
    args, geo = _slab(48, 40, nz, 64, torch.float32)
    ex = torch.zeros_like(args[4])
    ctx.sc_sweep(*args, exit_I=ex, J=torch.zeros_like(args[0]), noalloc=noalloc, **geo)
    over = list(args)
    over[4] = args[4].clone()
    ctx.sc_sweep(*over, exit_I=over[4], J=torch.zeros_like(args[0]), noalloc=noalloc, **geo)
    torch.cuda.synchronize()
    assert float((over[4] - ex).abs().max()) <= 1e-6 * float(ex.abs().max())
