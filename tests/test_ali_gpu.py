"""The NLTE ALI driver (dispatch_amd.ali) on small boxes of its workload generator:
one iteration's rate sums and departure coefficients against the oracle's
composition of the same steps (tests/ali_cases.py); convergence; the LTE limit
under strong collisional coupling."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def small(**kw):
    from dispatch_amd.ali import AliConfig
    base = dict(nx=6, ny=6, nz=48, nq=16, nbound=4, nline=6, ncont=4, lines_per_window=3, nphi=2, ncont_f=8)
    base.update(kw)
    return AliConfig(**base)


def test_ali_iteration_matches_oracle(ctx):
    from dispatch_amd.ali import NlteProblem
    from ali_cases import oracle_rates, oracle_update
    p = NlteProblem(ctx, small())
    print("ali iteration vs oracle, 6x6x48, 5 levels, 6 lines, 4 continua, 8 rays", flush=True)
    for it in range(2):
        gij, gji = p.rates()
        torch.cuda.synchronize()
        rij, rji = oracle_rates(p)
        for got, ref, what in ((gij, rij, "gamma_ij"), (gji, rji, "gamma_ji")):
            g = got.double().cpu().numpy()
            scale = np.abs(ref).max(axis=1, keepdims=True) + 1e-300
            err = np.abs(g - ref) / scale
            assert err.max() < 2e-4, f"iteration {it} {what}: {err.max():.3e} (row {np.unravel_index(err.argmax(), err.shape)})"
        b_ref, res_ref = oracle_update(p, rij, rji)
        res = p.update(gij, gji)
        b = p.b.cpu().numpy()
        assert np.abs(b / b_ref - 1).max() < 2e-4, f"iteration {it} b: {np.abs(b / b_ref - 1).max():.3e}"
        assert abs(res["maxerr"] - res_ref["maxerr"]) <= 2e-4 * abs(res_ref["maxerr"]) + 1e-6
        p.b.copy_(torch.from_numpy(b_ref))   # both continue from the oracle's populations


def test_ali_converges_and_departs_from_lte(ctx):
    from dispatch_amd.ali import NlteProblem
    p = NlteProblem(ctx, small(max_iter=40))
    n = p.solve(log=lambda m: print(m, flush=True))
    errs = [abs(e) for e, _ in p.history]
    assert errs[-1] < 1e-4 and n <= 40, errs
    b = p.b.cpu().numpy()
    assert np.abs(b - 1).max() > 1e-2   # the lines' NLTE departures are there


def test_ali_strong_collisions_give_lte(ctx):
    """With the electron density raised 1e7-fold the lower half of the box, where
    collisions then dominate every transition, is in LTE (b within 1e-3 of 1)."""
    from dispatch_amd.ali import NlteProblem
    cfg = small(ne_scale=1e7, max_iter=40)
    p = NlteProblem(ctx, cfg)
    p.solve()
    b = p.b.cpu().numpy().reshape(p.atom.nk, cfg.nz, -1)
    assert np.abs(b[:, :cfg.nz // 2] - 1).max() < 1e-3, np.abs(b[:, :cfg.nz // 2] - 1).max()


@pytest.mark.parametrize("kw", [{}, dict(nq=50, lines_per_window=4)])
def test_window_opacity_equals_the_sequence(ctx, kw):
    """m3drt_window_opacity against the sequence it fuses (the continuum product,
    convert_to_work_units, the seeded split tracking, bb_opacity, work_to_transfer) on
    every window and direction of the small problem at non-LTE populations: chi, S and
    the six tracking arrays bit for bit (both round every product and sum apart).  With
    50 frequencies per line a window of 4 lines has 200 frequencies, which the kernel
    splits into runs of 67 per lane, their ends inside line windows."""
    from dispatch_amd.ali import NlteProblem
    from dispatch_amd import synth
    p = NlteProblem(ctx, small(**kw))
    g = torch.Generator(device="cuda").manual_seed(3)
    p.b.mul_(torch.exp(0.3 * torch.randn(p.b.shape, generator=g, dtype=torch.float64, device="cuda")))
    print(f"window opacity fused vs sequence {kw}", flush=True)
    for wi, w in enumerate(p.windows):
        l0, l1 = w.lines[0], w.lines[-1] + 1
        nf, nc = w.nf, p.ncell
        for r, v in enumerate(p.vec):
            vproj = (p.vz * (v[2] / synth.C_LIGHT)).float().contiguous()
            d = dict(w.const, vproj=vproj, b=p.b, nstar=p.nstar, pop_ratio=p.pop_ratio, inv_df=p.inv_df,
                     e_kT=p.e_kT32, adamp=p.adamp[l0:l1])
            out = []
            for fused in (False, True):
                xhat = torch.full((nf, nc), 7.0, dtype=torch.float32, device="cuda")
                ehat = torch.full_like(xhat, 7.0)
                sp = dict(split_opac1=torch.full_like(xhat, 7.0), split_opac2=torch.full_like(xhat, 7.0),
                          split_chi1=torch.full_like(xhat, 7.0), split_chi2=torch.full_like(xhat, 7.0),
                          split_id=torch.full((nf, nc), 7, dtype=torch.int32, device="cuda"),
                          split_chi_id=torch.full((nf, nc), 7, dtype=torch.int32, device="cuda"))
                if fused:
                    ctx.window_opacity(d, w.chi_c, w.Bnu, w.beta, xhat, ehat, split=sp, split_offset=0)
                else:
                    xhat.zero_()
                    torch.mul(w.chi_c, w.Bnu, out=ehat)
                    ctx.convert_to_work_units(w.chi_c, xhat, ehat, w.beta)
                    sp["split_opac1"].copy_(ehat)
                    sp["split_chi1"].copy_(xhat)
                    for k in ("split_opac2", "split_chi2", "split_id", "split_chi_id"):
                        sp[k].zero_()
                    ctx.bb_opacity(d, xhat, ehat, split=sp, split_offset=0)
                    ctx.work_to_transfer(xhat, ehat, w.beta, split_opac1=sp["split_opac1"],
                                         split_opac2=sp["split_opac2"])
                out.append(dict(sp, chi=xhat, S=ehat))
            torch.cuda.synchronize()
            for k in out[0]:
                assert torch.equal(out[0][k], out[1][k]), (wi, r, k, float((out[0][k] - out[1][k]).abs().max()))


def _overlapping(p, w, seed):
    """The window's lines with windows that overlap: every line's start drawn anew, so
    that a frequency holds none, one or several lines."""
    g = np.random.default_rng(seed)
    nline, nf, nq = len(w.lines), w.nf, p.cfg.nq
    const = {k: v.clone() for k, v in w.const.items()}
    q = np.linspace(-p.cfg.qmax, p.cfg.qmax, nq).astype(np.float32)
    const["q"].zero_()
    for l in range(nline):
        f0 = int(g.integers(0, nf - nq + 1))
        const["iblue"][l], const["ired"][l] = f0 + 1, f0 + nq
        const["q"][l, f0:f0 + nq] = torch.from_numpy(q).cuda()
        const["wnu"][l] = 1.0 / nq
        const["wq"][l] = 2.0 * p.cfg.qmax / nq
    return const


@pytest.mark.parametrize("kw,overlap,off", [({}, False, 0), (dict(nq=50, lines_per_window=4), True, 3),
                                            (dict(nq=7, nline=70, lines_per_window=70, nbound=20), True, 0)])
def test_rates_with_the_tracking_formed_again(ctx, kw, overlap, off):
    """window_opacity(track) and bb_rates_window against window_opacity with its tracking
    arrays and bb_rates reading them: chi, S and the rate sums bit for bit, with lines
    alone at their frequencies and overlapping, and with more lines than the covering
    mask holds."""
    from dispatch_amd.ali import NlteProblem
    from dispatch_amd import synth
    p = NlteProblem(ctx, small(**kw))
    g = torch.Generator(device="cuda").manual_seed(5)
    p.b.mul_(torch.exp(0.3 * torch.randn(p.b.shape, generator=g, dtype=torch.float64, device="cuda")))
    print(f"rates with the tracking formed again {kw} overlap={overlap}", flush=True)
    w = p.windows[0]
    l0, l1, nf, nc = w.lines[0], w.lines[-1] + 1, w.nf, p.ncell
    const = _overlapping(p, w, 4) if overlap else w.const
    vproj = (p.vz * (p.vec[0][2] / synth.C_LIGHT)).float().contiguous()
    d = dict(const, vproj=vproj, b=p.b, nstar=p.nstar, pop_ratio=p.pop_ratio, inv_df=p.inv_df, e_kT=p.e_kT32,
             adamp=p.adamp[l0:l1])
    rnd = lambda: torch.rand((nf, nc), generator=g, device="cuda")
    Irem, esc, I = rnd() * w.Bnu, rnd(), rnd() * w.Bnu
    out = []
    for retrack in (False, True):
        chi, S = torch.empty_like(w.chi_c), torch.empty_like(w.chi_c)
        sp = {}
        if not retrack:
            sp = {k: torch.empty_like(w.chi_c) for k in ("split_opac1", "split_opac2", "split_chi1", "split_chi2")}
            sp.update({k: torch.empty((nf, nc), dtype=torch.int32, device="cuda") for k in ("split_id", "split_chi_id")})
        ctx.window_opacity(d, w.chi_c, w.Bnu, w.beta, chi, S, split=None if retrack else sp, split_offset=off,
                           track=retrack)
        Psi = torch.where(I < 0.05 * w.Bnu, torch.zeros_like(chi), esc / chi.abs())
        gij, gji = torch.zeros((l1 - l0, nc), device="cuda"), torch.zeros((l1 - l0, nc), device="cuda")
        dr, parts = dict(d, Inu=I, Psi=Psi, Bnu=w.Bnu, beta=w.beta), dict(sp, Irem=Irem, escape=esc, chi=chi)
        if retrack:
            ctx.bb_rates_window(dr, w.chi_c, 0.3, 1.0, gij, gji, own_norm=True, split=parts, split_offset=off)
        else:
            ctx.bb_rates(dr, 0.3, 1.0, gij, gji, precond=True, largest=True, own_norm=True, split=parts,
                         split_offset=off)
        out.append((chi, S, gij, gji))
    torch.cuda.synchronize()
    assert float(out[0][2].abs().max()) > 0
    for a, b, what in zip(*out, ("chi", "S", "gamma_ij", "gamma_ji")):
        assert torch.equal(a, b), (what, float((a - b).abs().max()))


@pytest.mark.parametrize("layout", ["native", "reference"])
@pytest.mark.parametrize("offs,scat,flags", [(True, False, False), (False, True, False), (False, False, True),
                                             (True, True, True)])
def test_tracking_formed_again_in_every_form(ctx, layout, offs, scat, flags):
    """The same comparison for lines that blend, with lower levels off their term's
    (lower_off, an exponential a line and cell), line scattering, psi flags read and
    raised, and both layouts: chi, S, the rate sums and the raised flags bit for bit."""
    from dispatch_amd import synth
    from dispatch_amd.ali import NlteProblem
    p = NlteProblem(ctx, small(nq=50, lines_per_window=6))
    g = torch.Generator(device="cuda").manual_seed(7)
    p.b.mul_(torch.exp(0.3 * torch.randn(p.b.shape, generator=g, dtype=torch.float64, device="cuda")))
    w = p.windows[0]
    l0, l1, nf, nc = w.lines[0], w.lines[-1] + 1, w.nf, p.ncell
    nl = l1 - l0
    print(f"tracking formed again {layout} lower_off={offs} scat={scat} flags={flags}", flush=True)
    const = _overlapping(p, w, 9)
    cover = torch.zeros(nf, dtype=torch.int32)
    for a, b in zip(const["iblue"].tolist(), const["ired"].tolist()):
        cover[a - 1:b] += 1
    assert int(cover.max()) > 1
    if offs:
        const["lower_off"] = (0.1 * torch.randn(nl, generator=g, device="cuda")).contiguous()
        const["lower_off"][::3] = 0.0
    lay = (lambda t: t) if layout == "native" else (lambda t: t.T.contiguous())
    d = dict(const, vproj=(p.vz * (p.vec[0][2] / synth.C_LIGHT)).float().contiguous(), b=p.b, nstar=p.nstar,
             pop_ratio=p.pop_ratio, inv_df=p.inv_df, e_kT=p.e_kT32, adamp=p.adamp[l0:l1])
    rnd = lambda: torch.rand((nf, nc), generator=g, device="cuda")
    cont, B, beta = lay(w.chi_c), lay(w.Bnu), lay(w.beta)
    I, Irem, esc = lay(rnd() * w.Bnu), lay(rnd() * w.Bnu), lay(rnd())
    extra = {}
    if scat:
        extra.update(chi_scat=lay(0.1 * rnd() * w.chi_c), dJnu=lay(rnd() * w.Bnu))
    raised = torch.randint(0, 1 << 20, (2, nc), generator=g, device="cuda", dtype=torch.int32)
    if flags:
        extra.update(ntrans=torch.arange(30, 30 + nl, dtype=torch.int32, device="cuda"),
                     psi_flags_in=torch.randint(0, 1 << 30, (2, nc), generator=g, device="cuda", dtype=torch.int32))
    out = []
    for retrack in (False, True):
        chi, S = torch.empty_like(cont), torch.empty_like(cont)
        sp = {}
        if not retrack:
            sp = {k: torch.empty_like(cont) for k in ("split_opac1", "split_opac2", "split_chi1", "split_chi2")}
            sp.update({k: torch.empty(cont.shape, dtype=torch.int32, device="cuda") for k in ("split_id", "split_chi_id")})
        ctx.window_opacity(d, cont, B, beta, chi, S, split=None if retrack else sp, split_offset=5, track=retrack,
                           layout=layout)
        Psi = torch.where(I < 0.05 * B, torch.zeros_like(chi), esc / chi.abs())
        gij, gji = torch.zeros((nl, nc), device="cuda"), torch.zeros((nl, nc), device="cuda")
        up = raised.clone()
        parts = dict(sp, Irem=Irem, escape=esc, chi=chi, **extra, **({"psi_flags_out": up} if flags else {}))
        dr = dict(d, Inu=I, Psi=Psi, Bnu=B, beta=beta)
        if retrack:
            ctx.bb_rates_window(dr, cont, 0.3, 1.0, gij, gji, own_norm=True, split=parts, split_offset=5, layout=layout)
        else:
            ctx.bb_rates(dr, 0.3, 1.0, gij, gji, precond=True, largest=True, own_norm=True, split=parts, split_offset=5,
                         layout=layout)
        out.append((chi, S, gij, gji, up))
    torch.cuda.synchronize()
    assert float(out[0][2].abs().max()) > 0 and (not flags or not torch.equal(out[0][4], raised))
    for a, b, what in zip(*out, ("chi", "S", "gamma_ij", "gamma_ji", "raised flags")):
        assert torch.equal(a, b), (what, float((a.double() - b.double()).abs().max()))


def test_tracking_flags_that_contradict_are_refused(ctx):
    """Tracking arrays together with M3DRT_BBOP_TRACK would stay unwritten, and
    m3drt_bb_opacity has no such form: both are errors, and nothing is written."""
    import ctypes as C
    from dispatch_amd import m3drt, synth
    from dispatch_amd.ali import NlteProblem
    p = NlteProblem(ctx, small())
    w = p.windows[0]
    l0, l1, nf, nc = w.lines[0], w.lines[-1] + 1, w.nf, p.ncell
    d = dict(w.const, vproj=(p.vz * (p.vec[0][2] / synth.C_LIGHT)).float().contiguous(), b=p.b, nstar=p.nstar,
             pop_ratio=p.pop_ratio, inv_df=p.inv_df, e_kT=p.e_kT32, adamp=p.adamp[l0:l1])
    chi, S = torch.full_like(w.chi_c, 3.0), torch.full_like(w.chi_c, 3.0)
    sp = {k: torch.full_like(w.chi_c, 3.0) for k in ("split_opac1", "split_opac2", "split_chi1", "split_chi2")}
    sp.update({k: torch.full((nf, nc), 3, dtype=torch.int32, device="cuda") for k in ("split_id", "split_chi_id")})
    with pytest.raises(m3drt.M3drtError, match="one of the two"):
        ctx.window_opacity(d, w.chi_c, w.Bnu, w.beta, chi, S, split=sp, track=True)
    ptr = lambda t: C.c_void_p(t.data_ptr())
    a = m3drt.BbOpacityArgs(l1 - l0, nf, nc, p.b.shape[0], m3drt.M3DRT_BBOP_TRACK, 0, 0.0, nc, 1,
                            *[ptr(d[k]) for k in ("iblue", "ired", "lev_i", "lev_j", "Bij", "lower_off", "q")], None,
                            None, *[ptr(d[k]) for k in ("b", "nstar", "pop_ratio", "inv_df", "vproj", "e_kT", "adamp")],
                            ptr(chi), ptr(S), *[None] * 7)
    with pytest.raises(m3drt.M3drtError, match="m3drt_window_opacity's"):
        m3drt._check(m3drt._ali_lib().m3drt_bb_opacity(ctx._h, C.byref(a)), "m3drt_bb_opacity")
    torch.cuda.synchronize()
    for t in (chi, S, *sp.values()):
        assert bool((t == 3).all())


def test_graph_replays_of_the_rate_pass_match_eager(ctx):
    """AliConfig(graph=True): the rate pass captured once and replayed, with the
    statistical-equilibrium update (eager work) between the replays, gives the eager
    pass's rate sums and departure coefficients bit for bit, iteration after
    iteration."""
    from dispatch_amd.ali import NlteProblem
    pe = NlteProblem(ctx, small())
    pg = NlteProblem(ctx, small(graph=True))
    print("ali rate pass: graph replays vs eager", flush=True)
    for it in range(4):
        ge, je = pe.rates()
        gg, jg = pg.rates()
        torch.cuda.synchronize()
        assert torch.equal(ge, gg) and torch.equal(je, jg), it
        pe.update(ge, je)
        pg.update(gg, jg)
        torch.cuda.synchronize()
        assert torch.equal(pe.b, pg.b), it
    assert pg._graph is not None
