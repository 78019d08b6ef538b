"""GPU parity of the statistical-equilibrium update (m3drt_rate_solve_f64,
m3drt_normalize_rates) against the oracle's restatement of
setup_transition_matrix + lineq_no_pivot + update_populations.  FP64 throughout,
same operation order: departure coefficients to 1e-12 relative, the convergence
measure's cell and level exactly."""
import numpy as np
import pytest
import torch

from nlte_cases import make_se_case
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def dev(a, dt):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device="cuda")


@pytest.mark.parametrize("seed,ncell,kw", [(5, 1000, {}), (6, 777, dict(max_update=3.0)),
                                            (7, 300, dict(conv_pop_floor=1e-4, sor_w=0.7))])
def test_rate_solve_matches_oracle(ctx, seed, ncell, kw):
    from dispatch_amd import m3drt
    c = make_se_case(ncell=ncell, seed=seed)
    print(f"rate solve seed={seed} ncell={ncell} {kw}", flush=True)
    bref, rref = O.update_populations(c["atom"], c["e_kT"], c["T"], c["totn"], c["nstar"], c["b"], c["gij"],
                                      c["gji"], c["cup"], **kw)
    at = m3drt.AtomOnDevice(c["atom"])
    b = dev(c["b"], torch.float64)
    r = ctx.rate_solve(at, dev(c["e_kT"], torch.float64), dev(c["T"], torch.float64),
                       dev(c["totn"], torch.float64), dev(c["nstar"], torch.float64), b,
                       dev(c["gij"], torch.float32), dev(c["gji"], torch.float32),
                       dev(c["cup"], torch.float64), **kw)
    got = b.cpu().numpy()
    assert np.max(np.abs(got - bref) / np.abs(bref)) < 1e-12
    assert (r["epos"], r["elvl"]) == (rref["epos"], rref["elvl"])
    assert r["maxerr"] == pytest.approx(rref["maxerr"], rel=1e-12)
    assert r["nclamp"] == rref["nclamp"]
    assert np.allclose(r["lvlerr"], rref["lvlerr"], rtol=1e-10, atol=0)


def test_normalize_rates_matches_oracle(ctx):
    from dispatch_amd import m3drt, synth
    rng = np.random.default_rng(9)
    atom = synth.make_atom()
    ncell = 500
    T = rng.uniform(4500, 8000, ncell)
    nstar = synth.lte_populations(atom, T, 10 ** rng.uniform(12, 15, ncell), np.ones(ncell) * 1e8)
    gij = rng.uniform(0, 1, (len(atom.ti), ncell)).astype(np.float32)
    gji = rng.uniform(0, 1, (len(atom.ti), ncell)).astype(np.float32)
    wphi = rng.uniform(0.5, 2, (len(atom.ti), ncell)).astype(np.float32)
    rij, rji = O.normalize_rates(atom, nstar, gij, gji, wphi)
    dij, dji = dev(gij, torch.float32), dev(gji, torch.float32)
    ctx.normalize_rates(m3drt.AtomOnDevice(atom), dev(nstar, torch.float64), dij, dji, dev(wphi, torch.float32))
    torch.cuda.synchronize()
    assert np.array_equal(dij.cpu().numpy(), rij)
    assert np.array_equal(dji.cpu().numpy(), rji)


def test_rate_solve_lte_fixed_point(ctx):
    from dispatch_amd import m3drt
    c = make_se_case(ncell=2000, seed=10, lte=True)
    b = dev(c["b"], torch.float64)
    r = ctx.rate_solve(m3drt.AtomOnDevice(c["atom"]), dev(c["e_kT"], torch.float64), dev(c["T"], torch.float64),
                       dev(c["totn"], torch.float64), dev(c["nstar"], torch.float64), b,
                       dev(c["gij"], torch.float32), dev(c["gji"], torch.float32), dev(c["cup"], torch.float64))
    assert np.max(np.abs(b.cpu().numpy() - 1.0)) < 1e-5
    assert abs(r["maxerr"]) < 1e-5


@pytest.mark.parametrize("nbound,nline,ncont,ncell", [(2, 1, 2, 1), (4, 6, 4, 41), (15, 60, 15, 7), (20, 80, 20, 40),
                                                     (62, 300, 62, 9), (110, 400, 110, 3)])
def test_rate_solve_sizes(ctx, monkeypatch, nbound, nline, ncont, ncell):
    """Level counts below, at and above the sixteen lanes of a cell, workgroups of 40, 4 and
    1 cells, the last one partly filled: against the oracle as above (1e-10: the rounding of
    the elimination grows with the level count in both)."""
    import functools
    from dispatch_amd import m3drt, synth
    monkeypatch.setattr(synth, "make_atom", functools.partial(synth.make_atom, nbound=nbound))
    c = make_se_case(ncell=ncell, seed=ncell, nline=nline, ncont=ncont)
    print(f"rate solve nbound={nbound} nline={nline} ncell={ncell}", flush=True)
    bref, rref = O.update_populations(c["atom"], c["e_kT"], c["T"], c["totn"], c["nstar"], c["b"], c["gij"],
                                      c["gji"], c["cup"])
    b = dev(c["b"], torch.float64)
    r = ctx.rate_solve(m3drt.AtomOnDevice(c["atom"]), dev(c["e_kT"], torch.float64), dev(c["T"], torch.float64),
                       dev(c["totn"], torch.float64), dev(c["nstar"], torch.float64), b,
                       dev(c["gij"], torch.float32), dev(c["gji"], torch.float32), dev(c["cup"], torch.float64))
    assert np.max(np.abs(b.cpu().numpy() - bref) / np.abs(bref)) < 1e-10
    assert (r["epos"], r["elvl"]) == (rref["epos"], rref["elvl"])
    assert r["nclamp"] == rref["nclamp"]
    assert np.allclose(r["lvlerr"], rref["lvlerr"], rtol=1e-8, atol=1e-10)


@pytest.mark.parametrize("nbound,nline,ncont,ncell", [(2, 1, 2, 16385), (4, 5, 4, 16500), (8, 14, 8, 20000), (15, 60, 15, 16390),
                                                      (16, 60, 16, 16390)])
def test_rate_solve_of_many_cells_equals_few_at_a_time(ctx, monkeypatch, nbound, nline, ncont, ncell):
    """Four lanes a cell take many cells of up to 16 levels, sixteen the others, with the
    same operations in the same order: one call over all cells against calls of at most
    16 384, the populations bit for bit and the largest changes and their cells."""
    import functools
    from dispatch_amd import m3drt, synth
    monkeypatch.setattr(synth, "make_atom", functools.partial(synth.make_atom, nbound=nbound))
    c = make_se_case(ncell=ncell, seed=nbound, nline=nline, ncont=ncont)
    print(f"rate solve of many cells nbound={nbound} ncell={ncell}", flush=True)
    atom = m3drt.AtomOnDevice(c["atom"])

    def solve(cells):
        d = lambda k, dt: dev(c[k][..., cells], dt)
        b = d("b", torch.float64)
        r = ctx.rate_solve(atom, d("e_kT", torch.float64), d("T", torch.float64), d("totn", torch.float64),
                           d("nstar", torch.float64), b, d("gij", torch.float32), d("gji", torch.float32),
                           d("cup", torch.float64))
        return b, r

    b, r = solve(slice(0, ncell))
    parts = [(c0, *solve(slice(c0, min(ncell, c0 + 8192)))) for c0 in range(0, ncell, 8192)]
    assert torch.equal(b, torch.cat([p[1] for p in parts], 1))
    assert r["nclamp"] == sum(p[2]["nclamp"] for p in parts)
    c0, _, best = max(parts, key=lambda p: abs(p[2]["maxerr"]))
    assert (r["maxerr"], r["epos"], r["elvl"]) == (best["maxerr"], best["epos"] + c0, best["elvl"])
    assert np.max(np.abs(r["lvlerr"])) == np.max(np.abs([p[2]["lvlerr"] for p in parts]))
