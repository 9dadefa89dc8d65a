"""Amplitude-ratio kernels of the RBMs (csrc/rbmq.hpp) against the FP64 oracle
at the sizes where their tiling can go wrong: hidden units around a wavefront
and above the eight-sample tile's limit, strings that fill less than, exactly
and more than a pass, sample counts around a tile, operators whose strings
leave sites unchanged, repeat each other or change more than two sites, and
parameters outside the products' range (which take the log-cosh form).

Tolerance 1e-11 relative, as for every E_loc comparison: each term is a product
of H + 2 factors, each within a few rounding errors of exact."""
import numpy as np
import pytest
import torch

from oracle import nets as onets
from oracle import operator as oop
from oracle import sampler as osamp

from helpers import tfim_pair, to_np, xxz_pair

pytestmark = pytest.mark.gpu

jv = pytest.importorskip("vmc_jax_amd")

TOL = 1e-11


def _mixed_pair(L):
    """Strings of every kind the kernels tell apart: repeated and padded
    flips, flips that cancel, raising / lowering pairs (no flip on half the
    configurations), complex elements, a single diagonal string."""
    from vmc_jax_amd import operator as dop
    out = []
    for o in (dop, oop):
        H = o.BranchFreeOperator()
        for i in range(L):
            j = (i + 1) % L
            H.add(o.scal_opstr(0.3, (o.Sx(i),)))
            H.add(o.scal_opstr(0.2 + 0.1j, (o.Sy(i),)))
            H.add(o.scal_opstr(0.7, (o.Sp(i), o.Sm(j))))
            H.add(o.scal_opstr(0.5, (o.Sm(i), o.Sp(j))))
            H.add(o.scal_opstr(0.4, (o.Sx(i), o.Sz(j))))
        H.add(o.scal_opstr(0.9, (o.Sx(0), o.Sx(0))))
        H.add(o.scal_opstr(1.1, (o.Sz(1),)))
        out.append(H)
    return out


def _long_pair(L):
    """Three- and four-site strings (the general loop)."""
    from vmc_jax_amd import operator as dop
    out = []
    for o in (dop, oop):
        H = o.BranchFreeOperator()
        for i in range(L):
            a, b, c = (i + 1) % L, (i + 2) % L, (i + 3) % L
            H.add(o.scal_opstr(0.3, (o.Sx(i), o.Sx(a), o.Sx(b))))
            H.add(o.scal_opstr(0.2, (o.Sx(i), o.Sy(a), o.Sx(b), o.Sy(c))))
            H.add(o.scal_opstr(-0.5, (o.Sz(i), o.Sz(a))))
        out.append(H)
    return out


OPS = {"tfim": lambda L: tfim_pair((L,), -1.0, -0.7), "xxz": lambda L: xxz_pair(L, 0.6), "mixed": _mixed_pair,
       "long": _long_pair}


def _states(cpx, L, H, bias, vbias, P):
    if cpx:
        net, onet = jv.nets.CpxRBM(H, bias=bias, visibleBias=vbias), onets.CpxRBM((L,), H, bias=bias, visibleBias=vbias)
    else:
        net, onet = jv.nets.RBM(H, bias=bias), onets.RBM((L,), H, bias=bias)
    psi = jv.NQS(net)
    psi(torch.zeros((1, 1, L), dtype=torch.int32))
    psi.set_parameters(P)
    return psi, onets.NQS(onet, P)


def _num(cpx, L, H, bias, vbias):
    return (2 if cpx else 1) * (L * H + (H if bias else 0) + (L if vbias else 0))


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("cpx,L,H,bias,vbias,op,n", [
    (True, 10, 20, True, True, "tfim", 9), (True, 5, 1, False, False, "tfim", 1), (True, 8, 63, True, False, "xxz", 7),
    (True, 7, 64, False, True, "mixed", 8), (True, 33, 65, True, False, "tfim", 5), (False, 12, 130, True, False, "xxz", 20),
    (False, 6, 3, False, False, "mixed", 33), (True, 65, 40, True, False, "tfim", 6), (True, 70, 9, True, True, "xxz", 5),
    (True, 6, 257, True, False, "mixed", 5), (True, 9, 12, True, True, "long", 10), (False, 9, 70, True, False, "long", 3),
    (True, 4, 6, True, False, "mixed", 8200)])
def test_eloc(cpx, L, H, bias, vbias, op, n):
    rng = np.random.default_rng(L * 1000 + H)
    P = 0.3 / np.sqrt(L) * rng.normal(size=_num(cpx, L, H, bias, vbias))
    psi, opsi = _states(cpx, L, H, bias, vbias, P)
    Hd, Ho = OPS[op](L)
    s = rng.integers(0, 2, size=(n, L)).astype(np.int32)
    sd = torch.as_tensor(s[None], device="cuda")
    e = to_np(Hd.get_O_loc(sd, psi, psi(sd)))[0]
    ref = Ho.get_O_loc(s, opsi, opsi(s))
    assert _rel(e, ref) < TOL


@pytest.mark.parametrize("H,L,op", [(257, 6, "mixed"), (300, 48, "tfim"), (900, 17, "xxz")])
def test_eloc_two_sample_tiles(H, L, op):
    """More than 256 hidden units: two samples per workgroup of four waves, many
    full tiles; every sample keeps its own amplitude."""
    n = 301
    rng = np.random.default_rng(H)
    P = 0.3 / np.sqrt(L) * rng.normal(size=_num(True, L, H, True, False))
    P[2 * H:] *= 0.3  # |Re theta| and the sites' summed |Re W| stay in range
    psi, opsi = _states(True, L, H, True, False, P)
    Hd, Ho = OPS[op](L)
    s = rng.integers(0, 2, size=(n, L)).astype(np.int32)
    sd = torch.as_tensor(s[None], device="cuda")
    e = to_np(Hd.get_O_loc(sd, psi, psi(sd)))[0]
    ref = Ho.get_O_loc(s, opsi, opsi(s))
    assert np.max(np.abs(e - ref)) < TOL * np.max(np.abs(ref))


def _late_pair(L, where):
    """A transverse field with one string that flips no spin (two Sx on one
    site) at position `where` of the list."""
    from vmc_jax_amd import operator as dop
    out = []
    for o in (dop, oop):
        H = o.BranchFreeOperator()
        for k in range(2 * L):
            if k == where:
                H.add(o.scal_opstr(0.9, (o.Sx(1), o.Sx(1))))
            H.add(o.scal_opstr(0.3 + 0.01 * k, (o.Sx(k % L),)))
        out.append(H)
    return out


@pytest.mark.parametrize("cpx,H,strings,n", [(True, 64, 3, 2000), (True, 64, 3, 2001), (True, 65, 1, 3000), (True, 65, 2, 5),
                                             (False, 640, 1, 1200), (False, 256, 2, 1501), (False, 300, 1, 3000), (False, 641, 2, 5), (True, 5, 1, 6001)])
def test_eloc_few_strings(cpx, H, strings, n):
    """Either side of the rule that gives few strings on few samples to the
    log-cosh kernel."""
    from vmc_jax_amd import operator as dop
    L = 5
    rng = np.random.default_rng(H)
    P = 0.3 / np.sqrt(L) * rng.normal(size=_num(cpx, L, H, True, False))
    psi, opsi = _states(cpx, L, H, True, False, P)
    Hd, Ho = dop.BranchFreeOperator(), oop.BranchFreeOperator()
    for k in range(strings):
        Hd.add(dop.scal_opstr(0.5 + k, (dop.Sx(k), dop.Sz(4))))
        Ho.add(oop.scal_opstr(0.5 + k, (oop.Sx(k), oop.Sz(4))))
    s = rng.integers(0, 2, size=(n, L)).astype(np.int32)
    sd = torch.as_tensor(s[None], device="cuda")
    e = to_np(Hd.get_O_loc(sd, psi, psi(sd)))[0]
    assert _rel(e, Ho.get_O_loc(s, opsi, opsi(s))) < TOL


@pytest.mark.parametrize("L,H,n,where", [(2, 1, 9000, 0), (2, 1, 40, 3), (50, 5, 60, 0), (50, 5, 60, 63),
                                         (50, 5, 60, 64), (50, 5, 60, 99)])
def test_eloc_string_that_flips_nothing(L, H, n, where):
    """The workgroup's flag for such strings, set in the first pass of 64 strings
    or in a later one, with a theta phase too short to hide a late clear."""
    rng = np.random.default_rng(where)
    P = 0.3 * rng.normal(size=_num(True, L, H, True, False))
    psi, opsi = _states(True, L, H, True, False, P)
    Hd, Ho = _late_pair(L, where)
    s = rng.integers(0, 2, size=(n, L)).astype(np.int32)
    sd = torch.as_tensor(s[None], device="cuda")
    e = to_np(Hd.get_O_loc(sd, psi, psi(sd)))[0]
    ref = Ho.get_O_loc(s, opsi, opsi(s))
    assert np.max(np.abs(e - ref) / np.abs(ref)) < TOL


def test_eloc_more_tiles_than_a_launch_has_workgroups():
    """2^24 tiles and a few samples: as many workgroups of 256 threads are more
    threads than a launch takes."""
    L, H, n = 2, 1, (1 << 24) * 8 + 37
    rng = np.random.default_rng(2)
    P = 0.3 * rng.normal(size=_num(False, L, H, True, False))
    psi, opsi = _states(False, L, H, True, False, P)
    Hd, Ho = tfim_pair((L,), -1.0, -0.7)
    basis = np.array([[0, 0], [0, 1], [1, 0], [1, 1]], dtype=np.int32)
    table = torch.as_tensor(Ho.get_O_loc(basis, opsi, np.zeros(4)), device="cuda").to(torch.complex128)
    s = torch.randint(0, 2, (1, n, L), dtype=torch.int32, device="cuda")
    e = Hd.get_O_loc(s, psi, torch.zeros((1, n), dtype=torch.complex128, device="cuda"))[0]
    for a in range(0, n, 1 << 24):
        b = min(n, a + (1 << 24))
        ref = table[(2 * s[0, a:b, 0] + s[0, a:b, 1]).long()]
        assert float((e[a:b] - ref).abs().max()) < TOL


@pytest.mark.parametrize("big", [10.0, 60.0])
def test_eloc_out_of_range(big):
    """A site whose summed |Re W| (80, 480) or a unit whose |Re theta| leaves the
    ratio form's range: the log-cosh form gives the oracle's values."""
    L, H = 6, 8
    rng = np.random.default_rng(3)
    P = 0.1 * rng.normal(size=_num(True, L, H, False, False))
    P[:H] = big * np.sign(P[:H])  # Re W of site 0
    psi, opsi = _states(True, L, H, False, False, P)
    Hd, Ho = _mixed_pair(L)
    s = rng.integers(0, 2, size=(11, L)).astype(np.int32)
    sd = torch.as_tensor(s[None], device="cuda")
    e = to_np(Hd.get_O_loc(sd, psi, psi(sd)))[0]
    ref = Ho.get_O_loc(s, opsi, opsi(s))
    assert np.all(np.isfinite(ref))
    assert np.max(np.abs(e - ref) / np.abs(ref)) < TOL


@pytest.mark.parametrize("cpx,L,H,vbias,op,n", [
    (True, 5, 1, False, "tfim", 3), (False, 7, 65, False, "mixed", 9), (True, 9, 130, True, "long", 10),
    (True, 6, 257, False, "xxz", 5), (False, 5, 900, False, "mixed", 7), (True, 4, 6, True, "mixed", 8200)])
def test_eloc_out_of_range_sizes(cpx, L, H, vbias, op, n):
    """The form for parameters out of range over units per lane, samples per
    workgroup, real networks and strings of more than two sites."""
    rng = np.random.default_rng(L * 1000 + H)
    P = 0.3 / np.sqrt(L) * rng.normal(size=_num(cpx, L, H, True, vbias))
    P[(2 if cpx else 1) * H] = 90.0
    psi, opsi = _states(cpx, L, H, True, vbias, P)
    Hd, Ho = OPS[op](L)
    s = rng.integers(0, 2, size=(n, L)).astype(np.int32)
    lpo = opsi(s)
    e = to_np(Hd.get_O_loc(torch.as_tensor(s[None], device="cuda"), psi, torch.as_tensor(lpo[None], device="cuda")))[0]
    ref = Ho.get_O_loc(s, opsi, lpo)
    assert np.max(np.abs(e - ref)) < TOL * np.max(np.abs(ref))
    big = np.abs(ref) > 1e-3 * np.max(np.abs(ref))
    assert np.max(np.abs(e - ref)[big] / np.abs(ref)[big]) < 1e-10


@pytest.mark.parametrize("cpx,L,H,vbias,mu", [
    (True, 70, 1, False, 2.0), (False, 12, 65, False, 1.0), (True, 9, 128, True, 2.0), (True, 8, 256, False, 0.5),
    (False, 6, 256, False, 0.0)])
def test_chains_out_of_range_sizes(cpx, L, H, vbias, mu):
    rng = np.random.default_rng(L * 100 + H)
    P = 0.3 / np.sqrt(L) * rng.normal(size=_num(cpx, L, H, True, vbias))
    P[(2 if cpx else 1) * H] = 90.0
    psi, opsi = _states(cpx, L, H, True, vbias, P)
    kw = dict(numChains=6, numSamples=24, thermalizationSweeps=5, sweepSteps=45, mu=mu)
    ms = jv.sampler.MCSampler(psi, (L,), 17, updateProposer=jv.sampler.propose_spin_flip, **kw)
    mo = osamp.MCSampler(opsi, (L,), 17, **kw)
    for _ in range(2):
        assert np.array_equal(to_np(ms.sample()[0])[0], mo.sample()[0])
    assert np.array_equal(to_np(ms.states), mo.states)
    assert abs(float(ms.acceptance_ratio()[0]) - float(np.ravel(mo.acceptance_ratio())[0])) < 1e-15


def _hop_pair(L):
    """Hopping strings (they keep the number of up spins) and a diagonal one."""
    from vmc_jax_amd import operator as dop
    out = []
    for o in (dop, oop):
        H = o.BranchFreeOperator()
        for i in range(L):
            j = (i + 1) % L
            H.add(o.scal_opstr(0.7, (o.Sp(i), o.Sm(j))))
            H.add(o.scal_opstr(0.7, (o.Sm(i), o.Sp(j))))
        H.add(o.scal_opstr(1.1, (o.Sz(1),)))
        out.append(H)
    return out


@pytest.mark.parametrize("mu", [2.0, 0.0])
def test_large_visible_bias(mu):
    """|Re a| = 400 on every site: the factor of one flipped site over- or
    underflows, that of a hop (and every log) does not; with mu = 0 every
    proposal is accepted whatever the ratio."""
    L, H = 6, 8
    rng = np.random.default_rng(13)
    P = 0.1 * rng.normal(size=_num(True, L, H, True, True))
    P[-2 * L:-L] = 400.0  # Re a
    psi, opsi = _states(True, L, H, True, True, P)
    Hd, Ho = _hop_pair(L)
    s = rng.integers(0, 2, size=(20, L)).astype(np.int32)
    sd = torch.as_tensor(s[None], device="cuda")
    e = to_np(Hd.get_O_loc(sd, psi, psi(sd)))[0]
    ref = Ho.get_O_loc(s, opsi, opsi(s))
    assert np.all(np.isfinite(ref))
    # log psi is 2400 in size: its rounding error is the exponent's
    assert np.max(np.abs(e - ref) / np.abs(ref)) < 1e-10
    kw = dict(numChains=3, numSamples=9, thermalizationSweeps=2, sweepSteps=20, mu=mu)
    ms = jv.sampler.MCSampler(psi, (L,), 17, updateProposer=jv.sampler.propose_spin_flip, **kw)
    mo = osamp.MCSampler(opsi, (L,), 17, **kw)
    assert np.array_equal(to_np(ms.sample()[0])[0], mo.sample()[0])


def test_eloc_nan_parameters():
    L, H = 6, 8
    P = 0.1 * np.random.default_rng(4).normal(size=_num(True, L, H, True, False))
    P[3] = np.nan
    psi, _ = _states(True, L, H, True, False, P)
    Hd, _ = tfim_pair((L,), -1.0, -0.7)
    sd = torch.zeros((1, 5, L), dtype=torch.int32, device="cuda")
    e = to_np(Hd.get_O_loc(sd, psi, torch.zeros((1, 5), dtype=torch.complex128, device="cuda")))
    assert np.all(np.isnan(e))


def test_eloc_streams():
    """Calls on two streams of one thread, each with its own parameters, keep
    their tables apart."""
    L, H, n = 10, 20, 4000
    rng = np.random.default_rng(5)
    Hd, _ = tfim_pair((L,), -1.0, -0.7)
    Hd.compile()
    sd = torch.as_tensor(rng.integers(0, 2, size=(1, n, L)).astype(np.int32), device="cuda")
    psis = [_states(True, L, H, True, False, 0.1 * rng.normal(size=_num(True, L, H, True, False)))[0] for _ in range(2)]
    lps = [p(sd) for p in psis]
    ref = [Hd.get_O_loc(sd, p, lp).clone() for p, lp in zip(psis, lps)]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    out = [[], []]
    for _ in range(4):
        for k, st in enumerate(streams):
            with torch.cuda.stream(st):
                out[k].append(Hd.get_O_loc(sd, psis[k], lps[k]))
    torch.cuda.synchronize()
    for k in range(2):
        assert all(torch.equal(o, ref[k]) for o in out[k])


def test_eloc_many_streams():
    """Calls in turn on more streams than eight do not wait for the device."""
    L, H = 10, 20
    rng = np.random.default_rng(6)
    Hd, _ = tfim_pair((L,), -1.0, -0.7)
    psi, _ = _states(True, L, H, True, False, 0.1 * rng.normal(size=_num(True, L, H, True, False)))
    sd = torch.as_tensor(rng.integers(0, 2, size=(1, 40, L)).astype(np.int32), device="cuda")
    lp = psi(sd)
    ref = Hd.get_O_loc(sd, psi, lp)
    streams = [torch.cuda.Stream() for _ in range(20)]
    busy = torch.cuda.Stream()
    torch.cuda.synchronize()

    def turn():
        out = []
        for st in streams:
            with torch.cuda.stream(st):
                out.append(Hd.get_O_loc(sd, psi, lp))
        return out

    turn()  # buffers of every stream
    torch.cuda.synchronize()
    done = torch.cuda.Event()
    with torch.cuda.stream(busy):
        torch.cuda._sleep(200_000_000)  # 2 s at the 100 MHz counter, less at the core clock
        done.record()
    out = turn()
    waited = done.query()
    torch.cuda.synchronize()
    assert all(torch.equal(o, ref) for o in out)
    assert not waited


@pytest.mark.parametrize("cpx,L,H,bias,vbias,mu,big", [
    (True, 10, 20, True, True, 2.0, 0.0), (True, 7, 1, False, False, 1.0, 0.0), (False, 12, 65, True, False, 2.0, 0.0),
    (True, 65, 130, True, False, 2.0, 0.0), (False, 9, 256, False, False, 0.5, 0.0), (True, 6, 257, True, False, 2.0, 0.0),
    (True, 6, 8, False, False, 2.0, 10.0), (True, 8, 64, True, False, 0.0, 0.0)])
def test_chains(cpx, L, H, bias, vbias, mu, big):
    """Configurations, counters and walkers of the chains equal the oracle's
    (sites beyond one word of spins, several units per lane, the sizes and the
    weights that take the log-cosh form, every mu); long sweeps cross the
    interval after which theta is recomputed."""
    rng = np.random.default_rng(L * 100 + H)
    P = 0.3 / np.sqrt(L) * rng.normal(size=_num(cpx, L, H, bias, vbias))
    if big:
        P[:H] = big
    psi, opsi = _states(cpx, L, H, bias, vbias, P)
    kw = dict(numChains=6, numSamples=24, thermalizationSweeps=5, sweepSteps=45, mu=mu)
    ms = jv.sampler.MCSampler(psi, (L,), 17, updateProposer=jv.sampler.propose_spin_flip, **kw)
    mo = osamp.MCSampler(opsi, (L,), 17, **kw)
    for _ in range(2):
        s, lp, p = ms.sample()
        so, lpo, po = mo.sample()
        assert np.array_equal(to_np(s)[0], so)
        assert _rel(to_np(lp)[0], lpo) < TOL
    assert np.array_equal(to_np(ms.states), mo.states)
    assert abs(float(ms.acceptance_ratio()[0]) - float(np.ravel(mo.acceptance_ratio())[0])) < 1e-15


def _xxz_bond(L):
    """XXZ on one bond."""
    from vmc_jax_amd import operator as dop
    out = []
    for o in (dop, oop):
        H = o.BranchFreeOperator()
        for c, a in ((1.0, o.Sx), (1.0, o.Sy), (0.5, o.Sz)):
            H.add(o.scal_opstr(c, (a(1), a(2))))
        out.append(H)
    return out


def _sym_states(cpx, L, H, names, P, **kw):
    import warnings

    from oracle import symmetries as osym
    with warnings.catch_warnings():
        warnings.simplefilter("ignore", UserWarning)
        orb = jv.util.symmetries.get_orbit_1D(L, *names, **kw)
        d, f = osym.orbit_1d(L, *names, **kw)
    net, onet = (jv.nets.CpxRBM(H, bias=True), onets.CpxRBM((L,), H, bias=True)) if cpx else \
        (jv.nets.RBM(H, bias=True), onets.RBM((L,), H, bias=True))
    psi = jv.NQS(net, orbit=orb)
    psi(torch.zeros((1, 1, L), dtype=torch.int32))
    psi.set_parameters(P)
    return psi, onets.NQS(osym.SymNet(onet, d, f, "exp"), P)


ALL = ("translation", "reflection", "spinflip")


@pytest.mark.parametrize("cpx,L,H,names,op,big", [
    (True, 5, 1, ("reflection",), "tfim", 0.0), (True, 17, 9, ALL, "xxz", 0.0), (False, 9, 33, ALL, "mixed", 0.0),
    (True, 12, 70, ("translation",), "tfim", 0.0), (True, 9, 150, ALL, "xxz", 0.0), (True, 6, 300, ("translation",), "mixed", 0.0),
    (True, 33, 8, ALL, "tfim", 0.0), (True, 6, 8, ALL, "mixed", 10.0), (True, 6, 5, ALL, "long", 0.0)])
def test_sym_resident(cpx, L, H, names, op, big):
    """Symmetrised RBMs: log psi, local energies and chains against the oracle
    over row counts below, at and above the kernels' chunks (2 to 132), units
    beyond one pass, the smaller row tiles, a group and unit count too large
    for one workgroup's chain, out-of-range weights, and strings the resident
    form leaves to the materialised one."""
    rng = np.random.default_rng(L * 1000 + H)
    P = 0.3 / np.sqrt(L) * rng.normal(size=_num(cpx, L, H, True, False))
    if big:
        P[2 * H:3 * H] = big
    psi, opsi = _sym_states(cpx, L, H, names, P)
    s = rng.integers(0, 2, size=(7, L)).astype(np.int32)
    sd = torch.as_tensor(s[None], device="cuda")
    lp, lpo = psi(sd), opsi(s)
    assert np.max(np.abs(to_np(lp)[0] - lpo)) < TOL * np.max(np.abs(lpo))
    Hd, Ho = OPS[op](L)
    e = to_np(Hd.get_O_loc(sd, psi, lp))[0]
    assert _rel(e, Ho.get_O_loc(s, opsi, lpo)) < TOL
    kw = dict(numChains=3, numSamples=9, thermalizationSweeps=3, sweepSteps=50)
    ms = jv.sampler.MCSampler(psi, (L,), 5, updateProposer=jv.sampler.propose_spin_flip, **kw)
    mo = osamp.MCSampler(opsi, (L,), 5, **kw)
    for _ in range(2):
        so = mo.sample()[0]
        assert np.array_equal(to_np(ms.sample()[0])[0], so)
    assert np.array_equal(to_np(ms.states), mo.states)
    assert float(ms.acceptance_ratio()[0]) == float(np.ravel(mo.acceptance_ratio())[0])


@pytest.mark.parametrize("big", [0.0, 90.0])
@pytest.mark.parametrize("cpx,L,H,names", [
    (True, 10, 1, ("reflection",)), (True, 11, 200, ("reflection",)), (False, 6, 300, ("reflection",)),
    (True, 8, 130, ("translation",)), (True, 16, 33, ("translation",)), (True, 24, 8, ALL), (False, 16, 32, ALL)])
def test_sym_log_psi(cpx, L, H, names, big):
    """log psi over every split of a row between threads (4 to 64 threads, one
    or four units each), weights of ordinary size and far outside the ratio
    form's range."""
    rng = np.random.default_rng(L * 1000 + H)
    P = 0.3 / np.sqrt(L) * rng.normal(size=_num(cpx, L, H, True, False))
    if big:
        P[(2 if cpx else 1) * H] = big
    psi, opsi = _sym_states(cpx, L, H, names, P)
    s = rng.integers(0, 2, size=(13, L)).astype(np.int32)
    lp, lpo = to_np(psi(torch.as_tensor(s[None], device="cuda")))[0], opsi(s)
    assert np.max(np.abs(lp - lpo)) < TOL * np.max(np.abs(lpo))


@pytest.mark.parametrize("cpx,L,H,names,op,mu", [
    (True, 10, 1, ("reflection",), "tfim", 2.0), (True, 11, 200, ("reflection",), "xxz", 2.0),
    (False, 6, 300, ("reflection",), "mixed", 1.0), (True, 8, 40, ("translation",), "mixed", 2.0),
    (True, 24, 8, ALL, "tfim", 0.5), (False, 16, 32, ALL, "xxz", 2.0)])
def test_sym_out_of_range(cpx, L, H, names, op, mu):
    """Local energies and chains with a weight far outside the ratio form's
    range, over the splits of a row between threads."""
    rng = np.random.default_rng(L * 1000 + H)
    P = 0.3 / np.sqrt(L) * rng.normal(size=_num(cpx, L, H, True, False))
    P[(2 if cpx else 1) * H] = 90.0
    psi, opsi = _sym_states(cpx, L, H, names, P)
    s = rng.integers(0, 2, size=(13, L)).astype(np.int32)
    sd = torch.as_tensor(s[None], device="cuda")
    Hd, Ho = OPS[op](L)
    lpo = opsi(s)
    e = to_np(Hd.get_O_loc(sd, psi, torch.as_tensor(lpo[None], device="cuda")))[0]
    ref = Ho.get_O_loc(s, opsi, lpo)
    # log psi is some 1e3 in size: its rounding error is the exponent's
    assert np.max(np.abs(e - ref)) < 1e-10 * np.max(np.abs(ref))
    kw = dict(numChains=3, numSamples=9, thermalizationSweeps=2, sweepSteps=30, mu=mu)
    ms = jv.sampler.MCSampler(psi, (L,), 5, updateProposer=jv.sampler.propose_spin_flip, **kw)
    mo = osamp.MCSampler(opsi, (L,), 5, **kw)
    for _ in range(2):
        assert np.array_equal(to_np(ms.sample()[0])[0], mo.sample()[0])
    assert np.array_equal(to_np(ms.states), mo.states)
    assert float(ms.acceptance_ratio()[0]) == float(np.ravel(mo.acceptance_ratio())[0])


@pytest.mark.parametrize("cpx,L,H,names", [(True, 10, 20, ("reflection",)), (True, 12, 70, ALL), (False, 16, 32, ALL),
                                           (True, 6, 200, ("reflection",))])
def test_sym_eloc_forms(cpx, L, H, names):
    """Local energies and log psi in each form the sizes choose between: one to
    many strings (with and without diagonal ones) on one to some hundred
    samples, whose strings share a workgroup or have several."""
    from vmc_jax_amd import operator as dop
    rng = np.random.default_rng(L * 1000 + H)
    P = 0.3 / np.sqrt(L) * rng.normal(size=_num(cpx, L, H, True, False))
    psi, opsi = _sym_states(cpx, L, H, names, P)
    s = rng.integers(0, 2, size=(520, L)).astype(np.int32)
    lpo = opsi(s)
    for strings, diag in ((1, 0), (2, 0), (3, 1), (4, 3)):
        Hd, Ho = dop.BranchFreeOperator(), oop.BranchFreeOperator()
        for k in range(strings):
            Hd.add(dop.scal_opstr(0.5 + k, (dop.Sx(k), dop.Sx(5 - k) if k == 1 else dop.Sz(5 - k))))
            Ho.add(oop.scal_opstr(0.5 + k, (oop.Sx(k), oop.Sx(5 - k) if k == 1 else oop.Sz(5 - k))))
        for k in range(diag):
            Hd.add(dop.scal_opstr(0.3 * (k + 1), (dop.Sz(k), dop.Sz(k + 1))))
            Ho.add(oop.scal_opstr(0.3 * (k + 1), (oop.Sz(k), oop.Sz(k + 1))))
        ref = Ho.get_O_loc(s, opsi, lpo)
        for n in (1, 5, 100, 257, 520):
            sd = torch.as_tensor(s[None, :n].copy(), device="cuda")
            lp = psi(sd)
            assert np.max(np.abs(to_np(lp)[0] - lpo[:n])) < TOL * np.max(np.abs(lpo))
            e = to_np(Hd.get_O_loc(sd, psi, lp))[0]
            assert np.max(np.abs(e - ref[:n])) < TOL * np.max(np.abs(ref))


@pytest.mark.parametrize("cpx,L,H,mu", [(True, 9, 12, 1.0), (False, 9, 33, 0.5), (True, 8, 5, 0.0)])
def test_sym_chains_mu(cpx, L, H, mu):
    rng = np.random.default_rng(L * 100 + H)
    P = 0.3 / np.sqrt(L) * rng.normal(size=_num(cpx, L, H, True, False))
    psi, opsi = _sym_states(cpx, L, H, ALL, P)
    kw = dict(numChains=3, numSamples=9, thermalizationSweeps=3, sweepSteps=50, mu=mu)
    ms = jv.sampler.MCSampler(psi, (L,), 5, updateProposer=jv.sampler.propose_spin_flip, **kw)
    mo = osamp.MCSampler(opsi, (L,), 5, **kw)
    for _ in range(2):
        assert np.array_equal(to_np(ms.sample()[0])[0], mo.sample()[0])
    assert np.array_equal(to_np(ms.states), mo.states)


@pytest.mark.parametrize("L,H,n", [(10, 12, 2000), (12, 70, 40)])
def test_sym_streams(L, H, n):
    """Symmetrised calls on two streams of one thread, each with its own
    parameters, keep their scratch memory apart: enough samples to overlap, and
    few enough for the materialised rows."""
    rng = np.random.default_rng(15)
    Hd, _ = tfim_pair((L,), -1.0, -0.7)
    Hd.compile()
    sd = torch.as_tensor(rng.integers(0, 2, size=(1, n, L)).astype(np.int32), device="cuda")
    psis = [_sym_states(True, L, H, ALL, 0.1 * rng.normal(size=_num(True, L, H, True, False)))[0] for _ in range(2)]
    kw = dict(numChains=64, numSamples=64, thermalizationSweeps=2, sweepSteps=20)

    def calls(p):
        ms = jv.sampler.MCSampler(p, (L,), 5, updateProposer=jv.sampler.propose_spin_flip, **kw)
        lp = p(sd)
        return lp, Hd.get_O_loc(sd, p, lp), ms.sample()[0]
    ref = [[t.clone() for t in calls(p)] for p in psis]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    out = [[], []]
    for _ in range(8):
        for k, st in enumerate(streams):
            with torch.cuda.stream(st):
                out[k].append(calls(psis[k]))
    torch.cuda.synchronize()
    for k in range(2):
        assert all(torch.equal(a, b) for o in out[k] for a, b in zip(o, ref[k]))


def test_sym_eloc_negative_sums():
    """A real network's negative sums have no logarithm: the local energy is NaN
    where any string with a matrix element leads to one, also where it cancels
    against another string with the same s' (X X against Y Y)."""
    L, H = 7, 5
    P = 0.5 * np.random.default_rng(3).normal(size=_num(False, L, H, True, False))
    psi, opsi = _sym_states(False, L, H, ("reflection",), P, reflection_factor=-1.0)
    s = ((np.arange(2 ** L)[:, None] >> np.arange(L)) & 1).astype(np.int32)
    sp = s.copy()
    sp[:, 1:3] ^= 1
    asym = np.any(s != s[:, ::-1], axis=1) & np.any(sp != sp[:, ::-1], axis=1)  # sums that do not cancel
    s = s[asym & np.isfinite(opsi(s))]
    lpo = opsi(s)
    Hd, Ho = _xxz_bond(L)
    e = to_np(Hd.get_O_loc(torch.as_tensor(s[None], device="cuda"), psi, torch.as_tensor(lpo[None], device="cuda")))[0]
    ref = Ho.get_O_loc(s, opsi, lpo)
    assert np.isnan(ref).any() and np.isfinite(ref).any()
    assert np.array_equal(np.isnan(e), np.isnan(ref))
    ok = np.isfinite(ref)
    assert np.max(np.abs(e - ref)[ok]) < TOL * np.max(np.abs(ref[ok]))


@pytest.mark.parametrize("cpx,seed", [(True, 5), (True, 6), (False, 7)])
def test_sym_chain_rows_far_apart(cpx, seed):
    """Two rows (a chain and its mirror image) whose weights differ by e^{860}
    at the start, parameters in range: the lighter one still counts once flips
    during the thermalisation have made it the heavier."""
    L, H = 24, 16
    rng = np.random.default_rng(seed)
    k = 2 if cpx else 1
    P = 0.01 * rng.normal(size=_num(cpx, L, H, True, False))
    P[k * H:k * H + 12 * H] = 4.5  # Re W of the left half
    psi, opsi = _sym_states(cpx, L, H, ("reflection",), P)
    init = np.array([1] * 12 + [0, 1] * 6, dtype=np.int32)
    kw = dict(numChains=4, numSamples=8, thermalizationSweeps=40, sweepSteps=50, mu=0.01, initState=init)
    ms = jv.sampler.MCSampler(psi, (L,), seed, updateProposer=jv.sampler.propose_spin_flip, **kw)
    mo = osamp.MCSampler(opsi, (L,), seed, **kw)
    assert np.array_equal(to_np(ms.sample()[0])[0], mo.sample()[0])
    assert float(ms.acceptance_ratio()[0]) == float(np.ravel(mo.acceptance_ratio())[0])


@pytest.mark.parametrize("cpx", [True, False])
def test_sym_rows_that_are_no_permutation(cpx):
    """An orbit element may read a site twice, or never: (g s)_i = s_{m_i} all
    the same."""
    from oracle import symmetries as osym
    L, H, n = 6, 5, 30
    maps = np.array([[0, 1, 2, 3, 4, 5], [0, 0, 2, 3, 4, 5], [1, 2, 2, 2, 0, 3], [5, 4, 3, 2, 1, 0]])
    signs = np.array([[1] * 6, [1, 1, -1, 1, 1, -1], [1, -1, 1, 1, 1, -1], [-1] * 6])
    orb = jv.util.symmetries.LatticeSymmetry(maps=maps, signs=signs, factor=np.array([1.0, 0.5, 0.25, 2.0]))
    net, onet = (jv.nets.CpxRBM(H, bias=True), onets.CpxRBM((L,), H, bias=True)) if cpx else \
        (jv.nets.RBM(H, bias=True), onets.RBM((L,), H, bias=True))
    rng = np.random.default_rng(21)
    P = 0.3 * rng.normal(size=_num(cpx, L, H, True, False))
    psi = jv.NQS(net, orbit=orb)
    psi(torch.zeros((1, 1, L), dtype=torch.int32))
    psi.set_parameters(P)
    opsi = onets.NQS(osym.SymNet(onet, orb.orbit, orb.factor, "exp"), P)
    s = rng.integers(0, 2, size=(n, L)).astype(np.int32)
    sd = torch.as_tensor(s[None], device="cuda")
    lp, lpo = psi(sd), opsi(s)
    assert np.max(np.abs(to_np(lp)[0] - lpo)) < TOL * np.max(np.abs(lpo))
    for op in ("tfim", "mixed"):
        Hd, Ho = OPS[op](L)
        assert _rel(to_np(Hd.get_O_loc(sd, psi, lp))[0], Ho.get_O_loc(s, opsi, lpo)) < TOL
    kw = dict(numChains=5, numSamples=20, thermalizationSweeps=3, sweepSteps=50)
    ms = jv.sampler.MCSampler(psi, (L,), 5, updateProposer=jv.sampler.propose_spin_flip, **kw)
    mo = osamp.MCSampler(opsi, (L,), 5, **kw)
    assert np.array_equal(to_np(ms.sample()[0])[0], mo.sample()[0])


def test_eloc_in_a_captured_graph():
    """A captured call keeps no pointer into the tables' scratch memory: calls
    with other sizes between the replays do not change its results."""
    L, H, n = 9, 14, 50
    rng = np.random.default_rng(8)
    Hd, Ho = xxz_pair(L, 0.6)
    P = 0.1 * rng.normal(size=_num(True, L, H, True, False))
    psi, opsi = _states(True, L, H, True, False, P)
    s = rng.integers(0, 2, size=(n, L)).astype(np.int32)
    sd = torch.as_tensor(s[None], device="cuda")
    lp = psi(sd)
    eager = Hd.get_O_loc(sd, psi, lp).clone()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        Hd.get_O_loc(sd, psi, lp)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = Hd.get_O_loc(sd, psi, lp)
    big, _ = _states(True, 40, 90, True, False, 0.05 * rng.normal(size=_num(True, 40, 90, True, False)))
    Hb, _ = tfim_pair((40,), -1.0, -0.7)
    sb = torch.as_tensor(rng.integers(0, 2, size=(1, 30, 40)).astype(np.int32), device="cuda")
    for _ in range(3):
        with torch.cuda.stream(stream):
            Hb.get_O_loc(sb, big, big(sb))
        torch.cuda.synchronize()
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert _rel(to_np(out), to_np(eager)) < TOL


@pytest.mark.parametrize("n", [50, 300])
def test_sym_calls_in_a_captured_graph(n):
    """Captured on a stream that no call has used before (a warm call on another
    one has sized the scratch memory); larger calls between the replays leave
    the captured ones' buffers alone.  n: with and without strings spread over
    several workgroups."""
    L, H = 8, 6
    rng = np.random.default_rng(9)
    Hd, Ho = xxz_pair(L, 0.6)
    P = 0.1 * rng.normal(size=_num(True, L, H, True, False))
    psi, opsi = _sym_states(True, L, H, ALL, P)
    s = rng.integers(0, 2, size=(n, L)).astype(np.int32)
    sd = torch.as_tensor(s[None], device="cuda")
    kw = dict(numChains=6, numSamples=24, thermalizationSweeps=2, sweepSteps=20)
    ms = jv.sampler.MCSampler(psi, (L,), 17, updateProposer=jv.sampler.propose_spin_flip, **kw)
    first = to_np(ms.sample()[0]).copy()
    lp = psi(sd).clone()
    eager = Hd.get_O_loc(sd, psi, lp).clone()
    ms.callIndex = 0
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        e = Hd.get_O_loc(sd, psi, lp)
        lp2 = psi(sd)
        c = ms.sample()[0]
    big, _ = _sym_states(True, 20, 40, ALL, 0.05 * rng.normal(size=_num(True, 20, 40, True, False)))
    Hb, _ = tfim_pair((20,), -1.0, -0.7)
    sb = torch.as_tensor(rng.integers(0, 2, size=(1, 30, 20)).astype(np.int32), device="cuda")
    for _ in range(3):
        Hb.get_O_loc(sb, big, big(sb))
        torch.cuda.synchronize()
        e.zero_()
        lp2.zero_()
        ms.states.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(e, eager)
        assert torch.equal(lp2, lp)
        assert np.array_equal(to_np(c), first)
    assert _rel(to_np(e)[0], Ho.get_O_loc(s, opsi, opsi(s))) < TOL
