"""Workloads for timing the variational Monte Carlo inner loop.

Each case is one call (or one whole step) that a program built on this package
makes over and over: evaluating log psi, drawing Metropolis samples, local
energies, log-derivatives, a TDVP right-hand side and a MinSR Euler step.  The
listed sizes are those of the package's own benchmark and tests; `draw` spreads
further cases over the same ranges (lattices of 6 to 48 sites for RBMs, 5x5 to
10x10 for CNNs, hidden units and channels that fill wavefronts and that do not,
a few to 16384 samples).

`exact` restates each case in plain torch (float64 / complex128), from the
Philox draws of the chains up to the regularised solves.
"""
import math

import numpy as np
import torch

import vmc_jax_amd as jv

# --------------------------------------------------------------------------- cases


def _case(**kw):
    c = {"path": "", "net": "cpxrbm", "Lx": 0, "Ly": 0, "hidden": 0, "bias": True, "channels": "", "samples": 0,
         "chains": 0, "therm": 10, "sweep": 10, "ham": "tfim", "layout": 0, "precision": "fp64"}
    c.update(kw)
    return c


def listed():
    return [
        # the smallest call: log psi of a handful of configurations, as a script probing a state makes it
        _case(name="logpsi_rbm_l10_16", path="logpsi", Lx=10, hidden=20, samples=16),
        # chains of the real-time RBM workload: 1024 walkers, 25 thermalisation sweeps of 32 proposals
        _case(name="sample_rbm_l32", path="sample", Lx=32, hidden=64, samples=16384, chains=1024, therm=25, sweep=32),
        # chains of the 10x10 ground-state workload with the sampler's default schedule
        _case(name="sample_cnn_10x10", path="sample", net="cnn", Lx=10, Ly=10, channels="8,8,8", samples=8192,
              chains=512),
        # chains of a network symmetrised over translations, reflection and spin flip (64 elements)
        _case(name="sample_sym_l16", path="sample", net="sym", Lx=16, hidden=32, samples=4096, chains=1024),
        # local energies of the same three families; the Ising chain flips single spins ...
        _case(name="eloc_rbm_l32", path="eloc", Lx=32, hidden=64, samples=16384),
        # ... the Heisenberg chain pairs of them, here at sizes that fill no wavefront
        _case(name="eloc_rbm_xxz_l45", path="eloc", Lx=45, hidden=90, samples=3000, ham="xxz"),
        # the CNN's in the mixed-precision form
        _case(name="eloc_cnn_10x10_mixed", path="eloc", net="cnn", Lx=10, Ly=10, channels="8,8,8", samples=8192,
              precision="mixed"),
        _case(name="eloc_sym_l16", path="eloc", net="sym", Lx=16, hidden=32, samples=4096),
        # log-derivatives in the layout the TDVP equation reads, and the compact ones of an odd-sized CNN
        _case(name="grad_rbm_l32", path="gradients", Lx=32, hidden=64, samples=16384, layout=1),
        _case(name="grad_cnn_9x7", path="gradients", net="cnn", Lx=9, Ly=7, channels="8,6,5", samples=5000),
        # a whole right-hand side of real-time TDVP: sampling, local energies, gradients, regularised solve
        _case(name="tdvp_rbm_l32", path="tdvp", Lx=32, hidden=64, samples=16384, chains=1024, therm=25, sweep=32),
        # a whole Euler step of the ground-state search with MinSR
        _case(name="minsr_step_cnn_10x10", path="minsr_step", net="cnn", Lx=10, Ly=10, channels="8,8,8",
              samples=8192, chains=512),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["logpsi", "sample", "sample", "sample", "eloc", "eloc", "eloc", "eloc", "gradients",
                       "gradients", "tdvp", "minsr_step"])
    c = _case(path=path)
    if path == "tdvp":
        c["net"] = "cpxrbm"
    elif path == "minsr_step":
        c["net"] = "cnn"
    else:
        c["net"] = rng.choice(["cpxrbm", "cpxrbm", "cnn", "cnn", "sym", "rbm"])
    if c["net"] == "cnn":
        c["Lx"], c["Ly"] = rng.randint(5, 10), rng.randint(5, 10)
        c["channels"] = rng.choice(["8,8,8", "8,8", "4,4", "6,5,4", "3,7", "8,4,8"])
        if path == "eloc":
            c["precision"] = rng.choice(["fp64", "mixed"])
    elif c["net"] == "sym":
        c["Lx"] = rng.randint(6, 16)
        c["hidden"] = rng.randint(6, 32)
    else:
        c["Lx"] = rng.randint(8, 32) if path == "tdvp" else rng.randint(6, 48)
        c["hidden"] = max(3, int(c["Lx"] * rng.uniform(0.5, 2.0)))
        c["bias"] = rng.random() < 0.7
        if path == "eloc":
            c["ham"] = rng.choice(["tfim", "xxz"])
    top = {"sym": 4096, "cnn": 8192}.get(c["net"], 16384)
    c["samples"] = _log_int(rng, 16, top)
    if path == "gradients":
        c["layout"] = 0 if c["net"] == "cnn" else rng.choice([0, 1])
        if c["net"] == "sym":
            c["samples"] = min(c["samples"], 1024)
    if path in ("tdvp", "minsr_step"):
        c["samples"] = _log_int(rng, 1024, top)
    if path in ("sample", "tdvp", "minsr_step"):
        c["chains"] = min(c["samples"], _log_int(rng, 32, {"cnn": 512}.get(c["net"], 1024)))
        spc = -(-c["samples"] // c["chains"])
        while spc > 16:  # no chain longer than the listed ones
            c["chains"] = min(1024 if c["net"] != "cnn" else 512, c["chains"] * 2)
            spc = -(-c["samples"] // c["chains"])
        if c["net"] in ("cpxrbm", "rbm"):
            c["sweep"] = rng.choice([10, c["Lx"]])
            c["sweep"] = min(c["sweep"], 32)
    if path == "minsr_step":  # more samples than parameters, as the dual solve of the benchmark has
        c["channels"] = rng.choice(["8,8,8", "8,8", "4,4", "6,5,4"])
        c["samples"] = max(c["samples"], 2048)
    return c


# --------------------------------------------------------------------------- inputs


def _dev():
    return torch.device("cuda") if torch.cuda.is_available() else torch.device("cpu")


def _sites(c):
    return c["Lx"] * max(1, c["Ly"])


def _channels(c):
    return [int(x) for x in c["channels"].split(",")]


def _emitted(c):
    return -(-c["samples"] // c["chains"]) * c["chains"]


def _data(c, seed):
    """Parameters (flat, float64) and configurations / walkers of a case, from the seed alone (numpy).
    Weights have the size they reach in a run: RBM pre-activations of order one half, He-normal kernels for CNNs
    with small biases."""
    rng = np.random.default_rng(seed)
    L, H = _sites(c), c["hidden"]
    if c["net"] == "cnn":
        leaves = []
        cin = 1
        for l, co in enumerate(_channels(c)):
            if l > 0:
                leaves.append(0.05 * rng.normal(size=co))
            leaves.append(rng.normal(size=9 * cin * co) * math.sqrt(2.0 / (9 * cin)))
            cin = co
        P = np.concatenate(leaves)
    else:
        m = 1 if c["net"] == "rbm" else 2
        s = 0.1 if c["path"] == "tdvp" else 0.5 / math.sqrt(L)
        P = s * rng.normal(size=m * (L * H + (H if c["bias"] else 0)))
    rows = c["chains"] if c["path"] in ("sample", "tdvp", "minsr_step") else c["samples"]
    return P, rng.integers(0, 2, size=(rows, L)).astype(np.int32)


def _shape(c):
    return (c["Lx"], c["Ly"]) if c["Ly"] else (c["Lx"],)


def _bonds(c):
    L = _sites(c)
    if not c["Ly"]:
        return [(l, (l + 1) % L) for l in range(L)]
    Lx, Ly = c["Lx"], c["Ly"]
    return [(i * Ly + j, nb) for i in range(Lx) for j in range(Ly)
            for nb in (((i + 1) % Lx) * Ly + j, i * Ly + (j + 1) % Ly)]


def _field(c):
    return -3.0 if c["Ly"] else -1.0


def _hamiltonian(c):
    op = jv.operator
    H = op.BranchFreeOperator()
    for a, b in _bonds(c):
        if c["ham"] == "xxz":
            H.add(op.scal_opstr(0.7, (op.Sz(a), op.Sz(b))))
            H.add(op.scal_opstr(1.0, (op.Sx(a), op.Sx(b))))
            H.add(op.scal_opstr(1.0, (op.Sy(a), op.Sy(b))))
        else:
            H.add(op.scal_opstr(-1.0, (op.Sz(a), op.Sz(b))))
    if c["ham"] != "xxz":
        for i in range(_sites(c)):
            H.add(op.scal_opstr(_field(c), (op.Sx(i),)))
    return H


def prepare(case, seed):
    c = case
    P, cfg = _data(c, seed)
    shape = _shape(c)
    orbit = None
    if c["net"] == "cnn":
        ch = _channels(c)
        net = jv.nets.CNN(F=(3, 3), channels=tuple(ch), strides=(1, 1))
    elif c["net"] == "rbm":
        net = jv.nets.RBM(numHidden=c["hidden"], bias=c["bias"])
    else:
        net = jv.nets.CpxRBM(numHidden=c["hidden"], bias=c["bias"])
        if c["net"] == "sym":
            orbit = jv.util.symmetries.get_orbit_1D(c["Lx"], "translation", "reflection", "spinflip")
    psi = jv.NQS(net, orbit=orbit, precision=c["precision"])
    psi(torch.zeros((1, 1) + shape, dtype=torch.int32))
    psi.set_parameters(P)
    s = torch.as_tensor(cfg, device="cuda")
    st = {"case": c, "psi": psi}
    if c["path"] in ("logpsi", "gradients", "eloc"):
        st["configs"] = s.reshape((1, s.shape[0]) + shape).contiguous()
    if c["path"] == "eloc":
        st["H"] = _hamiltonian(c)
        st["H"].compile()
        st["logpsi"] = psi(st["configs"])
    if c["path"] in ("sample", "tdvp", "minsr_step"):
        st["sampler"] = jv.sampler.MCSampler(psi, shape, 1000 + seed, updateProposer=jv.sampler.propose_spin_flip,
                                             numChains=c["chains"], numSamples=c["samples"],
                                             thermalizationSweeps=c["therm"], sweepSteps=c["sweep"])
        st["walkers"] = s
    if c["path"] == "tdvp":
        st["H"] = _hamiltonian(c)
        st["eq"] = jv.util.TDVP(st["sampler"], rhsPrefactor=1.j, makeReal="imag", pinvTol=1e-8, pinvCutoff=1e-4)
        st["theta"] = psi.get_parameters()
    if c["path"] == "minsr_step":
        st["H"] = _hamiltonian(c)
        st["eq"] = jv.util.MinSR(st["sampler"], pinvTol=1e-10, diagonalShift=1e-3)
        st["stepper"] = jv.util.stepper.Euler(timeStep=5e-3)
        st["theta"] = psi.get_parameters()
    return st


def _resume(st):
    """The chains continue from given walkers and proposal counter, as after a checkpoint."""
    st["sampler"].states = st["walkers"].clone()
    st["sampler"].callIndex = 0


def run(state):
    st = state
    c, psi = st["case"], st["psi"]
    if c["path"] == "logpsi":
        return psi(st["configs"])
    if c["path"] == "gradients":
        return psi.gradients(st["configs"], layout=c["layout"])
    if c["path"] == "eloc":
        return st["H"].get_O_loc(st["configs"], psi, st["logpsi"])
    _resume(st)
    if c["path"] == "sample":
        configs, logpsi, p = st["sampler"].sample()
        return {"configs": configs, "logpsi": logpsi, "weights": p, "walkers": st["sampler"].states}
    if c["path"] == "tdvp":
        eq = st["eq"]
        update = eq(st["theta"], 0.0, psi=psi, hamiltonian=st["H"], intStep=0)
        return {"update": update, "spectrum": eq.get_spectrum(), "energy": eq.get_energy_mean()}
    theta, _ = st["stepper"].step(0.0, st["eq"], st["theta"], hamiltonian=st["H"], psi=psi, numSamples=None)
    return {"theta": theta, "energy": st["eq"].get_energy_mean()}


# --------------------------------------------------------------------------- work


def _group_order(c):
    return 4 * c["Lx"] if c["net"] == "sym" else 1


def _forward_flops(c):
    """log psi of one configuration (a log-cosh counted as 20 operations)."""
    if c["net"] == "cnn":
        n, f, cin = _sites(c), 0, 1
        for co in _channels(c):
            f += n * co * (18 * cin + 20)
            cin = co
        return f
    m = 1 if c["net"] == "rbm" else 2
    return _group_order(c) * c["hidden"] * m * (2 * _sites(c) + 20)


def _flip_flops(c):
    """Change of log psi when one or two spins flip: a CNN recomputes the outputs that see the spin; an RBM
    multiplies one factor cosh(theta + d) / cosh(theta) per hidden unit (two complex multiply-adds)."""
    if c["net"] == "cnn":
        f, cin = 0, 1
        for l, co in enumerate(_channels(c)):
            w = min(3 + 2 * l, c["Lx"]) * min(3 + 2 * l, c["Ly"])
            f += w * co * (18 * cin + 20)
            cin = co
        return f
    return _group_order(c) * c["hidden"] * (4 if c["net"] == "rbm" else 16)


def _num_params(c):
    return _data(dict(c, samples=1, chains=1), 0)[0].size


def _flips(c):
    """Off-diagonal s' of one configuration."""
    return 2 * len(_bonds(c)) if c["ham"] == "xxz" else _sites(c)


def work(case):
    c = case
    L, P = _sites(c), _num_params(c)
    n = _emitted(c) if c["chains"] else c["samples"]
    cpx = 1 if c["net"] in ("rbm", "cnn") else 2
    base = 8 * P + 4 * n * L
    steps = c["therm"] * c["sweep"] + (n // c["chains"] if c["chains"] else 0) * c["sweep"]
    out = 8 * cpx
    mc = {"bytes": base + 4 * c["chains"] * L * 2 + n * (out + 8),
          "flops": c["chains"] * (steps * _flip_flops(c) + _forward_flops(c))}
    el = {"bytes": base + n * (out + 16), "flops": n * (_forward_flops(c) + _flips(c) * _flip_flops(c))}
    row = P * 16 if c["layout"] == 1 else (P // 2) * 16 if cpx == 2 else P * (4 if c["precision"] == "mixed" else 8)
    gr = {"bytes": base + n * row, "flops": n * (3 * _forward_flops(c) if c["net"] == "cnn"
                                                 else _forward_flops(c) + _group_order(c) * P)}
    if c["path"] == "logpsi":
        return {"bytes": base + n * out, "flops": n * _forward_flops(c)}
    if c["path"] in ("sample", "eloc", "gradients"):
        return {"sample": mc, "eloc": el, "gradients": gr}[c["path"]]
    if c["path"] == "tdvp":
        # Gram (Hermitian half), Pc x Pc complex eigenproblem with vectors, projection of the samples on them
        q = P // 2
        flops = 4.0 * n * q * q + 4 * (4.0 / 3 + 2) * q ** 3 + 8.0 * n * q * q
    else:
        # Gram (symmetric half) and a Cholesky solve
        flops = 1.0 * n * P * P + P ** 3 / 3.0
    return {"bytes": base + 16 * P, "flops": flops + mc["flops"] + el["flops"] + gr["flops"]}


# --------------------------------------------------------------------------- plain torch in 64 bits


def _log_cosh(z):
    if not z.is_complex():
        return z.abs() + torch.log1p(torch.exp(-2 * z.abs())) - math.log(2.0)
    y = torch.where(z.real < 0, -z, z)
    return y + torch.log(1 + torch.exp(-2 * y)) - math.log(2.0)


def _rbm_leaves(c, P):
    L, H = _sites(c), c["hidden"]
    m = 1 if c["net"] == "rbm" else 2
    nb = m * H if c["bias"] else 0

    def leaf(v):
        return v if m == 1 else torch.complex(v[:v.numel() // 2], v[v.numel() // 2:])
    W = leaf(P[nb:nb + m * L * H]).reshape(L, H)
    b = leaf(P[:nb]) if nb else torch.zeros(H, dtype=W.dtype, device=P.device)
    return W, b


def _cnn_layers(c, P):
    out, cin, o = [], 1, 0
    for l, co in enumerate(_channels(c)):
        b = None
        if l > 0:
            b, o = P[o:o + co], o + co
        out.append((P[o:o + 9 * cin * co].reshape(9, cin, co), b))
        o, cin = o + 9 * cin * co, co
    return out


def _cnn_forward(c, P, s):
    """Activations of every layer (B, Lx, Ly, C) and the pre-activations' tanh."""
    x = (2.0 * s.to(torch.float64) - 1.0).reshape(-1, c["Lx"], c["Ly"], 1)
    acts, tanhs = [x], []
    for K, b in _cnn_layers(c, P):
        z = 0
        for k in range(9):
            z = z + torch.matmul(torch.roll(x, (-(k // 3), -(k % 3)), (1, 2)), K[k])
        if b is not None:
            z = z + b
        x = _log_cosh(z)
        acts.append(x)
        tanhs.append(torch.tanh(z))
    return acts, tanhs


def _maps(c, device):
    """Site maps of the translations and reflections of the chain."""
    L = c["Lx"]
    i = torch.arange(L, device=device)
    return torch.stack([m for t in range(L) for m in ((i - t) % L, (L - 1 - i - t) % L)])


def _logpsi(c, P, s):
    """log psi of s (B, L)."""
    if c["net"] == "cnn":
        out = []
        for part in s.split(1 << 16):
            a = _cnn_forward(c, P, part)[0][-1]
            out.append(a.sum(dim=(1, 2, 3)) / math.sqrt(a[0].numel()))
        return torch.cat(out)
    W, b = _rbm_leaves(c, P)
    if c["net"] != "sym":
        x = (2 * s - 1).to(W.dtype)
        return torch.cat([_log_cosh(p @ W + b).sum(-1) for p in x.split(1 << 18)])
    m = _maps(c, s.device)
    out = []
    for part in s.split(1 << 14):
        x = (2 * part - 1).to(W.dtype)[:, m]  # (B, 2L, L)
        th = x @ W
        a = torch.cat([_log_cosh(th + b).sum(-1), _log_cosh(b - th).sum(-1)], dim=1)
        top = a.real.max(dim=1, keepdim=True).values
        out.append(torch.log(torch.exp(a - top).sum(dim=1)) + top[:, 0])
    return torch.cat(out)


def _eloc(c, P, s, lp):
    s = s.to(torch.int64)
    x = 2 * s - 1
    lp = lp.to(torch.complex128)
    E = torch.zeros(s.shape[0], dtype=torch.complex128, device=s.device)
    zz = sum((x[:, a] * x[:, b]).to(torch.float64) for a, b in _bonds(c))
    if c["ham"] == "xxz":
        E += 0.7 * zz
        for a, b in _bonds(c):
            t = s.clone()
            t[:, a] = 1 - t[:, a]
            t[:, b] = 1 - t[:, b]
            # (S+S- + h.c.): x x = 1 on every pair, y y = +1 on unlike pairs and -1 on like ones
            m = 1.0 - (x[:, a] * x[:, b]).to(torch.float64)
            E += torch.where(m != 0, m * torch.exp(_logpsi(c, P, t).to(torch.complex128) - lp), 0.0)
    else:
        E += -zz
        for i in range(s.shape[1]):
            t = s.clone()
            t[:, i] = 1 - t[:, i]
            E += _field(c) * torch.exp(_logpsi(c, P, t).to(torch.complex128) - lp)
    return E


def _gradients(c, P, s, layout):
    if c["net"] == "cnn":
        rows = []
        for part in s.split(2048):
            acts, tanhs = _cnn_forward(c, P, part)
            layers = _cnn_layers(c, P)
            B = part.shape[0]
            leaves = [None] * len(layers)
            d = tanhs[-1] / math.sqrt(acts[-1][0].numel())
            for l in range(len(layers) - 1, -1, -1):
                K, b = layers[l]
                x = acts[l]
                dd = d.reshape(B, -1, d.shape[-1])
                g = [torch.matmul(torch.roll(x, (-(k // 3), -(k % 3)), (1, 2)).reshape(B, -1, x.shape[-1])
                                  .transpose(1, 2).contiguous(), dd).reshape(B, -1) for k in range(9)]
                leaves[l] = torch.cat(([dd.sum(1)] if b is not None else []) + g, dim=1)
                if l > 0:
                    back = 0
                    for k in range(9):
                        back = back + torch.matmul(torch.roll(d, (k // 3, k % 3), (1, 2)), K[k].T.contiguous())
                    d = back * tanhs[l - 1]
            rows.append(torch.cat(leaves, dim=1))
        return torch.cat(rows)
    W, b = _rbm_leaves(c, P)
    x = (2 * s - 1).to(W.dtype)

    def leaves_of(x, sign):
        """(bias, kernel) derivatives at sign * x."""
        t = torch.tanh(sign * (x @ W) + b)
        return t, (sign * x)[:, :, None] * t[:, None, :]
    if c["net"] == "sym":
        m = _maps(c, s.device)
        lp = _logpsi(c, P, s)
        gb = gk = 0
        for j in range(m.shape[0]):
            for sign in (1, -1):
                xs = x[:, m[j]]
                w = torch.exp(_log_cosh(sign * (xs @ W) + b).sum(-1) - lp)
                t, k = leaves_of(xs, sign)
                gb, gk = gb + w[:, None] * t, gk + w[:, None, None] * k
    else:
        gb, gk = leaves_of(x, 1)
    parts = ([gb] if c["bias"] else []) + [gk.reshape(x.shape[0], -1)]
    if layout == 1 and c["net"] == "rbm":
        parts = [p.to(torch.complex128) for p in parts]
    if layout == 1 and c["net"] != "rbm":
        parts = [q for p in parts for q in (p, 1j * p)]
    return torch.cat(parts, dim=1)


def _draws(c, seed, steps):
    """Site and uniform number of each (step, chain): Philox4x32-10, key = seed, counter = (step, chain, call, stream)."""
    M = np.uint64(0xFFFFFFFF)
    n = c["chains"]
    ctr = [np.repeat(np.arange(steps, dtype=np.uint64), n), np.tile(np.arange(n, dtype=np.uint64), steps),
           np.zeros(steps * n, np.uint64), np.zeros(steps * n, np.uint64)]
    k0, k1 = seed & 0xFFFFFFFF, seed >> 32
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * ctr[0], np.uint64(0xCD9E8D57) * ctr[2]
        ctr = [(p1 >> np.uint64(32)) ^ ctr[1] ^ np.uint64(k0), p1 & M,
               (p0 >> np.uint64(32)) ^ ctr[3] ^ np.uint64(k1), p0 & M]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    site = (ctr[0] * np.uint64(_sites(c))) >> np.uint64(32)
    u = ((ctr[1] >> np.uint64(5)).astype(np.float64) * 67108864.0 + (ctr[2] >> np.uint64(6))) / 9007199254740992.0
    return site.astype(np.int64).reshape(steps, n), u.reshape(steps, n)


def _chains(c, P, walkers, seed):
    """Emitted configurations of the Metropolis chains."""
    spc = _emitted(c) // c["chains"]
    therm = c["therm"] * c["sweep"]
    steps = therm + spc * c["sweep"]
    site, u = (torch.as_tensor(v, device=P.device) for v in _draws(c, seed, steps))
    s = walkers.to(torch.int64)
    at = torch.arange(s.shape[0], device=P.device)
    re = _logpsi(c, P, s).real.to(torch.float64)
    out = []
    for t in range(steps):
        new = s.clone()
        new[at, site[t]] = 1 - new[at, site[t]]
        rn = _logpsi(c, P, new).real
        acc = u[t] < torch.exp(2.0 * (rn - re))
        s = torch.where(acc[:, None], new, s)
        re = torch.where(acc, rn, re)
        k = t + 1 - therm
        if k > 0 and k % c["sweep"] == 0:
            out.append(s)
    return torch.cat(out)


def _center(x):
    """sqrt(p) (x - <x>) with uniform weights."""
    return (x - x.mean(0)) / math.sqrt(x.shape[0])


def _tdvp_solve(E, O, pinv_tol, pinv_cutoff, snr_tol):
    """Real-time TDVP with the signal-to-noise regulariser: imaginary parts of the covariances."""
    n = O.shape[0]
    d, e = _center(O), _center(E)
    S = 1j * (d.conj().T @ d).imag
    F = 1j * ((-1j) * (d.conj().T @ e)).imag
    ev, V = torch.linalg.eigh(S)
    VtF = V.conj().T @ F
    q = ((-1j) * (d.conj() * e[:, None]) * n).imag  # imaginary parts of the samples of F
    qr = torch.complex(torch.matmul(q, V.imag), torch.matmul(q, V.real))  # i q conj(V)
    var = _center(qr).abs().square().sum(0)
    snr = torch.sqrt(n * VtF.abs().square() / var)
    r = (ev / ev[-1]).abs()
    inv = torch.where(r > 1e-14, 1.0 / ev, 0.0)
    residual, cutoff = 1.0, 1e-2
    while residual > pinv_tol and cutoff > pinv_cutoff:
        cutoff *= 0.8
        reg = 1.0 / (1.0 + (max(cutoff, pinv_cutoff) / r) ** 6) / (1.0 + (snr_tol / snr) ** 6)
        pe = inv * reg
        residual = float(torch.linalg.norm((pe * ev - 1.0) * VtF) / torch.linalg.norm(F))
    return (V @ (pe * VtF)).real, ev


def exact(case, seed):
    c = case
    if c["path"] == "sample" and c["precision"] == "mixed":
        return None  # the chains' decisions are taken in 32 bits
    P, cfg = _data(c, seed)
    P = torch.as_tensor(P, device=_dev())
    s = torch.as_tensor(cfg, device=_dev())
    if c["path"] == "logpsi":
        return _logpsi(c, P, s)[None]
    if c["path"] == "gradients":
        return _gradients(c, P, s, c["layout"])[None]
    if c["path"] == "eloc":
        return _eloc(c, P, s, _logpsi(c, P, s))[None]
    s = _chains(c, P, s, 1000 + seed)
    lp = _logpsi(c, P, s)
    n = s.shape[0]
    if c["path"] == "sample":
        return {"configs": None, "logpsi": lp[None],
                "weights": torch.full((1, n), 1.0 / n, dtype=torch.float64, device=P.device), "walkers": None}
    E = _eloc(c, P, s, lp)
    if c["path"] == "tdvp":
        update, ev = _tdvp_solve(E, _gradients(c, P, s, 1), 1e-8, 1e-4, 2.0)
        return {"update": update, "spectrum": ev, "energy": float(E.mean().real)}
    d, e = _center(_gradients(c, P, s, 0)), _center(E.real)
    S = d.T @ d + 1e-3 * torch.eye(d.shape[1], dtype=torch.float64, device=P.device)
    return {"theta": P - 5e-3 * torch.linalg.solve(S, d.T @ e), "energy": float(E.mean().real)}
