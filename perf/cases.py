"""The work this library does for its users, as cases that can be timed.

A case is one stretch of a simulation through the public binding
(``yukawacolourednoise_amd.Context``: the field goes in, Langevin steps run, a measurement
is taken where the run takes one, the field comes out), or one coloured-noise field
written to device memory (``abi.coloured_noise_noalloc``).  ``listed()`` names the stretches
users run, from the smallest lattice of an ``input.toml`` to the 1024 x 1024 workload;
``draw()`` gives more of the same ranges.

The start fields are Gaussian fields with a lattice propagator spectrum, cut at the coloured
noise's cutoff, around a mean: at the couplings below they give CG the iteration counts it
meets on thermalised fields.  ``exact()`` restates the model in 64-bit torch.
"""
import math

import numpy as np
import torch

import yukawacolourednoise_amd as Y
from yukawacolourednoise_amd import abi

# Couplings of the workloads: the action's m2, lambda, the Yukawa coupling g, the fermion
# mass M and Wilson parameter r, the step size eps; mean and spread of the start field.
COUPLINGS = {
    # 32 x 32 and 256 x 256 workloads, the driver's input files
    "plain": dict(m2=-0.2, lam=0.5, g=0.3, M=0.3, r=1.0, eps=0.01, mean=1.6, spread=0.45),
    # near the chiral point: the 512 x 512 and 1024 x 1024 workloads
    "chiral": dict(m2=-0.4, lam=1.0, g=0.5, M=0.05, r=1.0, eps=0.005, mean=0.45, spread=0.45),
    # the lattice-size sweep: naive fermions (r = 0), rescaled drift
    "sweep": dict(m2=-0.125, lam=0.3955, g=0.07, M=0.01, r=0.0, eps=0.005, mean=1.0, spread=0.55),
}

SOLVERS = {
    "fp64": (Y.YCN_CG_FP64, Y.YCN_PRECOND_NONE, 0),
    "mixed": (Y.YCN_CG_MIXED, Y.YCN_PRECOND_NONE, 0),
    "eo-fp64": (Y.YCN_CG_FP64, Y.YCN_PRECOND_NONE, 1),
    "eo-mixed": (Y.YCN_CG_MIXED, Y.YCN_PRECOND_NONE, 1),
    "learned": (Y.YCN_CG_MIXED, Y.YCN_PRECOND_CNN, 0),
}


def chain(name, Nt, Nx, solver, couplings, steps, *, chains=1, vectors=1, cut=0.5, adaptive=False, single=False,
          measure=False, relative=True, iters=100):
    """A stretch of `steps` Langevin steps of `chains` chains with `vectors` noise vectors per
    drift.  single: one call per step, as a program that reads every step size does;
    measure: a measurement at the end; relative: solves to a true relative residual of
    1e-10, else to the reference's absolute 1e-8; iters: about what a solve takes."""
    return dict(name=name, kind="chain", Nt=Nt, Nx=Nx, solver=solver, couplings=couplings, steps=steps,
                chains=chains, vectors=vectors, cut=cut, adaptive=adaptive, single=single, measure=measure,
                relative=relative, iters=iters)


def noise(name, Nt, Nx, *, chains=1, cut=0.5):
    return dict(name=name, kind="noise", Nt=Nt, Nx=Nx, chains=chains, cut=cut)


def listed():
    return [
        # the reference's default lattice and stopping rule, driven step by step
        chain("input-16x16", 16, 16, "fp64", "plain", 16, adaptive=True, single=True, measure=True, relative=False,
              iters=60),
        # one point of the lattice-size sweep: an odd time extent, which no tile divides
        chain("sweep-7x32", 7, 32, "fp64", "sweep", 16, adaptive=True, single=True, relative=False, iters=60),
        # the small workload between two exports
        chain("small-32x32", 32, 32, "fp64", "plain", 16, measure=True, iters=75),
        # a lattice of unequal extents, even-odd solver in double precision
        chain("eo-fp64-48x160", 48, 160, "eo-fp64", "plain", 8, adaptive=True, measure=True, iters=50),
        # the middle workload with the fastest solver
        chain("eo-mixed-256x256", 256, 256, "eo-mixed", "plain", 16, iters=50),
        # the near-critical workload in mixed precision
        chain("mixed-512x512", 512, 512, "mixed", "chiral", 8, iters=300),
        # flexible CG with a network trained on the chain's own solves
        chain("learned-256x256", 256, 256, "learned", "chiral", 8, iters=150),
        # the 64-chain scan in m2, 8 noise vectors per drift: 512 systems at once
        chain("scan-64x64x64", 64, 64, "eo-mixed", "plain", 8, chains=64, vectors=8, iters=50),
        # the large workload with the reference's solver
        chain("fp64-1024x1024", 1024, 1024, "fp64", "chiral", 2, iters=300),
        # the large workload with the fastest solver
        chain("eo-mixed-1024x1024", 1024, 1024, "eo-mixed", "chiral", 16, iters=115),
        # coloured noise into a device buffer: the large lattice, and a batch of ragged ones
        noise("noise-1024x1024", 1024, 1024),
        noise("noise-12x45x50", 45, 50, chains=12, cut=0.25),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _unnamed(case):
    return {k: v for k, v in case.items() if k != "name"}


def draw(rng):
    cut = rng.choice([1.0, 0.5, 0.25, 0.7])
    kind = rng.choice(["noise", "small", "plain", "even-odd", "even-odd", "scan", "learned"])
    if kind == "noise":
        chains = rng.choice([1, 1, 2, 5])
        # extents with small prime factors, odd ones among them
        Nt, Nx = (rng.choice([1, 2, 3, 5, 7, 9, 15]) * 2 ** rng.randint(2, 6) for _ in range(2))
        return _unnamed(noise("", Nt, min(Nx, 1024), chains=chains if chains * Nt * Nx < 2 ** 19 else 1, cut=cut))
    adaptive = rng.random() < 0.4
    if kind == "small":
        if rng.random() < 0.5:
            c = chain("", rng.randint(2, 22), 32, "fp64", "sweep", 8, adaptive=True, single=True, relative=False, iters=60)
        else:
            c = chain("", _spread(rng, 6, 48), _spread(rng, 8, 48), rng.choice(["fp64", "mixed"]), "plain", 8,
                      adaptive=adaptive, cut=cut, chains=rng.choice([1, 1, 2, 7]), vectors=rng.choice([1, 1, 3]), iters=70)
    elif kind == "plain":
        c = chain("", 2 * _spread(rng, 24, 256), 16 * _spread(rng, 3, 32), rng.choice(["fp64", "mixed"]),
                  rng.choice(["plain", "chiral"]), 4, adaptive=adaptive, cut=cut, iters=200)
    elif kind == "even-odd":
        Nt, Nx = 2 * _spread(rng, 4, 400), 32 * _spread(rng, 1, 25)
        if rng.random() < 0.5:
            Nt, Nx = 16 * _spread(rng, 1, 50), 16 * _spread(rng, 1, 50)
        c = chain("", Nt, Nx, rng.choice(["eo-fp64", "eo-mixed", "eo-mixed"]), rng.choice(["plain", "chiral"]), 8,
                  adaptive=adaptive, cut=cut, iters=100)
    elif kind == "scan":
        L = rng.choice([16, 32, 48, 64])
        c = chain("", L, L, rng.choice(["fp64", "mixed", "eo-fp64", "eo-mixed", "eo-mixed"]), "plain", 4,
                  chains=rng.choice([4, 10, 16, 33, 64]), vectors=rng.choice([1, 2, 4, 8]), cut=cut, iters=60)
    else:
        c = chain("", 16 * _spread(rng, 2, 16), 16 * _spread(rng, 2, 16), "learned", "chiral", 4, cut=cut, iters=120)
    return _unnamed(c)


# ---- inputs -----------------------------------------------------------------------------
def _m2(case):
    """Per-chain m2: the scan -1 ... 0.5 where there are several chains."""
    n, m2 = case["chains"], COUPLINGS[case["couplings"]]["m2"]
    return [m2] if n == 1 else [-1.0 + 1.5 * k / (n - 1) for k in range(n)]


def _seeds(case, seed):
    return [(1234 + 7919 * seed + k) % (1 << 31) for k in range(case["chains"])]


def _start_field(case, seed):
    """(chains, Nt, Nx): a Gaussian field with spectrum 1 / (p^2 + 0.3) below the cutoff."""
    w = COUPLINGS[case["couplings"]]
    R, Nt, Nx = case["chains"], case["Nt"], case["Nx"]
    z = np.fft.rfft2(np.random.default_rng(seed).standard_normal((R, Nt, Nx)))
    kt = 2 * np.pi * np.fft.fftfreq(Nt)[:, None]
    kx = 2 * np.pi * np.fft.rfftfreq(Nx)[None]
    z = z * (kt ** 2 + kx ** 2 <= 2 * (np.pi * case["cut"]) ** 2) / np.sqrt(4 * np.sin(kt / 2) ** 2 + 4 * np.sin(kx / 2) ** 2 + 0.3)
    f = np.fft.irfft2(z, s=(Nt, Nx))
    f = f - f.mean(axis=(1, 2), keepdims=True)
    return w["mean"] + w["spread"] * f / f.std()


def _params(case, seed):
    if case["kind"] == "noise":
        return Y.default_params(Nt=case["Nt"], Nx=case["Nx"], nReplicas=case["chains"], cutFraction=case["cut"])
    w = COUPLINGS[case["couplings"]]
    precision, precond, evenOdd = SOLVERS[case["solver"]]
    p = Y.default_params(Nt=case["Nt"], Nx=case["Nx"], nReplicas=case["chains"], nNoise=case["vectors"], m2=w["m2"],
                         lam=w["lam"], g=w["g"], M=w["M"], r=w["r"], cutFraction=case["cut"], epsBar=w["eps"],
                         driftMode=1 if case["couplings"] == "sweep" else 0, adaptive=int(case["adaptive"]),
                         seed=_seeds(case, seed)[0], cgPrecision=precision, precond=precond, evenOdd=evenOdd)
    if case["relative"]:
        p.cgTol, p.cgTolMode, p.cgMaxIter = 1e-10, Y.YCN_TOL_REL_TRUE, 20000
    return p


TRAINING_STEPS, PAIRS_PER_SOLVE = 16, 16


def prepare(case, seed):
    seeds = _seeds(case, seed)
    p = _params(case, seed)
    state = {"case": dict(case), "params": p, "step": 100 + seed % 1000}
    if case["kind"] == "noise":
        state["seeds"] = np.array(seeds, dtype=np.uint64)
        state["out"] = torch.empty((case["chains"], case["Nt"], case["Nx"]), dtype=torch.float64, device="cuda")
        return state
    ctx = Y.Context(p)
    ctx.set_replicas(_m2(case), np.array(seeds, dtype=np.uint64))
    phi = _start_field(case, seed)
    if case["solver"] == "learned":
        ctx.set_field(phi)
        ctx.precond_train(0, TRAINING_STEPS, pairs_per_solve=PAIRS_PER_SOLVE)
    state["ctx"], state["phi"] = ctx, phi
    return state


def run(state):
    case, step = state["case"], state["step"]
    if case["kind"] == "noise":
        rc = abi.coloured_noise_noalloc(state["params"], step, state["out"].data_ptr(),
                                        torch.cuda.current_stream().cuda_stream, state["seeds"])
        if rc != abi.YCN_OK:
            raise Y.YcnError(rc, abi.lib.ycn_last_error(None).decode())
        return state["out"]
    ctx, n = state["ctx"], case["steps"]
    ctx.set_field(state["phi"])
    out = {}
    if case["single"]:
        out["eps"] = np.stack([ctx.langevin_step(step + k).eps for k in range(n)])
    else:
        ctx.langevin_run(step, n)
    if case["measure"]:
        obs, out["slices"], out["corr"] = ctx.measure(0, step + n)
        out["obs"] = [obs[k] for k in ("magnetisation", "phi2", "trace", "eps")]
    out["phi"] = ctx.get_field()
    return out


# Operations per site: two Dirac applications on the real and imaginary-free spinor (56) and
# CG's three updates and two products, on every site or (even-odd) on half of them.
_FLOPS = {"fp64": 96, "mixed": 96, "learned": 96 + 2 * 4608, "eo-fp64": 76, "eo-mixed": 76}


def work(case):
    V = case["Nt"] * case["Nx"] * case["chains"]
    fft = 10.0 * V * math.log2(case["Nt"] * case["Nx"])
    if case["kind"] == "noise":
        return {"bytes": 8 * V, "flops": fft + 60 * V}
    solve = _FLOPS[case["solver"]] * case["iters"] * V * case["vectors"]
    return {"bytes": 16 * V * case["steps"], "flops": case["steps"] * (fft + solve)}


# ---- the model in 64 bits ----------------------------------------------------------------
_LOW = 0xFFFFFFFF


def _philox(counter, key):
    """Philox4x32-10 on int64 tensors holding 32-bit words."""
    c0, c1, c2, c3 = counter
    k0, k1 = key
    for i in range(10):
        if i:
            k0, k1 = (k0 + 0x9E3779B9) & _LOW, (k1 + 0xBB67AE85) & _LOW
        a, b = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = ((b >> 32) & _LOW) ^ c1 ^ k0, b & _LOW, ((a >> 32) & _LOW) ^ c3 ^ k1, a & _LOW
    return c0, c1, c2, c3


def _normals(seed, stream, step, n):
    q = torch.arange((n + 1) // 2, dtype=torch.int64, device="cuda")
    zero = torch.zeros_like(q)
    o = _philox((q, zero, zero + (step & _LOW), zero + (step >> 32)), (seed & _LOW, stream))
    u1 = ((((o[0] << 21) | (o[1] >> 11)) + 1).double()) * 2.0 ** -53
    u2 = ((o[2] << 21) | (o[3] >> 11)).double() * 2.0 ** -53
    rho = torch.sqrt(-2.0 * torch.log(u1))
    return torch.stack([rho * torch.cos(2 * math.pi * u2), rho * torch.sin(2 * math.pi * u2)], 1).reshape(-1)[:n]


def _coloured(case, seeds, step):
    Nt, Nx = case["Nt"], case["Nx"]
    xi = torch.stack([_normals(s, 0, step, Nt * Nx) for s in seeds]).reshape(-1, Nt, Nx)

    def momentum(n, count):
        k = np.arange(count, dtype=np.float64)
        k = np.where(np.arange(count) <= n // 2, k, k - n)
        return (k * 2.0 * math.pi / n) ** 2

    keep = momentum(Nt, Nt)[:, None] + momentum(Nx, Nx // 2 + 1)[None] <= (math.sqrt(2.0) * math.pi * case["cut"]) ** 2
    return torch.fft.irfft2(torch.fft.rfft2(xi) * torch.from_numpy(keep).cuda(), s=(Nt, Nx))


class _Model:
    """D on spinors (chains, vectors, flavour, spin, Nt, Nx), all real."""

    def __init__(self, case):
        self.w, self.case = COUPLINGS[case["couplings"]], case
        self.m2 = torch.tensor(_m2(case), dtype=torch.float64, device="cuda")[:, None, None]

    def dirac(self, phi, v, dagger):
        w, s = self.w, (-1 if dagger else 1)

        def hop(u, n, dim):   # the neighbour n sites ahead, antiperiodic in time
            u = torch.roll(u, -n, dim)
            if dim == -2:
                u.select(-2, -1 if n > 0 else 0).neg_()
            return u

        d = (2 * w["r"] + w["M"] + w["g"] * phi)[:, None, None]
        a, b = v[:, :, :, 0], v[:, :, :, 1]
        hp, hm, hr = 0.5 * (w["r"] + 1), 0.5 * (w["r"] - 1), 0.5 * w["r"]
        af, ab, bf, bb = (hop(u, n, -1) for u, n in ((a, s), (a, -s), (b, s), (b, -s)))
        oa = d * a - (hp * hop(a, -s, -2) + hr * (af + ab) + 0.5 * (bb - bf))
        ob = d * b - (hp * hop(b, s, -2) + hr * (bf + bb) + 0.5 * (ab - af))
        if hm:
            oa -= hm * hop(a, s, -2)
            ob -= hm * hop(b, -s, -2)
        return torch.stack([oa, ob], 3)

    def normal_solve(self, phi, b):
        """y with D^dag D y = b, to a relative residual of 1e-13."""
        dot = lambda u, v: (u * v).sum(dim=(2, 3, 4, 5), keepdim=True)  # noqa: E731
        x, r, p = torch.zeros_like(b), b.clone(), b.clone()
        rr = dot(r, r)
        stop = 1e-26 * rr
        for i in range(20000):
            Ap = self.dirac(phi, self.dirac(phi, p, False), True)
            alpha = torch.where(rr > stop, rr / dot(p, Ap), torch.zeros_like(rr))
            x += alpha * p
            r -= alpha * Ap
            new = torch.where(rr > stop, dot(r, r), rr)
            if i % 8 == 7 and not bool((new > stop).any()):
                break
            p = r + (new / rr) * p
            rr = new
        return x

    def force(self, phi, seeds, stream, step):
        c = self.case
        V, J = c["Nt"] * c["Nx"], c["vectors"]
        eta = torch.stack([torch.stack([_normals(s, stream + j, step, 4 * V) for j in range(J)]) for s in seeds])
        eta = eta.reshape(-1, J, c["Nt"], c["Nx"], 2, 2).permute(0, 1, 4, 5, 2, 3).contiguous()
        chi = self.dirac(phi, self.normal_solve(phi, eta), False)
        scale = c["cut"] ** 2 if c["couplings"] == "sweep" else 1.0
        return -self.w["g"] * scale * (chi * eta).sum(dim=(1, 2, 3)) / J

    def step(self, phi, seeds, step):
        w = self.w
        force = self.force(phi, seeds, 1, step)
        laplacian = sum(torch.roll(phi, n, d) for n in (1, -1) for d in (1, 2)) - 4 * phi
        drift = force + phi * (self.m2 + w["lam"] / 6 * phi * phi) - laplacian
        eps = torch.full_like(self.m2, w["eps"])
        if self.case["adaptive"]:
            eps = w["eps"] * 30 / drift.abs().amax(dim=(1, 2), keepdim=True).clamp(1e-5, 1e5)
        return phi - eps * drift - torch.sqrt(2 * eps) * _coloured(self.case, seeds, step), eps

    def correlator(self, phi):
        """Time slices of D^-1 src, src = (1, 1, 0, 0) at the origin."""
        src = torch.zeros((1, 1, 2, 2, *phi.shape[1:]), dtype=torch.float64, device="cuda")
        src[0, 0, 0, :, 0, 0] = 1.0
        # D^-1 = (D^dag D)^-1 D^dag
        return self.normal_solve(phi, self.dirac(phi, src, True)).sum(dim=(0, 1, 2, 3, 5))


def exact(case, seed):
    seeds, step = _seeds(case, seed), 100 + seed % 1000
    if case["kind"] == "noise":
        return _coloured(case, seeds, step)
    model, n = _Model(case), case["steps"]
    phi = torch.from_numpy(_start_field(case, seed)).cuda()
    eps = []
    for k in range(n):
        phi, e = model.step(phi, seeds, step + k)
        eps.append(e.reshape(-1))
    out = {}
    if case["single"]:
        out["eps"] = torch.stack(eps)
    if case["measure"]:
        one = phi[:1]
        trace = model.force(phi, seeds, 0x4D00, step + n)[0].sum() / model.w["g"]
        out["slices"], out["corr"] = one[0].sum(dim=1), model.correlator(one)
        out["obs"] = [float(v) for v in (one.sum(), (one * one).sum(), trace, eps[-1][0])]
    out["phi"] = phi if case["chains"] > 1 else phi[0]
    return out
