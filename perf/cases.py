"""Performance cases: the work that users of this framework have it do, at the sizes they do it.

Every case goes through the public entry points of ``rbmd_amd`` (``ForceContext``,
``BatchContext``, ``DifferentiableForce``) as a user's program does:

* ``md``      molecular dynamics through ``md_run``: the state stays on the GPU and is advanced
              in place (NVE of a plain LJ fluid, NVT Nose-Hoover of the LJ electrolyte);
* ``steps``   a host program with an integrator of its own (the Force module boundary): it writes
              the positions of each step into its arrays, asks for the force and applies it.  The
              positions of the steps are a short ballistic trajectory, long enough for the skin to
              run out, so lists are rebuilt at about their natural rate;
* ``rerun``   energies, virial and forces of stored, uncorrelated configurations with a given
              k-sample: every configuration rebuilds the lists;
* ``batch``   many small boxes in one evaluation;
* ``match``   force-matching training steps through autograd: two minibatches, each a stored
              configuration with the parameters of that step;
* ``adjoint`` force and its vector-Jacobian product on one large box.

Positions are an fcc lattice at liquid density with thermal-size displacements (a randomly
oriented rigid molecule per lattice site for water), made on the GPU from the seed.  LJ units but
for water (Angstrom, kcal/mol).
"""
import math

import numpy as np
import torch

DEV = "cuda:0"
RHO = 0.8          # reduced density of the LJ systems
SKIN = 0.3
QQR2E_REAL = 332.06371


# ---------------------------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------------------------
def listed():
    return [
        # The plain LJ fluid of the C1 configuration: FP64, full Verlet list, energies and virial
        # every step.  The smallest work: launches and latency.
        dict(name="lj-4k-nve-fp64", kind="md", system="lj", n=4000, precision="fp64",
             nsteps=20, energy=True),
        # A small electrolyte driven by a host program's integrator, RBL + RBE, P = 200.
        dict(name="salt-4k-steps", kind="steps", system="salt", n=4001, ions=0.1,
             neighbor="RBL", coulomb="RBE", P=200, frames=16, energy=False),
        # A medium electrolyte's NVT production run.
        dict(name="salt-27k-nvt", kind="md", system="salt", n=27013, precision="fp32", P=200,
             nsteps=10, energy=False),
        # The headline system: 200,000 particles, RBL + RBE with P = 200, NVT.
        dict(name="salt-200k-nvt", kind="md", system="salt", n=200000, precision="fp32", P=200,
             nsteps=10, energy=False),
        # Stored configurations of the headline system evaluated with energies and virial.
        dict(name="salt-200k-rerun", kind="rerun", n=200000, ions=0.1, P=200, frames=2),
        # A molten salt (every atom charged) with full lists, exact Ewald and energies.
        dict(name="molten-14k-ewald", kind="steps", system="salt", n=13824, ions=1.0,
             neighbor="Verlet-List", coulomb="EWALD", kmax=6, frames=4, energy=True),
        # SPC/E water, CVFF special bonds, RBL + RBE, energies every step: a small solvent box.
        dict(name="water-9k-rbe-energy", kind="steps", system="water", n=3000, neighbor="RBL",
             coulomb="RBE", P=300, frames=16, energy=True),
        # SPC/E water, CVFF special bonds, RBL + RBSOG at P = 512: the C3 configuration.
        dict(name="water-73k-rbsog", kind="steps", system="water", n=24327, neighbor="RBL",
             coulomb="RBSOG", P=512, frames=16, energy=False),
        # A few small replicas with their energies (replica exchange).
        dict(name="batch-24-energy", kind="batch", nrep=24, nmin=500, nmax=2000, P=100,
             energy=True),
        # 256 independent boxes of 500 to 8000 atoms: the C4 configuration.
        dict(name="batch-256", kind="batch", nrep=256, nmin=500, nmax=8000, P=100, energy=False),
        # Force-matching training steps on a medium box.
        dict(name="match-32k", kind="match", n=32000, P=200),
        # Force and adjoint of the 2,000,000-particle box, P = 400: the C5 configuration.
        dict(name="adjoint-2m", kind="adjoint", n=2000000, P=400),
    ]


def _logu(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["lj", "nvt", "salt", "rerun", "ewald", "water", "water", "batch", "match",
                       "adjoint"])
    if kind == "lj":
        return dict(kind="md", system="lj", n=_logu(rng, 1200, 60000),
                    precision=rng.choice(["fp64", "fp32"]), nsteps=rng.randint(5, 20),
                    energy=rng.random() < 0.5)
    if kind == "nvt":
        return dict(kind="md", system="salt", n=_logu(rng, 4000, 200000), precision="fp32",
                    P=rng.randint(60, 400), nsteps=rng.randint(5, 10),
                    energy=rng.random() < 0.25)
    if kind == "salt":
        return dict(kind="steps", system="salt", n=_logu(rng, 1500, 200000),
                    ions=round(rng.uniform(0.03, 0.4), 3), neighbor="RBL", coulomb="RBE",
                    P=rng.randint(60, 400), frames=rng.randint(6, 16),
                    energy=rng.random() < 0.25)
    if kind == "rerun":
        return dict(kind="rerun", n=_logu(rng, 3000, 200000), ions=round(rng.uniform(0.03, 0.4), 3),
                    P=rng.randint(60, 400), frames=rng.randint(1, 2))
    if kind == "ewald":
        return dict(kind="steps", system="salt", n=_logu(rng, 1500, 20000),
                    ions=rng.choice([1.0, round(rng.uniform(0.1, 0.9), 3)]),
                    neighbor="Verlet-List", coulomb="EWALD", kmax=rng.randint(3, 6),
                    frames=rng.randint(2, 6), energy=rng.random() < 0.5)
    if kind == "water":
        return dict(kind="steps", system="water", n=_logu(rng, 700, 24000),
                    neighbor=rng.choice(["RBL", "RBL", "Verlet-List"]),
                    coulomb=rng.choice(["RBE", "RBSOG"]), P=rng.randint(100, 512),
                    frames=rng.randint(6, 16), energy=rng.random() < 0.5)
    if kind == "batch":
        nmin = _logu(rng, 500, 2000)
        return dict(kind="batch", nrep=_logu(rng, 8, 200), nmin=nmin,
                    nmax=_logu(rng, nmin + 100, 8000), P=rng.randint(50, 200),
                    energy=rng.random() < 0.5)
    if kind == "match":
        return dict(kind="match", n=_logu(rng, 3000, 100000), P=rng.randint(100, 400))
    return dict(kind="adjoint", n=_logu(rng, 20000, 800000), P=rng.randint(100, 400))


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
class Sys:
    """One periodic box as a user's program holds it: per-atom arrays on the host, positions and
    velocities on the GPU (N, 3) in FP64."""


def _rng(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _fcc(n, gen, jitter=0.1):
    """n atoms on the sites of a near-cubic fcc block (a few sites left empty) at density RHO,
    each displaced uniformly within +-jitter per direction.  Box edges are FP32 numbers."""
    best = None
    c0 = max(5, int((n / 4.0) ** (1.0 / 3.0)))
    for a in range(max(5, c0 - 2), c0 + 3):
        for b in range(a, c0 + 4):
            c = max(a, -(-n // (4 * a * b)))
            cost = (4 * a * b * c - n) / n + 0.1 * (max(b, c) / a - 1)
            if best is None or cost < best[0]:
                best = (cost, (a, b, c))
    cells = best[1]
    a = (n / RHO / (cells[0] * cells[1] * cells[2])) ** (1.0 / 3.0)
    L = np.array([float(np.float32(a * c)) for c in cells])
    g = torch.stack(torch.meshgrid(*[torch.arange(c, device=DEV) for c in cells], indexing="ij"),
                    -1).reshape(-1, 1, 3).double()
    basis = torch.tensor([[0, 0, 0], [.5, .5, 0], [.5, 0, .5], [0, .5, .5]], device=DEV,
                         dtype=torch.float64) + 0.25
    pos = ((g + basis) * a).reshape(-1, 3)
    keep = torch.randperm(len(pos), generator=gen, device=DEV)[:n].sort().values
    pos = pos[keep] + jitter * (2 * torch.rand((n, 3), generator=gen, device=DEV,
                                               dtype=torch.float64) - 1)
    # the atoms' order in a file is not their order in space
    return pos[torch.randperm(n, generator=gen, device=DEV)], L


def _wrap32(x, L, dtype=torch.float32):
    """Positions folded into the box, as (3, N) contiguous arrays of the program's type."""
    Lt = torch.tensor(L, device=DEV, dtype=torch.float64)
    x = x - Lt * torch.floor(x / Lt)
    y = x.T.contiguous().to(dtype)
    hi = Lt.to(dtype)[:, None]
    return torch.where(y >= hi, y - hi, y)


def _lj_system(n, seed, ions=0.0):
    """n LJ particles; a share `ions` carries charges +1 and -1 in equal numbers.  Types: cation,
    anion, solvent (one type without ions)."""
    gen = _rng(seed)
    s = Sys()
    s.pos, s.L = _fcc(n, gen)
    s.n = n
    vel = torch.randn((n, 3), generator=gen, device=DEV, dtype=torch.float64)
    s.vel = vel - vel.mean(0)
    if ions > 0:
        half = int(n * ions / 2)
        t = torch.full((n,), 2, dtype=torch.int32, device=DEV)
        p = torch.randperm(n, generator=gen, device=DEV)
        t[p[:half]] = 0
        t[p[half:2 * half]] = 1
        if ions >= 1.0 and 2 * half < n:
            t[p[2 * half:]] = 0
        s.types = t.cpu().numpy()
        s.Q = np.array([1.0, -1.0, 0.0])
        s.eps, s.sigma = np.ones(3), np.ones(3)
    else:
        s.types = np.zeros(n, dtype=np.int32)
        s.Q = np.zeros(1)
        s.eps, s.sigma = np.ones(1), np.ones(1)
    s.charges = s.Q[s.types]
    s.ids = np.arange(n, dtype=np.int32)
    s.box_lo, s.box_len = np.zeros(3), s.L
    return s


def _water(nmol, seed):
    """nmol rigid SPC/E molecules at 33.4 / nm^3 on lattice sites, random orientations, atoms
    O, H1, H2 per molecule."""
    gen = _rng(seed)
    L = float(np.float32((nmol / 0.0334) ** (1.0 / 3.0)))
    m = int(math.ceil(nmol ** (1.0 / 3.0) - 1e-9))
    g = torch.stack(torch.meshgrid(*[torch.arange(m, device=DEV)] * 3, indexing="ij"),
                    -1).reshape(-1, 3)[:nmol]
    o = (g.double() + 0.5) * (L / m)
    o = o + 0.15 * (2 * torch.rand((nmol, 3), generator=gen, device=DEV, dtype=torch.float64) - 1)
    q = torch.randn((nmol, 4), generator=gen, device=DEV, dtype=torch.float64)
    w, x, y, z = (q / q.norm(dim=1, keepdim=True)).T
    rot = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                       2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                       2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)],
                      -1).reshape(nmol, 3, 3)
    h = math.radians(109.47) / 2
    ref = torch.tensor([[0, 0, 0], [math.sin(h), 0, math.cos(h)], [-math.sin(h), 0, math.cos(h)]],
                       device=DEV, dtype=torch.float64)
    s = Sys()
    s.pos = (o[:, None, :] + (rot[:, None] * ref[None, :, None, :]).sum(-1)).reshape(-1, 3)
    s.vel = torch.randn((nmol, 3), generator=gen, device=DEV, dtype=torch.float64)
    s.vel = 8.0 * s.vel.repeat_interleave(3, 0)  # the molecule's, by atom
    s.n = 3 * nmol
    s.L = np.array([L, L, L])
    s.box_lo, s.box_len = np.zeros(3), s.L
    s.types = np.tile(np.array([0, 1, 1], dtype=np.int32), nmol)
    s.ids = np.arange(s.n, dtype=np.int32)
    s.charges = np.tile(np.array([-0.8476, 0.4238, 0.4238]), nmol)
    s.eps, s.sigma = np.array([0.15535, 0.0]), np.array([3.166, 0.0])
    base = 3 * np.arange(nmol, dtype=np.int32)
    s.nspecial = np.tile(np.array([[2, 2, 2], [1, 2, 2], [1, 2, 2]], dtype=np.int32), (nmol, 1))
    s.special = np.empty((s.n, 2), dtype=np.int32)
    s.special[0::3] = np.stack([base + 1, base + 2], 1)
    s.special[1::3] = np.stack([base, base + 2], 1)
    s.special[2::3] = np.stack([base, base + 1], 1)
    return s


def _config(case, seed):
    """The RBMD JSON document of the case."""
    sysk = case.get("system", "salt")
    if sysk == "lj":
        return {"init_configuration": {"read_data": {"unit": "LJ", "atom_style": "atomic"}},
                "hyper_parameters": {
                    "force_field": {"type": "LJ/CUT"},
                    "neighbor": {"type": "Verlet-List", "cut_off": 2.5, "skin": SKIN},
                    "precision": case["precision"]},
                "execution": {"ensemble": "NVE", "integration_type": "vv", "timestep": 0.004}}
    neighbor, coulomb = case.get("neighbor", "RBL"), case.get("coulomb", "RBE")
    water = sysk == "water"
    nb = {"type": neighbor, "cut_off": 10.0 if water else 3.5, "skin": 2.0 if water else SKIN}
    if not water:
        nb["lj_cut_off"] = 2.5
    if neighbor == "RBL":
        nb.update({"r_core": 6.5 if water else 2.5, "neighbor_sample_num": 100 if water else 30,
                   "energy_rbl_flag": "no"})
    cl = {"type": coulomb, "alpha": 0.0784 if water else 0.09, "random_seed": seed % 4294967291}
    if coulomb == "RBE":
        cl.update({"coulomb_sample_num": case["P"], "energy_rbe_flag": "no"})
    elif coulomb == "RBSOG":
        cl.update({"coulomb_sample_num": case["P"], "rbsog_level": 1})
    else:
        cl["kmax"] = [case["kmax"]] * 3
    hp = {"force_field": {"type": "CVFF" if water else "LJ/CUT/COUL/LONG"}, "neighbor": nb,
          "coulomb": cl, "precision": case.get("precision", "fp32")}
    if water:
        hp["force_field"]["mixing_rule"] = "arithmetic"
        hp["extend"] = {"special_bonds": [0.0, 0.0, 0.0]}
    return {"init_configuration": {"read_data": {"unit": "REAL" if water else "LJ",
                                                 "atom_style": "full" if water else "charge"}},
            "hyper_parameters": hp,
            "execution": {"ensemble": "NVT", "integration_type": "vv",
                          "temp_ctrl_type": "NOSE_HOOVER", "temperature": [1.0, 1.0, 0.2],
                          "timestep": 0.002}}


def _context(case, s, seed):
    from rbmd_amd import ForceContext

    ctx = ForceContext(_config(case, seed), device=0)
    ctx.set_system(s.box_lo, s.box_len, s.types, s.ids, s.charges, s.eps, s.sigma)
    if case.get("system") == "water":
        ctx.set_special(s.nspecial, s.special)
    return ctx


def _kvectors(L, alpha, P, seed):
    """P integer k-vectors m != 0 of a box, each with the probability of RBE's sampling measure
    exp(-(2 pi m / L)^2 / 4 alpha)."""
    rng = np.random.default_rng(seed)
    out = np.zeros((0, 3), dtype=np.int32)
    sd = np.sqrt(alpha) * np.asarray(L) / (math.sqrt(2.0) * math.pi)
    while len(out) < P:
        m = np.rint(rng.normal(size=(2 * P + 16, 3)) * sd).astype(np.int32)
        out = np.concatenate([out, m[np.any(m != 0, axis=1)]])
    return out[:P]


def _positions(s, k):
    """Positions (N, 3) of step k of a host program's short trajectory."""
    return s.pos + (0.0025 * k) * s.vel


def _sizes(case):
    """Atom counts of a batch's boxes: log-uniform between nmin and nmax."""
    rng = np.random.default_rng((case["nrep"], case["nmin"], case["nmax"]))
    return np.rint(np.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"]),
                                      case["nrep"]))).astype(int)


def _match_params(seed):
    """Type charges, eps and sigma of the two training steps."""
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(2):
        q = 1.0 + 0.02 * rng.normal()
        out.append((np.array([q, -q, 0.0]), 1.0 + 0.02 * rng.normal(size=3),
                    1.0 + 0.005 * rng.normal(size=3)))
    return out


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "md":
        s = _lj_system(case["n"], seed, 0.1 if case["system"] == "salt" else 0.0)
        dt = torch.float64 if case["precision"] == "fp64" else torch.float32
        ctx = _context(case, s, seed)
        ctx.set_masses(np.ones(len(s.eps)))
        x = _wrap32(s.pos, s.L, dt)
        v = s.vel.T.contiguous().to(dt)
        f = torch.zeros_like(x)
        img = torch.zeros((3, s.n), dtype=torch.int32, device=DEV)
        st.update(ctx=ctx, x=x, v=v, f=f, img=img)
        ctx.md_init(tuple(x), tuple(v), tuple(f), image=tuple(img), energy=case["energy"])
    elif kind == "steps":
        s = (_water(case["n"], seed) if case["system"] == "water"
             else _lj_system(case["n"], seed, case["ions"]))
        frames = [_wrap32(_positions(s, k), s.L) for k in range(case["frames"])]
        st.update(ctx=_context(case, s, seed), frames=frames, x=frames[0].clone(),
                  v=torch.zeros_like(frames[0]), f=torch.zeros_like(frames[0]))
    elif kind == "rerun":
        ss = [_lj_system(case["n"], seed + 7919 * k, case["ions"]) for k in range(case["frames"])]
        s = ss[0]
        m = [torch.tensor(_kvectors(s.L, 0.09, case["P"], seed + k).reshape(-1), device=DEV)
             for k in range(case["frames"])]
        st.update(ctx=_context(case, s, seed), m=m,
                  frames=[_wrap32(q.pos, s.L) for q in ss],
                  f=[torch.zeros((3, s.n), device=DEV) for _ in ss])
    elif kind == "batch":
        from rbmd_amd import BatchContext

        reps = [_lj_system(int(n), seed + 31 * r, 0.1) for r, n in enumerate(_sizes(case))]
        b = BatchContext(_config(case, seed), device=0)
        b.set_systems(reps)
        x = torch.cat([_wrap32(s.pos, s.L) for s in reps], 1).contiguous()
        m = torch.tensor(np.concatenate([_kvectors(s.L, 0.09, case["P"], seed + r).reshape(-1)
                                         for r, s in enumerate(reps)]), device=DEV)
        st.update(ctx=b, x=x, f=torch.zeros_like(x), m=m)
    elif kind == "match":
        from rbmd_amd.autograd import DifferentiableForce

        ss = [_lj_system(case["n"], seed + 7919 * k, 0.1) for k in range(2)]
        # one labelled system: the same atoms in two configurations
        s = ss[0]
        model = DifferentiableForce(_config(case, seed), s)
        gen = _rng(seed + 5)
        st.update(model=model, pos=[_wrap32(q.pos, s.L).T.contiguous() for q in ss],
                  target=[5.0 * torch.randn((s.n, 3), generator=gen, device=DEV)
                          for _ in range(2)],
                  par=[[torch.tensor(a, device=DEV) for a in p] for p in _match_params(seed)],
                  m=[torch.tensor(_kvectors(s.L, 0.09, case["P"], seed + k).reshape(-1),
                                  device=DEV) for k in range(2)])
    else:
        s = _lj_system(case["n"], seed, 0.1)
        x = _wrap32(s.pos, s.L)
        G = torch.randn((3, s.n), generator=_rng(seed + 5), device=DEV)
        m = torch.tensor(_kvectors(s.L, 0.09, case["P"], seed).reshape(-1), device=DEV)
        st.update(ctx=_context(case, s, seed), x=x, f=torch.zeros_like(x), G=G,
                  d=torch.zeros_like(x), m=m,
                  dparam=torch.zeros(9, dtype=torch.float64, device=DEV))
    return st


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------
def _thermo(ctx):
    t = ctx.thermo()
    return np.array([t["e_vdwl"], t["e_coul"], t["e_kspace"], *t["virial"]])


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "md":
        x, v, f, img = st["x"], st["v"], st["f"], st["img"]
        st["ctx"].md_run(case["nsteps"], tuple(x), tuple(v), tuple(f), image=tuple(img),
                         energy=case["energy"])
        return [x, v, f]
    if kind == "steps":
        # the host program's loop: write the step's positions, evaluate, apply the force
        ctx, x, v, f = st["ctx"], st["x"], st["v"], st["f"]
        px, py, pz = x
        fx, fy, fz = f
        v.zero_()
        for k, fr in enumerate(st["frames"]):
            x.copy_(fr)
            ctx.force(k, px, py, pz, fx, fy, fz, energy=case["energy"])
            v.add_(f, alpha=0.0025)
        return [v, f, _thermo(ctx)] if case["energy"] else [v, f]
    if kind == "rerun":
        out = []
        for k, x in enumerate(st["frames"]):
            f = st["f"][k]
            st["ctx"].force(k, x[0], x[1], x[2], f[0], f[1], f[2], m_samples=st["m"][k],
                            energy=True)
            out += [f, _thermo(st["ctx"])]
        return out
    if kind == "batch":
        x, f = st["x"], st["f"]
        st["ctx"].force(1, x[0], x[1], x[2], f[0], f[1], f[2], m_samples=st["m"],
                        energy=case["energy"])
        return [f, st["ctx"].energies()] if case["energy"] else [f]
    if kind == "match":
        out = []
        for k in range(2):
            leaves = [st["pos"][k].detach().requires_grad_(True)]
            leaves += [p.detach().requires_grad_(True) for p in st["par"][k]]
            F = st["model"](*leaves, step=k, m_samples=st["m"][k])
            ((F - st["target"][k]) ** 2).sum().backward()
            out += [F.detach()] + [p.grad for p in leaves]
        return out
    x, f, G, d = st["x"], st["f"], st["G"], st["d"]
    st["ctx"].force(1, x[0], x[1], x[2], f[0], f[1], f[2], m_samples=st["m"])
    st["ctx"].force_vjp(1, x[0], x[1], x[2], G[0], G[1], G[2], d[0], d[1], d[2], st["dparam"])
    return [f, d, st["dparam"]]


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------
def _ball(r):
    return 4.0 / 3.0 * math.pi * r ** 3


def work(case):
    """Bytes: positions in and forces out (and what the integrator reads and writes) once per
    evaluation.  Operations: about 27 per LJ pair inside the cutoff and 45 per charged pair the
    force keeps, with energies 20 more for each pair inside the cutoff, and 30 per charged atom
    and k-vector (phase, sine and cosine, structure factor and force)."""
    kind = case["kind"]
    fp = 8 if case.get("precision") == "fp64" else 4
    e = 20 if case.get("energy") or kind == "rerun" else 0
    if kind == "batch":
        n = case["nrep"] * (case["nmax"] - case["nmin"]) / math.log(case["nmax"] / case["nmin"])
    else:
        n = case["n"] * (3 if case.get("system") == "water" else 1)
    if case.get("system") == "lj":
        flops = n * RHO * _ball(2.5) * (27 + e)
        return {"bytes": case["nsteps"] * n * fp * 15.0, "flops": case["nsteps"] * flops}
    if case.get("system") == "water":
        dens = 0.1002
        full = _ball(10.0) * dens
        kept = full if case["neighbor"] != "RBL" else _ball(6.5) * dens + 100
        pairs = n * (kept * 45 + full * e)
        nq = n
    else:
        ions = case.get("ions", 0.1)
        nq = n * ions
        full = RHO * ions * _ball(3.5)
        kept = full if case.get("neighbor", "RBL") != "RBL" else min(
            full, RHO * ions * _ball(2.5) + 30 * ions)
        lj = n * RHO * _ball(2.5)
        pairs = lj * (27 + e) + nq * (kept * 45 + full * e)
    K = (2 * case["kmax"] + 1) ** 3 - 1 if case.get("coulomb") == "EWALD" else case["P"]
    flops = pairs + 30.0 * nq * K
    per = {"md": case.get("nsteps", 1), "steps": case.get("frames", 1),
           "rerun": case.get("frames", 1), "match": 2}.get(kind, 1)
    if kind == "md":
        return {"bytes": per * n * 4 * 15.0, "flops": per * flops}
    if kind in ("match", "adjoint"):
        # the adjoint reads positions and cotangents, writes gradients, and evaluates about twice
        # the forward's operations
        return {"bytes": per * n * 4 * 15.0, "flops": per * 3 * flops}
    return {"bytes": per * n * 4 * (9.0 if kind == "steps" else 6.0), "flops": per * flops}


# ---------------------------------------------------------------------------------------------
# tolerances
# ---------------------------------------------------------------------------------------------
def tolerance(case):
    # A correct FP32 evaluation is 1e-6 to 7e-6 from FP64 (the most where one close pair across a
    # box edge carries much of the norm; about 1e-5 for water, whose Coulomb terms nearly cancel).
    # The same system with its atoms in another order, hence all sums in another order, is 1e-7
    # from the first.  The largest difference sits at an atom whose terms cancel: 1e-4 to 5e-4 of
    # the root mean square.  About four times what is seen.
    kind = case["kind"]
    if kind == "md":
        if case["precision"] == "fp64":
            return {"rel": 1e-11, "max": 1e-8}
        # rounding grows along the steps of a pass, and a pair at r_core may change its class
        return {"rel": 5e-5, "max": 5e-2}
    if case.get("system") == "water":
        return {"rel": 3e-5, "max": 3e-3}
    return {"rel": 2e-5, "max": 2e-3}


# ---------------------------------------------------------------------------------------------
# results in 64 bits
# ---------------------------------------------------------------------------------------------
_M64 = (1 << 64) - 1


def _i64(v):
    v &= _M64
    return v - (1 << 64) if v >> 63 else v


def _shr(v, s):
    return (v >> s) & ((1 << (64 - s)) - 1)


def _mix64(v):
    """The 64-bit finaliser of the shell selection (int64 tensors, wrapping arithmetic)."""
    v = v + _i64(0x9e3779b97f4a7c15)
    v = (v ^ _shr(v, 30)) * _i64(0xbf58476d1ce4e5b9)
    v = (v ^ _shr(v, 27)) * _i64(0x94d049bb133111eb)
    return v ^ _shr(v, 31)


def _selected(f, step, hi, hj):
    """Whether the shell keeps directed pairs with hash halves hi, hj: hash mod f == 0."""
    h = _mix64(hi ^ hj ^ step)
    # unsigned h mod f from its halves
    up, lo = _shr(h, 32), h & 0xffffffff
    return ((up % f) * ((1 << 32) % f) + lo) % f == 0


def _frequency(n, L, r_core, rc, samples):
    """Every how many shell atoms one is kept, so that about `samples` are."""
    f4 = np.float32
    rho = f4(n) / (f4(L[0]) * f4(L[1]) * f4(L[2]))
    co = int(np.round(np.float64(f4(1.0 + (0.05 / float(rho) - 0.05)))))
    num = [int(float(f4(co) * rho) * math.ceil(4.0 / 3.0 * math.pi * float(f4(r)) ** 3) + 1)
           for r in (r_core, rc)]
    shell = num[1] - num[0]
    return 1 if shell <= samples else int(math.ceil(f4(shell) / f4(samples)))


def _pair_chunks(x, L, rc, most=1 << 25):
    """Directed pairs (i, j) closer than about rc, in chunks, from a cell table."""
    n = len(x)
    nc = [max(1, int(L[d] / (rc * 1.001))) for d in range(3)]
    if min(nc) < 3:
        nc = [1, 1, 1]
    Lt = torch.tensor(L, device=DEV, dtype=torch.float64)
    u = x.double()
    c = torch.stack([(u[:, d] / L[d] * nc[d]).long().clamp(0, nc[d] - 1) for d in range(3)], 1)
    cid = (c[:, 2] * nc[1] + c[:, 1]) * nc[0] + c[:, 0]
    ncell = nc[0] * nc[1] * nc[2]
    order = cid.argsort(stable=True)
    cnt = torch.bincount(cid, minlength=ncell)
    M = int(cnt.max())
    start = cnt.cumsum(0) - cnt
    slot = torch.arange(n, device=DEV) - start[cid[order]]
    table = torch.full((ncell, M), -1, dtype=torch.long, device=DEV)
    table[cid[order], slot] = order
    offs = [(0, 0, 0)] if ncell == 1 else [(a, b, e) for a in (-1, 0, 1) for b in (-1, 0, 1)
                                           for e in (-1, 0, 1)]
    if ncell == 1:
        for a in range(0, n, max(1, most // n)):
            i = torch.arange(a, min(n, a + max(1, most // n)), device=DEV)
            d = u[None, :, :] - u[i][:, None, :]
            d = d - Lt * torch.round(d / Lt)
            d2 = (d * d).sum(-1)
            ii, j = torch.nonzero(d2 < (rc * 1.0001) ** 2, as_tuple=True)
            i = i[ii]
            keep = i != j
            yield i[keep], j[keep]
        return
    step = max(1, most // (M * M * 3))
    cc = torch.arange(ncell, device=DEV)
    cx, cy, cz = cc % nc[0], (cc // nc[0]) % nc[1], cc // (nc[0] * nc[1])
    for o in offs:
        nb = (((cz + o[2]) % nc[2]) * nc[1] + (cy + o[1]) % nc[1]) * nc[0] + (cx + o[0]) % nc[0]
        for a in range(0, ncell, step):
            ti, tj = table[a:a + step], table[nb[a:a + step]]
            d = u[tj.clamp(min=0)][:, None, :, :] - u[ti.clamp(min=0)][:, :, None, :]
            d = d - Lt * torch.round(d / Lt)
            d2 = (d * d).sum(-1)
            ok = (d2 < (rc * 1.0001) ** 2) & (ti[:, :, None] >= 0) & (tj[:, None, :] >= 0) & (
                ti[:, :, None] != tj[:, None, :])
            w = torch.nonzero(ok, as_tuple=True)
            yield ti[w[0], w[1]], tj[w[0], w[2]]


def _exact_force(x, L, s, cfg, step, kv, kw, G=None, params=None):
    """The total force (N, 3) in FP64 of FP32 positions x (N, 3), with [E_lj, E_coul, E_k,
    virial] and, for a cotangent G (N, 3), dL/dr and dL/d(Q, eps, sigma) per type."""
    hp = cfg["hyper_parameters"]
    nb, cl = hp["neighbor"], hp.get("coulomb")
    real = cfg["init_configuration"]["read_data"]["unit"] == "REAL"
    qqr2e = QQR2E_REAL if real else 1.0
    rc, rlj = nb["cut_off"], nb.get("lj_cut_off", nb["cut_off"])
    rbl = nb["type"] == "RBL"
    n = len(x)
    f32 = np.float32
    T = lambda a, t=torch.float64: torch.tensor(np.asarray(a), device=DEV, dtype=t)  # noqa: E731
    types = T(s.types, torch.long)
    ids = T(s.ids, torch.long)
    Q, eps, sigma = ([T(a) for a in params] if params else
                     [T(getattr(s, "Q", np.zeros(len(s.eps)))), T(s.eps), T(s.sigma)])
    q = Q[types] if params or hasattr(s, "Q") else T(s.charges)
    alpha = float(f32(cl["alpha"])) if cl else 0.0
    g = math.sqrt(cl["alpha"]) if cl else 0.0
    rs2 = f32(nb.get("r_core", 0)) * f32(nb.get("r_core", 0))
    rc2, rl2 = f32(rc) * f32(rc), f32(rlj) * f32(rlj)
    e4 = f32(1e-4)
    freq = _frequency(n, L, nb["r_core"], rc, nb["neighbor_sample_num"]) if rbl else 1
    hi = _mix64(ids)
    hj = _mix64(ids + _i64(0xd1b54a32d192ed03))
    L32 = T(L, torch.float32)
    fp64in = x.dtype == torch.float64
    xd = x.double()
    Lt = T(L)
    F = torch.zeros((n, 3), dtype=torch.float64, device=DEV)
    th = torch.zeros(9, dtype=torch.float64, device=DEV)
    dr = torch.zeros_like(F)
    dp = [torch.zeros_like(Q), torch.zeros_like(eps), torch.zeros_like(sigma)]
    Gm = None
    if G is not None:
        Gm = G.double()
        Gm = Gm - Gm.mean(0) if rbl else Gm

    def classes(i, j):
        # the squared distance that decides a pair's class is rounded to the program's precision
        if fp64in:
            d = xd[j] - xd[i]
            d = d - Lt * torch.round(d / Lt)
            return (d * d).sum(-1)
        d = x[j] - x[i]
        d = torch.where(d.abs() > 0.5 * L32, d - torch.copysign(L32.expand_as(d), d), d).double()
        t = (d[:, 0] * d[:, 0]).float().double()
        t = (d[:, 1] * d[:, 1] + t).float().double()
        return (d[:, 2] * d[:, 2] + t).float().double()

    for i, j in _pair_chunks(x, L, max(rc, rlj) if cl else rlj):
        qq = q[i] * q[j]
        c2 = classes(i, j)
        keep = (c2 < float(rc2)) & ((c2 < float(rl2)) | (qq != 0))
        i, j, c2, qq = i[keep], j[keep], c2[keep], qq[keep]
        w = torch.ones_like(c2)
        if rbl:
            core = c2 < float(f32(rs2 - e4))
            sel = _selected(freq, step, hi[i], hj[j])
            w = torch.where(core, ((c2 < float(rs2)) & (c2 > float(e4))).double(),
                            ((c2 < float(f32(rc2 - e4))) & (c2 > float(rs2)) & sel).double()
                            * freq)
        inlj = c2 < float(rl2)

        def terms(xx, Qt, et, sg):
            d = xx[j] - xx[i]
            d = d - Lt * torch.round(d.detach() / Lt)
            u = (d * d).sum(-1)
            ee = torch.sqrt(et[types[i]] * et[types[j]])
            ss = (sg[types[i]] + sg[types[j]]) / 2
            s6 = (ss * ss / u) ** 3
            z = torch.zeros_like(u)
            fl = torch.where(inlj, -24 * ee * (2 * s6 - 1) * s6 / u, z)
            el = torch.where(inlj, 2 * ee * (s6 - 1) * s6, z)
            if cl is None:
                return d, fl, el, z
            r = torch.sqrt(u)
            ec = torch.erfc(g * r)
            pq = qq if Qt is None else Qt[types[i]] * Qt[types[j]] * (qq != 0)
            fc = -qqr2e * pq * (ec / u + 2 * g / math.sqrt(math.pi) * torch.exp(-alpha * u) / r) / r
            return d, fl + fc, el, 0.5 * qqr2e * pq * ec / r

        with torch.no_grad():
            d, f, el, ec = terms(xd, None, eps, sigma)
            F.index_add_(0, i, (w * f)[:, None] * d)
            th[0] += el.sum()
            th[1] += ec.sum()
            for k, (a, b) in enumerate(((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))):
                th[3 + k] += (-0.5 * f * d[:, a] * d[:, b]).sum()
        if Gm is not None:
            # chunks of pairs through autograd (the adjoint of the weighted pair sum)
            lv = [xd.clone().requires_grad_(True)] + [p.clone().requires_grad_(True)
                                                      for p in (Q, eps, sigma)]
            d, f, _, _ = terms(*lv)
            out = torch.autograd.grad(((Gm[i] * d).sum(-1) * w * f).sum(), lv)
            dr += out[0]
            for a, b in zip(dp, out[1:]):
                a += b
    if rbl:
        F -= F.mean(0)
    if cl is not None:
        ci = torch.nonzero(q)[:, 0]
        V = float(np.prod(L))
        kvec = 2 * math.pi * T(kv) / Lt
        k2 = (kvec ** 2).sum(1)
        A = T(kw) * (-4 * math.pi * qqr2e) / (V * k2)
        xc, qc, tc = xd[ci], q[ci], types[ci]
        Fk = torch.zeros_like(xc)
        step_k = max(1, (1 << 24) // max(1, len(ci)))
        for a in range(0, len(kvec), step_k):
            kk, Ak = kvec[a:a + step_k], A[a:a + step_k]

            def kforce(xx, qv):
                ph = xx @ kk.T
                cs, sn = torch.cos(ph), torch.sin(ph)
                re, im = qv @ cs, qv @ sn
                return (qv[:, None] * Ak * (im * cs - re * sn)) @ kk, re, im

            with torch.no_grad():
                fk, re, im = kforce(xc, qc)
                Fk += fk
                base = qqr2e * 2 * math.pi / V * T(kw)[a:a + step_k] * (re ** 2 + im ** 2) / \
                    k2[a:a + step_k]
                th[2] += base.sum()
                cc = 2 * (1 / (4 * cl["alpha"]) + 1 / k2[a:a + step_k])
                for m, (b, e) in enumerate(((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))):
                    th[3 + m] += (base * (float(b == e) - cc * kk[:, b] * kk[:, e])).sum()
            if G is not None:
                lx = xc.clone().requires_grad_(True)
                lq = Q.clone().requires_grad_(True)
                fk, _, _ = kforce(lx, lq[tc])
                gx, gq = torch.autograd.grad((G.double()[ci] * fk).sum(), (lx, lq))
                dr.index_add_(0, ci, gx)
                dp[0] += gq
        F.index_add_(0, ci, Fk)
        th[2] += -qqr2e * (math.sqrt(cl["alpha"] / math.pi) * (q * q).sum() +
                           0.5 * math.pi * q.sum() ** 2 / (cl["alpha"] * V))
    return F, th.cpu().numpy(), dr, dp


def _rbe_weight(L, alpha, P):
    h = 1.0
    for Ld in L:
        t = alpha * Ld * Ld
        h *= math.sqrt(t / math.pi) * sum(math.exp(-m * m * t) for m in range(-10, 11))
    return np.full(P, (h - 1.0) / P)


def exact(case, seed):
    kind = case["kind"]
    cfg = _config(case, seed)
    if kind == "md":
        if case["system"] != "lj" or case["precision"] != "fp64" or case["n"] > 20000:
            return None  # chaotic in FP32; the sampled k-vectors are the framework's own stream
        s = _lj_system(case["n"], seed)
        dt = cfg["execution"]["timestep"]
        x = _wrap32(s.pos, s.L, torch.float64).T.contiguous()
        v = s.vel.clone()
        Lt = torch.tensor(s.L, device=DEV, dtype=torch.float64)
        f = _exact_force(x, s.L, s, cfg, 0, None, None)[0]
        for _ in range(case["nsteps"]):
            v = v + 0.5 * dt * f
            x = x + dt * v
            x = torch.where(x >= Lt, x - Lt, x)
            x = torch.where(x < 0, x + Lt, x)
            f = _exact_force(x, s.L, s, cfg, 0, None, None)[0]
            v = v + 0.5 * dt * f
        return [a.T.contiguous() for a in (x, v, f)]
    if kind == "steps":
        if case["coulomb"] != "EWALD":
            return None  # the k-sample of each step is the framework's own stream
        s = _lj_system(case["n"], seed, case["ions"])
        km = case["kmax"]
        r = np.arange(-km, km + 1)
        kv = np.stack(np.meshgrid(r, r, r, indexing="ij"), -1).reshape(-1, 3)
        kv = kv[np.any(kv != 0, axis=1)]
        k2 = ((2 * np.pi * kv / s.L) ** 2).sum(1)
        kw = np.exp(-k2 / (4 * cfg["hyper_parameters"]["coulomb"]["alpha"]))
        imp = torch.zeros((s.n, 3), dtype=torch.float64, device=DEV)
        for k in range(case["frames"]):
            x = _wrap32(_positions(s, k), s.L).T.contiguous()
            F, th, _, _ = _exact_force(x, s.L, s, cfg, k, kv, kw)
            imp += 0.0025 * F
        out = [imp.T.contiguous(), F.T.contiguous()]
        return out + [th] if case["energy"] else out
    if kind == "rerun":
        ss = [_lj_system(case["n"], seed + 7919 * k, case["ions"]) for k in range(case["frames"])]
        s, out = ss[0], []
        for k, q in enumerate(ss):
            kv = _kvectors(s.L, 0.09, case["P"], seed + k)
            x = _wrap32(q.pos, s.L).T.contiguous()
            F, th, _, _ = _exact_force(x, s.L, s, cfg, k, kv, _rbe_weight(s.L, 0.09, case["P"]))
            out += [F.T.contiguous(), th]
        return out
    if kind == "batch":
        out, en = [], []
        for r, n in enumerate(_sizes(case)):
            s = _lj_system(int(n), seed + 31 * r, 0.1)
            kv = _kvectors(s.L, 0.09, case["P"], seed + r)
            x = _wrap32(s.pos, s.L).T.contiguous()
            F, th, _, _ = _exact_force(x, s.L, s, cfg, 1, kv, _rbe_weight(s.L, 0.09, case["P"]))
            out.append(F.T)
            en.append(th)
        f = torch.cat(out, 1).contiguous()
        return [f, np.stack(en)] if case["energy"] else [f]
    if kind == "match":
        ss = [_lj_system(case["n"], seed + 7919 * k, 0.1) for k in range(2)]
        s, out = ss[0], []
        gen = _rng(seed + 5)
        target = [5.0 * torch.randn((s.n, 3), generator=gen, device=DEV) for _ in range(2)]
        for k, par in enumerate(_match_params(seed)):
            kv = _kvectors(s.L, 0.09, case["P"], seed + k)
            x = _wrap32(ss[k].pos, s.L).T.contiguous()
            kw = _rbe_weight(s.L, 0.09, case["P"])
            F = _exact_force(x, s.L, s, cfg, k, kv, kw, params=par)[0]
            G = 2.0 * (F - target[k].double())
            _, _, dr, dp = _exact_force(x, s.L, s, cfg, k, kv, kw, G=G, params=par)
            out += [F, dr, *dp]
        return out
    s = _lj_system(case["n"], seed, 0.1)
    x = _wrap32(s.pos, s.L).T.contiguous()
    G = torch.randn((3, s.n), generator=_rng(seed + 5), device=DEV).T.contiguous()
    kv = _kvectors(s.L, 0.09, case["P"], seed)
    F, _, dr, dp = _exact_force(x, s.L, s, cfg, 1, kv, _rbe_weight(s.L, 0.09, case["P"]), G=G,
                                params=[s.Q, s.eps, s.sigma])
    return [F.T.contiguous(), dr.T.contiguous(), torch.cat(dp)]
