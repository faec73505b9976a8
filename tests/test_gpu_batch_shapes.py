"""Replica batch at the edges of its work split: launch shapes from one wave to
four per workgroup and one to 64 lanes per charged atom, replicas without
charges, with a single ion pair and with every atom charged, an LJ cutoff
beyond r_core (RBL shell pairs in the LJ pass), and a dense replica whose
brick neighbourhood exceeds the LDS stage (several windows).  Every replica
against the FP64 oracle of its box; forces 2e-5 relative RMS, energies 1e-5
of the terms they add up (as tests/test_gpu_batch.py).
"""
import numpy as np
import pytest

from rbmd_amd import BatchContext, rbe_sample_host, systems
from tests.refs import coul_abs_scale, reference_force, rel_rms

pytestmark = pytest.mark.gpu

SHAPES = [dict(bw=2, pair_block=256, grid_per_cu=8, qlanes=16),
          dict(bw=1, pair_block=64, grid_per_cu=1, qlanes=64),
          dict(bw=2, pair_block=64, grid_per_cu=16, qlanes=1),
          dict(bw=2, pair_block=128, grid_per_cu=2, qlanes=2)]


def _replicas(kind):
    if kind == "ions":
        return [systems.electrolyte(n, frac_ion=f, seed=90 + k)
                for k, (n, f) in enumerate([(501, 0.0), (640, 0.002), (777, 0.5), (2300, 0.05)])]
    # dense: neighbourhoods of 64 cells of more than 24 atoms
    return [systems.electrolyte(900, rho=1.5, d_min=0.6, seed=95),
            systems.electrolyte(2400, rho=1.5, d_min=0.6, seed=96)]


@pytest.mark.parametrize("kind,lj_cut", [("ions", 2.5), ("ions", 3.2), ("dense", 2.5)])
@pytest.mark.parametrize("shape", SHAPES)
def test_batch_shapes_match_the_oracle(device, kind, lj_cut, shape):
    import torch

    P, step = 70, 3
    cfg = systems.ljsalt_config(P=P, lj_cut_off=lj_cut)
    reps = _replicas(kind)
    b = BatchContext(cfg, device=0)
    b.set_systems(reps)
    b.set_shape(**shape)
    p = torch.tensor(np.concatenate([s.pos for s in reps]).astype(np.float32), device=device)
    px, py, pz = (p[:, d].contiguous() for d in range(3))
    f = [torch.zeros(b.n, dtype=torch.float32, device=device) for _ in range(3)]
    ms = [rbe_sample_host(0.09, s.box_len, P, 17 + r, step) for r, s in enumerate(reps)]
    m = torch.tensor(np.concatenate(ms).reshape(-1).astype(np.int32), device=device)
    out = []
    for energy in (False, True):
        b.force(step, px, py, pz, *f, m_samples=m, energy=energy, sync=True)
        out.append(np.stack([t.double().cpu().numpy() for t in f], 1))
    E = b.energies()
    for r, s in enumerate(reps):
        a, e = b.offsets[r], b.offsets[r + 1]
        Fo, en, vir, ek, vk = reference_force(s, s.pos.astype(np.float32), cfg, step, ms[r])
        for F in out:
            assert rel_rms(F[a:e], Fo) < 2e-5
        np.testing.assert_allclose(E[r, 0], en[0], rtol=1e-5)
        # the Coulomb terms' signs cancel: bounded by the sum of their sizes
        scale = coul_abs_scale(s, 3.5, 0.09, 1.0) if np.any(s.charges) else 0.0
        np.testing.assert_allclose(E[r, 1], en[1], rtol=0, atol=1e-6 * scale + 1e-12)
        np.testing.assert_allclose(E[r, 2], ek, rtol=1e-5, atol=1e-9)
        w = np.asarray(vir) + np.asarray(vk)
        np.testing.assert_allclose(E[r, 3:], w, rtol=1e-5, atol=1e-5 * np.abs(w).max())


def _pair_box(L, pos, q):
    s = systems.electrolyte(2, frac_ion=0.0, seed=1)
    s.box_len = np.array([L, L, L], dtype=np.float64)
    s.box_lo = np.zeros(3)
    s.pos = pos.astype(np.float64)
    s.types = np.array([0, 1] if q else [2, 2], dtype=np.int32)
    s.charges = np.array([1.0, -1.0] if q else [0.0, 0.0])
    return s


@pytest.mark.parametrize("q,rc,cells", [(0, 2.5, 3), (1, 3.5, 3), (1, 2.5, 5)])
def test_pairs_at_the_cutoff_across_an_edge(device, q, rc, cells):
    """Boxes of three and four cells per dimension (of five and six for the LJ
    term of two ions) holding one pair across an edge, within rounding of the
    cutoff: it carries a force exactly when the FP32 square of its minimum image
    (one subtraction of L from r_j - r_i) is below the cutoff's."""
    import torch

    f32 = np.float32
    rng = np.random.default_rng(5 + q)
    reps, want = [], []
    for r in range(192):
        L = float(f32(rng.uniform(2.53 * cells, 2.48 * (cells + 2))))
        u = rng.normal(size=3)
        u[r % 3] = 3.0 * np.sign(u[r % 3])
        u /= np.linalg.norm(u)
        x0 = rng.uniform(0.3, 0.7, 3) * L
        x0[r % 3] = L - 0.3 if u[r % 3] > 0 else 0.3
        x1 = x0 + u * (rc + rng.uniform(-6e-7, 6e-7))
        x0, x1 = x0.astype(f32), (x1 - L * np.floor(x1 / L)).astype(f32)
        d = x1 - x0
        d = np.where(np.abs(d) > f32(0.5) * f32(L), d - np.copysign(f32(L), d), d)
        t = f32(d[0] * d[0])
        for k in (1, 2):  # fused: one rounding
            t = f32(np.float64(d[k]) * np.float64(d[k]) + np.float64(t))
        want.append(bool(t < f32(rc) * f32(rc)))
        reps.append(_pair_box(L, np.stack([x0, x1]), q))
    assert 40 < sum(want) < 152
    cfg = systems.ljsalt_config(P=8)
    cfg["hyper_parameters"]["neighbor"].update(type="Verlet-List")
    b = BatchContext(cfg, device=0)
    b.set_systems(reps)
    p = torch.tensor(np.concatenate([s.pos for s in reps]).astype(f32), device=device)
    px, py, pz = (p[:, d].contiguous() for d in range(3))
    m = torch.zeros(3 * 8 * len(reps), dtype=torch.int32, device=device)
    m[0::3] = 1
    f = [torch.zeros(b.n, dtype=torch.float32, device=device) for _ in range(3)]
    b.force(1, px, py, pz, *f, m_samples=m, energy=True, sync=True)
    E = b.energies()
    # the pair's own energy term: the k-space force of a charged pair is never 0
    got = E[:, 1 if rc == 3.5 else 0] != 0.0
    assert got.tolist() == want
    # the pass without energies takes the same pairs (a class is 0.04 of force;
    # the terms of the two passes differ by a few roundings of at most 1)
    fe = [t.clone() for t in f]
    b.force(1, px, py, pz, *f, m_samples=m, energy=False, sync=True)
    for t, te in zip(f, fe):
        assert float((t - te).abs().max()) < 1e-5


@pytest.mark.parametrize("lj_cut", [2.5, 3.2])
def test_core_pairs_across_an_edge(device, lj_cut):
    """RBL: pairs of two (weakly charged) ions across an edge of five or six cells,
    within rounding of the core's bound r_core^2 - 1e-4: the LJ force is there exactly
    when the FP32 square of the minimum image is below it, in the pass with energies
    as in the one without.  Beyond it, up to r_core, no class holds the pair."""
    import torch

    f32 = np.float32
    rng = np.random.default_rng(11)
    t_core = f32(f32(2.5) * f32(2.5) - f32(1e-4))
    reps, want = [], []
    for r in range(192):
        L = float(f32(rng.uniform(5.05 * lj_cut, 5.4 * lj_cut)))
        u = rng.normal(size=3)
        u[r % 3] = 3.0 * np.sign(u[r % 3])
        u /= np.linalg.norm(u)
        x0 = rng.uniform(0.3, 0.7, 3) * L
        x0[r % 3] = L - 0.3 if u[r % 3] > 0 else 0.3
        x1 = x0 + u * (np.sqrt(float(t_core)) + rng.uniform(-6e-7, 6e-7))
        x0, x1 = x0.astype(f32), (x1 - L * np.floor(x1 / L)).astype(f32)
        d = x1 - x0
        d = np.where(np.abs(d) > f32(0.5) * f32(L), d - np.copysign(f32(L), d), d)
        t = f32(d[0] * d[0])
        for k in (1, 2):  # fused: one rounding
            t = f32(np.float64(d[k]) * np.float64(d[k]) + np.float64(t))
        want.append(bool(t < t_core))
        s = _pair_box(L, np.stack([x0, x1]), 1)
        s.charges = 1e-3 * s.charges
        reps.append(s)
    assert 40 < sum(want) < 152
    b = BatchContext(systems.ljsalt_config(P=8, lj_cut_off=lj_cut), device=0)
    b.set_systems(reps)
    p = torch.tensor(np.concatenate([s.pos for s in reps]).astype(f32), device=device)
    px, py, pz = (p[:, d].contiguous() for d in range(3))
    m = torch.zeros(3 * 8 * len(reps), dtype=torch.int32, device=device)
    m[0::3] = 1
    f = [torch.zeros(b.n, dtype=torch.float32, device=device) for _ in range(3)]
    for energy in (False, True):
        b.force(1, px, py, pz, *f, m_samples=m, energy=energy, sync=True)
        # the LJ force at the bound is 0.039, all charged terms are below 1e-5
        F = torch.stack(f, 1).norm(dim=1).cpu().numpy().reshape(-1, 2)
        got = F > 0.02
        assert got[:, 0].tolist() == got[:, 1].tolist() == want


def test_box_edge_of_a_power_of_two(device):
    """Fewer than three cells per dimension (minimum image per pair), edges a
    power of two, full lists, as many atoms as leave lanes idle."""
    import torch

    cfg = systems.ljsalt_config(P=8, lj_cut_off=3.5)
    cfg["hyper_parameters"]["neighbor"].update(type="Verlet-List")
    s = systems.electrolyte(9, frac_ion=0.0, seed=3)
    g = np.stack(np.meshgrid([0, 1, 2], [0, 1, 2], [0], indexing="ij"), -1).reshape(-1, 3)
    s.box_lo, s.box_len = np.zeros(3), np.array([8.0, 8.0, 8.0])
    s.pos = 0.4 + 1.3 * g + 0.05 * np.random.default_rng(4).normal(size=(9, 3))
    b = BatchContext(cfg, device=0)
    b.set_systems([s])
    p = torch.tensor(s.pos.astype(np.float32), device=device)
    px, py, pz = (p[:, d].contiguous() for d in range(3))
    f = [torch.zeros(b.n, dtype=torch.float32, device=device) for _ in range(3)]
    kv = np.tile(np.array([[1, 0, 0]], dtype=np.int32), (8, 1))
    m = torch.tensor(kv.reshape(-1), device=device)
    Fo, en, _, _, _ = reference_force(s, s.pos.astype(np.float32), cfg, 1, kv)
    for energy in (False, True):
        b.force(1, px, py, pz, *f, m_samples=m, energy=energy, sync=True)
        assert rel_rms(np.stack([t.double().cpu().numpy() for t in f], 1), Fo) < 2e-5
    np.testing.assert_allclose(b.energies()[0, 0], en[0], rtol=1e-5)
