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
