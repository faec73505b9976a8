"""Sizes at which the launch rules change: lanes per atom over list A (8, 4, 2, 1),
single-cell bricks, the one-block rebuild (at most 16,384 atoms), systems without
list-A pairs, selection frequencies that are and are not powers of two, and the
parameters of a training step set on the stream.

Forces against the FP64 oracle at 2e-5 relative RMS (FP32 terms of about 1e-7
relative, sums of about 100 of them), energies at 1e-5.
"""
import numpy as np
import pytest

from rbmd_amd import ForceContext, RbmdxError, rbe_sample_host, systems
from tests.refs import reference_force, rel_rms
from tests.test_gpu_vjp import _oracle as adjoint_oracle, _run as adjoint

pytestmark = pytest.mark.gpu


def _ctx(s, cfg):
    ctx = ForceContext(cfg, device=0)
    ctx.set_system(s.box_lo, s.box_len, s.types, s.ids, s.charges, s.eps, s.sigma)
    return ctx


def _rows(a, device, dtype):
    import torch

    t = torch.tensor(np.ascontiguousarray(a.T), dtype=dtype, device=device)
    return list(t.unbind())


def _wrap32(pos, L):
    p = (pos - L * np.floor(pos / L)).astype(np.float32)
    return np.where(p >= L.astype(np.float32), np.float32(0), p)


@pytest.mark.parametrize("n,ions,P", [(130, 0.1, 60), (1500, 0.1, 60), (4100, 0.1, 60),
                                      (8193, 0.1, 60), (16384, 0.1, 60), (16385, 0.1, 60),
                                      (33000, 0.1, 60), (16384, 0.5, 1000), (16384, 0.5, 1040)])
def test_forces_where_the_launch_rules_change(device, n, ions, P):
    """Also around 1,024 S(k) blocks (every atom charged, 1,000 and 1,040 k's)."""
    import torch

    s = systems.electrolyte(n, frac_ion=ions, seed=21)
    cfg = systems.ljsalt_config(P=P, cut_off=2.4 if n < 500 else 3.5,
                                lj_cut_off=2.2, r_core=2.2, skin=0.2)
    m = rbe_sample_host(0.09, s.box_len, P, 5, 0)
    mt = torch.tensor(m.reshape(-1).astype(np.int32), device=device)
    ctx = _ctx(s, cfg)
    rng = np.random.default_rng(n)
    f = [torch.zeros(n, device=device) for _ in range(3)]
    # lists built, reused (a tenth of the skin), rebuilt
    for step, amp in enumerate((0.0, 0.01, 0.15)):
        p32 = _wrap32(s.pos + amp * rng.uniform(-1, 1, (n, 3)), s.box_len)
        p = _rows(p32, device, torch.float32)
        ctx.force(step, *p, *f, m_samples=mt, energy=step != 1, sync=True)
        Fo, en, vir, ek, vk = reference_force(s, p32, cfg, step, m)
        assert rel_rms(torch.stack(f, 1).double().cpu().numpy(), Fo) < 2e-5
        if step != 1:
            th = ctx.thermo()
            assert th["e_vdwl"] == pytest.approx(en[0], rel=1e-5)
            assert th["e_kspace"] == pytest.approx(ek, rel=1e-5)
            w = np.asarray(vir) + np.asarray(vk)
            np.testing.assert_allclose(th["virial"], w, rtol=1e-5, atol=1e-5 * np.abs(w).max())
    assert ctx.thermo()["rebuilds"] >= 2


@pytest.mark.parametrize("rho", [0.08, 0.3, 0.5])
def test_sparse_cells(device, rho):
    """Cells of 2, 7 and 11 atoms on average (8 and 16 lanes stage a cell, some cells
    holding more), with lists shorter than a group of entries per lane.  No pair is
    closer than sigma, where rounding a coordinate shifted across the edge (4e-6)
    would move the energy by 12 times as much as r."""
    import torch

    n = 5000
    s = systems.electrolyte(n, rho=rho, frac_ion=0.1, d_min=1.0, seed=13)
    cfg = systems.ljsalt_config(P=40)
    m = rbe_sample_host(0.09, s.box_len, 40, 5, 0)
    mt = torch.tensor(m.reshape(-1).astype(np.int32), device=device)
    ctx = _ctx(s, cfg)
    p32 = _wrap32(s.pos, s.box_len)
    p = _rows(p32, device, torch.float32)
    f = [torch.zeros_like(t) for t in p]
    Fo, en, _, _, _ = reference_force(s, p32, cfg, 2, m)
    for energy in (False, True):
        ctx.force(2, *p, *f, m_samples=mt, energy=energy, sync=True)
        assert rel_rms(torch.stack(f, 1).double().cpu().numpy(), Fo) < 2e-5
    assert ctx.thermo()["e_vdwl"] == pytest.approx(en[0], rel=1e-5)


@pytest.mark.parametrize("n,precision", [(2600, "fp32"), (5000, "fp32"), (2600, "fp64")])
def test_neighbourhoods_beyond_the_stage(device, n, precision):
    """Long cutoffs: neighbourhoods beyond the LDS stage, with lists (2,600 atoms in
    FP32) and beyond the lists' 16-bit offsets (direct scans over an atom's lanes).
    Forces and energies as above, the adjoint as in test_gpu_vjp."""
    import torch

    s = systems.electrolyte(n, frac_ion=0.1, seed=12)
    s.sigma = np.array([1.0, 0.95, 1.05])
    cfg = systems.ljsalt_config(P=40, cut_off=6.0, lj_cut_off=6.0, precision=precision)
    m = rbe_sample_host(0.09, s.box_len, 40, 5, 0)
    mt = torch.tensor(m.reshape(-1).astype(np.int32), device=device)
    ctx = _ctx(s, cfg)
    dt = torch.float32 if precision == "fp32" else torch.float64
    p32 = _wrap32(s.pos, s.box_len)
    p = _rows(p32, device, dt)
    f = [torch.zeros_like(t) for t in p]
    Fo, en, _, _, _ = reference_force(s, p32, cfg, 2, m)
    for energy in (False, True):
        ctx.force(2, *p, *f, m_samples=mt, energy=energy, sync=True)
        assert rel_rms(torch.stack(f, 1).double().cpu().numpy(), Fo) < 2e-5
    assert ctx.thermo()["e_vdwl"] == pytest.approx(en[0], rel=1e-5)
    if precision == "fp32":
        s.pos = p32.astype(np.float64)
        G = np.random.default_rng(7).normal(size=(n, 3))
        _, dr, dp = adjoint(ctx, s, device, 2, m, G)
        _, (dro, *dpo) = adjoint_oracle(s, cfg, 2, m, G)
        assert rel_rms(dr, dro) < 1e-4
        for k, want in enumerate(dpo):
            np.testing.assert_allclose(dp[3 * k:3 * k + 3], want, rtol=0,
                                       atol=1e-4 * np.abs(want).max())


@pytest.mark.parametrize("samples", [1000, 40, 30, 20])
def test_all_charged_selection_frequencies(device, samples):
    """Every atom charged (no list A): frequencies 1, 3, 4 and 5."""
    import torch

    n = 3000
    s = systems.electrolyte(n, frac_ion=0.5, seed=8)
    assert np.all(s.charges != 0)
    cfg = systems.ljsalt_config(P=40, sample_num=samples)
    m = rbe_sample_host(0.09, s.box_len, 40, 5, 0)
    mt = torch.tensor(m.reshape(-1).astype(np.int32), device=device)
    ctx = _ctx(s, cfg)
    f = [torch.zeros(n, device=device) for _ in range(3)]
    p32 = _wrap32(s.pos, s.box_len)
    p = _rows(p32, device, torch.float32)
    for energy in (False, True):
        ctx.force(3, *p, *f, m_samples=mt, energy=energy, sync=True)
        Fo, en, _, _, _ = reference_force(s, p32, cfg, 3, m)
        assert rel_rms(torch.stack(f, 1).double().cpu().numpy(), Fo) < 2e-5
    th = ctx.thermo()
    assert th["e_vdwl"] == pytest.approx(en[0], rel=1e-5)
    assert th["pairs_a"] == 0 and th["rbl_frequency"] == {1000: 1, 40: 3, 30: 4, 20: 5}[samples]


def test_md_runs_split_anywhere(device):
    """NVE (no thermostat factor): one run of 9 steps equals runs of 0, 4, 1 and
    4 bit for bit, with image flags and without."""
    import torch

    s = systems.electrolyte(700, frac_ion=0.0, seed=4)
    cfg = systems.lj_config()
    cfg["execution"] = {"ensemble": "NVE", "timestep": 0.004, "integration_type": "vv"}
    out = []
    for runs, flags in (((9,), True), ((0, 4, 1, 4), True), ((9,), False)):
        ctx = _ctx(s, cfg)
        ctx.set_masses(np.ones(len(s.eps)))
        x, v = (_rows(a, device, torch.float64) for a in (s.pos, s.vel))
        f = [torch.zeros_like(t) for t in x]
        img = tuple(torch.zeros(s.n, dtype=torch.int32, device=device) for _ in range(3))
        ctx.md_init(x, v, f, image=img if flags else None)
        for k in runs:
            ctx.md_run(k, x, v, f, image=img if flags else None)
        assert ctx.md_state()["step"] == 9
        out.append(torch.stack([*x, *v, *f]))
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])


def test_thermostatted_runs_split_anywhere(device):
    """NVT: a run's end applies the factor that the next step would have taken into its
    opening one, which rounds each velocity once more (1.1e-16, FP64) per split; nine
    steps of a liquid multiply a difference by less than ten."""
    import torch

    s = systems.electrolyte(700, frac_ion=0.0, seed=4)
    cfg = systems.lj_config()
    cfg["execution"] = {"ensemble": "NVT", "temp_ctrl_type": "NOSE_HOOVER", "timestep": 0.004,
                        "temperature": [1.5, 1.2, 0.1], "integration_type": "vv",
                        "num_steps": 9}
    out, st = [], []
    for runs in ((9,), (0, 4, 1, 4)):
        ctx = _ctx(s, cfg)
        ctx.set_masses(np.ones(len(s.eps)))
        x, v = (_rows(a, device, torch.float64) for a in (s.pos, s.vel))
        f = [torch.zeros_like(t) for t in x]
        ctx.md_init(x, v, f)
        for k in runs:
            ctx.md_run(k, x, v, f)
        st.append(ctx.md_state())
        out.append(torch.stack([*x, *v]))
    assert st[0]["step"] == st[1]["step"] == 9
    for q in ("temperature", "ke", "t_target", "eta", "eta_dot", "thermostat_energy"):
        np.testing.assert_allclose(st[1][q], st[0][q], rtol=1e-13, atol=1e-15)
    assert float((out[1] - out[0]).abs().max()) < 1e-13


def test_type_parameters_on_the_stream(device):
    """The parameters of a training step: forces bit for bit those of set_charges
    and set_lj, the energies too (the charge sums per type), and a type may not
    become charged or neutral."""
    import torch

    from rbmd_amd.autograd import DifferentiableForce

    s = systems.electrolyte(2000, frac_ion=0.1, seed=6)
    cfg = systems.ljsalt_config(P=40)
    m = rbe_sample_host(0.09, s.box_len, 40, 5, 0)
    mt = torch.tensor(m.reshape(-1).astype(np.int32), device=device)
    pos = torch.tensor(_wrap32(s.pos, s.box_len), device=device)
    model = DifferentiableForce(cfg, s)
    ref = _ctx(s, cfg)
    f = [torch.zeros(s.n, device=device) for _ in range(3)]
    rng = np.random.default_rng(3)
    for k in range(3):
        a = 1.0 + 0.1 * rng.normal()
        Q, e, g = (np.array([a, -a, 0.0]), 1 + 0.1 * rng.normal(size=3),
                   1 + 0.02 * rng.normal(size=3))
        par = [torch.tensor(t, device=device) for t in (Q, e, g)]
        if k == 2:
            par = [t.cpu() for t in par]
        F = model(pos, *par, step=k, m_samples=mt)
        ref.set_charges(Q[s.types])
        ref.set_lj(e, g)
        ref.force(k, *pos.t().contiguous().unbind(), *f, m_samples=mt, energy=True, sync=True)
        # (the reference adds energies: another kernel, the same force terms)
        assert rel_rms(F.double().cpu().numpy(), torch.stack(f, 1).double().cpu().numpy()) < 1e-6
        model.ctx.force(k, *pos.t().contiguous().unbind(), *f, m_samples=mt, energy=True,
                        sync=True)
        a, b = model.ctx.thermo(), ref.thermo()
        for q in ("e_vdwl", "e_coul", "e_kspace"):
            assert a[q] == pytest.approx(b[q], rel=1e-12)
    with pytest.raises(RbmdxError, match="which atoms are charged"):
        model(pos, par[0] + 0.5, par[1], par[2], step=0, m_samples=mt)
