"""The engine's host logic over a stand-in for the HIP runtime (host/hip_stub.cpp, built
here from the library's own sources): orders of launches and copies, and failures
half-way, without a GPU."""
import ctypes
import json
import os
import re
import subprocess

import numpy as np
import pytest

import rbmd_amd
from rbmd_amd import RbmdxError, build, systems

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host") / "libhost.so")
    src = [os.path.join(build.CSRC, f) for f in ("api.cpp", "batch.cpp", "sampler.cpp", "sog.cpp",
                                                 "data_api.cpp", "lammps_data.cpp", "output.cpp")]
    flags = ["-O0" if f == "-O2" else f for f in build.CXX_FLAGS]
    # -Bsymbolic: the stand-in, not the HIP runtime that torch has loaded
    subprocess.run(["g++", *flags, "-shared", "-Wl,-Bsymbolic", "-Wno-unused-result", "-o", out, *src,
                    os.path.join(HERE, "host", "hip_stub.cpp"), "-lpthread"], check=True)
    h = rbmd_amd.load_library(out)
    h.stub_log.restype = ctypes.c_char_p
    return h


@pytest.fixture
def stub(lib, monkeypatch):
    monkeypatch.setattr(rbmd_amd, "_lib", lib)
    lib.stub_counts(0)
    lib.stub_clear()

    class Stub:
        def log(self):
            out = lib.stub_log().decode().split("\n")[:-1]
            lib.stub_clear()
            return out

        fail = staticmethod(lambda name, after: lib.stub_fail(name.encode(), after))
        counts = staticmethod(lib.stub_counts)

    return Stub()


class _Row(np.ndarray):
    """A host array that the bindings take as a device tensor."""

    def data_ptr(self):
        return self.ctypes.data


def _rows(n, dtype=np.float32):
    return [np.zeros(n, dtype).view(_Row) for _ in range(3)]


def _ctx(n=600, **md):
    s = systems.electrolyte(n, seed=3)
    cfg = systems.ljsalt_config(P=8)
    if md:
        cfg["execution"] = md
    ctx = rbmd_amd.ForceContext(cfg, device=0)
    ctx.set_system(s.box_lo, s.box_len, s.types, s.ids, s.charges, s.eps, s.sigma)
    return s, ctx


A, B = 16, 32  # two streams


def _ordered(log, first, then):
    """Whether every `then` that follows a `first` has a wait in between."""
    pending = False
    for e in log:
        if e.startswith("sync"):
            pending = False
        elif e.startswith(then) and pending:
            return False
        if e.startswith(first):
            pending = True
    return True


def test_type_parameters_and_what_follows_them(stub):
    """The parameters set on a stream are in place before charges copied from the host,
    or parameters set on another stream."""
    s, ctx = _ctx()
    p = (np.array([1.1, -1.1, 0.0]), np.ones(3), np.ones(3))
    stub.log()
    ctx.set_type_params(*p, A)
    ctx.set_charges(1.2 * s.charges)
    assert _ordered(stub.log(), "type_params", "h2d")
    ctx.set_type_params(*p, A)
    ctx.set_lj(np.ones(3), np.ones(3))
    assert _ordered(stub.log(), "type_params", "h2d")
    ctx.set_type_params(*p, A)
    ctx.set_type_params(*p, B)
    log = stub.log()
    assert log.index("type_params s16") < log.index("sync") < log.index("type_params s32")
    # on one stream nothing waits
    ctx.set_type_params(*p, B)
    assert stub.log() == ["type_params s32"]


def test_type_parameters_are_checked(stub, lib):
    """One value per type; no system and no context are errors."""
    s, ctx = _ctx()
    for bad in ((s.charges, s.eps, s.sigma), ([1.0, -1.0], s.eps, s.sigma)):
        with pytest.raises(ValueError, match="one per type"):
            ctx.set_type_params(*bad, A)
    new = rbmd_amd.ForceContext(systems.ljsalt_config(P=8), device=0)
    with pytest.raises(RbmdxError, match="set_system first"):
        new.set_type_params([1.0, -1.0, 0.0], s.eps, s.sigma, A)
    h = ctypes.c_void_p()
    assert lib.rbmdx_create(b"{", 0, ctypes.byref(h)) != 0
    one = (ctypes.c_double * 1)(1.0)
    assert lib.rbmdx_set_type_params(h, one, one, one, None) != 0
    assert b"not created" in lib.rbmdx_last_error(h)
    lib.rbmdx_destroy(h)


@pytest.mark.parametrize("ensemble", ["NVT", "NVE"])
def test_md_run_that_fails_half_way(stub, ensemble):
    """A step that fails (its graph's launch) leaves the completed steps: their state is
    closed with its factor applied, step and thermostat agree, and a later run goes on."""
    md = dict(ensemble=ensemble, timestep=0.002, integration_type="vv")
    if ensemble == "NVT":
        md.update(temp_ctrl_type="NOSE_HOOVER", temperature=[1.0, 1.0, 0.1])
    s, ctx = _ctx(**md)
    ctx.set_masses(np.ones(3))
    x, v, f = _rows(s.n), _rows(s.n), _rows(s.n)
    ctx.md_init(x, v, f, stream=A)
    ctx.md_run(2, x, v, f, stream=A)
    st = ctx.md_state()
    assert (st["step"], st["temperature"]) == (2, 2.0)
    stub.log()
    stub.fail("hipGraphLaunch", 3)
    with pytest.raises(RbmdxError):
        ctx.md_run(5, x, v, f, stream=A)
    log = stub.log()
    assert log.count("md_thermostat s16") == 3 and log[-1] == "md_apply s16"
    st = ctx.md_state()
    assert (st["step"], st["temperature"]) == (5, 5.0)
    # before its first step: nothing done, nothing pending
    stub.log()
    stub.fail("hipGraphLaunch", 0)
    with pytest.raises(RbmdxError):
        ctx.md_run(5, x, v, f, stream=A)
    assert "md_apply s16" not in stub.log()
    ctx.md_run(2, x, v, f, stream=A)
    st = ctx.md_state()
    assert (st["step"], st["temperature"]) == (7, 7.0)
    # a state that cannot be closed is not taken for one
    stub.fail("hipGraphLaunch", 1)
    stub.fail("md_apply", 0)
    with pytest.raises(RbmdxError):
        ctx.md_run(5, x, v, f, stream=A)
    with pytest.raises(RbmdxError, match="md_init first"):
        ctx.md_run(1, x, v, f, stream=A)


def test_lists_that_cannot_grow(stub):
    """Lists that an evaluation outgrew are replaced by the next one; if that fails
    (allocation, or the capture after it), no later evaluation reads freed lists, and
    none reads new ones before they are built."""
    s, ctx = _ctx()
    x, f = _rows(s.n), _rows(s.n)
    stub.counts(100)
    ctx.force(0, *x, *f, stream=A)
    ctx.force(1, *x, *f, stream=A)
    stub.log()
    for k, call in enumerate(("hipMalloc", "hipGraphInstantiate", "hipGraphLaunch")):
        stub.counts(200 << k)
        ctx.force(2, *x, *f, stream=A)  # outgrown: the next call allocates
        stub.fail(call, 0)
        with pytest.raises(RbmdxError):
            ctx.force(3, *x, *f, stream=A)
        assert "force s16" not in stub.log()[2:]
        with pytest.raises(RbmdxError, match="no lists built yet|neighbour lists"):
            if call == "hipMalloc":
                ctx.force_noalloc(3, *x, *f, stream=A)
            else:
                ctx.export_candidates()
        for step in (4, 5):
            ctx.force(step, *x, *f, stream=A)
        log = stub.log()
        assert "force reads freed lists" not in log and log.count("rebuild") == 1
        assert log.index("rebuild") == log.index("force s16") + 1


@pytest.mark.parametrize("order", ["rows", "columns", "column of one", "one atom"])
def test_positions_changed_between_forward_and_backward(stub, monkeypatch, order):
    """The positions of the backward pass are the forward pass's in any memory order of
    the argument, also when the caller changes its array in between."""
    import torch

    from rbmd_amd import autograd

    for m in (rbmd_amd, autograd):
        monkeypatch.setattr(m, "_current_stream", lambda device: A)
    s = systems.electrolyte(600, frac_ion=0.05, seed=3)
    model = autograd.DifferentiableForce(systems.ljsalt_config(P=8), s)
    seen = []
    monkeypatch.setattr(model.ctx, "force_vjp", lambda step, *a, **k: (
        seen.extend(t.clone() for t in a[:3]), [t.zero_() for t in (*a[6:9], a[9])]))
    p = torch.tensor(s.pos.astype(np.float32))
    base, pos = {"rows": (p, p), "columns": (q := p.t().contiguous(), q.t()),
                 "column of one": (p, p.unsqueeze(2)), "one atom": (p, p[:1])}[order]
    want = pos.clone()
    par = [torch.tensor(a, requires_grad=True) for a in ([1.0, -1.0, 0.0], s.eps, s.sigma)]
    F = model(pos, *par)
    assert F.shape == pos.shape
    base += 1.0
    F.sum().backward()
    assert torch.equal(torch.stack(seen, 1), want)


def test_stored_launch_shapes_are_those_of_the_kernels(stub, tmp_path):
    """A shape stored for other kernels (a key without this version) is measured again;
    one stored for these is taken."""
    path = tmp_path / "tune.json"

    def tuned():
        b = rbmd_amd.BatchContext(systems.ljsalt_config(P=8), device=0)
        b.set_systems([systems.electrolyte(600, seed=3)])
        x, f = _rows(b.n), _rows(b.n)
        stub.log()
        out = b.autotune(0, *x, *f, m_samples=np.ones(24, np.int32).view(_Row),
                         cache_path=path, stream=A)
        return out, "batch s16" in stub.log()

    (_, us), measured = tuned()
    assert measured and us > 0
    (_, us), measured = tuned()
    assert not measured and us == 0
    entries = json.loads(path.read_text())
    (key, shape), = entries.items()
    other = re.sub(r"\|v\d+$", "", key)
    shape.update(pair_block=64, grid_per_cu=1)
    path.write_text(json.dumps({other: shape, re.sub(r"\|v\d+$", "|v1", key): shape}))
    (shape, us), measured = tuned()
    assert measured and us > 0 and shape["grid_per_cu"] > 1
    assert set(entries) < set(json.loads(path.read_text()))
