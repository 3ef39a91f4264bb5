"""The forms a run's steps take: within a run the march is that of w = v +
dt/2 a, whose field the first step forms from (v, a) unless the last run left
it, and from which the last step writes (v, a); the steps between are replayed
several to a graph.  A run of n steps equals n runs of one step bit by bit,
for n around the lengths where the form or the graph changes, on a solid with
receivers of few and of several hundred orders and on a fluid layer with 3D
coupling and 3D masses (points marched by other kernels).  Where the program
sets the velocity and the acceleration in between, w follows them: the run
equals that of a solver that starts from those fields.  And w is what the
velocity and the acceleration give: a run that goes on from fields read from a
solver, in another or set again in the same, is the unbroken run bit by bit.
Receivers ride on the step's first element launch, or, where that launch has
large blocks and they are many, take one of their own."""
import math

import numpy as np
import pytest

from axisem3d_amd import preloop

pytestmark = pytest.mark.gpu


def _solid(nsteps):
    sp = preloop.spherical_regional(
        ntheta=4, nrad=3, theta_max_deg=6.0, depth=300e3, nu_min=5,
        nu_max=410, nsteps=nsteps, attenuation=False, corr_len=100e3,
        bound_nr=False)
    sp._courant /= 60.0
    sp._build_3d((np.arange(sp.n_solid_elements) % 3) == 0)
    preloop.finish_regional(sp, nsteps, src_depth=50e3, f_peak=1.0,
                            n_receivers=5, theta_max_deg=6.0)
    return sp


def _fluid(nsteps):
    mesh = preloop.StructuredMesh(np.linspace(0, 4e3, 5),
                                  np.linspace(0, 6e3, 7))

    def mat(r, rc):
        inl = (rc > 2e3) & (rc < 4e3)
        one = np.ones_like(r)
        return (np.where(inl, 1000.0, 2600.0) * one,
                np.where(inl, 1500.0, 6000.0) * one,
                np.where(inl, 0.0, 3464.0) * one)
    sp = preloop.build_domain(
        mesh, mat, lambda s, z: 3.0 + 8.0 * (s / 4e3) + 0.0 * z, courant=0.4)
    _, iz = mesh.element_ix_iz()
    zc = (iz + 0.5) * 1e3
    preloop.make_fluid(sp, (zc > 2e3) & (zc < 4e3))
    preloop.make_mass3d(sp, np.arange(0, sp.n_solid_points, 3), seed=3)
    preloop.make_fluid_mass3d(sp, np.arange(0, len(sp.fluid_nr), 4), seed=4)
    preloop.make_coupling3d(sp, np.arange(0, len(sp.sf_solid), 2), seed=5)
    mt = np.array([1.0, 0.7, 0.4, 0.3, 0.2, 0.1]) * 1e15
    preloop.add_axial_moment_source(sp, 1e3, mt, 1.628 / (2 * math.pi),
                                    1.628, nsteps)
    preloop.add_receivers(sp, np.array([0.5e3, 2e3]), np.array([5.5e3, 1.5e3]),
                          np.array([0.3, 1.1]))
    return sp


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("case", ["solid", "fluid"])
@pytest.mark.parametrize("n", [2, 3, 9, 10, 11, 27])
def test_run_equals_single_steps(case, prec, n):
    from axisem3d_amd.solver import GpuSolver
    spec = (_solid if case == "solid" else _fluid)(n)
    fields = ["displ", "veloc", "accel"]
    if case == "fluid":
        fields += ["fdispl", "fveloc", "faccel"]
    a, b, c = (GpuSolver(spec, prec) for _ in range(3))
    rng = np.random.default_rng(7)

    def state():
        out = {}
        for f in fields:
            x = a.get_field(f)
            x = rng.standard_normal(x.shape) + \
                1j * rng.standard_normal(x.shape)
            out[f] = x * {"d": 1.0, "v": 1.0 / spec.dt,
                          "a": 1.0 / spec.dt ** 2}[f.lstrip("f")[0]] * 1e-3
        return out

    start, later = state(), state()
    for f in fields:
        a.set_field(f, start[f])
        b.set_field(f, start[f])
    a.run(n)
    for _ in range(n):
        b.run(1)
    for f in fields:
        assert np.array_equal(a.get_field(f), b.get_field(f)), f
    s, t = a.seismograms(), b.seismograms()
    assert np.abs(t).max() > 0 and np.array_equal(s, t)
    # other velocities and accelerations: what w was no longer holds
    a.step = 0
    for f in fields:
        later[f] = a.get_field(f) if f.endswith("displ") else later[f]
        c.set_field(f, later[f])
        if not f.endswith("displ"):
            a.set_field(f, later[f])
    a.run(n)
    c.run(n)
    for f in fields:
        assert np.array_equal(a.get_field(f), c.get_field(f)), f
    for g in (a, b, c):
        g.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("case", ["solid", "fluid"])
@pytest.mark.parametrize("n", [1, 12])
def test_run_from_saved_fields_equals_unbroken_run(case, prec, n):
    from axisem3d_amd.solver import GpuSolver
    m = 14
    spec = (_solid if case == "solid" else _fluid)(n + m)
    fields = ["displ", "veloc", "accel"]
    if case == "fluid":
        fields += ["fdispl", "fveloc", "faccel"]
    a, b, c = (GpuSolver(spec, prec) for _ in range(3))
    rng = np.random.default_rng(8)
    for f in fields:
        x = a.get_field(f)
        x = rng.standard_normal(x.shape) + 1j * rng.standard_normal(x.shape)
        x *= {"d": 1.0, "v": 1.0 / spec.dt,
              "a": 1.0 / spec.dt ** 2}[f.lstrip("f")[0]] * 1e-3
        a.set_field(f, x)
        b.set_field(f, x)
    a.run(n + m)
    b.run(n)
    for f in fields:
        x = b.get_field(f)
        b.set_field(f, x)
        c.set_field(f, x)
    c.step = n
    b.run(m)
    c.run(m)
    for g in (b, c):
        for f in fields:
            assert np.array_equal(a.get_field(f), g.get_field(f)), f
        s = a.seismograms()[n:]
        assert np.abs(s).max() > 0
        assert np.array_equal(s, g.seismograms()[n:])
    for g in (a, b, c):
        g.close()


# one-kernel form: at most 512 x 1024 threads of receivers' blocks ride.  Nr
# 90: 1024 threads in FP32; Nr 50: 512 in FP64; Nr 9: 128
@pytest.mark.parametrize("prec,nr,nrec,own", [
    ("fp32", 90, 512, False), ("fp32", 90, 513, True),
    ("fp64", 50, 1024, False), ("fp64", 50, 1025, True),
    ("fp32", 9, 1500, False)])
def test_many_receivers(prec, nr, nrec, own):
    from axisem3d_amd import capi
    from axisem3d_amd.solver import GpuSolver
    n = 12
    mesh = preloop.StructuredMesh(np.linspace(0, 4e3, 4),
                                  np.linspace(0, 3e3, 4))
    _, prof = preloop.layered_profile(3, 3e3, 0.)
    sp = preloop.build_domain(mesh, prof, lambda s, z: nr + 0. * s,
                              courant=0.4 / nr, bound_nr=False)
    field = preloop.RandomField(5, corr_len=3e3)
    preloop.make_3d_isotropic(sp, field, None,
                              np.ones(sp.n_solid_elements, bool))
    mt = np.array([1.0, 0.7, 0.4, 0.3, 0.2, 0.1]) * 1e15
    preloop.add_axial_moment_source(sp, 1.7e3, mt, 3 * sp.dt, 1.628, n)
    s = 4e3 * (np.arange(nrec) + 0.5) / nrec
    phi = np.linspace(0.0, 6.0, nrec)
    preloop.add_receivers(sp, s, np.full(nrec, 3e3), phi)
    g = GpuSolver(sp, prec)
    assert g.autotune_info()["fused_elements"] == sp.n_solid_elements
    g.profile(True)
    g.run(n)
    assert (g.profile_read(capi.KERNEL_RECORD)[1] > 0) == own
    sel = np.r_[0:20, nrec // 2, nrec - 20:nrec]
    preloop.add_receivers(sp, s[sel], np.full(len(sel), 3e3), phi[sel])
    few = GpuSolver(sp, prec)
    few.run(n)
    a, b = g.seismograms()[:, sel], few.seismograms()
    # the same field; a receiver's sum of 25 points and up to 46 orders in
    # another order
    assert np.abs(b).max() > 0
    assert np.abs(a - b).max() < 25 * 46 * 2.3e-16 * np.abs(
        few.get_field("displ")).max()
    for x in (g, few):
        x.close()
