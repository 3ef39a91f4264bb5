"""3D elements of small Nr in the one-kernel form of the cardinal path
(displacement to element forces with the strain series of all GLL points in
LDS) against the FP64 oracle: stage stiffness from a random state, twice, so
that the SLS memory enters the second, and seismograms of a short run with
the source inside such an element.

Domains: a spherical sector of three by two elements, axial ones among them,
with element Nr 1 to 5 (single butterflies, even and odd, orders that are
mean or Nyquist only), a ramp of small Nr with points of fewer orders than
their element, primes, and ramps over the Nr from which six elements take the
three kernels; all media, with no, CG4 and FULL attenuation of 5 and of 3
solids.  Larger ones: 48 elements at the largest Nr of either precision, a
sector in which the two forms run side by side, and one whose elements make
two launch groups.  Each asserts how many elements take the one-kernel form.

Tolerances as for the other element kernels: relative 1e-13 (FP64) and 1e-5
(FP32+FP64) per stage, 1e-12 and 1e-4 over the run."""
import numpy as np
import pytest

import oracle
from axisem3d_amd import preloop

pytestmark = pytest.mark.gpu
STEPS = 30


def _spec(nr0, nr1, mtype, att, nsls, ntheta=3, nrad=2):
    sp = preloop.spherical_regional(
        ntheta=ntheta, nrad=nrad, theta_max_deg=3.0, depth=100e3, nu_min=1, nu_max=1,
        nsteps=STEPS, attenuation=att is not None, cg4=att == "cg4",
        nsls=nsls, corr_len=40e3, bound_nr=False)
    s_max = 6371e3 * np.sin(np.radians(3.0))
    mesh = sp._mesh
    _, prof = preloop.layered_profile(11, 6371e3, 6271e3)
    field, a = sp._field, sp._att_in
    sp = preloop.build_domain(
        mesh, prof, lambda s, z: nr0 + (nr1 - nr0) * s / s_max, courant=0.5,
        lucky=nr1 > 7, bound_nr=False)
    sp._courant /= max(1.0, 0.4 * nr1)
    E = sp.n_solid_elements
    mt = {"iso": 0, "ti": 1, "aniso": 2}.get(mtype)
    types = np.arange(E) % 3 if mt is None else np.full(E, mt)
    preloop.make_media(sp, types.astype(np.uint8), field=field,
                       mask3d=np.ones(E, bool), att=a, seed=4)
    preloop.finish_regional(sp, STEPS, src_depth=30e3, f_peak=1.0,
                            n_receivers=3, theta_max_deg=3.0)
    return sp


def _fused(sp, prec):
    """How many elements should take the one-kernel form: up to Nr 168 (FP32)
    or 83 (FP64); of each medium, if there are larger ones in the domain, at
    least 256, and at least 48 if one of them has Nr 120 (58) or more."""
    top, big = {"fp32": (168, 120), "fp64": (83, 58)}[prec]
    nr = np.asarray(sp.elem_nr)
    n = 0
    for mt in range(3):
        q = nr[(np.asarray(sp.elem_mtype) == mt) & (nr <= top)]
        few = (nr > top).any() and len(q) < 256
        few |= len(q) < 48 and len(q) > 0 and q.max() >= big
        n += 0 if few else len(q)
    return n


def _rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


CASES = [(1, 1, "iso", None, 0), (2, 2, "mixed", "cg4", 5),
         (3, 3, "ti", "full", 3), (4, 4, "aniso", "cg4", 5),
         (5, 5, "mixed", "full", 5), (4, 16, "mixed", "cg4", 5),
         (9, 45, "mixed", "cg4", 3), (13, 13, "iso", None, 0),
         (60, 91, "mixed", "full", 5), (70, 90, "ti", "cg4", 5),
         (150, 190, "iso", "cg4", 5), (64, 64, "aniso", None, 0)]


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp32", 1e-5)])
@pytest.mark.parametrize("nr0,nr1,mtype,att,nsls", CASES)
def test_small_nr_matches_oracle(prec, tol, nr0, nr1, mtype, att, nsls):
    from axisem3d_amd.solver import GpuSolver
    sp = _spec(nr0, nr1, mtype, att, max(nsls, 1))
    o = oracle.Oracle(sp)
    g = GpuSolver(sp, prec)
    assert g.autotune_info()["fused_elements"] == _fused(sp, prec)
    assert (_fused(sp, prec) > 0) == (nr1 < (190 if prec == "fp32" else 64))
    rng = np.random.default_rng(21)
    for k in range(2):
        u = rng.standard_normal((o.nmodes, 3)) + 1j * rng.standard_normal(
            (o.nmodes, 3))
        g.set_field("displ", u)
        g.set_field("stiff", np.zeros_like(u))
        g.computeStiffness()
        e = _rel(g.get_field("stiff"), o.stiffness(u))
        print(f"Nr {nr0}..{nr1} {mtype} {att} {prec} pass {k}: {e:.2e}")
        assert e < tol
    g.close()
    o = oracle.Oracle(sp)
    ref = o.run(STEPS)
    g = GpuSolver(sp, prec)
    g.run(STEPS)
    es, eu = _rel(g.seismograms(), ref), _rel(g.get_field("displ"), o.displ)
    print(f"  run: seismograms {es:.2e}, field {eu:.2e}")
    assert np.abs(o.displ).max() > 0
    assert eu < (1e-12 if prec == "fp64" else 1e-4)
    if np.abs(ref).max() > 0:
        assert es < (1e-12 if prec == "fp64" else 1e-4)
    g.close()


# the form each element should take: the LDS holds Nr 168 in FP32 and 83 in
# FP64; from Nr 120 and 58 (112 KiB) fewer than 48 of a medium take the three
# kernels
@pytest.mark.parametrize("prec,nr,ntheta,nrad,fused", [
    ("fp32", 117, 3, 2, 6), ("fp32", 120, 3, 2, 0), ("fp32", 120, 47, 1, 0),
    ("fp32", 120, 8, 6, 48), ("fp32", 168, 8, 6, 48), ("fp32", 175, 8, 6, 0),
    ("fp64", 56, 3, 2, 6), ("fp64", 60, 3, 2, 0), ("fp64", 60, 47, 1, 0),
    ("fp64", 60, 8, 6, 48), ("fp64", 81, 8, 6, 48), ("fp64", 84, 8, 6, 0)])
def test_form_by_count_and_size(prec, nr, ntheta, nrad, fused):
    from axisem3d_amd.solver import GpuSolver
    # the largest Nr with the media and attenuation of most operands
    mtype, att, nsls = {168: ("aniso", "full", 5), 81: ("ti", "full", 3)}.get(
        nr, ("iso", "cg4", 5))
    sp = _spec(nr, nr, mtype, att, nsls, ntheta, nrad)
    assert set(sp.elem_nr.tolist()) == {nr}
    o = oracle.Oracle(sp)
    g = GpuSolver(sp, prec)
    assert g.autotune_info()["fused_elements"] == fused
    rng = np.random.default_rng(23)
    for k in range(2):
        u = rng.standard_normal((o.nmodes, 3)) + 1j * rng.standard_normal(
            (o.nmodes, 3))
        g.set_field("displ", u)
        g.set_field("stiff", np.zeros_like(u))
        g.computeStiffness()
        e = _rel(g.get_field("stiff"), o.stiffness(u))
        print(f"{sp.n_solid_elements} of Nr {nr} {prec} pass {k}: {e:.2e}")
        assert e < (1e-13 if prec == "fp64" else 1e-5)
    g.close()


def _stages(sp, prec, seed):
    """Two stages against the oracle; the launches of the one-kernel form."""
    from axisem3d_amd import capi
    from axisem3d_amd.solver import GpuSolver
    o = oracle.Oracle(sp)
    g = GpuSolver(sp, prec)
    fused = g.autotune_info()["fused_elements"]
    assert fused == _fused(sp, prec)
    g.profile(True)
    rng = np.random.default_rng(seed)
    for k in range(2):
        u = rng.standard_normal((o.nmodes, 3)) + 1j * rng.standard_normal(
            (o.nmodes, 3))
        g.set_field("displ", u)
        g.set_field("stiff", np.zeros_like(u))
        g.computeStiffness()
        e = _rel(g.get_field("stiff"), o.stiffness(u))
        print(f"{fused} of {sp.n_solid_elements} {prec} pass {k}: {e:.2e}")
        assert e < (1e-13 if prec == "fp64" else 1e-5)
    n = [g.profile_read(k)[1] for k in (capi.KERNEL_CD_FUSED,
                                        capi.KERNEL_CD_STRESS)]
    g.close()
    return fused, n[0] / 2, n[1] / 2


@pytest.mark.parametrize("prec,nr1", [("fp32", 200), ("fp64", 100)])
def test_two_forms_side_by_side(prec, nr1):
    sp = _spec(9, nr1, "ti", "cg4", 5, 33, 10)
    fused, one, three = _stages(sp, prec, 24)
    assert 256 <= fused < sp.n_solid_elements
    assert one == 1 and three >= 1


# groups of at least 512: the second begins where two of its elements fit the
# LDS of one of the first's largest
@pytest.mark.parametrize("prec,nr1", [("fp32", 120), ("fp64", 81)])
def test_two_launch_groups(prec, nr1):
    sp = _spec(8, nr1, "iso", None, 0, 75, 20)
    fused, one, three = _stages(sp, prec, 25)
    assert fused == sp.n_solid_elements
    assert one == 2 and three == 0
