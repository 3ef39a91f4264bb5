"""Blocks of the cardinal path's stress kernel, which take one to five GLL
points of an element: stage stiffness from a random state, twice (the SLS
memory enters the second), against the FP64 oracle.

The ranges of Nr are those in which a block takes five, four, three, two and
one points in either precision, each with odd Nr among them, so that the last
block of an element is short (25 = 12 x 2 + 1 = 8 x 3 + 1 = 6 x 4 + 1) and the
sixteen bytes a lane reads or writes end on a row's padding (in FP32 the
lowest range, 84 to 110, takes the one-kernel form; the others assert that
none does).

Tolerances as for the other element kernels: relative 1e-13 (FP64) and 1e-5
(FP32+FP64)."""
import numpy as np
import pytest

import oracle
from axisem3d_amd import preloop

pytestmark = pytest.mark.gpu


def _spec(nr0, nr1, mtype, att, nsls):
    sp = preloop.spherical_regional(
        ntheta=3, nrad=2, theta_max_deg=3.0, depth=100e3, nu_min=1, nu_max=1,
        nsteps=4, attenuation=att is not None, cg4=att == "cg4", nsls=nsls,
        corr_len=40e3, bound_nr=False)
    s_max = 6371e3 * np.sin(np.radians(3.0))
    mesh = sp._mesh
    _, prof = preloop.layered_profile(11, 6371e3, 6271e3)
    field, a = sp._field, sp._att_in
    sp = preloop.build_domain(
        mesh, prof, lambda s, z: nr0 + (nr1 - nr0) * s / s_max, courant=0.5,
        bound_nr=False)
    E = sp.n_solid_elements
    mt = {"iso": 0, "ti": 1, "aniso": 2}.get(mtype)
    types = np.arange(E) % 3 if mt is None else np.full(E, mt)
    preloop.make_media(sp, types.astype(np.uint8), field=field,
                       mask3d=np.ones(E, bool), att=a, seed=4)
    preloop.finish_regional(sp, 4, src_depth=30e3, f_peak=1.0,
                            n_receivers=3, theta_max_deg=3.0)
    return sp


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp32", 1e-5)])
@pytest.mark.parametrize("nr0,nr1,mtype,att,nsls", [
    (84, 110, "mixed", "cg4", 5), (115, 165, "ti", "full", 3),
    (169, 231, "mixed", "cg4", 5), (243, 330, "aniso", "full", 5),
    (351, 440, "iso", None, 0), (560, 810, "mixed", "cg4", 3),
    (900, 1000, "ti", "cg4", 5)])
def test_stress_blocks_match_oracle(prec, tol, nr0, nr1, mtype, att, nsls):
    from axisem3d_amd.solver import GpuSolver
    sp = _spec(nr0, nr1, mtype, att, max(nsls, 1))
    o = oracle.Oracle(sp)
    g = GpuSolver(sp, prec)
    one = prec == "fp32" and nr1 <= 110
    assert g.autotune_info()["fused_elements"] == (
        sp.n_solid_elements if one else 0)
    rng = np.random.default_rng(22)
    for k in range(2):
        u = rng.standard_normal((o.nmodes, 3)) + 1j * rng.standard_normal(
            (o.nmodes, 3))
        g.set_field("displ", u)
        g.set_field("stiff", np.zeros_like(u))
        g.computeStiffness()
        ref = o.stiffness(u)
        e = np.linalg.norm(g.get_field("stiff") - ref) / np.linalg.norm(ref)
        print(f"Nr {nr0}..{nr1} {mtype} {att} {prec} pass {k}: {e:.2e}")
        assert e < tol
    g.close()


@pytest.mark.parametrize("prec,nr", [
    ("fp32", 180), ("fp32", 231), ("fp32", 288), ("fp32", 375),
    ("fp32", 378), ("fp32", 525), ("fp32", 528), ("fp32", 810),
    ("fp64", 150), ("fp64", 189), ("fp64", 240), ("fp64", 405)])
def test_blocks_per_cu(prec, nr):
    """The points of a block leave LDS for five blocks of a CU (four in
    FP64), the kernel's own arrays included: as the runtime counts them, at Nr
    on either side of where a block takes one point less."""
    from axisem3d_amd.solver import GpuSolver
    sp = _spec(nr, nr, "iso", "cg4", 5)
    assert set(sp.elem_nr.tolist()) == {nr}
    g = GpuSolver(sp, prec)
    info = g.autotune_info()
    g.close()
    assert info["fused_elements"] == 0
    # of the chip's 256 CUs
    assert info["cardinal_blocks"] >= (5 if prec == "fp32" else 4) * 256
