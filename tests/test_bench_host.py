"""Host side of bench.py (CPU only): the one-GPU refusal, the algorithmic
byte model's parts, and the profile lookups the bench line uses."""
import os
import subprocess
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)


def test_more_than_one_gpu_is_refused():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"),
                        "--gpus", "2"], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 2
    assert "one GPU" in r.stderr
    assert r.stdout == ""


def test_bytes_per_step_counts_each_array_once():
    import bench
    from axisem3d_amd import preloop
    sp = preloop.cartesian_homogeneous(
        nx=4, nz=4, width=4e3, depth=4e3, nsteps=5, src_depth=2e3,
        n_receivers=2, nodal_nr=lambda s, z: np.full(s.shape, 5.0))
    b = bench.bytes_per_step(sp, 4)
    nupd = sp.n_updates_per_step()
    # Fourier path only: no cardinal bytes; the point kernel reads the
    # element forces and reads and writes u, v, a (FP64) per point-mode
    assert b["cd_grad"] == b["cd_stress"] == b["cd_quad"] == 0
    assert b["point"] >= nupd * (6 * 4 + 6 * 48)
    assert b["fr"] > nupd * 48
    # a run marches u and w = v + dt/2 a, and writes v and a in its last step;
    # with absorbing boundaries, or in the symplectic scheme, it does not
    r = bench.bytes_per_step(sp, 4, run_steps=20)
    assert b["point"] - r["point"] == nupd * 2 * 48 - nupd * 2 * 48 // 20
    sp.time_scheme = "symplectic"
    assert bench.bytes_per_step(sp, 4, run_steps=20) == b
    sp.time_scheme = "newmark"
    sp._abc_abi = {"sponge_solid": {0: [1.0]}}
    assert bench.bytes_per_step(sp, 4, run_steps=20) == b


def test_the_timed_replays_are_replays():
    """Eight steps a graph: the run that captures is long enough for one
    whatever came before it (the first step may form w, the last writes v and
    a), and in the timed one all but the last step are replayed."""
    import bench
    assert bench.CAPTURE_RUN - 2 == bench.GRAPH_STEPS == 8
    for steps in (1, 7, 8, 9, 20, 60):
        n = bench.replay_run(steps)
        assert n > steps and (n - 1) % bench.GRAPH_STEPS == 0
        assert n - 1 < steps + bench.GRAPH_STEPS
        assert bench.bench_steps(steps, 5) == 5 + steps + bench.CAPTURE_RUN + n


def test_profile_lookups():
    import bench
    t = bench.pmc_traffic("k_cd_stress", "regional")
    assert t is None or t > 1e9
    v = bench.pmc_valu_busy("k_cd_stress", "regional")
    assert v is None or 0.0 < v <= 1.0
    assert bench.pmc_traffic("no_such_kernel", "regional") is None
