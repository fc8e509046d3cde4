"""Forward dynamics by leg elimination (spi_fwd.h): the host build against the FP64 oracle over
random states in and out of contact, and the rollout kernels built on it at the edges of their
workgroups and horizons."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT, random_state

SRC = os.path.join(ROOT, "tests", "host_dyn", "spi_fwd_host.cpp")


def _build(tmp, double):
    out = str(tmp / ("fwd_d.so" if double else "fwd_f.so"))
    cmd = ["/opt/rocm/bin/hipcc", "--offload-host-only", "-O2", "-std=c++17", "-fPIC", "-shared", "-w",
           "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "spi-active_amd", "csrc"), SRC, "-o", out]
    if double:
        cmd.insert(1, "-DSPI_HOST_DOUBLE")
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        pytest.skip("hipcc host build unavailable: " + r.stderr[-300:])
    return C.CDLL(out)


# double: the simulation settings are floats and the contact and friction tanh a float expf (1e-7
# relative each, times the contact stiffness' share of the accelerations); float: 1e-7 per
# operation, amplified by the condition of the mass matrix (about 1e2) and a stiff contact.
@pytest.mark.parametrize("double,median,worst", [(True, 1e-6, 2e-5), (False, 2e-6, 2e-4)])
@pytest.mark.parametrize("height", [0.22, 0.26, 0.6])
def test_host_elimination_matches_oracle(tmp_path, model, sim, theta0, double, median, worst, height):
    import spio
    from spi_amd._lib import sim_args
    L, o, a = _build(tmp_path, double), spio.Oracle(model, sim), sim_args(sim)
    dp = C.POINTER(C.c_double)
    ptr = lambda x: x.ctypes.data_as(dp)
    rng = np.random.default_rng(int(100 * height))
    off = []
    for _ in range(100):
        par = theta0 * (1 + 0.2 * rng.normal(size=25))
        par[1:4] += 0.02 * rng.normal(size=3)
        s = random_state(rng, sim, height=height)
        s[25:37] = 4.0 * rng.normal(size=12)
        par, s = (np.asarray(x, np.float32).astype(np.float64) for x in (par, s))
        s[3:7] /= np.linalg.norm(s[3:7])
        tau = np.asarray(8.0 * rng.normal(size=12), np.float32).astype(np.float64)
        a0, qdd, force = o.forward(s[:13], s[13:25], s[25:37], tau, par)[:3]
        acc, ff = np.zeros(18), np.zeros(12)
        L.spi_host_forward_elim(C.byref(a), ptr(par), ptr(s), ptr(tau), ptr(acc), ptr(ff))
        want = np.concatenate([np.ravel(a0), np.ravel(qdd)])
        off.append(max(np.linalg.norm(acc - want) / np.linalg.norm(want),
                       np.linalg.norm(ff - np.ravel(force)) / max(np.linalg.norm(force), 1.0)))
    assert np.median(off) < median and np.max(off) < worst, (np.median(off), np.max(off))


@pytest.mark.gpu
@pytest.mark.parametrize("n,horizon", [(1, 1), (255, 2), (257, 1), (300, 60)])
def test_rollout_cost_at_edges(gpu, model, sim, theta0, n, horizon):
    """One lane per rollout at workgroup edges and a short and a long horizon: every cost against the
    record mode (which candidate and segment it belongs to; both inline the same step), and up to two
    steps a sample against the FP64 oracle (its value)."""
    import spio
    import torch
    from spi_amd.agents.sysid import identification_prior
    from spi_amd.data import synthetic_segments
    from spi_amd.params import params_soa
    from spi_amd.rollout import RolloutEngine
    eng = RolloutEngine(sim)
    segs = synthetic_segments(eng.simulate_np, theta0, sim, n_seg=3, horizon=horizon, seed=horizon)
    pr = identification_prior()
    rng = np.random.default_rng(n)
    rows = np.clip(pr.mean + 0.2 * pr.std * rng.normal(size=(n, 25)), pr.lo, pr.hi).astype(np.float32)
    got = eng.segment_costs(torch.from_numpy(params_soa(rows)).to(gpu), n, eng.upload_segments(segs), horizon,
                            physics="lanes").cpu().numpy()
    w = np.repeat(np.asarray(eng.weights, np.float32).astype(np.float64), [3, 4, 3, 3, 12, 12])
    for s in range(3):
        y = eng.simulate_np(rows, np.repeat(segs.init[s:s + 1], n, 0), np.repeat(segs.actions[s:s + 1], n, 0))
        want = (w * (y.astype(np.float64) - segs.targets[s]) ** 2).sum((1, 2))
        # both kernels inline the same step; contraction may differ (1e-6 of the state, which the
        # squared error at the noise floor turns into 1e-3 at most where nothing is chaotic)
        ok = np.abs(got[s] - want) <= 2e-3 * want + 1e-4
        assert ok.mean() > (0.99 if horizon <= 20 else 0.9), np.abs(got[s] / want - 1).max()
    if horizon <= 2:
        at = np.unique(np.clip([0, 1, n // 3, 63, n - 2, n - 1], 0, n - 1))
        ref = spio.Oracle(model, sim).rollout_cost(rows[at].astype(np.float64), segs.init, segs.actions, segs.targets, 0,
                                                   np.asarray(eng.cargs.w[:], np.float64))
        assert (np.abs(got[:, at].T - ref) <= 2e-3 * ref + 1e-4).all()
