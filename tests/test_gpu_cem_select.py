"""Elite selection of the CEM update at its edges: one sample, every sample an elite, more elites
than the selection holds, ties across the threshold (few, and more than its list), NaN, infinities
and signed zeros, against numpy's stable order and float64 moments."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _costs(rng, n, kind):
    c = np.exp(rng.normal(size=n)).astype(np.float32)
    if kind == "ties":
        c = np.round(c * 4).astype(np.float32) / 4
    elif kind == "one value":
        c[:] = 1.5
    elif kind == "special":
        c -= 1.0
        c[rng.random(n) < 0.3] = np.inf
        c[rng.random(n) < 0.1] = np.nan
        c[rng.random(n) < 0.1] = -0.0
        c[rng.random(n) < 0.1] = 0.0
    elif kind == "mostly diverged":
        c[rng.random(n) < 0.97] = np.inf
    return c


@pytest.mark.parametrize("kind", ["smooth", "ties", "one value", "special", "mostly diverged"])
@pytest.mark.parametrize("n,elites", [(1, 1), (65, 65), (1000, 100), (4096, 410), (8192, 820), (8192, 1024), (8191, 1025),
                                      (64, 32), (65, 32), (128, 64), (128, 65), (2048, 1024), (2049, 1), (8192, 1)])
def test_selection_matches_numpy(gpu, n, elites, kind):
    import torch
    from spi_amd import _lib
    rng = np.random.default_rng(n + elites)
    c = _costs(rng, n, kind)
    theta = rng.normal(size=(25, n)).astype(np.float32)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    cost, th = d(c), d(theta)
    mean, std, best = (torch.zeros(25, device=gpu) for _ in range(3))
    min_std, best_cost = torch.zeros(25, device=gpu), torch.full((1,), float("inf"), device=gpu)
    idx = torch.full((elites,), -1, dtype=torch.int32, device=gpu)
    _lib.check(_lib.lib().spi_cem_update(_lib.ptr(cost), _lib.ptr(th), n, 25, n, elites, 0.0, _lib.ptr(min_std),
                                         _lib.ptr(mean), _lib.ptr(std), _lib.ptr(best), _lib.ptr(best_cost),
                                         _lib.ptr(idx, torch.int32), _lib.stream()), "spi_cem_update")
    key = np.where(np.isnan(c), np.inf, c)
    want = np.lexsort((np.arange(n), key))[:elites]
    assert np.array_equal(idx.cpu().numpy(), want)
    el = theta[:, want].astype(np.float64)
    # float32 sums of up to 1025 unit normals over 64 lanes: 17 terms a lane, 6 levels, 1e-7 each
    assert np.allclose(mean.cpu().numpy(), el.mean(1), atol=3e-6)
    assert np.allclose(std.cpu().numpy(), el.std(1), atol=3e-6)
    if np.isfinite(key[want[0]]):
        assert float(best_cost) == key[want[0]] and np.array_equal(best.cpu().numpy(), theta[:, want[0]])


def test_tied_costs_take_no_longer(gpu):
    """A population whose costs all tie (every rollout diverged) or mostly do, against distinct costs."""
    import torch
    from spi_amd.agents.cem import CEMConfig, DeviceCEM
    one = np.ones(22)

    def time(cost):
        cem = DeviceCEM(0 * one, one, -3 * one, 3 * one, 0.01 * one, CEMConfig(n_samples=4096))
        cem.ask()
        c = torch.from_numpy(cost).to(gpu)
        out = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                cem.tell(c)
            b.record()
            b.synchronize()
            out.append(a.elapsed_time(b))
        return min(out)

    smooth = time(_costs(np.random.default_rng(0), 4096, "smooth"))
    for kind in ("one value", "mostly diverged", "ties"):
        assert time(_costs(np.random.default_rng(0), 4096, kind)) < 2 * smooth
