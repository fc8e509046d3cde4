"""Window packing and command sequences where their kernels change path: groups across the end of
a trajectory, trajectories of one window, records longer than the staging, trajectories no longer
than the horizon; trials shorter and longer than a workgroup, odd command widths."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths,horizon", [((65, 64, 200), 1), ((21, 22, 40, 85, 21), 20), ((150, 129, 300), 128),
                                             ((400, 371), 320), ((30, 5, 90), 20), ((700,), 7)])
def test_store_windows_equal_the_rows(gpu, lengths, horizon):
    from spi_amd.store import SegmentStore
    rng = np.random.default_rng(sum(lengths))
    store, data = SegmentStore(), []
    for i, T in enumerate(lengths):
        s, a = rng.normal(size=(T, 37)).astype(np.float32), rng.normal(size=(T, 12)).astype(np.float32)
        store.add_arrays(s, a, kp=20.0 + i, kd=0.5 + i)
        data.append((s, a))
    for which in (None, list(range(len(lengths)))[::-1]):
        b = store.windows(horizon, which)
        want, src, start, ends = [], [], [], []
        for i in (range(len(lengths)) if which is None else which):
            s, a = data[i]
            for t in range(len(s) - horizon):
                rec = np.concatenate([a[t:t + horizon], s[t + 1:t + horizon + 1]], 1).reshape(-1)
                want.append(np.concatenate([s[t], rec]))
                src.append(i)
                start.append(t)
                ends.append(t == len(s) - horizon - 1)
        assert np.array_equal(b.segments.cpu().numpy(), np.stack(want))
        assert np.array_equal(b.source, src) and np.array_equal(b.start, start) and np.array_equal(b.motion_ends, ends)
        assert np.array_equal(b.kp, 20.0 + np.array(src)) and np.array_equal(b.kd, np.float32(0.5) + np.array(src))


@pytest.mark.parametrize("horizon", [1, 4, 5, 20, 21, 330])     # 20: the longest short record
@pytest.mark.parametrize("n", [1, 2, 3, 65, 130])
@pytest.mark.parametrize("order", ["run", "random", "reversed"])
def test_row_tables_equal_the_rows(gpu, horizon, n, order):
    """Windows of any rows, rows outside the buffer (NaN records) among them."""
    import torch
    from spi_amd import _lib
    rng = np.random.default_rng(horizon + n)
    R = 500
    s, a = rng.normal(size=(R, 37)).astype(np.float32), rng.normal(size=(R, 12)).astype(np.float32)
    rows = {"run": 7 + np.arange(n), "random": rng.integers(-3, R, n), "reversed": R - 1 - np.arange(n)}[order].astype(np.int32)
    d = lambda x: torch.from_numpy(x).to(gpu)
    sd, ad, rd = d(s), d(a), d(rows)
    out = torch.empty((n, 37 + 49 * horizon), device=gpu)
    _lib.check(_lib.lib().spi_pack_windows_rows(_lib.ptr(sd), _lib.ptr(ad), R, _lib.ptr(rd, torch.int32), n, horizon,
                                                _lib.ptr(out), _lib.stream()), "spi_pack_windows_rows")
    out = out.cpu().numpy()
    for w, r in enumerate(rows):
        if r < 0 or r + horizon >= R:
            assert np.isnan(out[w]).all()
        else:
            rec = np.concatenate([a[r:r + horizon], s[r + 1:r + horizon + 1]], 1).reshape(-1)
            assert np.array_equal(out[w], np.concatenate([s[r], rec]))


def test_short_records_of_scattered_rows_take_no_longer(gpu):
    """Rows in any order read element by element: one-step records within a few times consecutive rows'."""
    import torch
    from spi_amd import _lib
    R, n = 20000, 5000
    s, a, out = torch.randn((R, 37), device=gpu), torch.randn((R, 12), device=gpu), torch.empty((n, 86), device=gpu)

    def time(rows):
        rd, best = torch.from_numpy(rows.astype(np.int32)).to(gpu), []
        for _ in range(9):
            t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            t0.record()
            for _ in range(20):
                _lib.check(_lib.lib().spi_pack_windows_rows(_lib.ptr(s), _lib.ptr(a), R, _lib.ptr(rd, torch.int32), n, 1,
                                                            _lib.ptr(out), _lib.stream()), "spi_pack_windows_rows")
            t1.record()
            t1.synchronize()
            best.append(t0.elapsed_time(t1))
        return min(best)

    assert time(np.arange(n)[::-1]) < 1.7 * time(np.arange(n))


@pytest.mark.parametrize("mode", ["constant", "polynomial", "bezier"])
@pytest.mark.parametrize("trials,steps,width", [(1, 38, 14), (33, 39, 13), (5, 51, 14), (1, 52, 13), (2100, 50, 13), (3, 250, 11),
                                                (2100, 53, 14), (40, 76, 13), (40, 77, 13), (9, 125, 11)])
def test_command_sequences_at_edges(gpu, mode, trials, steps, width):
    import torch
    import spio_commands as oc
    from spi_amd.agents.commands import CommandGenerator
    from test_commands_oracle import DEFAULT, IDX, RANGES
    gen = CommandGenerator(RANGES[:width], DEFAULT[:width], IDX, mode, rollout_length=5.0, horizon_length=1.0,
                           dt=1.0 / steps)
    U, S = gen.n_updates, gen.steps
    rng = np.random.default_rng(trials)
    b = gen.param_bounds()
    P = rng.uniform(b[:, 0], b[:, 1], size=(trials, b.shape[0])).astype(np.float32)
    out = gen.generate(torch.from_numpy(P)).cpu().numpy()
    for k in sorted({0, trials // 2, trials - 1}):
        ref = oc.commands_from_params(P[k], mode, RANGES[:width], DEFAULT[:width], IDX, U, S)
        assert np.abs(out[k] - ref).max() < 2e-6


def test_command_time_is_even_over_the_steps(gpu):
    """A few steps past 256 do not cost a second workgroup per trial."""
    import torch
    from spi_amd.agents.commands import CommandGenerator
    from test_commands_oracle import DEFAULT, IDX, RANGES

    def time(steps):
        gen = CommandGenerator(RANGES, DEFAULT, IDX, "polynomial", rollout_length=5.0, horizon_length=1.0, dt=1.0 / steps)
        p = torch.rand((4096, len(gen.param_names())), device=gpu)
        out = []
        for _ in range(9):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                gen.generate(p)
            b.record()
            b.synchronize()
            out.append(a.elapsed_time(b))
        return min(out)

    assert time(53) < 1.35 * time(51)
