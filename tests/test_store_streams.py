"""The store's joined buffers are kept between calls: a call on one stream builds them, later calls
on any stream read them, with nothing that the caller could order."""
import numpy as np
import pytest


class _Stream:
    def __init__(self, log, name):
        self.log, self.name, self.cuda_stream = log, name, ord(name)

    def synchronize(self):
        self.log.append("synchronize " + self.name)


def test_joined_buffers_are_complete_before_they_are_kept(monkeypatch):
    """On host tensors with a recorded stream: both copies, then the stream's synchronisation, then
    the buffers are kept; a rebuild after an add goes the same way; a call on another stream builds
    nothing and marks the kept buffers as used there."""
    import torch
    from spi_amd import _lib, store as S
    log, used = [], []
    streams = {"now": _Stream(log, "a")}
    monkeypatch.setattr(_lib, "require_gpu", lambda: None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: streams["now"])
    cat = torch.cat
    monkeypatch.setattr(torch, "cat", lambda ts: (log.append("cat"), cat(ts))[1])
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda t, s: used.append((t.data_ptr(), s.name)), raising=False)

    class Store(S.SegmentStore):
        def __setattr__(self, name, value):
            if name == "_joined" and value is not None:
                log.append("kept")
            object.__setattr__(self, name, value)

    store = Store(device="cpu")
    for n_traj in (1, 2):
        store.add_arrays(np.ones((9, 37)), np.ones((9, 12)))
        del log[:]
        states, actions, first = store._joined_buffers()
        assert log == ["cat", "cat", "synchronize a", "kept"] and states.shape == (9 * n_traj, 37)
    assert not used
    streams["now"] = _Stream(log, "b")
    del log[:]
    assert store._joined_buffers()[0].data_ptr() == states.data_ptr() and not log
    assert {p for p, _ in used} >= {states.data_ptr(), actions.data_ptr()} and {n for _, n in used} == {"b"}


@pytest.mark.gpu
def test_second_stream_reads_the_finished_buffers(gpu):
    """First call on a stream with work queued before it, second call on another stream."""
    import torch
    from spi_amd.store import SegmentStore
    rng = np.random.default_rng(0)
    H, data = 7, [(rng.normal(size=(T, 37)).astype(np.float32), rng.normal(size=(T, 12)).astype(np.float32))
                  for T in (300, 41, 900)]
    store = SegmentStore()
    for s, a in data:
        store.add_arrays(s, a)
    one, two = torch.cuda.Stream(), torch.cuda.Stream()
    busy = torch.ones(1 << 26, device=gpu)
    torch.cuda.synchronize()
    with torch.cuda.stream(one):
        for _ in range(50):
            busy.mul_(1.0001)
        x = store.windows(H)
    with torch.cuda.stream(two):
        y = store.windows(H)
    torch.cuda.synchronize()
    want = [np.concatenate([s[t], np.concatenate([a[t:t + H], s[t + 1:t + H + 1]], 1).reshape(-1)])
            for s, a in data for t in range(len(s) - H)]
    assert np.array_equal(x.segments.cpu().numpy(), np.stack(want))
    assert np.array_equal(y.segments.cpu().numpy(), np.stack(want))
