"""Set means and log-determinants over Fisher matrices at the edges of their kernel: sets around the
16 groups loaded ahead and the strides of the count, matrices around the workgroup sizes, invalid
groups (NaN inside) at the ends of batches and in the tail, sets with none valid, indefinite matrices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [1, 4, 8, 9, 16, 17, 22, 32])
@pytest.mark.parametrize("size", [1, 15, 16, 17, 33, 600])
def test_set_means_and_logdets(gpu, P, size):
    import torch
    from spi_amd import _lib
    rng = np.random.default_rng(100 * P + size)
    n_sets, reg = 7, 1e-6
    A = rng.normal(size=(n_sets, size, P, P + 3))
    F = (A @ A.transpose(0, 1, 3, 2)).astype(np.float32)
    status = np.zeros((n_sets, size), np.int32)
    for s, bad in enumerate(([], [0], [15, 16], [size - 1], list(range(0, size, 2)), list(range(size)), [])):
        status[s, [k for k in bad if k < size]] = 1
    F[status != 0] = np.nan
    F[6, :, 0, 0] *= -1.0                                   # a negative first pivot
    scale = np.exp(rng.normal(size=P))
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    Fd, st, sc = d(F), d(status), d(scale)
    mean = torch.empty((n_sets, P, P), dtype=torch.float64, device=gpu)
    ld = torch.empty(n_sets, dtype=torch.float64, device=gpu)
    nv = torch.empty(n_sets, dtype=torch.int32, device=gpu)
    _lib.check(_lib.lib().spi_fim_logdet(_lib.ptr(Fd), _lib.ptr(st, torch.int32), n_sets, size, P,
                                         _lib.ptr(sc, torch.float64), reg, _lib.ptr(mean, torch.float64),
                                         _lib.ptr(ld, torch.float64), _lib.ptr(nv, torch.int32), _lib.stream()), "logdet")
    mean, ld, nv = mean.cpu().numpy(), ld.cpu().numpy(), nv.cpu().numpy()
    for s in range(n_sets):
        ok = status[s] == 0
        assert nv[s] == ok.sum()
        want = (F[s, ok].astype(np.float64).sum(0) / ok.sum() if ok.any() else np.zeros((P, P))) * np.outer(scale, scale)
        want = want + reg * max(np.trace(want), 0.0) / P * np.eye(P)
        # float64 sums of up to 600 terms: 600 roundings of 1e-16 of the largest
        assert np.abs(mean[s] - want).max() <= 1e-12 * max(np.abs(want).max(), 1e-300)
        if not ok.any() or s == 6:
            assert ld[s] == -np.inf
        else:
            sign, ref = np.linalg.slogdet(want)
            # the ridge bounds the condition at P / 1e-6: 1e-16 * 3e7 per eigenvalue
            assert sign > 0 and abs(ld[s] - ref) <= 1e-7 * P
