"""The actor's layers on split products at the edges of their tiles: row counts around a tile, widths
that leave part of one, inputs of three magnitudes, of few non-zero values, of one sign and from either
end of the range, and non-finite inputs in every tile shape, dense and from a ring, against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _net(dims, seed):
    from spi_amd.agents.policy import PolicyMLP
    return PolicyMLP.random(dims[0], dims[-1], dims[1:-1], seed=seed)


def _f64(net, x):
    h = x.astype(np.float64)
    L = net.layers()
    for i, (W, b) in enumerate(L):
        h = h @ W.cpu().numpy().astype(np.float64).T + b.cpu().numpy().astype(np.float64)
        if i < len(L) - 1:
            h = np.where(h > 0, h, np.expm1(np.minimum(h, 0)))
    return h


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 200])
@pytest.mark.parametrize("dims", [(64, 64, 64), (900, 512, 12), (68, 65, 100), (100, 192, 64)])
@pytest.mark.parametrize("scale", [1e-3, 1.0, 1e4])
def test_split_layers_match_float64(gpu, rows, dims, scale):
    import torch
    net = _net(dims, rows)
    x = (scale * np.random.default_rng(rows).normal(size=(rows, dims[0]))).astype(np.float32)
    got = net(torch.from_numpy(x).to(gpu)).cpu().numpy()
    want = _f64(net, x)
    # two layers of at most 900 float32 accumulations of random sign: 1e-7 sqrt(900) of the scale
    assert np.abs(got - want).max() <= 5e-6 * np.abs(want).max()


def test_non_finite_inputs_stay_in_their_row(gpu):
    import torch
    net = _net((900, 512, 12), 3)
    x = np.random.default_rng(0).normal(size=(130, 900)).astype(np.float32)
    clean = net(torch.from_numpy(x).to(gpu)).cpu().numpy()
    bad = x.copy()
    bad[5, 7], bad[70, 899], bad[129, 0] = np.inf, np.nan, 3.4e38
    got = net(torch.from_numpy(bad).to(gpu)).cpu().numpy()
    keep = [i for i in range(130) if i not in (5, 70, 129)]
    assert np.array_equal(got[keep], clean[keep])
    assert np.isnan(got[70]).all() and not np.isfinite(got[5]).any()
    want = _f64(net, bad[129:])[0]                       # 1e37 per unit, 1e36 per output
    assert np.abs(want).max() < 3e38 and np.abs(got[129] - want).max() <= 5e-6 * np.abs(want).max()
    # one hidden layer of an infinite input: each unit is its weight's sign times infinity
    one = _net((64, 64), 1)
    y = np.zeros((1, 64), np.float32)
    y[0, 3] = np.inf
    W = one.layers()[0][0].cpu().numpy()
    assert np.array_equal(one(torch.from_numpy(y).to(gpu)).cpu().numpy()[0], np.sign(W[:, 3]) * np.inf)


def _one_layer(W):
    from spi_amd.agents.policy import PolicyMLP
    return PolicyMLP([(W, np.zeros(W.shape[0], np.float32))])


@pytest.mark.parametrize("non_zero", [1, 4])
def test_rows_of_few_inputs_round_like_float32(gpu, non_zero):
    """A sum of n float32 products is off by at most n roundings of 2^-24 of the products' magnitudes,
    and a single product by one."""
    import torch
    rng = np.random.default_rng(non_zero)
    W = rng.normal(size=(512, 900)).astype(np.float32)
    x = np.zeros((520, 900), np.float32)
    for row in x:
        row[rng.choice(900, non_zero, replace=False)] = rng.normal(size=non_zero)
    got = _one_layer(W)(torch.from_numpy(x).to(gpu)).cpu().numpy().astype(np.float64)
    x, W = x.astype(np.float64), W.astype(np.float64)
    assert (np.abs(got - x @ W.T) <= 1.02 * non_zero * 2.0 ** -24 * (np.abs(x) @ np.abs(W).T)).all()


def test_positive_sums_are_not_biased(gpu):
    """130 x 512 sums of 900 positive products: their mean relative error is far below a rounding."""
    import torch
    rng = np.random.default_rng(5)
    x, W = (np.abs(rng.normal(size=(n, 900))).astype(np.float32) for n in (130, 512))
    got = _one_layer(W)(torch.from_numpy(x).to(gpu)).cpu().numpy().astype(np.float64)
    assert abs((got / (x.astype(np.float64) @ W.astype(np.float64).T) - 1).mean()) < 2.0 ** -27


@pytest.mark.parametrize("scale_x,scale_w", [(1e-36, 1), (1, 1e-36), (1e-36, 1e30), (1e30, 1e-36), (1e-39, 1e30),
                                             (1e37, 1e-37), (1e18, 1e18), (1e25, 1e5)])
def test_magnitudes_over_the_whole_range(gpu, scale_x, scale_w):
    """64 products of operands near either end of float32: 64 roundings of 2^-24 would be 4e-6."""
    import torch
    rng = np.random.default_rng(9)
    x, W = (scale_x * rng.normal(size=(70, 64))).astype(np.float32), (scale_w * rng.normal(size=(64, 64))).astype(np.float32)
    got = _one_layer(W)(torch.from_numpy(x).to(gpu)).cpu().numpy().astype(np.float64)
    want = x.astype(np.float64) @ W.astype(np.float64).T
    assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)


def _times(f, n=7):
    import torch
    out = []
    for _ in range(n + 2):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        f()
        b.record()
        b.synchronize()
        out.append(a.elapsed_time(b))
    return min(out[2:])


def test_non_finite_rows_do_not_stall_the_batch(gpu):
    """Sixteen NaN rows among 2048: no more than a few times the clean batch."""
    import torch
    net = _net((900, 512, 256, 128, 12), 4)
    x = torch.randn((2048, 900), device=gpu)
    bad = x.clone()
    bad[:48:3, 5] = float("nan")
    assert _times(lambda: net(bad)) < 4 * _times(lambda: net(x))


# a tile shape each: two groups, one group, 128 columns (70 and 192: part of a tile)
@pytest.mark.parametrize("rows,width", [(130, 70), (6000, 192), (22000, 192)])
@pytest.mark.parametrize("ring", [None, 0, 1])
def test_non_finite_and_huge_operands_in_every_tile_shape(gpu, rows, width, ring):
    """inf, NaN and 3e38 in single rows against float64 (an infinite sum stays infinite, a NaN one
    NaN), dense and from a ring (lines aligned, and one row on); the rows between are as without them."""
    import torch
    rng = np.random.default_rng(rows)
    K = 68
    net = _one_layer(rng.normal(size=(width, K)).astype(np.float32))
    W = net.layers()[0][0].cpu().numpy().astype(np.float64)
    x = rng.normal(size=(rows, K)).astype(np.float32)
    bad = x.copy()
    at = {5: np.inf, 63: -np.inf, 64: np.nan, rows // 2: 3e38, rows - 1: np.inf}
    for i, (r, v) in enumerate(at.items()):
        bad[r, (7 * i) % K] = v

    def run(a):
        if ring is None:
            return net(torch.from_numpy(a).to(gpu)).cpu().numpy()
        buf = torch.zeros((3, K, rows + 2 + ring), device=gpu)     # the newest line holds the rows
        buf[1, :, ring:ring + rows] = torch.from_numpy(a.T.copy()).to(gpu)
        kmap = torch.stack([torch.zeros(K, dtype=torch.int32), torch.arange(K, dtype=torch.int32)], 1).to(gpu).contiguous()
        return net.forward_ring(buf, 1, kmap, 3.3e38, rows, row0=ring).cpu().numpy()

    clean, got = run(x), run(bad)
    assert np.array_equal(clean, net(torch.from_numpy(x).to(gpu)).cpu().numpy())   # ring and dense: the same bits
    keep = np.setdiff1d(np.arange(rows), list(at))
    assert np.array_equal(got[keep], clean[keep])
    if ring is not None:
        bad = np.where(np.isnan(bad), np.float32(-3.3e38), np.clip(bad, np.float32(-3.3e38), np.float32(3.3e38)))
    with np.errstate(all="ignore"):
        for r in at:
            want = (bad[r].astype(np.float64)[None] * W).sum(1).astype(np.float32)
            finite = np.isfinite(want)
            assert np.array_equal(np.isnan(want), np.isnan(got[r])) and np.array_equal(want[~finite], got[r][~finite], equal_nan=True)
            assert np.allclose(got[r][finite], want[finite], rtol=1e-5, atol=0)
    # 68 terms of about 1, 2e-6 of their sum's scale
    assert np.abs(clean - x.astype(np.float64) @ W.T).max() < 1e-4
