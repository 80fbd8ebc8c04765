"""The projections on int8 digits (linear_tile 64) against the f64 contract.

Sizes sit at the edges of the form: one row and column, either side of its 64 x 64 tiles and
32-row blocks, one K stage, K in one, two and four register groups and beyond them. Values sit
at the edges of the digits: weights in three digits (below 0.498), in four (up to 127) and
past them, rows whose elements span more binades than the six digits, rows with infinities
and NaN. Products whose operands the digits hold exactly must give the f64 sum rounded once:
at most 1 ulp (two f64 sums may straddle a rounding boundary) on a handful of elements, as
test_gpu_model_ops.py asks of the f64 kernels.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = np.float32(1e-6)


def _ulps(a, b):
    # signed-magnitude order, so that -0.0 and 0.0 are neighbours of the smallest values
    def key(x):
        i = x.astype(np.float32).view(np.int32).astype(np.int64)
        return np.where(i < 0, -(i & 0x7FFFFFFF), i)
    return np.abs(key(a) - key(b))


def _check(got, want):
    d = _ulps(got, want)
    assert d.max() <= 1, f"{d.max()} ulps"
    assert int((d > 0).sum()) <= max(2, got.size // 20000)


def _h(x, nw):
    if nw is None:
        return x.astype(np.float64)
    x64 = x.astype(np.float64)
    scale = 1.0 / np.sqrt((x64 * x64).mean(axis=1, keepdims=True) + np.float64(EPS))
    return ((x64 * scale).astype(np.float32) * nw).astype(np.float64)


def _run(gpu, dev, x, w, nw=None, resid=None, w_up=None):
    out = torch.full((x.shape[0], w.shape[0]), np.nan, dtype=torch.float32, device=dev)
    t = [None if a is None else torch.from_numpy(a).to(dev) for a in (x, w, nw, resid, w_up)]
    if w_up is not None:
        gpu.linear_swiglu_f64acc(t[0], t[1], t[4], out, norm_w=t[2], eps=float(EPS))
    else:
        gpu.linear_f64acc(t[0], t[1], out, norm_w=t[2], eps=float(EPS), resid=t[3])
    return out.cpu().numpy()


@pytest.mark.parametrize("rows,n_out,k_in", [(1, 1, 64), (31, 33, 128), (64, 64, 64),
                                             (65, 127, 512), (130, 200, 576), (96, 40, 1088),
                                             (33, 65, 2048), (40, 130, 2112)])
@pytest.mark.parametrize("norm", [False, True])
def test_shapes(gpu, dev, tune, rows, n_out, k_in, norm):
    tune(linear_tile=64)
    rng = np.random.default_rng(rows + n_out + k_in)
    x = rng.standard_normal((rows, k_in), dtype=np.float32)
    w = (rng.standard_normal((n_out, k_in)) * 0.02).astype(np.float16)
    nw = (1 + 0.1 * rng.standard_normal(k_in)).astype(np.float32) if norm else None
    want = (_h(x, nw) @ w.astype(np.float64).T).astype(np.float32)
    got = _run(gpu, dev, x, w, nw)
    _check(got, want)
    assert np.array_equal(got, _run(gpu, dev, x, w, nw)), "not deterministic"
    r = rng.standard_normal((rows, n_out), dtype=np.float32)
    assert np.array_equal(_run(gpu, dev, x, w, nw, resid=r), r + got)


@pytest.mark.parametrize("rows,hidden,k_in", [(1, 1, 64), (33, 17, 128), (70, 100, 704)])
def test_swiglu(gpu, dev, tune, rows, hidden, k_in):
    tune(linear_tile=64)
    rng = np.random.default_rng(hidden)
    x = rng.standard_normal((rows, k_in), dtype=np.float32)
    wg, wu = ((rng.standard_normal((hidden, k_in)) * 0.05).astype(np.float16) for _ in range(2))
    nw = np.ones(k_in, np.float32)
    h = _h(x, nw)
    g, u = ((h @ w.astype(np.float64).T).astype(np.float32) for w in (wg, wu))
    want = (g / (np.float32(1.0) + np.exp(-g))) * u
    got = _run(gpu, dev, x, wg, nw, w_up=wu)
    # exp may differ by an ulp between libraries: a few ulps of the product at most
    assert np.all(np.abs(got - want) <= 8 * 2.0 ** -24 * np.abs(want) + 1e-30)


@pytest.mark.parametrize("scale", [0.45, 0.5, 30.0, 127.0, 128.0, 60000.0])
def test_weight_ranges(gpu, dev, tune, scale):
    """Weights up to each digit count's limit and past it (f64 sums there), with fp16
    subnormals among them, in one column block; the other block keeps three digits."""
    tune(linear_tile=64)
    rng = np.random.default_rng(int(scale * 10))
    x = rng.standard_normal((40, 192), dtype=np.float32)
    w = (rng.standard_normal((64, 192)) * 0.02).astype(np.float16)
    w[:32] = (rng.uniform(-1, 1, (32, 192)) * scale).astype(np.float16)
    w[3, :] = np.float16(scale)
    w[5, ::2] = np.float16(2.0 ** -24)
    w[6, ::3] = -np.float16(scale)
    _check(_run(gpu, dev, x, w), (x.astype(np.float64) @ w.astype(np.float64).T).astype(np.float32))


@pytest.mark.parametrize("spread", [1.0, 2.0 ** 10, 2.0 ** 15, 2.0 ** 21, 2.0 ** 40])
def test_rows_with_outliers(gpu, dev, tune, spread):
    """One element `spread` times the others: the digits hold every bit up to a spread of 2^22
    (the last one of them past 2^14); past it every other element is rounded and the row's
    block takes f64 sums."""
    tune(linear_tile=64)
    rng = np.random.default_rng(11)
    x = rng.uniform(0.5, 1.0, (64, 256)).astype(np.float32)
    x[::5, 17] *= np.float32(spread)
    w = (rng.standard_normal((48, 256)) * 0.02).astype(np.float16)
    w[::2, 17] = 0  # columns that do not see the outlier keep the others' bits
    _check(_run(gpu, dev, x, w), (x.astype(np.float64) @ w.astype(np.float64).T).astype(np.float32))


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan, 3e38, 1e-38])
def test_unusual_rows(gpu, dev, tune, bad):
    """Rows outside the digits' range give what f64 sums give, and leave the other rows' bits
    alone (a block of 32 rows takes f64 sums together, in another order: 1 ulp)."""
    tune(linear_tile=64)
    rng = np.random.default_rng(13)
    x = rng.standard_normal((70, 128), dtype=np.float32)
    w = (rng.standard_normal((64, 128)) * 0.02).astype(np.float16)
    x[5] *= 0 if abs(bad) < 1 else 1
    x[5, 40] = bad
    x[6] = 0
    got = _run(gpu, dev, x, w)
    with np.errstate(invalid="ignore", over="ignore"):
        want = (x.astype(np.float64) @ w.astype(np.float64).T).astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    fine = np.isfinite(want)
    assert np.array_equal(got[~fine & ~np.isnan(want)], want[~fine & ~np.isnan(want)])
    d = _ulps(got[fine], want[fine])
    assert d.max() <= 1
    assert np.array_equal(got[32:64], _run(gpu, dev, x[32:64], w)), "another block changed"


@pytest.mark.parametrize("spread,others", [(2.0 ** 47, 255), (2.0 ** 60, 255), (2.0 ** 100, 255),
                                           (2.0 ** 40, 10), (2.0 ** 60, 1)])
def test_outliers_out_of_sight(gpu, dev, tune, spread, others):
    """Elements below the last digit of their row's largest, all of them or the few that are not
    zero: columns that do not see the largest get the others' f64 sums."""
    tune(linear_tile=64)
    rng = np.random.default_rng(17)
    x = np.zeros((64, 256), np.float32)
    x[:, :others] = rng.uniform(0.5, 1.0, (64, others)) * 2.0 ** -41
    x[:, 255] = spread * 2.0 ** -41
    w = (rng.standard_normal((48, 256)) * 0.02).astype(np.float16)
    w[::2, 255] = 0
    _check(_run(gpu, dev, x, w), (x.astype(np.float64) @ w.astype(np.float64).T).astype(np.float32))


@pytest.mark.parametrize("size,weight", [(1e-38, 1e-8), (1e-37, 2e-6), (0.0, 1.0)])
def test_norm_lifts_products_out_of_the_subnormals(gpu, dev, tune, size, weight):
    """x * norm_w is zero or subnormal, the normalised row is not."""
    tune(linear_tile=64)
    rng = np.random.default_rng(19)
    x = (rng.uniform(0.5, 1.0, (40, 128)) * size).astype(np.float32)
    nw = np.full(128, weight, np.float32)
    w = (rng.uniform(50, 100, (40, 128))).astype(np.float16)
    want = (_h(x, nw) @ w.astype(np.float64).T).astype(np.float32)
    assert (size == 0.0) == (not want.any())
    _check(_run(gpu, dev, x, w, nw), want)


@pytest.mark.parametrize("small", [2.0 ** -20, 1e-8, 1e-10, 1e-12, 1e-14, 1e-30])
@pytest.mark.parametrize("count", [1, 2, 5, 16, 17, 40])
@pytest.mark.parametrize("norm", [False, True])
def test_columns_that_see_only_small_elements(gpu, dev, tune, small, count, norm):
    """`count` elements of a row far below its largest (what the digits round off, listed up to
    16 a row, f64 sums past that), and columns whose weights are nonzero only there, one-hot
    columns among them: the f64 sum, rounded once."""
    tune(linear_tile=64)
    rng = np.random.default_rng(count)
    rows, k_in = 70, 768
    x = rng.standard_normal((rows, k_in), dtype=np.float32)
    x[::3] = np.abs(x[::3]) + 0.5  # rows without small elements of their own
    w = (rng.standard_normal((96, k_in)) * 0.02).astype(np.float16)
    at = rng.choice(k_in, count, replace=False)
    x[1:, at] = (rng.uniform(0.5, 1.0, (rows - 1, count)) * small).astype(np.float32)
    x[2:, at[0]] *= -1
    keep = w[:40, at].copy()
    w[:40] = 0
    w[:40, at] = keep
    w[40:50] = 0
    w[np.arange(40, 50), at[np.arange(10) % count]] = 1
    nw = (1 + 0.1 * rng.standard_normal(k_in)).astype(np.float32) if norm else None
    want = (_h(x, nw) @ w.astype(np.float64).T).astype(np.float32)
    got = _run(gpu, dev, x, w, nw)
    _check(got, want)
    assert np.array_equal(got, _run(gpu, dev, x, w, nw)), "not deterministic"


@pytest.mark.parametrize("eps", [0.0, 1e-6])
def test_zero_rows_under_the_norm(gpu, dev, tune, eps):
    """A zero row normalised with eps = 0 is 0 times infinity, NaN as in the f64 forms; other
    rows of its block are untouched."""
    x = torch.randn(40, 128, device=dev)
    x[7] = 0
    w = torch.randn(64, 128, device=dev).mul_(0.02).half()
    nw = torch.ones(128, device=dev)
    outs = []
    for tile in (64, 32):
        tune(linear_tile=tile)
        out = torch.zeros(40, 64, device=dev)
        gpu.linear_f64acc(x, w, out, norm_w=nw, eps=eps)
        outs.append(out)
    assert bool(outs[1][7].isnan().all()) == (eps == 0.0)
    assert torch.equal(outs[0].isnan(), outs[1].isnan())
    d = _ulps(*(o.nan_to_num(nan=0.0).cpu().numpy() for o in outs))
    assert d.max() <= 1


@pytest.mark.parametrize("rows", [40, 130])
def test_identity_weights_give_the_rows_back(gpu, dev, tune, rows):
    """One-hot columns: every element of every row is an exact product by itself, whatever its
    size beside the row's largest."""
    tune(linear_tile=64)
    rng = np.random.default_rng(23)
    k_in = 512
    x = rng.standard_normal((rows, k_in), dtype=np.float32)
    x[1::4] *= rng.standard_normal(x[1::4].shape, dtype=np.float32) ** 2
    x[2::4] = np.exp(x[2::4] * 3)
    x[3::4, 7] *= 3000
    w = np.eye(k_in, dtype=np.float16)
    assert np.array_equal(_run(gpu, dev, x, w), x)


def test_subnormal_rows_that_round_past_the_bound(gpu, dev, tune):
    """x * scale = 0.5000001 steps of f32's smallest rounds up to one, and a huge norm weight
    lifts it: twice what x * norm_w * scale says."""
    tune(linear_tile=64)
    eps = np.float32(3.999999)
    x = np.full((40, 64), 2.0 ** -149, np.float32)
    x[::3, ::5] *= -1
    nw = np.full(64, 1.99995 * 2.0 ** 99, np.float32)
    w = np.random.default_rng(29).uniform(0.5, 1, (40, 64)).astype(np.float16)
    x64 = x.astype(np.float64)
    scale = 1.0 / np.sqrt((x64 * x64).mean(axis=1, keepdims=True) + np.float64(eps))
    h = (x64 * scale).astype(np.float32) * nw
    assert np.abs(h).max() > 1.9 * np.abs(x * nw).max() * scale.max()
    out = torch.zeros(40, 40, device=dev)
    gpu.linear_f64acc(*(torch.from_numpy(a).to(dev) for a in (x, w)), out,
                      norm_w=torch.from_numpy(nw).to(dev), eps=float(eps))
    _check(out.cpu().numpy(), (h.astype(np.float64) @ w.astype(np.float64).T).astype(np.float32))


@pytest.mark.parametrize("mode", ["plain", "residual", "swiglu"])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("rows,n_out,k_in", [(1, 1, 64), (100, 72, 192), (130, 200, 1088)])
@pytest.mark.parametrize("bad_rows", [(), (3,), (40,), (3, 40), (99, 129)])
@pytest.mark.parametrize("bad_cols", [(), (1,), (33, 70)])
def test_blocks_of_f64_sums_beside_digits(gpu, dev, tune, mode, norm, rows, n_out, k_in, bad_rows, bad_cols):
    """Row blocks and column blocks outside the digits, alone and beside others in a 64 x 64 tile:
    the f64 kernel's outputs, bit for bit in those blocks."""
    rng = np.random.default_rng(31)
    x = rng.standard_normal((rows, k_in), dtype=np.float32)
    w, up = ((rng.standard_normal((n_out, k_in)) * 0.02).astype(np.float16) for _ in range(2))
    nw = (1 + 0.1 * rng.standard_normal(k_in)).astype(np.float32) if norm else None
    bad_rows = [r for r in bad_rows if r < rows]
    bad_cols = [c for c in bad_cols if c < n_out]
    for r in bad_rows:  # one in four elements is rounded
        x[r, ::4] = (rng.uniform(0.5, 1, x[r, ::4].shape) * 1e-12).astype(np.float32)
    for c in bad_cols:
        (up if mode == "swiglu" else w)[c, 5] = 200.0
    resid = rng.standard_normal((rows, n_out), dtype=np.float32) if mode == "residual" else None
    outs = []
    for tile in (64, 32):
        tune(linear_tile=tile)
        outs.append(_run(gpu, dev, x, w, nw, resid=resid, w_up=up if mode == "swiglu" else None))
    d = _ulps(*outs)
    same = np.zeros((rows, n_out), bool)
    for r in bad_rows:
        same[r // 32 * 32:r // 32 * 32 + 32] = True
    per = 16 if mode == "swiglu" else 32
    for c in bad_cols:
        same[:, c // per * per:c // per * per + per] = True
    assert not d[same].any()
    assert d.max() <= (8 if mode == "swiglu" else 1) and int((d > 0).sum()) <= max(2, d.size // 5000)


def test_workspace_is_checked(gpu, dev):
    """A workspace below the size asked for is refused before any launch; a null one means the
    plain product."""
    from crucible_amd import _lib
    lib = _lib.load()
    rows, n, k = 2048, 768, 768
    need = lib.crucible_linear_workspace_bytes(rows, n, k, 0, 0)
    assert need > 0
    assert lib.crucible_linear_workspace_bytes(16, n, k, 0, 0) == 0
    x = torch.randn(rows, k, device=dev)
    w = torch.randn(n, k, device=dev).mul_(0.02).half()
    out = torch.zeros(rows, n, device=dev)
    ws = torch.empty(need, dtype=torch.uint8, device=dev)
    args = (x.data_ptr(), k, None, 1e-6, w.data_ptr(), n, k, None, out.data_ptr(), n, rows)
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.crucible_linear_f64acc_ws(*args, ws.data_ptr(), need - 1, stream) == _lib.ERR_WORKSPACE
    assert lib.crucible_linear_f64acc_ws(*args, ws.data_ptr() + 8, need, stream) == _lib.ERR_INVALID
    assert not out.any()
    assert lib.crucible_linear_f64acc_ws(*args, None, 0, stream) == 0
    plain = out.clone()
    assert lib.crucible_linear_f64acc_ws(*args, ws.data_ptr(), need, stream) == 0
    d = (out.view(torch.int32).long() - plain.view(torch.int32).long()).abs()
    assert int(d.max()) <= 1 and int((d > 0).sum()) <= out.numel() // 20000


def test_no_room_for_the_digits(gpu, dev):
    """Where the digits' scratch does not fit the device's memory, the product is made without
    it, as it was before it took any."""
    rows, hidden, k_in = 2048, 2048, 768
    need = gpu.lib.crucible_linear_workspace_bytes(rows, hidden, k_in, 1, 1)
    assert need > 20 << 20
    x = torch.randn(rows, k_in, device=dev)
    w, up = (torch.randn(hidden, k_in, device=dev).mul_(0.02).half() for _ in range(2))
    nw = torch.ones(k_in, device=dev)
    outs = [torch.zeros(rows, hidden, device=dev) for _ in range(4)]

    def both(a, b):
        gpu.linear_f64acc(x, w, a, norm_w=nw)
        gpu.linear_swiglu_f64acc(x, w, up, b, norm_w=nw)

    both(*outs[:2])
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(dev).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(dev) + (4 << 20)) / total, dev)
    try:
        held = []  # blocks that the allocator still had
        with pytest.raises(torch.OutOfMemoryError):
            for _ in range(1000):
                held.append(torch.empty(need, dtype=torch.uint8, device=dev))
        both(*outs[2:])
    finally:
        held = None
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
    assert int((outs[0] - outs[2]).abs().gt(0).sum()) <= outs[0].numel() // 20000
    torch.testing.assert_close(outs[1], outs[3], rtol=1e-6, atol=1e-9)
