"""The MFMA attention of head dimensions that are multiples of 32 (hd_attend.hpp) against the
one-row generic kernels, which take the same calls when a buffer is not 16-byte aligned.

Both compute the same attention over the same fp16 pages; they differ in the order of f32 sums
and in carrying P (and an f32 query) as fp16 hi + lo, about 2^-22 of each: outputs of N(0,1)
values agree to 1e-5. Sizes sit at the edges: one key, one page, either side of a 16-page split
and of a 32-row tile, more than 16 query heads a group, every dimension.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _unaligned(t):
    """The same values one element into a larger buffer."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    out = flat[1:].view(t.shape)
    out.copy_(t)
    return out


def _case(dev, seed, hd, n_head, n_kv, lens, n_layer=2, dtype=torch.float32):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    stride = max(-(-max(max(lens), 1) // 16), 1) + 1
    n_pages = len(lens) * stride + 3
    kv = n_kv * hd
    pools = [torch.randn(n_pages * n_layer * 16 * kv, generator=g, device=dev).half() for _ in "kv"]
    perm = torch.randperm(n_pages, generator=g, device=dev)[:len(lens) * stride]
    tables = perm.view(len(lens), stride).int().contiguous()
    q = torch.randn(len(lens), n_head * hd, generator=g, device=dev).to(dtype)
    return g, stride, kv, pools, tables, q


@pytest.mark.parametrize("hd,n_head,n_kv", [(32, 4, 4), (32, 24, 1), (96, 12, 3), (128, 40, 2),
                                            (160, 6, 2), (192, 4, 1), (224, 2, 2), (256, 8, 2)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_decode_against_generic(gpu, dev, hd, n_head, n_kv, dtype):
    lens = [1, 15, 16, 17, 255, 256, 257, 0, 600]
    b, layer = len(lens), 1
    g, stride, kv, (kp, vp), tables, q = _case(dev, hd + n_head, hd, n_head, n_kv, lens, dtype=dtype)
    d_len = torch.tensor(lens, dtype=torch.int32, device=dev)

    def run(q, k, v):
        out = torch.full((b, n_head * hd), 7.0, device=dev)
        gpu.attention_decode_paged(q, k, v, out, tables, d_len, b, n_head, n_kv, hd, stride, 2,
                                   layer, kv, stride * 16)
        return out

    got, want = run(q, kp, vp), run(_unaligned(q), kp, vp)
    assert torch.all(got[7] == 7.0), "an inactive request's output was written"
    assert float((got - want).abs().max()) <= TOL
    # without scratch one workgroup walks the splits: the same bits
    from crucible_amd import _lib
    lib = _lib.load()
    alone = torch.full_like(got, 7.0)
    _lib.check(lib.crucible_attention_decode_paged(
        q.data_ptr(), 0 if dtype == torch.float32 else 1, kp.data_ptr(), vp.data_ptr(),
        alone.data_ptr(), 0, tables.data_ptr(), d_len.data_ptr(), b, n_head, n_kv, hd, stride, 2,
        layer, kv, stride * 16, None, 0, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(alone, got)


@pytest.mark.parametrize("hd,n_head,n_kv", [(32, 24, 1), (96, 12, 3), (128, 12, 3), (256, 4, 2)])
@pytest.mark.parametrize("kv_dtype", [torch.float32, torch.float16])
def test_append_against_separate_calls(gpu, dev, hd, n_head, n_kv, kv_dtype):
    """Positions inside the attended keys, just past them, in a page the length does not reach,
    in the table's last page and outside it; inactive requests append too."""
    lens = [1, 16, 17, 300, 40, 0, 260, 30]
    pos = [0, 15, 16, 299, 40, 3, 16 * 19 - 1, 10 ** 6]
    b, layer = len(lens), 0
    g, stride, kv, (kp, vp), tables, q = _case(dev, hd, hd, n_head, n_kv, lens)
    assert stride == 20
    d_len = torch.tensor(lens, dtype=torch.int32, device=dev)
    d_pos = torch.tensor(pos, dtype=torch.int32, device=dev)
    new = [torch.randn(b, kv, generator=g, device=dev).to(kv_dtype) for _ in "kv"]
    k1, v1, k2, v2 = kp.clone(), vp.clone(), kp.clone(), vp.clone()
    o1 = torch.full((b, n_head * hd), 7.0, device=dev)
    o2 = o1.clone()
    gpu.attention_decode_paged_append(q, new[0], new[1], k1, v1, o1, tables, d_pos, d_len, b, n_head,
                                      n_kv, hd, stride, 2, layer, kv, 300)
    for src, pool, kind in ((new[0], k2, "k"), (new[1], v2, "v")):
        gpu.cache_store_rows_paged(src, pool, tables, d_pos, b, kv, stride, 2, layer, kind=kind)
    gpu.attention_decode_paged(q, k2, v2, o2, tables, d_len, b, n_head, n_kv, hd, stride, 2, layer,
                               kv, 300)
    assert torch.equal(k1, k2) and torch.equal(v1, v2)
    assert torch.equal(o1, o2)


@pytest.mark.parametrize("hd", [32, 96, 128, 160, 192, 224, 256])
@pytest.mark.parametrize("entry", ["append", "noalloc", "qkv"])
def test_rows_of_one_batch_that_share_pages(gpu, dev, hd, entry):
    """Sixteen consecutive positions of one sequence in one call, as in the verification of
    several tokens: every row sees the earlier rows' appends, and the outputs are those of the
    separate calls. Four more rows share a page of another sequence in descending order."""
    from crucible_amd import _lib
    lib = _lib.load()
    n_head, n_kv, layer = 4, 2, 1
    pos = list(range(500, 516)) + [43, 42, 41, 40]
    lens = [p + 1 for p in pos]
    b = len(pos)
    g, stride, kv, (kp, vp), two, _ = _case(dev, hd + 3, hd, n_head, n_kv, [516, 44])
    tables = two[torch.tensor([0] * 16 + [1] * 4, device=dev)].contiguous()
    qkv = torch.randn(b, n_head * hd + 2 * kv, generator=g, device=dev)
    q = qkv[:, :n_head * hd].contiguous()
    new = [qkv[:, n_head * hd + i * kv:n_head * hd + (i + 1) * kv].contiguous() for i in range(2)]
    d_len, d_pos = (torch.tensor(x, dtype=torch.int32, device=dev) for x in (lens, pos))
    k1, v1, k2, v2 = kp.clone(), vp.clone(), kp.clone(), vp.clone()
    for src, pool, kind in ((new[0], k2, "k"), (new[1], v2, "v")):
        gpu.cache_store_rows_paged(src, pool, tables, d_pos, b, kv, stride, 2, layer, kind=kind)
    o1, o2, o3 = (torch.full((b, n_head * hd), 7.0, device=dev) for _ in range(3))
    geometry = (b, n_head, n_kv, hd, stride, 2, layer, kv, stride * 16)
    gpu.attention_decode_paged(q, k2, v2, o2, tables, d_len, *geometry)
    gpu.attention_decode_paged(_unaligned(q), k2, v2, o3, tables, d_len, *geometry)
    if entry == "append":
        gpu.attention_decode_paged_append(q, *new, k1, v1, o1, tables, d_pos, d_len, *geometry)
    elif entry == "qkv":
        gpu.attention_decode_qkv_paged_append(qkv, None, None, k1, v1, o1, tables, d_pos, d_len,
                                              *geometry)
    else:
        _lib.check(lib.crucible_attention_decode_paged_append_noalloc(
            q.data_ptr(), 0, new[0].data_ptr(), new[1].data_ptr(), 0, k1.data_ptr(), v1.data_ptr(),
            o1.data_ptr(), 0, tables.data_ptr(), d_pos.data_ptr(), d_len.data_ptr(), *geometry,
            torch.cuda.current_stream().cuda_stream))
    assert torch.equal(k1, k2) and torch.equal(v1, v2)
    assert torch.equal(o1, o2)
    assert float((o1 - o3).abs().max()) <= TOL


@pytest.mark.parametrize("hd", [32, 96, 128, 160, 256])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_prefill_against_generic(gpu, dev, hd, dtype):
    lens = [1, 16, 31, 32, 33, 65, 300]
    n_head, n_kv, layer = 4, 2, 1
    g, stride, kv, (kp, vp), tables, _ = _case(dev, hd, hd, n_head, n_kv, lens)
    owners = np.repeat(np.arange(len(lens), dtype=np.int32), lens)
    positions = np.concatenate([np.arange(n, dtype=np.int32) for n in lens])
    rows = len(owners)
    q = torch.randn(rows, n_head * hd, generator=g, device=dev).to(dtype)
    d_own, d_pos = (torch.from_numpy(a).to(dev) for a in (owners, positions))

    def run(q, v):
        out = torch.full((rows, n_head * hd), 7.0, device=dev)
        gpu.attention_prefill_packed(q, kp, v, out, tables, d_own, d_pos, rows, stride, n_head, n_kv,
                                     hd, 2, layer, kv, stride * 16)
        return out

    got = run(q, vp)
    assert float((got - run(_unaligned(q), vp)).abs().max()) <= TOL
    # packed tiles hold rows of several requests: one request's NaN stays its own
    bad = vp.clone().view(-1, 2, kv, 16)
    bad[tables[2, :1].long(), layer] = float("nan")
    touched = torch.from_numpy(owners == 2).to(dev)
    other = run(q, bad.view(-1))
    assert torch.equal(other[~touched], got[~touched])
    assert torch.all(torch.isnan(other[touched]))


@pytest.mark.parametrize("hd", [32, 128, 256])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_prefill_rows_before_an_infinite_value(gpu, dev, hd, bad):
    """V values that are not finite reach the rows that see them, and no earlier row of the tile;
    positions descend within the second request."""
    lens, at = [70, 40], [37, 8]
    n_head, n_kv, layer = 4, 2, 1
    g, stride, kv, (kp, vp), tables, _ = _case(dev, hd + 1, hd, n_head, n_kv, lens)
    owners = np.repeat(np.arange(2, dtype=np.int32), lens)
    positions = np.concatenate([np.arange(70), np.arange(40)[::-1]]).astype(np.int32)
    pool = vp.view(-1, 2, kv, 16)
    for r, t in enumerate(at):
        pool[tables[r, t // 16].long(), layer, :, t % 16] = bad
    q = torch.randn(110, n_head * hd, generator=g, device=dev)
    d_own, d_pos = (torch.from_numpy(a).to(dev) for a in (owners, positions))

    def run(q):
        out = torch.full((110, n_head * hd), 7.0, device=dev)
        gpu.attention_prefill_packed(q, kp, vp, out, tables, d_own, d_pos, 110, stride, n_head, n_kv,
                                     hd, 2, layer, kv, stride * 16)
        return out

    got, want = run(q), run(_unaligned(q))
    sees = torch.from_numpy(positions >= np.array(at)[owners]).to(dev)
    assert not torch.isfinite(got[sees]).any() and not torch.isfinite(want[sees]).any()
    assert float((got[~sees] - want[~sees]).abs().max()) <= TOL


def _same_special(got, want):
    """NaN and infinities in the same places, the rest to TOL."""
    assert torch.equal(got.isnan(), want.isnan())
    inf = want.isinf()
    assert torch.equal(got.isinf(), inf) and torch.equal(got[inf], want[inf])
    fine = want.isfinite()
    assert float((got[fine] - want[fine]).abs().max()) <= TOL


def _spoil(pools, tables, layer, kv, request, key, what, value):
    """`value` into one key of a request: its whole V row, the first half of it, or one K element."""
    page = tables[request, key // 16].long()
    if what == "k":
        pools[0].view(-1, 2, 16, kv)[page, layer, key % 16, ::32] = value
    else:
        pools[1].view(-1, 2, kv, 16)[page, layer, :kv // (2 if what == "half" else 1), key % 16] = value


SPECIAL = [("v", 3, float("inf")), ("half", 290, float("-inf")), ("half", 40, float("nan")),
           ("k", 5, float("inf")), ("k", 299, float("-inf"))]


@pytest.mark.parametrize("hd", [32, 96, 128, 160, 192, 224, 256])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("what,key,value", SPECIAL)
def test_decode_of_infinite_values(gpu, dev, hd, dtype, what, key, value):
    """A visible infinity gives what the generic kernels' f32 sums give: an infinite V value an
    infinite output, and NaN only where they have one."""
    from crucible_amd import _lib
    lib = _lib.load()
    lens, n_head, n_kv, layer = [300, 70, 600, 17], 4, 2, 1
    g, stride, kv, pools, tables, q = _case(dev, hd + 7, hd, n_head, n_kv, lens, dtype=dtype)
    _spoil(pools, tables, layer, kv, 0, key, what, value)
    _spoil(pools, tables, layer, kv, 2, key, what, value)
    _spoil(pools, tables, layer, kv, 2, 555, "half", float("inf"))
    d_len = torch.tensor(lens, dtype=torch.int32, device=dev)
    outs = []
    for x in (q, _unaligned(q)):
        out = torch.full((4, n_head * hd), 7.0, device=dev)
        gpu.attention_decode_paged(x, *pools, out, tables, d_len, 4, n_head, n_kv, hd, stride, 2, layer,
                                   kv, stride * 16)
        outs.append(out)
    _same_special(*outs)
    alone = torch.full_like(outs[0], 7.0)
    _lib.check(lib.crucible_attention_decode_paged(
        q.data_ptr(), 0 if dtype == torch.float32 else 1, pools[0].data_ptr(), pools[1].data_ptr(),
        alone.data_ptr(), 0, tables.data_ptr(), d_len.data_ptr(), 4, n_head, n_kv, hd, stride, 2,
        layer, kv, stride * 16, None, 0, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(alone.nan_to_num(nan=5.0), outs[0].nan_to_num(nan=5.0))


@pytest.mark.parametrize("hd", [32, 96, 128, 160, 192, 224, 256])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("hybrid", [False, True])
@pytest.mark.parametrize("what,key,value", SPECIAL)
def test_prefill_of_infinite_values(gpu, dev, hd, dtype, hybrid, what, key, value):
    """The same for prefill rows before, at and after the key, in pairs of pages that a tile's
    rows see whole and in part; hybrid chunks also bring a V value past fp16's range."""
    starts, lens = [250, 0], [60, 45]
    n_head, n_kv, layer = 4, 2, 1
    g, stride, kv, pools, tables, _ = _case(dev, hd + 9, hd, n_head, n_kv,
                                            [s + n for s, n in zip(starts, lens)])
    _spoil(pools, tables, layer, kv, 0, key, what, value)
    if key < 45:
        _spoil(pools, tables, layer, kv, 1, key, what, value)
    rows = sum(lens)
    segments = torch.tensor([[0, lens[0], starts[0], 0], [lens[0], lens[1], starts[1], 1]],
                            dtype=torch.int32, device=dev)
    q = torch.randn(rows, n_head * hd, generator=g, device=dev).to(dtype)
    cur = [torch.randn(rows, kv, generator=g, device=dev) for _ in "kv"]
    cur[1][40, :kv // 4] = 1e6
    outs = []
    for x in (q, _unaligned(q)):
        out = torch.full((rows, n_head * hd), 7.0, device=dev)
        gpu.attention_prefill_tiled(x, *pools, *(cur if hybrid else (None, None)), out, tables, segments,
                                    2, max(lens), stride, n_head, n_kv, hd, 2, layer, kv, hybrid=hybrid)
        outs.append(out)
    _same_special(*outs)


@pytest.mark.parametrize("hd,n_head,n_kv,lens", [
    (128, 2, 2, [200, 16]), (160, 4, 2, [256, 1]), (256, 4, 1, [100]), (96, 8, 8, [40] * 64),
    (160, 4, 4, [300] * 64), (128, 8, 8, [300] * 64), (128, 8, 8, [300] * 63), (160, 4, 2, [257, 8])])
def test_decode_forms_by_shape(gpu, dev, hd, n_head, n_kv, lens):
    """Shapes on both sides of the line between the one-head and the shared-K/V kernels: outputs
    to TOL of the generic kernel's, equal bits with and without scratch and from the fused entry."""
    from crucible_amd import _lib
    lib = _lib.load()
    b, layer = len(lens), 1
    g, stride, kv, (kp, vp), tables, q = _case(dev, hd + b, hd, n_head, n_kv, lens)
    d_len = torch.tensor(lens, dtype=torch.int32, device=dev)
    max_seq = 16 * -(-max(lens) // 16)
    geometry = (b, n_head, n_kv, hd, stride, 2, layer, kv, max_seq)
    outs = [torch.full((b, n_head * hd), 7.0, device=dev) for _ in range(4)]
    gpu.attention_decode_paged(q, kp, vp, outs[0], tables, d_len, *geometry)
    gpu.attention_decode_paged(_unaligned(q), kp, vp, outs[1], tables, d_len, *geometry)
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(lib.crucible_attention_decode_paged(
        q.data_ptr(), 0, kp.data_ptr(), vp.data_ptr(), outs[2].data_ptr(), 0, tables.data_ptr(),
        d_len.data_ptr(), *geometry, None, 0, stream))
    k = kp.view(-1, 2, 16, kv)
    v = vp.view(-1, 2, kv, 16)
    last = d_len.long() - 1
    page = tables.gather(1, (last // 16)[:, None])[:, 0].long()
    k_new, v_new = k[page, layer, last % 16].contiguous(), v[page, layer, :, last % 16].contiguous()
    gpu.attention_decode_paged_append(q, k_new, v_new, kp, vp, outs[3], tables, last.int(), d_len, *geometry)
    assert float((outs[0] - outs[1]).abs().max()) <= TOL
    assert torch.equal(outs[2], outs[0]) and torch.equal(outs[3], outs[0])


@pytest.mark.parametrize("hd", [32, 96, 128, 160, 192, 224, 256])
@pytest.mark.parametrize("n_head,n_kv", [(4, 2), (40, 2)])
@pytest.mark.parametrize("kind", ["distinct", "alternating", "runs"])
def test_prefill_tiles_of_many_owners(gpu, dev, hd, n_head, n_kv, kind):
    """Packed rows of as many requests as rows, of three requests in turn, and of runs longer and
    shorter than a tile: a tile's owners are dealt out over workgroups (more of them with few
    heads), and every row is its request's alone."""
    rng = np.random.default_rng(37)
    owners = {"distinct": rng.permutation(70), "alternating": np.arange(70) % 3,
              "runs": np.repeat(np.arange(5), [1, 40, 2, 24, 3])}[kind].astype(np.int32)
    lens = rng.integers(1, 90, owners.max() + 1).tolist()
    positions = np.array([rng.integers(0, lens[o]) for o in owners], np.int32)
    positions[5] = -1
    g, stride, kv, (kp, vp), tables, _ = _case(dev, hd + 11, hd, n_head, n_kv, lens)
    q = torch.randn(70, n_head * hd, generator=g, device=dev).half()
    d_own, d_pos = (torch.from_numpy(a).to(dev) for a in (owners, positions))
    outs = []
    for x in (q, _unaligned(q)):
        out = torch.full((70, n_head * hd), 7.0, device=dev)
        gpu.attention_prefill_packed(x, kp, vp, out, tables, d_own, d_pos, 70, stride, n_head, n_kv, hd,
                                     2, 1, kv, stride * 16)
        outs.append(out)
    assert bool((outs[0][5] == 7.0).all())
    assert float((outs[0] - outs[1]).abs().max()) <= TOL


def test_large_and_tiny_f32_queries(gpu, dev):
    """f32 queries outside fp16's range: the operands are scaled by a power of two."""
    hd, n_head, n_kv, lens = 128, 4, 2, [70, 33]
    g, stride, kv, (kp, vp), tables, q = _case(dev, 5, hd, n_head, n_kv, lens)
    d_len = torch.tensor(lens, dtype=torch.int32, device=dev)
    for factor in (2.0 ** -60, 1e-6, 1e5):
        kp2 = (kp.float() * min(1.0, 1.0 / factor)).half() if factor > 1 else kp
        qq = (q * factor).contiguous()
        outs = []
        for x in (qq, _unaligned(qq)):
            out = torch.zeros(2, n_head * hd, device=dev)
            gpu.attention_decode_paged(x, kp2, vp, out, tables, d_len, 2, n_head, n_kv, hd, stride, 2,
                                       0, kv, stride * 16)
            outs.append(out)
        assert torch.isfinite(outs[0]).all()
        # scores of 1e5 x 1e-5 products keep 2^-22 of their magnitude (about 11): 1e-4 of weight
        assert float((outs[0] - outs[1]).abs().max()) <= (1e-4 if factor > 1 else TOL)


@pytest.mark.parametrize("hd", [32, 128])
@pytest.mark.parametrize("power", [-140, -119, -100, 22, 26, 28, 30, 40, 80, 91, 110, 119])
def test_f32_queries_over_the_whole_range(gpu, dev, hd, power):
    """Scores past 2^18 put all the weight on the largest, scores below 2^-80 weigh every key the
    same: either way the outputs are the generic kernels' (their largest two scores are 2^-12
    apart or more), in decode and in prefill."""
    n_head, n_kv, lens = 4, 2, [70, 33]
    g, stride, kv, (kp, vp), tables, q = _case(dev, 5, hd, n_head, n_kv, lens)
    q = torch.ldexp(q, torch.tensor(power, device=dev)) if power > -126 else \
        torch.ldexp(torch.ldexp(q, torch.tensor(-100, device=dev)), torch.tensor(power + 100, device=dev))
    assert q.isfinite().all() and bool((q != 0).any())
    if power > 0:
        k = kp.view(-1, 2, 16, n_kv, hd)
        for b, n in enumerate(lens):
            keys = k[tables[b].long(), 0].reshape(-1, n_kv, hd)[:n].double()
            s = (q[b].double().view(1, n_head, hd) * keys.repeat_interleave(2, 1)).sum(2).t().sort(1).values
            assert bool(((s[:, -1] - s[:, -2]) > s.abs().amax(1) * 2.0 ** -12).all())
    d_len = torch.tensor(lens, dtype=torch.int32, device=dev)
    d_own = torch.tensor([0, 1], dtype=torch.int32, device=dev)
    outs = []
    for x in (q, _unaligned(q)):
        a, b = torch.zeros(2, n_head * hd, device=dev), torch.zeros(2, n_head * hd, device=dev)
        gpu.attention_decode_paged(x, kp, vp, a, tables, d_len, 2, n_head, n_kv, hd, stride, 2, 0, kv,
                                   stride * 16)
        gpu.attention_prefill_packed(x, kp, vp, b, tables, d_own, d_len - 1, 2, stride, n_head, n_kv, hd,
                                     2, 0, kv, stride * 16)
        outs.append((a, b))
    for got, want in zip(*outs):
        assert want.isfinite().all()
        assert float((got - want).abs().max()) <= TOL


@pytest.mark.parametrize("hd,n_head,n_kv", [(32, 12, 3), (96, 12, 3), (128, 12, 3), (160, 6, 2), (192, 6, 2),
                                            (224, 6, 2), (256, 6, 2)])
def test_decode_of_long_contexts(gpu, dev, hd, n_head, n_kv):
    """Nine and seventeen splits: the combine takes its partials in two and three batches."""
    from crucible_amd import _lib
    lib = _lib.load()
    lens = [2048, 2049, 4200, 100]
    g, stride, kv, (kp, vp), tables, q = _case(dev, hd + 13, hd, n_head, n_kv, lens)
    d_len = torch.tensor(lens, dtype=torch.int32, device=dev)
    geometry = (4, n_head, n_kv, hd, stride, 2, 1, kv, stride * 16)
    outs = [torch.zeros(4, n_head * hd, device=dev) for _ in range(3)]
    gpu.attention_decode_paged(q, kp, vp, outs[0], tables, d_len, *geometry)
    gpu.attention_decode_paged(_unaligned(q), kp, vp, outs[1], tables, d_len, *geometry)
    _lib.check(lib.crucible_attention_decode_paged(
        q.data_ptr(), 0, kp.data_ptr(), vp.data_ptr(), outs[2].data_ptr(), 0, tables.data_ptr(),
        d_len.data_ptr(), *geometry, None, 0, torch.cuda.current_stream().cuda_stream))
    assert float((outs[0] - outs[1]).abs().max()) <= TOL
    assert torch.equal(outs[2], outs[0])


@pytest.mark.parametrize("hd", [32, 96, 128, 160, 192, 224, 256])
@pytest.mark.parametrize("kv_dtype", [torch.float32, torch.float16])
def test_fused_entries_at_every_dimension(gpu, dev, hd, kv_dtype):
    """RoPE and both appends: pools byte for byte those of the RoPE split and the appends, outputs
    to TOL of the generic kernel's on them."""
    lens = [1, 16, 17, 300, 40, 0]
    pos = [0, 15, 16, 299, 10, 3]
    b, n_head, n_kv, layer = len(lens), 6, 2, 1
    g, stride, kv, (kp, vp), tables, _ = _case(dev, hd + 15, hd, n_head, n_kv, lens)
    d_len, d_pos = (torch.tensor(x, dtype=torch.int32, device=dev) for x in (lens, pos))
    angle = torch.randn(stride * 16, hd // 2, generator=g, device=dev)
    cos, sin = angle.cos().contiguous(), angle.sin().contiguous()
    qkv = torch.randn(b, n_head * hd + 2 * kv, generator=g, device=dev)
    q = torch.empty(b, n_head * hd, device=dev)
    k, v = torch.empty(b, kv, device=dev), torch.empty(b, kv, device=dev)
    gpu.rope_split_qkv(qkv, q, k, v, cos, sin, d_pos, n_head, n_kv, hd)
    k, v = k.to(kv_dtype), v.to(kv_dtype)
    geometry = (b, n_head, n_kv, hd, stride, 2, layer, kv, stride * 16)
    pools = [[kp.clone(), vp.clone()] for _ in range(3)]
    outs = [torch.full((b, n_head * hd), 7.0, device=dev) for _ in range(3)]
    for src, pool, kind in ((k, pools[0][0], "k"), (v, pools[0][1], "v")):
        gpu.cache_store_rows_paged(src, pool, tables, d_pos, b, kv, stride, 2, layer, kind=kind)
    gpu.attention_decode_paged(_unaligned(q), *pools[0], outs[0], tables, d_len, *geometry)
    gpu.attention_decode_paged_append(q, k, v, *pools[1], outs[1], tables, d_pos, d_len, *geometry)
    gpu.attention_decode_qkv_paged_append(qkv, cos, sin, *pools[2], outs[2], tables, d_pos, d_len, *geometry)
    for i in (1, 2):
        assert torch.equal(pools[i][0], pools[0][0]) and torch.equal(pools[i][1], pools[0][1])
        assert float((outs[i] - outs[0]).abs().max()) <= TOL
        assert bool((outs[i][5] == 7.0).all())


@pytest.mark.parametrize("hd", [128, 256])
def test_workspace_shared_with_head_dim_64(gpu, dev, hd):
    """Calls of other head dimensions leave the counters and the unit plan of a workspace alone,
    so a caller's head_dim 64 launches around them give the bits they give by themselves."""
    from crucible_amd import _lib
    lib = _lib.load()
    lens, n_head, n_kv = [600, 33, 257], 12, 3
    b = len(lens)
    d_len = torch.tensor(lens, dtype=torch.int32, device=dev)
    wide, usual = (_case(dev, d, d, n_head, n_kv, lens) for d in (hd, 64))
    max_seq = usual[1] * 16
    nbytes = lib.crucible_attention_decode_workspace_bytes(b, n_head, max_seq) + 4 * b * n_head * (hd + 2)
    fixed = lib.crucible_attention_decode_workspace_bytes(1, 1, 1) - 4 * 66  # one split's partials
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=dev)

    def run(case, d):
        _, stride, kv, (kp, vp), tables, q = case
        out = torch.zeros(b, n_head * d, device=dev)
        _lib.check(lib.crucible_attention_decode_paged(
            q.data_ptr(), 0, kp.data_ptr(), vp.data_ptr(), out.data_ptr(), 0, tables.data_ptr(),
            d_len.data_ptr(), b, n_head, n_kv, d, stride, 2, 1, kv, max_seq, ws.data_ptr(), nbytes,
            torch.cuda.current_stream().cuda_stream))
        return out

    before = ws.clone()
    first = run(wide, hd)
    assert torch.equal(ws[:fixed], before[:fixed]), "the counters or the plan were written"
    assert not torch.equal(ws[fixed:], before[fixed:]), "the partials are not where they should be"
    want = run(usual, 64)
    assert torch.equal(run(wide, hd), first)
    assert torch.equal(run(usual, 64), want)


@pytest.mark.parametrize("hd", [128, 256])
def test_the_callers_workspace_is_used(gpu, dev, hd):
    """A call that brings a workspace which holds its partials allocates nothing and writes them
    there; one that is too small is left alone; one that is not on the device is refused."""
    from crucible_amd._lib import CrucibleError
    lens, n_head, n_kv = [600, 33, 257], 12, 3
    b = len(lens)
    g, stride, kv, (kp, vp), tables, q = _case(dev, hd, hd, n_head, n_kv, lens)
    d_len = torch.tensor(lens, dtype=torch.int32, device=dev)
    max_seq = stride * 16
    need = gpu.lib.crucible_attention_decode_workspace_bytes(b, n_head, max_seq) + 4 * b * n_head * (hd + 2)

    def run(ws):
        out = torch.zeros(b, n_head * hd, device=dev)
        before = torch.cuda.memory_stats(dev)["allocation.all.allocated"]
        gpu.attention_decode_paged(q, kp, vp, out, tables, d_len, b, n_head, n_kv, hd, stride, 2, 1, kv,
                                   max_seq, workspace=ws)
        return out, torch.cuda.memory_stats(dev)["allocation.all.allocated"] - before

    want, allocated = run(None)
    assert allocated > 0
    ws = torch.zeros(need, dtype=torch.uint8, device=dev)
    out, allocated = run(ws)
    assert allocated == 0 and bool(ws.any()) and torch.equal(out, want)
    small = torch.zeros(1 << 20, dtype=torch.uint8, device=dev)
    out, _ = run(small)
    assert not small.any() and torch.equal(out, want)
    with pytest.raises(CrucibleError):
        run(torch.zeros(need, dtype=torch.uint8))


@pytest.mark.parametrize("hd", [128, 256])
def test_captured_calls_replay(gpu, dev, hd):
    """The fused decode with scratch of its own, and a projection on digits, captured in a graph:
    every replay on new inputs, with eager work between, gives the eager calls' outputs."""
    lens, n_head, n_kv, layer = [600, 33, 257], 12, 3, 1
    b = len(lens)
    g, stride, kv, (kp, vp), tables, q = _case(dev, hd + 17, hd, n_head, n_kv, lens)
    d_len = torch.tensor(lens, dtype=torch.int32, device=dev)
    new = [torch.randn(b, kv, generator=g, device=dev) for _ in "kv"]
    x = torch.randn(300, 768, generator=g, device=dev)
    w = torch.randn(1152, 768, generator=g, device=dev).mul_(0.02).half()
    nw = torch.ones(768, device=dev)
    out, y = torch.zeros(b, n_head * hd, device=dev), torch.zeros(300, 1152, device=dev)
    assert gpu.lib.crucible_linear_workspace_bytes(300, 1152, 768, 1, 0) > 0

    def step(o, p):
        gpu.attention_decode_paged_append(q, *new, kp, vp, o, tables, d_len - 1, d_len, b, n_head, n_kv, hd,
                                          stride, 2, layer, kv, stride * 16)
        gpu.linear_f64acc(x, w, p, norm_w=nw)

    step(out, y)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(out, y)
    for _ in range(4):
        for t in (q, *new, x):
            t.copy_(torch.randn(t.shape, generator=g, device=dev))
        x[5] *= 1e-3
        x[5, 0] = float("inf")  # f64 sums for its block
        want, wy = torch.zeros_like(out), torch.zeros_like(y)
        step(want, wy)
        torch.cuda.synchronize()
        out.zero_(), y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(y.nan_to_num(nan=7.0), wy.nan_to_num(nan=7.0))
