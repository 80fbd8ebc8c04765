"""The two forms of the RoPE split (16-byte accesses, 4 pairs a thread; scalar for unaligned
buffers and head dimensions that are not a multiple of 8) and the V append's row groups, at the
edges of both: bit for bit against each other and against the K append's rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _shift(t):
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    out = flat[1:].view(t.shape)
    out.copy_(t)
    return out


@pytest.mark.parametrize("rows,nh,nkv,hd", [(1, 1, 1, 8), (3, 12, 3, 64), (70, 5, 2, 24),
                                            (2, 40, 8, 128), (1030, 4, 4, 32)])
def test_rope_split_forms_agree(gpu, dev, rows, nh, nkv, hd):
    g = torch.Generator(device=dev)
    g.manual_seed(rows + hd)
    qkv = torch.randn(rows, (nh + 2 * nkv) * hd, generator=g, device=dev)
    cos, sin = (torch.randn(50, hd // 2, generator=g, device=dev) for _ in "cs")
    pos = torch.randint(0, 50, (rows,), generator=g, device=dev).int()
    pos[rows // 2] = 50 if rows > 2 else pos[rows // 2]  # outside the tables: NaN rows
    outs = []
    for x in (qkv, _shift(qkv)):
        o = [torch.full((rows, n * hd), 7.0, device=dev) for n in (nh, nkv, nkv)]
        gpu.rope_split_qkv(x, *o, cos, sin, pos, nh, nkv, hd)
        outs.append(o)
    for a, b in zip(*outs):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    assert torch.equal(outs[0][2], qkv[:, (nh + nkv) * hd:])
    assert bool(torch.isnan(outs[0][0]).any()) == (rows > 2)


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 100])
@pytest.mark.parametrize("kv", [8, 12, 192])
def test_v_append_is_the_k_append_transposed(gpu, dev, rows, kv):
    g = torch.Generator(device=dev)
    g.manual_seed(rows * kv)
    stride, n_layer, layer = 8, 2, 1
    table = torch.randperm(stride, generator=g, device=dev).view(1, stride).int().contiguous()
    pos = (torch.arange(rows, device=dev) + 5).int()
    pos[rows // 3] = -1  # skipped
    own = torch.zeros(rows, dtype=torch.int32, device=dev)
    src = torch.randn(rows, kv, generator=g, device=dev)
    pools = {}
    for kind in "kv":
        pools[kind] = torch.full((stride * n_layer * 16 * kv,), 7.0, dtype=torch.float16, device=dev)
        gpu.cache_store_packed_paged(src, pools[kind], table, own, pos, rows, kv, stride, n_layer,
                                     layer, kind=kind)
    k = pools["k"].view(stride, n_layer, 16, kv)
    v = pools["v"].view(stride, n_layer, kv, 16)
    assert torch.equal(k, v.transpose(2, 3))
    assert int((k != 7.0).sum()) <= (rows - 1) * kv
