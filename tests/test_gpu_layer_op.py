"""rcsa_attention's native op against its general path (serial, separate
selection), bit for bit: dtypes, block shapes, views, masks, budgets, the
LSE, gathered sources and V in other types."""
import pytest
import torch

pytestmark = pytest.mark.gpu

FIELDS = ("out", "indices", "counts", "score", "qhat", "khat", "lse", "q_i8", "q_scale", "k_i8",
          "k_scale", "kmean", "k_mask")


def _same(a, b):
    for name in FIELDS:
        x, y = getattr(a, name), getattr(b, name)
        assert (x is None) == (y is None), name
        if x is not None:
            assert x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y), name


@pytest.mark.parametrize("int8", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,bs", [(128, 128), (128, 64), (64, 128), (64, 64)])
def test_layer_op_matches_general_path(dev, D, bs, dtype, int8):
    from cast_amd.pipeline import rcsa_attention
    g = torch.Generator().manual_seed(D + bs)
    B, H, nq, nk = 2, 3, 3, 9
    wide = torch.randn(B, H, nk * bs, 2 * D, generator=g).to(dtype).to(dev)
    q = torch.randn(B, nq * bs, H, D, generator=g).to(dtype).to(dev).transpose(1, 2)
    k, v = wide[..., :D], wide[..., D:].flip(2)
    qv = torch.rand(nq * bs, generator=g) > 0.2
    kv = torch.rand(nk * bs, generator=g) > 0.2
    forced = torch.rand(nq, nk, generator=g) < 0.2
    allowed = torch.rand(B * H, nq, nk, generator=g) < 0.8
    rows = torch.randint(0, 7, (nq,), generator=g)
    for kw in (dict(k_select=5), dict(k_select=rows, max_k=6, forced=forced.to(dev)),
               dict(k_select=4, allowed=allowed.to(dev), forced=forced.to(dev), n_split=2),
               dict(k_select=4, sm_scale=0.2)):
        for valid in ((None, None), (qv.to(dev), kv.to(dev))):
            args = dict(block_size=bs, int8=int8, return_lse=True, **kw)
            _same(rcsa_attention(q, k, v.half(), *valid, **args),
                  rcsa_attention(q, k, v.half(), *valid, overlap=False, fuse_select=False,
                                 **args))


@pytest.mark.parametrize("int8", [True, False])
def test_gathered_layer_op_matches_general_path(dev, int8):
    from cast_amd import layout
    from cast_amd.pipeline import rcsa_attention
    g = torch.Generator().manual_seed(9)
    H, hw, shape = 2, (8, 16), (4, 4, 8)
    lq = layout.compact_layout(range(5), 0, *hw, shape, dev)
    lk = layout.compact_layout(range(11), 6, *hw, shape, dev)
    n = hw[0] * hw[1]
    q, k, v = (torch.randn(1, f * n, H, 128, generator=g).bfloat16().to(dev) for f in (5, 11, 11))
    args = dict(block_size=128, k_select=3, int8=int8, return_lse=True,
                q_slot_token=lq.slot_token, k_slot_token=lk.slot_token)
    _same(rcsa_attention(q, k, v, None, None, **args),
          rcsa_attention(q, k, v, None, None, overlap=False, fuse_select=False, **args))


def test_layer_op_refuses_as_before(dev):
    from cast_amd.pipeline import rcsa_attention
    q = torch.zeros(1, 1, 128, 128, dtype=torch.bfloat16, device=dev)
    args = dict(block_size=128, k_select=1)
    with pytest.raises(ValueError, match="valid mask"):
        rcsa_attention(q, q, q, torch.ones(5, device=dev), None, **args)
    with pytest.raises(ValueError, match="multiple of block_size"):
        rcsa_attention(q[:, :, :100], q, q, None, None, **args)
    with pytest.raises(ValueError, match="mask shape"):
        rcsa_attention(q, q, q, None, None, forced=torch.ones(3, 1, device=dev), **args)
    with pytest.raises(TypeError):
        rcsa_attention(q, q.float(), q, None, None, **args)


@pytest.mark.parametrize("int8", [True, False])
def test_layer_op_refuses_maps_that_are_no_vectors(dev, int8):
    from cast_amd.pipeline import rcsa_attention
    q = torch.zeros(1, 256, 1, 128, dtype=torch.bfloat16, device=dev)
    slots = torch.arange(256, dtype=torch.int32, device=dev)
    for qm, km in ((slots.view(2, 128), slots), (slots, slots.view(2, 128))):
        with pytest.raises(ValueError, match="slot map must be a vector"):
            rcsa_attention(q, q, q, None, None, block_size=128, k_select=1, int8=int8,
                           q_slot_token=qm, k_slot_token=km)
