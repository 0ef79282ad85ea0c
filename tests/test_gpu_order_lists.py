"""rcsa_order_lists: ascending lists and validity bits against a plain sort."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _want(idx, cnt, nkb, rows):
    B, H, N, K = idx.shape
    out = torch.full((B, H, len(rows), K), -1, dtype=torch.int32)
    lens = torch.zeros(B, H, len(rows), dtype=torch.int32)
    for b in range(B):
        for h in range(H):
            for i, r in enumerate(rows):
                n = min(max(int(cnt[b, h, r]), 0), K)
                live = sorted(j for j in idx[b, h, r, :n].tolist() if 0 <= j < nkb)
                out[b, h, i, :len(live)] = torch.tensor(live, dtype=torch.int32)
                lens[b, h, i] = len(live)
    return out, lens


# block counts at the edges of a wavefront's 64 tallies and of the LDS they take
@pytest.mark.parametrize("nkb", [1, 63, 64, 65, 303, 4096])
@pytest.mark.parametrize("k", [1, 64, 97])
def test_order_lists(nkb, k):
    from cast_amd import ops
    g = torch.Generator().manual_seed(nkb * 100 + k)
    # padding, repeats and numbers past the keys among the entries
    idx = torch.randint(-1, nkb + 2, (2, 3, 5, k), generator=g, dtype=torch.int32)
    cnt = torch.randint(-1, k + 2, (2, 3, 5), generator=g, dtype=torch.int32)
    valid = torch.rand(nkb * 64, generator=g) > 0.4
    for rows in (None, torch.tensor([4, 0, 2])):
        got, lens, bits = ops.order_lists(idx.cuda(), cnt.cuda(), nkb, rows=rows,
                                          valid=valid.cuda())
        want, want_lens = _want(idx, cnt, nkb, range(5) if rows is None else rows.tolist())
        assert torch.equal(got.cpu(), want) and torch.equal(lens.cpu(), want_lens)
        assert torch.equal(bits.cpu(), ops.valid_bits(valid, 64).reshape(-1))
        assert torch.equal(ops.valid_bits(valid.cuda(), 64).cpu(), ops.valid_bits(valid, 64))


def test_order_lists_views():
    """Lists shared by heads and batches (stride 0) and views of wider tables."""
    from cast_amd import ops
    g = torch.Generator().manual_seed(1)
    wide = torch.randint(0, 40, (1, 4, 7, 50), generator=g, dtype=torch.int32)
    cnt = torch.randint(0, 21, (1, 1, 7), generator=g, dtype=torch.int32)
    idx = wide[:, 1:3, :, 10:30]
    got, lens = ops.order_lists(idx.cuda(), cnt.cuda(), 40)
    want, want_lens = _want(idx, cnt.expand(1, 2, 7), 40, range(7))
    assert torch.equal(got.cpu(), want) and torch.equal(lens.cpu(), want_lens)
    shared = wide[:, :1].expand(2, 5, 7, 50)
    got, lens = ops.order_lists(shared.cuda()[:, :1].expand(2, 5, 7, 50),
                                cnt.cuda().expand(2, 5, 7), 40)
    want, want_lens = _want(shared, cnt.expand(2, 5, 7), 40, range(7))
    assert torch.equal(got.cpu(), want) and torch.equal(lens.cpu(), want_lens)


def test_order_lists_refuses():
    from cast_amd import ops
    idx = torch.zeros(1, 1, 2, 4, dtype=torch.int32, device="cuda")
    cnt = torch.ones(1, 1, 2, dtype=torch.int32, device="cuda")
    with pytest.raises(RuntimeError, match="sizes"):
        ops.order_lists(idx, cnt, 4097)
    with pytest.raises(TypeError):
        ops.order_lists(idx.long(), cnt, 4)
    with pytest.raises(ValueError):
        ops.order_lists(idx, cnt[:, :, :1], 4)


@pytest.mark.parametrize("int8", [False, True])
def test_attention_over_ordered_lists(int8):
    """The attention orders lists whose keys exceed an XCD's L2: the result is that
    of the given order up to the rounding of its sums (bf16 output: half a unit in
    the last place either side, 2^-8 relative, of values below 1)."""
    from cast_amd import ops
    g = torch.Generator(device="cuda").manual_seed(2)
    H, Lq, Lk, D = 2, 256, 128 * 90, 128
    q, k, v = (torch.randn(1, H, n, D, device="cuda", generator=g).bfloat16()
               for n in (Lq, Lk, Lk))
    idx = torch.rand(1, H, 2, 90, device="cuda", generator=g).argsort(-1)[..., :40].int()
    idx = idx.contiguous()
    cnt = torch.tensor([[[40, 33], [0, 7]]], dtype=torch.int32, device="cuda")
    assert ops.order_helps(H, Lk, (3 if int8 else 4) * D, 128, 40)
    if int8:
        _, q8, qs = ops.pool_query(q, None, 128, quantize=True)
        _, ks, kn, kx = ops.pool_key(k, None, 128, stats=True)
        k8, sc, _ = ops.quantize_key(k, None, 128, ks, kn, kx)
        run = lambda **kw: ops.sparse_attn_int8(q8, qs, k8, sc, v, idx, cnt, **kw)
    else:
        run = lambda **kw: ops.sparse_attn_bf16(q, k, v, idx, cnt, **kw)
    a, b = run().float(), run(ordered=True).float()
    assert torch.allclose(a, b, rtol=2 ** -7, atol=2 ** -9)
    assert not a[0, 1, :128].any()  # the empty list
