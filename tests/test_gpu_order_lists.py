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
    """Lists in ascending order, for keys that exceed an XCD's L2: the result is that
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
        run = lambda i, c: ops.sparse_attn_int8(q8, qs, k8, sc, v, i, c, ordered=True)
    else:
        run = lambda i, c: ops.sparse_attn_bf16(q, k, v, i, c, ordered=True)
    a = run(*ops.order_for_attention(idx, cnt, q.shape, Lk, 128, 128)).float()
    b = run(idx, cnt).float()
    assert torch.allclose(a, b, rtol=2 ** -7, atol=2 ** -9)
    assert not a[0, 1, :128].any()  # the empty list


@pytest.mark.parametrize("ns", [2, 3, 7, 16])
@pytest.mark.parametrize("N,H", [(28, 24), (5, 3), (64, 4)])
def test_lists_of_a_split_launch(ns, N, H):
    """The lists of an XCD's query blocks past its full rounds, which the launch cuts into
    shares, keep every share's entries (those that name no block last, as -1) and are
    ascending within it; the others are ascending."""
    from cast_amd import ops
    cux = torch.cuda.get_device_properties(0).multi_processor_count // 8
    g = torch.Generator().manual_seed(ns + N)
    nkb, K = 70, 50
    idx = torch.randint(-1, nkb + 2, (1, 1, N, K), generator=g, dtype=torch.int32)
    cnt = torch.randint(0, K + 3, (1, 1, N), generator=g, dtype=torch.int32)
    cnt[0, 0, :4] = torch.tensor([0, 1, ns, ns + 1])  # shares without an entry
    got, lens = ops.order_lists(idx.cuda().expand(1, H, N, K), cnt.cuda().expand(1, H, N), nkb,
                                n_split=ns)
    want, want_lens = _want(idx, cnt, nkb, range(N))
    cut = torch.full((N, K), -1, dtype=torch.int32)  # the lists as the launch cuts them
    for r in range(N):
        n = min(int(cnt[0, 0, r]), K)
        for s in range(ns):
            a, b = n * s // ns, n * (s + 1) // ns
            live = sorted(j for j in idx[0, 0, r, a:b].tolist() if 0 <= j < nkb)
            cut[r, a:a + len(live)] = torch.tensor(live, dtype=torch.int32)
    per = -(-H * N // 8)
    item = torch.arange(H * N)
    tail = (item % per >= per // cux * cux)[:, None]
    row = item % N
    assert torch.equal(got.cpu().reshape(H * N, K), torch.where(tail, cut[row], want[0, 0, row]))
    assert torch.equal(lens.cpu().reshape(-1),
                       torch.where(tail[:, 0], cnt[0, 0].clamp_max(K)[row], want_lens[0, 0, row]))


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("H,Lq,ns", [(1, 128, 4), (2, 256, None), (8, 512, 2)])
def test_ordered_shares_round_no_further(int8, H, Lq, ns):
    """Split lists that the library orders stay as close to float64 as in the random
    order they came in, for values that resemble each other within a frame (a share's
    partial output is rounded to bf16; contiguous shares of an ascending list are 10 to
    20 per cent further off).  Both sides round the same partial outputs, up to the order
    of the sums in them; each is a mean over at least 16384 values, whose error varies by
    less than 1 per cent."""
    from cast_amd import ops
    dev, D, nkb, keys = "cuda", 128, 210, 90
    g = torch.Generator(device=dev).manual_seed(4)

    def tokens(n):
        frames = torch.randn(1, H, -(-n // 880), D, device=dev, generator=g) * 0.3
        x = torch.randn(1, H, n, D, device=dev, generator=g) / D ** 0.5
        return (x + frames.repeat_interleave(880, 2)[:, :, :n]).bfloat16()
    q, k, v = tokens(Lq), tokens(nkb * 128), tokens(nkb * 128)
    rows = Lq // 128
    idx = torch.rand(1, H, rows, nkb, device=dev, generator=g).argsort(-1)[..., :keys].int()
    idx = idx.contiguous()
    cnt = torch.full((1, H, rows), keys, dtype=torch.int32, device=dev)
    assert ops.order_helps(H, nkb * 128, (3 if int8 else 4) * D, 128, keys)
    if int8:
        _, q8, qs = ops.pool_query(q, None, 128, quantize=True)
        _, ks, kn, kx = ops.pool_key(k, None, 128, stats=True)
        k8, sc, kmean = ops.quantize_key(k, None, 128, ks, kn, kx)
        qd = q8.double().view(1, H, rows, 128, D) * qs.view(1, H, rows, 1, 1).double()
        kd = k8.double().view(1, H, nkb, 128, D) * sc.view(1, H, nkb, 1, 1).double()
        qd, kd = qd.view(1, H, Lq, D), kd.view(1, H, nkb * 128, D)
        run = lambda i, c: ops.sparse_attn_int8(q8, qs, k8, sc, v, i, c, n_split=ns, ordered=True)
    else:
        qd, kd = q.double(), k.double()
        run = lambda i, c: ops.sparse_attn_bf16(q, k, v, i, c, n_split=ns, ordered=True)
    ref = torch.empty(1, H, Lq, D, dtype=torch.float64, device=dev)
    for h in range(H):
        for r in range(rows):
            tok = (idx[0, h, r].long()[:, None] * 128 + torch.arange(128, device=dev)).reshape(-1)
            p = torch.softmax(qd[0, h, r * 128:(r + 1) * 128] @ kd[0, h, tok].T / D ** 0.5, -1)
            ref[0, h, r * 128:(r + 1) * 128] = p @ v[0, h, tok].double()
    err = lambda x: ((x.double() - ref).norm() / ref.norm()).item()
    given = err(run(idx, cnt))
    ours = err(run(*ops.order_for_attention(idx, cnt, q.shape, nkb * 128, 128, 128, ns)))
    print(f"ordered shares int8 {int8} H {H} n_split {ns}: {given:.4e} as given, {ours:.4e}",
          flush=True)
    assert ours <= 1.02 * given


@pytest.mark.parametrize("int8", [False, True])
def test_rows_past_the_query_blocks(int8):
    """Lists and lengths may each have more rows than the query has blocks, whether the
    call orders them or not; fewer are refused by the attention."""
    from cast_amd import ops
    from cast_amd.kernel import longcat_asymmetric
    g = torch.Generator(device="cuda").manual_seed(6)
    H, Lq, D, K = 2, 1024, 128, 300
    nqb = Lq // 64
    for nkb in (20, 400):
        q, k, v = (torch.randn(1, H, n, D, device="cuda", generator=g).bfloat16()
                   for n in (Lq, nkb * 128, nkb * 128))
        idx = torch.rand(1, H, nqb + 2, 400, device="cuda", generator=g).argsort(-1)[..., :K]
        idx = idx.int().contiguous()  # (the short keys: most entries name no block)
        cnt = torch.full((1, H, nqb + 1), K, dtype=torch.int32, device="cuda")
        if int8:
            _, q8, qs = ops.pool_query(q, None, 64, quantize=True)
            _, ks, kn, kx = ops.pool_key(k, None, 128, stats=True)
            k8, sc, _ = ops.quantize_key(k, None, 128, ks, kn, kx)
            run = lambda i, c: ops.sparse_attn_int8(q8, qs, k8, sc, v, i, c, block_m=64)
        else:
            run = lambda i, c: ops.sparse_attn_bf16(q, k, v, i, c, block_m=64)
        i0, c0 = idx[:, :, :nqb].contiguous(), cnt[:, :, :nqb].contiguous()
        want = run(i0, c0)
        assert ops.order_pays(H, Lq, nkb * 128, (3 if int8 else 4) * D, 64, 128, K,
                              int8) == (nkb == 400)
        for i, c in ((idx, cnt), (idx[:, :, :nqb], cnt), (idx, c0)):
            assert torch.equal(run(i, c), want)
        with pytest.raises(RuntimeError, match="spans"):
            run(idx[:, :, :1].contiguous(), cnt)
        if not int8:
            flags = torch.ones(nkb * 128, dtype=torch.bool, device="cuda")
            got = [longcat_asymmetric(q, k, v, i, c, flags, query_block_size=64,
                                      key_block_size=128) for i, c in ((idx, cnt), (i0, c0))]
            assert torch.equal(*got)


# either side of every line of the two rules (bytes of a listed block: 64 KiB bf16)
@pytest.mark.parametrize("bm,H,Lq,nkb,K,int8,pays", [
    (64, 8, 1760, 161, 28, False, True), (64, 8, 1760, 161, 27, False, False),
    (64, 8, 1760, 160, 28, False, False), (128, 24, 3520, 129, 19, False, True),
    (128, 24, 3520, 129, 18, False, False), (128, 24, 3520, 128, 19, False, False),
    (128, 24, 1760, 303, 90, False, False), (128, 24, 3520, 303, 66, True, True),
    (128, 24, 3520, 303, 65, True, False), (128, 8, 3520, 60, 60, False, False)])
def test_order_rule(bm, H, Lq, nkb, K, int8, pays):
    from cast_amd import ops
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("sizes for 256 compute units")
    assert ops.order_pays(H, Lq, nkb * 128, (3 if int8 else 4) * 128, bm, 128, K, int8) == pays


def test_asymmetric_flags_from_the_host():
    """Key flags in host memory are taken whatever the size of the call."""
    from cast_amd import kernel
    g = torch.Generator(device="cuda").manual_seed(8)
    H, D, nkb, Lq, K = 8, 128, 80, 1792, 20
    assert kernel.ops.listed_bytes(H, Lq, 4 * D, 64, 128, K) > 28 << 20
    q, k, v = (torch.randn(1, H, n, D, device="cuda", generator=g).bfloat16()
               for n in (Lq, nkb * 128, nkb * 128))
    idx = torch.rand(1, H, Lq // 64, nkb, device="cuda", generator=g).argsort(-1)[..., :K].int()
    cnt = torch.full((1, H, Lq // 64), K, dtype=torch.int32, device="cuda")
    flags = torch.rand(nkb * 128, device="cuda", generator=g) > 0.1
    run = lambda f: kernel.longcat_asymmetric(q, k, v, idx.contiguous(), cnt, f,
                                              query_block_size=64, key_block_size=128)
    torch.testing.assert_close(run(flags.cpu()).float(), run(flags).float(), rtol=2.0 ** -7,
                               atol=2.0 ** -9)
