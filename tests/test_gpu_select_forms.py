"""The block scores' query tiles, the selection's register forms with ties and
either class cut, the local rank order and the certificate sums, against plain
torch on the CPU."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# 16-, 32- and 64-row tiles (by the rows and the workgroups they leave), their
# remainders, one row and one column
@pytest.mark.parametrize("nbh,nq,nk", [(1, 1, 1), (2, 17, 65), (24, 28, 853), (24, 33, 330),
                                       (24, 65, 700), (3, 130, 63)])
@pytest.mark.parametrize("d", [64, 128])
def test_block_scores_tiles(dev, nbh, nq, nk, d):
    from cast_amd import ops
    g = torch.Generator().manual_seed(nq + nk)
    q, k = (torch.nn.functional.normalize(torch.randn(nbh, n, d, generator=g), dim=-1)
            for n in (nq, nk))
    got = ops.block_scores(q.to(dev), k.to(dev)).cpu()
    # unit vectors: a chain of d FMAs is within d 2^-24 of the exact product
    want = q.double() @ k.double().transpose(1, 2)
    assert float((got.double() - want).abs().max()) <= d * 2.0 ** -24


def _want(score, k, forced, allowed, local_rank):
    """Order of preference: forced, then score (or, local_rank, the forced by
    fl(score + 1e6)), ties to the lower index."""
    nbh, nq, nk = score.shape
    rank = torch.where(forced, (score + 1e6) - 1e6, score) if local_rank else score
    lists = []
    for b in range(nbh):
        for i in range(nq):
            cols = [j for j in range(nk) if allowed is None or bool(allowed[i, j])]
            cols.sort(key=lambda j: (not bool(forced[i, j]), -float(rank[b, i, j]), j))
            lists.append(cols[:max(0, min(int(k[i]), len(cols)))])
    return lists


@pytest.mark.parametrize("nk", [5, 64, 130, 300, 330, 400, 513, 1100, 2100])
@pytest.mark.parametrize("order", ["index", "rank", "rank_local"])
def test_select_forms(dev, nk, order):
    from cast_amd import ops
    g = torch.Generator().manual_seed(nk)
    nq, max_k = 9, min(nk, 200)
    score = torch.randn(2, nq, nk, generator=g)
    score[:, ::2] = (score[:, ::2] * 2).round() / 2  # many equal scores
    score[0, 1, : nk // 2] = -float("inf")
    score[0, 3, nk - 1] = float("nan")
    forced = torch.rand(nq, nk, generator=g) < 0.02
    forced[4] = torch.rand(nk, generator=g) < 0.7  # more forced than selected
    allowed = torch.rand(nq, nk, generator=g) < 0.9
    k = torch.randint(0, max_k + 1, (nq,), generator=g)
    k[0], k[1] = max_k, 0
    for al in (None, allowed):
        idx, cnt = ops.select_topk(score.to(dev), k.to(dev), forced=forced.to(dev),
                                   allowed=None if al is None else al.to(dev), max_k=max_k,
                                   order=order)
        ref = score.clone()
        ref[torch.isnan(ref)] = float("inf")  # NaN ranks highest
        want = _want(ref, k, forced, al, order == "rank_local")
        idx, cnt = idx.cpu().reshape(-1, max_k), cnt.cpu().reshape(-1)
        for r, w in enumerate(want):
            w = sorted(w) if order == "index" else w
            assert int(cnt[r]) == len(w)
            assert idx[r].tolist() == w + [-1] * (max_k - len(w)), (r, order)


@pytest.mark.parametrize("nbh,nq,nk", [(24, 28, 130), (3, 130, 65), (2, 9, 40)])
def test_select_split_order(dev, nbh, nq, nk):
    """Rank order for the rows past the full rounds of an XCD's run, index order for the
    others (all, some and none of the rows)."""
    from cast_amd import ops
    g = torch.Generator().manual_seed(nk)
    score = torch.randn(nbh, nq, nk, generator=g).to(dev)
    forced = (torch.rand(nq, nk, generator=g) < 0.1).to(dev)
    k = torch.randint(0, 30, (nq,), generator=g).to(dev)
    args = dict(forced=forced, max_k=30)
    got, cnt = ops.select_topk(score, k, order="split", **args)
    rank, want_cnt = ops.select_topk(score, k, order="rank", **args)
    index, _ = ops.select_topk(score, k, order="index", **args)
    per = -(-nbh * nq // 8)
    cux = torch.cuda.get_device_properties(0).multi_processor_count // 8
    tail = (torch.arange(nbh * nq) % per >= per // cux * cux).view(nbh, nq, 1).to(dev)
    assert torch.equal(cnt, want_cnt)
    assert torch.equal(got, torch.where(tail, rank, index))


def test_select_check_sums(dev):
    from cast_amd import ops
    g = torch.Generator().manual_seed(3)
    nbh, nq, nk, mk = 5, 130, 201, 70
    sel = torch.randint(0, nk, (nbh, nq, mk), generator=g, dtype=torch.int32)
    sel[:, ::3, 5] = sel[:, ::3, 4]
    cnt = torch.randint(0, mk + 1, (nbh, nq), generator=g, dtype=torch.int32)
    local = torch.rand(nq, nk, generator=g) < 0.1
    score = torch.randn(nbh, nq, nk, generator=g)
    got = ops.select_check(sel.to(dev), cnt.to(dev), local.to(dev), score.to(dev)).cpu()
    live = torch.arange(mk) < cnt[..., None]
    dup = ((sel[..., 1:] == sel[..., :-1]) & live[..., 1:]).sum()
    kept = (torch.gather(local.expand(nbh, -1, -1), -1, sel.long()) & live).sum()
    assert int(got[0]) == int(dup) and int(got[1]) == int(kept)
    assert abs(float(got[2]) - float(score.double().sum())) < 1e-8


def test_select_overlapping_rows_take_the_packed_path(dev):
    """Rows a stride of zero apart and unequal dtypes still select as their copies."""
    from cast_amd.selector import BlockSelector
    g = torch.Generator().manual_seed(4)
    hw, shape, frames, nb = (8, 16), (4, 4, 8), 4, 4
    L = frames * hw[0] * hw[1]
    q = torch.randn(1, 2, L, 64, generator=g).to(dev)
    k = torch.randn(1, 2, 1, 64, generator=g).to(dev).expand(1, 2, L, 64)
    counts = torch.full((1, 1, nb), 4, dtype=torch.long)
    for kk, ref in ((k, k.contiguous()), (q.bfloat16(), None)):
        s = BlockSelector(shape, 4, nb)
        s.compile_budgets(token_h=hw[0], token_w=hw[1])
        args = dict(geometry_indices=None, geometry_counts=counts, latent_hw=hw,
                    block_shape=shape)
        got = s.select(q, kk, **args)
        if ref is not None:
            want = s.select(q, ref, **args)
            assert torch.equal(got[0], want[0])
        assert got[0].shape == (1, 2, nb, 4)
