"""The many-workgroups form of the attention's other block shapes (head_dim 64 or
64-row / 64-key blocks), which needs two rounds of query blocks per XCD, and key
validity bits set past K_LEN, in a last block whose later steps lie past it.

Tolerances of the other attention tests (test_gpu_attn_forms)."""
import pytest
import torch

from oracle import rcsa_oracle as orc

pytestmark = pytest.mark.gpu

SHAPES = [(128, 128, 64), (128, 64, 128), (128, 64, 64), (64, 128, 128), (64, 128, 64),
          (64, 64, 128), (64, 64, 64)]


@pytest.mark.parametrize("int8", [True, False])
@pytest.mark.parametrize("D,bm,bn", SHAPES)
def test_many_form_matches_oracle(dev, D, bm, bn, int8):
    from cast_amd import ops
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    nqb, nkb, kmax = 32, 5, 4
    H = -(-2 * cus // nqb)
    g = torch.Generator().manual_seed(D + 2 * bm + 4 * bn + int(int8))
    lq, lk = nqb * bm - 9, nkb * bn - bn + 7  # the last key block holds seven keys
    idx = torch.rand(1, H, nqb, nkb, generator=g).argsort(-1)[..., :kmax].int().contiguous()
    cnt = torch.randint(0, kmax + 1, (1, H, nqb), generator=g, dtype=torch.int32)
    kv = torch.rand(lk, generator=g) < 0.9
    wide = torch.ones(nkb * bn, dtype=torch.bool)  # the bits past K_LEN are set
    wide[:lk] = kv
    v = torch.randn(1, H, lk, D, generator=g).bfloat16()
    print(f"attention shapes: {D} {bm} {bn} int8 {int8}", flush=True)
    if int8:
        q8 = torch.randint(-127, 128, (1, H, lq, D), generator=g, dtype=torch.int8)
        k8 = torch.randint(-127, 128, (1, H, lk, D), generator=g, dtype=torch.int8)
        qs = torch.rand(H, nqb, generator=g) * 0.02 + 0.005
        ks = torch.rand(H, nkb, generator=g) * 0.02 + 0.005
        q = q8.float() * qs[:, torch.arange(lq) // bm][None, :, :, None]
        k = k8.float() * ks[:, torch.arange(lk) // bn][None, :, :, None]

        def run(**kw):
            return ops.sparse_attn_int8(q8.to(dev), qs.to(dev), k8.to(dev), ks.to(dev), v.to(dev),
                                        idx.to(dev), cnt.to(dev), block_m=bm, block_n=bn,
                                        return_lse=True, **kw)
        cos_min, rel = 0.9999, 5e-3
    else:
        q, k = (torch.randn(1, H, n, D, generator=g).bfloat16() for n in (lq, lk))

        def run(**kw):
            return ops.sparse_attn_bf16(q.to(dev), k.to(dev), v.to(dev), idx.to(dev),
                                        cnt.to(dev), block_m=bm, block_n=bn, return_lse=True,
                                        **kw)
        cos_min, rel = 0.999, 1e-2
    ref, rlse = orc.sparse_attention(q.float(), k.float(), v.float(), idx, cnt, kv, block_m=bm,
                                     block_n=bn)
    for kw in (dict(block_mask=ops.valid_bits(wide.to(dev), bn)), dict(valid=kv.to(dev))):
        out, lse = run(**kw)
        st = orc.equivalence_stats(ref, out.float().cpu())
        assert st["cosine"] >= cos_min and st["max_abs"] <= 3e-2 and st["relative_l2"] <= rel, st
        fin = torch.isfinite(rlse)
        assert torch.equal(fin, torch.isfinite(lse.cpu()))
        torch.testing.assert_close(lse.cpu()[fin], rlse[fin], atol=2e-2, rtol=0)


@pytest.mark.parametrize("int8", [True, False])
def test_bits_past_the_keys_are_ignored(dev, int8):
    """D 128, 128 x 128 blocks, both forms: set bits past K_LEN change nothing."""
    from cast_amd import ops
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    g = torch.Generator().manual_seed(5)
    for H in (1, -(-2 * cus // 32)):
        lq, lk = 32 * 128, 3 * 128 + 5
        v = torch.randn(1, H, lk, 128, generator=g).bfloat16().to(dev)
        idx = torch.tensor([3, 0], dtype=torch.int32).expand(1, H, 32, 2).contiguous().to(dev)
        cnt = torch.full((1, H, 32), 2, dtype=torch.int32, device=dev)
        outs = []
        for past in (True, False):
            flags = torch.full((4 * 128,), past)
            flags[:lk] = True
            kw = dict(block_mask=ops.valid_bits(flags.to(dev), 128))
            if int8:
                gg = torch.Generator().manual_seed(6)
                q8, k8 = (torch.randint(-127, 128, (1, H, n, 128), generator=gg,
                                        dtype=torch.int8).to(dev) for n in (lq, lk))
                outs.append(ops.sparse_attn_int8(q8, torch.full((H, 32), 0.01, device=dev), k8,
                                                 torch.full((H, 4), 0.01, device=dev), v, idx,
                                                 cnt, **kw))
            else:
                gg = torch.Generator().manual_seed(6)
                q, k = (torch.randn(1, H, n, 128, generator=gg).bfloat16().to(dev)
                        for n in (lq, lk))
                outs.append(ops.sparse_attn_bf16(q, k, v, idx, cnt, **kw))
        assert torch.equal(*outs)
