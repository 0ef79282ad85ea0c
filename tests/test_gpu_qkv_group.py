"""rcsa_int8_linear_group and the row quantiser's register forms against the
oracle, bit for bit: both tile sizes, their remainders, K steps that do not fill
the copy ring, projections of unequal width, missing biases, fp32 outputs."""
import pytest
import torch

from oracle import rcsa_oracle as orc

pytestmark = pytest.mark.gpu


# 128 x 128 tiles (few tokens) and 256 x 256 tiles (many), rows at the tiles'
# edges; K of 1, 3, 4, 5 and 6 ring steps
@pytest.mark.parametrize("M,K,widths", [
    (1, 128, (256,)), (127, 384, (256, 512, 768)), (129, 512, (512, 256)),
    (257, 640, (256, 256, 256, 256)), (5633, 256, (3072, 3072, 3072)), (5887, 768, (3072, 512)),
])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_int8_linear_group_matches_oracle(dev, M, K, widths, out_dtype):
    from cast_amd import ops
    g = torch.Generator().manual_seed(M + K)
    x = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
    xs = torch.rand(M, generator=g) * 0.01 + 1e-4
    projs = []
    for i, n in enumerate(widths):
        w = torch.randint(-127, 128, (n, K), generator=g, dtype=torch.int8)
        bias = None if i == 1 else torch.randn(n, generator=g).bfloat16()
        projs.append((w, torch.rand(n, generator=g) * 0.01 + 1e-4, bias))
    print(f"int8 linear group {M} {K} {widths} {out_dtype}", flush=True)
    got = ops.int8_linear_group(
        x.to(dev), xs.to(dev), [tuple(t if t is None else t.to(dev) for t in p) for p in projs],
        out_dtype=out_dtype)
    torch.cuda.synchronize()
    for o, (w, ws, bias) in zip(got, projs):
        assert o.dtype == out_dtype
        assert torch.equal(o.cpu(), orc.int8_linear(x, xs, w, ws, bias).to(out_dtype))


def test_int8_linear_leaves_a_wide_output_alone(dev):
    """A view of a wider output: the columns past the projection stay as they were."""
    from cast_amd import ops
    g = torch.Generator().manual_seed(2)
    for M in (130, 5700):
        x = torch.randint(-127, 128, (M, 128), generator=g, dtype=torch.int8)
        w = torch.randint(-127, 128, (3072, 128), generator=g, dtype=torch.int8)
        xs, ws = torch.rand(M, generator=g), torch.rand(3072, generator=g)
        wide = torch.full((M + 3, 3072 + 8), 7.0, dtype=torch.bfloat16, device=dev)
        ops.int8_linear(x.to(dev), xs.to(dev), w.to(dev), ws.to(dev), out=wide[:M, :3072])
        wide = wide.cpu()
        assert torch.equal(wide[:M, :3072], orc.int8_linear(x, xs, w, ws, None))
        assert (wide[M:] == 7).all() and (wide[:, 3072:] == 7).all()


@pytest.mark.parametrize("stride", [(1 << 22) - 4, 1 << 22, (1 << 22) + 4])
def test_int8_linear_rows_far_apart(dev, stride):
    """Output rows on either side of the stride from which they go one by one."""
    from cast_amd import ops
    g = torch.Generator().manual_seed(3)
    M, N = 3, 512
    x = torch.randint(-127, 128, (M, 256), generator=g, dtype=torch.int8)
    w = torch.randint(-127, 128, (N, 256), generator=g, dtype=torch.int8)
    xs, ws = torch.rand(M, generator=g), torch.rand(N, generator=g)
    bias = torch.randn(N, generator=g).bfloat16()
    wide = torch.full((M, stride), 7.0, dtype=torch.bfloat16, device=dev)
    ops.int8_linear(x.to(dev), xs.to(dev), w.to(dev), ws.to(dev), bias.to(dev),
                    out=wide[:, :N])
    wide = wide.cpu()
    assert torch.equal(wide[:, :N], orc.int8_linear(x, xs, w, ws, bias))
    assert (wide[:, N:] == 7).all()


# the widest stride of a tile's own stores, and the first past it, in bytes: 8 MiB
@pytest.mark.parametrize("past", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N", [512, 49408])
def test_int8_linear_whole_tile_of_far_rows(dev, N, dtype, past):
    """All rows of a tile, 128 (few channels) and 256 (many: more than three rounds of the
    small tiles): the last of the 256 begins just below 2^31 bytes from the first."""
    from cast_amd import _lib
    g = torch.Generator().manual_seed(7)
    M = 256
    stride = (8 << 20) // dtype.itemsize - (0 if past else 4)
    x = torch.randint(-127, 128, (M, 128), generator=g, dtype=torch.int8)
    w = torch.randint(-127, 128, (N, 128), generator=g, dtype=torch.int8)
    xs, ws = torch.rand(M, generator=g), torch.rand(N, generator=g)
    bias = torch.randn(N, generator=g).bfloat16()
    print(f"int8 linear, {N} channels, rows {stride} of {dtype}", flush=True)
    wide = torch.full((M, stride), 7.0, dtype=dtype, device=dev)
    _lib.torch_ops().int8_linear_group(x.to(dev), xs.to(dev), [w.to(dev)], [ws.to(dev)],
                                       [bias.to(dev)], [wide[:, :N]])
    assert torch.equal(wide[:, :N].cpu(), orc.int8_linear(x, xs, w, ws, bias).to(dtype))
    assert bool((wide[:, N:] == 7).all())


@pytest.mark.parametrize("C", [8, 1016, 1032, 2048, 3064, 5120, 5128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_quantize_rows_lengths(dev, C, dtype):
    from cast_amd import ops
    g = torch.Generator().manual_seed(C)
    x = (torch.randn(37, C, generator=g) * torch.rand(37, 1, generator=g) * 4).to(dtype)
    x[5] = 0
    q, s = ops.quantize_rows_int8(x.to(dev))
    wq, ws = orc.quantize_rows_int8(x)
    assert torch.equal(q.cpu(), wq) and torch.equal(s.cpu(), ws)
