"""GPU tests of the W4A4 GEMM's small block tiles against the 256 x 128 tiles.

Every tile runs the same per-output arithmetic in the same order (exact group sums, exact scale
products, the rescale FMAs in group order, hi / lo low-rank products 16 ranks at a time, one bf16
rounding), so outputs must be bit-identical whatever the tile.  The 256 x 128 tiles are held to the
oracle by ``test_gpu_e3m2_shapes.py`` and ``test_gpu_kernels.py``.
"""
import pytest
import torch

from .test_gpu_wide_tiles import _tiles

pytestmark = pytest.mark.gpu

# (M, N, K, group, rank, bias): single rows and columns, tile edges and remainders in M and N, K of one
# group, of a part of a 256-column stage, of one stage, of 3-5 stages (the ring of four filling and
# wrapping) and of many; odd N (padded operand rows, element stores); ranks in one, two and three chunks
SHAPES = [(1, 1, 64, 64, 32, False), (1, 33, 128, 128, 32, True), (2, 31, 192, 64, 32, False),
          (31, 64, 256, 64, 64, True), (32, 65, 320, 64, 32, False), (33, 96, 512, 128, 32, False),
          (63, 127, 704, 64, 96, True), (64, 128, 768, 128, 64, False), (65, 129, 832, 64, 32, False),
          (97, 200, 1024, 64, 32, True), (127, 300, 1152, 128, 32, False), (129, 1000, 1280, 64, 64, False),
          (200, 264, 1792, 128, 32, True), (257, 1537, 6144, 64, 32, False), (77, 640, 16384, 128, 64, True)]


def _layer(dev, n, k, group, rank, bias):
    from krea2_svdquant_amd.kernels.hip import backend
    from krea2_svdquant_amd.runtime.krea2_standin import random_quantized_state
    gen = torch.Generator(device=dev).manual_seed(n + k)
    st = random_quantized_state(n, k, rank=rank, group_size=group, device=dev, generator=gen)
    if bias:
        st.bias = torch.randn(n, device=dev, generator=gen).to(torch.bfloat16)
    return backend.prepare_layer(st, (), dev)


def _x(dev, m, k, seed=5):
    gen = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(m, k, device=dev, generator=gen)
    x[:, ::53] *= 20
    return x.to(torch.bfloat16)


@pytest.mark.parametrize("out_f32", [False, True])
@pytest.mark.parametrize("m,n,k,group,rank,bias", SHAPES)
def test_small_tiles_bit_identical(dev, m, n, k, group, rank, bias, out_f32):
    from krea2_svdquant_amd.kernels.hip.backend import forward_prepared
    prep, x = _layer(dev, n, k, group, rank, bias), _x(dev, m, k)
    with _tiles("256x128"):
        want = forward_prepared(x, prep, out_f32=out_f32)
    assert torch.isfinite(want.float()).all()
    for tile in ("32x32", "64x64", "128x64"):
        with _tiles(tile):
            got = forward_prepared(x, prep, out_f32=out_f32)
        assert torch.equal(got, want), tile
    assert torch.equal(forward_prepared(x, prep, out_f32=out_f32), want)


@pytest.mark.parametrize("m,k", [(48, 1536), (70, 320)])
def test_small_tiles_siblings(dev, m, k):
    """Sibling layers in one launch of small tiles, at any K, against a launch per layer."""
    from krea2_svdquant_amd.kernels.hip.backend import forward_prepared, forward_prepared_siblings
    preps = [_layer(dev, n, k, 64, rank, False) for n, rank in ((300, 32), (64, 64), (129, 32))]
    x = _x(dev, m, k)
    with _tiles("256x128"):
        want = [forward_prepared(x, p) for p in preps]
    for tile in ("32x32", "64x64", "128x64", "auto"):
        with _tiles(tile):
            got = forward_prepared_siblings(x, preps)
        for g, w in zip(got, want):
            assert torch.equal(g, w), tile


@pytest.mark.parametrize("m,n,k,group,rank", [(40, 100, 256, 64, 160), (65, 192, 512, 128, 256), (130, 300, 320, 64, 288)])
def test_small_tiles_large_ranks(dev, m, n, k, group, rank):
    from krea2_svdquant_amd.kernels.hip.backend import forward_prepared
    prep, x = _layer(dev, n, k, group, rank, True), _x(dev, m, k)
    with _tiles("256x128"):
        want = forward_prepared(x, prep)
    for tile in ("32x32", "64x64", "128x64", "auto"):
        with _tiles(tile):
            assert torch.equal(forward_prepared(x, prep), want), tile
