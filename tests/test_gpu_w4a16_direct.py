"""GPU tests of the W4A16 tiles that dequantize into MFMA operands (``w4a16_direct_kernel``).

Each output is the same chain of bf16 MFMAs as on the register-staged tiles
(``SVDQ_W4A16_KERNEL=wide``, 32768 columns here so that every M takes them): the same weights, 16
columns of K at a time, then the low-rank term, bias and store.  So the outputs are bit-identical on
every tile (``SVDQ_W4A16_TILES``), alone and as sibling layers.  Parity of the default path with the
oracle: ``test_gpu_kernels.py``, ``test_gpu_config2_shapes.py``.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

TILES = ["32x128", "64x128", "128x128", "192x128", "128x256"]


def _operands(dev, m, n, k, group, rank, seed):
    from krea2_svdquant_amd.kernels.hip import ops
    from krea2_svdquant_amd.kernels.hip.backend import prepare_layer
    from krea2_svdquant_amd.runtime.krea2_standin import random_quantized_state
    gen = torch.Generator(device=dev).manual_seed(seed)
    st = random_quantized_state(n, k, rank=rank, group_size=group, device=dev, generator=gen)
    p = prepare_layer(st, (), dev)
    x = torch.randn(m, k, device=dev, generator=gen).to(torch.bfloat16)
    _, _, _, xh, mid = ops.act_quant(x, p.srs, p.l2, None, None, group, p.rtp, -1, False, True, False)
    bias = (torch.randn(n, device=dev, generator=gen) * 0.1).to(torch.bfloat16)
    return xh, p.qweight, p.weight_scales, mid, p.l1cat, bias


# M around the tiles' 32 / 64 / 128 / 192 rows; N = 32768 and not a multiple of a tile or of 8; stages of 64
# columns: 1, fewer than the ring and the unrolled loop (8) hold, a partial slot of codes (4), many
@pytest.mark.parametrize("m,n,k,group,rank,out_f32", [
    (1, 32768, 64, 64, 32, False),
    (31, 32641, 128, 128, 32, True),
    (33, 32768, 192, 64, 64, False),
    (64, 32515, 320, 64, 96, False),
    (77, 32768, 384, 128, 64, True),
    (129, 32644, 512, 64, 32, False),
    (193, 32768, 576, 64, 32, True),
    (257, 32769, 640, 128, 128, False),
    (400, 32768, 1088, 64, 32, False),
])
def test_tiles_bit_identical_to_register_staged(dev, monkeypatch, m, n, k, group, rank, out_f32):
    from krea2_svdquant_amd.kernels.hip import ops
    print(f"w4a16 direct: M={m} N={n} K={k} G={group} r={rank} f32={out_f32}", flush=True)
    xh, qw, sw, mid, l1, bias = _operands(dev, m, n, k, group, rank, seed=m + k)
    monkeypatch.delenv("SVDQ_W4A16_TILES", raising=False)
    monkeypatch.setenv("SVDQ_W4A16_KERNEL", "wide")
    want = ops.w4a16_gemm(xh, qw, sw, mid, l1, bias, group, out_f32)
    monkeypatch.delenv("SVDQ_W4A16_KERNEL")
    assert torch.isfinite(want.float()).all()
    assert torch.equal(ops.w4a16_gemm(xh, qw, sw, mid, l1, bias, group, out_f32), want)
    for tile in TILES:
        monkeypatch.setenv("SVDQ_W4A16_TILES", tile)
        for _ in range(3):   # back to back: each launch's LDS starts as the one before left it
            got = ops.w4a16_gemm(xh, qw, sw, mid, l1, bias, group, out_f32)
            assert torch.equal(got, want), tile


@pytest.mark.parametrize("m,k,group", [(16, 256, 64), (77, 512, 128), (300, 320, 64)])
def test_siblings_bit_identical_to_single_layers(dev, monkeypatch, m, k, group):
    from krea2_svdquant_amd.kernels.hip import ops
    print(f"w4a16 direct siblings: M={m} K={k} G={group}", flush=True)
    layers = [_operands(dev, m, n, k, group, 32 * (1 + i % 2), seed=n) for i, n in enumerate((6144, 1536, 1531, 300))]
    xh, qw, sw, mid, l1, bias = map(list, zip(*layers))
    bias[1] = None
    for tile in [None] + TILES:
        monkeypatch.delenv("SVDQ_W4A16_TILES", raising=False)
        own = [ops.w4a16_gemm(*o, group, False) for o in zip(xh, qw, sw, mid, l1, bias)]
        if tile:
            monkeypatch.setenv("SVDQ_W4A16_TILES", tile)
        for got, want in zip(ops.w4a16_gemm_siblings(xh, qw, sw, mid, l1, bias, group, False), own):
            assert torch.equal(got, want), tile


@pytest.mark.parametrize("m,n,k,group,rank,out_f32", [
    (1, 130, 64, 64, 32, False), (127, 128, 128, 128, 256, True), (129, 257, 320, 64, 160, False),
    (300, 1000, 512, 64, 256, False), (513, 640, 1088, 64, 32, True)])
def test_every_kernel_bit_identical_on_small_grids(dev, monkeypatch, m, n, k, group, rank, out_f32):
    """Fewer than 128 tiles of 256 x 256: the 128 x 128 register-staged tiles and each other kernel, ranks
    up to eight chunks of 32."""
    from krea2_svdquant_amd.kernels.hip import ops
    print(f"w4a16 kernels: M={m} N={n} K={k} G={group} r={rank} f32={out_f32}", flush=True)
    o = _operands(dev, m, n, k, group, rank, seed=m + n)
    monkeypatch.delenv("SVDQ_W4A16_KERNEL", raising=False)
    monkeypatch.setenv("SVDQ_W4A16_TILES", "128x128staged")
    want = ops.w4a16_gemm(*o, group, out_f32)
    assert torch.isfinite(want.float()).all()
    for tile in [None, "192x256", "256x256"] + TILES:
        monkeypatch.delenv("SVDQ_W4A16_TILES", raising=False)
        if tile:
            monkeypatch.setenv("SVDQ_W4A16_TILES", tile)
        assert torch.equal(ops.w4a16_gemm(*o, group, out_f32), want), tile
