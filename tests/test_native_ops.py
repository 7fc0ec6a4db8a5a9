"""The native operators svdq::linear and svdq::linear_siblings: shape functions on the CPU; on the GPU
the same bits as the activation and GEMM operators they replace, the same refusals, and no silent
gradient."""
import pytest
import torch

from krea2_svdquant_amd.kernels.hip import lib, ops


@pytest.mark.skipif(not lib.TORCH_LIB_PATH.exists(), reason="library not built")
def test_shape_functions():
    from torch._subclasses.fake_tensor import FakeTensorMode
    ops.load_native()
    with FakeTensorMode():
        x = torch.empty(2, 3, 128, dtype=torch.bfloat16)
        l1 = torch.empty(40, 32, dtype=torch.bfloat16)
        y = ops.linear(x, x, x, None, None, 64, 32, x, x, l1, None, ops.OPERAND_E3M2, False, False)
        assert y.shape == (2, 3, 40) and y.dtype == torch.bfloat16
        ys = ops.linear_siblings(x, [x, x], [x, x], [None, None], [None, None], 64, [32, 32], [x, x], [x, x], [l1, l1],
                                 [None, None], ops.OPERAND_NONE, True, False)
        assert [t.shape for t in ys] == [(2, 3, 40)] * 2 and ys[0].dtype == torch.float32


def _prepared(dev, n, k, group, lora=0):
    from krea2_svdquant_amd.kernels.hip import backend
    from krea2_svdquant_amd.runtime.krea2_standin import random_quantized_state
    from krea2_svdquant_amd.runtime.linear import SVDQuantLoRAAdapter
    gen = torch.Generator(device=dev).manual_seed(n)
    st = random_quantized_state(n, k, rank=32, group_size=group, device=dev, generator=gen)
    st.bias = torch.randn(n, device=dev, generator=gen).to(torch.bfloat16)
    ads = []
    if lora:
        ads = [SVDQuantLoRAAdapter(torch.randn(lora, k, device=dev, generator=gen).to(torch.bfloat16) * 0.02,
                                   torch.randn(n, lora, device=dev, generator=gen).to(torch.bfloat16) * 0.02)]
    return backend.prepare_layer(st, ads, dev)


@pytest.mark.gpu
@pytest.mark.parametrize("group,operand,k,lora", [(64, "e3m2", 320, 0), (64, "e4m3", 256, 16), (128, "i8", 256, 0),
                                                  (32, "i8", 192, 0), (64, None, 320, 16), (128, None, 256, 0)])
def test_linear_is_the_two_operators(dev, group, operand, k, lora):
    from krea2_svdquant_amd.kernels.hip.backend import forward_prepared, forward_prepared_siblings
    p = _prepared(dev, 72, k, group, lora)
    x = torch.randn(5, 7, k, device=dev).to(torch.bfloat16)
    x2 = x.reshape(35, k)
    fast = group in (64, 128)
    if operand is None:
        _, _, _, xhat, mid = ops.act_quant(x2, p.srs, p.l2, p.lora_down, p.lora_mult, group, p.rtp, ops.OPERAND_NONE,
                                           False, True, False)
        want = ops.w4a16_gemm(xhat, p.qweight, p.weight_scales, mid, p.l1cat, p.bias, group, False)
    else:
        opc = ops.OPERAND_NAMES[operand]
        qa, sx, _, _, mid = ops.act_quant(x2, p.srs, p.l2, p.lora_down, p.lora_mult, group, p.rtp, opc, False,
                                          not fast, False, True)
        want = ops.w4a4_gemm(qa, sx, p.weight_operand(opc), p.weight_scale_pairs(opc), mid, p.l1cat, p.bias, group,
                             opc, False)
    kw = {"mode": "w4a16"} if operand is None else {"operand": operand}
    y = forward_prepared(x, p, **kw)
    assert y.shape == (5, 7, 72) and torch.equal(y.reshape(35, 72), want)
    assert torch.equal(forward_prepared(x.transpose(0, 1), p, **kw), y.transpose(0, 1))   # any strides
    if fast:
        for z in forward_prepared_siblings(x, [p, p], **kw):
            assert torch.equal(z, y)


@pytest.mark.gpu
def test_refusals(dev):
    from krea2_svdquant_amd.kernels.hip.backend import forward_prepared
    p = _prepared(dev, 72, 256, 64)
    flat = torch.randn(257 * 4 + 1, device=dev).to(torch.bfloat16)
    with pytest.raises(lib.SVDQError) as e:   # contiguous rows that do not start on 16 bytes
        forward_prepared(flat[1:1 + 4 * 256].view(4, 256), p)
    assert e.value.status == -3
    with pytest.raises(lib.SVDQError):
        forward_prepared(flat[:0].view(0, 256), p)
    with pytest.raises(ValueError):
        forward_prepared(torch.zeros(4, 320, device=dev, dtype=torch.bfloat16), p)
    with pytest.raises(ValueError):
        forward_prepared(torch.zeros(256, device=dev, dtype=torch.bfloat16), p)
    with pytest.raises(TypeError):
        forward_prepared(torch.zeros(4, 256, device=dev), p)
    x = torch.randn(4, 256, device=dev).to(torch.bfloat16).requires_grad_()
    with pytest.raises(RuntimeError):
        forward_prepared(x, p).sum().backward()


@pytest.mark.skipif(not lib.TORCH_LIB_PATH.exists(), reason="library not built")
def test_operators_of_another_torch_are_refused_before_loading(tmp_path, monkeypatch):
    mark = b"svdq_torch built with torch "
    data = lib.TORCH_LIB_PATH.read_bytes()
    assert mark + torch.__version__.encode() + b"\0" in data
    other = tmp_path / "libsvdq_torch.so"
    monkeypatch.setattr(lib, "TORCH_LIB_PATH", other)
    monkeypatch.setattr(torch.ops, "load_library", lambda path: pytest.fail("loaded"))
    for content, needle in ((data.replace(mark + torch.__version__[:1].encode(), mark + b"0"), "built with torch 0"),
                            (data.replace(mark, b"x" * len(mark)), "built with torch unknown")):
        other.write_bytes(content)
        with pytest.raises(RuntimeError, match=needle):
            lib.load_torch_ops()
