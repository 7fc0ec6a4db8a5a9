"""GPU tests of the sibling x_hat passes in one launch (``svdq_act_xhat_siblings``): W4A16 sibling
linears against each layer by itself, bit for bit.  Row blocks of 64 and their remainders, one K group
up to several per split, ranks of one and two column tiles (one launch), of three, of unequal tiles and
with a LoRA adapter (a pass per layer), IEEE division.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _layers(dev, k, group, ranks, seed):
    from krea2_svdquant_amd.kernels.hip.backend import prepare_layer
    from krea2_svdquant_amd.runtime.krea2_standin import random_quantized_state
    gen = torch.Generator(device=dev).manual_seed(seed)
    return gen, [prepare_layer(random_quantized_state(n, k, rank=r, group_size=group, device=dev, generator=gen), (), dev)
                 for n, r in zip((512, 256, 320, 64), ranks)]


@pytest.mark.parametrize("m,k,group,ranks", [
    (1, 64, 64, (32, 32)),
    (63, 128, 128, (16, 32, 8, 32)),
    (65, 512, 64, (64, 48, 33, 64)),
    (130, 1088, 64, (32, 32, 32)),
    (1000, 6144, 128, (32, 32, 32, 32)),
    (77, 512, 64, (32, 64)),
    (77, 512, 64, (96, 96)),
    (64, 512, 64, (32,)),
])
@pytest.mark.parametrize("exact", [False, True])
def test_xhat_siblings_match_single_layers(dev, m, k, group, ranks, exact):
    from krea2_svdquant_amd.kernels.hip.backend import forward_prepared, forward_prepared_siblings
    print(f"x_hat siblings: M={m} K={k} G={group} ranks={ranks} exact={exact}", flush=True)
    gen, preps = _layers(dev, k, group, ranks, seed=m + k)
    x = torch.randn(m, k, device=dev, generator=gen).to(torch.bfloat16)
    x[0, :3] = torch.tensor([1e30, 1e-38, 0.0], dtype=torch.bfloat16)   # the division's range test
    for y, p in zip(forward_prepared_siblings(x, preps, mode="w4a16", exact_div=exact), preps):
        want = forward_prepared(x, p, mode="w4a16", exact_div=exact)
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))


def test_xhat_siblings_with_an_adapter(dev):
    from krea2_svdquant_amd.kernels.hip import ops
    gen, preps = _layers(dev, 512, 64, (32, 32), seed=9)
    x = torch.randn(70, 512, device=dev, generator=gen).to(torch.bfloat16)
    p = preps[0]
    down = (torch.randn(32, 512, device=dev, generator=gen) * 0.05).to(torch.bfloat16)
    mult = torch.full((32,), 0.5, device=dev)
    l1 = torch.cat((p.l1cat, (torch.randn(p.n, 32, device=dev, generator=gen) * 0.05).to(torch.bfloat16)), 1)
    args = (64, 64, *p.gemm_weights(ops.OPERAND_NONE), l1.contiguous(), None, ops.OPERAND_NONE, False, False)
    want = ops.linear(x, p.srs, p.l2, down, mult, *args)
    w, s = zip(*(q.gemm_weights(ops.OPERAND_NONE) for q in preps))
    got = ops.linear_siblings(x, [q.srs for q in preps], [q.l2 for q in preps], [down, None], [mult, None], 64,
                              [64, preps[1].rtp], list(w), list(s), [l1.contiguous(), preps[1].l1cat], [None, None],
                              ops.OPERAND_NONE, False, False)
    assert torch.equal(got[0], want)
