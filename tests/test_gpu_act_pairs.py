"""GPU tests of the activation pass with groups of 128, whose halves go to a pair of waves: codes and
scales bit-exact against the oracle quantizer with odd and even group counts per split, values that
leave the smoothing's fast range in one half of a group only, and every rank tile count."""
import numpy as np
import pytest
import torch

from oracle import sim, synth
from .gpu_util import bf16_tensor, e3m2_codes_of, operand_bytes, sx_pairs_ok, to_device_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,rank,extreme", [(1, 128, 32, False), (3, 384, 64, False), (64, 640, 32, True),
                                              (65, 1280, 64, True), (130, 6144, 96, False), (700, 1920, 128, True)])
def test_codes_scales_and_down_projection(dev, m, k, rank, extreme):
    from krea2_svdquant_amd.kernels.hip import backend, ops
    x = synth.make_activation(m, k, seed=m + k)
    if extreme:   # one half of some groups below 2^-90, above 2^100, or zero
        x[:, 64:128] *= np.float32(2.0 ** -100)
        x[0, 256:320] = np.float32(2.0 ** 105)
        x[m // 2, 128:192] = 0.0
    st = synth.make_layer(64, k, np.clip(x, -100, 100), rank=rank, group_size=128, seed=3)
    prep = backend.prepare_layer(to_device_state(st, dev), (), dev)
    xd = bf16_tensor(x, dev)
    x_hat, _, sx_ref, codes = sim.quantize_activations(x, st)
    for fmt, op in (("e3m2", ops.OPERAND_E3M2), ("i8", ops.OPERAND_I8)):
        qa, sxp, _, _, mid = ops.act_quant(xd, prep.srs, prep.l2, None, None, 128, prep.rtp, op, False, False, False,
                                           True)
        got = qa.cpu().numpy()
        assert np.array_equal(e3m2_codes_of(got, m, k) if fmt == "e3m2" else got,
                              codes if fmt == "e3m2" else operand_bytes(codes, fmt))
        assert sx_pairs_ok(sxp, sx_ref)
        # f32 sums of K products in another order: K 2^-24 of the sum of magnitudes
        want = np.asarray(x_hat, np.float64) @ np.asarray(st.l2, np.float64).T
        bound = np.abs(np.asarray(x_hat, np.float64)) @ np.abs(np.asarray(st.l2, np.float64)).T * (k * 2.0 ** -24 + 2.0 ** -16)
        err = np.abs(ops.mid_values(mid).cpu().numpy()[:, :rank] - want)
        assert np.all(err <= bound + 1e-30)


# rank tiles of 32 split over launches: 4 (one launch up to M K = 3 << 20, then 2 + 2), 5 (2 + 3), 6 (3 + 3), 7 (3 + 4) and
# 9 (2 + 4 + 3), with and without LoRA tiles among the first
@pytest.mark.parametrize("m,k,r,rl", [(70, 1280, 128, 0), (700, 6144, 128, 0), (700, 6144, 32, 96), (65, 640, 160, 0),
                                      (129, 1280, 64, 128), (64, 640, 192, 32), (33, 384, 256, 32)])
@pytest.mark.parametrize("fmt,packed", [("e3m2", False), ("e3m2", True), ("i8", False), ("e4m3", False)])
def test_rank_tiles_over_launches(dev, m, k, r, rl, fmt, packed):
    """Codes and scales as with one rank tile; the down projections within the bound of sums of K
    products in any order."""
    from krea2_svdquant_amd.kernels.hip import ops
    print(f"rank tiles: M={m} K={k} r={r}+{rl} {fmt} packed={packed}", flush=True)
    gen = torch.Generator(device=dev).manual_seed(m + r)
    x = torch.randn(m, k, device=dev, generator=gen).to(torch.bfloat16)
    s = (torch.rand(k, device=dev, generator=gen) + 0.5).to(torch.bfloat16)
    srs = ops.prepare_smooth(s)
    l2 = (torch.randn(r, k, device=dev, generator=gen) * 0.05).to(torch.bfloat16)
    down = (torch.randn(rl, k, device=dev, generator=gen) * 0.05).to(torch.bfloat16) if rl else None
    mult = torch.linspace(0.5, 1.5, rl, device=dev) if rl else None
    op = ops.OPERAND_NAMES[fmt]
    one = ops.act_quant(x, srs, l2[:32].contiguous(), None, None, 128, 32, op, packed, False, False, True)
    got = ops.act_quant(x, srs, l2, down, mult, 128, ops.rank_padded(r + rl), op, packed, False, False, True)
    qa = [t.cpu().numpy() for t in (one[0], got[0])]
    if fmt == "e3m2":   # (an odd row count pads the planes with a row that is not written)
        qa = [e3m2_codes_of(t, m, k) for t in qa]
    assert np.array_equal(*qa) and all(torch.equal(a, b) for a, b in zip(one[1:3], got[1:3]))
    xh = (x.float() / s.float()).to(torch.bfloat16).double()
    want, mag = xh @ l2.double().T, xh.abs() @ l2.double().abs().T
    if rl:
        want = torch.cat((want, mult.double() * (x.double() @ down.double().T)), 1)
        mag = torch.cat((mag, mult.double() * (x.double().abs() @ down.double().abs().T)), 1)
    v = ops.mid_values(got[4]).double()
    assert bool(((v[:, : r + rl] - want).abs() <= mag * (k * 2.0 ** -24 + 2.0 ** -16)).all())
    assert not v[:, r + rl:].any()


@pytest.mark.parametrize("m", [4095, 4096, 4100])
def test_two_rank_tiles_around_the_prefetch_limit(dev, m):
    """Group 64, ranks 33-64: x is prefetched up to 4096 rows; the same codes, x_hat and sums either way, so
    the rows that both sides hold have the same bits (K = 256: one split for any M)."""
    from krea2_svdquant_amd.kernels.hip import ops
    gen = torch.Generator(device=dev).manual_seed(7)
    k = 256
    x = torch.randn(4100, k, device=dev, generator=gen).to(torch.bfloat16)
    srs = ops.prepare_smooth((torch.rand(k, device=dev, generator=gen) + 0.5).to(torch.bfloat16))
    l2 = (torch.randn(48, k, device=dev, generator=gen) * 0.05).to(torch.bfloat16)
    for op, xhat in ((ops.OPERAND_NONE, True), (ops.OPERAND_I8, False)):
        few = ops.act_quant(x[:64].contiguous(), srs, l2, None, None, 64, 64, op, False, xhat, False)
        got = ops.act_quant(x[:m].contiguous(), srs, l2, None, None, 64, 64, op, False, xhat, False)
        for i in (0, 1, 3):
            assert got[i].numel() == 0 or torch.equal(got[i][:64], few[i])
        assert torch.equal(ops.mid_values(got[4])[:64], ops.mid_values(few[4]))
