"""GPU tests of the attention's last round of workgroups: items cut into key pieces where there is
room for two of each, whole items otherwise (``svdq_attn.hip``, ``attn_plan``).

The workspace tells which it is: 16 bytes of flags per item, and more than that only with pieces.
48 query heads over 256-query items; tolerance as in ``test_gpu_attention.py``.
"""
import math

import pytest
import torch

from tests.test_gpu_attention import _check, _fast_flags, _inputs

pytestmark = pytest.mark.gpu


def _in_pieces(t, heads):
    from krea2_svdquant_amd.kernels.hip import lib
    return lib.load().svdq_attention_workspace(t, heads) > 16 * heads * ((t + 255) // 256)


@pytest.mark.parametrize("t,pieces", [
    (1, False),       # a single key
    (64, False),      # one key tile: nothing to cut
    (65, True),       # two pieces, the second of one key
    (448, True),      # 7 tiles in two pieces
    (449, True),
    (512, True),
    (513, False),     # 144 items: no room for two pieces
    (1279, False),    # 240 items, a partial key tile and query block
    (1281, True),     # one whole round and 32 items in 8 pieces
])
def test_last_round_matches_float32(dev, t, pieces):
    print(f"attention round: T={t}", flush=True)
    assert _in_pieces(t, 48) == pieces
    _check(*_inputs(t, 48, 12, dev, seed=t))


@pytest.mark.parametrize("t,pieces", [(64, False), (300, True), (512, True), (700, False)])
def test_overflowing_products_hand_over(dev, t, pieces):
    """Keys 32.. score 56 log2 units above the first 32 (the fixed exponent offset) and every v is
    2^73: p v passes the f32 range while the row sum stays below 2^64.  The waves hand over to the
    running-maximum kernel, and the average of equal values is exact."""
    assert _in_pieces(t, 48) == pieces
    q = torch.ones(t, 48, 128, device=dev, dtype=torch.bfloat16)
    k = torch.full((t, 12, 128), 56.0 * math.log(2.0) * math.sqrt(128) / 128, device=dev)
    k[:32] = 0.0
    v = torch.full((t, 12, 128), 2.0 ** 73, device=dev, dtype=torch.bfloat16)
    out, flags = _fast_flags(q, k.to(torch.bfloat16), v, 1.0 / math.sqrt(128))
    assert bool((flags[:, : (t + 63) // 64] == 1).all())
    assert torch.equal(out, torch.full_like(out, 2.0 ** 73))
