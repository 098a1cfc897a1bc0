"""A gate that forgets the state at a chunk's last token: the state after it
is that token's own update, however far its decay lies outside the fp32 range
of the chunk's recentred gates (g given as the chunk-local log2 cumsum, which
has no lower bound, kernels.py:673-674).

kg = bf16(k^ * 2^(G_last - G)) has an exponential of its own
(kernels.py:285-286): G_last - G is never positive, while the grams' factors
2^(G - G_mid) and 2^(G_mid - G) leave the range beyond 126 bits.
"""

from __future__ import annotations

import pytest
import torch

from kda_bt16 import forward_choice, kda_bt16_fwd
from kda_oracle import recurrent_gold
from kda_testlib import assert_close_rel

pytestmark = pytest.mark.gpu

T, H = 44, 2


@pytest.mark.parametrize("fused", [False, True])
# the last row of a full and of a partial chunk; 2^-126.5 is no normal number, 2^200 infinite
@pytest.mark.parametrize("at,bits", [(31, 126.5), (31, 200.0), (43, 126.5)])
def test_state_after_a_hard_decay(fused, at, bits, gpu_device):
    gen = torch.Generator().manual_seed(at)
    q, k, v = (torch.randn(1, T, H, 128, generator=gen).bfloat16() for _ in range(3))
    beta = torch.randn(1, T, H, generator=gen)
    h0 = 0.05 * torch.randn(1, H, 128, 128, generator=gen)
    d = -0.01 * torch.rand(1, T, H, 128, generator=gen)  # log2 decay of each token
    d[:, at] = -bits
    g = torch.cat([c.cumsum(1) for c in d.split(16, dim=1)], dim=1)
    with forward_choice(fused=fused):
        o, ht = kda_bt16_fwd(
            *(x.to(gpu_device) for x in (q, k, v, g, beta)), scale=0.1, initial_state=h0.to(gpu_device),
            output_final_state=True, use_qk_l2norm_in_kernel=True, use_gate_in_kernel=False,
            use_beta_sigmoid_in_kernel=True)
    o_gold, ht_gold = recurrent_gold(q, k, v, g, beta, 0.1, initial_state=h0, use_gate=False, dtype=torch.float64)
    # bf16 operands over fp32 sums: the bar of the reference's tests for the chunked path
    assert_close_rel("ht", ht_gold, ht, 0.01)
    rows = [t for t in range(T) if t != at]  # (the token's own o is outside the recentred gram's range)
    assert_close_rel("o", o_gold[:, rows], o[:, rows].float(), 0.01)
