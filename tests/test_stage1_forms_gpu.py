"""Stage 1 forms the forward's records in one pass over the columns or in
passes of their own, by the launch's chunks: the two-stage forward on both
sides of each line against the fused one (always one pass), bit for bit."""

from __future__ import annotations

import pytest
import torch

from kda_bt16 import chunk_kda, forward_choice

pytestmark = pytest.mark.gpu


def _both(B, T, H, lens, gate_dtype, dev):
    gen = torch.Generator(device=dev).manual_seed(T)

    def r(*s):
        return torch.randn(*s, generator=gen, device=dev)

    q, k, v = (r(B, T, H, 128).bfloat16() for _ in range(3))
    g, beta = r(B, T, H, 128).to(gate_dtype), r(B, T, H).to(gate_dtype)
    cu = None
    if lens:
        cu = torch.tensor([0, *lens], device=dev).cumsum(0)
    kw = dict(scale=0.1, initial_state=0.05 * r(len(lens) if lens else B, H, 128, 128), output_final_state=True,
              use_qk_l2norm_in_kernel=True, use_gate_in_kernel=True, use_beta_sigmoid_in_kernel=True, safe_gate=True,
              lower_bound=-5.0, A_log=r(H), dt_bias=0.1 * r(H * 128), state_v_first=True, cu_seqlens=cu)
    for fused in (False, True):
        with forward_choice(fused=fused):
            yield chunk_kda(q, k, v, g, beta, **kw)


# chunks = 16 rows x H heads x T / 16, or, packed, H x (T / 16 + sequences)
@pytest.mark.parametrize("B,T,H,lens,gate_dtype", [
    (16, 240, 16, (), torch.bfloat16),    # 3840 whole chunks
    (16, 256, 16, (), torch.bfloat16),    # 4096
    (16, 448, 16, (), torch.bfloat16),    # 7168
    (16, 464, 16, (), torch.bfloat16),    # 7424
    (16, 448, 16, (), torch.float32),
    (16, 255, 12, (), torch.bfloat16),    # 3072, the last of each row partial
    (16, 257, 12, (), torch.bfloat16),    # 3264
    (16, 767, 12, (), torch.bfloat16),    # 9216
    (16, 769, 12, (), torch.bfloat16),    # 9408
    (1, 2960, 16, (1000, 0, 17, 5, 16, 1922, 0), torch.bfloat16),  # 3072 slots, gaps among them
    (1, 2976, 16, (1000, 0, 33, 5, 16, 1922, 0), torch.bfloat16),  # 3088
    (1, 2976, 16, (1000, 0, 33, 5, 16, 1922, 0), torch.float32),
])
def test_either_form_gives_the_same_bits(B, T, H, lens, gate_dtype, gpu_device):
    (o, ht), (o_fused, ht_fused) = _both(B, T, H, lens, gate_dtype, gpu_device)
    assert torch.isfinite(o).all() and torch.isfinite(ht).all()
    assert torch.equal(o, o_fused)
    assert torch.equal(ht, ht_fused)
