"""The forward's q^ and k^, bit for bit: bf16(x * (1 / sqrt(sum x^2 + eps)))
with the sum a chain of fp32 fused multiply-adds per lane, then over the
lanes, and root, quotient and product correctly rounded (kernels.py:108-113).

The two are read off the outputs: with an identity state, no decay and beta =
0, o is q^; with a zero state, beta = 1 and v the first unit vector, one
token's final state holds k^ in its first row."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from kda_bt16 import forward_choice, kda_bt16_fwd

pytestmark = pytest.mark.gpu


def _unit(x: torch.Tensor) -> torch.Tensor:
    """The kernel's arithmetic in numpy: lane (row, q4) sums the columns
    16 * kt + 4 * q4 + i in order of kt, i.  The fused multiply-add is formed
    in 64 bits, where a bf16 square is exact."""
    f32 = np.float32
    a = x.float().numpy().reshape(-1, 8, 4, 4)  # [row, kt, q4, i]
    s = np.zeros((a.shape[0], 4), f32)
    for kt in range(8):
        for i in range(4):
            e = a[:, kt, :, i].astype(np.float64)
            s = (s.astype(np.float64) + e * e).astype(f32)
    s = (s[:, 0] + s[:, 1]) + (s[:, 2] + s[:, 3])
    rn = f32(1) / np.sqrt(s + f32(1e-6))
    return torch.from_numpy(a.reshape(-1, 128) * rn[:, None]).to(torch.bfloat16).reshape(x.shape)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("std", [1.0, 1e-3])  # 1e-3: eps counts beside the sum
def test_unit_vectors_bit_for_bit(fused, std, gpu_device):
    H, T, dev = 4, 333, gpu_device
    gen = torch.Generator().manual_seed(7)
    x = (std * torch.randn(1, T, H, 128, generator=gen)).bfloat16()
    kw = dict(scale=1.0, output_final_state=True, use_qk_l2norm_in_kernel=True, use_gate_in_kernel=False,
              use_beta_sigmoid_in_kernel=False)
    eye = torch.eye(128, device=dev).expand(1, H, 128, 128).contiguous()
    zero = torch.zeros(1, T, H, device=dev)
    with forward_choice(fused=fused):
        o, _ = kda_bt16_fwd(x.to(dev), x.to(dev), x.to(dev), torch.zeros(1, T, H, 128, device=dev), zero,
                            initial_state=eye, **kw)
        k1 = x.reshape(T, 1, H, 128).to(dev)  # one-token sequences
        v1 = torch.zeros_like(k1)
        v1[..., 0] = 1
        _, ht = kda_bt16_fwd(k1, k1, v1, torch.zeros(T, 1, H, 128, device=dev), torch.ones(T, 1, H, device=dev), **kw)
    want = _unit(x)
    assert torch.equal(o.cpu(), want)
    assert torch.equal(ht[:, :, 0, :].cpu(), want[0].float())
