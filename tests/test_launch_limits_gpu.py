"""Launches whose threads exceed 2^32: packed calls of more sequences than
2^32 threads of one dimension hold at the kernel's threads a sequence, nearly
all of them empty."""

from __future__ import annotations

import pytest
import torch

from kda_bt16 import kda_bt16_fwd, kda_recurrent_fwd

pytestmark = pytest.mark.gpu


def _packed(n, dev):
    """n sequences, four of which have tokens (3, 17, 2, 21 of them), among them
    the first and the last; and the call on those four alone."""
    at, lens = torch.tensor([0, 5, n - 4096, n - 1]), torch.tensor([3, 17, 2, 21])
    gen = torch.Generator(device=dev).manual_seed(n)
    T = int(lens.sum())
    x = [torch.randn(1, T, 1, 128, generator=gen, device=dev).bfloat16() for _ in range(4)]
    x.append(torch.randn(1, T, 1, generator=gen, device=dev))
    size = torch.zeros(n + 1, dtype=torch.int64)
    size[at + 1] = lens
    few = torch.cat([torch.zeros(1, dtype=torch.int64), lens.cumsum(0)])
    kw = dict(scale=0.1, use_qk_l2norm_in_kernel=True, use_gate_in_kernel=True, use_beta_sigmoid_in_kernel=True,
              lower_bound=-5.0, A_log=torch.zeros(1, device=dev))
    return x, size.cumsum(0).to(dev), few.to(dev), kw


@pytest.mark.parametrize("vfirst", [True, False])
def test_recurrence_over_more_than_2_pow_22_sequences(vfirst, gpu_device):
    # two work-groups of 512 threads a sequence: 2^22 of them are 2^32 threads
    x, cu, few, kw = _packed((1 << 22) + 4096, gpu_device)
    o, _ = kda_recurrent_fwd(*x, cu_seqlens=cu, state_v_first=vfirst, **kw)
    want, _ = kda_recurrent_fwd(*x, cu_seqlens=few, state_v_first=vfirst, **kw)
    assert torch.isfinite(want).all()
    assert torch.equal(o, want)


def test_fused_forward_over_more_sequences_than_2_pow_32_threads(gpu_device):
    # one work-group of 768 threads a sequence
    x, cu, few, kw = _packed((1 << 32) // 768 + 4096, gpu_device)
    o, _ = kda_bt16_fwd(*x, cu_seqlens=cu, use_fused_kernel=True, **kw)
    want, _ = kda_bt16_fwd(*x, cu_seqlens=few, use_fused_kernel=True, **kw)
    assert torch.isfinite(want).all()
    assert torch.equal(o, want)
