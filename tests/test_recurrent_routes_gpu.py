"""Which of the two token-recurrence kernels a call takes, on both sides of each
line, and that it gives the bits of its tokens' decode steps there."""

from __future__ import annotations

import pytest
import torch
from torch.profiler import ProfilerActivity, profile

from kda_bt16 import kda_decode_step, kda_recurrent_fwd

pytestmark = pytest.mark.gpu

WHOLE, ROWS = "recurrent_kernel", "recurrent_rows_kernel"
HV = 32


@pytest.mark.parametrize("N,T,vfirst,packed,kernel", [
    (8, 1, True, True, ROWS),      # 256 pairs: one round of either kernel
    (9, 1, True, True, WHOLE),     # one token each, packed: a serving step
    (20, 1, False, True, WHOLE),
    (20, 2, True, True, WHOLE),
    (20, 2, False, True, WHOLE),
    (24, 3, True, True, WHOLE),
    (10, 2, True, True, ROWS),     # 320 pairs
    (11, 2, False, False, WHOLE),
    (20, 3, True, False, ROWS),    # 640 pairs
    (28, 3, True, False, ROWS),    # 896: a second round with little in it
    (24, 8, False, False, WHOLE),  # 768 pairs, a full round
    (24, 9, False, False, ROWS),
    (28, 3, False, False, ROWS),
    (18, 5, False, False, WHOLE),  # K-first, the rows kernel's second batch of tokens
    (32, 5, False, False, ROWS),
    (36, 5, False, True, WHOLE),
    (88, 4, True, False, ROWS),    # 2816 pairs
    (90, 4, True, True, WHOLE),
    (36, 6, False, True, ROWS),
])
def test_route_and_bits(N, T, vfirst, packed, kernel, gpu_device):
    dev = gpu_device
    gen = torch.Generator(device=dev).manual_seed(N * T)

    def r(*s):
        return torch.randn(*s, generator=gen, device=dev)

    x = [r(N, T, HV, 128).bfloat16() for _ in range(4)] + [r(N, T, HV).bfloat16()]
    kw = dict(scale=0.1, use_qk_l2norm_in_kernel=True, use_gate_in_kernel=True, use_beta_sigmoid_in_kernel=True,
              lower_bound=-5.0, A_log=r(HV), dt_bias=0.1 * r(HV * 128), state_v_first=vfirst)
    h0 = 0.05 * r(N, HV, 128, 128)
    cu = torch.arange(0, N * T + 1, T, device=dev) if packed else None
    ins = [t.flatten(0, 1)[None] if packed else t for t in x]

    def call():
        return kda_recurrent_fwd(*ins, initial_state=h0, output_final_state=True, cu_seqlens=cu, **kw)

    call()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        o, ht = call()
        torch.cuda.synchronize()
    state = h0.clone()
    steps = [kda_decode_step(*(t[:, i:i + 1].contiguous() for t in x), state, **kw) for i in range(T)]
    assert torch.equal(o.reshape(N, T, HV, 128), torch.cat(steps, dim=1))
    assert torch.equal(ht, state)
    ran = [e.key for e in prof.key_averages() if "recurrent" in e.key]
    if not ran:
        pytest.skip("the profiler recorded no kernel")
    assert len(ran) == 1 and f"::{kernel}<" in ran[0], ran


def test_unequal_packed_sequences_take_the_rows(gpu_device):
    """Twenty sequences whose tokens are no multiple of them: a long one may be
    among them (here it is), and it runs row by row."""
    lens = [1] * 19 + [40]
    gen = torch.Generator(device=gpu_device).manual_seed(3)
    T = sum(lens)
    q, k, v, g = (torch.randn(1, T, HV, 128, generator=gen, device=gpu_device).bfloat16() for _ in range(4))
    beta = torch.randn(1, T, HV, generator=gen, device=gpu_device)
    cu = torch.tensor([0, *lens], device=gpu_device).cumsum(0)
    kw = dict(scale=0.1, use_qk_l2norm_in_kernel=True, use_gate_in_kernel=True, lower_bound=-5.0, output_final_state=True,
              A_log=torch.zeros(HV, device=gpu_device))
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        o, ht = kda_recurrent_fwd(q, k, v, g, beta, cu_seqlens=cu, **kw)
        torch.cuda.synchronize()
    o1, ht1 = kda_recurrent_fwd(*(t[:, 19:].contiguous() for t in (q, k, v, g, beta)), **kw)
    assert torch.equal(o[:, 19:], o1) and torch.equal(ht[19:], ht1)
    ran = [e.key for e in prof.key_averages() if "recurrent" in e.key]
    if not ran:
        pytest.skip("the profiler recorded no kernel")
    assert f"::{ROWS}<" in ran[0], ran
