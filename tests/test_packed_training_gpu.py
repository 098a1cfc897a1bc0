"""A training step over packed sequences against one step per sequence, where
the (sequence, head) pairs outnumber the CUs' eighths: stage 2 and the reverse
chain then take the sequences longest first (up to 64 of them), and each must
be taken once.  o, ht and every gradient of an input bit for bit; the gradients
of A_log and dt_bias, sums over the sequences in another order, to 1e-5."""

from __future__ import annotations

import pytest
import torch

from kda_bt16 import chunk_kda, set_backward_recompute

pytestmark = pytest.mark.gpu

CASES = {
    # ties, empty ones, the longest in the middle; 35 pairs, no multiple of 8
    "n7_h5": (5, 5, [33, 0, 17, 257, 17, 64, 33]),
    "n7_h3_hv6": (3, 6, [1, 128, 0, 128, 300, 16, 5]),
    # more than 64 sequences: in their own order
    "n70_h1": (1, 1, [7 + 13 * (i % 9) if i % 11 else 0 for i in range(70)]),
}


def _step(x, par, h0, do, dht, cu):
    x = [t.detach().requires_grad_(True) for t in x]
    par = [t.detach().requires_grad_(True) for t in par]
    h0 = h0.detach().requires_grad_(True)
    o, ht = chunk_kda(*x, scale=0.1, initial_state=h0, output_final_state=True, use_qk_l2norm_in_kernel=True,
                      use_gate_in_kernel=True, use_beta_sigmoid_in_kernel=True, safe_gate=True, lower_bound=-5.0,
                      A_log=par[0], dt_bias=par[1], state_v_first=True, cu_seqlens=cu)
    grads = torch.autograd.grad([o, ht], [*x, h0, *par], [do, dht])
    return [o.detach(), ht.detach(), *grads]


@pytest.mark.parametrize("recompute", [False, True])
@pytest.mark.parametrize("name", list(CASES))
def test_packed_step_equals_one_step_per_sequence(name, recompute, gpu_device):
    H, HV, lens = CASES[name]
    dev, T, N = gpu_device, sum(lens), len(lens)
    assert N * HV * 8 > 256
    gen = torch.Generator(device=dev).manual_seed(T)

    def r(*s):
        return torch.randn(*s, generator=gen, device=dev)

    x = [r(1, T, H, 128).bfloat16(), r(1, T, H, 128).bfloat16(), r(1, T, HV, 128).bfloat16(),
         r(1, T, HV, 128).bfloat16(), r(1, T, HV)]
    par = [torch.log(1 + 15 * torch.rand(HV, generator=gen, device=dev)), 0.1 * r(HV * 128)]
    h0, do, dht = 0.05 * r(N, HV, 128, 128), r(1, T, HV, 128).bfloat16(), 0.1 * r(N, HV, 128, 128)
    cu = torch.tensor([0, *lens], device=dev).cumsum(0)
    set_backward_recompute(recompute)
    try:
        got = _step(x, par, h0, do, dht, cu)
        each, at = [], 0
        for n, size in enumerate(lens):
            rows, at = slice(at, at + size), at + size
            if size == 0:
                assert torch.equal(got[1][n], h0[n]) and torch.equal(got[7][n], dht[n])
                continue
            one = _step([t[:, rows].contiguous() for t in x], par, h0[n:n + 1], do[:, rows].contiguous(),
                        dht[n:n + 1], None)
            each.append((n, rows, one))
    finally:
        set_backward_recompute(False)
    names = ("o", "ht", "dq", "dk", "dv", "dg", "dbeta", "dh0")
    for n, rows, one in each:
        for i, what in enumerate(names):
            mine = got[i][n:n + 1] if what in ("ht", "dh0") else got[i][:, rows]
            assert torch.equal(mine, one[i]), (n, what)
    for i in (8, 9):
        want = torch.stack([one[i].double() for _, _, one in each]).sum(0)
        err = (got[i].double() - want).norm() / want.norm()
        assert err < 1e-5, (i, err)
