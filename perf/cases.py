"""What a user of this package has it do, as cases to time and to compare.

Every case is one pass through the public entry points (``kda_bt16_fwd``,
``chunk_kda`` and its autograd, ``fused_recurrent_kda``, ``kda_decode_step``)
on inputs of the shapes and distributions that the tests and ``bench.py``
use: bf16 q, k, v ~ N(0, 1); the raw gate ~ N(0, 1) or N(0, 2); raw beta
~ N(0, 1); A_log = log U(1, 16); dt_bias std 0.1; states std 0.05.

A case is a dict of plain values:

* ``path``: ``fwd`` (``kda_bt16_fwd``), ``chunk`` (``chunk_kda``, FLA's
  convention), ``train`` (``chunk_kda`` and its backward), ``recurrent``
  (``fused_recurrent_kda``) or ``decode`` (``kda_decode_step``);
* ``B, T, H, HV``: batch rows, tokens, q/k heads and value heads;
* ``lens``: lengths of the packed sequences (B = 1), or "" for batch rows;
* ``gdtype``: the dtype of g and beta, ``bf16`` or ``f32``;
* ``gate``: ``kernel`` (raw gate, A_log, dt_bias) or ``log`` (g is the
  per-token log decay);
* ``gstd``: the raw gate's standard deviation;
* ``h0``: whether there is an initial state;
* ``v_first``: the state layout.
"""

from __future__ import annotations

import math
import os
import sys

import torch
import torch.utils.checkpoint

for _p in (os.path.join(os.getcwd(), "kda-ascendc_amd"),):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import kda_bt16  # noqa: E402

D = 128  # K = V, the head size the kernels serve
LOWER_BOUND = -5.0
SCALE = D ** -0.5
L2_EPS = 1e-6


def _case(name, path, B, T, H, HV=None, lens="", gdtype="bf16", gate="kernel", gstd=1.0, h0=False,
          v_first=True):
    c = {"path": path, "B": B, "T": T, "H": H, "HV": HV or H, "lens": lens, "gdtype": gdtype,
         "gate": gate, "gstd": gstd, "h0": h0, "v_first": v_first}
    return {"name": name, **c} if name else c


def listed():
    return [
        # One decode step of a single conversation: the smallest call, where
        # the launch and the host path count.
        _case("decode_b1", "decode", 1, 1, 32, h0=True),
        # One decode step of a full serving batch: the state streamed once
        # each way.
        _case("decode_b128", "decode", 128, 1, 32, h0=True),
        # A few tokens at once from a kept state (a draft to verify, the tail
        # of a prompt), in FLA's default K-first layout.
        _case("recurrent_t24", "recurrent", 4, 24, 16, h0=True, v_first=False),
        # A short prompt batch on a small model (or one rank's few heads).
        _case("fwd_b2_t1024_h4", "fwd", 2, 1024, 4, h0=True),
        # A ragged prompt with grouped value heads, fp32 gate and beta.
        _case("chunk_t3001_h8_hv16", "chunk", 1, 3001, 8, HV=16, gdtype="f32", v_first=False),
        # Two medium prompts continued from a state.
        _case("fwd_b2_t4096_h8", "fwd", 2, 4096, 8, h0=True),
        # Packed prefill: 16 prompts of uneven lengths in 8192 tokens.
        _case("chunk_packed16_t8192_h32", "chunk", 1, 8192, 32,
              lens="611,212,505,377,1403,148,540,731,66,818,459,283,640,512,475,412"),
        # The headline: one long prompt, 32 heads.
        _case("fwd_b1_t8192_h32", "fwd", 1, 8192, 32),
        # The same length with 96 heads.
        _case("fwd_b1_t8192_h96", "fwd", 1, 8192, 96),
        # Batched prefill continued from states, a wide gate: the largest.
        _case("fwd_b16_t2048_h32", "fwd", 16, 2048, 32, gstd=2.0, h0=True),
        # A training step over packed, ragged documents with grouped heads.
        _case("train_packed6_t4000_h8_hv16", "train", 1, 4000, 8, HV=16,
              lens="1311,97,640,1024,33,895", v_first=False),
        # A training step at the headline shape.
        _case("train_b1_t8192_h32", "train", 1, 8192, 32),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["fwd", "fwd", "chunk", "chunk", "train", "train", "decode", "recurrent"])
    gdtype = rng.choice(["bf16", "bf16", "f32"])
    v_first = rng.random() < 0.5
    h0 = rng.random() < 0.5
    gate = "kernel" if path in ("fwd", "decode") or rng.random() < 0.8 else "log"
    if path == "decode":
        return _case("", path, _log_int(rng, 1, 128), 1, rng.choice([8, 16, 32]), gdtype=gdtype, h0=True,
                     v_first=v_first)
    H = rng.choice([4, 8, 16, 32])
    HV = H * rng.choice([1, 1, 1, 2])
    if path == "recurrent":
        return _case("", path, _log_int(rng, 1, 32), rng.randint(2, 64), H, HV=HV, gdtype=gdtype,
                     gate=gate, h0=True, v_first=v_first)
    # token-heads: at most those of the largest listed case of the path
    most = 8192 * 32 if path == "train" else 16 * 2048 * 32
    if path in ("chunk", "train") and rng.random() < 0.6:
        n = rng.randint(2, 16)
        total = min(_log_int(rng, 1024, 8192), most // HV)
        cuts = sorted(rng.randint(1, total) for _ in range(n - 1))
        lens = [b - a for a, b in zip([0] + cuts, cuts + [total]) if b > a]
        return _case("", path, 1, sum(lens), H, HV=HV, lens=",".join(map(str, lens)), gdtype=gdtype,
                     gate=gate, h0=h0, v_first=v_first)
    T = _log_int(rng, 300, 8192)
    if rng.random() < 0.3:
        T = max(16, T // 16 * 16)
    B = min(_log_int(rng, 1, 16), max(1, most // (T * HV)))
    return _case("", path, B, T, H, HV=HV, gdtype=gdtype, gate=gate, gstd=rng.choice([1.0, 2.0]), h0=h0,
                 v_first=v_first)


def _lens(case):
    return [int(x) for x in case["lens"].split(",")] if case["lens"] else None


def _states(case):
    return len(_lens(case)) if case["lens"] else case["B"]


def _inputs(case, seed):
    dev = torch.device("cuda", 0)
    gen = torch.Generator(device=dev).manual_seed(seed)
    B, T, H, HV = case["B"], case["T"], case["H"], case["HV"]
    gt = torch.bfloat16 if case["gdtype"] == "bf16" else torch.float32

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=dev, dtype=torch.float32)

    x = {
        "q": randn(B, T, H, D).bfloat16(),
        "k": randn(B, T, H, D).bfloat16(),
        "v": randn(B, T, HV, D).bfloat16(),
    }
    g = randn(B, T, HV, D) * case["gstd"]
    if case["gate"] == "log":
        g = LOWER_BOUND * torch.sigmoid(g)
    x["g"] = g.to(gt)
    x["beta"] = randn(B, T, HV).to(gt)
    x["A_log"] = x["dt_bias"] = x["h0"] = x["do"] = x["dht"] = x["cu"] = None
    if case["gate"] == "kernel":
        x["A_log"] = torch.log(1.0 + 15.0 * torch.rand(HV, generator=gen, device=dev))
        x["dt_bias"] = 0.1 * randn(HV * D)
    if case["h0"]:
        x["h0"] = 0.05 * randn(_states(case), HV, D, D)
    if case["path"] == "train":
        x["do"] = randn(B, T, HV, D).bfloat16()
        x["dht"] = 0.1 * randn(_states(case), HV, D, D)
    lens = _lens(case)
    if lens:
        offs = [0]
        for n in lens:
            offs.append(offs[-1] + n)
        x["cu"] = torch.tensor(offs, dtype=torch.int64, device=dev)
    return x


_GRAD_OF = ("q", "k", "v", "g", "beta", "A_log", "dt_bias", "h0")


def prepare(case, seed):
    x = _inputs(case, seed)
    kw = dict(scale=SCALE, use_qk_l2norm_in_kernel=True, use_beta_sigmoid_in_kernel=True,
              use_gate_in_kernel=case["gate"] == "kernel", lower_bound=LOWER_BOUND, A_log=x["A_log"],
              dt_bias=x["dt_bias"], state_v_first=case["v_first"])
    if case["path"] == "train":
        for n in _GRAD_OF:
            if x[n] is not None:
                x[n].requires_grad_(True)
    if case["path"] in ("chunk", "train"):
        kw["safe_gate"] = True
    if case["path"] in ("chunk", "train", "recurrent") and x["cu"] is not None:
        kw["cu_seqlens"] = x["cu"]
    return {"case": case, "x": x, "kw": kw}


def run(state):
    case, x, kw = state["case"], state["x"], state["kw"]
    seq = (x["q"], x["k"], x["v"], x["g"], x["beta"])
    path = case["path"]
    if path == "decode":
        o = kda_bt16.kda_decode_step(*seq, x["h0"], **kw)
        return {"o": o, "state": x["h0"]}
    fn = {"fwd": kda_bt16.kda_bt16_fwd, "chunk": kda_bt16.chunk_kda, "train": kda_bt16.chunk_kda,
          "recurrent": kda_bt16.fused_recurrent_kda}[path]
    o, ht = fn(*seq, initial_state=x["h0"], output_final_state=True, **kw)
    if path != "train":
        return {"o": o, "ht": ht}
    wrt = [n for n in _GRAD_OF if x[n] is not None]
    grads = torch.autograd.grad([o, ht], [x[n] for n in wrt], [x["do"], x["dht"]])
    return {"o": o, "ht": ht, **{"d" + n: g for n, g in zip(wrt, grads)}}


def work(case):
    B, T, H, HV = case["B"], case["T"], case["H"], case["HV"]
    tok, S = B * T, _states(case)
    gs = 2 if case["gdtype"] == "bf16" else 4
    # q, k (bf16) per q/k head; v, o (bf16), g, beta per value head
    qk, vo, gb = tok * H * D * 2 * 2, tok * HV * D * 2, tok * HV * (D + 1) * gs
    st = S * HV * D * D * 4
    par = HV * (D + 1) * 4 if case["gate"] == "kernel" else 0
    nbytes = qk + 2 * vo + gb + par + st * (2 if case["h0"] else 1)
    if case["path"] in ("decode", "recurrent"):
        # decay, S k, the rank-one update and S q of one token
        return {"bytes": nbytes, "flops": tok * HV * 7 * D * D}
    # matmul flops of a 16-token chunk: two grams, u, w, and w h, qg h,
    # Aqk v_new and the state update
    lens = _lens(case) or [T] * B
    chunks = sum((n + 15) // 16 for n in lens) * HV
    flops = chunks * (4 * 2 * 16 * 16 * D + 3 * 2 * 16 * D * D + 2 * 16 * 16 * D)
    if case["path"] == "train":
        # the backward also reads dO and dht and writes a gradient of every input
        nbytes += vo + st + qk + vo + gb + par + (st if case["h0"] else 0)
        flops *= 3
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # bf16 outputs over fp32 sums; the chunked paths also round their
    # operands (q^, k^, w, u, v_new, the state copy) to bf16 where the
    # reference rounds them.  Seen against exact(): o 1.7e-3 for the token
    # recurrence, 4.2e-3 for the chunked paths, gradients up to 4.3e-3; the
    # limits are about four times that.
    return {"rel": 7e-3 if case["path"] in ("decode", "recurrent") else 1.7e-2}


def _recurrence(q, k, v, a, beta, S, live):
    """Tokens in order, fp64: q, k [S, HV, T, K], v [S, HV, T, V], the decay
    a [S, HV, T, K], beta [S, HV, T], the state S [S, HV, V, K]; ``live``
    [S, T] marks the tokens of each sequence (None: all).  (o, final state)."""
    out = []
    for t in range(q.shape[2]):
        kt = k[:, :, t]
        D_ = S * a[:, :, t].unsqueeze(-2)
        pred = (D_ * kt.unsqueeze(-2)).sum(-1)
        vn = beta[:, :, t].unsqueeze(-1) * (v[:, :, t] - pred)
        N_ = D_ + vn.unsqueeze(-1) * kt.unsqueeze(-2)
        S = N_ if live is None else torch.where(live[:, t, None, None, None], N_, S)
        out.append(SCALE * (S * q[:, :, t].unsqueeze(-2)).sum(-1))
    return torch.stack(out, 2), S


def exact(case, seed):
    x = _inputs(case, seed)
    train = case["path"] == "train"
    lens = _lens(case)
    B, T, H, HV = case["B"], case["T"], case["H"], case["HV"]
    f = {}
    for n in _GRAD_OF:
        f[n] = None if x[n] is None else x[n].double().requires_grad_(train)

    def rows(t):
        """[B, T, heads, ...] to [S, heads, Tmax, ...], padded."""
        if lens:
            parts = torch.split(t[0], lens)
            t = torch.nn.utils.rnn.pad_sequence(parts, batch_first=True)
        return t.transpose(1, 2).contiguous()

    def l2(t):
        return t / torch.sqrt((t * t).sum(-1, keepdim=True) + L2_EPS)

    with torch.set_grad_enabled(train):
        rep = HV // H
        q = l2(f["q"]).repeat_interleave(rep, 2)
        k = l2(f["k"]).repeat_interleave(rep, 2)
        if case["gate"] == "kernel":
            lin = f["g"] + f["dt_bias"].view(HV, D)
            a = torch.exp(LOWER_BOUND * torch.sigmoid(torch.exp(f["A_log"])[:, None] * lin))
        else:
            a = torch.exp(f["g"])
        q, k, v, a = (rows(t) for t in (q, k, f["v"], a))
        beta = rows(torch.sigmoid(f["beta"]).unsqueeze(-1)).squeeze(-1)
        live = None
        if lens:
            n = torch.tensor(lens, device=q.device)
            live = torch.arange(q.shape[2], device=q.device)[None, :] < n[:, None]
        S = torch.zeros(_states(case), HV, D, D, dtype=torch.float64, device=q.device)
        if f["h0"] is not None:
            S = f["h0"] if case["v_first"] else f["h0"].transpose(-1, -2)
        os_ = []
        for t0 in range(0, q.shape[2], 64):
            sl = slice(t0, t0 + 64)
            part = (q[:, :, sl], k[:, :, sl], v[:, :, sl], a[:, :, sl], beta[:, :, sl], S,
                    None if live is None else live[:, sl])
            if train:
                o, S = torch.utils.checkpoint.checkpoint(_recurrence, *part, use_reentrant=False)
            else:
                o, S = _recurrence(*part)
            os_.append(o)
        o = torch.cat(os_, 2).transpose(1, 2)
        if lens:
            o = torch.cat([o[i, :n] for i, n in enumerate(lens)])[None]
        ht = S if case["v_first"] else S.transpose(-1, -2)
        if case["path"] == "decode":
            return {"o": o, "state": ht}
        out = {"o": o, "ht": ht}
        if train:
            wrt = [n for n in _GRAD_OF if f[n] is not None]
            grads = torch.autograd.grad([o, ht], [f[n] for n in wrt], [x["do"].double(), x["dht"].double()])
            out.update({"d" + n: g for n, g in zip(wrt, grads)})
        return {n: t.detach() for n, t in out.items()}
