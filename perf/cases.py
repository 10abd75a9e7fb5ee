"""The work a serving program has the token-selection library do, as measurable cases.

A case is a dict of plain values; `kind` names the entry point:
  sample        PreparedSample / sample_rows: Sampler.sample for B logits rows, parameters and histories on the device
  serve         DeviceSamplers.step: Sampler.choose for B requests whose state lives on the device (ids back on the host)
  verify        PreparedVerify: greedy speculative verify of B blocks of T positions
  propose       PreparedPropose: the drafter's top-16 and walk for n blocks of 7 slots
  head_verify   lmhead_verify_greedy: the bf16 lm_head with greedy verify fused in
  head_sample   lmhead_sample: the bf16 lm_head with top-k sampling fused in

The out_flags word is not among the outputs: it names the internal route a row took and diagnostics of it. A row that
failed shows the token -1.
"""
import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "volundr-mlx_amd"))

from volundr_amd import DeviceSamplers, Sampler, Sampling, ops  # noqa: E402

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SLOTS, RANK = 7, 256  # the drafter's block and codebook rank
MASK = (1 << 64) - 1


def listed():
    """The twelve standing cases, smallest calls first."""
    return [
        # one interactive request: a top-k 20 draw from one fp32 row
        dict(name="sample-1", kind="sample", B=1, V=163840, ld=163840, dtype="f32", mix="topk", dist="spikes", H=0,
             pairs=False, prepared=True),
        # a few requests on a vocabulary of odd size (rows not 16-byte aligned), bf16, raw histories, biases, masks
        dict(name="sample-6-ragged", kind="sample", B=6, V=100003, ld=100003, dtype="bf16", mix="chat", dist="chat",
             H=1000, pairs=False, prepared=False),
        # the decode batch the library's headline metric is quoted on
        dict(name="sample-16-mixed", kind="sample", B=16, V=163840, ld=163840, dtype="f32", mix="mixed",
             dist="student", H=4096, pairs=True, prepared=True),
        # the same batch when the model is unsure of everything: whole-vocabulary nucleus, long histories
        dict(name="sample-16-flat", kind="sample", B=16, V=163840, ld=163840, dtype="f32", mix="flat", dist="flat",
             H=32768, pairs=True, prepared=True),
        # a full server: every kind of request in one decode step
        dict(name="sample-128-chat", kind="sample", B=128, V=163840, ld=163840, dtype="f32", mix="chat", dist="chat",
             H=1024, pairs=True, prepared=True),
        # an engine's decode step with the request state on the device, model vocabulary, bf16 logits
        dict(name="serve-64", kind="serve", B=64, V=248320, vv=248077, ld=248320, dtype="bf16", mix="chat",
             dist="chat", H=512),
        # one speculative verify block (16 drafts and the bonus position)
        dict(name="verify-1x17", kind="verify", B=1, T=17, V=163840, vv=163840, ld=163840, dtype="bf16"),
        # verify blocks of a batch of speculating requests, model vocabulary
        dict(name="verify-16x17", kind="verify", B=16, T=17, V=248320, vv=248077, ld=248320, dtype="bf16"),
        # the drafter's proposal for one request and for a batch of them
        dict(name="propose-1", kind="propose", n=1, V=248320, vv=248077, ld=248320, dtype="bf16"),
        dict(name="propose-16", kind="propose", n=16, V=248320, vv=248077, ld=248320, dtype="bf16"),
        # the head with verify, and the head with a decode batch's sampling, at the model's size
        dict(name="head-verify-1x17", kind="head_verify", B=1, T=17, K=5120, V=248320, vv=248077),
        dict(name="head-sample-16", kind="head_sample", R=16, K=5120, V=248320),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: batch sizes and vocabularies log-uniform over the served range, odd sizes and row strides
    among them."""
    kind = rng.choice(["sample"] * 5 + ["serve"] * 2 + ["verify"] * 2 + ["propose"] * 2 + ["head_verify", "head_sample"])
    V = _log_int(rng, 32000, 262144)
    aligned = rng.random() < 0.6
    if aligned:
        V = (V + 63) // 64 * 64
    ld = V if rng.random() < 0.7 else V + 8 * rng.randint(1, 64)  # padded rows
    dt = rng.choice(["f32", "f32", "bf16", "bf16", "f16"])
    if kind == "sample":
        mix = rng.choice(["topk", "mixed", "chat", "chat", "flat", "greedy", "nucleus"])
        dist = {"flat": "flat", "mixed": "student"}.get(mix) or rng.choice(["chat", "spikes"])
        return dict(kind=kind, B=_log_int(rng, 1, 128), V=V, ld=ld, dtype="f32" if mix == "flat" else dt, mix=mix,
                    dist=dist, H=_log_int(rng, 16, 16384), pairs=rng.random() < 0.5, prepared=rng.random() < 0.7)
    if kind == "serve":
        return dict(kind=kind, B=_log_int(rng, 1, 96), V=V, vv=V - rng.randint(0, 256), ld=ld, dtype=dt,
                    mix=rng.choice(["chat", "mixed", "topk"]), dist="chat", H=_log_int(rng, 16, 2048))
    if kind == "verify":
        return dict(kind=kind, B=_log_int(rng, 1, 16), T=rng.randint(1, 17), V=V, vv=V - rng.randint(0, 256), ld=ld,
                    dtype=dt)
    if kind == "propose":
        return dict(kind=kind, n=_log_int(rng, 1, 16), V=V, vv=V - rng.randint(0, 256), ld=ld, dtype=dt)
    V = (V + 15) // 16 * 16
    K = 256 * rng.randint(4, 20)
    if kind == "head_verify":
        B = rng.randint(1, 4)
        return dict(kind=kind, B=B, T=rng.randint(1, 17), K=K, V=V, vv=V - rng.randint(0, 243))
    return dict(kind=kind, R=rng.randint(1, 16), K=K, V=V)


# ---------------------------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------------------------
def _samplings(mix, B, V, rng):
    """Request parameters: `mixed` the headline batch's, `chat` what a chat server sees (greedy, top-k, nucleus and
    min-p requests, some with penalties, biases, suppressed ids and a stop mask)."""
    out = []
    for _ in range(B):
        if mix == "topk":
            sp = Sampling(temperature=1.0, top_k=20)
        elif mix == "greedy":
            sp = Sampling(temperature=0.0, repetition_penalty=float(rng.uniform(1.0, 1.2)))
        elif mix == "nucleus":
            sp = Sampling(temperature=float(rng.uniform(0.6, 1.2)), top_p=float(rng.choice([0.8, 0.9, 0.95])))
        elif mix == "flat":
            sp = Sampling(temperature=1.0, top_k=0, top_p=0.95, repetition_penalty=1.1)
        elif mix == "mixed":
            sp = Sampling(temperature=float(rng.uniform(0.6, 1.2)), top_k=int(rng.choice([0, 20, 50])),
                          top_p=float(rng.choice([0.8, 0.95, 1.0])),
                          repetition_penalty=float(rng.uniform(1.05, 1.2)),
                          presence_penalty=float(rng.uniform(0.0, 0.5)))
        else:
            p = rng.random()
            sp = Sampling(temperature=float(rng.uniform(0.6, 1.1)))
            if p < 0.2:
                sp.temperature = 0.0
            elif p < 0.6:
                sp.top_k, sp.top_p = int(rng.choice([20, 40, 50, 64])), float(rng.choice([0.8, 0.9, 0.95, 1.0]))
            elif p < 0.85:
                sp.top_p = float(rng.choice([0.8, 0.9, 0.95]))
            else:
                sp.min_p = float(rng.choice([0.02, 0.05, 0.1]))
            if rng.random() < 0.5:
                sp.repetition_penalty = float(rng.uniform(1.02, 1.15))
            if rng.random() < 0.25:
                sp.presence_penalty, sp.frequency_penalty = float(rng.uniform(0, 0.5)), float(rng.uniform(0, 0.2))
            if rng.random() < 0.2:
                sp.logit_bias = [(int(t), float(b)) for t, b in zip(rng.integers(0, V, 8), rng.uniform(-3, 3, 8))]
            if rng.random() < 0.2:
                sp.suppress_tokens = [int(t) for t in rng.integers(0, V, 4)]
            if rng.random() < 0.3:
                sp.min_new_tokens, sp.stop_token_ids = 1 << 20, [int(t) for t in rng.integers(0, V, 3)]
        out.append(sp)
    return out


def _histories(case, rng):
    """Zipf-like histories, as text has (the near-flat batch: uniform over the vocabulary)."""
    H, V, B = case["H"], case["V"], case["B"]
    if not H:
        return None
    if case["mix"] == "flat":
        return [rng.integers(0, V, H).astype(np.int32) for _ in range(B)]
    return [((rng.zipf(1.1, H) - 1) % V).astype(np.int32) for _ in range(B)]


def _rows(case, rows, seed, dist):
    """[rows, V] logits (a view with row stride ld) of the case's dtype on the GPU."""
    V, ld = case["V"], case["ld"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(rows, V, generator=g, device="cuda")
    if dist == "student":  # 3 * Student-t with 3 degrees of freedom
        q = torch.zeros(rows, V, device="cuda")
        for _ in range(3):
            q += torch.randn(rows, V, generator=g, device="cuda").square_()
        x = 3.0 * x / (q / 3.0).sqrt_()
        del q
    elif dist == "flat":
        x *= 0.1
    elif dist == "spikes":
        x *= 3.0
        x.scatter_(1, torch.randint(0, V, (rows, 5), generator=g, device="cuda"), 12.0)
    else:  # chat: a few hundred plausible tokens above a wide floor, as a language model's next-token logits have
        x *= 2.0
        at = torch.randint(0, V // 200, (rows, 200), generator=g, device="cuda")
        at += torch.arange(200, device="cuda") * (V // 200)  # distinct positions
        at = at.gather(1, torch.rand(rows, 200, generator=g, device="cuda").argsort(1))
        top = 16.0 - torch.arange(200, device="cuda") ** 0.4 * torch.rand(rows, 1, generator=g, device="cuda") * 1.2
        x.scatter_(1, at, top + 0.3 * torch.randn(rows, 200, generator=g, device="cuda"))
    y = torch.empty(rows, ld, dtype=DTYPES[case["dtype"]], device="cuda")[:, :V]
    y.copy_(x)
    return y


def _verify_rows(case, seed):
    """Logits [B, T, V] with a clear winner per position (now and then an exact tie at a higher index) and drafts that
    agree with it for a random prefix."""
    B, T, vv = case["B"], case["T"], case["vv"]
    x = _rows(case, B * T, seed, "chat")
    rng = np.random.default_rng(seed)
    win = rng.integers(0, vv, B * T)
    x[torch.arange(B * T, device="cuda"), torch.from_numpy(win).cuda()] = 22.0
    tied = np.nonzero(rng.random(B * T) < 0.05)[0]
    if tied.size:
        hi = win[tied] + ((vv - win[tied]) * rng.random(tied.size)).astype(np.int64)
        x[torch.from_numpy(tied).cuda(), torch.from_numpy(hi).cuda()] = 22.0
    return x.unflatten(0, (B, T)), _drafts(win.reshape(B, T), vv, rng)


def _drafts(win, vv, rng):
    B, T = win.shape
    d = rng.integers(0, vv, (B, max(T - 1, 0)))
    for b, n in enumerate(rng.integers(0, T, B)):
        d[b, :n] = win[b, :n]
        if n < T - 1:
            d[b, n] = (win[b, n] + 1) % vv
    return torch.from_numpy(d.astype(np.int32)).cuda()


def _head(case, R, seed):
    """Hidden rows that point at one token each, as a trained model's do, and a random head weight."""
    V, K = case["V"], case["K"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    W = torch.empty(V, K, dtype=torch.bfloat16, device="cuda")
    for a in range(0, V, 32768):
        W[a:a + 32768] = torch.randn(min(32768, V - a), K, generator=g, device="cuda") / math.sqrt(K)
    win = np.random.default_rng(seed).integers(0, case.get("vv", V), R)
    h = 2.0 * torch.randn(R, K, generator=g, device="cuda") + 16.0 * W[torch.from_numpy(win).cuda()].float()
    return h.to(torch.bfloat16), W, win


def prepare(case, seed):
    kind, rng = case["kind"], np.random.default_rng(seed)
    s = SimpleNamespace(case=case)
    if kind == "sample":
        B, V = case["B"], case["V"]
        sps, hists, s.u = _samplings(case["mix"], B, V, rng), _histories(case, rng), rng.random(B)
        s.x = _rows(case, B, seed, case["dist"])
        s.rows = ops.pack_rows(sps, s.u, V, hists, hist_pairs=case["pairs"]).to("cuda")
        s.sps, s.hists = sps, hists
        s.call = ops.PreparedSample([s.x], s.rows) if case["prepared"] else None
    elif kind == "serve":
        B, V = case["B"], case["V"]
        s.sps, s.hists = _samplings(case["mix"], B, V, rng), _histories(case, rng)
        s.seeds = [int(v) | 1 for v in rng.integers(1, 1 << 62, B)]
        reqs = []
        for sp, h, sd in zip(s.sps, s.hists, s.seeds):
            sp.seed = sd
            q = Sampler(sp, vocab_valid=case["vv"])
            for t in h.tolist():
                q.accept(t)
            reqs.append(q)
        s.x = _rows(case, B, seed, case["dist"])
        s.ds = DeviceSamplers(reqs, V, hist_cap=8192)
    elif kind == "verify":
        s.x, s.drafts = _verify_rows(case, seed)
        s.call = ops.PreparedVerify([s.x], s.drafts, case["vv"])
    elif kind == "propose":
        n, V = case["n"], case["V"]
        s.x = _rows(case, n * SLOTS, seed, "chat").unflatten(0, (n, SLOTS))
        g = torch.Generator(device="cuda").manual_seed(seed + 1)
        s.A = (torch.randn(V, RANK, generator=g, device="cuda") * 0.1).to(torch.bfloat16)
        s.Bc = (torch.randn(V, RANK, generator=g, device="cuda") * 0.1).to(torch.bfloat16)
        s.hp = torch.randn(n, SLOTS, RANK, generator=g, device="cuda")
        s.anchor = torch.randint(0, case["vv"], (n,), generator=g, device="cuda", dtype=torch.int32)
        s.call = ops.PreparedPropose([s.x], s.hp, s.A, s.Bc, s.anchor, case["vv"])
    elif kind == "head_verify":
        B, T = case["B"], case["T"]
        h, s.W, win = _head(case, B * T, seed)
        s.h = h.unflatten(0, (B, T))
        s.drafts = _drafts(win.reshape(B, T), case["vv"], rng) if T > 1 else None
    else:
        s.h, s.W, _ = _head(case, case["R"], seed)
        R = case["R"]
        s.sps = [Sampling(temperature=float(rng.uniform(0.6, 1.2)), top_k=int(rng.choice([20, 50])),
                          top_p=float(rng.choice([0.8, 0.95, 1.0]))) if r % 8 != 7 else Sampling(temperature=0.0)
                 for r in range(R)]
        s.u = rng.random(R)
    return s


def run(s):
    kind = s.case["kind"]
    if kind == "sample":
        o = s.call() if s.call is not None else ops.sample_rows(s.x, s.rows)
        return {"ids": o.ids, "logprobs": o.logprobs, "keep": o.keep}
    if kind == "serve":
        o = s.ds.step(s.x).out
        return {"ids": o.ids, "logprobs": o.logprobs, "keep": o.keep}
    if kind == "propose":
        return {"drafts": s.call()}
    if kind == "head_sample":
        o = ops.lmhead_sample(s.h, s.W, s.sps, s.u)
        return {"ids": o.ids, "logprobs": o.logprobs, "keep": o.keep}
    o = s.call() if kind == "verify" else ops.lmhead_verify_greedy(s.h, s.W, s.drafts, s.case["vv"])
    return {"argmax": o.argmax, "accept": o.accept, "logprobs": o.logprobs}


def work(case):
    """Each input read once, each output written once; the head's products."""
    kind, V = case["kind"], case["V"]
    es = {"f32": 4}.get(case.get("dtype"), 2)
    if kind in ("sample", "serve"):
        B = case["B"]
        # 96 bytes of parameters and 16 of results a row; the penalty counts as 4 bytes a token
        return {"bytes": B * (V * es + 4 * case["H"] + 96 + 16), "flops": 0}
    if kind == "verify":
        R = case["B"] * case["T"]
        return {"bytes": R * (case["vv"] * es + 12), "flops": 0}
    if kind == "propose":
        n = case["n"]
        rows = 1 + (SLOTS - 1) * 16 + SLOTS * 16  # codebook rows the walk can touch
        return {"bytes": n * (SLOTS * (case["vv"] * es + RANK * 4 + 4) + rows * RANK * 2), "flops": 0}
    R, K = (case["R"] if kind == "head_sample" else case["B"] * case["T"]), case["K"]
    return {"bytes": V * K * 2 + R * K * 2 + R * 16, "flops": 2.0 * R * V * K}


def tolerance(case):
    """Tokens, counts and accept lengths are whole numbers: the same, but for draws and cuts within rounding of a
    cumulative boundary. Log-probabilities come from 32-bit quotients, exponentials and sums (1e-7 to 4e-6 off the
    64-bit values)."""
    if case["kind"] == "propose":
        return {"rel": 0.0, "differ": 0.01}
    return {"rel": 1e-5, "max": 1e-4, "differ": 0.01}


# ---------------------------------------------------------------------------------------------------------------
# The results in 64 bits
# ---------------------------------------------------------------------------------------------------------------
def _edit(x, sp, hist, V):
    """The logit edits of the sampler, which are defined in float32."""
    for t, b in sp.logit_bias:
        x[t] += np.float32(b)
    if sp.suppress_tokens:
        x[torch.tensor(sp.suppress_tokens, device=x.device)] = -math.inf
    if hist is not None and (sp.repetition_penalty != 1.0 or sp.frequency_penalty or sp.presence_penalty):
        ids, c = np.unique(hist, return_counts=True)
        ids, c = torch.from_numpy(ids.astype(np.int64)).to(x.device), torch.from_numpy(c.astype(np.float32)).to(x.device)
        v = x[ids]
        if sp.repetition_penalty != 1.0:
            r = torch.tensor(sp.repetition_penalty, dtype=torch.float32, device=x.device)
            v = torch.where(v > 0, v / r, v * r)
        f = torch.tensor(sp.frequency_penalty, dtype=torch.float32, device=x.device)
        p = torch.tensor(sp.presence_penalty, dtype=torch.float32, device=x.device)
        x[ids] = v - (f * c + p)
    return x


def _exact_row(x, sp, u):
    """(token, logprob, kept) of one edited row, in float64."""
    d = x.double()
    if sp.greedy:
        j = int(torch.nonzero(d == d.max())[0])
        return j, float(d[j] - torch.logsumexp(d[torch.isfinite(d)], 0)), 0
    idx = torch.nonzero(torch.isfinite(d))[:, 0]
    val, o = torch.sort(d[idx], descending=True, stable=True)
    idx = idx[o]
    k = sp.top_k if sp.top_k else idx.numel()
    t = float(np.float32(sp.temperature))
    if k < idx.numel():
        val, idx = val[:k], idx[:k]
    elif idx.numel() > 4096:
        keep = val / t >= val[0] / t - 40.0
        val, idx = val[keep], idx[keep]
    pr = torch.exp(val / t - val[0] / t)
    pr /= pr.sum()
    n, c = pr.numel(), torch.cumsum(pr, 0)
    if sp.top_p < 1.0:
        hit = torch.nonzero(c >= sp.top_p)
        n = int(hit[0]) + 1 if hit.numel() else n
    if sp.min_p > 0.0:
        below = torch.nonzero(pr < pr[0] * sp.min_p)
        n = min(n, max(int(below[0]), 1) if below.numel() else pr.numel())
    z = pr[:n].sum()
    j = min(int(torch.searchsorted(c[:n].contiguous(), (u * z).reshape(1))), n - 1)
    return int(idx[j]), float(torch.log(pr[j] / z)), n


def _exact_sample(x, sps, us, hists, V, vvs=None):
    ids, lps, keep = [], [], []
    for r, sp in enumerate(sps):
        row = x[r].float().clone()
        if vvs is not None and sp.greedy and not sp.needs_logits(vvs, 0):
            row = row[:vvs]  # a request that needs no logits: the argmax over the valid ids
        else:
            row = _edit(row, sp, None if hists is None else hists[r], V)
            if sp.min_new_tokens > (len(hists[r]) if vvs is not None else 0) and sp.stop_token_ids:
                row[torch.tensor(sp.stop_token_ids, device=row.device)] = -math.inf
        j, lp, n = _exact_row(row, sp, float(us[r]))
        ids.append(j), lps.append(lp), keep.append(n)
    return {"ids": np.array(ids), "logprobs": np.array(lps), "keep": np.array(keep)}


def _exact_logits(s):
    """bf16(h @ W^T): products and sums in float64, then the head's rounding to bf16, widened."""
    h, out = s.h.reshape(-1, s.h.shape[-1]).double(), []
    for a in range(0, s.W.shape[0], 16384):
        out.append((h @ s.W[a:a + 16384].double().T).to(torch.bfloat16).double())
    return torch.cat(out, 1)


def _exact_verify(x, drafts, B, T):
    x = x.double()
    top = x.max(-1, keepdim=True).values
    am = torch.argmax((x == top).to(torch.uint8), -1)  # the first maximum
    lp = (top[..., 0] - torch.logsumexp(x, -1)).reshape(B, T)
    am = am.reshape(B, T)
    acc = torch.cumprod((drafts.reshape(B, T - 1).long() == am[:, :-1]).long(), 1).sum(1) if T > 1 else am[:, 0] * 0
    return {"argmax": am.cpu().numpy(), "accept": acc.cpu().numpy(), "logprobs": lp.cpu().numpy()}


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]
    if kind == "sample":
        return _exact_sample(s.x, s.sps, s.u, s.hists, case["V"])
    if kind == "serve":
        us = []
        for r in s.seeds:
            r ^= r >> 12
            r ^= (r << 25) & MASK
            r ^= r >> 27
            us.append((((r * 0x2545F4914F6CDD1D) & MASK) >> 11) / float(1 << 53))
        return _exact_sample(s.x, s.sps, us, s.hists, case["V"], case["vv"])
    if kind == "verify":
        rows = [_exact_verify(x[..., :case["vv"]], d, 1, case["T"]) for x, d in
                zip(s.x, s.drafts if case["T"] > 1 else [None] * case["B"])]
        return {k: np.concatenate([r[k] for r in rows]) for k in rows[0]}
    if kind == "propose":
        return None  # token ids alone
    x = _exact_logits(s)
    if kind == "head_verify":
        return _exact_verify(x[:, :case["vv"]], s.drafts, case["B"], case["T"])
    return _exact_sample(x, s.sps, s.u, None, case["V"])
