"""GPU parity of the batches that take more rows than one launch of vs_sample_kernel holds (csrc/vs_batch.hip): the
streaming pass, the finish from the lists and the open rows, against the NumPy oracle. B = 70 and 130 rows of 8192 and
more logits always go that way (at most 64 rows fit one launch of the other kernel); 130 rows also use the second half
of the workspace rows and the second launch of a batch."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from oracle import draft_ref as DR
from oracle import sampler_ref as S
from parity import check_sample
from volundr_amd import DeviceSamplers, Sampler, _lib, ops, sample_batch, topk_batch
from volundr_amd.session import Sampling

pytestmark = pytest.mark.gpu


def rows_on(dev, x, dtype, pad):
    """x as a device view whose row stride is V + pad elements."""
    B, V = x.shape
    t = torch.empty(B, V + pad, dtype=dtype, device=dev)[:, :V]
    t.copy_(torch.from_numpy(x).to(dev))
    return t, t.float().cpu().numpy()


def plan(dev, dtype, B, V, pad=0):
    """How the launches split such a batch on this device: rows, logits per lane, workgroups per row, list length."""
    L, out = _lib.load(), np.zeros(7, np.int32)
    ws = L.vs_sample_workspace_bytes(B, V)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    _lib.check(L.vs_batch_plan(ops._DTYPES[dtype], V, V + pad, 0, B, ws, cus, out.ctypes.data), "vs_batch_plan")
    return dict(zip(("rows", "E", "G", "CH", "kcap", "kmax", "nv"), out.tolist()))


def check(dev, x, ps, u, hists=None, dtype=torch.float32, pad=0, pairs=False, label="", max_excused=2, some=None):
    """All rows of the call, or the rows `some`, against the oracle (boundary rows excused: draws of flat rows now and
    then, 1e-6 of the mass on either side of a logit's 1e-5 to 1e-4)."""
    xt, xr = rows_on(dev, x, dtype, pad)
    print(f"[{label}] B={x.shape[0]} V={x.shape[1]} {dtype} pad={pad} pairs={pairs}", flush=True)
    out = sample_batch(xt, ps, u, hists, hist_pairs=pairs)
    torch.cuda.synchronize()
    some = range(x.shape[0]) if some is None else some
    refs = [S.sample(xr[i], ps[i], float(u[i]), S.counts_from_history(hists[i]) if hists is not None else {})
            for i in some]
    at = torch.tensor(list(some), device=dev)
    part = SimpleNamespace(ids=out.ids[at], logprobs=out.logprobs[at], flags=out.flags[at], keep=out.keep[at])
    check_sample(part, refs, label, max_excused)
    return out, refs


def mixed_params(rng, n, V):
    out = []
    for _ in range(n):
        sp = Sampling(temperature=float(rng.choice([0.0, 0.6, 1.0, 1.0, 1.6])),
                      top_k=int(rng.choice([0, 0, 0, 1, 20, 64, 65, 128, 256, 257, 300])),
                      top_p=float(rng.choice([1.0, 0.95, 0.8, 0.3])), min_p=float(rng.choice([0.0, 0.0, 0.05, 0.5])),
                      repetition_penalty=float(rng.choice([1.0, 1.1, 1.3])),
                      presence_penalty=float(rng.choice([0.0, 0.3])), frequency_penalty=float(rng.choice([0.0, 0.1])))
        if rng.random() < 0.3:
            sp.logit_bias = [(int(t), float(b)) for t, b in zip(rng.integers(0, V, 5), rng.uniform(-4, 4, 5))]
        if rng.random() < 0.3:
            sp.suppress_tokens = [0, int(rng.integers(0, V)), V - 1]
        if rng.random() < 0.3:
            sp.min_new_tokens, sp.stop_token_ids = 5, [1, V - 2]
        out.append(sp)
    return out


# chunks of up to 8192 positions: one whole chunk, a few logits in the next, several; rows off the 16-byte lines
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,V,pad", [(70, 8192, 0), (70, 8195, 1), (130, 16391, 0), (66, 24577, 7), (130, 16384, 8)])
def test_mixed_rows(dev, B, V, pad, dtype):
    rng = np.random.default_rng(V + pad)
    scale = rng.choice([0.05, 0.3, 1.0, 3.0, 6.0], size=(B, 1))
    x = (rng.standard_normal((B, V)) * scale).astype(np.float32)
    hists = [rng.integers(0, V, size=int(rng.integers(0, 2500))) for _ in range(B)]
    assert plan(dev, dtype, B, V, pad)["E"] == 16
    check(dev, x, mixed_params(rng, B, V), rng.random(B), hists, dtype, pad, pairs=bool(pad % 2 == 0),
          label=f"batch mix {B}x{V}+{pad}")


# chunks of up to 16384 positions, the batches of a full server: nine and more lists per row (two per wave of the finish
# kernel), a whole last chunk, a few logits in it, rows off the 16-byte lines, a second launch of few rows
@pytest.mark.parametrize("dtype,B,V,pad", [(torch.float32, 66, 163840, 0), (torch.float32, 130, 147461, 3),
                                           (torch.bfloat16, 130, 163840, 8), (torch.bfloat16, 66, 248327, 1),
                                           (torch.float16, 66, 248320, 0), (torch.float16, 100, 163843, 5)])
def test_mixed_rows_of_a_full_server(dev, dtype, B, V, pad):
    p = plan(dev, dtype, B, V, pad)
    assert p["E"] == 32 and p["G"] > 8, p
    rng = np.random.default_rng(V + B)
    scale = rng.choice([0.05, 1.0, 2.0, 3.0], size=(B, 1)).astype(np.float32)
    x = rng.standard_normal((B, V), dtype=np.float32) * scale
    hists = [rng.integers(0, V, size=int(rng.integers(0, 4000))) for _ in range(B)]
    some = sorted({*range(0, B, 5), 0, 63, 64, 65, B - 2, B - 1} & set(range(B)))
    check(dev, x, mixed_params(rng, B, V), rng.random(B), hists, dtype, pad, pairs=bool(pad % 2 == 0),
          label=f"server mix {B}x{V}+{pad}", some=some)


@pytest.mark.parametrize("dtype,pad", [(torch.float32, 3), (torch.bfloat16, 0)])
def test_open_rows_read_again(dev, dtype, pad):
    """More open rows than leave each a cluster that holds the row in LDS (40 and more at V = 163840): every pass streams
    and edits the row again."""
    rng = np.random.default_rng(44)
    B, V = 66, 163840
    x = rng.standard_normal((B, V), dtype=np.float32) * np.float32(0.1)
    x[1::4] = np.round(x[1::4] * 8) / 8  # tied values: the general method
    x[2::4] *= 20.0
    kinds = [dict(top_p=0.95), dict(top_p=0.9, min_p=0.5), dict(top_k=3000, top_p=0.9), dict(temperature=0.8)]
    ps = [Sampling(repetition_penalty=1.1, presence_penalty=0.02, **kinds[r % 4]) for r in range(B)]
    for r in range(0, B, 3):
        ps[r].logit_bias = [(int(t), 0.3) for t in rng.integers(0, V, 6)]
        ps[r].suppress_tokens = [int(t) for t in rng.integers(0, V, 5)]
    hists = [rng.integers(0, V, size=int(rng.integers(1, 6000))) for _ in range(B)]
    u = (np.floor(rng.random(B) * 4000) + 0.37) / 4000
    check(dev, x, ps, u, hists, dtype, pad, pairs=not pad, label="open rows read again", some=range(0, B, 3))
    row = _lib.load().vs_sample_workspace_bytes(1, V)
    ws = ops.workspace(dev, 64 * row)
    open_rows = int((ws[64:64 + 56] != 0).sum()) + int((ws[row + 64:row + 64 + B - 56] != 0).sum())
    assert open_rows >= 43, open_rows  # 256 // 43 = 5 workgroups of 24576 logits hold less than a row


def odd_rows(rng, V):
    """Rows that lists, bounds and value bins find hard."""
    n = lambda s: (rng.standard_normal(V) * s).astype(np.float32)  # noqa: E731
    rows = [np.zeros(V, np.float32), np.full(V, -3.5, np.float32), np.round(n(1.0)), np.round(n(3.0) * 2) / 2]
    few = np.full(V, -np.inf, np.float32)
    few[rng.choice(V, 40, replace=False)] = n(2.0)[:40]
    one = np.full(V, -np.inf, np.float32)
    one[V - 1] = 1.0
    none = np.full(V, -np.inf, np.float32)
    nan = n(2.0)
    nan[V // 3] = np.nan
    inf = n(2.0)
    inf[V // 2] = np.inf
    low = n(1.0)
    low[:700] += 12.0 + rng.random(700).astype(np.float32)  # the largest logits all in one chunk
    huge = n(1.0)
    huge[5], huge[V - 5] = 2e38, -2e38
    half = n(1.0)
    half[::2] = -np.inf
    zero = n(1e-3)
    zero[zero < 0] = -0.0
    return rows + [few, one, none, nan, inf, low, huge, half, zero]


@pytest.mark.parametrize("pad", [0, 3])
@pytest.mark.parametrize("sp", [dict(top_k=20), dict(top_k=200, top_p=0.9), dict(top_p=0.9), dict(), dict(min_p=0.05),
                                dict(top_p=0.95, min_p=0.01, temperature=0.7), dict(temperature=0.0),
                                dict(top_k=700), dict(min_p=1.0)], ids=str)
def test_odd_rows(dev, sp, pad):
    rng = np.random.default_rng(7 + pad)
    V = 8192 + 40
    base = odd_rows(rng, V)
    x = np.stack((base * 6)[:70])
    # equal masses have draw boundaries at multiples of 1 / n: keep the draws off them
    u = (np.floor(rng.random(70) * 4000) + 0.37) / 4000
    with np.errstate(all="ignore"):
        check(dev, x, [Sampling(**sp)] * 70, u, pad=pad, label=f"odd rows {sp}")


def test_large_counts_and_many_tokens(dev):
    """Table counts that do not fit the edit words, and a token repeated through a long raw history."""
    rng = np.random.default_rng(3)
    B, V = 66, 9000
    x = (rng.standard_normal((B, V)) * 2).astype(np.float32)
    ps = [Sampling(top_k=30, repetition_penalty=1.2, frequency_penalty=1e-9, presence_penalty=0.1)] * B
    u = rng.random(B)
    tables = [{int(np.argsort(-x[r])[0]): (1 << 28) + 5, int(np.argsort(-x[r])[1]): 3, 7: (1 << 30)} for r in range(B)]
    xt = torch.from_numpy(x).to(dev)
    out = sample_batch(xt, ps, u, tables, hist_pairs=True)
    check_sample(out, [S.sample(x[r], ps[r], float(u[r]), tables[r]) for r in range(B)], "large counts")
    hists = [np.concatenate([np.full(20000, int(np.argmax(x[r]))), rng.integers(0, V, 700)]) for r in range(B)]
    check(dev, x, ps, u, hists, label="repeated token", max_excused=1)


@pytest.mark.parametrize("pairs", [False, True])
def test_lengths_of_the_edit_lists(dev, pairs):
    """Tables, histories, masks and biases that end at, before and past what a lane loads ahead (512 ids of a list, 2048
    table entries, 4096 raw tokens, then rounds of 12288), with the row's largest logits among their ids."""
    rng = np.random.default_rng(9)
    B, V = 66, 33000
    x = (rng.standard_normal((B, V)) * 2).astype(np.float32)
    top = np.argsort(-x, axis=1)[:, :4000]
    lens = [1, 3, 511, 512, 513, 2047, 2048, 2049, 4095, 4096, 4103, 16384, 16391, 30000]
    few = [0, 1, 511, 512, 513, 1100]
    ps, hists = [], []
    for r in range(B):
        n, m = lens[r % len(lens)], few[r % len(few)]
        ids = np.concatenate([top[r][: min(n, 300)], rng.permutation(V)])  # unique once cut, in an order of no kind
        ids = ids[np.sort(np.unique(ids, return_index=True)[1])][:n]
        if not pairs:
            ids = np.concatenate([ids[: n - n // 3], rng.choice(ids, n // 3)]) if n > 3 else ids
        hists.append(rng.permutation(ids))
        sp = Sampling(temperature=0.9, top_k=[40, 0, 64][r % 3], top_p=0.95, repetition_penalty=1.2, presence_penalty=0.2,
                      frequency_penalty=0.05)
        if m:
            sp.suppress_tokens = [int(i) for i in rng.choice(top[r], m, replace=False)]
            sp.logit_bias = [(int(i), float(b)) for i, b in zip(rng.choice(top[r], m), rng.uniform(-2, 2, m))]
            sp.min_new_tokens, sp.stop_token_ids = 5, [int(i) for i in rng.choice(top[r], m, replace=False)]
        ps.append(sp)
    check(dev, x, ps, rng.random(B), hists, pairs=pairs, pad=3, label="edit lists")


def test_state_rows(dev):
    """70 requests with their state on the device: draws, accepted tokens, stop masks and forced rows over steps."""
    V, B = 8200, 70
    rng = np.random.default_rng(5)
    sps = mixed_params(rng, B, V)
    for i, sp in enumerate(sps):
        sp.seed = 1000 + i
    ds = DeviceSamplers([Sampler(sp, vocab_valid=V - 8) for sp in sps], V, hist_cap=64, device=dev)
    state = [(S.seed_state(1000 + i), [], 0) for i in range(B)]
    for step in range(4):
        print(f"[batch state] step {step}", flush=True)
        x = (rng.standard_normal((B, V)) * 2.5).astype(np.float32)
        res = ds.step(torch.from_numpy(x).to(dev))
        refs, nxt = [], []
        for i, sp in enumerate(sps):
            rs, u = S.xorshift64s_next(state[i][0])
            r = S.choose(x[i], sp, V - 8, u, state[i][1])
            refs.append(r)
            nxt.append((rs if r.kind == "sample" else state[i][0], state[i][1] + [res.ids[i]], state[i][2] + 1))
        check_sample(res.out, refs, f"batch state step {step}", max_excused=1)
        state = nxt
    st = ds.host_state()
    for i in range(B):
        assert int(st[i]["rng"]) == state[i][0] and int(st[i]["produced"]) == 4
        assert ds.history(i) == state[i][1]


@pytest.mark.parametrize("k", [1, 16, 64])
def test_top_lists(dev, k):
    rng = np.random.default_rng(k)
    V = 8192 + 24
    x = np.stack((odd_rows(rng, V) * 6)[:70])
    xt = torch.from_numpy(x).to(dev)
    ids, vals = topk_batch(xt, k)
    ids, vals = ids.cpu().numpy(), vals.cpu().numpy()
    for r in range(70):
        ri, rv = DR.topk_sorted(x[r], k)
        assert np.array_equal(ids[r], ri), (k, r)
        assert np.array_equal(vals[r], rv), (k, r)


def test_graph_replays(dev):
    """The three launches captured: every replay on refilled logits equals the eager call."""
    rng = np.random.default_rng(9)
    B, V = 70, 16500
    sps = mixed_params(rng, B, V)
    rows = ops.pack_rows(sps, rng.random(B), V).to(dev)
    xs = [torch.from_numpy((rng.standard_normal((B, V)) * s).astype(np.float32)).to(dev) for s in (0.2, 2.0, 5.0)]
    x = xs[0].clone()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        call = ops.PreparedSample([x], rows)
        call()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        call()
    for i in (1, 2, 0, 1):
        x.copy_(xs[i])
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        got = call.out.block.clone()
        want = ops.sample_rows(xs[i], rows).block
        torch.cuda.synchronize()
        assert torch.equal(got, want), i


def test_tag_words_left_alone(dev):
    """The words that hold the other kernel's tags keep what it left there, whatever a large batch does: that kernel
    takes a partial for this call's own by them."""
    rng = np.random.default_rng(12)
    B, V = 70, 8200
    row = _lib.load().vs_sample_workspace_bytes(1, V)
    x = torch.from_numpy((rng.standard_normal((B, V)) * 2).astype(np.float32)).to(dev)
    ps = mixed_params(rng, B, V)
    sample_batch(x, ps, rng.random(B))  # the workspace is as large as it gets
    sample_batch(x[:16], ps[:16], rng.random(16))
    ws = ops.workspace(dev, 64 * row)
    at = torch.tensor([r * row + 128 + 96 * g + 20 + i for r in range(64) for g in range(64) for i in range(4)], device=dev)
    before = ws[at].clone()
    print("[tags] 70 rows", flush=True)
    sample_batch(x, ps, rng.random(B))
    torch.cuda.synchronize()
    assert torch.equal(ws[at], before)


def hard_lists(rng, V, n):
    """n rows whose chunks have more candidates than their lists hold: continuous values, values in steps (thousands of
    ties at the cut), one value, the largest logits side by side, few finite logits."""
    rows = []
    for r in range(n):
        x = (rng.standard_normal(V) * 2).astype(np.float32)
        if r % 5 == 1:
            x = np.round(x * 2) / 2
        elif r % 5 == 2:
            x[:] = -1.25 if r % 2 else 0.0
            x[::7] = -0.0 if r % 2 == 0 else -1.25
        elif r % 5 == 3:
            at = int(rng.integers(0, V - 3000))
            x[at:at + 3000] += 12.0
        elif r % 5 == 4:
            x[rng.random(V) < 0.99] = -np.inf
        rows.append(x)
    return np.stack(rows)


@pytest.mark.parametrize("B,V,pad,dtype", [(20, 248320, 0, torch.bfloat16), (66, 163840, 0, torch.float32),
                                           (40, 100003, 3, torch.float16), (70, 8192, 0, torch.float32)])
def test_top_k_above_what_a_bound_lists(dev, B, V, pad, dtype):
    """top_k up to 256 where the chunks' bounds let more candidates through than a list holds."""
    rng = np.random.default_rng(B)
    x = hard_lists(rng, V, B)
    ps = [Sampling(top_k=int([256, 100, 200, 127, 129, 160, 128, 255, 64][r % 9]), top_p=float([1.0, 0.9][r % 2]), temperature=1.3)
          for r in range(B)]
    u = (np.floor(rng.random(B) * 4000) + 0.37) / 4000  # equal masses: draws off the multiples of 1 / n
    check(dev, x, ps, u, dtype=dtype, pad=pad, label=f"top-k lists {B}x{V}", max_excused=1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [16, 64])
def test_top_lists_of_tied_values(dev, k, dtype):
    rng = np.random.default_rng(k)
    B, V = 32, 100008
    xt, x = rows_on(dev, hard_lists(rng, V, B), dtype, 0)
    print(f"[tied lists] k={k} {dtype}", flush=True)
    ids, vals = topk_batch(xt, k)
    ids, vals = ids.cpu().numpy(), vals.cpu().numpy()
    for r in range(B):
        ri, rv = DR.topk_sorted(x[r], k)
        assert np.array_equal(ids[r], ri) and np.array_equal(vals[r], rv), (k, r)


@pytest.mark.parametrize("B,V,pad,dtype", [(24, 131072, 0, torch.float16), (66, 8192, 0, torch.float32),
                                           (66, 32771, 1, torch.float32), (48, 163840, 0, torch.bfloat16)])
def test_top_k_above_the_lists(dev, B, V, pad, dtype):
    """top_k above 256: gathered by one pass and finished in one workgroup up to 2048, by radix selects above and where
    too many keys share the cut's bin; rows whose tiles stay in LDS between the passes and (48 rows) rows read again."""
    rng = np.random.default_rng(V)
    x = np.concatenate([hard_lists(rng, V, B // 2), (rng.standard_t(3, (B - B // 2, V)) * 3).astype(np.float32)])
    low = -60000.0 if dtype == torch.float16 else -1e9
    for r in range(0, B, 4):
        x[r, rng.random(V) < 0.3] = low  # masked by a large negative value: the values' range says nothing
    ks = [257, 300, 1000, 2047, 2048, 2049, 5000, 512, 513]
    ps = [Sampling(top_k=ks[r % 9], top_p=float([1.0, 0.9, 0.3][r % 3]), min_p=float([0.0, 0.0, 0.02, 0.0, 0.3][r % 5]),
                   temperature=float([1.0, 0.6, 1.8][r % 3])) for r in range(B)]
    u = (np.floor(rng.random(B) * 4000) + 0.37) / 4000
    check(dev, x, ps, u, dtype=dtype, pad=pad, label=f"large top-k {B}x{V}", max_excused=1)


@pytest.mark.parametrize("kind", ["flat", "min_p", "tied", "top_k"])
def test_open_rows_repeat_bit_for_bit(dev, kind):
    """Rows that several workgroups finish together add their masses up in an order of no kind: the results must not
    depend on it."""
    rng = np.random.default_rng(21)
    B, V = 66, 40000
    x = (rng.standard_normal((B, V)) * (0.1 if kind != "top_k" else 2.0)).astype(np.float32)
    if kind == "tied":
        x = np.round(x * 20) / 20
    kw = dict(flat=dict(top_p=0.9), min_p=dict(min_p=0.7), tied=dict(top_p=0.9, min_p=0.7), top_k=dict(top_k=6000))[kind]
    rows = ops.pack_rows([Sampling(temperature=0.9, **kw)] * B, rng.random(B), V).to(dev)
    xt = torch.from_numpy(x).to(dev)
    print(f"[repeat] {kind}", flush=True)
    first = ops.sample_rows(xt, rows).block.clone()
    for _ in range(12):
        assert torch.equal(ops.sample_rows(xt, rows).block, first)


@pytest.mark.parametrize("down", [8.0, 10.0, 12.0])
def test_mass_of_the_unlisted_logits(dev, down):
    """Requests without a cut that draw a listed token: the logprob is the logarithm of the row's mass, half of it in
    tied logits far below the maximum that no list holds, at the temperatures where (x - max) (log2 e / t) in float32 is
    furthest from the quotients' difference. Each mass is within 2 ulp of its exponential (2.4e-7), a tree of four adds 2
    halves of an ulp (1.2e-7), on at most 0.55 of the mass; the float32 logarithm and the result add an ulp of the logprob
    (below 1) each: 0.55 * 3.6e-7 + 1.0e-7 = 3.0e-7 in all, for every temperature."""
    rng = np.random.default_rng(int(down))
    B, V = 66, 163840
    f = np.float32
    ts = rng.uniform(0.6, 1.4, 100000).astype(f)
    x0 = f(5) - f(down) * ts
    folded = np.exp2(((x0 - f(5)) * (f(np.log2(np.e)) / ts)).astype(np.float64))
    ts = ts[np.argsort(-np.abs(folded / np.exp((x0 / ts).astype(np.float64) - f(5) / ts) - 1))[:B]]
    x = np.empty((B, V), np.float32)
    for r in range(B):  # a maximum of 5, a floor whose mass is about 1, logits above it to list, the rest near nothing
        x[r] = 5.0 - 38.0 * ts[r]
        at = rng.permutation(V)
        x[r, at[:min(int(np.exp(down)), V - V // 50)]] = f(5) - f(down) * ts[r]
        x[r, at[V - V // 60:]] = 5.0 - ts[r] * (down - 0.5 - 0.3 * rng.random(V // 60))
        x[r, at[V - V // 60 - 1]] = 5.0
    rows = ops.pack_rows([Sampling(temperature=float(t)) for t in ts], np.full(B, 1e-9), V).to(dev)
    print(f"[mass] {down}", flush=True)
    o = ops.sample_rows(torch.from_numpy(x).to(dev), rows)
    lp = o.logprobs.cpu().numpy().astype(np.float64)
    assert np.array_equal(o.ids.cpu().numpy(), x.argmax(1))
    assert np.all(o.keep.cpu().numpy() == V)
    done = ops.workspace(dev, 64 * _lib.load().vs_sample_workspace_bytes(1, V))[64:64 + 56]  # the rows' open flags
    assert int(done.sum()) == 0  # finished from the lists
    xs = x / ts[:, None]  # float32, as the sampler divides
    d = xs.astype(np.float64) - xs.max(1, keepdims=True)
    want = -np.log(np.where(d >= -40.0, np.exp(d), 0.0).sum(1))
    err = np.abs(lp - want)
    print(f"[mass] largest error {err.max():.2e}, mean {np.mean(lp - want):.2e}", flush=True)
    assert err.max() <= 3.0e-7


def test_logprobs_have_no_bias(dev):
    """Nucleus rows of a language model's shape: the logprob is the float32 difference the reference takes less the
    logarithm of the kept mass, rounded once. Masses (2 ulp), the logarithm and the result (an ulp of a few units) leave
    a row's error within about 2.5e-7 of no preferred sign, so the mean over 128 rows within 3 * 2.5e-7 / sqrt(128)."""
    rng = np.random.default_rng(31)
    B, V, n = 128, 32768, 900
    ts = rng.uniform(0.6, 1.1, B).astype(np.float32)
    x = (rng.standard_normal((B, V)) * 2).astype(np.float32)
    for r in range(B):
        x[r, rng.choice(V, n, replace=False)] = (16.0 - rng.random() * 0.6 * np.arange(n) ** 0.4
                                                 + 0.3 * rng.standard_normal(n)).astype(np.float32)
    ps = [Sampling(temperature=float(t), top_p=0.8) for t in ts]
    u = rng.random(B)
    print("[bias] 128 rows", flush=True)
    o = sample_batch(torch.from_numpy(x).to(dev), ps, u)
    refs = [S.sample(x[r], ps[r], float(u[r])) for r in range(B)]
    check_sample(o, refs, "logprobs", 1)
    lp, ids, keep = (t.cpu().numpy() for t in (o.logprobs, o.ids, o.keep))
    err = [float(lp[r]) - f.logprob for r, f in enumerate(refs) if ids[r] == f.token and keep[r] == f.keep]
    print(f"[bias] mean {np.mean(err):.2e}, largest {np.max(np.abs(err)):.2e}", flush=True)
    assert abs(np.mean(err)) <= 3 * 2.5e-7 / np.sqrt(B)
