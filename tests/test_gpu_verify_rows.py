"""vs_verify_greedy on blocks of many rows (one pass over all rows and a merge) against the NumPy oracle.

The logprob's bound is the one of the other verify tests; what this path adds to it are sums of at most 32 exponentials per
float accumulator (32 * 2^-24 = 2e-6 relative, in the logarithm of the sum an absolute error that small)."""
import numpy as np
import pytest
import torch

from oracle import verify_ref as VR
from volundr_amd import verify_greedy

pytestmark = pytest.mark.gpu
CUS = 256
TILE = {torch.float32: 256 * 32, torch.bfloat16: 256 * 64, torch.float16: 256 * 64}


def block(dev, B, T, V, ld, off, dtype, seed):
    """[B, T, V] view of rows ld apart that begins `off` logits after an allocation's start."""
    g = torch.Generator(device=dev).manual_seed(seed)
    base = torch.full((off + B * T * ld,), float("nan"), dtype=dtype, device=dev)  # what lies between rows is never used
    x = base[off:].view(B, T, ld)[:, :, :V]
    x.copy_(torch.randn((B, T, V), generator=g, device=dev) * 3.0)
    return x


def check(o, x, drafts, vv, label):
    ref = x.float().cpu().numpy()
    tok, acc, lp = VR.verify(ref, drafts, vv)
    assert np.array_equal(o.argmax.cpu().numpy(), tok), label
    assert np.array_equal(o.accept.cpu().numpy(), acc), label
    g = o.logprobs.cpu().numpy().astype(np.float64)
    ok = np.isfinite(lp) & np.isfinite(ref[..., :vv]).all(-1)
    assert np.all((np.abs(g - lp) <= 1e-5 * np.abs(lp) + 1e-6)[ok]), (label, np.max(np.abs(g - lp)[ok]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("edge", ["tile", "tile+1", "tile-1", "two+7", "wave"])
@pytest.mark.parametrize("mis", [(0, 0), (5, 0), (3, 1)])
def test_edges(dev, dtype, edge, mis):
    """Rows that end at a tile's edge, one before and one past it, in the middle of a wave's part, and aligned and
    unaligned starts of every kind; the maximum planted in the first and last places, ties across tiles."""
    tile = TILE[dtype]
    V = {"tile": tile, "tile+1": tile + 1, "tile-1": tile - 1, "two+7": 2 * tile + 7, "wave": tile + 700}[edge]
    off, pad = mis
    T = 7
    B = 8 * CUS // -(-V // tile) // T + 1  # more rows than one launch of the other path holds
    vv = V - (3 if edge == "wave" else 0)
    x = block(dev, B, T, V, V + pad, off, dtype, 3)
    r = torch.arange(B * T, device=dev)
    places = torch.tensor([0, vv - 1, min(tile, vv) - 1, min(tile, vv - 1), vv // 2, 8, vv - 2], device=dev)
    x[r // T, r % T, places[r % 7]] = 20.0
    x[:, 2, vv - 1] = 20.0  # a tie across tiles: the first one wins
    if vv < V:
        x[:, :, vv:] = 60.0 if dtype != torch.float16 else 100.0  # above everything, outside vocab_valid
    some = torch.tensor(sorted({*range(2 * T), *range(B - T, B)}), device=dev)  # the oracle's share of the requests
    tok = places[r % 7].view(B, T).cpu().numpy().astype(np.int32)
    drafts = tok[:, :-1].copy()
    for b in range(B):
        if b % T < T - 1:
            drafts[b, b % T] = (drafts[b, b % T] + 1) % vv
    print(f"[edges] {dtype} {edge} V={V} B={B} T={T} off={off} pad={pad}", flush=True)
    o = verify_greedy(x, torch.from_numpy(drafts).to(dev), vv)
    torch.cuda.synchronize()
    assert np.array_equal(o.argmax.cpu().numpy(), tok)
    assert np.array_equal(o.accept.cpu().numpy(), np.arange(B) % T)
    sub = some.cpu().numpy()
    part = type(o)(o.argmax[some], o.accept[some], o.logprobs[some])
    check(part, x[some], drafts[sub], vv, (dtype, edge, mis))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("pad", [0, 3])
def test_odd_values(dev, dtype, pad):
    """NaN ranks first, then +inf; rows of -inf alone give 0; values by the type's lowest; signed zeros tie."""
    V, T, B = 40007 if pad else 40008, 9, 120
    x = block(dev, B, T, V, V + pad, 0, dtype, 4)
    low = torch.finfo(dtype).min
    for b in range(0, B, 5):
        x[b, 0, 100] = 3.0
        x[b, 0, 30000] = float("nan")
        x[b, 1, 25000] = float("nan")
        x[b, 1, V - 1] = float("nan")
        x[b, 2, 35000] = float("inf")
        x[b, 2, 12000] = float("inf")
        x[b, 3, :] = float("-inf")
        x[b, 4, :] = float("-inf")
        x[b, 4, V - 1] = low
        x[b, 5, :] = low
        x[b, 6, :] = float("-inf")
        x[b, 6, 17:20000:3] = -1.5
        x[b, 7, :] = -60000.0 if dtype == torch.float16 else -2e38
        x[b, 7, 20011] = -59000.0 if dtype == torch.float16 else -1.9e38
        x[b, 8, :] = -1.0
        x[b, 8, 300] = -0.0
        x[b, 8, 20000] = 0.0
    ref = x.float().cpu().numpy()
    want = np.argmax(ref, -1).astype(np.int32)
    drafts = want[:, :-1].copy()
    print(f"[odd] {dtype} pad={pad} B={B} T={T} V={V}", flush=True)
    o = verify_greedy(x, torch.from_numpy(drafts).to(dev), V)
    torch.cuda.synchronize()
    assert np.array_equal(o.argmax.cpu().numpy(), want)
    assert (o.accept.cpu().numpy() == T - 1).all()
    lp = o.logprobs.cpu().numpy().astype(np.float64)
    r64 = ref.astype(np.float64)
    for b in range(B):
        for j in range(T):
            m = r64[b, j, want[b, j]]
            if not np.isfinite(m) or not (r64[b, j] < np.inf).all():
                assert lp[b, j] == 0.0 or not np.isfinite(m), (b, j)
                continue
            exp = -np.log(np.exp(np.maximum(r64[b, j] - m, -1e4)).sum())
            # the maximum's own rounding in m - (m + log S) is absorbed by evaluating it in 64 bits
            assert abs(lp[b, j] - exp) <= 1e-5 * abs(exp) + 1e-6 + abs(m) * 2.0 ** -52, (b, j, lp[b, j], exp)


@pytest.mark.parametrize("T", [1, 2, 70])
def test_block_lengths(dev, T):
    V = 30000
    B = 1200 // T + 1
    x = block(dev, B, T, V, V, 0, torch.bfloat16, T)
    tok = x.float().argmax(-1).cpu().numpy()
    drafts = tok[:, :-1].astype(np.int32).copy()
    for b in range(B):
        if T > 1 and b % T < T - 1:
            drafts[b, b % T] += 1
    print(f"[lengths] B={B} T={T}", flush=True)
    o = verify_greedy(x, torch.from_numpy(drafts).to(dev) if T > 1 else None, V)
    torch.cuda.synchronize()
    check(o, x, drafts, V, T)


def test_graph_replays_between_other_calls(dev):
    """Replays of a captured call, with calls of few rows on the same workspace between them."""
    B, T, V = 40, 17, 65536
    x = block(dev, B, T, V, V, 0, torch.bfloat16, 8)
    tok = x.float().argmax(-1)
    drafts = tok[:, :-1].to(torch.int32).contiguous()
    few, fd = x[:1].clone(), drafts[:1].clone()
    want_few = verify_greedy(few, fd, V).argmax.clone()
    verify_greedy(x, drafts, V)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        o = verify_greedy(x, drafts, V)
    for i in range(4):
        x.copy_(block(dev, B, T, V, V, 0, torch.bfloat16, 20 + i))
        d = x.float().argmax(-1)[:, :-1].to(torch.int32)
        d[:, i] += 1
        drafts.copy_(d)
        g.replay()
        assert torch.equal(verify_greedy(few, fd, V).argmax, want_few)
        torch.cuda.synchronize()
        check(o, x, drafts.cpu().numpy(), V, i)


@pytest.mark.parametrize("dtype,line", [(torch.float32, 4 << 20), (torch.bfloat16, 2 << 20), (torch.float16, 3 << 20)])
@pytest.mark.parametrize("V", [16381, 100003, 8193])
def test_unaligned_rows_around_the_line(dev, dtype, line, V):
    """Few unaligned rows take the one-launch kernel below a number of logits and the two launches from there on (rows
    that fill their workgroups badly keep to the first): both give the oracle's answer."""
    for n in (line // V, line // V + 1):
        T = 3
        B = -(-n // T)
        x = block(dev, B, T, V, V, 0, dtype, n)
        tok = x.float().argmax(-1).cpu().numpy()
        drafts = tok[:, :-1].astype(np.int32).copy()
        drafts[::2, 1] += 1
        print(f"[line] {dtype} V={V} B={B} T={T}", flush=True)
        o = verify_greedy(x, torch.from_numpy(drafts).to(dev), V)
        torch.cuda.synchronize()
        check(o, x, drafts, V, (dtype, V, n))
