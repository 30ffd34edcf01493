"""K8 (softmax-max of logit rows) and K9 (low-confidence unmasking) on the
GPU, through the C ABI, against the oracle (oracle/sampler.py).

x0 must equal the oracle's index on every row whose result does not depend
on the summation order of s (the oracle evaluated with s scaled by 1 +- 4e-6
agrees); that is all rows but a handful, and the test requires >= 99 %.  x0_p
is bf16(1/s): within one bf16 unit everywhere and equal on >= 98 % of rows.
The unmasking kernel is bit-exact against the oracle given the same
predictions and confidences."""
import numpy as np
import pytest
import torch

from helpers import bits

from oracle import sampler as osm
from oracle.bf16 import f32_to_bf16_bits
from dllm_serve_amd import _capi

pytestmark = pytest.mark.gpu

MASK = 126336


def _run_k8(logits):
    M, V = logits.shape
    x0 = torch.full((M,), -1, dtype=torch.int64, device=logits.device)
    p = torch.zeros(M, dtype=torch.bfloat16, device=logits.device)
    ws = torch.empty(max(16, _capi.softmax_max_workspace_size(M, V)), dtype=torch.uint8, device=logits.device)
    _capi.softmax_max(logits, x0, p, ws)
    torch.cuda.synchronize()
    return x0.cpu().numpy(), bits(p)


def _check_k8(logits_host_bits, x0, p):
    ox0, op = osm.softmax_max(logits_host_bits)
    lo0, _ = osm.softmax_max(logits_host_bits, 1 - 4e-6)
    hi0, _ = osm.softmax_max(logits_host_bits, 1 + 4e-6)
    robust = (lo0 == ox0) & (hi0 == ox0)
    assert robust.mean() >= 0.99
    bad = np.nonzero(robust & (x0 != ox0))[0]
    assert bad.size == 0, f"x0 differs on rows {bad[:8]}: got {x0[bad[:8]]} want {ox0[bad[:8]]}"
    d = np.abs(p.astype(np.int32) - op.astype(np.int32))
    assert d.max() <= 1 and np.mean(d == 0) >= 0.98, f"x0_p: max diff {d.max()}, equal {np.mean(d == 0):.4f}"


@pytest.mark.parametrize("M,V,sigma,pad", [
    (64, 126464, 1.3, 0),       # LLaDA vocabulary, logits of the random-weight model's scale
    (256, 126464, 3.0, 8),      # C2 cached step row count, strided rows
    (1024, 126464, 1.3, 0),     # C2 dense step row count
    (96, 152064, 2.0, 0),       # Dream vocabulary
    (300, 4096, 0.3, 0),        # |max| <= 2: the rounding-tie rescan runs on every row
    (513, 4104, 0.4, 8),        # more than 512 rows: 256-thread workgroups, rescan rows, strided
    (37, 264, 0.5, 8),
    (5, 8, 1.0, 0),
])
def test_softmax_max_matches_oracle(dev, M, V, sigma, pad):
    print(f"softmax_max M={M} V={V} sigma={sigma} pad={pad}", flush=True)
    g = torch.Generator().manual_seed(M * 7 + V)
    full = (torch.randn(M, V + pad, generator=g) * sigma).to(torch.bfloat16)
    full[:, V:] = 100.0                              # padding columns must be ignored
    logits = full.to(dev)[:, :V]
    x0, p = _run_k8(logits)
    _check_k8(bits(full[:, :V]), x0, p)


@pytest.mark.parametrize("M,V,sigma,pad,T", [
    (1, 126464, 2.0, 0, 0.0),        # one row over eight workgroups
    (20, 16384, 0.3, 0, 0.0),        # ranges merged by the second launch, rescan on every row
    (3, 8232, 1.0, 8, 0.0),          # 1029 chunks in two ranges, strided
    (64, 126464, 2.0, 0, 0.0),       # the most rows that are split
    (5, 33288, 2.0, 8, 1.0),         # noisy: sixteen ranges of 4161 chunks
    (128, 16392, 2.0, 0, 0.5),       # noisy: the most rows that are split
])
def test_softmax_max_split_rows(dev, M, V, sigma, pad, T):
    """Rows spread over several workgroups (a workspace given) against the
    oracle, and the same call with a null and a short workspace."""
    print(f"softmax_max split M={M} V={V} sigma={sigma} pad={pad} T={T}", flush=True)
    full = (torch.randn(M, V + pad, generator=torch.Generator().manual_seed(V)) * sigma).to(torch.bfloat16)
    full[:, V:] = 100.0                              # padding columns must be ignored
    logits = full.to(dev)[:, :V]
    temps = torch.full((M,), T, dtype=torch.float64, device=dev)
    need = _capi.softmax_max_split_workspace_size(M, V)
    assert need > 0
    for nbytes in (need, need - 1, 0):
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev) if nbytes else None
        x0 = torch.full((M,), -1, dtype=torch.int64, device=dev)
        p = torch.zeros(M, dtype=torch.bfloat16, device=dev)
        if T:
            _capi.softmax_max_sample(logits, temps, 31, 2, x0, p, ws)
            _check_sample(bits(full[:, :V]), np.full(M, T), 31, 2, x0.cpu().numpy(), bits(p))
        else:
            _capi.softmax_max(logits, x0, p, ws)
            _check_k8(bits(full[:, :V]), x0.cpu().numpy(), bits(p))


def test_softmax_max_ties_and_neg_inf(dev):
    print("softmax_max ties / -inf", flush=True)
    V = 126464
    g = torch.Generator().manual_seed(3)
    rows = (torch.randn(6, V, generator=g) * 1.5)
    rows[0, [5000, 17, 90000]] = 9.0                 # exact ties of the maximum: first index
    rows[1, :] = 0.75                                # uniform row: index 0
    rows[2, ::3] = -float("inf")                     # -inf columns
    rows[3, 100000:] = -float("inf")
    rows[3, 126463] = -float("inf")
    rows[4, :] = 0.28125                             # rounding tie: index 3 beats index 10
    rows[4, 3], rows[4, 10] = 1.0 - 2 ** -8, 1.0
    rows[5, 126463] = 12.0                           # maximum in the very last column
    t = rows.to(torch.bfloat16)
    x0, p = _run_k8(t.to(dev))
    ox0, op = osm.softmax_max(bits(t))
    assert x0[0] == 17 and x0[1] == 0 and x0[4] == 3 and x0[5] == 126463
    assert np.array_equal(x0, ox0)
    assert np.all(np.abs(p.astype(np.int32) - op.astype(np.int32)) <= 1)


def _unmask_case(rng, n_seq, max_win, tie_levels):
    tokens, params, rows = [], [], 0
    for b in range(n_seq):
        n = int(rng.integers(0, max_win + 1)) if b else max_win
        pad = int(rng.integers(0, 9))
        tok = rng.integers(0, 1000, n + pad)
        tok[pad:][rng.random(n) < rng.random()] = MASK
        steps = int(rng.integers(-1, 9))
        if b == 0:  # the longest window, masked to its last position, of which some are unmasked
            tok[-1] = MASK
            steps = 2
        params.append((len(tokens) + pad, n, rows, steps, int(rng.random() < 0.5)))
        tokens.extend(tok.tolist())
        rows += n
    conf = f32_to_bf16_bits(np.round(rng.random(rows) * tie_levels) / tie_levels) if tie_levels else \
        f32_to_bf16_bits(rng.random(rows).astype(np.float32))
    x0 = rng.integers(1000, 126000, rows)
    return np.array(tokens, np.int64), params, conf, x0


@pytest.mark.parametrize("n_seq,max_win,ties", [(64, 300, 0), (64, 300, 16), (8, 8192, 64), (3, 1, 0), (32, 64, 2),
                                               # edges of the one-wavefront forms (64, 256 and 1024 positions)
                                               (20, 65, 4), (20, 256, 0), (20, 257, 3), (20, 1024, 8),
                                               (20, 1025, 8)])
def test_unmask_matches_oracle(dev, n_seq, max_win, ties):
    print(f"unmask n_seq={n_seq} max_win={max_win} ties={ties}", flush=True)
    rng = np.random.default_rng(n_seq * 31 + max_win + ties)
    tokens, params, conf, x0 = _unmask_case(rng, n_seq, max_win, ties)
    assert max(w[1] for w in params) == max_win  # the kernel form goes by the longest window
    want, want_n = osm.unmask_step(tokens, params, x0, conf, MASK)
    assert want_n[0] > 0
    t = torch.from_numpy(tokens).to(dev)
    p = torch.tensor(params, dtype=torch.int32).to(dev)
    cf = torch.from_numpy(conf.view(np.int16)).view(torch.bfloat16).to(dev)
    xd = torch.from_numpy(x0).to(dev)
    nun = torch.full((n_seq,), -1, dtype=torch.int32, device=dev)
    _capi.lowconf_unmask(t, p, n_seq, max_win, xd, cf, MASK, nun)
    torch.cuda.synchronize()
    got = t.cpu().numpy()
    assert np.array_equal(nun.cpu().numpy(), want_n)
    bad = np.nonzero(got != want)[0]
    assert bad.size == 0, f"{bad.size} tokens differ, first at {bad[:8]}"


def test_remask_sampler_step_matches_oracle(dev):
    """RemaskSampler on a mixed batch (no SparseConfig, and sparse sequences
    in the full-attention, compute-cache and reuse states): LM head by torch
    (a library GEMM), K8 + K9 against the oracle on the same logits."""
    from dllm_serve_amd.engine.sampler import RemaskSampler, step_windows
    from dllm_serve_amd.engine.sequence import Sequence
    from dllm_serve_amd.sparse.state import SparseConfig

    print("remask sampler step", flush=True)
    H, V = 512, 126464
    g = torch.Generator().manual_seed(21)
    w = (torch.randn(V, H, generator=g) * 0.05).to(torch.bfloat16).to(dev)
    cfg = SparseConfig(enabled=True, default_block_len=32, retention_ratio=0.5, delay_step=1)
    seqs = [Sequence([1] * 40, 64, MASK, None, device=dev, steps=16),
            Sequence([2] * 50, 64, MASK, cfg, device=dev),
            Sequence([3] * 30, 70, MASK, cfg, device=dev),
            Sequence([4] * 20, 32, MASK, cfg, device=dev)]
    seqs[0].current_step = 5
    seqs[2].advance()                                 # compute-cache state
    for _ in range(2):
        seqs[3].advance()                             # reuse state
    # partly unmasked windows
    N = max(s.num_tokens for s in seqs)
    host = np.zeros((len(seqs), N), np.int64)
    rng = np.random.default_rng(4)
    for b, s in enumerate(seqs):
        tok = np.array(s.token_ids)
        tok[s.num_prompt_tokens:][rng.random(s.gen_length) < 0.3] = 777
        host[b, :s.num_tokens] = tok
    tokens = torch.from_numpy(host).to(dev)
    n_rows = sum(s.step_rows()[1] for s in seqs)
    hidden = torch.randn(n_rows, H, generator=g).to(torch.bfloat16).to(dev)
    sampler = RemaskSampler(lambda h: h @ w.t(), MASK, max_logprobs=64)
    nun = sampler(hidden, seqs, tokens)
    torch.cuda.synchronize()
    # oracle on the same logits
    win = step_windows(seqs)
    sel = torch.cat([torch.arange(h0, h0 + n) for h0, _, n, _, _ in win]).to(dev)
    rows = hidden.index_select(0, sel)
    logits = torch.cat([rows[a:a + 64] @ w.t() for a in range(0, rows.shape[0], 64)])  # the sampler's chunks
    lb = bits(logits)
    x0, p = _run_k8(logits)
    _check_k8(lb, x0, p)
    params, r = [], 0
    for b, (h0, lo, n, sr, first) in enumerate(win):
        params.append((b * N + lo, n, r, sr, first))
        r += n
    want, want_n = osm.unmask_step(host.reshape(-1), params, x0, p, MASK)
    assert np.array_equal(nun.cpu().numpy(), want_n)
    assert np.array_equal(tokens.cpu().numpy().reshape(-1), want)
    assert want_n.sum() > 0


def _run_k8_sample(logits, temps, seed, row_base):
    M, V = logits.shape
    x0 = torch.full((M,), -1, dtype=torch.int64, device=logits.device)
    p = torch.zeros(M, dtype=torch.bfloat16, device=logits.device)
    ws = torch.empty(max(16, _capi.softmax_max_workspace_size(M, V)), dtype=torch.uint8, device=logits.device)
    t = torch.tensor(temps, dtype=torch.float64, device=logits.device)
    _capi.softmax_max_sample(logits, t, seed, row_base, x0, p, ws)
    torch.cuda.synchronize()
    return x0.cpu().numpy(), bits(p)


def _check_sample(lb, temps, seed, row_base, x0, p):
    """x0 equal to the oracle's on >= 99 % of rows; elsewhere the kernel's
    choice must be a near-tie (its transformed value within one bf16 unit of
    the maximum, from last-place differences of f64 exp / log)."""
    ox0, op = osm.softmax_max_sample(lb, temps, seed, row_base)
    bad = np.nonzero(x0 != ox0)[0]
    assert len(bad) <= 0.01 * len(x0), f"{len(bad)} rows differ"
    for r in bad:
        T = temps[r]
        v = osm.gumbel_transform(lb[r], T, osm.uniforms(seed, row_base + r, lb.shape[1])) if T > 0 else lb[r]
        vv = v.astype(np.int32)
        assert abs(vv[x0[r]] - vv[ox0[r]]) <= 1, (r, x0[r], ox0[r])
    d = np.abs(p.astype(np.int32) - op.astype(np.int32))
    assert d.max() <= 1 and np.mean(d == 0) >= 0.98


def test_softmax_max_sample_matches_oracle(dev):
    print("softmax_max_sample V=126464", flush=True)
    M, V = 64, 126464
    g = torch.Generator().manual_seed(77)
    t = (torch.randn(M, V, generator=g) * 2.0).to(torch.bfloat16)
    temps = [[0.0, 0.5, 1.0, 2.0][r % 4] for r in range(M)]
    seed, row_base = 0x1234_5678_9ABC, 17
    x0, p = _run_k8_sample(t.to(dev), temps, seed, row_base)
    _check_sample(bits(t), np.array(temps), seed, row_base, x0, p)
    # rows split over two calls draw the same noise (counter = global row index)
    td = t.to(dev)
    a0, ap = _run_k8_sample(td[:40], temps[:40], seed, row_base)
    b0, bp = _run_k8_sample(td[40:], temps[40:], seed, row_base + 40)
    assert np.array_equal(np.concatenate([a0, b0]), x0) and np.array_equal(np.concatenate([ap, bp]), p)


def test_remask_sampler_with_temperature(dev):
    """RemaskSampler at temperature 1.0 for two sequences and 0 for one:
    x0 / x0_p from the oracle's Gumbel transform with the sampler's seed."""
    from dllm_serve_amd.engine.sampler import RemaskSampler, step_windows
    from dllm_serve_amd.engine.sequence import Sequence

    print("remask sampler temperature", flush=True)
    H, V = 256, 4096
    g = torch.Generator().manual_seed(5)
    w = (torch.randn(V, H, generator=g) * 0.2).to(torch.bfloat16).to(dev)
    seqs = [Sequence([1] * 30, 48, MASK, None, device=dev, steps=12) for _ in range(3)]
    N = seqs[0].num_tokens
    tok = torch.tensor([s.token_ids for s in seqs], dtype=torch.int64, device=dev)
    hidden = torch.randn(3 * N, H, generator=g).to(torch.bfloat16).to(dev)
    sampler = RemaskSampler(lambda h: h @ w.t(), MASK, seed=5)
    temps = [1.0, 0.0, 1.0]
    nun = sampler(hidden, seqs, tok, temperature=temps)
    torch.cuda.synchronize()
    win = step_windows(seqs)
    sel = torch.cat([torch.arange(h0, h0 + n) for h0, _, n, _, _ in win]).to(dev)
    logits = hidden.index_select(0, sel) @ w.t()
    lb = bits(logits)
    row_t = np.concatenate([np.full(n, temps[b]) for b, (_, _, n, _, _) in enumerate(win)])
    seed_used = (5 * 0x9E3779B97F4A7C15) & 0xFFFFFFFFFFFFFFFF
    ox0, op = osm.softmax_max_sample(lb, row_t, seed_used, 0)
    params, r = [], 0
    for b, (h0, lo, n, sr, first) in enumerate(win):
        params.append((b * N + lo, n, r, sr, first))
        r += n
    host = np.array([s.token_ids for s in seqs], np.int64).reshape(-1)
    want, want_n = osm.unmask_step(host, params, ox0, op, MASK)
    assert np.array_equal(nun.cpu().numpy(), want_n)
    got = tok.cpu().numpy().reshape(-1)
    assert np.mean(got == want) > 0.99   # rows whose f64 noise rounds differently may pick another token
    assert np.array_equal(got != MASK, want != MASK) or np.mean((got != MASK) == (want != MASK)) > 0.99


@pytest.mark.parametrize("M,V,sigma,T", [
    (3, 8, 1.0, 1.0),            # one chunk: lanes without logits
    (5, 520, 0.1, 1.0),          # 65 chunks, small values: nothing may be left out
    (9, 1032, 2.0, 0.25),
    (513, 4104, 3.0, 0.7),       # 256-thread workgroups
    (4, 33288, 6.0, 3.0),        # a second round of loads, partly past the row's end
])
def test_softmax_max_sample_bounds(dev, M, V, sigma, T):
    """The bound that leaves logits out of the f64 transform: row lengths at
    the edges of the chunk walk, values below and far above the gap."""
    print(f"softmax_max_sample bounds M={M} V={V} sigma={sigma} T={T}", flush=True)
    g = torch.Generator().manual_seed(M + V)
    t = (torch.randn(M, V, generator=g) * sigma).to(torch.bfloat16)
    t[0, ::3] = -float("inf")
    x0, p = _run_k8_sample(t.to(dev), [T] * M, 99, 5)
    _check_sample(bits(t), np.full(M, T), 99, 5, x0, p)


def test_softmax_max_sample_overflow(dev):
    """Values past the largest bf16 are infinite (the reference's too): the
    first infinite one is the token, its probability NaN."""
    print("softmax_max_sample overflow", flush=True)
    t = torch.zeros(2, 8200, dtype=torch.bfloat16)
    t[0, [700, 41, 8199]] = 95.0     # exp(95) / E > 3.4e38 for every draw (E < 37)
    t[1, [8199, 3000]] = 80.0        # large, finite
    x0, p = _run_k8_sample(t.to(dev), [1.0, 1.0], 7, 0)
    assert x0[0] == 41 and np.isnan(torch.from_numpy(p[:1].view(np.int16)).view(torch.bfloat16).float().item())
    _check_sample(bits(t[1:]), np.array([1.0]), 7, 1, x0[1:], p[1:])


@pytest.mark.parametrize("V", [64, 4104, 33288])
@pytest.mark.parametrize("workspace", [False, True])
def test_softmax_max_sample_without_a_threshold(dev, V, workspace):
    """Rows whose values stay below the gap are computed whole; one large value
    anywhere (first and last column, a later round of chunks) ends that."""
    print(f"softmax_max_sample no threshold V={V} workspace={workspace}", flush=True)
    g = torch.Generator().manual_seed(V)
    at = [None, 0, 7, V // 2, V - 9, V - 1]
    M, T = len(at), 0.4
    t = (torch.randn(M, V, generator=g) - 6.0).to(torch.bfloat16)
    for r, c in enumerate(at):
        if c is not None:
            t[r, c] = 12.0
    logits = t.to(dev)
    temps = torch.full((M,), T, dtype=torch.float64, device=dev)
    x0 = torch.full((M,), -1, dtype=torch.int64, device=dev)
    p = torch.zeros(M, dtype=torch.bfloat16, device=dev)
    need = _capi.softmax_max_split_workspace_size(M, V)
    ws = torch.empty(need, dtype=torch.uint8, device=dev) if workspace and need else None
    _capi.softmax_max_sample(logits, temps, 17, 0, x0, p, ws)
    assert all(int(x0[r]) == c for r, c in enumerate(at) if c is not None)
    _check_sample(bits(t), np.full(M, T), 17, 0, x0.cpu().numpy(), bits(p))
