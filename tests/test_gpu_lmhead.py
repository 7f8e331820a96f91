"""The fused lm-head product (lcs_lmhead, lcs_lmhead.hip) through the C ABI.

Two gates, as for every kernel here:
- the logits against the exact product: bit-exact on small-integer operands
  (every bf16 product and every partial sum is then an exactly representable
  f32 integer), and within K * 2^-24 * sum_k |x_k w_k| of the float64 product
  on random operands (f32 accumulation of exact bf16 x bf16 products);
- the epilogue's statistics against the kernel's own written logits: argmax
  bit-exact with the first-index rule (llama.cpp:1237-1245), the draft
  logprob and acceptance length against the oracle's verify
  (sampling.cpp:150-170, engine.cpp:357-383), log_z (returned in f32)
  within 1e-5 plus half an f32 spacing of the float64 log-sum-exp.
"""
import sys
from types import SimpleNamespace

import numpy as np
import pytest

from oracle import pyoracle as O
from tests.util import LOGPROB_TOL

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


@pytest.fixture(scope="module")
def sampler():
    from locus_amd.sampler import Sampler
    s = Sampler(device=0, max_rows=512, max_vocab=262144, max_hist=64, max_top=4)
    yield s
    s.close()


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def bf16(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(torch.bfloat16)


def run(sampler, x, w, draft=None, rows_per_seq=0, logits=True):
    """x (rows, hidden), w (vocab, hidden) bf16 on the device."""
    torch = sampler.torch
    rows, vocab = x.shape[0], w.shape[0]
    n_seq = rows // rows_per_seq if (rows_per_seq and draft is not None) else 0
    out = sampler.alloc_lmhead_out(rows, vocab, logits=logits, draft=draft is not None, n_seq=n_seq)
    sampler.lmhead_dev(x, w, out, draft=draft, rows_per_seq=rows_per_seq)
    torch.cuda.synchronize()
    return {k: v.cpu().numpy() for k, v in out.items()}


def logsumexp64(l):
    l = l.astype(np.float64)
    m = l.max(axis=1, keepdims=True)
    return (m + np.log(np.exp(l - m).sum(axis=1, keepdims=True)))[:, 0]


def check_epilogue(g, draft=None, rows_per_seq=0):
    """The fused statistics against the written logits."""
    lg = g["logits"]
    assert np.array_equal(g["argmax_ids"], np.argmax(lg, axis=1).astype(np.int32))
    # log_z is returned in f32: 1e-5 plus half an f32 spacing at its magnitude
    lz = logsumexp64(lg)
    assert (np.abs(g["log_z"] - lz) <= LOGPROB_TOL + 0.5 * np.spacing(np.abs(lz).astype(np.float32))).all()
    if draft is not None:
        rows, vocab = lg.shape
        R = rows_per_seq or 1
        w = SimpleNamespace(logits=lg, draft=draft, dtype="f32", n_seq=rows // R, rows_per_seq=R,
                            vocab=vocab, rows=rows)
        am, lp, acc = O.verify(w, threads=16)
        assert np.array_equal(g["argmax_ids"], am)
        assert np.abs(g["draft_lp"] - lp).max() <= LOGPROB_TOL
        if rows_per_seq:
            assert np.array_equal(g["accept_len"].astype(np.uint32), acc)


def test_integer_operands_are_exact(sampler):
    """Small integers: the product is exact, so the logits are bit-exact and
    ties between columns are frequent (the first index must win)."""
    torch = sampler.torch
    rng = np.random.default_rng(1)
    for rows, vocab, hidden in [(5, 1000, 128), (64, 4096, 64), (67, 300, 192), (1, 1, 64), (130, 257, 256)]:
        say("integer", rows, vocab, hidden)
        xi = rng.integers(-4, 5, (rows, hidden)).astype(np.float32)
        wi = rng.integers(-3, 4, (vocab, hidden)).astype(np.float32)
        ref = (xi.astype(np.int64) @ wi.astype(np.int64).T).astype(np.float32)
        g = run(sampler, bf16(torch, xi).cuda(), bf16(torch, wi).cuda())
        assert np.array_equal(g["logits"], ref)
        check_epilogue(g)
        if vocab > 1:
            ties = sum(int((ref[r] == ref[r].max()).sum() > 1) for r in range(rows))
            say("rows whose maximum is tied:", ties)


# (151936: a vocabulary the kernel serves with 320-column blocks, to fit one
# round of resident workgroups)
@pytest.mark.parametrize("rows,vocab,hidden", [(64, 32000, 1024), (130, 5000, 512), (8, 257, 4096),
                                               (8, 151936, 256)])
def test_random_operands_within_the_f32_bound(sampler, rows, vocab, hidden):
    torch = sampler.torch
    say("random", rows, vocab, hidden)
    rng = np.random.default_rng(rows * 7 + vocab)
    x = bf16(torch, rng.standard_normal((rows, hidden)))
    w = bf16(torch, rng.standard_normal((vocab, hidden)) * 0.05)
    g = run(sampler, x.cuda(), w.cuda())
    x64, w64 = x.double().numpy(), w.double().numpy()
    ref = x64 @ w64.T
    bound = hidden * U * (np.abs(x64) @ np.abs(w64).T)
    assert (np.abs(g["logits"] - ref) <= bound).all()
    check_epilogue(g)


# tiles of 64, 128 or 256 rows and 64 to 320 columns, with a row, a column and
# a k-step more or less than full ones; the last: row offsets past 32 bits
@pytest.mark.parametrize("rows,vocab,hidden", [
    (3, 63, 64), (64, 129, 192), (63, 20001, 64), (64, 50257, 128), (2, 80001, 64), (17, 100001, 64),
    (65, 255, 64), (128, 257, 128), (128, 50257, 64), (129, 256, 64), (255, 513, 192), (256, 50257, 64),
    (257, 2049, 128), (300, 700, 320), (300, 50001, 64), (512, 512, 64), (3, 5, (1 << 22) + 64)])
def test_row_tiles_are_exact(sampler, rows, vocab, hidden):
    torch = sampler.torch
    say("tiles", rows, vocab, hidden)
    rng = np.random.default_rng(rows + vocab)
    xi = rng.integers(-4, 5, (rows, hidden)).astype(np.float32)
    wi = rng.integers(-3, 4, (vocab, hidden)).astype(np.float32)
    ref = (xi.astype(np.int64) @ wi.astype(np.int64).T).astype(np.float32)
    draft = rng.integers(0, vocab, rows).astype(np.int32)
    draft[0], draft[rows - 1] = -1, vocab
    d = torch.from_numpy(draft).cuda()
    x, w = bf16(torch, xi).cuda(), bf16(torch, wi).cuda()
    g = run(sampler, x, w, draft=d)
    assert np.array_equal(g["logits"], ref)
    check_epilogue(g)
    # logprobs in f32 of values up to ~300: half a spacing beside the tolerance
    lp = ref[np.arange(1, rows - 1), draft[1:-1]].astype(np.float64) - logsumexp64(ref)[1:-1]
    assert (np.abs(g["draft_lp"][1:-1] - lp) <= LOGPROB_TOL + 0.5 * np.spacing(np.abs(lp).astype(np.float32))).all()
    assert g["draft_lp"][0] == 0.0 and g["draft_lp"][rows - 1] == 0.0
    # logits rows that are not 16-byte aligned, and no logits at all
    big = torch.full((rows, vocab + 5), -7.0, dtype=torch.float32, device="cuda")
    out = sampler.alloc_lmhead_out(rows, vocab, logits=False, draft=True)
    sampler.lmhead_dev(x, w, dict(out, logits=big[:, 1:1 + vocab]), draft=d)
    torch.cuda.synchronize()
    assert np.array_equal(big[:, 1:1 + vocab].cpu().numpy(), ref)
    assert (big[:, 0] == -7.0).all() and (big[:, 1 + vocab:] == -7.0).all()
    h = run(sampler, x, w, draft=d, logits=False)
    for k in ("argmax_ids", "log_z", "draft_lp"):
        assert np.array_equal(h[k], g[k]) and np.array_equal(out[k].cpu().numpy(), g[k]), k


# One or two cases per tile of lmhead_tile (rows, vocab, the tile's 64-column and
# row counts, k-steps a stage holds, stages of its ring), each run over more
# stages than the ring has; tests/test_lmhead_shape.py holds the choice of the
# tile to this list. 256 CUs.
STEADY = [
    (3, 300, 1, 64, 2, 6), (64, 20001, 2, 64, 2, 4), (64, 33001, 4, 64, 2, 4), (2, 80001, 5, 64, 2, 3),
    (17, 100001, 4, 64, 4, 2), (128, 257, 2, 128, 2, 4), (300, 1001, 2, 128, 2, 4), (128, 33001, 4, 128, 2, 3),
    (300, 50001, 4, 128, 2, 3), (255, 513, 2, 256, 2, 3), (512, 513, 2, 256, 2, 3), (256, 33001, 4, 256, 4, 2),
    (511, 50257, 4, 256, 4, 2)]


@pytest.mark.parametrize("hidden", [320, 384, 512])   # 5, 6 and 8 stages of 64 k, twice as many of 32
@pytest.mark.parametrize("rows,vocab", [c[:2] for c in STEADY])
def test_stages_past_the_ring_are_exact(sampler, rows, vocab, hidden):
    torch = sampler.torch
    say("stages", rows, vocab, hidden)
    rng = np.random.default_rng([rows, vocab, hidden])
    xi = rng.integers(-4, 5, (rows, hidden)).astype(np.float32)
    wi = rng.integers(-3, 4, (vocab, hidden)).astype(np.float32)
    # (float64 holds these integer sums exactly; on the device, where it is quick)
    x, w = torch.from_numpy(xi).cuda(), torch.from_numpy(wi).cuda()
    ref = (x.double() @ w.double().t()).float().cpu().numpy()
    cols = rng.choice(vocab, min(vocab, 500), replace=False)
    assert np.array_equal(ref[:, cols], xi.astype(np.float64) @ wi[cols].T.astype(np.float64))
    g = run(sampler, x.to(torch.bfloat16), w.to(torch.bfloat16))
    assert np.array_equal(g["logits"], ref)
    check_epilogue(g)


@pytest.mark.parametrize("rows,vocab", [(3, 1), (5, 70), (64, 300), (130, 513)])
def test_argmax_stays_in_range_for_nan_and_inf(sampler, rows, vocab):
    """Rows of NaN, of -inf and with one +inf: the argmax is an id of the
    vocabulary (a decode loop looks up its embedding)."""
    torch = sampler.torch
    hidden = 64
    x = torch.ones((rows, hidden), dtype=torch.bfloat16, device="cuda")
    w = torch.ones((vocab, hidden), dtype=torch.bfloat16, device="cuda")
    x[0] = float("nan")
    x[1] = float("-inf")
    x[2, 0] = float("inf")
    g = run(sampler, x, w)
    assert ((g["argmax_ids"] >= 0) & (g["argmax_ids"] < vocab)).all(), g["argmax_ids"]
    assert (g["argmax_ids"][3:] == 0).all()
    w[vocab // 2:] = float("nan")
    g = run(sampler, x, w)
    assert ((g["argmax_ids"] >= 0) & (g["argmax_ids"] < vocab)).all(), g["argmax_ids"]


@pytest.mark.parametrize("rows,vocab", [(3, 64), (5, 300), (64, 1000), (130, 1000), (256, 1000)])
def test_argmax_beside_nan_columns(sampler, rows, vocab):
    """Columns of NaN beside finite ones, also all of one wave's or of one
    block's: the argmax is the first of the greatest finite columns, and log z
    is NaN (one of the sum's terms is)."""
    torch = sampler.torch
    x = torch.ones((rows, 64), dtype=torch.bfloat16, device="cuda")
    best = vocab // 4 + 3
    for lo, hi in [(vocab // 2, vocab), (32, 64), (64, 128), (0, vocab // 4), (best - 1, best), (best + 1, best + 2)]:
        w = torch.full((vocab, 64), -1.0, dtype=torch.bfloat16, device="cuda")
        w[best:best + 2] = 1.0
        w[lo:hi] = float("nan")
        g = run(sampler, x, w)
        want = np.argmax(np.where(np.isnan(g["logits"]), -np.inf, g["logits"]), axis=1)
        assert np.array_equal(g["argmax_ids"], want), (lo, hi, g["argmax_ids"][:4], want[:4])
        if lo < vocab:
            assert np.isnan(g["log_z"]).all(), (lo, hi)


@pytest.mark.parametrize("rows,vocab", [(5, 300), (64, 1000), (130, 1000), (256, 1000)])
def test_log_z_of_rows_with_inf_blocks(sampler, rows, vocab):
    """Columns of -inf, whole blocks of them too, have no weight in log z; a
    row of nothing but -inf has none (as in logprobs_from, which then divides
    by the exponential of -inf - -inf)."""
    torch = sampler.torch
    x = torch.ones((rows, 64), dtype=torch.bfloat16, device="cuda")
    for lo, hi in [(0, vocab - 7), (0, vocab // 2), (vocab // 3, vocab), (40, 41), (0, vocab)]:
        w = torch.from_numpy(np.linspace(-0.1, 0.1, vocab, dtype=np.float32)[:, None].repeat(64, 1)).to(torch.bfloat16).cuda()
        w[lo:hi] = float("-inf")
        g = run(sampler, x, w)
        if (lo, hi) == (0, vocab):
            assert np.isnan(g["log_z"]).all()
        else:
            lz = logsumexp64(g["logits"])
            assert (np.abs(g["log_z"] - lz) <= LOGPROB_TOL).all(), (lo, hi, g["log_z"][0], lz[0])
            assert np.array_equal(g["argmax_ids"], np.argmax(g["logits"], axis=1))


@pytest.mark.parametrize("vocab", [20000, 140000])
def test_drafts_and_acceptance(sampler, vocab):
    """rows_per_seq = 8: each sequence's drafts agree with the argmax on a
    chosen prefix, then differ; the last row carries no draft (-1)."""
    torch = sampler.torch
    rng = np.random.default_rng(5)
    n_seq, R, hidden = 24, 8, 512
    rows = n_seq * R
    x = bf16(torch, rng.standard_normal((rows, hidden))).cuda()
    w = bf16(torch, rng.standard_normal((vocab, hidden)) * 0.05).cuda()
    first = run(sampler, x, w)
    am = first["argmax_ids"].reshape(n_seq, R)
    prefix = rng.integers(0, R, n_seq)
    prefix[:3] = [0, R - 1, 3]
    draft = rng.integers(0, vocab, (n_seq, R)).astype(np.int32)
    for s in range(n_seq):
        draft[s, :prefix[s]] = am[s, :prefix[s]]
        if draft[s, prefix[s]] == am[s, prefix[s]]:
            draft[s, prefix[s]] = (am[s, prefix[s]] + 1) % vocab
    draft[:, R - 1] = -1
    draft[5, 2] = vocab     # out of range: logprob 0
    d = torch.from_numpy(draft.reshape(-1)).cuda()
    g = run(sampler, x, w, draft=d, rows_per_seq=R)
    assert np.array_equal(g["logits"], first["logits"])   # deterministic
    check_epilogue(g, draft.reshape(-1), R)
    assert g["accept_len"].tolist() == [min(int(p), 2) if s == 5 else int(p) for s, p in enumerate(prefix)]
    assert g["draft_lp"][R - 1::R].tolist() == [0.0] * n_seq
    # the fused outputs do not depend on writing the logits
    h = run(sampler, x, w, draft=d, rows_per_seq=R, logits=False)
    for k in ("argmax_ids", "log_z", "draft_lp", "accept_len"):
        assert np.array_equal(h[k], g[k]), k


def test_padded_logits_rows(sampler):
    """ld_logits > vocab: the padding is left as it was."""
    torch = sampler.torch
    rng = np.random.default_rng(9)
    rows, vocab, hidden = 16, 700, 128
    x = bf16(torch, rng.standard_normal((rows, hidden))).cuda()
    w = bf16(torch, rng.standard_normal((vocab, hidden))).cuda()
    big = torch.full((rows, 768), -3.0, dtype=torch.float32, device="cuda")
    out = {"logits": big[:, :vocab], "argmax_ids": torch.zeros(rows, dtype=torch.int32, device="cuda")}
    sampler.lmhead_dev(x, w, out)
    torch.cuda.synchronize()
    b = big.cpu().numpy()
    assert (b[:, vocab:] == -3.0).all()
    assert np.array_equal(out["argmax_ids"].cpu().numpy(), np.argmax(b[:, :vocab], axis=1))


def test_invalid_arguments_are_rejected(sampler):
    from locus_amd.sampler import SamplerError
    torch = sampler.torch
    x = torch.zeros((4, 96), dtype=torch.bfloat16, device="cuda")
    w = torch.zeros((100, 96), dtype=torch.bfloat16, device="cuda")
    out = sampler.alloc_lmhead_out(4, 100)
    with pytest.raises(SamplerError, match="multiple of 64"):
        sampler.lmhead_dev(x, w, out)
    x = torch.zeros((6, 64), dtype=torch.bfloat16, device="cuda")
    w = torch.zeros((100, 64), dtype=torch.bfloat16, device="cuda")
    d = torch.zeros(6, dtype=torch.int32, device="cuda")
    out = sampler.alloc_lmhead_out(6, 100, draft=True, n_seq=1)
    with pytest.raises(SamplerError, match="divide rows"):
        sampler.lmhead_dev(x, w, out, draft=d, rows_per_seq=4)
    x = torch.zeros((600, 64), dtype=torch.bfloat16, device="cuda")
    out = sampler.alloc_lmhead_out(600, 100)
    with pytest.raises(SamplerError, match="context limits"):
        sampler.lmhead_dev(x, w, out)


def test_decode_shape_full_size(sampler):
    """B = 64, V = 128256, hidden 4096 (the decode batch of the sampling
    workloads): columns checked against float64 on a sample, the epilogue
    against the whole written logits."""
    torch = sampler.torch
    say("full size 64 x 128256 x 4096")
    gen = torch.Generator(device="cuda").manual_seed(3)
    rows, vocab, hidden = 64, 128256, 4096
    x = torch.randn((rows, hidden), generator=gen, device="cuda").to(torch.bfloat16)
    w = (torch.randn((vocab, hidden), generator=gen, device="cuda") * 0.02).to(torch.bfloat16)
    g = run(sampler, x, w)
    cols = np.random.default_rng(0).choice(vocab, 2048, replace=False)
    cols[:2] = [0, vocab - 1]
    x64 = x.double().cpu().numpy()
    w64 = w[torch.from_numpy(cols).cuda()].double().cpu().numpy()
    ref = x64 @ w64.T
    bound = hidden * U * (np.abs(x64) @ np.abs(w64).T)
    assert (np.abs(g["logits"][:, cols] - ref) <= bound).all()
    check_epilogue(g)
