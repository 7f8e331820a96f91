"""lcs_logprobs and greedy sampling with logprobs where a workgroup takes a whole
row (logprobs_from, sampling.cpp:150-190; argmax, llama.cpp:1237-1245), against
float64."""
import numpy as np
import pytest

from locus_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sampler():
    from locus_amd.sampler import Sampler
    s = Sampler(device=0, max_rows=300, max_vocab=262144, max_hist=64, max_top=20)
    yield s
    s.close()


# rows that end inside a group or a round, fewer ids than the top n, one lane's
# groups past 64 (V 262144), and rows cut into slices beside them (5 x 40000)
@pytest.mark.parametrize("V,rows,dtype,n_top", [(1, 70, "f32", 3), (13, 3, "bf16", 20), (257, 65, "f32", 20), (4099, 9, "bf16", 5),
                                                (32769, 64, "f32", 1), (65536, 2, "bf16", 20), (40000, 5, "f32", 5),
                                                (262141, 66, "bf16", 5), (128256, 64, "f32", 0)])
def test_rows_in_one_workgroup(sampler, V, rows, dtype, n_top):
    torch = sampler.torch
    g = np.random.default_rng([V, rows])
    x = (g.standard_normal((rows, V), dtype=np.float32) * 2).astype(np.float32)
    x[0] = np.round(x[0])                       # hundreds of values tied at the top
    if rows > 4 and V > 100:
        x[1] = 0.5                              # one value
        x[2, 50:] = -np.inf                     # fewer finite values than lanes
        x[3, :8] = 30.0                         # the whole top in one group
    logits = W.bf16_rne(x) if dtype == "bf16" else x
    f = (W.bf16_to_f32(logits) if dtype == "bf16" else x).astype(np.float64)
    chosen = g.integers(0, V, rows).astype(np.int32)
    chosen[-1] = V                              # outside: logprob 0
    w = W.Workload("lp", rows, V, dtype, logits, W.default_params(rows), None, np.zeros(rows), n_top=n_top,
                   want_logprobs=True)
    d = sampler.upload(w)
    m = f.max(1, keepdims=True)
    lz = (m + np.log(np.exp(f - m).sum(1, keepdims=True)))[:, 0]
    k = min(n_top, V)
    order = np.stack([np.lexsort((np.arange(V), -f[r]))[:k] for r in range(rows)])

    def check(o, lp_of):
        got = {n: o[n].cpu().numpy() for n in ("ids", "chosen_lp", "top_ids", "top_lp")}
        assert np.array_equal(got["ids"], f.argmax(1).astype(np.int32))
        want = np.array([f[r, t] - lz[r] if t < V else 0.0 for r, t in enumerate(lp_of)])
        fin = np.isfinite(want)
        assert (np.abs(got["chosen_lp"][fin] - want[fin]) <= 1e-5).all()
        assert np.array_equal(got["chosen_lp"][~fin], want[~fin].astype(np.float32))
        assert np.array_equal(got["top_ids"][:, :k], order)
        top = np.take_along_axis(f, order, 1) - lz[:, None]
        fin = np.isfinite(top)
        assert (np.abs(got["top_lp"][:, :k][fin] - top[fin]) <= 1e-5).all()

    o = sampler.alloc_out(rows, n_top, True, diag=False)
    sampler.logprobs_dev(d, o, chosen=torch.from_numpy(chosen).cuda())
    torch.cuda.synchronize()
    check(o, chosen)
    o = sampler.alloc_out(rows, n_top, True, diag=False)
    sampler.logprobs_dev(d, o)                  # of each row's argmax
    torch.cuda.synchronize()
    check(o, f.argmax(1))
    o = sampler.alloc_out(rows, n_top, True, diag=False)
    sampler.sample_dev(d, o, lp_ids=torch.from_numpy(chosen).cuda())   # greedy rows
    torch.cuda.synchronize()
    check(o, chosen)
    # the sliced path (asked for by diag) agrees, past the vocabulary's end too
    o2 = sampler.alloc_out(rows, n_top, True, diag=True)
    sampler.sample_dev(d, o2, lp_ids=torch.from_numpy(chosen).cuda())
    torch.cuda.synchronize()
    assert torch.equal(o["top_ids"], o2["top_ids"]) and torch.equal(o["ids"], o2["ids"])


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("NT,before", [(256, 0), (512, 8192)])   # threads per row, groups ahead of the last round
def test_verify_rows_that_end_in_any_slot_of_a_round(sampler, NT, before, dtype):
    """A row's last round takes 1, 2, 3, 4, 6 or 8 groups of 16 bytes a thread:
    rows that end with the first and the last group of each, the maximum among
    the row's last ids, against float64."""
    G, rows = 8 if dtype == "bf16" else 4, 4
    for k in range(8):
        for V in ((before + k * NT) * G + 1, (before + (k + 1) * NT) * G - 1, (before + (k + 1) * NT) * G):
            g = np.random.default_rng([V, NT])
            x = (g.standard_normal((rows, V), dtype=np.float32) * 2).astype(np.float32)
            x[0, V - 1] = x[1, V // 2] = x[1, V - 1] = 30.0
            logits = W.bf16_rne(x) if dtype == "bf16" else x
            f = (W.bf16_to_f32(logits) if dtype == "bf16" else x).astype(np.float64)
            draft = np.array([V - 1, V // 2, 0, V - 1], np.int32)
            w = W.Workload("rounds", rows, V, dtype, logits, None, None, None, n_seq=2, rows_per_seq=2, draft=draft)
            got = sampler.verify(w)
            am = f.argmax(1)
            m = f.max(1, keepdims=True)
            lp = f[np.arange(rows), draft] - (m + np.log(np.exp(f - m).sum(1, keepdims=True)))[:, 0]
            assert np.array_equal(got["argmax_ids"], am), (V, got["argmax_ids"], am)
            assert (np.abs(got["draft_lp"] - lp) <= 1e-5).all(), (V, got["draft_lp"], lp)
            hit = (am == draft).reshape(2, 2)
            assert got["accept_len"].tolist() == [int(h[0]) + int(h[0] and h[1]) for h in hit]
