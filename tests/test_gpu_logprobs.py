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
