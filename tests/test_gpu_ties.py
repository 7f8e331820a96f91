"""Nucleus rows whose deciding candidates tie by the hundred (bf16 or coarsely
quantised logits): the decisive group is larger than the finalize ranks at
once, so it is narrowed by rank key first. The reference leaves the order of
equal logits to its sort; this build orders them by id, so the expected id is
taken from a float64 walk of the reference's chain (sampling.cpp:87-147) in
that order."""
import numpy as np
import pytest

from locus_amd import workloads as W

pytestmark = pytest.mark.gpu

PATH_EXACT, PATH_NUCLEUS = 4, 6


@pytest.fixture(scope="module")
def sampler():
    from locus_amd.sampler import Sampler
    s = Sampler(device=0, max_rows=64, max_vocab=262144, max_hist=4096, max_top=20)
    yield s
    s.close()


def walk(logits, p, u):
    """(id, survivors, least relative distance of a decision from its threshold)."""
    order = np.lexsort((np.arange(len(logits)), -logits))
    inv_t = np.float32(1.0) / np.float32(p["temperature"])
    x = (logits[order] - logits[order[0]]) * inv_t
    w = np.exp(x.astype(np.float64))
    k = int(p["top_k"]) if 0 < p["top_k"] < len(w) else len(w)
    w = w[:k]
    s = w.sum()
    keep, near = k, 1.0
    if p["top_p"] < 1.0:
        cum = np.cumsum(w) / s
        keep = min(k, int(np.argmax(cum >= p["top_p"])) + 1)
        near = min(near, np.abs(cum - np.float64(p["top_p"])).min())
    if p["min_p"] > 0.0:
        keep = min(keep, max(1, int((w >= np.float64(p["min_p"])).sum())))
        near = min(near, np.abs(w - np.float64(p["min_p"])).min())
    c = np.cumsum(w[:keep])
    r = u * c[-1]
    hit = np.nonzero(c >= r)[0]
    at = int(hit[0]) if len(hit) else keep - 1
    return int(order[at]), keep, min(near, np.abs(c / c[-1] - u).min())


@pytest.mark.parametrize("V,dtype,step,params", [
    (151936, "bf16", 0.0, dict(temperature=1.5, top_p=0.98)),    # ~180 ids a value at the top-p cut
    (262144, "bf16", 0.0, dict(temperature=1.5, top_p=0.9)),     # ~490 at the top-p cut
    (262144, "bf16", 0.0, dict(temperature=1.0)),                # the draw alone
    (128256, "f32", 0.25, dict(temperature=1.0, top_p=0.95)),    # thousands a value: several narrowing steps
    (128256, "f32", 0.0625, dict(temperature=2.0, top_k=100000, top_p=0.7, min_p=0.02)),
    (32001, "f32", 0.125, dict(temperature=1.0, top_k=5000, top_p=0.9)),   # the K-th candidate inside a tie
    (8193, "bf16", 1.0, dict(temperature=1.3, top_p=0.8)),       # a value spans both slices
    (257, "f32", 8.0, dict(temperature=1.0, top_p=0.6)),         # one value more than the finalize ranks at once
])
def test_groups_of_equal_logits(sampler, V, dtype, step, params):
    rows = 12
    g = np.random.default_rng([V, int(step * 1000)])
    x = g.standard_normal((rows, V), dtype=np.float32)
    if step:
        x = np.round(x / np.float32(step)) * np.float32(step)
    logits = W.bf16_rne(x) if dtype == "bf16" else x
    p = W.default_params(rows)
    for k, v in params.items():
        p[k] = v
    u = g.random(rows)
    u[0], u[1] = 0.0, 0.999999   # the first candidate, and the far end of the list
    w = W.Workload("ties", rows, V, dtype, logits, p, None, u)
    got = sampler.sample(w)
    assert sampler.status() == 0
    f = W.bf16_to_f32(logits) if dtype == "bf16" else x
    checked = 0
    for r in range(rows):
        tok, keep, near = walk(f[r], p[r], u[r])
        if near < 1e-9:
            continue
        checked += 1
        assert got["ids"][r] == tok, (r, got["ids"][r], tok, got["diag"][r])
        assert got["diag"]["keep"][r] == keep, (r, got["diag"][r], keep)
    assert checked >= rows // 2
    assert (got["diag"]["path"] == PATH_NUCLEUS).all(), got["diag"]["path"].tolist()


def test_one_value_past_the_candidate_list(sampler):
    """Every logit equal: the plan's list cannot hold the row, the exact path takes it."""
    V, rows = 40000, 3
    p = W.default_params(rows)
    p["temperature"], p["top_p"] = 1.0, 0.9
    u = np.array([0.1, 0.5, 0.99])
    w = W.Workload("flat", rows, V, "f32", np.full((rows, V), 1.5, np.float32), p, None, u)
    got = sampler.sample(w)
    f = np.full(V, 1.5, np.float32)
    want = [walk(f, p[r], u[r])[0] for r in range(rows)]
    assert np.abs(got["ids"] - np.array(want)).max() <= 1, (got["ids"], want)   # (40000 u is a near tie)
    assert (got["diag"]["path"] == PATH_EXACT).all()
