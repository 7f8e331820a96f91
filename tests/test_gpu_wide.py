"""Min-p rows whose windows overflow their slices' records, handed by row_fin to
the nucleus kernels of the same call (sampling.cpp:99-147 decides them exactly
either way), and rows with heavily penalised ids, which the nucleus histogram
sums apart from its bins."""
import numpy as np
import pytest

from locus_amd import workloads as W
from oracle import pyoracle as O
from tests.test_gpu_sampling import compare

pytestmark = pytest.mark.gpu


def make(V, rows, dtype, seed, n_hist=600, **params):
    g = np.random.default_rng([V, rows, seed])
    x = g.standard_normal((rows, V), dtype=np.float32)
    p = W.default_params(rows)
    for k, v in params.items():
        p[k] = v
    # a few ids very often: frequency penalties of up to ~60 logits
    hist = np.where(g.random((rows, n_hist)) < 0.4, g.integers(0, min(V, 5), (rows, 1)),
                    g.integers(0, V, (rows, n_hist))).astype(np.int32)
    p["repeat_last_n"] = n_hist
    logits = W.bf16_rne(x) if dtype == "bf16" else x
    f32 = W.bf16_to_f32(logits) if dtype == "bf16" else x
    seeds = W._seeds(seed, 0, rows)
    kw = dict(hist_off=np.arange(rows + 1, dtype=np.uint32) * n_hist, hist_ids=hist.reshape(-1), n_top=5,
              want_logprobs=True)
    w = W.Workload("wide", rows, V, dtype, logits, p, seeds, W.uniforms(seeds), **kw)
    w32 = W.Workload("wide", rows, V, "f32", f32, p, seeds, W.uniforms(seeds), **kw)
    return w, w32


@pytest.fixture(scope="module")
def sampler():
    from locus_amd.sampler import Sampler
    s = Sampler(device=0, max_rows=300, max_vocab=262144, max_hist=4096, max_top=20)
    yield s
    s.close()


PEN = dict(repeat_penalty=1.1, frequency_penalty=0.25, presence_penalty=0.3)


@pytest.mark.parametrize("V,rows,dtype,params", [
    (128256, 4, "f32", dict(temperature=1.5, min_p=0.01, top_p=0.9, **PEN)),
    (128256, 3, "bf16", dict(temperature=1.5, min_p=0.02, top_p=1.0, **PEN)),
    (262144, 2, "f32", dict(temperature=1.5, min_p=0.01, top_p=0.9, **PEN)),
    (8193, 5, "f32", dict(temperature=2.0, min_p=0.1, top_p=1.0, **PEN)),          # two slices, a short one
    (700, 4, "f32", dict(temperature=3.0, min_p=0.2, top_p=0.8, **PEN)),           # one slice
    (9000, 270, "f32", dict(temperature=1.5, min_p=0.05, top_p=0.95, **PEN)),      # past one launch of 256 rows
    (50257, 4, "f32", dict(temperature=1.5, top_p=0.97, **PEN)),                    # top-p alone, outliers off the bins
    (50257, 4, "bf16", dict(temperature=1.0, top_p=1.0, **PEN)),                    # the draw alone
    (50257, 4, "f32", dict(temperature=0.2, top_p=0.99, **PEN)),
])
def test_wide_rows(sampler, V, rows, dtype, params):
    w, w32 = make(V, rows, dtype, 77, **params)
    o = O.sample_batch(w32, threads=16)
    g = sampler.sample(w)
    # (min-p rows: handed over and decided there; the others: in the bins, their
    # outliers summed apart, not on the exact path)
    compare(w32, g, o, "wide", expect_paths={4} if params.get("min_p") else {6})
    assert (g["diag"]["reserved"] == (1 if params.get("min_p") else 0)).all(), g["diag"]["reserved"].tolist()
    h = sampler.sample(w, use_host_params=False)   # modes unknown to the host: every kernel is launched
    assert np.array_equal(h["ids"], g["ids"]) and np.array_equal(h["top_ids"], g["top_ids"])


@pytest.mark.parametrize("V,dtype,params", [
    (50257, "f32", dict(temperature=1.5, min_p=0.02, top_p=0.9)),
    (9000, "bf16", dict(temperature=0.7, min_p=0.05)),
])
def test_constrained_min_p_rows_report_the_nucleus_path(sampler, V, dtype, params):
    """A min-p row under a mask is the nucleus kernels' own, not one handed over."""
    w, w32 = make(V, 4, dtype, 79, **params)
    w.mask = w32.mask = W.pack_mask(np.random.default_rng(V).random((4, V)) < 0.95)
    o = O.sample_batch(w32, threads=16)
    compare(w32, sampler.sample(w), o, "constrained", expect_paths={6})


@pytest.mark.parametrize("V,dtype,params", [
    (128256, "f32", dict(temperature=3.0, min_p=1e-6, top_p=1.0, **PEN)),
    (128256, "f32", dict(temperature=3.0, min_p=1e-6, top_p=0.9, **PEN)),
    (50257, "bf16", dict(temperature=2.0, min_p=1e-9, top_p=1.0, **PEN)),
    (50257, "f32", dict(temperature=2.0, min_p=1e-30, top_p=1.0, **PEN)),     # below every outlier
    (128256, "f32", dict(temperature=3.0, min_p=0.01, top_p=1.0, **PEN)),     # between the bins' end and the outliers
    (128256, "f32", dict(temperature=1.5, min_p=0.02, top_p=0.9, **PEN)),     # inside the bins
])
def test_min_p_cut_past_the_bins(sampler, V, dtype, params):
    """Constrained rows whose penalised outliers (one id 60 logits down, one 25)
    lie past the histogram's bins: a min-p cut between them or beyond is no
    reason for the exact path."""
    w, w32 = make(V, 8, dtype, 78, **params)
    bits = np.random.default_rng(V).random((8, V)) < 0.95
    bits[:, :10] = True
    w.hist_ids.reshape(8, -1)[:, ::6] = 7
    w.mask = w32.mask = W.pack_mask(bits)
    w.u[:] = w32.u[:] = np.linspace(0.02, 0.9, 8)   # (a draw in the last bin is one)
    assert w32.hist_ids is w.hist_ids
    o = O.sample_batch(w32, threads=16)
    g = sampler.sample(w)
    compare(w32, g, o, "past", expect_paths={6})


@pytest.mark.parametrize("V,dtype,params", [
    (32000, "f32", dict(temperature=1.5, min_p=0.01, top_p=0.9)),
    (32000, "bf16", dict(temperature=1.5, min_p=0.01, **PEN)),
    (128256, "f32", dict(temperature=0.8, min_p=0.05, top_p=0.95, **PEN)),
    (700, "f32", dict(temperature=1.0, min_p=0.1, top_k=600)),
])
def test_min_p_cut_in_an_empty_bin(sampler, V, dtype, params):
    """Constrained confident rows (eight ids far above the rest): no candidate
    in the min-p cut's own bin survives, which is no reason for the exact path."""
    rows = 16
    w, w32 = make(V, rows, "f32", 80, **params)
    g = np.random.default_rng(V)
    x = w.logits
    for r in range(rows):
        x[r, g.choice(np.arange(10, V), 8, replace=False)] += np.float32(12.0)
    if dtype == "bf16":
        w.dtype, w.logits = "bf16", W.bf16_rne(x)
        w32.logits = W.bf16_to_f32(w.logits)
    w.mask = w32.mask = W.pack_mask(g.random((rows, V)) < 0.95)
    o = O.sample_batch(w32, threads=16)
    compare(w32, sampler.sample(w), o, "empty bin", expect_paths={6})


def test_wide_rows_beside_others(sampler):
    """Greedy, top-k, narrow and wide min-p, top-p and masked rows in one batch."""
    w, _ = make(40000, 24, "f32", 5, **PEN)
    p = w.params
    p["temperature"][4:] = 1.5
    p["top_k"][4:8] = 30
    p["min_p"][8:16], p["top_p"][8:] = 0.01, 0.95
    w.logits[8:12] *= np.float32(6.0)   # (narrow windows)
    bits = np.random.default_rng(9).random((24, 40000)) < 0.3
    w.mask = W.pack_mask(bits)
    has = np.zeros(24, np.uint8)
    has[20:] = 1
    o = O.sample_batch(w, threads=16, has_mask=has)
    g = sampler.sample(w, has_mask=sampler.torch.from_numpy(has).cuda())
    compare(w, g, o, "beside")
    assert g["diag"]["reserved"].tolist() == [0] * 12 + [1] * 4 + [0] * 8
    path = g["diag"]["path"].tolist()
    assert set(path[:4]) == {1} and set(path[4:8]) == {5} and set(path[8:12]) <= {2, 3} and set(path[12:16]) == {4}, path


def test_wide_row_above_max_hist_is_reported():
    from locus_amd.sampler import Sampler
    small = Sampler(device=0, max_rows=4, max_vocab=20000, max_hist=100, max_top=5)
    try:
        w, _ = make(20000, 2, "f32", 3, temperature=1.5, min_p=0.01, **PEN)
        g = small.sample(w)
        assert (g["ids"] == -1).all() and small.status() == 1
    finally:
        small.close()
