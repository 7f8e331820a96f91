"""Workloads of the sampler that its users run, through its public entry points.

Each case is one call of the engine's token step on inputs that already lie in
device memory: sampling (lcs_sample), speculative verify (lcs_verify), the
fused lm-head product (lcs_lmhead), batched logprobs (lcs_logprobs) and n-gram
drafts (lcs_ngram_draft). listed() holds the cases themselves, draw() further
ones of the same ranges; prepare() builds a case's inputs from a seed, run()
makes the one call, exact() restates its floating outputs in 64 bits.

Logits are normal with the spreads of locus_amd.workloads' configurations,
histories are Zipf(1.1), masks are runs of 1..64 allowed ids.
"""
import ctypes
import functools
import math

import numpy as np
import torch

from locus_amd import sampler as S
from locus_amd.workloads import Workload, default_params

MAX_ROWS, MAX_VOCAB, MAX_HIST, MAX_TOP = 2048, 262144, 4096, 20


def listed():
    return [
        # one chat stream, the usual temperature 0.8 / top-k 40 / top-p 0.95:
        # the latency of a single step
        {"name": "topk_1", "kind": "sample", "preset": "topk", "rows": 1, "vocab": 128256, "dtype": "f32",
         "hist": 0, "n_top": 0},
        # a server's batch with the whole chain: penalties over 2048-id
        # histories, min-p, top-p, draw, top-5 logprobs (the headline workload)
        {"name": "full_64", "kind": "sample", "preset": "full", "rows": 64, "vocab": 128256, "dtype": "f32",
         "hist": 2048, "ragged": False, "n_top": 5},
        # a large batch at a high temperature with nothing but top-p: the
        # nucleus holds about 10^5 ids a row
        {"name": "topp_256", "kind": "sample", "preset": "topp", "rows": 256, "vocab": 151936, "dtype": "f32",
         "hist": 0, "n_top": 0},
        # constrained decoding: every row under its own JSON grammar mask
        {"name": "json_32", "kind": "sample", "preset": "json", "rows": 32, "vocab": 128256, "dtype": "f32",
         "hist": 0, "n_top": 1},
        # creative sampling: flat logits, a high temperature and a low min-p,
        # so that thousands of ids survive per row
        {"name": "minp_wide_64", "kind": "sample", "preset": "minp_wide", "rows": 64, "vocab": 128256,
         "dtype": "f32", "hist": 2048, "ragged": False, "n_top": 5},
        # a server's batch as requests come: greedy, top-k, the full chain and
        # plain top-p rows side by side, logits from a bf16 model
        {"name": "mixed_24", "kind": "sample", "preset": "mixed", "rows": 24, "vocab": 151936, "dtype": "bf16",
         "hist": 1024, "ragged": True, "n_top": 1},
        # speculative decoding of a large batch, logits from a bf16 model
        {"name": "verify_512x8", "kind": "verify", "n_seq": 512, "per_seq": 8, "vocab": 163840, "dtype": "bf16"},
        # speculative decoding of a few streams: four drafts and the bonus row
        {"name": "verify_4x5", "kind": "verify", "n_seq": 4, "per_seq": 5, "vocab": 128256, "dtype": "f32"},
        # the lm-head of a decode step: logits and the statistics that the
        # sampling call takes over
        {"name": "lmhead_64", "kind": "lmhead", "rows": 64, "vocab": 128256, "hidden": 4096, "per_seq": 0},
        # the lm-head of a speculative step: drafts verified in its epilogue,
        # no logits written
        {"name": "lmhead_1024", "kind": "lmhead", "rows": 1024, "vocab": 128256, "hidden": 4096, "per_seq": 8},
        # scoring a prompt: the logprob of each given token and the top 5
        {"name": "logprobs_1024", "kind": "logprobs", "rows": 1024, "vocab": 128256, "dtype": "bf16", "n_top": 5},
        # prompt-lookup drafts of a batch with contexts of up to 32k tokens
        {"name": "draft_64", "kind": "draft", "n_seq": 64, "ctx": 32768, "ngram": 3, "max_draft": 7},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _vocab(rng):
    # vocabularies of this repository's tests and configurations, or any size
    return rng.choice([32000, 128256, 151936, 163840, 262144, _log(rng, 4000, 262144), _log(rng, 20000, 262144)])


def draw(rng):
    kind = rng.choice(["sample", "sample", "sample", "verify", "lmhead", "logprobs", "draft"])
    if kind == "sample":
        preset = rng.choice(["greedy", "topk", "full", "topp", "json", "minp_wide", "mixed"])
        rows = _log(rng, 1, 64 if preset == "minp_wide" else 256)
        pen = preset in ("full", "minp_wide", "mixed")
        return {"kind": kind, "preset": preset, "rows": rows, "vocab": _vocab(rng),
                "dtype": rng.choice(["f32", "bf16"]), "hist": _log(rng, 16, 4096) if pen else 0,
                "ragged": True, "n_top": rng.choice([0, 1, 5, 20])}
    if kind == "verify":
        vocab, per = _vocab(rng), rng.randint(1, 16)
        dtype = rng.choice(["f32", "bf16"])
        most = int(1.3e9) // (vocab * per * (4 if dtype == "f32" else 2))
        return {"kind": kind, "n_seq": _log(rng, 1, max(1, min(512, most))), "per_seq": per, "vocab": vocab,
                "dtype": dtype}
    if kind == "lmhead":
        vocab, hidden = rng.choice([32000, 50257, 128256, 151936, _log(rng, 16000, 152000)]), 64 * rng.randint(16, 64)
        per = rng.choice([0, 0, 2, 4, 8])
        rows = _log(rng, 1, min(1024, 1024 * 128256 * 4096 // (vocab * hidden)))
        return {"kind": kind, "rows": max(1, rows // per) * per if per else rows, "vocab": vocab, "hidden": hidden,
                "per_seq": per}
    if kind == "logprobs":
        vocab, dtype = _vocab(rng), rng.choice(["f32", "bf16"])
        most = int(5e8) // (vocab * (4 if dtype == "f32" else 2))
        return {"kind": kind, "rows": _log(rng, 1, min(MAX_ROWS, most)), "vocab": vocab, "dtype": dtype,
                "n_top": rng.choice([0, 1, 5, 20])}
    return {"kind": kind, "n_seq": _log(rng, 1, 512), "ctx": _log(rng, 64, 131072), "ngram": rng.randint(2, 5),
            "max_draft": rng.randint(1, 16)}


# ------------------------------------------------------------------ inputs --
@functools.lru_cache(maxsize=None)
def _sampler():
    """The handle that a serving program creates once."""
    return S.Sampler(device=0, max_rows=MAX_ROWS, max_vocab=MAX_VOCAB, max_hist=MAX_HIST, max_top=MAX_TOP)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _stride(vocab, dtype):
    g = 8 if dtype == "bf16" else 4
    return (vocab + g - 1) // g * g


def _logits(gen, rows, vocab, dtype, sigma):
    """(rows, stride); the padding past the vocabulary holds values too."""
    x = torch.randn(rows, _stride(vocab, dtype), generator=gen, device="cuda",
                    dtype=torch.bfloat16 if dtype == "bf16" else torch.float32)
    return x.mul_(sigma)


def _ints(gen, lo, hi, shape):
    return torch.randint(lo, hi, shape, generator=gen, device="cuda")


@functools.lru_cache(maxsize=None)
def _zipf_cdf(vocab):
    w = np.arange(1, vocab + 1, dtype=np.float64) ** -1.1
    return torch.from_numpy(np.cumsum(w) / w.sum()).cuda()


def _zipf(gen, vocab, n):
    perm = torch.randperm(vocab, generator=gen, device="cuda")
    u = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64)
    return perm[torch.searchsorted(_zipf_cdf(vocab), u).clamp_(max=vocab - 1)].to(torch.int32)


def _mask(gen, rng, rows, vocab):
    """Per row: runs of 1..64 allowed ids, a log-uniform share in [5e-4, 0.3]."""
    words = (vocab + 31) // 32
    d = torch.zeros(rows, words * 32 + 64, device="cuda", dtype=torch.int32)
    for r in range(rows):
        runs = max(1, math.ceil(math.exp(rng.uniform(math.log(5e-4), math.log(0.3))) * vocab / 32.5))
        at = _ints(gen, 0, vocab, (runs,))
        one = torch.ones(runs, device="cuda", dtype=torch.int32)
        d[r].index_add_(0, at, one)
        d[r].index_add_(0, at + _ints(gen, 1, 65, (runs,)), -one)
    bits = (d.cumsum(1)[:, :vocab] > 0).to(torch.int64)
    bits = torch.nn.functional.pad(bits, (0, words * 32 - vocab)).view(rows, words, 32)
    packed = (bits << torch.arange(32, device="cuda")).sum(2)
    return torch.where(packed >= 1 << 31, packed - (1 << 32), packed).to(torch.int32)


def _params(preset, rows, hist):
    p = default_params(rows)
    p["repeat_last_n"] = max(hist, 1)

    def put(sel, **kw):
        for k, v in kw.items():
            p[k][sel] = v

    topk = dict(temperature=0.8, top_k=40, top_p=0.95)
    pen = dict(repeat_penalty=1.1, frequency_penalty=0.5, presence_penalty=0.3)
    full = dict(temperature=0.7, min_p=0.05, top_p=0.9, **pen)
    if preset == "topk":
        put(slice(None), **topk)
    elif preset == "full":
        put(slice(None), **full)
    elif preset == "topp":
        put(slice(None), temperature=1.5, top_p=0.98)
    elif preset == "json":
        put(slice(None), temperature=1.0, top_p=0.95)
    elif preset == "minp_wide":
        put(slice(None), temperature=1.5, min_p=0.01, top_p=0.9, **pen)
    elif preset == "mixed":   # rows in turn greedy, top-k, the full chain, top-p
        put(slice(1, None, 4), **topk)
        put(slice(2, None, 4), **full)
        put(slice(3, None, 4), temperature=1.0, top_p=0.95)
    return p


_SIGMA = {"greedy": 2.0, "topk": 2.0, "full": 3.0, "topp": 1.0, "json": 2.5, "minp_wide": 1.0, "mixed": 2.5}


def _sample_logits(c, gen):
    logits = _logits(gen, c["rows"], c["vocab"], c["dtype"], _SIGMA[c["preset"]])
    if c["preset"] in ("greedy", "topk"):   # a confident model: a few ids stand out
        at = _ints(gen, 0, c["vocab"], (c["rows"], 8))
        logits.scatter_(1, at, logits.gather(1, at) + 12.0)
    return logits


def _prepare_sample(c, seed):
    gen, rng = _gen(seed), np.random.default_rng(seed)
    rows, vocab, preset, hist = c["rows"], c["vocab"], c["preset"], c["hist"]
    logits = _sample_logits(c, gen)
    params = _params(preset, rows, hist)
    d = {"logits": logits, "stride": logits.shape[1], "params_host": params,
         "params": torch.from_numpy(params.view(np.uint8).copy()).cuda(),
         "u": torch.from_numpy(rng.random(rows)).cuda()}
    if hist:   # every history full, or of any length up to hist
        lens = rng.integers(0, hist + 1, rows) if c["ragged"] else np.full(rows, hist)
        off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        d["hist_off"] = torch.from_numpy(off).cuda()
        d["hist_ids"] = _zipf(gen, vocab, max(int(off[-1]), 1))
    if preset == "json":
        d["mask"] = _mask(gen, rng, rows, vocab)
    n_top = c["n_top"]
    d["w"] = Workload(preset, rows, vocab, c["dtype"], None, params, None, None, n_top=n_top,
                      want_logprobs=n_top > 0)
    s = _sampler()
    out = s.alloc_out(rows, n_top, n_top > 0, diag=False)
    return {"s": s, "launch": s.prepare(d, out), "out": out}


def _verify_inputs(c, seed):
    """Logits with one dominant id a row, and drafts that hit it three times in four."""
    gen = _gen(seed)
    rows = c["n_seq"] * c["per_seq"]
    logits = _logits(gen, rows, c["vocab"], c["dtype"], 2.0)
    dom = _ints(gen, 0, c["vocab"], (rows, 1))
    logits.scatter_(1, dom, logits.amax(1, keepdim=True) + 6.0)
    hit = torch.rand(rows, generator=gen, device="cuda") < 0.75
    draft = torch.where(hit, dom[:, 0], _ints(gen, 0, c["vocab"], (rows,))).to(torch.int32)
    return logits, draft


def _prepare_verify(c, seed):
    logits, draft = _verify_inputs(c, seed)
    rows = c["n_seq"] * c["per_seq"]
    w = Workload("verify", rows, c["vocab"], c["dtype"], None, None, None, None, n_seq=c["n_seq"],
                 rows_per_seq=c["per_seq"])
    s = _sampler()
    out = s.alloc_verify_out(w)
    launch = s.prepare_verify({"logits": logits, "stride": logits.shape[1], "draft": draft, "w": w}, out)
    return {"s": s, "launch": launch, "out": out}


def _lmhead_inputs(c, seed):
    gen = _gen(seed)
    x = torch.randn(c["rows"], c["hidden"], generator=gen, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(c["vocab"], c["hidden"], generator=gen, device="cuda", dtype=torch.bfloat16)
    w.mul_(2.5 / math.sqrt(c["hidden"]))
    draft = None
    if c["per_seq"]:   # three drafts in four are what the model says
        best = (x @ w.t()).argmax(1)
        hit = torch.rand(c["rows"], generator=gen, device="cuda") < 0.75
        draft = torch.where(hit, best, _ints(gen, 0, c["vocab"], (c["rows"],))).to(torch.int32)
    return x, w, draft


def _prepare_lmhead(c, seed):
    x, w, draft = _lmhead_inputs(c, seed)
    s, per = _sampler(), c["per_seq"]
    out = s.alloc_lmhead_out(c["rows"], c["vocab"], logits=not per, draft=bool(per),
                             n_seq=c["rows"] // per if per else 0, stats=not per)
    shown = dict(out)
    if not per:   # lcs_row_stats: f64 log_z, f32 max, i32 argmax
        st = shown.pop("stats")
        shown.update(stats_log_z=st[:, 0], stats_max=st.view(torch.float32)[:, 2],
                     stats_argmax=st.view(torch.int32)[:, 3])
    return {"s": s, "x": x, "w": w, "draft": draft, "per": per, "buf": out, "out": shown}


def _logprobs_inputs(c, seed):
    gen = _gen(seed)
    logits = _logits(gen, c["rows"], c["vocab"], c["dtype"], 2.0)
    chosen = _ints(gen, 0, c["vocab"], (c["rows"], 1))
    # the text's token is likely under the model in two rows of three
    lift = 8.0 * (torch.rand(c["rows"], 1, generator=gen, device="cuda") < 0.67)
    logits.scatter_(1, chosen, logits.gather(1, chosen) + lift.to(logits.dtype))
    return logits, chosen[:, 0].to(torch.int32)


def _prepare_logprobs(c, seed):
    logits, chosen = _logprobs_inputs(c, seed)
    w = Workload("logprobs", c["rows"], c["vocab"], c["dtype"], None, None, None, None, n_top=c["n_top"],
                 want_logprobs=True)
    s = _sampler()
    out = s.alloc_out(c["rows"], c["n_top"], True, diag=False)
    return {"s": s, "d": {"logits": logits, "stride": logits.shape[1], "w": w}, "chosen": chosen, "out": out}


def _prepare_draft(c, seed):
    """Contexts of log-uniform length; in half of them the last n-gram occurs earlier."""
    gen, rng = _gen(seed), np.random.default_rng(seed)
    n, ng = c["n_seq"], c["ngram"]
    lens = np.exp(rng.uniform(math.log(c["ctx"] / 16), math.log(c["ctx"]), n)).astype(np.int64)
    off = np.concatenate([[0], np.cumsum(lens)])
    ids = _zipf(gen, 32000, int(off[-1]))
    src, dst = [], []
    for i in range(n):
        if lens[i] > 2 * ng and rng.random() < 0.5:
            at = int(off[i] + rng.integers(0, lens[i] - 2 * ng))
            src.append(np.arange(off[i + 1] - ng, off[i + 1]))
            dst.append(np.arange(at, at + ng))
    if src:
        ids[torch.from_numpy(np.concatenate(dst)).cuda()] = ids[torch.from_numpy(np.concatenate(src)).cuda()]
    off_d = torch.from_numpy(off.astype(np.int32)).cuda()
    draft = torch.full((n, c["max_draft"]), -7, dtype=torch.int32, device="cuda")
    length = torch.full((n,), -7, dtype=torch.int32, device="cuda")
    b = S._DBatch(n, ng, c["max_draft"], off_d.data_ptr(), ids.data_ptr())
    o = S._DOut(draft.data_ptr(), length.data_ptr())
    return {"s": _sampler(), "b": ctypes.byref(b), "o": ctypes.byref(o), "keep": (off_d, ids),
            "out": {"draft": draft, "draft_len": length}}


def prepare(case, seed):
    state = {"sample": _prepare_sample, "verify": _prepare_verify, "lmhead": _prepare_lmhead,
             "logprobs": _prepare_logprobs, "draft": _prepare_draft}[case["kind"]](case, seed)
    state["kind"] = case["kind"]
    return state


def run(state):
    kind, s = state["kind"], state["s"]
    if kind in ("sample", "verify"):
        state["launch"](s.stream_handle())
    elif kind == "lmhead":
        s.lmhead_dev(state["x"], state["w"], state["buf"], draft=state["draft"], rows_per_seq=state["per"])
    elif kind == "logprobs":
        s.logprobs_dev(state["d"], state["out"], chosen=state["chosen"])
    else:
        rc = S.lib().lcs_ngram_draft(s.ctx, state["b"], state["o"], s.stream_handle())
        if rc != S.LCS_OK:
            raise S.SamplerError(f"lcs_ngram_draft: {rc}")
    return state["out"]


# -------------------------------------------------------------- accounting --
def work(case):
    c = case
    if c["kind"] == "draft":   # half of the contexts are searched to their start
        mean = c["ctx"] * (15 / 16) / math.log(16)
        return {"bytes": c["n_seq"] * (4 * 0.75 * mean + 4 * (c["max_draft"] + 1)), "flops": 0}
    if c["kind"] == "lmhead":
        r, v, h = c["rows"], c["vocab"], c["hidden"]
        out = r * 12 + c["rows"] // c["per_seq"] * 4 if c["per_seq"] else r * (4 * v + 24)
        return {"bytes": 2 * h * (r + v) + out, "flops": 2 * r * v * h}
    esz = 2 if c["dtype"] == "bf16" else 4
    if c["kind"] == "verify":
        rows = c["n_seq"] * c["per_seq"]
        return {"bytes": rows * (esz * c["vocab"] + 12) + 4 * c["n_seq"], "flops": 0}
    row = esz * c["vocab"] + (4 + 4 + 8 * c["n_top"] if c["n_top"] or c["kind"] == "logprobs" else 4)
    if c["kind"] == "sample":
        row += 40 + 4 * c["hist"]
        if c["preset"] == "json":
            row += 4 * ((c["vocab"] + 31) // 32)
    else:
        row += 4
    return {"bytes": c["rows"] * row, "flops": 0}


def tolerance(case):
    if case["kind"] == "draft":
        return "exact"
    # measured against exact(): 4e-7 of the lm-head's f32 accumulation (the
    # largest of its logits' differences near 6 sigma of that), 1e-7 of the
    # logprobs' f32 sums and rounding; sampled ids do not differ
    if case["kind"] == "lmhead":
        return {"rel": 2e-6, "max": 2e-5, "differ": 0.004}
    return {"rel": 5e-7, "max": 5e-6}


def _top(lp, n_top):
    return torch.topk(lp, n_top, dim=1).values if n_top else lp.new_zeros(lp.shape[0], 1)


def exact(case, seed):
    c = case
    if c["kind"] == "draft" or (c["kind"] == "sample" and not c["n_top"]):
        return None
    if c["kind"] == "lmhead":
        x, w, draft = _lmhead_inputs(c, seed)
        xd = x.double()
        z = torch.cat([xd @ w[i:i + 8192].double().t() for i in range(0, c["vocab"], 8192)], 1)
        lz = torch.logsumexp(z, 1)
        if draft is None:
            return {"argmax_ids": None, "log_z": lz, "logits": z, "stats_log_z": lz, "stats_max": z.amax(1),
                    "stats_argmax": None}
        return {"argmax_ids": None, "log_z": lz, "accept_len": None,
                "draft_lp": z.gather(1, draft.long()[:, None])[:, 0] - lz}
    if c["kind"] == "sample":
        logits, ids = _sample_logits(c, _gen(seed)), None
    elif c["kind"] == "verify":
        logits, ids = _verify_inputs(c, seed)
    else:
        logits, ids = _logprobs_inputs(c, seed)
    n_top = c.get("n_top", 0)
    top, lps = [], []
    for i in range(0, logits.shape[0], 128):
        lp = torch.log_softmax(logits[i:i + 128, :c["vocab"]].double(), 1)
        top.append(_top(lp, n_top))
        if ids is not None:
            lps.append(lp.gather(1, ids[i:i + 128].long()[:, None])[:, 0])
    if c["kind"] == "verify":
        return {"argmax_ids": None, "draft_lp": torch.cat(lps), "accept_len": None}
    return {"ids": None, "chosen_lp": torch.cat(lps) if lps else None, "top_ids": None, "top_lp": torch.cat(top)}
