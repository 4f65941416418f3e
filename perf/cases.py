"""The work that programs on this library have it do, as cases that can be timed and compared.

Every case goes through the public C ABI (``stratakv_amd`` and its ctypes handles): paged decode of one
sequence and of batches, chunked prefill, one whole decoder layer for a token and for prompts, and the
head with the token choice.  Sizes are those of bench.py's configurations, of the tests, or generic.
"""
import ctypes
import math

import numpy as np
import torch

import stratakv_amd as skv

DEV = "cuda"
BLOCK = 16
EPS = 1e-5

# (query heads, kv heads, head_dim) of the batch decode and prefill work; bench.py's geometries first.
GEOMS = [(32, 4, 64), (32, 8, 128), (64, 8, 128), (8, 2, 64), (16, 16, 64), (8, 1, 128)]
# Further shapes that the entry points take: other groups, head dims and block sizes (query heads, kv
# heads, head_dim, block_size).
OTHER_GEOMS = [(24, 8, 128, 16), (12, 4, 64, 16), (40, 8, 128, 16), (16, 4, 128, 32), (28, 4, 128, 16),
               (8, 2, 96, 16), (8, 1, 256, 16), (32, 4, 64, 8)]
# Decoder layers: hidden, query heads, kv heads, head_dim, intermediate, vocabulary.
LAYERS = {"2048": (2048, 32, 4, 64, 5632, 32000), "4096": (4096, 32, 8, 128, 14336, 32000)}


def listed():
    return [
        # One token of a short chat: the attention call of every layer of a small generation, launch-bound.
        dict(name="decode_one_short", kind="decode_one", hq=32, hkv=4, hd=64, bs=16, ctx=137),
        # One token of one long conversation: few heads, one long table.
        dict(name="decode_one_long", kind="decode_one", hq=32, hkv=4, hd=64, bs=16, ctx=4097),
        # A serving batch of mixed contexts at head_dim 64, the fused append + decode step.
        dict(name="decode_batch_mixed", kind="decode_batch", hq=32, hkv=4, hd=64, bs=16, batch=64, dist="uniform",
             lo=512, hi=8192, append=True, q="bf16", kv="bf16", shape_seed=3),
        # A full serving batch of long log-normal contexts at head_dim 128: the largest call, HBM-bound.
        dict(name="decode_batch_long", kind="decode_batch", hq=32, hkv=8, hd=128, bs=16, batch=128, dist="lognormal",
             lo=2048, hi=32768, append=False, q="bf16", kv="bf16", shape_seed=4),
        # A batch of a model whose query heads per kv head are not a power of two.
        dict(name="decode_batch_group3", kind="decode_batch", hq=24, hkv=8, hd=128, bs=16, batch=24, dist="uniform",
             lo=200, hi=4096, append=True, q="bf16", kv="bf16", shape_seed=5),
        # New prompts entering a large model: whole 2,048-token chunks appended, then attended causally.
        dict(name="prefill_chunks", kind="prefill", hq=64, hkv=8, hd=128, bs=16, batch=4, chunk_lo=2048, chunk_hi=2048,
             prior_lo=0, prior_hi=0, q="bf16", kv="bf16", shape_seed=6),
        # Follow-up turns: short ragged chunks over long cached contexts, fp32 rows as the layers produce them.
        dict(name="prefill_followup", kind="prefill", hq=32, hkv=4, hd=64, bs=16, batch=3, chunk_lo=37, chunk_hi=300,
             prior_lo=1000, prior_hi=6000, q="fp32", kv="fp32", shape_seed=7),
        # One decode token through one layer: norms, projections, attention, feed-forward.
        dict(name="layer_token", kind="layer", layer="2048", rows=1, prior=300),
        # A short prompt through one layer.
        dict(name="layer_prompt_16", kind="layer", layer="2048", rows=16, prior=0),
        # A paragraph of a prompt through one layer.
        dict(name="layer_prompt_100", kind="layer", layer="2048", rows=100, prior=0),
        # A long prompt through one layer of a wider model.
        dict(name="layer_prompt_500_wide", kind="layer", layer="4096", rows=500, prior=0),
        # The end of a step: final norm, lm_head and the sampled token.
        dict(name="head_sample", kind="head", layer="2048", temperature=0.8, top_k=40, top_p=0.95),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode_one", "decode_batch", "decode_batch", "decode_other", "prefill", "prefill", "layer",
                       "layer", "head"])
    if kind == "decode_one":
        hq, hkv, hd = rng.choice(GEOMS)
        return dict(kind=kind, hq=hq, hkv=hkv, hd=hd, bs=BLOCK, ctx=_log_int(rng, 1, 32768))
    if kind in ("decode_batch", "decode_other"):
        other = kind == "decode_other"
        hq, hkv, hd, bs = rng.choice(OTHER_GEOMS) if other else rng.choice(GEOMS) + (BLOCK,)
        # The batch's K/V rows: up to the largest listed call's 5 GB, an eighth of that for the other shapes.
        most = int((5e8 if other else 4e9) / (4 * hkv * hd))
        batch = _log_int(rng, 2, 64 if other else 256)
        hi = min(_log_int(rng, 64, 16384), max(64, most // batch))
        return dict(kind="decode_batch", hq=hq, hkv=hkv, hd=hd, bs=bs, batch=batch, dist="uniform",
                    lo=rng.randint(1, hi), hi=hi, append=rng.random() < 0.7, q=rng.choice(["bf16", "bf16", "fp32"]),
                    kv=rng.choice(["bf16", "fp32"]), shape_seed=rng.randrange(1 << 20))
    if kind == "prefill":
        if rng.random() < 0.2:
            hq, hkv, hd, bs = rng.choice(OTHER_GEOMS)
            batch, hi, prior = rng.randint(1, 4), _log_int(rng, 8, 128), _log_int(rng, 16, 1024)
        else:
            hq, hkv, hd = rng.choice(GEOMS)
            bs, batch, hi = BLOCK, rng.randint(1, 6), _log_int(rng, 8, 2048)
            prior = 0 if rng.random() < 0.4 else _log_int(rng, 16, 8192)
            # No more products than the listed 4 x 2,048 tokens of 64 heads of 128.
            while batch * hi * (prior + hi / 2) * hq * hd > 4 * 2048 * 1024 * 64 * 128:
                batch, hi, prior = max(1, batch - 1), max(8, hi * 3 // 4), prior * 3 // 4
        return dict(kind="prefill", hq=hq, hkv=hkv, hd=hd, bs=bs, batch=batch, chunk_lo=rng.randint(1, hi), chunk_hi=hi,
                    prior_lo=prior // 2, prior_hi=prior, q=rng.choice(["bf16", "fp32"]), kv=rng.choice(["bf16", "fp32"]),
                    shape_seed=rng.randrange(1 << 20))
    if kind == "layer":
        layer = rng.choice(["2048", "2048", "4096"])
        rows = 1 if rng.random() < 0.3 else _log_int(rng, 2, 500 if layer == "4096" else 2048)
        return dict(kind="layer", layer=layer, rows=rows, prior=rng.choice([0, _log_int(rng, 1, 2048)]))
    return dict(kind="head", layer=rng.choice(["2048", "4096"]), temperature=round(rng.uniform(0.3, 1.5), 2),
                top_k=rng.choice([0, 1, 40, 200]), top_p=rng.choice([1.0, 0.95, 0.5]))


# ---------------------------------------------------------------------------
# Shapes and inputs.
# ---------------------------------------------------------------------------
def _lens(case):
    """Context lengths of a decode batch; (prior, chunk) lengths of a prefill batch."""
    rng = np.random.default_rng(case["shape_seed"])
    b = case["batch"]
    if case["kind"] == "prefill":
        return (rng.integers(case["prior_lo"], case["prior_hi"] + 1, b),
                rng.integers(case["chunk_lo"], case["chunk_hi"] + 1, b))
    if case["dist"] == "lognormal":  # median a quarter of the largest, sigma 0.6
        return np.clip(np.round(case["hi"] / 4 * np.exp(0.6 * rng.standard_normal(b))), case["lo"], case["hi"]).astype(np.int64)
    return rng.integers(case["lo"], case["hi"] + 1, b)


def _tables(lens, bs, seed):
    """Block tables over a fragmented pool of exactly the blocks needed and a few more."""
    nbs = [-(-int(n) // bs) for n in lens]
    total = sum(nbs) + 7
    perm = np.random.default_rng(seed).permutation(total).astype(np.int32)
    t = np.full((len(nbs), max(nbs)), -1, np.int32)
    pos = 0
    for b, nb in enumerate(nbs):
        t[b, :nb] = perm[pos:pos + nb]
        pos += nb
    return t, total


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, dtype="fp32", std=1.0):
    x = torch.randn(shape, generator=g, device=DEV, dtype=torch.bfloat16 if dtype == "bf16" else torch.float32)
    return x.mul_(std) if std != 1.0 else x


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _dtype(name):
    return skv.DTYPE_BF16 if name == "bf16" else skv.DTYPE_FP32


def _workspace(nbytes):
    return torch.empty(int(nbytes), dtype=torch.uint8, device=DEV)


def _prepare_decode_one(case, seed):
    hq, hkv, hd, bs = case["hq"], case["hkv"], case["hd"], case["bs"]
    g = _gen(seed)
    t, total = _tables([case["ctx"]], bs, seed)
    nbytes = skv.lib().skv_paged_attention_decode_workspace_bytes(hq, hkv, hd)
    return dict(case=case, total=total, table=_dev(t), k=_normal(g, (total, bs, hkv, hd), "bf16"),
                v=_normal(g, (total, bs, hkv, hd), "bf16"), q=_normal(g, (hq, hd)), k_new=_normal(g, (hkv, hd)),
                v_new=_normal(g, (hkv, hd)), out=torch.empty((hq, hd), device=DEV), ws=_workspace(nbytes), wsb=nbytes)


def _run_decode_one(s):
    c = s["case"]
    skv.paged_attention_decode_append(
        s["q"].data_ptr(), s["k_new"].data_ptr(), s["v_new"].data_ptr(), skv.DTYPE_FP32, s["k"].data_ptr(),
        s["v"].data_ptr(), s["total"], s["table"].data_ptr(), s["out"].data_ptr(), c["ctx"], c["bs"], c["hq"], c["hkv"],
        c["hd"], c["hd"] ** -0.5, s["ws"].data_ptr(), s["wsb"], torch.cuda.current_stream().cuda_stream)
    return {"out": s["out"], "k": s["k"], "v": s["v"]}


def _prepare_decode_batch(case, seed):
    hq, hkv, hd, bs, b = case["hq"], case["hkv"], case["hd"], case["bs"], case["batch"]
    g = _gen(seed)
    lens = _lens(case)
    t, total = _tables(lens, bs, seed)
    nbytes = skv.decode_workspace_bytes(b, hq, hkv, hd)
    return dict(case=case, total=total, width=t.shape[1], table=_dev(t), lens=_dev(lens.astype(np.int32)),
                k=_normal(g, (total, bs, hkv, hd), "bf16"), v=_normal(g, (total, bs, hkv, hd), "bf16"),
                q=_normal(g, (b, hq, hd), case["q"]), k_new=_normal(g, (b, hkv, hd), case["kv"]),
                v_new=_normal(g, (b, hkv, hd), case["kv"]), out=torch.empty((b, hq, hd), device=DEV),
                ws=_workspace(nbytes), wsb=nbytes)


def _run_decode_batch(s):
    c = s["case"]
    stream = torch.cuda.current_stream().cuda_stream
    if c["append"]:
        skv.paged_decode_append(
            s["q"].data_ptr(), _dtype(c["q"]), s["k_new"].data_ptr(), s["v_new"].data_ptr(), _dtype(c["kv"]),
            s["k"].data_ptr(), s["v"].data_ptr(), s["total"], s["table"].data_ptr(), s["width"], s["lens"].data_ptr(),
            c["batch"], c["hq"], c["hkv"], c["hd"], c["bs"], c["hd"] ** -0.5, s["out"].data_ptr(), s["ws"].data_ptr(),
            s["wsb"], stream)
        return {"out": s["out"], "k": s["k"], "v": s["v"]}
    skv.paged_decode(s["q"].data_ptr(), _dtype(c["q"]), s["k"].data_ptr(), s["v"].data_ptr(), s["total"],
                     s["table"].data_ptr(), s["width"], s["lens"].data_ptr(), c["batch"], c["hq"], c["hkv"], c["hd"],
                     c["bs"], c["hd"] ** -0.5, s["out"].data_ptr(), s["ws"].data_ptr(), s["wsb"], stream)
    return {"out": s["out"]}


def _prepare_prefill(case, seed):
    hq, hkv, hd, bs, b = case["hq"], case["hkv"], case["hd"], case["bs"], case["batch"]
    g = _gen(seed)
    prior, chunk = _lens(case)
    n = int(chunk.sum())
    t, total = _tables(prior + chunk, bs, seed)
    offsets = np.concatenate([[0], np.cumsum(chunk)]).astype(np.int32)
    return dict(case=case, total=total, width=t.shape[1], table=_dev(t), n=n, longest=int(chunk.max()),
                offsets=_dev(offsets), positions=_dev(prior.astype(np.int32)),
                lens=_dev((prior + chunk).astype(np.int32)), k=_normal(g, (total, bs, hkv, hd), "bf16"),
                v=_normal(g, (total, bs, hkv, hd), "bf16"), q=_normal(g, (n, hq, hd), case["q"]),
                k_new=_normal(g, (n, hkv, hd), case["kv"]), v_new=_normal(g, (n, hkv, hd), case["kv"]),
                out=torch.empty((n, hq, hd), device=DEV))


def _run_prefill(s):
    c = s["case"]
    stream = torch.cuda.current_stream().cuda_stream
    skv.kv_append(s["k_new"].data_ptr(), s["v_new"].data_ptr(), _dtype(c["kv"]), s["k"].data_ptr(), s["v"].data_ptr(),
                  s["total"], s["table"].data_ptr(), s["width"], s["positions"].data_ptr(), c["batch"], s["longest"],
                  c["hkv"], c["hd"], c["bs"], token_offsets=s["offsets"].data_ptr(), stream=stream)
    skv.paged_prefill(s["q"].data_ptr(), _dtype(c["q"]), s["k"].data_ptr(), s["v"].data_ptr(), s["total"],
                      s["table"].data_ptr(), s["width"], s["offsets"].data_ptr(), s["lens"].data_ptr(), c["batch"],
                      s["n"], c["hq"], c["hkv"], c["hd"], c["bs"], c["hd"] ** -0.5, s["out"].data_ptr(), stream)
    return {"out": s["out"], "k": s["k"], "v": s["v"]}


def _prepare_layer(case, seed):
    hidden, hq, hkv, hd, inter, _ = LAYERS[case["layer"]]
    rows, prior, kvd = case["rows"], case["prior"], hkv * hd
    g = _gen(seed)
    t, total = _tables([prior + rows], BLOCK, seed)
    f = lambda *shape: torch.empty(shape, device=DEV)  # noqa: E731
    s = dict(case=case, total=total, table=_dev(t), width=t.shape[1],
             x=_normal(g, (rows, hidden)), gamma1=1 + _normal(g, (hidden,), std=0.1),
             gamma2=1 + _normal(g, (hidden,), std=0.1),
             # q, k, v and gate, up rows packed one after another, as the checkpoint loader lays them out.
             wqkv=_normal(g, (hq * hd + 2 * kvd, hidden), "bf16", 0.02), wo=_normal(g, (hidden, hq * hd), "bf16", 0.02),
             wgu=_normal(g, (2 * inter, hidden), "bf16", 0.02), wd=_normal(g, (hidden, inter), "bf16", 0.02),
             k=_normal(g, (total, BLOCK, hkv, hd), "bf16"), v=_normal(g, (total, BLOCK, hkv, hd), "bf16"),
             q=f(rows, hq * hd), k_new=f(rows, kvd), v_new=f(rows, kvd), ctx=f(rows, hq * hd), h=f(rows, hidden),
             act=f(rows, inter), up=f(rows, inter), norm=f(rows, hidden), y=f(rows, hidden),
             positions=_dev(np.array([prior], np.int32)), offsets=_dev(np.array([0, rows], np.int32)),
             lens=_dev(np.array([prior + rows], np.int32)), strides=(ctypes.c_int64 * 3)(hidden, hidden, hidden))
    if rows == 1:
        s["wsb"] = skv.lib().skv_paged_attention_decode_workspace_bytes(hq, hkv, hd)
    else:
        s["wsb"] = 0
        if rows >= 256:
            need = skv.gemm_lib().skv_prompt_gemm_workspace_bytes
            s["wsb"] = max(need(rows, hidden, hq * hd + 2 * kvd), need(rows, hq * hd, hidden),
                           need(rows, max(hidden, min(inter, 8192)), max(2 * inter, hidden)))
    s["ws"] = _workspace(s["wsb"] + 256)
    return s


def _taken(rc):
    """False when an entry point does not take the shape (nothing launched); raises on any other failure."""
    if rc == skv.SKV_ERR_UNSUPPORTED:
        return False
    if rc != skv.SKV_OK:
        raise skv.SkvError(rc, skv.lib().skv_last_error().decode(errors="replace"))
    return True


def _run_layer(s):
    c = s["case"]
    hidden, hq, hkv, hd, inter, _ = LAYERS[c["layer"]]
    rows, prior, kvd, qd = c["rows"], c["prior"], hkv * hd, hq * hd
    lib, bf16, st = skv.lib(), skv.DTYPE_BF16, torch.cuda.current_stream().cuda_stream
    p = {n: s[n].data_ptr() for n in ("x", "gamma1", "gamma2", "wqkv", "wo", "wgu", "wd", "k", "v", "q", "k_new",
                                      "v_new", "ctx", "h", "act", "up", "norm", "y", "table", "ws")}
    wk, wv, wu = p["wqkv"] + 2 * qd * hidden, p["wqkv"] + 2 * (qd + kvd) * hidden, p["wgu"] + 2 * inter * hidden
    ws = -(-p["ws"] // 256) * 256
    qkv = (p["gamma1"], EPS, p["wqkv"], wk, wv, bf16, 1, s["strides"], None, None, None, hidden, hq, hkv, hd, prior,
           p["q"], p["k_new"], p["v_new"])
    gate_up = (p["gamma2"], EPS, p["wgu"], wu, bf16, 1, hidden, hidden, None, None, hidden, inter, p["act"])
    if rows == 1:
        _taken(lib.skv_fused_qkv_f32(p["x"], *qkv, st))
        skv.paged_attention_decode_append(p["q"], p["k_new"], p["v_new"], skv.DTYPE_FP32, p["k"], p["v"], s["total"],
                                          p["table"], p["ctx"], prior + 1, BLOCK, hq, hkv, hd, hd ** -0.5, ws, s["wsb"], st)
        _taken(lib.skv_linear_residual_f32(p["ctx"], p["wo"], bf16, 1, qd, qd, hidden, None, p["x"], p["h"], st))
        _taken(lib.skv_fused_gate_up_swiglu_f32(p["h"], *gate_up, st))
        down = _taken(lib.skv_linear_residual_f32(p["act"], p["wd"], bf16, 1, inter, inter, hidden, None, p["h"], p["y"], st))
    else:
        # The entry points of the prompt's length: library GEMMs, matrix cores, or the row kernels.
        how = "gemm" if rows >= 256 else "mm" if rows >= 32 else "rows"
        src = skv.gemm_lib() if how == "gemm" else lib
        more = (ws, s["wsb"], st) if how == "gemm" else (st,)
        fused_qkv = getattr(src, "skv_fused_qkv_%s_f32" % how)
        residual = getattr(src, "skv_linear_residual_%s_f32" % how)
        _taken(fused_qkv(p["x"], rows, *qkv, p["norm"], *more))
        skv.kv_append(p["k_new"], p["v_new"], skv.DTYPE_FP32, p["k"], p["v"], s["total"], p["table"], s["width"],
                      s["positions"].data_ptr(), 1, rows, hkv, hd, BLOCK, stream=st)
        skv.paged_prefill(p["q"], skv.DTYPE_FP32, p["k"], p["v"], s["total"], p["table"], s["width"],
                          s["offsets"].data_ptr(), s["lens"].data_ptr(), 1, rows, hq, hkv, hd, BLOCK, hd ** -0.5,
                          p["ctx"], st)
        _taken(residual(p["ctx"], rows, p["wo"], bf16, 1, qd, qd, hidden, None, p["x"], p["h"], *more))
        if how == "gemm" and inter <= 8192:
            down = _taken(src.skv_ffn_swiglu_gemm_f32(p["h"], rows, p["gamma2"], EPS, p["wgu"], wu, p["wd"], bf16, 1,
                                                      hidden, hidden, inter, None, None, None, hidden, inter, p["y"],
                                                      p["norm"], *more))
        else:
            _taken(getattr(src, "skv_fused_gate_up_swiglu_%s_f32" % how)(p["h"], rows, *gate_up, p["norm"], *more))
            down = inter <= 8192 and _taken(residual(p["act"], rows, p["wd"], bf16, 1, inter, inter, hidden, None, p["h"],
                                                     p["y"], *more))
    if not down:  # wider than the fused projections take: the separate projection and add
        _taken(lib.skv_linear_f32(p["act"], rows, p["wd"], bf16, 1, inter, inter, hidden, None, p["y"], st))
        _taken(lib.skv_add_f32(p["y"], p["h"], rows * hidden, st))
    return {"y": s["y"], "k": s["k"], "v": s["v"]}


def _prepare_head(case, seed):
    hidden, vocab = LAYERS[case["layer"]][0], LAYERS[case["layer"]][5]
    g = _gen(seed)
    return dict(case=case, x=_normal(g, (1, hidden)), gamma=1 + _normal(g, (hidden,), std=0.1),
                w=_normal(g, (vocab, hidden), "bf16", 0.02), norm=torch.empty((1, hidden), device=DEV),
                logits=torch.empty(vocab, device=DEV), token=torch.zeros(1, dtype=torch.int32, device=DEV),
                flags=torch.zeros(1, dtype=torch.int32, device=DEV),
                uniform=float(np.random.default_rng(seed).random()))


def _run_head(s):
    c = s["case"]
    hidden, vocab = LAYERS[c["layer"]][0], LAYERS[c["layer"]][5]
    lib, st = skv.lib(), torch.cuda.current_stream().cuda_stream
    _taken(lib.skv_rmsnorm_f32(s["x"].data_ptr(), s["norm"].data_ptr(), s["gamma"].data_ptr(), 1, hidden, EPS, st))
    _taken(lib.skv_linear_f32(s["norm"].data_ptr(), 1, s["w"].data_ptr(), skv.DTYPE_BF16, 1, hidden, hidden, vocab, None,
                              s["logits"].data_ptr(), st))
    skv.sample(s["logits"].data_ptr(), vocab, c["temperature"], c["top_k"], c["top_p"], s["uniform"],
               s["token"].data_ptr(), 0, s["flags"].data_ptr(), st)
    return {"logits": s["logits"], "token": s["token"], "flags": s["flags"]}


def prepare(case, seed):
    kind = case["kind"]
    return {"decode_one": _prepare_decode_one, "decode_batch": _prepare_decode_batch, "prefill": _prepare_prefill,
            "layer": _prepare_layer, "head": _prepare_head}[kind](case, seed)


_RUN = {"decode_one": _run_decode_one, "decode_batch": _run_decode_batch, "prefill": _run_prefill, "layer": _run_layer,
        "head": _run_head}


def run(state):
    return _RUN[state["case"]["kind"]](state)


# ---------------------------------------------------------------------------
# What a pass cannot do without, and what its outputs are in 64 bits.
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "head":
        hidden, vocab = LAYERS[case["layer"]][0], LAYERS[case["layer"]][5]
        return {"bytes": 2 * hidden * vocab + 8 * hidden + 4 * vocab, "flops": 2 * hidden * vocab}
    if kind == "layer":
        hidden, hq, hkv, hd, inter, _ = LAYERS[case["layer"]]
        rows, prior = case["rows"], case["prior"]
        weights = hidden * (2 * hq * hd + 2 * hkv * hd + 3 * inter)
        keys = rows * prior + rows * (rows + 1) // 2
        return {"bytes": 2 * weights + 4 * hkv * hd * (prior + 2 * rows) + 8 * rows * hidden,
                "flops": 2 * rows * weights + 4 * hq * hd * keys}
    hq, hkv, hd = case["hq"], case["hkv"], case["hd"]
    if kind == "prefill":
        prior, chunk = _lens(case)
        keys = int((chunk * prior + chunk * (chunk + 1) // 2).sum())
        n, row = int(chunk.sum()), hkv * hd
        sq, skv_ = (4 if case["q"] == "fp32" else 2), (4 if case["kv"] == "fp32" else 2)
        return {"bytes": 4 * row * int((prior + chunk).sum()) + 2 * n * row * (skv_ + 2) + n * hq * hd * (sq + 4),
                "flops": 4 * hq * hd * keys}
    lens = np.array([case["ctx"]]) if kind == "decode_one" else _lens(case)
    b, tokens = len(lens), int(lens.sum())
    q32 = kind == "decode_one" or case["q"] == "fp32"
    new = 2 * b * hkv * hd * (2 + (4 if kind == "decode_one" or case["kv"] == "fp32" else 2))
    appends = kind == "decode_one" or case["append"]
    return {"bytes": 4 * hkv * hd * tokens + 4 * -(-tokens // case["bs"]) + b * hq * hd * (8 if q32 else 6) +
            (new if appends else 0), "flops": 4 * hq * hd * tokens}


def _bf16(x):
    return x.float().bfloat16()


def _rows_of(pool, table, n, bs):
    """The first n rows of one sequence, in 64 bits: [heads][n][head_dim]."""
    blocks = table[:-(-n // bs)].long()
    return pool[blocks].reshape(-1, pool.shape[2], pool.shape[3])[:n].double().transpose(0, 1).contiguous()


def _attend(q, k, v, first):
    """Causal attention of q [n][Hq][hd], row i at position first + i, over k, v [Hkv][len][hd]; 64 bits."""
    n, hq, hd = q.shape
    hkv, length = k.shape[0], k.shape[1]
    qh = (q.double() * hd ** -0.5).reshape(n, hkv, hq // hkv, hd)
    out = torch.empty((n, hkv, hq // hkv, hd), dtype=torch.float64, device=q.device)
    visible = torch.arange(length, device=q.device)[None, :] <= first + torch.arange(n, device=q.device)[:, None]
    for h in range(hkv):
        kt = k[h].t().contiguous()
        for g in range(hq // hkv):
            sc = (qh[:, h, g].contiguous() @ kt).masked_fill_(~visible, -math.inf)
            out[:, h, g] = torch.softmax(sc, 1) @ v[h]
    return out.reshape(n, hq, hd)


def _place(pool, table, first, rows, bs):
    """Writes rows [n][heads][head_dim] at positions first.. of one sequence."""
    pos = first + torch.arange(rows.shape[0], device=DEV)
    pool[table[pos // bs].long(), pos % bs] = rows if rows.dtype == torch.bfloat16 else _bf16(rows)


def _exact_layer(case, seed):
    hidden, hq, hkv, hd, inter, _ = LAYERS[case["layer"]]
    rows, prior, kvd = case["rows"], case["prior"], hkv * hd
    s = _prepare_layer(case, seed)

    def norm(x, gamma):
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * gamma.double()

    def product(x, w):
        return x @ w.double().t().contiguous()

    inv = (10000.0 ** (-2.0 * torch.arange(hd // 2, device=DEV, dtype=torch.float64) / hd)).float().double()
    angle = (prior + torch.arange(rows, device=DEV, dtype=torch.float64))[:, None] * inv
    cos, sin = torch.cos(angle)[:, None], torch.sin(angle)[:, None]

    def rope(x):
        a, b = x[..., :hd // 2], x[..., hd // 2:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    x = s["x"].double()
    qkv = product(norm(x, s["gamma1"]), s["wqkv"])
    q = rope(qkv[:, :hq * hd].reshape(rows, hq, hd))
    _place(s["k"], s["table"][0], prior, rope(qkv[:, hq * hd:hq * hd + kvd].reshape(rows, hkv, hd)), BLOCK)
    _place(s["v"], s["table"][0], prior, qkv[:, hq * hd + kvd:].reshape(rows, hkv, hd), BLOCK)
    n = prior + rows
    ctx = _attend(q, _rows_of(s["k"], s["table"][0], n, BLOCK), _rows_of(s["v"], s["table"][0], n, BLOCK), prior)
    h = x + product(ctx.reshape(rows, -1), s["wo"])
    gu = product(norm(h, s["gamma2"]), s["wgu"])
    gate, up = gu[:, :inter], gu[:, inter:]
    y = h + product(gate * torch.sigmoid(gate) * up, s["wd"])
    return {"y": y, "k": s["k"].double(), "v": s["v"].double()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "layer":
        return _exact_layer(case, seed)
    if kind == "head":
        s = _prepare_head(case, seed)
        x = s["x"].double()
        x = x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * s["gamma"].double()
        return {"logits": s["w"].double() @ x[0], "token": None, "flags": None}
    s = prepare(case, seed)
    bs, table = case["bs"], s["table"]
    if kind == "prefill":
        prior, chunk = _lens(case)
        off = np.concatenate([[0], np.cumsum(chunk)])
        out = []
        for b in range(case["batch"]):
            rows = slice(int(off[b]), int(off[b + 1]))
            first, n = int(prior[b]), int(prior[b] + chunk[b])
            _place(s["k"], table[b], first, s["k_new"][rows], bs)
            _place(s["v"], table[b], first, s["v_new"][rows], bs)
            out.append(_attend(s["q"][rows], _rows_of(s["k"], table[b], n, bs), _rows_of(s["v"], table[b], n, bs), first))
        return {"out": torch.cat(out), "k": s["k"].double(), "v": s["v"].double()}
    lens = [case["ctx"]] if kind == "decode_one" else _lens(case)
    one = (lambda x, b: x[None]) if kind == "decode_one" else (lambda x, b: x[b:b + 1])
    out = []
    for b, n in enumerate(int(x) for x in lens):
        if kind == "decode_one" or case["append"]:
            _place(s["k"], table[b], n - 1, one(s["k_new"], b), bs)
            _place(s["v"], table[b], n - 1, one(s["v_new"], b), bs)
        out.append(_attend(one(s["q"], b), _rows_of(s["k"], table[b], n, bs), _rows_of(s["v"], table[b], n, bs), n - 1))
    out = torch.cat(out)
    if kind == "decode_one":
        return {"out": out[0], "k": s["k"].double(), "v": s["v"].double()}
    return {"out": out, "k": s["k"].double(), "v": s["v"].double()} if case["append"] else {"out": out}


def tolerance(case):
    # About four times the errors against exact() that the cases show, or what one rounding step gives.
    kind = case["kind"]
    if kind == "head":
        return {"rel": 5e-6}            # fp32 sums of bf16 weights
    if kind == "layer":                 # K/V rows rounded to bf16, so one step of bf16 now and then; fp16 P in prompts
        return {"rel": 1e-3, "max": 1.6e-2}
    if kind == "prefill":               # probabilities rounded to fp16
        return {"rel": 1e-3, "max": 1.6e-2}
    return {"rel": 1e-5, "max": 4e-4}   # fp32 sums; an fp32 query keeps ~17 bits
