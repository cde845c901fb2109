"""What the performance of this package is measured on: the calls a speculative-decoding server
makes in a round, each through its public entry point, with inputs made on the GPU from a seed.

A case's ``kind`` names the call:

  greedy   accept_greedy: argmax acceptance of a temperature-0 round
  verify   verify_step: the fused sampled verification, dense or ragged rows
  topk     kernels.dspine.topk on verification rows
  probs    build_dspine_target_probs: the dense target distribution
  filter   filter_target_probs: the backend filter on given probabilities
  sparse   build_sparse_target, then accept_sparse on what it built
  table    serial_rs_table: the draft's float32 q table
  factor   factor_table: the draft's float64 q table from the per-model cache
  round    the small calls around a round: uniforms, the K-lane draft chain, the verify-length
           plan with its window index, and the commit of the accepted slots
"""

from __future__ import annotations

import math
from types import SimpleNamespace

import torch

DEV = "cuda"
TOP_K_ALL = 1 << 30
BIG = 64 * 17 * 151936  # logits of the largest verification batch

# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------


def listed():
    return [
        # one interactive user at temperature 0: the smallest verification there is, launch bound
        dict(name="greedy_1x17_f32", kind="greedy", bs=1, T=17, V=151936, dtype="f32"),
        # a busy server's round: greedy, top-k and nucleus requests mixed, penalties over a
        # 512-token history, KV slots
        dict(name="verify_64x17_mixed", kind="verify", bs=64, T=17, V=151936, dtype="bf16", mix="serving", hist=512,
             backend="pytorch", ragged=False, peak=0.0),
        # four users sampling with drafts that are mostly accepted: an ordinary interactive round
        dict(name="verify_4x17_deep", kind="verify", bs=4, T=17, V=151936, dtype="bf16", mix="serving", hist=512,
             backend="pytorch", ragged=False, peak=16.0),
        # float32 logits, every request top-k 20 with top-p 0.95
        dict(name="verify_32x17_topk_f32", kind="verify", bs=32, T=17, V=151936, dtype="f32", mix="topk", hist=0,
             backend="pytorch", ragged=False, peak=0.0),
        # verify lengths from a planner (4 to 16 rows a request) on compact rows, a wide vocabulary,
        # nucleus sampling of heavy-tailed logits
        dict(name="verify_32_ragged_262144", kind="verify", bs=32, T=17, V=262144, dtype="bf16", mix="heavy", hist=0,
             backend="pytorch", ragged=True, peak=0.0),
        # candidate lanes of every row of a round
        dict(name="topk20_1088", kind="topk", bs=64, T=17, V=151936, dtype="bf16", k=20),
        # the dense target distribution of that round, for callers that need P itself
        dict(name="probs_64x17_mixed", kind="probs", bs=64, T=17, V=151936, dtype="bf16", mix="serving",
             backend="pytorch"),
        # a caller's own probabilities filtered (its softmax ran elsewhere)
        dict(name="filter_32x17_mixed", kind="filter", bs=32, T=17, V=151936, mix="serving", backend="pytorch"),
        # the small-support joint target of a top-k batch, and chain rejection on it
        dict(name="sparse_24x16", kind="sparse", bs=24, T=16, V=151936, dtype="bf16"),
        # the draft side of a 64-request round: the float32 table of every block row
        dict(name="table_64x16", kind="table", bs=64, T=16, K=16, H=4096, R=512, C=1024, V=32768, RR=0),
        # the same table from the float64 factors
        dict(name="factor_64x16", kind="factor", bs=64, T=16, K=16, H=4096, R=512, C=1024, V=32768),
        # the launches of a few microseconds that surround every round
        dict(name="round_64x16", kind="round", bs=64, T=16, K=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _vocab(rng, lo=8192, hi=262144):
    v = _log(rng, lo, hi)
    # most vocabularies are padded to a multiple of 64; some are not padded at all
    return v if rng.random() < 0.3 else max(64, v // 64 * 64)


def draw(rng):
    kind = rng.choice(["greedy", "verify", "verify", "verify", "topk", "probs", "filter", "sparse", "table", "factor",
                       "round"])
    T = rng.randint(3, 17)
    c = dict(kind=kind, bs=_log(rng, 1, 64), T=T)
    if kind == "round":
        c.update(bs=_log(rng, 2, 64), K=rng.choice([5, 8, 16, 16, 32]))
        return c
    if kind in ("table", "factor"):
        c.update(K=rng.choice([5, 8, 16, 16]), H=rng.choice([512, 1024, 2048, 2560, 4096]),
                 R=rng.choice([64, 128, 192, 256, 512]), C=rng.choice([64, 272, 512, 1024]), V=_log(rng, 2048, 32768))
        if kind == "table":
            c.update(K=rng.choice([5, 8, 16, 16, 24]), RR=rng.choice([0, 0, 32]))
        return c
    c.update(V=_vocab(rng))
    size = {"bf16": 1, "f32": 2}
    dtype = rng.choice(["bf16", "bf16", "f32"])
    if kind == "greedy":
        c.update(dtype=dtype)
    elif kind == "verify":
        c.update(dtype=dtype, mix=rng.choice(["serving", "serving", "topk", "nucleus", "plain", "heavy"]),
                 hist=rng.choice([0, 64, 512]), backend=rng.choice(["pytorch", "pytorch", "flashinfer"]),
                 ragged=rng.random() < 0.3, peak=rng.choice([0.0, 16.0]))
    elif kind == "topk":
        c.update(dtype=dtype, k=rng.choice([1, 5, 16, 20, 33, 64]))
    elif kind == "probs":
        c.update(dtype=dtype, mix=rng.choice(["serving", "topk", "nucleus", "plain", "minp"]),
                 backend=rng.choice(["pytorch", "flashinfer"]))
    elif kind == "filter":
        c.update(mix=rng.choice(["serving", "topk", "nucleus", "minp"]),
                 backend=rng.choice(["pytorch", "flashinfer"]))
        dtype = "f32"
    else:
        c.update(dtype="bf16", T=16)
        dtype = "f32"  # its P is
    most = BIG // size[dtype]
    while c["bs"] > 1 and c["bs"] * c["T"] * c["V"] > most:
        c["bs"] //= 2
    return c


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _logits(g, rows, V, mix, dtype, peak):
    if mix == "heavy":  # 2 x Student-t, 3 degrees of freedom
        x = _randn(g, rows, V)
        chi = sum(_randn(g, rows, V).square_() for _ in range(3))
        x = 2.0 * x / (chi / 3.0).sqrt_()
    else:
        x = _randn(g, rows, V) * 2.5
    if peak:  # one likely next token a row
        at = torch.randint(0, V, (rows, 1), generator=g, device=DEV)
        x.scatter_(1, at, peak - 1.0 + 2.0 * torch.rand(rows, 1, generator=g, device=DEV))
    return x.to(torch.bfloat16 if dtype == "bf16" else torch.float32)


def _info(g, bs, mix):
    """The sampling parameters a server's batch carries, with the batch flags it knows."""
    pick = lambda values: torch.tensor(values, device=DEV)[  # noqa: E731
        torch.randint(0, len(values), (bs,), generator=g, device=DEV)]
    one = lambda v: torch.full((bs,), float(v), device=DEV)  # noqa: E731
    min_p = torch.zeros(bs, device=DEV)
    if mix == "serving":
        t, k, p = pick([0.0, 0.6, 1.0]), pick([0, 20]), pick([1.0, 0.95])
    elif mix == "topk":
        t, k, p = one(1.0), torch.full((bs,), 20, device=DEV), one(0.95)
    elif mix == "nucleus":
        t, k, p = pick([0.6, 1.0]), torch.zeros(bs, device=DEV, dtype=torch.int64), pick([0.9, 0.95])
    elif mix == "heavy":
        t, k, p = one(1.0), torch.zeros(bs, device=DEV, dtype=torch.int64), one(0.9)
    elif mix == "minp":
        t, k, p = pick([0.7, 1.0]), pick([0, 40]), pick([1.0, 0.95])
        min_p = pick([0.0, 0.05])
    else:  # plain sampling
        t, k, p = pick([0.8, 1.0]), torch.zeros(bs, device=DEV, dtype=torch.int64), one(1.0)
    greedy = t <= 0
    k = torch.where(k <= 0, torch.full_like(k, TOP_K_ALL), k)
    k = torch.where(greedy, torch.ones_like(k), k).to(torch.int32)
    t = torch.where(greedy, torch.ones_like(t), t)
    return SimpleNamespace(
        temperatures=t.view(-1, 1), top_ks=k, top_ps=p, min_ps=min_p,
        need_top_k_sampling=bool(((k > 1) & (k < TOP_K_ALL)).any()), need_top_p_sampling=bool((p < 1.0).any()),
        need_min_p_sampling=bool((min_p > 0).any()), is_any_greedy=bool((k <= 1).any()),
        is_all_greedy=bool((k <= 1).all()), max_top_k=int(k.max()))


def _draft(g, logits, row0, n, bs, T, K, noise):
    """Sparse q [bs, T-1, K] from noisy target rows (row row0[b] + s, the last of a short request
    repeated), and the drafts sampled from it."""
    V = logits.shape[1]
    step = torch.arange(T - 1, device=DEV)
    rows = (row0[:, None] + torch.minimum(step[None, :], (n - 1)[:, None])).reshape(-1)
    ids, q = [], []
    for part in rows.split(256):  # (bounded: a noisy float32 copy of the rows is made)
        noisy = logits[part].float() + noise * _randn(g, part.numel(), V)
        v, i = torch.topk(noisy, K, dim=-1)
        i, at = i.sort(-1)
        ids.append(i)
        q.append(torch.softmax(v.gather(-1, at), -1))
    ids, q = torch.cat(ids), torch.cat(q)
    lane = torch.multinomial(q, 1, generator=g)
    cand = torch.cat((torch.randint(0, V, (bs, 1), generator=g, device=DEV),
                      ids.gather(1, lane).view(bs, T - 1)), 1).contiguous()
    return cand, ids.view(bs, T - 1, K), q.view(bs, T - 1, K).contiguous()


def _outputs(bs, T):
    z = lambda shape, dt: torch.zeros(shape, device=DEV, dtype=dt)  # noqa: E731
    return (z(bs, torch.int32), z(bs, torch.int32), z(bs, torch.int64), z((bs, T), torch.int64), z(bs, torch.int32))


def _prefix(g, bs):
    return torch.randint(64, 4000, (bs,), generator=g, device=DEV).to(torch.int32)


def _prepare_greedy(c, g):
    bs, T, V = c["bs"], c["T"], c["V"]
    logits = _logits(g, bs * T, V, "plain", c["dtype"], 0.0)
    top = logits.argmax(-1).view(bs, T)
    cand = torch.zeros((bs, T), device=DEV, dtype=torch.int64)
    cand[:, 1:] = top[:, :-1]
    # one wrong draft a request
    at = 1 + torch.randint(0, T - 1, (bs, 1), generator=g, device=DEV)
    cand.scatter_(1, at, (cand.gather(1, at) + 1) % V)
    return SimpleNamespace(logits=logits, cand=cand, prefix=_prefix(g, bs), outs=_outputs(bs, T))


def _run_greedy(c, s):
    from dspine_amd.verification.caps import accept_greedy

    return accept_greedy(candidates=s.cand, next_token_logits=s.logits, prefix_lens=s.prefix, cap=c["T"],
                         outputs=s.outs)


def _lengths(T):
    """[lowest, highest + 1) verify length of a ragged request."""
    return min(4, T - 1), T


def _prepare_verify(c, g):
    from dspine_amd.verify import History, Workspace

    bs, T, V, K = c["bs"], c["T"], c["V"], 16
    if c["ragged"]:
        n = torch.randint(*_lengths(T), (bs,), generator=g, device=DEV)
        row0 = torch.cat((n.new_zeros(1), n.cumsum(0)))[:-1].contiguous()
        rows = int(n.sum())
    else:
        n = torch.full((bs,), T, device=DEV)
        row0, rows = torch.arange(bs, device=DEV) * T, bs * T
    logits = _logits(g, rows, V, c["mix"], c["dtype"], c["peak"])
    cand, q_ids, q = _draft(g, logits, row0, n, bs, T, K, 1.0)
    hist = None
    if c["hist"]:
        ids = torch.randint(0, V, (bs, c["hist"]), generator=g, device=DEV).to(torch.int32)
        hist = History(ids, torch.full((bs,), 0.5, device=DEV), torch.full((bs,), 1.1, device=DEV))
    page = torch.randint(0, 1 << 20, (bs, 4096 + 128), generator=g, device=DEV).to(torch.int32)
    u = torch.rand(bs, T, generator=g, device=DEV)
    return SimpleNamespace(
        logits=logits, info=_info(g, bs, c["mix"]), cand=cand, q_ids=q_ids, q=q, u=u[:, :-1].contiguous(),
        uf=u[:, -1].contiguous(), prefix=_prefix(g, bs), hist=hist, page=page, outs=_outputs(bs, T),
        kv=torch.zeros((bs, T), device=DEV, dtype=torch.int32), ws=Workspace(),
        lens=n.to(torch.int32) if c["ragged"] else None, row0=row0 if c["ragged"] else None)


def _run_verify(c, s):
    from dspine_amd.verify import verify_step

    outs, kv = verify_step(logits=s.logits, sampling_info=s.info, candidates=s.cand, q_ids=s.q_ids, q_values=s.q,
                           uniforms=s.u, uniform_final=s.uf, prefix_lens=s.prefix, verify_lens=s.lens,
                           row_offsets=s.row0, history=s.hist, page_table=s.page, outputs=s.outs, kv_slots=s.kv,
                           sampling_backend=c["backend"], workspace=s.ws)
    return {"outs": outs, "kv": kv}


def _prepare_topk(c, g):
    return SimpleNamespace(logits=_logits(g, c["bs"] * c["T"], c["V"], "plain", c["dtype"], 0.0))


def _run_topk(c, s):
    from dspine_amd.kernels.dspine import topk

    return topk(s.logits, c["k"])


def _prepare_probs(c, g):
    logits = _logits(g, c["bs"] * c["T"], c["V"], c["mix"], c["dtype"], 0.0)
    return SimpleNamespace(logits=logits, info=_info(g, c["bs"], c["mix"]))


def _run_probs(c, s):
    from dspine_amd.runtime.worker import build_dspine_target_probs

    return build_dspine_target_probs(next_token_logits=s.logits, sampling_info=s.info, block_size=c["T"], bs=c["bs"],
                                     sampling_backend=c["backend"])


def _prepare_filter(c, g):
    x = _logits(g, c["bs"] * c["T"], c["V"], c["mix"], "f32", 0.0)
    info = _info(g, c["bs"], c["mix"])
    t = info.temperatures.view(-1).repeat_interleave(c["T"])
    return SimpleNamespace(p=torch.softmax(x / t[:, None], -1), info=info)


def _run_filter(c, s):
    from dspine_amd.runtime.worker import filter_target_probs

    return filter_target_probs(s.p, s.info, c["T"], c["bs"], c["backend"])


def _prepare_sparse(c, g):
    bs, T, V = c["bs"], c["T"], c["V"]
    logits = _logits(g, bs * T, V, "plain", c["dtype"], 0.0)
    pick = lambda values: torch.tensor(values, device=DEV)[  # noqa: E731
        torch.randint(0, len(values), (bs,), generator=g, device=DEV)]
    info = SimpleNamespace(temperatures=pick([0.6, 1.0]).view(-1, 1), top_ks=pick([8, 20, 32]).to(torch.int32),
                           top_ps=pick([1.0, 0.95, 0.6]), min_ps=torch.zeros(bs, device=DEV),
                           need_top_k_sampling=True, need_top_p_sampling=True, need_min_p_sampling=False,
                           is_any_greedy=False, is_all_greedy=False, max_top_k=32)
    cand, q_ids, q = _draft(g, logits, torch.arange(bs, device=DEV) * T, torch.full((bs,), T, device=DEV), bs, T, 16,
                            0.5)
    u = torch.rand(bs, T, generator=g, device=DEV)
    return SimpleNamespace(logits=logits, info=info, cand=cand, q_ids=q_ids, q=q, u=u[:, :-1].contiguous(),
                           uf=u[:, -1].contiguous(), prefix=_prefix(g, bs), outs=_outputs(bs, T),
                           lens=torch.full((bs,), T, device=DEV, dtype=torch.int32))


def _run_sparse(c, s):
    from dspine_amd.sampling.sparse.accept import accept_sparse
    from dspine_amd.sampling.sparse.target import build_sparse_target

    t = build_sparse_target(s.logits, s.info, block_size=c["T"])
    accept_sparse(torch, candidates=s.cand, dense_p=t.dense_p, packed=t.packed, q_ids=s.q_ids, q_values=s.q,
                  verify_lens=s.lens, uniforms=s.u, uniform_final=s.uf, prefix_lens=s.prefix, outputs=s.outs)
    return {"packed": t.packed, "dense": t.dense_p, "outs": s.outs}


def _weights(c, g):
    H, R, C, V, bf = c["H"], c["R"], c["C"], c["V"], torch.bfloat16
    w = SimpleNamespace(
        codebook=(_randn(g, V, C) / math.sqrt(C)).to(bf), pg=_randn(g, R, C) / math.sqrt(C),
        pv=_randn(g, R, C) / math.sqrt(C), gb=_randn(g, R) * 0.1, w_last=_randn(g, H, R) / math.sqrt(R),
        norm_w=1.0 + 0.1 * _randn(g, H), lm=(_randn(g, V, H) / math.sqrt(H)).to(bf), res_emb=None, res_proj=None)
    if c.get("RR"):
        w.res_emb = (_randn(g, V, c["RR"]) / 4).to(bf)
        w.res_proj = _randn(g, R, c["RR"]) / math.sqrt(c["RR"])
    return w


def _draft_state(c, g):
    bs, T, K, bf = c["bs"], c["T"], c["K"], torch.bfloat16
    m, n = bs * T, bs * (T - 1)
    ids = torch.rand(n, c["V"], generator=g, device=DEV).topk(K, -1).indices.sort(-1).values
    return SimpleNamespace(
        w=_weights(c, g), raw=_randn(g, m, c["H"]).to(bf), rms=torch.rand(m, generator=g, device=DEV) + 0.5,
        query=_randn(g, m, c["R"]).to(bf), cand=ids.contiguous(),
        anchors=torch.randint(0, c["V"], (bs,), generator=g, device=DEV))


def _prepare_table(c, g):
    s = _draft_state(c, g)
    s.out = torch.zeros((s.cand.shape[0], c["K"], c["K"]), device=DEV)
    return s


def _run_table(c, s):
    from dspine_amd.kernels.dspine import serial_rs_table

    w = s.w
    return serial_rs_table(s.raw, s.rms, s.query, s.anchors, s.cand, w.codebook, w.pg, w.pv, w.gb, w.w_last, w.norm_w,
                           w.lm, 1e-6, c["T"], out=s.out, res_emb=w.res_emb, res_proj=w.res_proj)


def _prepare_factor(c, g):
    from dspine_amd.sampling.factorized.kernels import Workspace, build_cache

    s = _draft_state(c, g)
    n, w = s.cand.shape[0], s.w
    s.cache = build_cache(w.codebook, w.pg, w.pv, w.gb, w.w_last, w.norm_w, w.lm)
    s.ws = Workspace.allocate(n, c["K"], c["H"], c["R"], torch.device(DEV, torch.cuda.current_device()))
    s.out = torch.zeros((n, c["K"], c["K"]), device=DEV)
    s.base = torch.zeros((n, c["K"]), device=DEV, dtype=torch.float64)
    return s


def _run_factor(c, s):
    from dspine_amd.sampling.factorized.kernels import factor_table

    factor_table(s.raw, s.rms, s.query, s.anchors, s.cand, s.cache, 1e-6, c["T"], s.out, s.base, s.ws)
    return {"table": s.out, "base": s.base}


def _prepare_round(c, g):
    bs, T, K = c["bs"], c["T"], c["K"]
    n = bs * (T - 1)
    pick = lambda values: torch.tensor(values, device=DEV)[  # noqa: E731
        torch.randint(0, len(values), (bs,), generator=g, device=DEV)]
    cand = (torch.arange(K, device=DEV) * 1000
            + torch.randint(0, 1000, (n, K), generator=g, device=DEV)).contiguous()
    pool = bs + 8
    perm = torch.randperm(1 << 20, generator=g, device=DEV)
    return SimpleNamespace(
        seeds=torch.randint(0, 1 << 62, (bs,), generator=g, device=DEV),
        pos=torch.randint(0, 4096, (bs,), generator=g, device=DEV), table=_randn(g, n, K, K) * 2.0,
        inv_t=1.0 / pick([0.6, 1.0]), top_k=pick([5, K]).to(torch.int32), top_p=pick([0.9, 1.0]),
        min_p=pick([0.0, 0.02]), greedy=pick([0, 0, 0, 1]).to(torch.int32), cand=cand, gtok=cand[:, 0].clone(),
        tok=torch.zeros(n, device=DEV, dtype=torch.int64), q=torch.zeros((n, K), device=DEV),
        raw=torch.rand(bs, T - 1, generator=g, device=DEV),
        table_p=0.3 + 0.69 * torch.rand(T - 1, 64, generator=g, device=DEV),
        depth=torch.arange(T - 1, device=DEV), budget=bs * (1 + T // 3),
        cfg=SimpleNamespace(min_verify_len=1, survival_eps=0.0),
        accept=torch.randint(0, T, (bs,), generator=g, device=DEV).to(torch.int32),
        output=torch.zeros((bs, T), device=DEV, dtype=torch.int64), prefix=_prefix(g, bs),
        rows=torch.randperm(pool, generator=g, device=DEV)[:bs].contiguous(),
        table_t=torch.zeros((pool, 8192), device=DEV, dtype=torch.int32), loc=perm[:bs * T].to(torch.int64),
        seq=torch.zeros(pool, device=DEV, dtype=torch.int64),
        free=torch.zeros(bs * T, device=DEV, dtype=torch.int64), count=torch.zeros(1, device=DEV, dtype=torch.int32))


def _run_round(c, s):
    from dspine_amd.kernels.dspine import serial_sample_chain
    from dspine_amd.runtime.worker import commit_accept
    from dspine_amd.sampling.random import DRAFT, seeded_uniforms
    from dspine_amd.verification.sps import device_plan

    u = seeded_uniforms(s.seeds, s.pos, c["T"] - 1, DRAFT)
    serial_sample_chain(s.table, s.inv_t, s.top_k, s.top_p, s.min_p, s.greedy, u.view(-1), s.cand, s.gtok, s.tok, s.q,
                        c["T"])
    layout, index = device_plan(s.raw, s.table_p, s.depth, s.budget, s.cfg)
    commit_accept((s.accept, None, None, s.output, None), prefix_lens=s.prefix, req_pool_indices=s.rows,
                  req_to_token=s.table_t, out_cache_loc=s.loc, seq_lens=s.seq, free_slots=s.free, free_count=s.count)
    return {"u": u, "tok": s.tok, "q": s.q, "lens": layout.verify_lens, "qo": layout.qo_indptr_device, "index": index,
            "table": s.table_t, "seq": s.seq, "free": s.free, "count": s.count}


def prepare(case, seed):
    s = globals()["_prepare_" + case["kind"]](case, _gen(seed))
    s.case = case
    return s


def run(state):
    return globals()["_run_" + state.case["kind"]](state.case, state)


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------


def work(case):
    c, kind = case, case["kind"]
    bs, T = c["bs"], c["T"]
    if kind == "round":
        n, K = bs * (T - 1), c["K"]
        # the chain reads one K-lane row of each block row's table
        return {"bytes": n * K * (4 + 8 + 4) + n * 8 + bs * T * 40, "flops": n * K * 20}
    if kind in ("table", "factor"):
        K, H, R, C = c["K"], c["H"], c["R"], c["C"]
        n = bs * (T - 1)
        senders = bs * (1 + (T - 2) * K)  # a request's first block row has one sender
        head = n * K * H * 2
        if kind == "table":
            return {"bytes": head + n * H * 2 + 4 * (2 * R * C + H * R) + senders * C * 2 + n * K * K * 4,
                    "flops": 2.0 * (senders * C * 2 * R + senders * R * H + n * K * K * H)}
        # G and V rows of the senders, TG rows of the candidates, W and Gram, the head rows; x W, the
        # symmetric quadratic form, m . TG and the dot products with the head
        return {"bytes": head + n * H * 2 + 8 * (2 * senders * R + n * K * R + H * R + R * R) + n * K * K * 4,
                "flops": 2.0 * (n * H * R + senders * R * R / 2 + n * K * K * R + n * K * H)}
    rows = bs * T
    if kind == "verify" and c["ragged"]:
        rows = bs * (sum(_lengths(T)) - 1) / 2.0  # the mean of the drawn lengths
    e = 2 if c.get("dtype") == "bf16" else 4
    n = rows * c["V"]
    if kind == "greedy":
        return {"bytes": n * e, "flops": n}
    if kind == "verify":
        return {"bytes": n * e + bs * T * (16 * 12 + 40) + bs * c["hist"] * 4, "flops": 4 * n}
    if kind == "topk":
        return {"bytes": n * e + rows * c["k"] * 12, "flops": n}
    if kind == "filter":
        return {"bytes": n * 8, "flops": 2 * n}
    return {"bytes": n * (e + 4), "flops": 4 * n}  # probs, sparse: the logits read, P written


def tolerance(case):
    """Whole numbers: a sampled token turns on a comparison of float32 sums, so of a batch's outputs a
    request may differ where two sums meet; everything else whole is the same."""
    kind = case["kind"]
    if kind in ("greedy", "topk"):
        return "exact"
    if kind == "verify":
        return {"rel": 0.0, "differ": 0.01}
    if kind in ("probs", "filter"):
        # float32 softmax over the vocabulary, where 1.5e-7 is seen against 64 bits; the value at a
        # nucleus' edge may fall on either side of it, and a batch with such rows is seen 1.7e-5 off
        return {"rel": 7e-5, "max": 0.2}
    if kind == "sparse":
        return {"rel": 2e-6, "max": 4e-5, "differ": 0.01}  # 3.6e-7 is seen
    if kind == "table":
        return {"rel": 2.5e-6, "max": 5e-5}  # 5.5e-7 is seen
    if kind == "factor":
        return {"rel": 1e-7, "max": 2e-6}  # float64 sums, rounded to float32 once: 2.5e-8 is seen
    return {"rel": 1e-6, "max": 1e-5, "differ": 0.01}


# ---------------------------------------------------------------------------------------------
# the same in 64 bits, with plain torch
# ---------------------------------------------------------------------------------------------


def _filter64(p, info, c, b):
    """One request's rows filtered (float64) and renormalised: entries in descending order, lower ids
    first among equals."""
    k, top_p, min_p = int(info.top_ks[b]), float(info.top_ps[b]), float(info.min_ps[b])
    v, at = torch.sort(p, dim=-1, descending=True, stable=True)
    rank = torch.arange(v.shape[1], device=v.device)[None, :]
    ahead = v.cumsum(-1) - v
    if c["backend"] == "pytorch":
        keep = (rank < k) & (ahead <= top_p)
        if info.need_min_p_sampling:
            keep &= v >= v[:, :1] * min_p
    elif info.need_min_p_sampling:
        w = torch.where(rank < k, v, 0.0)
        w = w / w.sum(-1, keepdim=True)
        keep = (rank < k) & (w.cumsum(-1) - w <= top_p) & (v >= v[:, :1] * min_p)
    else:
        keep = (rank < k) & (ahead <= top_p)
    w = torch.where(keep, v, 0.0)
    return torch.zeros_like(p).scatter_(1, at, w / w.sum(-1, keepdim=True))


def _exact_probs(c, s):
    T, info = c["T"], s.info
    out = torch.empty((c["bs"], T, c["V"]), device=DEV, dtype=torch.float64)
    filtered = info.need_top_k_sampling or info.need_top_p_sampling or info.need_min_p_sampling
    for b in range(c["bs"]):
        x = s.logits[b * T:(b + 1) * T]
        p = torch.softmax(x.double() / info.temperatures.view(-1)[b].double(), -1)
        if filtered:
            p = _filter64(p, info, c, b)
        if info.is_any_greedy and int(info.top_ks[b]) <= 1:
            p = torch.zeros_like(p).scatter_(1, x.float().argmax(-1, keepdim=True), 1.0)
        out[b] = p
    return out


def _exact_filter(c, s):
    T = c["T"]
    info = s.info
    out = torch.empty((c["bs"], T, c["V"]), device=DEV, dtype=torch.float64)
    for b in range(c["bs"]):
        out[b] = _filter64(s.p[b * T:(b + 1) * T].double(), info, c, b)
    return out


def _exact_topk(c, s):
    return (torch.topk(s.logits.double(), c["k"], dim=-1).values, None)


def _exact_sparse(c, s):
    bs, T, V, cap = c["bs"], c["T"], c["V"], 32
    dense = torch.empty((bs * T, V), device=DEV, dtype=torch.float64)
    vals = torch.zeros((bs * T, cap), device=DEV, dtype=torch.float64)
    for b in range(bs):
        r = slice(b * T, (b + 1) * T)
        p = torch.softmax(s.logits[r].double() / s.info.temperatures.view(-1)[b].double(), -1)
        v, at = torch.sort(p, dim=-1, descending=True, stable=True)
        v, at = v[:, :cap + 1], at[:, :cap + 1]
        cut = v[:, int(s.info.top_ks[b]) - 1:int(s.info.top_ks[b])]
        higher = (v[:, None, :] * (v[:, None, :] > v[:, :, None])).sum(-1)
        top_p = float(s.info.top_ps[b])
        keep = (v >= cut) & ((higher < top_p) | (top_p >= 1))
        kept = torch.where(keep, v, 0.0)
        kept = kept / kept.sum(-1, keepdim=True)
        order = torch.where(keep, at, V + 1).sort(-1).indices
        vals[r] = torch.where(keep, kept, 0.0).gather(1, order)[:, :cap]
        over = keep.sum(-1) > cap
        full = torch.where(p >= cut, p, 0.0)
        dense[r] = torch.where(over[:, None], full / full.sum(-1, keepdim=True), p)
    return {"packed": (None, vals, None, None), "dense": dense, "outs": (None,) * 5}


def _table64(c, s):
    """(table, base) from the formula itself, block row by block row."""
    w, T, K, R = s.w, c["T"], c["K"], c["R"]
    n = s.cand.shape[0]
    row = torch.arange(n, device=DEV)
    state = row // (T - 1) * T + 1 + row % (T - 1)
    prev = torch.cat((s.cand[:1], s.cand[:-1]))
    sender = torch.where((row % (T - 1) == 0)[:, None], s.anchors[row // (T - 1)][:, None].expand(n, K), prev)
    x, q = s.raw[state].double(), s.query[state].double()
    pg, pv, wl, nw = w.pg.double(), w.pv.double(), w.w_last.double(), w.norm_w.double()
    table = torch.empty((n, K, K), device=DEV, dtype=torch.float64)
    base = torch.empty((n, K), device=DEV, dtype=torch.float64)
    for a in range(0, n, 64):
        z = slice(a, min(n, a + 64))
        m = z.stop - a
        e = w.codebook[sender[z]].double().view(m * K, -1) * math.sqrt(c["C"])
        gate = torch.sigmoid(q[z].repeat_interleave(K, 0) + e @ pg.t() + w.gb.double())
        value = e @ pv.t()
        if w.res_emb is not None:
            value = value + w.res_emb[sender[z]].double().view(m * K, -1) @ w.res_proj.double().t()
        y = x[z].repeat_interleave(K, 0) + s.rms[state[z]].double().repeat_interleave(K)[:, None] * (
            (gate * value) @ wl.t())
        y = y / (y.square().mean(-1, keepdim=True) + 1e-6).sqrt() * nw
        head = w.lm[s.cand[z]].double()  # [m, K, H]
        for i in range(m):
            table[a + i] = y[i * K:(i + 1) * K] @ head[i].t()
            base[a + i] = head[i] @ (x[a + i] * nw)
    return table, base


def _exact_table(c, s):
    return _table64(c, s)[0]


def _exact_factor(c, s):
    table, base = _table64(c, s)
    return {"table": table, "base": base}


def _exact_round(c, s):
    """The chain's q: every request walked in step, one block row at a time."""
    from dspine_amd.sampling.random import DRAFT, seeded_uniforms

    bs, steps, K = c["bs"], c["T"] - 1, c["K"]
    u = seeded_uniforms(s.seeds, s.pos, steps, DRAFT).double()  # (an input of the chain, checked as whole bits)
    table, cand = s.table.double().view(bs, steps, K, K), s.cand.view(bs, steps, K)
    q = torch.empty((bs, steps, K), device=DEV, dtype=torch.float64)
    lane = torch.zeros(bs, device=DEV, dtype=torch.int64)
    col = lambda x: x.double()[:, None]  # noqa: E731
    for i in range(steps):
        p = torch.softmax(table[torch.arange(bs, device=DEV), i, lane] * col(s.inv_t), -1)
        v, at = torch.sort(p, dim=-1, descending=True, stable=True)
        keep = ((torch.arange(K, device=DEV)[None] < col(s.top_k)) & (v.cumsum(-1) - v <= col(s.top_p))
                & (v >= v[:, :1] * col(s.min_p)))
        w = torch.zeros_like(p).scatter_(1, at, torch.where(keep, v, 0.0))
        q[:, i] = w / w.sum(-1, keepdim=True)
        cdf = q[:, i].cumsum(-1)
        last = torch.where(w > 0, torch.arange(K, device=DEV)[None], 0).amax(-1)
        lane = torch.minimum((cdf <= u[:, i:i + 1] * cdf[:, -1:]).sum(-1), last)
    greedy = s.greedy.bool()[:, None, None]
    q = torch.where(greedy, (cand == s.gtok.view(bs, steps, 1)).double(), q)
    return {"u": None, "tok": None, "q": q.view(bs * steps, K), "lens": None, "qo": None, "index": None, "table": None,
            "seq": None, "free": None, "count": None}


def exact(case, seed):
    f = globals().get("_exact_" + case["kind"])
    return None if f is None else f(case, prepare(case, seed))
