"""Parity of the HIP path (through the C ABI) with the CPU oracle on identical inputs.

Integer outputs must match bit-exactly.  A request may differ only when the oracle itself
reports a decision margin below MARGIN (tests/parity.py: an accept test u*q vs p or a bonus CDF
boundary within the measured probability error); every comparison records how many requests
were near such a margin and how many differed, and the run prints the table at its end.
The benchmark workloads (top-k rows, rejection, serving and ragged rounds) are compared in
full: every row or request.
"""

import numpy as np
import pytest
import torch

import parity
from dspine_amd import workloads as W
from parity import MARGIN

pytestmark = pytest.mark.gpu


def _oracle():
    import oracle.verify_oracle as O

    return O


def compare_outputs(gpu, ref, requests, tag):
    """gpu/ref: dicts of numpy arrays (accept, bonus, output, new_seq, [kv_slots]); returns the
    list of near-margin requests that differ (asserts every other request is identical)."""
    return parity.compare_requests(gpu, ref, requests, tag)


def _padded(x, device, width):
    """x [rows, V] on the device as a view of a [rows, width] buffer (row stride `width`)."""
    buf = torch.full((x.shape[0], width), float("nan"), dtype=x.dtype, device=device)
    buf[:, : x.shape[1]] = x.to(device)
    return buf[:, : x.shape[1]]


def run_gpu_verify(batch, device, backend="pytorch", row_stride=None):
    from dspine_amd.verify import History, verify_step

    d = W.to_device(batch, device)
    if row_stride is not None:
        d["logits"] = _padded(batch["logits"], device, row_stride)
        assert d["logits"].stride(0) == row_stride
    hist = None
    if "hist_ids" in d:
        hist = History(d["hist_ids"], d["presence"], d["repetition"])
    outs, kv = verify_step(
        logits=d["logits"], sampling_info=d["info"], candidates=d["candidates"], q_ids=d["q_ids"],
        q_values=d["q_values"], uniforms=d["uniforms"], uniform_final=d["uniform_final"],
        prefix_lens=d["prefix_lens"], verify_lens=d.get("verify_lens"),
        row_offsets=d.get("row_offsets"), history=hist, page_table=d.get("page_table"),
        sampling_backend=backend)
    torch.cuda.synchronize()
    names = ("accept", "commit", "bonus", "output", "new_seq")
    res = {n: t.cpu().numpy() for n, t in zip(names, outs)}
    res["kv_slots"] = kv.cpu().numpy() if kv is not None else None
    return res


def run_oracle(batch, requests, backend="pytorch", exact_softmax=True):
    O = _oracle()
    bs, T = batch["candidates"].shape
    lens = batch.get("verify_lens")
    lens = np.full(bs, T) if lens is None else lens.numpy()
    return O.verify_step(
        batch["logits"], batch["info"], candidates=batch["candidates"].numpy(),
        q_ids=batch["q_ids"].numpy(), q_values=batch["q_values"].numpy(), verify_lens=lens,
        uniforms=batch["uniforms"].numpy(), uniform_final=batch["uniform_final"].numpy(),
        prefix_lens=batch["prefix_lens"].numpy(), hist_ids=batch.get("hist_ids"),
        presence=batch.get("presence"), repetition=batch.get("repetition"),
        page_table=batch.get("page_table"),
        row_offsets=None if batch.get("row_offsets") is None else batch["row_offsets"].numpy(),
        sampling_backend=backend, requests=requests, exact_softmax=exact_softmax)


# ------------------------------------------------------------------------------------------
# uniforms
# ------------------------------------------------------------------------------------------
@pytest.mark.parametrize("stream", [0, 1, 2, 3])
def test_uniforms_bitwise(device, stream):
    from dspine_amd.sampling.random import seeded_uniforms

    O = _oracle()
    seeds = torch.tensor([0, -1, -(2**63), 2**63 - 1, 2**40 + 7, 12345])
    positions = torch.tensor([0, 19, 214, 8192, 131071, 7], dtype=torch.int32)
    got = seeded_uniforms(seeds.to(device), positions.to(device), 15, stream).cpu().numpy()
    ref = O.seeded_uniforms(seeds.numpy(), positions.numpy(), 15, stream)
    assert np.array_equal(got, ref)
    got64 = seeded_uniforms(seeds.to(device), positions.long().to(device), 15, stream).cpu().numpy()
    assert np.array_equal(got64, ref)


# ------------------------------------------------------------------------------------------
# top-k
# ------------------------------------------------------------------------------------------
def _topk_check(x_cpu, k, device):
    from dspine_amd.kernels.dspine import topk, topk_ids

    O = _oracle()
    vals, ids = topk(x_cpu.to(device), k)
    rv, ri = O.topk(x_cpu.float(), k)
    assert torch.equal(ids.cpu(), ri), "ids differ from the stable (value desc, id asc) order"
    assert torch.equal(vals.cpu(), rv)
    srt = topk_ids(x_cpu.to(device), k).cpu()
    assert torch.equal(srt, ri.sort(-1).values)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [16, 128])
def test_topk_small_ties(device, dtype, k):
    # tests/test_topk_compat.py:70-84: 257-wide rows of i % 7 with a -inf tail
    scores = torch.arange(257).remainder(7).to(dtype).repeat(2, 1)
    scores[1, 254:] = -torch.inf
    _topk_check(scores, k, device)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [1, 20, 64])
def test_topk_serving_rows(device, dtype, k):
    x = W.topk_rows(rows=96, seed=11, dtype=dtype)["logits"]
    _topk_check(x, k, device)


@pytest.mark.parametrize("k", [1, 20, 64, 256])
def test_topk_degenerate_rows(device, k):
    V = 70001
    rows = torch.zeros(6, V)
    rows[1] = torch.arange(V).float()          # ascending: every block raises the threshold
    rows[2] = -torch.arange(V).float()         # descending
    rows[3, :] = -torch.inf
    rows[3, 5::1000] = 1.0                     # only 71 finite values
    rows[4, 1::2] = -0.0                       # +0 / -0 alternating, a zero bound that takes -0 in
    rows[4, ::3] = -1.0
    g = torch.Generator().manual_seed(7)
    rows[5] = -torch.rand(V, generator=g) * 4.0 - 0.5  # every value negative: a negative bound
    for dtype in (torch.float32, torch.bfloat16):
        _topk_check(rows.to(dtype), k, device)


@pytest.mark.parametrize("dtype,chunks,k,spread", [
    (torch.bfloat16, 4, 33, None), (torch.bfloat16, 4, 34, None),  # bf16 lists counted, and selected by radix
    (torch.float32, 41, 49, None), (torch.float32, 41, 50, None),  # 2009 slots in registers, 2050 not
    (torch.float32, 64, 5, None), (torch.float32, 65, 5, None),    # a chunk count a lane, and over
    (torch.float32, 9, 64, (63, 7)), (torch.float32, 9, 64, (63, 8)),  # 512 candidates left, and 513
    (torch.float32, 1, 64, None), (torch.float32, 8, 256, None), (torch.float32, 9, 256, None),
])
def test_topk_merge_edges(device, dtype, chunks, k, spread):
    """Both sides of every line between the merge's counting and its radix selection; a row whose last
    chunk holds one value, one of ties.  ``spread`` (a, b): a large values in every chunk but the last, b
    there, so that each list's smallest is a small one and the large ones all stay."""
    n = 20480 if dtype == torch.bfloat16 else 12288
    V = (chunks - 1) * n + (1 if chunks > 1 and spread is None else n)
    g = torch.Generator().manual_seed(chunks * k)
    x = torch.rand(3, V, generator=g)
    if spread is not None:
        for c in range(chunks):
            at = c * n + torch.randperm(n, generator=g)[:spread[0] if c < chunks - 1 else spread[1]]
            x[:, at] = 10.0 + torch.rand(3, at.numel(), generator=g)
    x[2] = (x[2] * 50).round()
    _topk_check(x.to(dtype), k, device)


# ------------------------------------------------------------------------------------------
# greedy verify (config: 1 x 17 x 151936 fp32)
# ------------------------------------------------------------------------------------------
def test_greedy_round(device):
    from dspine_amd.verification.caps import accept_greedy

    O = _oracle()
    batch = W.greedy_round()
    top1 = O.argmax_rows(batch["logits"])
    ref = O.greedy_accept(top1, batch["candidates"].numpy(), [17], batch["prefix_lens"].numpy())
    outs = accept_greedy(candidates=batch["candidates"].to(device),
                         next_token_logits=batch["logits"].to(device),
                         prefix_lens=batch["prefix_lens"].to(device), cap=17)
    got = [t.cpu().numpy() for t in outs]
    assert int(got[0][0]) == batch["mismatch"] == int(ref[0][0])
    for g, r in zip(got, ref):
        assert np.array_equal(g, r)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_greedy_ties_and_caps(device, dtype):
    from dspine_amd.verification.caps import accept_greedy

    O = _oracle()
    g = torch.Generator().manual_seed(5)
    bs, T, V = 9, 16, 997
    logits = torch.randint(-3, 3, (bs * T, V), generator=g).to(dtype)  # heavy ties
    logits[: 3 * T] = 0  # all-tie rows: first id wins
    top1 = O.argmax_rows(logits)
    cand = torch.zeros(bs, T, dtype=torch.int64)
    cand[:, 1:] = torch.as_tensor(top1).view(bs, T)[:, : T - 1]
    cand[4, 6] = (cand[4, 6] + 1) % V
    lens = (torch.arange(bs, dtype=torch.int32) % T) + 1
    prefix = torch.arange(bs, dtype=torch.int32) + 100
    for cap, vl in ((T, None), (7, None), (None, lens)):
        ref = O.greedy_accept(top1, cand.numpy(), (lens.numpy() if vl is not None else [cap] * bs),
                              prefix.numpy())
        outs = accept_greedy(candidates=cand.to(device), next_token_logits=logits.to(device),
                             prefix_lens=prefix.to(device), cap=cap,
                             verify_lens=None if vl is None else vl.to(device))
        for got, r in zip(outs, ref):
            assert np.array_equal(got.cpu().numpy(), r), (cap, vl)


@pytest.mark.parametrize("bs,T,V,dtype", [(2, 1, 64, torch.float32), (3, 17, 1 << 20, torch.bfloat16),
                                          (2, 1100, 40, torch.float32)])
def test_greedy_edges(device, bs, T, V, dtype):
    """A block without drafts, rows of more than 32 chunks, and more rows than the accept kernel
    keeps argmaxes of; with the optional argmaxes and without."""
    from dspine_amd.verification.caps import accept_greedy

    O = _oracle()
    g = torch.Generator().manual_seed(T)
    logits = torch.randint(-60, 60, (bs * T, V), generator=g).to(dtype)
    logits[0] = -float("inf")  # nothing above -inf: the first id
    top1 = O.argmax_rows(logits)
    cand = torch.zeros(bs, T, dtype=torch.int64)
    cand[:, 1:] = torch.as_tensor(top1).view(bs, T)[:, : T - 1]
    if T > 2:
        cand[1, T - 1] = (cand[1, T - 1] + 1) % V
    prefix = torch.arange(bs, dtype=torch.int32)
    ref = O.greedy_accept(top1, cand.numpy(), [T] * bs, prefix.numpy())
    for top in (None, torch.full((bs, T), -1, dtype=torch.int64, device=device)):
        outs = accept_greedy(candidates=cand.to(device), next_token_logits=logits.to(device),
                             prefix_lens=prefix.to(device), cap=T, top1=top)
        for got, r in zip(outs, ref):
            assert np.array_equal(got.cpu().numpy(), r)
        assert top is None or np.array_equal(top.cpu().numpy().reshape(-1), np.asarray(top1).reshape(-1))


@pytest.mark.parametrize("T,V", [(64, 64), (65, 64), (32, 20481), (33, 20481), (16, 61441), (8, 102401), (9, 102401),
                                 (4, 163841), (5, 163841), (1, 327681), (2, 327681)])
def test_greedy_lane_groups(device, T, V):
    """Every width of the accept kernel's lane groups (1, 2, 4, 8, 16 lanes and the wave a row) with the
    rows that just fit one wave and those that just do not: maxima tied over all chunks, or one in a
    chunk of its own, caps and verify lengths, with the argmaxes and without."""
    from dspine_amd.verification.caps import accept_greedy

    O = _oracle()
    g = torch.Generator().manual_seed(T)
    bs = 5
    logits = torch.randint(-60, 60, (bs * T, V), generator=g).to(torch.bfloat16)
    logits[torch.arange(1, bs * T, 2), torch.randint(0, V, (bs * T // 2,), generator=g)] = 64.0
    top1 = O.argmax_rows(logits)
    cand = torch.zeros(bs, T, dtype=torch.int64)
    cand[:, 1:] = torch.as_tensor(top1).view(bs, T)[:, : T - 1]
    for b in range(1, bs):  # the first request's drafts are all accepted
        if T > 1:
            cand[b, int(torch.randint(1, T, (1,), generator=g))] += 1
    prefix = torch.arange(bs, dtype=torch.int32)
    lens = torch.randint(1, T + 1, (bs,), generator=g).to(torch.int32)
    x, c, p = logits.to(device), cand.to(device), prefix.to(device)
    for vl in (None, lens):
        ref = O.greedy_accept(top1, cand.numpy(), [T] * bs if vl is None else vl.tolist(), prefix.numpy())
        for top in (None, torch.full((bs, T), -1, dtype=torch.int64, device=device)):
            outs = accept_greedy(candidates=c, next_token_logits=x, prefix_lens=p, top1=top,
                                 **({"cap": T} if vl is None else {"verify_lens": vl.to(device)}))
            for got, r in zip(outs, ref):
                assert np.array_equal(got.cpu().numpy(), r)
            assert top is None or np.array_equal(top.cpu().numpy().reshape(-1), np.asarray(top1).reshape(-1))


# ------------------------------------------------------------------------------------------
# fused sampled verify
# ------------------------------------------------------------------------------------------
def _small_batch(seed, bs=24, T=8, V=997, K=8, dtype=torch.float32, mixed=True, penalties=False,
                 ragged=False):
    g = torch.Generator().manual_seed(seed)
    rows_per = torch.full((bs,), T, dtype=torch.int64)
    if ragged:
        rows_per = torch.randint(1, T + 1, (bs,), generator=g)
    offsets = torch.cat((torch.zeros(1, dtype=torch.int64), rows_per.cumsum(0)))[:-1]
    nrows = int(rows_per.sum()) if ragged else bs * T
    logits = (torch.randn(nrows, V, generator=g) * 2.0).to(dtype)
    if mixed:
        temps = torch.tensor([0.0, 0.6, 1.0, 1.3])[torch.randint(0, 4, (bs,), generator=g)]
        ks = torch.tensor([0, 1, 5, 20, 64, 100])[torch.randint(0, 6, (bs,), generator=g)]
        ps = torch.tensor([1.0, 0.95, 0.8, 0.5])[torch.randint(0, 4, (bs,), generator=g)]
    else:
        temps = torch.full((bs,), 0.8)
        ks = torch.full((bs,), 20)
        ps = torch.full((bs,), 0.9)
    info = W.sampling_info(temps, ks, ps)
    q_ids = torch.stack([torch.randperm(V, generator=g)[:K] for _ in range(bs * (T - 1))]).view(bs, T - 1, K)
    # make the most likely target token a q lane often, so acceptances happen
    base = logits.float()
    for b in range(bs):
        r0 = int(offsets[b]) if ragged else b * T
        for s in range(T - 1):
            r = r0 + min(s, int(rows_per[b]) - 1)
            q_ids[b, s, 0] = int(base[r].argmax())
    q_ids, _ = q_ids.sort(-1)
    q = torch.softmax(torch.randn(bs, T - 1, K, generator=g) * 2, -1)
    lanes = torch.multinomial(q.view(-1, K), 1, generator=g).view(bs, T - 1)
    drafts = q_ids.gather(2, lanes[..., None]).squeeze(-1)
    cand = torch.cat((torch.zeros(bs, 1, dtype=torch.int64), drafts), 1)
    u = W.philox_uniforms(seed, bs, T)
    batch = dict(logits=logits, info=info, candidates=cand, q_ids=q_ids, q_values=q.float(),
                 uniforms=u[:, : T - 1].contiguous(), uniform_final=u[:, T - 1].contiguous(),
                 prefix_lens=torch.randint(0, 50, (bs,), generator=g, dtype=torch.int64).to(torch.int32),
                 page_table=torch.randperm(bs * 80, generator=g).view(bs, 80).to(torch.int32))
    if ragged:
        batch["verify_lens"] = rows_per.to(torch.int32)
        batch["row_offsets"] = offsets
    else:
        batch["verify_lens"] = torch.randint(1, T + 1, (bs,), generator=g, dtype=torch.int64).to(torch.int32)
    if penalties:
        batch["hist_ids"] = torch.randint(-1, V, (bs, 40), generator=g, dtype=torch.int64).to(torch.int32)
        batch["presence"] = torch.rand(bs, generator=g)
        batch["repetition"] = 1.0 + torch.rand(bs, generator=g)
    return batch


@pytest.mark.parametrize("seed", [0, 1, 2])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("penalties", [False, True])
def test_verify_small_mixed(device, seed, dtype, penalties):
    batch = _small_batch(seed, dtype=dtype, penalties=penalties)
    bs = batch["candidates"].shape[0]
    gpu = run_gpu_verify(batch, device)
    ref = run_oracle(batch, list(range(bs)))
    near = compare_outputs(gpu, ref, range(bs), f"small seed={seed}")
    assert len(near) <= 1


@pytest.mark.parametrize("seed", [0, 1])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_verify_small_mixed_flashinfer(device, seed, dtype):
    """The mixed small batches under the flashinfer backend without min-p (greedy rows present:
    the joint support by rank, not the sparse joint route), with penalties and verify lengths."""
    batch = _small_batch(seed, dtype=dtype, penalties=True)
    bs = batch["candidates"].shape[0]
    gpu = run_gpu_verify(batch, device, backend="flashinfer")
    ref = run_oracle(batch, list(range(bs)), backend="flashinfer")
    near = compare_outputs(gpu, ref, range(bs), f"small flashinfer seed={seed}")
    assert len(near) <= 1


@pytest.mark.parametrize("mix", ["greedy", "lists", "unfiltered", "nucleus", "lists_and_greedy"])
def test_verify_launch_sets(device, mix):
    """Batches of one kind of request, which launch different kernel sets: greedy-only and
    support-list-only batches finish every request in the row merge (no k_final launch);
    unfiltered and nucleus batches leave their dense accepted rows to k_final."""
    batch = _small_batch(40 + len(mix), dtype=torch.bfloat16, penalties=True)
    bs = batch["candidates"].shape[0]
    half = bs // 2
    temps, ks, ps = {
        "greedy": ([0.0] * bs, [0] * bs, [1.0] * bs),
        "lists": ([0.8] * bs, [20] * bs, [0.9] * bs),
        "unfiltered": ([0.8] * bs, [0] * bs, [1.0] * bs),
        "nucleus": ([0.8] * bs, [0] * bs, [0.9] * bs),
        "lists_and_greedy": ([0.0] * half + [1.0] * (bs - half), [0] * half + [5] * (bs - half), [1.0] * bs),
    }[mix]
    batch["info"] = W.sampling_info(temps, ks, ps)
    gpu = run_gpu_verify(batch, device)
    ref = run_oracle(batch, list(range(bs)))
    assert len(compare_outputs(gpu, ref, range(bs), f"launch set {mix}")) <= 1


@pytest.mark.parametrize("seed", [5, 6])
def test_verify_page_table_edges(device, seed):
    """KV slots where the committed positions run past the page table's columns (-1 there, as
    the oracle's kv_slots), from prefix 0 and from the last column."""
    batch = _small_batch(seed, dtype=torch.bfloat16, penalties=True)
    bs, T = batch["candidates"].shape
    g = torch.Generator().manual_seed(100 + seed)
    cols = 24
    batch["page_table"] = torch.randperm(bs * cols, generator=g).view(bs, cols).to(torch.int32)
    prefix = torch.randint(cols - T, cols + 2, (bs,), generator=g, dtype=torch.int64)
    prefix[0] = 0
    prefix[1] = cols - 1
    batch["prefix_lens"] = prefix.to(torch.int32)
    batch["verify_lens"] = torch.full((bs,), T, dtype=torch.int32)
    gpu = run_gpu_verify(batch, device)
    ref = run_oracle(batch, list(range(bs)))
    assert (ref["kv_slots"] == -1).any() and (ref["kv_slots"] >= 0).any()
    near = compare_outputs(gpu, ref, range(bs), f"page edges seed={seed}")
    assert len(near) <= 1


@pytest.mark.parametrize("seed", [3, 4])
def test_verify_small_ragged(device, seed):
    batch = _small_batch(seed, dtype=torch.bfloat16, ragged=True, penalties=True)
    bs = batch["candidates"].shape[0]
    gpu = run_gpu_verify(batch, device)
    ref = run_oracle(batch, list(range(bs)))
    assert len(compare_outputs(gpu, ref, range(bs), f"ragged seed={seed}")) <= 1


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V,stride", [(997, 1000), (20483, 20488), (41000, 41000), (5, 8)])
def test_verify_row_layouts(device, dtype, V, stride):
    # 16-byte aligned rows whose vocab leaves a partial last vector, a vocab that ends a
    # chunk exactly plus 3, a vocab ending inside the second chunk, and a vocab shorter than
    # one vector (the byte-wise load path)
    mixed = dtype == torch.bfloat16
    batch = _small_batch(11, bs=12, T=5, V=V, K=4, dtype=dtype, mixed=mixed, penalties=True)
    bs = batch["candidates"].shape[0]
    gpu = run_gpu_verify(batch, device, row_stride=stride)
    ref = run_oracle(batch, list(range(bs)))
    assert len(compare_outputs(gpu, ref, range(bs), f"layout V={V} stride={stride}")) <= 1


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("offset,V,stride", [(1, 20483, 20483), (3, 12289, 12291), (2, 997, 999), (7, 41003, 41006)])
def test_rows_of_any_alignment(device, dtype, offset, V, stride):
    """Rows that start at any element (an odd vocabulary, a view into a larger buffer), P written to rows
    of an odd stride: the same bits as rows copied to 16-byte boundaries."""
    from dspine_amd.kernels.dspine import topk
    from dspine_amd.verification.caps import accept_greedy
    from dspine_amd.verify import target_probs

    g = torch.Generator().manual_seed(V)
    bs, T = 4, 3
    x = (torch.randn(bs * T, V, generator=g) * 2.5).to(dtype)
    buf = torch.full((bs * T * stride + 16,), float("nan"), dtype=dtype, device=device)
    odd = buf[offset:].as_strided((bs * T, V), (stride, 1))
    odd.copy_(x)
    pad = torch.zeros(bs * T, (V + 63) // 64 * 64, dtype=dtype, device=device)[:, :V]
    pad.copy_(x)
    for a, b in zip(topk(odd, 20), topk(pad, 20)):
        assert torch.equal(a, b)
    cand = torch.randint(0, V, (bs, T), generator=g).to(device)
    cand[:, 1:] = pad.float().argmax(-1).view(bs, T)[:, :-1]
    prefix = torch.arange(bs, dtype=torch.int32, device=device)
    for a, b in zip(accept_greedy(candidates=cand, next_token_logits=odd, prefix_lens=prefix),
                    accept_greedy(candidates=cand, next_token_logits=pad, prefix_lens=prefix)):
        assert torch.equal(a, b)
    info = W.info_to(W.sampling_info([1.0, 0.0, 0.7, 1.0], [0, 0, 20, 0], [0.95, 1.0, 0.9, 1.0]), device)
    out = torch.full((bs * T, (V + 63) // 64 * 64), -1.0, device=device)
    ref = target_probs(pad, info, bs=bs, T=T, out=out[:, :V])
    raw = torch.full((bs * T * stride + 16,), -1.0, device=device)
    got = target_probs(odd, info, bs=bs, T=T, out=raw[offset:].as_strided((bs * T, V), (stride, 1)))
    assert torch.equal(got, ref)
    assert bool((out[:, V:] == -1).all()) and int((raw == -1).sum()) == raw.numel() - bs * T * V


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_verify_long_history(device, dtype):
    # a history of 6000 tokens over 20483 ids: more vectors hold a penalised value than a
    # wave's LDS slots, so every lane penalises its own elements in place
    batch = _small_batch(13, bs=8, T=5, V=20483, K=4, dtype=dtype, mixed=True, penalties=True)
    g = torch.Generator().manual_seed(14)
    bs = batch["candidates"].shape[0]
    batch["hist_ids"] = torch.randint(-1, 20483, (bs, 6000), generator=g, dtype=torch.int64).to(torch.int32)
    gpu = run_gpu_verify(batch, device)
    ref = run_oracle(batch, list(range(bs)))
    assert len(compare_outputs(gpu, ref, range(bs), f"long history {dtype}")) <= 1


@pytest.mark.parametrize("V,stride", [(997, 1000), (70001, 70008)])
def test_greedy_and_topk_row_layouts(device, V, stride):
    from dspine_amd.kernels.dspine import topk
    from dspine_amd.verification.caps import accept_greedy

    O = _oracle()
    g = torch.Generator().manual_seed(9)
    bs, T = 4, 6
    x = torch.randn(bs * T, V, generator=g).to(torch.bfloat16)
    xd = _padded(x, device, stride)
    vals, ids = topk(xd, 20)
    rv, ri = O.topk(x.float(), 20)
    assert torch.equal(ids.cpu(), ri) and torch.equal(vals.cpu(), rv)
    top1 = O.argmax_rows(x)
    cand = torch.zeros(bs, T, dtype=torch.int64)
    cand[:, 1:] = torch.as_tensor(top1).view(bs, T)[:, : T - 1]
    cand[1, 3] = (cand[1, 3] + 1) % V
    prefix = torch.arange(bs, dtype=torch.int32)
    ref = O.greedy_accept(top1, cand.numpy(), [T] * bs, prefix.numpy())
    outs = accept_greedy(candidates=cand.to(device), next_token_logits=xd, prefix_lens=prefix.to(device), cap=T)
    for got, r in zip(outs, ref):
        assert np.array_equal(got.cpu().numpy(), r)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("case", ["flat", "constant", "peaked", "wide_tail"])
def test_verify_nucleus_paths(device, case, dtype):
    # nucleus rows (top-k off, top-p < 1) that exercise each way the cut is found: "flat"
    # (temperature 40: the counted windows cannot reach the row floor -> full histogram),
    # "constant" (151936 equal values: more ties than a 16-bit counter holds), "peaked" (one
    # dominant token: every counted value is kept and the cut is the first value below the
    # windows), "wide_tail" (heavy-tailed logits, T = 1)
    V = 151936
    bs, T = 4, 3
    batch = _small_batch(21, bs=bs, T=T, V=V, K=4, dtype=dtype, mixed=False, penalties=True)
    g = torch.Generator().manual_seed(22)
    rows = bs * T
    if case == "flat":
        logits = torch.randn(rows, V, generator=g) * 2.0
        temps = [40.0] * bs
    elif case == "constant":
        logits = torch.zeros(rows, V)
        logits[:, ::7919] = 0.5
        temps = [1.0] * bs
    elif case == "peaked":
        logits = torch.randn(rows, V, generator=g)
        logits[torch.arange(rows), torch.randint(0, V, (rows,), generator=g)] = 30.0
        temps = [1.0] * bs
    else:
        logits = 2.0 * torch.distributions.StudentT(3.0).sample((rows, V))
        temps = [1.0] * bs
    batch["logits"] = logits.to(dtype)
    batch["info"] = W.sampling_info(temps, [0] * bs, [0.9, 0.5, 0.95, 0.99][:bs])
    base = batch["logits"].float()
    for b in range(bs):  # a likely token as a q lane, so some drafts are accepted
        for s_ in range(T - 1):
            batch["q_ids"][b, s_, 0] = int(base[b * T + s_].argmax())
    batch["q_ids"], _ = batch["q_ids"].sort(-1)
    gpu = run_gpu_verify(batch, device)
    # pinned against the exact softmax: CPU torch's float32 normaliser is off by ~1e-4 on the
    # flat and constant rows, which moves their cut by a few of the ~10^5 ties
    ref = run_oracle(batch, list(range(bs)), exact_softmax=True)
    assert len(compare_outputs(gpu, ref, range(bs), f"nucleus {case}")) <= 1


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_verify_full_histogram_rows_accepted(device, dtype):
    """Flat nucleus rows (temperature 40: the bf16 rows need the full histogram, the float32
    rows the radix descent) whose drafts are accepted: every q lane is 1e-7, below the ~7e-6
    of a kept token, so the chain runs through several such rows and the bonus of a later one
    is drawn after the accepted ones (the resumed scan of the request's rows)."""
    V = 151936
    bs, T = 4, 5
    batch = _small_batch(23, bs=bs, T=T, V=V, K=4, dtype=dtype, mixed=False, penalties=True)
    g = torch.Generator().manual_seed(24)
    batch["logits"] = (torch.randn(bs * T, V, generator=g) * 2.0).to(dtype)
    batch["info"] = W.sampling_info([40.0] * bs, [0] * bs, [0.9, 0.5, 0.95, 0.8])
    batch["q_values"] = torch.full_like(batch["q_values"], 1e-7)
    batch["verify_lens"] = torch.tensor([5, 3, 4, 5], dtype=torch.int32)
    gpu = run_gpu_verify(batch, device)
    ref = run_oracle(batch, list(range(bs)), exact_softmax=True)
    assert (ref["accept"] >= 2).any(), ref["accept"]
    assert len(compare_outputs(gpu, ref, range(bs), f"full-histogram rows accepted {dtype}")) <= 1


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("case", ["windows", "flat"])
def test_verify_flashinfer_min_p_nucleus(device, case, dtype):
    # flashinfer's min-p branch (tests/ref_utils.py:79-108): renormalise over the top-k, top-p
    # on that mass, then min-p against the max -- on nucleus rows (top-k off or > 64, one
    # support-list row beside them), min-p both dominating and negligible; "flat" (temperature
    # 40) sends the bf16 rows to the full histogram
    V = 151936
    bs, T = 6, 3
    batch = _small_batch(31, bs=bs, T=T, V=V, K=4, dtype=dtype, mixed=False, penalties=True)
    g = torch.Generator().manual_seed(32)
    batch["logits"] = (torch.randn(bs * T, V, generator=g) * 2.0).to(dtype)
    temps = [40.0] * bs if case == "flat" else [1.0, 0.7, 1.0, 0.7, 1.0, 0.7]
    batch["info"] = W.sampling_info(temps, [0, 100, 1000, 20, 5000, 0], [0.9, 0.8, 0.95, 0.5, 0.9, 1.0],
                                    min_ps=[0.05, 1e-4, 0.1, 3e-4, 0.01, 1e-5])
    base = batch["logits"].float()
    for b in range(bs):  # a likely token as a q lane, so some drafts are accepted
        for s_ in range(T - 1):
            batch["q_ids"][b, s_, 0] = int(base[b * T + s_].argmax())
    batch["q_ids"], _ = batch["q_ids"].sort(-1)
    gpu = run_gpu_verify(batch, device, backend="flashinfer")
    ref = run_oracle(batch, list(range(bs)), backend="flashinfer", exact_softmax=True)
    assert len(compare_outputs(gpu, ref, range(bs), f"flashinfer min-p {case}")) <= 1


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_verify_large_vocab(device, dtype):
    """262144-wide rows (26 float32 / 13 bf16 chunks a row), ragged, mixed list / nucleus /
    greedy rows with penalties."""
    batch = _small_batch(41, bs=6, T=4, V=262144, K=8, dtype=dtype, ragged=True, penalties=True)
    bs = batch["candidates"].shape[0]
    gpu = run_gpu_verify(batch, device)
    ref = run_oracle(batch, list(range(bs)), exact_softmax=True)
    assert len(compare_outputs(gpu, ref, range(bs), f"large vocab {dtype}")) <= 1


def test_verify_unfiltered(device):
    batch = _small_batch(7, dtype=torch.bfloat16, mixed=False)
    batch["info"] = W.sampling_info([0.7] * 24, [0] * 24, [1.0] * 24)
    bs = 24
    gpu = run_gpu_verify(batch, device)
    ref = run_oracle(batch, list(range(bs)))
    assert len(compare_outputs(gpu, ref, range(bs), "unfiltered")) <= 1


def _full(batch, device, tag, backend="pytorch"):
    """Every request against the oracle with its exact softmax (the parity bound), then against
    its literal float32 softmax (recorded, tests/parity.py)."""
    bs = batch["candidates"].shape[0]
    gpu = run_gpu_verify(batch, device, backend=backend)
    ref = run_oracle(batch, list(range(bs)), backend=backend)
    compare_outputs(gpu, ref, range(bs), tag)
    literal = run_oracle(batch, list(range(bs)), backend=backend, exact_softmax=False)
    parity.compare_literal(gpu, literal, ref, range(bs), tag)
    return gpu, ref


def test_verify_serving_round_full(device):
    """The benchmark's serving workload (64 x 17 x 151936 bf16, penalties, mixed modes, KV
    slots): every request against the oracle."""
    _full(W.serving_round(), device, "serving 64x17x151936 bf16")


def test_verify_serving_round_full_flashinfer(device):
    """The serving workload under the flashinfer backend: its greedy requests keep the batch off
    the sparse joint route, so every sampled row takes the joint support by rank (top-k, then the
    top-p test on the mass ranked ahead); every request against the oracle."""
    _full(W.serving_round(), device, "serving 64x17x151936 bf16 flashinfer", backend="flashinfer")


def test_verify_serving_round_deep_accept(device):
    """The serving workload with a planted likely token per row (the bench's --accept deep):
    deep accepted prefixes, so the accepted row and the bonus draw lie far down the requests."""
    gpu, ref = _full(W.serving_round(peak=16.0), device, "serving deep-accept 64x17x151936 bf16")
    assert ref["accept"].mean() > 4.0, ref["accept"].mean()


@pytest.mark.parametrize("sigma", [0.5, 1.5])
def test_verify_rejection_round_full(device, sigma):
    """The rejection workload (32 x 17 x 151936 fp32, top-k 20, top-p 0.95): every request."""
    _full(W.rejection_round(sigma_draft=sigma), device, f"rejection 32x17x151936 fp32 sigma={sigma}")


def test_verify_ragged_round_full(device):
    """The ragged workload (32 requests x U{4..16} rows x 262144 bf16, Student-t): every request."""
    _full(W.ragged_round(), device, "ragged 32x(4..16)x262144 bf16")


def test_verify_rejection_and_ragged_flashinfer(device):
    """The rejection (top-k 20, top-p 0.95; 20 q lanes, so not the sparse joint route) and ragged
    (top-p 0.9 over the whole vocabulary) workloads under the flashinfer backend: every request."""
    _full(W.rejection_round(sigma_draft=0.5), device, "rejection 32x17x151936 fp32 sigma=0.5 flashinfer",
          backend="flashinfer")
    _full(W.ragged_round(), device, "ragged 32x(4..16)x262144 bf16 flashinfer", backend="flashinfer")


def test_topk_rows_full(device):
    """The top-k workload ([1088, 151936] bf16, planted peaks, ~1% duplicates): all rows for
    k in {1, 20, 64}, ids and values bit-exact in (value desc, id asc) order."""
    from dspine_amd.kernels.dspine import topk, topk_ids

    O = _oracle()
    x = W.topk_rows()["logits"]
    rv, ri = O.topk(x.float(), 64)  # the first k of one stable order are the top-k for every k
    xd = x.to(device)
    for k in (1, 20, 64):
        vals, ids = topk(xd, k)
        srt = topk_ids(xd, k)
        torch.cuda.synchronize()
        bad = (ids.cpu() != ri[:, :k]).any(-1) | (vals.cpu() != rv[:, :k]).any(-1)
        assert int(bad.sum()) == 0, (k, torch.nonzero(bad).view(-1)[:10].tolist())
        assert torch.equal(srt.cpu(), ri[:, :k].sort(-1).values)
        parity.record(f"topk [1088, 151936] bf16 k={k} (rows)", x.shape[0], 0, [])


def test_target_p_error_bounds_margin(device):
    """The dense target P of the HIP path against the float64 softmax (rounded once) and
    against CPU torch's float32 softmax on the serving workload's rows (all four modes): the
    largest relative error against the exact softmax on entries >= 1e-6 of the row max stays
    below half of MARGIN, so a decision further than MARGIN from its boundary (as the
    oracle's exact softmax places it) cannot come out differently."""
    from dspine_amd.runtime.worker import build_dspine_target_probs

    O = _oracle()
    batch = W.serving_round()
    T = batch["candidates"].shape[1]
    reqs = 16
    x = batch["logits"][: reqs * T]
    info = batch["info"]
    sub = W.sampling_info(info.temperatures.view(-1)[:reqs].clone(), info.top_ks[:reqs].clone(),
                          info.top_ps[:reqs].clone())
    sub.temperatures = info.temperatures[:reqs].clone()
    gp = build_dspine_target_probs(next_token_logits=x.to(device), sampling_info=W.info_to(sub, device),
                                   block_size=T, bs=reqs, sampling_backend="pytorch")
    got = gp.reshape(reqs * T, -1).double().cpu()
    errs = {}
    for exact in (True, False):
        ref = O.build_target_probs(x, sub, T, reqs, "pytorch", exact_softmax=exact).reshape(reqs * T, -1).double()
        both = (ref > 0) & (got > 0) & (ref >= ref.amax(-1, keepdim=True) * 1e-6)
        rel = ((got - ref).abs() / ref.clamp_min(1e-300))[both]
        # rows whose kept support differs (a top-p cut within the error of its boundary)
        cut_rows = int(((got > 0) != (ref > 0)).any(-1).sum())
        errs[exact] = (float(rel.max()), cut_rows)
    print(f"[p-error] vs float64 softmax {errs[True][0]:.3g} ({errs[True][1]} rows with another cut), "
          f"vs CPU torch float32 {errs[False][0]:.3g} ({errs[False][1]} rows with another cut)", flush=True)
    # the parity tests compare against the exact softmax: the HIP path's P must sit well inside
    # MARGIN of it, with the same cut on every row
    assert errs[True][0] < MARGIN / 2, errs
    assert errs[True][1] == 0, errs
    # CPU torch's float32 normaliser is itself ~1e-5 off on these 151936-wide rows and cuts
    # some top-p rows inside a bf16 tie group elsewhere (the reason the oracle's exact softmax
    # is the parity reference); bounded here only to keep the figure on record
    assert errs[False][0] < parity.LITERAL_MARGIN, errs
