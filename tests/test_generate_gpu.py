"""Sampling kernels, the Python entry points and the scheduler on the GPU."""
import math
import random

import numpy as np
import pytest
import torch

import helpers
from plain import llama as plain
from plain import sampler as psampler

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# ------------------------------------------------------------------ sampling kernels
def test_argmax_first_maximum_wins():
    from glassbox_amd import ops
    g = torch.Generator().manual_seed(0)
    for vocab in (5, 331, 49152):
        logits = torch.randn(6, vocab, generator=g)
        logits[1, 3] = logits[1, vocab - 1] = 9.0            # a tie: the first one
        logits[2, vocab - 1] = 10.0
        logits[3, :] = -1.5                                  # all equal: token 0
        logits[4, 0] = 11.0
        logits[5] = -logits[5].abs()                         # zeros of both signs are one value: the first of them
        logits[5, 2], logits[5, 4] = -0.0, 0.0
        out = torch.empty(6, dtype=torch.int32, device=DEV)
        ops.argmax(logits.to(DEV), out)
        assert out.tolist() == [psampler.argmax(r) for r in logits.tolist()]
        assert out.tolist()[1:] == [3, vocab - 1, 0, 0, 2]


def test_sampler_vectors_of_the_reference_on_the_device():
    # crates/glassbox-core/src/sampler.rs:188-218
    from glassbox_amd.sampling import SamplerConfig, sample_rows
    logits = torch.tensor([[1.0, 3.0, 2.0, 0.0, -1.0]] * 4, device=DEV)
    cfgs = [SamplerConfig(), SamplerConfig(temperature=1.0, top_k=2), SamplerConfig(temperature=1.0, top_p=0.5),
            SamplerConfig(temperature=1.0, min_p=0.3)]
    toks, cands = sample_rows(logits.clone(), cfgs, [0.99] * 4)
    assert cands == [1, 2, 1, 2]
    assert toks == [1, 2, 1, 2]            # u = 0.99 falls on the last candidate of each distribution
    toks, _ = sample_rows(logits.clone(), cfgs, [0.0] * 4)
    assert toks == [1, 1, 1, 1]
    # p0 = 1 / (1 + e^-1) = 0.731 with top_k = 2: the draw turns at that value
    assert sample_rows(logits[:1].clone(), [cfgs[1]], [0.73])[0] == [1]
    assert sample_rows(logits[:1].clone(), [cfgs[1]], [0.7320])[0] == [2]
    # repetition penalty 4 on token 1 makes token 2 the maximum (sampler.rs:213-217)
    toks, _ = sample_rows(logits[:1].clone(), [SamplerConfig(repetition_penalty=4.0)], [0.0], [[1]])
    assert toks == [2]


def check_sampled(row, context, c, u, token, candidates):
    """One row's token and number of candidates against the plain sampler.  The reference adds its probabilities in
    32-bit, one after the other (sampler.rs:118-146,155-163); the kernel adds whole numbers, which is exact.  Where the
    two differ, the 32-bit sums' rounding decides (a cut or a draw that falls within it of a boundary), so the kernel
    must give either the plain sampler's answer or the one of the same formulas in 64-bit, within 2e-6 of a boundary."""
    dist = psampler.distribution(row, context, c.temperature, c.top_k, c.top_p, c.min_p, c.repetition_penalty)
    if c.temperature <= 0.0:
        assert (token, candidates) == (dist[0][0], 1), c
        return
    delta = 2e-6
    # the candidates before top-p, most likely first (min-p keeps a prefix of the top k), and exp(l - max) in 64-bit
    kept = len(psampler.distribution(row, context, c.temperature, c.top_k, 1.0, c.min_p, c.repetition_penalty))
    top = psampler.distribution(row, context, c.temperature, c.top_k, 1.0, 0.0, c.repetition_penalty)
    l = np.array(row, dtype=np.float32)
    if c.repetition_penalty != 1.0:
        for t in context:
            l[t] = l[t] / np.float32(c.repetition_penalty) if l[t] > 0 else l[t] * np.float32(c.repetition_penalty)
    l = (l / np.float32(c.temperature)).astype(np.float32)
    order = [t for t, _ in top]
    e = np.exp(l[order].astype(np.float64) - float(l[order[0]]))
    if c.top_p < 1.0:
        run = np.cumsum(e[:kept]) / e.sum()                 # the softmax over the top k, min-p's prefix of it
        n = candidates
        exact = 1 <= n <= kept and (run[n - 1] >= c.top_p - delta or n == kept) and (n == 1 or run[n - 2] < c.top_p + delta)
        assert exact or n == len(dist), (c, n, len(dist))
    else:
        n = candidates
        assert n == len(dist), (c, n, len(dist))
    if n == 1:
        assert token == order[0], (c, token)
        return
    run = np.cumsum(e[:n]) / e[:n].sum()
    at = order.index(token)
    assert at < n, (c, token, at, n)
    exact = (run[at - 1] if at else 0.0) <= u + delta and (run[at] >= u - delta or at == n - 1)
    # the plain sampler's own draw, from its 32-bit running sum
    acc, plain_draw = np.float32(0), dist[-1][0]
    for t, p in dist:
        acc = np.float32(acc + np.float32(p))
        if u < acc:
            plain_draw = t
            break
    assert exact or token == plain_draw, (c, token, at, plain_draw, u)


@pytest.mark.parametrize("vocab,spread", [(97, 3.0), (331, 3.0), (49152, 3.0), (2500, 0.05), (49152, 0.2), (128256, 2.0)])
def test_sampling_kernel_agrees_with_the_plain_sampler(vocab, spread):
    """Rows of peaked and of nearly flat logits (random weights give the latter: the draw then falls among thousands
    of tokens of almost one probability), with every filter on and off, against the plain sampler."""
    from glassbox_amd.sampling import SamplerConfig, sample_rows
    g = torch.Generator().manual_seed(vocab + int(spread * 100))
    rng = random.Random(vocab + int(spread * 100))
    rows = 24 if vocab < 1000 else 6
    logits = torch.randn(rows, vocab, generator=g) * spread
    logits[0, 5] = logits[0, 9] = logits[0].max() + 1         # ties at the top go by token id
    logits[1, :] = 0.25                                        # every logit equal
    if rows > 2:
        logits[2] = (logits[2] * 2).round() / 2                # few values, many ties, zeros of both signs
    cfgs, ctxs, us = [], [], []
    for r in range(rows):
        cfgs.append(SamplerConfig(temperature=rng.choice([0.0, 0.6, 1.0, 2.0]), top_k=rng.choice([0, 0, 1, 7, 50]),
                                  top_p=rng.choice([1.0, 1.0, 0.95, 0.6, 0.1]), min_p=rng.choice([0.0, 0.0, 0.02, 0.3]),
                                  repetition_penalty=rng.choice([1.0, 1.0, 1.2, 3.0])))
        ctxs.append([rng.randrange(vocab) for _ in range(rng.randrange(0, 30))] + [5, 5])
        us.append(rng.random())
    toks, cands = sample_rows(logits.to(DEV), cfgs, us, ctxs)
    for r in range(rows):
        check_sampled(logits[r].tolist(), ctxs[r], cfgs[r], us[r], toks[r], cands[r])
    # the same left on the device (what a step launched ahead takes its tokens from), drawn and greedy rows
    from glassbox_amd.sampling import sample_rows_pending
    late_toks, late_cands = sample_rows_pending(logits.to(DEV), cfgs, us, ctxs)
    assert late_toks.tolist() == toks and late_cands.tolist() == cands and late_toks[3].value() == toks[3]
    greedy = [SamplerConfig(repetition_penalty=c.repetition_penalty) for c in cfgs]
    want, _ = sample_rows(logits.to(DEV), greedy, us, ctxs)
    late_toks, late_cands = sample_rows_pending(logits.to(DEV), greedy, us, ctxs)
    assert late_toks.tolist() == want and late_cands is None


def test_sampling_kernel_on_rows_of_ties_and_edge_settings():
    """Rows that are all one value, two values, or a few (with zeros of both signs, which are one value and go by
    token id), with filters at their edges: top-k of 1 and beyond the vocabulary, top-p of 0 and just below 1, min-p
    of 1, uniform numbers of 0 and just below 1."""
    from glassbox_amd.sampling import SamplerConfig, sample_rows
    checked = 0
    for seed in range(12):
        rng = random.Random(seed)
        g = torch.Generator().manual_seed(seed)
        vocab = rng.choice([17, 150, 1025, 2500, 4099])
        spread = rng.choice([0.02, 0.3, 1.0, 8.0])
        logits = torch.randn(16, vocab, generator=g) * spread
        mode = seed % 3
        if mode == 0:
            logits = (logits * 2).round() / 2
        elif mode == 1:
            logits = logits.sign() * spread
        else:
            logits[:] = rng.choice([0.0, -3.5, 7.25])
        cfgs, ctxs, us = [], [], []
        for r in range(16):
            cfgs.append(SamplerConfig(temperature=rng.choice([0.0, 0.05, 0.6, 2.0, 5.0]), top_k=rng.choice([0, 1, 2, 50, vocab, vocab + 5]),
                                      top_p=rng.choice([1.0, 0.95, 0.1, 0.0, 0.999]), min_p=rng.choice([0.0, 0.02, 0.9, 1.0]),
                                      repetition_penalty=rng.choice([1.0, 1.2, 3.0])))
            ctxs.append([rng.randrange(vocab) for _ in range(rng.randrange(0, 30))])
            us.append(rng.choice([rng.random(), 0.0, 0.999999]))
        toks, cands = sample_rows(logits.clone().to(DEV), cfgs, us, ctxs)
        for r in range(16):
            check_sampled(logits[r].tolist(), ctxs[r], cfgs[r], us[r], toks[r], cands[r])
            checked += 1
    assert checked == 192


@pytest.mark.parametrize("rows", [7, 256, 257])
@pytest.mark.parametrize("vocab", [1, 2, 3, 6, 1023, 1026, 4097, 16387, 20006])
def test_argmax_of_rows_that_begin_anywhere(rows, vocab):
    """Rows that begin at every place in a word of 16 bytes, from one token on; the maximum at either end and in the words between,
    the first of two."""
    from glassbox_amd import ops
    g = torch.Generator().manual_seed(vocab)
    for shift in range(4):
        flat = torch.randn(rows * vocab + 4, generator=g)
        logits = flat[shift:shift + rows * vocab].view(rows, vocab)
        for r, at in enumerate((0, vocab - 1, vocab // 2, max(0, vocab - 2), min(1, vocab - 1), min(3, vocab - 1), max(0, vocab - 4))):
            logits[r, at] = 9.0
            logits[r, vocab - 1] = 9.0
        out = torch.empty(rows, dtype=torch.int32, device=DEV)
        ops.argmax(flat.to(DEV)[shift:shift + rows * vocab].view(rows, vocab), out)
        first = (logits == logits.max(dim=1, keepdim=True).values).int().argmax(dim=1)
        assert out.tolist() == first.tolist()


@pytest.mark.parametrize("vocab", [1023, 1024, 1027, 4099, 49152])
@pytest.mark.parametrize("ties", [False, True])
def test_sampling_kernel_where_few_candidates_are_sorted(vocab, ties):
    """Top-k on either side of where the candidates are found first and sorted (512), with more of one value than the kernel
    sorts (1,024), and of rows with few more tokens than it has threads; the other filters behind it."""
    from glassbox_amd.sampling import SamplerConfig, sample_rows
    rng = random.Random(vocab)
    g = torch.Generator().manual_seed(vocab)
    ks = [1, 2, 50, 63, 64, 500, 511, 512, 513, 1000, 1022]
    logits = torch.randn(len(ks) + 3, vocab, generator=g)
    if ties:
        logits = (logits * 8).round() / 8
    logits[-1, 1000:] -= 20.0                                  # a thousand before all others
    logits[-2, :] = 1.0                                        # all equal: more of one value than are sorted, or just as many
    logits[-3] = logits[-3] * 6
    cfgs = [SamplerConfig(temperature=0.9, top_k=k, top_p=rng.choice([1.0, 0.97, 0.5]), min_p=rng.choice([0.0, 0.0, 0.05])) for k in ks]
    cfgs += [SamplerConfig(temperature=1.0, top_k=20, top_p=0.9, min_p=0.2), SamplerConfig(temperature=1.0, top_k=9, top_p=0.5),
             SamplerConfig(temperature=1.0, top_k=40, top_p=0.7)]
    us = [rng.random() for _ in cfgs]
    toks, cands = sample_rows(logits.clone().to(DEV), cfgs, us, [[]] * len(cfgs))
    for r, c in enumerate(cfgs):
        check_sampled(logits[r].tolist(), [], c, us[r], toks[r], cands[r])


@pytest.mark.parametrize("vocab", [1025, 2048, 5000])
def test_sampling_kernel_on_many_rows_with_more_ties_than_are_sorted(vocab):
    """Rows of few values, more than 1,024 tokens of them at or above the k-th: no thread may go on to the searches before all
    have seen how many there are.  Every row against the reference, and a second time."""
    from glassbox_amd.sampling import SamplerConfig, sample_rows
    rng = random.Random(vocab)
    g = torch.Generator().manual_seed(vocab)
    n = 96
    logits = torch.zeros(n, vocab)
    logits[1::3] = torch.randint(0, 2, (n // 3, vocab), generator=g) * 0.001      # apart below the bound's 16 bits
    logits[2::3, :12] += torch.randn(n // 3, 12, generator=g).abs()
    cfgs = [SamplerConfig(temperature=1.0, top_k=rng.choice([13, 40, 300, 512]), top_p=rng.choice([1.0, 0.9]), min_p=rng.choice([0.0, 0.05]))
            for _ in range(n)]
    us = [rng.random() for _ in cfgs]
    first = sample_rows(logits.clone().to(DEV), cfgs, us, [[]] * n)
    assert list(map(list, first)) == list(map(list, sample_rows(logits.clone().to(DEV), cfgs, us, [[]] * n)))
    for r, c in enumerate(cfgs):
        check_sampled(logits[r].tolist(), [], c, us[r], first[0][r], first[1][r])


@pytest.mark.parametrize("vocab", [1024, 1025, 4099, 16384])
@pytest.mark.parametrize("mask", [-math.inf, -3.3e38, -1e4])
def test_sampling_kernel_behind_masks_that_leave_few_tokens(vocab, mask):
    """One token fewer than top-k left, as many, one more, a thousand: which way a row takes depends on that."""
    from glassbox_amd.sampling import SamplerConfig, sample_rows
    rng = random.Random(vocab)
    g = torch.Generator().manual_seed(vocab)
    cfgs, rows = [], []
    for k in (1, 2, 40, 256, 257, 511):
        for left in (k - 1, k, k + 1, 1000):
            row = torch.full((vocab,), mask)
            keep = torch.randperm(vocab, generator=g)[:left]
            row[keep] = torch.randn(left, generator=g) * 2
            rows.append(row)
            cfgs.append(SamplerConfig(temperature=1.0, top_k=k, top_p=rng.choice([1.0, 0.9]), min_p=rng.choice([0.0, 0.02])))
    us = [rng.random() for _ in cfgs]
    toks, cands = sample_rows(torch.stack(rows).to(DEV), cfgs, us, [[]] * len(cfgs))
    for r, c in enumerate(cfgs):
        if bool((rows[r] > mask).any()) or mask > -math.inf:      # (a row without any token left has no answer)
            check_sampled(rows[r].tolist(), [], c, us[r], toks[r], cands[r])


def test_temperature_draws_follow_the_softmax():
    from glassbox_amd.sampling import Rng, SamplerConfig, sample_rows
    logits = torch.tensor([[0.0, math.log(2.0), math.log(5.0), -30.0]], device=DEV).repeat(64, 1)
    rng, counts = Rng(3), np.zeros(4)
    cfg = [SamplerConfig(temperature=1.0)] * 64
    for _ in range(60):
        toks, _ = sample_rows(logits.clone(), cfg, [rng.next_f32() for _ in range(64)])
        for t in toks:
            counts[t] += 1
    assert np.abs(counts / counts.sum() - np.array([1, 2, 5, 0]) / 8).max() < 0.03
    # temperature 2 flattens: p ~ (1, sqrt 2, sqrt 5)
    counts = np.zeros(4)
    for _ in range(60):
        toks, _ = sample_rows(logits.clone(), [SamplerConfig(temperature=2.0)] * 64, [rng.next_f32() for _ in range(64)])
        for t in toks:
            counts[t] += 1
    want = np.array([1, math.sqrt(2), math.sqrt(5), 0])
    assert np.abs(counts / counts.sum() - want / want.sum()).max() < 0.03


# ------------------------------------------------------------------- entry points
def assert_greedy(folder, prompts, outs, steps, dtype, what):
    """Every reply is the greedy continuation by the plain implementation on the weights the engine holds.  Two
    logits can lie within rounding of each other; a token that differs where the plain margin is below ``margin``
    ends that reply's comparison (in 32-bit that does not happen with these models; in bfloat16 rarely)."""
    cfg, w = helpers._load_rounded(folder) if dtype == "bfloat16" else helpers._load(folder)
    margin = 1e-4 if dtype == "float32" else 1e-2
    compared = 0
    for p, out in zip(prompts, outs):
        assert len(out) == steps
        toks = list(p)
        for i, t in enumerate(out):
            logits = plain.forward(w, cfg, toks)[-1]
            if t != int(torch.argmax(logits)):
                top2 = torch.topk(logits, 2).values
                assert (top2[0] - top2[1]).item() < margin, f"{what}, {dtype}, prompt of {len(p)} tokens, step {i}: wrong token"
                break
            toks.append(t)
            compared += 1
    assert compared >= 0.6 * steps * len(prompts), f"{what}, {dtype}: the comparison ended early too often"


@pytest.mark.parametrize("dtype,graphs", [("bfloat16", True), ("bfloat16", False), ("float32", True)])
def test_a_step_takes_sampled_tokens_from_the_device(model_dirs, dtype, graphs):
    """``greedy_pending`` leaves a step's tokens on the device and ``Engine.step`` takes them from there (the host reads
    their values after the launch): the same logits, bit for bit, as with tokens read back first.  Rows in another
    order than the sampler left them, a request that sits a step out, a pending token beside another request's
    prompt portion (the general path), and the cache manager's record of the tokens, which a later request with the
    same beginning finds."""
    from glassbox_amd.engine import Engine
    from glassbox_amd.sampling import PendingToken, greedy_pending
    folder = model_dirs.get("B")
    vocab = helpers.TINY["B"]["vocab_size"]
    prompts = {r: helpers.random_tokens(vocab, n, seed=80 + i) for i, (r, n) in enumerate({"a": 30, "b": 17, "c": 44}.items())}
    late, first = (Engine(folder, dtype=dtype, max_tokens=1024, max_seqs=8, graph_decode=graphs, prefix_caching=True)
                   for _ in range(2))
    wants = [(r, p, [len(p) - 1]) for r, p in prompts.items()]
    order = ["a", "b", "c"]
    sampled = greedy_pending(late.step(wants))
    tok_late = {r: sampled[i] for i, r in enumerate(order)}               # each request's newest token: on the device
    tok_first = dict(zip(order, first.step(wants).argmax(-1).tolist()))   # and read back
    history = {r: [] for r in order}
    schedule = [["a", "b", "c"], ["c", "a", "b"], ["b", "c"], ["b", "c"], ["c", "b"]] + [["c", "b"]] * 20
    for step, live in enumerate(schedule):
        e_late = [(r, [tok_late[r]], [0]) for r in live]
        e_first = [(r, [tok_first[r]], [0]) for r in live]
        if step == 3:     # request a comes back with a prompt portion beside the others' pending tokens
            extra = helpers.random_tokens(vocab, 9, seed=99)
            e_late.insert(0, ("a", [tok_late["a"]] + extra, [9]))
            e_first.insert(0, ("a", [tok_first["a"]] + extra, [9]))
            live = ["a"] + live
        assert all(isinstance(toks[0], PendingToken) for _, toks, _ in e_late)
        for r, toks, _ in e_first:
            history[r] += toks
        l_late, l_first = late.step(e_late), first.step(e_first)
        assert torch.equal(l_late, l_first), f"step {step}: logits differ with tokens taken from the device"
        sampled = greedy_pending(l_late)
        tok_first.update(zip(live, l_first.argmax(-1).tolist()))
        tok_late.update({r: sampled[i] for i, r in enumerate(live)})
        assert sampled.tolist() == [tok_first[r] for r in live]
    if graphs:
        assert late.decode_graphs.replays >= 15
    with pytest.raises(Exception, match="only the first"):
        late.step([("b", [5, tok_late["b"]], [1])])
    # what the cache manager recorded are the values: a request with the same beginning finds the pages
    for eng in (late, first):
        eng.cache.check_invariants()
        whole = prompts["c"] + history["c"]
        assert eng.request_len("c") == len(whole)
        assert eng.add_request("again", whole) == (len(whole) - 1) // 16 * 16
        for r in ("a", "b", "c", "again"):
            eng.end_request(r)
        assert eng.cache.used_pages() == 0


@pytest.mark.parametrize("name", ["A", "B", "D"])
def test_greedy_generation_through_the_entry_point(model_dirs, name):
    """generate() against the plain implementation's greedy decoding: the first tiny configuration with its
    prompts of 5, 17 and 33 tokens and 16 steps, the second with 1, 9, 40 and 70 tokens in portions of sixteen."""
    from glassbox_amd import Engine, generate
    folder = model_dirs.get(name)
    vocab = helpers.TINY[name]["vocab_size"]
    prompts = [helpers.random_tokens(vocab, n, seed=n) for n in ((5, 17, 33) if name == "A" else (1, 9, 40, 70))]
    steps = 16 if name == "A" else 24
    for dtype in ("float32", "bfloat16"):
        eng = Engine(folder, dtype=dtype, max_tokens=1024, max_seqs=8)
        outs = generate(eng, prompts, max_tokens=steps, token_budget=256 if name == "A" else 16)
        assert_greedy(folder, prompts, outs, steps, dtype, f"generate() on {name}")
        if name != "A":   # the reply must say something about the context (the tied tiny model echoes its last token)
            assert any(out != [p[-1]] * steps for p, out in zip(prompts, outs))
        eng.cache.check_invariants()
        assert eng.cache.used_pages() == 0


def test_batched_equals_unbatched_on_the_device(model_dirs):
    """crates/glassbox-server/tests/scheduler.rs:84-123 with the real model in 32-bit, where every
    output cell is summed in an order that does not depend on the batch: exact equality.  On the untied tiny
    model, whose replies depend on the context, through a pool so small that requests are preempted."""
    from glassbox_amd import Engine, generate, greedy
    folder = model_dirs.get("B")
    rng = random.Random(4)
    jobs = [([rng.randrange(384) for _ in range(1 + rng.randrange(60))], 1 + rng.randrange(24)) for _ in range(10)]
    eng = Engine(folder, dtype="float32", max_tokens=14 * 16, max_seqs=12, prefix_caching=True)
    alone = [greedy(eng, p, n) for p, n in jobs]
    assert any(ref != [p[-1]] * n for (p, n), ref in zip(jobs, alone)), "replies that echo the prompt show nothing"
    assert eng.cache.used_pages() == 0
    outs, sched = generate(eng, [p for p, _ in jobs], max_tokens=24, token_budget=16, return_scheduler=True)
    for (p, n), out, ref in zip(jobs, outs, alone):
        assert out[:n] == ref
    assert sched.metrics["preemptions"] > 0, "14 pages for 10 requests should force preemption"
    assert_greedy(folder, [p for p, _ in jobs], outs, 24, "float32", "batched")
    eng.cache.check_invariants()
    assert eng.cache.used_pages() == 0


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_prefix_sharing_on_the_device(model_dirs, dtype):
    """A shared 70-token prefix is computed once; outputs equal those without sharing
    (tests/scheduler.rs:165-186): in 32-bit exactly, in bfloat16 both are the plain implementation's replies."""
    from glassbox_amd import Engine, generate
    folder = model_dirs.get("B")
    rng = random.Random(11)
    system = [(i * 13) % 384 for i in range(70)]
    prompts = [system + [rng.randrange(384) for _ in range(1 + rng.randrange(40))] for _ in range(8)]
    res = {}
    for share in (True, False):
        eng = Engine(folder, dtype=dtype, max_tokens=128 * 16, max_seqs=4, prefix_caching=share)
        res[share] = generate(eng, prompts, max_tokens=12, token_budget=48, max_seqs=4, return_scheduler=True)
        assert_greedy(folder, prompts, res[share][0], 12, dtype, f"prefix cache {share}")
        assert eng.cache.used_pages() == 0
    if dtype == "float32":
        assert res[True][0] == res[False][0]
    assert any(out != [p[-1]] * 12 for p, out in zip(prompts, res[True][0]))
    assert res[True][1].metrics["prefix_hit_tokens"] >= 64 and res[False][1].metrics["prefix_hit_tokens"] == 0


def test_fork_copies_the_shared_page_on_the_device(model_dirs):
    """kv.rs:336-349 end to end: a forked request continues from its parent's cache, and the parent's
    partial page is copied before the child writes into it."""
    from glassbox_amd import Engine
    folder = model_dirs.get("B")
    toks = helpers.random_tokens(384, 41, seed=8)
    eng = Engine(folder, dtype="float32", max_tokens=512, max_seqs=4)
    eng.step([("p", toks[:20], [])])
    eng.fork_request("p", "c")
    a = eng.step([("c", [7, 8, 9], [0, 1, 2])]).cpu().numpy().copy()
    b = eng.step([("p", toks[20:], list(range(21)))]).cpu().numpy().copy()
    assert np.abs(a - helpers.plain_logits(folder, tuple(toks[:20] + [7, 8, 9]))[20:]).max() < 1e-4
    assert np.abs(b - helpers.plain_logits(folder, tuple(toks))[20:]).max() < 1e-4
    eng.end_request("p"); eng.end_request("c")
    eng.cache.check_invariants()
    assert eng.cache.used_pages() == 0


def test_seeded_temperature_generation_repeats(model_dirs):
    """The same seeds give the same replies, in bfloat16 too (what the replies must be is checked in 32-bit, against
    the plain sampler, in test_scheduler_gpu.py)."""
    from glassbox_amd import Engine, SamplerConfig, generate
    eng = Engine(model_dirs.get("B"), dtype="bfloat16", max_tokens=2048, max_seqs=8)
    prompts = [helpers.random_tokens(384, n, seed=n) for n in (1, 9, 40, 70)]
    cfgs = [SamplerConfig(temperature=0.8, seed=s) for s in (1, 2, 3, 4)]
    a = generate(eng, prompts, 24, cfgs, token_budget=16)
    b = generate(eng, prompts, 24, cfgs, token_budget=16)
    c = generate(eng, prompts, 24, [SamplerConfig(temperature=0.8, seed=s + 10) for s in (1, 2, 3, 4)], token_budget=16)
    assert a == b and a != c and all(len(o) == 24 for o in a)


def test_a_warm_up_leaves_nothing_behind(model_dirs):
    """``Engine.warm_up`` runs a throwaway request: afterwards no page is held, no request is live, the decode graph of
    that length is there, and a request's logits are what they are without it; a pool too small for it is left alone."""
    from glassbox_amd.engine import Engine
    folder = model_dirs.get("B")
    prompt = helpers.random_tokens(384, 21, seed=2)
    plain_engine = Engine(folder, dtype="float32", max_tokens=128, max_seqs=2)
    want = plain_engine.step([("a", prompt, [20])]).clone()
    eng = Engine(folder, dtype="float32", max_tokens=128, max_seqs=2)
    eng.warm_up(len(prompt))
    assert eng.cache.used_pages() == 0 and not eng._ids
    assert eng.decode_graphs is None or eng.decode_graphs.shapes
    assert torch.equal(eng.step([("a", prompt, [20])]), want)
    eng.end_request("a")
    tiny = Engine(folder, dtype="float32", max_tokens=16, max_seqs=1)   # one page
    tiny.warm_up(64)
    assert tiny.cache.used_pages() == 0


def _glassbox(*args, stdin=None):
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    return subprocess.run([sys.executable, os.path.join(root, "bin", "glassbox"), *args], capture_output=True, text=True,
                          timeout=600, input=stdin)


@pytest.fixture(scope="module")
def cli_model(tmp_path_factory):
    """The second tiny configuration written by ``glassbox random``."""
    import json
    base = tmp_path_factory.mktemp("cli")
    cfg = base / "cfg.json"
    cfg.write_text(json.dumps(helpers.TINY_B))
    out = base / "model"
    r = _glassbox("random", "--config", str(cfg), "--out", str(out), "--seed", "5")
    assert r.returncode == 0, r.stderr
    return str(out)


def test_the_command_line_generates(cli_model):
    r = _glassbox("generate", "--model", cli_model, "--prompt", "5,17,3,300,41", "-n", "8", "--dtype", "float32")
    assert r.returncode == 0, r.stderr
    toks = [int(t) for t in r.stdout.split()]
    c, w = plain.load_folder(cli_model)
    want = plain.greedy(w, c, [5, 17, 3, 300, 41], 8)
    assert want != [41] * 8, "a reply that echoes the prompt shows nothing"
    assert toks == want and "prefill 5 tokens" in r.stderr
    # sampling options reach the sampler: temperature with a seed repeats, another seed differs
    runs = [_glassbox("generate", "--model", cli_model, "--prompt", "5 17 3", "-n", "12", "--dtype", "float32", "--temp", "0.9",
                      "--top-k", "40", "--seed", s).stdout.split() for s in ("3", "3", "4")]
    assert runs[0] == runs[1] and runs[0] != runs[2] and len(runs[0]) == 12


def test_the_command_line_batches(cli_model, tmp_path):
    """``glassbox batch``: one prompt a line, continuous batching, replies in the order of the prompts."""
    prompts = [helpers.random_tokens(384, n, seed=30 + n) for n in (3, 41, 18, 70, 9)]
    f = tmp_path / "prompts.txt"
    f.write_text("\n".join(" ".join(map(str, p)) for p in prompts) + "\n")
    r = _glassbox("batch", "--model", cli_model, "--prompts", str(f), "-n", "10", "--dtype", "float32", "--budget", "16",
                  "--max-seqs", "3", "--blocks", "64")
    assert r.returncode == 0, r.stderr
    got = [[int(t) for t in line.split()] for line in r.stdout.strip().splitlines()]
    c, w = plain.load_folder(cli_model)
    assert got == [plain.greedy(w, c, p, 10) for p in prompts]
    assert "5 requests, 50 tokens" in r.stderr


def test_the_command_line_benchmarks_and_replays(cli_model, tmp_path):
    """``glassbox bench single``, ``bench serve`` and ``replay`` run and report what they say they report."""
    import json
    out = tmp_path / "single.json"
    r = _glassbox("bench", "single", "--model", cli_model, "--label", "tiny", "--out", str(out))
    assert r.returncode == 0, r.stderr
    res = json.loads(out.read_text())
    assert res["label"] == "tiny" and res["pp512_tok_s"] > 0 and res["tg128_tok_s"] > 0 and res["meta"]["gpu"]
    r = _glassbox("bench", "serve", "--model", cli_model, "--workload", "system", "--requests", "6", "--rates", "inf",
                  "--blocks", "256", "--budget", "64", "--max-seqs", "4")
    assert r.returncode == 0, r.stderr
    res = json.loads(r.stdout)
    modes = {run["mode"]: run["result"] for run in res["runs"]}
    assert set(modes) == {"prefix cache", "no prefix cache"}
    assert modes["prefix cache"]["prefix_hit_tokens"] >= 384 and modes["no prefix cache"]["prefix_hit_tokens"] == 0
    assert all(m["requests"] == 6 and m["throughput_tok_s"] > 0 for m in modes.values())
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": [5, 17, 3, 9], "want": [3]}], "end": []},
             {"step": 1, "entries": [{"id": "a", "tokens": [8], "want": [0]}], "end": ["a"]}]
    r = _glassbox("replay", "--model", cli_model, "--dtype", "float32", "--out", str(tmp_path / "logits"), "--max-tokens", "64",
                  stdin="".join(json.dumps(s) + "\n" for s in steps))
    assert r.returncode == 0 and r.stdout.split() == ["done", "0", "done", "1"], r.stderr
    got = np.fromfile(tmp_path / "logits" / "1.f32", dtype="<f4")
    c, w = plain.load_folder(cli_model)
    assert np.abs(got - plain.forward(w, c, [5, 17, 3, 9, 8])[-1].numpy()).max() < 1e-4


@pytest.mark.parametrize("name,dtype", [("B", "bfloat16"), ("M", "bfloat16"), ("A", "float32")])
def test_steps_of_single_tokens_replay_graphs_like_plain_steps(model_dirs, name, dtype):
    """Engine.step replays steps of one token per request from HIP graphs.  The same steps through an engine
    without graphs give the same logits: with the number of live requests changing (1, 2, 3 and 5 rows, so that
    filler rows stand beside the live ones), prompts of other requests between the replays (their steps take the
    general path and their buffers grow), a request ending and its pages going to the next, and a context that
    crosses from one bucket of 1,024 tokens into the next."""
    from glassbox_amd.engine import Engine
    folder = model_dirs.get(name)
    vocab = helpers.TINY[name]["vocab_size"]
    long = 1015 if name == "M" else 50
    lens = {"a": long, "b": 37, "c": 70 if name != "M" else 300, "d": 9, "e": 21, "f": 40}
    prompts = {r: helpers.random_tokens(vocab, n, seed=60 + i) for i, (r, n) in enumerate(lens.items())}
    engs = [Engine(folder, dtype=dtype, max_tokens=2048, max_seqs=8, graph_decode=g) for g in (True, False)]
    assert engs[0].decode_graphs is not None and engs[1].decode_graphs is None
    nxt = {r: 7 + i for i, r in enumerate(prompts)}
    tol = 2e-5 if dtype == "float32" else 8e-3

    def both(entries, what):
        outs = [e.step(entries).float().cpu() for e in engs]
        if outs[0].numel():
            scale = max(1.0, float(outs[1].abs().max()))
            err = float((outs[0] - outs[1]).abs().max())
            assert err <= tol * scale, f"{what}: graphs and plain steps differ by {err:.3e} (largest logit {scale:.2f})"
        return outs[1]

    def decode(live, steps, what):
        for s in range(steps):
            logits = both([(r, [nxt[r]], [0]) for r in live], f"{what}, step {s}, requests {live}")
            for r, row in zip(live, logits):
                nxt[r] = int(row.argmax())

    both([("a", prompts["a"], [])], "prompt a")
    decode(["a"], 4, "one request")
    both([("b", prompts["b"], [len(prompts["b"]) - 1])], "prompt b")
    decode(["a", "b"], 5, "two requests")
    both([("c", prompts["c"], []), ("a", [nxt["a"]], [0]), ("b", [nxt["b"]], [0])], "prompt c beside single tokens")
    decode(["b", "c", "a"], 6, "three requests and a filler")
    for e in engs:
        e.end_request("b")
    both([("d", prompts["d"], []), ("e", prompts["e"], [3])], "prompts d and e")
    decode(["a", "c", "d", "e"], 3, "four requests")
    both([("f", prompts["f"], [])], "prompt f")
    decode(["f", "a", "c", "d", "e"], 7, "five requests and three fillers")
    decode(["a"], 3, "one request again")
    graphs = engs[0].decode_graphs
    assert graphs.replays >= 12 and len({rows for rows, _ in graphs.shapes}) >= 4
    if name == "M":
        assert len({bucket for _, bucket in graphs.shapes}) == 2
    for e in engs:
        for r in ("a", "c", "d", "e", "f"):
            e.end_request(r)
        e.cache.check_invariants()
        assert e.cache.used_pages() == 0


@pytest.mark.parametrize("name", ["B", "M"])
def test_single_token_steps_leave_the_final_norm_to_the_products(model_dirs, name, monkeypatch):
    """In a bfloat16 step of a few single tokens, each wanting its logits, no norm runs as a kernel of its own: the
    first is computed by the first product, the others are prepared by the product that makes the residual before
    them, the final norm (crates/glassbox-core/src/model.rs:350-361) by the last block's, and the vocabulary
    product scales by its factor.  A step that wants other rows, or more than sixteen, norms the wanted rows as
    before; the logits are those of the plain kernels either way."""
    from glassbox_amd import ops
    from glassbox_amd.engine import Engine
    folder = model_dirs.get(name)
    vocab = helpers.TINY[name]["vocab_size"]
    fused, plain_eng = (Engine(folder, dtype="bfloat16", max_tokens=2048, max_seqs=24, graph_decode=False, kernels=k)
                        for k in ("auto", "plain"))
    calls = []
    real = ops.rmsnorm
    monkeypatch.setattr(ops, "rmsnorm", lambda *a, **k: (calls.append(a[0].shape[0]), real(*a, **k))[1])

    def step(entries):
        calls.clear()
        got = fused.step(entries).float().cpu()
        n = len(calls)
        want = plain_eng.step(entries).float().cpu()
        assert (got - want).abs().max().item() <= 8e-3 * max(1.0, want.abs().max().item())
        return n

    prompts = {r: helpers.random_tokens(vocab, 20 + 3 * i, seed=80 + i) for i, r in enumerate("abcdefghijklmnopqr")}
    assert step([(r, p, [len(p) - 1]) for r, p in prompts.items()]) >= 1          # portions: the wanted rows are normed
    few = list(prompts)[:5]
    assert step([(r, [9], [0]) for r in few]) == 0                                # five single tokens: no norm kernel
    assert step([(r, [11], [0] if i else []) for i, r in enumerate(few)]) >= 1    # one of them wants nothing
    assert step([(r, [12], [0]) for r in prompts]) >= 1                           # eighteen rows: beyond the limit
    assert step([(few[0], [13], [0])]) == 0


def test_decode_graph_shapes_are_kept_up_to_a_limit(model_dirs, monkeypatch):
    """Only so many shapes keep their buffers and graph; the least recently used one makes room, and a shape that
    comes back is warmed and captured again.  The logits stay those of an engine without graphs."""
    from glassbox_amd.engine import Engine, decode_graphs
    monkeypatch.setattr(decode_graphs, "MAX_SHAPES", 2)
    folder = model_dirs.get("A")
    vocab = helpers.TINY["A"]["vocab_size"]
    prompts = {r: helpers.random_tokens(vocab, n, seed=80 + i) for i, (r, n) in enumerate({"a": 20, "b": 9, "c": 31}.items())}
    engs = [Engine(folder, dtype="bfloat16", max_tokens=1024, max_seqs=4, graph_decode=g) for g in (True, False)]
    nxt = {"a": 3, "b": 4, "c": 5}
    for r, toks in prompts.items():
        for e in engs:
            e.step([(r, toks, [])])
    for live in (["a"], ["a", "b"], ["a", "b", "c"], ["a"], ["b", "c"], ["c", "a", "b"]):
        for _ in range(4):
            outs = [e.step([(r, [nxt[r]], [0]) for r in live]).float().cpu() for e in engs]
            assert float((outs[0] - outs[1]).abs().max()) <= 8e-3 * max(1.0, float(outs[1].abs().max())), live
            for r, row in zip(live, outs[1]):
                nxt[r] = int(row.argmax())
        assert len(engs[0].decode_graphs.shapes) <= 2
    assert engs[0].decode_graphs.replays >= 6


def test_graphs_die_with_their_engine_and_nothing_is_collected_during_a_capture(model_dirs):
    """A graph that dies synchronises the device, which is not allowed while a stream captures.  The graphs hold
    their engine weakly, so an engine that is dropped frees them at once, by reference count, with the garbage
    collector off; and the collector is held off for the length of a capture all the same, and is back on after."""
    import gc
    import weakref
    import torch
    from glassbox_amd.engine import Engine
    folder = model_dirs.get("B")
    toks = helpers.random_tokens(helpers.TINY["B"]["vocab_size"], 12, seed=5)

    def decode(eng, steps, seen=None):
        eng.step([("r", toks, [])])
        if seen is not None:
            plain_forward = eng.model.forward
            def spy(ctx, layers):
                if torch.cuda.is_current_stream_capturing():
                    seen.append(gc.isenabled())
                return plain_forward(ctx, layers)
            eng.model.forward = spy
        nxt = 7
        for _ in range(steps):
            nxt = int(eng.step([("r", [nxt], [0])])[0].argmax())
        eng.end_request("r")
        return nxt

    gc.collect()
    gc.disable()
    try:
        first = Engine(folder, dtype="bfloat16", max_tokens=256, max_seqs=2)
        want = decode(first, 5)
        assert first.decode_graphs.replays >= 3
        gone, graphs_gone = weakref.ref(first), weakref.ref(first.decode_graphs)
        del first
        assert gone() is None and graphs_gone() is None, "engine and graphs must not keep each other alive"
    finally:
        gc.enable()
    seen = []
    second = Engine(folder, dtype="bfloat16", max_tokens=256, max_seqs=2)
    assert decode(second, 5, seen) == want
    assert seen and not any(seen), "the collector was on during a capture"
    assert gc.isenabled()
