"""The expansion step of the tree sampler on the device (multi-draw top-k sampler, unique / fork bookkeeping) against the
oracle's restatement of mcts.py:115-152, and the whole search loop against a host loop that does the same bookkeeping
with the oracle and forks by copying K/V rows."""
import pytest
import torch

from oracle import q40_oracle as O

pytestmark = pytest.mark.gpu


def test_multi_draw_sampler_matches_oracle_and_single_draws():
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(80)
    logits = (torch.randn((5, 32016), generator=g) * 2).half()
    counts = torch.tensor([3, 0, 40, 1, 6], dtype=torch.int32)
    u = torch.rand(50, generator=g)
    got = K.sample_topk_counts(logits.cuda(), 0.3, 32, counts.cuda(), u.cuda()).cpu()
    want = O.sample_topk_counts(logits, 0.3, 32, counts.tolist(), u)
    assert torch.equal(got, want)
    # the same draws one row at a time through the single-draw kernel
    rows = torch.repeat_interleave(torch.arange(5), counts.long())
    single = K.sample_topk(logits[rows].cuda(), 0.3, 32, uniform=u.cuda()).cpu()
    assert torch.equal(got, single)


def test_counts_beyond_the_buffers_are_cut():
    """counts that add up to more than uniform / out hold: the draws that fit are made, nothing is written past them;
    the bookkeeping kernel likewise ignores draws its buffer does not hold and a branch counter outside the batch"""
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(82)
    logits = (torch.randn((4, 4096), generator=g) * 2).half()
    counts = torch.tensor([6, 9, 30, 5], dtype=torch.int32)
    u = torch.rand(50, generator=g)
    full = K.sample_topk_counts(logits.cuda(), 0.7, 16, counts.cuda(), u.cuda()).cpu()
    out = torch.full((40,), -1, dtype=torch.int64, device="cuda:0")
    K.sample_topk_counts(logits.cuda(), 0.7, 16, counts.cuda(), u[:20].contiguous().cuda(), out=out)
    assert torch.equal(out[:20].cpu(), full[:20]) and bool((out[20:] == -1).all())
    # bookkeeping: 4 branches want 50 draws, the buffer holds 8 (6 of branch 0, 2 of branch 1); curr_b says 9 of a batch of 6
    draws = full[:8].contiguous().cuda()
    oc = torch.zeros((2, 6), dtype=torch.int32)
    oc[1, :4] = counts
    oc_d = oc.cuda()
    alive = torch.ones(6, dtype=torch.bool, device="cuda:0")
    curr = torch.tensor([9], dtype=torch.int32, device="cuda:0")
    results = torch.zeros((6, 4), dtype=torch.int64, device="cuda:0")
    K.tree_fork(draws, oc_d, alive, curr, results, 0)
    assert 1 <= int(curr) <= 6
    assert int(results[0, 0]) == int(full[:6].min())              # branch 0 keeps its smallest distinct draw


@pytest.mark.parametrize("big", [(1, 2**31 - 1), (2**31 - 1, 2**31 - 1, 7), (2**30, 2**30, 2**30, 2**30, 2**30), (-5, 3, -2**31, 2**31 - 1, 2**31 - 1)])
@pytest.mark.parametrize("row_temps", [False, True])
def test_counts_whose_sum_passes_32_bits_are_cut(big, row_temps):
    """the rows' offsets are sums of counts cut at the buffer, so a sum beyond 2^31 (or 2^32) makes no draw outside it; the draws that
    fit are those of counts cut on the host"""
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(83)
    n, rows = 12, 70                                              # (more rows than lanes: a lane adds two counts)
    logits = (torch.randn((rows, 4096), generator=g) * 2).half()
    counts = torch.tensor(list(big) + [2**31 - 1] * (rows - len(big)), dtype=torch.int32)
    left, cut = n, []
    for c in counts.tolist():
        cut.append(min(max(c, 0), left))
        left -= cut[-1]
    u = torch.rand(n, generator=g)
    temp = torch.full((rows,), 0.7).cuda() if row_temps else 0.7
    want = K.sample_topk_counts(logits.cuda(), temp, 16, torch.tensor(cut, dtype=torch.int32).cuda(), u.cuda()).cpu()
    buf = torch.full((3 * n,), -1, dtype=torch.int64, device="cuda:0")
    K.sample_topk_counts(logits.cuda(), temp, 16, counts.cuda(), u.cuda(), out=buf[n:2 * n])
    assert torch.equal(buf[n:2 * n].cpu(), want)
    assert bool((buf[:n] == -1).all()) and bool((buf[2 * n:] == -1).all())


def test_row_temperature_sampler_matches_oracle():
    """The sampler's temp <= 0 mode: one temperature per branch, quotients and probabilities in float32."""
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(81)
    logits = (torch.randn((6, 32016), generator=g) * 2).half()
    counts = torch.tensor([5, 1, 0, 30, 2, 12], dtype=torch.int32)
    temps = O.ramp_temperature(-0.9, 50, counts)
    assert temps.dtype == torch.float32 and float(temps[1]) == pytest.approx(0.1) and float(temps.max()) < 0.9
    u = torch.rand(50, generator=g)
    got = K.sample_topk_counts(logits.cuda(), temps.cuda(), 32, counts.cuda(), u.cuda()).cpu()
    want = O.sample_topk_counts(logits, temps, 32, counts.tolist(), u)
    assert torch.equal(got, want)
    # one temperature for all rows, a power of two (the fp16 quotient is exact): the float32 mode draws what the fp16 mode
    # draws wherever the fp16 rounding of the probabilities does not move a boundary across the uniform number
    flat = torch.full((6,), 0.5)
    a = K.sample_topk_counts(logits.cuda(), flat.cuda(), 32, counts.cuda(), u.cuda()).cpu()
    b = K.sample_topk_counts(logits.cuda(), 0.5, 32, counts.cuda(), u.cuda()).cpu()
    assert int((a != b).sum()) <= 1


@pytest.mark.parametrize("seed", range(8))
def test_tree_fork_kernel_matches_oracle(seed):
    """random trees: random multiplicities that sum to the batch size, a few dead branches, few distinct tokens (many
    duplicates) or many (rows run out), with and without a page table"""
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(900 + seed)
    B = int(torch.randint(1, 120, (1,), generator=g))
    steps, t = 7, int(torch.randint(0, 7, (1,), generator=g))
    cur = int(torch.randint(1, B + 1, (1,), generator=g))
    # multiplicities: cur positive integers that sum to B
    cuts = torch.sort(torch.randperm(B - 1, generator=g)[: cur - 1] + 1).values.tolist() if B > 1 else []
    cnt = [b - a for a, b in zip([0] + cuts, cuts + [B])]
    oc = torch.zeros((2, B), dtype=torch.int32)
    oc[1, :cur] = torch.tensor(cnt, dtype=torch.int32)
    oc[0, :cur] = torch.randint(0, 1000, (cur,), generator=g, dtype=torch.int32)
    vocab = 3 if seed % 2 == 0 else 32016
    draws = torch.randint(0, vocab, (B,), generator=g)
    alive = torch.rand(B, generator=g) > 0.2
    results = torch.zeros((B, steps), dtype=torch.int64)
    results[:cur, :t] = torch.randint(1, 32016, (cur, t), generator=g)
    use_pages = seed % 3 != 0
    Smax = 9
    pages = (torch.arange(B * Smax, dtype=torch.int32).view(B, Smax) * 7 % 1000) if use_pages else None
    n_rows = min(t, Smax)
    want_oc, want_res, want_pages = oc.clone(), results.clone(), pages.clone() if use_pages else None
    want_cur, want_origin = O.tree_fork(draws, want_oc, alive, cur, B, want_res, t, want_pages, n_rows)
    d_oc, d_res, d_cur = oc.cuda(), results.cuda(), torch.tensor([cur], dtype=torch.int32).cuda()
    d_pages = pages.cuda() if use_pages else None
    origin = K.tree_fork(draws.cuda(), d_oc, alive.cuda(), d_cur, d_res, t, pages=d_pages, n_rows=n_rows)
    assert int(d_cur) == want_cur
    assert origin.cpu().tolist() == want_origin
    assert torch.equal(d_oc.cpu(), want_oc)
    assert torch.equal(d_res.cpu(), want_res)
    if use_pages:
        assert torch.equal(d_pages.cpu(), want_pages)


CFG = dict(dim=256, n_layers=2, n_heads=2, vocab_size=320, multiple_of=128, max_batch_size=12, max_seq_len=10, max_prompt_seq_len=16)


def _temperature(temp, batch_size, counts):
    return temp if temp > 0.0 else O.ramp_temperature(temp, batch_size, counts)


def _host_search(model, prompt, batch_size, depth, top_k, temp, uniforms):
    """The reference's search loop (mcts.py:67-182) with the oracle's bookkeeping on the host and row-copy forks."""
    from spec_mcts_amd import kernels as K
    model.resetSeq()
    steps = min(depth, model.params.max_seq_len)
    results = torch.zeros((batch_size, steps), dtype=torch.int64)
    alive = torch.ones(batch_size, dtype=torch.bool)
    oc = torch.zeros((2, batch_size), dtype=torch.int32)
    oc[1, 0] = batch_size
    state = torch.zeros(batch_size, dtype=torch.int32)
    results_len = torch.zeros(batch_size, dtype=torch.int32)
    terminal = torch.tensor((29961, 29914, 20055, 4690, 1164, 29962))
    cur, pos, stats = 1, 0, []
    for t in range(steps):
        if pos == 0:
            logits = model(prompt.cuda(), 0)
            pos = prompt.shape[1]
        else:
            logits = model(results[:cur, t - 1:t].cuda(), pos)
            pos += 1
        # (the draws come from the device sampler, held against the oracle's in the test above: a probability on a rounding
        # boundary must not decide whether the two LOOPS agree)
        tt = _temperature(temp, batch_size, oc[1])
        draws = K.sample_topk_counts(logits[:, -1].contiguous(), tt.cuda() if isinstance(tt, torch.Tensor) else tt, top_k, oc[1].cuda(), uniforms[t].cuda()).cpu()
        new_cur, origin = O.tree_fork(draws, oc, alive, cur, batch_size, results, t)
        r = cur
        while r < new_cur:                                   # consecutive new rows of one origin = one model.fork call
            n = 1
            while r + n < new_cur and origin[r + n] == origin[r]:
                n += 1
            model.fork(origin[r], r, n)
            r += n
        cur = new_cur
        ends, state = O.detect_terminal(results[:, t], state, terminal, 2)
        results_len += alive.int()
        alive = ~(ends | ~alive)
        stats.append(cur)
        if int((~alive).sum()) == cur:
            return results[:cur, :t + 1], results_len, stats
    return results[:cur], results_len, stats


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("seed,temp", [(0, 0.8), (1, 1.5), (2, 3.0), (3, -2.5)])
def test_device_search_equals_host_search(seed, temp, use_graph):
    """mcts.search on the device (decode steps replayed from per-bucket HIP graphs, or issued launch by launch) against the
    reference's loop with host bookkeeping, row-copy forks and plain model(tokens, pos) calls, on the same uniform numbers:
    the same tokens, lengths and branch counts, bit for bit."""
    from spec_mcts_amd import ModelArgs
    from spec_mcts_amd.load_q40 import load_q40
    from spec_mcts_amd.mcts import mcts
    sd = O.random_q40_state_dict(O.OracleArgs(**CFG), seed=60 + seed, std=0.05)
    dev_model = load_q40(dict(sd), ModelArgs(**CFG))
    host_model = load_q40(dict(sd), ModelArgs(**CFG))
    host_model.paged_kv = False                                # forks copy K/V rows, as the reference's do
    prompt = torch.randint(0, CFG["vocab_size"], (1, 9), generator=torch.Generator().manual_seed(seed))
    B, depth = 12, 8
    tree = mcts(dev_model, depth, top_k=8, temp=temp)
    tree.use_graph = use_graph
    tree.generator = torch.Generator(device="cuda:0").manual_seed(1234 + seed)
    res, res_len, stats = tree.search(prompt, B)
    assert tree.last_replays == (tree.last_steps if use_graph else 0)
    assert int(tree.last_counts[1].sum()) == B
    # the same uniform numbers, step by step, for the host loop
    gen = torch.Generator(device="cuda:0").manual_seed(1234 + seed)
    uniforms = [torch.rand(B, device="cuda:0", dtype=torch.float32, generator=gen).cpu() for _ in range(depth)]
    want, want_len, want_stats = _host_search(host_model, prompt, B, depth, 8, temp, uniforms)
    assert stats.cpu().tolist() == want_stats
    assert torch.equal(res.cpu(), want)
    assert torch.equal(res_len.cpu(), want_len)
    assert want_stats[-1] > 1, "the tree did not branch: the test would not exercise the fork"
    # every row's history up to its fork point is its ancestor's: rows share first tokens
    assert int((res[:, 0] == res[0, 0]).sum()) >= 1
    if use_graph:
        # a second search on the same object replays the graphs captured by the first (same prompt length): same result
        tree.generator = torch.Generator(device="cuda:0").manual_seed(1234 + seed)
        res2, res_len2, stats2 = tree.search(prompt, B)
        assert torch.equal(res2, res) and torch.equal(res_len2, res_len) and torch.equal(stats2, stats)


def test_row_temperature_that_is_not_positive_draws_the_largest_logit():
    """a ramp that reaches 0 (or a NaN) has no softmax: the row returns its argmax for every draw, the other rows are unaffected"""
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(5)
    logits = torch.randn((4, 500), generator=g).half().cuda()
    counts = torch.tensor([3, 2, 4, 1], dtype=torch.int32).cuda()
    u = torch.rand(10, generator=g).cuda()
    temps = torch.tensor([0.7, 0.0, float("nan"), -1.0]).cuda()
    good = torch.tensor([0.7, 0.7, 0.7, 0.7]).cuda()
    got = K.sample_topk_counts(logits, temps, 8, counts, u).cpu()
    ref = K.sample_topk_counts(logits, good, 8, counts, u).cpu()
    top = logits.float().argmax(1).cpu()
    assert torch.equal(got[:3], ref[:3])
    assert got[3:5].tolist() == [int(top[1])] * 2 and got[5:9].tolist() == [int(top[2])] * 4 and got[9:].tolist() == [int(top[3])]


@pytest.mark.parametrize("seed", range(4))
def test_tree_fork_first_step_of_a_wide_search(seed):
    """the first step: one branch owns all batch_size draws (up to 1024), the case the workgroup-wide sort is for; and a
    later step with many branches, empty segments and dead branches"""
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(300 + seed)
    for B, cur, hot in ((1024, 1, 40), (777, 1, 3), (1000, 37, 12)):
        steps = 6
        results = torch.randint(1, 1000, (B, steps), generator=g)
        oc = torch.zeros((2, B), dtype=torch.int32)
        if cur == 1:
            oc[1, 0] = B
        else:
            cut = torch.sort(torch.randint(0, B + 1, (cur - 1,), generator=g)).values
            edges = torch.cat((torch.tensor([0]), cut, torch.tensor([B])))
            oc[1, :cur] = (edges[1:] - edges[:-1]).int()                 # some multiplicities are 0
        alive = torch.ones(B, dtype=torch.bool)
        if cur > 1:
            alive[torch.randint(0, cur, (5,), generator=g)] = False
        n = int(oc[1, :cur].sum())
        draws = torch.randint(0, hot, (n,), generator=g)
        t = 3
        want_oc, want_res = oc.clone(), results.clone()
        want_cur, want_origin = O.tree_fork(draws, want_oc, alive, cur, B, want_res, t)
        d_oc, d_res, d_cur = oc.cuda(), results.cuda(), torch.tensor([cur], dtype=torch.int32).cuda()
        origin = K.tree_fork(draws.cuda(), d_oc, alive.cuda(), d_cur, d_res, t)
        assert int(d_cur) == want_cur
        assert origin.cpu().tolist() == want_origin
        assert torch.equal(d_oc.cpu(), want_oc)
        assert torch.equal(d_res.cpu(), want_res)


@pytest.mark.parametrize("B", [200, 255, 256, 257, 300])
@pytest.mark.parametrize("huge", [False, True])
def test_tree_step_on_either_side_of_the_small_batch_kernel(B, huge):
    """Batches (and draws) of up to 256 take the one kernel, larger ones the other: both against the oracle, with rows that run out.
    huge: the last live branch's multiplicity is 2^31 - 1, of which the draws that the buffer holds exist."""
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(1700 + B)
    cur, steps, t = B // 3, 5, 3
    cuts = torch.sort(torch.randperm(B - 1, generator=g)[: cur - 1] + 1).values.tolist()
    cnt = [b - a for a, b in zip([0] + cuts, cuts + [B])]
    oc = torch.zeros((2, B), dtype=torch.int32)
    oc[1, :cur] = torch.tensor(cnt, dtype=torch.int32)
    draws = torch.randint(0, 40, (B,), generator=g)
    alive = torch.rand(B, generator=g) > 0.1
    alive[cur - 1] = True
    results = torch.zeros((B, steps), dtype=torch.int64)
    results[:cur, :t] = torch.randint(1, 32016, (cur, t), generator=g)
    want_oc, want_res = oc.clone(), results.clone()
    want_cur, want_origin = O.tree_fork(draws, want_oc, alive, cur, B, want_res, t, None, 0)
    d_oc = oc.clone()
    if huge:
        d_oc[1, cur - 1] = 2**31 - 1
    d_oc, d_res, d_cur = d_oc.cuda(), results.cuda(), torch.tensor([cur], dtype=torch.int32).cuda()
    origin = K.tree_fork(draws.cuda(), d_oc, alive.cuda(), d_cur, d_res, t)
    assert int(d_cur) == want_cur and origin.cpu().tolist() == want_origin
    assert torch.equal(d_oc.cpu(), want_oc) and torch.equal(d_res.cpu(), want_res)


@pytest.mark.parametrize("cur", [1, 15, 16, 17, 63, 64, 65, 128, 129])
def test_tree_fork_of_branches_without_draws(cur):
    """Branches with no draws or less than none between the others, at the edges of the rows and the waves of the prefix sums: the one kernel's draws go to
    the branches that the other kernel (more than 256 rows) gives them to"""
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(cur)
    cnt = torch.randint(-2, 4, (cur,), generator=g).to(torch.int32)
    cnt[cur - 1] = 3
    n = int(cnt.clamp(min=0).sum())
    draws = torch.randint(0, 5, (n,), generator=g).cuda()
    res = []
    for B in (256, 300):
        oc = torch.zeros((2, B), dtype=torch.int32)
        oc[1, :cur] = cnt
        results = torch.zeros((B, 6), dtype=torch.int64)
        results[:cur] = torch.arange(cur * 6).view(cur, 6)
        alive = torch.ones(B, dtype=torch.bool)
        alive[cur // 2] = cur < 3
        d_oc, d_res, d_cur = oc.cuda(), results.cuda(), torch.tensor([cur], dtype=torch.int32).cuda()
        origin = K.tree_fork(draws, d_oc, alive.cuda(), d_cur, d_res, 2)
        assert cur <= int(d_cur) <= 256
        res.append((int(d_cur), origin.cpu()[:256], d_oc.cpu()[:, :256], d_res.cpu()[:256]))
    assert res[0][0] == res[1][0] and all(torch.equal(a, b) for a, b in zip(res[0][1:], res[1][1:]))
