"""fused_moe_bf16 on the GPU vs the fp32 CPU oracle on identical seeded inputs.
Gate: max |got - ref| / max(|ref|, 1) <= 2e-2."""
import math

import pytest
import torch

from helpers import BF16_GATE, oracle_schedule, reference_routing, rel_clamp
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu


def _inputs(T, K, E, N, device, seed, x_std=1.0):
    g = torch.Generator(device=device).manual_seed(seed)
    x = (torch.randn((T, K), device=device, generator=g) * x_std).to(torch.bfloat16)
    w1 = (torch.randn((E, N, K), device=device, generator=g) / math.sqrt(K)).to(torch.bfloat16)
    w2 = (torch.randn((E, K, N // 2), device=device, generator=g) / math.sqrt(N // 2)).to(torch.bfloat16)
    return g, x, w1, w2


def _run_case(T, K, E, N, top_k, split, device, seed=0, use_op_align=True, exact=False, hot_last=True,
              prefill_out=None):
    import prime_moe
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed)
    ids, wts = reference_routing(T, E, top_k, device, g, hot_last=hot_last)
    if use_op_align:
        sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    else:
        sched = oracle_schedule(ids, E, 128, exact=exact)
    if prefill_out is None:
        out = torch.zeros((T, K), dtype=torch.bfloat16, device=device) if not split else \
            torch.full((T, K), float("nan"), dtype=torch.bfloat16, device=device)
    else:
        out = prefill_out.clone()
    ret = prime_moe.fused_moe_bf16(x, w1, w2, *sched, wts, out, top_k, 128, 64, 4, 2, 1, 1, split)
    torch.cuda.synchronize()
    assert ret is out
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())
    if prefill_out is not None and not split:
        ref = ref + prefill_out.float().cpu()
    got = out.float().cpu()
    assert torch.isfinite(got).all()
    err = rel_clamp(got, ref, 1.0)
    assert err <= BF16_GATE, f"rel_clamp_1 {err:.4g} > {BF16_GATE}"
    return err


@pytest.mark.parametrize("split", [True, False])
def test_readme_shape(split, device):
    # T=256 K=4096 E=8 N=512 top_k=4 with top-4 of N(0,1) logits and softmax weights
    import prime_moe
    from prime_moe.workloads import CONFIGS, make_inputs
    cfg = CONFIGS["c1_readme_bf16"]
    inp = make_inputs(cfg, device, seed=1)
    sched = torch.ops.prime_moe.moe_align(inp["topk_ids"], cfg.E, 128, 1)
    out = torch.zeros((cfg.T, cfg.K), dtype=torch.bfloat16, device=device)
    prime_moe.fused_moe_bf16(inp["x"], inp["w1"], inp["w2"], *sched, inp["topk_weights"], out, cfg.top_k,
                             128, 64, 4, 2, 1, 1, split)
    torch.cuda.synchronize()
    ref = O.fused_moe_dense(inp["x"].cpu(), inp["w1"].cpu(), inp["w2"].cpu(), inp["topk_ids"].cpu(),
                            inp["topk_weights"].cpu())
    err = rel_clamp(out.float().cpu(), ref, 1.0)
    assert err <= BF16_GATE, err


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("T,K,E,N", [
    (8, 4096, 257, 256), (32, 7168, 8, 512), (128, 4096, 37, 256), (256, 7168, 37, 512),
    (200, 1024, 8, 768), (1, 128, 1, 256), (130, 384, 3, 256),
])
def test_reference_sweep_shapes(T, K, E, N, split, device):
    # the reference's own sweep grid (test/test.py:133-146), top_k = 9 with a hot last expert,
    # plus ragged cases: K % 256 == 128, a single token, one expert
    top_k = 9 if E > 1 else 1
    _run_case(T, K, E, N, top_k, split, device, seed=T + E)


@pytest.mark.parametrize("split", [True, False])
def test_exact_size_schedule_from_python_restatement(split, device):
    _run_case(64, 1024, 8, 512, 4, split, device, use_op_align=False, exact=True)
    _run_case(64, 1024, 8, 512, 4, split, device, use_op_align=False, exact=False)


def test_split_overwrites_and_fused_accumulates(device):
    T, K = 96, 512
    pre = torch.randn((T, K), device=device).to(torch.bfloat16)
    _run_case(T, K, 4, 256, 2, True, device, prefill_out=pre, hot_last=False)   # overwritten
    _run_case(T, K, 4, 256, 2, False, device, prefill_out=pre, hot_last=False)  # added to


def test_tokens_beyond_m_are_dropped(device):
    import prime_moe
    T, K, E, N, top_k = 64, 512, 4, 256, 2
    g, x, w1, w2 = _inputs(T, K, E, N, device, 3)
    ids, wts = reference_routing(T, E, top_k, device, g, hot_last=False)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    keep = 40  # x with fewer rows than the schedule refers to: rows of tokens >= keep are skipped
    out = torch.zeros((keep, K), dtype=torch.bfloat16, device=device)
    prime_moe.fused_moe_bf16(x[:keep].contiguous(), w1, w2, *sched, wts, out, top_k, 128, 32, 8, 1, 1, 1, True)
    torch.cuda.synchronize()
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())[:keep]
    assert rel_clamp(out.float().cpu(), ref, 1.0) <= BF16_GATE


def shuffle_runs(s, counts, gen):
    """The rows of every expert's run in another order: what is dropped then leaves holes between live rows."""
    s, at = s.clone(), 0
    for c in counts:
        s[at:at + c] = s[at:at + c][torch.randperm(c, device=s.device, generator=gen)]
        at += (c + 127) // 128 * 128
    return s


@pytest.mark.parametrize("T,K,E,N", [
    (1625, 256, 5, 8192),  # up kernel: 10 row tiles x 32 weight tiles, workgroups go from tile to tile
    (1625, 8192, 5, 256),  # down kernel: likewise; up kernel: deep split
])
def test_tokens_beyond_m_are_dropped_on_tall_tiles(T, K, E, N, device):
    import prime_moe
    top_k, keep = 2, 1000
    assert T * top_k > 32 * E  # the rule of the dispatch: tall tiles
    g, x, w1, w2 = _inputs(T, K, E, N, device, 5)
    ids, wts = reference_routing(T, E, top_k, device, g, hot_last=False)
    s, e, n = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    s = shuffle_runs(s, torch.bincount(ids.flatten(), minlength=E).tolist(), g)
    n_tiles, _ = _tall_plan(x, w1, w2, (s, e, n), wts, torch.empty_like(x), top_k)
    cus = torch.cuda.get_device_properties(device).multi_processor_count
    assert n_tiles * (N // 256 if N > K else K // 256) > cus
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())[:keep]
    # the whole schedule, and the rows that its length names and no more (no padding behind them)
    for length in (s.numel(), int(n[0])):
        torch.empty((32 << 20,), dtype=torch.float32, device=device).fill_(float("nan"))  # dirty the allocator's blocks
        out = torch.empty((keep, K), dtype=torch.bfloat16, device=device)
        prime_moe.fused_moe_bf16(x[:keep].contiguous(), w1, w2, s[:length].contiguous(), e[:length // 128].contiguous(), n, wts,
                                 out, top_k, 128, 32, 8, 1, 1, 1, True)
        torch.cuda.synchronize()
        assert rel_clamp(out.float().cpu(), ref, 1.0) <= BF16_GATE


def test_validation_errors(device):
    import prime_moe
    T, K, E, N, top_k = 16, 256, 2, 256, 2
    g, x, w1, w2 = _inputs(T, K, E, N, device, 0)
    ids, wts = reference_routing(T, E, top_k, device, g, hot_last=False)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    out = torch.zeros((T, K), dtype=torch.bfloat16, device=device)
    ok = dict(top_k=top_k, block_m=128, block_n=64, warp_n=4, stages=2, bpc=1, cpc=1, split=True)

    def call(**kw):
        a = dict(ok)
        a.update(kw)
        prime_moe.fused_moe_bf16(kw.pop("x", x), w1, w2, *sched, kw.pop("wts", wts), kw.pop("out", out),
                                 a["top_k"], a["block_m"], a["block_n"], a["warp_n"], a["stages"], a["bpc"],
                                 a["cpc"], a["split"])

    call()
    for bad in (dict(block_m=64), dict(block_n=64, warp_n=8), dict(stages=0), dict(stages=6),
                dict(stages=5, split=True), dict(bpc=2), dict(cpc=2)):
        with pytest.raises(RuntimeError):
            call(**bad)
    call(stages=5, split=False)
    with pytest.raises(RuntimeError):
        call(x=x.float())
    with pytest.raises(RuntimeError):
        call(out=out.float())
    with pytest.raises(RuntimeError):
        call(wts=wts.double())
    with pytest.raises(RuntimeError):
        call(x=x.t().contiguous().t())
    with pytest.raises(RuntimeError):
        call(x=x[:, :192].contiguous())
    # a tensor that is not on x's GPU is rejected on the host (its pointer never reaches a kernel)
    with pytest.raises(RuntimeError, match="is on cpu"):
        call(wts=wts.cpu())
    with pytest.raises(RuntimeError, match="is on cpu"):
        call(out=out.cpu())
    with pytest.raises(RuntimeError, match="is on cpu"):
        prime_moe.fused_moe_bf16(x, w1, w2, sched[0].cpu(), sched[1], sched[2], wts, out, top_k, 128, 64, 4, 2, 1, 1, True)
    # x starting 2 bytes into an allocation: the 16-byte copies of the loaders would be misaligned
    shifted = torch.empty((T * K + 1,), dtype=torch.bfloat16, device=device)[1:].view(T, K)
    with pytest.raises(RuntimeError, match="aligned"):
        call(x=shifted)


def test_result_is_bitwise_reproducible(device):
    """No atomics anywhere in the pipeline: two calls on the same inputs agree bit for bit."""
    import prime_moe
    g, x, w1, w2 = _inputs(300, 512, 8, 512, device, seed=5)
    ids, wts = reference_routing(300, 8, 4, device, g)
    sched = torch.ops.prime_moe.moe_align(ids, 8, 128, 1)
    outs = []
    for _ in range(3):
        out = torch.empty((300, 512), dtype=torch.bfloat16, device=device)
        prime_moe.fused_moe_bf16(x, w1, w2, *sched, wts, out, 4, 128, 64, 4, 2, 1, 1, True)
        outs.append(out)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


def test_experts_with_one_and_with_several_row_tiles(device):
    # expert 0: 276 rows = a full row tile and a tail of 20 rows that reads the same weight rows; expert 1:
    # 200 rows in one tile of two blocks; expert 2: 56 rows; expert 3: 20 rows, alone on its weight rows
    # (decode-style tile, other cache policy of the weight copies); expert 4: none
    import prime_moe
    from test_gpu_mxfp8 import _routing_by_counts
    counts, top_k = [276, 200, 56, 20, 0], 2
    K, E, N = 1024, 5, 512
    ids, wts = _routing_by_counts(counts, top_k, device, seed=6)
    T = ids.shape[0]
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=22)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    for split in (True, False):
        out = torch.zeros((T, K), dtype=torch.bfloat16, device=device)
        prime_moe.fused_moe_bf16(x, w1, w2, *sched, wts, out, top_k, 128, 64, 4, 2, 1, 1, split)
        torch.cuda.synchronize()
        ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())
        assert rel_clamp(out.float().cpu(), ref, 1.0) <= BF16_GATE


def test_block_without_expert_and_duplicate_pair(device):
    """Schedules the fused op must survive: a block whose expert id is out of range is not computed and
    its pairs contribute nothing (never whatever the workspace held); a pair id listed twice in one block
    contributes once; listed again in a block of another expert, one of the two experts' rows (unspecified
    which) stands for the pair, and nothing faults."""
    import prime_moe
    T, K, E, N, top_k = 300, 512, 6, 512, 2
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=9)
    ids, wts = reference_routing(T, E, top_k, device, g, hot_last=False)
    s, e, n = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    dropped = 1  # second block of the schedule loses its expert
    e_bad = e.clone()
    e_bad[dropped] = -1
    pairs = s[dropped * 128:(dropped + 1) * 128]
    pairs = pairs[pairs >= 0].long()
    w_ref = wts.clone().flatten()
    w_ref[pairs] = 0.0  # the oracle drops the same pairs through their routing weights
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), w_ref.view(T, top_k).cpu())
    for fill in (float("nan"), 1e30):  # whatever an earlier call left in the caching allocator's blocks
        junk = torch.full((64 << 20,), fill, dtype=torch.bfloat16, device=device)
        del junk
        out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
        prime_moe.fused_moe_bf16(x, w1, w2, s, e_bad, n, wts, out, top_k, 128, 64, 4, 2, 1, 1, True)
        torch.cuda.synchronize()
        got = out.float().cpu()
        assert torch.isfinite(got).all()
        assert rel_clamp(got, ref, 1.0) <= BF16_GATE
    # a pair id listed twice (in a padding slot of its own block): counted once
    s_dup = s.clone()
    blk = int((s[:128] < 0).nonzero()[0]) if bool((s[:128] < 0).any()) else None
    if blk is not None:
        s_dup[blk] = s[0]
        ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())
        out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
        prime_moe.fused_moe_bf16(x, w1, w2, s_dup, e, n, wts, out, top_k, 128, 64, 4, 2, 1, 1, True)
        torch.cuda.synchronize()
        assert rel_clamp(out.float().cpu(), ref, 1.0) <= BF16_GATE
    # the same pair id once more in a padding slot of another expert's block: two workgroups write y[pair]; the
    # result for that token is one of the two candidates, the rest of the output is untouched
    other = [b for b in range(1, int(n[0]) // 128) if int(e[b]) != int(e[0]) and bool((s[b * 128:(b + 1) * 128] < 0).any())]
    if other:
        b = other[0]
        slot = b * 128 + int((s[b * 128:(b + 1) * 128] < 0).nonzero()[0])
        s_far = s.clone()
        s_far[slot] = s[0]
        ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())
        out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
        prime_moe.fused_moe_bf16(x, w1, w2, s_far, e, n, wts, out, top_k, 128, 64, 4, 2, 1, 1, True)
        torch.cuda.synchronize()
        got = out.float().cpu()
        assert torch.isfinite(got).all()
        tok = int(s[0]) // top_k
        keep = torch.ones(T, dtype=torch.bool)
        keep[tok] = False
        assert rel_clamp(got[keep], ref[keep], 1.0) <= BF16_GATE


def _takes_deep(pairs, E, blocks, K, N):
    """The rules of the dispatch, on 256 CUs."""
    n_wt = N // 256
    if K < 2048 or blocks > 64 or blocks * n_wt > 128:
        return False
    if blocks * n_wt <= 32:
        return pairs > 32 * E
    return pairs > (64 if K < 4096 or n_wt > 2 else 34 if 3 * E * N * K >= 112e6 else 48) * E


@pytest.mark.parametrize("T,K,E,N,top_k,exact,deep", [
    (256, 4096, 8, 512, 4, False, True),    # the README shape: 8 - 16 row tiles x 2 weight tiles, every tile split 8 ways
    (100, 2048, 4, 256, 2, False, True),    # one weight tile, tiles of two to four fragments
    (130, 6144, 3, 512, 3, True, True),     # exact-size schedule, a second block with two live rows
    (33, 2048, 1, 256, 1, False, True),     # one weight tile, a second fragment with one live row
    (300, 2176, 2, 1024, 2, False, True),   # 17 slabs: parts of unequal length
    (700, 4096, 8, 512, 4, False, True),    # 30 blocks x 2: tiles of two pairs of fragments
    (180, 4096, 37, 256, 9, False, True),   # 50 blocks, a fragment or two each
    (900, 2304, 2, 2048, 1, True, True),    # exact-size schedule, 8 weight tiles
    (40, 2048, 4, 256, 2, False, False),    # up to 32 rows per expert: the streaming kernels, no deep split
    (1, 2048, 1, 256, 1, False, False),     # one row, likewise
])
def test_few_jobs_deep_split_and_join_kernel(T, K, E, N, top_k, exact, deep, device):
    """Few up jobs for the chip and a long contraction: every up tile is split over up to 8 workgroups that
    only store their partial sums, and a kernel of its own joins them and applies SwiGLU.  Against the
    oracle, and bit for bit the same on a second call (the join adds the parts in part order)."""
    import prime_moe
    n_blocks = (T * top_k + E * 127 + 127) // 128
    assert deep == _takes_deep(T * top_k, E, n_blocks, K, N)
    for split in (True, False):
        _run_case(T, K, E, N, top_k, split, device, seed=T + K, use_op_align=not exact, exact=exact, hot_last=False)
    g, x, w1, w2 = _inputs(T, K, E, N, device, T + K)
    ids, wts = reference_routing(T, E, top_k, device, g, hot_last=False)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    if deep:
        plan = _prologue_workspace(x, w1, w2, sched, wts, torch.empty_like(x), top_k)[:16].view(torch.int32).tolist()
        assert plan[1] >= 2 and plan[3] == 1  # (row tiles, parts, split jobs, deep) of the up kernel
    outs = []
    for _ in range(2):
        torch.empty((32 << 20,), dtype=torch.float32, device=device).fill_(float("nan"))  # dirty the allocator's blocks
        out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
        prime_moe.fused_moe_bf16(x, w1, w2, *sched, wts, out, top_k, 128, 64, 4, 2, 1, 1, True)
        outs.append(out)
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.parametrize("K,N,counts", [
    (2048, 256, [40] * 9 + [1, 0, 63, 64, 65, 127, 128, 129, 0, 33]),  # 28 blocks: most runs a block long, some experts without rows
    (2304, 768, [385, 3]),                                            # a run of four blocks with one row in the last, two tiles
    (4096, 512, [0, 700, 0]),                                         # two runs of six blocks
    (4096, 256, [48] * 24 + [1, 0, 63, 64, 65, 127, 128, 129, 0, 33, 200, 257]),  # 57 blocks, 41 of them live, most runs a block long
    (2304, 512, [385, 900, 3, 2300, 700]),                            # 58 blocks x 2, runs of up to 18
])
def test_deep_up_kernel_cuts_and_plans(K, N, counts, device):
    """The tiles that every workgroup of the deep up kernel works out for itself: also with tokens beyond M (holes in a block),
    a block of an expert that does not exist and a schedule cut behind its last pair."""
    from test_gpu_mxfp8 import _routing_by_counts
    import prime_moe
    E, top_k = len(counts) + 1, 2
    counts = counts + [max(counts) + sum(counts + [max(counts)]) % 2]  # (no expert has more rows than there are tokens)
    ids, wts = _routing_by_counts(counts, top_k, device, seed=K)
    T = ids.shape[0]
    keep = T - T // 8
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=N)
    s, e, n = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    last = int((s >= 0).nonzero().max()) + 1
    assert _takes_deep(T * top_k, E, s.numel() // 128, K, N) and _takes_deep(keep * top_k, E, (last + 127) // 128, K, N)
    e_bad = e.clone()
    e_bad[1] = E + 3
    w_ref = wts.clone()
    lost = s[128:256]
    w_ref.view(-1)[lost[lost >= 0].long()] = 0.0
    for e_, w_, m, length in ((e, wts, T, s.numel()), (e_bad, w_ref, keep, last)):
        ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), w_.cpu())[:m]
        torch.empty((32 << 20,), dtype=torch.float32, device=device).fill_(float("nan"))  # dirty the allocator's blocks
        out = torch.empty((m, K), dtype=torch.bfloat16, device=device)
        prime_moe.fused_moe_bf16(x[:m].contiguous(), w1, w2, s[:length].contiguous(), e_, n, wts, out, top_k, 128, 64, 4, 2, 1, 1, True)
        torch.cuda.synchronize()
        got = out.float().cpu()
        assert torch.isfinite(got).all() and rel_clamp(got, ref, 1.0) <= BF16_GATE


def _deep_cut(f2, K, N, device):
    """(tiles, parts) of the up kernel in deep mode, of runs with f2 pairs of fragments each."""
    cus = torch.cuda.get_device_properties(device).multi_processor_count // 8 * 8
    pairs, n_wt = sum(f2), N // 256
    tiles = pairs if pairs <= 64 and pairs * n_wt * 8 <= cus else sum((f + 1) // 2 for f in f2)
    return tiles, max(1, min(8, K // 64 // 4, cus // (tiles * n_wt), 1024 // (2 * pairs * n_wt)))


@pytest.mark.parametrize("K,N,counts", [
    (2048, 512, [193, 512, 130, 126]),         # 4 + 8 + 3 + 2 = 17 pairs of fragments x 2 weight tiles: one more than tiles of one pair
    (2048, 512, [192, 512, 130, 126]),         # 16: the most that tiles of one pair take
    (2048, 256, [64] * 10 + [700, 640, 65]),   # 33 pairs x 1
    (4096, 256, [64] * 10 + [700, 640]),       # 31 pairs x 1
    (2304, 1024, [300, 129]),                  # 8 pairs x 4: as many as there is room for; a share of 4 or 5 slabs
    (2048, 1280, [321, 63]),                   # 7 pairs x 5: one tile of two pairs and a single one
    (2048, 512, [8065]),                       # 64 blocks, the most, x 2: two parts each, as many sums as the workspace holds
    (2048, 512, [8066]),                       # 65: the resident kernel
    (2304, 256, [4000, 3, 1500, 129, 64]),     # 49 blocks: five parts of 7 or 8 slabs
    (2048, 2048, [700, 600, 200]),             # 15 blocks x 8
    (2048, 2048, [700, 600, 367]),             # 16 blocks x 8: the most pairs
    (2048, 2048, [700, 600, 368]),             # 17 x 8: the resident kernel
])
def test_deep_up_kernel_tiles_of_one_pair_and_two(K, N, counts, device):
    """The edge between tiles of one pair of fragments and of two (256 CUs: pairs x weight tiles x 8 parts), against the oracle."""
    import prime_moe
    E = len(counts)
    ids = torch.repeat_interleave(torch.arange(E, dtype=torch.int32, device=device), torch.tensor(counts, device=device))
    ids = ids[torch.randperm(ids.numel(), generator=torch.Generator().manual_seed(K)).to(device)].view(-1, 1).contiguous()
    T = ids.shape[0]
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=N)
    wts = torch.rand((T, 1), generator=g, device=device)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    blocks = sched[0].numel() // 128
    assert T > 64 * E and K >= 2048  # the rules of the dispatch
    assert (blocks <= 64 and blocks * (N // 256) <= 128) == (counts not in ([8066], [700, 600, 368]))
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())
    plan = _prologue_workspace(x, w1, w2, sched, wts, torch.empty_like(x), 1)[:16].view(torch.int32).tolist()
    if counts not in ([8066], [700, 600, 368]):
        assert (plan[0], plan[1], plan[3]) == (*_deep_cut([(c + 63) // 64 for c in counts], K, N, device), 1)
    else:
        assert plan[3] == 0
    out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
    prime_moe.fused_moe_bf16(x, w1, w2, *sched, wts, out, 1, 128, 64, 4, 2, 1, 1, True)
    torch.cuda.synchronize()
    got = out.float().cpu()
    assert torch.isfinite(got).all() and rel_clamp(got, ref, 1.0) <= BF16_GATE


@pytest.mark.parametrize("counts", [
    [8065],       # 64 blocks, 127 pairs of fragments: the table of the cut has room for 64 tiles
    [4096],       # 64 pairs: all of one pair
    [4097],       # 65
    [65] * 33,    # 33 blocks, 66 pairs
])
def test_deep_up_kernel_on_more_cus_than_its_table_has_tiles(counts, device):
    """From 520 CUs on there would be a workgroup for every part of more tiles of one pair of fragments than the table holds."""
    from prime_moe import _native
    import prime_moe
    K, N, E, lib = 2048, 256, len(counts), _native.load()
    ids = torch.repeat_interleave(torch.arange(E, dtype=torch.int32, device=device), torch.tensor(counts, device=device)).view(-1, 1).contiguous()
    T = ids.shape[0]
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=T)
    wts = torch.rand((T, 1), generator=g, device=device)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    assert 32 < sched[0].numel() // 128 <= 64 and T > 64 * E  # the rules of the dispatch
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())
    for cus in (512, 520, 1024):
        lib.pmoe_set_compute_units(cus)
        try:
            out = torch.full((T, K), float("nan"), dtype=torch.bfloat16, device=device)
            prime_moe.fused_moe_bf16(x, w1, w2, *sched, wts, out, 1, 128, 64, 4, 2, 1, 1, True)
        finally:
            lib.pmoe_set_compute_units(0)
        torch.cuda.synchronize()
        got = out.float().cpu()
        assert torch.isfinite(got).all() and rel_clamp(got, ref, 1.0) <= BF16_GATE, cus


@pytest.mark.parametrize("counts,order", [
    ([0, 700, 0, 700], None),                            # ascending, expert 0 without rows: two runs of six blocks
    ([130, 60, 40, 230], [4, 0, 1, 2, 3, 5]),            # experts 3 0 0 1 2 3: another expert in front of expert 0
    ([130, 60, 40, 230], [2, 0, 4, 1, 5, 3]),            # experts 1 0 3 0 3 2: no expert's blocks side by side
    ([40, 230, 60, 130], [1, 2, 0, 4, 5, 3]),            # experts 1 1 0 3 3 2
    ([900, 1300, 1100, 700, 1300], "any"),               # 45 blocks: neighbours of one expert by chance, short blocks inside a run
    ([60] * 30 + [900, 900], "any"),                     # 46
])
def test_deep_up_kernel_takes_blocks_in_any_order(counts, order, device):
    """expert_ids says which expert a block belongs to, in whatever order the blocks come; neighbours of one expert are one run."""
    from test_gpu_mxfp8 import _routing_by_counts
    import prime_moe
    K, N, E, top_k = 2048, 256, len(counts), 2
    ids, wts = _routing_by_counts(counts, top_k, device, seed=sum(counts))
    T = ids.shape[0]
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=N)
    s, e, n = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    assert _takes_deep(T * top_k, E, s.numel() // 128, K, N)
    n_live = int(n[0]) // 128
    if order == "any":
        order = torch.randperm(n_live, generator=torch.Generator().manual_seed(E)).tolist()
    if order is not None:
        assert len(order) == n_live
        s, e = s.clone(), e.clone()
        s.view(-1, 128)[:n_live] = s.view(-1, 128)[order]
        e[:n_live] = e[order]
    # pairs of fragments of every run: whole blocks and the rows of the last one
    f2, exp, rows = [], e[:n_live].tolist(), (s.view(-1, 128)[:n_live] >= 0).sum(1).tolist()
    for b in range(n_live):
        if b == 0 or exp[b] != exp[b - 1]:
            start = b
        if b + 1 == n_live or exp[b + 1] != exp[b]:
            f2.append((128 * (b - start) + rows[b] + 63) // 64)
    ws = _prologue_workspace(x, w1, w2, (s, e, n), wts, torch.empty_like(x), top_k)
    plan = ws[:36].view(torch.int32).tolist()
    assert (plan[0], plan[1]) == _deep_cut(f2, K, N, device) and plan[3] == 1  # the up kernel's tiles and parts, deep
    assert plan[8] == 2 * sum(f2)                                     # fragments
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())
    out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
    prime_moe.fused_moe_bf16(x, w1, w2, s, e, n, wts, out, top_k, 128, 64, 4, 2, 1, 1, True)
    torch.cuda.synchronize()
    got = out.float().cpu()
    assert torch.isfinite(got).all() and rel_clamp(got, ref, 1.0) <= BF16_GATE


@pytest.mark.parametrize("K,E,N,rows", [
    (4096, 37, 256, 34),   # 116 MB of weights, more than 32 blocks
    (4096, 16, 512, 48),   # 101 MB
    (2048, 24, 512, 64),   # a shorter contraction
    (4096, 8, 512, 32),    # up to 32 (block, weight tile) pairs
])
@pytest.mark.parametrize("more", [0, 1])
def test_line_between_streaming_and_deep_mode(K, E, N, rows, more, device):
    import prime_moe
    T = rows * E + more
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=E)
    ids, wts = reference_routing(T, E, 1, device, g, hot_last=False)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    assert _takes_deep(T, E, sched[0].numel() // 128, K, N) == bool(more)
    plan = _prologue_workspace(x, w1, w2, sched, wts, torch.empty_like(x), 1)[:16].view(torch.int32).tolist()
    assert plan[3] == more
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())
    out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
    prime_moe.fused_moe_bf16(x, w1, w2, *sched, wts, out, 1, 128, 64, 4, 2, 1, 1, True)
    torch.cuda.synchronize()
    got = out.float().cpu()
    assert torch.isfinite(got).all() and rel_clamp(got, ref, 1.0) <= BF16_GATE


@pytest.mark.parametrize("cus", [8, 16, 24, 40, 64, 256])
def test_few_up_jobs_on_fewer_cus(cus, device):
    """Every job runs, also where there are more of them than workgroups: 16 here (8 experts of one block, 2 weight tiles)."""
    from test_gpu_mxfp8 import _routing_by_counts
    import prime_moe
    from prime_moe import _native
    counts, K, N, top_k = [90, 100, 70, 128, 1, 90, 111, 66], 2048, 512, 2
    E = len(counts)
    ids, wts = _routing_by_counts(counts, top_k, device, seed=cus)
    T = ids.shape[0]
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=cus)
    s, e, n = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    assert T * top_k > 32 * E and s.numel() // 128 * (N // 256) <= 32 and int(n[0]) == 8 * 128  # the rules of the dispatch
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())
    torch.empty((32 << 20,), dtype=torch.float32, device=device).fill_(float("nan"))  # dirty the allocator's blocks
    out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
    try:
        _native.load().pmoe_set_compute_units(cus)
        prime_moe.fused_moe_bf16(x, w1, w2, s, e, n, wts, out, top_k, 128, 64, 4, 2, 1, 1, True)
    finally:
        _native.load().pmoe_set_compute_units(0)
    torch.cuda.synchronize()
    got = out.float().cpu()
    assert torch.isfinite(got).all() and rel_clamp(got, ref, 1.0) <= BF16_GATE


@pytest.mark.parametrize("counts,N,cus", [
    ([65] * 33, 2048, 1024),   # 33 tiles of two pairs of fragments x 8 weight tiles: 264 jobs, a round of 256 and 8
    ([65] * 33, 2048, 512),
    ([400] * 5, 1024, 32),     # 40 jobs: 8 behind a round of 32, 40 behind no round of 256
    ([400] * 5, 1024, 128),    # one round that is not full on either
    ([700] * 5, 2048, 64),     # 80 jobs
    ([700] * 5, 2048, 256),
])
def test_last_round_of_the_resident_kernels_on_other_numbers_of_cus(counts, N, cus, device):
    """The part of the last round that is shared by rows is the one that the walk of the jobs leaves over, on any number of CUs."""
    import prime_moe
    from prime_moe import _native
    K, E, lib = 512, len(counts), _native.load()
    ids = torch.repeat_interleave(torch.arange(E, dtype=torch.int32, device=device), torch.tensor(counts, device=device)).view(-1, 1).contiguous()
    T = ids.shape[0]
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=T)
    wts = torch.rand((T, 1), generator=g, device=device)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    assert T > 64 * E and K < 2048  # the rules of the dispatch: prologue and resident kernels
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())
    torch.empty((32 << 20,), dtype=torch.float32, device=device).fill_(float("nan"))  # dirty the allocator's blocks
    out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
    lib.pmoe_set_compute_units(cus)
    try:
        prime_moe.fused_moe_bf16(x, w1, w2, *sched, wts, out, 1, 128, 64, 4, 2, 1, 1, True)
    finally:
        lib.pmoe_set_compute_units(0)
    torch.cuda.synchronize()
    got = out.float().cpu()
    assert torch.isfinite(got).all() and rel_clamp(got, ref, 1.0) <= BF16_GATE


def _prologue_workspace(x, w1, w2, sched, wts, out, top_k):
    """The workspace after the prologue of the tall-tile path: it starts with the plan, the run list and the table of row
    tiles (bf16_workspace in csrc/fused_moe_bf16.hip)."""
    from prime_moe import _native
    lib = _native.load()
    (M, K), (E, N, _) = x.shape, w1.shape
    s, e, n = sched
    nbytes = lib.pmoe_fused_moe_bf16_workspace_bytes(M, K, N, E, s.numel(), top_k, 1)
    ws = torch.zeros((nbytes,), dtype=torch.uint8, device=x.device)
    try:
        lib.pmoe_set_phase_mask(1)  # the prologue alone
        _native.check(lib.pmoe_fused_moe_bf16(
            x.data_ptr(), w1.data_ptr(), w2.data_ptr(), out.data_ptr(), s.data_ptr(), e.data_ptr(), n.data_ptr(),
            wts.data_ptr(), top_k, M, K, N, E, s.numel(), 128, 64, 4, 2, 1, 1, 1, ws.data_ptr(), nbytes,
            torch.cuda.current_stream().cuda_stream))
    finally:
        lib.pmoe_set_phase_mask(15)
    torch.cuda.synchronize()
    return ws


def _tall_plan(x, w1, w2, sched, wts, out, top_k):
    """(number of row tiles, the up kernel's table of row tiles) that the prologue of the tall-tile path builds."""
    ws = _prologue_workspace(x, w1, w2, sched, wts, out, top_k)
    up = lambda b: (b + 255) // 256 * 256
    at = 256 + up((sched[0].numel() // 128 + 1) * 20)
    n_tiles = int(ws[:4].view(torch.int32)[0])
    return n_tiles, ws[at:at + 16 * n_tiles].view(torch.int32).view(-1, 4)[:, :3].cpu()


@pytest.mark.parametrize("E", [130, 1000, 1024])
def test_row_tiles_of_one_size_keep_their_order(E, device):
    """The place of a row tile decides where the K loops of its jobs start, that is the order of their sums: tiles of
    one size come in the order of the schedule, whichever wave of the prologue is first."""
    from test_gpu_mxfp8 import _routing_by_counts
    K, N, top_k = 128, 256, 2
    counts = [36 if e % 3 else 100 for e in range(E)]  # one and two pairs of fragments
    counts[-1] += sum(counts) % 2
    ids, wts = _routing_by_counts(counts, top_k, device, seed=E)
    T = ids.shape[0]
    assert T * top_k > 32 * E and E >= 128  # the rule of the dispatch: tall tiles
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=E)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
    want = [[4 * e, 2 - (c <= 64), e] for e, c in enumerate(counts)]
    want.sort(key=lambda t: (-t[1], t[0]))
    for _ in range(4):
        n_tiles, tiles = _tall_plan(x, w1, w2, sched, wts, out, top_k)
        assert n_tiles == E
        assert torch.equal(tiles, torch.tensor(want, dtype=torch.int32))


def test_many_tiles_of_one_size_are_bitwise_reproducible(device):
    import prime_moe
    T, K, E, N, top_k = 640, 2048, 128, 512, 8
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=4)
    ids = torch.topk(torch.randn((T, E), device=device, generator=g), top_k).indices.to(torch.int32).contiguous()
    wts = torch.softmax(torch.randn((T, top_k), device=device, generator=g), -1)
    assert T * top_k > 32 * E  # tall tiles
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    first = None
    for _ in range(20):
        out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
        prime_moe.fused_moe_bf16(x, w1, w2, *sched, wts, out, top_k, 128, 64, 4, 2, 1, 1, True)
        first = out if first is None else first
        assert torch.equal(first.view(torch.int16), out.view(torch.int16))
