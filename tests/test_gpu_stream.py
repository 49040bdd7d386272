"""The weight-streaming kernels (few rows per expert, csrc/moe_stream.h and moe_stream_mx.h) at the sizes where they can go wrong:
live rows around the 4-row, 32-row, 64-row and 128-row edges, blocks of one expert that take several passes, one slab
and more slabs than stages, the short-contraction down kernels (H = 128, 256) and the general ones, tiles of one
and of two units of weight rows, and the mxfp8 ring kernels without a work list."""
import pytest
import torch

from helpers import (BF16_GATE, MX_COS_GATE, MX_FLIP_DELTA, MX_RELL2_GATE, cosine, mx_elementwise_gates, rel_clamp,
                     rel_l2)
from oracle import moe_oracle as O
from test_gpu_bf16 import _inputs, shuffle_runs
from test_gpu_mxfp8 import _quantised_inputs, _routing_by_counts

pytestmark = pytest.mark.gpu

EDGES = [1, 4, 5, 31, 32, 33, 63, 64, 65, 96, 97, 128, 129]


@pytest.mark.parametrize("K,N,E,split", [
    (128, 256, 40, True),     # one slab up, H = 128 down
    (384, 512, 40, False),    # three slabs, H = 256 down
    (640, 768, 40, True),     # H = 384: general down kernel, three slabs
    (3072, 256, 40, True),    # more slabs than stages
    (512, 1024, 64, False),   # jobs of two units of weight rows in both kernels
])
def test_stream_kernels_at_row_edges(K, N, E, split, device):
    import prime_moe
    counts = EDGES + [0] * (E - len(EDGES))
    ids, wts = _routing_by_counts(counts, 2, device, seed=K)
    T = ids.shape[0]
    assert 2 * T <= 32 * E  # the rule of the dispatch
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=N)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())
    outs = []
    for _ in range(2):
        torch.empty((32 << 20,), dtype=torch.float32, device=device).fill_(float("nan"))  # dirty the allocator's blocks
        out = torch.zeros((T, K), dtype=torch.bfloat16, device=device)
        prime_moe.fused_moe_bf16(x, w1, w2, *sched, wts, out, 2, 128, 64, 4, 2, 1, 1, split)
        outs.append(out)
    torch.cuda.synchronize()
    got = outs[0].float().cpu()
    assert torch.isfinite(got).all() and rel_clamp(got, ref, 1.0) <= BF16_GATE
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


def test_stream_kernels_with_dropped_rows_and_blocks(device):
    """Holes in a block (tokens beyond M), a block without an expert, a misaligned end of the schedule."""
    import prime_moe
    T, K, E, N, top_k = 24, 256, 6, 512, 2
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=3)
    ids = torch.randint(0, E, (T, top_k), device=device, generator=g, dtype=torch.int32)
    wts = torch.softmax(torch.randn((T, top_k), device=device, generator=g), -1)
    s, e, n = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    keep = 17
    e_bad = e.clone()
    e_bad[1] = E + 3
    w_ref = wts.clone()
    w_ref[ids == int(e[1])] = 0.0
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), w_ref.cpu())[:keep]
    for length in (s.numel(), int(n[0]) - 100):  # (the cut rows are padding of the last block)
        assert bool((s[length:int(n[0])] < 0).all())
        out = torch.empty((keep, K), dtype=torch.bfloat16, device=device)
        prime_moe.fused_moe_bf16(x[:keep].contiguous(), w1, w2, s[:length].contiguous(), e_bad, n, wts, out, top_k,
                                 128, 64, 4, 2, 1, 1, True)
        torch.cuda.synchronize()
        got = out.float().cpu()
        assert torch.isfinite(got).all() and rel_clamp(got, ref, 1.0) <= BF16_GATE


@pytest.mark.parametrize("K,N,E,T,top_k,hot,want", [
    (1024, 768, 246, 1960, 4, 73, 3),    # general down kernel: all pairs on 73 experts, 107 rows each
    (1024, 768, 246, 1960, 4, 246, 0),   # the same call with its pairs spread out
    (1024, 768, 168, 1340, 4, 50, 0),    # crowded, but too small to enqueue the tall kernels
    (2048, 512, 150, 1200, 4, 80, 2),    # short down kernel (H = 256): 60 rows per block crowd it, not the up kernel
    (4096, 256, 150, 1200, 4, 30, 3),    # H = 128, blocks of one expert
    (7168, 512, 60, 60, 32, 1, 2),       # one expert named 32 times by each token: only the tall down kernel is enqueued
])
def test_crowded_schedules_take_the_tall_kernels(K, N, E, T, top_k, hot, want, device):
    """Few rows per expert on average, all of them on few experts: the kernels decide on the device which of them work
    (1: the tall up kernel, 2: the tall down kernel), and whichever did, every pair is computed once."""
    from prime_moe import _native
    lib = _native.load()
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=K)
    perm = torch.randperm(E, device=device, generator=g)[:hot].to(torch.int32)
    pick = torch.randn((T, max(hot, top_k)), device=device, generator=g).topk(top_k).indices % hot
    ids = perm[pick].contiguous()
    wts = torch.softmax(torch.randn((T, top_k), device=device, generator=g), -1)
    assert T * top_k <= 32 * E  # the rule of the dispatch: streaming kernels are enqueued
    s, e, n = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    nbytes = lib.pmoe_fused_moe_bf16_workspace_bytes(T, K, N, E, s.numel(), top_k, 1)
    ws = torch.full((nbytes,), 0xff, dtype=torch.uint8, device=device)
    out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
    _native.check(lib.pmoe_fused_moe_bf16(
        x.data_ptr(), w1.data_ptr(), w2.data_ptr(), out.data_ptr(), s.data_ptr(), e.data_ptr(), n.data_ptr(),
        wts.data_ptr(), top_k, T, K, N, E, s.numel(), 128, 64, 4, 2, 1, 1, 1, ws.data_ptr(), nbytes,
        torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    # the plan of the tall kernels: two descriptions of 16 bytes, then the next slot of every queue (8 up, 8 down)
    up, down = ws[32:96].view(torch.int32).view(2, 8).cpu()
    first = torch.cuda.get_device_properties(device).multi_processor_count // 8
    took = (1 if bool((up > first).any()) else 0) | (2 if bool((down > first).any()) else 0)
    assert took == want
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())
    got = out.float().cpu()
    assert torch.isfinite(got).all() and rel_clamp(got, ref, 1.0) <= BF16_GATE


SPARSE = [129, 65, 64, 33, 32, 5] + [1] * 60


@pytest.mark.parametrize("K,N,E,counts,split", [
    (256, 256, 40, EDGES, True),       # streaming up kernel with one slab, H = 128 down
    (512, 512, 40, EDGES, False),      # H = 256 down
    (2304, 512, 40, EDGES, True),      # more slabs than stages, a last group of turns that is not full
    (256, 2048, 40, EDGES, False),     # ring kernels without a work list
    (256, 768, 256, SPARSE, True),     # general streaming down kernel, H = 384: the last slab has one half
    (1024, 512 + 256, 256, SPARSE, False),  # ring down kernel: two rows a tile, four tiles per CU
    (1024, 512 + 256, 60, [33, 16, 5] + [2] * 40, True),  # general streaming down kernel, up to four rows a tile
    (1024, 512 + 256, 300, [1] * 200, False),             # likewise, a row each and more tiles than CUs
    (2048, 8192, 11, [129, 33, 31, 20, 15, 10, 8, 6, 5, 4, 3], True),  # ring kernels, activation rows of 4 KB: 32 phases of the K walk
])
def test_mx_kernels_without_a_schedule_at_row_edges(K, N, E, counts, split, device):
    import prime_moe
    counts = counts + [0] * (E - len(counts))
    counts[-1] += sum(counts) % 2
    ids, wts = _routing_by_counts(counts, 2, device, seed=K)
    T = ids.shape[0]
    g, a, deq = _quantised_inputs(T, K, E, N, device, seed=N)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    outs = []
    for _ in range(2):
        torch.empty((32 << 20,), dtype=torch.float32, device=device).fill_(float("nan"))  # dirty the allocator's blocks
        out = torch.zeros((T, K), dtype=torch.bfloat16, device=device)
        prime_moe.fused_moe_mxfp8(a["x"], a["x_scales"], a["w1"], a["w1_scales"], a["w2"], a["w2_scales"], *sched, wts,
                                  out, 2, 128, 64, 4, 2, 1, split)
        outs.append(out)
    torch.cuda.synchronize()
    ref, bound = O.fused_moe_dense(deq["x"], deq["w1"], deq["w2"], ids.cpu(), wts.cpu(), act_mx=True,
                                   flip_delta=MX_FLIP_DELTA)
    got = outs[0].float().cpu()
    assert torch.isfinite(got).all()
    assert cosine(got, ref) >= MX_COS_GATE and rel_l2(got, ref) <= MX_RELL2_GATE
    mx_elementwise_gates(got, ref, bound)
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.parametrize("counts,lists", [
    ([180, 180, 130, 128, 75, 75, 75, 21], True),  # 79 rows per block: the lists of the prologue, paired blocks
    ([24] * 36, False),                            # the same call spread out: jobs by arithmetic
    ([216] * 4, False),                            # crowded, but on fewer jobs than CUs
])
def test_mx_crowded_schedules_use_work_lists(counts, lists, device):
    """Few rows per expert on average, all of them on few experts: the prologue and the two kernels decide on the device
    whether there are work lists."""
    import prime_moe
    from prime_moe import _native
    lib = _native.load()
    K, E, N, top_k = 256, 36, 8192, 4
    counts = counts + [0] * (E - len(counts))
    ids, wts = _routing_by_counts(counts, top_k, device, seed=sum(counts[:3]))
    T = ids.shape[0]
    cus, n_wt = torch.cuda.get_device_properties(device).multi_processor_count, N // 256
    assert T > 128 and T * top_k <= 24 * E and T * top_k // 96 * n_wt > cus  # the rules of the dispatch
    n_live = sum(-(-c // 128) for c in counts)
    assert lists == (T * top_k > 64 * n_live and n_live * n_wt > cus)
    g, a, deq = _quantised_inputs(T, K, E, N, device, seed=N)
    s, e, n = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    nbytes = lib.pmoe_fused_moe_mxfp8_workspace_bytes(T, K, N, E, s.numel(), top_k, 1)
    ws = torch.full((nbytes,), 0xff, dtype=torch.uint8, device=device)
    out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
    _native.check(lib.pmoe_fused_moe_mxfp8(
        *(a[k].data_ptr() for k in ("x", "x_scales", "w1", "w1_scales", "w2", "w2_scales")), out.data_ptr(), s.data_ptr(),
        e.data_ptr(), n.data_ptr(), wts.data_ptr(), top_k, T, K, N, E, s.numel(), 128, 64, 4, 2, 1, 1, ws.data_ptr(), nbytes,
        torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    n_tiles = int(ws[:4].view(torch.int32)[0])  # the workspace starts with the number of row tiles of the lists
    assert n_tiles == (sum(-(-c // 256) for c in counts) if lists else -1)
    ref, bound = O.fused_moe_dense(deq["x"], deq["w1"], deq["w2"], ids.cpu(), wts.cpu(), act_mx=True,
                                   flip_delta=MX_FLIP_DELTA)
    got = out.float().cpu()
    assert torch.isfinite(got).all()
    assert cosine(got, ref) >= MX_COS_GATE and rel_l2(got, ref) <= MX_RELL2_GATE
    mx_elementwise_gates(got, ref, bound)


@pytest.mark.parametrize("K,N,E,counts,rows", [
    (256, 256, 40, EDGES, "stream"),    # streaming up kernel, H = 128 down
    (512, 512, 40, EDGES, "stream"),    # H = 256 down
    (256, 768, 256, SPARSE, "mixed"),    # ring up kernel, general streaming down kernel with half a slab (H = 384)
    (512, 768, 64, [33, 16, 12] + [1] * 9, "stream"),  # general streaming kernels in both directions
    (256, 2048, 40, EDGES, "ring"),     # ring kernels without a work list
    (256, 512, 4, [400, 300, 257, 129], "list"),  # ring kernels with one
])
def test_mx_kernels_with_dropped_rows_and_blocks(K, N, E, counts, rows, device):
    """x with fewer rows than the schedule names (single holes and whole groups of four rows inside live fragments: a copy
    instruction of the loaders each), a block of an expert that does not exist, a schedule cut behind its last pair."""
    import prime_moe
    counts = counts + [0] * (E - len(counts))
    counts[-1] += sum(counts) % 2
    ids, wts = _routing_by_counts(counts, 2, device, seed=K + N)
    T = ids.shape[0]
    keep = (3 * T) // 5
    jobs, cus = min(E, 2 * keep) * (N // 256), torch.cuda.get_device_properties(device).multi_processor_count
    assert (rows == "list") == (2 * keep > (64 if jobs < cus // 2 else 24) * E)  # the rules of the dispatch
    assert rows != "ring" or (jobs >= cus and N > 512 and 2 * keep > 4 * E)
    g, a, deq = _quantised_inputs(T, K, E, N, device, seed=N)
    s, e, n = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    s = shuffle_runs(s, counts, g)
    at = groups = 0
    for c in counts:  # rows 4 .. 7 of a run: a group without a token where the run has four dropped rows
        gone = (s[at:at + c] >= 2 * keep).nonzero().flatten()[:4]
        if c >= 12 and gone.numel() == 4:
            run = s[at:at + c].clone()
            rest = torch.ones(c, dtype=torch.bool, device=device)
            rest[gone] = False
            s[at:at + c] = torch.cat([run[rest][:4], run[gone], run[rest][4:]])
            groups += 1
        at += (c + 127) // 128 * 128
    assert groups >= 2
    e_bad = e.clone()
    e_bad[1] = E + 3
    w_ref = wts.clone()
    lost = s[128:256]
    w_ref.view(-1)[lost[lost >= 0].long()] = 0.0
    ref, bound = O.fused_moe_dense(deq["x"], deq["w1"], deq["w2"], ids.cpu(), w_ref.cpu(), act_mx=True, flip_delta=MX_FLIP_DELTA)
    ref, bound = ref[:keep], bound[:keep]
    last = int((s >= 0).nonzero().max()) + 1
    for length in (s.numel(), last):
        torch.empty((32 << 20,), dtype=torch.float32, device=device).fill_(float("nan"))  # dirty the allocator's blocks
        out = torch.empty((keep, K), dtype=torch.bfloat16, device=device)
        prime_moe.fused_moe_mxfp8(a["x"][:keep].contiguous(), a["x_scales"][:keep].contiguous(), a["w1"], a["w1_scales"], a["w2"],
                                  a["w2_scales"], s[:length].contiguous(), e_bad, n, wts, out, 2, 128, 64, 4, 2, 1, True)
        torch.cuda.synchronize()
        got = out.float().cpu()
        assert torch.isfinite(got).all()
        assert cosine(got, ref) >= MX_COS_GATE and rel_l2(got, ref) <= MX_RELL2_GATE
        mx_elementwise_gates(got, ref, bound)
