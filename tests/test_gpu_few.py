"""One token or two through the bf16 layer (csrc/moe_few.h): one step of the contraction, whole batches of steps and a remainder,
one to forty blocks (of four or fewer, several waves share a contraction, of more than eight a wave takes several), experts named
by both tokens, a token that names an expert more than twice, tokens beyond M, blocks of experts that do not exist, pairs listed
twice; calls on both sides of the lines behind which other kernels run."""
import pytest
import torch

from helpers import BF16_GATE, rel_clamp
from oracle import moe_oracle as O
from test_gpu_bf16 import _inputs

pytestmark = pytest.mark.gpu


def _run(x, w1, w2, sched, wts, top_k, split, device):
    import prime_moe
    M, K = x.shape
    torch.empty((8 << 20,), dtype=torch.float32, device=device).fill_(float("nan"))  # dirty the allocator's blocks
    out = torch.full((M, K), float("nan") if split else 0.25, dtype=torch.bfloat16, device=device)
    prime_moe.fused_moe_bf16(x, w1, w2, *sched, wts, out, top_k, 128, 64, 4, 2, 1, 1, split)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("K,N,E,ids", [
    (128, 256, 4, [[2]]),                                   # one step, one block: eight parts of one step
    (1024, 2048, 6, [[5, 0]]),                              # whole batches of 8 steps, two blocks
    (1152, 2304, 8, [[0, 1, 2], [2, 1, 0]]),                # a remainder of one step, three blocks of two rows
    (4096, 512, 8, [[7, 6, 5, 4], [3, 2, 1, 0]]),           # eight blocks
    (256, 768, 40, [list(range(0, 9)), list(range(5, 14))]),  # fourteen blocks, four of them with two rows
    (384, 256, 3, [[1, 1, 1], [1, 0, 1]]),                  # an expert with five rows
    (640, 512, 40, [list(range(32)), list(range(8, 40))]),  # 64 pairs (streaming kernels, as the fourteen blocks above)
    (512, 768, 12, [list(range(8)), list(range(4, 12))]),   # sixteen pairs on twelve blocks, four of them with two rows
    (2048, 1024, 40, [list(range(32)), list(range(8, 40))]),  # 64 pairs on forty blocks
])
def test_one_and_two_tokens(K, N, E, ids, split, device):
    import prime_moe  # noqa: F401 (registers the ops)
    ids = torch.tensor(ids, dtype=torch.int32, device=device)
    T, top_k = ids.shape
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=K + N)
    wts = torch.softmax(torch.randn((T, top_k), device=device, generator=g), -1)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu()) + (0.0 if split else 0.25)
    outs = [_run(x, w1, w2, sched, wts, top_k, split, device) for _ in range(2)]
    got = outs[0].float().cpu()
    assert torch.isfinite(got).all() and rel_clamp(got, ref, 1.0) <= BF16_GATE
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


def test_odd_schedules(device):
    import prime_moe  # noqa: F401 (registers the ops)
    K, N, E, top_k = 512, 512, 6, 3
    ids = torch.tensor([[0, 3, 5], [3, 1, 0], [3, 5, 2]], dtype=torch.int32, device=device)  # the third token is beyond M
    g, x, w1, w2 = _inputs(3, K, E, N, device, seed=1)
    wts = torch.softmax(torch.randn((3, top_k), device=device, generator=g), -1)
    s, e, n = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    ref = lambda w: O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), w.cpu())[:2]
    check = lambda sched, w, want: rel_clamp(_run(x[:2].contiguous(), w1, w2, sched, w, top_k, True, device).float().cpu(), want, 1.0) <= BF16_GATE
    assert check((s, e, n), wts, ref(wts))
    last = int((s >= 0).nonzero().max()) + 1
    assert check((s[:last].contiguous(), e, n), wts, ref(wts))  # cut behind the last pair
    e_bad = e.clone()
    e_bad[0] = E + 1  # expert 0's block
    w_ref = wts.clone()
    w_ref[ids == 0] = 0.0
    assert check((s, e_bad, n), wts, ref(w_ref))
    s_dup = s.clone()
    s_dup[1 if int(s[1]) < 0 else int((s[:128] >= 0).sum())] = s[0]  # a pair id twice in its block contributes once
    assert check((s_dup, e, n), wts, ref(wts))
    assert check((s, e, torch.zeros_like(n)), wts, torch.zeros_like(ref(wts)))  # nothing scheduled


@pytest.mark.parametrize("ids,place", [
    ([[0, 1]], 1),                       # two blocks: four waves per contraction
    ([[1, 0, 3], [3, 0, 2]], 2),         # four blocks: two
    ([list(range(9))], 5),               # nine: one, and two blocks of one wave
])
def test_pair_under_two_experts(ids, place, device):
    """One of the two rows stands for the pair, for every column of its token."""
    import prime_moe  # noqa: F401 (registers the ops)
    K, N, E = 2048, 2048, 9
    ids = torch.tensor(ids, dtype=torch.int32, device=device)
    T, top_k = ids.shape
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=place)
    wts = torch.softmax(torch.randn((T, top_k), device=device, generator=g), -1)
    s, e, n = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    n_live = int(n[0]) // 128
    for src, dst in ((0, n_live - 1), (n_live - 1, 0), (place - 1, place)):
        pair, s_far, ids_far = int(s[128 * src]), s.clone(), ids.clone()
        s_far[128 * dst + int((s[128 * dst:128 * dst + 128] >= 0).sum())] = pair
        ids_far.view(-1)[pair] = int(e[dst])
        refs = [O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), i.cpu(), wts.cpu()) for i in (ids, ids_far)]
        for _ in range(4):
            got = _run(x, w1, w2, (s_far, e, n), wts, top_k, True, device).float().cpu()
            assert min(rel_clamp(got, r, 1.0) for r in refs) <= BF16_GATE


def test_rows_behind_the_end_of_the_schedule_are_no_pairs(device):
    """num_tokens_post_padded may end inside a block: what lies behind it is not part of the schedule."""
    import prime_moe  # noqa: F401 (registers the ops)
    K, N, E, top_k = 512, 512, 6, 3
    ids = torch.tensor([[0, 3, 5], [3, 1, 5]], dtype=torch.int32, device=device)
    g, x, w1, w2 = _inputs(2, K, E, N, device, seed=2)
    wts = torch.softmax(torch.randn((2, top_k), device=device, generator=g), -1)
    s, e, n = torch.ops.prime_moe.moe_align(ids, E, 128, 1)  # blocks of experts 0, 1, 3 (two rows), 5 (two rows)
    for end in (1, 129, 257, 258, 385, 386):
        w_ref = wts.clone()
        lost = s[end:]
        w_ref.view(-1)[lost[lost >= 0].long()] = 0.0
        ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), w_ref.cpu())
        got = _run(x, w1, w2, (s, e, torch.full_like(n, end)), wts, top_k, True, device).float().cpu()
        assert rel_clamp(got, ref, 1.0) <= BF16_GATE, end


def _few_runs(T, K, N, top_k, device):
    """Whether a call takes the kernels of moe_few.h: with finalize masked off they alone write `out`."""
    from prime_moe import _native
    import prime_moe
    E = max(2, T * top_k)
    g, x, w1, w2 = _inputs(T, K, E, N, device, seed=N)
    ids = torch.randperm(E, generator=g, device=device)[:T * top_k].view(T, top_k).to(torch.int32)
    wts = torch.softmax(torch.randn((T, top_k), device=device, generator=g), -1)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    out = torch.full((T, K), float("nan"), dtype=torch.bfloat16, device=device)
    lib = _native.load()
    try:
        lib.pmoe_set_phase_mask(6)  # the up and the down kernel
        prime_moe.fused_moe_bf16(x, w1, w2, *sched, wts, out, top_k, 128, 64, 4, 2, 1, 1, True)
    finally:
        lib.pmoe_set_phase_mask(15)
    torch.cuda.synchronize()
    written = torch.isfinite(out.float()).all().item()
    assert written or torch.isnan(out.float()).all().item()
    got = _run(x, w1, w2, sched, wts, top_k, True, device).float().cpu()
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())
    assert torch.isfinite(got).all() and rel_clamp(got, ref, 1.0) <= BF16_GATE
    return written


@pytest.mark.parametrize("T,K,N,top_k,few", [
    (2, 256, 8192, 2, True), (1, 256, 8192, 5, False),      # four pairs of any size; more, and most CUs idle
    (1, 512, 2048, 16, True), (1, 512, 2304, 16, False),    # the idle CUs' share
    (2, 640, 512, 8, True), (1, 640, 512, 17, False), (2, 640, 512, 32, False),  # short rows of W2: 16 pairs, 17, 64
    (1, 2048, 8192, 5, True), (2, 2048, 1024, 32, True), (1, 2048, 1024, 65, False), (2, 2048, 768, 9, False),  # no idle CU
    (2, 1792, 1024, 24, True), (2, 1664, 1024, 24, False),  # few idle CUs, more than 16 pairs
    (2, 2176, 1536, 4, True), (1, 2176, 1536, 9, False), (1, 2176, 1792, 5, False), (2, 4096, 2048, 2, True),  # K beyond the CUs
    (1, 4224, 256, 1, False), (3, 256, 256, 1, False),      # K beyond 4096, three tokens
])
def test_which_calls_take_these_kernels(T, K, N, top_k, few, device):
    cus = torch.cuda.get_device_properties(device).multi_processor_count
    if cus != 256:
        pytest.skip("the lines are drawn for 256 CUs")
    assert _few_runs(T, K, N, top_k, device) == few
