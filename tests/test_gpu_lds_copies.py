"""The direct-to-LDS copies of the GEMM kernels are issued from inline assembly that sets M0 itself (csrc/moe_ring.h).
If a compiler ever kept a value of its own in M0 across such a statement, copies would land in the wrong place.  These
cases run the tile paths with the longest runs of copies between two barriers (bf16: tiles of 384 token rows, ten
copies per wave and slab; mxfp8: row tiles of two full blocks, nine per wave and stage, with two to four stages in
flight) right after every CU's LDS has been filled with NaN patterns, so a misplaced copy shows up here, by name, as
a NaN or a parity failure, and not somewhere in the grids.

The streaming kernels read token fragments and scale dwords past the live rows, that is LDS that the job never wrote; what they
find there may only reach output columns that nobody stores."""
import pytest
import torch

import test_gpu_bf16 as B
import test_gpu_mxfp8 as M
from helpers import BF16_GATE, MX_COS_GATE, MX_FLIP_DELTA, MX_RELL2_GATE, cosine, mx_elementwise_gates, rel_clamp, rel_l2
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu


def _poison(device):
    from prime_moe import _native
    word = torch.zeros(1, dtype=torch.int32, device=device)
    _native.check(_native.load().pmoe_poison_lds(word.data_ptr(), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert int(word[0]) == 0


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("K,N", [(256, 256), (2048, 512)])
def test_bf16_tall_tiles_on_poisoned_lds(K, N, split, device):
    # 2 experts x ~800 rows: tiles of 5 and 6 pairs of fragments; K = 256 has four slabs (the ring's first and last
    # stages only), K = 2048 runs the steady state
    _poison(device)
    B._run_case(800, K, 2, N, 2, split, device, seed=11, hot_last=False)


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("K,N", [(256, 256), (2048, 512)])
def test_mxfp8_full_tiles_on_poisoned_lds(K, N, split, device):
    _poison(device)
    M._run_case(800, K, 2, N, 2, split, device, seed=12, hot_last=False)


@pytest.mark.parametrize("r", [1, 5, 33])
@pytest.mark.parametrize("K,N", [(256, 256), (512, 512), (384, 768)])
def test_bf16_streaming_kernels_on_poisoned_lds(K, N, r, device):
    # short down kernels (H = 128, 256) and the general one, `r` live rows in every block
    import prime_moe
    E = 40
    ids, wts = M._routing_by_counts([r] * 16 + [0] * 24, 2, device, seed=r)
    T = ids.shape[0]
    assert 2 * T <= 32 * E  # the rule of the dispatch
    g, x, w1, w2 = B._inputs(T, K, E, N, device, seed=K + r)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
    _poison(device)
    prime_moe.fused_moe_bf16(x, w1, w2, *sched, wts, out, 2, 128, 64, 4, 2, 1, 1, True)
    torch.cuda.synchronize()
    got = out.float().cpu()
    ref = O.fused_moe_dense(x.cpu(), w1.cpu(), w2.cpu(), ids.cpu(), wts.cpu())
    assert torch.isfinite(got).all() and rel_clamp(got, ref, 1.0) <= BF16_GATE


@pytest.mark.parametrize("r", [1, 5, 33])
@pytest.mark.parametrize("K,N,E", [(256, 256, 40), (512, 512, 40), (256, 768, 256)])
def test_mxfp8_streaming_kernels_on_poisoned_lds(K, N, E, r, device):
    # as above; H = 384 ends in half a slab
    import prime_moe
    ids, wts = M._routing_by_counts([r] * 16 + [0] * (E - 16), 2, device, seed=r)
    T = ids.shape[0]
    assert 2 * T <= 24 * E and (N <= 512 or 2 * T <= 4 * min(E, 2 * T))  # the rules of the dispatch: no list, streaming down
    g, a, deq = M._quantised_inputs(T, K, E, N, device, seed=K + r)
    sched = torch.ops.prime_moe.moe_align(ids, E, 128, 1)
    out = torch.empty((T, K), dtype=torch.bfloat16, device=device)
    _poison(device)
    prime_moe.fused_moe_mxfp8(a["x"], a["x_scales"], a["w1"], a["w1_scales"], a["w2"], a["w2_scales"], *sched, wts, out, 2, 128, 64,
                              4, 2, 1, True)
    torch.cuda.synchronize()
    got = out.float().cpu()
    ref, bound = O.fused_moe_dense(deq["x"], deq["w1"], deq["w2"], ids.cpu(), wts.cpu(), act_mx=True, flip_delta=MX_FLIP_DELTA)
    assert torch.isfinite(got).all()
    assert cosine(got, ref) >= MX_COS_GATE and rel_l2(got, ref) <= MX_RELL2_GATE
    mx_elementwise_gates(got, ref, bound)
