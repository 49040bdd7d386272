"""moe_align at the edges of its launch shapes (one workgroup, slices of 1024 .. 8192 ids), the scratch sizes that choose
between them, and the router's one-kernel form: bit-exact against the oracle."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from test_gpu_route import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,E", [(8192, 8), (8193, 37), (9000, 700), (65536, 128), (65537, 128), (131073, 600), (262145, 5)])
def test_align_at_slice_edges_with_every_scratch(n, E, device):
    import prime_moe
    from prime_moe import _native
    lib = _native.load()
    ids = np.random.default_rng(n).integers(-1, E, size=n).astype(np.int32)
    ids[: n // 3] = E // 2  # a hot expert
    keep = np.flatnonzero(ids >= 0)
    s_c, e_c, t_c = O.moe_align_fast(ids[keep], E, 128, 1)
    pad_to, max_padded, max_blocks = prime_moe.align_sizes(n, E, 128, 1)
    s_w = np.full(max_padded, -1, dtype=np.int32)
    s_w[: s_c.size] = np.where(s_c >= 0, keep[np.maximum(s_c, 0)], -1)
    e_w = np.full(max_blocks, E - 1, dtype=np.int32)
    e_w[: e_c.size] = e_c
    dev_ids = torch.from_numpy(ids).to(device)
    small, fast = lib.pmoe_moe_align_workspace_bytes(n, E), lib.pmoe_moe_align_workspace_bytes_fast(n, E)
    assert fast >= small and (fast > 0) == (n > 8192)
    for nbytes in sorted({0, 4, small, (small + fast) // 2, fast}):
        s = torch.full((max_padded,), 0x5a5a5a5a, dtype=torch.int32, device=device)
        e = torch.full((max_blocks,), 0x5a5a5a5a, dtype=torch.int32, device=device)
        t = torch.full((1,), 0x5a5a5a5a, dtype=torch.int32, device=device)
        ws = torch.full((max(nbytes, 4),), 0x5a, dtype=torch.uint8, device=device)
        _native.check(lib.pmoe_moe_align_ws(dev_ids.data_ptr(), s.data_ptr(), e.data_ptr(), t.data_ptr(), n, E, 128, pad_to,
                                            max_padded, max_blocks, ws.data_ptr() if nbytes else None, nbytes,
                                            torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        for got, want in zip((s, e, t), (s_w, e_w, t_c)):
            np.testing.assert_array_equal(got.cpu().numpy(), want, err_msg=f"{nbytes} bytes of scratch")


@pytest.mark.parametrize("n,E,short,refused", [(8193, 37, 0, False), (16384, 8, 0, False), (16385, 8, 4, False), (16385, 8, 0, True)])
def test_a_misaligned_workspace_is_an_error_only_where_scratch_is_needed(n, E, short, refused, device):
    """The first query asks for no scratch up to 16384 ids, and a smaller one than it asks for is as good as none: such a
    pointer may be anything."""
    import prime_moe
    from prime_moe import _native
    lib = _native.load()
    ids = np.random.default_rng(n).integers(0, E, size=n).astype(np.int32)
    pad_to, max_padded, max_blocks = prime_moe.align_sizes(n, E, 128, 1)
    need = lib.pmoe_moe_align_workspace_bytes(n, E)
    assert (need == 0) == (n <= 16384)
    nbytes = (need or 1 << 20) - short
    ws = torch.full((nbytes + 8,), 0x5a, dtype=torch.uint8, device=device)
    dev_ids = torch.from_numpy(ids).to(device)
    s, e, t = (torch.empty((c,), dtype=torch.int32, device=device) for c in (max_padded, max_blocks, 1))
    rc = lib.pmoe_moe_align_ws(dev_ids.data_ptr(), s.data_ptr(), e.data_ptr(), t.data_ptr(), n, E, 128, pad_to, max_padded,
                               max_blocks, ws.data_ptr() + 1, nbytes, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert (rc != 0) == refused
    if not refused:
        for got, want in zip((s, e, t), O.moe_align_fast(ids, E, 128, 1)):
            np.testing.assert_array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("n,E,words", [
    ((1 << 21) + 1, 1024, "all"),  # the kernel that turns counts into bases: 257 slices, 16 workgroups of experts
    ((1 << 22) - 77, 100, "all"),  # its last workgroup has experts to spare
    ((1 << 23) + 5, 17, "all"),    # one workgroup, 32 columns
    ((1 << 22) - 77, 100, "counts"),  # scratch for the counts alone: the scatter kernel adds them up
])
def test_align_of_very_many_ids(n, E, words, device):
    import prime_moe
    from prime_moe import _native
    lib = _native.load()
    slices = -(-n // 8192)
    assert slices * slices * E > 1 << 24  # the rule of the dispatch
    ids = np.random.default_rng(n).integers(0, E, size=n).astype(np.int32)
    ids[n // 2: n // 2 + n // 8] = E // 2
    pad_to, max_padded, max_blocks = prime_moe.align_sizes(n, E, 128, 1)
    nbytes = lib.pmoe_moe_align_workspace_bytes(n, E) if words == "all" else 4 * slices * E
    ws = torch.full((nbytes,), 0x5a, dtype=torch.uint8, device=device)
    dev_ids = torch.from_numpy(ids).to(device)
    s, e, t = (torch.full((c,), 0x5a5a5a5a, dtype=torch.int32, device=device) for c in (max_padded, max_blocks, 1))
    _native.check(lib.pmoe_moe_align_ws(dev_ids.data_ptr(), s.data_ptr(), e.data_ptr(), t.data_ptr(), n, E, 128, pad_to,
                                        max_padded, max_blocks, ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    for got, want in zip((s, e, t), O.moe_align_fast(ids, E, 128, 1)):
        np.testing.assert_array_equal(got.cpu().numpy(), want)


def test_align_next_to_2_31_blocks_by_one_workgroup(device):
    """Blocks of one row and padding to 2^30 - 1: two of them make 2^31 - 2 blocks, and every loop over rows or blocks steps
    past 2^31 before it ends."""
    import prime_moe  # noqa: F401
    bpc = (1 << 30) - 1
    s, e, t = torch.ops.prime_moe.moe_align(torch.zeros((8,), dtype=torch.int32, device=device), 1, 1, bpc)
    assert s.numel() == e.numel() == 2 * bpc and int(t) == bpc
    assert torch.equal(s[:8], torch.arange(8, dtype=torch.int32, device=device))
    for at in range(0, 2 * bpc, 1 << 29):
        assert int(s[max(at, 8):at + (1 << 29)].max()) == -1 == int(s[max(at, 8):at + (1 << 29)].min())
        assert int(e[at:at + (1 << 29)].max()) == 0 == int(e[at:at + (1 << 29)].min())


def test_align_next_to_2_31_ids_by_many_workgroups(device):
    import prime_moe  # noqa: F401
    n, step = (1 << 31) - 1, 1 << 29
    ids = torch.empty((n,), dtype=torch.int32, device=device)
    for at in range(0, n, step):
        ids[at:at + step] = torch.arange(at, min(at + step, n), dtype=torch.int32, device=device).bitwise_and_(1)
    s, e, t = torch.ops.prime_moe.moe_align(ids, 2, 1, 1)
    half = (n + 1) // 2  # the even ids, then the odd ones
    assert s.numel() == e.numel() == int(t) == n
    for at in range(0, n, step):
        end = min(at + step, n)
        want = torch.arange(at, end, dtype=torch.int64, device=device)
        owner = (want >= half).to(torch.int32)
        want = torch.where(want < half, 2 * want, 2 * (want - half) + 1).to(torch.int32)
        assert torch.equal(s[at:end], want) and torch.equal(e[at:end], owner)


@pytest.mark.parametrize("T,E,k", [(16, 512, 32), (17, 512, 8), (8, 513, 32), (9, 1024, 4), (16, 64, 32), (2, 33, 32)])
def test_route_around_the_one_kernel_form(T, E, k, device):
    g = torch.Generator(device=device).manual_seed(T + E + k)
    _check(torch.randn((T, E), generator=g, device=device), k, bias=torch.randn((E,), generator=g, device=device))
    _check(torch.randint(-2, 3, (T, E), generator=g, device=device).to(torch.bfloat16), k, block_m=32, bpc=2)
