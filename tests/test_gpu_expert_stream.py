"""GPU: the grouped GEMM's weight stream for short groups, and the choice between it, the 128-row tiles and the
ping-pong kernel.

All of them take the same v_mfma_f32_16x16x32_bf16 sequence per output element in ascending K and round once, as the
drained kernel does (an output 2 bytes off 16-byte alignment runs that one): equal bit for bit, so no tolerance.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

EDGES = [1, 31, 32, 33, 0, 63, 64, 65, 127, 128, 129, 0, 200, 2]  # edges of the 32-, 64- and 128-row tiles


def _case(pkg, dev, sizes, K, N, swiglu, gather, seed):
    g = torch.Generator().manual_seed(seed)
    M = sum(sizes)
    w = (torch.randn(len(sizes), N, K, generator=g) * 0.05).to(torch.bfloat16).to(dev)
    offs = pkg.ops.group_offsets_from_splits(sizes, dev)
    ncols = N // 2 if swiglu else N
    if gather:
        x = torch.randn(77, K, generator=g).to(torch.bfloat16).to(dev)
        rows = torch.randint(-1, 78, (M,), generator=g, dtype=torch.int32).to(dev)  # -1 and 77: zero rows
        call = lambda **kw: pkg.ops.grouped_gemm_gather(x, rows, w, offs, swiglu=swiglu, **kw)
    else:
        x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(dev)
        call = lambda **kw: pkg.ops.grouped_gemm(x, w, offs, swiglu=swiglu, **kw)
    buf = torch.full((M * ncols + 16,), float("nan"), dtype=torch.bfloat16, device=dev)
    drained = call(out=buf[1:1 + M * ncols].view(M, ncols))
    guarded = torch.full((M + 2, ncols), 3.0, dtype=torch.bfloat16, device=dev)
    return call, drained, guarded


def _same(got, ref, what):
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16)), what


@pytest.mark.parametrize("swiglu,gather", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("sizes,K,N", [
    (EDGES + [0] * 16, 192, 528),          # 3 K steps: the rings run across units; 264 / 33 columns of 8
    (EDGES + [0] * 16, 1024, 16),          # units of one 16-column slab, fewer units than workgroups
    ([5] * 3 + [0] * 61 + [40, 0, 9] * 30, 256, 1040),  # 154 groups: three chunks of 64 lanes
    ([1], 448, 2048),                      # one group, one row
    ([3, 0, 17] * 40, 512, 4096),          # several rounds of units
])
def test_stream_matches_drained_kernel(pkg, dev, sizes, K, N, swiglu, gather):
    assert sum(sizes) <= 32 * len(sizes)
    call, drained, guarded = _case(pkg, dev, sizes, K, N, swiglu, gather, sum(sizes) + K + N)
    M = sum(sizes)
    call(out=guarded[1:M + 1])
    torch.cuda.synchronize()
    _same(guarded[1:M + 1], drained, f"K={K} N={N}")
    assert torch.all(guarded[0] == 3.0) and torch.all(guarded[M + 1] == 3.0), "stored outside out"


@pytest.mark.parametrize("swiglu,gather", [(False, False), (True, True)])
@pytest.mark.parametrize("sizes", [
    [64] * 5 + [20],                       # every group at most 64 rows
    [65, 40, 40, 40],                      # one more than that
    [128] * 7 + [1],                       # every group at most 128 rows
    [129, 40, 0, 90],                      # one more than that
    [700] + [3] * 9 + [0] * 6,             # skewed: nearly all rows in one group
    [40] * 300,                            # more groups than a wavefront's lanes
    [300] + [40] * 299,
])
def test_choice_by_group_sizes(pkg, dev, sizes, swiglu, gather):
    # More than 32 and at most 128 rows per group on average: with a workspace (stale contents) the launch looks at
    # the groups; without one it does not.
    M, G = sum(sizes), len(sizes)
    assert 32 * G < M <= 128 * G
    call, drained, _ = _case(pkg, dev, sizes, 320, 272, swiglu, gather, M + G)
    nbytes = pkg._lib.lib().moe_grouped_gemm_workspace_size(M, 320, 272, G)
    assert nbytes > 0
    ws = torch.full((nbytes,), 0xAB, dtype=torch.uint8, device=dev)
    for _ in range(2):  # the second call finds the first one's list
        _same(call(workspace=ws), drained, "with a workspace")
    _same(call(workspace=torch.empty(0, dtype=torch.uint8, device=dev)), drained, "without one")


@pytest.mark.parametrize("sizes", [[128, 40, 0, 90, 64, 100, 30], [129, 40, 0, 90, 64, 100, 30], [700, 3, 0, 9, 130, 1, 2]])
def test_choice_by_group_sizes_plain_large(pkg, dev, sizes):
    # A rows in place, plain: the launch looks at the groups from 2^28 weights on.
    M, G, N, K = sum(sizes), len(sizes), 8192, 4736
    assert 32 * G < M <= 128 * G and G * N * K >= 1 << 28
    g = torch.Generator(device=dev).manual_seed(M)
    x = torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16)
    w = torch.stack([(torch.randn(N, K, generator=g, device=dev) * 0.05).to(torch.bfloat16) for _ in range(G)])
    offs = pkg.ops.group_offsets_from_splits(sizes, dev)
    buf = torch.full((M * N + 16,), float("nan"), dtype=torch.bfloat16, device=dev)
    drained = pkg.ops.grouped_gemm(x, w, offs, out=buf[1:1 + M * N].view(M, N))
    ws = torch.full((512,), 0xAB, dtype=torch.uint8, device=dev)
    for _ in range(2):
        _same(pkg.ops.grouped_gemm(x, w, offs, workspace=ws), drained, "with a workspace")


@pytest.mark.parametrize("N,K,sizes,tiles", [
    (8192, 2048, [100] * 16 + [0], True),             # 2^24 weights a group: a row tile each
    (8192, 2048, [129] + [100] * 15 + [0], False),    # one row tile more
    (4096, 2048, [257, 0] + [100] * 31, True),        # 2^23: 34 row tiles of 32 groups, less than an eighth more
    (4096, 2048, [257, 0, 257] + [90] * 30, False),   # 36 of 32: an eighth
    (2048, 2048, [640, 0] + [90] * 19 + [640, 0] + [90] * 11 + [40] * 32, True),     # below: 72 of 64
    (2048, 2048, [1200, 1200] + [40] * 62, False),    # 82 of 64: more than a quarter
])
def test_choice_by_row_tiles_plain_large(pkg, dev, N, K, sizes, tiles):
    # The 128-row tiles keep groups of several row tiles where these are few for the size of a group's weights. Word 33
    # of the workspace says who computed the groups; the results are the same bit for bit.
    M, G = sum(sizes), len(sizes)
    assert 32 * G < M <= 128 * G and G * N * K >= 1 << 28
    g = torch.Generator(device=dev).manual_seed(M)
    x = torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(G, N, K, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    offs = pkg.ops.group_offsets_from_splits(sizes, dev)
    drained = pkg.ops.grouped_gemm(x, w, offs, workspace=torch.empty(0, dtype=torch.uint8, device=dev))
    nbytes = pkg._lib.lib().moe_grouped_gemm_workspace_size(M, K, N, G)
    ws = torch.full((nbytes,), 0xAB, dtype=torch.uint8, device=dev)
    for _ in range(2):
        _same(pkg.ops.grouped_gemm(x, w, offs, workspace=ws), drained, "with a workspace")
    assert int(ws.view(torch.int32)[33]) == (1 if tiles else 0)
