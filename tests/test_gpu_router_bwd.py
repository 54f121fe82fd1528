"""GPU parity of the tf32 router backward GEMMs (case39 dgrad, case31 wgrad).

The golden (reference_tf32, case39...:61-68 / case31...:61-68) multiplies tf32-rounded operands
exactly and accumulates in fp32.  Here every tf32 product is one exact product of fp16 values scaled
by powers of two (dgrad: per grad_output row and per weight column; wgrad: per operand column),
accumulated in fp32 in another order, so the bound is
|ours - golden| <= 1e-4 * sum_k |a_k b_k| + 1e-5.  The cases' own checks against an explicit sum
(case39: 1e-3, case31: 1e-2 absolute) are applied as written at full size; the full-size goldens
are computed on the CPU.
"""
from __future__ import annotations

import pytest
import torch

from oracle import ref_torch

pytestmark = pytest.mark.gpu


def _bound_check(got, ref, absprod, what):
    err = (got.cpu().double() - ref.double()).abs()
    bound = 1e-4 * absprod.double() + 1e-5
    assert bool((err <= bound).all()), f"{what}: worst err/bound {(err / bound).max().item():.3f}"


# Reductions of whole and partial 64-wide steps (K = 40, 1000, 1200), output columns past a column tile, row
# tiles with 1-127 valid rows, grad_output rows longer than the 1024 values the row conversion keeps in registers.
@pytest.mark.parametrize("M,K,N", [(64, 64, 256), (5, 8, 8), (300, 320, 520), (1000, 64, 8192), (130, 1000, 264),
                                   (700, 192, 1000), (129, 40, 72), (300, 1200, 136)])
def test_router_dgrad_tf32_shapes(pkg, dev, M, K, N):
    g = torch.Generator().manual_seed(M + K + N)
    go = torch.randn(M, K, generator=g)
    w = torch.randn(K, N, generator=g).to(torch.bfloat16).float()
    got = pkg.ops.router_dgrad_tf32(go.to(dev), w.to(dev))
    ref = ref_torch.router_dgrad_tf32(go, w)
    absprod = ref_torch.round_tf32_rne(go).abs() @ ref_torch.round_tf32_rne(w).abs()
    _bound_check(got, ref, absprod, f"dgrad M={M} K={K} N={N}")


@pytest.mark.parametrize("M,N,K", [(64, 64, 256), (5, 8, 8), (1000, 320, 520), (4096, 64, 1000), (0, 16, 24)])
def test_router_wgrad_tf32_shapes(pkg, dev, M, N, K):
    g = torch.Generator().manual_seed(3 * M + N + K)
    go = torch.randn(M, N, generator=g)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).float()
    got = pkg.ops.router_wgrad_tf32(go.to(dev), x.to(dev))
    assert got.shape == (N, K)
    ref = ref_torch.router_wgrad_tf32(go, x)
    absprod = ref_torch.round_tf32_rne(go).abs().t() @ ref_torch.round_tf32_rne(x).abs()
    _bound_check(got, ref, absprod, f"wgrad M={M} N={N} K={K}")


def test_case39_full_size(pkg, dev):
    case = pkg.cases.case39_ref_musa_asm_tf32_ssgemm_nn_384x256
    go, w = case.make_inputs(seed=0, device=dev)
    got = case.kernel_function(go, w)
    assert got.shape == (case.M, case.N) and got.dtype == torch.float32
    a, b = ref_torch.round_tf32_rne(go.cpu()), ref_torch.round_tf32_rne(w.cpu())
    ref = ref_torch.router_dgrad_tf32(go.cpu(), w.cpu())
    bound = 1e-4 * (a.abs() @ b.abs()) + 1e-5
    assert bool(((got.cpu() - ref).abs() <= bound).all())
    a, b = a.to(dev), b.to(dev)
    rows = torch.tensor([0, case.M // 2, case.M - 1], device=dev)
    manual = (a[rows].double().unsqueeze(-1) * b.double().unsqueeze(0)).sum(dim=1)
    assert (got[rows].double() - manual).abs().max().item() <= 1e-3


def test_case31_full_size(pkg, dev):
    case = pkg.cases.case31_ref_musa_asm_tf32_ssgemm_tn_128x256
    go, x = case.make_inputs(seed=0, device=dev)
    got = case.kernel_function(go, x)
    assert got.shape == (case.N, case.K) and got.dtype == torch.float32
    a, b = ref_torch.round_tf32_rne(go.cpu()), ref_torch.round_tf32_rne(x.cpu())
    ref = ref_torch.router_wgrad_tf32(go.cpu(), x.cpu())
    bound = 1e-4 * (a.abs().t() @ b.abs()) + 1e-5
    assert bool(((got.cpu() - ref).abs() <= bound).all())
    a, b = a.to(dev), b.to(dev)
    cols = torch.tensor([0, case.N // 2, case.N - 1], device=dev)
    manual = torch.stack([(a[:, c].double().unsqueeze(1) * b.double()).sum(dim=0) for c in cols.tolist()])
    assert (got[cols].double() - manual).abs().max().item() <= 1e-2


def test_router_wgrad_tf32_columns_of_any_scale(pkg, dev):
    # Each operand column is scaled by its own power of two into the fp16 range: columns of grad_output
    # near 1e-30 and 1e18, and of inp near 1e-20 and 1e15, keep the relative accuracy of the others
    # (the bound without its absolute term on the scaled rows and columns of dw).
    M, N, K = 1000, 64, 520
    g = torch.Generator().manual_seed(77)
    go = torch.randn(M, N, generator=g)
    x = torch.randn(M, K, generator=g)
    go[:, 3] *= 1e-30
    go[:, 5] *= 1e18
    x[:, 7] *= 1e-20
    x[:, 9] *= 1e15
    got = pkg.ops.router_wgrad_tf32(go.to(dev), x.to(dev)).cpu().double()
    ref = ref_torch.router_wgrad_tf32(go.double(), x.double())
    absprod = ref_torch.round_tf32_rne(go).abs().t().double() @ ref_torch.round_tf32_rne(x).abs().double()
    rel = (got - ref).abs() / absprod.clamp(min=1e-300)
    assert bool(torch.isfinite(got).all())
    for what, sel in (("row 3", rel[3]), ("row 5", rel[5]), ("column 7", rel[:, 7]), ("column 9", rel[:, 9]),
                      ("all", rel)):
        assert rel.numel() and bool((sel <= 1e-4).all()), f"{what}: worst relative error {sel.max().item():.3e}"


def test_router_dgrad_tf32_rows_and_columns_of_any_scale(pkg, dev):
    # grad_output's rows and weight's columns are each scaled by their own power of two into the fp16 range:
    # rows near 1e-30, 1e-25 and 1e18, columns near 1e-20 and 1e15 keep the relative accuracy of the others.
    # Reference: the float64 sum of the tf32-rounded operands' products; outputs in fp32's subnormal range
    # (row 600 x column 7, ~1e-44) are held to an absolute 2^-126, fp32's smallest normal.
    M, K, N = 700, 320, 520
    g = torch.Generator().manual_seed(78)
    go = torch.randn(M, K, generator=g)
    w = torch.randn(K, N, generator=g)
    go[3] *= 1e-30
    go[5] *= 1e18
    go[600] *= 1e-25
    w[:, 7] *= 1e-20
    w[:, 9] *= 1e15
    got = pkg.ops.router_dgrad_tf32(go.to(dev), w.to(dev)).cpu().double()
    a, b = ref_torch.round_tf32_rne(go).double(), ref_torch.round_tf32_rne(w).double()
    ref = a @ b
    excess = (got - ref).abs() - (1e-4 * (a.abs() @ b.abs()) + 2.0 ** -126)
    assert bool(torch.isfinite(got).all())
    for what, sel in (("row 3", excess[3]), ("row 5", excess[5]), ("row 600", excess[600]),
                      ("column 7", excess[:, 7]), ("column 9", excess[:, 9]), ("all", excess)):
        assert bool((sel <= 0).all()), f"{what}: error above the bound by {sel.max().item():.3e}"


@pytest.mark.parametrize("which", ["dgrad", "wgrad"])
def test_router_tf32_inf_and_nan_entries(pkg, dev, which):
    # A row / column holding Inf (or NaN) and finite values above fp16's range: the scale comes from the largest
    # finite magnitude, so the finite values convert exactly and the Inf / NaN entries stay Inf / NaN; the
    # outputs match torch's fp32 product of the tf32-rounded operands in their Inf (with sign) and NaN
    # positions, and the finite ones within the bound.
    g = torch.Generator().manual_seed(91)
    if which == "dgrad":
        M, K, N = 300, 320, 264
        a = torch.randn(M, K, generator=g)
        b = torch.randn(K, N, generator=g)
        a[10, 0], a[10, 1], a[10, 2] = float("inf"), 1e6, -3e5  # one grad_output row: Inf and large finite values
        a[11, 5] = float("nan")
        b[3, 20], b[4, 20] = float("-inf"), 2e5                 # one weight column
        got = pkg.ops.router_dgrad_tf32(a.to(dev), b.to(dev)).cpu()
        ra, rb = ref_torch.round_tf32_rne(a), ref_torch.round_tf32_rne(b)
        ref = ref_torch.router_dgrad_tf32(a, b)
        absprod = ra.abs() @ rb.abs()
    else:
        M, N, K = 1000, 64, 520
        a = torch.randn(M, N, generator=g)
        b = torch.randn(M, K, generator=g)
        a[0, 6], a[1, 6], a[2, 6] = float("inf"), 1e6, -3e5     # one grad_output column
        a[7, 8] = float("nan")
        b[3, 30], b[4, 30] = float("-inf"), 2e5                 # one inp column
        got = pkg.ops.router_wgrad_tf32(a.to(dev), b.to(dev)).cpu()
        ra, rb = ref_torch.round_tf32_rne(a), ref_torch.round_tf32_rne(b)
        ref = ref_torch.router_wgrad_tf32(a, b)
        absprod = ra.abs().t() @ rb.abs()
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(torch.isposinf(got), torch.isposinf(ref)) and torch.equal(torch.isneginf(got), torch.isneginf(ref))
    fin = torch.isfinite(ref)
    assert int((~fin).sum()) > 0 and int(fin.sum()) > 0
    err = (got[fin].double() - ref[fin].double()).abs()
    assert bool((err <= 1e-4 * absprod[fin].double() + 1e-5).all())

@pytest.mark.parametrize("M,N,K", [
    (1, 8, 8),          # one reduction row
    (63, 64, 264),      # less than a stage, one column past a column tile
    (193, 72, 256),     # four stages: the ring's slots wrap; 5 row blocks of the 8
    (700, 256, 1000),   # chunks of the reduction, the last one shorter
    (2049, 320, 72),    # a chunk of one row
    (300, 648, 512),    # three row tiles
])
def test_router_wgrad_tf32_edges_and_growing_columns(pkg, dev, M, N, K):
    # Columns of inp whose magnitudes grow along the rows (the scale found first does not hold), a column that is zero
    # until the last row, a value that tf32 rounds to Inf's neighbour, and zero columns; the reference is the float64
    # sum of the tf32-rounded operands' products, at the bound of this file.
    g = torch.Generator().manual_seed(M + 3 * N + K)
    go = torch.randn(M, N, generator=g)
    x = torch.randn(M, K, generator=g)
    x[:, 1] *= 10.0 ** torch.linspace(-20, 18, M)
    x[:, 2] = 0.0
    x[M - 1, 2] = 1e-12
    x[:, 3] = 0.0
    x[:, 5] *= 10.0 ** torch.linspace(12, -25, M)
    x[M // 2, 6] = 3.4e38
    go[M // 2] *= 1e-3  # keeps column 6 finite
    got = pkg.ops.router_wgrad_tf32(go.to(dev), x.to(dev)).cpu().double()
    a, b = ref_torch.round_tf32_rne(go).double(), ref_torch.round_tf32_rne(x).double()
    ref = a.t() @ b
    excess = (got - ref).abs() - (1e-4 * (a.abs().t() @ b.abs()) + 2.0 ** -126)
    assert bool(torch.isfinite(got).all())
    assert bool((excess <= 0).all()), f"worst excess {excess.max().item():.3e}"


@pytest.mark.parametrize("M,K,N", [
    (1, 64, 8),         # one row, one lane's columns
    (65, 256, 520),     # a stage and a row; a column past a column tile
    (4100, 128, 1032),  # chunks of several stages: the ring's slots wrap
    (12345, 192, 2056), # five column tiles, uneven chunks
    (70, 320, 64),      # the longest reduction of the weight-stationary kernel
    (70, 328, 64),      # and one past it (128-row tiles)
])
def test_router_dgrad_tf32_edges(pkg, dev, M, K, N):
    # Against the float64 sum of the tf32-rounded operands' products, at the bound of this file; guard rows around
    # the output stay as they are.
    g = torch.Generator(device=dev).manual_seed(M + 3 * K + N)
    go = torch.randn(M, K, generator=g, device=dev) * 10.0 ** torch.linspace(-20, 10, M, device=dev)[:, None]
    w = torch.randn(K, N, generator=g, device=dev) * 10.0 ** torch.linspace(-8, 8, N, device=dev)
    nbytes = pkg._lib.lib().moe_router_dgrad_tf32_workspace_size(M, K, N)
    ws = torch.full((nbytes,), 0xAB, dtype=torch.uint8, device=dev)
    buf = torch.full((M + 2, N), 3.0, device=dev)
    pkg._lib.call("moe_router_dgrad_tf32", pkg._lib.ptr(go), M, K, pkg._lib.ptr(w), N, pkg._lib.ptr(buf[1:]), pkg._lib.ptr(ws), nbytes,
                  pkg._lib.stream_handle())
    a, b = ref_torch.round_tf32_rne(go.cpu()).double(), ref_torch.round_tf32_rne(w.cpu()).double()
    excess = (buf[1:M + 1].cpu().double() - a @ b).abs() - (1e-4 * (a.abs() @ b.abs()) + 2.0 ** -126)
    assert bool((excess <= 0).all()), f"worst excess {excess.max().item():.3e}"
    assert bool((buf[0] == 3.0).all()) and bool((buf[M + 1] == 3.0).all()), "stored outside grad_input"


@pytest.mark.parametrize("M", [1, 33])
def test_router_wgrad_tf32_rows_of_64_bit_offsets(pkg, dev, M):
    # Rows of inp so long that 64 of them take 64-bit addresses, whose loads are left out where a wavefront has no row
    # (M = 1: 31 of 32, and the second half of the stage) or no column (the last tile has 8): grad_output's tile is
    # still complete in LDS before any wavefront multiplies it. Reference: float64 on the device, the bound of this file.
    N, K = 8, (1 << 22) + 8
    g = torch.Generator(device=dev).manual_seed(M)
    go = torch.randn(M, N, generator=g, device=dev)
    x = torch.randn(M, K, generator=g, device=dev)
    got = pkg.ops.router_wgrad_tf32(go, x)
    a, b = ref_torch.round_tf32_rne(go).double(), ref_torch.round_tf32_rne(x)
    for at in range(0, K, 1 << 20):
        bk = b[:, at:at + (1 << 20)].double()
        err = (got[:, at:at + (1 << 20)].double() - a.t() @ bk).abs()
        assert bool((err <= 1e-4 * (a.abs().t() @ bk.abs()) + 1e-5).all()), f"columns from {at}: worst error {err.max().item():.3e}"


def test_router_wgrad_tf32_small_values_beside_a_large_one(pkg, dev):
    # Column 5 of inp holds 2^27 in its first row and values of [1, 2) below, 2^27 to 2^28 smaller: scaled by the power
    # of two that brings the large one to 2^14 they are fp16 normal numbers, so they keep all 11 significant bits. The
    # first 32 outputs have grad_output 0 in the large one's row and see the small ones alone; the bound is that of a
    # sum of M exact products in fp32, M 2^-24 sum |a b| over those products.
    M, N, K = 120, 64, 264
    g = torch.Generator().manual_seed(17)
    go = torch.randn(M, N, generator=g)
    x = torch.randn(M, K, generator=g)
    x[:, 5] = (1 + torch.rand(M, generator=g)) * torch.sign(torch.randn(M, generator=g))
    x[0, 5] = 2.0 ** 27
    go[0, :32] = 0.0
    # columns that grow up to the largest value that their first scale takes, and past it
    x[:, 6] = 1.0
    x[40, 6] = 65504.0 / 2 ** 14
    x[:, 7] = 1.0
    x[40, 7] = 65520.0 / 2 ** 14
    got = pkg.ops.router_wgrad_tf32(go.to(dev), x.to(dev)).cpu().double()
    a, b = ref_torch.round_tf32_rne(go).double(), ref_torch.round_tf32_rne(x).double()
    err = (got - a.t() @ b).abs()
    bound = M * 2.0 ** -24 * (a.abs().t() @ b.abs())
    assert bool((err[:32] <= bound[:32]).all()), f"worst err/bound {(err[:32] / bound[:32]).max().item():.1f}"
    assert bool((err[:, 6:8] <= bound[:, 6:8]).all())


def test_router_wgrad_tf32_sums_of_chunks_beyond_fp32(pkg, dev):
    # The reduction of 512 rows runs in chunks. Their sums alone lie beyond fp32's range (64 products of 2^126 and more
    # of one sign), the total does not: the chunks are added while scaled. Columns that are zero in all chunks but one,
    # with values near the smallest there are, and a column of zeros check what a chunk without a scale adds.
    M, N, K = 512, 64, 256
    go = torch.full((M, N), 2.0 ** 60)
    x = torch.full((M, K), 2.0 ** 66)
    x[M // 2:] *= -1.0
    x[M - 1] *= 0.5              # total: 2^125
    x[:, 1] = 0.0
    x[M - 1, 1] = 2.0 ** -136    # the smallest value that the rounding to tf32 leaves, an fp32 subnormal
    x[:, 2] = 0.0
    x[0, 2] = -(2.0 ** -133)
    x[:, 3] = 0.0
    got = pkg.ops.router_wgrad_tf32(go.to(dev), x.to(dev)).cpu().double()
    ref = go.double().t() @ x.double()  # all values are tf32 values
    assert torch.equal(got, ref), (got[0, :5], ref[0, :5])


@pytest.mark.parametrize("M,K,N", [(3, 8, 264), (65, 40, 520), (130, 200, 1032), (67, 264, 72)])
def test_router_dgrad_tf32_partial_reduction_steps_and_tiny_rows(pkg, dev, M, K, N):
    # Reductions that are not whole 64-value steps: what lies past a row's values is the next row's, here Inf and NaN, and
    # must not reach the sums. Rows of subnormals only, down to the smallest that the rounding to tf32 leaves, take the
    # largest exponent of their byte and stay exact (a sum of M exact products in fp32; results below 2^-126 round once
    # more).
    g = torch.Generator().manual_seed(M + K + N)
    go = torch.randn(M, K, generator=g)
    w = torch.randn(K, N, generator=g) * 2.0 ** 20
    go[M // 2] = float("inf")
    go[M // 2, 1::2] = float("nan")
    go[0] = 2.0 ** -136
    go[M - 1] *= 2.0 ** -127
    w[:, N - 2] = float("nan")
    got = pkg.ops.router_dgrad_tf32(go.to(dev), w.to(dev)).cpu().double()
    rows = [m for m in range(M) if m != M // 2]
    cols = [n for n in range(N) if n != N - 2]
    assert bool(torch.isnan(got[M // 2]).all()) and bool(torch.isnan(got[:, N - 2]).all())
    a, b = ref_torch.round_tf32_rne(go[rows]).double(), ref_torch.round_tf32_rne(w[:, cols]).double()
    excess = (got[rows][:, cols] - a @ b).abs() - (K * 2.0 ** -24 * (a.abs() @ b.abs()) + 2.0 ** -149)
    assert bool((excess <= 0).all()), f"worst excess {excess.max().item():.3e}"


@pytest.mark.parametrize("M,N,K", [
    (1024, 320, 1024),  # planes for 3 chunks instead of 8
    (700, 320, 520),    # 2 instead of 5
    (200, 72, 8),       # one chunk
    (4096, 64, 1000),   # all of them
    (1, 1024, 8), (65, 520, 8), (70, 72, 24),  # the copy of grad_output is the larger part of the workspace
])
def test_router_wgrad_tf32_workspace_of_the_least_size(pkg, dev, M, N, K):
    # fp16 copies of both operands, their exponents and column-max slabs and the planes of chunks of 512 rows or more are
    # enough at every size, and nothing is stored past them. Inf and NaN in some columns of grad_output: the next row of
    # its transposed copy is not read as the end of one.
    def up(b):
        return (b + 255) // 256 * 256
    def slabs(rows):
        s = max(1, min(64, -(-rows // 64)))
        return -(-rows // -(-rows // s))
    tiles = -(-N // 256) * -(-K // 256)
    chunks = min(-(-256 // tiles), max(1, M // 512), 64)
    if chunks > 1:
        chunks = -(-M // (-(-(-(-M // chunks)) // 64) * 64))
    least = (up(2 * M * N) + up(2 * M * K) + up(4 * N) + up(4 * K) + up(4 * slabs(M) * N) + up(4 * slabs(M) * K) + up(4 * chunks * N * K))
    assert least <= pkg._lib.lib().moe_router_wgrad_tf32_workspace_size(M, N, K)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    go = torch.randn(M, N, generator=g, device=dev)
    x = torch.randn(M, K, generator=g, device=dev)
    go[0, 4] = float("inf")
    go[M - 1, 6] = float("nan")
    guard = 4096
    ws = torch.full((least + guard,), 0xAB, dtype=torch.uint8, device=dev)
    out = torch.empty(N, K, device=dev)
    args = (pkg._lib.ptr(go), M, N, pkg._lib.ptr(x), K, pkg._lib.ptr(out), pkg._lib.ptr(ws))
    with pytest.raises(pkg._lib.MoeError):
        pkg._lib.call("moe_router_wgrad_tf32", *args, least - 1, pkg._lib.stream_handle())
    pkg._lib.call("moe_router_wgrad_tf32", *args, least, pkg._lib.stream_handle())
    assert bool((ws[least:] == 0xAB).all()), "stored past the workspace"
    rows = [n for n in range(N) if n not in (4, 6)]
    a, b = ref_torch.round_tf32_rne(go.cpu()[:, rows]).double(), ref_torch.round_tf32_rne(x.cpu()).double()
    err = (out.cpu().double()[rows] - a.t() @ b).abs()
    assert bool((err <= 1e-4 * (a.abs().t() @ b.abs()) + 1e-5).all()), f"worst error {err.max().item():.3e}"
    assert not bool(torch.isfinite(out[4]).any()) and bool(torch.isnan(out[6]).all())


def test_router_wgrad_tf32_chunks_that_do_not_fit_the_workspace(pkg, dev):
    # inp of 2 GiB takes two chunks for its 32-bit offsets; a workspace without room for two planes of 2 GiB takes one,
    # with 64-bit addresses. Some rows of the result against float64, at the bound of this file.
    M, N, K = 8192, 8192, 65536
    def up(b):
        return (b + 255) // 256 * 256
    least = up(2 * M * N) + up(2 * M * K) + up(4 * N) + up(4 * K) + up(4 * 64 * N) + up(4 * 64 * K) + up(4 * N * K)
    assert least < pkg._lib.lib().moe_router_wgrad_tf32_workspace_size(M, N, K)
    g = torch.Generator(device=dev).manual_seed(5)
    go = torch.randn(M, N, generator=g, device=dev)
    x = torch.randn(M, K, generator=g, device=dev)
    ws = torch.empty(least, dtype=torch.uint8, device=dev)
    out = torch.empty(N, K, device=dev)
    pkg._lib.call("moe_router_wgrad_tf32", pkg._lib.ptr(go), M, N, pkg._lib.ptr(x), K, pkg._lib.ptr(out), pkg._lib.ptr(ws), least,
                  pkg._lib.stream_handle())
    del ws
    rows = torch.tensor([0, 63, 64, 4097, N - 1], device=dev)
    a = ref_torch.round_tf32_rne(go[:, rows]).double()
    for at in range(0, K, 8192):
        b = ref_torch.round_tf32_rne(x[:, at:at + 8192]).double()
        err = (out[rows, at:at + 8192].double() - a.t() @ b).abs()
        assert bool((err <= 1e-4 * (a.abs().t() @ b.abs()) + 1e-5).all()), f"columns from {at}: worst error {err.max().item():.3e}"


@pytest.mark.parametrize("M,K,N", [
    (1000, 320, 1032), (1, 8, 136),      # two wavefronts a workgroup: 9 column tiles, and one column past a tile
    (3000, 320, 1032), (1100, 72, 3848), # four
    (12800, 264, 1032),                  # eight, units of several stages
])
def test_router_dgrad_tf32_workgroups_of_fewer_columns(pkg, dev, M, K, N):
    test_router_dgrad_tf32_edges(pkg, dev, M, K, N)


def test_router_dgrad_tf32_rows_near_the_largest_value(pkg, dev):
    # The smallest exponent that a row's byte holds: largest magnitudes in [2^127, 2^128). The bound of a sum of K exact
    # products in fp32.
    M, K, N = 70, 64, 136
    g = torch.Generator().manual_seed(3)
    go = torch.randn(M, K, generator=g) * 2.0 ** 120
    go[:, 5] = 1.5 * 2.0 ** 127
    w = torch.randn(K, N, generator=g) * 2.0 ** -30
    got = pkg.ops.router_dgrad_tf32(go.to(dev), w.to(dev)).cpu().double()
    a, b = ref_torch.round_tf32_rne(go).double(), ref_torch.round_tf32_rne(w).double()
    assert bool(((got - a @ b).abs() <= K * 2.0 ** -24 * (a.abs() @ b.abs())).all())
