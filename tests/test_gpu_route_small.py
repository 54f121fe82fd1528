"""GPU: the top-k's slot lists and the row-id map's one-launch form, at the sizes where they can go wrong; whole numbers
and copies, so equal bit for bit to the oracle."""
from __future__ import annotations

import pytest
import torch

from oracle import ref_torch
from conftest import assert_bits_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E", [1, 60, 64, 65, 128, 129, 192, 193, 257, 320, 321, 384, 448, 449, 512, 513, 1024])
@pytest.mark.parametrize("levels", [2, 7, 0])
def test_topk_slots_and_ties(pkg, dev, E, levels):
    # Few distinct values: ties inside a lane's list, between lanes, and between both; signed zeros, infinities, NaN.
    g = torch.Generator().manual_seed(E + levels)
    T, k = 37, min(E, 64)
    x = torch.randint(0, levels, (T, E), generator=g).float() - levels // 2 if levels else torch.randn(T, E, generator=g)
    special = torch.tensor([0.0, -0.0, float("inf"), float("-inf"), float("nan"), 3.4e38])
    hit = torch.rand(T, E, generator=g) < 0.1
    x[hit] = special[torch.randint(0, 6, (int(hit.sum()),), generator=g)]
    for kk in {1, min(E, 8), k}:
        values, indices, mask = pkg.ops.topk(x.to(dev), kk, with_mask=True)
        rv, ri = ref_torch.topk(x, kk)
        assert torch.equal(indices.cpu(), ri), f"E={E} k={kk}"
        assert_bits_equal(values, rv, f"E={E} k={kk}")
        assert torch.equal(mask.cpu(), torch.zeros(T, E, dtype=torch.bool).scatter_(1, ri, True))


@pytest.mark.parametrize("T", [1, 63, 64, 65, 255, 256, 257])
@pytest.mark.parametrize("E", [1, 31, 32, 33, 60, 64, 80, 256, 272, 1024])
def test_row_id_map_one_launch_sizes(pkg, dev, T, E):
    # T <= 256 and a mask of at most 64 KiB (16 KiB without 16-byte loads) is one launch; the sizes lie on both sides.
    g = torch.Generator().manual_seed(T * 1000 + E)
    for rm in (torch.rand(T, E, generator=g) < 0.15, torch.ones(T, E, dtype=torch.bool), torch.zeros(T, E, dtype=torch.bool)):
        R = int(rm.sum())
        row_em, row_tm = ref_torch.row_id_map(rm)
        m = rm.to(torch.uint8) * torch.randint(1, 256, (T, E), generator=g).to(torch.uint8)  # any nonzero byte selects
        got = pkg.ops.row_id_map(m.to(dev), expert_major_i32=True, expert_offsets=True, src_rows=R)
        assert torch.equal(got["expert_major"].cpu(), row_em) and torch.equal(got["token_major"].cpu(), row_tm)
        assert torch.equal(got["expert_major_i32"].cpu().long(), row_em)
        assert torch.equal(got["expert_offsets"].cpu(), ref_torch.expert_offsets(rm))
        assert torch.equal(got["src_token"].cpu().long(), rm.t().nonzero()[:, 1])


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("T,E", [(63, 32), (255, 64), (257, 32), (1023, 96), (4097, 320), (16641, 64)])
def test_row_id_map_paired_stores(pkg, dev, T, E, shift):
    # Whole groups of 32 experts: token-major rows in pairs on a 16-byte aligned output, one at a time on another; nothing
    # outside the output is written.
    L = pkg._lib
    g = torch.Generator().manual_seed(T + E)
    rm = torch.rand(T, E, generator=g) < 0.1
    m = rm.to(torch.uint8).to(dev)
    buf = torch.full((T * E + 4,), -7, dtype=torch.int64, device=dev)
    out = buf[2 + shift:2 + shift + T * E]
    n = L.lib().moe_row_id_map_workspace_size(T, E)
    ws = torch.empty(n, dtype=torch.uint8, device=dev)
    L.call("moe_row_id_map", m.data_ptr(), T, E, None, out.data_ptr(), None, None, None, 0, ws.data_ptr(), n, L.stream_handle())
    assert torch.equal(out.view(T, E).cpu(), ref_torch.row_id_map(rm)[1])
    assert (buf[:2 + shift] == -7).all() and (buf[2 + shift + T * E:] == -7).all()


@pytest.mark.parametrize("T", [16129, 16384])
@pytest.mark.parametrize("E", [256, 257, 288, 300, 304, 320])
def test_row_id_map_more_than_one_round(pkg, dev, T, E):
    # 64 (63 or 64) super-chunks: up to 8 expert groups make 512 blocks of 1024 threads, 9 and more take 512 threads.
    g = torch.Generator().manual_seed(T + E)
    rm = torch.rand(T, E, generator=g) < 0.03
    row_em, row_tm = ref_torch.row_id_map(rm)
    got = pkg.ops.row_id_map(rm.to(torch.uint8).to(dev), expert_major_i32=True, expert_offsets=True, src_rows=int(rm.sum()))
    assert torch.equal(got["expert_major"].cpu(), row_em) and torch.equal(got["token_major"].cpu(), row_tm)
    assert torch.equal(got["expert_major_i32"].cpu().long(), row_em)
    assert torch.equal(got["expert_offsets"].cpu(), ref_torch.expert_offsets(rm))
    assert torch.equal(got["src_token"].cpu().long(), rm.t().nonzero()[:, 1])


@pytest.mark.parametrize("E", [320, 321, 384, 385, 448, 449, 512])
@pytest.mark.parametrize("levels", [2, 0])
def test_topk_one_or_two_of_many_rows(pkg, dev, E, levels):
    # From 1024 rows on, lists of 6 to 8 elements a lane are searched for k = 1 and 2 and sorted for more; ties and special
    # values as above. The router's fused top-k takes the same forms on its own logits.
    g = torch.Generator().manual_seed(E + levels)
    T = 1025
    x = torch.randint(0, levels, (T, E), generator=g).float() if levels else torch.randn(T, E, generator=g)
    special = torch.tensor([0.0, -0.0, float("inf"), float("-inf"), float("nan"), 3.4e38])
    hit = torch.rand(T, E, generator=g) < 0.02
    x[hit] = special[torch.randint(0, 6, (int(hit.sum()),), generator=g)]
    inp = torch.randn(T, 64, generator=g).to(torch.bfloat16).to(dev)
    weight = (torch.randint(0, 3, (E, 64), generator=g) - 1).to(torch.bfloat16).to(dev) if levels else torch.randn(E, 64, generator=g).to(torch.bfloat16).to(dev)
    logits = pkg.ops.router_logits(inp, weight)
    for k in (1, 2, 3):
        for rows in (T, 1023):
            values, indices, mask = pkg.ops.topk(x[:rows].to(dev), k, with_mask=True)
            rv, ri = ref_torch.topk(x[:rows], k)
            assert torch.equal(indices.cpu(), ri), f"E={E} k={k} rows={rows}"
            assert_bits_equal(values, rv, f"E={E} k={k} rows={rows}")
            assert torch.equal(mask.cpu(), torch.zeros(rows, E, dtype=torch.bool).scatter_(1, ri, True))
        fused = pkg.ops.router_topk(inp, weight, k)
        rv, ri = ref_torch.topk(logits.cpu(), k)
        assert torch.equal(fused[1].cpu(), ri), f"fused E={E} k={k}"
        assert_bits_equal(fused[0], rv, f"fused E={E} k={k}")
