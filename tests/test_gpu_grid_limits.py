"""Launches past a grid's y and z limits (65535 rows or KV heads), which number their units and
merges along x instead, and rows of 65536 tiles and more, whose split bounds are computed in 64
bits: against the fp32 oracle of the few distinct rows or heads that each case repeats."""
import math

import pytest
import torch

from oracle import attention as oracle
from paged_cases import assert_parity, make_case

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16


@pytest.mark.parametrize("rows", [65535, 65540])
@pytest.mark.parametrize("page,splits", [(16, 1), (16, 3), (24, 2)])
def test_many_rows(ext, gpu, rows, page, splits):
    lengths = [100, 1, 64, 97, 33, 0, 130]  # the distinct rows, in turn
    case = make_case(lengths, 2, 1, page, F16, seed=page + splits)
    n, of = len(lengths), torch.arange(rows) % len(lengths)
    dev = lambda x: x[of].contiguous().to(gpu)
    out = torch.full((rows, 2, 128), float("nan"), dtype=F16, device=gpu)
    ws = torch.empty(rows * 2 * splits * 130 if splits > 1 else 0, device=gpu)
    ext.paged_attention_masked(dev(case.q), case.k_pages.to(gpu), case.v_pages.to(gpu),
                               dev(case.block_table), dev(case.seq_lens), out, ws, max(lengths),
                               page, splits)
    ref = oracle.paged_decode(case.q, case.k_pages, case.v_pages, case.block_table, case.seq_lens,
                              torch.arange(n), torch.arange(n), n)
    ref[lengths.index(0)] = 0.0
    assert_parity(out, ref[of])


@pytest.mark.parametrize("heads,splits", [(65535, 2), (65540, 1), (65540, 2)])
def test_many_kv_heads(ext, gpu, heads, splits):
    case = make_case([37, 70], 7, 7, 16, BF16, seed=heads)  # the distinct heads, in turn
    of = torch.arange(heads) % 7
    pool = lambda x: x.to(gpu)[:, of.to(gpu)].contiguous()
    out = torch.full((2, heads, 128), float("nan"), dtype=BF16, device=gpu)
    ws = torch.empty(2 * heads * splits * 130 if splits > 1 else 0, device=gpu)
    ext.paged_attention_masked(pool(case.q), pool(case.k_pages), pool(case.v_pages),
                               case.block_table.to(gpu), case.seq_lens.to(gpu), out, ws, 70, 16, splits)
    ref = oracle.paged_decode(case.q, case.k_pages, case.v_pages, case.block_table, case.seq_lens,
                              torch.arange(2), torch.arange(2), 2)
    assert_parity(out, ref[:, of])


@pytest.mark.parametrize("tiles,splits", [(65535, 65535), (65536, 65536), (65611, 65600), (65611, 7)])
def test_long_row_split_bounds(ext, gpu, tiles, splits):
    page, pages, hq = 64, 5, 2
    n = 32 * tiles - 9
    gen = torch.Generator().manual_seed(tiles)
    q = torch.randn(1, hq, 128, generator=gen).half()
    k, v = (torch.randn(pages, 1, page, 128, generator=gen).half() for _ in range(2))
    cols = -(-n // page)
    order = torch.arange(cols) * pages // cols  # each page fills a fifth of the row
    out = torch.empty(1, hq, 128, dtype=F16, device=gpu)
    ws = torch.full((hq * splits * 130,), float("nan"), device=gpu)
    ext.paged_attention_masked(q.to(gpu), k.to(gpu), v.to(gpu), order[None].to(torch.int32).to(gpu),
                               torch.tensor([n], dtype=torch.int32, device=gpu), out, ws, n, page, splits)
    # softmax over the distinct tokens, each as often as the row holds it
    count = torch.zeros(pages * page, dtype=torch.float64)
    tokens = order.repeat_interleave(page)[:n] * page + torch.arange(n) % page
    count.index_add_(0, tokens, torch.ones(n, dtype=torch.float64))
    p = torch.exp(q[0].double() @ k.reshape(-1, 128).double().T / math.sqrt(128)) * count
    ref = (p / p.sum(1, keepdim=True)) @ v.reshape(-1, 128).double()
    assert_parity(out, ref.float()[None])
