"""Page sizes that are not multiples of 16 through every grid and queue launch shape, against
the fp32 oracle: pages of one token (64-entry table windows crossed every two tiles), pages
that split 16-token blocks unevenly, pages longer than a window, rows ending inside a tile,
and K/V past each row's end (in its last page and in pages of no row) holding NaN."""
import pytest
import torch

import pkv_native
from oracle import attention as oracle
from paged_cases import assert_parity, make_case

pytestmark = pytest.mark.gpu

LENGTHS = [2900, 1, 31, 33, 640, 1537, 65]


def _poisoned(page, hq, hkv, dtype, lengths, seed):
    """A case whose K/V hold NaN wherever no row has a token, and the clean oracle output."""
    case = make_case(lengths, hq, hkv, page, dtype, seed=seed)
    n = len(lengths)
    ref = oracle.paged_decode(case.q, case.k_pages, case.v_pages, case.block_table, case.seq_lens,
                              torch.arange(n), torch.arange(n), n)
    used = torch.zeros(case.k_pages.shape[0], page, dtype=torch.bool)
    for length, pages in zip(lengths, case.page_lists):
        for t in range(length):
            used[pages[t // page], t % page] = True
    for pool in (case.k_pages, case.v_pages):
        pool.masked_fill_(~used[:, None, :, None], float("nan"))
    return case, ref


@pytest.mark.parametrize("page", [1, 3, 8, 24, 100])
@pytest.mark.parametrize("hq,hkv,dtype,splits", [
    (8, 2, torch.float16, 1), (16, 2, torch.bfloat16, 3), (40, 2, torch.float16, 2),
    (64, 32, torch.float16, 4)])
def test_grid_ops(gpu, ext, page, hq, hkv, dtype, splits):
    case, ref = _poisoned(page, hq, hkv, dtype, LENGTHS, seed=page * 7 + splits)
    b, ctx = len(LENGTHS), max(LENGTHS)
    out = torch.empty(b, hq, 128, dtype=dtype, device=gpu)
    ws = torch.empty(b * hq * splits * 130 if splits > 1 else 0, device=gpu)
    ext.paged_attention_masked(case.q.to(gpu), case.k_pages.to(gpu), case.v_pages.to(gpu),
                               case.block_table.to(gpu), case.seq_lens.to(gpu), out, ws, ctx, page,
                               splits)
    assert_parity(out, ref)


@pytest.mark.parametrize("page", [1, 8, 40])
@pytest.mark.parametrize("hq", [8, 48])
def test_work_queue(gpu, ext, page, hq):
    hkv = 2
    case, ref = _poisoned(page, hq, hkv, torch.float16, LENGTHS, seed=page)
    b = len(LENGTHS)
    meta = pkv_native.build_workqueue(LENGTHS, list(range(b)), case.page_lists, page, 6, False, hkv)
    t = lambda x: torch.as_tensor(meta[x], dtype=torch.int32, device=gpu)
    out = torch.empty(b, hq, 128, dtype=torch.float16, device=gpu)
    ws = torch.empty(meta["total_partial_slots"] * hq * 130, device=gpu)
    counters = torch.zeros(b, hkv, dtype=torch.int32, device=gpu)
    ext.paged_attention_workqueue(
        case.q.to(gpu), case.k_pages.to(gpu), case.v_pages.to(gpu), t("block_table"),
        t("seq_lens"), t("work_items"), t("split_offsets"), counters, t("q_indices"),
        t("out_indices"), out, ws, meta["bucket_length"], page, meta["total_partial_slots"], False)
    assert_parity(out, ref)


@pytest.mark.parametrize("page", [1, 8, 24, 100])
@pytest.mark.parametrize("lengths,hq,hkv,splits", [
    ([2000, 0, 33, 1555], 12, 3, 1),   # 12 units: slices of 32 dims
    ([700, 1, 64, 640, 513] * 4, 20, 5, 1),  # 100 units: slices of 64 dims
    ([4000, 97], 32, 8, 4)])           # 64 units, split
def test_few_units(gpu, ext, page, lengths, hq, hkv, splits):
    """Launches that share the CUs out by output dims (at most half as many units as CUs)."""
    dtype = torch.bfloat16 if page == 8 else torch.float16
    case, ref = _poisoned(page, hq, hkv, dtype, lengths, seed=page + splits)
    b = len(lengths)
    out = torch.empty(b, hq, 128, dtype=dtype, device=gpu)
    ws = torch.empty(b * hq * splits * 130 if splits > 1 else 0, device=gpu)
    ext.paged_attention_masked(case.q.to(gpu), case.k_pages.to(gpu), case.v_pages.to(gpu),
                               case.block_table.to(gpu), case.seq_lens.to(gpu), out, ws,
                               max(lengths), page, splits)
    assert_parity(out, ref)
