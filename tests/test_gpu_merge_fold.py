"""The merges at the sizes where their fold changes: state counts around a pair (1, 2, 3), a row
of lanes (16, 17), a chunk of 32 (31, 32, 33) and several chunks, at odd head counts, for the
grid-split ops (num_splits given; every split written) and the work queue's per-item schedule
(pages of 8) and balanced one, with states that underflow to weight 0 (one split's scores 120
above the rest's, e^-120 < 2^-149), against the fp32 oracle.  The workspace holds NaN before
each call."""
import pytest
import torch

import pkv_native
from oracle import attention as oracle
from paged_cases import assert_parity, make_case

pytestmark = pytest.mark.gpu


def _split_weights(case, row, head, kv_head, splits):
    """fp32 merge weights of the row's non-empty splits, exp(m_s - max m)."""
    n, ps = int(case.seq_lens[row]), case.page_size
    k = case.k_pages[case.page_lists[row], kv_head].float().reshape(-1, 128)[:n]
    scores = k @ case.q[row, head].float() / 128 ** 0.5
    tiles = -(-n // 32)
    ends = [32 * (tiles * s // splits) for s in range(splits + 1)]
    m = torch.stack([scores[a:b].max() for a, b in zip(ends, ends[1:]) if a < min(b, n)])
    return torch.exp(m - m.max())


def _case(lengths, hq, hkv, dtype, seed, spike, splits, page=16):
    case = make_case(lengths, hq, hkv, page, dtype, seed=seed)
    if spike:  # one page of each row along its queries' direction: the other splits underflow
        for row, pages in enumerate(case.page_lists):
            for h in range(hkv):
                q = case.q[row, h * (hq // hkv)].float()
                case.k_pages[pages[len(pages) // 2], h, 3] = (q * (1400.0 / q.dot(q))).to(dtype)
        w = _split_weights(case, lengths.index(max(lengths)), 0, 0, splits)
        assert len(w) == 1 or (w == 0).any()
    n = len(lengths)
    ref = oracle.paged_decode(case.q, case.k_pages, case.v_pages, case.block_table, case.seq_lens,
                              torch.arange(n), torch.arange(n), n)
    return case, ref


@pytest.mark.parametrize("splits", [2, 3, 16, 17, 31, 32, 33, 65, 100])
@pytest.mark.parametrize("dtype,spike", [(torch.float16, False), (torch.bfloat16, True)])
def test_grid_split(ext, gpu, splits, dtype, spike):
    lengths, hq, hkv = [32 * splits, 32 * splits + 77, 3300], 15, 3
    case, ref = _case(lengths, hq, hkv, dtype, splits, spike, splits)
    out = torch.empty(3, hq, 128, dtype=dtype, device=gpu)
    ws = torch.full((3 * hq * splits * 130,), float("nan"), device=gpu)
    ext.paged_attention_masked(case.q.to(gpu), case.k_pages.to(gpu), case.v_pages.to(gpu),
                               case.block_table.to(gpu), case.seq_lens.to(gpu), out, ws, max(lengths),
                               16, splits)
    assert_parity(out, ref)


@pytest.mark.parametrize("splits", [1, 2, 17, 33, 70])
@pytest.mark.parametrize("balanced", [False, True])
@pytest.mark.parametrize("spike", [False, True])
def test_work_queue(ext, gpu, splits, balanced, spike):
    # 40 tokens: fewer tiles than splits, so empty slots hold NaN and must be skipped
    lengths, hq, hkv, page = [40, 5000, 1, 2600], 12, 4, 16 if balanced else 8
    case, ref = _case(lengths, hq, hkv, torch.float16, splits, spike, splits, page)
    b = len(lengths)
    meta = pkv_native.build_workqueue(lengths, list(range(b)), case.page_lists, page, splits, False, hkv)
    t = lambda x: torch.as_tensor(meta[x], dtype=torch.int32, device=gpu)
    floats = meta["total_partial_slots"] * hq * 130
    if balanced:
        floats = max(floats, pkv_native.workqueue_balanced_workspace_bytes(b, hq, hkv) // 4)
    assert ext.workqueue_schedule(b, hq, hkv, page, floats, False) == int(balanced)
    ws = torch.full((floats,), float("nan"), device=gpu)
    out = torch.empty(b, hq, 128, dtype=torch.float16, device=gpu)
    ext.paged_attention_workqueue(
        case.q.to(gpu), case.k_pages.to(gpu), case.v_pages.to(gpu), t("block_table"), t("seq_lens"),
        t("work_items"), t("split_offsets"), torch.zeros(b, hkv, dtype=torch.int32, device=gpu),
        t("q_indices"), t("out_indices"), out, ws, meta["bucket_length"], page,
        meta["total_partial_slots"], False)
    assert_parity(out, ref)
