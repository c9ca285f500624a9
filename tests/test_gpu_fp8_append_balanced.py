"""The work-queue op with fp8 K/V and the append, on the balanced schedule, whose decode writes
each row's newest token itself: outputs and pools equal append_kv_fp8 followed by the op, bit
for bit, for newest tokens in the first, second and later tiles of a wave's range, values that
saturate, underflow, are infinite or NaN, and rows whose append is skipped (no tokens, a length
past the table, a page outside the pool)."""
import pytest
import torch

import pkv_native
from paged_cases import make_case

pytestmark = pytest.mark.gpu

F8 = torch.float8_e4m3fn


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lengths,hq,hkv,page", [
    ([1, 32, 33, 64, 65, 96, 97, 128, 161], 12, 3, 16),
    ([20000, 31, 5000, 700, 16, 17], 32, 8, 32),
    ([300] * 40, 16, 4, 64),
    ([33000], 8, 8, 16),
])
def test_equals_append_then_op(ext, gpu, dtype, lengths, hq, hkv, page):
    ks, vs, b = 0.05, 0.03, len(lengths)
    case = make_case(lengths, hq, hkv, page, torch.float16, seed=b + page)
    gen = torch.Generator().manual_seed(b)
    kn, vn = (torch.randn(b, hkv, 128, generator=gen) for _ in range(2))
    for x in (kn, vn):
        x[:, :, 3], x[:, :, 4], x[:, :, 5], x[:, :, 6] = 1e4, -1e4, 1e-5, -3e-4
    vn[b // 2, 0, 7], vn[b // 2, 0, 8], vn[b // 2, 0, 9] = float("inf"), float("nan"), -float("nan")
    kn, vn = kn.to(dtype).to(gpu), vn.to(dtype).to(gpu)
    meta = pkv_native.build_workqueue(lengths, list(range(b)), case.page_lists, page, 4, False, hkv)
    t = lambda x: torch.as_tensor(meta[x], dtype=torch.int32, device=gpu)
    floats = max(meta["total_partial_slots"] * hq * 130,
                 pkv_native.workqueue_balanced_workspace_bytes(b, hq, hkv) // 4)
    assert ext.workqueue_schedule(b, hq, hkv, page, floats, False) == 1
    table, lens = t("block_table"), t("seq_lens").clone()
    if b > 4:  # skipped appends: past the table (the row is read to the table's end), bad page
        lens[1] = table.shape[1] * page + 5
        table[2, (lengths[2] - 1) // page] = case.k_pages.shape[0] + 3
        lens[3] = 0
    results = []
    for fused in (True, False):
        k = (case.k_pages.float() / ks).clamp(-448, 448).to(F8).to(gpu)
        v = (case.v_pages.float() / vs).clamp(-448, 448).to(F8).to(gpu)
        ws = torch.full((floats,), float("nan"), device=gpu)
        out = torch.empty(b, hq, 128, dtype=dtype, device=gpu)
        args = (case.q.to(dtype).to(gpu), k, v, table, lens, t("work_items"), t("split_offsets"),
                torch.zeros(b, hkv, dtype=torch.int32, device=gpu), t("q_indices"), t("out_indices"),
                out, ws, meta["bucket_length"], page, meta["total_partial_slots"], False, ks, vs)
        if fused:
            ext.paged_attention_workqueue_fp8_append(*args, kn, vn)
        else:
            ext.append_kv_fp8(kn, vn, k, v, table, lens, ks, vs)
            ext.paged_attention_workqueue_fp8(*args)
        results.append([x.view(torch.int16 if x is out else torch.uint8).cpu() for x in (out, k, v)])
    for a, c in zip(*results):
        assert torch.equal(a, c)


def test_scales_are_checked_before_launch(ext, gpu):
    case = make_case([64], 8, 2, 16, torch.float16, seed=2)
    k, v = (torch.zeros(case.k_pages.shape, dtype=torch.uint8, device=gpu).view(F8) for _ in range(2))
    meta = pkv_native.build_workqueue([64], [0], case.page_lists, 16, 1, False, 2)
    t = lambda x: torch.as_tensor(meta[x], dtype=torch.int32, device=gpu)
    ws = torch.empty(pkv_native.workqueue_balanced_workspace_bytes(1, 8, 2) // 4, device=gpu)
    new = torch.ones(1, 2, 128, dtype=torch.float16, device=gpu)
    out = torch.zeros(1, 8, 128, dtype=torch.float16, device=gpu)
    for ks, vs in ((1.0, 0.0), (1.0, -1.0), (0.0, 1.0), (1.0, float("inf"))):
        with pytest.raises(RuntimeError, match="finite"):
            ext.paged_attention_workqueue_fp8_append(
                case.q.to(gpu), k, v, t("block_table"), t("seq_lens"), t("work_items"),
                t("split_offsets"), torch.zeros(1, 2, dtype=torch.int32, device=gpu), t("q_indices"),
                t("out_indices"), out, ws, 64, 16, meta["total_partial_slots"], False, ks, vs, new, new)
    torch.cuda.synchronize()
    assert not k.view(torch.uint8).any() and not out.any()
