"""Launches of at most one unit per CU on the whole-line K path, at the edges of its rule on a
256-CU card: units of 32 output dims (up to 64 units), of 64 (up to 128) and undivided (up to
224, or 256 for rows of their own lengths), with unit counts that are not multiples of 8, rows
that are empty, of one or two tiles, of odd and even tile counts and ending inside a tile, over
paged, contiguous and appending K/V, unsplit and split, against the fp32 oracle.  The appending
ops also equal the append followed by the op bit for bit, outputs and pools."""
import pytest
import torch

from oracle import attention as oracle
from paged_cases import assert_parity, make_case

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16
EDGES = [0, 1, 32, 33, 64, 65, 96, 127, 640, 1023, 1555]


def _lengths(batch):
    return [EDGES[(3 * i + 10) % len(EDGES)] for i in range(batch)]


# (batch, Hq, Hkv, dtype, splits): batch * Hkv * splits units
SHAPES = [
    (3, 24, 6, F16, 1), (11, 80, 5, BF16, 1),      # 4 slices, G = 4 and 16
    (13, 25, 5, F16, 1), (16, 8, 8, BF16, 1),      # 2 slices, 65 and 128 units, G = 5 and 1
    (43, 9, 3, F16, 1), (32, 32, 8, BF16, 1),      # undivided, 129 and 256 units
    (5, 8, 2, F16, 3), (7, 16, 4, BF16, 3), (11, 12, 4, F16, 3), (16, 16, 8, BF16, 2),
]


@pytest.mark.parametrize("batch,hq,hkv,dtype,splits", SHAPES)
def test_masked(ext, gpu, batch, hq, hkv, dtype, splits):
    lengths = _lengths(batch)
    case = make_case(lengths, hq, hkv, 16, dtype, seed=batch + splits)
    ctx = max(lengths)
    out = torch.full((batch, hq, 128), float("nan"), dtype=dtype, device=gpu)
    ws = torch.empty(batch * hq * splits * 130 if splits > 1 else 0, device=gpu)
    ext.paged_attention_masked(case.q.to(gpu), case.k_pages.to(gpu), case.v_pages.to(gpu),
                               case.block_table.to(gpu), case.seq_lens.to(gpu), out, ws, ctx, 16,
                               splits)
    ref = oracle.paged_decode(case.q, case.k_pages, case.v_pages, case.block_table, case.seq_lens,
                              torch.arange(batch), torch.arange(batch), batch)
    ref[[i for i, n in enumerate(lengths) if n == 0]] = 0.0
    assert_parity(out, ref)


@pytest.mark.parametrize("batch,hq,hkv,dtype,splits", SHAPES)
def test_append_equals_append_then_op(ext, gpu, batch, hq, hkv, dtype, splits):
    lengths = _lengths(batch)
    case = make_case(lengths, hq, hkv, 32, dtype, seed=7 * batch + splits)
    gen = torch.Generator().manual_seed(batch)
    kn, vn = (torch.randn(batch, hkv, 128, generator=gen).to(dtype).to(gpu) for _ in range(2))
    q, bt, sl = case.q.to(gpu), case.block_table.to(gpu), case.seq_lens.to(gpu)
    ws = torch.empty(batch * hq * splits * 130 if splits > 1 else 0, device=gpu)
    results = []
    for fused in (True, False):
        k, v = case.k_pages.to(gpu).clone(), case.v_pages.to(gpu).clone()
        out = torch.full((batch, hq, 128), float("nan"), dtype=dtype, device=gpu)
        args = (q, k, v, bt, sl, out, ws, max(lengths), 32, splits)
        if fused:
            ext.paged_attention_masked_append(*args, kn, vn)
        else:
            ext.append_kv(kn, vn, k, v, bt, sl)
            ext.paged_attention_masked(*args)
        results.append((out, k, v))
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize("batch,hq,hkv,n,dtype", [
    (3, 12, 3, 545, F16), (10, 64, 8, 1000, BF16), (27, 40, 8, 1555, F16), (1, 48, 3, 33000, BF16)])
def test_contiguous(ext, gpu, batch, hq, hkv, n, dtype):
    gen = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(*s, 128, generator=gen).to(dtype)
               for s in ((batch, hq), (batch, hkv, n), (batch, hkv, n)))
    out = torch.full((batch, hq, 128), float("nan"), dtype=dtype, device=gpu)
    ext.attention_contiguous(q.to(gpu), k.to(gpu), v.to(gpu), out, torch.empty(0, device=gpu), 1)
    ref = torch.stack([oracle.sdpa_row(q[b], k[b], v[b]) for b in range(batch)])
    assert_parity(out, ref)
