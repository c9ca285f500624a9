"""Unsplit calls of few units whose output is one of their own inputs: q itself, or (Hq = Hkv)
the new tokens' rows.  A unit's rows are read before its output is written, so such a call
gives what the call with an output of its own gives.  Units shared out over several workgroups
would break that where one of them starts after another has finished, so each call here runs
while a launch on a second stream holds every CU and lets go of them one after the other."""
import pytest
import torch

from oracle import attention as oracle
from paged_cases import assert_parity, make_case

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16


class Busy:
    """256 workgroups, one per CU, over rows of 512 to 16384 tokens, on a stream of their own."""

    def __init__(self, ext, gpu):
        self.ext, self.stream = ext, torch.cuda.Stream()
        rows, hkv, pages = 32, 8, 1024
        self.q = torch.randn(rows, hkv, 128, device=gpu).half()
        self.k = torch.randn(pages, hkv, 16, 128, device=gpu).half()
        self.v = torch.randn(pages, hkv, 16, 128, device=gpu).half()
        self.table = torch.arange(pages, dtype=torch.int32, device=gpu).repeat(rows, 1)
        self.lens = torch.arange(1, rows + 1, dtype=torch.int32, device=gpu) * 512
        self.out = torch.empty_like(self.q)
        self.ws = torch.empty(0, device=gpu)
        torch.cuda.synchronize()

    def start(self):
        with torch.cuda.stream(self.stream):
            self.ext.paged_attention_masked(self.q, self.k, self.v, self.table, self.lens, self.out,
                                            self.ws, 16384, 16, 1)


@pytest.fixture(scope="module")
def busy(ext, gpu):
    return Busy(ext, gpu)


def _lengths(batch):
    return [(700, 3, 1500, 64, 1023, 545)[i % 6] for i in range(batch)]


# batch * Hkv units: 4 and 2 workgroups per unit up to 64 and 128 units on a 256-CU card
SHAPES = [(1, 32, 8, 16, F16), (3, 24, 6, 32, BF16), (8, 40, 8, 16, F16), (13, 25, 5, 16, BF16),
          (16, 8, 8, 16, F16), (2, 16, 8, 24, F16)]


@pytest.mark.parametrize("batch,hq,hkv,page,dtype", SHAPES)
def test_output_is_q(ext, gpu, busy, batch, hq, hkv, page, dtype):
    lengths = _lengths(batch)
    case = make_case(lengths, hq, hkv, page, dtype, seed=batch)
    q, k, v = case.q.to(gpu), case.k_pages.to(gpu), case.v_pages.to(gpu)
    bt, sl = case.block_table.to(gpu), case.seq_lens.to(gpu)
    ws, apart = torch.empty(0, device=gpu), torch.empty_like(q)
    ext.paged_attention_masked(q, k, v, bt, sl, apart, ws, max(lengths), page, 1)
    ref = oracle.paged_decode(case.q, case.k_pages, case.v_pages, case.block_table, case.seq_lens,
                              torch.arange(batch), torch.arange(batch), batch)
    assert_parity(apart, ref)
    for _ in range(4):
        both = q.clone()
        torch.cuda.synchronize()
        busy.start()
        ext.paged_attention_masked(both, k, v, bt, sl, both, ws, max(lengths), page, 1)
        torch.cuda.synchronize()
        if page % 16 == 0:
            assert torch.equal(both, apart)
        else:  # other waves share out an odd page size's rows when the unit is undivided
            assert_parity(both, ref)


@pytest.mark.parametrize("batch,hq,hkv,n,dtype", [(1, 32, 8, 2048, F16), (12, 30, 10, 600, BF16)])
def test_contiguous_output_is_q(ext, gpu, busy, batch, hq, hkv, n, dtype):
    gen = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(*s, 128, generator=gen).to(dtype).to(gpu)
               for s in ((batch, hq), (batch, hkv, n), (batch, hkv, n)))
    apart, ws = torch.empty_like(q), torch.empty(0, device=gpu)
    ext.attention_contiguous(q, k, v, apart, ws, 1)
    for _ in range(4):
        both = q.clone()
        torch.cuda.synchronize()
        busy.start()
        ext.attention_contiguous(both, k, v, both, ws, 1)
        torch.cuda.synchronize()
        assert torch.equal(both, apart)


@pytest.mark.parametrize("which", ["q", "k_new", "v_new"])
def test_append_output_is_an_input(ext, gpu, busy, which):
    lengths, heads = _lengths(6), 16
    case = make_case(lengths, heads, heads, 16, F16, seed=5)
    gen = torch.Generator().manual_seed(6)
    kn, vn = (torch.randn(6, heads, 128, generator=gen).half().to(gpu) for _ in range(2))
    bt, sl, ws = case.block_table.to(gpu), case.seq_lens.to(gpu), torch.empty(0, device=gpu)

    def step(shared):
        rows = {"q": case.q.to(gpu), "k_new": kn.clone(), "v_new": vn.clone()}
        k, v = case.k_pages.to(gpu), case.v_pages.to(gpu)
        out = rows[which] if shared else torch.empty_like(rows["q"])
        torch.cuda.synchronize()
        busy.start()
        ext.paged_attention_masked_append(rows["q"], k, v, bt, sl, out, ws, max(lengths), 16, 1,
                                          rows["k_new"], rows["v_new"])
        torch.cuda.synchronize()
        return out, k, v

    apart = step(False)
    for _ in range(4):
        for a, b in zip(step(True), apart):
            assert torch.equal(a, b)
