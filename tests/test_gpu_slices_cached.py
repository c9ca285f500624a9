"""Few units over K/V that was just written, and so comes from the Infinity Cache, which a CU
reads almost twice as fast as HBM: units shared out over several workgroups must not take
longer there than undivided ones.  A call whose output is its q runs undivided, with the same
waves, and is the yardstick.  The shared-out calls take 0.81 and 0.80 of its time; with V's
lines fetched once for each of the two slices that share them they took 1.32 and 1.44."""
import statistics

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,n", [(8, 4096), (4, 9008)])
def test_no_slower_than_undivided(ext, gpu, rows, n):
    hkv, page = 8, 16
    pages = rows * n // page
    q = torch.randn(rows, 4 * hkv, 128, device=gpu).half()
    k, v = (torch.randn(pages, hkv, page, 128, device=gpu).half() for _ in range(2))
    table = torch.randperm(pages, device=gpu).to(torch.int32).reshape(rows, -1)
    out, ws = torch.empty_like(q), torch.empty(0, device=gpu)

    def took(target):
        times = []
        for i in range(24):
            k.neg_(), v.neg_()
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            ext.paged_attention(q, k, v, table, target, ws, n, page, 1)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return statistics.median(times[4:])

    apart, in_place = took(out), took(q)
    print(f"{rows * hkv} units of {n} tokens: {1e3 * apart:.1f} us, undivided {1e3 * in_place:.1f} us")
    assert apart < 1.1 * in_place
