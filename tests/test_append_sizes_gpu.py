"""paged_kv_append at the sizes where its split over workgroups changes: rows
of one 16-byte piece (64 rows per workgroup) up to rows of several workgroup
passes (one row per workgroup), and batches around the size whose prefix sums
fit LDS.  Bytes are copied, so the caches equal a host scatter bit for bit."""

import pytest
import torch

import workloads as W

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need an MI355X")
    from kernels import _fa2
    _fa2.lib()
    yield


@pytest.mark.parametrize("B,H,D,dtype", [(7, 1, 8, torch.bfloat16), (7, 2, 64, torch.float16),
                                         (5, 8, 128, torch.bfloat16), (3, 40, 256, torch.float32),
                                         (511, 1, 64, torch.bfloat16), (512, 1, 64, torch.bfloat16),
                                         (513, 1, 64, torch.bfloat16)])
def test_append_equals_host_scatter(B, H, D, dtype):
    from kernels.paged_cache import paged_kv_append
    page = 16
    g = torch.Generator().manual_seed(B + H)
    add = torch.randint(0, 70 if B < 100 else 4, (B,), generator=g).tolist()
    start = torch.randint(0, 40, (B,), generator=g, dtype=torch.int32)
    width = (40 + 70) // page + 1
    pages = B * width
    tables = [torch.randperm(pages, generator=g).to(torch.int32).view(B, width) for _ in range(2)]
    new = [torch.randn((sum(add), H, D), generator=g).to(dtype) for _ in range(2)]
    caches = [torch.zeros((pages * page, H, D), dtype=dtype) for _ in range(2)]
    dev = [c.to(DEV) for c in caches]
    paged_kv_append(dev[0], dev[1], tables[0].to(DEV), tables[1].to(DEV), new[0].to(DEV),
                    new[1].to(DEV), W.indptr(add).to(DEV), page, start_pos=start.to(DEV))
    torch.cuda.synchronize()
    at = 0
    for b, n in enumerate(add):
        pos = int(start[b]) + torch.arange(n)
        for c, t, x in zip(caches, tables, new):
            c[t[b].long()[pos // page] * page + pos % page] = x[at:at + n]
        at += n
    assert all(torch.equal(d.cpu(), c) for d, c in zip(dev, caches))
