"""fp32 tensors of flash_attention_v2 on the 16-bit kernels, which round Q
themselves (one head per workgroup) or read a copy (two heads) and write the
fp32 output: partial q-blocks and waves, several units per workgroup with the
next unit prefetched across the output stores, splits.  A capped grid keeps the
two-head kernel and must equal the uncapped one-head kernel bit for bit; both
pass the bars of test_attention_gpu.py."""

import pytest
import torch

from attn_cases import make_case, pack, unpack
from test_attention_gpu import check_all

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need an MI355X")
    from kernels import _fa2
    _fa2.lib()
    yield


@pytest.mark.parametrize("splits", [0, 2])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("layout", ["dense", "ragged"])
def test_capped_grids_equal_the_one_head_kernel(layout, D, causal, splits):
    from kernels import flash_attention_v2
    case = make_case(3, 8, 2, D, "self", torch.float32, layout, 8100 + D,
                     q_range=(1, 420), dense_q_range=(333, 333))
    q, k, v, kw = pack(case, layout, device=DEV)
    outs = [flash_attention_v2(q, k, v, is_causal=causal, max_workgroups=w, num_splits=splits, **kw)
            for w in (0, 1, 8)]
    torch.cuda.synchronize()
    assert all(torch.equal(outs[0].view(torch.int32), o.view(torch.int32)) for o in outs[1:])
    check_all(case, layout, causal, unpack(case, layout, outs[0].cpu(), kw))
