"""fp32 attention whose scores are too large for their product with the softmax
scale to be rounded harmlessly (past 2^31 in log2 units an ulp of it is 2^8): the
largest weight must still be finite and not zero.

Such a row's softmax is one key's weight of 1: where the scores of the two
largest keys differ by more than fp32 sums can (2 D 2^-24 sum |q k|) and by more
than exp2 reaches (150), the output is that key's row of V, bit for bit, however
the keys are cut into pieces.
"""

import pytest
import torch

from decode_cases import LAYOUTS, make_decode_case
from test_decode_gpu import run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need an MI355X")
    from kernels import _fa2
    _fa2.lib()
    yield


def check_one_hot(q, k, v, out, off):
    """q/out [QH, M, D], k/v [N, KVH, D]; row i sees keys j <= i + off."""
    QH, M, D = q.shape
    N, KVH, _ = k.shape
    k = k.double().transpose(0, 1).repeat_interleave(QH // KVH, 0)
    v = v.transpose(0, 1).repeat_interleave(QH // KVH, 0)
    s = torch.matmul(q.double(), k.transpose(1, 2))
    err = 2 * D * 2.0 ** -24 * torch.matmul(q.double().abs(), k.abs().transpose(1, 2)).amax(-1)
    hide = torch.arange(N)[None, :] > torch.arange(M)[:, None] + off
    s = s.masked_fill(hide, float("-inf"))
    top, at = s.topk(min(2, N), -1)
    sure = torch.ones_like(top[..., 0], dtype=torch.bool)
    if N > 1:
        sure = top[..., 0] - top[..., 1] > err + 150 * D ** 0.5
    # (about one row in 700 falls below the bound at D = 256; cases have as few as 4)
    assert sure.double().mean() > 0.5
    expect = torch.gather(v, 1, at[..., :1].expand(-1, -1, D))
    assert torch.isfinite(out).all()
    assert torch.equal(out[sure], expect[sure])


def scaled_case(B, QH, KVH, D, M, layout, size, lens):
    case = make_decode_case(B, QH, KVH, D, M, torch.float32, layout, seed=8200 + M, causal=M > 1,
                            ctx_lens=lens)
    case.qs = [q * size for q in case.qs]
    case.ctx_k = [k * size for k in case.ctx_k]
    case.draft_k = [k * size for k in case.draft_k]
    return case


@pytest.mark.parametrize("splits", [0, 3], ids=["walk", "forced"])
@pytest.mark.parametrize("size", [5e4, 1e5])
@pytest.mark.parametrize("heads,M", [((4, 4), 1), ((8, 2), 1), ((4, 4), 8), ((8, 2), 8)],
                         ids=["rows1", "rows4", "rows8", "rows32"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_fp32_decode_of_large_scores(layout, D, heads, M, size, splits):
    lens = [1100] * 2 if layout == "dense" else [300, 5, 1100]
    case = scaled_case(len(lens), *heads, D, M, layout, size, lens)
    for b, out in enumerate(run(case, layout, num_splits=splits)):
        k = case.ks[b]
        check_one_hot(case.qs[b], k, case.vs[b], out, k.shape[0] - M if M > 1 else k.shape[0])


@pytest.mark.parametrize("splits", [0, 3], ids=["auto", "forced"])
@pytest.mark.parametrize("heads,M", [((4, 4), 1), ((8, 2), 8)], ids=["rows1", "rows32"])
@pytest.mark.parametrize("D", [16, 32, 256])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_fp32_decode_of_large_scores_other_head_dims(layout, D, heads, M, splits):
    test_fp32_decode_of_large_scores(layout, D, heads, M, 1e5, splits)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [16, 64, 128, 256])
def test_flash_attention_v1_of_large_scores(D, causal):
    from kernels import flash_attention_v1
    g = torch.Generator().manual_seed(8300 + D)
    q, k, v = (torch.randn((2, h, 300, D), generator=g) for h in (4, 2, 2))
    q, k = q * 1e5, k * 1e5
    out = flash_attention_v1(q.cuda(), k.cuda(), v.cuda(), is_causal=causal).cpu()
    for b in range(2):
        check_one_hot(q[b], k[b].transpose(0, 1), v[b].transpose(0, 1), out[b],
                      0 if causal else 300)
