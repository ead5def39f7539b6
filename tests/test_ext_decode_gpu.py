"""The two launch paths of the decode entry points and of paged_kv_append (the
C++ extension and ctypes) enqueue the same library call with the same
parameters: bit-equal outputs and the same errors."""

import pytest
import torch

import workloads as W
from decode_cases import LAYOUTS, make_decode_case, pack_decode

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need an MI355X")
    from kernels import _launch
    assert _launch.ext() is not None, _launch._EXT_ERROR
    yield


def both(module, fn):
    module.USE_EXT = True
    a = fn()
    module.USE_EXT = False
    try:
        b = fn()
    finally:
        module.USE_EXT = True
    torch.cuda.synchronize()
    return a, b


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,splits", [(1, 0), (1, 3), (5, 0)])
def test_decode_extension_equals_ctypes(layout, dtype, M, splits):
    import kernels.decode as D
    from kernels import decode_attention, speculative_decode_attention
    case = make_decode_case(4, 8, 2, 128, M, dtype, layout, seed=7300 + M, causal=M > 1,
                            kv_range=(1, 900))
    q, k, v, kw = pack_decode(case, layout, device=DEV, squeeze_m=M == 1,
                              cache4d=layout == "paged")
    if M == 1:
        fn = lambda: decode_attention(q, k, v, num_splits=splits, **kw)  # noqa: E731
    else:
        # heads-inner strides: the wrapper copies q
        qt = q.transpose(1, 2).contiguous().transpose(1, 2)
        fn = lambda: speculative_decode_attention(qt, k, v, causal=True, **kw)  # noqa: E731
    a, b = both(D, fn)
    assert a.stride() == b.stride() and torch.equal(a, b)


def test_decode_extension_reports_the_librarys_errors():
    from kernels import _fa2, decode_attention
    q = torch.randn((2, 4, 64), device=DEV, dtype=torch.float16)
    k = torch.randn((2, 2, 10, 64), device=DEV, dtype=torch.float16)
    with pytest.raises(_fa2.Fa2Error) as e:
        decode_attention(q, k, k, num_splits=65)
    assert e.value.code == 11


@pytest.mark.parametrize("with_v,start", [(True, True), (False, False)])
def test_append_extension_equals_ctypes(with_v, start):
    import kernels.paged_cache as P
    g = torch.Generator().manual_seed(5)
    add, page = [3, 0, 20], 16
    new = torch.randn((sum(add), 4, 64), generator=g).to(torch.bfloat16).to(DEV)
    tbl = torch.randperm(12, generator=g).view(3, 4).to(DEV)  # int64: converted
    sp = torch.tensor([5, 0, 9], device=DEV) if start else None

    def run():
        kc = torch.zeros((12 * page, 4, 64), dtype=torch.bfloat16, device=DEV)
        vc = torch.zeros_like(kc) if with_v else None
        P.paged_kv_append(kc, vc, tbl, tbl.flip(0) if with_v else None, new,
                          new * 2 if with_v else None, W.indptr(add).to(DEV), page, start_pos=sp)
        return torch.stack([kc, vc]) if with_v else kc
    a, b = both(P, run)
    assert torch.equal(a, b) and bool((a != 0).any())
