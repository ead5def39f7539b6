"""GPU checks of the decode kernels' balanced walk (csrc/fa2_decode_walk.h) at
the sizes where it can go wrong: lengths around the 16-key wave tiles and the
64-key tiles the cuts count in, empty sequences, units cut into many pieces,
row counts around the 16-row blocks and several blocks per unit.

Every case passes the bars of test_decode_gpu.py (the reference tolerance, and
errors against fp64 within 4x / 2x of the reference arithmetic's).  A forced
split count runs one split per workgroup instead of the walk; the two differ
by the order of fp32 sums (and, in 16 bits, by softmax weights rounded after
different maxima), so they agree within the strict bar's own floor.
"""

import pytest
import torch

from decode_cases import LAYOUTS, make_decode_case, pack_decode
from test_decode_gpu import check, run

pytestmark = pytest.mark.gpu

LENS = [0, 1, 15, 16, 17, 63, 64, 65, 300, 1100, 0]


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need an MI355X")
    from kernels import _fa2
    _fa2.lib()
    yield


def lens_of(layout):
    return [1100] * 3 if layout == "dense" else LENS


@pytest.mark.parametrize("heads,M", [((4, 4), 1), ((16, 4), 4), ((17, 1), 1), ((8, 2), 8),
                                     ((33, 1), 1), ((8, 1), 8)],
                         ids=["rows1", "rows16", "rows17", "rows32", "rows33", "rows64"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_walk_rows_and_lengths_f32(layout, D, heads, M):
    QH, KVH = heads
    case = make_decode_case(len(lens_of(layout)), QH, KVH, D, M, torch.float32, layout, seed=5100,
                            causal=M > 1, ctx_lens=lens_of(layout))
    check(case, layout, run(case, layout))


@pytest.mark.parametrize("page", [1, 5, 16, 64])
def test_walk_page_sizes_f32(page):
    case = make_decode_case(6, 8, 2, 128, 2, torch.float32, "paged", seed=5200 + page,
                            causal=True, kv_range=(1, 700))
    check(case, "paged", run(case, "paged", shuffled=True, page=page))


@pytest.mark.parametrize("n", [130, 5000])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_walk_one_sequence_in_many_pieces_f32(layout, n):
    """One unit per kv head: every segment cuts it (up to 40 pieces)."""
    case = make_decode_case(1, 8, 2, 64, 1, torch.float32, layout, seed=5300, ctx_lens=[n])
    a = run(case, layout, decode=True)
    check(case, layout, a)
    b = run(case, layout, decode=True)
    assert all(torch.equal(x, y) for x, y in zip(a, b))
    c = run(case, layout, decode=True, num_splits=3)
    for x, y in zip(a, c):  # 5000 fp32 additions of rounding 2^-24, either order
        torch.testing.assert_close(x, y, rtol=0, atol=5000 ** 0.5 * 2.0 ** -24 * 4)


# ---- 16-bit: units of up to 16 rows on the wave-streaming kernel (17: the ring kernel) ----

@pytest.mark.parametrize("heads,M", [((4, 4), 1), ((8, 2), 1), ((10, 2), 1), ((16, 4), 4),
                                     ((17, 1), 1)],
                         ids=["rows1", "rows4", "rows5", "rows16", "rows17"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_walk_rows_and_lengths_16bit(layout, D, heads, M):
    QH, KVH = heads
    dt = torch.bfloat16 if D == 128 else torch.float16
    case = make_decode_case(len(lens_of(layout)), QH, KVH, D, M, dt, layout, seed=5400,
                            causal=M > 1, ctx_lens=lens_of(layout))
    check(case, layout, run(case, layout))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("page", [1, 2, 5, 8, 64])
def test_walk_page_sizes_16bit(page, D):
    """Pages below and above the rows of one load, a size that is no power of two,
    and (64 streams of long segments, one-row pages) windows of the table."""
    heads = 64 if page == 1 else 4
    case = make_decode_case(2, heads, heads, D, 2, torch.bfloat16, "paged", seed=5500 + page,
                            causal=True, ctx_lens=[1500, 700])
    check(case, "paged", run(case, "paged", shuffled=True, page=page))


@pytest.mark.parametrize("n", [130, 5000])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_walk_one_sequence_in_many_pieces_16bit(layout, n):
    case = make_decode_case(1, 8, 2, 128, 1, torch.bfloat16, layout, seed=5600, ctx_lens=[n])
    a = run(case, layout, decode=True)
    check(case, layout, a)
    assert all(torch.equal(x, y) for x, y in zip(a, run(case, layout, decode=True)))


# ---- short units, which stay whole: up to 12 tiles of 64 keys in 16 bits, 4 in fp32 (6: cut) ----

@pytest.mark.parametrize("dt,top", [(torch.bfloat16, 12 * 64), (torch.float16, 12 * 64),
                                    (torch.float32, 6 * 64), (torch.float32, 4 * 64)],
                         ids=["bf16", "fp16", "fp32", "fp32-4"])
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("past", [0, 1], ids=["whole", "cut"])
def test_short_units_stay_whole(layout, dt, top, past):
    """The longest unit at the limit and one key past it; 128 kv heads leave two
    segments per stream, so that a workgroup walks several units."""
    lens = [top + past] * 5 if layout == "dense" else [top + past, 0, 1, 64, 65, 300, 17, 0, 130]
    case = make_decode_case(len(lens), 128, 128, 64, 2, dt, layout, seed=5700, ctx_lens=lens)
    check(case, layout, run(case, layout))


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("QH,KVH,n", [(5, 5, 200), (12, 12, 700), (48, 48, 230), (3, 3, 1900)])
def test_streams_that_do_not_divide_the_grid(layout, dt, QH, KVH, n):
    """Whole units that go round all workgroups (fp32: also those past the
    streams' segments), and units long enough to be cut."""
    lens = [n] * 11 if layout == "dense" else [max(0, n - 37 * i) for i in range(11)]
    case = make_decode_case(len(lens), QH, KVH, 64, 1, dt, layout, seed=5750 + KVH, ctx_lens=lens)
    check(case, layout, run(case, layout, decode=True))


# ---- fp32 calls of many units: four-wave workgroups, blocks of 64 rows ----

@pytest.mark.parametrize("heads,M", [((6, 6), 1), ((24, 6), 4), ((8, 1), 8), ((33, 1), 1),
                                     ((16, 1), 8), ((18, 2), 5)],
                         ids=["rows1", "rows16", "rows64", "rows33", "rows128", "rows45"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("splits", [0, 3])
def test_many_units_f32(layout, D, heads, M, splits):
    """Over 3/2 units per CU with up to 16 rows, and over 1/2 per CU of 64 rows."""
    QH, KVH = heads
    B = 130 if QH // KVH * M > 16 else 70
    lens = [330] * B if layout == "dense" else [LENS[:-1][i % 10] if i % 13 else 700 + i
                                               for i in range(B)]
    case = make_decode_case(B, QH, KVH, D, M, torch.float32, layout, seed=5850 + M, causal=M > 1,
                            ctx_lens=lens)
    check(case, layout, run(case, layout, num_splits=splits))


# ---- more sequences than lanes: several per lane of the locating wave ----

@pytest.mark.parametrize("B", [65, 129, 700])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("layout", ["ragged", "paged"])
def test_cut_units_among_many_sequences(layout, dt, B):
    """Mostly short and empty sequences and a few of 47 tiles, which are cut: the
    starts of the segments lie inside the lanes' groups of sequences."""
    lens = [7 * i % 40 for i in range(B)]
    for i in (0, 3, B // 2, B - 2):
        lens[i] = 3000 + i % 64
    case = make_decode_case(B, 4, 2, 64, 1, dt, layout, seed=5900 + B, ctx_lens=lens)
    check(case, layout, run(case, layout, decode=True))


@pytest.mark.parametrize("B", [4096, 4097])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
def test_cut_units_among_thousands_of_sequences(dt, B):
    lens = [i % 3 for i in range(B)]
    lens[B // 2] = 3000
    case = make_decode_case(B, 2, 2, 64, 1, dt, "ragged", seed=5950 + B, ctx_lens=lens)
    check(case, "ragged", run(case, "ragged", decode=True))


@pytest.mark.parametrize("B", [65536, 65537])
@pytest.mark.parametrize("dt", [torch.float16, torch.float32], ids=["fp16", "fp32"])
def test_sequences_at_the_walks_limit(dt, B):
    """One past it the other decode kernels run, with a plan by list (dense: none)."""
    from kernels import decode_attention
    g = torch.Generator().manual_seed(B)
    q, k, v = (torch.randn(s, generator=g).to(dt) for s in ((B, 2, 64), (B, 1, 3, 64), (B, 1, 3, 64)))
    out = decode_attention(q.cuda(), k.cuda(), v.cuda()).cpu().double()
    s = torch.matmul(q.double(), k[:, 0].double().transpose(1, 2).contiguous()) / 8
    ref = torch.matmul(torch.softmax(s, -1), v[:, 0].double())
    # fp16: weights and output rounded to 11 bits, |v| < 6; fp32: a few ulps of it
    assert (out - ref).abs().max().item() < (6 * 2.0 ** -9 if dt == torch.float16 else 1e-5)


# ---- strides: heads outside the rows ----

@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("M", [1, 3])
def test_strided_caches_equal_contiguous_ones(layout, D, dt, M):
    """Head-major pools and token rows, dense K and V as views of [B, N, H, D], a K
    whose rows lie further apart than V's: no copy is made, the same bits."""
    from kernels import speculative_decode_attention
    lens = [1100] * 3 if layout == "dense" else LENS
    case = make_decode_case(len(lens), 8, 4, D, M, dt, layout, seed=5980 + M, causal=M > 1,
                            ctx_lens=lens)
    pk = dict(shuffled=True, page=16) if layout == "paged" else {}
    q, k, v, kw = pack_decode(case, layout, device="cuda", **pk)
    a = speculative_decode_attention(q, k, v, causal=M > 1, **kw)
    i, j = (1, 2) if layout == "dense" else (0, 1)
    ks, vs = (t.transpose(i, j).contiguous().transpose(i, j) for t in (k, v))
    wide = torch.full((*k.shape[:-1], 3 * D), float("nan"), dtype=dt, device="cuda")
    wide[..., D:2 * D] = k
    for kk, vv in ((ks, vs), (ks, v), (wide[..., D:2 * D], vs)):
        b = speculative_decode_attention(q, kk, vv, causal=M > 1, **kw)
        # (an empty sequence's rows are NaN in both)
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(0), b.nan_to_num(0))
