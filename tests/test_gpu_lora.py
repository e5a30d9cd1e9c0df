"""The low-rank adapter delta on the GPU, through the C ABI, against the oracle.

Mirrors tests/ltx25-lora-apply-test.cc (layer one, :383-470): every shape of
its table, including the three the published adapters run (the x2
upscaler's rank 32 at 128 tokens over 4096 and 16384 columns, and the
distilled adapter's rank 450), with its bar -- rel-L2 < 2e-2 against f64 over
the unrounded draws -- and the north-star bar against the oracle, which
applies the same bf16 rounding of r: max|y - ref| / max|ref| <= 1e-2. Plus the
shapes that take the element-wise load path, an adapter wider than one launch
(rank > 512), the matrix-core GEMM pair (rank >= 96), the r-first route (many
tokens: r by the dense GEMM, then the fused kernel's second phase), the
empty-shape no-op and A = 0 (y bit-identical).
"""
import zlib

import numpy as np
import pytest
import torch

import orc
from gpu_util import dev_bf16, host_bits, say

pytestmark = pytest.mark.gpu

MAX_REL = 1e-2   # normwise max relative error vs the oracle
REL_L2 = 2e-2    # the reference's bar (tests/ltx25-lora-apply-test.cc:456-465)

F, RF, P = "fused", "rfirst", "pair"
SHAPES = [  # name, M, K, N, rank, the route AUTO takes
    ("square self-attention projection", 12, 64, 64, 3, F),
    ("cross-attention key (narrow in)", 8, 32, 64, 3, F),
    ("cross-attention key (wide in)", 12, 64, 32, 3, F),
    ("the per-head gate (4 columns out)", 12, 64, 4, 3, F),
    ("the feed-forward widening", 12, 64, 256, 5, F),
    ("rank 1", 6, 64, 64, 1, F),
    ("x2 upscaler: attn projection", 128, 4096, 4096, 32, F),
    ("x2 upscaler: ff widening", 128, 4096, 16384, 32, F),
    ("distilled adapter: rank 450", 64, 1024, 1024, 450, F),
    # beyond the reference's table
    ("odd K, odd N (element-wise loads)", 45, 37, 30, 6, F),
    ("video tokens, rank 64", 1000, 512, 768, 64, RF),
    ("two launches (rank 600)", 70, 256, 192, 600, F),
    ("two launches, padded rank (530)", 96, 256, 320, 530, F),
    ("N not a multiple of 8 (element-wise y)", 40, 128, 4100, 16, F),
    # the GEMM pair (M >= 256, rank >= 96): rank padded to 64 with zero rows / columns
    ("GEMM pair, rank 128, no padding", 300, 2048, 1024, 128, P),
    ("GEMM pair, rank 450 padded to 512", 512, 1024, 2048, 450, P),
    ("GEMM pair, ragged M and N", 777, 512, 1000, 200, P),
    ("GEMM pair, rank 1000", 256, 512, 640, 1000, P),
    # r first (M >= 512, rank % 8 == 0, rank < 96): r = x . A^T by the dense GEMM, then the
    # fused kernel's second phase reads it
    ("r first: rank 32 at the FFN width", 1024, 4096, 16384, 32, RF),
    ("r first: rank 40, ragged M", 777, 1024, 2048, 40, RF),
    ("r first: rank 8", 600, 512, 1024, 8, RF),
    # N not a multiple of the 512-column super-block stride: the y loads issued four
    # super blocks ahead (ranks up to 64) run past the column split's end
    ("r first: rank 16, ragged N", 640, 1024, 1000, 16, RF),
    ("r first: rank 64, N = 4104", 520, 256, 4104, 64, RF),
    # more rows, so more of r's panels; ragged M, a rank that is not a multiple of 16, K that is
    # not a multiple of 512
    ("r first, 2085 rows: rank 40, K = 2624", 2085, 2624, 1024, 40, RF),
    ("r first, 2112 rows: rank 8, K = 1088", 2112, 1088, 256, 8, RF),
    ("r first, 2048 rows: rank 64, K = 4096", 2048, 4096, 512, 64, RF),
]


def draws(tag, M, K, N, rank):
    rng = np.random.default_rng(zlib.crc32(tag.encode()))
    x = rng.standard_normal((M, K)).astype(np.float32)
    a = (rng.standard_normal((rank, K)) * 0.5).astype(np.float32)
    b = (rng.standard_normal((N, rank)) * 0.5).astype(np.float32)
    y = rng.standard_normal((M, N)).astype(np.float32)
    return x, a, b, y


def max_rel(got, ref):
    return float(np.max(np.abs(got - ref)) / max(np.max(np.abs(ref)), 1e-30))


ROUTE = {F: 3, RF: 2, P: 1}   # LTX25_LORA_FUSED / _RFIRST / _PAIR


def run_and_check(pkg, what, M, K, N, rank):
    x, a, b, y0 = draws(what, M, K, N, rank)
    xb, ab, bb, yb = (orc.bf16_rne(t) for t in (x, a, b, y0))
    xd, ad, bd, yd = (dev_bf16(t) for t in (xb, ab, bb, yb))
    route = pkg.lora_route(xd, ad, bd, yd, M, K, N, rank)
    pkg.lora_add(xd, ad, bd, yd, M, K, N, rank)
    torch.cuda.synchronize()
    got = orc.bf16_to_f32(host_bits(yd))
    ref = orc.bf16_to_f32(orc.lora_add(xb, ab, bb, yb))
    assert max_rel(got, ref) <= MAX_REL, what
    want = y0.astype(np.float64) + (x.astype(np.float64) @ a.T.astype(np.float64)) @ b.T
    assert orc.rel_l2(got, want) < REL_L2, what
    # and it ADDED: y changed where the delta is not negligible
    assert not np.array_equal(host_bits(yd), yb)
    return route


@pytest.mark.parametrize("what,M,K,N,rank,route", SHAPES, ids=[s[0] for s in SHAPES])
def test_lora_add_against_oracle_and_f64(pkg, dev, what, M, K, N, rank, route):
    say(f"lora_add {what}: M={M} K={K} N={N} rank={rank}")
    assert pkg.lora_on_matrix_cores(M, K, N, rank) == (route == P)
    assert run_and_check(pkg, what, M, K, N, rank) == ROUTE[route]


@pytest.mark.parametrize("M,N,rank,tile", [(256, 640, 1000, 2), (64, 264, 16384, 0)])
def test_pair_with_a_split_k_second_gemm(pkg, dev, M, N, rank, tile):
    """y = bf16(y + r . b^T) with r . b^T split over K (128 x 128 tiles; the M <= 128 kernel): y is
    added once, by the launch that sums the partials."""
    pkg.set_tile(tile)
    pkg.set_lora_route(pkg.LORA_PAIR)
    try:
        assert pkg.linear_route(M, (rank + 63) & ~63, N, 16)["splits"] > 1
        say(f"lora_add pair, split-K second GEMM M={M} N={N} rank={rank} tile={tile}")
        assert run_and_check(pkg, f"split second {M}", M, 512, N, rank) == ROUTE[P]
    finally:
        pkg.set_tile(pkg.TILE_AUTO)
        pkg.set_lora_route(pkg.LORA_AUTO)


# the same shapes on every route that can take them (the A/B hook, ltx25_set_lora_route)
FORCED = [s for s in SHAPES if s[0] in (
    "x2 upscaler: attn projection", "distilled adapter: rank 450", "video tokens, rank 64",
    "GEMM pair, ragged M and N", "r first: rank 32 at the FFN width", "r first: rank 16, ragged N")]


@pytest.mark.parametrize("forced", [P, RF, F])
@pytest.mark.parametrize("what,M,K,N,rank,route", FORCED, ids=[s[0] for s in FORCED])
def test_lora_forced_routes_agree(pkg, dev, what, M, K, N, rank, route, forced):
    say(f"lora_add forced {forced}: {what}: M={M} K={K} N={N} rank={rank}")
    pkg.set_lora_route(ROUTE[forced])
    try:
        if forced == RF and rank % 8 != 0:
            # r first needs rank % 8 == 0: refused before any device use, y untouched
            yd = torch.ones((M, N), dtype=torch.bfloat16, device="cuda")
            xd = torch.zeros((M, K), dtype=torch.bfloat16, device="cuda")
            ad = torch.zeros((rank, K), dtype=torch.bfloat16, device="cuda")
            bd = torch.zeros((N, rank), dtype=torch.bfloat16, device="cuda")
            with pytest.raises(pkg.Ltx25Error) as e:
                pkg.lora_add(xd, ad, bd, yd, M, K, N, rank)
            assert e.value.code == pkg.E_UNSUPPORTED
            return
        assert run_and_check(pkg, what, M, K, N, rank) == ROUTE[forced]
    finally:
        pkg.set_lora_route(pkg.LORA_AUTO)


def test_lora_zero_adapter_leaves_y_bit_identical(pkg, dev):
    M, K, N, rank = 96, 256, 320, 16
    x, a, b, y0 = draws("zero", M, K, N, rank)
    yb = orc.bf16_rne(y0)
    yd = dev_bf16(yb)
    say("lora_add with A = 0")
    pkg.lora_add(dev_bf16(orc.bf16_rne(x)), torch.zeros((rank, K), dtype=torch.bfloat16,
                                                          device="cuda"),
                 dev_bf16(orc.bf16_rne(b)), yd, M, K, N, rank)
    torch.cuda.synchronize()
    assert np.array_equal(host_bits(yd), yb)


def test_lora_empty_shape_is_a_no_op(pkg, dev):
    yb = orc.bf16_rne(np.ones((4, 8), np.float32))
    yd = dev_bf16(yb)
    say("lora_add with M = 0 and rank = 0")
    pkg.lora_add(yd, yd, yd, yd, 0, 8, 8, 4)
    pkg.lora_add(yd, yd, yd, yd, 4, 8, 8, 0)
    torch.cuda.synchronize()
    assert np.array_equal(host_bits(yd), yb)
    assert not pkg.lora_on_matrix_cores(0, 8, 8, 4)


def test_lora_is_deterministic(pkg, dev):
    M, K, N, rank = 256, 1024, 2048, 32
    x, a, b, y0 = draws("determinism", M, K, N, rank)
    xd, ad, bd = (dev_bf16(orc.bf16_rne(t)) for t in (x, a, b))
    outs = []
    for i in range(2):
        yd = dev_bf16(orc.bf16_rne(y0))
        say(f"lora_add determinism run {i}")
        pkg.lora_add(xd, ad, bd, yd, M, K, N, rank)
        torch.cuda.synchronize()
        outs.append(host_bits(yd))
    assert np.array_equal(outs[0], outs[1])


# the plans under the FUSED answer: r by the dense GEMM ahead of the y phase, both products on the
# dense GEMM (from rank 96 and K = 512), one pass below; at each line's sides, ranks that are not
# multiples of 8 or 64, one token, ragged N
PLANS = [  # M, K, N, rank
    (128, 1344, 1032, 32), (128, 1280, 1032, 32), (23, 2112, 1032, 32), (23, 2048, 1032, 32),
    (255, 1024, 1032, 32), (255, 960, 1032, 32), (70, 1088, 264, 40), (70, 1024, 264, 40),
    # b copied
    (1, 11456, 520, 5), (1, 11392, 520, 5), (33, 1024, 8, 90), (20, 1088, 512, 95),
    (20, 960, 512, 95), (255, 1472, 4104, 17), (255, 1408, 4104, 17), (300, 2560, 96, 12),
    (40, 1536, 1000, 1), (700, 3008, 264, 6), (700, 2944, 264, 6), (600, 1984, 4104, 6),
    (600, 1920, 4104, 6), (600, 1024, 264, 90), (3000, 3904, 40, 6), (64, 512, 2056, 90),
    # many columns
    (1, 10944, 2056, 8), (1, 4096, 2056, 8), (64, 1152, 2056, 8), (64, 1088, 2056, 8),
    (64, 384, 2056, 64), (64, 320, 2056, 64),
    # both on the dense GEMM
    (255, 1024, 264, 96), (255, 512, 264, 96), (64, 512, 264, 128), (1, 512, 264, 128),
    (3, 512, 1000, 450), (3, 448, 1000, 450), (255, 512, 264, 128), (255, 512, 2056, 128),
    (200, 640, 264, 192), (200, 576, 264, 192), (200, 512, 264, 450), (200, 512, 264, 225),
    (100, 512, 264, 100), (1, 512, 264, 100), (32, 768, 264, 104), (16, 768, 264, 104),
    (70, 1600, 200, 512), (64, 1600, 200, 520),
]


@pytest.mark.parametrize("M,K,N,rank", PLANS)
def test_fused_plans_against_oracle(pkg, dev, M, K, N, rank):
    say(f"lora_add plan M={M} K={K} N={N} rank={rank}")
    assert run_and_check(pkg, f"plan {M} {K} {N} {rank}", M, K, N, rank) == ROUTE[F]


@pytest.mark.parametrize("M,K,N,rank", PLANS + [(45, 64, 30, 6)])
def test_gelu_after_the_adapter_is_the_sequence(pkg, dev, M, K, N, rank):
    """linear_q_lora where the fold does not take: the GELU inside the adapter's last kernel
    gives the bits of linear_q, lora_add, gelu_tanh."""
    from gpu_util import make_qweight, rng_normal
    if pkg.lora_fold_takes(M, K, N, rank, 8):
        pytest.skip("the fold takes it")
    rng = np.random.default_rng(M + K + N + rank)
    qw = make_qweight(pkg, rng_normal(rng, (N, K), 0.02), 8, 64)[0]
    x, a, b, _ = draws(f"gelu {M} {K} {N} {rank}", M, K, N, rank)
    xd, ad, bd = (dev_bf16(orc.bf16_rne(t * s)) for t, s in ((x, 1.0), (a, 0.1), (b, 0.1)))
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    seq = torch.empty_like(y)
    say(f"linear_q_lora + GELU M={M} K={K} N={N} rank={rank}")
    pkg.linear_q_lora(xd, qw, None, ad, bd, rank, y, M, K, N, pkg.EPI_GELU_TANH)
    pkg.linear_q(xd, qw, None, seq, M, K, N)
    pkg.lora_add(xd, ad, bd, seq, M, K, N, rank)
    pkg.gelu_tanh(seq, seq)
    torch.cuda.synchronize()
    assert np.array_equal(host_bits(y), host_bits(seq))


# the reference's caller scratch r ([M][rank]): the r-first route, and the GEMM pair at a
# rank that is a multiple of 64, compute r into it instead of the library's scratch
CALLER_R = [("r first: rank 40, ragged M", 777, 1024, 2048, 40, RF),
            ("r first: rank 56, 2085 rows", 2085, 2624, 512, 56, RF),
            ("GEMM pair, rank 128, no padding", 300, 2048, 1024, 128, P)]


@pytest.mark.parametrize("what,M,K,N,rank,route", CALLER_R, ids=[s[0] for s in CALLER_R])
def test_lora_caller_r_holds_r(pkg, dev, what, M, K, N, rank, route):
    say(f"lora_add with the caller's r: {what}: M={M} K={K} N={N} rank={rank}")
    x, a, b, y0 = draws(what, M, K, N, rank)
    xb, ab, bb, yb = (orc.bf16_rne(t) for t in (x, a, b, y0))
    xd, ad, bd = (dev_bf16(t) for t in (xb, ab, bb))
    assert pkg.lora_route(xd, ad, bd, dev_bf16(yb), M, K, N, rank) == ROUTE[route]
    # the library's scratch, then the caller's r (NaN-filled first): same kernels, same bits
    y_lib = dev_bf16(yb)
    pkg.lora_add(xd, ad, bd, y_lib, M, K, N, rank)
    r = torch.full((M, rank), float("nan"), dtype=torch.bfloat16, device="cuda")
    y_r = dev_bf16(yb)
    pkg.lora_add(xd, ad, bd, y_r, M, K, N, rank, r=r)
    torch.cuda.synchronize()
    assert np.array_equal(host_bits(y_r), host_bits(y_lib))
    got = orc.bf16_to_f32(host_bits(y_r))
    ref = orc.bf16_to_f32(orc.lora_add(xb, ab, bb, yb))
    assert max_rel(got, ref) <= MAX_REL
    # r = bf16(x . a^T) landed in the caller's buffer
    r_got = orc.bf16_to_f32(host_bits(r))
    r_ref = orc.bf16_to_f32(xb).astype(np.float64) @ orc.bf16_to_f32(ab).astype(np.float64).T
    assert np.isfinite(r_got).all()
    assert max_rel(r_got, r_ref) <= MAX_REL


# the plans' scratch is the stream's own: ranks and K of both two-launch plans
OWN = [(128, 4096, 1032, 32), (100, 2048, 1000, 200)]


def own_operands(M, K, N, rank):
    x, a, b, y0 = draws(f"own {M} {K} {N} {rank}", M, K, N, rank)
    return tuple(dev_bf16(orc.bf16_rne(t)) for t in (x, a, b, y0))


@pytest.mark.parametrize("M,K,N,rank", OWN)
def test_plans_under_capture_run_in_one_pass(pkg, dev, M, K, N, rank):
    """A capture without a call before it: the one-pass kernel, which needs no scratch."""
    x, a, b, y0 = own_operands(M, K, N, rank)
    want = y0.clone()
    pkg.set_lora_route(pkg.LORA_FUSED)
    pkg.lora_add(x, a, b, want, M, K, N, rank)
    pkg.set_lora_route(pkg.LORA_AUTO)
    y, eager = y0.clone(), y0.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    say(f"lora_add captured first M={M} K={K} N={N} rank={rank}")
    with torch.cuda.graph(graph):
        pkg.lora_add(x, a, b, y, M, K, N, rank)
    for _ in range(3):
        y.copy_(y0)
        graph.replay()
        eager.copy_(y0)
        pkg.lora_add(x, a, b, eager, M, K, N, rank)   # the plan's own scratch meanwhile
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))
        assert (eager.float() - want.float()).norm() < 3e-3 * want.float().norm()


# ranks whose b is copied with its rows padded: r ahead, and both products on the dense GEMM
COPIED = [(128, 4352, 1032, 12), (33, 4096, 4104, 17), (64, 1024, 1024, 450)]


@pytest.mark.parametrize("M,K,N,rank", COPIED)
def test_plans_before_a_capture(pkg, dev, M, K, N, rank):
    """A call, then the same captured: the one-pass kernel, whose copy of b the call has allocated."""
    x, a, b, y0 = own_operands(M, K, N, rank)
    want, y, eager = y0.clone(), y0.clone(), y0.clone()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    say(f"lora_add before its capture M={M} K={K} N={N} rank={rank}")
    with torch.cuda.stream(side):
        pkg.lora_add(x, a, b, eager, M, K, N, rank)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        pkg.lora_add(x, a, b, y, M, K, N, rank)
    pkg.set_lora_route(pkg.LORA_FUSED)
    pkg.lora_add(x, a, b, want, M, K, N, rank)
    pkg.set_lora_route(pkg.LORA_AUTO)
    torch.cuda.synchronize()
    for _ in range(3):
        y.copy_(y0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))
        eager.copy_(y0)
        pkg.lora_add(x, a, b, eager, M, K, N, rank)
        torch.cuda.synchronize()
        assert (eager.float() - want.float()).norm() < 3e-3 * want.float().norm()


@pytest.mark.parametrize("M,K,N,rank", OWN + COPIED)
def test_eight_streams_have_their_plans(pkg, dev, M, K, N, rank):
    """Eight streams at once, each with an adapter of its own: all idle before, so all hold scratch,
    and each result has the bits of the plan alone."""
    n = 8
    x, a, b, y0 = own_operands(M, K, N, rank)
    bs = [(b.float() * (1.0 + 0.1 * i)).to(torch.bfloat16) for i in range(n)]
    alone = []
    for bi in bs:
        alone.append(y0.clone())
        pkg.lora_add(x, a, bi, alone[-1], M, K, N, rank)
    streams = [torch.cuda.Stream() for _ in range(n)]
    ys = [[y0.clone() for _ in range(6)] for _ in range(n)]
    torch.cuda.synchronize()
    say(f"lora_add, eight streams M={M} K={K} N={N} rank={rank}")
    for t in range(6):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                pkg.lora_add(x, a, bs[i], ys[i][t], M, K, N, rank)
    torch.cuda.synchronize()
    for i in range(n):
        for y in ys[i]:
            assert torch.equal(y.view(torch.int16), alone[i].view(torch.int16)), i


@pytest.mark.parametrize("M,K,N,rank", OWN)
def test_plans_overlap_on_streams(pkg, dev, M, K, N, rank):
    """Calls on ten streams at once, more than have scratch of their own: each result is the one
    it has alone, the plan's or the one-pass kernel's."""
    n = 10
    x, a, b, y0 = own_operands(M, K, N, rank)
    xs = [x * (i + 1) for i in range(n)]
    alone = []
    for xi in xs:
        plan, one = y0.clone(), y0.clone()
        pkg.lora_add(xi, a, b, plan, M, K, N, rank)
        pkg.set_lora_route(pkg.LORA_FUSED)
        pkg.lora_add(xi, a, b, one, M, K, N, rank)
        pkg.set_lora_route(pkg.LORA_AUTO)
        alone.append((plan, one))
    streams = [torch.cuda.Stream() for _ in range(n)]
    ys = [[y0.clone() for _ in range(6)] for _ in range(n)]
    torch.cuda.synchronize()
    say(f"lora_add on {n} streams M={M} K={K} N={N} rank={rank}")
    for t in range(6):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                pkg.lora_add(xs[i], a, b, ys[i][t], M, K, N, rank)
    torch.cuda.synchronize()
    for i in range(n):
        for y in ys[i]:
            assert any(torch.equal(y.view(torch.int16), w.view(torch.int16)) for w in alone[i])
