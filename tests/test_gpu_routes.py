"""Every GEMM route at the same shapes, through the C ABI's tile switch
(ltx25_set_tile, the A/B hook the reference keeps as VPIPE_LTX25_MMA_TILE,
src/ltx25-metal-ops.cc:193-231), and the row slabs that keep each operand of
a launch under 2 GiB (the reference's operand limit, :342-374).

Each forced route is asserted through ltx25_linear_route before it runs, so a
test cannot pass on a route it did not mean to measure. Bars as in
test_gpu_qlinear.py: max|y - ref| / max|ref| <= 1e-2 against the oracle's f64
GEMM over the dequantized weight on sampled rows, rel-L2 < 3e-3 on all rows
against torch fp32 of the same operands; within one route the quantized
weight and its GPU-dequantized bf16 copy give bit-identical outputs.
"""
import numpy as np
import pytest
import torch

import orc
from gpu_util import dev_bf16, dev_f32, host_bits, host_f32, make_qweight, rng_normal, say
from test_gpu_qlinear import check_full_vs_torch, check_rows_vs_oracle, sample_rows

pytestmark = pytest.mark.gpu

SHAPES = [  # name, M, K, N, bias
    ("audio qkv", 126, 2048, 6144, True),
    ("audio ff_down (split K)", 126, 8192, 2048, True),
    ("config 0", 320, 4096, 4096, True),
    ("text kv", 1024, 4096, 8192, True),
    ("ragged M and N", 777, 2048, 1000, False),
    ("N not a multiple of 256", 192, 16384, 260, False),
]
TILES = [("tall", 1), ("mid", 2), ("skinny", 3)]


@pytest.fixture(autouse=True)
def _reset_tile(pkg):
    torch.backends.cuda.matmul.allow_tf32 = False
    yield
    pkg.set_tile(pkg.TILE_AUTO)


@pytest.mark.parametrize("tile_name,tile", TILES, ids=[t[0] for t in TILES])
@pytest.mark.parametrize("name,M,K,N,has_bias", SHAPES, ids=[s[0] for s in SHAPES])
def test_forced_tile(pkg, name, M, K, N, has_bias, tile_name, tile):
    rng = np.random.default_rng(40 + M + N)
    x_bits = orc.bf16_rne(rng_normal(rng, (M, K)))
    w = rng_normal(rng, (N, K), 0.02)
    b = rng_normal(rng, (N,), 0.01) if has_bias else None
    qw, codes, scales, biases, wb = make_qweight(pkg, w, 8, 64)
    pkg.set_tile(tile)
    route = pkg.linear_route(M, K, N)
    want = tile if (tile != 3 or M <= 128) else route["tile"]
    assert route["tile"] == want, route
    say(f"forced tile {tile_name}: {name} {M}x{K}->{N} route={route}")
    x_dev = dev_bf16(x_bits)
    b_dev = dev_f32(b) if b is not None else None
    y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    pkg.linear_q(x_dev, qw, b_dev, y, M, K, N)
    w_deq = torch.empty((N, K), dtype=torch.bfloat16, device="cuda")
    pkg.dequant(qw, w_deq, N, K)
    yd = torch.empty_like(y)
    pkg.linear(x_dev, w_deq, b_dev, yd, M, K, N)
    torch.cuda.synchronize()
    assert pkg.linear_route(M, K, N, bits=16)["tile"] == route["tile"]
    assert np.array_equal(host_bits(y), host_bits(yd)), "quantized and dense differ"
    wf, _ = orc.dequant(codes, scales, biases, N, K, 8, 64)
    check_rows_vs_oracle(y, orc.bf16_to_f32(x_bits), wf, b, sample_rows(M, 12))
    check_full_vs_torch(y, x_dev, dev_bf16(wb), b_dev)


@pytest.mark.parametrize("quantized", [False, True], ids=["dense", "w8g64"])
def test_row_slabs_past_2gib(pkg, quantized):
    """X of 2.2 GB: two row slabs, each launch's operands under 2 GiB. Rows on both
    sides of the slab boundary and the last row against the oracle."""
    M, K, N = 270000, 4096, 256
    route = pkg.linear_route(M, K, N, bits=8 if quantized else 16)
    assert route["slabs"] == 2, route
    edge = route["slab_rows"]
    say(f"row slabs: {M}x{K}->{N} quantized={quantized} slab_rows={edge}")
    rng = np.random.default_rng(41)
    w = rng_normal(rng, (N, K), 0.02)
    g = torch.Generator(device="cuda")
    g.manual_seed(42)
    x = torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16)
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    if quantized:
        qw, codes, scales, biases, wb = make_qweight(pkg, w, 8, 64)
        pkg.linear_q(x, qw, None, y, M, K, N)
        wf, _ = orc.dequant(codes, scales, biases, N, K, 8, 64)
    else:
        wb = orc.bf16_rne(w)
        pkg.linear(x, dev_bf16(wb), None, y, M, K, N)
        wf = orc.bf16_to_f32(wb)
    torch.cuda.synchronize()
    assert not torch.isnan(y.float()).any(), "rows left unwritten"
    rows = np.array([0, 1, edge - 2, edge - 1, edge, edge + 1, M - 2, M - 1] +
                    list(rng.integers(0, M, 8)))
    xr = orc.bf16_to_f32(host_bits(x[torch.from_numpy(rows).cuda()]))
    ref = orc.linear_f64_d(xr, wf)
    got = host_f32(y)[rows]
    assert orc.max_rel(got, ref) <= 1e-2
    assert orc.rel_l2(got, ref) < 3e-3


# where the planner leaves the 128 x 128 tile with one K split for larger ones: 128 x 256 tiles
# (dense weights, from K = 1024) and 256 x 256 tiles that do not fill the CUs; 1, 2, 3 and many K
# steps, ragged M and N
LARGER = [  # M, K, N, tile
    (1024, 64, 8192, 2), (300, 960, 16392, 2), (300, 1024, 16392, 2), (897, 1152, 8008, 2),
    (1000, 1088, 8192, 2), (257, 1024, 16000, 2), (700, 64, 16384, 1), (900, 128, 12296, 1), (641, 960, 13000, 1),
]


@pytest.mark.parametrize("M,K,N,tile", LARGER)
@pytest.mark.parametrize("bias,epi", [("f32", 0), ("bf16", 1), (None, 1)])
def test_larger_tiles_give_the_same_bits(pkg, M, K, N, tile, bias, epi):
    """AUTO's choice against the forced 128 x 128 and 256 x 256 tiles: the same sums in the same
    K order, so the same bits; dense, w8 and w4."""
    rng = np.random.default_rng(M + K + N)
    x = dev_bf16(orc.bf16_rne(rng_normal(rng, (M, K))))
    b = None if bias is None else rng_normal(rng, (N,), 0.05)
    bd = None if b is None else dev_f32(b) if bias == "f32" else dev_bf16(orc.bf16_rne(b))
    for bits, group in ((16, 64), (8, 64), (4, 32)):
        w = rng_normal(rng, (N, K), 0.05)
        if bits == 16:
            keep = dev_bf16(orc.bf16_rne(w))
            cw = pkg.dense_weight(keep)
        else:
            qw = make_qweight(pkg, w, bits, group)[0]
            cw = qw.c()
        assert pkg.linear_route(M, K, N, bits)["tile"] == tile
        outs = []
        for force in (pkg.TILE_AUTO, pkg.TILE_MID, pkg.TILE_TALL):
            pkg.set_tile(force)
            y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
            say(f"larger tiles {M}x{K}->{N} w{bits} bias={bias} epi={epi} forced={force} "
                f"route={pkg.linear_route(M, K, N, bits)}")
            pkg.linear_qc(x, cw, bd, y, M, K, N, epi)
            torch.cuda.synchronize()
            outs.append(host_bits(y))
        pkg.set_tile(pkg.TILE_AUTO)
        assert np.array_equal(outs[0], outs[1])
        assert np.array_equal(outs[0], outs[2])


@pytest.mark.parametrize("M,K,N", [(1024, 1408, 8192), (1024, 1536, 8192), (300, 1664, 16392),
                                   (1000, 1792, 8200), (1500, 384, 9000)])
def test_larger_int8_tiles_are_exact(pkg, M, K, N):
    """int8 on 128 x 256 tiles and on 256 x 256 tiles that do not fill the CUs: int32 accumulators
    and bf16 outputs exact."""
    rng = np.random.default_rng(M + K)
    xq = torch.from_numpy(rng.integers(-127, 128, (M, K), dtype=np.int8)).cuda()
    wq = torch.from_numpy(rng.integers(-127, 128, (N, K), dtype=np.int8)).cuda()
    sx = torch.from_numpy(rng.random(M, dtype=np.float32) * 0.01).cuda()
    sw = torch.from_numpy(rng.random(N, dtype=np.float32) * 0.01).cuda()
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    acc = torch.empty((M, N), dtype=torch.int32, device="cuda")
    say(f"larger int8 tiles {M}x{K}->{N}")
    pkg.i8_gemm(xq, sx, wq, sw, None, y, acc, M, K, N)
    torch.cuda.synchronize()
    exact = (xq.double() @ wq.double().t())
    assert torch.equal(acc.double(), exact)
    want = acc.float() * (sx[:, None] * sw[None, :])
    assert torch.equal(y, want.to(torch.bfloat16))


@pytest.mark.parametrize("rank,K", [(100, 256), (1000, 192), (1088, 1024)])
def test_larger_tiles_under_the_lora_pair(pkg, rank, K):
    """The pair's second GEMM, accumulators seeded from y (from 1024 columns of rank), and the
    fold's two-part activation on 128 x 256 tiles: the bits of the forced 256 x 256 tile."""
    M, N = 1024, 8192
    rng = np.random.default_rng(rank)
    x, a, b = (dev_bf16(orc.bf16_rne(rng_normal(rng, s, 0.1))) for s in ((M, K), (rank, K), (N, rank)))
    y0 = dev_bf16(orc.bf16_rne(rng_normal(rng, (M, N))))
    qw = make_qweight(pkg, rng_normal(rng, (N, K), 0.05), 8, 64)[0]
    assert pkg.lora_on_matrix_cores(M, K, N, rank) and pkg.lora_fold_takes(M, K, N, rank, 8)
    outs = []
    for force in (pkg.TILE_AUTO, pkg.TILE_TALL):
        pkg.set_tile(force)
        y = y0.clone()
        say(f"larger tiles under the LoRA pair, rank {rank}, forced={force}")
        pkg.lora_add(x, a, b, y, M, K, N, rank)
        f = torch.empty_like(y)
        pkg.linear_q_lora(x, qw, None, a, b, rank, f, M, K, N, pkg.EPI_GELU_TANH)
        torch.cuda.synchronize()
        outs.append((host_bits(y), host_bits(f)))
    assert np.array_equal(outs[0][0], outs[1][0])
    assert np.array_equal(outs[0][1], outs[1][1])


# a last round of 256 x 256 tiles that leaves half of the CUs idle or more goes out as 128 x 256
# tiles of the last columns or rows: ragged M and N on both sides of the cut. The forced 128 x 128
# tile gives the same sums in one launch.
ROUNDS = [  # M, K, N
    (2040, 2048, 12288),   # 8 x 48: 32 columns of tiles, then 16
    (6000, 2048, 4096),    # 24 x 16: 16 rows of tiles, then 8
    (4500, 2112, 4360),    # 18 x 18, N past the last whole column
    (2570, 2048, 6664),    # 11 x 27: 256 + 41
]


@pytest.mark.parametrize("M,K,N", ROUNDS)
@pytest.mark.parametrize("bias,epi", [("f32", 1), ("bf16", 0)])
def test_the_last_round_gives_the_same_bits(pkg, M, K, N, bias, epi):
    rng = np.random.default_rng(M + K + N)
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N)
    x = torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn((N, K), device="cuda", generator=g) * 0.05).to(torch.bfloat16)
    b = rng_normal(rng, (N,), 0.05)
    bd = dev_f32(b) if bias == "f32" else dev_bf16(orc.bf16_rne(b))
    assert pkg.linear_route(M, K, N, 16)["tile"] == pkg.TILE_TALL
    outs = []
    for force in (pkg.TILE_AUTO, pkg.TILE_MID):
        pkg.set_tile(force)
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        say(f"last round {M}x{K}->{N} bias={bias} epi={epi} forced={force}")
        pkg.linear_qc(x, pkg.dense_weight(w), bd, y, M, K, N, epi)
        torch.cuda.synchronize()
        outs.append(y)
    pkg.set_tile(pkg.TILE_AUTO)
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.parametrize("M,K,N", [(2040, 4096, 12296), (6000, 4096, 4096)])
def test_the_last_int8_round_is_exact(pkg, M, K, N):
    rng = np.random.default_rng(M + K)
    xq = torch.from_numpy(rng.integers(-127, 128, (M, K), dtype=np.int8)).cuda()
    wq = torch.from_numpy(rng.integers(-127, 128, (N, K), dtype=np.int8)).cuda()
    sx = torch.from_numpy(rng.random(M, dtype=np.float32) * 0.01).cuda()
    sw = torch.from_numpy(rng.random(N, dtype=np.float32) * 0.01).cuda()
    b = torch.from_numpy(rng.random(N, dtype=np.float32)).cuda()
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    acc = torch.empty((M, N), dtype=torch.int32, device="cuda")
    say(f"last int8 round {M}x{K}->{N}")
    pkg.i8_gemm(xq, sx, wq, sw, b, y, acc, M, K, N)
    torch.cuda.synchronize()
    assert torch.equal(acc.double(), xq.double() @ wq.double().t())
    want = torch.addcmul(b.double()[None, :], acc.double(),
                         (sx[:, None] * sw[None, :]).double())   # one fma, then one rounding
    assert torch.equal(y, want.float().to(torch.bfloat16))


@pytest.mark.parametrize("M,N", [(2040, 12288), (6000, 4096)])
def test_the_last_round_under_the_lora_pair(pkg, M, N):
    """y-seeded accumulators (rank 2048 as the second GEMM's K) and the two-part activation: the
    forced 128 x 128 tile's bits."""
    K, rank = 2048, 2048
    g = torch.Generator(device="cuda")
    g.manual_seed(M)
    x, a, b, y0 = ((torch.randn(s, device="cuda", generator=g) * 0.1).to(torch.bfloat16)
                   for s in ((M, K), (rank, K), (N, rank), (M, N)))
    rng = np.random.default_rng(M)
    qw = make_qweight(pkg, rng_normal(rng, (N, K), 0.05), 8, 64)[0]
    assert pkg.lora_on_matrix_cores(M, K, N, rank)
    outs = []
    for force in (pkg.TILE_AUTO, pkg.TILE_MID):
        pkg.set_tile(force)
        y = y0.clone()
        f = torch.empty_like(y)
        say(f"last round under the LoRA pair {M}x{K}->{N} forced={force}")
        pkg.lora_add(x, a, b, y, M, K, N, rank)
        pkg.linear_q_lora(x, qw, None, a, b, rank, f, M, K, N, 0)
        torch.cuda.synchronize()
        outs.append((y, f))
    pkg.set_tile(pkg.TILE_AUTO)
    assert torch.equal(outs[0][0].view(torch.int16), outs[1][0].view(torch.int16))
    assert torch.equal(outs[0][1].view(torch.int16), outs[1][1].view(torch.int16))
