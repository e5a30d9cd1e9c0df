"""The panel kernel (panel.hip) on the GPU, through the C ABI: linears from 1024 of K whose panels
of 32 to 128 rows x 32 or 64 columns fit the CUs in one round of workgroups.

Pinned as the M <= 128 kernel is: a selection GEMM (row m of X holds a single 1.0 at column
k(m), so y[m][n] = bf16(w[n][k(m)] + bias[n]) exactly, whatever the summation order), whose
columns walk the chunks, the four waves' ranges and the K splits; random data against the
oracle and, bit for bit, against the dense linear over the dequantized weight. The shapes sit
where the kernel can go wrong: one row or column past a panel, chunk counts that leave the waves
uneven, group rows that start at odd places of a 16-byte scale window, windows that wrap, scale
tensors off 16-byte alignment, K splits, N that is not a multiple of 8.
"""
import numpy as np
import pytest
import torch

import orc
from gpu_util import dev_bf16, dev_bytes, dev_f32, host_bits, host_f32, make_qweight, rng_normal, say
from test_gpu_skinny import make_bias, selection_x

pytestmark = pytest.mark.gpu

MAX_REL = 1e-2

# M, K, N, bits, group, bias, splits
CASES = [
    (129, 1024, 64, 8, 64, "f32", 1),        # 32 x 32: the smallest K, one row past four panels
    (160, 1088, 1000, 8, 64, "none", 1),     # 32 x 32: 17 chunks (4 4 4 5), 17 groups per row
    (250, 1600, 2046, 8, 32, "bf16", 1),     # 64 x 32: 50 groups per row, N % 8 != 0
    (200, 2112, 300, 4, 32, "f32", 1),       # 33 chunks, 66 groups: four windows wrap
    (1000, 2112, 500, 4, 64, "none", 1),     # 64 x 32
    (161, 4160, 4097, 8, 64, "bf16", 1),     # 128 x 32 or 64 x 64: one column past a panel
    (250, 4096, 4096, 8, 64, "none", 1),
    (257, 4096, 5000, 4, 32, "f32", 1),      # 128 x 64: one row past two panels
    (320, 4160, 4090, 8, 32, "bf16", 1),     # 128 x 64: N % 8 != 0
    (320, 4096, 4096, 16, 64, "f32", 1),     # dense
    (150, 1024, 40, 16, 64, "bf16", 1),      # dense, 32 x 32
    (1000, 1088, 300, 16, 64, "none", 1),    # dense, 64 x 32
    (160, 4160, 4100, 16, 64, "f32", 1),     # dense, N % 8 == 4
    (129, 1088, 8190, 8, 64, "bf16", 1),     # the wide panels at few chunks: 128 x 64, 17 chunks
    (300, 1088, 5000, 4, 32, "f32", 1),
    (250, 1088, 4100, 16, 64, "none", 1),
    (260, 1024, 3000, 8, 32, "f32", 1),      # 64 x 64
    (1500, 2048, 513, 4, 64, "bf16", 1),     # 128 x 32
    (1, 4096, 8192, 8, 64, "f32", 1),        # at most 128 rows where the M <= 128 kernel
    (31, 4160, 12290, 4, 64, "bf16", 1),     #   would need two rounds: 32 x 32, 32 x 64
    (126, 4096, 8192, 8, 32, "none", 1),
    (100, 4096, 16380, 4, 32, "f32", 1),     # 128 x 64
    (2, 9280, 3792, 8, 64, "bf16", None),    # K splits: uneven runs
    (99, 16320, 2688, 4, 32, "none", None),
    (150, 16384, 700, 8, 64, "f32", None),
    (300, 10368, 1168, 16, 64, "bf16", None),
]


def case_id(c):
    return f"M{c[0]}-K{c[1]}-N{c[2]}-w{c[3]}g{c[4]}-{c[5]}"


def weight(pkg, rng, N, K, bits, group, std):
    """-> call(x, bias, y, M, epi), the f32 weight of the oracle's bar, the bf16 weight as f32"""
    w = rng_normal(rng, (N, K), std)
    if bits == 16:
        wb = orc.bf16_rne(w)
        wd = dev_bf16(wb)
        return (lambda x, b, y, M, epi=0: pkg.linear(x, wd, b, y, M, K, N), orc.bf16_to_f32(wb),
                orc.bf16_to_f32(wb).reshape(N, K))
    qw, codes, scales, biases, wb = make_qweight(pkg, w, bits, group)
    wf, _ = orc.dequant(codes, scales, biases, N, K, bits, group)
    return (lambda x, b, y, M, epi=0: pkg.linear_q(x, qw, b, y, M, K, N, epi), wf,
            orc.bf16_to_f32(wb).reshape(N, K))


@pytest.mark.parametrize("case", CASES, ids=[case_id(c) for c in CASES])
def test_selection_gemm_is_bit_exact(pkg, dev, case):
    M, K, N, bits, group, bias, splits = case
    route = pkg.linear_route(M, K, N, bits)
    assert route["tile"] == pkg.TILE_MID, route
    assert route["splits"] == splits if splits is not None else route["splits"] > 1, route
    rng = np.random.default_rng(M * 31 + K + N * 7 + bits)
    call, _, w16 = weight(pkg, rng, N, K, bits, group, 0.05)
    b, bd = make_bias(rng, N, bias)
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    say(f"panel selection {case_id(case)} route={route}")
    for shift in (0, 7):
        x, cols = selection_x(M, K)
        if shift:
            x = np.roll(x, K // 2 + shift, axis=1)
            cols = (cols + K // 2 + shift) % K
        call(dev_bf16(orc.bf16_rne(x)), bd, y, M)
        torch.cuda.synchronize()
        sel = np.asarray(w16, np.float32)[:, cols].T
        want = sel + (np.asarray(b, np.float32)[None, :] if b is not None else 0.0)
        assert np.array_equal(host_bits(y), orc.bf16_rne(want.astype(np.float32))), shift


RANDOM = [c for c in CASES if c[0] * c[1] * c[2] < 2.5e9]


@pytest.mark.parametrize("case", RANDOM, ids=[case_id(c) for c in RANDOM])
def test_random_data_against_oracle_and_dense(pkg, dev, case):
    M, K, N, bits, group, bias, _ = case
    rng = np.random.default_rng(K * 3 + N)
    call, wf, w16 = weight(pkg, rng, N, K, bits, group, 0.02)
    xb = orc.bf16_rne(rng_normal(rng, (M, K)))
    b, bd = make_bias(rng, N, bias)
    x = dev_bf16(xb)
    epi = 1 if bits != 16 else 0
    y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    say(f"panel random {case_id(case)}")
    call(x, bd, y, M, epi)
    torch.cuda.synchronize()
    rows = np.unique(np.linspace(0, M - 1, 12).astype(int))
    ref = orc.linear_f64_d(orc.bf16_to_f32(xb)[rows], wf, b)
    if epi:
        ref = orc.gelu(ref.astype(np.float32)).astype(np.float64)
    assert orc.max_rel(host_f32(y)[rows], ref) <= MAX_REL
    if bits != 16:
        # the same plan over the dequantized weight, and the same call again: the same bits
        yd, yq, again = (torch.empty_like(y) for _ in range(3))
        wd = dev_bf16(orc.bf16_rne(w16))
        pkg.linear(x, wd, bd, yd, M, K, N)
        call(x, bd, yq, M, 0)
        call(x, bd, again, M, epi)
        torch.cuda.synchronize()
        assert np.array_equal(host_bits(yq), host_bits(yd))
        assert np.array_equal(host_bits(again), host_bits(y))


@pytest.mark.parametrize("bits,group", [(8, 64), (8, 32), (4, 64), (4, 32)])
@pytest.mark.parametrize("M,K,N", [(200, 1088, 1000), (320, 4160, 4096), (2, 9280, 3792)])
def test_scales_off_16_byte_alignment(pkg, dev, M, K, N, bits, group):
    """Scales and zero points as views one and three elements into their storage: the same bits."""
    assert pkg.linear_route(M, K, N, bits)["tile"] == pkg.TILE_MID
    rng = np.random.default_rng(M + K + bits)
    codes, scales, biases, _ = orc.quantize_affine(rng_normal(rng, (N, K), 0.02), bits, group)
    x = dev_bf16(orc.bf16_rne(rng_normal(rng, (M, K))))
    outs = []
    for s_off, q_off in ((0, 0), (1, 3)):
        def place(v, off):
            t = torch.full((v.size + off + 8,), float("nan"), dtype=torch.bfloat16, device="cuda")
            t[off:off + v.size] = dev_bf16(v).view(-1)
            return t[off:off + v.size]
        qw = pkg.QWeight(dev_bytes(codes), place(scales, s_off), place(biases, q_off), bits, group)
        y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
        say(f"panel scales at {s_off}, zero points at {q_off}: {M}x{K}->{N} w{bits}g{group}")
        pkg.linear_q(x, qw, None, y, M, K, N)
        torch.cuda.synchronize()
        outs.append(host_bits(y))
    assert np.array_equal(outs[0], outs[1])


def test_accumulating_output(pkg, dev):
    """The LoRA pair's second GEMM at a rank from 1024: y += r . B^T on a panel, ragged M and N."""
    M, K, N, rank = 300, 128, 264, 1024
    rng = np.random.default_rng(9)
    xb = orc.bf16_rne(rng_normal(rng, (M, K)))
    ab = orc.bf16_rne(rng_normal(rng, (rank, K), 0.05))
    bb = orc.bf16_rne(rng_normal(rng, (N, rank), 0.05))
    yb = orc.bf16_rne(rng_normal(rng, (M, N)))
    assert pkg.lora_on_matrix_cores(M, K, N, rank)
    y = dev_bf16(yb)
    say("panel accumulating into y: LoRA pair, rank 1024")
    pkg.lora_add(dev_bf16(xb), dev_bf16(ab), dev_bf16(bb), y, M, K, N, rank)
    torch.cuda.synchronize()
    r = orc.bf16_to_f32(orc.bf16_rne(orc.linear_f64(orc.bf16_to_f32(xb), orc.bf16_to_f32(ab))))
    ref = orc.bf16_to_f32(yb).astype(np.float64) + orc.linear_f64_d(r, orc.bf16_to_f32(bb))
    assert orc.max_rel(host_f32(y), ref) <= MAX_REL
