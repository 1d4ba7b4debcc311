"""GPU parity of the HIP path against the CPU oracle (run on the MI355X box).

Bars (written in each test):
  * quantize_per_channel, repack, int8-dyn int32 accumulators and outputs:
    bit-exact.
  * int8 weight-only outputs: relative L2 <= 1e-3 against the oracle (the
    fp32-accumulation tolerance of the path; fp16/bf16 activations are used
    exactly, fp32 activations as bf16 hi + lo).
Full-size shapes are checked on sampled output rows (the oracle on all rows
would take minutes); int8-dyn parameters always come from the whole tensor.
"""
from pathlib import Path

import numpy as np
import pytest
import torch

import oracle
from conftest import announce
from sbq import quant

pytestmark = pytest.mark.gpu

GOLD = Path(__file__).resolve().parent / "golden"
W8_TOL = 1e-3

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def make_weights(N, K, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(N, K, generator=g) * 0.02


def make_x(M, K, seed, outliers=False):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g)
    if outliers:
        idx = torch.randperm(K, generator=g)[: max(1, K // 100)]
        x[:, idx] *= 20
    return x


# ---------------------------------------------------------------------------
# quantize_per_channel + repack
# ---------------------------------------------------------------------------
def test_quantize_golden_bitexact(dev):
    announce("quantize golden fixture")
    d = np.load(GOLD / "quantize_per_channel.npz")
    q, s = quant.quantize_per_channel_gpu(torch.from_numpy(d["f32_w"]).to(dev))
    np.testing.assert_array_equal(q.cpu().numpy(), d["f32_q"])
    np.testing.assert_array_equal(s.cpu().numpy().view(np.uint32), d["f32_scale"].view(np.uint32))
    wb = torch.from_numpy(d["bf16_w_bits"]).view(torch.bfloat16)
    q, s = quant.quantize_per_channel_gpu(wb.to(dev))
    np.testing.assert_array_equal(q.cpu().numpy(), d["bf16_q"])
    np.testing.assert_array_equal(s.cpu().numpy(), d["bf16_scale"])


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("N,K", [(1, 1), (5, 3), (257, 300), (1024, 4096)])
def test_quantize_bitexact(dev, dtype, N, K):
    announce(f"quantize {dtype} {N}x{K}")
    w = make_weights(N, K, N * 7 + K).to(DT[dtype])
    if N > 2:
        w[1] = 0
    q, s = quant.quantize_per_channel_gpu(w.to(dev))
    qo, so = oracle.quantize_per_channel_c(w.float().numpy())
    np.testing.assert_array_equal(q.cpu().numpy(), qo)
    np.testing.assert_array_equal(s.cpu().numpy(), so)


def test_quantize_reference_api_returns_on_weight_device(dev):
    announce("quantize api devices")
    w = make_weights(33, 70, 5)
    q, s = quant.quantize_per_channel(w)
    assert q.device.type == "cpu" and q.dtype == torch.int8 and s.dtype == torch.float32
    qo, so = oracle.quantize_per_channel(w.numpy())
    np.testing.assert_array_equal(q.numpy(), qo)
    q2, _ = quant.quantize_per_channel(w.to(dev))
    assert q2.is_cuda


@pytest.mark.parametrize("N,K", [(4, 4096), (13, 200), (64, 96), (16, 64), (4096, 128), (130, 2560)])
def test_repack_roundtrip_and_colsum(dev, N, K):
    announce(f"repack {N}x{K}")
    g = torch.Generator().manual_seed(N + K)
    q = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    packed, colsum = quant.repack(q.to(dev))
    np.testing.assert_array_equal(packed.cpu().numpy(), oracle.pack_w8(q.numpy()))
    np.testing.assert_array_equal(colsum.cpu().numpy(), q.numpy().astype(np.int64).sum(1))
    np.testing.assert_array_equal(quant.unpack(packed, N, K).cpu().numpy(), q.numpy())


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("N,K", [(1, 1), (17, 15), (5, 1000), (33, 1025), (16, 2560), (40, 4095), (130, 4100), (21, 9728),
                                 (18, 12300)])
def test_quantize_pack_one_pass(dev, dtype, N, K):
    """Scales, int8 rows, packed tiles and column sums of one pass, for every
    number of chunks a lane holds, K and row starts of any alignment, and
    values on and next to every half of the scale (rows of maximum 127: scale
    1): bit-equal to the oracle and to the separate entry points."""
    announce(f"quantize pack {dtype} {N}x{K}")
    w = make_weights(N, K, N + K)
    if K > 600:  # half-way values and their neighbours, both signs
        half = torch.arange(-126.5, 127, 1.0)
        ties = torch.cat([half, torch.nextafter(half, half + 1), torch.nextafter(half, half - 1)])[:K - 1]
        w[0, 0] = 127.0
        w[0, 1:] = 0.0
        w[0, 1:1 + len(ties[:K - 1])] = ties[:K - 1]
    if N > 2:
        w[2] = 0
    wide = torch.zeros(N, K + 3, dtype=DT[dtype], device=dev)
    wide[:, 1:K + 1] = w.to(DT[dtype]).to(dev)
    qo, so = oracle.quantize_per_channel_c(w.to(DT[dtype]).float().numpy())
    for wd in (wide[:, 1:K + 1], w.to(DT[dtype]).to(dev)):
        q, s, packed, colsum = quant._quantize_pack(wd, True, True)
        np.testing.assert_array_equal(q.cpu().numpy(), qo)
        np.testing.assert_array_equal(s.cpu().numpy(), so)
        np.testing.assert_array_equal(packed.cpu().numpy(), oracle.pack_w8(qo))
        np.testing.assert_array_equal(colsum.cpu().numpy(), qo.astype(np.int64).sum(1))
        p2, c2 = quant.repack(q)
        assert torch.equal(p2, packed) and torch.equal(c2, colsum)
        q1, s1 = quant.quantize_per_channel_gpu(wd)
        assert torch.equal(q1, q) and torch.equal(s1, s) and torch.equal(quant.unpack(packed, N, K), q)


@pytest.mark.parametrize("N,K", [(1, 577), (16, 4097), (17, 65536), (300, 9728), (1000, 4608), (4081, 4160)])
def test_repack_of_few_long_rows(dev, N, K):
    """K split over workgroups: tiles and (added up) column sums are the oracle's."""
    announce(f"repack {N}x{K}")
    q = torch.randint(-127, 128, (N, K), dtype=torch.int8, generator=torch.Generator().manual_seed(N + K))
    packed, colsum = quant.repack(q.to(dev))
    alone, _ = quant.repack(q.to(dev), with_colsum=False)
    np.testing.assert_array_equal(packed.cpu().numpy(), oracle.pack_w8(q.numpy()))
    assert torch.equal(alone, packed)
    np.testing.assert_array_equal(colsum.cpu().numpy(), q.numpy().astype(np.int64).sum(1))


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("N,K", [(1, 1), (5, 63), (2048, 65), (3, 1024), (7, 2001), (2048, 1027), (6, 12289)])
def test_quantize_few_rows(dev, dtype, N, K):
    """A wavefront per row: bit-equal to the oracle and to the one pass with the packing, an all-zero row and
    rows of inf and NaN included."""
    announce(f"quantize rows {dtype} {N}x{K}")
    w = make_weights(N, K, N * K).to(DT[dtype])
    if N > 4:
        w[1] = 0
    q, s = quant.quantize_per_channel_gpu(w.to(dev))
    qo, so = oracle.quantize_per_channel_c(w.float().numpy())
    np.testing.assert_array_equal(q.cpu().numpy(), qo)
    np.testing.assert_array_equal(s.cpu().numpy(), so)
    if N > 4:
        w[2, K // 2], w[3, K // 3] = float("inf"), float("nan")
    q, s = quant.quantize_per_channel_gpu(w.to(dev))
    q2, s2, _, _ = quant._quantize_pack(w.to(dev), True, False)
    assert torch.equal(q, q2) and torch.equal(s.view(torch.int32), s2.view(torch.int32))


# ---------------------------------------------------------------------------
# int8 weight-only
# ---------------------------------------------------------------------------
W8_CASES = [
    # (M, N, K): decode GEMV (M <= 64) and prefill GEMM (M > 64), odd shapes of
    # the real checkpoint (router N=4, lora K=128, K=2560) and tails.
    (1, 4096, 4096), (1, 4, 2560), (1, 64, 4096), (1, 4096, 128), (2, 200, 96), (4, 6144, 256),
    (16, 1024, 4096), (17, 300, 512), (33, 96, 1000), (64, 512, 2560),
    (65, 256, 512), (128, 1024, 1024), (200, 130, 4096), (512, 2048, 512), (300, 13, 200),
]


@pytest.mark.parametrize("xd", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("M,N,K", W8_CASES)
def test_w8_parity(dev, M, N, K, xd):
    announce(f"w8 M={M} N={N} K={K} x={xd}")
    w = make_weights(N, K, 1000 + N + K)
    x = make_x(M, K, 2000 + M + K).to(DT[xd])
    q, s = oracle.quantize_per_channel(w.numpy())
    ref = oracle.int8_linear(x.float().numpy(), q, s)
    lin = quant.Int8Linear(w, None)
    y = lin(x.to(dev))
    assert y.dtype == torch.float32 and y.shape == (M, N) and y.is_contiguous()
    err = oracle.rel_l2(y.cpu().numpy(), ref)
    assert err <= W8_TOL, err
    if xd != "f32":
        # exact inputs: only fp32 summation order differs (and, for the fp16
        # prefill GEMM, the rounding of its offset-encoded weights' row-sum term)
        assert err <= 2e-6, err


@pytest.mark.parametrize("M,N,K", [(64, 512, 2560), (200, 130, 4096), (512, 2048, 512), (300, 4096, 12288),
                                   (2048, 1024, 4096)])
def test_w8_f16_prefill_row_sum_paths(dev, M, N, K):
    """The fp16 prefill GEMM feeds the weights to the MFMA as subnormals
    (q + 128) * 2^-24 and removes 128 * rowsum(x) in its epilogue.  The row
    sums come from a pre-pass when a workspace is given and from the GEMM's
    own K loop when none is: both paths match the oracle, also for all-positive
    activations (the largest offset term)."""
    announce(f"w8 f16 row sums M={M} N={N} K={K}")
    w = make_weights(N, K, 7000 + N + K)
    q, s = oracle.quantize_per_channel(w.numpy())
    lin = quant.Int8Linear(w, None)
    none = torch.empty(0, dtype=torch.uint8, device=dev)
    for positive in (False, True):
        x = make_x(M, K, 8000 + M + K).half()
        if positive:
            x = x.abs()
        ref = oracle.int8_linear(x.float().numpy(), q, s)
        xd = x.to(dev)
        y_pre = quant.linear_w8(xd, lin.packed, lin.scale, None, N)
        y_loop = quant.linear_w8(xd, lin.packed, lin.scale, None, N, workspace=none)
        e_pre = oracle.rel_l2(y_pre.cpu().numpy(), ref)
        e_loop = oracle.rel_l2(y_loop.cpu().numpy(), ref)
        # a float64 model of the cancellation bounds it by 1.1e-4 (all-positive x, K = 12288)
        bound = 3e-4 if positive else 2e-6
        assert e_pre <= bound and e_loop <= bound, (positive, e_pre, e_loop)


# fp16 W-only GEMM shapes at short K (the oracle stays fast): the picks here
# are mostly the small blocks, since at short K the per-launch cost dominates
# (every configuration in use is run at K = 4096 in test_configs_gpu.py);
# ragged M and N, the 64x64 and 128x64 K-split blocks at M <= 128.
W8_GEMM_CFG = [(2048, 4096, 128), (2048, 12288, 128), (1024, 12288, 192), (1000, 12290, 256), (512, 12288, 256),
               (500, 12300, 192), (512, 8192, 256), (512, 6144, 320), (450, 6100, 320), (256, 8192, 448),
               (100, 1000, 320), (384, 6144, 320), (768, 4096, 320)]


@pytest.mark.parametrize("M,N,K", W8_GEMM_CFG)
def test_w8_gemm_block_configs(dev, M, N, K):
    """Every fp16 W-only block configuration, with row sums from the pre-pass
    (workspace), from the K loop (no workspace), and over fp32 activations
    staged as fp16 planes; the activations are fp16 values, so all three must
    match the oracle to fp32 summation order."""
    announce(f"w8 gemm config M={M} N={N} K={K}")
    w = make_weights(N, K, 7300 + N + K)
    x = make_x(M, K, 7400 + M + K).half()
    q, s = oracle.quantize_per_channel(w.numpy())
    ref = oracle.int8_linear(x.float().numpy(), q, s)
    lin = quant.Int8Linear(w, None)
    xd = x.to(dev)
    none = torch.empty(0, dtype=torch.uint8, device=dev)
    for xin, ws in ((xd, None), (xd, none), (xd.float(), None)):
        y = quant.linear_w8(xin, lin.packed, lin.scale, None, N, workspace=ws)
        err = oracle.rel_l2(y.cpu().numpy(), ref)
        assert err <= 2e-6, (xin.dtype, ws is None, err)


@pytest.mark.parametrize("xd", ["f32", "bf16"])
@pytest.mark.parametrize("M,N,K", [(64, 512, 2560), (200, 130, 4096), (512, 2048, 512), (300, 4096, 4096)])
def test_w8_staged_prefill_rows(dev, M, N, K, xd):
    """fp32 / bf16 prefill activations are staged as a power-of-two scaled
    fp16 plane for the fp16 GEMM when a workspace is given; rows span
    1e-30 .. 1e30, and each row must match the oracle on its own.  The paths
    without a workspace are held to the weight-only tolerance."""
    announce(f"w8 staged M={M} N={N} K={K} x={xd}")
    w = make_weights(N, K, 9000 + N + K)
    q, s = oracle.quantize_per_channel(w.numpy())
    lin = quant.Int8Linear(w, None)
    mags = torch.pow(10.0, torch.linspace(-30.0, 30.0, M, dtype=torch.float64)).float()
    x = (make_x(M, K, 9100 + M + K) * mags[:, None]).to(DT[xd])
    ref = oracle.int8_linear(x.float().numpy(), q, s).astype(np.float64)
    xd_dev = x.to(dev)
    none = torch.empty(0, dtype=torch.uint8, device=dev)
    for ws in (None, none):
        y = quant.linear_w8(xd_dev, lin.packed, lin.scale, None, N, workspace=ws).cpu().numpy().astype(np.float64)
        row_err = np.linalg.norm(y - ref, axis=1) / np.linalg.norm(ref, axis=1)
        # staged bf16 is exact; staged fp32 keeps 11 significant bits: a relative rounding error of at most
        # 2^-11 per value, about 3e-4 relative L2 on a row's outputs (6e-4 allows for the row's spread)
        bar = (6e-4 if xd == "f32" else 2e-6) if ws is None else W8_TOL
        assert row_err.max() <= bar, (ws is None, float(row_err.max()), int(row_err.argmax()))


@pytest.mark.parametrize("yd", ["f16", "bf16"])
@pytest.mark.parametrize("M", [1, 9, 100])
def test_w8_low_precision_output(dev, M, yd):
    announce(f"w8 out={yd} M={M}")
    N, K = 264, 1024
    w = make_weights(N, K, 7)
    x = make_x(M, K, 8).half()
    q, s = oracle.quantize_per_channel(w.numpy())
    ref = oracle.int8_linear(x.float().numpy(), q, s)
    lin = quant.Int8Linear(w, None)
    y = quant.linear_w8(x.to(dev), lin.packed, lin.scale, None, N, DT[yd])
    assert y.dtype == DT[yd]
    assert oracle.rel_l2(y.float().cpu().numpy(), ref) <= 4e-3


@pytest.mark.parametrize("M,N,K", [(1, 4096, 12288), (1, 6144, 4096), (1, 24, 128), (2, 300, 6144), (3, 1000, 4096)])
def test_w8_decode_fp32_rows_split(dev, M, N, K):
    """fp32 decode activations run as bf16 hi + remainder (16 significant bits,
    fp32 range): a single row that fits in LDS is split once, in place; several
    rows are split per tile.  Rows of 1e-30, 1 and 1e30 magnitude each match
    the oracle to that precision; a NaN poisons its own row only."""
    bound = 2e-5
    announce(f"w8 fp32 split M={M} N={N} K={K}")
    w = make_weights(N, K, 7600 + N + K)
    b = torch.randn(N)
    q, s = oracle.quantize_per_channel(w.numpy())
    lin = quant.Int8Linear(w, b)
    base = make_x(M, K, 7700 + M + K, outliers=True)
    for shift in range(3):
        scales = torch.tensor([[1e-30], [1.0], [1e30]]).roll(shift, 0)[:M] if M > 1 else \
            torch.tensor([[(1e-30, 1.0, 1e30)[shift]]])
        x = (base * scales).float()
        ref = oracle.int8_linear(x.numpy(), q, s)
        y = quant.linear_w8(x.to(dev), lin.packed, lin.scale, None, N).cpu().numpy()
        for m in range(M):
            err = oracle.rel_l2(y[m], ref[m])
            assert err <= bound, (shift, m, err)
    x = base.clone()
    x[0, K // 3] = float("nan")
    y = quant.linear_w8(x.to(dev), lin.packed, lin.scale, lin.bias, N).cpu().numpy()
    assert np.isnan(y[0]).all()
    if M > 1:
        ref = oracle.int8_linear(x[1:].numpy(), q, s, b.numpy())
        assert oracle.rel_l2(y[1:], ref) <= bound


def test_w8_bias_and_strided_input(dev):
    announce("w8 bias + strided")
    N, K, M = 96, 512, 20
    w = make_weights(N, K, 9)
    b = torch.randn(N)
    big = make_x(M, K + 64, 10)
    x = big[:, 32:32 + K]  # row stride K + 64, 16-byte aligned rows
    q, s = oracle.quantize_per_channel(w.numpy())
    ref = oracle.int8_linear(x.numpy(), q, s, b.numpy())
    lin = quant.Int8Linear(w, b)
    x_dev = big.to(dev)[:, 32:32 + K]
    y = quant.linear_w8(x_dev, lin.packed, lin.scale, lin.bias, N)
    assert oracle.rel_l2(y.cpu().numpy(), ref) <= 1e-5
    # misaligned row start (offset of one element) takes the scalar path
    x_dev2 = big.to(dev)[:, 1:1 + K]
    ref2 = oracle.int8_linear(big[:, 1:1 + K].numpy(), q, s, b.numpy())
    y2 = quant.linear_w8(x_dev2, lin.packed, lin.scale, lin.bias, N)
    assert oracle.rel_l2(y2.cpu().numpy(), ref2) <= 1e-5


FAST_CASES = [
    # decode fast path (M <= 16, K % 64 == 0, aligned rows): odd tile counts
    # with two row tiles per wave, ragged N, M on both sides of 4, long K;
    # 257..383 row tiles, which take two row tiles per wave for weight-only
    # (the checkpoint's grouped 2 x 2560 x 4096 output projections among them)
    (1, 6152, 4096), (3, 6160, 4096), (5, 6144, 4096), (8, 4100, 12288), (16, 6152, 2560), (2, 24, 64),
    (1, 4, 128), (1, 5120, 4096), (4, 4610, 2560), (7, 6100, 4096),
    # M = 4 .. 8 over more than 1024 row tiles at short K: five row tiles per
    # workgroup with x in LDS (ragged last workgroup; 1025 row tiles)
    (8, 19456, 2560), (4, 18820, 2560), (6, 16400, 2560), (12, 19456, 2560), (16, 18820, 2560),
]


FAST_F32_CASES = [
    # fp32 activations at decode shapes: x in LDS as bf16 high / remainder
    # planes (M <= 8, x <= 24 KiB, or 48 KiB for one row), M = 2..8 filling
    # the planes' MFMA columns partly or wholly, and direct steps beyond
    (1, 6152, 4096), (1, 2560, 9728), (1, 19456, 2560), (2, 24, 64), (5, 1000, 1024), (8, 4096, 128),
    (8, 130, 704), (3, 6160, 4096), (8, 2560, 2560), (12, 1000, 512), (16, 4096, 128), (1, 4096, 12288),
    (8, 19456, 2560), (5, 16400, 2560),  # five row tiles per workgroup, x split from registers
]


@pytest.mark.parametrize("M,N,K", FAST_F32_CASES)
def test_w8_fast_path_f32_planes(dev, M, N, K):
    """fp32 x runs as high + remainder parts (x in LDS: row-scaled fp16, 22
    significant bits; direct steps: bf16, 16 bits): every row, at magnitudes
    from 1e-20 to 1e20, within 2e-5 of the float64 product of the oracle's
    quantized weights, on activations no 2-byte type holds exactly.  Dropping
    the remainder part would leave about 1e-3."""
    announce(f"w8 fast f32 planes M={M} N={N} K={K}")
    w = make_weights(N, K, 5200 + N + K)
    b = torch.randn(N, generator=torch.Generator().manual_seed(N + 1))
    x = make_x(M, K, 6200 + M + K) * (1.0 + 1e-3 * torch.rand(M, K, generator=torch.Generator().manual_seed(M)))
    x = x * torch.pow(10.0, torch.linspace(-20.0, 20.0, M, dtype=torch.float64)).float()[:, None]  # rows 1e-20 .. 1e20
    for m in range(M):  # one element per row 1000x the rest: a row scale that missed it would overflow fp16
        x[m, (K - 1 - 131 * m) % K] *= 1000.0
    q, s = oracle.quantize_per_channel(w.numpy())
    ref = (x.double().numpy() @ q.astype(np.float64).T) * s.astype(np.float64) + b.double().numpy()
    lin = quant.Int8Linear(w, b)
    y = quant.linear_w8(x.to(dev), lin.packed, lin.scale, lin.bias, N).cpu().numpy().astype(np.float64)
    row_err = np.linalg.norm(y - ref, axis=1) / np.linalg.norm(ref, axis=1)
    assert row_err.max() <= 2e-5, (float(row_err.max()), int(row_err.argmax()))


@pytest.mark.parametrize("xd", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("M,N,K", FAST_CASES)
def test_w8_fast_path_bias_strided(dev, M, N, K, xd):
    announce(f"w8 fast M={M} N={N} K={K} x={xd}")
    w = make_weights(N, K, 5000 + N + K)
    b = torch.randn(N, generator=torch.Generator().manual_seed(N))
    big = make_x(M, K + 64, 6000 + M + K).to(DT[xd])
    x = big[:, 64:]  # row stride K + 64 elements, rows stay 16-byte aligned
    q, s = oracle.quantize_per_channel(w.numpy())
    ref = oracle.int8_linear(x.float().numpy(), q, s, b.numpy())
    lin = quant.Int8Linear(w, b)
    y = quant.linear_w8(big.to(dev)[:, 64:], lin.packed, lin.scale, lin.bias, N)
    err = oracle.rel_l2(y.cpu().numpy(), ref)
    assert err <= (W8_TOL if xd == "f32" else 1e-5), err
    y16 = quant.linear_w8(big.to(dev)[:, 64:], lin.packed, lin.scale, lin.bias, N, torch.float16)
    assert oracle.rel_l2(y16.float().cpu().numpy(), ref) <= 4e-3


def test_w8_golden_fixture(dev):
    announce("w8 golden fixture")
    d = np.load(GOLD / "int8_linear.npz")
    for i in range(len(d["cases"])):
        x, q, s, y = d[f"c{i}_x"], d[f"c{i}_q"], d[f"c{i}_scale"], d[f"c{i}_y"]
        packed, _ = quant.repack(torch.from_numpy(q).to(dev))
        out = quant.linear_w8(torch.from_numpy(x).to(dev), packed, torch.from_numpy(s).to(dev), None, q.shape[0])
        assert oracle.rel_l2(out.cpu().numpy(), y) <= 1e-5, i


def test_w8_integer_activations_exact(dev):
    """Small-integer activations: every product and partial sum is exact in
    fp32, so the GPU result must equal fp32(sum) * scale bit for bit."""
    announce("w8 integer activations")
    N, K, M = 200, 1024, 12
    w = make_weights(N, K, 11)
    g = torch.Generator().manual_seed(12)
    x = torch.randint(-3, 4, (M, K), generator=g).half()
    q, s = oracle.quantize_per_channel(w.numpy())
    exact = (x.numpy().astype(np.int64) @ q.astype(np.int64).T).astype(np.float32) * s
    lin = quant.Int8Linear(w, None)
    np.testing.assert_array_equal(lin(x.to(dev)).cpu().numpy(), exact)
    xb = x.float().repeat(8, 1).half()  # M = 96 -> GEMM path
    exact_b = np.tile(exact, (8, 1))
    np.testing.assert_array_equal(lin(xb.to(dev)).cpu().numpy(), exact_b)
    # rows starting one element off 16-byte alignment -> general GEMV kernel
    big = torch.zeros((M, K + 8), dtype=torch.float16)
    big[:, 1:1 + K] = x
    y_mis = quant.linear_w8(big.to(dev)[:, 1:1 + K], lin.packed, lin.scale, None, N)
    np.testing.assert_array_equal(y_mis.cpu().numpy(), exact)


# ---------------------------------------------------------------------------
# int8-dyn (W8A8, fbgemm semantics): bit-exact
# ---------------------------------------------------------------------------
W8A8_CASES = [(1, 4096, 4096), (1, 4, 2560), (5, 64, 4096), (16, 13, 96), (33, 512, 256), (64, 100, 1000),
              (65, 64, 4096), (128, 1024, 4096), (300, 130, 200),
              (3, 6152, 4096), (8, 4100, 12288), (16, 6144, 4096), (2, 24, 64), (4, 16400, 4096), (1, 4100, 12288),
              (1, 4096, 128), (8, 4096, 256), (1, 2560, 9728), (8, 19456, 2560), (5, 16400, 2560)]


@pytest.mark.parametrize("xd", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("M,N,K", W8A8_CASES)
def test_w8a8_bitexact(dev, M, N, K, xd):
    announce(f"w8a8 M={M} N={N} K={K} x={xd}")
    w = make_weights(N, K, 3000 + N + K)
    x = make_x(M, K, 4000 + M + K, outliers=True).to(DT[xd])
    q, s = oracle.quantize_per_channel(w.numpy())
    ref, info = oracle.dyn_linear(x.float().numpy(), q, s, return_intermediates=True)
    lin = quant.DynamicInt8Linear(w, None)
    acc = torch.empty((M, N), dtype=torch.int32, device=dev)
    y = quant.linear_w8a8(x.to(dev), lin.packed, lin.scale, lin.colsum, None, N, acc_out=acc)
    np.testing.assert_array_equal(acc.cpu().numpy(), info["acc"])
    np.testing.assert_array_equal(y.cpu().numpy(), ref)
    sx, zp = quant.act_qparams(x.to(dev))
    assert (np.float32(sx), zp) == (np.float32(info["scale"]), info["zero_point"])


# W8A8 GEMM shapes at short K (the oracle stays fast), with odd K-tile counts
# and ragged M and N; two long-K shapes (K = 6208) as well.  Every
# configuration the picker uses runs at K = 4096 in test_configs_gpu.py.
W8A8_GEMM_CFG = [(2048, 24576, 128), (2048, 24576, 192), (2048, 12288, 128), (1024, 12288, 256), (1024, 8192, 256),
                 (1024, 8192, 320), (512, 12288, 256), (512, 12288, 320), (512, 8192, 256), (512, 8192, 448),
                 (256, 8192, 448), (384, 6144, 256), (256, 4096, 448), (448, 4096, 6208), (384, 6144, 6208),
                 (1000, 12290, 256),
                 (500, 12300, 192)]


@pytest.mark.parametrize("M,N,K", W8A8_GEMM_CFG)
def test_w8a8_gemm_block_configs(dev, M, N, K):
    announce(f"w8a8 gemm config M={M} N={N} K={K}")
    w = make_weights(N, K, 3700 + N + K)
    x = make_x(M, K, 3800 + M + K, outliers=True).half()
    q, s = oracle.quantize_per_channel(w.numpy())
    ref, info = oracle.dyn_linear(x.float().numpy(), q, s, return_intermediates=True)
    lin = quant.DynamicInt8Linear(w, None)
    acc = torch.empty((M, N), dtype=torch.int32, device=dev)
    y = quant.linear_w8a8(x.to(dev), lin.packed, lin.scale, lin.colsum, None, N, acc_out=acc)
    np.testing.assert_array_equal(acc.cpu().numpy(), info["acc"])
    np.testing.assert_array_equal(y.cpu().numpy(), ref)


@pytest.mark.parametrize("M,N,K", [(2048, 24576, 128), (1000, 12290, 256), (512, 12288, 256), (256, 8192, 448)])
def test_w8a8_token_gemm_block_configs(dev, M, N, K):
    announce(f"w8a8 token gemm config M={M} N={N} K={K}")
    w = make_weights(N, K, 3900 + N + K)
    x = make_x(M, K, 3950 + M + K, outliers=True).half()
    q, s = oracle.quantize_per_channel(w.numpy())
    ref, info = oracle.dyn_linear_token(x.float().numpy(), q, s, return_intermediates=True)
    lin = quant.DynamicInt8Linear(w, None, granularity="token")
    acc = torch.empty((M, N), dtype=torch.int32, device=dev)
    y = quant.linear_w8a8_token(x.to(dev), lin.packed, lin.scale, None, N, acc_out=acc)
    np.testing.assert_array_equal(acc.cpu().numpy(), info["acc"])
    np.testing.assert_array_equal(y.cpu().numpy(), ref)


@pytest.mark.parametrize("M", [1, 8, 64, 512])
def test_w8a8_quantizer_ties(dev, M):
    """Activations that land exactly on .5 after fma(x, 1/s_x, zp): x >= 0
    with max 255/16 gives s_x = 1/16, zp = 0, and x = (k + 0.5)/16 rounds half
    to even.  The fused GEMV (M=1), the partials GEMV (M=8) and the GEMM paths
    must match fbgemm's quantizer bit for bit."""
    announce(f"w8a8 ties M={M}")
    N, K = 256, 4096
    w = make_weights(N, K, 3300)
    kk = torch.arange(K).view(1, K)
    mm = torch.arange(M).view(M, 1)
    x = (((kk * 7 + mm * 13) % 255).float() + 0.5) / 16.0
    x[:, 0] = 255.0 / 16.0
    x = x.half()
    q, s = oracle.quantize_per_channel(w.numpy())
    ref, info = oracle.dyn_linear(x.float().numpy(), q, s, return_intermediates=True)
    assert (float(info["scale"]), int(info["zero_point"])) == (1.0 / 16.0, 0)
    lin = quant.DynamicInt8Linear(w, None)
    acc = torch.empty((M, N), dtype=torch.int32, device=dev)
    y = quant.linear_w8a8(x.to(dev), lin.packed, lin.scale, lin.colsum, None, N, acc_out=acc)
    np.testing.assert_array_equal(acc.cpu().numpy(), info["acc"])
    np.testing.assert_array_equal(y.cpu().numpy(), ref)


@pytest.mark.parametrize("xd", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (5, 64, 1000), (33, 512, 256), (128, 1024, 4096), (300, 130, 200),
                                   (2048, 512, 4096), (8, 4100, 2560), (16, 1000, 1024), (3, 6160, 4096),
                                   (1, 19456, 2560), (2, 24, 64)])
def test_w8a8_token_bitexact(dev, M, N, K, xd):
    """Per-token symmetric W8A8 (opt-in granularity): int32 accumulators and
    fp32 outputs bit-exact against the oracle, on every activation dtype,
    ragged K and small M; with 1% outlier channels x20."""
    announce(f"w8a8 token M={M} N={N} K={K} x={xd}")
    w = make_weights(N, K, 3500 + N + K)
    x = make_x(M, K, 3600 + M + K, outliers=True).to(DT[xd])
    q, s = oracle.quantize_per_channel(w.numpy())
    ref, info = oracle.dyn_linear_token(x.float().numpy(), q, s, return_intermediates=True)
    lin = quant.DynamicInt8Linear(w, None, granularity="token")
    acc = torch.empty((M, N), dtype=torch.int32, device=dev)
    y = quant.linear_w8a8_token(x.to(dev), lin.packed, lin.scale, None, N, acc_out=acc)
    np.testing.assert_array_equal(acc.cpu().numpy(), info["acc"])
    np.testing.assert_array_equal(y.cpu().numpy(), ref)
    np.testing.assert_array_equal(lin(x.to(dev)).cpu().numpy(), ref)


@pytest.mark.parametrize("xd", ["f32", "f16"])
def test_w8a8_token_rows_edge_cases(dev, xd):
    """Per-token decode with each row quantized in the GEMV: a zero row (scale
    1e-8 / 127), rows of tiny and huge magnitude and a row whose largest value
    sits in its last column, bit-exact against the oracle with a bias."""
    announce(f"w8a8 token edge rows x={xd}")
    M, N, K = 6, 2000, 2560
    w = make_weights(N, K, 3710)
    b = torch.randn(N, generator=torch.Generator().manual_seed(3711))
    x = make_x(M, K, 3712)
    x[0] = 0.0
    x[1] *= 1e-30 if xd == "f32" else 1e-3
    x[2] *= 1e30 if xd == "f32" else 1e3
    x[4, K - 1] = 50.0
    x = x.to(DT[xd])
    q, s = oracle.quantize_per_channel(w.numpy())
    ref, info = oracle.dyn_linear_token(x.float().numpy(), q, s, bias=b.numpy(), return_intermediates=True)
    lin = quant.DynamicInt8Linear(w, b.to(dev), granularity="token")
    acc = torch.empty((M, N), dtype=torch.int32, device=dev)
    y = quant.linear_w8a8_token(x.to(dev), lin.packed, lin.scale, lin.bias, N, acc_out=acc)
    np.testing.assert_array_equal(acc.cpu().numpy(), info["acc"])
    np.testing.assert_array_equal(y.cpu().numpy(), ref)


def test_w8a8_token_bias_and_default_granularity(dev):
    announce("w8a8 token bias")
    M, N, K = 64, 300, 4096
    w = make_weights(N, K, 3700)
    b = torch.randn(N, generator=torch.Generator().manual_seed(3701))
    x = make_x(M, K, 3702, outliers=True)
    q, s = oracle.quantize_per_channel(w.numpy())
    ref = oracle.dyn_linear_token(x.numpy(), q, s, bias=b.numpy())
    lin = quant.DynamicInt8Linear(w, b, granularity="token")
    np.testing.assert_array_equal(lin(x.to(dev)).cpu().numpy(), ref)
    # the default stays the reference's per-tensor semantics
    assert quant.DynamicInt8Linear(w, None).granularity == "tensor"
    with pytest.raises(ValueError):
        quant.DynamicInt8Linear(w, None, granularity="row")


def test_w8a8_golden_fixture(dev):
    announce("w8a8 golden fixture")
    d = np.load(GOLD / "int8_dyn.npz")
    for i, kind in enumerate(d["kinds"]):
        x, q, s, yref = d[f"c{i}_x"], d[f"c{i}_q"], d[f"c{i}_scale"], d[f"c{i}_y"]
        bias = torch.from_numpy(d[f"c{i}_bias"]).to(dev) if f"c{i}_bias" in d else None
        packed, colsum = quant.repack(torch.from_numpy(q).to(dev))
        y = quant.linear_w8a8(torch.from_numpy(x).to(dev), packed, torch.from_numpy(s).to(dev), colsum, bias,
                              q.shape[0])
        np.testing.assert_array_equal(y.cpu().numpy(), yref, err_msg=str(kind))


def test_w8a8_token_golden_fixture(dev):
    announce("w8a8 token golden fixture")
    d = np.load(GOLD / "int8_dyn_token.npz")
    for i in range(len(d["cases"])):
        x, q, s = d[f"c{i}_x"], d[f"c{i}_q"], d[f"c{i}_scale"]
        packed, _ = quant.repack(torch.from_numpy(q).to(dev), with_colsum=False)
        acc = torch.empty((x.shape[0], q.shape[0]), dtype=torch.int32, device=dev)
        y = quant.linear_w8a8_token(torch.from_numpy(x).to(dev), packed, torch.from_numpy(s).to(dev), None,
                                    q.shape[0], acc_out=acc)
        np.testing.assert_array_equal(acc.cpu().numpy(), d[f"c{i}_acc"], err_msg=f"case {i}")
        np.testing.assert_array_equal(y.cpu().numpy(), d[f"c{i}_y"], err_msg=f"case {i}")


@pytest.mark.parametrize("kind", ["zeros", "tiny", "tinypos", "tinyneg", "positive", "negative", "const", "huge"])
def test_w8a8_qparams_edge_cases(dev, kind):
    announce(f"qparams {kind}")
    g = torch.Generator().manual_seed(5)
    x = torch.randn(6, 700, generator=g)
    x = {"zeros": x * 0, "tiny": x * 1e-6, "tinypos": x.abs() * 1e-6, "tinyneg": -x.abs() * 1e-6,
         "positive": x.abs() + 1, "negative": -x.abs() - 1, "const": torch.full_like(x, 0.37),
         "huge": x * 3e4}[kind]
    sx, zp = quant.act_qparams(x.to(dev))
    so, zo = oracle.act_qparams(x.numpy())
    assert (np.float32(sx), zp) == (np.float32(so), zo)
    w = make_weights(40, 700, 6)
    q, s = oracle.quantize_per_channel(w.numpy())
    lin = quant.DynamicInt8Linear(w, None)
    np.testing.assert_array_equal(lin(x.to(dev)).cpu().numpy(), oracle.dyn_linear(x.numpy(), q, s))


ACT_QUANT_CASES = [  # (M, K, x dtype, row stride pad, xq row stride pad, kind)
    (1, 4096, "f32", 0, 0, "outliers"), (7, 700, "f16", 0, 3, "normal"), (33, 4096, "bf16", 64, 0, "outliers"),
    (128, 2560, "f32", 8, 16, "normal"), (5, 13, "f32", 3, 1, "normal"), (300, 1000, "f16", 0, 0, "tiny"),
    (2, 64, "f32", 0, 0, "zeros"), (64, 12288, "f16", 0, 0, "positive"),
]


@pytest.mark.parametrize("M,K,xd,xpad,qpad,kind", ACT_QUANT_CASES)
def test_act_quant_per_tensor_matches_oracle(dev, M, K, xd, xpad, qpad, kind):
    """sbq_act_quant_per_tensor (the quantization step of linear_dynamic,
    quant.py:65): scale, zero point and every uint8 value bit-exact against
    the oracle, strided rows in and out (ragged K, unaligned strides); and
    sbq_linear_w8a8's int32 accumulators equal sum_k (xq - zp) * q."""
    announce(f"act quant M={M} K={K} x={xd} pads={xpad},{qpad} {kind}")
    g = torch.Generator().manual_seed(M * 7 + K)
    x = torch.randn(M, K, generator=g)
    if kind == "outliers":
        x[:, torch.randperm(K, generator=g)[: max(1, K // 100)]] *= 20
    elif kind == "tiny":
        x *= 1e-6
    elif kind == "zeros":
        x *= 0
    elif kind == "positive":
        x = x.abs() + 0.5
    x = x.to(DT[xd])
    xs = torch.zeros((M, K + xpad), dtype=x.dtype)
    xs[:, :K] = x
    xd_dev = xs.to(dev)[:, :K]
    buf = torch.full((M, K + qpad), 77, dtype=torch.uint8, device=dev)
    xq, s, z = quant.act_quant_per_tensor(xd_dev, out=buf)
    so, zo = oracle.act_qparams(x.float().numpy())
    assert (np.float32(s.item()), int(z.item())) == (np.float32(so), zo)
    np.testing.assert_array_equal(xq.cpu().numpy(), oracle.quantize_act(x.float().numpy(), so, zo))
    if qpad:
        assert bool((buf[:, K:] == 77).all())  # the padding columns are left alone
    N = 48
    w = make_weights(N, K, 9)
    q, _ = oracle.quantize_per_channel(w.numpy())
    lin = quant.DynamicInt8Linear(w, None)
    acc = torch.empty((M, N), dtype=torch.int32, device=dev)
    quant.linear_w8a8(xd_dev, lin.packed, lin.scale, lin.colsum, None, N, acc_out=acc)
    ref = (xq.cpu().numpy().astype(np.int64) - zo) @ q.astype(np.int64).T
    np.testing.assert_array_equal(acc.cpu().numpy(), ref.astype(np.int32))


def test_w8a8_bias_fused(dev):
    announce("w8a8 bias")
    N, K = 72, 512
    w = make_weights(N, K, 21)
    b = torch.randn(N)
    for M in (3, 150):
        x = make_x(M, K, 22 + M, outliers=True)
        q, s = oracle.quantize_per_channel(w.numpy())
        lin = quant.DynamicInt8Linear(w, b)
        np.testing.assert_array_equal(lin(x.to(dev)).cpu().numpy(), oracle.dyn_linear(x.numpy(), q, s, b.numpy()))


# ---------------------------------------------------------------------------
# full-size shapes (sampled rows)
# ---------------------------------------------------------------------------
FULL_W8 = [(1, 4096, 4096), (1, 6144, 4096), (4, 24576, 4096), (16, 4096, 12288), (2048, 12288, 4096),
           (2048, 24576, 4096), (512, 4096, 4096)]


@pytest.mark.parametrize("M,N,K", FULL_W8)
def test_w8_full_size_sampled(dev, M, N, K):
    announce(f"w8 full M={M} N={N} K={K}")
    w = (torch.randn(N, K, generator=torch.Generator().manual_seed(0)) * 0.02)
    x = make_x(M, K, 1).half()
    lin = quant.Int8Linear(w.to(dev), None)
    y = lin(x.to(dev)).cpu().numpy()
    q = lin.qweight.cpu().numpy()
    s = lin.scale.cpu().numpy()
    rows = np.unique(np.linspace(0, M - 1, min(M, 24)).astype(int))
    ref = oracle.int8_linear(x.float().numpy()[rows], q, s)
    assert oracle.rel_l2(y[rows], ref) <= 2e-6


@pytest.mark.parametrize("M,N", [(1, 4096), (128, 12288), (2048, 12288)])
def test_w8a8_full_size_sampled(dev, M, N):
    announce(f"w8a8 full M={M} N={N}")
    K = 4096
    w = torch.randn(N, K, generator=torch.Generator().manual_seed(0)) * 0.02
    x = make_x(M, K, 1, outliers=True).half()
    lin = quant.DynamicInt8Linear(w.to(dev), None)
    acc = torch.empty((M, N), dtype=torch.int32, device=dev)
    y = quant.linear_w8a8(x.to(dev), lin.packed, lin.scale, lin.colsum, None, N, acc_out=acc)
    q, s = oracle.quantize_per_channel(w.numpy())
    xf = x.float().numpy()
    sx, zp = oracle.act_qparams(xf)  # parameters of the WHOLE tensor
    rows = np.unique(np.linspace(0, M - 1, min(M, 24)).astype(int))
    xq = oracle.quantize_act(xf[rows], sx, zp)
    acc_ref = ((xq.astype(np.int64) - zp) @ q.astype(np.int64).T).astype(np.int32)
    np.testing.assert_array_equal(acc.cpu().numpy()[rows], acc_ref)
    np.testing.assert_array_equal(y.cpu().numpy()[rows], oracle.dyn_epilogue(acc_ref, sx, s))


# ---------------------------------------------------------------------------
# the reference module API as the loader and the model use it
# ---------------------------------------------------------------------------
def test_int8_state_dict_roundtrip(dev):
    """quant.py:36-38: the state_dict holds qweight / scale (/ bias); loading
    one into another module must make it compute with the loaded weights."""
    announce("state_dict roundtrip")
    N, K = 96, 512
    w1, w2 = make_weights(N, K, 31), make_weights(N, K, 32)
    b = torch.randn(N)
    lin1, lin2 = quant.Int8Linear(w1, b), quant.Int8Linear(w2, torch.zeros(N))
    sd = lin1.state_dict()
    assert set(sd) == {"qweight", "scale", "bias"}
    assert sd["qweight"].dtype == torch.int8 and sd["scale"].dtype == torch.float32
    assert set(quant.Int8Linear(w1, None).state_dict()) == {"qweight", "scale"}
    lin2.load_state_dict(sd)
    x = make_x(3, K, 33)
    np.testing.assert_array_equal(lin2(x.to(dev)).cpu().numpy(), lin1(x.to(dev)).cpu().numpy())


def test_mismatched_operands_raise_before_launch(dev):
    """The C ABI sees raw pointers: the Python layer rejects operands whose
    sizes, dtypes or devices do not match (N, K) before any kernel runs, and
    the modules raise RuntimeError for an input that does not end in
    in_features, as the reference's matmul does."""
    announce("operand validation")
    N, K, M = 64, 256, 3
    w = make_weights(N, K, 51)
    lin = quant.Int8Linear(w, None)
    dyn = quant.DynamicInt8Linear(w, None)
    x = make_x(M, K, 52).to(dev)
    ok = quant.linear_w8(x, lin.packed, lin.scale, None, N)
    with pytest.raises(ValueError):  # tiles of a smaller weight
        quant.linear_w8(x, lin.packed[: quant.packed_bytes(N - 16, K)], lin.scale, None, N)
    with pytest.raises(ValueError):  # scale too short
        quant.linear_w8(x, lin.packed, lin.scale[:N - 1], None, N)
    with pytest.raises(ValueError):  # fp16 bias
        quant.linear_w8(x, lin.packed, lin.scale, torch.zeros(N, device=dev, dtype=torch.float16), N)
    with pytest.raises(ValueError):  # output of the wrong shape
        quant.linear_w8(x, lin.packed, lin.scale, None, N, out=torch.empty((M, N - 4), device=dev))
    with pytest.raises(ValueError):  # x on the CPU
        quant.linear_w8(x.cpu(), lin.packed, lin.scale, None, N)
    with pytest.raises(ValueError):  # colsum too short
        quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum[:8], None, N)
    with pytest.raises(ValueError):
        quant.linear_w8a8_token(x, dyn.packed, dyn.scale[:8], None, N)
    with pytest.raises(ValueError):
        quant.unpack(lin.packed[:1024], N, K)
    for mod in (lin, dyn, quant.fuse_linears([lin, quant.Int8Linear(w, None)])):
        with pytest.raises(RuntimeError):
            mod(make_x(M, K + 64, 53).to(dev))
    np.testing.assert_array_equal(quant.linear_w8(x, lin.packed, lin.scale, None, N).cpu().numpy(), ok.cpu().numpy())


def test_single_row_views_with_small_row_stride(dev):
    """One-row operands viewed from a column ([1, n] with stride(0) = 1, as
    t() of an [n, 1] tensor gives): a weight row, an activation row and the
    output row, in both formats; equal to the contiguous copies."""
    announce("single-row views")
    N, K = 96, 512
    w1 = torch.randn(K, 1, generator=torch.Generator().manual_seed(61)).to(dev).t()  # [1, K], stride (1, 1)
    q1, s1 = quant.quantize_per_channel_gpu(w1)
    q2, s2 = quant.quantize_per_channel_gpu(w1.contiguous())
    assert torch.equal(q1, q2) and torch.equal(s1, s2)
    w = make_weights(N, K, 62)
    x1 = make_x(K, 1, 63).to(dev).t()  # [1, K], stride (1, 1)
    for fmt in ("int8", "int8-dyn"):
        lin = quant.make_linear(fmt, w, None)
        out = torch.empty((N, 1), dtype=torch.float32, device=dev).t()  # [1, N], stride (1, 1)
        if fmt == "int8":
            quant.linear_w8(x1, lin.packed, lin.scale, None, N, out=out)
        else:
            quant.linear_w8a8(x1, lin.packed, lin.scale, lin.colsum, None, N, out=out)
        np.testing.assert_array_equal(out.cpu().numpy(), lin(x1.contiguous()).cpu().numpy(), err_msg=fmt)


@pytest.mark.parametrize("M,K,xd", [(1, 16384, "f16"), (4, 24576, "f32"), (1, 40000, "bf16"), (3, 65536, "f16"),
                                    (20, 20000, "f32")])
def test_long_k_beyond_the_gemv(dev, M, K, xd):
    """K beyond the decode GEMVs' 12288 (no model layer has it; a caller
    might): the tiled GEMM serves even one token; both formats against the
    oracle."""
    announce(f"long K M={M} K={K} x={xd}")
    N = 200
    w = make_weights(N, K, 81)
    q, s = oracle.quantize_per_channel(w.numpy())
    x = make_x(M, K, 82, outliers=True).to(DT[xd])
    xv = x.float().numpy()
    y = quant.Int8Linear(w, None)(x.to(dev))
    assert oracle.rel_l2(y.cpu().numpy(), oracle.int8_linear(xv, q, s)) <= W8_TOL
    yd = quant.DynamicInt8Linear(w, None)(x.to(dev))
    np.testing.assert_array_equal(yd.cpu().numpy(), oracle.dyn_linear(xv, q, s))


@pytest.mark.parametrize("M,K,xd", [(1, 12289, "f32"), (4, 13000, "f16"), (16, 20001, "bf16"), (2, 20000, "f32")])
def test_long_ragged_k_at_decode_sizes(dev, M, K, xd):
    """The same with K % 64 != 0, weight-only: the layer, and two layers fused
    (outputs stored as parts)."""
    announce(f"long ragged K M={M} K={K} x={xd}")
    N = 200
    w = make_weights(N, K, 84)
    q, s = oracle.quantize_per_channel(w.numpy())
    x = make_x(M, K, 85, outliers=True).to(DT[xd])
    want = oracle.int8_linear(x.float().numpy(), q, s)
    lin = quant.Int8Linear(w, None)
    assert oracle.rel_l2(lin(x.to(dev)).cpu().numpy(), want) <= W8_TOL
    fused = quant.fuse_linears([quant.Int8Linear(w[:132], None), quant.Int8Linear(w[132:], None)])
    assert oracle.rel_l2(torch.cat(fused(x.to(dev)), -1).cpu().numpy(), want) <= W8_TOL


@pytest.mark.parametrize("M,N,K,xd", [(65536, 16, 4096, "f16"), (100003, 8, 512, "f32"), (40000, 3, 1000, "bf16")])
def test_many_tokens_few_outputs(dev, M, N, K, xd):
    """Very tall, narrow calls (a router over a long prompt): grids of many
    row blocks and one column block; sampled rows against the oracle, int8-dyn
    with the parameters of the whole tensor."""
    announce(f"many tokens M={M} N={N} K={K} x={xd}")
    w = make_weights(N, K, 83)
    q, s = oracle.quantize_per_channel(w.numpy())
    x = make_x(M, K, 84, outliers=True).to(DT[xd])
    xg = x.to(dev)
    rows = np.unique(np.concatenate([np.arange(0, M, max(1, M // 97)), [M - 1]]))
    xv = x.float().numpy()
    y = quant.Int8Linear(w, None)(xg)
    assert oracle.rel_l2(y.cpu().numpy()[rows], oracle.int8_linear(xv[rows], q, s)) <= W8_TOL
    dyn = quant.DynamicInt8Linear(w, None)
    acc = torch.empty((M, N), dtype=torch.int32, device=dev)
    yd = quant.linear_w8a8(xg, dyn.packed, dyn.scale, dyn.colsum, None, N, acc_out=acc)
    sx, zp = oracle.act_qparams(xv)
    xq = oracle.quantize_act(xv[rows], sx, zp)
    acc_ref = ((xq.astype(np.int64) - zp) @ q.astype(np.int64).T).astype(np.int32)
    np.testing.assert_array_equal(acc.cpu().numpy()[rows], acc_ref)
    np.testing.assert_array_equal(yd.cpu().numpy()[rows], oracle.dyn_epilogue(acc_ref, sx, s))


def test_empty_inputs(dev):
    """No tokens: [0, K] and [2, 0, K] inputs give [0, N] and [2, 0, N] fp32
    outputs as the reference's matmul does, on GPU and CPU tensors, in both
    formats; no logits rows give no tokens."""
    announce("empty inputs")
    N, K = 48, 256
    w = make_weights(N, K, 71)
    for fmt in ("int8", "int8-dyn"):
        mod = quant.make_linear(fmt, w, None)
        for shape in ((0, K), (2, 0, K)):
            for x in (torch.empty(shape, device=dev), torch.empty(shape)):
                y = mod(x)
                assert y.shape == shape[:-1] + (N,) and y.dtype == torch.float32 and y.device == x.device, (fmt, shape)
    none = torch.empty((0, 1000), device=dev)
    assert quant.greedy_tokens(none).shape == (0,)
    assert quant.sample_tokens(none, 0.7, 0.9).shape == (0,)


def test_cpu_tensors_in_and_out(dev):
    """The reference model feeds CPU fp32 [T, B, K] tensors and views the
    fp32 contiguous result (model.py:262-264): same contract here."""
    announce("cpu in / cpu out")
    N, K = 64, 256
    w = make_weights(N, K, 41)
    x = make_x(6, K, 42).reshape(2, 3, K)
    q, s = oracle.quantize_per_channel(w.numpy())
    ref = oracle.int8_linear(x.reshape(-1, K).numpy(), q, s).reshape(2, 3, N)
    for fmt in ("int8", "int8-dyn"):
        y = quant.make_linear(fmt, w, None)(x)
        assert y.device.type == "cpu" and y.dtype == torch.float32 and y.shape == (2, 3, N) and y.is_contiguous()
        tol = 1e-5 if fmt == "int8" else 2e-2  # int8-dyn quantizes the activations too
        assert oracle.rel_l2(y.numpy(), ref) <= tol, fmt


@pytest.mark.parametrize("fmt", list(quant.FORMATS))
def test_make_linear_every_format(dev, fmt):
    announce(f"make_linear {fmt}")
    N, K = 48, 320
    w = make_weights(N, K, 51)
    b = torch.randn(N)
    x = make_x(5, K, 52)
    ref = x.double() @ w.double().t() + b.double()
    y = quant.make_linear(fmt, w, b)(x.to(dev))
    assert y.dtype == torch.float32 and y.shape == (5, N)
    tol = {"float32": 1e-6, "bfloat16": 2e-2, "float16": 2e-3, "int8": 2e-2, "int8-dyn": 3e-2}[fmt]
    assert oracle.rel_l2(y.cpu().double().numpy(), ref.numpy()) <= tol


def test_loader_style_swap(dev):
    """loader.py:43-51 replaces every nn.Linear (including nn.Sequential
    children) by make_linear(fmt, weight, None) in place."""
    announce("loader-style swap")
    torch.manual_seed(61)
    model = torch.nn.ModuleDict({
        "q_proj": torch.nn.Linear(256, 128, bias=False),
        "lora": torch.nn.Sequential(torch.nn.Linear(256, 32, bias=False), torch.nn.Linear(32, 128, bias=False)),
    })
    x = torch.randn(4, 256)
    ref_q = model["q_proj"](x).detach()
    ref_l = model["lora"](x).detach()
    for name, mod in list(model.named_modules()):
        if isinstance(mod, torch.nn.Linear):
            parent_name, _, child = name.rpartition(".")
            parent = model.get_submodule(parent_name) if parent_name else model
            setattr(parent, child, quant.make_linear("int8", mod.weight.detach(), None))
    assert not any(isinstance(m, torch.nn.Linear) for m in model.modules())
    with torch.inference_mode():
        assert oracle.rel_l2(model["q_proj"](x).numpy(), ref_q.numpy()) <= 2e-2
        assert oracle.rel_l2(model["lora"](x).numpy(), ref_l.numpy()) <= 3e-2


# ---------------------------------------------------------------------------
# exact N-fusion of layers that read the same input
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("M", [1, 5, 70])
def test_fused_w8a8_bitexact_and_parts(dev, M):
    """int8-dyn: one activation quantization for the same x and exact int32
    sums, so the fused layer must equal the separate layers bit for bit."""
    announce(f"fused w8a8 M={M}")
    K = 512
    sizes = (256, 64, 64, 4)
    ws = [make_weights(n, K, 70 + i) for i, n in enumerate(sizes)]
    bs = [torch.randn(n) if i == 1 else None for i, n in enumerate(sizes)]
    mods = [quant.DynamicInt8Linear(w, b) for w, b in zip(ws, bs)]
    fused = quant.fuse_linears(mods)
    assert fused.out_features == sum(sizes)
    x = make_x(M, K, 80, outliers=True).to(dev)
    outs = fused(x)
    for m, o in zip(mods, outs):
        assert o.is_contiguous() and o.shape == (M, m.out_features)
        np.testing.assert_array_equal(o.cpu().numpy(), m(x).cpu().numpy())
    parts = [fused.part(i) for i in range(len(sizes))]
    for m, pmod in zip(mods, parts):
        np.testing.assert_array_equal(pmod(x).cpu().numpy(), m(x).cpu().numpy())
    x.mul_(0.5)  # in-place change: the parts must not reuse the earlier launch
    for m, pmod in zip(mods, parts):
        np.testing.assert_array_equal(pmod(x).cpu().numpy(), m(x).cpu().numpy())


@pytest.mark.parametrize("M", [1, 3, 40])
def test_fused_w8_matches_parts(dev, M):
    announce(f"fused w8 M={M}")
    K = 1024
    sizes = (512, 128, 128)
    ws = [make_weights(n, K, 90 + i) for i, n in enumerate(sizes)]
    mods = [quant.Int8Linear(w, None) for w in ws]
    fused = quant.fuse_linears(mods)
    x = make_x(M, K, 99).reshape(1, M, K)
    outs = fused(x)  # CPU in, CPU out, [1, M, n]
    for w, m, o in zip(ws, mods, outs):
        assert o.device.type == "cpu" and o.shape == (1, M, m.out_features)
        q, s = oracle.quantize_per_channel(w.numpy())
        # fp32 x: bf16 high + remainder on the decode paths (M <= 16), one staged fp16 plane (11 bits) in the GEMM
        bar = 1e-5 if M <= 16 else 6e-4
        assert oracle.rel_l2(o.reshape(M, -1).numpy(), oracle.int8_linear(x.reshape(M, K).numpy(), q, s)) <= bar


def test_fuse_linears_rejects_mixed_parts(dev):
    a = quant.Int8Linear(make_weights(16, 64, 1), None)
    with pytest.raises(ValueError):
        quant.fuse_linears([a, quant.DynamicInt8Linear(make_weights(16, 64, 2), None)])
    with pytest.raises(ValueError):
        quant.fuse_linears([a, quant.Int8Linear(make_weights(16, 128, 3), None)])


# ---------------------------------------------------------------------------
# greedy token selection on the GPU (engine.py:30-31)
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("cls", ["Int8Linear", "DynamicInt8Linear"])
def test_fused_layer_saved_whole_before_the_parts_table(dev, cls):
    """A fused layer pickled without the column table (as layers once were)
    loads and slices its outputs: the same values."""
    announce(f"fused saved whole {cls}")
    fused = quant.fuse_linears([getattr(quant, cls)(make_weights(n, 256, n).to(dev), None) for n in (64, 20)])
    state = fused.__getstate__() if hasattr(fused, "__getstate__") else fused.__dict__
    state = {k: v for k, v in state.items() if k != "_pstart"}
    state["_buffers"] = {k: v for k, v in state["_buffers"].items() if k != "_parts"}
    state["_non_persistent_buffers_set"] = state["_non_persistent_buffers_set"] - {"_parts"}
    old = quant.FusedLinear.__new__(quant.FusedLinear)
    old.__setstate__(state)
    x = torch.randn(3, 256, device=dev, generator=torch.Generator(dev).manual_seed(5))
    assert all(torch.equal(a, b) for a, b in zip(old(x), fused(x)))
    assert all(torch.equal(a, b) for a, b in zip(old(x[:1]), fused(x[:1])))


def test_greedy_tokens_match_torch_argmax(dev):
    announce("greedy tokens")
    g = torch.Generator().manual_seed(3)
    V = 151936
    logits = torch.randn(3, V, generator=g)
    logits[1, 5] = logits[1, 100] = 50.0           # tie: the first index wins
    logits[2, 7] = float("nan")                     # NaN ranks above numbers
    logits[2, 9] = float("nan")
    got = quant.greedy_tokens(logits.to(dev)).cpu()
    np.testing.assert_array_equal(got.numpy(), torch.argmax(logits, dim=-1).numpy())
    assert got.tolist()[1:] == [5, 7]
    neg = torch.full((2, 1000), float("-inf"))
    assert quant.greedy_tokens(neg.to(dev)).tolist() == [0, 0]
    # rows that do not start 16-byte aligned take the scalar path
    wide = torch.randn(4, 1003, generator=g)
    sub = wide.to(dev)[:, 1:]
    np.testing.assert_array_equal(quant.greedy_tokens(sub).cpu().numpy(),
                                  torch.argmax(wide[:, 1:], dim=-1).numpy())


def test_greedy_tokens_after_lm_head(dev):
    """lm_head (model.py:447) then greedy sampling: the token equals torch's
    argmax of the same fp32 logits."""
    announce("lm_head + greedy")
    V, H = 32000, 1024
    lm = quant.Int8Linear(make_weights(V, H, 123), None)
    x = make_x(2, H, 124).to(dev)
    logits = lm(x)
    np.testing.assert_array_equal(quant.greedy_tokens(logits).cpu().numpy(),
                                  torch.argmax(logits.cpu(), dim=-1).numpy())


# ---------------------------------------------------------------------------
# pre-quantized weights: no re-quantization at load
# ---------------------------------------------------------------------------
def test_from_quantized_and_safetensors_roundtrip(dev, tmp_path):
    announce("prequantized load")
    N, K = 80, 384
    w = make_weights(N, K, 131)
    b = torch.randn(N)
    lin = quant.Int8Linear(w, b)
    dyn = quant.DynamicInt8Linear(w, None)
    x = make_x(4, K, 132).to(dev)
    same = quant.Int8Linear.from_quantized(lin.qweight, lin.scale, lin.bias)
    np.testing.assert_array_equal(same(x).cpu().numpy(), lin(x).cpu().numpy())
    path = str(tmp_path / "layers.safetensors")
    quant.save_quantized({"mlp.up": lin, "attn.q": dyn}, path)
    w8 = quant.load_quantized(path, "int8")
    np.testing.assert_array_equal(w8["mlp.up"](x).cpu().numpy(), lin(x).cpu().numpy())
    dy = quant.load_quantized(path, "int8-dyn")
    np.testing.assert_array_equal(dy["attn.q"](x).cpu().numpy(), dyn(x).cpu().numpy())
    with pytest.raises(ValueError):
        quant.load_quantized(path, "float8")


# (N, K, weight dtype, bias): ragged N and K (neither a multiple of the 16 x 64
# tile), a tile-aligned layer, and bf16 weights as loader.py:40,49 hands them
# to make_linear
SAVED_LAYERS = [(77, 200, "f32", True), (130, 4100, "bf16", False), (64, 256, "f32", False),
                (1000, 2560, "bf16", True)]


def test_saved_file_matches_oracle_quantization(dev, tmp_path):
    """The on-disk pre-quantized format against the oracle, not against this
    build's own layers: every <name>.qweight / <name>.scale in a
    save_quantized file equals the oracle's quantize_per_channel of the source
    weight (quant.py:25-29, the buffers of quant.py:36-37) bit for bit, for
    Int8Linear and for DynamicInt8Linear (saved from its packed tiles through
    unpack); <name>.bias is the fp32 bias.  The layers load_quantized builds
    from the file then match the oracle: int8 within the weight-only bar
    (rel-L2 1e-3; 2e-6 for fp16-valued inputs, which the kernels use exactly),
    int8-dyn int32 accumulators and outputs bit-exact."""
    from safetensors import safe_open

    announce("saved pre-quantized file vs oracle")
    srcs, mods = {}, {}
    for i, (N, K, wd, has_b) in enumerate(SAVED_LAYERS):
        w = make_weights(N, K, 150 + i).to(DT[wd])
        b = torch.randn(N, generator=torch.Generator().manual_seed(160 + i)) if has_b else None
        for kind, cls in (("w8", quant.Int8Linear), ("dyn", quant.DynamicInt8Linear)):
            name = f"layer{i}.{kind}"
            srcs[name] = (w, b)
            mods[name] = cls(w.to(dev), None if b is None else b.to(dev))
    path = str(tmp_path / "prequant.safetensors")
    quant.save_quantized(mods, path)
    with safe_open(path, framework="pt") as f:
        keys = set(f.keys())
        for name, (w, b) in srcs.items():
            q_ref, s_ref = oracle.quantize_per_channel(w.float().numpy())
            q = f.get_tensor(name + ".qweight")
            s = f.get_tensor(name + ".scale")
            assert q.dtype == torch.int8 and s.dtype == torch.float32, name
            np.testing.assert_array_equal(q.numpy(), q_ref, err_msg=name)
            np.testing.assert_array_equal(s.numpy().view(np.uint32), s_ref.view(np.uint32), err_msg=name)
            if b is None:
                assert name + ".bias" not in keys, name
            else:
                np.testing.assert_array_equal(f.get_tensor(name + ".bias").numpy(), b.float().numpy(), err_msg=name)
    loaded = {"int8": quant.load_quantized(path, "int8"), "int8-dyn": quant.load_quantized(path, "int8-dyn")}
    for i, (N, K, wd, has_b) in enumerate(SAVED_LAYERS):
        for name in (f"layer{i}.w8", f"layer{i}.dyn"):
            w, b = srcs[name]
            q_ref, s_ref = oracle.quantize_per_channel(w.float().numpy())
            bn = None if b is None else b.float().numpy()
            for M, xd in ((1, torch.float32), (5, torch.float16), (40, torch.float32), (300, torch.float16)):
                x = make_x(M, K, 170 + M, outliers=True).to(xd)
                xv = x.float().numpy()
                lin8 = loaded["int8"][name]
                assert isinstance(lin8, quant.Int8Linear)
                np.testing.assert_array_equal(lin8.qweight.cpu().numpy(), q_ref)
                y = lin8(x.to(dev)).cpu().numpy()
                tol = W8_TOL if xd == torch.float32 else 2e-6
                assert oracle.rel_l2(y, oracle.int8_linear(xv, q_ref, s_ref, bn)) <= tol, (name, M)
                dyn = loaded["int8-dyn"][name]
                assert isinstance(dyn, quant.DynamicInt8Linear)
                acc = torch.empty((M, N), dtype=torch.int32, device=dev)
                xg = x.to(dev)
                yd = quant.linear_w8a8(xg, dyn.packed, dyn.scale, dyn.colsum, dyn.bias, N, acc_out=acc)
                y_ref, info = oracle.dyn_linear(xv, q_ref, s_ref, bn, return_intermediates=True)
                np.testing.assert_array_equal(acc.cpu().numpy(), info["acc"], err_msg=f"{name} M={M}")
                np.testing.assert_array_equal(yd.cpu().numpy(), y_ref, err_msg=f"{name} M={M}")
                np.testing.assert_array_equal(dyn(xg).cpu().numpy(), y_ref, err_msg=f"{name} M={M} forward")


# ---------------------------------------------------------------------------
# HIP graph capture: every entry point replays correctly with eager work between
# ---------------------------------------------------------------------------
def test_graph_replays_match_eager(dev):
    announce("graph replays")
    K = 1024
    w = make_weights(320, K, 141)
    lin = quant.Int8Linear(w, torch.randn(320))
    dyn = quant.DynamicInt8Linear(w, None)
    shapes = [(1, True), (3, False), (96, True)]  # fast GEMV, general GEMV (misaligned rows), GEMM
    xs = []
    for M, aligned in shapes:
        big = make_x(M, K + 8, 142 + M).to(dev)
        xs.append(big[:, :K] if aligned else big[:, 1:1 + K])
    ws_dyn = [quant.w8a8_workspace(x.shape[0], K, dev) for x in xs]
    outs = {}

    def body():
        for i, x in enumerate(xs):
            outs[("w8", i)] = quant.linear_w8(x, lin.packed, lin.scale, lin.bias, 320)
            outs[("dyn", i)] = quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum, None, 320,
                                                 workspace=ws_dyn[i])
        outs["tok"] = quant.greedy_tokens(outs[("w8", 0)])

    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        body()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        body()
    for rep in range(3):
        for x in xs:  # eager work between replays: new activations in place
            x.mul_(-1.25).add_(0.5 * rep)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for i, x in enumerate(xs):
            eager_w8 = quant.linear_w8(x, lin.packed, lin.scale, lin.bias, 320)
            eager_dyn = quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum, None, 320)
            np.testing.assert_array_equal(outs[("w8", i)].cpu().numpy(), eager_w8.cpu().numpy(),
                                          err_msg=f"w8 replay {rep} M={x.shape[0]}")
            np.testing.assert_array_equal(outs[("dyn", i)].cpu().numpy(), eager_dyn.cpu().numpy(),
                                          err_msg=f"w8a8 replay {rep} M={x.shape[0]}")
        assert outs["tok"].item() == int(torch.argmax(outs[("w8", 0)][0]).item())


def test_graph_replays_size_dependent_paths(dev):
    """Paths chosen by activation size, replayed from a HIP graph with new
    activations written between replays: the in-kernel W8A8 min/max over 24
    and 48 KiB of x, the prefill quantizer at 1 and 2 chunks per thread with
    256- and 512-thread min/max workgroups, and the 48 KiB fp32 split of the
    decode GEMV."""
    announce("graph replays, size-dependent paths")
    N = 320
    cases = [(1, 12288, torch.float16), (2, 12288, torch.float16), (128, 4096, torch.float16),
             (512, 4096, torch.float16), (1, 12288, torch.float32)]
    mods = {}
    for _, K, _ in cases:
        if K not in mods:
            w = make_weights(N, K, 150 + K)
            mods[K] = (quant.Int8Linear(w, None), quant.DynamicInt8Linear(w, None))
    xs = [make_x(M, K, 160 + M + K, outliers=True).to(xd).to(dev) for M, K, xd in cases]
    wss = [quant.w8a8_workspace(M, K, dev) for M, K, _ in cases]
    outs = {}

    def body():
        for i, (x, (M, K, _)) in enumerate(zip(xs, cases)):
            lin, dyn = mods[K]
            outs[("w8", i)] = quant.linear_w8(x, lin.packed, lin.scale, None, N)
            outs[("dyn", i)] = quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum, None, N, workspace=wss[i])

    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        body()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        body()
    for rep in range(3):
        for x in xs:
            x.mul_(-1.5).add_(0.25 * rep)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for i, (x, (M, K, xd)) in enumerate(zip(xs, cases)):
            lin, dyn = mods[K]
            eager_w8 = quant.linear_w8(x, lin.packed, lin.scale, None, N)
            eager_dyn = quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum, None, N)
            np.testing.assert_array_equal(outs[("w8", i)].cpu().numpy(), eager_w8.cpu().numpy(),
                                          err_msg=f"w8 replay {rep} M={M} K={K} {xd}")
            np.testing.assert_array_equal(outs[("dyn", i)].cpu().numpy(), eager_dyn.cpu().numpy(),
                                          err_msg=f"w8a8 replay {rep} M={M} K={K} {xd}")


# ---------------------------------------------------------------------------
# concurrency: the library keeps no state, so calls on two streams at once
# give the same results as the same calls one after the other
# ---------------------------------------------------------------------------
def test_concurrent_streams_match_sequential(dev):
    announce("two streams")
    K = 4096
    layers = [quant.Int8Linear(make_weights(N, K, 160 + i), None) for i, N in enumerate((6144, 4096))]
    dyns = [quant.DynamicInt8Linear(make_weights(N, K, 170 + i), None) for i, N in enumerate((4096, 1024))]
    xs = [make_x(M, K, 180 + M).to(dev).half() for M in (1, 8, 300)]
    # a workspace is scratch of one call at a time: one per stream and size
    wss = {(i, M): quant.w8a8_workspace(M, K, dev) for i in range(2) for M in (1, 8, 300)}

    def work(i, x):
        lin, dyn = layers[i], dyns[i]
        return (quant.linear_w8(x, lin.packed, lin.scale, None, lin.out_features),
                quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum, None, dyn.out_features,
                                  workspace=wss[(i, x.shape[0])]))

    ref = [[work(i, x) for x in xs] for i in range(2)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]  # default priority
    got = [[None] * len(xs) for _ in range(2)]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    for j, x in enumerate(xs):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i][j] = work(i, x)
    torch.cuda.synchronize()
    for i in range(2):
        for j, x in enumerate(xs):
            for a, b in zip(got[i][j], ref[i][j]):
                np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy(), err_msg=f"stream {i} M={x.shape[0]}")


def test_concurrent_host_threads_match_sequential(dev):
    """Host threads calling the library at once, each on its own stream with
    its own workspaces (ctypes releases the GIL for every call, so the calls
    overlap on the host as well as on the GPU): module calls, the greedy
    token (separate and fused with lm_head) and the sampler give the results
    of the same calls made one after the other."""
    import threading

    announce("four host threads")
    K, V = 2560, 20000
    lins = [quant.Int8Linear(make_weights(N, K, 190 + i), None) for i, N in enumerate((9728, 1024))]
    dyns = [quant.DynamicInt8Linear(make_weights(N, K, 195 + i), None) for i, N in enumerate((4096, 640))]
    head = quant.Int8Linear(make_weights(V, K, 199), None)
    xs = [make_x(M, K, 200 + M).to(dev).half() for M in (1, 4, 24, 160)]
    uni = torch.rand(4, generator=torch.Generator().manual_seed(205)).to(dev)
    torch.cuda.synchronize()  # inputs and packed weights made on the default stream

    def work(t, reps):
        s = torch.cuda.Stream()  # default priority
        out = []
        with torch.cuda.stream(s):
            for _ in range(reps):
                res = []
                for j, x in enumerate(xs):
                    lin, dyn = lins[(t + j) % 2], dyns[(t + j) % 2]
                    res.append(lin(x))
                    res.append(dyn(x))
                logits = head(xs[1])
                res.append(quant.greedy_tokens(logits))
                res.append(quant.sample_tokens(logits, 0.7, top_p=0.9, u=uni))
                res.extend(head.forward_greedy(xs[1]))  # a fused-argmax state per stream
                out = res
        s.synchronize()
        return out

    ref = [work(t, 1) for t in range(4)]
    got = [None] * 4
    errs = []

    def run(t):
        try:
            got[t] = work(t, 3)
        except Exception as e:  # reported below, not lost in the thread
            errs.append(repr(e))

    threads = [threading.Thread(target=run, args=(t,)) for t in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not errs, errs
    for t in range(4):
        assert len(got[t]) == len(ref[t])
        for k, (a, b) in enumerate(zip(got[t], ref[t])):
            np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy(), err_msg=f"thread {t} result {k}")


# ---------------------------------------------------------------------------
# model-level fidelity, as the reference's loader test checks its formats
# (tests/test_model.py:180-192: logits of a tiny random model in each format
# against float32, cosine > 0.99, > 0.95 for int8-dyn)
# ---------------------------------------------------------------------------
def _toy_model_logits(fmt, weights, emb, tokens, heads=4):
    """Embedding, then two blocks of q/k/v/o projections around causal
    attention and a gated MLP (the projection pattern of model.py:240-270),
    then the tied lm_head; every linear comes from make_linear(fmt) and runs
    on CPU fp32 tensors, as the reference model calls them."""
    lin = {name: quant.make_linear(fmt, w) for name, w in weights.items()}
    lin["lm_head"] = quant.make_linear(fmt, emb)
    x = emb[tokens]  # [T, H]
    T, H = x.shape
    d = H // heads
    mask = torch.full((T, T), float("-inf")).triu(1)

    def norm(t):
        return t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + 1e-6)

    for blk in range(2):
        h = norm(x)
        q, k, v = (lin[f"{blk}.{p}"](h).view(T, heads, d).transpose(0, 1) for p in ("q", "k", "v"))
        att = torch.softmax(q @ k.transpose(1, 2) / d ** 0.5 + mask, dim=-1) @ v
        x = x + lin[f"{blk}.o"](att.transpose(0, 1).reshape(T, H))
        h = norm(x)
        x = x + lin[f"{blk}.down"](torch.nn.functional.silu(lin[f"{blk}.gate"](h)) * lin[f"{blk}.up"](h))
    return lin["lm_head"](norm(x))[-1]


@pytest.mark.parametrize("T", [40, 1])
def test_toy_model_fidelity_per_format(dev, T):
    announce(f"toy model fidelity T={T}")
    g = torch.Generator().manual_seed(4)
    H, F, V = 512, 1536, 1000
    shapes = {"q": (H, H), "k": (H, H), "v": (H, H), "o": (H, H), "gate": (F, H), "up": (F, H), "down": (H, F)}
    weights = {f"{b}.{n}": torch.randn(*s, generator=g) * 0.02 for b in range(2) for n, s in shapes.items()}
    emb = torch.randn(V, H, generator=g)
    tokens = torch.randint(0, V, (T,), generator=g)
    ref = _toy_model_logits("float32", weights, emb, tokens)
    for fmt in ("bfloat16", "float16", "int8", "int8-dyn"):
        got = _toy_model_logits(fmt, weights, emb, tokens)
        assert got.device.type == "cpu" and got.dtype == torch.float32
        cos = float(torch.nn.functional.cosine_similarity(got, ref, dim=0))
        assert cos > (0.95 if fmt == "int8-dyn" else 0.99), (fmt, cos)  # the reference's bar
        # the oracle's arithmetic in the same toy model reaches 0.99995 (int8-dyn) and 0.99998 (int8)
        assert cos > (0.999 if fmt == "int8-dyn" else 0.9999), (fmt, cos)


# ---------------------------------------------------------------------------
# fp16 / bf16 outputs of the prefill GEMM leave through an LDS-staged
# epilogue; fp32 outputs are stored directly.  Both compute the same fp32
# value, so the 2-byte output must equal the fp32 output rounded on the host,
# for every block configuration, ragged M and N, and strided / misaligned rows.
# ---------------------------------------------------------------------------
def _bits(t):
    """Raw 16-bit patterns of a 2-byte tensor (numpy has no bfloat16)."""
    return t.contiguous().view(torch.int16).cpu().numpy()


LEPI_CASES = [(2048, 12288, 128), (2048, 4096, 192), (1024, 4096, 256), (100, 1000, 320), (1000, 12290, 256),
              (2048, 24576, 128), (256, 8192, 448), (512, 12288, 256), (500, 12300, 192), (512, 6144, 320)]


@pytest.mark.parametrize("M,N,K", LEPI_CASES)
def test_gemm_2byte_outputs_equal_rounded_fp32(dev, M, N, K):
    """Also with a bias: the last fma of the epilogue must round to fp32 before
    the 16-bit conversion (a fused fma-to-fp16 rounds once and differs in about
    one output in 20000)."""
    announce(f"gemm 2-byte outputs M={M} N={N} K={K}")
    w = make_weights(N, K, 4100 + N + K)
    x = make_x(M, K, 4200 + M + K, outliers=True).half().to(dev)
    lin = quant.Int8Linear(w, None)
    dyn = quant.DynamicInt8Linear(w, None)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(4300 + N)).to(dev)
    for b in (None, bias):
        y32 = quant.linear_w8(x, lin.packed, lin.scale, b, N)
        d32 = quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum, b, N)
        t32 = quant.linear_w8a8_token(x, dyn.packed, dyn.scale, b, N)
        for od in (torch.float16, torch.bfloat16):
            wide = torch.empty((M, N + 3), dtype=od, device=dev)
            for out in (None, wide[:, :N]):  # dense rows; rows with an odd stride (no 16-byte stores)
                got = quant.linear_w8(x, lin.packed, lin.scale, b, N, od, out=out)
                np.testing.assert_array_equal(_bits(got), _bits(y32.to(od)))
                got = quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum, b, N, od, out=out)
                np.testing.assert_array_equal(_bits(got), _bits(d32.to(od)))
                got = quant.linear_w8a8_token(x, dyn.packed, dyn.scale, b, N, od, out=out)
                np.testing.assert_array_equal(_bits(got), _bits(t32.to(od)))
    xb = x.to(torch.bfloat16)  # bf16 activations without a workspace: the bf16 kernel
    ref = quant.linear_w8(xb, lin.packed, lin.scale, None, N, workspace=torch.empty(0, dtype=torch.uint8, device=dev))
    got = quant.linear_w8(xb, lin.packed, lin.scale, None, N, torch.bfloat16,
                          workspace=torch.empty(0, dtype=torch.uint8, device=dev))
    np.testing.assert_array_equal(_bits(got), _bits(ref.to(torch.bfloat16)))


@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (4, 6144, 4096), (16, 1000, 2560), (24, 4096, 4096), (1, 4096, 12288)])
def test_gemv_2byte_outputs_equal_rounded_fp32(dev, M, N, K):
    """Decode GEMVs (fast path for M <= 16, general kernel beyond): fp16 /
    bf16 outputs, with and without a bias, equal the fp32 output rounded."""
    announce(f"gemv 2-byte outputs M={M} N={N} K={K}")
    w = make_weights(N, K, 4400 + N + K)
    x = make_x(M, K, 4500 + M + K, outliers=True).half().to(dev)
    lin = quant.Int8Linear(w, None)
    dyn = quant.DynamicInt8Linear(w, None)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(4600 + N)).to(dev)
    for b in (None, bias):
        y32 = quant.linear_w8(x, lin.packed, lin.scale, b, N)
        d32 = quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum, b, N)
        for od in (torch.float16, torch.bfloat16):
            got = quant.linear_w8(x, lin.packed, lin.scale, b, N, od)
            np.testing.assert_array_equal(_bits(got), _bits(y32.to(od)))
            got = quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum, b, N, od)
            np.testing.assert_array_equal(_bits(got), _bits(d32.to(od)))


def test_graph_replays_lds_epilogue(dev):
    """fp16 outputs of one-group GEMM blocks (the LDS-staged epilogue, W-only
    and W8A8) replayed from a HIP graph with eager work between replays."""
    announce("graph replays, LDS-staged epilogue")
    M, N, K = 1024, 4096, 1024
    w = make_weights(N, K, 190)
    lin = quant.Int8Linear(w, None)
    dyn = quant.DynamicInt8Linear(w, None)
    x = make_x(M, K, 191).half().to(dev)
    ws8 = quant.w8_workspace(M, K, dev)
    wsd = quant.w8a8_workspace(M, K, dev)
    y8 = torch.empty((M, N), dtype=torch.float16, device=dev)
    yd = torch.empty((M, N), dtype=torch.float16, device=dev)

    def body():
        quant.linear_w8(x, lin.packed, lin.scale, None, N, torch.float16, out=y8, workspace=ws8)
        quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum, None, N, torch.float16, workspace=wsd, out=yd)

    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        body()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        body()
    for rep in range(3):
        x.mul_(-1.5).add_(0.25 * rep)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        ref8 = quant.linear_w8(x, lin.packed, lin.scale, None, N).to(torch.float16)
        refd = quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum, None, N).to(torch.float16)
        np.testing.assert_array_equal(_bits(y8), _bits(ref8), err_msg=f"w8 replay {rep}")
        np.testing.assert_array_equal(_bits(yd), _bits(refd), err_msg=f"w8a8 replay {rep}")


# ---------------------------------------------------------------------------
# seeded random shapes: every dispatch path (fast / general GEMV, each GEMM
# block configuration, the register-staged GEMM) against the oracle, with
# random activation and output dtypes and aligned or misaligned row strides
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("M,N,K,xd,yd,pad", [
    (31, 51, 15, "f16", "f16", 1), (17, 942, 64, "f32", "f16", 8), (32, 100, 256, "bf16", "f32", 1),
    (20, 33, 128, "f16", "bf16", 3), (17, 64, 64, "f32", "f32", 1), (24, 300, 200, "f32", "f32", 0),
])
def test_general_gemv_two_row_tiles_short_k(dev, M, N, K, xd, yd, pad):
    """17..32 tokens at short K on the general GEMV (ragged K or misaligned
    rows keep them off the fast paths): one wave covers K, and the second row
    tile of x still gets its outputs (a workgroup of one wave once left rows
    16..M-1 unwritten).  Both formats against the oracle."""
    announce(f"general gemv two row tiles M={M} N={N} K={K} x={xd} y={yd} pad={pad}")
    w = make_weights(N, K, 7100 + M)
    big = torch.zeros((M, K + pad), dtype=DT[xd])
    big[:, pad:] = make_x(M, K, 7200 + M, outliers=True).to(DT[xd])
    x = big.to(dev)[:, pad:]
    xv = x.float().cpu().numpy()
    q, s = oracle.quantize_per_channel(w.numpy())
    lin = quant.Int8Linear(w, None)
    dyn = quant.DynamicInt8Linear(w, None)
    y = torch.full((M, N), float("nan"), dtype=DT[yd], device=dev)
    quant.linear_w8(x, lin.packed, lin.scale, None, N, out=y)
    err = oracle.rel_l2(y.float().cpu().numpy(), oracle.int8_linear(xv, q, s))
    assert err <= {"f32": W8_TOL, "f16": W8_TOL, "bf16": 5e-3}[yd], err
    acc = torch.full((M, N), -7, dtype=torch.int32, device=dev)
    yd8 = quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum, None, N, acc_out=acc)
    refd, info = oracle.dyn_linear(xv, q, s, return_intermediates=True)
    np.testing.assert_array_equal(acc.cpu().numpy(), info["acc"])
    np.testing.assert_array_equal(yd8.cpu().numpy(), refd)


def _random_cases(n, seed):
    g = np.random.default_rng(seed)
    cases = []
    for i in range(n):
        M = int(g.choice([1, 2, 3, 5, 8, 13, 16, 17, 31, 33, 64, 65, 100, 128, 200, 257, 300, 384]))
        N = int(g.integers(1, 2049))
        K = int(g.choice([int(g.integers(1, 2049)), 64 * int(g.integers(1, 33))]))
        xd = str(g.choice(["f32", "f16", "bf16"]))
        yd = str(g.choice(["f32", "f16", "bf16"]))
        pad = int(g.choice([0, 0, 1, 8]))  # extra row elements; odd pads misalign the rows
        cases.append((i, M, N, K, xd, yd, pad))
    return cases


@pytest.mark.parametrize("i,M,N,K,xd,yd,pad", _random_cases(40, 2024))
def test_random_shapes_match_oracle(dev, i, M, N, K, xd, yd, pad):
    announce(f"random case {i}: M={M} N={N} K={K} x={xd} y={yd} pad={pad}")
    w = make_weights(N, K, 5000 + i)
    xf = make_x(M, K, 5100 + i, outliers=True)
    big = torch.zeros((M, K + pad), dtype=DT[xd])
    big[:, pad:] = xf.to(DT[xd])
    x = big.to(dev)[:, pad:]  # row stride K + pad, first row offset by pad elements
    xv = x.float().cpu().numpy()
    q, s = oracle.quantize_per_channel(w.numpy())
    lin = quant.Int8Linear(w, None)
    dyn = quant.DynamicInt8Linear(w, None)
    # int8 weight-only: rel-L2 against the oracle.  fp32 outputs: the path's 1e-3, and fp32 summation order only
    # for exact (fp16 / bf16) inputs; 2-byte outputs add one output rounding (rms 2^-11 / sqrt 3 for fp16,
    # 2^-8 / sqrt 3 for bf16)
    y = quant.linear_w8(x, lin.packed, lin.scale, None, N, DT[yd])
    ref = oracle.int8_linear(xv, q, s)
    err = oracle.rel_l2(y.float().cpu().numpy(), ref)
    bound = {"f32": 2e-6 if xd != "f32" else W8_TOL, "f16": W8_TOL, "bf16": 5e-3}[yd]
    assert err <= bound, err
    # int8-dyn: int32 accumulators bit-exact, fp32 outputs bit-exact
    acc = torch.empty((M, N), dtype=torch.int32, device=dev)
    yd8 = quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum, None, N, acc_out=acc)
    refd, info = oracle.dyn_linear(xv, q, s, return_intermediates=True)
    np.testing.assert_array_equal(acc.cpu().numpy(), info["acc"])
    np.testing.assert_array_equal(yd8.cpu().numpy(), refd)


def _random_prefill_cases(n, seed):
    """Prefill-sized shapes (grids of every block configuration), M*N*K <= 3e9."""
    g = np.random.default_rng(seed)
    cases = []
    for i in range(n):
        while True:
            M = int(g.choice([33, 100, 128, 250, 256, 384, 500, 512, 640, 1000, 1024, 1536, 2048]))
            N = int(g.choice([int(g.integers(16, 16385)), 16 * int(g.integers(1, 1025)), 4096, 6144, 12288]))
            K = 64 * int(g.integers(1, 33)) if g.random() < 0.8 else int(g.integers(1, 2049))
            if M * N * K <= 3 * 10 ** 9:
                break
        xd = str(g.choice(["f32", "f16", "bf16"]))
        ws = str(g.choice(["auto", "none"]))
        cases.append((i, M, N, K, xd, ws))
    return cases


@pytest.mark.parametrize("i,M,N,K,xd,ws", _random_prefill_cases(40, 2025))
def test_random_prefill_shapes_match_oracle(dev, i, M, N, K, xd, ws):
    """Seeded prefill shapes across the GEMM block configurations, with and
    without a workspace: W-only to fp32 summation order for fp16 / bf16
    inputs (1e-3 for fp32 inputs), W8A8 acc and y bit-exact."""
    announce(f"random prefill case {i}: M={M} N={N} K={K} x={xd} ws={ws}")
    w = make_weights(N, K, 5200 + i)
    x = make_x(M, K, 5300 + i, outliers=True).to(DT[xd]).to(dev)
    xv = x.float().cpu().numpy()
    q, s = oracle.quantize_per_channel(w.numpy())
    lin = quant.Int8Linear(w, None)
    dyn = quant.DynamicInt8Linear(w, None)
    kw = {} if ws == "auto" else {"workspace": torch.empty(0, dtype=torch.uint8, device=dev)}
    y = quant.linear_w8(x, lin.packed, lin.scale, None, N, **kw)
    err = oracle.rel_l2(y.cpu().numpy(), oracle.int8_linear(xv, q, s))
    assert err <= (2e-6 if xd != "f32" else W8_TOL), err
    acc = torch.empty((M, N), dtype=torch.int32, device=dev)
    yd8 = quant.linear_w8a8(x, dyn.packed, dyn.scale, dyn.colsum, None, N, acc_out=acc)
    refd, info = oracle.dyn_linear(xv, q, s, return_intermediates=True)
    np.testing.assert_array_equal(acc.cpu().numpy(), info["acc"])
    np.testing.assert_array_equal(yd8.cpu().numpy(), refd)
