"""Which kernels the C ABI launches, without a GPU (tests/host/dispatch.py):
the library's host code runs over a recorder in place of the HIP runtime, on
made-up addresses that nothing reads."""
import json
import math
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HOST = ROOT / "tests" / "host"
PKG = ROOT / "spikingbrain-cpu_amd" / "sbq"


@pytest.fixture(scope="module")
def dispatch(tmp_path_factory):
    so = tmp_path_factory.mktemp("trace") / "launch_trace.so"
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-std=c++17", "-Wall", str(HOST / "launch_trace.cpp"),
                    "-o", str(so)], check=True)

    def run(calls, axes=1):
        """[(status, [kernel name with template arguments, ...], [(workgroups, threads of one), ...])]; the
        workgroups counted along x, or over the given number of axes"""
        r = subprocess.run([sys.executable, str(HOST / "dispatch.py"), str(so), str(PKG / "libsbq.so"), str(PKG)],
                           input=json.dumps(calls), capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        return [(t["rc"], [ln[0] for ln in t["launches"]], [(math.prod(ln[1][:axes]), ln[2][0]) for ln in t["launches"]])
                for t in json.loads(r.stdout)]

    return run


def kernels(names):
    return [n.split("<")[0] for n in names]


def test_ragged_k_beyond_the_decode_gemv_is_staged(dispatch):
    """K % 64 != 0 beyond the decode GEMVs' 12288: every weight-only entry point
    takes decode sizes (they run the tiled GEMM on rows of whole tiles)."""
    calls = [{"op": op, "M": M, "N": 1000, "K": K, "x": x, "ws": ws}
             for op in ("linear_w8", "linear_w8_parts", "linear_w8_argmax") for M in (1, 2, 4, 16)
             for K in (12289, 13000, 20001) for x in ("f32", "f16", "bf16") for ws in ("base", "full")]
    for c, (rc, names, _) in zip(calls, dispatch(calls)):
        assert rc == 0 and kernels(names)[:2] == ["pad_rows_kernel", "gemm_dl_kernel"], (c, rc, names)


@pytest.mark.parametrize("fmt", ["w8", "w8a8"])
def test_greedy_logits_take_the_route_of_the_linear(dispatch, fmt):
    """The greedy entry points compute the logits with the launches of the plain
    linear (decode, ragged K, long K, mid-sized and prefill M, with and without
    the workspace): the bits of forward."""
    ws = (None, "base", "full") if fmt == "w8" else ("base", "full")
    shapes = [{"M": M, "N": N, "K": K, "x": x, "ws": w, "off": off} for M in (1, 2, 5, 8, 16, 17, 20, 40, 100)
              for N, K in ((2999, 2500), (1000, 130), (18820, 128), (151936, 2561), (4096, 4096), (700, 13000))
              for x in ("f32", "f16", "bf16") for w in ws for off in (0, 1)]
    plain = dispatch([dict(s, op=f"linear_{fmt}") for s in shapes])
    greedy = dispatch([dict(s, op=f"linear_{fmt}_argmax") for s in shapes])
    for s, p, g in zip(shapes, plain, greedy):
        assert p[0] == 0 and g[0] == 0, (s, p, g)
        n = len(p[1])
        assert g[1][:n] == p[1] and g[2][:n] == p[2], (s, p, g)
        assert all("argmax" in k for k in g[1][n:]), (s, g)


def test_every_aligned_decode_pick_launches(dispatch):
    """The configuration picked for an aligned decode call (whole K tiles) is
    one its K leaves enough waves for: the fast GEMV runs, never the general
    one behind it (which weight-only fp16 / bf16 keeps at M > 8 and up to four
    K tiles).  Workgroups of five and six row tiles need as many waves, each
    with a K tile."""
    calls = [{"op": op, "M": M, "N": N, "K": 64 * Kc, "x": x, "ws": "full"}
             for op in ("linear_w8", "linear_w8a8") for x in ("f32", "f16", "bf16") for M in (1, 2, 3, 4, 6, 8, 9, 12, 16)
             for Kc in (1, 2, 3, 4, 5, 6, 7, 9, 10, 11, 13, 17, 25, 33, 40, 49, 64, 65, 127, 128, 192)
             for N in (64, 3000, 4097, 6144, 12000, 16385, 17000, 18820, 20480, 20500, 24576, 24600, 30000, 151936)
             if op == "linear_w8a8" or x == "f32" or M <= 8 or Kc > 4]
    for c, (rc, names, _) in zip(calls, dispatch(calls)):
        assert rc == 0 and kernels(names)[-1] == "gemv_fast_kernel", (c, rc, names)


def test_wide_grouped_int8_dyn_is_one_launch(dispatch):
    """Groups of more than 4096 row tiles in all with more than 32 KiB of x: all
    inputs quantized in one launch (a workgroup each) and one GEMV when every
    linear has its share of the workspace; without it, the fused launch."""
    for n, M, N, K, x in ((3, 4, 27866, 2688, "f32"), (3, 8, 71403, 1216, "f32"), (2, 8, 40000, 4096, "f16"),
                          (4, 5, 33000, 4096, "bf16")):
        c = {"op": "linear_w8a8_grouped", "M": M, "N": N, "K": K, "x": x, "count": n}
        (rc, names, grids), (rc1, names1, _) = dispatch([dict(c, ws=str(n)), dict(c, ws="base")])
        assert rc == 0 and kernels(names) == ["quantize_small_kernel", "gemv_fast_kernel"] and grids[0][0] == n, (c, names)
        assert rc1 == 0 and kernels(names1) == ["gemv_fast_kernel"], (c, names1)


# (M, N, K, x, off, kernels): both sides of each line of pad_ragged_rows
GENERAL, PADDED, STAGED = (["gemv_kernel"], ["pad_rows_kernel", "gemv_fast_kernel"], ["pad_rows_kernel", "gemm_dl_kernel"])
RAGGED_LINES = [
    (1, 300, 4095, "f32", 0, GENERAL), (1, 300, 4097, "f32", 0, PADDED), (1, 20000, 2500, "f16", 0, GENERAL),
    (2, 300, 383, "f32", 0, GENERAL), (2, 300, 385, "f32", 0, PADDED), (2, 300, 2500, "f32", 0, GENERAL),
    (2, 300, 2500, "f32", 1, PADDED), (2, 4000, 2500, "f32", 0, PADDED),
    (4, 20, 631, "f32", 0, GENERAL), (8, 300, 1025, "f32", 0, PADDED), (8, 300, 1028, "f32", 0, PADDED),
    (5, 20000, 500, "f32", 0, PADDED), (16, 300, 4095, "f32", 0, GENERAL), (16, 300, 4097, "f32", 0, PADDED),
    (2, 300, 1535, "f16", 0, GENERAL), (2, 300, 1537, "f16", 0, PADDED), (2, 300, 2504, "bf16", 0, GENERAL),
    (11, 36683, 72, "f16", 0, GENERAL), (11, 36683, 160, "f16", 0, GENERAL), (11, 36683, 161, "f16", 0, GENERAL),
    (8, 300, 769, "bf16", 0, PADDED), (8, 300, 776, "bf16", 0, GENERAL), (8, 300, 776, "bf16", 1, PADDED),
    (16, 4000, 2504, "f16", 0, GENERAL), (16, 5000, 2504, "f16", 0, PADDED), (4, 300, 6152, "f16", 0, PADDED),
    (20, 300, 631, "f32", 0, GENERAL), (20, 300, 1025, "f32", 0, STAGED), (20, 2692, 313, "f32", 0, GENERAL),
    (20, 300, 127, "f16", 0, GENERAL), (20, 300, 129, "f16", 0, STAGED), (28, 2431, 2168, "f16", 0, GENERAL),
    (28, 2431, 2168, "f16", 1, STAGED), (32, 12780, 3000, "f16", 0, STAGED), (33, 300, 65, "f16", 0, STAGED),
]


@pytest.mark.parametrize("op", ["linear_w8", "linear_w8_argmax"])
def test_ragged_rows_are_padded_where_it_pays(dispatch, op):
    """Ragged weight-only calls that the general GEMV takes run it until K or
    the layer outweighs the padding launch; misaligned rows sooner than rows
    it reads with vector loads.  Without the workspace nothing is padded."""
    calls = [{"op": op, "M": M, "N": N, "K": K, "x": x, "off": off, "ws": "full"} for M, N, K, x, off, _ in RAGGED_LINES]
    for c, (*_, want), (rc, names, _) in zip(calls, RAGGED_LINES, dispatch(calls)):
        assert rc == 0 and kernels(names)[:len(want)] == want, (c, names)
    for c, (rc, names, _) in zip(calls, dispatch([dict(c, ws=None) for c in calls])):
        assert rc == 0 and kernels(names)[0] in ("gemv_kernel", "gemm_w8_kernel"), (c, names)


def test_small_activations_are_quantized_in_one_launch(dispatch):
    """int8-dyn beyond the fused capacity: one quantizing launch up to 20 chunks
    of dense x per thread (81920 values), 32768 values of rows that are not
    dense, and two beyond."""
    one, two = "quantize_small_kernel", ("minmax_partial_kernel", "minmax_dense_kernel")
    for M, K, off, want in ((8, 4033, 0, one), (8, 4096, 1, one), (9, 4033, 0, two), (9, 4096, 1, two), (20, 4096, 0, one),
                            (21, 4096, 0, two), (32, 1024, 1, one), (33, 1023, 0, two), (3, 77, 0, one)):
        for x in ("f32", "f16", "bf16"):
            c = {"op": "linear_w8a8", "M": M, "N": 5000, "K": K, "x": x, "off": off, "ws": "full"}
            if x != "f32" and M <= 8 and K % 64 == 0 and not off:
                continue  # within the fused capacity
            rc, names, _ = dispatch([c])[0]
            assert rc == 0 and kernels(names)[0] in want, (c, names)


# (op, M, N, K, x, template of the GEMV: D, G, x in LDS, waves): both sides of
# the lines between picks, where the other one was measured slower
PICKS = [
    ("linear_w8", 2, 97455, 4864, "f32", (4, 2, False, 4)), ("linear_w8", 2, 8000, 4864, "f32", (4, 2, True, 8)),
    ("linear_w8", 2, 97455, 4096, "f32", (4, 2, True, 8)), ("linear_w8", 1, 97455, 4864, "f32", (4, 2, True, 8)),
    ("linear_w8", 1, 10000, 1024, "f16", (8, 1, True, 2)), ("linear_w8", 1, 10000, 1536, "f16", (8, 1, True, 4)),
    ("linear_w8", 1, 10000, 2560, "f16", (8, 1, True, 2)),
    ("linear_w8a8", 1, 19456, 2560, "f16", (8, 1, False, 2)), ("linear_w8a8", 1, 19456, 384, "f16", (4, 2, False, 3)),
    ("linear_w8a8", 2, 19456, 1024, "f16", (4, 2, False, 4)), ("linear_w8a8", 2, 19456, 2560, "f16", (8, 1, False, 2)),
    ("linear_w8a8", 3, 60000, 1024, "bf16", (4, 2, False, 4)), ("linear_w8a8", 3, 60000, 1024, "f32", (8, 1, False, 2)),
    ("linear_w8a8", 1, 12288, 1024, "f16", (4, 2, False, 4)), ("linear_w8a8", 1, 12288, 2688, "f16", (4, 1, False, 4)),
    ("linear_w8a8", 1, 12288, 1024, "f32", (4, 1, False, 4)), ("linear_w8a8", 1, 5120, 1024, "f16", (8, 2, False, 4)),
    ("linear_w8a8", 1, 7000, 1024, "f16", (4, 2, False, 4)), ("linear_w8a8", 1, 7000, 5248, "f32", (8, 1, True, 4)),
    ("linear_w8a8", 1, 14000, 5248, "f32", (4, 2, False, 4)), ("linear_w8a8", 4, 25661, 5888, "f16", (4, 2, False, 8)),
    ("linear_w8a8", 7, 36840, 3072, "f16", (2, 5, True, 8)), ("linear_w8a8_token", 7, 25661, 3072, "f16", (2, 5, True, 8)),
    ("linear_w8a8_token", 2, 40000, 1024, "f16", (4, 2, False, 4)), ("linear_w8a8_token", 1, 12288, 2688, "f16", (4, 2, False, 4)),
    ("linear_w8a8_token", 1, 40000, 1024, "bf16", (8, 1, False, 2)), ("linear_w8a8_token", 2, 40000, 1024, "f32", (8, 1, False, 2)),
]


def test_decode_picks_around_their_lines(dispatch):
    for (op, M, N, K, x, want) in PICKS:
        rc, names, dims = dispatch([{"op": op, "M": M, "N": N, "K": K, "x": x, "ws": "full"}])[0]
        assert rc == 0 and kernels(names) == ["gemv_fast_kernel"], (op, M, N, K, x, names)
        _, D, G, xl, *_ = [v.strip() for v in names[0].split("<")[1].split(">")[0].split(",")]
        assert (int(D), int(G), xl == "true", dims[0][1] // 64) == want, (op, M, N, K, x, names, dims)


def test_short_per_token_rows_are_quantized_first(dispatch):
    """Up to four K tiles, beyond a dozen tiles of x: the row quantizer's launch."""
    for M, Kc, first in ((3, 4, "gemv_fast_kernel"), (4, 4, "quantize_rows_sym_kernel"), (12, 1, "gemv_fast_kernel"),
                         (13, 1, "quantize_rows_sym_kernel"), (16, 4, "quantize_rows_sym_kernel"), (3, 5, "gemv_fast_kernel")):
        for x in ("f32", "f16"):
            rc, names, _ = dispatch([{"op": "linear_w8a8_token", "M": M, "N": 4096, "K": 64 * Kc, "x": x, "ws": "full"}])[0]
            assert rc == 0 and kernels(names)[0] == first and kernels(names)[-1] == "gemv_fast_kernel", (M, Kc, x, names)


def test_repack_spreads_few_long_rows(dispatch):
    """A repack of few row tiles takes a workgroup of 8 waves for about every 8
    tiles of K (16 rows of 65536 were one workgroup's serial walk); sums
    along K start from a launch that clears them where K is split."""
    calls = [{"op": "repack_w8", "N": N, "K": K, "colsum": cs} for cs in (False, True)
             for N in (1, 16, 17, 64, 300, 1000, 4096, 9728) for K in (1, 64, 600, 4096, 4097, 12288, 65536)]
    for c, (rc, names, grids) in zip(calls, dispatch(calls, axes=3)):
        tiles, per = -(-c["N"] // 16), -(-(-(-c["K"] // 64)) // 8)
        split = grids[-1][0] // tiles
        assert rc == 0 and kernels(names)[-1] == "pack_weight_kernel" and grids[-1][0] % tiles == 0, (c, names)
        assert kernels(names)[:-1] == (["zero_ints_kernel"] if c["colsum"] and split > 1 else []), (c, names)
        if not c["colsum"] or per > 8:
            assert split == 1 if tiles >= 256 else split == min(per, -(-512 // tiles)), (c, grids)


def test_quantize_few_rows_takes_a_wave_each(dispatch):
    """Few short rows of 2-byte values, or at odd 2-byte addresses, quantized
    alone: four rows per workgroup; else sixteen."""
    calls = [{"op": "quantize_per_channel", "N": N, "K": K, "x": x} for x in ("f32", "f16", "bf16")
             for N in (1, 16, 999, 2048, 2049) for K in (1, 64, 1000, 1001, 1024, 1026, 2001, 2500)]
    for c, (rc, names, grids) in zip(calls, dispatch(calls)):
        few = c["x"] != "f32" and c["N"] <= 2048 and (c["K"] <= 1024 or c["K"] % 2)
        assert rc == 0 and kernels(names) == ["quantize_few_rows_kernel" if few else "pack_weight_kernel"], (c, names)
        assert grids[0][0] == -(-c["N"] // (4 if few else 16)), (c, grids)


def test_row_argmax_below_8192_values_is_one_launch(dispatch):
    """Three launches cost the host more than one row of fewer values gains."""
    calls = [{"op": "argmax_rows", "M": M, "N": N} for M in (1, 8, 128, 129) for N in (1, 4096, 4097, 8191, 8192, 151936)]
    for c, (rc, names, _) in zip(calls, dispatch(calls)):
        want = 3 if c["N"] >= 8192 and c["M"] <= 128 else 1
        assert rc == 0 and len(names) == want and all("argmax" in n for n in names), (c, names)
