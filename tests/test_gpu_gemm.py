"""GPU parity of the batched prefill GEMM (rows > 1, MFMA path) against the oracle.

X f32 N(0,1) with N = 16 / 64 / 512 token rows, W Q8_0
and Q4_0 at 4096x4096 and 11008x4096 (N(0,0.02), reference quantiser); Q4_1
and ragged shapes in addition.  Bound: tests/tolerance.py (BASELINE and the
reference's own criterion)."""

import os
import sys

import numpy as np
import pytest

import oracle
from tolerance import check_close

pytestmark = pytest.mark.gpu

FMTS = {"q8_0": oracle.Q8_0, "q4_0": oracle.Q4_0, "q4_1": oracle.Q4_1}
THREADS = min(16, os.cpu_count() or 1)


def run(hip, orc, qt, m, k, n, seed=0, scale_rows=None):
    rng = np.random.default_rng(500 + m + k + n + seed)
    w = (rng.standard_normal((m, k), dtype=np.float32) * np.float32(0.02)).astype(np.float32)
    x = rng.standard_normal((n, k), dtype=np.float32)
    if scale_rows is not None:
        x *= np.asarray(scale_rows, np.float32)[:, None]
    blocks = orc.quantize(qt, w, threads=THREADS)
    want = orc.linear(qt, x, blocks, m, threads=THREADS)
    name = hip.kernel_name(qt, n, m, k)
    print(f"gemm qt={qt} M={m} K={k} N={n} kernel={name}", flush=True)
    wt = hip.Weight.upload(qt, blocks, m, k)
    got = wt.linear_host(x)
    wt.free()
    return name, check_close(got, want, x, qt, blocks, f"gemm qt={qt} {m}x{k} N={n}")


@pytest.mark.parametrize("n", [16, 64, 512])
@pytest.mark.parametrize("shape", [(4096, 4096), (11008, 4096)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_gemm_baseline_config4(hip, orc, shape, n):
    for fmt in ("q8_0", "q4_0"):
        name, _ = run(hip, orc, FMTS[fmt], *shape, n)
        assert name.startswith("gemm_mfma"), name


@pytest.mark.parametrize("shape", [(4096, 4096), (4096, 11008)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_gemm_256_tokens_two_splits(hip, orc, shape):
    """256 token rows: two K splits of the large-tile kernel and their reduction."""
    for fmt, qt in FMTS.items():
        name, _ = run(hip, orc, qt, *shape, 256)
        assert "splitk2" in name, name


@pytest.mark.parametrize("m,k,n", [(4096, 4096, 16), (64, 64, 2), (33, 4096, 17), (300, 896, 40),
                                   (4864, 896, 7), (17, 64, 100), (1000, 11008, 3), (520, 4096, 130),
                                   (300, 896, 200), (200, 4096, 96),
                                   # either side of 128 token rows (the workspace rule changes there)
                                   (300, 4096, 128), (300, 4096, 129),
                                   # 130 blocks per row: not a whole number of 4-block chunks
                                   (300, 4160, 40), (300, 4160, 200)])
def test_gemm_q4_1_and_ragged(hip, orc, m, k, n):
    for fmt, qt in FMTS.items():
        run(hip, orc, qt, m, k, n)


@pytest.mark.parametrize("m,k,n", [(4097, 1664, 333),   # 13 steps (an odd count), one row and 13 tokens past a tile
                                   (3999, 2048, 257),   # short last row tile, one token past a tile
                                   (4097, 4096, 129),   # two K splits
                                   (11009, 4096, 65),   # below the chunk kernel's old limit of 128 tokens
                                   (4095, 11008, 64)])  # 86 steps over eight uneven K splits
def test_gemm_large_tile_edges(hip, orc, m, k, n):
    """The large-tile kernel at the edges of its tile (128 rows x 64 tokens), of its
    steps (128 k) and of its K split."""
    for fmt, qt in FMTS.items():
        name, _ = run(hip, orc, qt, m, k, n)
        assert "_tile_" in name, name


@pytest.mark.parametrize("m,k,n", [(1, 256, 129), (257, 11008, 256), (2048, 2048, 192), (129, 1024, 1030)])
def test_gemm_chunk_above_128_tokens(hip, orc, m, k, n):
    """Small products above 128 token rows: the chunk kernel, x split in it."""
    for fmt, qt in FMTS.items():
        name, _ = run(hip, orc, qt, m, k, n)
        assert "_chunk_" in name, name


def test_gemm_large_tile_needs_dword_weights(hip, orc):
    """Weights wrapped two bytes off a dword take the chunk kernel instead."""
    m, k, n = 4097, 1664, 333
    rng = np.random.default_rng(31)
    x = rng.standard_normal((n, k), dtype=np.float32)
    xb, y = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer(4 * n * m)
    for fmt, qt in FMTS.items():
        assert "_tile_" in hip.kernel_name(qt, n, m, k)
        blocks = orc.quantize(qt, rng.standard_normal((m, k), dtype=np.float32) * np.float32(0.02), threads=THREADS)
        buf = hip.DeviceBuffer(blocks.nbytes + 4)
        buf.upload(blocks, 2)
        print(f"gemm qt={qt} weights at +2 bytes", flush=True)

        class At:  # the blocks inside the allocation
            ptr, nbytes = buf.ptr + 2, blocks.nbytes

        wt = hip.Weight.wrap(qt, At, blocks.shape[0], m, k)
        wt.linear_device(xb, y, rows=n)
        want = orc.linear(qt, x, blocks, m, threads=THREADS)
        check_close(y.download(np.float32, n * m).reshape(n, m), want, x, qt, blocks, f"qt={qt} unaligned weights")
        wt.free()
        buf.free()


class Inside:
    """A device buffer's bytes from an offset on, as the binding takes buffers."""

    def __init__(self, hip, a, offset):
        a = np.ascontiguousarray(a)
        self.buf = hip.DeviceBuffer(a.nbytes + offset)
        self.buf.upload(a, offset)
        self.ptr, self.nbytes = self.buf.ptr + offset, a.nbytes


@pytest.mark.parametrize("ms,k,n", [((4097,), 1664, 333), ((300,), 896, 40), ((300,), 896, 2), ((300,), 4160, 40),
                                    ((256, 128, 72), 896, 40), ((4096, 4096, 300), 1664, 333)])
def test_gemm_unaligned_operands(hip, orc, ms, k, n):
    """Weights two bytes off a dword and x four off 16 bytes, each and both, one
    linear or a group: the operands' addresses move no output past the bound."""
    rng = np.random.default_rng(77)
    x = rng.standard_normal((n, k), dtype=np.float32)
    for fmt, qt in FMTS.items():
        blocks = [orc.quantize(qt, rng.standard_normal((m, k), dtype=np.float32) * np.float32(0.02), threads=THREADS)
                  for m in ms]
        want = [orc.linear(qt, x, b, m, threads=THREADS) for b, m in zip(blocks, ms)]
        for wo, xo in ((2, 0), (0, 4), (2, 4)):
            print(f"gemm {fmt} Ms={ms} K={k} N={n} weights at +{wo} x at +{xo}", flush=True)
            xb = Inside(hip, x, xo)
            ws = [hip.Weight.wrap(qt, Inside(hip, b, wo), b.shape[0], m, k) for b, m in zip(blocks, ms)]
            ys = [hip.DeviceBuffer(4 * n * m) for m in ms]
            calls = hip.make_calls([(w, xb, y, n) for w, y in zip(ws, ys)])
            if len(ms) > 1:
                hip.linear_fused(calls)
            else:
                hip.linear_many(calls)
            hip.synchronize(hip.stream(0))
            for y, v, b, m in zip(ys, want, blocks, ms):
                check_close(y.download(np.float32, n * m).reshape(n, m), v, x, qt, b, f"{fmt} M={m} +{wo} +{xo}")


@pytest.mark.parametrize("k", [4092, 4090, 20032, 20476, 20474])
@pytest.mark.parametrize("xo", [0, 4])
def test_gemm_split_rows(hip, orc, k, xo):
    """The x split of rows that are not whole blocks (whole float4s or not), and past
    the 16 384 elements held in registers, from x on 16 bytes or on a float."""
    m, n = 70, 33
    rng = np.random.default_rng(k + xo)
    x = rng.standard_normal((n, k), dtype=np.float32)
    x[:, -3:] *= 50  # a row's maximum among its last elements
    for fmt, qt in FMTS.items():
        blocks = orc.quantize(qt, rng.standard_normal((m, k), dtype=np.float32) * np.float32(0.02), threads=THREADS)
        print(f"gemm {fmt} M={m} K={k} N={n} x at +{xo}", flush=True)
        wt, y = hip.Weight.upload(qt, blocks, m, k), hip.DeviceBuffer(4 * n * m)
        wt.linear_device(Inside(hip, x, xo), y, rows=n)
        hip.synchronize(hip.stream(0))
        want = orc.linear(qt, x, blocks, m, threads=THREADS)
        check_close(y.download(np.float32, n * m).reshape(n, m), want, x, qt, blocks, f"{fmt} K={k} +{xo}")
        wt.free()


def close64(orc, got, x, qt, blocks, m, label):
    """2-norm of the difference to the 64-bit product over the product's.  Every block
    of a row adds one f32 rounding (2^-24, signs at random: the root of their number)
    and the hi / lo halves carry 22 bits of x, so a lost lo half (2^-12) or a sum in
    fewer bits shows where the 1e-3 of the other checks does not see it."""
    k = x.shape[1]
    want = x.astype(np.float64) @ orc.dequantize(qt, blocks, m, k).reshape(m, k).astype(np.float64).T
    err = float(np.linalg.norm(got - want) / np.linalg.norm(want))
    bound = np.sqrt(k / 32) * 2.0 ** -24 + 2.0 ** -22
    print(f"{label}: {err:.2e} of {bound:.2e}", flush=True)
    assert err <= bound, label


@pytest.mark.parametrize("m,k,n,part", [(4097, 1664, 333, "_tile_"), (4097, 4096, 129, "_tile_"), (300, 896, 16, "_chunk_"),
                                        (300, 896, 40, "_chunk_"), (300, 4160, 40, "_bm64_"), (300, 4160, 333, "_bm128_")])
def test_gemm_against_64_bits(hip, orc, m, k, n, part):
    """Each kernel's rounding, in every format."""
    rng = np.random.default_rng(64)
    x = rng.standard_normal((n, k), dtype=np.float32)
    for fmt, qt in FMTS.items():
        name = hip.kernel_name(qt, n, m, k)
        assert part in name, name
        blocks = orc.quantize(qt, rng.standard_normal((m, k), dtype=np.float32) * np.float32(0.02), threads=THREADS)
        wt = hip.Weight.upload(qt, blocks, m, k)
        close64(orc, wt.linear_host(x), x, qt, blocks, m, name)
        wt.free()


@pytest.mark.parametrize("ms,k,n", [((3072, 1000), 4096, 333),       # one split, a short last weight
                                    ((2048, 256, 200), 4096, 333),   # two splits
                                    ((1024, 1024, 72), 11008, 100)])  # seven
def test_gemm_large_tile_group(hip, orc, ms, k, n):
    """Two and three weights in one launch of the large-tile kernel: each row tile's
    weight, output and size, with and without a K split."""
    rng = np.random.default_rng(sum(ms))
    x = rng.standard_normal((n, k), dtype=np.float32)
    xb = hip.DeviceBuffer.from_array(x)
    for fmt, qt in FMTS.items():
        name = hip.kernel_name(qt, n, sum(ms), k)
        assert "_tile_" in name and ("splitk1" in name) == (len(ms) == 2), name
        blocks = [orc.quantize(qt, rng.standard_normal((m, k), dtype=np.float32) * np.float32(0.02), threads=THREADS)
                  for m in ms]
        ws = [hip.Weight.upload(qt, b, m, k) for b, m in zip(blocks, ms)]
        ys = [hip.DeviceBuffer(4 * n * m) for m in ms]
        print(f"gemm group {name} Ms={ms}", flush=True)
        for _ in range(2):  # the second launch finds the counters that the first left
            for y in ys:
                y.fill(0xFF)
            hip.linear_fused(hip.make_calls([(w, xb, y, n) for w, y in zip(ws, ys)]))
            hip.synchronize()
            for y, b, m in zip(ys, blocks, ms):
                close64(orc, y.download(np.float32, n * m).reshape(n, m), x, qt, b, m, f"{fmt} M={m}")


@pytest.mark.parametrize("m,k,n,part", [(4097, 1664, 333, "_tile_"), (300, 896, 40, "_chunk_")])
def test_gemm_nonfinite_x(hip, orc, m, k, n, part):
    """An infinity or a NaN in a token's x makes that token's outputs non-finite, as the
    oracle's, and leaves every other token's bits alone."""
    rng = np.random.default_rng(5)
    x = rng.standard_normal((n, k), dtype=np.float32)
    bad = x.copy()
    bad[3, 5], bad[n - 1, k - 1], bad[n // 2, 64] = np.inf, np.nan, -np.inf
    rows = [3, n // 2, n - 1]
    for fmt, qt in FMTS.items():
        assert part in hip.kernel_name(qt, n, m, k)
        blocks = orc.quantize(qt, rng.standard_normal((m, k), dtype=np.float32) * np.float32(0.02), threads=THREADS)
        print(f"gemm {fmt} M={m} K={k} N={n} with infinities", flush=True)
        wt = hip.Weight.upload(qt, blocks, m, k)
        clean, got = wt.linear_host(x), wt.linear_host(bad)
        wt.free()
        want = orc.linear(qt, bad[rows], blocks, m, threads=THREADS)
        assert not np.isfinite(want).any() and not np.isfinite(got[rows]).any()
        assert np.array_equal(np.delete(got, rows, axis=0), np.delete(clean, rows, axis=0))


# The kernel of each shape: (out, in, rows, name part).
KERNELS = [(4097, 1664, 333, "_tile_"), (300, 896, 40, "_chunk_"), (300, 4160, 40, "_q4_1_bm")]


@pytest.mark.parametrize("m,k,n,part", KERNELS)
def test_gemm_q4_1_offsets_in_f32(hip, m, k, n, part):
    """Q4_1's offset term carries the block sums of x in 32 bits: with scales of 0 and
    one offset of 1 per row, an output is one block's sum, here one 24-bit value."""
    qt, nb = FMTS["q4_1"], k // 32
    assert part in hip.kernel_name(qt, n, m, k)
    rng = np.random.default_rng(8)
    x = np.zeros((n, nb, 32), np.float32)
    sums = (1 + rng.integers(0, 1 << 22, (n, nb)) * 2.0 ** -22 + 2.0 ** -23).astype(np.float32)
    x[:, :, 5] = sums
    at = np.arange(m) % nb
    blocks = rng.integers(0, 256, (m, nb, 20), dtype=np.uint8)
    head = blocks[:, :, :4].copy().view(np.float16)
    head[:] = 0
    head[np.arange(m), at, 1] = 1
    blocks[:, :, :4] = head.view(np.uint8)
    print(f"gemm q4_1 offsets M={m} K={k} N={n}", flush=True)
    wt = hip.Weight.upload(qt, blocks.reshape(m * nb, 20), m, k)
    got = wt.linear_host(x.reshape(n, k))
    wt.free()
    assert np.array_equal(got, sums[:, at])


@pytest.mark.parametrize("m,k,n,part", KERNELS)
def test_gemm_q4_1_infinite_offset(hip, orc, m, k, n, part):
    """An infinite offset gives infinite outputs, not NaN."""
    qt, nb = FMTS["q4_1"], k // 32
    rng = np.random.default_rng(9)
    x = np.abs(rng.standard_normal((n, k), dtype=np.float32)) + np.float32(0.01)
    w = rng.standard_normal((m, k), dtype=np.float32) * np.float32(0.02)
    blocks = orc.quantize(qt, w, threads=THREADS).reshape(m, nb, 20)
    for row, b, v in ((0, 0, np.inf), (7, nb - 1, -np.inf), (m - 1, nb // 2, np.inf)):
        blocks[row, b, 2:4] = np.array([v], np.float16).view(np.uint8)
    blocks = blocks.reshape(m * nb, 20)
    want = orc.linear(qt, x, blocks, m, threads=THREADS)
    assert np.isinf(want[:, [0, 7, m - 1]]).all()
    print(f"gemm q4_1 infinite offset M={m} K={k} N={n}", flush=True)
    wt = hip.Weight.upload(qt, blocks, m, k)
    got = wt.linear_host(x)
    wt.free()
    assert np.array_equal(got[:, [0, 7, m - 1]], want[:, [0, 7, m - 1]])
    assert np.isfinite(np.delete(got, [0, 7, m - 1], axis=1)).all()


def test_gemm_wide_dynamic_range(hip, orc):
    """Per-token power-of-two scaling keeps the hi/lo split exact across token
    magnitudes from 1e-6 to 1e4 (and an all-zero token)."""
    scales = [1e-6, 1.0, 1e4, 0.0, 3.5, 1e-3, 250.0, 1.0]
    for fmt, qt in FMTS.items():
        run(hip, orc, qt, 512, 4096, len(scales), scale_rows=scales)


def test_gemm_odd_block_count_uses_gemv_rows(hip, orc):
    # K=4095 has an even block count (tail 31); K=100 has 4 blocks; K=4064+32 odd count -> GEMV per row
    for m, k, n in [(64, 4095, 5), (64, 100, 3), (48, 4128, 4)]:
        for fmt, qt in FMTS.items():
            run(hip, orc, qt, m, k, n)


def test_graph_replay_after_workspace_growth(hip, orc):
    """A graph recorded with a stream's batched-call workspace keeps working
    after a larger eager call on the same stream grows that workspace (the old
    buffer is retired, not freed): every replay equals the eager result bit
    for bit."""
    qt, m, k = oracle.Q4_0, 4096, 4096
    rng = np.random.default_rng(77)
    w = (rng.standard_normal((m, k), dtype=np.float32) * np.float32(0.02)).astype(np.float32)
    blocks = orc.quantize(qt, w, threads=THREADS)
    wt = hip.Weight.upload(qt, blocks, m, k)
    sp = hip.stream_create(0)  # a stream with no workspace yet
    x16 = hip.DeviceBuffer.from_array(rng.standard_normal((16, k), dtype=np.float32))
    y16 = hip.DeviceBuffer(16 * m * 4)
    x512 = hip.DeviceBuffer.from_array(rng.standard_normal((512, k), dtype=np.float32))
    y512 = hip.DeviceBuffer(512 * m * 4)
    print("gemm workspace growth: eager N=16, record, eager N=512, replays", flush=True)
    wt.linear_device(x16, y16, rows=16, stream=sp)  # creates the stream's workspace (N=16 size)
    hip.synchronize(sp)
    want = y16.download(np.float32)
    g = hip.Graph(hip.make_calls([(wt, x16, y16, 16)]), sp)
    wt.linear_device(x512, y512, rows=512, stream=sp)  # grows the workspace
    hip.synchronize(sp)
    for i in range(3):
        y16.fill(0)
        g.launch(sp)
        hip.synchronize(sp)
        got = y16.download(np.float32)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), f"replay {i} differs"
        wt.linear_device(x512, y512, rows=512, stream=sp)  # eager work between replays
        hip.synchronize(sp)
    g.destroy()
    hip.stream_destroy(sp)
    wt.free()


def _fused_rows(hip, orc, qt, ms, k, n, seed):
    """mlq_hip_quant_linear_fused with `n` token rows over weights of ms rows
    sharing x: every output against the oracle, and the per-call results of
    mlq_hip_quant_linear for comparison."""
    rng = np.random.default_rng(900 + seed)
    x = rng.standard_normal((n, k), dtype=np.float32)
    blocks = [orc.quantize(qt, (rng.standard_normal((m, k), dtype=np.float32) * np.float32(0.02)), threads=THREADS)
              for m in ms]
    ws = [hip.Weight.upload(qt, b, m, k) for b, m in zip(blocks, ms)]
    xb = hip.DeviceBuffer.from_array(x)
    ys = [hip.DeviceBuffer(4 * n * m) for m in ms]
    print(f"fused gemm qt={qt} Ms={ms} K={k} N={n}", flush=True)
    hip.linear_fused(hip.make_calls([(w, xb, y, n) for w, y in zip(ws, ys)]))
    hip.synchronize()
    got = [y.download(np.float32, n * m).reshape(n, m) for y, m in zip(ys, ms)]
    single = [w.linear_host(x) for w in ws]
    for g, b, m in zip(got, blocks, ms):
        check_close(g, orc.linear(qt, x, b, m, threads=THREADS), x, qt, b, f"fused qt={qt} M={m} N={n}")
    for w in ws:
        w.free()
    xb.free()
    for y in ys:
        y.free()
    return got, single


@pytest.mark.parametrize("ms,k,n", [((256, 128, 72), 896, 16), ((256, 128, 72), 896, 40), ((256, 128, 72), 896, 300),
                                    ((128, 256), 4096, 64), ((100, 128, 64), 896, 40), ((64, 64, 64, 64), 896, 20)],
                         ids=["g3_n16", "g3_n40", "g3_n300", "g2_n64", "ragged_first", "four_calls"])
def test_fused_batched_rows(hip, orc, ms, k, n):
    """Batched rows through the fused entry: the grouped GEMM (up to three
    weights, each but the last a whole number of row tiles) or, where the
    shapes do not allow it (a first weight of 100 rows, four calls), one
    launch per call -- every output within the tolerance of the oracle."""
    for fmt, qt in FMTS.items():
        _fused_rows(hip, orc, qt, ms, k, n, seed=len(ms) + n)


def test_fused_batched_qkv_512_rows_bit_identical(hip, orc):
    """q/k/v-shaped group at 512 rows: one K split at both the single-call and
    the group's total M, so the grouped launch must give every row the bits of
    mlq_hip_quant_linear."""
    for fmt in ("q4_0", "q8_0"):
        got, single = _fused_rows(hip, orc, FMTS[fmt], (4096, 4096, 4096), 4096, 512, seed=7)
        for i, (g, s) in enumerate(zip(got, single)):
            assert np.array_equal(g.view(np.uint32), s.view(np.uint32)), f"{fmt} call {i}"
