"""flk_q8_matvec on the GPU against the Q8_0 oracle, bit for bit.

The kernel follows q8_coop.wgsl's summation order (coop(64) in
cpuMatmulQ8F32, kernels/lib.ts:196-278) with one-rounding FMAs, so every
output must equal the oracle's (fused=True) exactly. Shapes cover the Qwen3
projections (q 2048x1024, k/v 1024x1024, o 1024x2048, gate/up 3072x1024,
down 1024x3072, LM head 151936x1024), every lanes-per-row layout (1..64 and
2-4 blocks per lane), the wide fallback (> 8192 columns), batched tokens and
the f16 scale edge cases (subnormal, exponent 31). Batches of 8 or more
tokens go through the tile kernel that reuses each weight block across
tokens; it is held to the same exactness.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

from flock_amd import ops  # noqa: E402


def run_gpu(packed, x, rows, cols, n_tokens=1):
    w = ops.Q8Matrix.from_packed(packed, rows, cols)
    xb = ops.DeviceBuffer.from_array(np.ascontiguousarray(x, np.float32))
    ob = ops.DeviceBuffer(n_tokens * rows * 4)
    ops.q8_matvec(w, xb, ob, n_tokens)
    ops.sync()
    return ob.download(n_tokens * rows)


def problem(rng, rows, cols, n_tokens=1, wscale=0.05):
    packed = oracle.quant_matrix_q8((rng.standard_normal(rows * cols) * wscale).astype(np.float32),
                                    rows, cols)
    x = rng.standard_normal(n_tokens * cols).astype(np.float32)
    return packed, x


@pytest.mark.parametrize("rows,cols", [
    (2048, 1024), (1024, 1024), (1024, 2048), (3072, 1024), (1024, 3072),  # Qwen3 projections
    (4096, 1024),                                   # q, k, v stacked
    (64, 32), (33, 64), (17, 96), (9, 160), (5, 288), (130, 512),  # 1..16 lanes per row
    (70, 4096), (40, 6144), (24, 8192),             # 2, 3, 4 blocks per lane
    (13, 8224),                                     # wide path (257 blocks)
    (1, 1024), (3, 1024),                           # fewer rows than a wave covers
])
def test_matches_oracle_exactly(rng, rows, cols):
    packed, x = problem(rng, rows, cols)
    got = run_gpu(packed, x, rows, cols)
    want = oracle.q8_matvec(packed, x, rows, cols, 64, fused=True)
    assert np.array_equal(got, want), np.flatnonzero(got != want)[:8]
    # The reference's own CPU model (two roundings per fma32) agrees too.
    assert np.array_equal(got, oracle.q8_matvec(packed, x, rows, cols, 64, fused=False))


@pytest.mark.parametrize("n_tokens", [2, 3, 7])
def test_batched_tokens(rng, n_tokens):
    rows, cols = 1024, 1024
    packed, x = problem(rng, rows, cols, n_tokens)
    got = run_gpu(packed, x, rows, cols, n_tokens)
    want = oracle.q8_matvec(packed, x, rows, cols, 64, fused=True)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("rows,cols,n_tokens", [
    (96, 1024, 8), (100, 1024, 13),                 # one chunk; ragged row and token tiles
    (1024, 2048, 9), (33, 1536, 8),                 # two leaves per lane (the second partial)
    (70, 3072, 17), (13, 8224, 8), (24, 8192, 10),  # three and more chunks
    (40, 512, 10), (5, 32, 8), (3, 96, 11),         # fewer blocks than lanes
])
def test_token_tiles_match_oracle(rng, rows, cols, n_tokens):
    """Batches of 8 or more tokens take the weight-reusing tile kernel; its
    sums keep the coop(64) order, so it is exact too."""
    packed, x = problem(rng, rows, cols, n_tokens)
    got = run_gpu(packed, x, rows, cols, n_tokens)
    want = oracle.q8_matvec(packed, x, rows, cols, 64, fused=True)
    assert np.array_equal(got, want), np.flatnonzero(got != want)[:8]


@pytest.mark.parametrize("mode,rows,n", [
    ("plain", 4096, 1024), ("norm", 4096, 1024), ("gate_up", 4096, 1024),  # 8 row tiles
    ("norm", 2050, 256), ("gate_up", 2050, 256),  # 2 row tiles, ragged last group and tile
])
def test_row_streaming_matches_small_batches(rng, mode, rows, n):
    """Large batches stream several row tiles through one staged token tile
    (8 at 1024 tokens x 4096 rows, 2 at 256 x 2050); they must equal the same
    tokens projected 8 at a time (one row tile per workgroup), which the tests
    above hold to the oracle -- and the first tokens are held to it here too."""
    cols = 1024
    packed = random_packed(rng, rows, cols)
    w = ops.Q8Matrix.from_packed(packed, rows, cols)
    x = rng.standard_normal(n * cols).astype(np.float32)
    gain = rng.normal(1, 0.1, cols).astype(np.float32)
    xb = ops.DeviceBuffer.from_array(x)
    gb = ops.DeviceBuffer.from_array(gain)
    n_out = rows // 2 if mode == "gate_up" else rows

    def project(xbuf, ntok, out):
        if mode == "plain":
            ops.q8_matvec(w, xbuf, out, ntok)
        elif mode == "norm":
            ops.q8_matvec_ex(w, xbuf, out, ntok, norm_gain=gb, eps=oracle.QWEN3_EPS)
        else:
            ops.q8_gate_up_swiglu(w, xbuf, out, ntok, norm_gain=gb, eps=oracle.QWEN3_EPS)

    big = ops.DeviceBuffer(n * n_out * 4)
    project(xb, n, big)
    small = ops.DeviceBuffer(8 * n_out * 4)
    xs = ops.DeviceBuffer(8 * cols * 4)
    got = big.download(n * n_out).reshape(n, n_out)
    for t0 in range(0, n, 8):
        xs.upload(x[t0 * cols:(t0 + 8) * cols])
        project(xs, 8, small)
        ops.sync()
        assert np.array_equal(got[t0:t0 + 8], small.download(8 * n_out).reshape(8, n_out)), t0
    xin = x[:8 * cols]
    if mode != "plain":
        xin = oracle.rmsnorm(xin, gain, cols, 8, oracle.QWEN3_EPS)
    want = oracle.q8_matvec(packed, xin, rows, cols, 64, fused=True).reshape(8, rows)
    if mode == "gate_up":  # rows 2i, 2i + 1 are a (gate, up) pair
        want = oracle.swiglu(want[:, 0::2].ravel(), want[:, 1::2].ravel()).reshape(8, n_out)
    assert np.array_equal(got[:8], want)


def test_tile_kernels_equal_per_token_kernel_on_random_shapes():
    """Seeded random shapes and fusions: a batch of >= 8 tokens (tile kernels,
    any row tiling) equals the same tokens projected at most 7 at a time (the
    per-token kernel), bit for bit."""
    rng = np.random.default_rng(2024)
    for case in range(24):
        rows = int(rng.integers(1, 2600))
        cols = 32 * int(rng.integers(1, 130))
        n = int(rng.integers(8, 300))
        fuse = ["plain", "norm", "up", "res", "gate_up"][case % 5]
        if fuse == "gate_up":
            rows += rows % 2
            cols = min(cols, 1024)
        packed = random_packed(rng, rows, cols)
        w = ops.Q8Matrix.from_packed(packed, rows, cols)
        x = rng.standard_normal(n * cols).astype(np.float32)
        aux = rng.standard_normal(n * max(rows, cols)).astype(np.float32)
        gain = ops.DeviceBuffer.from_array(rng.normal(1, 0.1, cols).astype(np.float32))
        n_out = rows // 2 if fuse == "gate_up" else rows

        def run(t0, t1):
            k = t1 - t0
            xb = ops.DeviceBuffer.from_array(x[t0 * cols:t1 * cols])
            ob = ops.DeviceBuffer(k * n_out * 4)
            if fuse == "plain":
                ops.q8_matvec(w, xb, ob, k)
            elif fuse == "norm":
                ops.q8_matvec_ex(w, xb, ob, k, norm_gain=gain, eps=oracle.QWEN3_EPS)
            elif fuse == "up":
                ub = ops.DeviceBuffer.from_array(aux[t0 * cols:t1 * cols])
                ops.q8_matvec_ex(w, xb, ob, k, up=ub)
            elif fuse == "res":
                rb = ops.DeviceBuffer.from_array(aux[t0 * rows:t1 * rows])
                ops.q8_matvec_ex(w, xb, ob, k, res=rb)
            else:
                ops.q8_gate_up_swiglu(w, xb, ob, k, norm_gain=gain, eps=oracle.QWEN3_EPS)
            ops.sync()
            return ob.download(k * n_out)

        big = run(0, n)
        small = np.concatenate([run(t, min(t + 7, n)) for t in range(0, n, 7)])
        assert np.array_equal(big, small), (case, rows, cols, n, fuse)


# Every instance of q8_mfma_kernel: 32 and 64 tokens per tile, the three input
# fusions, one block per leaf of the tree (8, 16, 32 or 64 blocks per row) and the
# general walk; one row in the last row tile wherever the plan allows it.
@pytest.mark.parametrize("rows,cols,n,fuse,tile", [
    (513, 256, 1696, "plain", 32),
    (513, 2080, 1696, "res", 32),     # 65 blocks: one leaf of two
    (704, 1024, 1236, "up", 32),
    (513, 2080, 1696, "up", 32),
    (1473, 1024, 1945, "norm", 32),
    (961, 2080, 1944, "norm", 32),
    (4096, 1024, 1000, "norm", 32),
    (6144, 1024, 500, "gate_up", 32),
    (4100, 96, 700, "plain", 32),     # fewer blocks than the 8 leaves written out
    (1537, 1024, 1068, "res", 64),
    (1537, 96, 1068, "plain", 64),
    (1537, 4224, 1068, "plain", 64),  # leaves of two and of three blocks
    (1537, 1024, 1068, "up", 64),
    (832, 3072, 1973, "up", 64),
    (1024, 3072, 2048, "res", 64),    # a layer's down projection
    (3457, 1024, 2108, "norm", 64),
    (6144, 1024, 2048, "gate_up", 64),
    (2497, 2080, 1457, "norm", 64),
    # And the VALU tiles: few and many row tiles per workgroup, rows past a tile.
    (4097, 256, 601, "up", -8),
    (4096, 1024, 777, "norm", -8),
    (2050, 2080, 1100, "res", -1),
    (1000, 3072, 2100, "norm", -1),
])
def test_matrix_core_tiles_match_small_batches(rng, rows, cols, n, fuse, tile):
    """Batches that fill the GPU with 64-row tiles (q8_mfma_kernel) equal the
    same tokens projected 7 at a time (the per-token kernel), bit for bit."""
    assert ops.lib().flock_q8_batch_tile(rows, cols, n, fuse in ("norm", "gate_up")) == tile
    w = ops.Q8Matrix.from_packed(random_packed(rng, rows, cols), rows, cols)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    x[:, 3] *= 1e-39  # subnormal products
    aux = rng.standard_normal((n, max(rows, cols))).astype(np.float32)
    gain = ops.DeviceBuffer.from_array(rng.normal(1, 0.1, cols).astype(np.float32))
    n_out = rows // 2 if fuse == "gate_up" else rows

    def run(t0, t1):
        k = t1 - t0
        xb = ops.DeviceBuffer.from_array(np.ascontiguousarray(x[t0:t1]))
        ob = ops.DeviceBuffer.from_array(np.full(k * n_out, np.nan, np.float32))
        if fuse == "gate_up":
            ops.q8_gate_up_swiglu(w, xb, ob, k, norm_gain=gain, eps=oracle.QWEN3_EPS)
        else:
            kw = {"norm": dict(norm_gain=gain, eps=oracle.QWEN3_EPS), "plain": {}}.get(fuse)
            if kw is None:
                a = np.ascontiguousarray(aux[t0:t1, :cols if fuse == "up" else rows])
                kw = {fuse: ops.DeviceBuffer.from_array(a)}
            ops.q8_matvec_ex(w, xb, ob, k, **kw)
        ops.sync()
        return ob.download(k * n_out)

    big = run(0, n)
    small = np.concatenate([run(t, min(t + 7, n)) for t in range(0, n, 7)])
    assert np.array_equal(big, small)


def random_packed(rng, rows, cols):
    """Q8_0 bytes with random int8 quants and f16 scales around 4e-4 (what
    quantRowQ8 gives for N(0, 0.05) weights), built without the quantizer."""
    blocks = np.empty((rows * cols // 32, 34), np.uint8)
    sc = (np.abs(rng.standard_normal(blocks.shape[0])) * 4e-4 + 1e-5).astype(np.float16)
    blocks[:, :2] = sc.view(np.uint8).reshape(-1, 2)
    blocks[:, 2:] = rng.integers(0, 256, (blocks.shape[0], 32), dtype=np.uint8)
    return blocks.ravel()


def test_lm_head_shape(rng):
    # Qwen3-0.6B's tied LM head: 151936 x 1024 (165 MB of Q8_0).
    rows, cols = 151936, 1024
    packed = random_packed(rng, rows, cols)
    x = rng.standard_normal(cols).astype(np.float32)
    got = run_gpu(packed, x, rows, cols)
    want = oracle.q8_matvec(packed, x, rows, cols, 64, fused=True)
    assert np.array_equal(got, want)
    assert oracle.argmax(got) == oracle.argmax(want)


def test_scale_edge_cases(rng):
    # Subnormal, tiny normal, largest finite and exponent-31 scales (inf and
    # nan patterns read as +-FLT_MAX); x small so products stay finite.
    rows, cols = 8, 64
    scales = [0x0001, 0x03FF, 0x0400, 0x7BFF, 0x7C00, 0xFC00, 0x7E00, 0x3C00]
    q = rng.integers(-128, 128, (rows, cols))
    parts = []
    for r in range(rows):
        for b in range(cols // 32):
            h = scales[r]
            parts.append(bytes([h & 0xFF, h >> 8]) +
                         bytes((q[r, 32 * b:32 * b + 32] & 0xFF).astype(np.uint8)))
    packed = np.frombuffer(b"".join(parts), np.uint8)
    x = (rng.standard_normal(cols) * 1e-3).astype(np.float32)
    got = run_gpu(packed, x, rows, cols)
    want = oracle.q8_matvec(packed, x, rows, cols, 64, fused=True)
    assert np.array_equal(got, want)


def test_integer_problem_is_exact(rng):
    # Integer quants, unit scales, integer x: the exact product, whatever the order.
    rows, cols = 512, 2048
    q = rng.integers(-128, 128, (rows, cols))
    x = rng.integers(-8, 9, cols).astype(np.float32)
    packed = np.frombuffer(b"".join(
        bytes([0x00, 0x3C]) + bytes((q[r, 32 * b:32 * b + 32] & 0xFF).astype(np.uint8))
        for r in range(rows) for b in range(cols // 32)), np.uint8)
    got = run_gpu(packed, x, rows, cols)
    assert np.array_equal(got, (q @ x.astype(np.int64)).astype(np.float32))


# ---------------------------------------------------------------- argmax / head
def gpu_argmax(x):
    n = x.size
    xb = ops.DeviceBuffer.from_array(np.ascontiguousarray(x, np.float32))
    ov, oi = ops.DeviceBuffer(4), ops.DeviceBuffer(4)
    ws = ops.DeviceBuffer(ops.argmax_ws_bytes(n))
    ops.argmax(xb, n, ov, oi, ws)
    ops.sync()
    return float(ov.download(1)[0]), int(oi.download(1, np.uint32)[0])


@pytest.mark.parametrize("n", [1, 100, 256, 257, 4096, 151936, 1 << 20])
def test_argmax_matches_oracle(rng, n):
    x = rng.standard_normal(n).astype(np.float32)
    assert gpu_argmax(x) == oracle.argmax_wgsl(x)


def test_argmax_ties_nan_and_sentinel(rng):
    n = 151936
    x = rng.standard_normal(n).astype(np.float32)
    top = float(x.max()) + 1.0
    for i in (90000, 1234, 150000, 70001):  # equal maxima in different workgroups
        x[i] = top
    assert gpu_argmax(x) == (top, 1234) == oracle.argmax_wgsl(x)
    x[5] = np.nan
    x[1233] = np.nan
    assert gpu_argmax(x) == oracle.argmax_wgsl(x) == (top, 1234)
    y = np.full(1000, -np.inf, np.float32)
    y[::7] = np.nan
    assert gpu_argmax(y) == oracle.argmax_wgsl(y) == (-np.finfo(np.float32).max, 0xFFFFFFFF)
    y[400] = -np.finfo(np.float32).max
    assert gpu_argmax(y) == oracle.argmax_wgsl(y)


def run_head(x, gain, packed, vocab, hidden, with_logits=True):
    w = ops.Q8Matrix.from_packed(packed, vocab, hidden)
    xb = ops.DeviceBuffer.from_array(x)
    gb = ops.DeviceBuffer.from_array(gain)
    normed = ops.DeviceBuffer(hidden * 4)
    logits = ops.DeviceBuffer(vocab * 4) if with_logits else None
    ov, oi = ops.DeviceBuffer(4), ops.DeviceBuffer(4)
    ws = ops.DeviceBuffer(ops.lm_head_ws_bytes(vocab, hidden))
    ops.lm_head(xb, gb, oracle.QWEN3_EPS, w, normed, logits, ov, oi, ws)
    ops.sync()
    return (normed.download(hidden), logits.download(vocab) if with_logits else None,
            float(ov.download(1)[0]), int(oi.download(1, np.uint32)[0]))


@pytest.mark.parametrize("vocab,hidden", [(151936, 1024), (1000, 64), (5003, 2048), (300, 8224)])
def test_lm_head_matches_oracle(rng, vocab, hidden):
    packed = random_packed(rng, vocab, hidden)
    x = rng.standard_normal(hidden).astype(np.float32)
    gain = rng.normal(1, 0.1, hidden).astype(np.float32)
    normed, logits, v, i = run_head(x, gain, packed, vocab, hidden)
    w_normed, w_logits, w_v, w_i = oracle.lm_head(x, gain, oracle.QWEN3_EPS, packed, vocab, hidden)
    assert np.array_equal(normed, w_normed)
    assert np.array_equal(logits, w_logits)
    assert (v, i) == (w_v, w_i)
    # Without a logits buffer: the same token.
    assert run_head(x, gain, packed, vocab, hidden, with_logits=False)[2:] == (w_v, w_i)


@pytest.mark.parametrize("vocab,hidden", [
    (500, 32), (333, 1024), (100, 2080), (40, 8192),  # short matrices, every row width
    (65535, 64), (65536, 64), (65537, 1024),          # tall: apart, or one norm per workgroup
    (40, 8224),                                       # too wide to hold x: its own norm launch
])
def test_lm_head_with_the_norm_fused_or_apart(rng, vocab, hidden):
    """x and gain at 16-byte boundaries (the projection forms the norm) give the
    bits of unaligned ones and of a norm in place (a launch of its own)."""
    packed = random_packed(rng, vocab, hidden)
    w = ops.Q8Matrix.from_packed(packed, vocab, hidden)
    x = rng.standard_normal(hidden).astype(np.float32)
    gain = rng.normal(1, 0.1, hidden).astype(np.float32)
    ws = ops.DeviceBuffer(ops.lm_head_ws_bytes(vocab, hidden))

    def run(x_off=0, gain_off=0, in_place=False):
        xb, gb = (ops.DeviceBuffer.from_array(np.concatenate([np.zeros(o, np.float32), a]))
                  for o, a in ((x_off, x), (gain_off, gain)))
        normed = xb if in_place else ops.DeviceBuffer.from_array(np.full(hidden, np.nan, np.float32))
        logits = ops.DeviceBuffer.from_array(np.full(vocab, np.nan, np.float32))
        ov, oi = ops.DeviceBuffer(4), ops.DeviceBuffer(4)
        ops.lm_head(xb.ptr + 4 * x_off, gb.ptr + 4 * gain_off, oracle.QWEN3_EPS, w, normed, logits,
                    ov, oi, ws)
        ops.sync()
        return (normed.download(hidden), logits.download(vocab), ov.download(1),
                oi.download(1, np.uint32))

    want = run()
    assert np.array_equal(want[0], oracle.rmsnorm(x, gain, hidden, 1, oracle.QWEN3_EPS))
    for other in (run(x_off=1), run(gain_off=3), run(in_place=True)):
        assert all(np.array_equal(a, b) for a, b in zip(want, other))


@pytest.mark.parametrize("inner", ["x", "gain"])
@pytest.mark.parametrize("vocab,hidden", [(333, 1024), (65537, 1024)])
def test_lm_head_of_inputs_inside_the_workspace(rng, vocab, hidden, inner):
    """Workgroups write argmax partials to ws while others still read x and the
    gain: where those lie inside it, the norm gets a launch of its own."""
    w = ops.Q8Matrix.from_packed(random_packed(rng, vocab, hidden), vocab, hidden)
    x = rng.standard_normal(hidden).astype(np.float32)
    gain = rng.normal(1, 0.1, hidden).astype(np.float32)
    xb, gb = ops.DeviceBuffer.from_array(x), ops.DeviceBuffer.from_array(gain)
    ws = ops.DeviceBuffer(ops.lm_head_ws_bytes(vocab, hidden) + 4 * hidden)

    def run(xp, gp):
        normed, logits = ops.DeviceBuffer(4 * hidden), ops.DeviceBuffer(4 * vocab)
        ov, oi = ops.DeviceBuffer(4), ops.DeviceBuffer(4)
        ops.lm_head(xp, gp, oracle.QWEN3_EPS, w, normed, logits, ov, oi, ws)
        ops.sync()
        return (normed.download(hidden), logits.download(vocab), ov.download(1),
                oi.download(1, np.uint32))

    want = run(xb, gb)
    ws.upload(x if inner == "x" else gain)
    got = run(ws.ptr if inner == "x" else xb, ws.ptr if inner == "gain" else gb)
    assert all(np.array_equal(a, b) for a, b in zip(want, got))


def test_lm_head_tie_picks_lowest_row(rng):
    vocab, hidden = 151936, 1024
    packed = random_packed(rng, vocab, hidden).reshape(vocab, -1)
    x = rng.standard_normal(hidden).astype(np.float32)
    gain = np.ones(hidden, np.float32)
    _, logits, _, m = oracle.lm_head(x, gain, oracle.QWEN3_EPS, packed.ravel(), vocab, hidden)
    for r in (3, m // 2, vocab - 1):  # identical rows give identical logits
        packed[r] = packed[m]
    want = oracle.lm_head(x, gain, oracle.QWEN3_EPS, packed.ravel(), vocab, hidden)
    assert want[3] == min(3, m)
    got = run_head(x, gain, packed.ravel(), vocab, hidden)
    assert got[2:] == want[2:]
