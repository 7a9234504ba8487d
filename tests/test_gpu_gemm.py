"""GPU parity of the multi-token matmuls (prompt prefill) against the oracle.

The reference computes a prompt token by token; the oracle's matmul_batch is
the same M independent matmuls. Bars: fp32 outputs max|Δ|/max|ref| <= 1e-5;
crafted inputs whose outputs are exact integers pin the int8 matrix-core sums
(Q4_K) and the fp16 hi/lo path (Q6_K) bit for bit.
"""
import numpy as np
import pytest

from hako_amd import synth
from helpers import maxabs_rel

pytestmark = pytest.mark.gpu

TOL = 1e-5
Q4, Q6 = synth.TYPE_Q4_K, synth.TYPE_Q6_K
HAKO_TUNE_Q6K_GEMM_TN = 13   # include/hako_gpu.h
HAKO_TUNE_Q6K_GEMM_SK = 15
HAKO_TUNE_Q6K_GEMM_TM = 20


def run_batch(gpu, qtype, w, x, n_out, n_in, bias=None):
    m = x.shape[0]
    dw, dx, dy = gpu.upload(w), gpu.upload(x), gpu.alloc(m * n_out * 4)
    db = gpu.upload(bias) if bias is not None else None
    gpu.matmul_batch(dy, dx, qtype, dw, db, m, n_out, n_in)
    y = gpu.download(dy, np.float32, (m, n_out))
    for b in (dw, dx, dy, db):
        if b is not None:
            b.free()
    return y


def run_q4k_gemm(gpu, w, xq, xs, n_out, n_in):
    m = xq.shape[0]
    dw, dq, ds, dy = gpu.upload(w), gpu.upload(xq), gpu.upload(xs), gpu.alloc(m * n_out * 4)
    gpu.q4k_gemm(dy, dw, dq, ds, None, m, n_out, n_in)
    y = gpu.download(dy, np.float32, (m, n_out))
    for b in (dw, dq, ds, dy):
        b.free()
    return y


GEMM_SHAPES = [(64, 64, 256), (130, 200, 2048), (17, 100, 3584), (64, 512, 3584), (200, 37, 1280),
               (96, 300, 11008),
               # up to 16 tokens: the skinny kernels (batched decode)
               (2, 64, 256), (5, 100, 2048), (16, 512, 3584), (16, 1000, 1280), (1 + 15, 37, 2048), (3, 18944, 3584),
               # one split per 64-row tile, two passes of the weight prefetch ring
               (16, 32832, 2048)]


@pytest.mark.parametrize("m,n_out,n_in", GEMM_SHAPES)
def test_q4k_batch_vs_oracle(gpu, oracle, m, n_out, n_in):
    rng = np.random.default_rng(m * 1000 + n_out + n_in)
    w = synth.q4k_weight(rng, n_out, n_in)
    x = rng.standard_normal((m, n_in)).astype(np.float32)
    bias = 0.1 * rng.standard_normal(n_out).astype(np.float32)
    got = run_batch(gpu, Q4, w, x, n_out, n_in, bias)
    want = oracle.matmul(Q4, w, x, n_out, n_in, bias=bias, f64=True)
    assert maxabs_rel(got, want) < TOL


@pytest.mark.parametrize("m,n_out,n_in", GEMM_SHAPES + [(70, 100, 18944), (16, 100, 18944), (7, 3584, 11008)])
def test_q6k_batch_vs_oracle(gpu, oracle, m, n_out, n_in):
    rng = np.random.default_rng(m * 1001 + n_out + n_in)
    w = synth.q6k_weight(rng, n_out, n_in)
    x = rng.standard_normal((m, n_in)).astype(np.float32)
    bias = 0.1 * rng.standard_normal(n_out).astype(np.float32)
    got = run_batch(gpu, Q6, w, x, n_out, n_in, bias)
    want = oracle.matmul(Q6, w, x, n_out, n_in, bias=bias, f64=True)
    assert maxabs_rel(got, want) < TOL


def test_q6k_batch_token_rows_of_any_magnitude(gpu, oracle):
    """Each token row is scaled by its own power of two: rows of 1e-30, 1e4
    and subnormal-only values stay within tolerance of their own outputs."""
    rng = np.random.default_rng(5)
    n_out, n_in = 128, 2048
    w = synth.q6k_weight(rng, n_out, n_in)
    x = rng.standard_normal((6, n_in)).astype(np.float32)
    x[1] *= 1e-30
    x[2] *= 1e4
    x[3] = np.float32(1e-42) * np.sign(x[3])   # subnormal
    x[4] = 0.0
    x[5, ::7] *= 1e3                           # wide range within a row
    got = run_batch(gpu, Q6, w, x, n_out, n_in)
    want = oracle.matmul(Q6, w, x, n_out, n_in, f64=True)
    for t in range(6):
        ref = np.max(np.abs(want[t]))
        if ref == 0:
            assert np.all(got[t] == 0)
        else:
            assert np.max(np.abs(got[t] - want[t])) / ref < TOL, t


def _one_hot_scales(n_blocks, sb, which):
    """12 scale bytes giving (s, m) = (1, 0) (which='s') or (0, 1) (which='m')
    for sub-block sb and (0, 0) elsewhere (packing of reference quant.c:57-66)."""
    sc = np.zeros(12, np.uint8)
    if sb < 4:
        sc[sb if which == "s" else sb + 4] = 1
    else:
        sc[sb + 4] = 1 if which == "s" else 0x10
    return np.tile(sc, (n_blocks, 1))


@pytest.mark.parametrize("m", [80, 16, 5])
@pytest.mark.parametrize("sb", [0, 3, 4, 7])
@pytest.mark.parametrize("which", ["s", "m"])
def test_q4k_gemm_integer_sums_exact(gpu, oracle, m, sb, which):
    """d = 1, dmin = 1, one (s, m) = (1, 0) or (0, 1) per block and xs = 1:
    each output is Σ over blocks of the sub-block's iqx (or −ix), an integer
    the fp32 fold represents exactly — bit-exact against the oracle's sums."""
    rng = np.random.default_rng(sb * 3 + (which == "m") + m)
    n_out, n_in = 96, 3584
    nb = n_in // 256
    w = synth.q4k_weight(rng, n_out, n_in).reshape(n_out * nb, 144).copy()
    w[:, 0:2] = np.frombuffer(np.float16(1.0).tobytes(), np.uint8)
    w[:, 2:4] = np.frombuffer(np.float16(1.0).tobytes(), np.uint8)
    w[:, 4:16] = _one_hot_scales(n_out * nb, sb, which)
    w = w.reshape(n_out, nb * 144)
    xq = rng.integers(-127, 128, (m, n_in)).astype(np.int8)
    xs = np.ones((m, n_in // 32), np.float32)
    got = run_q4k_gemm(gpu, w, xq, xs, n_out, n_in)
    want = np.empty((m, n_out), np.float64)
    for t in range(m):
        iqx, ix = oracle.q4k_isums(w, xq[t], n_out, n_in)
        sel = iqx if which == "s" else -ix
        want[t] = sel[:, sb::8].sum(axis=1)
    assert np.array_equal(got, want.astype(np.float32))


@pytest.mark.parametrize("m", [70, 16, 3])
def test_q6k_gemm_exact_integers(gpu, oracle, m):
    """Small-integer activations (exact in fp16, lo = 0) and d = 1: outputs are
    integers the fp32 accumulation holds exactly — bit-exact against the
    oracle's double-precision result."""
    rng = np.random.default_rng(9 + m)
    n_out, n_in = 90, 2048
    nb = n_in // 256
    w = synth.q6k_weight(rng, n_out, n_in).reshape(n_out * nb, 210).copy()
    w[:, 208:210] = np.frombuffer(np.float16(1.0).tobytes(), np.uint8)
    w = w.reshape(n_out, nb * 210)
    x = rng.integers(-8, 9, (m, n_in)).astype(np.float32)
    got = run_batch(gpu, Q6, w, x, n_out, n_in)
    want = oracle.matmul(Q6, w, x, n_out, n_in, f64=True)
    assert np.array_equal(got, want)


def test_q4k_gemm_full_7b_shape_sampled_rows(gpu, oracle):
    """The 7B ffn_up prefill shape (512 tokens x 18944 x 3584); rows sampled
    for the oracle, plus batch == per-token GEMV consistency on all of it."""
    rng = np.random.default_rng(77)
    m, n_out, n_in = 512, 18944, 3584
    w = synth.q4k_weight(rng, n_out, n_in)
    x = rng.standard_normal((m, n_in)).astype(np.float32)
    got = run_batch(gpu, Q4, w, x, n_out, n_in)
    rows = np.unique(np.concatenate([np.arange(64), rng.integers(0, n_out, 128), [n_out - 1]]))
    want = oracle.matmul(Q4, w[rows], x, rows.size, n_in, f64=True)
    assert maxabs_rel(got[:, rows], want) < TOL
    # every token against the single-token GEMV of the same weights
    dw, dx, do = gpu.upload(w), gpu.upload(x[[0, 255, 511]]), gpu.alloc(n_out * 4)
    for i, t in enumerate((0, 255, 511)):
        gpu.matmul(do, dx.offset(i * n_in * 4), Q4, dw, None, n_out, n_in)
        assert maxabs_rel(got[t], gpu.download(do, np.float32, (n_out,))) < TOL
    for b in (dw, dx, do):
        b.free()


@pytest.mark.parametrize("m,n_out,n_in", [(64, 128, 256), (130, 200, 2048), (77, 3648, 1024), (512, 384, 4608),
                                         (17, 65, 768), (500, 3001, 512), (130, 9000, 768)])
def test_q6k_gemm_tile_widths_agree_bit_exact(gpu, oracle, m, n_out, n_in):
    """The 64-row and the 128-row (double-buffered) tiles and the 256-row tiles
    of 64 and 128 tokens do the same arithmetic per output in the same order
    while K is not split, so their outputs are bit-identical, ragged token and
    row edges included, and so is whichever of them the shape is given by
    itself (64 and 128 rows here); within the bar of the oracle."""
    rng = np.random.default_rng(m + n_out + n_in)
    w = synth.q6k_weight(rng, n_out, n_in)
    x = rng.standard_normal((m, n_in)).astype(np.float32)
    bias = 0.1 * rng.standard_normal(n_out).astype(np.float32)
    got = {}
    gpu.tune(HAKO_TUNE_Q6K_GEMM_SK, 0)
    try:
        for tn, tm in ((64, 0), (128, 0), (0, 64), (0, 128), (0, 0)):
            gpu.tune(HAKO_TUNE_Q6K_GEMM_TN, tn)
            gpu.tune(HAKO_TUNE_Q6K_GEMM_TM, tm)
            got[tn, tm] = run_batch(gpu, Q6, w, x, n_out, n_in, bias)
    finally:
        gpu.tune(HAKO_TUNE_Q6K_GEMM_TN, 0)
        gpu.tune(HAKO_TUNE_Q6K_GEMM_TM, 0)
        gpu.tune(HAKO_TUNE_Q6K_GEMM_SK, 2)
    for form, y in got.items():
        assert np.array_equal(y.view(np.uint32), got[64, 0].view(np.uint32)), form
    want = oracle.matmul(Q6, w, x, n_out, n_in, bias=bias, f64=True)
    assert maxabs_rel(got[128, 0], want) < TOL


@pytest.mark.parametrize("tm", [64, 128])
@pytest.mark.parametrize("m,n_out,n_in", [(130, 200, 2048), (77, 3648, 1024), (512, 384, 4608), (64, 128, 512),
                                         (512, 3584, 4608)])
def test_q6k_gemm_split_k(gpu, oracle, m, n_out, n_in, tm):
    """256-row tiles whose K is split over workgroups (a tile's ranges of its
    super-blocks meet in a second launch, in order of K) against the same
    tiles whole: within 1e-6, and the GEMM bar of the oracle. The shapes give
    tiles of one to many workgroups, ranges of one super-block and of unequal
    length, ragged token and row edges; twice in a row, the second call on
    other inputs, so no stale sum passes. With the knob at 1 only the decoder
    splits."""
    rng = np.random.default_rng(3 * m + n_out + n_in)
    w = synth.q6k_weight(rng, n_out, n_in)
    bias = 0.1 * rng.standard_normal(n_out).astype(np.float32)
    gpu.tune(HAKO_TUNE_Q6K_GEMM_TM, tm)
    try:
        for call in range(2):
            x = rng.standard_normal((m, n_in)).astype(np.float32) * (1.0 + 9.0 * call)
            got = {}
            for sk in (0, 1, 2):
                gpu.tune(HAKO_TUNE_Q6K_GEMM_SK, sk)
                got[sk] = run_batch(gpu, Q6, w, x, n_out, n_in, bias)
            assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
            assert maxabs_rel(got[2], got[0]) < 1e-6
            want = oracle.matmul(Q6, w, x, n_out, n_in, bias=bias, f64=True)
            assert maxabs_rel(got[2], want) < TOL
    finally:
        gpu.tune(HAKO_TUNE_Q6K_GEMM_TM, 0)
        gpu.tune(HAKO_TUNE_Q6K_GEMM_SK, 2)


@pytest.mark.parametrize("m,n_out,n_in", [(17, 1, 512), (32, 33, 768), (33, 65, 2048), (77, 2048, 2048),
                                         (77, 4608, 1280), (200, 3000, 3584), (512, 2048, 3840), (512, 2048, 2048),
                                         (64, 512, 3584), (200, 2048, 3584)])
def test_q4k_gemm_shared_units(gpu, oracle, m, n_out, n_in):
    """Few 32-row units per workgroup, so that several waves share one: 2, 3, 8,
    8, 5, 4, 3, 1 (the first shape past the rule), 12 and 6 of them, some with
    fewer super-blocks than waves. Integer inputs with one
    (s, m) = (1, 0) per block and unit scales: every output is exact in
    fp32 whatever the order of the sums."""
    rng = np.random.default_rng(m + n_out + n_in)
    nb = n_in // 256
    w = synth.q4k_weight(rng, n_out, n_in).reshape(n_out * nb, 144).copy()
    w[:, 0:4] = np.frombuffer(np.float16([1.0, 1.0]).tobytes(), np.uint8)
    w[:, 4:16] = _one_hot_scales(n_out * nb, 5, "s")
    w = w.reshape(n_out, nb * 144)
    xq = rng.integers(-127, 128, (m, n_in)).astype(np.int8)
    got = run_q4k_gemm(gpu, w, xq, np.ones((m, n_in // 32), np.float32), n_out, n_in)
    q = (w.reshape(n_out, nb, 144)[:, :, 16 + 64:16 + 96] >> 4).astype(np.float64)   # sub-block 5: high nibbles
    want = xq.reshape(m, nb, 8, 32)[:, :, 5].reshape(m, -1).astype(np.float64) @ q.reshape(n_out, -1).T
    assert np.array_equal(got, want.astype(np.float32))
    if m * n_out * n_in < 1 << 29:   # and random inputs against the oracle
        w = synth.q4k_weight(rng, n_out, n_in)
        x = rng.standard_normal((m, n_in)).astype(np.float32)
        bias = 0.1 * rng.standard_normal(n_out).astype(np.float32)
        got = run_batch(gpu, Q4, w, x, n_out, n_in, bias)
        assert maxabs_rel(got, oracle.matmul(Q4, w, x, n_out, n_in, bias=bias, f64=True)) < TOL


@pytest.mark.parametrize("m,n_out,n_in", [(17, 1, 256), (33, 257, 512), (64, 255, 1024), (65, 256, 1280),
                                         (128, 520, 4096), (129, 300, 4352), (161, 513, 2816)])
def test_q6k_gemm_wide_tile_edges(gpu, oracle, m, n_out, n_in):
    """256-row tiles at the edges of their token tiles (32, 64, 128), rows, and
    the activation layouts (rows of up to 1024, 4096 and more values), K whole
    and split, with rows of very different magnitude. Per output, hi + lo is
    within 2^-22 of a row's largest activation and the sums are fp32: within
    the bar of the other GEMM tests."""
    rng = np.random.default_rng(m + n_out + n_in)
    w = synth.q6k_weight(rng, n_out, n_in)
    x = rng.standard_normal((m, n_in)).astype(np.float32) * np.exp2(rng.integers(-20, 20, (m, 1))).astype(np.float32)
    bias = 0.1 * rng.standard_normal(n_out).astype(np.float32)
    want = oracle.matmul(Q6, w, x, n_out, n_in, bias=bias, f64=True)
    scale = np.max(np.abs(want), axis=1, keepdims=True)
    try:
        for tm in (64, 128):
            gpu.tune(HAKO_TUNE_Q6K_GEMM_TM, tm)
            for sk in (0, 2):
                gpu.tune(HAKO_TUNE_Q6K_GEMM_SK, sk)
                got = run_batch(gpu, Q6, w, x, n_out, n_in, bias)
                assert np.max(np.abs(got - want) / scale) < TOL
    finally:
        gpu.tune(HAKO_TUNE_Q6K_GEMM_TM, 0)
        gpu.tune(HAKO_TUNE_Q6K_GEMM_SK, 2)


def test_q6k_gemm_rows_past_16m_values(gpu, oracle):
    """Rows of more than 65536 super-blocks, whose packed token tile passes 2 GB:
    activations are zero but in 64 blocks, the first and the last among them, so
    the oracle needs these only."""
    rng = np.random.default_rng(16)
    m, n_out, nb = 32, 3, 65536 + 2
    at = np.unique(np.concatenate([[0, 32767, 32768, 65535, 65536, nb - 1], rng.integers(0, nb, 58)]))
    part = synth.q6k_weight(rng, n_out, 256 * at.size).reshape(n_out, at.size, 210)
    w = np.zeros((n_out, nb, 210), np.uint8)
    w[:, at] = part
    xs = rng.standard_normal((m, at.size, 256)).astype(np.float32)
    x = np.zeros((m, nb, 256), np.float32)
    x[:, at] = xs
    got = run_batch(gpu, Q6, w.reshape(n_out, -1), x.reshape(m, -1), n_out, 256 * nb)
    want = oracle.matmul(Q6, part.reshape(n_out, -1), xs.reshape(m, -1), n_out, 256 * at.size, f64=True)
    assert maxabs_rel(got, want) < TOL


def test_q6k_gemm_full_7b_shape_sampled_rows(gpu, oracle):
    rng = np.random.default_rng(78)
    m, n_out, n_in = 512, 3584, 18944
    w = synth.q6k_weight(rng, n_out, n_in)
    x = rng.standard_normal((m, n_in)).astype(np.float32)
    got = run_batch(gpu, Q6, w, x, n_out, n_in)
    rows = np.unique(np.concatenate([np.arange(32), rng.integers(0, n_out, 64), [n_out - 1]]))
    want = oracle.matmul(Q6, w[rows], x, rows.size, n_in, f64=True)
    assert maxabs_rel(got[:, rows], want) < TOL


def test_gemm_bad_shapes_are_rejected(gpu):
    from hako_amd.gpu import HakoGpuError
    dw, dx, dy = gpu.alloc(1 << 16), gpu.alloc(1 << 16), gpu.alloc(1 << 16)
    with pytest.raises(HakoGpuError, match="256"):
        gpu.matmul_batch(dy, dx, Q4, dw, None, 4, 4, 100)
    with pytest.raises(HakoGpuError, match="256"):
        gpu.matmul_batch(dy, dx, Q6, dw, None, 4, 4, 300)
    with pytest.raises(HakoGpuError, match="m > 0"):
        gpu.matmul_batch(dy, dx, Q6, dw, None, 0, 4, 256)
    for b in (dw, dx, dy):
        b.free()


_CAPTURED = """
import sys
import numpy as np
sys.path.insert(0, sys.argv[1])
from hako_amd import synth
from hako_amd.gpu import Gpu
gpu, rng = Gpu(0), np.random.default_rng(4)
wm, wk, m, n_out, n_in = int(sys.argv[2]), int(sys.argv[3]), 32, 256, 4096

def operands(m, n_out, n_in):
    x = rng.standard_normal((m, n_in)).astype(np.float32)
    return gpu.alloc(4 * m * n_out), gpu.upload(x), synth.TYPE_Q6_K, gpu.upload(synth.q6k_weight(rng, n_out, n_in)), None, m, n_out, n_in

first, call = operands(wm, 64, wk), operands(m, n_out, n_in)
gpu.matmul_batch(*first)
gpu.sync()
gpu.capture_begin()
gpu.matmul_batch(*call)
graph = gpu.capture_end()
eager = gpu.alloc(4 * m * n_out)
for _ in range(3):
    gpu.h2d(call[0], np.zeros((m, n_out), np.float32))
    gpu.graph_launch(graph)
    got = gpu.download(call[0], np.float32, (m, n_out))
    gpu.matmul_batch(eager, *call[1:])
    want = gpu.download(eager, np.float32, (m, n_out))
    assert np.any(want) and np.array_equal(got.view(np.uint32), want.view(np.uint32))
    print("replayed", flush=True)
"""


@pytest.mark.parametrize("wm,wk", [(512, 256), (16, 18944)])
def test_q6k_gemm_is_captured_after_another_shape(wm, wk):
    """A Q6_K matmul whose activation fits the workspace of an earlier call can
    be captured, also where it splits K and the earlier call (one super-block;
    16 tokens) did not: the room for the sums is there since the first call. In
    a process of its own, whose workspaces hold nothing else."""
    import os
    import subprocess
    import sys
    repo = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", _CAPTURED, repo, str(wm), str(wk)], capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
