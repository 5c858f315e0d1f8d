"""Batched (skinny) K-quant matvec on the gfx950 f16 matrix cores vs the oracle.

The reference has no batched matvec (its decode loops tokens one by one,
src/vbs_specializer.c:353-357), so the oracle of vbs_gfx950_linear_batch is
`batch` independent vbs_host_linear_tile calls (src/vbs_host_math.h:223-267):
every vector must meet the single matvec's bar, relative L2 <= 1e-5.
"""
import ctypes
import threading

import numpy as np
import pytest

import vbs_gfx950 as V
from test_gpu_kernels import LIN_TOL, SEED, Mem, lin_err, mem, rel_l2, synth_x  # noqa: F401 (mem: fixture)

pytestmark = pytest.mark.gpu

KQ = [V.Q4_K, V.Q6_K]


def run_batch(dev, mem, t, w, X, rows, cols, xs=None, ys=None):
    """Y = W X^T through the C ABI; X rows padded to stride xs, Y rows at
    stride ys pre-filled with -3 (so untouched entries are visible)."""
    batch = X.shape[0]
    xs, ys = xs or cols, ys or rows
    Xp = np.zeros((batch, xs), np.float32)
    Xp[:, :cols] = X
    pw, px = mem.up(w), mem.up(Xp)
    py = mem.up(np.full(batch * ys, -3.0, np.float32))
    dev.linear_batch(t, pw, px, xs, py, ys, cols, rows, batch)
    return dev.download(py, (batch, ys), np.float32)


def vectors(host, batch, cols, stream):
    return np.stack([synth_x(host, cols, stream + b) for b in range(batch)])


@pytest.mark.parametrize("t", KQ, ids=lambda t: V.TYPE_NAMES[t])
@pytest.mark.parametrize("batch", [1, 2, 5, 8, 11, 16])
@pytest.mark.parametrize("rows,cols", [(1, 256), (37, 4352), (700, 8192), (19, 11008),
                                       (96, 28672), (1030, 4096)])
def test_batch_parity(dev, host, oracle, mem, t, batch, rows, cols):
    """Row counts that leave tiles, waves and workgroups partly idle, one to
    eight blocks per wave, one and two launches of eight vectors."""
    w = V.synth_matrix(host, t, rows, cols, SEED, 71)
    X = vectors(host, batch, cols, 80)
    Y = run_batch(dev, mem, t, w, X, rows, cols)
    for b in range(batch):
        assert lin_err(Y[b], oracle.linear(t, w, X[b], cols, rows)) <= LIN_TOL, b


@pytest.mark.parametrize("t", KQ, ids=lambda t: V.TYPE_NAMES[t])
def test_batch_strides(dev, host, oracle, mem, t):
    """x and y strides wider than the row; entries past `rows` untouched."""
    rows, cols, batch = 300, 4096, 6
    w = V.synth_matrix(host, t, rows, cols, SEED, 72)
    X = vectors(host, batch, cols, 90)
    Y = run_batch(dev, mem, t, w, X, rows, cols, xs=cols + 40, ys=rows + 13)
    assert np.all(Y[:, rows:] == -3.0)
    for b in range(batch):
        assert lin_err(Y[b, :rows], oracle.linear(t, w, X[b], cols, rows)) <= LIN_TOL


@pytest.mark.parametrize("t", KQ, ids=lambda t: V.TYPE_NAMES[t])
def test_batch_activation_edge_cases(dev, host, oracle, mem, t):
    """Per-vector scaling: an all-zero vector, a vector of 1e-30 scale, one of
    1e30 scale, outliers, zero and subnormal-scale sub-blocks; every vector
    meets the bar on its own."""
    rows, cols = 128, 4096
    w = V.synth_matrix(host, t, rows, cols, SEED, 73)
    X = vectors(host, 8, cols, 100)
    X[0] = 0.0
    X[1] *= 1e-30
    X[2] *= 1e30
    X[3, 40] = 1.0e4
    X[4, 0:32] = 0.0
    X[4, 64:96] *= 1e-40
    X[5, 96:128] *= 1e30
    X[6, 7] = -0.0
    Y = run_batch(dev, mem, t, w, X, rows, cols)
    assert np.all(Y[0] == 0.0)
    for b in range(1, 8):
        want = oracle.linear(t, w, X[b], cols, rows)
        assert np.all(np.isfinite(Y[b])), b
        assert lin_err(Y[b], want) <= LIN_TOL, b


@pytest.mark.parametrize("t", KQ, ids=lambda t: V.TYPE_NAMES[t])
def test_batch_non_finite_vector(dev, host, oracle, mem, t):
    """A vector holding inf or NaN gives NaN rows (as the batch-1 matrix-core
    kernel does for such a sub-block); the other vectors are unaffected."""
    rows, cols = 64, 4096
    w = V.synth_matrix(host, t, rows, cols, SEED, 74)
    X = vectors(host, 4, cols, 110)
    X[1, 300] = np.inf
    X[2, 5] = np.nan
    Y = run_batch(dev, mem, t, w, X, rows, cols)
    assert np.all(np.isnan(Y[1])) and np.all(np.isnan(Y[2]))
    for b in (0, 3):
        assert lin_err(Y[b], oracle.linear(t, w, X[b], cols, rows)) <= LIN_TOL


@pytest.mark.parametrize("t,rows,cols", [(V.Q4_K, 28672, 8192), (V.Q6_K, 8192, 28672),
                                         (V.Q6_K, 32000, 8192)],
                         ids=["q4k_70b_gate", "q6k_70b_down", "q6k_70b_head"])
def test_batch_70b_shapes(dev, host, oracle, mem, t, rows, cols):
    """The Llama-70B layer shapes at batch 8, the oracle on the first and last
    192 rows (the packed rows are sliced out of the full matrix)."""
    w = V.synth_matrix(host, t, rows, cols, SEED, 75)
    X = vectors(host, 8, cols, 120)
    Y = run_batch(dev, mem, t, w, X, rows, cols)
    k = 192
    for lo in (0, rows - k):
        ws = np.ascontiguousarray(w[lo:lo + k])
        for b in range(8):
            assert lin_err(Y[b, lo:lo + k], oracle.linear(t, ws, X[b], cols, k)) <= LIN_TOL, (lo, b)


@pytest.mark.parametrize("rows,cols", [(4096, 11008), (3000, 8448), (4100, 28672), (5000, 25088)])
@pytest.mark.parametrize("batch", [3, 8, 11])
def test_batch_q6k_ring_shapes(dev, host, oracle, mem, rows, cols, batch):
    """Q6_K rows of 33-48 blocks over 2049-4096 rows and of 97-112 blocks
    over 4097-8192 rows take the batched LDS-DMA ring kernel: whole and short
    row ranges per workgroup, 33-112 blocks, one and two launches of eight
    vectors; every row of every vector against the oracle."""
    w = V.synth_matrix(host, V.Q6_K, rows, cols, SEED, 77)
    X = vectors(host, batch, cols, 130)
    Y = run_batch(dev, mem, V.Q6_K, w, X, rows, cols)
    for b in range(batch):
        assert lin_err(Y[b], oracle.linear(V.Q6_K, w, X[b], cols, rows, threads=16)) <= LIN_TOL, b


@pytest.mark.parametrize("rows", [11008, 22016])
@pytest.mark.parametrize("batch", [5, 8])
def test_batch_7b_gate_shape(dev, host, oracle, mem, batch, rows):
    """Q4_K 11008x4096 and 22016x4096 (the Llama-7B gate, and gate/up as one
    launch): 688 and 1376 tiles of 16-block rows, three tiles per workgroup
    (the last workgroup partly idle), every row against the oracle."""
    cols = 4096
    w = V.synth_matrix(host, V.Q4_K, rows, cols, SEED, 77)
    X = vectors(host, batch, cols, 130)
    Y = run_batch(dev, mem, V.Q4_K, w, X, rows, cols)
    for b in range(batch):
        assert lin_err(Y[b], oracle.linear(V.Q4_K, w, X[b], cols, rows)) <= LIN_TOL, b


def test_batch_ranged_qkv_every_row(dev, host, oracle, mem):
    """The 70B Q/K/V shape at batch 5 takes the ranged plan (an even range of
    42 rows of one matrix per workgroup, 246 workgroups, the last range of
    each matrix shorter): every row of every matrix against the oracle, per
    vector, and entries past each matrix's rows untouched."""
    shapes, cols, batch, pad = [8192, 1024, 1024], 8192, 5, 7
    ws = [V.synth_matrix(host, V.Q4_K, r, cols, SEED, 160 + m) for m, r in enumerate(shapes)]
    X = vectors(host, batch, cols, 170)
    px = mem.up(X)
    pws = [mem.up(w) for w in ws]
    pys = [mem.up(np.full(batch * (r + pad), -3.0, np.float32)) for r in shapes]
    dev.linear_batch_multi(V.Q4_K, pws, shapes, px, cols, pys, [r + pad for r in shapes], cols, batch)
    for m, (w, r) in enumerate(zip(ws, shapes)):
        Y = dev.download(pys[m], (batch, r + pad), np.float32)
        assert np.all(Y[:, r:] == -3.0), m
        for b in range(batch):
            want = oracle.linear(V.Q4_K, w, X[b], cols, r, threads=16)
            assert lin_err(Y[b, :r], want) <= LIN_TOL, (m, b)
            # a row of a wrong range would stand out even inside the L2 norm
            assert np.max(np.abs(Y[b, :r] - want)) <= 1e-4 * (np.max(np.abs(want)) + 1.0), (m, b)


@pytest.mark.parametrize("t,shapes,cols", [
    (V.Q4_K, [8192, 1024, 1024], 8192), (V.Q4_K, [4096, 1024, 1024], 4096),
    (V.Q4_K, [28672, 28672], 8192), (V.Q6_K, [4096, 1000, 13], 4096), (V.Q4_K, [37], 512)],
    ids=["q4k_70b_qkv", "q4k_7b_qkv", "q4k_70b_gate_up", "q6k_ragged", "q4k_one"])
@pytest.mark.parametrize("batch", [5, 8, 11])
def test_batch_multi_matrix_launch(dev, host, oracle, mem, t, shapes, cols, batch):
    """vbs_gfx950_linear_batch_multi: Q/K/V (or gate/up) of one layer over the
    same vectors in one launch. Workgroups of several tiles span the
    boundaries between the matrices (70B Q/K/V: 640 tiles, three per
    workgroup, the last one partly idle). The first and last 64 rows of every
    matrix (so the rows on both sides of each boundary, and the last
    workgroup's) against the oracle, per vector; entries past each matrix's
    rows untouched."""
    ws = [V.synth_matrix(host, t, r, cols, SEED, 140 + m) for m, r in enumerate(shapes)]
    X = vectors(host, batch, cols, 150)
    px = mem.up(X)
    pad = 7
    pws = [mem.up(w) for w in ws]
    pys = [mem.up(np.full(batch * (r + pad), -3.0, np.float32)) for r in shapes]
    dev.linear_batch_multi(t, pws, shapes, px, cols, pys, [r + pad for r in shapes], cols, batch)
    for m, (w, r) in enumerate(zip(ws, shapes)):
        Y = dev.download(pys[m], (batch, r + pad), np.float32)
        assert np.all(Y[:, r:] == -3.0), m
        spans = sorted({(0, min(64, r)), (max(0, r - 64), r)})
        for lo, hi in spans:
            wsl = np.ascontiguousarray(w[lo:hi])
            for b in range(batch):
                want = oracle.linear(t, wsl, X[b], cols, hi - lo)
                assert lin_err(Y[b, lo:hi], want) <= LIN_TOL, (m, lo, b)


BLK = [V.Q4_0, V.Q4_1, V.Q8_0, V.F16]


@pytest.mark.parametrize("t", BLK, ids=lambda t: V.TYPE_NAMES[t])
@pytest.mark.parametrize("shapes,cols,batch", [
    ([1], 2304, 3), ([16], 256, 16), ([17, 33], 96, 9), ([300], 4384, 8), ([3000], 4384, 8), ([4097], 288, 2),
    ([4113, 80, 15], 544, 5), ([8209], 256, 7), ([12301], 320, 11)])
def test_batch_block_types(dev, host, oracle, mem, t, shapes, cols, batch):
    """The matrix-core batched kernel of the 32-element block types and F16:
    one, two and three tiles per workgroup (up to 256, 512 and more tiles),
    launches across matrix boundaries, partial last tiles, workgroups and
    256-element units (rows of 96 to 4384 elements at every 2-byte offset),
    one and two groups of eight vectors, strides wider than the row; every
    row against the oracle, the padding untouched."""
    xs, pad = cols + 4, 3
    ws = [V.synth_matrix(host, t, r, cols, SEED, 180 + m) for m, r in enumerate(shapes)]
    X = vectors(host, batch, cols, 190)
    Xp = np.zeros((batch, xs), np.float32)
    Xp[:, :cols] = X
    pws = [mem.up(w) for w in ws]
    pys = [mem.up(np.full(batch * (r + pad), -3.0, np.float32)) for r in shapes]
    dev.linear_batch_multi(t, pws, shapes, mem.up(Xp), xs, pys, [r + pad for r in shapes], cols, batch)
    for m, (w, r) in enumerate(zip(ws, shapes)):
        Y = dev.download(pys[m], (batch, r + pad), np.float32)
        assert np.all(Y[:, r:] == -3.0), m
        for b in range(batch):
            want = oracle.linear(t, w, X[b], cols, r)
            assert lin_err(Y[b, :r], want) <= LIN_TOL, (m, b)


@pytest.mark.parametrize("t", BLK, ids=lambda t: V.TYPE_NAMES[t])
@pytest.mark.parametrize("rows,cols,batch", [
    (3072, 8192, 2), (3072, 8192, 3), (3073, 3040, 2), (4096, 3072, 4), (3074, 2048, 4), (8209, 1056, 7), (3071, 1056, 8),
    (3072, 544, 5), (24576, 512, 8), (24576, 32, 9), (8192, 64, 9), (1920, 4096, 8), (1919, 4096, 8), (2048, 2048, 16),
    (1024, 8192, 12), (1023, 8192, 16), (1024, 8192, 5)])
def test_batch_block_types_rule(dev, host, oracle, mem, t, rows, cols, batch):
    """One matrix on both sides of each limit between the general kernel and the
    matrix cores, there with one to three tiles per workgroup."""
    w = V.synth_matrix(host, t, rows, cols, SEED, 184)
    X = vectors(host, batch, cols, 195)
    Y = run_batch(dev, mem, t, w, X, rows, cols)
    for b in range(batch):
        assert lin_err(Y[b], oracle.linear(t, w, X[b], cols, rows, threads=8)) <= LIN_TOL, b


@pytest.mark.parametrize("t", BLK, ids=lambda t: V.TYPE_NAMES[t])
@pytest.mark.parametrize("shapes,cols,batch", [
    ([1000, 24], 2080, 4), ([1000, 25], 2080, 4), ([2000, 48], 2048, 3), ([1025, 1024], 2048, 3), ([3000, 2000], 512, 4),
    ([3000, 2000], 544, 4), ([1500, 548], 5120, 1), ([2000, 2096], 4096, 1), ([2000, 2096], 4128, 1), ([9000, 7400], 288, 1),
    ([9000, 7384], 1056, 1), ([9000, 7384], 1056, 2), ([300, 212], 4096, 8), ([300, 213], 4096, 5), ([300, 70], 4096, 9),
    ([300, 70, 142], 4096, 2), ([300, 70, 143], 4096, 1), ([300, 70, 20], 4096, 3), ([3000, 1000, 96], 4096, 1)])
def test_batch_multi_rule(dev, host, oracle, mem, t, shapes, cols, batch):
    """Two and three matrices on both sides of each limit between the general
    kernel and the matrix cores."""
    ws = [V.synth_matrix(host, t, r, cols, SEED, 186 + m) for m, r in enumerate(shapes)]
    X = vectors(host, batch, cols, 197)
    for w, r, Y in zip(ws, shapes, run_multi(dev, mem, t, ws, X, shapes, cols)):
        for b in range(batch):
            assert lin_err(Y[b], oracle.linear(t, w, X[b], cols, r, threads=8)) <= LIN_TOL, b


@pytest.mark.parametrize("t", BLK, ids=lambda t: V.TYPE_NAMES[t])
def test_batch_block_types_non_finite(dev, host, oracle, mem, t):
    """inf and NaN in a vector and in a row's scales give the oracle's inf and
    NaN rows; the other vectors and rows stay within the bar."""
    rows, cols = 64, 1024
    w = V.synth_matrix(host, t, rows, cols, SEED, 74)
    w[7, :2] = np.array([0x7C00], np.uint16).view(np.uint8)  # an infinite scale (F16: weight)
    w[9, :2] = np.array([0x7E00], np.uint16).view(np.uint8)  # NaN
    X = vectors(host, 6, cols, 110)
    X[1, 300], X[2, 5], X[3, 1000] = np.inf, np.nan, -np.inf
    Y = run_batch(dev, mem, t, w, X, rows, cols)
    for b in range(6):
        with np.errstate(invalid="ignore"):
            want = oracle.linear(t, w, X[b], cols, rows)
        fine = np.isfinite(want)
        assert np.array_equal(np.isnan(Y[b]), np.isnan(want)), b
        assert np.array_equal(Y[b][~fine & ~np.isnan(want)], want[~fine & ~np.isnan(want)]), b
        if fine.any():
            assert lin_err(Y[b][fine], want[fine]) <= LIN_TOL, b


def run_multi(dev, mem, t, ws, X, shapes, cols, base=0):
    """Y of each matrix through one matrix-core launch, the matrices at a base
    that is only `base` bytes past 16-byte alignment."""
    batch = X.shape[0]
    pws = [mem.up(np.concatenate([np.zeros(base, np.uint8), w.reshape(-1)])) + base for w in ws]
    pys = [mem.zeros(batch * r) for r in shapes]
    dev.linear_batch_multi(t, pws, shapes, mem.up(X), cols, pys, shapes, cols, batch)
    return [dev.download(py, (batch, r), np.float32) for py, r in zip(pys, shapes)]


# (test_batch_block_types' [1], [16], [300] and [4097] and the one matrix of
# test_batch_block_types_non_finite run in the general kernel, as do two matrices
# of few rows and at most four vectors; three of such rows take k_mvbb)
@pytest.mark.parametrize("t", BLK, ids=lambda t: V.TYPE_NAMES[t])
@pytest.mark.parametrize("batch", [1, 6, 11])
def test_batch_mfma_non_finite(dev, host, oracle, mem, t, batch):
    """Infinities and NaN on the matrix cores: in vectors, and as scales,
    weights and Q4_1 mins, also in a row's partly filled last unit, give the
    oracle's inf and NaN; every other result stays within the bar."""
    shapes, cols = [40, 33, 5], 1056
    ws = [V.synth_matrix(host, t, r, cols, SEED, 260 + m) for m, r in enumerate(shapes)]
    bb = V.GEOMETRY[t][1]
    f16 = lambda v: np.array([v], np.uint16).view(np.uint8)  # noqa: E731
    ws[0][3, :2], ws[0][39, -bb:][:2], ws[1][7, -bb:][:2] = f16(0x7C00), f16(0x7C00), f16(0x7E00)
    if t == V.Q4_1:
        ws[1][32, -bb + 2:][:2] = f16(0xFC00)
    X = vectors(host, batch, cols, 270)
    X[0, 300] = np.inf
    if batch > 1:
        X[2, 1040], X[4, 1055], X[batch - 1, 0] = np.nan, -np.inf, np.inf
    for w, r, Y in zip(ws, shapes, run_multi(dev, mem, t, ws, X, shapes, cols)):
        for b in range(batch):
            with np.errstate(invalid="ignore"):
                want = oracle.linear(t, w, X[b], cols, r)
            fine = np.isfinite(want)
            assert np.array_equal(np.isnan(Y[b]), np.isnan(want)), b
            assert np.array_equal(Y[b][np.isinf(want)], want[np.isinf(want)]), b
            if fine.any():
                assert lin_err(Y[b][fine], want[fine]) <= LIN_TOL, b


@pytest.mark.parametrize("t", BLK, ids=lambda t: V.TYPE_NAMES[t])
@pytest.mark.parametrize("base", [0, 2, 6, 14])
def test_batch_mfma_activation_edges(dev, host, oracle, mem, t, base):
    """The per-unit scaling of the block types' vectors (all zero, 1e-30, 1e30,
    outliers, zero and subnormal sub-blocks) with the matrices at every kind of
    2-byte base (F16 off 16 bytes takes the general kernel)."""
    shapes, cols = [70, 17], 1120
    ws = [V.synth_matrix(host, t, r, cols, SEED, 290 + m) for m, r in enumerate(shapes)]
    X = vectors(host, 8, cols, 300)
    X[0] = 0.0
    X[1] *= 1e-30
    X[2] *= 1e30
    X[3, 40] = 1.0e4
    X[4, 0:32] = 0.0
    X[4, 64:96] *= 1e-40
    X[5, 96:128] *= 1e30
    X[6, 7] = -0.0
    X[7, 1100:] *= 1e-38
    for w, r, Y in zip(ws, shapes, run_multi(dev, mem, t, ws, X, shapes, cols, base)):
        assert np.all(Y[0] == 0.0)
        for b in range(1, 8):
            want = oracle.linear(t, w, X[b], cols, r)
            assert np.all(np.isfinite(Y[b])), b
            assert lin_err(Y[b], want) <= LIN_TOL, b


def test_scratch_growth_keeps_captured_graphs(dev, host, oracle, mem):
    """The batched matvec keeps its prepared x in the library's scratch. A
    graph captured from the library's stream holds the scratch address of the
    capture, so a later call that grows the scratch (a long attention: its
    per-chunk partials live there too) must leave that memory valid: every
    replay still meets the oracle. A call under capture that would need more
    scratch fails with a reason and launches nothing (growing allocates)."""
    hip, stream = V.Hip(), dev.stream()
    t, rows, cols, batch = V.Q4_K, 96, 4096, 4
    w = V.synth_matrix(host, t, rows, cols, SEED, 78)
    X = vectors(host, batch, cols, 140)
    pw, px, py = mem.up(w), mem.up(X), mem.zeros(batch * rows)
    want = [oracle.linear(t, w, X[b], cols, rows) for b in range(batch)]
    nqh, nkh, hd = 8, 1, 128
    pq, po = mem.up(synth_x(host, nqh * hd, 141)), mem.zeros(nqh * hd)

    # zero keys and values for the long attentions below, allocated before any capture
    caches = {seq: (mem.zeros(seq * hd, np.uint16), mem.zeros(seq * hd, np.uint16))
              for seq in (520_000, 1_100_000)}

    def attention(seq):
        """Attention over `seq` zero keys and values: per-chunk partials of
        8 x seq/64 x 130 floats (32 MiB at 520,000 positions)."""
        kc, vc = caches[seq]
        return dev._attention(pq, kc, vc, po, seq, 0, seq, nqh, nkh, hd, ctypes.c_float(0.088))

    dev.linear_batch(t, pw, px, cols, py, rows, cols, rows, batch)  # sizes the scratch
    graph = hip.capture(stream, lambda: dev.linear_batch(t, pw, px, cols, py, rows, cols, rows,
                                                         batch))
    try:
        for rep in range(3):
            dev.write(py, np.zeros(batch * rows, np.float32))
            if rep == 1:  # grows the scratch well past anything the other tests use
                assert attention(520_000) == 1, dev.error()
                assert np.all(dev.download(po, nqh * hd, np.float32) == 0.0)
            hip.launch(graph, stream)
            Y = dev.download(py, (batch, rows), np.float32)
            for b in range(batch):
                assert lin_err(Y[b], want[b]) <= LIN_TOL, (rep, b)
    finally:
        hip.destroy(graph)
    rc = []
    failed = hip.capture(stream, lambda: rc.append(attention(1_100_000)))
    hip.destroy(failed)
    assert rc == [0] and "capturing" in dev.error(), dev.error()
    # the stream works on after the refused call
    dev.linear_batch(t, pw, px, cols, py, rows, cols, rows, batch)
    Y = dev.download(py, (batch, rows), np.float32)
    assert lin_err(Y[0], want[0]) <= LIN_TOL


def test_batch_calls_of_several_threads(dev, host, mem):
    """Batched matvecs and a chunked attention issued by several threads at once
    (they share the library's stream and scratch): every result has the bits
    of the same call alone."""
    calls = []
    for i, (t, rows, cols, batch) in enumerate([(V.Q8_0, 3072, 1280, 8), (V.Q4_1, 4096, 1024, 16),
                                                (V.F16, 3104, 2048, 6), (V.Q4_K, 512, 2048, 8)]):
        pw, px = mem.up(V.synth_matrix(host, t, rows, cols, SEED, 210 + i)), mem.up(vectors(host, batch, cols, 220 + 20 * i))
        py = mem.zeros(batch * rows)
        calls.append((lambda a=(t, pw, px, cols, py, rows, cols, rows, batch): dev.linear_batch(*a), py, batch * rows))
    nqh, nkh, hd, seq = 16, 2, 64, 3000
    pk = mem.up(V.synth_normal_f16(host, seq * nkh * hd, SEED, 230))
    pq, po = mem.up(synth_x(host, nqh * hd, 231)), mem.zeros(nqh * hd)
    calls.append((lambda: dev.attention(pq, pk, pk, po, seq, 0, seq, nqh, nkh, hd, np.float32(0.125)), po, nqh * hd))
    want = []
    for call, p, n in calls:
        call()
        want.append(dev.download(p, n, np.float32))
    for _ in range(10):
        for _, p, n in calls:
            dev.write(p, np.full(n, 7.0, np.float32))
        go = threading.Barrier(len(calls))

        def work(call):
            go.wait()
            for _ in range(20):
                call()

        threads = [threading.Thread(target=work, args=(c[0],)) for c in calls]
        for th in threads:
            th.start()
        for th in threads:
            th.join()
        for (_, p, n), w in zip(calls, want):
            assert np.array_equal(dev.download(p, n, np.float32).view(np.uint32), w.view(np.uint32))


def test_batch_graphs_beside_each_other(dev, host, mem):
    """Captured batched matvecs of the block types, replayed on two streams at
    once and beside uncaptured calls: each keeps its prepared vectors in its
    own graph's memory, so every result has the uncaptured call's bits."""
    hip, stream = V.Hip(), dev.stream()
    hip.h.hipStreamCreateWithFlags.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_uint]
    hip.h.hipStreamSynchronize.argtypes = hip.h.hipStreamDestroy.argtypes = [ctypes.c_void_p]
    calls, want, graphs, streams = [], [], [], []
    for i, (t, rows, cols, batch) in enumerate([(V.Q8_0, 3072, 1280, 8), (V.Q4_1, 4096, 1280, 16),
                                                (V.Q4_0, 3072, 1280, 5)]):
        pw, px = mem.up(V.synth_matrix(host, t, rows, cols, SEED, 240 + i)), mem.up(vectors(host, batch, cols, 250 + 20 * i))
        py = mem.zeros(batch * rows)
        calls.append((lambda a=(t, pw, px, cols, py, rows, cols, rows, batch): dev.linear_batch(*a), py, batch * rows))
        calls[-1][0]()
        want.append(dev.download(py, batch * rows, np.float32))
    try:
        for call, _, _ in calls[:2]:
            graphs.append(hip.capture(stream, lambda: [call() for _ in range(20)]))
            s = ctypes.c_void_p()
            assert hip.h.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
            streams.append(s.value)
        for _ in range(10):
            for _, p, n in calls:
                dev.write(p, np.full(n, 7.0, np.float32))
            dev.sync()
            for g, s in zip(graphs, streams):
                hip.launch(g, s)
            for _ in range(20):
                calls[2][0]()
            for s in streams:
                assert hip.h.hipStreamSynchronize(s) == 0
            for (_, p, n), w in zip(calls, want):
                assert np.array_equal(dev.download(p, n, np.float32).view(np.uint32), w.view(np.uint32))
    finally:
        for g in graphs:
            hip.destroy(g)
        for s in streams:
            hip.h.hipStreamDestroy(s)


def test_batch_capture_needs_no_sizing_call(dev, host, oracle, mem):
    """A capture of calls whose prepared vectors (17 MB and 9 MB) no uncaptured
    call has sized: the graph's bits are those of the calls alone, replay after
    replay; captured again and again, its memory is given back."""
    hip, stream = V.Hip(), dev.stream()
    hip.h.hipMemGetInfo.argtypes = [ctypes.POINTER(ctypes.c_size_t)] * 2

    def free_bytes():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.h.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    t, rows, cols, batch = V.Q4_0, 1040, 262144, 16
    w = V.synth_matrix(host, t, rows, cols, SEED, 280)
    X = vectors(host, batch, cols, 281)
    pw, px, py = mem.up(w), mem.up(X), mem.zeros(batch * rows)

    def enqueue():
        dev.linear_batch(t, pw, px, cols, py, rows, cols, rows, 8)  # (and a smaller one before it)
        dev.linear_batch(t, pw, px, cols, py, rows, cols, rows, batch)

    before, got = free_bytes(), []
    for rep in range(12):
        graph = hip.capture(stream, enqueue)
        for _ in range(2):
            dev.write(py, np.zeros(batch * rows, np.float32))
            hip.launch(graph, stream)
            got.append(dev.download(py, (batch, rows), np.float32))
        hip.destroy(graph)
        dev.sync()
    assert before - free_bytes() <= 8 * (48 << 20)  # (the graphs', idle ones among them; each holds 16 + 32 MiB)
    dev.linear_batch(t, pw, px, cols, py, rows, cols, rows, batch)
    alone = dev.download(py, (batch, rows), np.float32)
    for Y in got:
        assert np.array_equal(Y.view(np.uint32), alone.view(np.uint32))
    ws = np.ascontiguousarray(w[:32])
    for b in (0, 9, 15):
        assert lin_err(alone[b, :32], oracle.linear(t, ws, X[b], cols, 32)) <= LIN_TOL, b
