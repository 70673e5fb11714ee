"""GPU prefill matmul (MFMA, f16 operands, fp32 accumulation) against the fp64
oracle X @ dequant(W)^T and the reference's own batched-matmul outputs.

Tolerance: weights are decoded exactly and rounded once to f16, x rows are
scaled by a power of two and rounded to f16, so each product carries at most
2^-11 relative error and each output at most about 2^-11 * sum|w*x| (fp32
accumulation adds K * 2^-24 of the same sum). Gates: every output within
1e-3 * sum_k |w_k x_k| (the dot-product error bound, which holds however much
the sum cancels), and the path's max-rel 1e-3 target (normwise:
max|y - y_ref| / max|y_ref|) for tiles of at least 64 outputs, where the
typical figure is near 2e-4."""
import ctypes

import numpy as np
import pytest

from oracle import quant
from tests.conftest import normwise_rel
from tests.gpu_util import random_ggml

pytestmark = pytest.mark.gpu

TYPES = (2, 8, 12, 13, 14)
MAX_REL = 1e-3


def check(got, raw, t, rows, cols, xs):
    ref = quant.matmul_exact(raw, t, rows, cols, xs)
    w = quant.dequantize(raw, t, (rows, cols)).astype(np.float64)
    absdot = np.abs(np.asarray(xs, dtype=np.float64)) @ np.abs(w).T
    assert np.all(np.abs(got - ref) <= MAX_REL * absdot + 1e-30)
    if ref.size >= 64:
        assert normwise_rel(got, ref) < MAX_REL
    return ref


def gpu_matmul(raw, t, rows, cols, xs, rows_major=False):
    from localai_amd import device
    q = device.QMat.from_ggml(raw, t, rows, cols)
    y = q.matmul(device.to_device_f32(xs), rows_major=rows_major).cpu().numpy()
    q.close()
    return y


@pytest.mark.parametrize('t', TYPES)
def test_golden_matmul(golden, t):
    """The reference test-suite matmul case (64 x 512, 5 tokens, tests/test_dequant.py:160-177)."""
    raw, xs = golden[f'raw_mm_{t}'].tobytes(), golden['vectors']
    got = gpu_matmul(raw, t, 64, 512, xs)
    assert got.shape == (5, 64)
    check(got, raw, t, 64, 512, xs)
    assert normwise_rel(got, golden[f'matmul_{t}']) < MAX_REL


@pytest.mark.parametrize('t', TYPES)
@pytest.mark.parametrize('rows,tokens', [(1, 1), (200, 37), (128, 128), (300, 130), (129, 257)])
def test_ragged_tiles(t, rows, tokens):
    rng = np.random.default_rng(rows * 7 + tokens + t)
    block, _ = quant.block_layout(t)
    cols = 512 if block == 256 else 160      # Q8_0/Q4_0: 5 blocks, an odd number of 64-value units
    raw = random_ggml(rng, t, rows * cols)
    xs = rng.standard_normal((tokens, cols)).astype(np.float32)
    got = gpu_matmul(raw, t, rows, cols, xs)
    assert got.shape == (tokens, rows)
    check(got, raw, t, rows, cols, xs)


@pytest.mark.parametrize('t', (8, 12, 14))
@pytest.mark.parametrize('nblocks', (1, 3, 8, 17))
def test_k_lengths(t, nblocks):
    rng = np.random.default_rng(nblocks * 5 + t)
    block, _ = quant.block_layout(t)
    rows, cols, tokens = 96, block * nblocks, 40
    raw = random_ggml(rng, t, rows * cols)
    xs = rng.standard_normal((tokens, cols)).astype(np.float32)
    got = gpu_matmul(raw, t, rows, cols, xs)
    check(got, raw, t, rows, cols, xs)


@pytest.mark.parametrize('rows,cols,tokens', [(112, 256, 256), (113, 512, 257), (300, 160, 300), (16, 768, 600),
                                            (1000, 1024, 512), (1800, 256, 256)])
def test_q8_0_workgroup_tiles(rows, cols, tokens):
    """Q8_0 with 256 tokens or more: ragged row and token edges, K padded up to
    whole 256-value blocks (cols 160), one and several tiles each way, and both
    output layouts."""
    rng = np.random.default_rng(rows + cols + tokens)
    raw = random_ggml(rng, 8, rows * cols)
    xs = rng.standard_normal((tokens, cols)).astype(np.float32)
    got = gpu_matmul(raw, 8, rows, cols, xs)
    assert got.shape == (tokens, rows)
    check(got, raw, 8, rows, cols, xs)
    if rows * tokens <= 300 * 300:
        np.testing.assert_array_equal(gpu_matmul(raw, 8, rows, cols, xs, rows_major=True), got.T)


@pytest.mark.parametrize('t', TYPES)
@pytest.mark.parametrize('rows,nblocks,tokens', [(16, 1, 1), (257, 2, 17), (272, 5, 49), (300, 6, 81), (40, 16, 113),
                                                 (512, 24, 130), (8192, 4, 32)])
def test_dense_tiles_and_splits(t, rows, nblocks, tokens):
    """The dense kernel's edges: odd and even block counts per split, one and
    many splits, token tiles of 1 to 8 MFMA tiles, rows past the last row tile;
    and a workspace with no room for splits (the size of the converted x),
    which takes one split: the same products, summed in another order."""
    from localai_amd import _lib, device
    rng = np.random.default_rng(rows + 31 * nblocks + tokens + t)
    cols = 256 * nblocks
    raw = random_ggml(rng, t, rows * cols)
    xs = rng.standard_normal((tokens, cols)).astype(np.float32)
    ref = check(gpu_matmul(raw, t, rows, cols, xs), raw, t, rows, cols, xs)
    q = device.QMat.from_ggml(raw, t, rows, cols)
    xd = device.to_device_f32(xs)
    torch = device.torch()
    least = (tokens + 15) // 16 * 16 * cols * 2 + tokens * 4
    ws = torch.empty(least, dtype=torch.uint8, device=xd.device)
    y = torch.empty((tokens, rows), dtype=torch.float32, device=xd.device)
    lib = _lib.load()
    args = (q.handle, 0, device.ptr(xd), tokens, device.ptr(y), 0, device.ptr(ws))
    _lib.check(lib.localai_hip_matmul(*args, least, device.stream_ptr()))
    check(y.cpu().numpy(), raw, t, rows, cols, xs)
    assert lib.localai_hip_matmul(*args, least - 1, device.stream_ptr()) != 0
    assert int(lib.localai_hip_matmul_workspace_size(q.handle, tokens)) >= least
    assert np.isfinite(ref).all()
    q.close()


@pytest.mark.parametrize('t,rows,nblocks,tokens', [(12, 4112, 3, 2000), (14, 4096, 2, 2048), (8, 3900, 4, 2100),
                                                   (13, 4112, 2, 2000), (2, 4100, 3, 1990)])
def test_dense_rounds_of_tiles(t, rows, nblocks, tokens):
    """More than 256 output tiles of few blocks of K: one whole round, none or some
    tiles left over (the Q4_K and Q8_0 shapes run the 128-row tile kernel), ragged
    edges; both output layouts hold the same values."""
    rng = np.random.default_rng(rows + tokens)
    cols = 256 * nblocks
    raw = random_ggml(rng, t, rows * cols)
    xs = rng.standard_normal((tokens, cols)).astype(np.float32)
    got = gpu_matmul(raw, t, rows, cols, xs)
    check(got, raw, t, rows, cols, xs)
    np.testing.assert_array_equal(gpu_matmul(raw, t, rows, cols, xs, rows_major=True), got.T)


@pytest.mark.parametrize('t,nblocks', [(12, 10), (12, 11), (14, 10), (14, 11), (8, 10), (8, 11), (13, 6), (13, 7),
                                       (2, 6), (2, 7)])
@pytest.mark.parametrize('rows,tokens', [(8200, 2100), (8192, 2048)])
def test_dense_two_rounds_and_parts(t, nblocks, rows, tokens):
    """Two whole rounds of 256 tiles (a whole tile's first requests in flight while
    the whole tile before it is stored), then 49 tiles in parts of K, which only
    some workgroups have (561 tiles, ragged edges), or nothing (512 tiles); odd
    and even block counts; every output against 64-bit products of the same
    weights, in both layouts."""
    from localai_amd import _lib, device
    torch = device.torch()
    rng = np.random.default_rng(t + nblocks + rows)
    cols = 256 * nblocks
    block, size = quant.block_layout(t)
    part = np.frombuffer(random_ggml(rng, t, 257 * cols), np.uint8).reshape(-1, size)
    raw = np.resize(part, (rows * cols // block, size)).tobytes()
    q = device.QMat.from_ggml(raw, t, rows, cols)
    least = (tokens + 15) // 16 * 16 * cols * 2 + tokens * 4
    parts = int(_lib.load().localai_hip_matmul_workspace_size(q.handle, tokens)) - least
    assert (parts >= 2 * 49 * 256 * 128 * 4) == (rows == 8200)
    x = device.to_device_f32(rng.standard_normal((tokens, cols)))
    got = q.matmul(x)
    assert torch.equal(q.matmul(x, rows_major=True), got.T)
    w, x = q.dequant().double().T.contiguous(), x.double()
    ref = x @ w
    err = (got.double() - ref).abs()
    assert bool(err.le(MAX_REL * (x.abs() @ w.abs())).all())
    assert float(err.max() / ref.abs().max()) < MAX_REL
    q.close()


@pytest.mark.parametrize('t,rows,cols,tokens', [(2, 3, (1 << 25) + 32, 66), (8, 3, (1 << 25) + 32, 66),
                                                (2, 1, (1 << 28) + 32, 1)])
def test_rows_past_32_bit_offsets(t, rows, cols, tokens):
    """More than 4 GiB of f16 rows of x under one token tile (33.6 million columns,
    66 tokens): several launches, each with offsets of 32 bits, the same products
    in both layouts; and a row of 268 million columns. x holds zeros but for
    2^16 values (the row's ends among them), so that fp32 sums over millions of
    products stay exact enough to compare."""
    from localai_amd import device
    torch = device.torch()
    rng = np.random.default_rng(t)
    block, size = quant.block_layout(t)
    part = np.frombuffer(random_ggml(rng, t, 1 << 20), np.uint8).reshape(-1, size)
    raw = np.resize(part, (rows * cols // block, size)).tobytes()
    q = device.QMat.from_ggml(raw, t, rows, cols)
    at = np.unique(np.concatenate([rng.integers(0, cols, 1 << 16), np.arange(64), np.arange(cols - 64, cols)]))
    vals = device.to_device_f32(rng.standard_normal((tokens, len(at))))
    at = torch.from_numpy(at).to(vals.device)
    x = torch.zeros((tokens, cols), dtype=torch.float32, device=vals.device)
    x[:, at] = vals
    got = q.matmul(x)
    assert torch.equal(q.matmul(x, rows_major=True), got.T)
    w = q.dequant()[:, at].double()
    for tok in range(tokens):
        terms = w * vals[tok].double()
        # products of random sign, x and w each rounded by up to 2^-11 of them,
        # evenly: five standard deviations of their sum
        bound = 5 * 2.0 ** -11 * (2 / 3) ** 0.5 * terms.square().sum(1).sqrt()
        assert bool((got[tok].double() - terms.sum(1)).abs().le(bound).all())
    q.close()


@pytest.mark.parametrize('t', TYPES)
@pytest.mark.parametrize('rows_major', (False, True))
def test_parts_of_huge_activations_cancel(t, rows_major):
    """Rows of x near fp32's largest values whose halves cancel in the product:
    each half's sum exceeds fp32, the whole does not, however K is divided.
    One positive weight throughout (its type's bytes), so every output of a
    token is the sum of its x times that weight."""
    from localai_amd import device
    rows, cols, tokens = 300, 4096, 33
    block, size = quant.block_layout(t)
    b = np.zeros((rows * cols // block, size), np.uint8)
    d = 208 if t == 14 else 0
    b[:, d:d + 2] = np.frombuffer(np.float16(0.002).tobytes(), np.uint8)
    if t in (12, 13):
        b[:, 4:12], b[:, 12:16] = 1, 0x11   # scales 1 (of dmin, which is 0, too)
        b[:, 16:48] = 0x11 if t == 12 else 0
        b[:, 48:] = 0x11                    # quants 1
    elif t == 14:
        b[:, 128:192], b[:, 192:208] = 0xAA, 1   # high bits 2: quants 32 - 32 + 1
        b[:, :128] = 0x11
    else:
        b[:, 2:] = 1 if t == 8 else 0x99    # quants 1 (Q4_0: 9 - 8)
    raw = b.tobytes()
    w = quant.dequantize(raw, t, (rows, cols)).astype(np.float64)
    assert w.min() == w.max() > 0.0019
    # exact in f16: with values that are not, the rounding of each half (up to
    # 2^-11 of it) would be 15 times that of the whole in normwise_rel
    xs = np.full((tokens, cols), 2.0 ** 127, np.float32)
    xs[:, cols // 2:] *= np.float32(-0.875)
    xs[1] = 1.0
    q = device.QMat.from_ggml(raw, t, rows, cols)
    got = q.matmul(device.to_device_f32(xs), rows_major=rows_major).cpu().numpy()
    q.close()
    check(got.T if rows_major else got, raw, t, rows, cols, xs)


@pytest.mark.parametrize('t', (12, 14, 8))
@pytest.mark.parametrize('rows,cols,tokens', [(300, 512, 130), (129, 1280, 33), (16, 768, 7), (200, 160, 257)])
def test_handles_without_the_tile_form(monkeypatch, t, rows, cols, tokens):
    """LOCALAI_HIP_MFMA_MATVEC=0 when a handle is made: Q4_K, Q6_K and Q8_0 hold
    row planes, and their products, in both layouts, through the handle and
    through the legacy export, come from those."""
    from localai_amd import _lib, device
    if cols % quant.block_layout(t)[0]:
        cols += 256 - cols % 256
    rng = np.random.default_rng(rows + cols + t)
    raw = random_ggml(rng, t, rows * cols)
    xs = rng.standard_normal((tokens, cols)).astype(np.float32)
    monkeypatch.setenv('LOCALAI_HIP_MFMA_MATVEC', '0')
    q = device.QMat.from_ggml(raw, t, rows, cols)
    xd = device.to_device_f32(xs)
    got = q.matmul(xd).cpu().numpy()
    check(got, raw, t, rows, cols, xs)
    np.testing.assert_array_equal(q.matmul(xd, rows_major=True).cpu().numpy(), got.T)
    assert normwise_rel(q.matvec(xd[0].contiguous()).cpu().numpy(), quant.matmul_exact(raw, t, rows, cols, xs[:1])[0]) < 1e-5
    q.close()
    lib = _lib.load()
    out = np.zeros((rows, tokens), np.float32)
    buf = np.frombuffer(raw, np.uint8)
    f32 = ctypes.POINTER(ctypes.c_float)
    getattr(lib, {12: 'localai_q4k_matmul', 14: 'localai_q6k_matmul', 8: 'localai_q8_0_matmul'}[t])(
        buf.ctypes.data_as(ctypes.POINTER(ctypes.c_uint8)), xs.ctypes.data_as(f32), out.ctypes.data_as(f32), rows,
        cols, tokens, 4)
    assert lib.localai_hip_last_status() == 0
    check(out.T, raw, t, rows, cols, xs)


@pytest.mark.parametrize('t', (12, 14, 8))
@pytest.mark.parametrize('rows,nblocks,tokens', [(1, 1, 33), (16, 1, 40), (129, 3, 257), (300, 2, 130), (4112, 2, 2000),
                                                 (81001, 1, 5)])
def test_short_k_on_128_row_tiles(t, rows, nblocks, tokens):
    """Products of few blocks of K, more than 32 tokens (or very many rows): the 128 x
    128 tiles of the tile form's older kernel. Ragged row and token edges, one to several
    hundred workgroups, Q8_0 rows that end inside a block; no room for parts in
    the workspace, both output layouts."""
    from localai_amd import _lib, device
    rng = np.random.default_rng(rows + 31 * nblocks + tokens + t)
    cols = 256 * nblocks - (32 if t == 8 else 0)
    raw = random_ggml(rng, t, rows * cols)
    xs = rng.standard_normal((tokens, cols)).astype(np.float32)
    q = device.QMat.from_ggml(raw, t, rows, cols)
    least = (tokens + 15) // 16 * 16 * 256 * nblocks * 2 + tokens * 4
    assert int(_lib.load().localai_hip_matmul_workspace_size(q.handle, tokens)) == least
    xd = device.to_device_f32(xs)
    got = q.matmul(xd).cpu().numpy()
    check(got, raw, t, rows, cols, xs)
    np.testing.assert_array_equal(q.matmul(xd, rows_major=True).cpu().numpy(), got.T)
    q.close()


@pytest.mark.parametrize('t', (2, 8))
@pytest.mark.parametrize('cols', (32, 64, 96, 2144, 4128, 4192))
@pytest.mark.parametrize('tokens', (33, 20))
def test_dense_rows_of_partial_blocks(t, cols, tokens):
    """32-value blocks: rows that end inside a 256-value block or a 64-value unit,
    around the 4096-value chunks of the row planes; the last block's scale is
    infinite in one row, whose outputs must not leak into others."""
    rng = np.random.default_rng(cols + t)
    rows = 37
    raw = random_ggml(rng, t, rows * cols)
    xs = rng.standard_normal((tokens, cols)).astype(np.float32)
    got = gpu_matmul(raw, t, rows, cols, xs)
    check(got, raw, t, rows, cols, xs)
    b = np.frombuffer(raw, np.uint8).copy().reshape(rows, -1)
    size = 18 if t == 2 else 34
    b[5, -size:-size + 2] = (0x00, 0x7c)
    inf = gpu_matmul(b.tobytes(), t, rows, cols, xs)
    keep = np.arange(rows) != 5
    np.testing.assert_array_equal(inf[:, keep], got[:, keep])


@pytest.mark.parametrize('cols', (2304, 4096, 4352, 8192, 12544, 16384, 16640))
def test_long_rows_of_x(cols):
    """Activation rows past 2048 values (one workgroup per row, each group count)
    and past 16384 (one wave, read twice), with a row of zeros."""
    rng = np.random.default_rng(cols)
    raw = random_ggml(rng, 12, 48 * cols)
    xs = rng.standard_normal((5, cols)).astype(np.float32)
    xs[3] = 0.0
    got = gpu_matmul(raw, 12, 48, cols, xs)
    check(got, raw, 12, 48, cols, xs)
    assert not got[3].any()


@pytest.mark.parametrize('t,rows,nblocks,tokens', [(12, 512, 16, 77), (13, 300, 9, 40)])
def test_dense_parts_replayed_from_a_graph(t, rows, nblocks, tokens):
    """A product in several parts of K, captured and replayed with eager work
    between the replays: every replay equals the eager call bit for bit."""
    from localai_amd import device
    torch = device.torch()
    rng = np.random.default_rng(rows + tokens)
    cols = 256 * nblocks
    q = device.QMat.from_ggml(random_ggml(rng, t, rows * cols), t, rows, cols)
    x = device.to_device_f32(rng.standard_normal((tokens, cols)).astype(np.float32))
    want = q.matmul(x).clone()
    out = torch.empty_like(want)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        q.matmul(x, out=out)
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        q.matmul(x, out=out)
    for _ in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        q.matmul(x[:17].contiguous())
        torch.cuda.synchronize()
    q.close()


def test_rows_major_layout_matches_reference_convention():
    """y_layout 1 is the [rows, tokens] buffer of localai_*_matmul (engine/native_quant.cpp:492)."""
    rng = np.random.default_rng(11)
    raw = random_ggml(rng, 8, 70 * 256)
    xs = rng.standard_normal((9, 256)).astype(np.float32)
    a = gpu_matmul(raw, 8, 70, 256, xs)
    b = gpu_matmul(raw, 8, 70, 256, xs, rows_major=True)
    assert b.shape == (70, 9)
    np.testing.assert_array_equal(a, b.T)


def test_token_rows_of_very_different_magnitude():
    """Each token row gets its own power-of-two scale into f16 range, so rows
    far outside f16's range (1e6, 1e-7) keep full relative accuracy."""
    rng = np.random.default_rng(5)
    rows, cols = 64, 512
    raw = random_ggml(rng, 12, rows * cols)
    xs = rng.standard_normal((4, cols)).astype(np.float32)
    xs[1] *= 1e6
    xs[2] *= 1e-7
    xs[3, :] = 0.0
    got = gpu_matmul(raw, 12, rows, cols, xs)
    ref = quant.matmul_exact(raw, 12, rows, cols, xs)
    w = quant.dequantize(raw, 12, (rows, cols)).astype(np.float64)
    absdot = np.abs(xs.astype(np.float64)) @ np.abs(w).T
    for r in range(3):
        assert normwise_rel(got[r], ref[r]) < MAX_REL
        assert np.all(np.abs(got[r] - ref[r]) <= MAX_REL * absdot[r])
    assert np.all(got[3] == 0.0)


def test_q8_0_prefill_shape_sampled_rows():
    """The Q8_0 prefill workload at full size (512 tokens x 4096 -> 14336 rows):
    every output is computed on the GPU; rows sampled every 97 are checked
    against the fp64 oracle, and all outputs must be finite."""
    from localai_amd import device
    from localai_amd import synth
    rows, cols, tokens = 14336, 4096, 512
    raw = synth.quant_tensor(np.random.default_rng(3), 8, rows, cols)
    xs = np.random.default_rng(4).standard_normal((tokens, cols)).astype(np.float32)
    q = device.QMat.from_ggml(raw, 8, rows, cols)
    got = q.matmul(device.to_device_f32(xs)).cpu().numpy()
    q.close()
    assert np.all(np.isfinite(got))
    sample = np.arange(0, rows, 97)
    _, bpb = quant.block_layout(8)
    row_bytes = cols // 32 * bpb
    buf = np.frombuffer(raw, dtype=np.uint8).reshape(rows, row_bytes)[sample]
    check(got[:, sample], buf.tobytes(), 8, len(sample), cols, xs)
