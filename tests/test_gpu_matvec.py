"""GPU decode-matvec parity against the fp64 oracle (exactly decoded weights),
the reference's golden outputs and the reference's own test tolerances.

Tolerance: fp32 accumulation of exact products gives errors of order 1e-6 of
the output scale; the gate is the path's max-rel 1e-3 target (normwise:
max|y - y_ref| / max|y_ref|) plus an elementwise check at the reference
test suite's tolerances."""
import ctypes

import numpy as np
import pytest

from oracle import quant
from tests.conftest import normwise_rel
from tests.gpu_util import random_ggml

pytestmark = pytest.mark.gpu

TYPES = (2, 8, 12, 13, 14)
MAX_REL = 1e-3


def gpu_matvec(raw, t, rows, cols, x):
    from localai_amd import device
    q = device.QMat.from_ggml(raw, t, rows, cols)
    y = q.matvec(device.to_device_f32(x)).cpu().numpy()
    q.close()
    return y


@pytest.mark.parametrize('t', TYPES)
def test_golden_cases(golden, t):
    """The reference test-suite cases (300 x 512, tests/test_dequant.py:119-230)."""
    raw, x = golden[f'raw_{t}'].tobytes(), golden[f'x_{t}']
    got = gpu_matvec(raw, t, 300, 512, x)
    exact = quant.matvec_exact(raw, t, 300, 512, x)
    assert normwise_rel(got, exact) < 1e-5
    np.testing.assert_allclose(got, exact, rtol=2e-5, atol=2e-4)
    if t in (2, 8, 14):   # reference kernels that are exact up to rounding: same tolerance vs AVX2
        rtol, atol = (2e-5, 2e-4) if t == 8 else (2e-4, 2e-3)
        np.testing.assert_allclose(got, golden[f'matvec_{t}'], rtol=rtol, atol=atol)


@pytest.mark.parametrize('t', TYPES)
@pytest.mark.parametrize('rows', (1, 63, 64, 65, 300, 1000))
def test_ragged_rows(t, rows):
    rng = np.random.default_rng(rows * 31 + t)
    block, _ = quant.block_layout(t)
    cols = 512 if block == 256 else 96
    raw = random_ggml(rng, t, rows * cols)
    x = rng.standard_normal(cols).astype(np.float32)
    got = gpu_matvec(raw, t, rows, cols, x)
    assert normwise_rel(got, quant.matvec_exact(raw, t, rows, cols, x)) < 1e-5


@pytest.mark.parametrize('t', TYPES)
@pytest.mark.parametrize('nblocks', (1, 2, 7, 17, 56))
def test_k_lengths(t, nblocks):
    rng = np.random.default_rng(nblocks * 13 + t)
    block, _ = quant.block_layout(t)
    cols = block * nblocks
    raw = random_ggml(rng, t, 70 * cols)
    x = rng.standard_normal(cols).astype(np.float32)
    got = gpu_matvec(raw, t, 70, cols, x)
    assert normwise_rel(got, quant.matvec_exact(raw, t, 70, cols, x)) < 1e-5


@pytest.mark.parametrize('nsb', (1, 3, 8, 17, 33, 56, 72))
def test_q8_0_mfma_k_lengths(nsb):
    """Q8_0 rows of whole 256-value super-blocks take the i8-MFMA matvec over
    the tile form (every launch plan: 1..32 super-blocks per row at once,
    33..72 streamed through two register sets); ragged row count."""
    rng = np.random.default_rng(nsb * 7 + 1)
    cols = 256 * nsb
    raw = random_ggml(rng, 8, 70 * cols)
    x = rng.standard_normal(cols).astype(np.float32)
    got = gpu_matvec(raw, 8, 70, cols, x)
    assert normwise_rel(got, quant.matvec_exact(raw, 8, 70, cols, x)) < 1e-5


@pytest.mark.parametrize('t', (12, 14, 8))
@pytest.mark.parametrize('ntok', (1, 2, 3, 5, 8, 11))
def test_multi_vector(t, ntok):
    from localai_amd import device
    rng = np.random.default_rng(ntok + t)
    rows, cols = 200, 1024
    raw = random_ggml(rng, t, rows * cols)
    x = rng.standard_normal((ntok, cols)).astype(np.float32)
    q = device.QMat.from_ggml(raw, t, rows, cols)
    got = q.matvec(device.to_device_f32(x)).cpu().numpy()
    want = quant.matmul_exact(raw, t, rows, cols, x)
    assert got.shape == (ntok, rows)
    assert normwise_rel(got, want) < 1e-5


@pytest.mark.parametrize('t', (12, 14, 8))
@pytest.mark.parametrize('rows,cols,ntok', [(200, 1024, 7), (14336, 4096, 3), (4096, 14336, 5), (300, 256 * 60, 2),
                                            (48, 256 * 33, 4), (200, 256 * 65, 9), (40, 256 * 72, 3)])
def test_multi_vector_on_the_tile_form(t, rows, cols, ntok):
    """Several vectors through a Q4_K / Q6_K / Q8_0 handle run the tile-form
    kernel: every y[t] equals the one-vector call on x[t] bit for bit, the
    oracle within 1e-5 normwise, and the handle builds no row planes (its
    device bytes do not change)."""
    from localai_amd import _lib, device
    rng = np.random.default_rng(rows + ntok + t)
    raw = random_ggml(rng, t, rows * cols)
    x = rng.standard_normal((ntok, cols)).astype(np.float32)
    q = device.QMat.from_ggml(raw, t, rows, cols)
    lib = _lib.load()
    before = int(lib.localai_hip_qmat_device_bytes(q.handle))
    xd = device.to_device_f32(x)
    got = q.matvec(xd).cpu().numpy()
    assert int(lib.localai_hip_qmat_device_bytes(q.handle)) == before
    for i in range(ntok):
        one = q.matvec(xd[i].contiguous()).cpu().numpy()
        np.testing.assert_array_equal(got[i].view(np.uint32), one.view(np.uint32))
    sel = np.arange(rows) if rows <= 4096 else np.unique(rng.choice(rows, 1500, replace=False))
    rowb = len(raw) // rows
    sub = np.frombuffer(raw, np.uint8).reshape(rows, rowb)[sel].tobytes()
    want = quant.matmul_exact(sub, t, len(sel), cols, x)
    assert normwise_rel(got[:, sel], want) < 1e-5
    q.close()


@pytest.mark.parametrize('t', (12, 14, 8))
@pytest.mark.parametrize('rows,nsb,ntok', [(16 * 260 - 3, 3, 6), (16 * 600 + 5, 2, 9), (16 * 780, 1, 31), (16 * 1100 + 1, 2, 4),
                                           (40, 1, 13), (16 * 900 - 3, 12, 5), (16 * 1000 - 9, 9, 7),
                                           (16 * 1030 + 1, 10, 2)])
def test_multi_vector_groups_and_row_tiles(t, rows, nsb, ntok):
    """Vector counts around the groups of four, one, two and four row tiles per
    workgroup, ragged last tiles: each y[t] equals the one-vector call bit
    for bit."""
    from localai_amd import device
    rng = np.random.default_rng(rows + nsb + ntok + t)
    cols = 256 * nsb
    raw = random_ggml(rng, t, rows * cols)
    x = rng.standard_normal((ntok, cols)).astype(np.float32)
    q = device.QMat.from_ggml(raw, t, rows, cols)
    xd = device.to_device_f32(x)
    got = q.matvec(xd).cpu().numpy()
    for i in range(ntok):
        one = q.matvec(xd[i].contiguous()).cpu().numpy()
        np.testing.assert_array_equal(got[i].view(np.uint32), one.view(np.uint32))
    q.close()


@pytest.mark.parametrize('name,t,rows,cols', [
    ('ffn_gate', 12, 14336, 4096), ('ffn_down', 14, 4096, 14336), ('attn_v', 14, 1024, 4096),
    ('attn_k', 12, 1024, 4096)])
def test_llama3_8b_shapes(name, t, rows, cols):
    from localai_amd import synth
    rng = np.random.default_rng(11)
    raw = synth.quant_tensor(rng, t, rows, cols)
    x = synth.activations(rng, cols)
    got = gpu_matvec(raw, t, rows, cols, x)
    err = normwise_rel(got, quant.matvec_exact(raw, t, rows, cols, x))
    assert err < MAX_REL
    assert err < 1e-5, f'{name}: {err}'


@pytest.mark.parametrize('t', (14, 12))
def test_vocab_head_128256x4096(t):
    """The Llama-3-8B vocabulary head (engine/model.py:235-237, output.weight
    128256 x 4096: Q6_K in a Q4_K_M file, Q4_K checked too), 8016 row tiles
    in one launch: the first and last 64 rows and 3000 sampled rows against
    the oracle (its rows sliced out of the GGML bytes), and every output
    finite and repeatable bit for bit."""
    from localai_amd import device, synth
    rows, cols = 128256, 4096
    rng = np.random.default_rng(128 + t)
    raw = synth.quant_tensor(rng, t, rows, cols)
    x = synth.activations(rng, cols)
    q = device.QMat.from_ggml(raw, t, rows, cols)
    xd = device.to_device_f32(x)
    y = q.matvec(xd).cpu().numpy()
    y2 = q.matvec(xd).cpu().numpy()
    q.close()
    assert np.isfinite(y).all()
    np.testing.assert_array_equal(y.view(np.uint32), y2.view(np.uint32))
    rowb = (cols // 256) * (210 if t == 14 else 144)
    sel = np.unique(np.concatenate([np.arange(64), np.arange(rows - 64, rows),
                                    rng.choice(rows, 3000, replace=False)]))
    buf = np.frombuffer(raw, np.uint8).reshape(rows, rowb)
    want = quant.matvec_exact(buf[sel].tobytes(), t, len(sel), cols, x)
    err = normwise_rel(y[sel], want)
    print(f'vocab head type {t}: normwise {err:.2e} over {len(sel)} rows', flush=True)
    assert err < 1e-5


@pytest.mark.parametrize('t', (12, 14, 8))
def test_many_tile_loop_kernel(t):
    """From 2048 row tiles a one-vector matvec runs the tile-looping kernel:
    2049 tiles (an odd count, the last one 5 rows deep) at K = 2048 (eight
    waves). Sampled rows and the last tile against the oracle, and the first
    and last 64 rows bit for bit equal to the one-tile-per-workgroup kernel
    run on those rows alone (same products, same summation order; the last
    64 start mid-tile in the big matrix)."""
    from localai_amd import device, synth
    rows, cols = 2048 * 16 + 5, 2048
    rng = np.random.default_rng(40 + t)
    raw = synth.quant_tensor(rng, t, rows, cols)
    x = synth.activations(rng, cols)
    xd = device.to_device_f32(x)
    q = device.QMat.from_ggml(raw, t, rows, cols)
    y = q.matvec(xd).cpu().numpy()
    q.close()
    assert np.isfinite(y).all()
    rowb = len(raw) // rows
    buf = np.frombuffer(raw, np.uint8).reshape(rows, rowb)
    sel = np.unique(np.concatenate([np.arange(rows - 21, rows), rng.choice(rows, 1500, replace=False)]))
    want = quant.matvec_exact(buf[sel].tobytes(), t, len(sel), cols, x)
    assert normwise_rel(y[sel], want) < 1e-5
    for lo, hi in ((0, 64), (rows - 64, rows)):
        small = device.QMat.from_ggml(buf[lo:hi].tobytes(), t, hi - lo, cols)
        ys = small.matvec(xd).cpu().numpy()
        small.close()
        # a row's arithmetic does not depend on which rows share its tile
        np.testing.assert_array_equal(y[lo:hi].view(np.uint32), ys.view(np.uint32))


def test_expert_slices_of_a_3d_tensor():
    """[E, rows, cols] tensor; expert e is the byte slice of engine/zaya.py:144-150."""
    from localai_amd import device
    rng = np.random.default_rng(5)
    E, rows, cols = 4, 96, 512
    raw = random_ggml(rng, 14, E * rows * cols)
    q = device.QMat.from_ggml(raw, 14, rows, cols, batch=E)
    x = rng.standard_normal(cols).astype(np.float32)
    per = len(raw) // E
    for e in range(E):
        got = q.matvec(device.to_device_f32(x), expert=e).cpu().numpy()
        want = quant.matvec_exact(raw[e * per:(e + 1) * per], 14, rows, cols, x)
        assert normwise_rel(got, want) < 1e-5


# -------------------------------------------- drop-in Python API (native_quant)

def test_native_quant_mirror_contract():
    from localai_amd import native_quant as nq
    assert nq.get_native() is not None
    rng = np.random.default_rng(9)
    raw = random_ggml(rng, 12, 300 * 512)
    x = rng.standard_normal(512).astype(np.float32)
    y = nq.matvec(raw, x, 300, 512, 12)
    assert y.dtype == np.float32 and y.shape == (300,)
    assert normwise_rel(y, quant.matvec_exact(raw, 12, 300, 512, x)) < 1e-5
    # unsupported type / misaligned cols -> None (engine/native_quant.py:104-111)
    assert nq.matvec(raw, x, 300, 512, 3) is None
    assert nq.matvec(raw, x[:100], 300, 100, 12) is None
    # size mismatch -> ValueError (engine/native_quant.py:115-116)
    with pytest.raises(ValueError):
        nq.matvec(raw[:-144], x, 300, 512, 12)
    with pytest.raises(ValueError):
        nq.matvec(raw, x[:256], 300, 512, 12)
    v = rng.standard_normal((5, 512)).astype(np.float32)
    m = nq.matmul(raw, v, 300, 512, 12)
    assert m.shape == (5, 300)
    assert normwise_rel(m, quant.matmul_exact(raw, 12, 300, 512, v)) < 1e-5
    with pytest.raises(ValueError):
        nq.matmul(raw, v[:, :256], 300, 512, 12)
    # from 32 tokens the MFMA GEMM path (f16 operands): the GEMM tolerance
    v = rng.standard_normal((40, 512)).astype(np.float32)
    m = nq.matmul(raw, v, 300, 512, 12)
    assert m.shape == (40, 300)
    assert normwise_rel(m, quant.matmul_exact(raw, 12, 300, 512, v)) < 1e-3


def test_native_quant_cache_reuses_immutable_weights():
    from localai_amd import native_quant as nq
    rng = np.random.default_rng(10)
    raw = random_ggml(rng, 14, 128 * 512)   # bytes: immutable
    x = rng.standard_normal(512).astype(np.float32)
    nq.clear_cache()
    y1 = nq.matvec(raw, x, 128, 512, 14)
    assert len(nq._cache) == 1
    y2 = nq.matvec(raw, x, 128, 512, 14)
    assert len(nq._cache) == 1
    np.testing.assert_array_equal(y1, y2)
    mutable = bytearray(raw)               # writable: never cached
    y3 = nq.matvec(mutable, x, 128, 512, 14)
    np.testing.assert_array_equal(y1, y3)
    assert len(nq._cache) == 1
    mutable[208:210] = np.float16(0.0).tobytes()   # change the scale of block 0 of row 0
    y4 = nq.matvec(mutable, x, 128, 512, 14)
    assert y4[0] != y1[0]
    nq.clear_cache()


# ------------------------------------------------------ legacy C exports


def _legacy(lib, name, raw, x, rows, cols, tokens=None):
    u8p, f32p = ctypes.POINTER(ctypes.c_uint8), ctypes.POINTER(ctypes.c_float)
    rawa = np.frombuffer(raw, dtype=np.uint8)
    xa = np.ascontiguousarray(x, dtype=np.float32)
    if tokens is None:
        out = np.empty(rows, np.float32)
        getattr(lib, f'localai_{name}_matvec')(rawa.ctypes.data_as(u8p), xa.ctypes.data_as(f32p),
                                               out.ctypes.data_as(f32p), rows, cols, 4)
    else:
        out = np.empty((rows, tokens), np.float32)
        getattr(lib, f'localai_{name}_matmul')(rawa.ctypes.data_as(u8p), xa.ctypes.data_as(f32p),
                                               out.ctypes.data_as(f32p), rows, cols, tokens, 4)
    assert lib.localai_hip_last_status() == 0, lib.localai_hip_last_error()
    return out


@pytest.mark.parametrize('name,t', [('q8_0', 8), ('q4_0', 2), ('q4k', 12), ('q5k', 13), ('q6k', 14)])
def test_legacy_exports(name, t):
    from localai_amd import _lib
    lib = _lib.load()
    rng = np.random.default_rng(t)
    rows, cols = 300, 512
    raw = random_ggml(rng, t, rows * cols)
    x = rng.standard_normal(cols).astype(np.float32)
    got = _legacy(lib, name, raw, x, rows, cols)
    assert normwise_rel(got, quant.matvec_exact(raw, t, rows, cols, x)) < 1e-5
    v = rng.standard_normal((5, cols)).astype(np.float32)
    got = _legacy(lib, name, raw, v, rows, cols, tokens=5)        # [rows, tokens]
    assert normwise_rel(got.T, quant.matmul_exact(raw, t, rows, cols, v)) < 1e-5
    v = rng.standard_normal((33, cols)).astype(np.float32)       # MFMA GEMM path
    got = _legacy(lib, name, raw, v, rows, cols, tokens=33)
    assert normwise_rel(got.T, quant.matmul_exact(raw, t, rows, cols, v)) < 1e-3


def test_legacy_registered_range_uses_cached_copy():
    from localai_amd import _lib
    lib = _lib.load()
    rng = np.random.default_rng(21)
    rows, cols = 256, 1024
    buf = np.frombuffer(bytearray(random_ggml(rng, 12, rows * cols)), dtype=np.uint8)
    x = rng.standard_normal(cols).astype(np.float32)
    assert lib.localai_hip_register_host(ctypes.c_void_p(buf.ctypes.data), buf.size) == 0
    y1 = _legacy(lib, 'q4k', buf, x, rows, cols)
    y2 = _legacy(lib, 'q4k', buf, x, rows, cols)
    np.testing.assert_array_equal(y1, y2)
    assert normwise_rel(y1, quant.matvec_exact(buf.tobytes(), 12, rows, cols, x)) < 1e-5
    assert lib.localai_hip_unregister_host(ctypes.c_void_p(buf.ctypes.data)) == 0
    assert lib.localai_hip_unregister_host(ctypes.c_void_p(buf.ctypes.data)) == 1
    assert lib.localai_hip_cache_clear() == 0


@pytest.mark.parametrize('t,rows,cols', [(12, 14336, 4096), (14, 4096, 14336), (14, 1024, 4096), (8, 512, 4096)])
def test_repeated_launches_are_bit_identical(t, rows, cols):
    """The waves of a workgroup meet in LDS in a fixed order (no atomics), so
    30 back-to-back launches at the Llama-3-8B shapes must give identical bits."""
    import torch
    from localai_amd import device, synth
    rng = np.random.default_rng(77)
    raw = synth.quant_tensor(rng, t, rows, cols)
    x = device.to_device_f32(synth.activations(rng, cols))
    q = device.QMat.from_ggml(raw, t, rows, cols)
    outs = [q.matvec(x) for _ in range(30)]
    torch.cuda.synchronize()
    first = outs[0].cpu().numpy()
    for o in outs[1:]:
        np.testing.assert_array_equal(o.cpu().numpy().view(np.uint32), first.view(np.uint32))
    assert normwise_rel(first, quant.matvec_exact(raw, t, rows, cols, x.cpu().numpy())) < 1e-5


@pytest.mark.parametrize('t,rows,cols', [(12, 5 * 64, 16384), (14, 7 * 64 - 3, 14336), (12, 9 * 64, 8192),
                                         (8, 13 * 64 + 1, 8192), (14, 3 * 64, 4096), (12, 17 * 64, 4096)])
def test_tile_counts_not_multiple_of_xcds(t, rows, cols):
    """Row-tile counts that are not multiples of the 8 XCDs and long rows (up
    to 64 super-blocks, the 768-thread plan): each launch matches the oracle
    and every launch gives the same bits."""
    import torch
    from localai_amd import device, synth
    rng = np.random.default_rng(rows + cols)
    raw = synth.quant_tensor(rng, t, rows, cols)
    xh = synth.activations(rng, cols)
    x = device.to_device_f32(xh)
    q = device.QMat.from_ggml(raw, t, rows, cols)
    outs = [q.matvec(x) for _ in range(40)]
    torch.cuda.synchronize()
    first = outs[0].cpu().numpy()
    assert normwise_rel(first, quant.matvec_exact(raw, t, rows, cols, xh)) < 1e-5
    for o in outs[1:]:
        np.testing.assert_array_equal(o.cpu().numpy().view(np.uint32), first.view(np.uint32))


@pytest.mark.parametrize('shapes', [
    # attn_q / attn_k / attn_v of a Q4_K_M decode step (v in Q6_K): one mixed launch
    [(12, 512, 4096), (12, 128, 4096), (14, 128, 4096)],
    # the same mix with the Q6_K job first and ragged Q4_K jobs: their
    # workgroups take two tiles each, the last one only one (63 and 4 tiles)
    [(14, 77, 4096), (12, 1000, 4096), (12, 53, 4096)],
    # ffn_gate / ffn_up shape family, ragged rows, long K (768-thread plan)
    [(12, 100, 14336), (14, 37, 14336)],
    # a matrix without a tile form (Q8_0) runs beside the fused Q4_K / Q6_K launch
    [(8, 64, 2048), (14, 200, 2048), (12, 1, 2048), (12, 33, 2048)],
    # two Q4_K matrices of one shape with the paired-tile launch (tile i of
    # each per workgroup) and, singly, the two-tile plan: ragged last tile
    [(12, 12300, 4096), (12, 12300, 4096)],
])
def test_matvec_many_matches_single(shapes):
    """localai_hip_matvec_many gives bit-identical results to one matvec per
    matrix (the same per-tile arithmetic), and both match the oracle."""
    from localai_amd import device
    rng = np.random.default_rng(len(shapes) * 1000 + shapes[0][1])
    cols = shapes[0][2]
    x = rng.standard_normal(cols).astype(np.float32)
    raws = [random_ggml(rng, t, rows * cols) for t, rows, _ in shapes]
    mats = [device.QMat.from_ggml(r, t, rows, cols) for r, (t, rows, _) in zip(raws, shapes)]
    xd = device.to_device_f32(x)
    try:
        fused = [o.cpu().numpy() for o in device.matvec_many(mats, xd)]
        single = [m.matvec(xd).cpu().numpy() for m in mats]
    finally:
        for m in mats:
            m.close()
    for (t, rows, _), raw, f, s in zip(shapes, raws, fused, single):
        np.testing.assert_array_equal(f, s)
        assert normwise_rel(f, quant.matvec_exact(raw, t, rows, cols, x)) < 1e-5


def test_matvec_many_experts_and_errors():
    """Expert selection per job, and the argument checks of the fused entry."""
    from localai_amd import _lib, device
    rng = np.random.default_rng(77)
    E, rows, cols = 3, 48, 1024
    raw = random_ggml(rng, 14, E * rows * cols)
    m = device.QMat.from_ggml(raw, 14, rows, cols, batch=E)
    other = device.QMat.from_ggml(random_ggml(rng, 12, rows * 512), 12, rows, 512)
    x = rng.standard_normal(cols).astype(np.float32)
    xd = device.to_device_f32(x)
    try:
        outs = device.matvec_many([m, m], xd, experts=[2, 0])
        per = rows * cols * 210 // 256
        for o, e in zip(outs, (2, 0)):
            ref = quant.matvec_exact(raw[e * per:(e + 1) * per], 14, rows, cols, x)
            assert normwise_rel(o.cpu().numpy(), ref) < 1e-5
        with pytest.raises(ValueError):
            device.matvec_many([m, other], xd)
        lib = _lib.load()
        h = (ctypes.c_void_p * 1)(m.handle.value)
        ex = (ctypes.c_int64 * 1)(E)
        ys = (ctypes.c_void_p * 1)(device.ptr(outs[0]))
        assert lib.localai_hip_matvec_many(1, h, ex, device.ptr(xd), ys, None) != 0
        assert lib.localai_hip_matvec_many(9, h, None, device.ptr(xd), ys, None) != 0
    finally:
        m.close()
        other.close()


@pytest.mark.parametrize('group', [
    # ffn_gate / ffn_up of one Llama-3-8B decode step (engine/model.py:232): the
    # two-matrix Q4_K launch of the decode-layer benchmark
    [('ffn_gate', 12, 14336, 4096), ('ffn_up', 12, 14336, 4096)],
    # attn_q / attn_k / attn_v (engine/model.py:185-187), Q4_K / Q4_K / Q6_K
    [('attn_q', 12, 4096, 4096), ('attn_k', 12, 1024, 4096), ('attn_v', 14, 1024, 4096)],
])
def test_matvec_many_llama3_8b_groups(group):
    """The fused launches of the decode-layer benchmark at their exact shapes
    and input distributions: each output bit-identical to a single-matrix
    launch and within 1e-5 normwise of the fp64 oracle."""
    from localai_amd import device, synth
    rng = np.random.default_rng(2024 + len(group))
    cols = group[0][3]
    raws = [synth.quant_tensor(rng, t, rows, cols) for _, t, rows, _ in group]
    x = synth.activations(rng, cols)
    mats = [device.QMat.from_ggml(r, t, rows, cols) for r, (_, t, rows, _) in zip(raws, group)]
    xd = device.to_device_f32(x)
    try:
        fused = [o.cpu().numpy() for o in device.matvec_many(mats, xd)]
        single = [m.matvec(xd).cpu().numpy() for m in mats]
    finally:
        for m in mats:
            m.close()
    for (name, t, rows, _), raw, f, s in zip(group, raws, fused, single):
        np.testing.assert_array_equal(f.view(np.uint32), s.view(np.uint32), err_msg=name)
        err = normwise_rel(f, quant.matvec_exact(raw, t, rows, cols, x))
        assert err < 1e-5, f'{name}: {err}'


@pytest.mark.parametrize('t', (12, 13))
def test_deviation_from_avx2_is_the_int8_activation_error(golden, t):
    """The reference's AVX2 Q4_K / Q5_K matvecs quantise x to int8 per 32
    values (engine/native_quant.cpp:84-109, :183-278); the GPU keeps x exact.
    Reported, not gated to the AVX2 output: on the reference test-suite case
    (300 x 512, tests/test_dequant.py:202-216) the GPU differs from the
    reference's own output by about 6e-3 (Q4_K) / 7e-3 (Q5_K) normwise, and
    that difference is the activation-quantisation term: GPU - AVX2 equals
    exact - (oracle model of the int8 activations) to within 1e-3 of its size."""
    raw, x = golden[f'raw_{t}'].tobytes(), golden[f'x_{t}']
    got = gpu_matvec(raw, t, 300, 512, x)
    avx2 = golden[f'matvec_{t}']
    exact = quant.matvec_exact(raw, t, 300, 512, x)
    model = quant.q8_activation_matvec(raw, t, 300, 512, x)
    dev = normwise_rel(got, avx2)
    print(f'type {t}: GPU vs reference AVX2 normwise {dev:.3e}; GPU vs exact {normwise_rel(got, exact):.2e}')
    assert 2e-3 < dev < 2e-2
    assert normwise_rel(got - avx2, exact - model) < 1e-3


def test_deviation_from_avx2_at_ffn_gate_size():
    """Q4_K 14336 x 4096 (the single-matvec workload): the GPU against the
    reference's own AVX2 kernel built from source (oracle/_ref), reported as
    above. Skipped where the reference library or AVX2 is absent."""
    from oracle import ref
    from localai_amd import synth
    if not ref.available():
        pytest.skip('reference library not built')
    if ' avx2 ' not in open('/proc/cpuinfo').read():
        pytest.skip('host without AVX2')
    rng = np.random.default_rng(11)
    raw = synth.quant_tensor(rng, 12, 14336, 4096)
    x = synth.activations(rng, 4096)
    got = gpu_matvec(raw, 12, 14336, 4096, x)
    avx2 = ref.matvec(raw, x, 14336, 4096, 12, threads=8)
    exact = quant.matvec_exact(raw, 12, 14336, 4096, x)
    model = quant.q8_activation_matvec(raw, 12, 14336, 4096, x)
    dev = normwise_rel(got, avx2)
    print(f'Q4_K 14336x4096: GPU vs reference AVX2 normwise {dev:.3e}; GPU vs exact {normwise_rel(got, exact):.2e}; '
          f'AVX2 vs exact {normwise_rel(avx2, exact):.3e}')
    assert dev < 2e-2
    assert normwise_rel(got - avx2, exact - model) < 1e-3
