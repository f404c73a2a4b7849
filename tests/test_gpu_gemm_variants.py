"""GPU parity of every gemm16 wave tile (osh_config_set("gemm_variant", v)) and
of the LDS-staged tile (v = -2) against the oracle's FMA-chain GEMM, on shapes
that exercise partial row/column tiles, K tails shorter than one chunk, padded
leading dimensions, row bias, column scale and fused activations.  Every tile
sums k in order with one rounding per product, so outputs must be
bit-identical to the chain (and within the conftest tolerance, relative 1e-4,
absolute 1e-5, in any case)."""
import ctypes as C

import numpy as np
import pytest

from conftest import assert_fp32_close
from onnxsharp_amd import synth

pytestmark = pytest.mark.gpu


def _t(x, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev)


def _variants():
    from onnxsharp_amd import native as N
    n = C.c_int()
    N.call("osh_config_get", b"gemm_variants", C.byref(n))
    return [-2] + list(range(n.value))


@pytest.fixture()
def variant_reset():
    yield
    from onnxsharp_amd import native as N
    N.call("osh_config_set", b"gemm_variant", -1)


# (m, k, n, lda_pad, ldc_pad): K tails shorter than a chunk, K < 4, partial tiles in both directions
CASES = [(1024, 768, 768, 0, 0), (70, 36, 96, 0, 0), (33, 4, 8, 0, 0), (5, 13, 132, 3, 4),
         (200, 100, 260, 4, 8), (97, 64, 36, 0, 0)]


def _gemm(cuda, m, k, n, lda, ldc, a, b, col_bias=None, row_bias=None, col_scale=None, act=0):
    import torch
    from onnxsharp_amd import native as N
    a_pad = np.zeros((m, lda), np.float32)
    a_pad[:, :k] = a
    da, db = _t(a_pad, cuda), _t(b, cuda)
    dc = torch.full((m, ldc), 7.0, dtype=torch.float32, device=cuda)
    ptr = lambda t: C.c_void_p(t.data_ptr()) if t is not None else None
    keep = [_t(x, cuda) if x is not None else None for x in (col_bias, row_bias, col_scale)]
    N.call("osh_gemm_f32", m, n, k, ptr(da), lda, ptr(db), n, ptr(keep[0]), ptr(keep[1]), ptr(keep[2]), act,
           ptr(dc), ldc, C.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    out = dc.cpu().numpy()
    assert (out[:, n:] == 7.0).all(), "wrote past n into the padding of C"
    return out[:, :n]


@pytest.mark.parametrize("m,k,n,lpad,cpad", CASES)
def test_gemm_variants_column_bias(cuda, oracle, variant_reset, m, k, n, lpad, cpad):
    from onnxsharp_amd import native as N
    a = synth.uniform(m * 7 + k, (m, k), -1, 1)
    b = synth.uniform(n * 5 + k, (k, n), -1, 1)
    bias = synth.uniform(m + n, (n,), -1, 1)
    ref = oracle.gemm_f32(a, b, col_bias=bias)
    for v in _variants():
        print(f"gemm variant {v}: m={m} k={k} n={n} lda=k+{lpad} ldc=n+{cpad}", flush=True)
        N.call("osh_config_set", b"gemm_variant", v)
        y = _gemm(cuda, m, k, n, k + lpad, n + cpad, a, b, col_bias=bias)
        assert_fp32_close(y, ref, f"variant {v} gemm {m}x{k}x{n}")
        assert np.array_equal(y, ref), f"variant {v} gemm {m}x{k}x{n}: not bit-identical"


@pytest.mark.parametrize("m,k,n,off", [(1, 1, 1, 1), (17, 31, 2, 1), (16, 33, 47, 3), (33, 65, 49, 2), (35, 97, 131, 1)])
def test_gemm_variants_ragged_rows(cuda, oracle, variant_reset, m, k, n, off):
    """Odd rows at odd addresses: one chain of fmafs, bit for bit, and nothing
    of what surrounds the operands (NaN here: a leading dimension's padding,
    the floats before and after) reaches the result."""
    import torch
    from onnxsharp_amd import native as N
    a = synth.uniform(m * 11 + k, (m, k), -1, 1)
    b = synth.uniform(n * 3 + k, (k, n), -1, 1)
    res = synth.uniform(m + n + k, (n,), -1, 1)
    lda, ldb, ldc = k + off, n + off, n + 1

    def held(x, ld):  # NaN around and between the rows
        buf = np.full((off + x.shape[0] * ld + 80,), np.nan, np.float32)
        buf[off:off + x.shape[0] * ld].reshape(-1, ld)[:, :x.shape[1]] = x
        return _t(buf, cuda)

    da, db, bias = held(a, lda), held(b, ldb), _t(res, cuda)
    at = lambda t, o: C.c_void_p(t.data_ptr() + 4 * o)
    ref = oracle.gemm_f32(a, b, col_bias=res)
    for v in _variants()[1:] + [-1]:
        print(f"gemm variant {v}: m={m} k={k} n={n} offset={off}", flush=True)
        N.call("osh_config_set", b"gemm_variant", v)
        dc = torch.full((off + m * ldc,), 7.0, dtype=torch.float32, device=cuda)
        N.call("osh_gemm_f32", m, n, k, at(da, off), lda, at(db, off), ldb, at(bias, 0), None, None, 0, at(dc, off),
               ldc, C.c_void_p(torch.cuda.current_stream().cuda_stream))
        y = dc.cpu().numpy()
        assert (y[:off] == 7.0).all() and (y[off:].reshape(m, ldc)[:, n:] == 7.0).all(), "wrote past n"
        assert np.array_equal(y[off:].reshape(m, ldc)[:, :n], ref), f"variant {v}: not bit-identical"


@pytest.mark.parametrize("m,k,n", [(17, 33, 5), (35, 19, 50), (16, 65, 67), (33, 70, 131)])
def test_gemm_variants_ragged_epilogues(cuda, oracle, variant_reset, m, k, n):
    """Rows that end inside a lane's columns through every epilogue of every
    tile: column scale and bias, a residual (a 1x1 conv's; the lanes of a row's
    end write some columns twice), and batches at odd strides."""
    import torch
    from onnxsharp_amd import native as N
    from onnxsharp_amd.layers import ConvLayer
    batch = 3
    a = synth.uniform(m * 13 + k, (batch, m, k), -1, 1)
    b = synth.uniform(n * 17 + k, (batch, k, n), -1, 1)
    cs, cb = synth.uniform(m + n, (n,), 1e-3, 1e-1), synth.uniform(m + k, (n,), -1, 1)
    rb, res = synth.uniform(n + k, (m,), -1, 1), synth.uniform(m + n + k, (batch, m, n), -1, 1)
    st = lambda: C.c_void_p(torch.cuda.current_stream().cuda_stream)
    ptr = lambda t: C.c_void_p(t.data_ptr())
    ref_scale = oracle.relu(oracle.gemm_f32(a[0], b[0], col_bias=cb, col_scale=cs))
    ref_batch = np.stack([oracle.gemm_f32(a[i], b[i], col_bias=cb) for i in range(batch)])
    ref_conv = np.stack([oracle.gemm_f32(a[0], b[i], row_bias=rb) + res[i] for i in range(batch)])

    def strided(x, stride):
        buf = np.full((x.shape[0], stride), np.nan, np.float32)
        buf[:, :x[0].size] = x.reshape(x.shape[0], -1)
        return _t(buf, cuda)

    sa, sb, sc = m * k + 1, k * n + 3, m * n + 1
    da, db, dcb = strided(a, sa), strided(b, sb), _t(cb, cuda)
    layer = ConvLayer(group=1, strides=[1, 1], pads=[0] * 4)
    dx, dw, drb, dres = (_t(v, cuda) for v in (b.reshape(batch, k, 1, n), a[0].reshape(m, k, 1, 1), rb,
                                               res.reshape(batch, m, 1, n)))
    for v in _variants() + [-1]:
        print(f"gemm variant {v}: ragged epilogues m={m} k={k} n={n}", flush=True)
        N.call("osh_config_set", b"gemm_variant", v)
        y = _gemm(cuda, m, k, n, k, n + 1, a[0], b[0], col_bias=cb, col_scale=cs, act=N.ACT_RELU)
        assert np.array_equal(y, ref_scale), f"variant {v}: column scale"
        dc = torch.full((batch, sc), 7.0, device=cuda)
        N.call("osh_gemm_f32_batched", batch, m, n, k, ptr(da), k, sa, ptr(db), n, sb, ptr(dcb), 0, ptr(dc), n, sc, st())
        y = dc.cpu().numpy()
        assert np.array_equal(y[:, :m * n].reshape(batch, m, n), ref_batch) and (y[:, m * n:] == 7.0).all(), \
            f"variant {v}: batch"
        p, packed = layer.prepack_weights((batch, k, 1, n), dw)
        dy = torch.full((batch, m, 1, n), 7.0, device=cuda)
        N.call("osh_conv2d_add_f32", C.byref(p), ptr(dx), ptr(packed), ptr(drb), N.ACT_NONE, ptr(dres), ptr(dy), st())
        assert np.array_equal(dy.cpu().numpy().reshape(batch, m, n), ref_conv), f"variant {v}: residual"


def test_gemm_variants_row_bias_silu_and_column_scale(cuda, oracle, variant_reset):
    from onnxsharp_amd import native as N
    m, k, n = 128, 256, 640
    a = synth.uniform(301, (m, k), -1, 1)
    b = synth.uniform(302, (k, n), 0, 1)
    rb = synth.normal(303, (m,), 0, 0.1)
    cs = synth.uniform(304, (n,), 1e-3, 1e-1)
    cb = synth.uniform(305, (n,), -1, 1)
    ref_silu = oracle.silu_ref(oracle.gemm_f32(a, b, row_bias=rb))
    ref_scale = oracle.relu(oracle.gemm_f32(a, b, col_bias=cb, col_scale=cs))
    N.call("osh_config_set", b"exact_silu", 1)
    try:
        for v in _variants():
            print(f"gemm variant {v}: row bias + SiLU, column scale + Relu", flush=True)
            N.call("osh_config_set", b"gemm_variant", v)
            y = _gemm(cuda, m, k, n, k, n, a, b, row_bias=rb, act=N.ACT_SILU)
            assert_fp32_close(y, ref_silu, f"variant {v} row bias + silu")
            assert np.array_equal(y, ref_silu), f"variant {v} row bias + silu: not bit-identical"
            y = _gemm(cuda, m, k, n, k, n, a, b, col_bias=cb, col_scale=cs, act=N.ACT_RELU)
            assert_fp32_close(y, ref_scale, f"variant {v} column scale + relu")
            assert np.array_equal(y, ref_scale), f"variant {v} column scale + relu: not bit-identical"
    finally:
        N.call("osh_config_set", b"exact_silu", 0)


def test_gemm_variants_batched_broadcast(cuda, oracle, variant_reset):
    import torch
    from onnxsharp_amd import native as N
    batch, m, k, n = 3, 40, 72, 64
    a = synth.uniform(311, (batch, m, k), -1, 1)
    b = synth.uniform(312, (k, n), -1, 1)  # broadcast over the batch (stride 0)
    bias = synth.uniform(313, (n,), -1, 1)
    ref = np.stack([oracle.gemm_f32(a[i], b, col_bias=bias) for i in range(batch)])
    da, db, dbias = _t(a, cuda), _t(b, cuda), _t(bias, cuda)
    for v in _variants():
        print(f"gemm variant {v}: batched {batch}x{m}x{k}x{n}", flush=True)
        N.call("osh_config_set", b"gemm_variant", v)
        dc = torch.empty((batch, m, n), dtype=torch.float32, device=cuda)
        N.call("osh_gemm_f32_batched", batch, m, n, k, C.c_void_p(da.data_ptr()), k, m * k,
               C.c_void_p(db.data_ptr()), n, 0, C.c_void_p(dbias.data_ptr()), 0, C.c_void_p(dc.data_ptr()), n,
               m * n, C.c_void_p(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert_fp32_close(dc.cpu().numpy(), ref, f"variant {v} batched")
        assert np.array_equal(dc.cpu().numpy(), ref), f"variant {v} batched: not bit-identical"


def test_gemm_variant_option_range():
    from onnxsharp_amd import native as N
    with pytest.raises(N.OshError):
        N.call("osh_config_set", b"gemm_variant", 1000)


@pytest.mark.parametrize("batch,m,k,n,kc", [
    (1, 1946, 448, 2560, 32), (1, 207, 448, 5376, 32), (14, 436, 128, 436, 32), (1, 1881, 300, 7796, 32),  # 3 to 20 waves a SIMD
    (1, 16, 3566, 1223, 64), (1, 4, 3040, 4960, 64),  # a few waves, each waiting for memory
])
def test_gemm_chunk_length_rule(cuda, batch, m, k, n, kc):
    """64-k chunks hide a wave's own trips to memory and are for products of few
    waves: where a SIMD has several, the tile is one of 32-k chunks."""
    import torch
    from onnxsharp_amd import native as N
    a, b, c = (torch.zeros(s, device=cuda) for s in ((batch, m, k), (batch, k, n), (batch, m, n)))
    ptr = lambda t: C.c_void_p(t.data_ptr())
    N.kernel_log(reset=True)
    N.call("osh_gemm_f32_batched", batch, m, n, k, ptr(a), k, m * k, ptr(b), n, k * n, None, 0, ptr(c), n, m * n,
           C.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    names = N.kernel_log(reset=True)
    assert len(names) == 1 and names[0].startswith("gemm16_kernel<") and int(names[0].split(",")[3]) == kc, names
