"""GPU parity of MatMulInteger (MatMulIntegerLayer, src/OnnxSharp/Ops/QuantOps.cs:235-428):
int32 accumulators bit-exact against the oracle's int64 sum of
(a - a_zp)(b - b_zp[col]), for u8 and s8 activations and weights, scalar and
per-column weight zero points, and the reference's known answer."""
import json
import os

import numpy as np
import pytest

from onnxsharp_amd import synth

pytestmark = pytest.mark.gpu


def _t(x, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev)


def test_matmul_integer_known_answer(cuda):
    from onnxsharp_amd.layers import MatMulIntegerLayer
    g = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "known_answers.json")))["matmul_integer"]
    a = np.array(g["a"], np.uint8)
    b = np.array(g["b"], np.uint8)
    y = MatMulIntegerLayer().forward(_t(a, cuda), _t(b, cuda)).cpu().numpy()
    assert y.tolist() == g["c"]


CASES = [
    (5, 17, 33, "u8", 0, "u8", None),
    (64, 64, 64, "u8", 37, "s8", "scalar"),
    (70, 96, 45, "s8", -5, "s8", "column"),
    (33, 260, 130, "s8", 0, "u8", "column"),
    (256, 512, 2048, "u8", 128, "s8", None),
    (1, 40, 7, "u8", 255, "u8", "column"),
]


@pytest.mark.parametrize("m,k,n,adt,azp,bdt,bzp", CASES)
def test_matmul_integer_parity(cuda, oracle, m, k, n, adt, azp, bdt, bzp):
    from onnxsharp_amd.layers import MatMulIntegerLayer
    print(f"matmulinteger m={m} k={k} n={n} A {adt} zp {azp} B {bdt} zp {bzp}", flush=True)
    seed = m + 3 * k + 7 * n
    lo, hi, dt = (0, 255, np.uint8) if adt == "u8" else (-128, 127, np.int8)
    a = synth.randint(seed, (m, k), lo, hi, dt)
    lo, hi, dt = (0, 255, np.uint8) if bdt == "u8" else (-128, 127, np.int8)
    b = synth.randint(seed + 1, (k, n), lo, hi, dt)
    zps = None
    base = 128 if bdt == "u8" else 0  # a zero point has the weights' element type
    if bzp == "scalar":
        zps = [base + int(synth.randint(seed + 2, (1,), -20, 20, np.int32)[0])]
    elif bzp == "column":
        zps = [base + int(v) for v in synth.randint(seed + 2, (n,), -20, 20, np.int32)]
    y = MatMulIntegerLayer().forward(_t(a, cuda), _t(b, cuda), [azp], zps).cpu().numpy()
    ref = oracle.matmul_integer(a, b, azp, None if zps is None else np.array(zps, np.int32))
    assert y.dtype == np.int32
    assert np.array_equal(y, ref), f"max |d| {np.abs(y.astype(np.int64) - ref).max()}"


@pytest.mark.parametrize("m,k,n,offset,adt", [
    (1, 1, 5, 0, "u8"), (1, 2, 33, 1, "s8"), (3, 1, 7, 2, "u8"), (1, 4, 9, 3, "s8"),  # A of 1 to 4 bytes
    (2, 31, 40, 1, "u8"), (33, 33, 65, 3, "s8"), (32, 64, 129, 0, "u8"), (32, 64, 129, 8, "u8"),  # odd rows, odd bases
    (65, 130, 33, 2, "s8"), (31, 257, 70, 0, "u8"), (5, 288, 40, 0, "s8"),  # two stages and one k-step more
    (2047, 2050, 40, 1, "u8"), (1028, 96, 6500, 0, "u8"),  # many workgroups; 64-row tiles
])
def test_matmul_integer_any_address(cuda, oracle, m, k, n, offset, adt):
    """Activations at every byte offset and row length: the bytes before and
    after them (all ones) reach no sum."""
    import torch
    from onnxsharp_amd.layers import MatMulIntegerLayer
    print(f"matmulinteger m={m} k={k} n={n} offset={offset} A {adt}", flush=True)
    dt, lo, hi = (np.uint8, 0, 255) if adt == "u8" else (np.int8, -128, 127)
    a = synth.randint(m + k, (m, k), lo, hi, dt)
    b = synth.randint(n + k, (k, n), -128, 127, np.int8)
    buf = torch.full((offset + m * k + 64,), -1, dtype=torch.int8, device=cuda)
    buf[offset:offset + m * k] = _t(a.view(np.int8).reshape(-1), cuda)
    da = buf[offset:offset + m * k].view(torch.uint8 if adt == "u8" else torch.int8).view(m, k)
    assert da.is_contiguous() and da.data_ptr() == buf.data_ptr() + offset
    y = MatMulIntegerLayer().forward(da, _t(b, cuda), [7]).cpu().numpy()
    assert np.array_equal(y, oracle.matmul_integer(a, b, 7))


def test_matmul_integer_batch1_3d_and_errors(cuda, oracle):
    from onnxsharp_amd import native as N
    from onnxsharp_amd.layers import MatMulIntegerLayer
    a = synth.randint(11, (1, 9, 20), 0, 255, np.uint8)
    b = synth.randint(12, (20, 6), -128, 127, np.int8)
    y = MatMulIntegerLayer().forward(_t(a, cuda), _t(b, cuda), [3]).cpu().numpy()
    assert y.shape == (1, 9, 6)
    assert np.array_equal(y[0], oracle.matmul_integer(a[0], b, 3))
    with pytest.raises(N.OshError, match="K mismatch"):
        MatMulIntegerLayer().forward(_t(a[0], cuda), _t(b[:5], cuda))
