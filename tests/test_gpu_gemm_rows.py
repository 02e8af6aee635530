"""The streaming dequant-GEMM of up to 64 activation rows (csrc/gguf_gemm_rows.hip) on a GPU.

A group of matrices takes the kernel at any size, so the edges of its tiles, steps and slices are
tested there.  One-hot activations read single staged weights back exactly; random ones are checked
against fp16 operands and fp64 sums with fp32's summation bound.
"""

import numpy as np
import pytest

from oracle import gguf_ref as R
from tensor_amd.gguf import quant as Q
from tests import gguf_cases as cases

pytestmark = pytest.mark.gpu

ENCODINGS = ["q4_0", "q4_1", "q5_0", "q5_1", "q8_0", "q2_k", "q3_k", "q4_k", "q5_k", "q6_k"]


def group(device, encoding, x, raws):
    exe = device.load("gguf_gemm_group_noalloc", encoding=encoding, out_dtype="float32", count=len(raws))
    buffers = [device.from_numpy(a) for a in (x, *raws)]
    outs = [device.empty((x.shape[0], raw.shape[0]), "float32") for raw in raws]
    args = buffers[:1]
    for w, out in zip(buffers[1:], outs):
        device.fill_bytes(out, 0xFF)  # NaN
        args += [w, out]
    exe.launch(*args)
    result = [out.to_numpy() for out in outs]
    for b in buffers + outs:
        b.release()
    return result


def weights(encoding, raw, n, k):
    return R.dequantize(raw, Q.ggml_type(encoding), n, k).astype(np.float16)


def check(got, x, w, what):
    """Exact fp32 products of fp16 operands: K 2^-24 sum |x w| bounds any order of their sum."""
    xd, wd = x.astype(np.float16).astype(np.float64), w.astype(np.float64)
    bound = x.shape[1] * 2.0 ** -24 * (np.abs(xd) @ np.abs(wd).T) + 1e-12
    assert not np.isnan(got).any(), what
    assert (np.abs(got - xd @ wd.T) <= bound).all(), what


def check_sums(got, x, w, what):
    """Relative L2 against fp64: a sum rounds a few dozen times by at most 2^-24 of a partial sum, errors of
    independent signs (random terms), so 2^-20 leaves a factor of ten.  The last step of 256 columns is far more of the
    sums than that: a kernel that left it out would miss."""
    xd, wd = x.astype(np.float16).astype(np.float64), w.astype(np.float64)
    last, want = (x.shape[1] - 1) // 256 * 256, xd @ wd.T
    bound = 2.0 ** -20 * np.linalg.norm(want)
    assert np.linalg.norm(xd[:, last:] @ wd[:, last:].T) > 1000 * bound, what
    assert np.linalg.norm(got - want) <= bound, what


@pytest.mark.parametrize("encoding", ENCODINGS)
def test_one_hot_rows_give_the_fp16_weights(hip_device, encoding):
    lengths = (32, 96, 1056) if Q.GEOMETRY[Q.ggml_type(encoding)][0] == 32 else (256, 768)
    for k in lengths:
        rows = (70, 1)
        raws = [cases.random_blocks(encoding, n, k, 61 + i) for i, n in enumerate(rows)]
        for m in (16, 40):
            print("[gemm-rows] one-hot", encoding, m, k, flush=True)
            at = np.random.default_rng(62 + m).integers(0, k, m)
            x = np.zeros((m, k), np.float16)
            x[np.arange(m), at] = 1.0
            for got, raw, n in zip(group(hip_device, encoding, x, raws), raws, rows):
                assert np.array_equal(got, weights(encoding, raw, n, k).astype(np.float32)[:, at].T), (k, m, n)


@pytest.mark.parametrize("encoding", ENCODINGS)
@pytest.mark.parametrize("m", [9, 17, 33, 64])
def test_tiles_and_steps(hip_device, encoding, m):
    lengths = (288, 2592) if Q.GEOMETRY[Q.ggml_type(encoding)][0] == 32 else (512, 3328)
    for k in lengths:
        rows = (1, 17, 300)
        print("[gemm-rows] edges", encoding, m, rows, k, flush=True)
        raws = [cases.weight(n, k, encoding, 71 + i) for i, n in enumerate(rows)]
        x = cases.activation(m, k, 72)
        for got, raw, n in zip(group(hip_device, encoding, x, raws), raws, rows):
            check(got, x, weights(encoding, raw, n, k), (encoding, m, n, k))


@pytest.mark.parametrize("encoding,m,rows,k", [
    ("q8_0", 32, (48, 16), 16416),    # many slices, the last one short
    ("q4_k", 20, (12288, 40), 512),   # several row tiles per workgroup
    ("q6_k", 64, (24600, 33), 256),   # twelve tiles or 64 activation rows per workgroup, ragged
    ("q3_k", 50, (4100, 10), 768),    # activation rows over workgroups, a ragged last share
    ("q4_k", 48, (64, 64), 8192),     # narrow: no plan reaches its grid, the streaming kernel stays
])
def test_launch_shapes(hip_device, encoding, m, rows, k):
    print("[gemm-rows] shape", encoding, m, rows, k, flush=True)
    raws = [cases.weight(n, k, encoding, 81 + i) for i, n in enumerate(rows)]
    x = cases.activation(m, k, 82)
    for got, raw, n in zip(group(hip_device, encoding, x, raws), raws, rows):
        check(got, x, weights(encoding, raw, n, k), (encoding, m, n, k))
        check_sums(got, x, weights(encoding, raw, n, k), (encoding, m, n, k))


@pytest.mark.parametrize("encoding,m,k", [("q8_0", 32, 16416), ("q5_1", 64, 8224), ("q6_k", 40, 9472)])
def test_every_step_of_long_rows_is_multiplied_once(hip_device, encoding, m, k):
    """One-hot activations at the first and last column of every step of 256, so on both sides of every slice
    boundary and in the short last step: each output is one fp16 weight, exactly."""
    print("[gemm-rows] long rows, one-hot", encoding, m, k, flush=True)
    rows = (48, 16)
    raws = [cases.random_blocks(encoding, n, k, 85 + i) for i, n in enumerate(rows)]
    steps = range(0, k, 256)
    columns = sorted({*steps, *(min(s + 255, k - 1) for s in steps)})
    for first in range(0, len(columns), m):
        at = [columns[min(first + i, len(columns) - 1)] for i in range(m)]
        x = np.zeros((m, k), np.float16)
        x[np.arange(m), at] = 1.0
        for got, raw, n in zip(group(hip_device, encoding, x, raws), raws, rows):
            assert np.array_equal(got, weights(encoding, raw, n, k).astype(np.float32)[:, at].T), (n, at)


@pytest.mark.parametrize("encoding,m,n,k", [("q6_k", 2, 300, 768), ("q4_k", 33, 1030, 2560), ("q5_0", 64, 77, 1056)])
def test_packed_call_rounds_its_activations_to_fp16(hip_device, encoding, m, n, k):
    print("[gemm-rows] packed", encoding, m, n, k, flush=True)
    raw = cases.weight(n, k, encoding, 91)
    x = np.random.default_rng(92).standard_normal((m, k)).astype(np.float32)
    exe = hip_device.load("gguf_linear", encoding=encoding, m=m, n=n, k=k)
    xb, wb = hip_device.from_numpy(x.reshape(-1)), hip_device.from_numpy(raw.reshape(-1))
    out = hip_device.empty((m * n,), "float32")
    exe.launch(xb, wb, out)
    check(out.to_numpy().reshape(m, n), x, weights(encoding, raw, n, k), (encoding, m, n, k))
    for b in (xb, wb, out):
        b.release()
