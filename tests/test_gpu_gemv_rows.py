"""The matrix-core decode GEMV (csrc/gguf_gemv_rows.hip) through the entries that reach it, on a GPU.

A group of two or three matrices takes the kernel at any size (but the tuned M = 1 shapes), so the
edges of its tiles, steps, slices and launch shapes are tested there.  Every output is checked
against fp64 with the bound that any order of fp32 summation keeps, K * 2^-24 times the sum of the
terms' magnitudes.  A weight is the difference of a scaled code and a minimum, which the kernel sums apart:
each is at most twice the row's largest weight (the codes of a row span their range), so the terms
of element k are at most 3 max |w| |x[k]| together.
"""

import numpy as np
import pytest

from oracle import gguf_ref as R
from tensor_amd.gguf import quant as Q
from tests import gguf_cases as cases

pytestmark = pytest.mark.gpu

ENCODINGS = ["q4_0", "q4_1", "q5_0", "q5_1", "q8_0", "q2_k", "q3_k", "q4_k", "q5_k", "q6_k"]


def run(device, kernel, x, raws, encoding, rows, **options):
    exe = device.load(kernel, encoding=encoding, out_dtype="float32", **options)
    buffers = [device.from_numpy(a) for a in (x, *raws)]
    outs = [device.empty((x.shape[0], n), "float32") for n in rows]
    for out in outs:
        device.fill_bytes(out, 0xFF)  # NaN
    args = buffers[:1]
    if kernel == "gguf_gemv_group":
        for w, out in zip(buffers[1:], outs):
            args += [w, out]
    else:
        args = buffers + outs
    exe.launch(*args)
    result = [out.to_numpy() for out in outs]
    for b in buffers + outs:
        b.release()
    return result


def reference(x, raw, encoding, n, k):
    """(x W^T, its summation bound) in fp64."""
    w = R.dequantize(raw, Q.ggml_type(encoding), n, k).astype(np.float64)
    x = x.astype(np.float64)
    return x @ w.T, k * 2.0 ** -24 * 3 * np.abs(x).sum(1)[:, None] * np.abs(w).max(1)[None, :] + 1e-12


def check_sums(got, want, tail, what):
    """Relative L2 against fp64 of sums over random terms: each rounds a few dozen times by at most 2^-24 of a
    partial sum, errors of independent signs, so 2^-20 leaves a factor of ten.  tail, the part of the sums that the last
    step adds, is far more than that: a kernel that left it out would miss."""
    bound = 2.0 ** -20 * np.linalg.norm(want)
    assert np.linalg.norm(tail) > 1000 * bound, what
    assert np.linalg.norm(got - want) <= bound, what


def check(got, x, raw, encoding, n, k, what):
    want, bound = reference(x, raw, encoding, n, k)
    assert not np.isnan(got).any(), what
    over = np.abs(got - want) > bound
    assert not over.any(), (what, int(over.sum()), float(np.abs(got - want).max()))


def note(*what):
    print("[gemv-rows]", *what, flush=True)


@pytest.mark.parametrize("encoding", ENCODINGS)
@pytest.mark.parametrize("source", ["quantized", "random_bits"])
def test_every_encoding_at_the_edges_of_tiles_and_steps(hip_device, encoding, source):
    """One row, a ragged tile and several tiles; rows of one block, of a part of a step, of whole
    steps and of steps with a ragged last one (every block alignment); one to eight activation rows."""
    qk = Q.GEOMETRY[Q.ggml_type(encoding)][0]
    lengths = (32, 64, 96, 288, 1056, 2592) if qk == 32 else (256, 512, 768, 2304, 3328)
    rows = (1, 17, 100)
    for k in lengths:
        make = (lambda n, seed: cases.weight(n, k, encoding, seed)) if source == "quantized" else \
               (lambda n, seed: cases.random_blocks(encoding, n, k, seed))
        raws = [make(n, 11 + i) for i, n in enumerate(rows)]
        for m in (1, 2, 4, 5, 8):
            note(encoding, source, m, rows, k)
            x = cases.activation(m, k, 20 + m)
            for got, raw, n in zip(run(hip_device, "gguf_gemv_group", x, raws, encoding, rows, count=3), raws, rows):
                check(got, x, raw, encoding, n, k, (encoding, source, m, n, k))


@pytest.mark.parametrize("encoding,m,rows,k", [
    ("q8_0", 8, (33, 16), 16416),    # activations staged in slices, the last one short
    ("q2_k", 7, (48, 5), 24832),
    ("q4_k", 8, (16401, 7), 512),    # over 1024 tiles: four tiles per workgroup, 8 waves, a ragged last workgroup
    ("q6_k", 4, (16401, 7), 768),
    ("q4_0", 3, (4100, 4100), 320),  # three tiles per workgroup
    ("q5_k", 1, (8200, 40), 1280),   # four tiles per workgroup, three ranges of K
])
def test_launch_shapes(hip_device, encoding, m, rows, k):
    note("shape", encoding, m, rows, k)
    raws = [cases.weight(n, k, encoding, 31 + i) for i, n in enumerate(rows)]
    x = cases.activation(m, k, 33)
    last = (k - 1) // 256 * 256  # the last step's first column
    for got, raw, n in zip(run(hip_device, "gguf_gemv_group", x, raws, encoding, rows, count=2), raws, rows):
        check(got, x, raw, encoding, n, k, (encoding, m, n, k))
        w = R.dequantize(raw, Q.ggml_type(encoding), n, k).astype(np.float64)
        xd = x.astype(np.float64)
        check_sums(got, xd @ w.T, xd[:, last:] @ w[:, last:].T, (encoding, m, n, k))


@pytest.mark.parametrize("encoding,m,rows,k", [("q8_0", 8, (33, 16), 16416), ("q2_k", 7, (48, 5), 24832),
                                               ("q5_1", 5, (17, 1), 30752), ("q4_k", 6, (20, 3), 26880)])
def test_every_step_of_long_rows_is_multiplied_once(hip_device, encoding, m, rows, k):
    """Rows whose activations are staged in slices: one-hot activations at the first and last column of every step of
    256, so on both sides of every slice boundary and in the short last step.  An output is one weight, scale * code +
    low: at most eight roundings of terms that are together at most 3 max |w|."""
    note("long rows, one-hot", encoding, m, rows, k)
    raws = [cases.weight(n, k, encoding, 35 + i) for i, n in enumerate(rows)]
    ws = [R.dequantize(raw, Q.ggml_type(encoding), n, k).astype(np.float64) for raw, n in zip(raws, rows)]
    steps = range(0, k, 256)
    columns = sorted({*steps, *(min(s + 255, k - 1) for s in steps)})
    for first in range(0, len(columns), m):
        at = [columns[min(first + i, len(columns) - 1)] for i in range(m)]
        x = np.zeros((m, k), np.float16)
        x[np.arange(m), at] = 1.0
        for got, w in zip(run(hip_device, "gguf_gemv_group", x, raws, encoding, rows, count=2), ws):
            want, bound = w[:, at].T, 8 * 2.0 ** -24 * 3 * np.abs(w).max(1)[None, :]
            assert not np.isnan(got).any() and (np.abs(got - want) <= bound).all(), at
            assert (np.abs(want) > 1000 * bound).mean() > 0.5  # a step left out would be seen


@pytest.mark.parametrize("encoding,m,n,k", [("q4_0", 5, 4100, 1056), ("q8_0", 8, 4100, 1056), ("q3_k", 3, 1300, 2816),
                                            ("q6_k", 2, 1030, 2304), ("q5_0", 4, 1530, 3104), ("q4_k", 1, 300, 2304)])
def test_single_matrices(hip_device, encoding, m, n, k):
    """Sizes above the lines from which a single matrix takes the kernel."""
    note("single", encoding, m, n, k)
    raw, x = cases.weight(n, k, encoding, 41), cases.activation(m, k, 42)
    got, = run(hip_device, "gguf_gemv", x, [raw], encoding, (n,))
    check(got, x, raw, encoding, n, k, (encoding, m, n, k))


@pytest.mark.parametrize("encoding,m,n,k", [("q4_k", 2, 1, 256), ("q4_k", 3, 33, 4096), ("q4_k", 8, 300, 2816),
                                            ("q5_k", 1, 1000, 2304), ("q8_0", 6, 2100, 1056), ("q2_k", 4, 4130, 512)])
def test_swiglu_pairs(hip_device, encoding, m, n, k):
    """silu(g) * u of two bounded sums: the bound of the product's first-order terms, |silu'| <= 1.1,
    and 1e-5 of the result for the epilogue's own fp32 operations."""
    note("swiglu", encoding, m, n, k)
    gate, up = (cases.weight(n, k, encoding, 51 + i) for i in range(2))
    x = cases.activation(m, k, 53)
    got, = run(hip_device, "gguf_gemv_swiglu", x, [gate, up], encoding, (n,))
    (g, eg), (u, eu) = (reference(x, raw, encoding, n, k) for raw in (gate, up))
    want = R.silu(g) * u
    assert not np.isnan(got).any()
    assert (np.abs(got - want) <= 1.2 * eg * np.abs(u) + 1.2 * eu * np.abs(R.silu(g)) + 2 * eg * eu
            + 1e-5 * np.abs(want) + 1e-9).all()


@pytest.mark.parametrize("encoding", ENCODINGS)
def test_sums_keep_fp32_precision(hip_device, encoding):
    """Against fp64 over all outputs: sums in the precision of 16-bit exponent-aligned products would miss the
    bound of check_sums by another ten, as they would at activations that are all fp16 subnormals (2^-16 times normal ones)
    if those lost bits to their leading zeros."""
    m, rows, k = 3, (512, 512), 2560
    note("precision", encoding, m, rows, k)
    raws = [cases.weight(n, k, encoding, 77 + i) for i, n in enumerate(rows)]
    for scale in (1.0, 2.0 ** -16):
        x = (scale * np.random.default_rng(78).standard_normal((m, k))).astype(np.float16)
        for got, raw, n in zip(run(hip_device, "gguf_gemv_group", x, raws, encoding, rows, count=2), raws, rows):
            want, _ = reference(x, raw, encoding, n, k)
            check_sums(got, want, want, (encoding, scale))


def by_elements(x, w):
    """x W^T element by element: what an infinity or a NaN in either makes of each output."""
    with np.errstate(all="ignore"):
        return np.stack([(row.astype(np.float64) * w.astype(np.float64)).sum(1) for row in x])


def same_kind(got, want):
    return (np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want))
            and np.array_equal(np.isneginf(got), np.isneginf(want)))


@pytest.mark.parametrize("encoding", ["q4_1", "q5_0", "q5_1", "q2_k", "q3_k", "q5_k"])
@pytest.mark.parametrize("m", [1, 3, 8])
def test_infinities_and_nans_are_those_of_the_elements_products(hip_device, encoding, m):
    """An infinite activation gives infinities of the weights' signs (NaN at a zero weight, and for two that
    disagree), an infinite scale what its elements' products sum to; other rows stay as they are."""
    k, rows = 2592 if Q.GEOMETRY[Q.ggml_type(encoding)][0] == 32 else 2304, (200, 33)
    note("infinities", encoding, m, rows, k)
    raws = [cases.weight(n, k, encoding, 61 + i) for i, n in enumerate(rows)]
    size = Q.GEOMETRY[Q.ggml_type(encoding)][1]
    offset = cases.HALF_FIELDS[Q.ggml_type(encoding)][0]
    raws[1] = raws[1].copy()
    raws[1][5, 3 * size + offset:3 * size + offset + 2] = np.array([np.inf], np.float16).view(np.uint8)
    raws[1][32, offset:offset + 2] = np.array([np.nan], np.float16).view(np.uint8)
    with np.errstate(all="ignore"):
        weights = [R.dequantize(raw, Q.ggml_type(encoding), n, k) for raw, n in zip(raws, rows)]
    for special in ((np.inf,), (-np.inf,), (np.inf, np.inf), (np.nan,), ()):
        x = cases.activation(m, k, 63)
        for i, value in enumerate(special):
            x[0, 700 + 800 * i] = value
        group = run(hip_device, "gguf_gemv_group", x, raws, encoding, rows, count=2)
        for got, w, n in zip(group, weights, rows):
            want = by_elements(x, w)
            assert same_kind(got, want), (encoding, m, n, special)
            finite = np.isfinite(want)
            with np.errstate(all="ignore"):
                bound = k * 2.0 ** -24 * 3 * np.abs(x.astype(np.float64)).sum(1)[:, None] * np.abs(w).max(1)[None, :] + 1e-12
            assert (np.abs(got[finite] - want[finite]) <= bound[finite]).all()
    # the SwiGLU pair takes its own two sums
    gate, up = cases.weight(4130, k, encoding, 65), cases.weight(4130, k, encoding, 66)
    x = cases.activation(m, k, 67)
    x[0, 700] = np.inf
    got, = run(hip_device, "gguf_gemv_swiglu", x, [gate, up], encoding, (4130,))
    g, u = (by_elements(x, R.dequantize(raw, Q.ggml_type(encoding), 4130, k)).astype(np.float32) for raw in (gate, up))
    with np.errstate(all="ignore"):
        want = g / (1 + np.exp(-g)) * u
    assert same_kind(got, want), (encoding, m)
