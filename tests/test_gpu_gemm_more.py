"""The pipelined prefill GEMM of Q4_1, Q5_0, Q5_1, Q2_K and Q3_K (csrc/gguf_gemm_pipe_more.hip) on a GPU.

One-hot activations read single staged weights back, so every code, scale, minimum, high bit and
position is compared exactly (fp16 of the fp32 dequantization); random activations cover the tiles
against the prefill numerics (fp16 operands, fp64 sums) with fp32's summation bound.
"""

import numpy as np
import pytest

from oracle import gguf_ref as R
from tensor_amd.gguf import quant as Q
from tests import gguf_cases as cases

pytestmark = pytest.mark.gpu

ENCODINGS = ["q4_1", "q5_0", "q5_1", "q2_k", "q3_k"]


def group(device, encoding, x, raws):
    rows = [raw.shape[0] for raw in raws]
    exe = device.load("gguf_gemm_group", encoding=encoding, out_dtype="float32", count=len(raws))
    need = device.gemm_workspace(encoding, x.shape[0], x.shape[1], rows)
    assert need == 0  # K is not split across workgroups
    buffers = [device.from_numpy(a) for a in (x, *raws)]
    outs = [device.empty((x.shape[0], n), "float32") for n in rows]
    workspace = device.empty((256,), "uint8")
    args = buffers[:1]
    for w, out in zip(buffers[1:], outs):
        device.fill_bytes(out, 0xFF)
        args += [w, out]
    exe.launch(*args, workspace)
    result = [out.to_numpy() for out in outs]
    for b in buffers + outs + [workspace]:
        b.release()
    return result


@pytest.mark.parametrize("encoding", ENCODINGS)
@pytest.mark.parametrize("k,n", [(256, 70), (768, 70), (1024, 4200)])  # 64 x 64, unsplit and split K; wider tiles
def test_one_hot_rows_give_the_fp16_weights(hip_device, encoding, k, n):
    print("[gemm-more] one-hot", encoding, k, n, flush=True)
    raw = cases.random_blocks(encoding, n, k, 81)
    x = np.zeros((k, k), np.float16)
    order = np.random.default_rng(82).permutation(k)
    x[np.arange(k), order] = 1.0
    got, = group(hip_device, encoding, x, [raw])
    want = R.dequantize(raw, Q.ggml_type(encoding), n, k).astype(np.float16).astype(np.float32)
    assert np.array_equal(got, want[:, order].T)


@pytest.mark.parametrize("encoding", ENCODINGS)
@pytest.mark.parametrize("m,k,rows", [(65, 256, (33, 1)), (100, 1024, (300, 70)), (129, 1280, (8300,)),
                                      (300, 512, (2000, 1000, 64)), (520, 256, (12288,))])
def test_tiles_against_the_prefill_numerics(hip_device, encoding, m, k, rows):
    print("[gemm-more] tiles", encoding, m, k, rows, flush=True)
    x = cases.activation(m, k, 91)
    raws = [cases.weight(n, k, encoding, 92 + i) for i, n in enumerate(rows)]
    for got, raw, n in zip(group(hip_device, encoding, x, raws), raws, rows):
        w = R.dequantize(raw, Q.ggml_type(encoding), n, k).astype(np.float16).astype(np.float64)
        xd = x.astype(np.float64)
        # exact fp32 products of fp16 operands: K 2^-24 sum |x w| bounds any order of their sum
        bound = k * 2.0 ** -24 * (np.abs(xd) @ np.abs(w).T) + 1e-12
        assert not np.isnan(got).any()
        assert (np.abs(got - xd @ w.T) <= bound).all()


@pytest.mark.parametrize("encoding", ENCODINGS)
@pytest.mark.parametrize("units", [2, 3, 5, 7])  # K in pairs of steps or super-blocks: shares of 1-2 over 2 or 4 wave groups
def test_uneven_shares_of_k(hip_device, encoding, units):
    k = units * (128 if Q.GEOMETRY[Q.ggml_type(encoding)][0] == 32 else 256)
    for m, rows in ((100, (70, 33)), (333, (2560,)), (140, (12000,))):
        print("[gemm-more] uneven", encoding, m, k, rows, flush=True)
        x = cases.activation(m, k, 95)
        raws = [cases.weight(n, k, encoding, 96 + i) for i, n in enumerate(rows)]
        for got, raw, n in zip(group(hip_device, encoding, x, raws), raws, rows):
            w = R.dequantize(raw, Q.ggml_type(encoding), n, k).astype(np.float16).astype(np.float64)
            xd = x.astype(np.float64)
            bound = k * 2.0 ** -24 * (np.abs(xd) @ np.abs(w).T) + 1e-12
            assert not np.isnan(got).any()
            assert (np.abs(got - xd @ w.T) <= bound).all(), (encoding, m, n, k)
