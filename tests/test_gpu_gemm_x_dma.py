"""The 256 x 128 prefill tile with its activations by LDS DMA (csrc/gguf_gemm_pipe.h) on a GPU: the
shortest K its loop runs and an odd number of step pairs, ragged rows and columns, every encoding.
fp16 operands and fp64 sums, fp32's summation bound."""

import numpy as np
import pytest

from oracle import gguf_ref as R
from tensor_amd.gguf import quant as Q
from tests import gguf_cases as cases

pytestmark = pytest.mark.gpu

ENCODINGS = ["q4_0", "q4_1", "q5_0", "q5_1", "q8_0", "q2_k", "q3_k", "q4_k", "q5_k", "q6_k"]


@pytest.mark.parametrize("encoding", ENCODINGS)
@pytest.mark.parametrize("pairs", [1, 3])
def test_ragged_tiles(hip_device, encoding, pairs):
    # 110 column tiles by two row tiles: one round of 256 x 128 tiles against two of 256 x 96
    m, n = 300, 14000
    k = pairs * (128 if Q.GEOMETRY[Q.ggml_type(encoding)][0] == 32 else 256)
    print("[gemm-x-dma]", encoding, m, n, k, flush=True)
    raw, x = cases.weight(n, k, encoding, 51), cases.activation(m, k, 52)
    exe = hip_device.load("gguf_gemm_group_noalloc", encoding=encoding, out_dtype="float32", count=1)
    xb, wb, out = hip_device.from_numpy(x), hip_device.from_numpy(raw), hip_device.empty((m, n), "float32")
    hip_device.fill_bytes(out, 0xFF)
    exe.launch(xb, wb, out)
    got = out.to_numpy()
    for b in (xb, wb, out):
        b.release()
    w = R.dequantize(raw, Q.ggml_type(encoding), n, k).astype(np.float16).astype(np.float64)
    xd = x.astype(np.float64)
    assert not np.isnan(got).any()
    assert (np.abs(got - xd @ w.T) <= k * 2.0 ** -24 * (np.abs(xd) @ np.abs(w).T) + 1e-12).all(), (encoding, k)
