"""The order in which the prefill GEMM adds: on a tile whose waves do not split
K, an output is the sum over K in steps of 16 values, one MFMA each, so its
bits do not depend on the tile's shape.  The checksums are those of the
256 x 256 tile with fp16 weights in LDS that served every prefill shape
before the tiles of today, on the same inputs."""
import zlib

import numpy as np
import pytest

from tests.test_gpu_parity import check_rows, down, note, up

pytestmark = pytest.mark.gpu

Q8_0, Q4_K, Q6_K = 8, 12, 14
M, N = 512, 27648


@pytest.fixture(scope="module")
def dev():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


# (type, K, checksum of the fp32 outputs, of the fp16 ones); Q8_0 also with a K
# that is no multiple of 256
GOLD = [(Q4_K, 512, 0x25fd91cd, 0x8b23f6a5), (Q6_K, 512, 0xc761892f, 0xff7b19bb),
        (Q8_0, 512, 0x99d9f1d9, 0x8e5e78eb), (Q8_0, 448, 0xf13335c7, 0x85cfd41c)]


@pytest.mark.parametrize("qtype,K,crc32,crc16", GOLD)
def test_sums_run_over_k_in_order(orc, dev, qtype, K, crc32, crc16):
    import torch
    from inferflux_amd import ops, synth
    note(f"prefill order type={qtype} M={M} N={N} K={K}")
    w = synth.blocks(qtype, N, K, seed=5)
    a = orc.quantize_q8_1(synth.activations(M, K, seed=6, outlier_frac=0.01))
    W, A = up(w, dev), up(a, dev)
    y = down(ops.qgemm_prefill_kernel(qtype, W, A, M, N, K, ops.PREFILL_F16))
    idx = np.arange(0, N, 31)
    check_rows(y[:, idx], orc.gemv_exact(qtype, w[idx], a, M, len(idx), K))
    assert zlib.crc32(y.tobytes()) == crc32
    y = down(ops.qgemm_prefill_kernel(qtype, W, A, M, N, K, ops.PREFILL_F16,
                                      out_dtype=torch.float16))
    assert zlib.crc32(y.tobytes()) == crc16


# Long prompts' narrow projections (K and V), fp16
@pytest.mark.parametrize("qtype,N,K,crc", [
    (Q4_K, 1024, 512, 0x567f4461), (Q4_K, 1024, 5120, 0x2351e596),
    (Q6_K, 1024, 512, 0xdf22c5d3), (Q6_K, 1024, 2560, 0x7367ad3b)])
def test_long_prompt_sums_run_over_k_in_order(orc, dev, qtype, N, K, crc):
    import torch
    from inferflux_amd import ops, synth
    note(f"prefill order type={qtype} M=1999 N={N} K={K}")
    w = synth.blocks(qtype, N, K, seed=5)
    a = orc.quantize_q8_1(synth.activations(1999, K, seed=6, outlier_frac=0.01))
    y = ops.qgemm_prefill_kernel(qtype, up(w, dev), up(a, dev), 1999, N, K, ops.PREFILL_F16,
                                 out_dtype=torch.float16)
    assert zlib.crc32(down(y).tobytes()) == crc
