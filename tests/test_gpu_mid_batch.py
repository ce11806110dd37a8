"""Batches between the decode and the fp16 prefill kernels on the int8 MFMA
GEMM: one to four wave groups a tile with fewer, as many and more super-blocks
than groups, ragged last tiles, and up to three projections in one launch;
within 1e-3 * ||y_row||_2 of the fp64 oracle, the bar of the decode tests
(2e-3 for fp16 outputs, whose rounding is 2^-11 of the largest value)."""
import numpy as np
import pytest

from tests.test_gpu_parity import check_rows, down, note, up

pytestmark = pytest.mark.gpu

Q4_K, Q8_0 = 12, 8


@pytest.fixture(scope="module")
def dev():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


# The bar is a part of a row's norm: Q4_K's fp16 activation sums alone are
# 2^-11 of each min term off, which a row of a few outputs can fall short of,
# so a Q4_K row has 63 outputs or more here (Q8_0 has no such term).
# 64 x 64 tiles: up to 256 (four groups), 512 (two), more (one), and one with few
# super-blocks; 512 large tiles with a batch of 64 and less stay on small ones
CASES = [
    (Q4_K, 33, (63,), 256), (Q4_K, 64, (65, 63, 64), 768), (Q4_K, 65, (200, 130), 1280),
    (Q4_K, 95, (300,), 2048), (Q4_K, 40, (16389,), 512), (Q4_K, 64, (11000, 11009), 768),
    (Q4_K, 34, (32800,), 256), (Q4_K, 60, (65473,), 256), (Q4_K, 66, (65473,), 256),
    (Q8_0, 33, (1, 2, 3), 256), (Q8_0, 127, (513, 64), 1280), (Q8_0, 64, (65,), 768),
    (Q8_0, 63, (16500,), 4096), (Q8_0, 63, (16500,), 512), (Q8_0, 50, (65473,), 256),
    (Q4_K, 64, (11000, 11009), 1280), (Q4_K, 40, (16389,), 1280), (Q8_0, 100, (8300,), 4352),
]


@pytest.mark.parametrize("qtype,M,Ns,K", CASES)
def test_mid_batch(orc, dev, qtype, M, Ns, K):
    import torch
    from inferflux_amd import ops, synth
    note(f"mid batch type={qtype} M={M} N={Ns} K={K}")
    ws = [synth.blocks(qtype, N, K, seed=N + K + i) for i, N in enumerate(Ns)]
    a = orc.quantize_q8_1(synth.activations(M, K, seed=M + K, outlier_frac=0.01))
    Ws, A = [up(w, dev) for w in ws], up(a, dev)
    rng = np.random.default_rng(M)
    idx = [np.unique(np.concatenate([[0, N - 1], rng.choice(N, min(N, 96))])) for N in Ns]
    want = [orc.gemv_exact(qtype, w[i], a, M, len(i), K) for w, i in zip(ws, idx)]
    with ops.launch_log() as lg:
        ys = ops.qgemv_grouped(qtype, Ws, A, M, list(Ns), K)
    assert len(lg.kernels) == 1 and lg.kernels[0].startswith("k_gemm_mfma<"), lg.kernels
    for y, i, e in zip(ys, idx, want):
        check_rows(down(y)[:, i], e)
    again = ops.qgemv_grouped(qtype, Ws, A, M, list(Ns), K)
    assert all(torch.equal(p, q) for p, q in zip(ys, again))
    base = [rng.standard_normal((M, N)).astype(np.float32) for N in Ns]
    ys = ops.qgemv_grouped(qtype, Ws, A, M, list(Ns), K, outs=[up(b, dev) for b in base],
                           mode=ops.ACCUM)
    for y, b, i, e in zip(ys, base, idx, want):
        check_rows(down(y)[:, i], e + b[:, i])
    y = ops.qgemv(qtype, Ws[0], A, M, Ns[0], K, out_dtype=torch.float16)
    check_rows(down(y)[:, idx[0]].astype(np.float64), want[0], tol=2e-3)
    bias = rng.standard_normal(Ns[0]).astype(np.float32)
    y = ops.qgemv(qtype, Ws[0], A, M, Ns[0], K, mode=ops.BIAS, bias=up(bias, dev))
    check_rows(down(y)[:, idx[0]], want[0] + bias[None, idx[0]])
