"""The slot-packed decode GEMV on raw rows, whose super-blocks are loaded along
the rows and turned into the lane layout in LDS: last row groups of 1, 31 and
32 rows, one super-block and more than the waves, the fused gate/up form; the
same bits as on the tiled copy (the same sums in the same order), and within
1e-3 * ||y_row||_2 of the fp64 oracle, the bar of the decode tests."""
import numpy as np
import pytest

from tests.test_gpu_parity import check_rows, down, note, up

pytestmark = pytest.mark.gpu

Q4_K, Q6_K = 12, 14


@pytest.fixture(scope="module")
def dev():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


@pytest.mark.parametrize("qtype,M,N,K", [
    (Q4_K, 4, 1, 256), (Q4_K, 8, 33, 2048), (Q4_K, 5, 8223, 512), (Q6_K, 5, 8192, 256),
    (Q6_K, 8, 8225, 768), (Q4_K, 6, 63, 2304), (Q6_K, 7, 31, 1024),
    (Q6_K, 8, 1000, 2048), (Q6_K, 4, 33, 6144),  # eight waves: LDS past 64 KB
])
def test_slot_raw_rows(orc, dev, qtype, M, N, K):
    from inferflux_amd import ops, synth
    note(f"slot raw type={qtype} M={M} N={N} K={K}")
    w = synth.blocks(qtype, N, K, seed=N + K)
    a = orc.quantize_q8_1(synth.activations(M, K, seed=M + K, outlier_frac=0.01))
    W, A = up(w, dev), up(a, dev)
    with ops.launch_log() as lg:
        y = down(ops.qgemv(qtype, W, A, M, N, K))
    assert lg.kernels[0].startswith("k_gemv_slot<"), lg.kernels
    check_rows(y, orc.gemv_exact(qtype, w, a, M, N, K))
    tt, T = ops.repack_tiled(qtype, W, N, K)
    yt = down(ops.qgemv(tt, T, A, M, N, K))
    assert np.array_equal(y.view(np.uint32), yt.view(np.uint32))


@pytest.mark.parametrize("qtype,M,N,K", [(Q4_K, 3, 32, 256), (Q6_K, 8, 96, 1280)])
def test_slot_raw_gate_up(orc, dev, qtype, M, N, K):
    from inferflux_amd import ops, synth
    note(f"slot raw gate/up type={qtype} M={M} N={N} K={K}")
    wg, wu = synth.blocks(qtype, N, K, seed=1), synth.blocks(qtype, N, K, seed=2)
    a = orc.quantize_q8_1(synth.activations(M, K, seed=3))
    G, U, A = up(wg, dev), up(wu, dev), up(a, dev)
    h, q = ops.qgemv_gate_up_silu(qtype, G, U, A, M, N, K)
    tt, Gt = ops.repack_tiled(qtype, G, N, K)
    Ut = ops.repack_tiled(qtype, U, N, K)[1]
    ht, qt = ops.qgemv_gate_up_silu(tt, Gt, Ut, A, M, N, K)
    assert np.array_equal(down(h).view(np.uint32), down(ht).view(np.uint32))
    assert np.array_equal(down(q), down(qt))
