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
    (Q4_K, 5, 131073, 512), (Q4_K, 8, 65537, 768), (Q4_K, 6, 32769, 1280),  # one, two, four waves
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


@pytest.mark.parametrize("M,N,K,lanes", [
    (8, 33, 256, True), (6, 8223, 1024, True), (4, 8193, 1280, False), (5, 31, 2048, False),
    (8, 65, 11008, True), (7, 31, 16384, True), (6, 33, 16640, False)])
def test_slot_raw_lane_loads(orc, dev, M, N, K, lanes):
    """Q4_K rows too short a wave to pay for the way through LDS are loaded in the
    lane layout: up to one super-block a wave, two where K is split (from 25
    super-blocks on); stored, accumulated and with the ordered split."""
    import torch
    from inferflux_amd import ops, synth
    note(f"slot raw lane loads M={M} N={N} K={K}")
    w = synth.blocks(Q4_K, N, K, seed=N + K)
    a = orc.quantize_q8_1(synth.activations(M, K, seed=M + K, outlier_frac=0.01))
    W, A = up(w, dev), up(a, dev)
    ye = orc.gemv_exact(Q4_K, w, a, M, N, K)
    tt, T = ops.repack_tiled(Q4_K, W, N, K)
    ws = torch.zeros(max(256, ops.qgemv_workspace_bytes(Q4_K, [N], M, K)), dtype=torch.uint8, device=dev)
    with ops.launch_log() as lg:
        y = down(ops.qgemv(Q4_K, W, A, M, N, K))
        yo = down(ops.qgemv(Q4_K, W, A, M, N, K, workspace=ws))
    slot = [k for k in lg.kernels if k.startswith("k_gemv_slot<")]
    assert len(slot) == 2 and all(k.endswith(",0,0,1>") == lanes for k in slot), lg.kernels
    check_rows(y, ye)
    yt = down(ops.qgemv(tt, T, A, M, N, K, workspace=ws))
    assert np.array_equal(yo.view(np.uint32), yt.view(np.uint32))
    base = torch.full((M, N), 2.0, device=dev)
    check_rows(down(ops.qgemv(Q4_K, W, A, M, N, K, out=base, mode=ops.ACCUM)), ye + 2.0)
    y16 = down(ops.qgemv(Q4_K, W, A, M, N, K, out_dtype=torch.float16))
    bar = 2e-3 * np.linalg.norm(ye, axis=1, keepdims=True)
    assert np.all(np.abs(y16.astype(np.float64) - ye) <= bar)
