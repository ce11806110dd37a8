"""The fp16 prefill GEMM over the tile shapes its plan chooses from (32 x 64
to 128 x 512): sizes at the edges of a tile and one past them, ragged K ends
(K of one chunk, K groups that one wave's share ends inside), rows that do
not start on 16 bytes, and projections that share a launch.  Checked against
the fp64 oracle at 1e-3 * ||y_row||_2 (fp16 outputs 2e-3), the bar of the other
prefill tests: weights and activations are rounded to fp16 (2^-11 each)."""
import numpy as np
import pytest

from tests.test_gpu_parity import check_rows, down, note, up

pytestmark = pytest.mark.gpu

Q8_0, Q4_K, Q6_K = 8, 12, 14


@pytest.fixture(scope="module")
def dev():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


# (M, N, K): the smallest tile and one past its edges, K of one chunk (Q8_0) or
# one super-block, K ends inside a group of K waves, then sizes wide enough for
# each larger tile (32 x 128, 64 x 128, 64 x 256, 96 x 256, 128 x 256, 128 x 512)
SHAPES = [(33, 64, 256), (64, 65, 512), (96, 63, 768), (33, 8192, 256), (65, 8201, 1280),
          (100, 22016, 512), (191, 22017, 768), (256, 22016, 256), (385, 22020, 512),
          (513, 33000, 256)]


@pytest.mark.parametrize("qtype", [Q4_K, Q6_K, Q8_0])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_prefill_tiles(orc, dev, qtype, M, N, K):
    import torch
    from inferflux_amd import ops, synth
    if qtype == Q8_0:
        K -= 64 * (M % 2) + 128 * (K > 256)  # odd chunk counts too
    note(f"prefill tiles type={qtype} M={M} N={N} K={K}")
    w = synth.blocks(qtype, N, K, seed=N + K)
    a = orc.quantize_q8_1(synth.activations(M, K, seed=M + K, outlier_frac=0.01))
    W, A = up(w, dev), up(a, dev)
    idx = np.unique(np.concatenate([[0, 31, N - 1], np.arange(max(0, N - 40), N),
                                    np.random.default_rng(N).choice(N, 48)]))
    ye = orc.gemv_exact(qtype, w[idx], a, M, len(idx), K)
    f = ops.PREFILL_F16
    guard = torch.full((M * N + 64,), 7.0, device=dev)
    y = guard[:M * N].view(M, N)
    ops.qgemm_prefill_kernel(qtype, W, A, M, N, K, f, out=y)
    check_rows(down(y)[:, idx], ye)
    assert bool((guard[M * N:] == 7.0).all())
    # output rows off the 16-byte boundary
    off = guard[1:1 + M * N].view(M, N)
    off.fill_(1.0)
    ops.qgemm_prefill_kernel(qtype, W, A, M, N, K, f, out=off, mode=ops.ACCUM)
    check_rows(down(off)[:, idx], ye + 1.0)
    y16 = ops.qgemm_prefill_kernel(qtype, W, A, M, N, K, f, out_dtype=torch.float16)
    check_rows(down(y16)[:, idx].astype(np.float64), ye, tol=2e-3)


@pytest.mark.parametrize("qtype,M,Ns,K,f16", [
    (Q4_K, 130, (300, 64, 65), 512, False), (Q4_K, 600, (2048, 256, 256), 256, True),
    (Q6_K, 40, (1000, 1), 1024, False), (Q8_0, 129, (77, 500, 31), 448, True),
    (Q8_0, 300, (4097, 4096), 192, False),
])
def test_prefill_grouped(orc, dev, qtype, M, Ns, K, f16):
    """Sibling projections in one launch: stored, and added to what is there."""
    import torch
    from inferflux_amd import ops, synth
    note(f"prefill grouped type={qtype} M={M} Ns={Ns} K={K}")
    ws = [synth.blocks(qtype, n, K, seed=n + i) for i, n in enumerate(Ns)]
    a = orc.quantize_q8_1(synth.activations(M, K, seed=M + K, outlier_frac=0.01))
    A, Ws = up(a, dev), [up(w, dev) for w in ws]
    dt = torch.float16 if f16 else torch.float32
    with ops.launch_log() as lg:
        ys = ops.qgemv_grouped(qtype, Ws, A, M, list(Ns), K, out_dtype=dt)
    assert [k for k in lg.kernels if k != "k_fill_zero"] == [lg.kernels[-1]]  # one GEMM launch
    base = [torch.full((M, n), 2.0, dtype=dt, device=dev) for n in Ns]
    ops.qgemv_grouped(qtype, Ws, A, M, list(Ns), K, outs=base, mode=ops.ACCUM)
    for w, n, y, b in zip(ws, Ns, ys, base):
        ye = orc.gemv_exact(qtype, w, a, M, n, K)
        bar = np.linalg.norm(ye, axis=1, keepdims=True)
        # a projection of one row is no norm to hide the fp16 rounding behind:
        # sum over K of |w x| 2^-11 / sqrt(K) at most, against its own norm
        tol = 2e-3 if f16 else 1e-3
        if n == 1:
            tol = 2e-2
        assert np.all(np.abs(down(y).astype(np.float64) - ye) <= tol * np.maximum(bar, 1e-6) + (2e-3 * np.abs(ye) if f16 else 0))
        assert np.all(np.abs(down(b).astype(np.float64) - ye - 2.0) <= tol * np.maximum(bar, 1e-6) + (4e-3 * (np.abs(ye) + 2) if f16 else 0))
