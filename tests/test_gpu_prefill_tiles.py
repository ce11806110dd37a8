"""The fp16 prefill GEMM over the tile shapes its plan chooses from (32 x 64 to
128 x 512 and 256 x 256): sizes at the edges of a tile and one past them, ragged K ends
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


# (M, N, K): the smallest tile and one past its edges, K of one super-block, K
# ends inside a group of K waves, then sizes wide enough for each larger tile
# (32 x 128, 64 x 128, 64 x 256, 96 x 256, 128 x 256, 128 x 512 or 256 x 256).
# test_prefill_splits.py checks which tiles these reach.
SHAPES = [(33, 64, 256), (64, 65, 512), (96, 63, 768), (65, 8201, 1280), (257, 4100, 512),
          (100, 22016, 512), (191, 22017, 768), (256, 22016, 256), (385, 22020, 512),
          (513, 33000, 256)]
# and a long prompt's 64 x 128 tile in order (Q4_K, Q6_K).
LONG = (1025, 1030, 512)
# Q8_0 takes any K of whole 64-value chunks: one, and odd counts
CASES = [(t, M, N, K) for t in (Q4_K, Q6_K) for M, N, K in SHAPES + [LONG]] + \
    [(Q8_0, M, N, K - 64 * (M % 2) - 128 * (K > 256)) for M, N, K in SHAPES] + \
    [(Q8_0, 35, 70, 64), (Q8_0, 300, 11009, 64)]


@pytest.mark.parametrize("qtype,M,N,K", CASES)
def test_prefill_tiles(orc, dev, qtype, M, N, K):
    import torch
    from inferflux_amd import ops, synth
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


# fp16 outputs do not split K; of the fp32 ones the first three do, into
# outputs that the launch before clears
GROUPED = [
    (Q4_K, 130, (512, 64, 65), 2048, False), (Q6_K, 40, (1000, 33), 4096, False),
    (Q8_0, 130, (300, 64, 65), 2048, False),
    (Q4_K, 130, (300, 64, 65), 512, False), (Q4_K, 600, (2048, 256, 256), 256, True),
    (Q6_K, 40, (1000, 1), 1024, False), (Q8_0, 129, (77, 500, 31), 768, True),
    (Q8_0, 300, (4097, 4096), 256, False),
]


@pytest.mark.parametrize("qtype,M,Ns,K,f16", GROUPED)
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
    assert lg.kernels[-1].startswith("k_gemm_f16<"), lg.kernels
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


# The fp16 copy of the activations (wide projections with a workspace), and
# K splits of the wider tiles: added with atomics, or in order
@pytest.mark.parametrize("qtype,M,N,K", [
    (Q4_K, 96, 16387, 256), (Q4_K, 96, 18432, 1280), (Q4_K, 200, 27648, 512), (Q4_K, 100, 49152, 256),
    (Q6_K, 33, 16384, 256), (Q6_K, 33, 18435, 768), (Q6_K, 66, 49152, 256), (Q6_K, 129, 49152, 256),
    (Q8_0, 128, 16384, 320), (Q8_0, 128, 18432, 192), (Q8_0, 129, 22020, 64), (Q8_0, 129, 49152, 256),
])
def test_prefill_workspace(orc, dev, qtype, M, N, K):
    import torch
    from inferflux_amd import ops, synth
    note(f"prefill workspace type={qtype} M={M} N={N} K={K}")
    w = synth.blocks(qtype, N, K, seed=N + K)
    a = orc.quantize_q8_1(synth.activations(M, K, seed=M + K, outlier_frac=0.01))
    W, A = up(w, dev), up(a, dev)
    ws = torch.empty(ops.prefill_workspace_bytes(qtype, M, N, K), dtype=torch.uint8, device=dev)
    with ops.launch_log() as lg:
        y = ops.qgemm_prefill_ws(qtype, W, A, M, N, K, ws)
    assert lg.kernels[0] == "k_q8_1_to_f16" and lg.kernels[-1].endswith(",1>"), lg.kernels
    assert torch.equal(y, ops.qgemm_prefill_kernel(qtype, W, A, M, N, K, ops.PREFILL_F16))
    idx = np.unique(np.concatenate([[0, 31, N - 1], np.random.default_rng(N).choice(N, 96)]))
    check_rows(down(y)[:, idx], orc.gemv_exact(qtype, w[idx], a, M, len(idx), K))


@pytest.mark.parametrize("qtype,M,N,K", [
    (Q4_K, 96, 1025, 5120), (Q4_K, 100, 2052, 13824), (Q6_K, 65, 1536, 8192), (Q6_K, 100, 1030, 13824),
    (Q8_0, 129, 4100, 4160), (Q8_0, 128, 1027, 11008),
])
def test_prefill_wide_splits(orc, dev, qtype, M, N, K):
    import torch
    from inferflux_amd import ops, synth
    note(f"prefill wide splits type={qtype} M={M} N={N} K={K}")
    w = synth.blocks(qtype, N, K, seed=N + K)
    a = orc.quantize_q8_1(synth.activations(M, K, seed=M + K, outlier_frac=0.01))
    W, A = up(w, dev), up(a, dev)
    idx = np.unique(np.concatenate([[0, N - 1], np.random.default_rng(N).choice(N, 96)]))
    ye = orc.gemv_exact(qtype, w[idx], a, M, len(idx), K)
    with ops.launch_log() as lg:
        y = ops.qgemm_prefill_kernel(qtype, W, A, M, N, K, ops.PREFILL_F16)
    assert lg.kernels[0] == "k_fill_zero" and ",1,0>" in lg.kernels[1], lg.kernels
    check_rows(down(y)[:, idx], ye)
    ws = torch.empty(ops.prefill_ordered_workspace_bytes(qtype, M, N, K), dtype=torch.uint8,
                     device=dev)
    y = torch.full((M, N), 1.0, device=dev)
    with ops.launch_log() as lg:
        ops.qgemm_prefill_ordered(qtype, W, A, M, N, K, ws, out=y, mode=ops.ACCUM)
    assert ",2,0>" in lg.kernels[0] and lg.kernels[1] == "k_split_sum", lg.kernels
    check_rows(down(y)[:, idx], ye + 1.0)


# Rows that do not start on 16 bytes, on tiles with one, two, four and eight K waves
@pytest.mark.parametrize("qtype,M,N,K", [
    (Q4_K, 130, 16385, 256), (Q4_K, 743, 16385, 512), (Q6_K, 600, 12290, 512), (Q6_K, 300, 6146, 512), (Q6_K, 65, 4101, 256),
    (Q8_0, 600, 12290, 512), (Q8_0, 257, 8201, 320), (Q8_0, 129, 1027, 192), (Q4_K, 97, 70, 256),
])
@pytest.mark.parametrize("f16", [False, True])
def test_prefill_unaligned_rows(orc, dev, qtype, M, N, K, f16):
    """Stored, added to what is there, and with a bias: the same sums each time."""
    import torch
    from inferflux_amd import ops, synth
    note(f"prefill unaligned rows type={qtype} M={M} N={N} K={K} f16={f16}")
    w = synth.blocks(qtype, N, K, seed=N + K)
    a = orc.quantize_q8_1(synth.activations(M, K, seed=M + K, outlier_frac=0.01))
    W, A, f = up(w, dev), up(a, dev), ops.PREFILL_F16
    dt = torch.float16 if f16 else torch.float32
    y = ops.qgemm_prefill_kernel(qtype, W, A, M, N, K, f, splits=1)
    idx = np.unique(np.concatenate([[0, 31, 32, N - 1], np.random.default_rng(N).choice(N, min(N, 96))]))
    check_rows(down(y)[:, idx], orc.gemv_exact(qtype, w[idx], a, M, len(idx), K))
    rng = torch.Generator().manual_seed(N)
    base = torch.randn(M, N, generator=rng).to(dt).to(dev)
    bias = torch.randn(N, generator=rng).to(dt).to(dev)
    got = ops.qgemm_prefill_kernel(qtype, W, A, M, N, K, f, splits=1, out_dtype=dt)
    assert torch.equal(got, y.to(dt))  # one rounding of the same fp32 sum
    got = ops.qgemm_prefill_kernel(qtype, W, A, M, N, K, f, splits=1, out=base.clone(), mode=ops.ACCUM)
    assert torch.equal(got, (y + base.float()).to(dt))
    got = ops.qgemm_prefill_kernel(qtype, W, A, M, N, K, f, splits=1, out_dtype=dt, mode=ops.BIAS, bias=bias)
    assert torch.equal(got, (y + bias.float()).to(dt))
