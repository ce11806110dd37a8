"""K splits and tiles of the fp16 prefill GEMM, planned on the host: the ordered
entry asks for no more workspace than the documented line (a grid of 256 x 256 tiles, 512 values of
K a split), so a buffer sized for a shape once stays large enough, and a
shape that never split still runs without one; and the GPU tests' shapes reach
every tile."""
import ctypes
import itertools

import pytest
import torch

from inferflux_amd import ops

Q4_K, Q6_K, Q8_0 = 12, 14, 8


def _line(M, N, K):
    tiles = -(-M // 256) * -(-N // 256)
    n64 = K // 64
    sp = max(1, min(256 // tiles, n64 // 8)) if tiles < 192 else 1
    sp = -(-n64 // -(-n64 // sp))
    return sp * M * N * 4 if sp > 1 else 0


@pytest.mark.parametrize("qt", [Q4_K, Q6_K, Q8_0])
def test_ordered_workspace_within_the_line(qt):
    Ms = [128, 173, 256, 257, 512, 1024, 1999]
    Ns = [1, 64, 300, 512, 2048, 5120, 13824, 27648, 49152, 151936]
    Ks = [256, 512, 2048, 5120, 13824, 27648]
    for M, N, K in itertools.product(Ms, Ns, Ks):
        need = ops.prefill_ordered_workspace_bytes(qt, M, N, K)
        copy = ops.prefill_workspace_bytes(qt, M, N, K)
        line = _line(M, N, K)  # the slots follow the fp16 copy, 256-byte aligned
        assert need <= (-(-copy // 256) * 256 + line if line else copy), (M, N, K)
        assert ops.prefill_ordered_workspace_bytes(qt, M, N, K, torch.float16) <= copy


def _instances(call, qt, M, N, K, *more, f16=False):
    """Instances that an entry of one projection would launch."""
    p = [ctypes.c_void_p(0x100000 * (i + 1)) for i in range(4)]
    from inferflux_amd import _lib
    with ops.launch_log(dry=True) as lg:
        rc = getattr(_lib.load(), call)(qt, p[0], p[1], p[2], ops.OUT_F16 if f16 else ops.OUT_F32, ops.STORE, None, M, N, K,
                                        *[p[3] if m == "ws" else m for m in more], None)
    assert rc == 0
    return lg.instances


# 32-row and 32-column MFMA tiles, waves along the columns, waves along K
TILES = {(3, 2, 4, 2), (2, 2, 4, 2), (2, 2, 2, 4), (1, 2, 2, 4),
         (1, 2, 1, 8)}
LARGE = {Q4_K: {(4, 2, 8, 1), (4, 2, 4, 2)}, Q6_K: {(8, 1, 8, 1), (4, 1, 8, 1)},
         Q8_0: {(8, 1, 8, 1), (4, 2, 4, 2)}}
ORDERED = (2, 1, 4, 1)  # Q4_K, Q6_K


def _tile(name):
    return tuple(int(v) for v in name.split("[")[1][:-1].split(","))[:4]


@pytest.mark.parametrize("qt", [Q4_K, Q6_K, Q8_0])
def test_gpu_shapes_reach_every_tile(qt):
    from tests.test_gpu_prefill_tiles import CASES
    got = {_tile(_instances("ifx_qgemm_prefill_kernel", qt, M, N, K, ops.PREFILL_F16, 0)[-1])
           for t, M, N, K in CASES if t == qt}
    assert got == TILES | LARGE[qt] | (set() if qt == Q8_0 else {ORDERED})


@pytest.mark.parametrize("qt", [Q4_K, Q6_K])
@pytest.mark.parametrize("M,N,K", [(1999, 1024, 5120), (2048, 1024, 5120), (1025, 1030, 512),
                                   (1999, 5120, 5120), (1999, 13824, 5120)])
def test_long_prompts_sum_in_order(qt, M, N, K):
    """fp16 outputs of a long prompt's layer: no waves along K."""
    call = _instances("ifx_qgemm_prefill_kernel", qt, M, N, K, ops.PREFILL_F16, 0, f16=True)
    assert len(call) == 1 and _tile(call[0])[3] == 1, call


@pytest.mark.parametrize("qt,M,N,K", [(Q4_K, 1023, 1024, 5120), (Q4_K, 1999, 256, 2048),
                                      (Q6_K, 1999, 256, 2048), (Q8_0, 1999, 1024, 5120)])
def test_other_launches_keep_the_k_waves(qt, M, N, K):
    call = _instances("ifx_qgemm_prefill_kernel", qt, M, N, K, ops.PREFILL_F16, 0, f16=True)
    assert _tile(call[0])[3] > 1, call


@pytest.mark.parametrize("qt", [Q4_K, Q6_K, Q8_0])
def test_ordered_launches_use_no_atomics(qt):
    """The ordered entry splits into slots or not at all."""
    Ms, Ns, Ks = [128, 200, 300, 512, 1024, 1999], [1, 300, 1024, 2048, 5120, 11008, 27648], [512, 2048, 5120, 11008]
    split = 0
    for M, N, K in itertools.product(Ms, Ns, Ks):
        need = ops.prefill_ordered_workspace_bytes(qt, M, N, K)
        call = _instances("ifx_qgemm_prefill_ordered", qt, M, N, K, "ws", need)
        gemm = [k for k in call if k.startswith("k_gemm_f16<")]
        epi = gemm[0].split("<")[1].split(",")[3]
        assert len(gemm) == 1 and epi != "1" and "k_fill_zero" not in call, call
        assert (epi == "2") == ("k_split_sum" in call), call
        split += epi == "2"
    assert split > 40
    # wide enough for a split to gain in slots only
    call = _instances("ifx_qgemm_prefill_ordered", Q8_0, 200, 5120, 5120, "ws", 1 << 40)
    assert call[-1] == "k_split_sum"


@pytest.mark.parametrize("qt", [Q4_K, Q6_K, Q8_0])
def test_copy_ends_below_the_zero_offset(qt):
    """Chunks past K read zeros at byte 0xF0000000, so no fp16 copy reaches it."""
    N, K = 16384, 27648
    for M, copied in ((72810, 1), (72817, 1), (72819, 0), (72900, 0), (77000, 0)):
        assert (2 * M * K < 0xF0000000) == bool(copied)
        nbytes = ops.prefill_workspace_bytes(qt, M, N, K)
        assert nbytes == 2 * M * K  # what a caller hands over does not change
        call = _instances("ifx_qgemm_prefill_ws", qt, M, N, K, "ws", nbytes)
        assert call[-1].split("[")[0].endswith(f",{copied}>"), call
        assert ("k_q8_1_to_f16" in call) == bool(copied)


@pytest.mark.parametrize("qt,M,N,K,groups", [
    (Q4_K, 60, 2048, 256, 1), (Q4_K, 60, 2048, 512, 4), (Q4_K, 60, 16384, 768, 4),
    (Q4_K, 60, 16385, 768, 1), (Q4_K, 60, 24576, 1024, 2), (Q4_K, 60, 32769, 2048, 1),
    (Q8_0, 60, 2048, 256, 1), (Q8_0, 60, 16384, 768, 1), (Q8_0, 60, 16384, 1024, 4),
    (Q8_0, 64, 27648, 5120, 1), (Q8_0, 65, 13824, 5120, 2), (Q8_0, 127, 16384, 3840, 1)])
def test_int8_wave_groups(qt, M, N, K, groups):
    """Few super-blocks, or weights that no second tile shares, keep one wave group."""
    call = _instances("ifx_qgemm_prefill_kernel", qt, M, N, K, ops.PREFILL_INT8, 0)
    assert call == [f"k_gemm_mfma<{qt},1,0>[{groups}]"]


def test_int8_gpu_shapes_reach_every_group_count():
    from tests.test_gpu_mid_batch import CASES
    for qt in (Q4_K, Q8_0):
        got = {k for t, M, Ns, K in CASES if t == qt
               for k in _instances("ifx_qgemm_prefill_kernel", qt, M, Ns[0], K, ops.PREFILL_INT8, 0)}
        want = {f"k_gemm_mfma<{qt},1,0>[{kw}]" for kw in (1, 2, 4)}
        assert want <= got, got
