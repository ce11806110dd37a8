"""K splits of the fp16 prefill GEMM: the ordered entry asks for no more
workspace than the documented line (a grid of 256 x 256 tiles, 512 values of
K a split), so a buffer sized for a shape once stays large enough, and a
shape that never split still runs without one."""
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
