"""The few-row prompt GEMM (16 to 128 weight rows per block) against the
row-tiled kernel on the same inputs: a row's bits must not depend on which of
the two a call takes, because a prompt's chunks mix them. Sizes are the edges
of its tiles: one row, a 16-row block and one more, 64 / 128 rows (the row tile
of its two forms) and one more, weight rows that end inside a tile, one stage
of k and many. PEREGRINE_GEMM_DMA=0 keeps the row-tiled kernel. Outputs have
one guard row, which stays untouched.
"""
import numpy as np
import pytest

from peregrine_amd.synth import random_bf16, random_q4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1, 16, 256), (16, 100, 512), (17, 320, 768), (43, 4096, 1024), (64, 1000, 4096),
                                   (65, 4104, 256), (128, 264, 1280), (129, 8192, 512), (300, 96, 2048)])
def test_few_rows_equal_row_tiles(gpu, monkeypatch, M, N, K):
    from peregrine_amd import ops
    from peregrine_amd.device import DeviceArray
    from peregrine_amd.ops import Q4Linear

    print(f"[few rows] M={M} N={N} K={K}", flush=True)
    rng = np.random.default_rng(M * 5 + N + K)
    g, u = (Q4Linear.upload(random_q4(rng, N, K, zero_mean=True)) for _ in range(2))
    x = DeviceArray.from_numpy(random_bf16(rng, (M, K), std=2.0))
    res = DeviceArray.from_numpy(random_bf16(rng, (M, N), std=3.0))
    guard = np.full((M + 1, N), 0x7FC1, np.uint16)

    def outputs():
        outs = [DeviceArray.from_numpy(guard) for _ in range(3)]
        g.encode_prefill_qmm(x, outs[0], M)
        g.encode_prefill_qmm_residual_add(x, res, outs[1], M)
        ops.prefill_gate_up_silu(g, u, x, outs[2], M)
        gpu.synchronize()
        return [o.numpy() for o in outs]

    few = outputs()
    monkeypatch.setenv("PEREGRINE_GEMM_DMA", "0")
    for a, b, what in zip(few, outputs(), ("store", "residual", "silu pair")):
        np.testing.assert_array_equal(a, b, err_msg=what)
        assert (a[M] == 0x7FC1).all() and not (a[:M] == 0x7FC1).any(), what
