"""The few-row prompt GEMM (16 to 128 weight rows per block) against the
row-tiled kernel on the same inputs: a row's bits must not depend on which of
the two a call takes, because a prompt's chunks mix them. Every form the
launcher picks, for plain outputs (10 t + m = 16 t weight rows and 64 m
activation rows per block) and for the SiLU pair, at the edges of its tiles: one
row, a 16-row block and one more, 64 / 128 rows and one more, weight rows that
end inside a tile, one stage of k and many. PEREGRINE_GEMM_DMA=0 keeps the
row-tiled kernel. Outputs have one guard row, which stays untouched.
"""
import numpy as np
import pytest

from helpers import PAIR, RESIDUAL, STORE, qmm_route
from peregrine_amd.synth import random_bf16, random_q4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,plain,pair", [
    (1, 16, 256, 11, 41), (16, 100, 512, 11, 41), (17, 320, 768, 11, 41), (43, 4096, 1024, 11, 41),
    (64, 1000, 4096, 11, 41), (65, 4104, 256, 41, 81), (128, 264, 1280, 11, 41), (129, 8192, 512, 42, 82),
    (300, 96, 2048, 11, 41), (17, 6152, 512, 21, 41), (65, 4096, 768, 21, 41), (100, 4100, 256, 41, 81),
    (128, 4090, 1280, 21, 41), (129, 1364, 256, 21, 41), (1, 8260, 1024, 41, 81), (64, 12300, 512, 41, 81),
    (384, 1360, 768, 12, 81), (321, 1357, 256, 12, 81), (322, 2720, 1280, 22, 41), (384, 2711, 256, 22, 41),
    (65, 8260, 768, 42, 82), (128, 8250, 256, 42, 82), (100, 12300, 512, 42, 82), (193, 4104, 256, 42, 82)])
def test_few_rows_equal_row_tiles(gpu, monkeypatch, M, N, K, plain, pair):
    from peregrine_amd import ops
    from peregrine_amd.device import DeviceArray
    from peregrine_amd.ops import Q4Linear

    print(f"[few rows] M={M} N={N} K={K}", flush=True)
    monkeypatch.delenv("PEREGRINE_GEMM_DMA", raising=False)

    def routes():
        return [qmm_route(STORE, M, [N], K), qmm_route(RESIDUAL, M, [N], K), qmm_route(PAIR, M, [N, N], K)]

    assert routes() == [plain, plain, pair]
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
    assert all(r in (192, 256) for r in routes())
    for a, b, what in zip(few, outputs(), ("store", "residual", "silu pair")):
        np.testing.assert_array_equal(a, b, err_msg=what)
        assert (a[M] == 0x7FC1).all() and not (a[:M] == 0x7FC1).any(), what


@pytest.mark.parametrize("M,qkv,gdn", [(1, 41, 41), (43, 41, 41), (64, 41, 41), (65, 42, 42), (128, 42, 42),
                                       (129, 41, 192)])
def test_several_weights_in_a_launch(gpu, monkeypatch, M, qkv, gdn):
    """q / k / v and the Gated DeltaNet's input projections share a launch (3 and
    4 weights, the last two of 32 rows): a prompt leaves the same states through
    the few-row kernel as through the row-tiled one. The second period of layers
    carries what the first one's q and z outputs change."""
    from peregrine_amd.model import DeviceModel, ModelConfig, ModelState

    print(f"[few rows] model prompt of {M}", flush=True)
    monkeypatch.delenv("PEREGRINE_GEMM_DMA", raising=False)
    cfg = ModelConfig(num_layers=8, hidden=1024, intermediate=2048, vocab=4096)
    assert qmm_route(STORE, M, [8192, 1024, 1024], 1024) == qkv
    assert qmm_route(STORE, M, [8192, 4096, 32, 32], 1024) == gdn
    m = DeviceModel(cfg, seed=5)
    prompt = np.random.default_rng(M).integers(0, cfg.vocab, M).astype(np.uint32)
    names = [f"layers.{i}.{n}" for i in range(cfg.num_layers)
             for n in (("recur", "conv") if cfg.is_linear(i) else ("cache_k", "cache_v"))]

    def ingest():
        st = ModelState(m, 256)
        first = st.prefill(prompt)
        out = [st.read(n, np.uint16) for n in names]
        st.close()
        return first, out

    first, few = ingest()
    monkeypatch.setenv("PEREGRINE_GEMM_DMA", "0")
    first_ref, ref = ingest()
    m.close()
    assert first == first_ref
    for n, a, b in zip(names, few, ref):
        np.testing.assert_array_equal(a, b, err_msg=n)
