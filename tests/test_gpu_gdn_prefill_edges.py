"""Gated DeltaNet prompt kernels against the oracle at the edges of their
chunks: conv1d around its 16-token chunk and its 3-entry state (the first
chunk's threads publish the state), the recurrence around its 32-token chunks
(k.q is formed while a chunk is staged, 8 tokens a step). Bounds as in test_gpu_prefill: state
and outputs of the conv exact / bf16, recurrence outputs bf16, state rel 1e-3."""
import numpy as np
import pytest

from helpers import assert_bf16_close
from peregrine_amd.synth import bf16_to_f32, random_bf16
from test_gpu_prefill import _gdn_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,has_prev", [(1, False), (2, True), (3, True), (16, True), (16, False), (18, True), (48, True)])
def test_conv1d_state_edges(gpu, orc, T, has_prev):
    from peregrine_amd import ops
    from peregrine_amd.device import DeviceArray

    rng = np.random.default_rng(T + has_prev)
    state = bf16_to_f32(random_bf16(rng, (3, 8192), std=2.0))
    w, x = random_bf16(rng, (8192, 4), std=0.5), random_bf16(rng, (T, 8192), std=2.0)
    sd, out = DeviceArray.from_numpy(state), DeviceArray((T, 8192), np.uint16)
    ops.conv1d_silu_prefill(sd, DeviceArray.from_numpy(x), DeviceArray.from_numpy(w), out, T, has_prev)
    gpu.synchronize()
    ro, rs = orc.conv1d_prefill(state, x, w, has_prev)
    assert_bf16_close(out.numpy(), ro, min_exact=0.999, what="conv prefill")
    np.testing.assert_array_equal(sd.numpy(), rs)


@pytest.mark.parametrize("T,has_prev", [(8, True), (9, False), (24, True), (31, True), (32, False), (33, True), (95, True)])
def test_recurrence_chunk_edges(gpu, orc, T, has_prev):
    from peregrine_amd import ops
    from peregrine_amd.device import DeviceArray

    rng = np.random.default_rng(T)
    co, a, b, A_log, dtb, state = _gdn_inputs(rng, T)
    qn, kn = orc.qk_l2norm_prefill(co)
    g, beta = orc.gating_many(A_log, a, dtb, b)
    d = DeviceArray.from_numpy
    sd, y = d(state), DeviceArray((T, 4096), np.uint16)
    ops.gated_delta_prefill(sd, d(qn), d(kn), d(co), d(g), d(beta), y, T, has_prev)
    gpu.synchronize()
    ry, rs = orc.gated_delta_prefill(state, qn, kn, co, g, beta, has_prev)
    assert_bf16_close(y.numpy(), ry, min_exact=0.95, what=f"gdn prefill y T={T}")
    gs = sd.numpy().astype(np.float64)
    assert np.linalg.norm(gs - rs) / np.linalg.norm(rs) <= 1e-3
