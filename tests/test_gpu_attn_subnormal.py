"""Prefill attention where probabilities are bf16 subnormals (below 2^-126):
they carry weight when the values behind them are large, and are kept. Row
maximum 0 at slot 0, whose values are zero; every other score is -86 .. -91.5, so
its probability is e^-86 = 2^-124.07 .. e^-91.5 = 2^-132.01, and its values are
+-2^118 .. 2^120: contexts of about 1e-2.

Bound: a probability's f32 bits may differ by an ulp between the two exp2,
which flips its bf16 rounding now and then, by 2^-133 (the spacing of bf16
subnormals) times a value of up to 2^120 = 2^-13; two such flips to a row and
head, plus one ulp of the context and one of the output."""
import numpy as np
import pytest

from peregrine_amd.synth import bf16_to_f32, f32_to_bf16, random_bf16

pytestmark = pytest.mark.gpu


# each split of the value dims, and a register window of the row statistics beyond the first
@pytest.mark.parametrize("T,prefix", [(2, 40), (2, 2100), (270, 0), (513, 0)])
def test_subnormal_probabilities_count(gpu, orc, T, prefix):
    from peregrine_amd import ops
    from peregrine_amd.device import DeviceArray

    print(f"[attn subnormal] T={T} prefix={prefix}", flush=True)
    rng = np.random.default_rng(T + prefix)
    L, stride = prefix + T, (prefix + T + 63) // 64 * 64
    q = np.zeros((T, 16, 256), np.float32)
    q[:, :, 0] = 16.0
    k = np.zeros((4, stride, 256), np.float32)
    k[:, 1:, 0] = -(86.0 + 0.5 * rng.integers(0, 12, (4, stride - 1)))
    v = np.ldexp(rng.choice([-1.0, 1.0], (4, 256, stride)), rng.integers(118, 121, (4, 256, stride)))
    v[:, :, 0] = 0.0
    v[:, :, L:] = 0.0
    q, k, v = (f32_to_bf16(a.astype(np.float32)) for a in (q.reshape(T, 4096), k, v))
    gate = random_bf16(rng, (T, 4096), std=2.0)
    d = DeviceArray.from_numpy
    out = DeviceArray((T, 4096), np.uint16)
    scores = DeviceArray((ops.attn_prefill_scores_bytes(T, prefix) // 2,), np.uint16)
    ops.attn_prefill(d(q), d(k), d(v), d(gate), out, scores, T, prefix, stride)
    gpu.synchronize()
    # sampled rows: the oracle's row t of T tokens is its only row of one token after prefix + t
    rows = np.unique(np.concatenate([np.arange(min(T, 2)), rng.integers(0, T, 6), [T - 1]]))
    ref = np.concatenate([orc.sigmoid_mul_pair(orc.attn_prefill(q[t:t + 1], k, v, 1, prefix + int(t), stride),
                                               gate[t:t + 1]) for t in rows])
    g, r = (bf16_to_f32(a).astype(np.float64) for a in (out.numpy()[rows], ref))
    rms = float(np.sqrt(np.mean(r * r)))
    print(f"exact {np.mean(out.numpy()[rows] == ref):.5f}, rms {rms:.3e}, max err {np.abs(g - r).max():.3e}")
    assert rms > 1e-3
    assert (np.abs(g - r) <= 2.0 ** -7 * np.abs(r) + 2 * 2.0 ** -13).all()
