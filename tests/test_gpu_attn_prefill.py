"""Prefill attention against the oracle where its kernels change form: each
split of the value dims (few, some and many tokens), each register window of
the row statistics (contexts around 2048, 6144 and past 16384), score blocks of
2, 3, 4 and 16 tiles, contexts that end inside a 64-slot tile and inside a
16-byte chunk, and cache strides that are not a multiple of the tile. Cache slots past the context hold NaN. The
bound is test_gpu_prefill's: one output ulp plus one flipped probability."""
import numpy as np
import pytest

from peregrine_amd.synth import random_bf16
from test_gpu_prefill import _check_attn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,prefix,stride", [(1, 0, 8), (33, 30, 64), (257, 3, 264), (513, 0, 520), (5, 2044, 2056),
                                             (2, 6142, 6144), (3, 6150, 6400), (1, 16383, 16384), (2, 16400, 16448)])
def test_attn_prefill_forms_vs_oracle(gpu, orc, T, prefix, stride):
    from peregrine_amd import ops
    from peregrine_amd.device import DeviceArray

    print(f"[attn forms] T={T} prefix={prefix} stride={stride}", flush=True)
    rng = np.random.default_rng(T * 7 + prefix)
    L = prefix + T
    q, gate = random_bf16(rng, (T, 4096)), random_bf16(rng, (T, 4096), std=2.0)
    kc, vc = random_bf16(rng, (4, stride, 256)), random_bf16(rng, (4, 256, stride))
    kc[:, L:] = 0x7FC0
    vc[:, :, L:] = 0x7FC0
    d = DeviceArray.from_numpy
    guard = np.full((T + 1, 4096), 0x7FC1, np.uint16)
    out = d(guard)
    scores = DeviceArray((ops.attn_prefill_scores_bytes(T, prefix) // 2,), np.uint16)
    ops.attn_prefill(d(q), d(kc), d(vc), d(gate), out, scores, T, prefix, stride)
    gpu.synchronize()
    got = out.numpy()
    assert (got[T] == 0x7FC1).all()
    vz = vc.copy()
    vz[:, :, L:] = 0
    ref = orc.sigmoid_mul_pair(orc.attn_prefill(q, kc, vz, T, prefix, stride), gate)
    _check_attn(got[:T], ref, vz, f"attn prefill T={T} prefix={prefix}")


@pytest.mark.parametrize("T,prefix", [(513, 3000), (1600, 0), (1021, 15003)])
def test_attn_prefill_long_segments_vs_oracle(gpu, orc, T, prefix):
    """Score blocks that walk 3, 4 and 16 tiles, so that each K buffer is used
    again. Sampled rows: the oracle's row t of T tokens is its only row of one
    token after prefix + t."""
    from peregrine_amd import ops
    from peregrine_amd.device import DeviceArray

    print(f"[attn segments] T={T} prefix={prefix}", flush=True)
    rng = np.random.default_rng(T + prefix)
    stride = (prefix + T + 63) // 64 * 64
    q, gate = random_bf16(rng, (T, 4096)), random_bf16(rng, (T, 4096), std=2.0)
    kc, vc = random_bf16(rng, (4, stride, 256)), random_bf16(rng, (4, 256, stride))
    d = DeviceArray.from_numpy
    out = DeviceArray((T, 4096), np.uint16)
    scores = DeviceArray((ops.attn_prefill_scores_bytes(T, prefix) // 2,), np.uint16)
    ops.attn_prefill(d(q), d(kc), d(vc), d(gate), out, scores, T, prefix, stride)
    gpu.synchronize()
    rows = np.unique([0, 31, 32, T // 2, T - 33, T - 1])
    ref = np.concatenate([orc.sigmoid_mul_pair(orc.attn_prefill(q[t:t + 1], kc, vc, 1, prefix + int(t), stride),
                                               gate[t:t + 1]) for t in rows])
    _check_attn(out.numpy()[rows], ref, vc, f"attn prefill T={T} prefix={prefix}")


@pytest.mark.parametrize("T,start,stride", [(1, 0, 8), (63, 5, 72), (64, 0, 64), (65, 100, 168)])
def test_prepare_aligned_equals_general(gpu, T, start, stride):
    """16-byte aligned operands take the vector kernel, others the general one:
    the same q, gate and cache bits (slots outside the call's and the memory around
    each output stay untouched)."""
    from peregrine_amd import ops
    from peregrine_amd.device import DeviceArray

    rng = np.random.default_rng(T)
    ins = [random_bf16(rng, (n,), std=std, mean=mean) for n, std, mean in
           [(T * 8192, 2.0, 0.0), (256, 0.1, 1.0), (T * 1024, 2.0, 0.0), (256, 0.1, 1.0), (T * 1024, 1.0, 0.0)]]
    sizes = [T * 4096, T * 4096, 4 * stride * 256, 4 * 256 * stride]

    def run(shift):  # operands `shift` values past a 16-byte boundary
        def dev(a):
            return DeviceArray.from_numpy(np.concatenate([np.zeros(shift, np.uint16), a, np.zeros(8, np.uint16)]))

        arrays = [dev(a) for a in ins] + [dev(np.full(n, 0x7FC1, np.uint16)) for n in sizes]
        p = [a.ptr + 2 * shift for a in arrays]
        ops.attn_prefill_prepare(*p, T, start, start, stride)
        gpu.synchronize()
        got = [a.numpy() for a in arrays[5:]]
        for a, n in zip(got, sizes):  # nothing before or past an output
            assert not a[:shift].any() and a.size == shift + n + 8 and not a[shift + n:].any()
        return [a[shift:shift + n] for a, n in zip(got, sizes)]

    for a, b, what in zip(run(0), run(1), ("q", "gate", "K cache", "V cache")):
        np.testing.assert_array_equal(a, b, err_msg=what)
