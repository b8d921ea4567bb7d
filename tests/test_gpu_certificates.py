"""GPU parity where the full-order path's error intervals do not decide: rows
whose double denominator lies within rounding error of a boundary between two
floats of 1 / den, so that only the sequential sum (src/generation.cpp:97)
says which float the probabilities are scaled by."""
import ctypes

import numpy as np
import pytest

from gemmaedge_amd import workloads as W
from gpu_util import assert_parity, rows_left, run_gpu, run_oracle, small_workload

pytestmark = pytest.mark.gpu

_libm = ctypes.CDLL("libm.so.6")
_libm.expf.restype = ctypes.c_float
_libm.expf.argtypes = [ctypes.c_float]


def _expf(v):
    return float(_libm.expf(float(v)))


def _sum_exp(x):
    """The double sum of the sampler's own float exponentials (numpy's differ in some last bits)."""
    values, counts = np.unique(x, return_counts=True)
    return float(np.sum(np.array([_expf(v) for v in values]) * counts))


@pytest.fixture(scope="module")
def sampler():
    import torch

    from gemmaedge_amd import Sampler, available

    assert torch.cuda.is_available(), "GPU test run without a GPU"
    assert available(), "no gfx950 device visible to the HIP library"
    s = Sampler(max_rows=8, max_vocab=W.VOCAB, max_history=64)
    yield s
    s.close()


def _on_a_boundary(base, dtype):
    """`base` (maximum 0) with its last 16 tokens chosen so that the sum of the
    exponentials comes as near as they allow to 1 / (midpoint of two floats)."""
    x = base.astype(np.float32).copy()
    x[-16:] = -80.0
    rounded = W.bf16_bits_to_f32(W.f32_to_bf16_bits(x)) if dtype == "bf16" else x
    s = _sum_exp(rounded)
    inv = np.float32(1.0 / s)
    below = np.nextafter(inv, np.float32(0.0))
    mid = (float(inv) + float(below)) / 2  # 1 / mid lies above s: terms can only be added
    rest = 1.0 / mid - s
    while rest < 0:
        below, inv = np.nextafter(below, np.float32(0.0)), below
        rest = 2.0 / (float(inv) + float(below)) - s
    for i in range(16):
        if rest <= 1e-30:
            break
        v = np.float32(np.log(rest))
        if dtype == "bf16":
            v = W.bf16_bits_to_f32(W.f32_to_bf16_bits(np.array([v], np.float32)))[0]
        while _expf(v) > rest:
            v = W.bf16_bits_to_f32(W.f32_to_bf16_bits(np.array([v * np.float32(1.004)], np.float32)))[0] \
                if dtype == "bf16" else np.nextafter(v, np.float32(-200.0))
        x[x.size - 16 + i] = v
        rest -= _expf(v)
    return x, rest, s


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("vocab", [5000, W.VOCAB])
def test_denominator_between_two_floats(sampler, dtype, vocab):
    rng = np.random.default_rng(vocab + len(dtype))
    rows = []
    for r in range(4):
        base = np.minimum(rng.standard_normal(vocab) * 3 - 14, -0.5)
        base[r] = 0.0
        x, rest, s = _on_a_boundary(base, dtype)
        # well inside the interval that the device allows the two sums to differ by
        assert 0 <= rest < 500 * 2.0**-53 * s, (rest, s)
        rows.append(x)
    x = np.stack(rows)
    logits = W.f32_to_bf16_bits(x) if dtype == "bf16" else x
    w = small_workload(f"boundary-{dtype}-{vocab}", logits, dict(temperature=1.0, top_k=0, top_p=0.999),
                       uniforms=np.array([0.2, 0.9, 0.9999, 0.6], np.float32), dtype=dtype)
    print(f"[certificates] {w.name}", flush=True)
    ora = run_oracle(w)
    assert_parity(w, run_gpu(sampler, w), ora)
    if dtype == "f32":  # only the sort has the sequential sum
        assert rows_left(sampler, 4) == [0, 1, 2, 3]
