"""GPU parity of f32 rows with top-k off whose values are built so that the
reference's float sums round in a chosen way: q = exp(l) / denominator of the
tokens is set by its distance from a half ulp of the running sum
(src/generation.cpp:103-126)."""
import ctypes

import numpy as np
import pytest

from gpu_util import assert_parity, rows_left, run_gpu, run_oracle, small_workload

pytestmark = pytest.mark.gpu

_libm = ctypes.CDLL("libm.so.6")
_libm.expf.restype = ctypes.c_float
_libm.expf.argtypes = [ctypes.c_float]
U = 2.0**-24  # the ulp of a sum in [1/2, 1)


def _exps(v):
    return np.array([_libm.expf(float(x)) for x in v], np.float32)


def _logits_below(inv, targets):
    """Per target probability, the largest logit whose q = exp(l) * inv lies below it."""
    out = []
    for t in targets:
        v = np.float32(np.log(t / float(inv)))
        q = lambda x: float(np.float32(_libm.expf(float(x))) * inv)  # noqa: E731
        while q(v) >= t:
            v = np.nextafter(v, np.float32(-200))
        while q(np.nextafter(v, np.float32(0))) < t:
            v = np.nextafter(v, np.float32(0))
        out.append(v)
    return np.array(out, np.float32)


def _scaled_to(inv, values, counts, low):
    """The row of `values` (each `counts` times, the largest 0), with as many
    tokens below exp = 0.5 added as bring the denominator's reciprocal to `inv`;
    the first of them lie at `low` and the last takes up the rest."""
    e = _exps(values).astype(np.float64)
    rest = 1.0 / float(inv) - float(np.sum(e * counts))
    assert rest > 0.0
    more = []
    pe = float(_libm.expf(float(low)))
    while rest > 1.5 * pe:
        more.append(low)
        rest -= pe
    for _ in range(8):  # each takes up what the one before leaves
        v = np.float32(np.log(rest))
        while float(_libm.expf(float(v))) > rest:
            v = np.nextafter(v, np.float32(-200))
        more.append(v)
        rest -= float(_libm.expf(float(v)))
        if rest < 1e-9:
            break
    row = np.concatenate([np.repeat(values, counts), np.array(more, np.float32)])
    s = float(np.sum(_exps(np.unique(row)).astype(np.float64) * np.unique(row, return_counts=True)[1]))
    assert np.float32(1.0 / s) == inv
    return row


@pytest.fixture(scope="module")
def sampler():
    import torch

    from gemmaedge_amd import Sampler, available

    assert torch.cuda.is_available(), "GPU test run without a GPU"
    assert available(), "no gfx950 device visible to the HIP library"
    s = Sampler(max_rows=8, max_vocab=262144, max_history=64)
    yield s
    s.close()


def test_bins_that_add_nothing_in_the_expected_binade(sampler):
    # Thousands of tokens a little below (k + 1/2) ulps: the sum falls 2e-3 short
    # of 1.0, where an even spread of the addends would take it past 1.0. There
    # the tail's addends (just above half an ulp of [1/2, 1)) would add nothing;
    # in truth each adds an ulp.
    inv = np.float32(4e-4)
    k = np.array([89, 84, 80, 76, 72, 67, 63, 59, 46, 44, 42, 40, 31, 29, 27, 25, 24, 9, 8])
    mid = _logits_below(inv, (k + 0.5) * U * (1 - 2e-6))
    tail = np.log(np.linspace(5.6e-8, 4.4e-8, 24600) / float(inv)).astype(np.float32)
    head = np.log(np.linspace(1.0, 0.1, 3480)).astype(np.float32)
    head[0] = 0.0
    values = np.concatenate([head, mid, tail])
    counts = np.concatenate([np.ones(3480, int), np.full(18, 4222), [4000], np.ones(24600, int)])
    row = _scaled_to(inv, values, counts, np.float32(-0.9))
    rng = np.random.default_rng(1)
    rng.shuffle(row)
    u = np.array([0.001, 0.05, 0.1, 0.2, 0.3, 0.35, 0.5, 0.9], np.float32)
    w = small_workload("gap", np.repeat(row[None], 8, 0), dict(temperature=1.0, top_k=0, top_p=2.0), uniforms=u)
    print(f"[binned exact] {w.name} V={w.vocab}", flush=True)
    assert_parity(w, run_gpu(sampler, w), run_oracle(w))


def test_a_large_bin_of_ties(sampler):
    # 6,000 tokens of one value half way between two ulps of the sum: a bin that
    # the cumulative sum was to pass as whole ulps, and too large to order.
    inv = np.float32(2.0**-11 * 1.3)
    v = np.float32(np.log(100.5 * U / float(inv)))
    for _ in range(1 << 20):
        q = float(np.float32(_libm.expf(float(v))) * inv) / U
        if q % 1.0 == 0.5:
            break
        v = np.nextafter(v, np.float32(0))
    else:
        pytest.fail("no tie found")
    head = np.log(np.linspace(1.0, 0.1, 2000)).astype(np.float32)
    head[0] = 0.0
    tail = np.linspace(v - 3, v - 0.5, 40000).astype(np.float32)
    row = _scaled_to(inv, np.concatenate([head, [v], tail]), np.concatenate([np.ones(2000, int), [6000], np.ones(40000, int)]),
                     np.float32(-1.2))
    rng = np.random.default_rng(2)
    rng.shuffle(row)
    u = np.array([0.01, 0.3, 0.6, 0.9], np.float32)
    w = small_workload("large tie", np.repeat(row[None], 4, 0), dict(temperature=1.0, top_k=0, top_p=0.99), uniforms=u)
    print(f"[binned exact] {w.name} V={w.vocab} q={q} ulps", flush=True)
    assert_parity(w, run_gpu(sampler, w), run_oracle(w))
    assert rows_left(sampler, 4) == [0, 1, 2, 3]
