"""GPU parity of the single-pass selection kernel where a wave's candidates do
not fit its list: it then lists down to a bound of its own (its q-th lane
maximum, or its largest), which the row's merge takes into account. Rows with
many large logits in one lane, in one wave, equal ones, and more than a lane
stages (which the rescans serve)."""
import numpy as np
import pytest

from gemmaedge_amd import workloads as W
from gpu_util import assert_parity, run_gpu, run_oracle, small_workload

pytestmark = pytest.mark.gpu

CHUNK = 256 * 64


@pytest.fixture(scope="module")
def sampler():
    import torch

    from gemmaedge_amd import Sampler, available

    assert torch.cuda.is_available(), "GPU test run without a GPU"
    assert available(), "no gfx950 device visible to the HIP library"
    s = Sampler(max_rows=16, max_vocab=W.VOCAB, max_history=256)
    yield s
    s.close()


def _slot(chunk, thread, s, w):
    """Index of slot s of a thread: w consecutive tokens per 16-byte load."""
    return chunk * CHUNK + ((s // w) * 256 + thread) * w + s % w


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("vocab", [20011, 50000, 131072, W.VOCAB])
@pytest.mark.parametrize("k", [5, 40, 64])
def test_crowded_waves(sampler, dtype, vocab, k):
    rng = np.random.default_rng(vocab + k)
    w = 4 if dtype == "f32" else 8
    rows = 12
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    chunks = vocab // CHUNK  # whole ones
    H = 40
    hist = rng.integers(0, vocab, size=(rows, H)).astype(np.int32)
    for r in range(rows):
        c = int(rng.integers(0, chunks))
        if r < 4:  # r + 4 large logits in one lane (4: fits; 7: more than it stages)
            t = int(rng.integers(0, 256))
            at = [_slot(c, t, int(s), w) for s in rng.choice(64, r + 4, replace=False)]
        elif r < 8:  # 20 to 62 in one wave
            n = (20, 24, 40, 62)[r - 4]
            base = 64 * int(rng.integers(0, 4))
            at = [_slot(c, base + int(t), int(rng.integers(0, 64)), w) for t in rng.choice(64, n, replace=False)]
        elif r < 10:  # 40 in one wave of every chunk
            at = [_slot(cc, 64 * (r - 8) + int(t), int(rng.integers(0, 64)), w) for cc in range(chunks) for t in range(40)]
        else:  # equal values: no bound of the wave's own separates them
            at = [_slot(c, int(t), s, w) for t in range(64) for s in (range(2) if r == 10 else range(6))]
        x[r, at] = 15.0 if r >= 10 else rng.uniform(12, 16, len(at)).astype(np.float32)
        hist[r, :len(at[:20])] = at[:20]
    logits = W.f32_to_bf16_bits(x) if dtype == "bf16" else x
    for pen in (1.0, 1.3):
        wl = small_workload(f"crowded-{dtype}-{vocab}-k{k}-r{pen}", logits,
                            dict(temperature=1.0, top_k=k, top_p=0.99, softcap=30.0, repetition_penalty=pen),
                            history=hist.reshape(-1), offsets=np.arange(rows + 1) * H, uniforms=W.mt_uniforms(k, rows),
                            dtype=dtype)
        print(f"[stream] {wl.name}", flush=True)
        for _ in range(3):  # list areas in turn
            assert_parity(wl, run_gpu(sampler, wl), run_oracle(wl), wl.name)
