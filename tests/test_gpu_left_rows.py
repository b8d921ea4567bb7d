"""GPU parity of the f32 rows that the sort-free path leaves to the sort: from
one row to more than the tiled sort takes, one tile to many, beside served rows,
with penalties, per-row parameters, a device ring, and in graph replays."""
import numpy as np
import pytest

from gemmaedge_amd import workloads as W
from gpu_util import assert_parity, oracle_params, rows_left, run_gpu, run_oracle, small_workload, to_device

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sampler():
    import torch

    from gemmaedge_amd import Sampler, available

    assert torch.cuda.is_available(), "GPU test run without a GPU"
    assert available(), "no gfx950 device visible to the HIP library"
    s = Sampler(max_rows=200, max_vocab=W.VOCAB, max_history=4096)
    yield s
    s.close()


def _left(rng, rows, vocab):
    """Rows with too many equal values, or NaN: none is served without a sort."""
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    for r in range(rows):
        if r % 3 == 0:
            x[r] = np.where(rng.random(vocab) < 0.5, np.float32(1.0), np.float32(1.25))
        elif r % 3 == 1:
            x[r, rng.integers(0, vocab)] = np.nan
        else:
            x[r] = 0.5
            x[r, : vocab // 100] = np.float32(-4.0)
    return x


@pytest.mark.parametrize("rows,vocab", [(1, 9500), (1, W.VOCAB), (2, 12289), (3, 65536), (9, 100003), (30, 20001)])
@pytest.mark.parametrize("penalty", [1.0, 1.3])
def test_every_row_left(sampler, rows, vocab, penalty):
    rng = np.random.default_rng(vocab + rows)
    H = 300
    hist = rng.integers(0, vocab, size=rows * H).astype(np.int32)
    w = small_workload(f"left-{rows}", _left(rng, rows, vocab),
                       dict(temperature=0.9, top_k=0, top_p=0.93, softcap=30.0, repetition_penalty=penalty),
                       history=hist, offsets=np.arange(rows + 1) * H, uniforms=W.mt_uniforms(vocab, rows))
    print(f"[left] {w.name} V={vocab}", flush=True)
    assert_parity(w, run_gpu(sampler, w), run_oracle(w))
    assert rows_left(sampler, rows) == list(range(rows))


@pytest.mark.parametrize("vocab", [1025, 4096, 4097])
def test_few_tiles(sampler, vocab):
    # (at most 4,096 equal values are ordered: here only NaN leaves a row)
    rng = np.random.default_rng(vocab)
    x = (rng.standard_normal((3, vocab)) * 3).astype(np.float32)
    x[0, 7] = x[2, vocab - 1] = np.nan
    w = small_workload(f"tiles-{vocab}", x, dict(temperature=1.0, top_k=0, top_p=0.95), uniforms=W.mt_uniforms(3, 3))
    print(f"[left] {w.name}", flush=True)
    assert_parity(w, run_gpu(sampler, w), run_oracle(w))
    assert rows_left(sampler, 3) == [0, 2]


@pytest.mark.parametrize("step", [1, 2, 40])
def test_some_rows_left(sampler, step):
    # 200 rows, every step-th left: the tiles of up to 160 rows, a workgroup a row above
    rng = np.random.default_rng(step)
    rows, vocab = 200, 9500
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    x[::step] = _left(rng, len(range(0, rows, step)), vocab)
    w = small_workload(f"some-{step}", x, dict(temperature=1.0, top_k=0, top_p=0.9, softcap=30.0),
                       uniforms=W.mt_uniforms(step, rows))
    print(f"[left] {w.name}", flush=True)
    assert_parity(w, run_gpu(sampler, w), run_oracle(w))
    assert rows_left(sampler, rows) == list(range(0, rows, step))


def test_per_row_parameters(sampler):
    import torch

    import ge_oracle as O
    from gemmaedge_amd import SamplingConfig

    rng = np.random.default_rng(5)
    rows, vocab = 12, 50257
    x = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    x[3] = _left(rng, 1, vocab)[0]
    cfgs = [dict(top_k=(3000, 0, 50256, 0, 40, 1025)[r % 6], temperature=(1.0, 0.0)[r == 5], top_p=(0.95, 1.0)[r % 2])
            for r in range(rows)]
    cfgs = [dict(dict(min_p=0.0, softcap=30.0, repetition_penalty=1.0), **c) for c in cfgs]
    uni = W.mt_uniforms(12, rows)
    print("[left] per row", flush=True)
    tok, pr, fl = sampler.sample(torch.from_numpy(x).cuda(), [SamplingConfig(**c) for c in cfgs],
                                 uniforms=torch.from_numpy(uni).cuda())
    torch.cuda.synchronize()
    left = rows_left(sampler, rows)
    for r in range(rows):
        w = small_workload(f"row{r}", x[r], cfgs[r], uniforms=uni[r:r + 1])
        got = tuple(t[r:r + 1].cpu().numpy() for t in (tok, pr, fl))
        assert_parity(w, got, O.run(w.logits, oracle_params(w.params), uniforms=w.uniforms), w.name)
    assert left == [r for r in range(rows) if r % 6 in (0, 2) or r in (3, 11)]


def test_replays_and_rings(sampler):
    # a graph of two calls, the second with the history that the first extends
    import torch

    from gemmaedge_amd import SamplingConfig

    rng = np.random.default_rng(6)
    rows, vocab, H = 5, 40001, 60
    x = _left(rng, rows, vocab)
    x[4] = (rng.standard_normal(vocab) * 3).astype(np.float32)
    hist = rng.integers(0, vocab, size=rows * H).astype(np.int32)
    p = dict(temperature=1.0, top_k=0, top_p=0.95, softcap=30.0, repetition_penalty=1.2)
    w = small_workload("ring", x, p, history=hist, offsets=np.arange(rows + 1) * H, uniforms=W.mt_uniforms(8, rows))
    first = run_oracle(w)
    both = np.concatenate([hist.reshape(rows, H), first.tokens.reshape(rows, 1)], 1).reshape(-1).astype(np.int32)
    w2 = small_workload("ring2", x, p, history=both, offsets=np.arange(rows + 1) * (H + 1), uniforms=w.uniforms)
    second = run_oracle(w2)
    logits, _, _, uni = to_device(w)
    ring = torch.zeros(rows, H + 2, dtype=torch.int32, device="cuda")
    ring[:, :H] = torch.from_numpy(hist.reshape(rows, H)).cuda()
    full = torch.full((rows,), H, dtype=torch.int32, device="cuda")
    ring_len = full.clone()
    out = [[torch.empty(rows, dtype=d, device="cuda") for d in (torch.int32, torch.float32, torch.int32)] for _ in range(2)]
    side = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side), torch.cuda.graph(g, stream=side):
        torch.add(full, 0, out=ring_len)
        for t, pr, fl in out:
            sampler.sample(logits, SamplingConfig(**p), uniforms=uni, ring=ring, ring_len=ring_len, tokens=t, probs=pr, flags=fl)
    torch.cuda.synchronize()
    for _ in range(4):
        print("[left] replay", flush=True)
        for t, _, _ in out:
            t.fill_(-7)
        g.replay()
        torch.cuda.synchronize()
        assert_parity(w, tuple(o.cpu().numpy() for o in out[0]), first, "first call")
        assert_parity(w2, tuple(o.cpu().numpy() for o in out[1]), second, "second call")
        assert_parity(w, run_gpu(sampler, w), first, "between")


@pytest.mark.parametrize("rows,vocab", [(3, 30000), (70, 30000), (2, W.VOCAB)])
def test_denominators_to_replay(sampler, rows, vocab):
    # the denominators' maps, of tiled rows and of rows with a workgroup each
    from test_gpu_certificates import _on_a_boundary

    rng = np.random.default_rng(vocab)
    base = np.minimum(rng.standard_normal(vocab) * 3 - 14, -0.5)
    base[0] = 0.0
    row, rest, s = _on_a_boundary(base, "f32")
    assert 0 <= rest < 500 * 2.0**-53 * s
    x = np.stack([rng.permutation(row) for _ in range(rows)])
    w = small_workload(f"replay-{rows}-{vocab}", x, dict(temperature=1.0, top_k=0, top_p=0.999), uniforms=W.mt_uniforms(4, rows))
    print(f"[left] {w.name}", flush=True)
    assert_parity(w, run_gpu(sampler, w), run_oracle(w))
    assert rows_left(sampler, rows) == list(range(rows))
