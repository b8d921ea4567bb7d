"""GPU parity of the f32 full-order rows that take no sort (top-k off): the
sizes where the histogram's bins, the parts of a row and the batch rule change,
draws at both ends of the row, cuts inside and between bins, and the rows that
are left to the sort-based pass. Checked against the CPU oracle: tokens and
probabilities bit-identical, near-boundary flags equal."""
import numpy as np
import pytest

import ge_oracle as O
from gemmaedge_amd import workloads as W
from gpu_util import assert_parity, oracle_params, rows_left, run_gpu, run_oracle, small_workload, to_device

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sampler():
    import torch

    from gemmaedge_amd import Sampler, available

    assert torch.cuda.is_available(), "GPU test run without a GPU"
    assert available(), "no gfx950 device visible to the HIP library"
    s = Sampler(max_rows=136, max_vocab=W.VOCAB, max_history=4096)
    yield s
    s.close()


def _check(sampler, w, left=None):
    """Parity, and which rows were left to the sort (None: any; the results are the same)."""
    print(f"[binned] {w.name} rows={w.rows} V={w.vocab} {w.params}", flush=True)
    assert_parity(w, run_gpu(sampler, w), run_oracle(w), w.name)
    if left is not None:
        assert rows_left(sampler, w.rows) == left


def _rows(rng, rows, vocab, kind):
    x = rng.standard_normal((rows, vocab)) * {"flat": 0.1, "wide": 3.0, "huge": 40.0, "same": 1e-4}[kind]
    if kind == "wide":
        for r in range(rows):
            x[r, rng.integers(0, vocab, 10)] += rng.uniform(6, 10, 10)
    return x.astype(np.float32)


@pytest.mark.parametrize("vocab", [1025, 4095, 4096, 4097, 16385, 32767, 32768, 65535, 65536, 131071, 131072, 200003])
@pytest.mark.parametrize("kind", ["flat", "wide", "huge", "same"])
def test_vocabularies(sampler, vocab, kind):
    rng = np.random.default_rng(vocab + len(kind))
    H = 200
    hist = rng.integers(0, vocab, size=6 * H).astype(np.int32)
    w = small_workload(f"{kind}-{vocab}", _rows(rng, 6, vocab, kind),
                       dict(temperature=0.9, top_k=0, top_p=0.93, softcap=30.0, repetition_penalty=1.15),
                       history=hist, offsets=np.arange(7) * H, uniforms=W.mt_uniforms(vocab, 6))
    _check(sampler, w, left=[])


@pytest.mark.parametrize("rows,vocab", [(1, W.VOCAB), (127, 131075), (128, 131075), (129, 40001), (136, 5003)])
def test_batches(sampler, rows, vocab):
    rng = np.random.default_rng(rows)
    x = np.concatenate([_rows(rng, (rows + 1) // 2, vocab, "wide"), _rows(rng, rows // 2, vocab, "flat")])
    _check(sampler, small_workload(f"batch-{rows}", x, dict(temperature=1.1, top_k=0, top_p=0.9, softcap=30.0),
                                   uniforms=W.mt_uniforms(rows, rows)), left=[])


@pytest.mark.parametrize("kind", ["flat", "wide"])
@pytest.mark.parametrize("params", [dict(top_p=1.0), dict(top_p=2.0), dict(top_p=0.0), dict(top_p=0.9999, min_p=0.02),
                                    dict(top_p=1.0, min_p=0.9), dict(top_p=1.0, min_p=1.5), dict(top_p=0.3, softcap=0.0),
                                    dict(top_p=0.97, repetition_penalty=0.7)])
def test_ends_and_cuts(sampler, kind, params):
    # the first and last tokens, the smallest draws, a cut inside a bin
    vocab = 70001
    u = np.array([0.0, 1e-12, 1e-6, 1e-4, 0.02, 0.5, 0.97, 0.9999, float(np.float32(1 - 2**-24))], np.float32)
    rng = np.random.default_rng(len(kind))
    x = np.repeat(_rows(rng, 3, vocab, kind), 3, axis=0)
    hist = rng.integers(0, vocab, size=9 * 64).astype(np.int32)
    w = small_workload(f"ends-{kind}", x, dict(dict(temperature=1.0, top_k=0, softcap=30.0), **params),
                       history=hist, offsets=np.arange(10) * 64, uniforms=u)
    # (the largest draws of an open nucleus end among the tail's many tokens)
    _check(sampler, w, left=[7, 8] if kind == "wide" and params["top_p"] >= 1.0 and "min_p" not in params else [])


@pytest.mark.parametrize("vocab,top", [(W.VOCAB, 0.0), (131071, 0.0), (65537, 0.0), (W.VOCAB, 1.5), (W.VOCAB, 12.0)])
def test_bins_of_every_size(sampler, vocab, top):
    # Near-uniform rows whose bins hold from one token to a few hundred, the
    # chains' binade changes and the draw at many places among them; with `top`
    # a few larger values widen the bins until a key takes more than 32 bits.
    # Quantised rows: equal exps, told apart by the index.
    rng = np.random.default_rng(vocab + int(top))
    u = np.linspace(0.01, 0.99, 9).astype(np.float32)
    for sigma, step in ((0.1, 0.0), (0.02, 0.0), (0.3, 0.0), (0.1, 2.0**-16)):
        x = (rng.standard_normal((9, vocab)) * sigma).astype(np.float32)
        if step:
            x = (np.round(x / step) * step).astype(np.float32)
        x[:, :3] += np.float32(top)
        for top_p in (0.6, 0.95):
            _check(sampler, small_workload(f"bins-{sigma}-{step}-{top_p}", x,
                                           dict(temperature=1.1, top_k=0, top_p=top_p, softcap=30.0), uniforms=u),
                   left=[] if top == 0.0 else None)  # (a few larger values can leave all others in one bin)


def test_ties_and_quantised_values(sampler):
    # bf16 values in f32 (hundreds of equal tokens a value), and a coarser grid
    rng = np.random.default_rng(3)
    x = _rows(rng, 4, 100003, "wide")
    x[0] = W.bf16_bits_to_f32(W.f32_to_bf16_bits(x[0]))
    x[1] = np.round(x[1] * 16) / 16
    x[2] = W.bf16_bits_to_f32(W.f32_to_bf16_bits(x[2] * np.float32(0.03)))
    for T in (1.0, 8.0):  # a hot temperature gives many logits one exp
        _check(sampler, small_workload(f"ties-T{T}", x, dict(temperature=T, top_k=0, top_p=0.95, softcap=30.0),
                                       uniforms=W.mt_uniforms(11, 4)), left=[])


def test_rows_left_to_the_sort(sampler):
    # beside an ordinary row: NaN, an infinite maximum, all equal, two values,
    # all masked but a few
    rng = np.random.default_rng(4)
    x = _rows(rng, 6, 50021, "wide")
    x[1, 17] = np.nan
    x[2, 5] = np.inf
    x[3] = 0.25
    x[4] = np.where(rng.random(50021) < 0.5, 1.0, 1.5)
    x[5, 40:] = -np.inf
    _check(sampler, small_workload("left", x, dict(temperature=1.0, top_k=0, top_p=0.95, softcap=30.0),
                                   uniforms=W.mt_uniforms(5, 6)), left=[1, 3, 4])


def test_replays_of_a_graph(sampler):
    import torch

    from gemmaedge_amd import SamplingConfig

    rng = np.random.default_rng(6)
    H = 100
    hist = rng.integers(0, W.VOCAB, size=3 * H).astype(np.int32)
    p = dict(temperature=1.0, top_k=0, top_p=0.95, softcap=30.0, repetition_penalty=1.2)
    w = small_workload("graph", _rows(rng, 3, W.VOCAB, "wide"), p, history=hist, offsets=np.arange(4) * H,
                       uniforms=W.mt_uniforms(8, 3))
    other = small_workload("other", _rows(rng, 3, 30011, "flat"), p, uniforms=W.mt_uniforms(9, 3))
    logits, h, offs, uni = to_device(w)
    tok = torch.empty(3, dtype=torch.int32, device="cuda")
    pr = torch.empty(3, dtype=torch.float32, device="cuda")
    fl = torch.empty(3, dtype=torch.int32, device="cuda")
    side = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side), torch.cuda.graph(g, stream=side):
        sampler.sample(logits, SamplingConfig(**w.params), uniforms=uni, history=h, history_offsets=offs, tokens=tok, probs=pr,
                       flags=fl)
    torch.cuda.synchronize()
    ora = run_oracle(w)
    for _ in range(4):
        tok.fill_(-7)
        g.replay()
        torch.cuda.synchronize()
        assert_parity(w, (tok.cpu().numpy(), pr.cpu().numpy(), fl.cpu().numpy()), ora, "replay")
        assert rows_left(sampler, 3) == []
        _check(sampler, other, left=[])  # other sizes on the same workspace in between


def test_per_row_parameters_take_one_kernel(sampler):
    import torch

    from gemmaedge_amd import SamplingConfig

    rng = np.random.default_rng(7)
    rows, vocab = 9, 131072
    x = np.concatenate([_rows(rng, 5, vocab, "wide"), _rows(rng, 4, vocab, "flat")])
    x[8, 3] = np.nan
    cfgs = [dict(temperature=0.8, top_k=0, top_p=0.9, softcap=30.0), dict(temperature=0.0), dict(top_k=3000, softcap=30.0),
            dict(top_k=40), dict(top_k=0, top_p=1.0, min_p=0.01, softcap=5.0), dict(top_k=vocab, top_p=0.5),
            dict(temperature=1.3, top_k=0, top_p=0.9, softcap=30.0), dict(top_k=0, top_p=0.99), dict(top_k=0)]
    cfgs = [dict(dict(temperature=1.0, top_k=0, top_p=0.95, min_p=0.0, softcap=0.0, repetition_penalty=1.0), **c) for c in cfgs]
    uni = W.mt_uniforms(12, rows)
    tok, pr, fl = sampler.sample(torch.from_numpy(x).cuda(), [SamplingConfig(**c) for c in cfgs],
                                 uniforms=torch.from_numpy(uni).cuda())
    torch.cuda.synchronize()
    # (of the full-order rows: the one with 1024 < k < V, and NaN)
    assert [r for r in rows_left(sampler, rows) if r not in (1, 3)] == [2, 8]
    for r in range(rows):
        w = small_workload(f"row{r}", x[r], cfgs[r], uniforms=uni[r:r + 1])
        got = tuple(t[r:r + 1].cpu().numpy() for t in (tok, pr, fl))
        assert_parity(w, got, O.run(w.logits, oracle_params(w.params), uniforms=w.uniforms), w.name)


@pytest.mark.parametrize("vocab", [32003, 50257, 65536, W.VOCAB])
@pytest.mark.parametrize("temperature,top_p", [(0.5, 1.0), (0.7, 0.9999), (1.0, 0.9999), (1.0, 1.0), (1.0, 2.0)])
def test_open_nuclei_take_no_sort(sampler, vocab, temperature, top_p):
    # most of the vocabulary lies in the last 2^-14 of the probability mass
    rng = np.random.default_rng(vocab)
    x = _rows(rng, 4, vocab, "wide")
    w = small_workload(f"open-{vocab}", x, dict(temperature=temperature, top_k=0, top_p=top_p, softcap=30.0),
                       uniforms=np.array([0.07, 0.43, 0.86, 0.99], np.float32))
    _check(sampler, w, left=[])


@pytest.mark.parametrize("vocab", [5003, 50257, W.VOCAB])
@pytest.mark.parametrize("allowed", [1, 2, 300, 0.1])
@pytest.mark.parametrize("params", [dict(top_p=0.9), dict(top_p=1.0), dict(top_p=0.0), dict(top_p=2.0),
                                    dict(top_p=1.0, min_p=0.05), dict(top_p=0.9, min_p=1e-6)])
def test_masked_rows_take_no_sort(sampler, vocab, allowed, params):
    # tokens at -inf (constrained decoding), all but a few or a tenth
    rng = np.random.default_rng(vocab + int(10 * allowed))
    x = _rows(rng, 4, vocab, "wide")
    n = allowed if allowed >= 1 else int(vocab * allowed)
    for r in range(4):
        x[r, rng.permutation(vocab)[n:]] = -np.inf
    x[3] = np.where(np.isinf(x[3]), np.float32(-1e30), x[3])
    w = small_workload(f"masked-{vocab}-{n}", x, dict(dict(temperature=1.0, top_k=0, softcap=0.0), **params),
                       uniforms=np.array([0.0, 0.3, 0.9, 0.995], np.float32))
    _check(sampler, w, left=[])
    w.uniforms[:] = np.float32(1 - 2**-24)  # the last kept token, wherever it lies
    _check(sampler, w)


@pytest.mark.parametrize("vocab", [5003, 32003, W.VOCAB])
@pytest.mark.parametrize("first", [9.0, 14.0, 20.0, 30.0])
@pytest.mark.parametrize("top_p", [0.95, 1.0])
def test_one_probability_holds_the_nucleus(sampler, vocab, first, top_p):
    # a confident row: its first probability reaches top_p, or nearly 1, alone
    rng = np.random.default_rng(vocab)
    x = (rng.standard_normal((6, vocab)) * 1.2).astype(np.float32)
    x[:, 7] = first
    u = np.array([0.0, 0.55, 0.8, 0.96, 0.9999, float(np.float32(1 - 2**-24))], np.float32)
    _check(sampler, small_workload(f"confident-{vocab}", x, dict(temperature=0.7, top_k=0, top_p=top_p), uniforms=u))
    assert [r for r in rows_left(sampler, 6) if r < 4] == []
