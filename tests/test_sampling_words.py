"""What a draw takes beside the logits, as the host lays it out in one array of 32-bit words, against the same values row by row."""
import random

import numpy as np
import pytest

from inferrs_amd.sampling import Sampler, SamplingParams
from inferrs_amd.sampling.rng import rand_f32, rand_f32_many


def test_random_numbers_of_many_rows_are_those_of_each():
    rng = random.Random(3)
    seeds = [0, 1, -1, (1 << 64) - 1, 1 << 64] + [rng.randrange(-(1 << 70), 1 << 70) for _ in range(500)]
    steps = [0, 1, 7, 2 ** 31, 2 ** 40] + [rng.randrange(1 << 20) for _ in range(500)]
    out = np.zeros(len(seeds), np.float32)
    rand_f32_many(seeds, steps, out.ctypes.data)
    assert out.tolist() == [rand_f32(a, b) for a, b in zip(seeds, steps)]


@pytest.mark.parametrize("case", ["penalties", "biases", "both", "neither", "one row"])
def test_words_hold_every_rows_values(case):
    kw = [dict(), dict(temperature=0.0), dict(repetition_penalty=1.0), dict(repeat_last_n=3, frequency_penalty=0.5), dict(repeat_last_n=0),
          dict(temperature=0.0, repetition_penalty=1.0, presence_penalty=-1.0, top_k=0, min_p=0.25)]
    if case in ("biases", "neither"):
        kw = [dict(k, repetition_penalty=1.0, frequency_penalty=0.0, presence_penalty=0.0) for k in kw]
    if case in ("biases", "both"):
        kw[1]["logit_bias"], kw[4]["logit_bias"] = {9: 1e39, 2: -0.5}, {7: 1.25}
    params = [SamplingParams(**k) for k in kw[:1 if case == "one row" else None]]
    rows = len(params)
    previous = [list(range(100 + i, 100 + i + n)) for i, n in zip(range(rows), (70, 5, 9, 8, 4, 0))]
    seeds = [11 * i + 1 for i in range(rows)]
    words, width, n_bias, penalized = Sampler("cpu")._pack(params, previous, seeds)
    words = words.numpy()
    takes = [min(p.repeat_last_n, len(prev)) if p.has_penalty else 0 for p, prev in zip(params, previous)]
    assert (width, n_bias) == (max(takes), max(len(p.logit_bias) for p in params)) and penalized == bool(width or n_bias)
    at = 0

    def column(count, dtype):
        nonlocal at
        part = words[at:at + rows * count].view(dtype).reshape(rows, count)
        at += rows * count
        return part

    if penalized:
        window = column(width, np.int32)
        rep, freq, pres = (column(1, np.float32)[:, 0] for _ in range(3))
        ids, vals = column(n_bias, np.int32), column(n_bias, np.float32)
        for i, (p, prev, take) in enumerate(zip(params, previous, takes)):
            assert window[i].tolist() == prev[len(prev) - take:] + [-1] * (width - take)
            want = (p.repetition_penalty, p.frequency_penalty, p.presence_penalty) if take else (1.0, 0.0, 0.0)
            assert (rep[i], freq[i], pres[i]) == tuple(np.float32(v) for v in want)
            biases = sorted(p.logit_bias.items())
            assert ids[i].tolist() == [t for t, _ in biases] + [-1] * (n_bias - len(biases))
            with np.errstate(over="ignore"):
                assert vals[i].tolist() == [np.float32(v) for _, v in biases] + [0.0] * (n_bias - len(biases))
    temperature = column(1, np.float32)[:, 0]
    assert temperature.tolist() == [np.float32(p.draw_temperature(len(prev))) for p, prev in zip(params, previous)]
    assert column(1, np.int32)[:, 0].tolist() == [p.top_k for p in params]
    assert column(1, np.float32)[:, 0].tolist() == [np.float32(p.top_p) for p in params]
    assert column(1, np.float32)[:, 0].tolist() == [np.float32(p.min_p) for p in params]
    u = column(1, np.float32)[:, 0]
    for i, (prev, seed) in enumerate(zip(previous, seeds)):
        assert u[i] == (rand_f32(seed, len(prev)) if temperature[i] >= 1e-5 else 0.0)
    assert column(1, np.int32)[:, 0].tolist() == [-1] * rows and at == words.size


def test_words_of_parameters_in_other_number_types():
    """Whole numbers that come as floats or NumPy's, and a temperature that is no number beside rows at 0: every row as alone."""
    params = [SamplingParams(top_k=50.0), SamplingParams(top_k=np.int64(7), temperature=np.float32(0.5)), SamplingParams(temperature=float("nan")),
              SamplingParams(temperature=0.0), SamplingParams(temperature=0.0, repetition_penalty=1.0)]
    previous, seeds = [(1, 2, 3), [4, 5], range(8), [6], [7]], [1, 2, 3, 4, 5]
    words, width, _, _ = Sampler("cpu")._pack(params, previous, seeds)
    draw = words.numpy()[-6 * len(params):].reshape(6, -1)
    assert width == 8 and draw[1].tolist() == [50, 7, 50, 50, 50]
    for i, (p, prev, seed) in enumerate(zip(params, previous, seeds)):
        alone = Sampler("cpu")._pack([p], [prev], [seed])[0].numpy()[-6:]
        assert draw[:, i].tolist() == alone.tolist()
        t = p.draw_temperature(len(prev))
        assert np.array_equal(draw[0, i:i + 1].view(np.float32)[0], np.float32(t), equal_nan=True)
        assert draw[4, i:i + 1].view(np.float32)[0] == (rand_f32(seed, len(prev)) if t >= 1e-5 else 0.0)
