"""Turns rows of logits into tokens on the device, one row per request, in the reference's
order of operations (`inferrs/src/sampler.rs:146-335`): logit bias, repetition, frequency and
presence penalties over the last `repeat_last_n` tokens, temperature, softmax, top-k, top-p,
min-p, and the walk to a random number that depends on the request's seed and step only."""
from __future__ import annotations

from array import array
from struct import pack
from typing import List, Optional, Sequence

import numpy as np
import torch

from .. import ops
from .params import SAMPLING_EPS, SamplingParams, TokenLogprob
from .rng import rand_f32, rand_f32_many


class Sampler:
    def __init__(self, device):
        self.device = torch.device(device)

    def _upload(self, *arrays: Optional[np.ndarray]) -> List[Optional[torch.Tensor]]:
        """Arrays of 32-bit numbers on the device, in one copy that the host does not wait for (a draw of 24 rows brought
        nine arrays, each with a copy and a wait of its own: 317 us against 227 with this one)."""
        flat = [None if a is None else np.ascontiguousarray(a).reshape(-1) for a in arrays]
        host = torch.empty(max(1, sum(a.size for a in flat if a is not None)), dtype=torch.int32,
                           pin_memory=self.device.type == "cuda")
        words, at = host.numpy(), 0
        for a in flat:
            if a is not None:
                words[at:at + a.size] = a.view(np.int32)
                at += a.size
        dev, at, out = host.to(self.device, non_blocking=True), 0, []
        for array, a in zip(arrays, flat):
            if a is None:
                out.append(None)
                continue
            part = dev[at:at + a.size]
            out.append((part.view(torch.float32) if array.dtype == np.float32 else part).view(array.shape))
            at += a.size
        return out

    def _pack(self, params: Sequence[SamplingParams], previous: Sequence[Sequence[int]], seeds: Sequence[int]):
        """What a draw takes beside the logits, laid out as `ops.sample_packed` reads it, on its way to the device: (words, the
        windows' width, biases a row, whether there are penalties or biases).  A field at a time over all rows and one array of the
        interpreter's for each kind of number: 24 rows with windows of 64 had taken 110 us as NumPy rows and a random number each."""
        rows, lens = len(params), [len(prev) for prev in previous]
        last = [p.repeat_last_n for p in params]
        rep, freq, pres = ([p.repetition_penalty for p in params], [p.frequency_penalty for p in params],
                           [p.presence_penalty for p in params])
        # (rows without a penalty, and those with no token yet, have no window)
        takes = [min(k, n) if k > 0 and n > 0 and (r != 1.0 or f != 0.0 or q != 0.0) else 0
                 for k, n, r, f, q in zip(last, lens, rep, freq, pres)]
        width, n_bias = max(takes), max([len(p.logit_bias) for p in params])
        penalized = bool(width or n_bias)
        whole, real = [], []                                    # the arrays in front: 32-bit numbers, and what follows them
        if penalized:
            for prev, take in zip(previous, takes):
                if take:
                    whole += prev[-take:]
                if take < width:
                    whole += [-1] * (width - take)
            real += [r if take else 1.0 for r, take in zip(rep, takes)]
            real += [f if take else 0.0 for f, take in zip(freq, takes)]
            real += [q if take else 0.0 for q, take in zip(pres, takes)]
        # (packing arguments is twice as fast as an array out of a list, which takes numbers beyond 32 bits as infinities)
        parts = [pack(f"{len(whole)}i", *whole), array("f", real).tobytes()]
        if n_bias:
            pairs = [sorted(p.logit_bias.items()) for p in params]
            pairs = [row + [(-1, 0.0)] * (n_bias - len(row)) for row in pairs]
            parts.append(pack(f"{rows * n_bias}i", *[int(t) for row in pairs for t, _ in row]))
            parts.append(array("f", [v for row in pairs for _, v in row]).tobytes())
        temperature = [p.temperature for p in params]
        if not min(temperature) >= SAMPLING_EPS:                 # (a temperature that is no number hides the ones behind it)
            temperature = [p.draw_temperature(n) for p, n in zip(params, lens)]
        parts += [array("f", temperature).tobytes(), pack(f"{rows}i", *[int(p.top_k) for p in params]),
                  array("f", [p.top_p for p in params] + [p.min_p for p in params]).tobytes()]
        front = b"".join(parts)
        at = len(front)
        host = torch.empty(at // 4 + 2 * rows, dtype=torch.int32, pin_memory=self.device.type == "cuda")
        view = memoryview(host.numpy()).cast("B")
        view[:at] = front
        # the step of a draw is the number of tokens before it (`sampler.rs:323-325`); rows of temperature 0 draw nothing
        rand_f32_many(seeds, lens, host.data_ptr() + at)
        for i, t in enumerate(temperature):
            if not t >= SAMPLING_EPS:
                view[at + 4 * i:at + 4 * i + 4] = b"\0\0\0\0"
        view[at + 4 * rows:] = pack(f"{rows}i", *[p.top_logprobs if p.logprobs else -1 for p in params])
        return host.to(self.device, non_blocking=True), width, n_bias, penalized

    def begin_chain(self, params: Sequence[SamplingParams], previous: Sequence[Sequence[int]],
                    seeds: Sequence[int], steps: int) -> "ChainDraw":
        """The draws of the next `steps` decode steps of these requests, prepared for the device."""
        return ChainDraw(self, params, previous, seeds, steps)

    def sample(self, logits: torch.Tensor, params: Sequence[SamplingParams], previous: Sequence[Sequence[int]],
               seeds: Sequence[int]) -> List[int]:
        """`logits` float32 [rows, vocab] on the device; row i belongs to a request with
        `params[i]`, whose prompt and output so far are `previous[i]` and whose seed is `seeds[i]`."""
        return self.sample_with_logprobs(logits, params, previous, seeds)[0]

    def sample_with_logprobs(self, logits: torch.Tensor, params: Sequence[SamplingParams],
                             previous: Sequence[Sequence[int]], seeds: Sequence[int]):
        """(tokens, per row a `TokenLogprob` or None): the log-probabilities for the rows whose
        parameters ask for them (`sampler.rs:285-352`)."""
        rows = logits.shape[0]
        if not (len(params) == len(previous) == len(seeds) == rows):
            raise ValueError("one parameter set, token history and seed per row of logits")
        if rows == 0:
            return [], []
        if all(p.is_plain_greedy for p in params):
            return ops.argmax(logits).cpu().tolist(), [None] * rows

        words, width, n_bias, penalized = self._pack(params, previous, seeds)
        top_k = [int(p.top_k) for p in params]
        reports = any([p.logprobs for p in params])
        narrow = all_narrow(min(top_k), max(top_k), logits.shape[1])
        # (rows that report entries of a list which top_p or min_p may not end, to within what 32 bits round: one call for all)
        open_rows = [p for p in params if p.top_logprobs > 1 and p.top_p > 0.999 and p.min_p < 1e-6] if reports else ()
        if narrow and open_rows:
            narrow = ops.sample_is_narrow(int(open_rows[0].top_k), logits.shape[1], min(p.temperature for p in open_rows), 1.0, 0.0, 2,
                                          any(p.logit_bias for p in open_rows))
        if not logits.is_contiguous():
            logits = logits.clone()
        # (penalties and bias are applied on the way: the logits stay as they are)
        if not reports:
            out = ops.sample_packed(logits, words, width, n_bias, penalized=penalized, narrow_only=narrow)
            return out.cpu().tolist(), [None] * rows
        sizes = ([rows * width] + [rows] * 3 + [rows * n_bias] * 2 if penalized else []) + [rows] * 6
        *pen, temperature, top_k, top_p, min_p, u, n_top = words.split(sizes)
        penalties = None
        if penalized:
            window, rep, freq, pres, bias_ids, bias_vals = pen
            penalties = (window.view(rows, width) if width else None, *(t.view(torch.float32) for t in (rep, freq, pres)),
                         *((bias_ids.view(rows, n_bias), bias_vals.view(torch.float32).view(rows, n_bias)) if n_bias else (None, None)))
        temperature, top_p, min_p, u = (t.view(torch.float32) for t in (temperature, top_p, min_p, u))
        out, lp, ids = ops.sample(logits, temperature, top_k, top_p, min_p, u, n_top, penalties=penalties, narrow_only=narrow)
        tokens, lp, ids = out.cpu().tolist(), lp.cpu().tolist(), ids.cpu().tolist()
        infos = []
        for i, p in enumerate(params):
            if not p.logprobs:
                infos.append(None)
                continue
            top = tuple((t, v) for t, v in zip(ids[i], lp[i][1:]) if t >= 0)[:p.top_logprobs]
            infos.append(TokenLogprob(tokens[i], lp[i][0], top))
        return tokens, infos


def all_narrow(least: int, most: int, vocab: int) -> bool:
    """Rows whose top_k lies in `least` .. `most` all go `ops.sample`'s shortest way, where they report no more than the token drawn
    and the first entry."""
    return 0 < least and most <= min(ops.sample_narrow_top(), vocab - 1)


class ChainDraw:
    """The draws of a run of decode steps that are queued without the host in between: what
    `Sampler.sample` works out from the token lists at every step is kept on the device here, the
    random numbers of all steps (they depend on seed and step only) and every row's penalty window,
    which takes the row's new token after each draw.  The tokens are those of single steps."""

    def __init__(self, sampler: "Sampler", params: Sequence[SamplingParams], previous: Sequence[Sequence[int]],
                 seeds: Sequence[int], steps: int):
        if any(p.logprobs for p in params):
            raise ValueError("log-probabilities are reported step by step, not from a run of steps")
        rows = len(params)
        self.greedy = all(p.is_plain_greedy for p in params)
        if self.greedy:
            return
        caps = np.asarray([p.repeat_last_n if p.has_penalty else 0 for p in params], dtype=np.int32)
        width = int(caps.max()) if rows else 0
        n_bias = max(len(p.logit_bias) for p in params)
        self.penalized = bool(width or n_bias)
        window = rep = freq = pres = ids = vals = None
        if self.penalized:
            rep, freq, pres = np.ones(rows, np.float32), np.zeros(rows, np.float32), np.zeros(rows, np.float32)
            window = np.full((rows, max(width, 1)), -1, dtype=np.int32)
            for i, (p, prev) in enumerate(zip(params, previous)):
                if p.has_penalty:
                    tail = list(prev[-p.repeat_last_n:])
                    window[i, :len(tail)] = tail
                    rep[i], freq[i], pres[i] = p.repetition_penalty, p.frequency_penalty, p.presence_penalty
            if n_bias:
                ids = np.full((rows, n_bias), -1, dtype=np.int32)
                vals = np.zeros((rows, n_bias), dtype=np.float32)
                for i, p in enumerate(params):
                    for j, (tid, b) in enumerate(sorted(p.logit_bias.items())):
                        ids[i, j], vals[i, j] = int(tid), float(b)
        # (a window that holds a token at the run's start holds one at every step of it)
        temperature = np.asarray([p.draw_temperature(len(prev)) for p, prev in zip(params, previous)], dtype=np.float32)
        top_k = np.asarray([p.top_k for p in params], dtype=np.int32)
        top_p = np.asarray([p.top_p for p in params], dtype=np.float32)
        min_p = np.asarray([p.min_p for p in params], dtype=np.float32)
        self.least_k, self.most_k = int(top_k.min()), int(top_k.max())
        # the step of a draw is the number of tokens before it (`sampler.rs:323-325`)
        u = np.asarray([[rand_f32(seed, len(prev) + i) if p.draw_temperature(len(prev)) >= SAMPLING_EPS else 0.0
                         for p, prev, seed in zip(params, previous, seeds)] for i in range(steps)],
                       dtype=np.float32).reshape(steps, rows)
        (self.window, self.caps, self.bias_ids, self.bias_vals, self.rep, self.freq, self.pres, self.temperature, self.top_k,
         self.top_p, self.min_p, self.u) = sampler._upload(window if width else None, caps if width else None, ids, vals, rep, freq,
                                                            pres, temperature, top_k, top_p, min_p, u)

    def pick(self, logits: torch.Tensor, step: int, out: torch.Tensor) -> None:
        """The tokens of the run's `step`-th step from its logits, into `out` (int32 [rows], on the device)."""
        if self.greedy:
            ops.argmax(logits, out=out)
            return
        penalties = (self.window, self.rep, self.freq, self.pres, self.bias_ids, self.bias_vals) if self.penalized else None
        ops.sample(logits, self.temperature, self.top_k, self.top_p, self.min_p, self.u[step], penalties=penalties,
                   narrow_only=all_narrow(self.least_k, self.most_k, logits.shape[1]), out=out)
        if self.window is not None:
            ops.window_push(self.window, self.caps, out)
