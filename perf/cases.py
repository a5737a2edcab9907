"""The work a user of the tensor API has it do, case by case, for timing and for comparing outputs.

A case names a stored tensor (dtype, shape), the view of it that is worked on and the calls made on that
view, in order. Inputs are device memory of the caller (`Tensor.from_raw`); every result is the fresh
tensor that the call returns, handed on without a copy. `listed()` are the sizes that the benchmark and the
tests use; `draw()` spreads the same calls over the whole range, from calls that are all latency to ones
of a few hundred megabytes, with odd sizes among them.
"""
from __future__ import annotations

import math

import torch

import hpt_amd as hpt

_DTYPES = {
    "f32": (hpt.f32, torch.float32),
    "f16": (hpt.f16, torch.float16),
    "bf16": (hpt.bf16, torch.bfloat16),
    "i32": (hpt.i32, torch.int32),
}
# how a result is described to torch (bf16 travels as its bits)
_TYPESTR = {"f32": "<f4", "f16": "<f2", "bf16": "<i2", "i32": "<i4", "i64": "<i8"}
_SIZE = {"f32": 4, "f16": 2, "bf16": 2, "i32": 4}

_EPS = 1e-5
_SCALE = 0.125  # of attention scores, 1 / sqrt(64)


def listed():
    return [
        # A small problem, 4 MB that sit in cache: the time is launches and host work (one head's scores,
        # a classifier's batch).
        {"name": "small_rows_f32", "dtype": "f32", "shape": "1024x1024", "view": "whole", "calls": "softmax 1; sum 1; max 1"},
        # The normalisation of a transformer block in full precision: every token's hidden state.
        {"name": "layernorm_f32", "dtype": "f32", "shape": "8192x4096", "view": "whole", "calls": "layernorm"},
        # The same in half precision, with the residual added, at a hidden size that is no power of two.
        {"name": "add_layernorm_f16", "dtype": "f16", "shape": "13107x5120", "view": "whole", "calls": "add_layernorm"},
        # The output layer of a language model: log-probabilities over an odd vocabulary, and the greedy token.
        {"name": "vocabulary_f32", "dtype": "f32", "shape": "640x50257", "view": "whole", "calls": "log_softmax 1; argmax 1"},
        # Images: pooling, batch statistics, the strongest channel, the sum of everything.
        {"name": "images_f32", "dtype": "f32", "shape": "64x128x56x56", "view": "whole",
         "calls": "sum 2,3; mean 0,2,3; max 1; sum 0,1,2,3"},
        # Integer images: exact sums over the channels, the channel that wins.
        {"name": "images_i32", "dtype": "i32", "shape": "64x128x56x56", "view": "whole", "calls": "sum 1; argmax 1"},
        # Decoder attention, prefill: causal softmax of the scaled scores of 32 heads.
        {"name": "causal_bf16", "dtype": "bf16", "shape": "32x2048x2048", "view": "whole", "calls": "softmax_causal"},
        # Softmax along an axis in the middle of a large tensor (attention laid out otherwise, channels); the
        # largest case.
        {"name": "cube_softmax_f32", "dtype": "f32", "shape": "512x512x512", "view": "whole", "calls": "softmax 1"},
        # A transposed half-precision view, used as it is: nothing is made contiguous first.
        {"name": "transposed_f16", "dtype": "f16", "shape": "4096x8192", "view": "transposed",
         "calls": "layernorm; softmax 1; sum 0"},
        # Every second element of the rows of a half-precision tensor.
        {"name": "stepped_f16", "dtype": "f16", "shape": "4096x8192", "view": "stepped", "calls": "layernorm; softmax 1; sum 0"},
        # Down the columns, rows of odd length: bias gradients, weights over the tokens.
        {"name": "columns_f32", "dtype": "f32", "shape": "8190x4097", "view": "whole", "calls": "sum 0; softmax 0"},
        # Point clouds: a few coordinates per point, everything over the points.
        {"name": "points_f32", "dtype": "f32", "shape": "5592x2000x3", "view": "whole", "calls": "max 1; mean 1; softmax 1"},
    ]


# ---- drawn cases --------------------------------------------------------------------------------

_MOST = 1 << 25  # elements of a drawn tensor


def _spread(rng, lo, hi):
    """A size between lo and hi, spread over its logarithm; half of them rounded to what sizes mostly are."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        step = 64 if n >= 512 else 8 if n >= 32 else 1
        n = n // step * step
    return max(lo, min(hi, n))


def _floats(rng):
    return rng.choice(["f32", "f32", "f16", "bf16"])


def _draw_rows(rng):
    cols = _spread(rng, 64, 16384)
    rows = _spread(rng, 16, max(16, min(131072, _MOST // cols)))
    calls = rng.choice(["softmax 1; sum 1; max 1", "layernorm", "layernorm", "add_layernorm", "log_softmax 1"])
    return _floats(rng), (rows, cols), "whole", calls


def _draw_vocabulary(rng):
    cols = _spread(rng, 16384, 152000)
    return _floats(rng), (_spread(rng, 1, _MOST // cols), cols), "whole", "log_softmax 1; argmax 1"


def _draw_images(rng):
    side = _spread(rng, 7, 112)
    channels = _spread(rng, 3, 512)
    batch = _spread(rng, 1, max(1, min(64, _MOST // (channels * side * side))))
    if rng.random() < 0.3:
        return "i32", (batch, channels, side, side), "whole", "sum 1; argmax 1"
    return _floats(rng), (batch, channels, side, side), "whole", "sum 2,3; mean 0,2,3; max 1; sum 0,1,2,3"


def _draw_causal(rng):
    # prefill (as many queries as keys), a chunk of a longer context, or one step of decoding
    keys = _spread(rng, 64, 4096)
    queries = rng.choice([keys, keys, _spread(rng, 1, keys), 1])
    heads = _spread(rng, 8, max(8, min(512, _MOST // (keys * queries))))
    return rng.choice(["bf16", "bf16", "f16"]), (heads, queries, keys), "whole", "softmax_causal"


def _draw_cube(rng):
    a = _spread(rng, 8, 512)
    b = _spread(rng, 16, 512)
    c = _spread(rng, 16, max(16, min(4096, _MOST // (a * b))))
    return _floats(rng), (a, b, c), "whole", rng.choice(["softmax 1", "softmax 1", "softmax 0"])


def _draw_view(rng):
    cols = _spread(rng, 128, 16384)
    rows = _spread(rng, 128, max(128, min(16384, _MOST // cols)))
    return _floats(rng), (rows, cols), rng.choice(["transposed", "stepped"]), "layernorm; softmax 1; sum 0"


def _draw_columns(rng):
    cols = _spread(rng, 16, 8192)
    rows = _spread(rng, 256, max(256, min(1 << 20, _MOST // cols)))
    return _floats(rng), (rows, cols), "whole", rng.choice(["sum 0; softmax 0", "sum 0"])


def _draw_points(rng):
    width = rng.randint(2, 8)
    points = _spread(rng, 64, 4096)
    clouds = _spread(rng, 64, max(64, min(16384, _MOST // (points * width))))
    return _floats(rng), (clouds, points, width), "whole", "max 1; mean 1; softmax 1"


def draw(rng):
    kind = rng.choice([_draw_rows, _draw_rows, _draw_vocabulary, _draw_images, _draw_causal, _draw_cube, _draw_view,
                       _draw_columns, _draw_points])
    dtype, shape, view, calls = kind(rng)
    return {"dtype": dtype, "shape": "x".join(str(s) for s in shape), "view": view, "calls": calls}


# ---- one case -----------------------------------------------------------------------------------


def _shape(case):
    return [int(s) for s in case["shape"].split("x")]


def _view_shape(case):
    s = _shape(case)
    if case["view"] == "transposed":
        return s[::-1]
    if case["view"] == "stepped":
        return s[:-1] + [(s[-1] + 1) // 2]
    return s


def _calls(case):
    """[(method, axes)] of a case's calls."""
    out = []
    for c in case["calls"].split(";"):
        name, _, axes = c.strip().partition(" ")
        out.append((name, [int(a) for a in axes.split(",")] if axes else []))
    return out


def _values(case, shape, gen):
    """What the path meets in earnest: logits within +-10 or so, hidden states with an offset per row."""
    dtype = _DTYPES[case["dtype"]][1]
    if dtype == torch.int32:
        return torch.randint(-1000, 1001, shape, generator=gen, device="cuda", dtype=torch.int32)
    x = torch.empty(shape, device="cuda", dtype=dtype)
    first = _calls(case)[0][0]
    if first == "softmax_causal":
        return x.normal_(0, 3 / _SCALE, generator=gen)
    if first == "layernorm" and case["view"] == "whole":
        off = torch.empty(shape[:-1] + [1], device="cuda", dtype=dtype).uniform_(-5, 5, generator=gen)
        return x.normal_(0, 1, generator=gen).add_(off)
    if first in ("softmax", "log_softmax"):
        return x.normal_(0, 3, generator=gen)
    return x.normal_(0, 1 if case["view"] == "whole" else 2, generator=gen)


def _hpt(t, name):
    """The caller's device memory as a tensor of the framework; nothing is copied."""
    return hpt.Tensor.from_raw(t.data_ptr(), list(t.shape), _DTYPES[name][0])


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    name = case["dtype"]
    shape = _shape(case)
    stored = _values(case, shape, gen)
    x = _hpt(stored, name)
    if case["view"] == "transposed":
        x = x.permute([1, 0])
    elif case["view"] == "stepped":
        x = x[:, ::2]
    keep = [stored]
    calls = []
    for method, axes in _calls(case):
        if method in ("layernorm", "add_layernorm"):
            cols = x.shape[-1]
            dtype = _DTYPES[name][1]
            gamma = torch.empty([cols], device="cuda", dtype=dtype).normal_(1, 0.1, generator=gen)
            beta = torch.empty([cols], device="cuda", dtype=dtype).normal_(0, 0.1, generator=gen)
            keep += [gamma, beta]
            args = [[cols], _hpt(gamma, name), _hpt(beta, name), _EPS]
            if method == "add_layernorm":
                residual = torch.empty(shape, device="cuda", dtype=dtype).normal_(0, 1, generator=gen)
                keep.append(residual)
                args.insert(0, _hpt(residual, name))
        elif method == "softmax_causal":
            # the last query sees every key
            args = [_SCALE, x.shape[-1] - x.shape[-2]]
        elif method in ("softmax", "log_softmax", "argmax"):
            args = [axes[0]]
        else:
            args = [axes]
        calls.append((method, args))
    return {"x": x, "calls": calls, "keep": keep}


class _Result:
    """A result's device memory as torch takes it over: the torch tensor keeps the framework's alive."""

    def __init__(self, t):
        self.t = t
        self.__cuda_array_interface__ = {"shape": tuple(t.shape), "typestr": _TYPESTR[t.dtype.name], "data": (t.ptr, False),
                                         "strides": None, "version": 2}


def _torch(t):
    r = torch.as_tensor(_Result(t), device="cuda")
    return r.view(torch.bfloat16) if t.dtype.name == "bf16" else r


def run(state):
    x = state["x"]
    return [_torch(getattr(x, method)(*args)) for method, args in state["calls"]]


def work(case):
    """Every call reads its input once (the causal softmax what lies below the diagonal) and writes its
    result once; a few operations per element."""
    shape = _view_shape(case)
    n = math.prod(shape)
    size = _SIZE[case["dtype"]]
    total = flops = 0
    for method, axes in _calls(case):
        read, written, per = n * size, n * size, 5
        if method == "softmax_causal":
            queries, keys = shape[-2], shape[-1]
            live = sum(min(keys, q + keys - queries + 1) for q in range(queries))
            read = shape[0] * live * size
        elif method == "layernorm":
            read, per = read + 2 * shape[-1] * size, 8
        elif method == "add_layernorm":
            read, per = 2 * read + 2 * shape[-1] * size, 9
        elif method in ("sum", "mean", "max", "argmax"):
            kept = math.prod(s for i, s in enumerate(shape) if i not in axes)
            written, per = kept * (8 if method == "argmax" else size), 1
        total += read + written
        flops += n * per
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """About four times what the calls differ by from the same calls in 64 bits (rel, largest of listed and drawn
    cases: f32 8.4e-8, f16 2.4e-4, bf16 1.8e-3; largest single difference: 4.2e-7, 5e-4, 4e-3)."""
    if case["dtype"] == "i32":
        return "exact"
    return {"f32": {"rel": 4e-7, "max": 2e-6}, "f16": {"rel": 1e-3, "max": 2e-3}, "bf16": {"rel": 7e-3, "max": 1.6e-2}}[case["dtype"]]
