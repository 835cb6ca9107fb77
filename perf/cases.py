"""The work that users of this library have it do, as cases that can be timed.

A case is one call (or, where B is new on every call, a pack and a call) of the Python entry points: `dots_packed`,
`angulars_packed`, `euclideans_packed` over an image made by `dots_pack`, and the symmetric kinds over one set of vectors.
Operands and results live in GPU memory, the results in a matrix that the caller keeps (`out=`).

Sizes are those of this repository's configurations, tests and benchmark (2048^3, 8192^3, 8192 x 8191 x 1000, the retrieval
shape 1024 x 1,048,576 x 768) or generic ones for searching vectors: a few to a thousand queries against tens of thousands
to a million vectors of 100 to 1000 dimensions, depths that are a multiple of nothing among them.
"""
import math

import torch

import numkong_amd as nk

# op: dots, angular, euclidean (packed kinds: `m` queries against `n` packed vectors of depth `k`); fresh_dots (the same
# product, but B is packed in the pass: it is new each time); symmetric_dots, symmetric_angular, symmetric_euclidean (all
# pairs of `n` vectors of depth `k`, upper triangle; `m` equals `n`).


def listed():
    return [
        # One query against a small table, the call of an interactive search: latency, not throughput.
        {"name": "lookup_i8", "op": "dots", "dtype": "i8", "m": 1, "n": 10000, "k": 256},
        # A middling product of integers: quantised layers, and the smallest of this repository's configurations.
        {"name": "square_i8_2048", "op": "dots", "dtype": "i8", "m": 2048, "n": 2048, "k": 2048},
        # A server's batch of queries against an index of half-precision embeddings: the stream of the index is the work.
        {"name": "search_bf16", "op": "angular", "dtype": "bf16", "m": 32, "n": 262144, "k": 768},
        # The retrieval configuration: every score of a thousand queries against a million vectors.
        {"name": "retrieval_i8", "op": "dots", "dtype": "i8", "m": 1024, "n": 1048576, "k": 768},
        # Descriptors of bytes with an odd number of dimensions, rows that start on odd addresses, a ragged table.
        {"name": "descriptors_u8", "op": "euclidean", "dtype": "u8", "m": 1000, "n": 500009, "k": 301},
        # The three types that the headline metric names, at its size.
        {"name": "square_i8_8192", "op": "dots", "dtype": "i8", "m": 8192, "n": 8192, "k": 8192},
        {"name": "square_bf16_8192", "op": "dots", "dtype": "bf16", "m": 8192, "n": 8192, "k": 8192},
        {"name": "square_e4m3_8192", "op": "dots", "dtype": "e4m3", "m": 8192, "n": 8192, "k": 8192},
        # The ragged configuration: no dimension but the first is a multiple of a tile, rows of C off every line.
        {"name": "ragged_f16", "op": "dots", "dtype": "f16", "m": 8192, "n": 8191, "k": 1000},
        # All pairs of one collection, as clustering and the removal of duplicates ask for them.
        {"name": "pairs_bf16", "op": "symmetric_angular", "dtype": "bf16", "m": 8192, "n": 8192, "k": 768},
        # A table that is new: packed and asked once (packing is most of it).
        {"name": "index_i8", "op": "fresh_dots", "dtype": "i8", "m": 16, "n": 1048576, "k": 768},
        # Single-precision vectors with the results in double precision.
        {"name": "search_f32", "op": "angular", "dtype": "f32", "m": 1000, "n": 20001, "k": 300},
    ]


_FLOAT_BITS = {"bf16": 16, "f16": 16, "f32": 32, "f64": 64, "e4m3": 8, "e5m2": 8, "e2m3": 8, "e3m2": 8}
_INTEGER_BITS = {"i8": 8, "u8": 8, "i4": 4, "u4": 4, "u1": 1}
_TORCH = {"i8": torch.int8, "u8": torch.uint8, "bf16": torch.bfloat16, "f16": torch.float16, "e4m3": torch.float8_e4m3fn,
          "e5m2": torch.float8_e5m2, "f32": torch.float32, "f64": torch.float64}  # the others come as bytes


def _cost(case):
    """A rough time in seconds, for keeping drawn cases within the largest listed one."""
    rate = {"f32": 50e12, "f64": 5e12}.get(case["dtype"], 1e15)
    needed = work(case)
    return needed["flops"] / rate + needed["bytes"] / 4e12


def draw(rng):
    """One more case: any kind, any type, sizes over the whole range, a third of them plain multiples, the rest ragged."""
    def size(low, high, odd):
        value = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
        if odd:
            return max(low, value | 1)
        step = 256 if value >= 1024 else (64 if value >= 128 else 1)
        return max(low, value // step * step)

    op = rng.choice(["dots", "dots", "dots", "angular", "angular", "euclidean", "fresh_dots", "symmetric_dots",
                     "symmetric_angular", "symmetric_euclidean"])
    dtype = rng.choice(["i8", "i8", "u8", "bf16", "bf16", "f16", "e4m3", "e5m2", "e2m3", "e3m2", "i4", "u4", "u1", "f32", "f64"])
    if dtype == "u1" and op in ("angular", "euclidean"):
        op = "dots"
    if dtype == "u1" and op.startswith("symmetric"):
        op = "symmetric_dots"
    case = {"op": op, "dtype": dtype, "k": size(64, 8192, rng.random() < 0.5)}
    if op.startswith("symmetric"):
        case["n"] = size(256, 16384, rng.random() < 0.6)
        case["m"] = case["n"]
    else:
        case["m"] = size(1, 8192, rng.random() < 0.6)
        case["n"] = size(1024, 1048576, rng.random() < 0.6)
    limit = max(_cost(one) for one in listed())
    while _cost(case) > limit:  # the wider side shrinks until the case costs no more than the largest listed one
        if op.startswith("symmetric"):
            case["n"] = case["m"] = case["n"] * 3 // 4
        elif case["n"] >= case["m"]:
            case["n"] = case["n"] * 3 // 4
        else:
            case["m"] = case["m"] * 3 // 4
    return case


def _vectors(dtype, rows, k, generator, centres):
    """`rows` vectors as a user of the type has them. Floats are embeddings: half of a vector's length is one of a
    thousand common centres, the rest its own (cosines near zero between strangers, near a half between relatives).
    Integers fill their range, as quantised data does; the 8-bit floats span half of theirs, as scaled data does."""
    device = "cuda:0"
    if dtype == "i8":
        return torch.randint(-128, 128, (rows, k), dtype=torch.int8, device=device, generator=generator)
    if dtype == "u8":
        return torch.randint(0, 256, (rows, k), dtype=torch.uint8, device=device, generator=generator)
    if dtype in ("i4", "u4", "u1"):
        values = {"u1": 8}.get(dtype, 2)
        return torch.randint(0, 256, (rows, (k + values - 1) // values), dtype=torch.uint8, device=device, generator=generator)
    if dtype in ("e2m3", "e3m2"):
        return torch.randint(0, 64, (rows, k), dtype=torch.uint8, device=device, generator=generator)
    out = torch.empty((rows, k), dtype=_TORCH[dtype], device=device)
    slab = max(1, (1 << 27) // max(k, 1))
    for first in range(0, rows, slab):
        here = min(slab, rows - first)
        values = torch.randn((here, k), device=device, generator=generator)
        values.mul_(0.5 ** 0.5)
        which = torch.randint(0, centres.shape[0], (here,), device=device, generator=generator)
        values.add_(centres[which], alpha=0.5 ** 0.5)
        if dtype in ("e4m3", "e5m2"):
            top = 448.0 if dtype == "e4m3" else 57344.0
            values.mul_(0.5 * top).clamp_(-top, top)
        out[first:first + here] = values.to(_TORCH[dtype])
    return out


def _depth(case):
    """Sub-byte types come as whole bytes, so their depth is what these hold."""
    values = {"u1": 8, "i4": 2, "u4": 2}.get(case["dtype"], 1)
    return (case["k"] + values - 1) // values * values


def _result_dtype(case):
    if case["dtype"] in ("f32", "f64"):
        return torch.float64
    return torch.int32 if case["dtype"] in _INTEGER_BITS and case["op"].endswith("dots") else torch.float32


_CALLS = {"dots": nk.dots_packed, "angular": nk.angulars_packed, "euclidean": nk.euclideans_packed,
          "symmetric_dots": nk.dots_symmetric, "symmetric_angular": nk.angulars_symmetric,
          "symmetric_euclidean": nk.euclideans_symmetric}


def prepare(case, seed):
    """The queries, the packed table (or the table itself where the pass packs it) and the matrix for the results."""
    generator = torch.Generator(device="cuda:0").manual_seed(seed)
    centres = torch.randn((1024, case["k"]), device="cuda:0", generator=generator)
    state = {"op": case["op"], "dtype": case["dtype"]}
    if case["op"].startswith("symmetric"):
        state["vectors"] = _vectors(case["dtype"], case["n"], case["k"], generator, centres)
        state["out"] = torch.zeros((case["n"], case["n"]), dtype=_result_dtype(case), device="cuda:0")
        return state
    state["a"] = _vectors(case["dtype"], case["m"], case["k"], generator, centres)
    b = _vectors(case["dtype"], case["n"], case["k"], generator, centres)
    if case["op"] == "fresh_dots":
        state["b"] = b
    else:
        state["packed"] = nk.dots_pack(b, case["dtype"])
    state["out"] = torch.empty((case["m"], case["n"]), dtype=_result_dtype(case), device="cuda:0")
    return state


def run(state):
    """One pass."""
    op = state["op"]
    if op.startswith("symmetric"):
        return _CALLS[op](state["vectors"], state["dtype"], out=state["out"])
    if op == "fresh_dots":
        return nk.dots_packed(state["a"], nk.dots_pack(state["b"], state["dtype"]), out=state["out"])
    return _CALLS[op](state["a"], state["packed"], out=state["out"])


def work(case):
    """Operands read once at the caller's width, results written once (of the symmetric kinds the upper triangle), a
    multiplication and an addition per pair of values. The packed table counts at the caller's width as well: how it is
    held is the library's affair."""
    dtype, n, k = case["dtype"], case["n"], _depth(case)
    row = k * (_FLOAT_BITS.get(dtype) or _INTEGER_BITS[dtype]) // 8
    width = 8 if dtype in ("f32", "f64") else 4
    if case["op"].startswith("symmetric"):
        pairs = n * (n + 1) // 2
        return {"bytes": n * row + pairs * width, "flops": 2 * pairs * k}
    return {"bytes": (case["m"] + n) * row + case["m"] * n * width, "flops": 2 * case["m"] * n * k}


def tolerance(case):
    """Whole numbers are exact. The rest: the 2-norm of the error over that of the result, about four times the most that
    the path shows against the same arithmetic in 64 bits (sums of 32 bits 1.3e-7 at depth 8192, distances made from them
    4.3e-8; f32 and f64 inputs, summed in 64 bits, 4.4e-16 and 1.3e-16)."""
    if _result_dtype(case) == torch.int32:
        return "exact"
    sums = case["op"].endswith("dots")
    if case["dtype"] in ("f32", "f64"):
        return {"rel": 2e-15 if sums else 6e-16}
    return {"rel": 5e-7 if sums else 2e-7}
