"""The work a user of this encoder has it do, as timed cases through its public entry points.

Six kinds of call, over the sizes of the repository's own configurations (a 256 x 512 tiny expert, a 5120 x 1536
expert, a 7168 x 2048 expert and its 384-expert layer):

* ``tiles``   the tile quantizer alone (``quantize_tiles``), from one small matrix's row step to a layer's
* ``ldlq``    the batched mixed-rate feedback recursion (``ldlq_mixed_batched``) of a layer's experts
* ``encode``  a whole matrix from weight and captured Hessian to packed payload (``quantize_qsrt``)
* ``gram``    Hessian capture (``gram_``), bf16 calibration rows or float32 activations
* ``rotate``  the blockwise Hadamard rotations (``rotate_``), both sides, float32 and float64
* ``decode``  packed payloads back to weights: one matrix (``decode_words``) or a layer's (``DecodePlan``)
"""

from __future__ import annotations

import math

import torch

from qsrt_amd import exl3_encoder_backend as backend
from qsrt_amd.decode import DecodePlan, decode_words
from qsrt_amd.gemm import gram_
from qsrt_amd.hadamard import rotate_
from qsrt_amd.ldlq import make_shared_h
from qsrt_amd.sqg_e4m3 import sqg_xor_cheb_t12_bytes

DEV = "cuda:0"
RHO = 0.85  # correlation of neighbouring calibration channels


def listed():
    return [
        # One 16-row step of the tiny expert's gate (512 / 16 columns of tiles): far fewer tiles than compute units.
        {"name": "tiles_k2_tiny", "kind": "tiles", "n": 32, "bits": 2, "context": 128},
        # The K4 records of a layer step (40 members x 16 tiles).
        {"name": "tiles_k4_group", "kind": "tiles", "n": 640, "bits": 4, "context": 128},
        # The K3 records of a layer step (40 members x 112 tiles): the bulk of a layer's encode.
        {"name": "tiles_k3_layer", "kind": "tiles", "n": 4480, "bits": 3, "context": 128},
        # Eight members of a layer step, 14 K3 and 2 K4 records each, over the last 256 input channels.
        {"name": "ldlq_mixed", "kind": "ldlq", "members": 8, "k": 256, "n": 2048, "k4_records": 2},
        # The tiny expert's gate, whole.
        {"name": "encode_k2_tiny", "kind": "encode", "k": 256, "n": 512, "bits": 2},
        # A strip of the 5120 x 1536 expert's gate, whole.
        {"name": "encode_k3_strip", "kind": "encode", "k": 1024, "n": 1536, "bits": 3},
        # Calibration rows that a layer's average expert sees (65,536 tokens over 384 experts).
        {"name": "gram_routed", "kind": "gram", "rows": 171, "k": 7168, "dtype": "bf16"},
        # Calibration rows of a single encoded expert.
        {"name": "gram_capture", "kind": "gram", "rows": 16384, "k": 7168, "dtype": "bf16"},
        # The down projection's Hessian from the float32 activations of the reconstructed gate and up.
        {"name": "gram_activations", "kind": "gram", "rows": 16384, "k": 2048, "dtype": "f32"},
        # Change of basis of one expert matrix, sign vectors fused.
        {"name": "rotate_expert", "kind": "rotate", "k": 7168, "n": 2048, "block": 128, "dtype": "f32"},
        # One expert matrix decoded on its own.
        {"name": "decode_one", "kind": "decode", "k": 7168, "n": 2048, "bits": 3, "experts": 0, "dtype": "bf16"},
        # Sixteen experts of a mixed-rate layer through one prepared plan.
        {"name": "decode_layer", "kind": "decode", "k": 7168, "n": 2048, "bits": 3, "experts": 16, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["tiles", "tiles", "ldlq", "encode", "gram", "rotate", "decode"])
    if kind == "tiles":
        return {"kind": kind, "n": _log(rng, 1, 4000), "bits": rng.choice([2, 3, 4]),
                "context": rng.choice([128, 128, 128, rng.randint(1, 127)])}
    if kind == "ldlq":
        n = 128 * rng.randint(2, 16)
        return {"kind": kind, "members": rng.randint(1, 8), "k": 128 * rng.randint(1, 2), "n": n,
                "k4_records": rng.randint(1, n // 128 - 1)}
    if kind == "encode":
        return {"kind": kind, "k": 128 * rng.randint(1, 8), "n": 128 * rng.randint(1, 12), "bits": rng.choice([2, 3, 4])}
    if kind == "gram":
        dtype = rng.choice(["bf16", "bf16", "f32"])
        return {"kind": kind, "rows": _log(rng, 1, 16384), "k": 16 * _log(rng, 16, 448 if dtype == "bf16" else 128),
                "dtype": dtype}
    if kind == "rotate":
        block = rng.choice([64, 128, 128, 256, 512])
        dtype = rng.choice(["f32", "f64"])
        return {"kind": kind, "k": 512 * rng.randint(1, 14), "n": 512 * rng.randint(1, 14 if dtype == "f32" else 7),
                "block": block, "dtype": dtype}
    return {"kind": kind, "k": 128 * _log(rng, 1, 56), "n": 128 * _log(rng, 1, 56), "bits": rng.choice([2, 3, 4]),
            "experts": 0, "dtype": rng.choice(["bf16", "bf16", "f32"])}


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) + 1)


def _correlated(rows, k, gen):
    """``[rows, k]`` float32 rows whose neighbouring channels correlate like ``RHO ** distance``."""

    lag = torch.arange(k, device=DEV)
    cov = torch.pow(torch.tensor(RHO, device=DEV), (lag[:, None] - lag[None, :]).abs().float())
    return torch.randn((rows, k), generator=gen, device=DEV) @ torch.linalg.cholesky(cov).T


def _heavy_tailed(shape, gen):
    """Weights of a trained matrix: normal with a chi-square-like spread of scales (heavy tails), std about 0.02."""

    z = torch.randn(shape, generator=gen, device=DEV)
    s = torch.randn((5, *shape), generator=gen, device=DEV).square().mean(dim=0).sqrt()
    return 0.02 * math.sqrt(3 / 5) * z / s


def _quant_args(bits, seed):
    return {"K": bits, "seed": 1000 + seed, "sv_seed": 2000 + seed, "sigma_reg": 0.01, "devices": [DEV],
            "apply_out_scales": False, "tailbite_context": 128, "sqg_e4m3_lut": sqg_xor_cheb_t12_bytes(bits)}


def prepare(case, seed):
    gen, kind = _gen(seed), case["kind"]
    if kind == "tiles":
        return {"kind": kind, "tiles": torch.randn((case["n"], 256), generator=gen, device=DEV),
                "args": {"K": case["bits"], "devices": [DEV], "tailbite_context": case["context"],
                         "sqg_e4m3_lut": sqg_xor_cheb_t12_bytes(case["bits"])}}
    if kind == "ldlq":
        k, n, members = case["k"], case["n"], case["members"]
        weights = torch.randn((members, k, n), generator=gen, device=DEV).double()
        factors = []
        for _ in range(members):
            x = _correlated(2 * k, k, gen)
            shared = make_shared_h(k, torch.device(DEV), x.T @ x)
            shared["count"] = 2 * k
            factors.append(backend.finalize_capture_H(shared, _quant_args(3, seed), False)[2])
        bits = [3] * (n // 16)
        for record in range(case["k4_records"]):  # the low records take the higher rate
            bits[8 * record:8 * record + 8] = [4] * 8
        args = {"devices": [DEV], "mixed_rate_axis": "n", "mixed_tile_bits": bits, "tailbite_context": 128,
                "sqg_e4m3_luts_by_bits": {b: sqg_xor_cheb_t12_bytes(b) for b in (3, 4)}}
        return {"kind": kind, "weights": weights, "Ls": torch.stack(factors), "args": [args] * members}
    if kind == "encode":
        k, n = case["k"], case["n"]
        x = _correlated(4 * k, k, gen)
        return {"kind": kind, "weight": _heavy_tailed((k, n), gen), "hessian": x.T @ x, "count": 4 * k,
                "args": _quant_args(case["bits"], seed % 100000)}
    if kind == "gram":
        x = torch.randn((case["rows"], case["k"]), generator=gen, device=DEV)
        return {"kind": kind, "x": x.to(torch.bfloat16) if case["dtype"] == "bf16" else x}
    if kind == "rotate":
        dtype = torch.float32 if case["dtype"] == "f32" else torch.float64
        x = torch.randn((case["k"], case["n"]), generator=gen, device=DEV).to(dtype)
        signs = [torch.where(torch.rand(m, generator=gen, device=DEV) < 0.5, -1.0, 1.0).to(dtype)
                 for m in (case["k"], case["n"])]
        return {"kind": kind, "x": x, "su": signs[0], "sv": signs[1], "block": case["block"]}
    k, n, bits, experts = case["k"], case["n"], case["bits"], case["experts"]
    dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32

    def words(count):
        return torch.randint(-32768, 32768, (count,), generator=gen, device=DEV, dtype=torch.int32).to(torch.int16)

    def scales(count):
        return (0.5 + torch.rand(count, generator=gen, device=DEV)).half()

    if not experts:
        return {"kind": kind, "words": words(k * n // 16 * bits).reshape(k // 16, n // 16, 16 * bits), "su": scales(k),
                "sv": scales(n), "bits": bits, "lut": sqg_xor_cheb_t12_bytes(bits).to(DEV), "dtype": dtype}
    records = [4] * 2 + [bits] * (n // 128 - 2)  # along the intermediate axis: columns of gate and up, rows of down
    per = sum(8 * (k // 16) * 16 * b for b in records)
    out = [torch.empty((2 * experts, k, n), dtype=dtype, device=DEV), torch.empty((experts, n, k), dtype=dtype, device=DEV)]
    payloads = []
    for axis, stack in zip("nk", out):
        for one in stack:
            payloads.append((words(per), records, axis, scales(one.shape[0]).float() / 128.0,
                             scales(one.shape[1]).float(), one))
    plan = DecodePlan.for_records(payloads, {b: sqg_xor_cheb_t12_bytes(b).to(DEV) for b in set(records)},
                                  out_dtype=dtype)
    return {"kind": kind, "plan": plan, "out": out, "payloads": payloads}


def run(state):
    kind = state["kind"]
    if kind == "tiles":
        recon, states = backend.quantize_tiles(state["tiles"], state["args"])
        return {"recon": recon, "states": states}
    if kind == "ldlq":
        weight_q, encoded = backend.ldlq_mixed_batched(state["weights"], state["Ls"], state["args"], synchronize=False)
        return {"weight_q": weight_q, "encoded": encoded}
    if kind == "encode":  # the call consumes its weight and its Hessian record: each pass takes its own
        shared = make_shared_h(state["hessian"].shape[0], torch.device(DEV), state["hessian"])
        shared["count"] = state["count"]
        weight_q, proxy, tensors = backend.quantize_qsrt(state["weight"].clone(), shared, dict(state["args"]), True)
        return {"weight": weight_q, "proxy": proxy, **tensors}
    if kind == "gram":
        k = state["x"].shape[1]
        return gram_(torch.zeros((k, k), dtype=torch.float32, device=state["x"].device), state["x"],
                     alpha=1.0 / state["x"].shape[0])
    if kind == "rotate":
        rotate_(state["x"], state["block"], side="left", pre_mul=state["su"])
        return rotate_(state["x"], state["block"], side="right", post_mul=state["sv"])
    if "plan" in state:
        state["plan"].run()
        return state["out"]
    return decode_words(state["words"], state["su"], state["sv"], state["bits"], state["lut"], out_dtype=state["dtype"])


def _tile_flops(tiles, context=128):
    """Each of 256 + 2 * context steps scores 2^16 edges: a subtraction and a fused multiply-add each."""

    return 3.0 * 65536 * (256 + 2 * context) * tiles


def work(case):
    kind = case["kind"]
    if kind == "tiles":
        return {"bytes": case["n"] * 256 * 10 + 65536, "flops": _tile_flops(case["n"], case["context"])}
    k = case["k"]
    if kind == "gram":
        size = 2 if case["dtype"] == "bf16" else 4
        return {"bytes": case["rows"] * k * size + 4 * k * k, "flops": float(case["rows"]) * k * (k + 1)}
    n = case["n"]
    if kind == "ldlq":
        m = case["members"]
        return {"bytes": m * (k * n * (8 + 4 + 2) + 4 * k * k),
                "flops": _tile_flops(m * k * n // 256) + m * float(k) * k * n}
    if kind == "encode":
        sample = 3 * max(k, n) // 16
        tiles = k * n // 256 + 10 * (sample // 3) + 5 * sample
        return {"bytes": 4 * k * k + k * n * (8 + case["bits"] / 8),
                "flops": _tile_flops(tiles) + float(k) * k * n + k ** 3 / 3}
    if kind == "rotate":
        size = 4 if case["dtype"] == "f32" else 8
        return {"bytes": 2 * size * k * n, "flops": 2.0 * k * n * math.log2(case["block"])}
    count = max(1, 3 * case["experts"])
    bits = case["bits"] + (2 * (4 - case["bits"]) / (n // 128) if case["experts"] else 0.0)
    return {"bytes": count * (k * n * (bits / 8 + (2 if case["dtype"] == "bf16" else 4)) + 4 * (k + n)),
            "flops": count * 2.0 * 14 * k * n}


def tolerance(case):
    kind = case["kind"]
    if kind in ("tiles", "ldlq"):
        return "exact"  # codewords and their table values
    if kind == "encode":
        return {"rel": 2e-6, "max": 2e-5, "differ": 0.0}  # the payload is bytes; weight and error are float32
    if kind == "gram":
        # float32 sums of up to 16,384 products: 5e-7 (bf16 operands) and 2e-6 (float32 ones) from the exact sum
        return {"rel": 2e-6, "max": 2e-5} if case["dtype"] == "bf16" else {"rel": 8e-6, "max": 8e-5}
    if kind == "rotate":
        return {"rel": 1e-6, "max": 1e-5} if case["dtype"] == "f32" else {"rel": 2e-15, "max": 2e-14}
    # bf16: a value on a rounding boundary may go either way (about 3 in 100,000, one ulp each)
    return {"rel": 1e-4, "max": 1e-2} if case["dtype"] == "bf16" else {"rel": 1e-6, "max": 1e-5}


# ---------------------------------------------------------------------------
# The same values in 64 bits, from the definitions
# ---------------------------------------------------------------------------


def _viterbi64(tiles, labels, bits, context):
    """The tail-biting path of each tile with float64 path costs: a primer over positions 256-C .. 255, 0 .. C-1
    names the state before position 0, and a constrained pass closes the path through it.  Returns its labels."""

    n, K, P = tiles.shape[0], bits, 1 << bits
    S = 65536 >> K
    cost_of = labels.view(P, S)  # codeword (k << (16 - K)) | state
    preds = (torch.arange(P, device=DEV)[:, None] << (16 - 2 * K)) | (torch.arange(S, device=DEV)[None, :] >> K)
    lag = 0 if K == 2 else 1  # K2 scores the primer's last costs, the others the ones before

    def walk(positions, cost, keep):
        arg = torch.empty((len(positions) - keep, n, S), dtype=torch.uint8, device=DEV)
        before = cost
        for i, pos in enumerate(positions):
            before = cost
            c = (cost_of[None] - tiles[:, pos, None, None]).square() + (
                0.0 if cost is None else cost[:, preds.view(-1)].view(n, P, S))
            cost, a = c.min(dim=1)
            if i >= keep:
                arg[i - keep] = a.to(torch.uint8)
        return cost, before, arg

    def trace(arg, state, codewords=None):
        for pos in range(arg.shape[0] - 1, -1, -1):
            k = arg[pos].gather(1, state[:, None]).squeeze(1).long()
            if codewords is not None:
                codewords[:, pos] = (k << (16 - K)) | state
            state = (k << (16 - 2 * K)) | (state >> K)
        return state

    primer = list(range(256 - context, 256)) + list(range(context))
    last, before, arg = walk(primer, None, context)
    closing = trace(arg, (before if lag else last).argmin(dim=1))
    first = torch.full((n, S), math.inf, dtype=torch.float64, device=DEV)
    first[torch.arange(n, device=DEV), closing] = 0.0
    _, _, arg = walk(list(range(256)), first, 0)
    codewords = torch.empty((n, 256), dtype=torch.int64, device=DEV)
    trace(arg, closing, codewords)
    return labels[codewords]


def _hadamard64(size):
    i = torch.arange(size, device=DEV)
    x, parity = i[:, None] & i[None, :], 0
    for b in range(size.bit_length()):
        parity = parity ^ ((x >> b) & 1)
    return (1.0 - 2.0 * parity.double()) / math.sqrt(size)


def _decode64(words, bits, su, sv, lut):
    """``[rows, cols, 16 bits]`` words -> ``[16 rows, 16 cols]``: adjacent words swapped, MSB first; each state is the
    16 bits that end with its symbol, cyclically; labels in tensor-core order; both 128-block rotations."""

    rows, cols, count = words.shape
    w = (words.long() & 0xFFFF).view(rows, cols, count // 2, 2).flip(-1).reshape(rows, cols, count)
    stream = ((w[..., None] >> torch.arange(15, -1, -1, device=DEV)) & 1).reshape(rows, cols, 256 * bits)
    end = bits * (torch.arange(256, device=DEV) + 1)
    state = 0
    for b in range(16):
        state = (state << 1) | stream[..., (end - 16 + b) % (256 * bits)]
    lane = torch.arange(32, device=DEV)
    row = 2 * (lane % 4)[:, None] + torch.tensor([0, 1, 8, 9], device=DEV)
    place = torch.cat([row * 16 + (lane // 4)[:, None], row * 16 + (lane // 4)[:, None] + 8], dim=1).reshape(-1)
    tile = torch.empty((rows, cols, 256), dtype=torch.float64, device=DEV)
    tile[..., place] = lut.view(torch.float8_e4m3fn).double()[state]
    x = tile.view(rows, cols, 16, 16).permute(0, 2, 1, 3).reshape(16 * rows, 16 * cols)
    h = _hadamard64(128)
    x = (h @ x.view(rows // 8, 128, 16 * cols)).reshape(16 * rows, 16 * cols) * su.double()[:, None]
    return (x.view(16 * rows, cols // 8, 128) @ h).reshape(16 * rows, 16 * cols) * sv.double()[None, :]


def exact(case, seed):
    """What ``run`` returns in 64 bits.  None for ``ldlq`` and ``encode``: their outputs follow from thousands of
    discrete path choices, each made on the ones before (and their float64 walk would take minutes)."""

    kind = case["kind"]
    if kind in ("ldlq", "encode"):
        return None
    state = prepare(case, seed)
    if kind == "tiles":
        labels = state["args"]["sqg_e4m3_lut"].to(DEV).view(torch.float8_e4m3fn).double()
        tiles = state["tiles"].double()
        return {"recon": torch.cat([_viterbi64(t, labels, case["bits"], case["context"]) for t in tiles.split(64)]),
                "states": None}
    if kind == "gram":
        x = state["x"].double()
        return x.T @ x / case["rows"]
    if kind == "rotate":
        k, n, block = case["k"], case["n"], case["block"]
        h = _hadamard64(block)
        x = (h @ (state["x"].double() * state["su"].double()[:, None]).view(k // block, block, n)).reshape(k, n)
        return (x.view(k, n // block, block) @ h).reshape(k, n) * state["sv"].double()[None, :]
    if "plan" not in state:
        return _decode64(state["words"], state["bits"], state["su"], state["sv"], state["lut"])
    luts = {b: sqg_xor_cheb_t12_bytes(b).to(DEV) for b in (4, case["bits"])}
    full = [torch.empty(o.shape, dtype=torch.float64, device=DEV) for o in state["out"]]
    at = [one for stack in full for one in stack]
    for (words, records, axis, su, sv, _), one in zip(state["payloads"], at):
        cursor = 0
        for r, bits in enumerate(records):
            rows, cols = (8, one.shape[1] // 16) if axis == "k" else (one.shape[0] // 16, 8)
            part = words[cursor:cursor + rows * cols * 16 * bits].view(rows, cols, 16 * bits)
            cursor += part.numel()
            lines = slice(128 * r, 128 * r + 128)
            if axis == "k":
                one[lines] = _decode64(part, bits, 128.0 * su[lines], sv, luts[bits])
            else:
                one[:, lines] = _decode64(part, bits, 128.0 * su, sv[lines], luts[bits])
    return full
