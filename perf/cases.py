"""The workloads this package's speed is measured on.

One case per kind of call a serving program makes of the GDN state codec, at
sizes of the Qwen3.5 gated-delta-net state (128 x 128 heads, 32 value heads a
layer, batches of up to 256 sequences), plus ``draw`` for other sizes of the
same ranges: a single head to whole batches, odd counts, both tile layouts,
both pool types, ragged windows and token counts.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

_PACKAGE = str(Path(__file__).resolve().parents[1] / "gdn-state-codec_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from gdn_state_codec import capsule, codec  # noqa: E402
from gdn_state_codec._native import native  # noqa: E402
from gdn_state_codec.runtime import (  # noqa: E402
    QWEN_QUERY_SCALE, GdnStateCodecExperiment, GdnStateCodecRuntime)
from gdn_state_codec.window import WindowSlot, step_bf16  # noqa: E402

DIM, RANK, WINDOW = 128, 4, 16
TILE = DIM * DIM
ENCODED = TILE + 2 * 4 * DIM            # codes, smoothing and scales of one head
BASES = 2 * 2 * DIM * RANK              # fp16 rank-4 compensators, both sides
RECORDS = WINDOW * (4 + 2 * 2 * DIM)    # gate, key and correction of 16 records


def listed() -> list[dict]:
    return [
        # Admission of one request to one layer: its 32 heads encoded from the
        # provider's dense state, and given back dense when it falls back.
        {"name": "slot_codec", "kind": "codec", "heads": 32, "layout": 1},
        # Offload and reload of a batch's dense states: 8 layers x 240
        # sequences x 32 heads, capsule layout.
        {"name": "batch_codec", "kind": "codec", "heads": 61440, "layout": 0},
        # Slot-indexed bf16 state pool of a server (12 layers), 5% of the
        # batch entries padding: gather-encode, then decode-scatter.
        {"name": "pool_bf16", "kind": "pool", "layers": 12, "slots": 160, "heads": 32,
         "batch": 120, "dtype": "bf16", "layout": 1},
        # One decode token of 256 sequences read against the encoded state.
        {"name": "decode_projection", "kind": "project", "seqs": 256, "tokens": 1, "heads": 32,
         "query_heads": 16, "layout": 1},
        # A 64-token prefill chunk of 64 sequences read the same way.
        {"name": "chunk_projection", "kind": "project", "seqs": 64, "tokens": 64, "heads": 32,
         "query_heads": 32, "layout": 1},
        # The per-layer runtime as a model calls it: one request, one window of
        # 16 decode tokens, and the boundary refit the full window brings.
        {"name": "slot_decode", "kind": "runtime", "heads": 32, "power": 0},
        # A batch's window: 16 quant-only steps and the quant-only refit.
        {"name": "window_quant", "kind": "window", "states": 8192, "power": 0},
        # The compensated window: 16 steps and the rank-4 power refit.
        {"name": "window_power", "kind": "window", "states": 8192, "power": 4},
        # The device rank-4 chain over an encoded boundary and its requantize.
        {"name": "rank_chain", "kind": "chain", "states": 2048, "iterations": 8},
        # The capsule factory's boundary encode (rank-4 fit) of one request:
        # 30 layers x 32 heads.
        {"name": "capsule_fit", "kind": "fit", "heads": 960, "rank": 4},
        # The exact-SVD initializer for one request's 30 layers, and the dense
        # state its slots reconstruct to.
        {"name": "exact_svd", "kind": "svd", "heads": 960},
        # Hibernate and resume: 4,096 slot states at mixed window positions to
        # capsules (SHA-256 sealed) and back.
        {"name": "capsule", "kind": "capsule", "states": 4096},
    ]


def draw(rng) -> dict:
    def size(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    kind = rng.choice(["codec", "pool", "project", "runtime", "window", "chain", "fit", "svd",
                       "capsule"])
    if kind == "codec":
        return {"kind": kind, "heads": size(1, 61440), "layout": rng.randrange(2)}
    if kind == "pool":
        slots = size(4, 160)
        return {"kind": kind, "layers": rng.randint(1, 12), "slots": slots,
                "heads": rng.choice([8, 16, 24, 32]), "batch": rng.randint(1, min(slots, 120)),
                "dtype": rng.choice(["f32", "bf16"]), "layout": rng.randrange(2)}
    if kind == "project":
        tokens = rng.choice([1, size(2, 64)])
        query_heads = rng.choice([4, 8, 16])
        return {"kind": kind, "seqs": size(1, 256 if tokens == 1 else 64), "tokens": tokens,
                "heads": query_heads * rng.choice([1, 2]), "query_heads": query_heads,
                "layout": rng.randrange(2)}
    if kind == "runtime":
        # The quant-only refit's process-wide handle serves one head count.
        power = rng.randrange(6)
        return {"kind": kind, "heads": 2 * size(1, 32) if power else 32, "power": power}
    if kind == "window":
        return {"kind": kind, "states": 2 * size(1, 4096), "power": rng.choice([0, 1, 2, 4])}
    if kind == "chain":
        return {"kind": kind, "states": size(1, 2048), "iterations": rng.randint(1, 8)}
    if kind == "fit":
        return {"kind": kind, "heads": size(1, 960), "rank": rng.randint(0, 4)}
    if kind == "svd":
        return {"kind": kind, "heads": size(1, 960)}
    return {"kind": kind, "states": size(1, 4096)}


# ------------------------------------------------------------------- inputs

def _generator(seed: int, device) -> torch.Generator:
    return torch.Generator(device=device).manual_seed(seed)


def _device() -> torch.device:
    return torch.device("cuda", torch.cuda.current_device())


def _heads(shape, gen, dev) -> torch.Tensor:
    """State values: N(0, 0.05^2) with 0.1% outliers at +-2."""
    x = torch.randn(shape, generator=gen, device=dev).mul_(0.05)
    lottery = torch.rand(shape, generator=gen, device=dev)
    x[lottery < 0.0005] = 2.0
    x[lottery > 0.9995] = -2.0
    return x


def _half(shape, scale, gen, dev) -> torch.Tensor:
    return (torch.randn(shape, generator=gen, device=dev) * scale).to(torch.float16)


def _unit(shape, gen, dev) -> torch.Tensor:
    v = torch.randn(shape, generator=gen, device=dev)
    return v / v.norm(dim=-1, keepdim=True)


def _slot(states, compensated, gen, dev) -> WindowSlot:
    """An encoded boundary with an empty window."""
    slot = WindowSlot.allocate(states, dev)
    codec.encode(_heads((states, DIM, DIM), gen, dev), codec.LAYOUT_VALUE_KEY, slot.residual,
                 slot.smoothing, slot.scales)
    if compensated:
        slot.compensator_keys.copy_(_half((states, DIM, RANK), 0.01, gen, dev))
        slot.compensator_values.copy_(_half((states, DIM, RANK), 0.01, gen, dev))
    return slot


def _records(slot, gen, dev) -> None:
    """A full window of records at the magnitudes decode steps leave."""
    s = slot.states
    slot.record_decay.copy_(0.93 + 0.06 * torch.rand((s, WINDOW), generator=gen, device=dev))
    slot.record_keys.copy_(_unit((s, WINDOW, DIM), gen, dev))
    slot.record_corrections.copy_(_half((s, WINDOW, DIM), 0.25, gen, dev))


def _tokens(states, gen, dev) -> list[tuple]:
    """16 decode tokens: log decay, beta, keys, queries, values."""
    tokens = []
    for _ in range(WINDOW):
        tokens.append((
            torch.log(0.9 + 0.09 * torch.rand(states, generator=gen, device=dev)),
            (0.2 + 0.6 * torch.rand(states, generator=gen, device=dev)).to(torch.bfloat16),
            _unit((states // 2, DIM), gen, dev).to(torch.bfloat16),
            _unit((states // 2, DIM), gen, dev).to(torch.bfloat16),
            (0.5 * torch.randn((states, DIM), generator=gen, device=dev)).to(torch.bfloat16)))
    return tokens


def prepare(case: dict, seed: int) -> dict:
    dev = _device()
    gen = _generator(seed, dev)
    kind = case["kind"]
    state = {"case": case}
    if kind == "codec":
        state["x"] = _heads((case["heads"], DIM, DIM), gen, dev)
        state["codes"] = torch.empty((case["heads"], DIM, DIM), dtype=torch.int8, device=dev)
        state["smoothing"] = torch.empty((case["heads"], DIM), device=dev)
        state["scales"] = torch.empty((case["heads"], DIM), device=dev)
        state["dense"] = torch.empty_like(state["x"])
    elif kind == "pool":
        layers, slots, heads, batch = (case[k] for k in ("layers", "slots", "heads", "batch"))
        dtype = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
        shape = (layers, slots, heads, DIM, DIM)
        # Student-t(3) x 0.05 values, 2% of the heads still zero.
        pool = torch.empty(shape, dtype=dtype, device=dev)
        for layer in range(layers):
            chi = sum(torch.randn(shape[1:], generator=gen, device=dev).square_()
                      for _ in range(3))
            values = torch.randn(shape[1:], generator=gen, device=dev).mul_(0.05)
            values /= (chi / 3).sqrt_()
            values[torch.rand(shape[1:3], generator=gen, device=dev) < 0.02] = 0.0
            pool[layer] = values
        ids = torch.randperm(slots, generator=gen, device=dev)[:batch].to(torch.int32)
        ids[torch.rand(batch, generator=gen, device=dev) < 0.05] = -1
        state.update(pool=pool, ids=ids, restored=torch.zeros_like(pool),
                     codes=torch.zeros((layers, batch, heads, DIM, DIM), dtype=torch.int8,
                                       device=dev),
                     smoothing=torch.zeros((layers, batch, heads, DIM), device=dev),
                     scales=torch.zeros((layers, batch, heads, DIM), device=dev))
    elif kind == "project":
        seqs, tokens, heads = case["seqs"], case["tokens"], case["heads"]
        x = _heads((seqs, heads, DIM, DIM), gen, dev)
        state["codes"], state["smoothing"], state["scales"] = codec.encode(x, case["layout"])
        lead = (seqs,) if tokens == 1 else (seqs, tokens)
        state["queries"] = _unit(lead + (case["query_heads"], DIM), gen, dev).to(torch.bfloat16)
        state["out"] = torch.empty(lead + (heads, DIM), device=dev)
    elif kind == "runtime":
        heads, power = case["heads"], case["power"]
        experiment = GdnStateCodecExperiment(
            initializer="exact_svd" if power else "quant_only", boundary_power_iterations=power)
        state["runtime"] = GdnStateCodecRuntime(experiment)
        state["provider"] = _heads((1, heads, DIM, DIM), gen, dev)
        state["tokens"] = [
            (q.view(1, 1, heads // 2, DIM), k.view(1, 1, heads // 2, DIM),
             v.view(1, 1, heads, DIM), g.view(1, 1, heads), b.view(1, 1, heads))
            for g, b, k, q, v in _tokens(heads, gen, dev)]
        # The request has already decoded one window: its slot exists, full.
        for token in state["tokens"]:
            state["runtime"].step(state["provider"], 0, *token, QWEN_QUERY_SCALE)
    elif kind == "window":
        states = case["states"]
        state["slot"] = _slot(states, case["power"] > 0, gen, dev)
        state["next"] = WindowSlot.allocate(states, dev)
        state["workspace"] = torch.empty((states, DIM, DIM), device=dev)
        state["tokens"] = _tokens(states, gen, dev)
        state["outs"] = [torch.empty((states, DIM), dtype=torch.bfloat16, device=dev)
                         for _ in range(WINDOW)]
    elif kind == "chain":
        states = case["states"]
        slot = _slot(states, True, gen, dev)
        _records(slot, gen, dev)
        state["slot"] = slot
        state["seeds"] = _unit((states, RANK, DIM), gen, dev).to(torch.float16)
        for name in ("new_left", "new_right"):
            state[name] = torch.zeros((states, RANK, DIM), dtype=torch.float16, device=dev)
        state["corrected"] = torch.empty((states, RANK, DIM), device=dev)
        state["next"] = WindowSlot.allocate(states, dev)
        state["workspace"] = torch.empty((states, DIM, DIM), device=dev)
    elif kind in ("fit", "svd"):
        state["x"] = _heads((case["heads"], DIM, DIM), gen, dev)
    elif kind == "capsule":
        states = case["states"]
        slot = _slot(states, True, gen, dev)
        _records(slot, gen, dev)
        positions = torch.randperm(states, generator=gen, device=dev) % WINDOW
        slot.positions[:, 0] = positions.to(torch.int32)
        lengths = 21688 + 1536 * positions
        state.update(slot=slot, fresh=WindowSlot.allocate(states, dev),
                     identity=capsule.CapsuleIdentity("5d" * 32, 1 + seed % 1000, 3),
                     offsets=torch.cumsum(lengths, 0) - lengths,
                     buffer=torch.zeros(int(lengths.sum()), dtype=torch.uint8, device=dev),
                     lengths=torch.empty(states, dtype=torch.int32, device=dev),
                     expected=positions.to(torch.int32))
    else:
        raise ValueError(kind)
    return state


# --------------------------------------------------------------------- a pass

def _ok(status: int) -> None:
    if status != 0:
        raise RuntimeError(f"GDN State Codec launch failed: {status}")


def _boundary(slot) -> list:
    return [slot.residual, slot.smoothing, slot.scales, slot.compensator_keys,
            slot.compensator_values]


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "codec":
        out = codec.encode(state["x"], case["layout"], state["codes"], state["smoothing"],
                           state["scales"])
        return [*out, codec.decode(*out, case["layout"], out=state["dense"])]
    if kind == "pool":
        out = codec.pool_encode(state["pool"], state["ids"], case["layout"], state["codes"],
                                state["smoothing"], state["scales"])
        return [*out, codec.pool_decode(*out, state["ids"], state["restored"], case["layout"])]
    if kind == "project":
        project = codec.project_decode if case["tokens"] == 1 else codec.project_chunked
        return project(state["codes"], state["smoothing"], state["scales"], state["queries"],
                       QWEN_QUERY_SCALE, case["layout"], out=state["out"])
    if kind == "runtime":
        runtime = state["runtime"]
        for token in state["tokens"]:
            out = runtime.step(state["provider"], 0, *token, QWEN_QUERY_SCALE)
        window = runtime._slots[0].window
        return [out, *_boundary(window), window.record_decay, window.record_keys,
                window.record_corrections, window.positions]
    if kind == "window":
        slot, following = state["slot"], state["next"]
        for token, out in zip(state["tokens"], state["outs"]):
            step_bf16(slot, *token, out=out, quant_only=case["power"] == 0, validate=False)
        boundary = _boundary(following)
        _ok(native().window_boundary_launch_v1(
            torch.cuda.current_stream().cuda_stream, *slot.pointers(),
            *(t.data_ptr() for t in boundary), state["workspace"].data_ptr(), slot.states,
            case["power"]))
        return [*state["outs"], *boundary, *([state["workspace"]] if case["power"] else [])]
    if kind == "chain":
        slot, following = state["slot"], state["next"]
        stream, lib = torch.cuda.current_stream().cuda_stream, native()
        operands = [t.data_ptr() for t in (*_boundary(slot), slot.record_decay, slot.record_keys,
                                           slot.record_corrections)]
        bases = [state["new_left"], state["new_right"]]
        _ok(lib.encoded_rank_chain_launch_v4(
            stream, *operands, state["seeds"].data_ptr(), *(t.data_ptr() for t in bases),
            state["corrected"].data_ptr(), slot.states, case["iterations"]))
        boundary = _boundary(following)
        _ok(lib.encoded_requantize_launch_v1(
            stream, *operands, *(t.data_ptr() for t in (*bases, *boundary, state["workspace"])),
            slot.states))
        return [*bases, state["corrected"], *boundary, state["workspace"]]
    if kind == "fit":
        return list(codec.quantize_boundary(state["x"], case["rank"], check=False))
    if kind == "svd":
        codes, smoothing, scales, keys, values, residual, status = codec.exact_svd_boundary(
            state["x"], check=False)
        # Each (u, v) pair's common sign is the solver's own, so the
        # compensators come out as the state they reconstruct with the codes.
        dense = codec.decode(codes, smoothing, scales, codec.LAYOUT_VALUE_KEY, keys.float(),
                             values.float())
        return [codes, smoothing, scales, residual, status, dense]
    slot, fresh, identity = state["slot"], state["fresh"], state["identity"]
    buffer, offsets, lengths = state["buffer"], state["offsets"], state["lengths"]
    _ok(native().capsule_serialize_launch_v1(
        torch.cuda.current_stream().cuda_stream, *slot.pointers(), capsule.LAYOUT_VALUE_KEY,
        identity.geometry_bytes, identity.generation, identity.epoch, buffer.data_ptr(),
        offsets.data_ptr(), buffer.numel(), lengths.data_ptr(), slot.states))
    status = capsule.restore(fresh, buffer, offsets, lengths, identity, state["expected"])
    return [buffer, lengths, status, *_boundary(fresh), fresh.record_decay, fresh.record_keys,
            fresh.record_corrections, fresh.positions]


# ------------------------------------------------------- work and tolerances

def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "codec":
        return {"bytes": case["heads"] * 2 * (4 * TILE + ENCODED), "flops": case["heads"] * 8 * TILE}
    if kind == "pool":
        tiles = case["layers"] * case["batch"] * case["heads"]
        width = 4 if case["dtype"] == "f32" else 2
        return {"bytes": tiles * 2 * (width * TILE + ENCODED), "flops": tiles * 8 * TILE}
    if kind == "project":
        seqs, tokens, heads = case["seqs"], case["tokens"], case["heads"]
        return {"bytes": seqs * (heads * ENCODED + tokens * DIM * (2 * case["query_heads"]
                                                                  + 4 * heads)),
                "flops": 2 * seqs * heads * tokens * TILE}
    if kind in ("runtime", "window"):
        states = case["heads"] if kind == "runtime" else case["states"]
        power = case["power"] > 0
        boundary = ENCODED + (BASES if power else 0)
        # A step reads the boundary, the records so far and the token, and
        # writes its record and output.
        step = boundary + RECORDS // WINDOW * (WINDOW + 1) // 2 + DIM * (2 + 2 + 2 + 2) + 6
        refit = 2 * boundary + RECORDS + (4 * TILE if power else 0)
        flops = WINDOW * (4 * TILE + 8 * DIM * WINDOW) + (2 * WINDOW + 8) * TILE
        flops += RANK * (2 * case["power"] + 1) * 2 * TILE if power else 0
        return {"bytes": states * (WINDOW * step + refit), "flops": states * flops}
    if kind == "chain":
        read = ENCODED + BASES + RECORDS
        return {"bytes": case["states"] * (2 * read + 3 * BASES + ENCODED + 4 * TILE),
                "flops": case["states"] * TILE * (2 * RANK * (2 * case["iterations"] + 1)
                                                  + 2 * WINDOW + 4 * RANK + 8)}
    if kind == "fit":
        # 32 iterations of two products a rank, the singular value, the update.
        return {"bytes": case["heads"] * (2 * 4 * TILE + ENCODED + 2 * 4 * DIM * case["rank"]),
                "flops": case["heads"] * TILE * (case["rank"] * (32 * 4 + 5) + 8)}
    if kind == "svd":
        # The Gram matrix, its tridiagonal form, and the rank-4 products.
        flops = 2 * DIM ** 3 // 2 + 4 * DIM ** 3 // 3 + 8 * RANK * TILE
        return {"bytes": case["heads"] * (3 * 4 * TILE + 2 * ENCODED + 2 * BASES),
                "flops": case["heads"] * flops}
    states = case["states"]
    mean = 21688 + 1536 * (WINDOW - 1) // 2  # a capsule's bytes, positions 0..15
    slot = ENCODED + BASES + (WINDOW - 1) * RECORDS // WINDOW // 2 + 4
    return {"bytes": states * 2 * (mean + slot), "flops": states * 2 * mean // 64 * 2000}


def tolerance(case: dict):
    kind = case["kind"]
    if kind == "project":
        # fp32 sums over 128 keys; the chunked form's weights are split into
        # two bf16 parts, 16 bits of significand.
        return {"rel": 5e-7} if case["tokens"] == 1 else {"rel": 1e-5}
    if kind in ("runtime", "window"):
        # bf16 outputs and fp16 records: one rounding apart in a record moves
        # what follows, and a code at a rounding boundary.
        return {"rel": 4e-3, "max": 0.1, "differ": 2e-3}
    if kind == "svd":
        # The rank-4 product is exact to the fp32 rounding of its outputs; a
        # cell of the residual near a rounding boundary moves a code by one,
        # and a compensator near one moves by an fp16 rounding.
        return {"rel": 1e-4, "max": 1e-2, "differ": 1e-4}
    # Codes, smoothing, scales, fits and capsules are fixed bit for bit by the
    # order of operations that the format states.
    return "exact"


# ------------------------------------------------- the same in 64 bits (torch)

def _quantized(m, scale_dim):
    """m / absmax over scale_dim, in 127ths, rounded half away from zero."""
    scale = m.abs().amax(dim=scale_dim, keepdim=True)
    q = torch.where(scale == 0, torch.zeros_like(m), m / scale * 127)
    return torch.sign(q) * torch.floor(q.abs() + 0.5), scale


def _encode64(x, layout):
    """codes (None), smoothing, scales and the dequantized tiles of x."""
    key, value = (-2, -1) if layout == codec.LAYOUT_KEY_VALUE else (-1, -2)
    s = x.abs().mean(dim=value, keepdim=True).clamp_min(1e-8).sqrt()
    q, scale = _quantized(x / s, key)
    return None, s.squeeze(value), scale.squeeze(key), q * s * scale / 127


def _dense64(slot):
    """The dense [state][key][value] boundary of an encoded slot."""
    x = (slot.residual.double() * slot.scales.double()[:, :, None]
         * slot.smoothing.double()[:, None, :] / 127).transpose(1, 2).contiguous()
    return x + _pair(slot.compensator_keys.double(), slot.compensator_values.double())


def _pair(left, right):
    """sum over r of left[s][i][r] right[s][j][r], one rank at a time."""
    total = 0.0
    for r in range(left.shape[-1]):
        total = total + left[:, :, None, r] * right[:, None, :, r]
    return total


def _apply(x, v, transpose=False):
    return ((x * v[:, :, None]).sum(1) if transpose else (x * v[:, None, :]).sum(2))


def _step64(x, token):
    """One gated delta rule token: (new dense state, output)."""
    g, beta, keys, queries, values = (t.double() for t in token)
    keys, queries = (t.repeat_interleave(2, dim=0) for t in (keys, queries))
    x = x * g.exp()[:, None, None]
    correction = beta[:, None] * (values - _apply(x, keys, True))
    x += keys[:, :, None] * correction[:, None, :]
    return x, _apply(x, queries, True) * QWEN_QUERY_SCALE


def _exact_window(case, seed):
    state = prepare(case, seed)
    slot = state["slot"]
    x = _dense64(slot)
    outs = []
    for token in state["tokens"]:
        x, out = _step64(x, token)
        outs.append(out)
    if case["power"] == 0:
        smoothing = slot.smoothing.double()
        scales = (x / smoothing[:, :, None]).abs().amax(1)
        zeros = torch.zeros((slot.states, DIM, RANK), dtype=torch.float64, device=x.device)
        return [*outs, None, smoothing, scales, zeros, zeros]
    left, right = [], []
    for r in range(RANK):
        v = (((r + 1) * (torch.arange(DIM, device=x.device) + 3)) % 17 - 8).double()
        v = (v / v.norm()).expand(slot.states, DIM)
        for _ in range(case["power"]):
            u = _apply(x, v)
            v = _apply(x, u / u.norm(dim=1, keepdim=True), True)
            v = v / v.norm(dim=1, keepdim=True)
        left.append(_apply(x, v).half().double())
        right.append(v.half().double())
        x = x - left[-1][:, :, None] * right[-1][:, None, :]
    _, smoothing, scales, _ = _encode64(x, codec.LAYOUT_KEY_VALUE)
    return [*outs, None, smoothing, scales, torch.stack(left, 2), torch.stack(right, 2), x]


def _exact_chain(case, seed):
    state = prepare(case, seed)
    slot = state["slot"]
    # The slot's buffers read as [left][right], left the smoothing axis.
    codes, left_axis, right_axis = (slot.residual.double(), slot.smoothing.double(),
                                    slot.scales.double())
    decay = slot.record_decay.double()
    suffix = torch.flip(torch.cumprod(torch.flip(decay, (1,)), 1), (1,))
    whole, suffix = suffix[:, 0], torch.cat([suffix[:, 1:], torch.ones_like(decay[:, :1])], 1)
    x = _pair(slot.compensator_keys.double(), slot.compensator_values.double())
    x *= whole[:, None, None]
    for j in range(WINDOW):
        x += (slot.record_keys[:, j].double() * suffix[:, j, None])[:, :, None] * \
            slot.record_corrections[:, j].double()[:, None, :]

    def product(v, transpose):
        """The boundary's product with the int8-quantized vector, and the rest."""
        scaled = v * (left_axis if transpose else right_axis)
        q, top = _quantized(scaled, 1)
        out = _apply(codes, q, transpose) * (right_axis if transpose else left_axis)
        return out * top / 127 / 127 * whole[:, None] + _apply(x, v, transpose)

    lefts, rights, corrected = [], [], []
    for r in range(RANK):
        v = state["seeds"][:, r].double()
        for _ in range(case["iterations"]):
            for transpose in (False, True):
                v = product(v, transpose)
                v = (v / v.norm(dim=1, keepdim=True)).half().double()
        corrected.append(product(v, False))
        lefts.append(corrected[-1].half().double())
        rights.append(v)
        x -= lefts[-1][:, :, None] * rights[-1][:, None, :]
    x += codes * left_axis[:, :, None] * right_axis[:, None, :] / 127 * whole[:, None, None]
    _, smoothing, scales, _ = _encode64(x, codec.LAYOUT_KEY_VALUE)
    return [torch.stack(lefts, 1), torch.stack(rights, 1), torch.stack(corrected, 1), None,
            smoothing, scales, torch.stack(lefts, 2), torch.stack(rights, 2), x]


def _exact_fit(case, seed):
    x = prepare(case, seed)["x"].double()
    heads, rank = case["heads"], case["rank"]
    keys = torch.zeros((heads, DIM, rank), dtype=torch.float64, device=x.device)
    values = torch.zeros_like(keys)
    for r in range(rank):
        v = torch.sin(((r + 1.0) * torch.arange(1, DIM + 1, device=x.device)).double())
        v = (v / v.norm()).expand(heads, DIM)
        for _ in range(32):
            u = _apply(x, v)
            u = u / u.norm(dim=1, keepdim=True)
            v = _apply(x, u, True)
            v = v / v.norm(dim=1, keepdim=True)
        keys[:, :, r] = u * (u * _apply(x, v)).sum(1, keepdim=True)
        values[:, :, r] = v
        x = x - keys[:, :, None, r] * values[:, None, :, r]
    codes, smoothing, scales, _ = _encode64(x, codec.LAYOUT_KEY_VALUE)
    return [codes, smoothing, scales, keys, values, x, None]


def _exact_svd(case, seed):
    x = prepare(case, seed)["x"].double()  # [head][value][key]
    u, s, vt = np.linalg.svd(x.cpu().numpy())
    v = torch.from_numpy(np.ascontiguousarray(u[:, :, :RANK])).to(x.device)
    k = torch.from_numpy(np.ascontiguousarray(
        np.swapaxes(vt[:, :RANK] * s[:, :RANK, None], 1, 2))).to(x.device)
    residual = x - _pair(v, k)
    codes, smoothing, scales, dequantized = _encode64(residual, codec.LAYOUT_VALUE_KEY)
    return [codes, smoothing, scales, residual, None,
            dequantized + _pair(v.half().double(), k.half().double())]


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "codec":
        if case["heads"] > 16384:
            return None
        return list(_encode64(prepare(case, seed)["x"].double(), case["layout"]))
    if kind == "project":
        state = prepare(case, seed)
        s, scale = state["smoothing"].double(), state["scales"].double()
        codes = state["codes"].double()
        if case["layout"] == codec.LAYOUT_KEY_VALUE:
            codes = codes.transpose(-2, -1)
        x = codes * scale[..., :, None] * s[..., None, :] / 127  # [seq][head][value][key]
        group = case["heads"] // case["query_heads"]
        q = state["queries"].double().repeat_interleave(group, dim=-2) * QWEN_QUERY_SCALE
        if case["tokens"] == 1:
            return (x * q[:, :, None, :]).sum(-1)
        return torch.stack([(x * q[:, t, :, None, :]).sum(-1) for t in range(case["tokens"])], 1)
    if kind == "window":
        return _exact_window(case, seed)
    if kind == "chain":
        return _exact_chain(case, seed)
    if kind == "fit":
        return _exact_fit(case, seed)
    if kind == "svd":
        return _exact_svd(case, seed)
    return None
