"""The work users have this package do, as timed cases: the gated-delta operators forward and backward, the LSH bucket
sort, the hierarchical operator and the whole block, each through its public entry point.

A case is a dict of plain values; ``path`` names the entry point:

* ``recurrent``  ``fused_recurrent_gated_delta_rule``: a few tokens per sequence on top of a state, and the fp32 mode;
* ``chunk``      ``chunk_gated_delta_rule`` forward: one event, a batch, or events packed with ``cu_seqlens``;
* ``train``      the same operator with its backward pass (the output and every gradient come back);
* ``lsh``        ``lsh_bucket_sort`` with the hit features, one event or a padded batch;
* ``block``      ``LshgdBlock`` inference on one event;
* ``hgdn``       ``chunk_h_gated_delta_rule``: outputs over whole chunks, or a prefill of any length with its level states.
"""
import math

import torch

from lampa_amd import block, gated_delta, hgdn, lsh, synth

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
FEAT_DIM = 24  # features per hit


def listed():
    return [
        # one new token for each of 16 sequences on top of their states: the smallest call, latency only
        {"name": "recurrent_step", "path": "recurrent", "B": 16, "T": 1, "H": 8, "K": 64, "V": 64, "dtype": "bf16",
         "l2norm": True, "state": True, "decay": 1.0},
        # the token-serial operator in fp32 on a whole sequence (the exact mode)
        {"name": "recurrent_fp32", "path": "recurrent", "B": 1, "T": 8192, "H": 4, "K": 32, "V": 32, "dtype": "fp32",
         "l2norm": False, "state": False, "decay": 1.0},
        # one layer on a small event (the low end of 6-60 thousand hits), a ragged length
        {"name": "chunk_small_event", "path": "chunk", "B": 1, "T": 6007, "H": 8, "K": 64, "V": 64, "dtype": "bf16",
         "l2norm": True, "events": 0, "state": False, "decay": 0.05},
        # one layer on a full event: the benchmark's own shape
        {"name": "chunk_event", "path": "chunk", "B": 1, "T": 60000, "H": 8, "K": 64, "V": 64, "dtype": "bf16",
         "l2norm": False, "events": 0, "state": False, "decay": 1.0},
        # sixteen events of 6-60 thousand hits in one packed call, wide heads: the largest call
        {"name": "chunk_packed_wide", "path": "chunk", "B": 1, "T": 520000, "H": 8, "K": 128, "V": 128, "dtype": "bf16",
         "l2norm": False, "events": 16, "state": False, "decay": 1.0},
        # a training step's share of one layer on a full event
        {"name": "train_event", "path": "train", "B": 1, "T": 60000, "H": 8, "K": 64, "V": 64, "dtype": "bf16",
         "l2norm": True, "events": 0, "state": False, "decay": 1.0},
        # the same with the reference model's heads and operand type on its 15-thousand-hit events
        {"name": "train_small_heads", "path": "train", "B": 1, "T": 14983, "H": 6, "K": 16, "V": 32, "dtype": "fp16",
         "l2norm": True, "events": 0, "state": False, "decay": 0.05},
        # bucket sort of one event with its features, as inference on single events does it
        {"name": "lsh_event", "path": "lsh", "events": 1, "n": 60000, "tables": 3, "proj": 4, "feats": True},
        # bucket sort of a batch of events, as a data loader's batch does it
        {"name": "lsh_batch", "path": "lsh", "events": 32, "n": 60000, "tables": 3, "proj": 4, "feats": True},
        # the four-layer block on one event
        {"name": "block_event", "path": "block", "n": 60000, "layers": 4},
        # the hierarchical operator, outputs only (whole chunks)
        {"name": "hgdn_event", "path": "hgdn", "B": 1, "T": 60032, "H": 8, "K": 64, "V": 64, "prefill": False,
         "decay": 1.0},
        # the hierarchical operator's prefill at a length that is no multiple of the chunk, level states returned
        {"name": "hgdn_prefill", "path": "hgdn", "B": 1, "T": 15000, "H": 8, "K": 64, "V": 64, "prefill": True,
         "decay": 0.05},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _decay(rng):
    """Mean log-decay of a token over that of the benchmark's inputs: from states that forget within a chunk to states
    that carry over many."""
    return rng.choice([1.0, 0.3, 0.05])


def draw(rng):
    path = rng.choice(["recurrent", "chunk", "chunk", "train", "train", "lsh", "lsh", "block", "hgdn"])
    if path == "recurrent":
        if rng.random() < 0.5:  # a few tokens for many sequences
            return {"path": path, "B": _log_int(rng, 1, 128), "T": _log_int(rng, 1, 64), "H": rng.randint(2, 8),
                    "K": rng.choice([16, 32, 64, 128]), "V": rng.choice([32, 64, 128]),
                    "dtype": rng.choice(["bf16", "fp16", "fp32"]), "l2norm": rng.random() < 0.5, "state": True,
                    "decay": _decay(rng)}
        width = rng.choice([32, 64])  # one long sequence in fp32
        return {"path": path, "B": 1, "T": _log_int(rng, 1000, 30000), "H": rng.randint(2, 8), "K": width, "V": width,
                "dtype": "fp32", "l2norm": rng.random() < 0.5, "state": rng.random() < 0.5, "decay": _decay(rng)}
    if path == "chunk":
        events = rng.choice([0, 0, rng.randint(2, 16)])
        wide = rng.random() < 0.4
        k, v = (128, rng.choice([64, 128])) if wide else rng.choice([(64, 64), (64, 64), (64, 128), (32, 32), (16, 32)])
        return {"path": path, "B": 1 if events else rng.choice([1, 1, rng.randint(2, 4)]),
                "T": _log_int(rng, 6000 * max(1, events // 2), 30000 * events) if events else _log_int(rng, 500, 60000),
                "H": rng.randint(4, 8), "K": k, "V": v, "dtype": rng.choice(["bf16", "bf16", "fp16"]),
                "l2norm": rng.random() < 0.5, "events": events, "state": rng.random() < 0.3, "decay": _decay(rng)}
    if path == "train":
        events = rng.choice([0, 0, rng.randint(2, 8)])
        k, v = rng.choice([(64, 64), (64, 64), (32, 64), (16, 32)])
        return {"path": path, "B": 1 if events else rng.choice([1, 1, 2]),
                "T": _log_int(rng, 3000 * events, 12000 * events) if events else _log_int(rng, 1000, 60000),
                "H": rng.randint(4, 8), "K": k, "V": v, "dtype": rng.choice(["bf16", "fp16"]),
                "l2norm": rng.random() < 0.7, "events": events, "state": rng.random() < 0.3, "decay": _decay(rng)}
    if path == "lsh":
        if rng.random() < 0.5:
            return {"path": path, "events": 1, "n": _log_int(rng, 1000, 120000), "tables": rng.randint(2, 4), "proj": 4,
                    "feats": rng.random() < 0.8}
        return {"path": path, "events": rng.randint(2, 32), "n": _log_int(rng, 3000, 60000), "tables": rng.randint(2, 3),
                "proj": rng.choice([3, 4]), "feats": rng.random() < 0.8}
    if path == "block":
        return {"path": path, "n": _log_int(rng, 3000, 60000), "layers": rng.randint(1, 4)}
    prefill = rng.random() < 0.5
    t = _log_int(rng, 1000, 60000)
    return {"path": path, "B": 1, "T": t if prefill else (t + 63) // 64 * 64, "H": rng.randint(4, 8),
            "K": rng.choice([64, 64, 32]), "V": rng.choice([64, 64, 128]), "prefill": prefill,
            "decay": _decay(rng)}


# ---- inputs ------------------------------------------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda")


def _operands(gen, B, T, H, K, V, dtype, l2norm, decay):
    """q, k (raw when the operator normalises them, else unit rows), v ~ N(0,1), log-decay g = -decay softplus(N(0,1)),
    write strength beta = sigmoid(N(0,1)): the distributions of ``synth.gdr_inputs``."""
    q, k = _normal(gen, B, T, H, K), _normal(gen, B, T, H, K)
    if not l2norm:
        q, k = torch.nn.functional.normalize(q, dim=-1), torch.nn.functional.normalize(k, dim=-1)
    v = _normal(gen, B, T, H, V)
    g = -decay * torch.nn.functional.softplus(_normal(gen, B, T, H))
    beta = torch.sigmoid(_normal(gen, B, T, H))
    return q.to(dtype), k.to(dtype), v.to(dtype), g, beta


def _boundaries(seed, total, events):
    """Token boundaries of ``events`` packed events whose sizes spread over a factor of up to ten (int64, on the GPU)."""
    gen = torch.Generator().manual_seed(seed)
    share = torch.rand(events, generator=gen, dtype=torch.float64) * 0.9 + 0.1
    cu = torch.zeros(events + 1, dtype=torch.int64)
    cu[1:] = torch.round(torch.cumsum(share, 0) / share.sum() * total).to(torch.int64)
    cu[-1] = total
    return cu.cuda()


def _hits(gen, events, n):
    """Hits of ``events`` collider events on ten barrel layers (``synth.collider_event``), made on the GPU: coords
    [events, n, 4] = (eta, cos phi, sin phi, r / 1020), feats [events, n, 24]."""
    radii = torch.tensor(synth.BARREL_RADII_MM, device="cuda")
    r = radii[torch.randint(0, len(synth.BARREL_RADII_MM), (events, n), generator=gen, device="cuda")]
    eta = torch.rand(events, n, generator=gen, device="cuda") * 8.0 - 4.0
    phi = (torch.rand(events, n, generator=gen, device="cuda") * 2.0 - 1.0) * math.pi
    coords = torch.stack([eta, torch.cos(phi), torch.sin(phi), r / 1020.0], dim=-1).contiguous()
    return coords, _normal(gen, events, n, FEAT_DIM)


def prepare(case, seed):
    gen = _generator(seed)
    path = case["path"]
    state = {"case": case}
    if path in ("recurrent", "chunk", "train"):
        B, T, H, K, V = (case[x] for x in ("B", "T", "H", "K", "V"))
        events = case.get("events", 0)
        state["args"] = _operands(gen, B, T, H, K, V, DTYPES[case["dtype"]], case["l2norm"], case["decay"])
        state["h0"] = 0.3 * _normal(gen, events or B, H, K, V) if case["state"] else None
        state["cu"] = _boundaries(seed, T, events) if events else None
        if path == "train":
            state["leaves"] = [x.requires_grad_(True) for x in state["args"]]
            if state["h0"] is not None:
                state["leaves"].append(state["h0"].requires_grad_(True))
            state["do"] = _normal(gen, B, T, H, V).to(DTYPES[case["dtype"]])
    elif path == "lsh":
        coords, feats = _hits(gen, case["events"], case["n"])
        if case["events"] == 1:
            coords, feats = coords[0], feats[0]
        alpha, beta = synth.lsh_params(4, case["tables"], case["proj"], 0.5, seed)
        state.update(coords=coords, feats=feats if case["feats"] else None, alpha=alpha.cuda(), beta=beta.cuda())
    elif path == "block":
        torch.manual_seed(seed)
        state["block"] = block.LshgdBlock(n_layers=case["layers"]).cuda().to(torch.bfloat16)
        coords, feats = _hits(gen, 1, case["n"])
        state.update(coords=coords[0], feats=feats[0])
    else:
        B, T, H, K, V = (case[x] for x in ("B", "T", "H", "K", "V"))
        state["args"] = _operands(gen, B, T, H, K, V, torch.bfloat16, True, case["decay"])
        levels = hgdn.num_levels(T)
        state["lam"] = (torch.rand(B, T, H, levels, generator=gen, device="cuda") + 0.25).to(torch.bfloat16)
    return state


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "recurrent":
        return gated_delta.fused_recurrent_gated_delta_rule(*state["args"], initial_state=state["h0"],
                                                            output_final_state=True,
                                                            use_qk_l2norm_in_kernel=case["l2norm"])
    if path == "chunk":
        return gated_delta.chunk_gated_delta_rule(*state["args"], initial_state=state["h0"], output_final_state=True,
                                                  cu_seqlens=state["cu"], use_qk_l2norm_in_kernel=case["l2norm"])
    if path == "train":
        o, _ = gated_delta.chunk_gated_delta_rule(*state["args"], initial_state=state["h0"], cu_seqlens=state["cu"],
                                                  use_qk_l2norm_in_kernel=case["l2norm"])
        return (o.detach(),) + torch.autograd.grad(o, state["leaves"], state["do"])
    if path == "lsh":
        return lsh.lsh_bucket_sort(state["coords"], state["alpha"], state["beta"], 0.5, case["tables"], case["proj"],
                                   state["feats"])
    if path == "block":
        return state["block"](state["feats"], state["coords"])
    q, k, v, g, beta = state["args"]
    o, h = hgdn.chunk_h_gated_delta_rule(q, k, v, g, state["lam"], beta, output_final_state=case["prefill"],
                                         use_qk_l2norm_in_kernel=True)
    return o if h is None else (o, h.states, h.counts)


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
def _chunk_flops(K, V):
    """Per token and head of the chunkwise forward with chunks of 64 tokens."""
    return 2 * 64 * (3 * K + 2 * V) + 6 * K * V + 2 * 64 * 64 / 3


def work(case):
    path = case["path"]
    if path in ("recurrent", "chunk", "train"):
        B, T, H, K, V = (case[x] for x in ("B", "T", "H", "K", "V"))
        size = 4 if case["dtype"] == "fp32" else 2
        tokens = B * T * H
        states = (case.get("events", 0) or B) * H * K * V * 4
        read = tokens * (size * (2 * K + V) + 8) + (states if case["state"] else 0)
        if path == "train":  # q, k, v, g, beta, do once; o and the gradients of the inputs once
            return {"bytes": 2 * read + tokens * size * 2 * V, "flops": 3 * tokens * _chunk_flops(K, V)}
        flops = tokens * (8 * K * V if path == "recurrent" else _chunk_flops(K, V))
        return {"bytes": read + tokens * size * V + states, "flops": flops}
    if path == "lsh":
        hits, row = case["events"] * case["n"], 4 * FEAT_DIM if case["feats"] else 0
        return {"bytes": hits * (16 + row + case["tables"] * (4 * case["proj"] + 4 + 4 + row)),
                "flops": hits * case["tables"] * case["proj"] * 10}
    if path == "block":
        hidden, cols, width = 128, 4 * 512 + 16, 512
        per_layer = 2 * hidden * cols + 2 * width * hidden + 8 * _chunk_flops(64, 64)
        weights = case["layers"] * 2 * hidden * (cols + width)
        return {"bytes": case["n"] * (4 * FEAT_DIM + 16 + 2 * FEAT_DIM) + weights,
                "flops": case["n"] * (case["layers"] * per_layer + 4 * FEAT_DIM * hidden)}
    B, T, H, K, V = (case[x] for x in ("B", "T", "H", "K", "V"))
    levels, chunks = hgdn.num_levels(T), (T + 63) // 64
    live = sum(bin(c).count("1") for c in range(chunks))  # (chunk, level) pairs that hold a state
    moved = B * T * H * (2 * (2 * K + 2 * V + levels) + 8)
    if case["prefill"]:
        moved += B * H * K * V * levels * 4
    return {"bytes": moved, "flops": B * H * (chunks * 64 * _chunk_flops(K, V) + live * 2 * 64 * K * V)}


def tolerance(case):
    """Permutations, ids and copied features are exact. Elsewhere about four times what the roundings of the operand type
    were measured to give against the same pass in float64 on the host, over the three decays: relative 2-norms of at most
    4.9e-3 (bf16) and 6.2e-4 (fp16) for the chunk operators and their gradients, 1.7e-3 and 2.1e-4 for the token-serial
    operator (fp32 arithmetic, one rounding at the end), 6.7e-3 for the block; 4e-7 in fp32 at 4000 tokens, where sums in
    another order give up to 1e-5 on the longest sequences."""
    if case["path"] == "lsh":
        return "exact"
    if case["path"] == "block":
        return {"rel": 2.7e-2, "max": 0.15}
    dtype = case.get("dtype", "bf16")
    if dtype == "fp32":
        return {"rel": 1e-5, "max": 1e-4}
    if case["path"] == "recurrent":
        return {"rel": 7e-3, "max": 1.6e-2} if dtype == "bf16" else {"rel": 9e-4, "max": 2e-3}
    return {"rel": 2e-2, "max": 0.15} if dtype == "bf16" else {"rel": 2.5e-3, "max": 2e-2}
