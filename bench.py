#!/usr/bin/env python3
"""Benchmark of the hot path on one MI355X.

A step is one chunkwise gated-delta layer forward (B=1, H=8, T=60000, d_k=d_v=64, C=64, bf16 q/k/v, fp32 g/beta,
tokens in the LSH-sorted order of a 60000-hit event) with every input resident in HBM.
Prints one JSON line: `value` = hits/s over the timed steps (wall clock), `roofline` = the slowest kernel of the layer
against the HBM peak on its algorithmic bytes (duration from HIP events on the launch stream), `cpu_baseline` = the
pure-PyTorch token loop on this box's host cores, `layer` / `lsh` / `block` / `hgdn` = per-kernel times, the LSH stage on one
event and on a batch, the 4-layer block, and the hierarchical (level-weighted) forward.
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0       # MI355X HBM3E
MFMA_BF16_PEAK_TFLOPS = 2500.0

T, H, K, V = 60000, 8, 64, 64
N_HITS, N_TABLES, N_PROJ, W_BUCKET, FEAT_DIM = 60000, 3, 4, 0.5, 24
# algorithmic work per unit
LAYER_BYTES_PER_TOKEN_HEAD = 2 * K + 2 * K + 2 * V + 2 * V + 8                 # q,k,v,o bf16 + g,beta fp32 = 520
LAYER_FLOP_PER_TOKEN_HEAD = 2 * 64 * (3 * K + 2 * V) + 6 * K * V + (2 * 64 * 64) // 3  # 68.3 kFLOP
KERNEL_BYTES_PER_TOKEN_HEAD = {            # algorithmic bytes each kernel of the pipeline has to move
    "gdr_segment_kernel<output>": LAYER_BYTES_PER_TOKEN_HEAD,    # reads q, k, v, g, beta and writes o: the whole 520 B
    "gdr_segment_kernel<composite>": 2 * K + 2 * V + 8,           # reads k, v, g, beta
    "gdr_local_kernel": 2 * K + 8,                                # reads k, g, beta
}
LSH_BYTES_PER_HIT_TABLE = 224
# HBM bytes per launch at config 2 from rocprofv3 counters (FETCH_SIZE x 2.0 + WRITE_SIZE x 1.0, the factors a plain
# 256 MiB copy gives), read from the summary below. Counters cannot be read from inside a run.
TRAFFIC_PROFILE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "profiles",
                               "gdr_chunk_fwd_config2_hbm_traffic_pmc.md")


def measured_traffic():
    """HBM bytes per launch of every kernel of the layer from the counter summary under profiles/ (rows
    `| kernel | FETCH_SIZE KiB | WRITE_SIZE KiB | bytes |` under the line `commit: <hash>`): counters cannot be read
    from inside a run, so the figure is the last profiled one and says which commit it was measured at."""
    out, commit = {}, None
    try:
        with open(TRAFFIC_PROFILE) as fh:
            for ln in fh:
                if ln.lower().startswith("commit:"):
                    commit = ln.split(":", 1)[1].strip()
                cells = [c.strip() for c in ln.strip().strip("|").split("|")]
                if len(cells) == 4 and cells[0].startswith("gdr_"):
                    try:
                        out[cells[0]] = float(cells[3])
                    except ValueError:
                        pass
    except OSError:
        pass
    return out, commit


def _median(xs):
    xs = sorted(xs)
    return xs[len(xs) // 2]


def cpu_baseline_gdr(q, k, v, g, beta, sample_tokens, repeats=5, warmups=3):
    """The reference's CPU path for the layer: a token loop in plain PyTorch (port: oracle.gated_delta.recurrent_delta,
    fp32) on a prefix of the same inputs: `warmups` untimed passes over a 256-token prefix, then `repeats` timed passes
    over the first `sample_tokens` tokens; the median, scaled to hits/s (the loop is serial in the tokens)."""
    import torch
    from oracle import gated_delta as og

    sl = slice(0, sample_tokens)
    args = [x[:, sl].float() for x in (q, k, v, g, beta)]
    for _ in range(warmups):
        og.recurrent_delta(*[a[:, :256] for a in args], dtype=torch.float32)
    times = []
    for _ in range(repeats):
        t0 = time.perf_counter()
        og.recurrent_delta(*args, dtype=torch.float32)
        times.append(time.perf_counter() - t0)
    dt = _median(times)
    return sample_tokens / dt, dt


def cpu_baseline_lsh(coords, feats, alpha, offsets):
    """The reference's CPU path for the LSH stage in plain PyTorch: bmm -> + offset -> quantise -> pack -> stable sort
    -> gather (the function the GPU leg computes); 3 untimed passes, then the median of 5."""
    import torch

    times = []
    for it in range(8):
        t0 = time.perf_counter()
        proj = torch.bmm(coords[None], alpha[None])[0] + offsets[None, :]
        ids = torch.floor(proj / W_BUCKET).to(torch.int64).T.reshape(N_TABLES, N_PROJ, -1)
        lo = ids.amin(-1, keepdim=True)
        rng = ids.amax(-1, keepdim=True) - lo + 1
        stride = torch.cumprod(torch.cat([torch.ones_like(rng[:, :1]), rng[:, :-1]], 1), 1)
        keys = ((ids - lo) * stride).sum(1)
        perm = torch.sort(keys, dim=-1, stable=True).indices
        out = feats[None].expand(N_TABLES, -1, -1).gather(1, perm[..., None].expand(-1, -1, feats.shape[-1]))
        if it >= 3:
            times.append(time.perf_counter() - t0)
    del out
    return _median(times)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    # (a layer is ~0.12 ms: 50 + 200 steps take 30 ms; the clocks are settled by the untimed steps of --prewarm-ms)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=50)
    ap.add_argument("--cpu-sample-tokens", type=int, default=8192,
                    help="prefix of the workload the CPU baseline is timed on (median of 5 passes, scaled linearly)")
    ap.add_argument("--prewarm-ms", type=float, default=1000.0,
                    help="untimed steps run before the warm-up until this much wall clock has passed AND five batches "
                         "of 20 steps in a row agree within 2 % (at most three times as long), so that the clocks of a "
                         "GPU that was idle have settled whatever --warmup is")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baselines (for profiler runs)")
    ap.add_argument("--copy-probe", action="store_true",
                    help="first run one plain device copy of 256 MiB, the known-size kernel that scales a counter run")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py: this build runs the hot path on ONE GPU; --gpus must be 1 "
              "(heads, sequences and segments would shard across GPUs; that is not implemented).", file=sys.stderr)
        sys.exit(2)

    import torch
    from lampa_amd import _capi
    from lampa_amd import gated_delta as gd
    from lampa_amd import lsh, synth

    if not os.path.exists(_capi.LIB_PATH):
        from lampa_amd import build as lib_build
        lib_build.build()
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)

    if args.copy_probe:
        src = torch.empty(256 << 20, dtype=torch.uint8, device=dev).fill_(1)
        dst = torch.empty_like(src)
        torch.cuda.synchronize()
        dst.copy_(src)  # 256 MiB read + 256 MiB written by one elementwise copy kernel
        torch.cuda.synchronize()
        del src, dst

    # ---- inputs (synthetic, seeded) ----
    coords, feats, _ = synth.collider_event(N_HITS, seed=0)
    alpha, beta_h = synth.lsh_params(4, N_TABLES, N_PROJ, W_BUCKET, 1)
    q, k, v, g, beta = synth.gdr_inputs(1, T, H, K, V, torch.bfloat16, seed=0)
    coords_d, feats_d, alpha_d, beta_hd = (x.to(dev) for x in (coords, feats, alpha, beta_h))
    perm = lsh.lsh_bucket_sort(coords_d, alpha_d, beta_hd, W_BUCKET, N_TABLES, N_PROJ)["perm"][0].long().cpu()
    q, k, v, g, beta = (x[:, perm].contiguous() for x in (q, k, v, g, beta))
    qd, kd, vd, gd_, bd = (x.to(dev) for x in (q, k, v, g, beta))

    def step():
        return gd.chunk_gated_delta_rule(qd, kd, vd, gd_, bd, output_final_state=True)

    def settle(fn, ms=60.0):
        """Untimed calls of a leg's step for `ms` of wall clock before its own warm-up: every leg prepares its inputs on
        the host first, the GPU idles meanwhile, and for about 30 ms after an idle spell everything runs up to a third
        slower (clocks)."""
        t_ = time.perf_counter()
        while 1e3 * (time.perf_counter() - t_) < ms:
            fn()
            fn()
            torch.cuda.synchronize()

    # ---- clock settling (untimed, stated in the output), then W warm-up steps, then the timed region: exactly K steps ----
    # (On a box whose GPU had been idle, the first 20-step region timed 150 ms after the first launch read 146-150 us per
    # step twice where every later process read 120-123: the region is 2.4 ms long, and one power-state change of the
    # memory system inside it is a fifth of it. Hence the longer settling and the check that the step time is steady.)
    t_pre = time.perf_counter()
    n_pre = 0
    recent = []
    while True:
        tb = time.perf_counter()
        for _ in range(20):
            step()
        torch.cuda.synchronize()
        n_pre += 20
        recent = (recent + [time.perf_counter() - tb])[-5:]
        spent = 1e3 * (time.perf_counter() - t_pre)
        steady = len(recent) == 5 and max(recent) <= 1.02 * min(recent)
        if (spent >= args.prewarm_ms and steady) or spent >= 3 * args.prewarm_ms:
            break
    prewarm_ms = 1e3 * (time.perf_counter() - t_pre)
    import gc
    gc.disable()  # no collector pause inside the timed region (and no collection here: while the host is busy the GPU
                  # idles, its clocks drop, and the next ~200 steps are up to a third slower)
    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    gc.enable()
    ms_per_step = 1e3 * elapsed / args.steps
    hits_per_s = T / (elapsed / args.steps)

    # ---- per-kernel durations with HIP events on the launch stream (separate pass of the same steps) ----
    _capi.profile_begin()
    for _ in range(args.steps):
        step()
    prof = _capi.profile_end(max_entries=8 * args.steps + 8)
    stage = {}
    for name, ms in prof:
        stage.setdefault(name, []).append(ms)
    stage_us = {name: 1e3 * sum(v_) / len(v_) for name, v_ in stage.items()}
    dominant = max(stage_us, key=stage_us.get)
    token_heads = T * H
    dom_bytes = KERNEL_BYTES_PER_TOKEN_HEAD.get(dominant, LAYER_BYTES_PER_TOKEN_HEAD) * token_heads
    dom_gbs = dom_bytes / (stage_us[dominant] * 1e-6) / 1e9
    layer_us = ms_per_step * 1e3
    traffic_table, traffic_commit = measured_traffic()
    roofline = {"bound": "hbm", "kernel": dominant, "achieved": round(dom_gbs, 1), "peak": HBM_PEAK_GBS,
                "unit": "GB/s", "frac": round(dom_gbs / HBM_PEAK_GBS, 4), "traffic": traffic_table.get(dominant),
                "traffic_measured_at_commit": traffic_commit,
                "kernel_us": round(stage_us[dominant], 2), "algorithmic_bytes_per_launch": dom_bytes}
    # ---- what the output pass's access pattern costs with no arithmetic (memory-only twin of that kernel: same rows
    #      of q, k, v, the per-chunk records and the o rows per workgroup and chunk; whole chunks only) ----
    n_chunks_probe = T // 64
    rec = torch.zeros(n_chunks_probe * H * 5376, dtype=torch.uint8, device=dev)
    o_probe = torch.empty_like(vd)
    cps_probe = gd._default_chunks_per_segment([(T + 63) // 64], H, 2 * torch.cuda.get_device_properties(dev).multi_processor_count)

    def probe():
        _capi.check(_capi.lib().lampa_gdr_traffic_probe(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), rec.data_ptr(),
                                                        o_probe.data_ptr(), n_chunks_probe, H, cps_probe,
                                                        torch.cuda.current_stream().cuda_stream), "traffic probe")
    for _ in range(20):
        probe()
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    ev0.record()
    for _ in range(100):
        probe()
    ev1.record()
    torch.cuda.synchronize()
    probe_us = 1e3 * ev0.elapsed_time(ev1) / 100
    probe_bytes = n_chunks_probe * H * (4 * 64 * 64 * 2 + 4608)  # q, k, v, o rows and the T blocks of the record
    roofline["memory_only_twin"] = {
        "us": round(probe_us, 2), "bytes": probe_bytes, "GB/s": round(probe_bytes / (probe_us * 1e-6) / 1e9, 1),
        "kernel_over_twin": round(stage_us.get("gdr_segment_kernel<output>", float("nan")) / probe_us, 3),
        "note": "the output pass's loads and stores with no arithmetic (lampa_gdr_traffic_probe), 100 launches with "
                "HIP events: the practical floor of that kernel on this memory system"}
    # the same twin with the reads of a whole walk over the earlier composites in front of the first chunk (the second level of the
    # two-level scan runs inside the output pass): the floor of the kernel where no segment cuts off its past. At these inputs'
    # decays every segment does, and the kernel reads one composite or none: its own floor is the twin above.
    n_seg_probe = (n_chunks_probe + cps_probe - 1) // cps_probe
    comp = torch.zeros((n_seg_probe + (n_seg_probe + 7) // 8) * H * 24576, dtype=torch.uint8, device=dev)

    def probe_walk():
        _capi.check(_capi.lib().lampa_gdr_traffic_probe_walk(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), rec.data_ptr(),
                                                             comp.data_ptr(), o_probe.data_ptr(), n_chunks_probe, H,
                                                             cps_probe, torch.cuda.current_stream().cuda_stream),
                    "traffic probe (walk)")
    for _ in range(20):
        probe_walk()
    ev0.record()
    for _ in range(100):
        probe_walk()
    ev1.record()
    torch.cuda.synchronize()
    walk_us = 1e3 * ev0.elapsed_time(ev1) / 100
    walk_steps = sum(s_ // 8 + s_ % 8 for s_ in range(n_seg_probe))
    walk_bytes = probe_bytes + walk_steps * H * 24576
    roofline["memory_only_twin_with_walk"] = {
        "us": round(walk_us, 2), "bytes": walk_bytes, "GB/s": round(walk_bytes / (walk_us * 1e-6) / 1e9, 1),
        "kernel_over_twin": round(stage_us.get("gdr_segment_kernel<output>", float("nan")) / walk_us, 3),
        "note": "the twin above plus the composites of a whole walk over the scan's second level before the first chunk "
                "(lampa_gdr_traffic_probe_walk: per step and wave 8 KiB of M' and 8 KiB of N, two steps ahead), which the "
                "kernel makes where no segment cuts off its past; at these inputs it starts behind the last one"}
    del rec, o_probe, comp
    # ---- per-step distribution (HIP events on the launch stream, one pair per step) and a cold variant that rotates
    #      among input sets totalling more than 512 MB, so that no step finds its inputs in the memory-side cache ----
    def event_times(fn, n):
        evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(n)]
        for i, (a, b) in enumerate(evs):
            a.record()
            fn(i)
            b.record()
        torch.cuda.synchronize()
        return sorted(1e3 * a.elapsed_time(b) for a, b in evs)

    def pct(xs, p):
        return round(xs[min(len(xs) - 1, int(p * len(xs)))], 2)

    n_dist = max(100, args.steps)
    warm = event_times(lambda i: step(), n_dist)
    sets = [(qd, kd, vd, gd_, bd)] + [tuple(x.clone() for x in (qd, kd, vd, gd_, bd)) for _ in range(2)]
    set_mb = sum(x.numel() * x.element_size() for x in sets[0]) / 1e6
    for i in range(6):
        gd.chunk_gated_delta_rule(*sets[i % 3], output_final_state=True)
    cold = event_times(lambda i: gd.chunk_gated_delta_rule(*sets[i % 3], output_final_state=True), n_dist)
    del sets
    timing = {
        "steps": n_dist, "unit": "us per layer, HIP events around each step",
        "warm": {"median": pct(warm, 0.5), "p10": pct(warm, 0.1), "p90": pct(warm, 0.9)},
        "cold": {"median": pct(cold, 0.5), "p10": pct(cold, 0.1), "p90": pct(cold, 0.9),
                 "input_sets": 3, "mb_per_set": round(set_mb, 1)},
    }
    layer = {
        "us_per_layer": round(layer_us, 2), "timing": timing,
        "hbm_frac": round(LAYER_BYTES_PER_TOKEN_HEAD * token_heads / (layer_us * 1e-6) / 1e9 / HBM_PEAK_GBS, 4),
        "mfma_frac": round(LAYER_FLOP_PER_TOKEN_HEAD * token_heads / (layer_us * 1e-6) / 1e12 / MFMA_BF16_PEAK_TFLOPS, 4),
        "kernel_us": {n: round(u, 2) for n, u in stage_us.items()},
        "kernel_us_sum": round(sum(stage_us.values()), 2),
        "kernel_us_note": "HIP-event intervals of a separate pass: each holds the kernel and the gap to the next launch, "
                          "and recording the events slows the pipeline by a few us, so their sum exceeds us_per_layer; "
                          "the kernel-trace durations are in profiles/",
    }

    # ---- LSH stage (config 1): ids + keys + stable sort + feature gather, 3 tables ----
    def lsh_step():
        return lsh.lsh_bucket_sort(coords_d, alpha_d, beta_hd, W_BUCKET, N_TABLES, N_PROJ, feats_d)

    settle(lsh_step)
    for _ in range(args.warmup):
        lsh_step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        lsh_step()
    torch.cuda.synchronize()
    lsh_us = 1e6 * (time.perf_counter() - t0) / args.steps
    _capi.profile_begin()
    for _ in range(args.steps):
        lsh_step()
    lprof = _capi.profile_end(max_entries=16 * args.steps + 16)
    lstage = {}
    for name, ms in lprof:
        lstage.setdefault(name, []).append(ms)
    lsh_bytes = LSH_BYTES_PER_HIT_TABLE * N_HITS * N_TABLES
    lsh_kernel_us = {n: round(1e3 * sum(v_) / args.steps, 2) for n, v_ in lstage.items()}
    lsh_gpu_us = sum(lsh_kernel_us.values())
    lsh_info = {
        "workload": f"config1: N={N_HITS}, {N_TABLES} tables x {N_PROJ} proj, w={W_BUCKET}, {FEAT_DIM} fp32 feats",
        "us_per_event": round(lsh_us, 2), "hits_per_s": round(N_HITS / (lsh_us * 1e-6), 1),
        "launches_per_event": round(len(lprof) / args.steps, 2),
        "sum_kernel_us": round(lsh_gpu_us, 2), "kernel_us_per_event": lsh_kernel_us,
        "roofline": {"bound": "hbm", "achieved": round(lsh_bytes / (lsh_us * 1e-6) / 1e9, 1), "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": round(lsh_bytes / (lsh_us * 1e-6) / 1e9 / HBM_PEAK_GBS, 4),
                     "algorithmic_bytes": lsh_bytes},
    }

    # ---- the same stage on a batch of events in one set of launches (throughput form of config 1) ----
    n_batch = 32
    bc, bf = [], []
    for e in range(n_batch):
        c_e, f_e, _ = synth.collider_event(N_HITS, seed=e)
        bc.append(c_e)
        bf.append(f_e)
    bc_d, bf_d = torch.stack(bc).to(dev), torch.stack(bf).to(dev)

    def lsh_batch_step():
        return lsh.lsh_bucket_sort(bc_d, alpha_d, beta_hd, W_BUCKET, N_TABLES, N_PROJ, bf_d)

    settle(lsh_batch_step)
    for _ in range(3):
        lsh_batch_step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(10):
        lsh_batch_step()
    torch.cuda.synchronize()
    batch_us = 1e6 * (time.perf_counter() - t0) / 10
    lsh_info["batch"] = {
        "events": n_batch, "us_per_event": round(batch_us / n_batch, 2),
        "hits_per_s": round(n_batch * N_HITS / (batch_us * 1e-6), 1),
        "roofline": {"bound": "hbm", "achieved": round(n_batch * lsh_bytes / (batch_us * 1e-6) / 1e9, 1),
                     "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": round(n_batch * lsh_bytes / (batch_us * 1e-6) / 1e9 / HBM_PEAK_GBS, 4)},
    }
    del bc_d, bf_d

    # ---- config 3: the 4-layer block on one event (input linear, LSH sort, layers, unsort, head), bf16 weights seed 2 ----
    from lampa_amd import block as lblock
    torch.manual_seed(2)
    blk = lblock.LshgdBlock().to(dev).to(torch.bfloat16)
    settle(lambda: blk(feats_d, coords_d))
    for _ in range(3):
        blk(feats_d, coords_d)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(10):
        blk(feats_d, coords_d)
    torch.cuda.synchronize()
    block_us = 1e6 * (time.perf_counter() - t0) / 10
    _capi.profile_begin()
    blk(feats_d, coords_d)
    bstage = {}
    for name, ms in _capi.profile_end(max_entries=512):
        bstage[name] = bstage.get(name, 0.0) + 1e3 * ms
    block_info = {
        "workload": f"config3: N={N_HITS} hits, linear 24->128, LSH sort, 4 gated-delta layers (H=8, d=64, conv 4, SiLU "
                    "gate, RMS norm), unsort, head 128->24; bf16 weights, seed 2",
        "us_per_event": round(block_us, 1), "hits_per_s": round(N_HITS / (block_us * 1e-6), 1),
        "own_kernel_us": {n: round(v_, 1) for n, v_ in bstage.items()},
        "note": "own_kernel_us: this package's kernels with HIP events; the rest of the time is the library GEMMs "
                "(projections) and launch gaps",
    }
    del blk

    # ---- hierarchical (level-weighted) forward on the config-2 shape padded to whole chunks ----
    from lampa_amd import hgdn
    T_H = (T + 63) // 64 * 64
    pad = T_H - T
    qh, kh, vh = (torch.nn.functional.pad(x, (0, 0, 0, 0, 0, pad)) for x in (qd, kd, vd))
    gh, bh = (torch.nn.functional.pad(x, (0, 0, 0, pad)) for x in (gd_, bd))
    L_H = hgdn.num_levels(T_H)
    lam = (torch.rand(1, T_H, H, L_H, generator=torch.Generator().manual_seed(3)) + 0.25).to(torch.bfloat16).to(dev)
    for _ in range(30):  # (long enough for the clocks to settle after the host-side work of the previous leg)
        hgdn.chunk_h_gated_delta_rule(qh, kh, vh, gh, lam, bh, use_qk_l2norm_in_kernel=True)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(100):
        hgdn.chunk_h_gated_delta_rule(qh, kh, vh, gh, lam, bh, use_qk_l2norm_in_kernel=True)
    torch.cuda.synchronize()
    hgdn_us = 1e6 * (time.perf_counter() - t0) / 100
    _capi.profile_begin()
    for _ in range(10):
        hgdn.chunk_h_gated_delta_rule(qh, kh, vh, gh, lam, bh, use_qk_l2norm_in_kernel=True)
    hstage = {}
    for name, ms in _capi.profile_end(max_entries=512):
        if name != "start":
            hstage[name] = hstage.get(name, 0.0) + 1e3 * ms / 10
    live = sum(bin(c).count("1") for c in range(T_H // 64)) * H  # (chunk, head, level) triples that hold a state
    hgdn_flop = (T_H // 64) * H * 2 * 64 * 64 * (3 * K + 2 * V + 42) + live * 6 * 64 * K * V
    # prefill (outputs + level states) and the single-token step that continues it
    for _ in range(3):
        _, hst = hgdn.chunk_h_gated_delta_rule(qh, kh, vh, gh, lam, bh, output_final_state=True,
                                               use_qk_l2norm_in_kernel=True)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(10):
        _, hst = hgdn.chunk_h_gated_delta_rule(qh, kh, vh, gh, lam, bh, output_final_state=True,
                                               use_qk_l2norm_in_kernel=True)
    torch.cuda.synchronize()
    prefill_us = 1e6 * (time.perf_counter() - t0) / 10
    one = [x[:, :1].contiguous() for x in (qh, kh, vh, gh, lam, bh)]
    import warnings as _w
    with _w.catch_warnings():
        _w.simplefilter("ignore")  # the operator warns when seq_len (1) < num_heads, as the reference does
        for _ in range(5):
            hgdn.chunk_h_gated_delta_rule(*one, initial_state=hst, output_final_state=True, use_qk_l2norm_in_kernel=True)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(50):
            hgdn.chunk_h_gated_delta_rule(*one, initial_state=hst, output_final_state=True, use_qk_l2norm_in_kernel=True)
        torch.cuda.synchronize()
    step_us = 1e6 * (time.perf_counter() - t0) / 50
    step_bytes = 2 * hst.states.numel() * 4
    del hst, one
    hgdn_info = {
        "workload": f"hierarchical gated-delta forward, B=1 H={H} T={T_H} K=V={K}, L={L_H} levels, bf16, weak "
                    "hierarchy base 2",
        "us": round(hgdn_us, 1), "hits_per_s": round(T / (hgdn_us * 1e-6), 1),
        "kernel_us": {n: round(v_, 1) for n, v_ in hstage.items()},
        "mfma_frac": round(hgdn_flop / (hgdn_us * 1e-6) / 2.5e15, 4),
        "prefill_us": round(prefill_us, 1),
        "step": {"us": round(step_us, 1), "state_bytes_read_and_written": step_bytes,
                 "hbm_frac": round(step_bytes / (step_us * 1e-6) / 1e9 / HBM_PEAK_GBS, 4)},
        "note": "wall clock of chunk_h_gated_delta_rule; mfma_frac = algorithmic flops "
                "(per chunk and head 2*64*64*(3K+2V+42) for the chunk-local products with triangular factors counted as such, 6*64*K*V per occupied level) "
                "over the bf16 dense peak",
    }
    del qh, kh, vh, gh, bh, lam

    # ---- config 0: the reference's own CPU-runnable case (B=1, H=4, T=8192, d_k=d_v=32, fp32, seed 0) on the fp32 paths ----
    q0, k0, v0, g0, b0 = synth.gdr_inputs(1, 8192, 4, 32, 32, torch.float32, seed=0)
    d0 = [x.to(dev) for x in (q0, k0, v0, g0, b0)]

    def time_us(fn, n=20, w=3):
        if w > 1:
            settle(fn)
        for _ in range(w):
            fn()
        torch.cuda.synchronize()
        t_ = time.perf_counter()
        for _ in range(n):
            fn()
        torch.cuda.synchronize()
        return 1e6 * (time.perf_counter() - t_) / n

    c0_us = time_us(lambda: gd.fused_recurrent_gated_delta_rule(*d0, output_final_state=True))
    _capi.profile_begin()
    for _ in range(5):
        gd.fused_recurrent_gated_delta_rule(*d0, output_final_state=True)
    c0_stage = {}
    for name, ms in _capi.profile_end(max_entries=64):
        if name != "start":
            c0_stage[name] = c0_stage.get(name, 0.0) + 1e3 * ms / 5
    # the same operator in fp32 at the headline shape (the fp32 mode of the chunk operator, allow_fp32=True)
    d2f = [x.to(dev) for x in synth.gdr_inputs(1, T, H, K, V, torch.float32, seed=0)]
    f32_us = time_us(lambda: gd.chunk_gated_delta_rule(*d2f, output_final_state=True, allow_fp32=True), n=5, w=2)
    del d2f
    config0 = {"workload": "config0: token-serial gated delta, B=1 H=4 T=8192 d_k=d_v=32, fp32, zero initial state",
               "us": round(c0_us, 1), "hits_per_s": round(8192 / (c0_us * 1e-6), 1),
               "kernel_us": {n: round(v_, 1) for n, v_ in c0_stage.items()},
               "fp32_mode_at_config2_shape": {"us": round(f32_us, 1), "hits_per_s": round(T / (f32_us * 1e-6), 1)},
               "note": "the sequence is cut into segments that run in parallel: every segment's affine map, a serial "
                       "scan over the maps, then every segment from its true initial state; fp32 throughout"}
    if not args.no_cpu:
        c0_cpu_hps, c0_cpu_dt = cpu_baseline_gdr(q0, k0, v0, g0, b0, 8192, repeats=5, warmups=3)
        config0["cpu_baseline"] = {"value": round(c0_cpu_hps, 1), "unit": "hits/s", "seconds": round(c0_cpu_dt, 3),
                                   "cores": torch.get_num_threads(), "kind": "port"}
    del d0

    # ---- config 4: 16 packed events of U[6000, 60000] hits, H = 8, K = V = 128, bf16 (varlen, two-level scan) ----
    lens4, cu4 = synth.varlen_lengths(16, 6000, 60000, seed=0)
    T4 = int(cu4[-1])
    d4 = [x.to(dev) for x in synth.gdr_inputs(1, T4, 8, 128, 128, torch.bfloat16, seed=4)]
    cu4d = cu4.to(dev)
    c4_us = time_us(lambda: gd.chunk_gated_delta_rule(*d4, output_final_state=True, cu_seqlens=cu4d), n=20, w=5)
    _capi.profile_begin()
    for _ in range(5):
        gd.chunk_gated_delta_rule(*d4, output_final_state=True, cu_seqlens=cu4d)
    c4_stage = {}
    for name, ms in _capi.profile_end(max_entries=64):
        c4_stage.setdefault(name, []).append(ms)
    th4 = T4 * 8
    config4 = {"workload": f"config4: 16 packed events ({T4} tokens), H=8, K=V=128, bf16, cu_seqlens",
               "us": round(c4_us, 1), "hits_per_s": round(T4 / (c4_us * 1e-6), 1),
               "hbm_frac": round(1032 * th4 / (c4_us * 1e-6) / 1e9 / HBM_PEAK_GBS, 4),
               "mfma_frac": round(182.9e3 * th4 / (c4_us * 1e-6) / 1e12 / MFMA_BF16_PEAK_TFLOPS, 4),
               "kernel_us": {n: round(1e3 * sum(v_) / len(v_), 1) for n, v_ in c4_stage.items()},
               "note": "algorithmic work per token-head: 1032 B and 182.9 kFLOP"}
    del d4

    # ---- backward pass of the layer at the headline shape and at the reference model's head sizes: the chunked form on
    #      the MFMA (lampa_gdr_chunk_fwd_train, then lampa_gdr_bwd_saved) and, beside it, the fp32 token-serial form
    #      (lampa_gdr_bwd) ----
    def backward_leg(T_, H_, K_, V_, dtype_):
        qb, kb, vb, gb_, bb = (x.to(dev) for x in synth.gdr_inputs(1, T_, H_, K_, V_, dtype_, seed=0))
        dob = torch.randn_like(vb)
        fn = lambda: gd._backward_launch(qb, kb, vb, gb_, bb, K_ ** -0.5, None, None, gd.L2_CHUNK, dob, None)
        out_ = {"workload": f"gradients of one gated-delta layer, B=1 H={H_} T={T_} K={K_} V={V_}, "
                            f"{str(dtype_).split('.')[-1]} q/k/v/do"}
        for form, flag in (("chunked", True), ("token_serial", False)):
            gd.CHUNKED_BACKWARD = flag
            try:
                us = time_us(fn, n=10 if flag else 5, w=3)
                _capi.profile_begin()
                fn()
                stage = {}
                for name, ms in _capi.profile_end(max_entries=64):
                    if name != "start":
                        stage[name] = stage.get(name, 0.0) + 1e3 * ms
            finally:
                gd.CHUNKED_BACKWARD = True
            out_[form] = {"us": round(us, 1), "hits_per_s": round(T_ / (us * 1e-6), 1),
                          "kernel_us": {n: round(v_, 1) for n, v_ in stage.items()}}
        out_["us"] = out_["chunked"]["us"]  # what chunk_gated_delta_rule's autograd takes
        return out_

    backward = {"config2_shape": backward_leg(T, H, K, V, torch.bfloat16),
                "reference_model_heads": backward_leg(30016, 6, 16, 32, torch.float16),
                "note": "chunked: the forward again, keeping records, states and segment maps, then one walk per "
                        "segment from the last chunk to the first on the MFMA; operands in the input type (heads below 64 x 64 zero-padded). token_serial: fp32, "
                        "parallel segments, a state kept every 8 tokens. Both: dq, dk, dv, dg, dbeta out, q/k "
                        "normalisation included"}

    # ---- the reference layer's own head sizes (d_k = 16, d_v = 32, H = 6, fp16, T = 30000): the chunk operator
    #      (zero-padded 32 x 32 heads) against the token-serial operator in parallel segments and as one run per head ----
    qs, ks, vs, gs, bs = (x.to(dev) for x in synth.gdr_inputs(1, 30000, 6, 16, 32, torch.float16, seed=48, g_scale=0.05))
    sm_chunk = time_us(lambda: gd.chunk_gated_delta_rule(qs, ks, vs, gs, bs), n=10, w=3)
    sm_seg = time_us(lambda: gd.fused_recurrent_gated_delta_rule(qs, ks, vs, gs, bs), n=10, w=3)
    keep = gd.SEGMENT_MIN_TOKENS
    gd.SEGMENT_MIN_TOKENS = None
    try:
        sm_loop = time_us(lambda: gd.fused_recurrent_gated_delta_rule(qs, ks, vs, gs, bs), n=1, w=1)
    finally:
        gd.SEGMENT_MIN_TOKENS = keep
    small_heads = {"workload": "B=1 H=6 T=30000 K=16 V=32 fp16 (the reference layer's head sizes)",
                   "chunk_us": round(sm_chunk, 1), "token_serial_segments_us": round(sm_seg, 1),
                   "token_serial_one_run_per_head_us": round(sm_loop, 1)}
    del qs, ks, vs, gs, bs

    # ---- CPU baseline (reported, not a target): the reference's pure-PyTorch path on this box's host cores ----
    cpu = None
    if not args.no_cpu:
        cores = torch.get_num_threads()
        n_cpu = min(T, max(64, args.cpu_sample_tokens))
        cpu_hits_per_s, cpu_dt = cpu_baseline_gdr(q, k, v, g, beta, n_cpu)
        lsh_cpu_s = cpu_baseline_lsh(coords, feats, alpha, beta_h)
        lsh_info["cpu_baseline_us"] = round(lsh_cpu_s * 1e6, 1)
        # the same loop on one thread, on a shorter prefix (the loop is serial in the tokens: time scales linearly)
        n_one = min(n_cpu, 2048)
        torch.set_num_threads(1)
        one_hits_per_s, one_dt = cpu_baseline_gdr(q, k, v, g, beta, n_one, repeats=3, warmups=1)
        torch.set_num_threads(cores)
        cpu_model = ""
        try:
            with open("/proc/cpuinfo") as fh:
                cpu_model = next((ln.split(":", 1)[1].strip() for ln in fh if ln.startswith("model name")), "")
        except OSError:
            pass
        cpu = {"value": round(cpu_hits_per_s, 1), "unit": "hits/s", "cores": cores, "kind": "port",
               "cpu_model": cpu_model,
               "one_thread": {"value": round(one_hits_per_s, 1),
                              "sample": f"first {n_one} tokens, median of 3 passes ({one_dt:.2f} s each)"},
               "sample": f"first {n_cpu} of {T} tokens, all {H} heads, fp32 token loop in PyTorch: 3 warm-ups on 256 "
                         f"tokens, median of 5 timed passes ({cpu_dt:.2f} s each)"
                         + ("" if n_cpu == T else ", scaled linearly to hits/s"),
               "cpu_count": os.cpu_count()}

    out = {
        "metric": "hits/s per gated-delta layer at T=60k (bf16); % HBM and MFMA roofline",
        "value": round(hits_per_s, 1), "unit": "hits/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "prewarm_ms": round(prewarm_ms, 1), "prewarm_steps": n_pre,
        "ms_per_step": round(ms_per_step, 5), "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "bf16", "data": "synthetic",
        "config": {"workload": "config2: chunk gated-delta forward, B=1 H=8 T=60000 K=V=64 C=64, bf16 q/k/v, fp32 "
                               "g/beta/state, LSH-sorted token order of a config-1 event"},
        "roofline": roofline, "cpu_baseline": cpu, "layer": layer, "lsh": lsh_info, "block": block_info, "hgdn": hgdn_info, "config0": config0, "config4": config4, "backward": backward, "small_heads": small_heads,
    }
    print(json.dumps(out))


if __name__ == "__main__":
    main()
