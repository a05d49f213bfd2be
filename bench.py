"""Benchmark of the FP8 block-scale MoE operator on one MI355X.

``python bench.py [--gpus 1] [--steps K] [--warmup W] [--workloads a,b,...]``

A step is one call of the operator (routing -> permute -> GEMM1+SwiGLU -> GEMM2 -> combine) on a
seeded synthetic batch already resident in HBM. Every BASELINE configuration is measured in one
run: the T=16 plumbing case, the decode-sized T=64 headline, the prefill-sized T=4096 case, the
skewed T=16384 case and the Qwen3-style T=1024 case. Each workload first runs W warm-up calls and
then keeps calling for at least ``--settle-ms`` of wall time (clocks settle over tens of ms of
load, whatever the call length), then times K (at least 20) back-to-back calls between two HIP
events. Consecutive calls cycle through ``--weight-sets`` (default 3) distinct weight sets, as
consecutive MoE layers would, so no call finds the previous call's weights in a cache.

Prints ONE JSON line. ``value`` is TFLOP/s of the headline workload over algorithmic FLOPs
(6*H*I per local (token, expert) pair, pairs counted from the routing of the run). Each workload
carries a ``roofline`` block for its dominant kernel (the stage with the largest time, from
events the library records on the operator's stream); the top-level ``roofline`` is the
headline's. Every workload also carries a ``cpu_baseline``: the CPU oracle (the
dequantise-then-fp32 PyTorch-CPU restatement of the operator) timed on all host cores on the same
inputs (median of 3; a single call for the skewed T=16384 batch); the top-level one is the
headline's.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

import torch

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)

from justgoal_amd import _lib  # noqa: E402
from justgoal_amd import inputs as jin  # noqa: E402
from justgoal_amd.geometry import BLOCK, bytes_per_token, flops_per_pair, weight_bytes_per_expert  # noqa: E402
from justgoal_amd.moe import bind, workspace_views  # noqa: E402

METRIC = "ms/call + TFLOPS, DS-V3 FP8 MoE at T=64 and T=4096; % of FP8 MFMA/HBM peak"
PEAK_HBM_GBS = 8000.0
PEAK_FP8_TFLOPS = 5000.0
PEAK_BF16_TFLOPS = 2500.0
STAGES = ("route", "permute", "gemm1_swiglu", "gemm2", "combine")
# Kernel-family thresholds of justgoal_amd/csrc/moe_gemm.hip (kStreamMaxRows, kBigRows,
# kG2TileMaxRows; tests/test_bench.py checks they match the source)
GEMM1_STREAM_MAX_ROWS = 4
GEMM1_BIG_ROWS = 16
GEMM2_TILE_MAX_ROWS = 7
# ... and of justgoal_amd/csrc/moe_wide.hip (kBigTileRows, kMinRounds), on 256 CUs
GEMM2_BIG_TILE_ROWS = 64
GEMM2_WIDE_MIN_ROUNDS = 5
GEMM2_TOKEN_MAX_ROWS, GEMM2_TOKEN_MAX_PAIRS, GEMM2_TOKEN_MIN_COLS = 16, 96, 16
CUS = 256


def log(msg):
    print(msg, file=sys.stderr, flush=True)


def routing_stats(geom, T, ws):
    """Routed pairs, active local experts and tokens with a local pair, read from the workspace
    of the call that just ran."""
    v = workspace_views(geom, T, ws)
    counts = v["counts"].cpu()
    pairs = int(counts.sum())
    active = int((counts > 0).sum())
    tok_local = int(((v["pair_of"].cpu() >= 0).any(dim=1)).sum())
    return pairs, active, tok_local


def algorithmic(geom, T, pairs, active, tok_local):
    """FLOPs and HBM bytes the operator must move (intermediates excluded), and the same for the
    two expert GEMMs on their own (each with the intermediates it must read or write once)."""
    H, I = geom.hidden, geom.intermediate
    flops = flops_per_pair(geom) * pairs
    bytes_ = active * weight_bytes_per_expert(geom) + T * bytes_per_token(geom) + 2 * geom.num_experts
    # GEMM1 + SwiGLU alone: W13 + S13 of active experts, routed fp8 rows + scales, bf16 C rows
    w13 = 2 * I * H + 4 * (2 * I // BLOCK) * (H // BLOCK)
    g1_bytes = active * w13 + tok_local * (H + 4 * H // BLOCK) + pairs * I * 2
    g1_flops = 2 * H * 2 * I * pairs
    return flops, bytes_, g1_flops, g1_bytes


def gemm2_algorithmic(geom, pairs, active):
    """GEMM2 alone: W2 + S2 of active experts, bf16 C rows read once, one bf16 row written per
    pair (its output or partial row); 2*I*H FLOPs per pair."""
    H, I = geom.hidden, geom.intermediate
    w2 = H * I + 4 * (H // BLOCK) * (I // BLOCK)
    return 2 * I * H * pairs, active * w2 + pairs * I * 2 + pairs * H * 2


def settle_and_time(call, steps, warmup, settle_ms, dev):
    """W warm-up calls, then more calls until ``settle_ms`` of wall time has passed, then
    ``steps`` back-to-back calls between two events. Returns (ms per call, warm-up calls run)."""
    for _ in range(warmup):
        call()
    torch.cuda.synchronize(dev)
    n = warmup
    t0 = time.perf_counter()
    while (time.perf_counter() - t0) * 1e3 < settle_ms:
        for _ in range(4):
            call()
        n += 4
        torch.cuda.synchronize(dev)
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record()
    for _ in range(steps):
        call()
    end.record()
    torch.cuda.synchronize(dev)
    return start.elapsed_time(end) / steps, n


def time_calls(call, steps, warmup, dev):
    return settle_and_time(call, steps, warmup, 0.0, dev)[0]


def stage_times(call, reps, dev):
    """Average per-stage milliseconds from hipEvents the library records on its own stream."""
    import ctypes
    n = len(STAGES) + 1
    sets = [[torch.cuda.Event(enable_timing=True) for _ in range(n)] for _ in range(reps)]
    for evs in sets:  # torch creates the underlying hipEvent on first record
        for e in evs:
            e.record()
    torch.cuda.synchronize(dev)
    L = _lib.lib()
    tot = [0.0] * len(STAGES)
    try:
        # calls go back to back (no host sync in between), as in the timed loop
        for evs in sets:
            arr = (ctypes.c_void_p * n)(*[e.cuda_event for e in evs])
            _lib.check(L.moe_set_stage_events(arr, n), "moe_set_stage_events")
            call()
        torch.cuda.synchronize(dev)
    finally:
        L.moe_set_stage_events(None, 0)
    for evs in sets:
        for i in range(len(STAGES)):
            tot[i] += evs[i].elapsed_time(evs[i + 1])
    return {s: tot[i] / reps for i, s in enumerate(STAGES)}


def roofline_block(stage, kernel, ms, flops, nbytes, peak_tflops, workload):
    """Roofline of one kernel: bound by whichever of FLOPs / peak and bytes / HBM peak is
    larger; ``achieved`` is the algorithmic rate over the kernel's average launch time."""
    t_mfma = flops / (peak_tflops * 1e12)
    t_hbm = nbytes / (PEAK_HBM_GBS * 1e9)
    if t_mfma >= t_hbm:
        bound, achieved, peak, unit = "mfma", flops / (ms * 1e-3) / 1e12, peak_tflops, "TFLOP/s"
    else:
        bound, achieved, peak, unit = "hbm", nbytes / (ms * 1e-3) / 1e9, PEAK_HBM_GBS, "GB/s"
    blk = {"bound": bound, "kernel": kernel, "stage": stage, "achieved": achieved, "peak": peak,
           "unit": unit, "frac": achieved / peak, "traffic": load_traffic(stage, workload),
           "algorithmic_bytes": nbytes, "algorithmic_flops": flops, "avg_launch_ms": ms}
    # The same figure from the committed rocprofv3 kernel trace of this bench (its average
    # duration for this kernel and workload), so the event-timed frac can be checked against it.
    us = load_rocprof_avg_us(kernel, workload)
    if us is not None:
        r_ms = us * 1e-3
        blk["rocprof_avg_launch_ms"] = r_ms
        blk["frac_rocprof"] = ((flops / (r_ms * 1e-3) / 1e12) if bound == "mfma"
                               else (nbytes / (r_ms * 1e-3) / 1e9)) / peak
    return blk


def measure(cfg, weight_sets, steps, warmup, settle_ms, dev, seed=None):
    """Times one workload. With several weight sets (distinct layers' weights), consecutive
    calls cycle through them, so no call finds the previous call's weights in a cache."""
    geom = cfg.geom
    seed = cfg.seed if seed is None else seed
    act = jin.make_activations(geom, cfg.tokens, seed=seed, device=dev,
                               skew_experts=cfg.skew_experts, skew_offset=cfg.skew_offset)
    calls = []
    for w13, s13, w2, s2 in weight_sets:
        kw = dict(act, gemm1_weights=w13, gemm1_weights_scale=s13, gemm2_weights=w2,
                  gemm2_weights_scale=s2, local_expert_offset=0,
                  routed_scaling_factor=2.5 if geom.routing_method == 0 else 1.0)
        calls.append(bind(**kw, geometry=geom))
    kw = dict(kw, gemm1_weights=weight_sets[0][0], gemm1_weights_scale=weight_sets[0][1],
              gemm2_weights=weight_sets[0][2], gemm2_weights_scale=weight_sets[0][3])
    call = calls[0]
    if len(calls) == 1:
        timed = call
    else:
        state = [0]

        def timed():
            state[0] = (state[0] + 1) % len(calls)
            return calls[state[0]]()
    ms, n_warm = settle_and_time(timed, steps, warmup, settle_ms, dev)
    st = stage_times(timed, min(steps, 20), dev)
    pairs, active, tok_local = routing_stats(geom, cfg.tokens, call.workspace)
    if pairs == 0:
        raise RuntimeError(f"{cfg.name}: no routed pairs read back from the call's workspace")
    flops, bytes_, g1_flops, g1_bytes = algorithmic(geom, cfg.tokens, pairs, active, tok_local)
    g2_flops, g2_bytes = gemm2_algorithmic(geom, pairs, active)
    tflops = flops / (ms * 1e-3) / 1e12
    gbs = bytes_ / (ms * 1e-3) / 1e9
    t_floor_ms = max(flops / (PEAK_FP8_TFLOPS * 1e12), bytes_ / (PEAK_HBM_GBS * 1e9)) * 1e3
    g1 = roofline_block("gemm1_swiglu", gemm1_kernel_name(cfg), st["gemm1_swiglu"], g1_flops,
                        g1_bytes, PEAK_FP8_TFLOPS, cfg.name)
    g2 = roofline_block("gemm2", gemm2_launch_name(cfg), st["gemm2"], g2_flops, g2_bytes,
                        PEAK_BF16_TFLOPS, cfg.name)
    res = dict(workload=cfg.name, geometry=geom.name, tokens=cfg.tokens, seed=seed,
               ms_per_call=ms, steps=steps, warmup_calls=n_warm, weight_sets=len(calls),
               tflops=tflops, gb_s=gbs,
               pairs=pairs, active_experts=active, algorithmic_flops=flops,
               algorithmic_bytes=bytes_, call_floor_ms=t_floor_ms,
               call_floor_frac=t_floor_ms / ms, hbm_frac=gbs / PEAK_HBM_GBS,
               fp8_mfma_frac=tflops / PEAK_FP8_TFLOPS, stage_ms=st,
               roofline=g1 if st["gemm1_swiglu"] >= st["gemm2"] else g2,
               kernels={"gemm1_swiglu": g1, "gemm2": g2})
    return res, kw


QUANT_GRAPH_CALLS = 20


def measure_quant(T, H, steps, warmup, dev):
    """The activation-quantisation kernel on a bf16 [T, H] batch already in HBM: algorithmic bytes
    = bf16 read + e4m3 write + fp32 scales (2 + 1 + 4/128 bytes per element)."""
    from justgoal_amd.moe import quantize_activations
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(2)).bfloat16().to(dev)
    q = torch.empty((T, H), dtype=torch.float8_e4m3fn, device=dev)
    sc = torch.empty((H // BLOCK, T), dtype=torch.float32, device=dev)
    call = lambda: quantize_activations(x, q, sc)
    # Eager calls from Python: at small T the host's per-call overhead (argument checks, ctypes)
    # is longer than the kernel, so the GPU waits on the host.
    host_ms = time_calls(call, steps, warmup, dev)
    # The kernel as a pipeline sees it: QUANT_GRAPH_CALLS launches captured in one HIP graph
    # and replayed, so the time per launch excludes the host.
    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream(dev).wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(QUANT_GRAPH_CALLS):
            call()
    ms = time_calls(graph.replay, max(5, steps // QUANT_GRAPH_CALLS), 2, dev) / QUANT_GRAPH_CALLS
    nbytes = T * H * 3 + T * (H // BLOCK) * 4
    gbs = nbytes / (ms * 1e-3) / 1e9
    return dict(tokens=T, hidden=H, ms_per_call=ms, bytes=nbytes, gb_s=gbs,
                hbm_frac=gbs / PEAK_HBM_GBS, host_call_ms=host_ms,
                timing=f"per launch in a replayed HIP graph of {QUANT_GRAPH_CALLS} launches; "
                       "host_call_ms: eager Python calls")


def _rows_hint(cfg):
    g = cfg.geom
    return cfg.tokens * g.top_k // g.num_experts


def gemm1_kernel_name(cfg):
    """The GEMM1+SwiGLU kernel family the library picks for this shape: the shape-only rule of
    justgoal_amd/csrc/moe_gemm.hip (expected pairs per expert T*top_k/E: <= GEMM1_STREAM_MAX_ROWS
    streaming, >= GEMM1_BIG_ROWS large tiles, else LDS tiles)."""
    rows = _rows_hint(cfg)
    return ("gemm1_stream_kernel" if rows <= GEMM1_STREAM_MAX_ROWS else
            "gemm1_tile_kernel" if rows < GEMM1_BIG_ROWS else "gemm1_big_kernel")


def gemm2_kernel_name(cfg):
    """GEMM2: LDS-tiled up to GEMM2_TILE_MAX_ROWS expected pairs per expert; above, 256-column
    tiles from GEMM2_BIG_TILE_ROWS, or where the experts' tiles fill the chip
    GEMM2_WIDE_MIN_ROUNDS times; else large tiles (every bench geometry has I >= 384)."""
    rows, g = _rows_hint(cfg), cfg.geom
    if rows <= GEMM2_TILE_MAX_ROWS:
        return "gemm2_tile_kernel"
    tiles = g.local_experts * -(-g.hidden // 256)
    wide = rows >= GEMM2_BIG_TILE_ROWS or tiles >= GEMM2_WIDE_MIN_ROUNDS * CUS
    return "gemm2_wide_kernel" if wide else "gemm2_big_kernel"


def gemm2_launch_name(cfg):
    """The kernel of the GEMM2 stage: that of gemm2_kernel_name, except for a few tokens, whose
    GEMM2 and combine are one launch (GEMM2_TOKEN_MAX_ROWS tokens and GEMM2_TOKEN_MAX_PAIRS expected
    local pairs at most; the rule of justgoal_amd/csrc/moe_stream.hip). Its combine stage is
    empty."""
    g = cfg.geom
    cols = -(-g.hidden // (4 * CUS)) * 4
    pairs = cfg.tokens * g.top_k * g.local_experts // g.num_experts
    few = (cfg.tokens <= GEMM2_TOKEN_MAX_ROWS and pairs <= GEMM2_TOKEN_MAX_PAIRS and
           GEMM2_TOKEN_MIN_COLS <= cols <= 32 and g.intermediate in (1024, 1536, 2048))
    return "gemm2_token_kernel" if few else gemm2_kernel_name(cfg)


def load_traffic(stage, name):
    """HBM bytes per launch measured by rocprofv3 --pmc (committed under profiles/), if present."""
    p = os.path.join(HERE, "profiles", f"traffic_{stage}_{name}.json")
    if not os.path.exists(p):
        return None
    with open(p) as f:
        return json.load(f).get("bytes_per_launch")


def load_rocprof_avg_us(kernel, name):
    """Average duration (us) of ``kernel`` in ``name``'s calls in the committed rocprofv3
    --kernel-trace summary of this bench, if present."""
    p = os.path.join(HERE, "profiles", "kernel_avg_us.json")
    if not os.path.exists(p):
        return None
    with open(p) as f:
        ent = json.load(f).get("workloads", {}).get(name, {}).get(kernel)
    return None if ent is None else ent["average_us"]


# CPU-baseline repetitions per workload: median of 3 (one warm-up call first for the small
# batches), and a single call for the skewed T=16384 batch (about 5 s per oracle call on the GPU
# host's 16 threads, minutes on a few cores). The six baselines add ~25 s to a default run.
CPU_BASELINE_REPS = {"ds_t16384_skew": (1, 0)}
CPU_BASELINE_DEFAULT = (3, 1)
CPU_BASELINE_BIG = (3, 0)  # batches whose oracle call takes seconds: no separate warm-up


def cpu_baseline(cfg, kw_dev, cpu_weights, flops):
    """The CPU oracle (torch-CPU fp32 dequantise-then-matmul restatement of the operator) on all
    of this host's cores, on the full workload with the same inputs as the GPU run (weight set 0,
    already on the host). Returns the bench line's ``cpu_baseline`` object."""
    import oracle
    cores = max(1, os.cpu_count() or 1)
    torch.set_num_threads(cores)
    kw = {k: (v.cpu() if isinstance(v, torch.Tensor) else v) for k, v in kw_dev.items()}
    kw.update(gemm1_weights=cpu_weights[0], gemm1_weights_scale=cpu_weights[1],
              gemm2_weights=cpu_weights[2], gemm2_weights_scale=cpu_weights[3])
    geom = cfg.geom
    reps, warm = CPU_BASELINE_REPS.get(
        cfg.name, CPU_BASELINE_BIG if cfg.tokens >= 4096 or geom.local_experts > 32
        else CPU_BASELINE_DEFAULT)
    for _ in range(warm):
        oracle.moe_reference(kw, geom)
    ts = []
    for _ in range(reps):
        t0 = time.perf_counter()
        oracle.moe_reference(kw, geom)
        ts.append(time.perf_counter() - t0)
    ts.sort()
    sec = ts[len(ts) // 2]
    what = f"median of {reps}" if reps > 1 else "one call"
    if warm:
        what += f" after {warm} warm-up"
    return {"value": flops / sec / 1e12, "unit": "TFLOPS", "cores": torch.get_num_threads(),
            "kind": "port", "ms_per_call": sec * 1e3,
            "sample": f"full {cfg.name} call (T={cfg.tokens}), {what}, torch-CPU fp32 "
                      "dequantise-then-matmul oracle, weight set 0"}


DEFAULT_WORKLOADS = ("ds_t16", "ds_t64", "ds_t1024", "ds_t4096", "ds_t16384_skew", "qwen3_t1024")


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--settle-ms", type=float, default=300.0,
                    help="wall time of calls after the warm-up calls, before timing")
    ap.add_argument("--config", default="ds_t64", choices=sorted(jin.CONFIGS),
                    help="headline workload (value, ms_per_step)")
    ap.add_argument("--workloads", default=",".join(DEFAULT_WORKLOADS),
                    help="comma-separated workloads to measure (the headline is always included)")
    ap.add_argument("--weight-sets", type=int, default=3,
                    help="distinct weight sets that consecutive calls cycle through (consecutive "
                         "MoE layers have different weights; with 1 set, repeated calls of a "
                         "small batch partly hit the previous call's weights in the 256 MB MALL)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-quant", action="store_true")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="only run 5 device-to-device copies of 1 GiB (reference kernel for "
                         "scaling rocprofv3 FETCH_SIZE / WRITE_SIZE readings) and exit")
    args = ap.parse_args()
    if args.copy_calibration:
        src = torch.ones(1 << 30, dtype=torch.uint8, device="cuda:0")
        dst = torch.empty_like(src)
        for _ in range(5):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"copy_bytes": 1 << 30, "copies": 5}))
        return
    if args.gpus != 1:
        print("bench.py measures one GPU only: this build runs the operator on a single MI355X "
              "(expert-parallel sharding across GPUs is a design note, not built); use --gpus 1.",
              file=sys.stderr)
        sys.exit(2)
    if not torch.cuda.is_available():
        print("bench.py needs a GPU", file=sys.stderr)
        sys.exit(2)
    steps = max(20, args.steps)
    dev = torch.device("cuda:0")
    _lib.lib()
    head_cfg = jin.CONFIGS[args.config]
    names = [n for n in args.workloads.split(",") if n]
    if args.config not in names:
        names.insert(0, args.config)
    results, head = {}, None
    weights = {}
    # group by geometry so each weight set is generated and resident once
    for geom in dict.fromkeys(jin.CONFIGS[n].geom for n in names):
        t0 = time.time()
        log(f"[bench] generating {geom.name} weights")
        wts_cpu = [jin.make_weights(geom, seed=k) for k in range(args.weight_sets)]
        wts = [tuple(t.to(dev) for t in w) for w in wts_cpu]
        cpu_w0 = wts_cpu[0]
        del wts_cpu
        log(f"[bench] weights ready in {time.time() - t0:.1f}s")
        for n in names:
            cfg = jin.CONFIGS[n]
            if cfg.geom != geom:
                continue
            r, kw = measure(cfg, wts, steps, args.warmup, args.settle_ms, dev)
            rl = r["roofline"]
            log(f"[bench] {n}: {r['ms_per_call']:.4f} ms ({r['warmup_calls']} warm-up calls), "
                f"{r['tflops']:.1f} TFLOPS, {r['gb_s']:.0f} GB/s, floor frac "
                f"{r['call_floor_frac']:.3f}; {rl['kernel']} {rl['frac']:.3f} of {rl['bound']}; "
                f"stages " + ", ".join(f"{k} {v * 1e3:.1f}us" for k, v in r["stage_ms"].items()))
            if not args.no_cpu_baseline:
                t1 = time.time()
                r["cpu_baseline"] = cpu_baseline(cfg, kw, cpu_w0, r["algorithmic_flops"])
                r["gpu_speedup_vs_cpu"] = r["cpu_baseline"]["ms_per_call"] / r["ms_per_call"]
                log(f"[bench] {n}: CPU oracle {r['cpu_baseline']['ms_per_call']:.1f} ms/call on "
                    f"{r['cpu_baseline']['cores']} threads ({time.time() - t1:.0f}s)")
            results[n] = r
            if n == args.config:
                head = r
            del kw
        del wts, cpu_w0
        torch.cuda.empty_cache()
    quant = [] if args.no_quant else [
        measure_quant(T, head_cfg.geom.hidden, steps, args.warmup, dev) for T in (4096, 64)]
    for r in quant:
        log(f"[bench] activation quant T={r['tokens']}: {r['ms_per_call'] * 1e3:.1f} us, "
            f"{r['gb_s']:.0f} GB/s (graph-replayed; eager Python call {r['host_call_ms'] * 1e3:.1f} us)")
    cpu = head.get("cpu_baseline")
    out = {
        "metric": METRIC, "value": head["tflops"], "unit": "TFLOPS", "n_gpus": 1,
        "steps": steps, "warmup": args.warmup, "ms_per_step": head["ms_per_call"],
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "fp8-e4m3 (GEMM1) / bf16 (GEMM2), fp32 accumulate",
        "data": f"synthetic (seed {head_cfg.seed}: N(0,1) activations/logits, N(0,0.1) bias, "
                f"N(0,0.02) weights, 128x128 block scales; {args.weight_sets} weight sets "
                "cycled call to call)",
        "config": {"workload": head_cfg.name, "geometry": head_cfg.geom.name,
                   "tokens": head_cfg.tokens, "seed": head_cfg.seed,
                   "local_pairs": head["pairs"], "active_local_experts": head["active_experts"],
                   "hidden": head_cfg.geom.hidden, "intermediate": head_cfg.geom.intermediate,
                   "local_experts": head_cfg.geom.local_experts, "top_k": head_cfg.geom.top_k,
                   "parallelism": "single GPU (EP rank 0 of 8: local experts 0..31)",
                   "settle_ms": args.settle_ms, "weight_sets": args.weight_sets},
        "roofline": head["roofline"],
        "cpu_baseline": cpu,
        "headline": head,
        "workloads": {n: r for n, r in results.items() if n != args.config},
        "activation_quant": quant,
    }
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
