"""TileMix fused attention benchmark on one MI355X.

Default workload: BASELINE config 3 (the headline): B=4 H=16 S=4096 D=128,
causal, 128x64 routing tiles (above-diagonal tiles skipped, the 8 key tiles
nearest the diagonal FP16, the rest INT8 with p=0.5), inputs N(0,1) fp16.

One step = the whole TileMix job on inputs already resident in HBM:
  1. tilemix_quantize_qk_batched on K (64-row blocks -> K8 + k_scales), then
  2. tilemix_attention_batched with quantize=2 (each workgroup quantizes its own
     128-row Q block in registers, routes every 16x32 cell to INT8 or FP16 MFMA
     or skip, online softmax, P.V on FP16 MFMA, fp32 O).
``value`` = effective TFLOP/s of the step: algorithmic ops counted from the
drawn mask (QK^T 2D per visible pair as INT8 or FP16 by route, P.V 2D FP16)
over the wall time of K steps. ``roofline`` covers the attention kernel alone:
its average duration from HIP events on its stream, against the blended
INT8/FP16 MFMA peak of the same op mix. ``cpu_baseline`` times the CPU PyTorch
restatement of the reference's CPU path (python/reference_attention.py) on a
bounded sample of heads on this host's cores.

Warm-up: the W requested steps, then more untimed steps until at least
--min-warmup-ms of wall time has passed since warm-up began. An MI355X
raises its clock over the first tens of milliseconds of sustained work (the
headline attention launch goes from about 0.39 ms to 0.31 ms after roughly
50 ms), so a few steps alone would time the ramp rather than the sustained
rate. The JSON line reports W as requested and the steps actually run; the
timed region is exactly K steps either way.

After the timed steps, the card's `pp_dpm_sclk` sysfs file is read while more untimed
steps run (``roofline.sclk_mhz_sampled``; plain file reads, no child process). Reading
the clock level slows the following launches for a while, so the sample never precedes
the timed region. The MFMA peaks are quoted at 2.4 GHz; with N(0,1) operands the card
holds a lower clock under its power limit (``--input-scale 0`` shows the same kernel at
2.4 GHz).

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--min-warmup-ms T] [--config 3]
                       [--precise] [--no-check] [--no-cpu-baseline] [--no-clock]
                       [--input-scale F] [--routing] [--per-head demo|config]
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT / "tilemix-cuda_amd"))

PEAK_FP16_TFLOPS = 2516.6   # MI355X dense FP16 MFMA (256 CU x 2.4 GHz x 4096 flop/clk)
PEAK_INT8_TOPS = 5033.2     # MI355X dense INT8 MFMA
PEAK_HBM_GBS = 8000.0


def parse_args():
    p = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=20)
    p.add_argument("--warmup", type=int, default=5)
    p.add_argument("--min-warmup-ms", type=float, default=150.0,
                   help="keep running untimed steps after the W warm-up steps until this much wall "
                        "time has passed since warm-up began (0 disables)")
    p.add_argument("--config", type=int, default=3, choices=[1, 2, 3, 4, 5])
    p.add_argument("--seed", type=int, default=20261201)
    p.add_argument("--precise", action="store_true", help="split-precision P.V (fp32-level accuracy)")
    p.add_argument("--no-check", action="store_true", help="skip the parity check against the oracle")
    p.add_argument("--no-cpu-baseline", action="store_true")
    p.add_argument("--cpu-budget", type=float, default=12.0, help="seconds of CPU-baseline work")
    p.add_argument("--check-rows", type=int, default=4096)
    p.add_argument("--copy-probe-mib", type=int, default=0,
                   help="after timing, run one device copy of this many MiB on the bench stream "
                        "(calibrates rocprofv3 FETCH_SIZE/WRITE_SIZE against known bytes)")
    p.add_argument("--no-clock", action="store_true",
                   help="skip the sysfs shader-clock sample taken after the timed steps")
    p.add_argument("--input-scale", type=float, default=1.0,
                   help="diagnostic: multiply Q, K and V by this factor after the routing codes are "
                        "drawn from the unscaled inputs (same routes, same INT8 codes, smaller "
                        "operands); used to show how the sustained clock depends on the data")
    p.add_argument("--routing", action="store_true",
                   help="time the device routing producer for --config's router instead (tile codes, "
                        "then route / skip words), with HBM rates against the algorithmic bytes")
    p.add_argument("--per-head", choices=["demo", "config"], default=None,
                   help="time the drop-in per-head API (launch_fused_fp16_attention, precise P.V) instead: "
                        "'demo' = the reference demo workload (M=1000 N=1003 d=128, g=2, mask 0xaaaa...), "
                        "'config' = a loop of per-head calls over --config's heads (no causal mask or "
                        "skip in that API: every pair is computed, skipped cells as FP16)")
    return p.parse_args()


def log(msg: str) -> None:
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def main() -> int:
    args = parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print(json.dumps({"error": "this build runs on one GPU only: the TileMix path would shard "
                          "across GPUs by head with no exchange between them, but multi-GPU runs are "
                          "not part of this build; run with --gpus 1"}))
        return 2

    import torch
    import tilemix
    from tilemix import workloads

    if not torch.cuda.is_available():
        print(json.dumps({"error": "no GPU visible"}))
        return 1
    torch.cuda.set_device(0)
    if args.per_head:
        print(json.dumps(per_head_bench(args)), flush=True)
        return 0
    if args.routing:
        print(json.dumps(routing_bench(args)), flush=True)
        return 0
    w = workloads.WORKLOADS[args.config]
    log(w.describe())
    Q, K, V = workloads.make_inputs(w, args.seed)
    codes = workloads.make_codes(w, args.seed, Q, K)
    if args.input_scale != 1.0:
        Q, K, V = ((x.float() * args.input_scale).to(torch.float16) for x in (Q, K, V))
        log(f"inputs scaled by {args.input_scale:g} (routing codes from the unscaled inputs)")
    route_np, skip_np = workloads.pack_heads(codes, w.key_tiles_per_group)
    work = workloads.work(w, codes)
    heads, S, D = w.heads, w.S, w.D
    dev = "cuda:0"
    route_words = torch.from_numpy(route_np.view(np.int64)).to(dev)
    skip_words = torch.from_numpy(skip_np.view(np.int64)).to(dev) if skip_np is not None else None
    O = torch.empty((heads, S, D), dtype=torch.float32, device=dev)
    K8 = torch.empty((heads, S, D), dtype=torch.int8, device=dev)
    k_scales = torch.empty((heads, (S + 63) // 64), dtype=torch.int16, device=dev)
    stream = torch.cuda.Stream()
    attn_args = tilemix.BatchedArgs(Q=Q, K=K, V=V, O=O, heads=heads, M=S, N=S, d=D,
                                    score_scale=w.score_scale, causal=w.causal, precise=args.precise,
                                    quantize=2, route_words=route_words, skip_words=skip_words,
                                    key_tiles_per_group=w.key_tiles_per_group, K8=K8, k_scales=k_scales)

    def step(events=None):
        tilemix.check(tilemix.quantize_tilemix_qk_batched(None, K, None, K8, None, k_scales, heads, S, S, D,
                                                          stream=stream), "quantize K")
        if events is not None:
            events[0].record(stream)
        tilemix.check(tilemix.attention_batched(attn_args, stream), "attention")
        if events is not None:
            events[1].record(stream)

    with torch.cuda.stream(stream):
        warm_start = time.perf_counter()
        for _ in range(args.warmup):
            step()
        torch.cuda.synchronize()
        warmup_run = args.warmup
        while (time.perf_counter() - warm_start) * 1e3 < args.min_warmup_ms and warmup_run < 100000:
            for _ in range(8):
                step()
            warmup_run += 8
            torch.cuda.synchronize()
        warmup_ms = (time.perf_counter() - warm_start) * 1e3
        log(f"warm-up: {warmup_run} steps in {warmup_ms:.1f} ms ({args.warmup} requested, "
            f"minimum {args.min_warmup_ms:g} ms)")
        pairs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
                 for _ in range(args.steps)]
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for k in range(args.steps):
            step(pairs[k])
        torch.cuda.synchronize()
        t1 = time.perf_counter()
        # The shader clock under sustained load, sampled while more untimed steps run after
        # the timed ones: reading the clock level slows the kernel for a while (measured: the
        # next 20 steps about 20 % slower), so it never precedes the timed region.
        sclk = None
        if not args.no_clock:
            sclk, sample_steps = sample_sclk_mhz(step, torch.cuda.synchronize)
            log(f"sampled shader clock: {sclk} MHz ({sample_steps} untimed steps after the timed ones)")
        if args.copy_probe_mib > 0:
            src = torch.ones(args.copy_probe_mib << 19, dtype=torch.float16, device=dev)
            dst = torch.empty_like(src)
            torch.cuda.synchronize()
            dst.copy_(src)
            torch.cuda.synchronize()
            log(f"copy probe: {args.copy_probe_mib} MiB read + {args.copy_probe_mib} MiB written")
            del src, dst
    ms_per_step = (t1 - t0) * 1e3 / args.steps
    attn_ms = float(np.mean([a.elapsed_time(b) for a, b in pairs]))
    log(f"step {ms_per_step:.4f} ms, attention kernel {attn_ms:.4f} ms (HIP events)")

    ops_total = work["ops_int8"] + work["flops_fp16"]
    t_min = work["ops_int8"] / (PEAK_INT8_TOPS * 1e12) + work["flops_fp16"] / (PEAK_FP16_TFLOPS * 1e12)
    blended_peak = ops_total / t_min / 1e12
    achieved = ops_total / (attn_ms * 1e-3) / 1e12
    value = ops_total / (ms_per_step * 1e-3) / 1e12

    result = {
        "metric": "effective TFLOP/s & % MFMA peak, TileMix attn B=4 H=16 S=4096 D=128",
        "value": round(value, 3),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "warmup_steps_run": warmup_run,
        "warmup_ms": round(warmup_ms, 1),
        "ms_per_step": round(ms_per_step, 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "i8+f16 (i32/f32 accumulate)",
        "data": "synthetic (seeded torch N(0,1)/outlier/Student-t fp16; seeded numpy routing masks)",
        "config": {
            "workload": w.describe(),
            "B": w.B, "H": w.H, "S": S, "D": D, "causal": w.causal,
            "key_tiles_per_group": w.key_tiles_per_group,
            "precise_pv": bool(args.precise),
            "visible_pairs_int8": work["pairs_int8"], "visible_pairs_fp16": work["pairs_fp16"],
            "ops_int8": work["ops_int8"], "flops_fp16": work["flops_fp16"],
            "step": "K pre-pass quantizer + attention (Q quantized in-kernel)",
        },
        "roofline": {
            "bound": "mfma",
            "kernel": attention_kernel_name(w, args.precise),
            "achieved": round(achieved, 3),
            "peak": round(blended_peak, 3),
            "unit": "TFLOP/s",
            "frac": round(achieved / blended_peak, 4),
            "traffic": None,
            "kernel_ms": round(attn_ms, 5),
            "achieved_hbm_gbs": None,
            "peak_basis": "blended: ops_int8/5033.2T + flops_fp16/2516.6T",
            "sclk_mhz_sampled": sclk,
            "sclk_mhz_peak_basis": 2400,
            # frac against the peaks scaled to the sampled clock: how close the kernel runs to
            # what the card delivers at the clock it holds under this load (frac itself stays
            # against the 2.4 GHz peaks)
            "frac_at_sampled_sclk": round(achieved / blended_peak * 2400.0 / sclk, 4) if sclk else None,
        },
    }
    if args.input_scale != 1.0:
        result["data"] += f"; Q, K, V scaled by {args.input_scale:g} after routing (diagnostic run)"

    measured = measured_traffic(w.describe())
    if measured is not None and "stale" in measured:
        result["roofline"]["traffic_stale"] = measured["stale"]
    elif measured is not None:
        result["roofline"]["traffic"] = measured["traffic_bytes"]
        result["roofline"]["achieved_hbm_gbs"] = round(measured["traffic_bytes"] / (attn_ms * 1e-3) / 1e9, 1)
        result["roofline"]["traffic_source"] = measured["source"]

    if not args.no_check:
        result["parity"] = parity_check(w, Q, K, V, O, K8, k_scales, codes, args)
        log(f"parity: {result['parity']}")

    if not args.no_cpu_baseline:
        result["cpu_baseline"] = cpu_baseline(w, Q, K, V, codes, args.cpu_budget)
        log(f"cpu baseline: {result['cpu_baseline']}")

    print(json.dumps(result), flush=True)
    return 0


def routing_bench(args) -> dict:
    """The device routing producer on --config's shape: stage 1 writes one code per tile
    (tilemix_tiles_bernoulli / _causal_band / _three_way, or the importance router, which
    reads all of Q and K for its tile maxima), stage 2 packs the codes into TileMixRouting
    words (tilemix_routes_from_tiles). Each stage is timed with HIP events over --steps
    calls after the clock warm-up; bytes are the algorithmic ones (inputs read once, codes
    and words written once). For the importance router the device codes are compared with
    the host router over the same data."""
    import torch
    import tilemix
    from tilemix import routing, workloads

    w = workloads.WORKLOADS[args.config]
    heads, S, D, g = w.heads, w.S, w.D, w.key_tiles_per_group
    tr, tk = (128, 64) if w.router in ("causal_band", "importance") else (64, 64)
    tq, tkk = (S + tr - 1) // tr, (S + tk - 1) // tk
    dev = "cuda:0"
    codes = torch.empty((heads, tq, tkk), dtype=torch.uint8, device=dev)
    words = tilemix.routing_word_count(S, S, g)
    route = torch.empty(heads * words, dtype=torch.int64, device=dev)
    skip = torch.empty_like(route)
    stream = torch.cuda.Stream()
    seed = args.seed
    if w.router == "importance":
        Q, K, _ = workloads.make_inputs(w, args.seed)
        need = tilemix.importance_workspace_bytes(heads, S, S, tr, tk)
        workspace = torch.empty(max(need // 4, 1), dtype=torch.float32, device=dev)
        stage1_bytes = 2 * heads * S * D * 2 + codes.numel()

        def stage1():
            tilemix.check(tilemix.tiles_importance(Q, K, heads, S, S, D, tr, tk, 0.25, workspace, need, codes,
                                                   stream=stream), "importance")
    else:
        stage1_bytes = codes.numel()

        def stage1():
            if w.router == "bernoulli":
                rc = tilemix.tiles_bernoulli(codes, heads, S, S, tr, tk, 0.5, seed, stream=stream)
            elif w.router == "causal_band":
                rc = tilemix.tiles_causal_band(codes, heads, S, tr, tk, 8, 0.5, seed, stream=stream)
            else:
                rc = tilemix.tiles_three_way(codes, heads, S, S, tr, tk, 0.3, 0.4, seed, stream=stream)
            tilemix.check(rc, w.router)

    def stage2():
        tilemix.check(tilemix.routes_from_tiles(codes, heads, S, S, tr, tk, g, route, skip, stream=stream), "pack")

    stage2_bytes = codes.numel() + 2 * route.numel() * 8

    def timed(fn):
        with torch.cuda.stream(stream):
            start = time.perf_counter()
            while (time.perf_counter() - start) * 1e3 < args.min_warmup_ms:
                for _ in range(8):
                    fn()
                torch.cuda.synchronize()
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record(stream)
            for _ in range(args.steps):
                fn()
            e1.record(stream)
            torch.cuda.synchronize()
        return e0.elapsed_time(e1) / args.steps

    stages = []
    for name, fn, nbytes in ((f"tile codes ({w.router})", stage1, stage1_bytes),
                             ("routes_from_tiles", stage2, stage2_bytes)):
        ms = timed(fn)
        gbs = nbytes / (ms * 1e-3) / 1e9
        stages.append({"stage": name, "ms": round(ms, 5), "bytes": int(nbytes), "gbs": round(gbs, 1),
                       "frac_hbm": round(gbs / PEAK_HBM_GBS, 4)})
    result = {"metric": "device routing producer, per call", "config": {"workload": w.describe(),
              "tile": [tr, tk], "key_tiles_per_group": g, "tiles_per_head": tq * tkk}, "steps": args.steps,
              "stages": stages}
    if w.router == "importance":
        got = codes.cpu().numpy()
        q_amax = Q.view(heads, tq, tr * D).abs().amax(-1).float().cpu().numpy()
        k_amax = K.view(heads, tkk, tk * D).abs().amax(-1).float().cpu().numpy()
        match = all(np.array_equal(got[h], routing.importance_top_fraction(
            q_amax[h], k_amax[h], S, S, D, tr, tk, 0.25)[:: tr // 16, :: tk // 32][:tq, :tkk]) for h in range(heads))
        result["codes_equal_host_router"] = bool(match)
    return result


def per_head_bench(args) -> dict:
    """The reference's own call pattern (src/main.cu:55-58, src/tests/tilemix_test.cu:487-500):
    quantize_tilemix_qk, then launch_fused_fp16_attention with a TileMixRouting mask, one head
    per call, precise (split fp16) P.V. Timed with HIP events over `steps` rounds on one
    stream; a round is one quantize + one attention call per head."""
    import torch
    import tilemix
    from tilemix import routing, workloads

    dev = "cuda:0"
    if args.per_head == "demo":
        # src/main.cu:22-58: M=1000, N=1003, d=128, key_tiles_per_group 2, every routing word
        # 0xaaaa... (odd 64-key groups INT8, even ones FP16), inputs periodic in the index.
        M, N, d, g, heads = 1000, 1003, 128, 2, 1
        # The demo's periodic inputs (periods 17, 19, 23; src/main.cu:38-40).
        idx = torch.arange(max(M, N) * d, dtype=torch.int64)
        Q = (0.125 * ((idx[: M * d] % 17) - 8).float()).to(torch.float16).reshape(1, M, d).to(dev)
        K = (0.125 * ((idx[: N * d] % 19) - 9).float()).to(torch.float16).reshape(1, N, d).to(dev)
        V = (0.1 * ((idx[: N * d] % 23) - 11).float()).to(torch.float16).reshape(1, N, d).to(dev)
        words = np.full(tilemix.routing_word_count(M, N, g), 0xAAAAAAAAAAAAAAAA, dtype=np.uint64)
        route = torch.from_numpy(words.view(np.int64)).to(dev).reshape(1, -1)
        kt = np.arange((N + 31) // 32)
        codes = np.repeat(((kt // g) % 2 == 1).astype(np.uint8)[None, :], (M + 15) // 16, axis=0)[None]
        name, scale = "reference demo (src/main.cu): M=1000 N=1003 d=128, g=2, mask 0xaaaa...", 1.0 / np.sqrt(d)
        causal = False
    else:
        w = workloads.WORKLOADS[args.config]
        Q, K, V = workloads.make_inputs(w, args.seed)
        codes = workloads.make_codes(w, args.seed, Q, K)
        codes = np.where(codes == routing.SKIP, routing.FP16, codes).astype(np.uint8)
        route_np, _ = workloads.pack_heads(codes, w.key_tiles_per_group)
        heads, M, N, d, g = w.heads, w.S, w.S, w.D, w.key_tiles_per_group
        route = torch.from_numpy(route_np.view(np.int64)).to(dev).reshape(heads, -1)
        name = (f"per-head loop over {w.describe()} as {heads} calls of the per-head API "
                "(non-causal, skipped cells FP16)")
        scale, causal = w.score_scale, False
    O = torch.empty((heads, M, d), dtype=torch.float32, device=dev)
    Q8 = torch.empty((heads, M, d), dtype=torch.int8, device=dev)
    K8 = torch.empty((heads, N, d), dtype=torch.int8, device=dev)
    qs = torch.empty((heads, (M + 127) // 128), dtype=torch.int16, device=dev)
    ks = torch.empty((heads, (N + 63) // 64), dtype=torch.int16, device=dev)
    stream = torch.cuda.Stream()
    words_per_head = route.shape[1]

    def one_round():
        for h in range(heads):
            tilemix.check(tilemix.quantize_tilemix_qk(Q[h], K[h], Q8[h], K8[h], qs[h], ks[h], M, N, d, stream),
                          "quantize_tilemix_qk")
            tilemix.check(tilemix.launch_fused_fp16_attention(
                Q[h], K[h], V[h], O[h], M, N, d, float(scale), stream,
                tilemix.TileMixRouting(route[h], words_per_head, g),
                tilemix.TileMixQuantized(Q8[h], K8[h], qs[h], ks[h])), "launch_fused_fp16_attention")

    with torch.cuda.stream(stream):
        t0 = time.perf_counter()
        while (time.perf_counter() - t0) * 1e3 < args.min_warmup_ms:
            one_round()
            torch.cuda.synchronize()
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record(stream)
        for _ in range(args.steps):
            one_round()
        end.record(stream)
        torch.cuda.synchronize()
    ms_per_round = start.elapsed_time(end) / args.steps
    work = {"ops_int8": 0, "flops_fp16": 0}
    for h in range(codes.shape[0]):
        one = routing.algorithmic_work(codes[h], M, N, d, causal)
        work["ops_int8"] += one["ops_int8"]
        work["flops_fp16"] += one["flops_fp16"]
    ops_total = work["ops_int8"] + work["flops_fp16"]
    t_min = work["ops_int8"] / (PEAK_INT8_TOPS * 1e12) + work["flops_fp16"] / (PEAK_FP16_TFLOPS * 1e12)
    achieved = ops_total / (ms_per_round * 1e-3) / 1e12
    return {"metric": "per-head API effective TFLOP/s (quantize_tilemix_qk + launch_fused_fp16_attention)",
            "value": round(achieved, 3), "unit": "TFLOP/s", "n_gpus": 1, "steps": args.steps,
            "ms_per_round": round(ms_per_round, 5), "calls_per_round": 2 * heads,
            "higher_is_better": True, "dtype": "i8+f16 (i32/f32 accumulate), precise P.V",
            "config": {"workload": name, "heads": heads, "M": M, "N": N, "d": d, "key_tiles_per_group": g},
            "roofline": {"bound": "mfma", "achieved": round(achieved, 3),
                         "peak": round(ops_total / t_min / 1e12, 3), "unit": "TFLOP/s",
                         "frac": round(t_min / (ms_per_round * 1e-3), 4),
                         "note": "time per round includes the quantizer launches"}}


def attention_kernel_name(w, precise: bool) -> str:
    """The kernel that the library's launch rules (csrc/attention_rules.h) choose for the workload:
    the 128-row kernel for the tiny one and for precise P.V, else the 256-row kernel."""
    return "attention_kernel" if precise or w.index == 1 else "attention_wide_kernel"


# Sources whose change invalidates a recorded traffic measurement.
STAMPED_SOURCES = ["tilemix-cuda_amd/csrc/attention.hip", "tilemix-cuda_amd/csrc/attention_common.h",
                   "tilemix-cuda_amd/csrc/attention_rules.h",
                   "tilemix-cuda_amd/csrc/tilemix_device.h", "tilemix-cuda_amd/csrc/tilemix_launch.h",
                   "tilemix-cuda_amd/csrc/quantize.hip", "tilemix-cuda_amd/build.py"]


def source_stamp() -> str:
    """First 16 hex digits of a SHA-256 over the kernel sources and build flags."""
    import hashlib

    h = hashlib.sha256()
    for name in STAMPED_SOURCES:
        h.update(name.encode() + b"\0" + (ROOT / name).read_bytes() + b"\0")
    return h.hexdigest()[:16]


def parse_dpm_sclk(text: str) -> float | None:
    """The current shader clock in MHz from an amdgpu `pp_dpm_sclk` sysfs file: one line per
    clock level ("0: 500Mhz", "1: 2100Mhz *"), the level in use marked with '*'. None when no
    line is marked or the marked line carries no number."""
    for line in text.splitlines():
        if line.rstrip().endswith("*"):
            _, _, level = line.partition(":")
            digits = "".join(ch for ch in level if ch.isdigit() or ch == ".")
            return float(digits) if digits else None
    return None


def sclk_files(device: int = 0) -> list[Path]:
    """The `pp_dpm_sclk` file of torch device `device`, found through its PCI address; when the
    address is unknown, the only such file under /sys/class/drm (several cards: none)."""
    try:
        import torch

        props = torch.cuda.get_device_properties(device)
        pattern = f"{props.pci_domain_id:04x}:{props.pci_bus_id:02x}:{props.pci_device_id:02x}.*"
        found = sorted(Path("/sys/bus/pci/devices").glob(f"{pattern}/pp_dpm_sclk"))
        if found:
            return found[:1]
    except Exception:  # no torch device properties, no sysfs
        pass
    cards = sorted(Path("/sys/class/drm").glob("card*/device/pp_dpm_sclk"))
    return cards if len(cards) == 1 else []


def sample_sclk_mhz(step, sync, files: list[Path] | None = None, reads: int = 5) -> tuple[float | None, int]:
    """Shader clock (MHz) read from sysfs while bench steps keep the GPU busy, and the number of
    steps run meanwhile. The median of `reads` reads of the card's `pp_dpm_sclk` (plain file
    reads on a helper thread: this process starts no other program, which would be an exec
    from a process that has initialised the GPU), or None when the file is missing or
    unreadable. The MI355X holds its 2.4 GHz maximum only while it is under its power limit;
    with N(0,1) operands this kernel runs below it (zero operands: at it)."""
    import threading

    paths = sclk_files() if files is None else files
    readings: list[float] = []

    def read():
        for _ in range(reads):
            time.sleep(0.1)
            try:
                mhz = parse_dpm_sclk(paths[0].read_text())
            except (OSError, IndexError):
                return
            if mhz is not None:
                readings.append(mhz)

    reader = threading.Thread(target=read, daemon=True)
    reader.start()
    start = time.perf_counter()
    steps = 0
    while reader.is_alive() and time.perf_counter() - start < 5.0:
        for _ in range(8):
            step()
        steps += 8
        sync()
    reader.join(timeout=1.0)
    return (float(np.median(readings)) if readings else None), steps


def measured_traffic(workload: str):
    """HBM bytes per attention launch measured with rocprofv3 FETCH_SIZE/WRITE_SIZE
    (calibrated on a copy of known size) for this workload, if recorded for the
    sources being run; {"stale": ...} when it was measured on other sources."""
    path = ROOT / "profiles" / "traffic.json"
    if not path.exists():
        return None
    entries = json.loads(path.read_text()).get("attention") or []
    entry = next((e for e in entries if e.get("workload") == workload), None)
    if entry is None:
        return None
    current = source_stamp()
    if entry.get("source_stamp") != current:
        return {"stale": f"profiled sources {entry.get('source_stamp')} differ from these sources {current}; "
                         "re-run the FETCH_SIZE / WRITE_SIZE passes"}
    return entry


def parity_check(w, Q, K, V, O, K8, k_scales, codes, args) -> dict:
    """K8/k_scales bit-exact vs the oracle quantizer (all heads); O vs the fp64
    oracle on a seeded sample of (head, row) pairs: max-abs <= 2e-3, mean-abs <= 2e-4."""
    import torch
    sys.path.insert(0, str(ROOT))
    import oracle

    oracle.build()
    heads, S, D = w.heads, w.S, w.D
    to_bits = lambda t: t.detach().cpu().view(torch.int16).numpy().view(np.uint16)
    q_all, k_all, v_all = to_bits(Q), to_bits(K), to_bits(V)
    k8_all = K8.cpu().numpy()
    ks_all = k_scales.cpu().numpy().view(np.uint16)
    o_all = O.cpu().numpy()
    rng = np.random.default_rng(args.seed + 7)
    sample_heads = sorted(set(rng.choice(heads, size=min(heads, 4), replace=False).tolist()))
    rows_per_head = max(1, args.check_rows // len(sample_heads))
    k8_exact = True
    max_abs, sum_abs, count = 0.0, 0.0, 0
    for h in range(heads):
        k8_ref, ks_ref = oracle.quantize(k_all[h], 64)
        k8_exact &= bool(np.array_equal(k8_ref, k8_all[h]) and np.array_equal(ks_ref, ks_all[h]))
    for h in sample_heads:
        q8_ref, qs_ref = oracle.quantize(q_all[h], 128)
        k8_ref, ks_ref = oracle.quantize(k_all[h], 64)
        rows = np.sort(rng.choice(S, size=min(S, rows_per_head), replace=False)).astype(np.int32)
        expected = oracle.tilemix(q_all[h], k_all[h], v_all[h], q8_ref, k8_ref, qs_ref, ks_ref, codes[h],
                                  w.score_scale, w.causal, rows=rows)
        err = np.abs(o_all[h][rows].astype(np.float64) - expected)
        max_abs = max(max_abs, float(err.max()))
        sum_abs += float(err.sum())
        count += err.size
    mean_abs = sum_abs / count
    return {"k8_kscales_bit_exact": k8_exact, "sampled_heads": sample_heads, "sampled_rows": count // D,
            "max_abs": max_abs, "mean_abs": mean_abs,
            "pass": bool(k8_exact and max_abs <= 2e-3 and mean_abs <= 2e-4)}


def cpu_baseline(w, Q, K, V, codes, budget_s: float) -> dict:
    """CPU PyTorch restatement of python/reference_attention.py on whole heads of the
    same workload until ``budget_s`` seconds of work; throughput over the sampled heads."""
    import torch
    sys.path.insert(0, str(ROOT))
    from oracle.torch_reference import reference_attention
    from tilemix import routing

    cores = len(os.sched_getaffinity(0))
    torch.set_num_threads(cores)
    model = ""
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    q_cpu, k_cpu, v_cpu = (t.cpu() for t in (Q, K, V))
    rows, cols = codes.shape[1:]

    def key_mask(h):
        if not (codes[h] == routing.SKIP).any():
            return None
        cell = np.repeat(np.repeat(codes[h] != routing.SKIP, 16, axis=0)[: w.S], 32, axis=1)[:, : w.S]
        return torch.from_numpy(np.ascontiguousarray(cell))

    with torch.inference_mode():
        reference_attention(q_cpu[0][:64].contiguous(), k_cpu[0][:64].contiguous(), v_cpu[0][:64].contiguous())
        done, ops, t_total = 0, 0, 0.0
        while done < w.heads and t_total < budget_s:
            mask = key_mask(done)
            t0 = time.perf_counter()
            reference_attention(q_cpu[done], k_cpu[done], v_cpu[done], causal=w.causal, key_mask=mask,
                                scale=w.score_scale)
            t_total += time.perf_counter() - t0
            one = routing.algorithmic_work(codes[done], w.S, w.S, w.D, w.causal)
            ops += one["ops_int8"] + one["flops_fp16"]
            done += 1
    return {"value": round(ops / t_total / 1e12, 5), "unit": "TFLOP/s", "cores": cores, "kind": "port",
            "sample": f"{done} of {w.heads} heads (full S={w.S}), torch {torch.__version__} CPU fp32 dense "
                      f"softmax attention (python/reference_attention.py restated, masked scores -inf), "
                      f"{t_total:.2f} s, cpu '{model}'",
            "seconds": round(t_total, 3), "heads": done}


if __name__ == "__main__":
    sys.exit(main())
