"""Benchmark: ms per 10-step Pi0 action chunk (hipGraph replay of the decoder loop).

`--workload encoder` measures the prefix encoder instead:
ms per encode of M = 768 rows through 18 layers, with the gated-FFN GEMM's
MFMA roofline and the CPU oracle on a one-layer sample. `--workload full`
times the whole one-graph forward (config 4) against the published H100 figure.

One "step" of this benchmark = one replay of the captured decoder loop: 10
Euler steps x 18 layers at M = 51 rows against 819 keys,
with weights, prefix K/V and inputs already resident in HBM.

Also measured, inside the same run:
  * the dominant kernel (the GeGLU gate/up GEMM, 47% of the bytes) timed with
    HIP events around a captured graph of launches cycling the 18 distinct
    layer weights (cold reads), -> `roofline`;
  * the CPU oracle (fp32 PyTorch restatement) on a bounded
    sample of whole chunks on the host cores, -> `cpu_baseline`.
"""
from __future__ import annotations

import argparse
import json
import os
import statistics
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
for _p in (ROOT, os.path.join(ROOT, "flash-vla_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

HBM_PEAK_GBS = 8000.0
LAYERS, STEPS, ENC_LEN, CHUNK = 18, 10, 768, 50
LAYER_WEIGHT_BYTES = 34_603_008            # qkv + o + gate + up + down, bf16
SMALL_PROJ_BYTES = 2_232_384               # in/mlp/out projections and biases per step
KV_READ_BYTES = LAYERS * 819 * 256 * 2 * 2
KV_WRITE_BYTES = LAYERS * 51 * 256 * 2 * 2
STEP_BYTES = LAYERS * LAYER_WEIGHT_BYTES + SMALL_PROJ_BYTES + KV_READ_BYTES + KV_WRITE_BYTES
CHUNK_BYTES = STEPS * STEP_BYTES           # 6,411,223,680 B
GATE_BYTES = 2 * 1024 * 4096 * 2           # gate + up weights of one layer (activations excluded)
# HBM bytes per launch from rocprofv3 FETCH_SIZE x 2.0 + WRITE_SIZE x 1.0 (KiB; factors from a
# plain 256 MiB copy); profiles/kernels_hbm_traffic_config2_config3.md
GATE_TRAFFIC_BYTES = (8645.0 * 2.0 + 408.0 * 1.0) * 1024
ENC_GATE_TRAFFIC_BYTES = (77941.8 * 2.0 + 24576.0 * 1.0) * 1024   # block_gemm_kernel at M = 768


def _time_graph(run, n_inner, reps, torch):
    """Median microseconds per call of `run(i)` captured n_inner times in one graph."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for i in range(3):
            run(i)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for i in range(n_inner):
            run(i)
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream()
    samples = []
    for _ in range(reps):
        s = torch.cuda.Event(enable_timing=True)
        e = torch.cuda.Event(enable_timing=True)
        s.record(stream)
        g.replay()
        e.record(stream)
        e.synchronize()
        samples.append(s.elapsed_time(e) * 1000.0 / n_inner)
    return statistics.median(samples)


def _timed_calls(call, steps, torch):
    """Run `call()` `steps` times on the current stream, each bracketed by its own pair of
    HIP events, the whole region by an outer pair. Returns (median ms, timing dict)."""
    stream = torch.cuda.current_stream()
    evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
           for _ in range(steps)]
    outer = (torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
    torch.cuda.synchronize()
    outer[0].record(stream)
    for s_ev, e_ev in evs:
        s_ev.record(stream)
        call()
        e_ev.record(stream)
    outer[1].record(stream)
    torch.cuda.synchronize()
    samples = sorted(s_ev.elapsed_time(e_ev) for s_ev, e_ev in evs)
    ms = statistics.median(samples)
    ms_mean = outer[0].elapsed_time(outer[1]) / steps
    if steps < 30:
        print(f"[bench] note: median of {steps} calls (>= 30 recommended)", file=sys.stderr,
              flush=True)
    return ms, {"statistic": f"median of {steps} individually timed calls",
                "ms_mean_bracket": round(ms_mean, 4), "ms_min": round(samples[0], 4),
                "ms_max": round(samples[-1], 4)}


def kernel_roofline(eng, torch):
    from flash_vla_amd.backends.hip import wrappers as W
    b, w = eng.buffers, eng.weights
    with W.use_pool(eng.pool):
        us = _time_graph(lambda i: W.decoder_norm_gated_ffn(
            b["decoder_x"], w["decoder_ffn_gate_w"][i % LAYERS], w["decoder_ffn_up_w"][i % LAYERS],
            b["decoder_hidden"], None), n_inner=LAYERS * 4, reps=20, torch=torch)
    achieved = GATE_BYTES / (us * 1e-6) / 1e9
    return {"kernel": "skinny_gemm_kernel<EPI_GATE> (decoder_norm_gated_ffn)",
            "bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
            "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": int(GATE_TRAFFIC_BYTES),
            "avg_launch_us": round(us, 3), "bytes_per_launch": GATE_BYTES}


def boundary_us(torch) -> float:
    """Cost of one dependent dispatch in a graph: median microseconds per launch of a
    graph of 256 chained one-element kernels (`x += 1`, no memory traffic to speak of)."""
    x = torch.zeros(1, device="cuda")
    return _time_graph(lambda i: x.add_(1.0), n_inner=256, reps=10, torch=torch)


def host_threads() -> int:
    """Threads for the CPU legs: the box's CPU share (OMP_NUM_THREADS, 16 on the GPU pool),
    capped by the cores the OS reports."""
    share = int(os.environ.get("OMP_NUM_THREADS", "16") or 16)
    return max(1, min(os.cpu_count() or 1, share))


def cpu_model() -> str:
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def host_info(threads: int) -> dict:
    return {"cores": threads, "host_cpus": os.cpu_count(), "cpu_model": cpu_model()}


def cpu_baseline(seconds_budget: float = 20.0):
    import torch
    from oracle import pi0_decoder as O
    from flash_vla_amd.weights import decoder_checkpoint, decoder_inputs

    threads = host_threads()
    torch.set_num_threads(threads)
    ck = decoder_checkpoint(seed=0)
    inp = decoder_inputs(seed=1)
    args = (ck, inp["observation_state_normalized"], inp["diffusion_noise"], inp["encoder_K"],
            inp["encoder_V"], ENC_LEN)
    O.decoder_packed(*args, steps=1, bf16=False)       # warm caches / thread pool
    times = []
    t_start = time.perf_counter()
    while len(times) < 3 or (time.perf_counter() - t_start < seconds_budget and len(times) < 10):
        t0 = time.perf_counter()
        O.decoder_packed(*args, steps=STEPS, bf16=False)
        times.append((time.perf_counter() - t0) * 1000.0)
        if time.perf_counter() - t_start > 3 * seconds_budget:
            break
    return {"value": round(statistics.median(times), 2), "unit": "ms per 10-step chunk",
            **host_info(threads), "kind": "port",
            "sample": f"median of {len(times)} full 10-step chunks (fp32 PyTorch oracle, "
                      f"config 1 maths on the packed bf16 weights)"}


ENC_M, ENC_LAYERS, ENC_W, ENC_FFN, ENC_QKV = 768, 18, 2048, 16384, 2560
MFMA_BF16_PEAK_TFLOPS = 2500.0


def encoder_flops(M=ENC_M, layers=ENC_LAYERS):
    """Algorithmic flops of one encode: 17 full layers + the last layer's QKV projection."""
    qkv = 2 * M * ENC_W * ENC_QKV
    attn = 2 * 2 * (M * 8) * M * 256
    o = 2 * M * ENC_W * ENC_W
    gate = 2 * M * ENC_W * 2 * ENC_FFN
    down = 2 * M * ENC_FFN * ENC_W
    return (layers - 1) * (qkv + attn + o + gate + down) + qkv, 2 * M * ENC_W * 2 * ENC_FFN


def encoder_cpu_baseline(ck_cpu, x_cpu):
    import torch
    from oracle import pi0_encoder as E
    threads = host_threads()
    torch.set_num_threads(threads)
    one = {k: v[:2] for k, v in ck_cpu.items()}
    E.encoder_packed(one, x_cpu[:64], layers=2, bf16=False)          # warm the thread pool
    t = {}
    for n in (1, 2):
        t0 = time.perf_counter()
        E.encoder_packed(one, x_cpu, layers=n, bf16=False)
        t[n] = (time.perf_counter() - t0) * 1000.0
    full_layer = t[2] - t[1]
    est = (ENC_LAYERS - 1) * full_layer + t[1]
    return {"value": round(est, 1), "unit": "ms per encode (M=768, 18 layers)", **host_info(threads),
            "kind": "port",
            "sample": f"fp32 PyTorch oracle timed on 1 full layer ({full_layer:.0f} ms) and the "
                      f"QKV-only last layer ({t[1]:.0f} ms) at M=768; value = 17 x full + last"}


def main_encoder(args, torch):
    from flash_vla_amd import Pi0EncoderEngine
    from flash_vla_amd.weights import encoder_checkpoint, encoder_inputs
    from flash_vla_amd.backends.hip import encoder_wrappers as EW
    from flash_vla_amd.backends.hip import wrappers as W

    t0 = time.time()
    ck = encoder_checkpoint(seed=2, device="cuda", draw_on_device=True)
    x = encoder_inputs(seed=3).cuda()
    eng = Pi0EncoderEngine(ck, encoder_seq_len=ENC_M, copy_weights=False)
    print(f"[bench] encoder engine captured, {time.time() - t0:.1f}s", file=sys.stderr, flush=True)
    for _ in range(max(args.warmup, 3)):
        eng.forward(x)
    # each call copies the [768, 2048] input into the static buffer and replays the graph
    ms, timing = _timed_calls(lambda: eng.forward(x), args.steps, torch)
    flops, gate_flops = encoder_flops()
    print(f"[bench] encoder {ms:.3f} ms/encode", file=sys.stderr, flush=True)

    roof = None
    if not args.no_kernel:
        b = eng.buffers
        with W.use_pool(eng.pool):
            us = _time_graph(lambda i: EW.encoder_norm_gated_ffn(
                b["encoder_x"], ck["encoder_ffn_gate_w"][i % ENC_LAYERS],
                ck["encoder_ffn_up_w"][i % ENC_LAYERS], b["encoder_hidden"], b["encoder_x_norm"]),
                n_inner=ENC_LAYERS, reps=10, torch=torch)
        achieved = gate_flops / (us * 1e-6) / 1e12
        roof = {"kernel": "block_gemm_kernel + rms_norm_kernel (encoder_norm_gated_ffn)",
                "bound": "mfma", "achieved": round(achieved, 1), "peak": MFMA_BF16_PEAK_TFLOPS,
                "unit": "TFLOP/s", "frac": round(achieved / MFMA_BF16_PEAK_TFLOPS, 4),
                "traffic": int(ENC_GATE_TRAFFIC_BYTES), "avg_launch_us": round(us, 3), "flops_per_launch": gate_flops}
    cpu = None
    if not args.no_cpu:
        ck_cpu = encoder_checkpoint(seed=2, layers=2)
        cpu = encoder_cpu_baseline(ck_cpu, encoder_inputs(seed=3))
    out = {
        "metric": "ms per prefix encode (18 layers, hipGraph)",
        "value": round(ms, 4), "unit": "ms", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(ms, 4), "higher_is_better": False,
        "scaling": "weak", "vs_baseline": None, "dtype": "bf16",
        "data": "synthetic (seeded N(0,0.02) packed weights, N(0,1) [768, 2048] input)",
        "config": {"workload": "Pi0 prefix encoder, BASELINE config 3: 18 Gemma layers at M=768, "
                               "width 2048, 8 q heads / 1 kv head x 256, GeGLU 2048 -> 2 x 16384, "
                               "bidirectional attention, last layer QKV only",
                   "global_batch": 1, "seq_len": ENC_M, "parallelism": "single GPU"},
        "tflops": round(flops / (ms * 1e-3) / 1e12, 1),
        "mfma_frac": round(flops / (ms * 1e-3) / 1e12 / MFMA_BF16_PEAK_TFLOPS, 4),
        "flops_per_encode": flops,
        "timing": timing,
        "roofline": roof,
        "cpu_baseline": cpu,
    }
    print(json.dumps(out), flush=True)


H100_FULL_FORWARD_MS = 15.18     # full Pi0 forward, fused, H100 SXM5 (README.md:108)


def main_full(args, torch):
    """the whole Pi0Inference.forward (3 views, empty prompt, chunk 50)."""
    from flash_vla_amd import Pi0Inference
    from flash_vla_amd.weights import random_checkpoint

    t0 = time.time()
    B, P = args.batch, args.prompt_tokens
    ck = random_checkpoint(prompt_len=0, seed=0, device="cuda", draw_on_device=True)
    gen = torch.Generator().manual_seed(4)
    lead = (B,) if B > 1 else ()
    images = (torch.rand(*lead, 3, 224, 224, 3, generator=gen) * 2 - 1).to(torch.bfloat16).cuda()
    state = torch.randn(*lead, 32, generator=gen).to(torch.bfloat16).cuda()
    noise = torch.randn(*lead, 50, 32, generator=gen).to(torch.bfloat16).cuda()
    ids = None
    if P:
        vocab = 257152
        ck["embed_tokens"] = (torch.randn(vocab, 2048, device="cuda",
                                          generator=torch.Generator(device="cuda").manual_seed(5))
                              * 0.05).to(torch.bfloat16)
        ids = torch.randint(0, vocab, (B, P), generator=gen, dtype=torch.int32).cuda()
    eng = Pi0Inference(ck, num_views=3, chunk_size=50, batch=B, prompt_tokens=P)
    del ck
    print(f"[bench] full forward captured, {time.time() - t0:.1f}s", file=sys.stderr, flush=True)
    for _ in range(max(args.warmup, 3)):
        eng.forward(images, state, noise, ids)
    # each call copies the inputs into the static buffers and replays the graph
    ms, timing = _timed_calls(lambda: eng.forward(images, state, noise, ids), args.steps, torch)
    print(f"[bench] full forward {ms:.3f} ms", file=sys.stderr, flush=True)
    config5 = B > 1 or P > 0
    M_enc = B * (768 + P)
    roof = None
    if not args.no_kernel:
        # the forward's largest kernel: the encoder's RMSNorm + gated FFN at M = B x prefix
        from flash_vla_amd.backends.hip import encoder_wrappers as EW
        from flash_vla_amd.backends.hip import wrappers as W
        b, w = eng.buffers, eng.weights
        with W.use_pool(eng.pool):
            us = _time_graph(lambda i: EW.encoder_norm_gated_ffn(
                b["encoder_x"], w["encoder_ffn_gate_w"][i % ENC_LAYERS],
                w["encoder_ffn_up_w"][i % ENC_LAYERS], b["encoder_hidden"], b["encoder_x_norm"]),
                n_inner=ENC_LAYERS, reps=10, torch=torch)
        gate_flops = 2 * M_enc * ENC_W * 2 * ENC_FFN
        achieved = gate_flops / (us * 1e-6) / 1e12
        roof = {"kernel": "block_gemm_kernel + rms_norm_kernel (encoder_norm_gated_ffn)",
                "bound": "mfma", "achieved": round(achieved, 1), "peak": MFMA_BF16_PEAK_TFLOPS,
                "unit": "TFLOP/s", "frac": round(achieved / MFMA_BF16_PEAK_TFLOPS, 4),
                "traffic": int(ENC_GATE_TRAFFIC_BYTES) if not config5 else None,
                "avg_launch_us": round(us, 3), "flops_per_launch": gate_flops}
    cpu = None if args.no_cpu else full_forward_cpu_baseline(B, P)
    workload = ("Pi0 full forward, BASELINE config 4: 3 views 224x224, SigLIP 27 layers, "
                "projector, 18-layer encoder at M=768, empty prompt, 10-step decoder, chunk 50")
    if config5:
        workload = (f"Pi0 full forward, BASELINE config 5 profile: batch {B} independent requests "
                    f"(3 views each), {P}-token prompt embedded from a 257152 x 2048 table x "
                    f"sqrt(2048) (prefix {768 + P}), decoder M={51 * B}, keys {768 + P + 51}, "
                    f"10 steps, chunk 50")
    out = {
        "metric": "ms per full Pi0 forward (vision + encoder + 10-step decoder, one hipGraph)",
        "value": round(ms, 4), "unit": "ms", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(ms, 4), "higher_is_better": False,
        "scaling": "weak", "dtype": "bf16",
        # the published H100 figure is for config 4 only
        "vs_baseline": None if config5 else round(ms / H100_FULL_FORWARD_MS, 4),
        "data": "synthetic (random_checkpoint N(0,1) x 0.05 weights, uniform[-1,1] images, "
                "N(0,1) state and noise" + (", uniform token ids)" if P else ")"),
        "config": {"workload": workload, "global_batch": B, "seq_len": 768 + P,
                   "parallelism": "single GPU"},
        "action_chunks_per_s": round(B * 1000.0 / ms, 2),
        "baseline_ms": None if config5 else H100_FULL_FORWARD_MS,
        "baseline_hw": None if config5 else "H100 SXM5 (published)",
        "timing": timing, "roofline": roof, "cpu_baseline": cpu,
    }
    print(json.dumps(out), flush=True)


def full_forward_cpu_baseline(batch: int, prompt: int):
    """The fp32 PyTorch oracles on the host cores, extrapolated per request from one timed
    SigLIP layer (x 27), one full encoder layer (x 17) plus the QKV-only last layer at the
    request's prefix length, and one whole 10-step decoder chunk; x `batch` requests."""
    import torch
    from oracle import pi0_decoder as O
    from oracle import pi0_encoder as E
    from oracle import pi0_vision as V
    from flash_vla_amd.weights import decoder_checkpoint, decoder_inputs, encoder_checkpoint
    threads = host_threads()
    torch.set_num_threads(threads)
    gen = torch.Generator().manual_seed(6)
    vw = {"vision_pre_attn_norm_w": torch.ones(1, 1152), "vision_pre_attn_norm_b": torch.zeros(1, 1152),
          "vision_attn_qkv_w": torch.randn(1, 1152, 3456, generator=gen) * 0.02,
          "vision_attn_qkv_b": torch.zeros(1, 3456),
          "vision_attn_o_w": torch.randn(1, 1152, 1152, generator=gen) * 0.02,
          "vision_attn_o_b": torch.zeros(1, 1152),
          "vision_pre_ffn_norm_w": torch.ones(1, 1152), "vision_pre_ffn_norm_b": torch.zeros(1, 1152),
          "vision_ffn_up_w": torch.randn(1, 1152, 4304, generator=gen) * 0.02,
          "vision_ffn_up_b": torch.zeros(1, 4304),
          "vision_ffn_down_w": torch.randn(1, 4304, 1152, generator=gen) * 0.02,
          "vision_ffn_down_b": torch.zeros(1, 1152)}
    vx = torch.randn(768, 1152, generator=gen)
    V.vision_layer(vx[:256], vw, 0, 1, bf16=False)                    # warm the thread pool
    vis_layer = float("inf")
    for _ in range(2):
        t0 = time.perf_counter()
        V.vision_layer(vx, vw, 0, 3, bf16=False)
        vis_layer = min(vis_layer, (time.perf_counter() - t0) * 1000.0)
    M = 768 + prompt
    ck = {k: v[:2] for k, v in encoder_checkpoint(seed=2, layers=2).items()}
    ex = torch.randn(M, 2048, generator=gen).to(torch.bfloat16)
    E.encoder_packed(ck, ex[:64], layers=2, bf16=False)              # warm-up
    t = {}
    for n in (1, 2):                     # best of two: the layer time is a difference
        best = float("inf")
        for _ in range(2):
            t0 = time.perf_counter()
            E.encoder_packed(ck, ex, layers=n, bf16=False)
            best = min(best, (time.perf_counter() - t0) * 1000.0)
        t[n] = best
    enc = (ENC_LAYERS - 1) * (t[2] - t[1]) + t[1]
    dck, inp = decoder_checkpoint(seed=0), decoder_inputs(seed=1)
    keys_pad = M - ENC_LEN
    K = inp["encoder_K"] if keys_pad == 0 else torch.cat(
        [inp["encoder_K"], inp["encoder_K"][:, :keys_pad]], dim=1)
    Vc = inp["encoder_V"] if keys_pad == 0 else torch.cat(
        [inp["encoder_V"], inp["encoder_V"][:, :keys_pad]], dim=1)
    O.decoder_packed(dck, inp["observation_state_normalized"], inp["diffusion_noise"], K, Vc, M,
                     steps=1, layers=2, bf16=False)                  # warm-up
    t0 = time.perf_counter()
    O.decoder_packed(dck, inp["observation_state_normalized"], inp["diffusion_noise"], K, Vc, M,
                     steps=STEPS, bf16=False)
    dec = (time.perf_counter() - t0) * 1000.0
    per_request = 27 * vis_layer + enc + dec
    return {"value": round(batch * per_request, 1), "unit": "ms per full forward", **host_info(threads),
            "kind": "port",
            "sample": f"fp32 PyTorch oracles, per request: 27 x one SigLIP layer ({vis_layer:.0f} ms), "
                      f"encoder at M={M} = 17 x one full layer ({t[2] - t[1]:.0f} ms) + the QKV-only "
                      f"layer ({t[1]:.0f} ms), one 10-step decoder chunk ({dec:.0f} ms); x {batch} "
                      f"request(s); patch embedding and projector omitted"}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--workload", choices=("decoder", "encoder", "full"), default="decoder",
                    help="decoder loop (the headline metric), the prefix encoder, or the "
                         "whole forward")
    ap.add_argument("--batch", type=int, default=1,
                    help="--workload full: independent requests per forward (config 5: 4)")
    ap.add_argument("--prompt-tokens", type=int, default=0,
                    help="--workload full: prompt length in token ids (config 5: 48)")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--no-kernel", action="store_true", help="skip the per-kernel roofline leg")
    ap.add_argument("--kernel-only", action="store_true",
                    help="decoder: only the gate-kernel roofline leg (no loop capture), so a "
                         "rocprofv3 trace of this command holds just that kernel's timed launches")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="only run a plain 256 MiB device copy (5x), to calibrate rocprofv3 "
                         "FETCH_SIZE / WRITE_SIZE against a kernel of known traffic")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only (the decoder loop is a single-GPU path); "
              f"--gpus {args.gpus} is not supported", file=sys.stderr)
        sys.exit(2)

    import torch
    if args.copy_calibration:
        src = torch.ones(64 << 20, dtype=torch.float32, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(5):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"copy_calibration_bytes_read": src.numel() * 4,
                          "copy_calibration_bytes_written": dst.numel() * 4, "launches": 5}))
        return

    if args.workload == "encoder":
        main_encoder(args, torch)
        return
    if args.workload == "full":
        main_full(args, torch)
        return

    from flash_vla_amd import Pi0DecoderEngine
    from flash_vla_amd.weights import decoder_checkpoint, decoder_inputs

    t0 = time.time()
    ck = decoder_checkpoint(seed=0)
    inp = decoder_inputs(seed=1)
    print(f"[bench] inputs generated in {time.time() - t0:.1f}s", file=sys.stderr, flush=True)
    if args.kernel_only:
        eng = Pi0DecoderEngine({k: v.cuda() for k, v in ck.items()}, steps=STEPS, layers=LAYERS,
                               capture=False)
        print(json.dumps({"roofline": kernel_roofline(eng, torch)}), flush=True)
        return
    eng = Pi0DecoderEngine({k: v.cuda() for k, v in ck.items()}, steps=STEPS, layers=LAYERS)
    eng.load_prefix(inp["encoder_K"].cuda(), inp["encoder_V"].cuda())
    state = inp["observation_state_normalized"].cuda()
    noise = inp["diffusion_noise"].cuda()
    eng.buffers["observation_state_normalized"].copy_(state)
    print(f"[bench] engine captured, {time.time() - t0:.1f}s", file=sys.stderr, flush=True)

    stream = torch.cuda.current_stream()
    for _ in range(max(args.warmup, 3)):
        eng.buffers["diffusion_noise"].copy_(noise)
        eng.replay()
    torch.cuda.synchronize()
    # timed region: exactly `steps` chunk replays, each bracketed by its own pair of HIP
    # events (the noise is not reset in between; each replay is a full 10-step denoise of
    # whatever the buffer holds). value = the median replay; the mean over the whole
    # bracket is reported beside it.
    ms, timing = _timed_calls(eng.replay, args.steps, torch)
    print(f"[bench] {ms:.3f} ms/chunk (median of {args.steps}; bracket mean "
          f"{timing['ms_mean_bracket']:.3f})", file=sys.stderr, flush=True)

    # lower-bound model of the loop: every kernel / copy node of the captured chain is one
    # dependent dispatch, and one dispatch costs at least an empty kernel's boundary
    nodes = eng.graph_nodes()
    launches = sum(v for k, v in nodes.items() if k in ("kernel", "memcpy", "memset"))
    b_us = boundary_us(torch)
    roof = None if args.no_kernel else kernel_roofline(eng, torch)
    if roof is not None:
        # the same launches with the graph boundary (an empty kernel's cost, measured above)
        # taken out: the kernel's own share of each launch (reported beside `frac`)
        own = roof["avg_launch_us"] - b_us
        roof["boundary_us"] = round(b_us, 3)
        roof["frac_excl_boundary"] = round(GATE_BYTES / (own * 1e-6) / 1e9 / HBM_PEAK_GBS, 4)
    cpu = None if args.no_cpu else cpu_baseline()

    gbs = CHUNK_BYTES / (ms * 1e-3) / 1e9
    out = {
        "metric": "ms per 10-step action chunk (decoder loop, hipGraph)",
        "value": round(ms, 4), "unit": "ms", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(ms, 4), "higher_is_better": False,
        "scaling": "weak", "vs_baseline": None, "dtype": "bf16",
        "data": "synthetic (seeded N(0,0.02) folded weights, N(0,1) prefix K/V, state, noise)",
        "config": {"workload": "Pi0 decoder loop, BASELINE config 2: 10 Euler steps x 18 layers, "
                               "M=51 rows (1 state + 50 actions), 8 q heads / 1 kv head x 256, "
                               "keys 819, width 1024, FFN 4096, batch 1",
                   "global_batch": 1, "seq_len": 51, "keys": 819, "parallelism": "single GPU",
                   # the engine default; the reference re-rounds a bf16 diffusion_noise every
                   # step (pipeline.py:105,132), selectable with fp32_euler=False
                   "euler_accumulator": "fp32"},
        "ms_per_decoder_step": round(ms / STEPS, 4),
        "launches_per_chunk": launches,
        "graph_nodes": nodes,
        "boundary_us": round(b_us, 3),
        "sync_floor_ms": round(launches * b_us / 1000.0, 4),
        "sync_floor_frac_of_value": round(launches * b_us / 1000.0 / ms, 4),
        "hbm_gbs": round(gbs, 1),
        "loop_roofline_frac": round(gbs / HBM_PEAK_GBS, 4),
        "bytes_per_chunk": CHUNK_BYTES,
        "timing": timing,
        "roofline": roof,
        "cpu_baseline": cpu,
    }
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
