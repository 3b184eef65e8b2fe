"""Throughput of the gfx950 BC4 decode GEMV on the 27B-class linear shapes (batch 1).

One "step" is one decode sweep: every q, k, v, o, gate, up and down linear of ``--layers``
distinct layer copies, each a batch-1 GEMV with a float32 output. The
copies are distinct device buffers, together far larger than the 256 MB Infinity Cache, so the
weights stream from HBM. A step is captured once as a HIP graph and replayed.

Prints one JSON line. ``value`` is the algorithmic HBM bytes of a step (BC4 payload + row
scales + bf16 x + fp32 y per linear) times the step count, divided by the timed wall time.
``roofline`` is the 5120->27648 (gate/up) GEMV alone: its algorithmic bytes divided by its
average launch time over back-to-back launches timed with HIP events on the launch stream.
``cpu_baseline`` is the CPU path on the host cores: per-shape medians of the C restatement's fused
decode + matvec, of the decode and of the matvec alone, and the config-3 fp32 GEMM.
``hbm_stream_read`` is a plain streaming read of the same launch size (the achievable HBM rate);
``roofline.frac_of_stream_read`` is the GEMV's rate against it.
``prefill_tok_s_512`` and ``decode_tok_s`` are the metric's other two figures on the 27B-class
decoder (64 layers, hidden 5120, linears BC4-encoded from random-init weights): the 512-token prefill
(``texelator_amd.prefill.benchmark_prefill``; null with ``prefill_gate_failed`` if the prefill path
fails the reference protocol's correctness gate) and graph-replayed greedy decode from 512 to
``--context`` with every step timed; ``model`` holds the details, ``model_3b`` the same for the
3B-class one, and ``model_3b_hf`` that one through the reference's own calling path (a Hugging Face
Qwen2 with TexelatorLinear modules: prefill protocol and greedy ``generate``).
"""
from __future__ import annotations

import argparse
import json
import os
import platform
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))

HBM_PEAK_GBS = 8000.0
SEED = 20260827
HIDDEN, INTER, KV = 5120, 27648, 1024
# (name, M = output features, K = input features)
LAYER = [("q", HIDDEN, HIDDEN), ("k", KV, HIDDEN), ("v", KV, HIDDEN), ("o", HIDDEN, HIDDEN),
         ("gate", INTER, HIDDEN), ("up", INTER, HIDDEN), ("down", HIDDEN, INTER)]
DOMINANT = ("gate", "up")
TRAFFIC_FILE = ROOT / "profiles" / "gemv_gate_up_5120x27648.md"


def gemv_bytes(m: int, k: int) -> int:
    """Algorithmic HBM bytes of one batch-1 GEMV: payload + scales + bf16 x + fp32 y."""
    return m * k // 2 + 4 * m + 2 * k + 4 * m


def log(message: str) -> None:
    print(f"[bench] {message}", file=sys.stderr, flush=True)


def encoded_weights(torch, shapes, lut):
    """BC4-encode one W ~ N(0, 0.02^2) * LogNormal(0, 0.3) per input channel for each shape."""
    from texelator_amd.encoder import encode_matrix

    out = {}
    generator = torch.Generator(device="cuda").manual_seed(SEED)
    for m, k in shapes:
        w = torch.randn((m, k), device="cuda", generator=generator) * 0.02
        s = torch.exp(0.3 * torch.randn(k, device="cuda", generator=generator))
        w *= s[None, :]
        hdiag = torch.ones(k, device="cuda")
        out[(m, k)] = encode_matrix(w, hdiag, lut, rows_per_chunk=2048)
        del w
    torch.cuda.synchronize()
    return out


def read_traffic():
    """HBM bytes per gate/up launch measured with rocprofv3 counters, if recorded."""
    if not TRAFFIC_FILE.exists():
        return None
    for line in TRAFFIC_FILE.read_text().splitlines():
        if line.startswith("traffic_bytes_per_launch:"):
            return float(line.split(":", 1)[1])
    return None


def cpu_model() -> str:
    """The host CPU's model name (``/proc/cpuinfo``, with its family/model/stepping numbers, which
    name the part where a virtualised host reports only a vendor string), or the platform's
    processor string."""
    fields = {}
    try:
        for line in Path("/proc/cpuinfo").read_text().splitlines():
            key, _, value = line.partition(":")
            key = key.strip()
            if key in ("model name", "cpu family", "model", "stepping") and key not in fields:
                fields[key] = value.strip()
            if not line.strip() and fields:
                break
    except OSError:
        pass
    if "model name" not in fields:
        return platform.processor() or platform.machine()
    ids = ", ".join(f"{k} {fields[k]}" for k in ("cpu family", "model", "stepping") if k in fields)
    return f"{fields['model name']} ({ids})" if ids else fields["model name"]


def cpu_quota() -> float | None:
    """CPUs' worth of time the cgroup allows this process (``cpu.max``), or None if unlimited."""
    for path in ("/sys/fs/cgroup/cpu.max",):
        try:
            quota, period = Path(path).read_text().split()[:2]
        except (OSError, ValueError):
            continue
        if quota != "max":
            return int(quota) / int(period)
    try:
        quota = int(Path("/sys/fs/cgroup/cpu/cpu.cfs_quota_us").read_text())
        period = int(Path("/sys/fs/cgroup/cpu/cpu.cfs_period_us").read_text())
        return quota / period if quota > 0 else None
    except (OSError, ValueError):
        return None


def cpu_threads() -> tuple[int, int, float | None]:
    """(threads used, cores in this process's affinity mask, cgroup CPU quota). Every affinity core
    is used unless the cgroup grants fewer CPUs' worth of time, where more threads than that only
    time-slice against each other."""
    affinity = len(os.sched_getaffinity(0))
    quota = cpu_quota()
    threads = affinity if quota is None else max(1, min(affinity, int(quota)))
    return threads, affinity, quota


def _median_seconds(fn, runs: int) -> float:
    import statistics

    samples = []
    for _ in range(runs):
        start = time.perf_counter()
        fn()
        samples.append(time.perf_counter() - start)
    return statistics.median(samples)


def cpu_baseline(weights, runs: int = 5) -> dict:
    """The CPU path on the host cores, bounded to ~10-30 s: per distinct config-2 shape, medians
    of ``runs`` runs of (a) the C restatement's fused BC4 decode + fp32 matvec
    (``oracle_decode_matvec_f32``, OpenMP), (b) the BC4 -> bf16 decode alone (``oracle_decode_bf16``)
    and (c) the fp32 matvec alone on the decoded weights (torch CPU); then the config-3 fp32 GEMM
    on the decoded weights at T = 32, 128, 512 (torch CPU). ``value`` is one layer's seven linears
    (algorithmic GEMV bytes) over the sum of their decode + matvec medians."""
    import numpy as np
    import torch

    from oracle import bc4, clib

    cores, affinity, quota = cpu_threads()
    clib.set_threads(cores)
    torch.set_num_threads(cores)
    rng = np.random.default_rng(SEED)
    x32 = {k: rng.standard_normal(k).astype(np.float32) for k in (HIDDEN, INTER)}
    xbits = {k: bc4.f32_to_bf16_bits(v) for k, v in x32.items()}
    per_shape, decoded = {}, {}
    started = time.perf_counter()
    for name, m, k in LAYER:
        if (m, k) in decoded:
            continue
        blocks, scales = weights[(m, k)]
        fused = _median_seconds(lambda: clib.decode_matvec_f32(blocks, scales, xbits[k]), runs)
        decode = _median_seconds(lambda: clib.decode_bf16_bits(blocks, scales), runs)
        w = torch.from_numpy(bc4.bf16_bits_to_f32(clib.decode_bf16_bits(blocks, scales)))
        xv = torch.from_numpy(bc4.bf16_bits_to_f32(xbits[k]))
        matvec = _median_seconds(lambda: torch.mv(w, xv), runs)
        decoded[(m, k)] = w
        per_shape[f"{k}x{m}"] = {
            "decode_matvec_ms": round(fused * 1e3, 3), "decode_ms": round(decode * 1e3, 3),
            "matvec_ms": round(matvec * 1e3, 3),
            "decode_matvec_GB/s": round(gemv_bytes(m, k) / fused / 1e9, 3), "runs": runs}
    layer_seconds = sum(per_shape[f"{k}x{m}"]["decode_matvec_ms"] / 1e3 for _, m, k in LAYER)
    layer_bytes = sum(gemv_bytes(m, k) for _, m, k in LAYER)
    gemm = {}
    for name in PREFILL_SHAPES:
        m, k = next((m, k) for n, m, k in LAYER if n == name)
        w = decoded[(m, k)]
        for tokens in PREFILL_TOKENS:
            xt = torch.from_numpy(rng.standard_normal((tokens, k)).astype(np.float32)).to(torch.bfloat16).float()
            seconds = _median_seconds(lambda: torch.mm(xt, w.t()), runs)
            gemm[f"{name}_{k}x{m}_T{tokens}"] = {"ms": round(seconds * 1e3, 2),
                                                 "GFLOP/s": round(2.0 * tokens * m * k / seconds / 1e9, 1),
                                                 "tokens_per_s": round(tokens / seconds, 1)}
    elapsed = time.perf_counter() - started
    return {
        "value": round(layer_bytes / layer_seconds / 1e9, 3),
        "unit": "GB/s",
        "cores": cores,
        "kind": "port",
        "cpu_model": cpu_model(),
        "affinity_cores": affinity,
        "host_cpus": os.cpu_count(),
        "cgroup_cpu_quota": quota,
        "sample": (f"one layer's 7 linears, medians of {runs} runs per distinct shape of the C restatement's "
                   f"fused BC4 decode + fp32 matvec ({cores} OpenMP threads); per-shape decode-only and "
                   f"matvec-only medians and the T=32/128/512 fp32 GEMM (torch CPU, {cores} threads) beside it; "
                   f"{elapsed:.1f} s in all"),
        "per_shape": per_shape,
        "prefill_gemm": gemm,
    }


COPY_BYTES = 1 << 30
MFMA_BF16_PEAK_TFLOPS = 2500.0
PREFILL_TOKENS = (32, 128, 512)
PREFILL_SHAPES = ("q", "gate", "down")


def timed_launches(torch, stream, launch, count: int) -> float:
    """Seconds per launch of ``count`` back-to-back launches, queued behind a spin kernel so that
    the host cost of issuing them is hidden, timed with events on ``stream``."""
    torch.cuda.synchronize()
    torch.cuda._sleep(20_000_000)
    begin = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    begin.record(stream)
    for i in range(count):
        launch(i)
    end.record(stream)
    torch.cuda.synchronize()
    return begin.elapsed_time(end) / 1e3 / count


def prefill_section(torch, ext, stream, handles, candidates=range(5, 10), repeats: int = 2) -> dict:
    """bf16 prefill GEMM per shape and token count: every tile candidate timed over the layer
    copies; reports the fastest, its TFLOP/s and MFMA utilisation against the dense bf16 peak."""
    out = {}
    generator = torch.Generator(device="cuda").manual_seed(SEED + 2)
    for name in PREFILL_SHAPES:
        group = [(m, k, h) for (n, m, k, h) in handles if n == name]
        m, k, _ = group[0]
        for tokens in PREFILL_TOKENS:
            x = torch.randn((tokens, k), device="cuda", generator=generator).to(torch.bfloat16)
            y = torch.empty((tokens, m), device="cuda", dtype=torch.bfloat16)
            nbytes = ext.workspace_bytes(group[0][2], tokens)
            ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device="cuda")
            times, outputs = {}, {}
            for cand in candidates:
                launch = lambda i, c=cand: ext.prefill_into(group[i % len(group)][2], c, x, y, ws)  # noqa: E731
                launch(0)
                outputs[cand] = y.clone()
                times[cand] = timed_launches(torch, stream, launch, repeats * len(group))
            first = outputs[min(outputs)]
            equal = all(torch.equal(first, value) for value in outputs.values())
            if not equal:
                log(f"prefill tiles differ on {name} T={tokens}")
            best = min(times, key=times.get)
            flops = 2.0 * tokens * m * k
            tflops = flops / times[best] / 1e12
            out[f"{name}_{k}x{m}_T{tokens}"] = {
                "best": ext.candidate_name(best), "us": round(times[best] * 1e6, 2),
                "TFLOP/s": round(tflops, 1), "mfma_util": round(tflops / MFMA_BF16_PEAK_TFLOPS, 4),
                "tokens_per_s": round(tokens / times[best], 1),
                "workspace_bytes": nbytes, "candidates_bitwise_equal": equal,
                "all_us": {ext.candidate_name(c): round(t * 1e6, 2) for c, t in times.items()},
            }
    return out


def stream_read(torch, stream, copies: int, repeats: int = 2) -> dict:
    """Achievable HBM read rate for the gate/up launch size: a plain streaming-read kernel over
    ``copies`` distinct buffers of the gate/up payload size, back-to-back launches between events
    (the GEMV's timing method)."""
    import ctypes

    from texelator_amd import _lib
    from texelator_amd._lib import check

    nbytes = INTER * HIDDEN // 2
    generator = torch.Generator(device="cuda").manual_seed(SEED + 3)
    bufs = [torch.randint(0, 256, (nbytes,), dtype=torch.uint8, device="cuda", generator=generator)
            for _ in range(copies)]
    sink = torch.empty(4096, dtype=torch.int32, device="cuda")
    lib = _lib.load()

    def launch(i):
        check(lib.tx_stream_read(ctypes.c_void_p(bufs[i % copies].data_ptr()), nbytes,
                                 ctypes.c_void_p(sink.data_ptr()), ctypes.c_void_p(stream.cuda_stream)))

    launch(0)
    seconds = timed_launches(torch, stream, launch, repeats * copies)
    del bufs
    return {"GB/s": round(nbytes / seconds / 1e9, 1), "bytes_per_launch": nbytes, "avg_launch_us": round(seconds * 1e6, 3),
            "launches": repeats * copies}


def kernel_only(torch, ext, runtime, hardware, device, args) -> int:
    """Launches for counter runs: the 5120->27648 GEMV on ``--layers`` distinct copies, three
    times each, then one device-to-device copy of COPY_BYTES (read COPY_BYTES, write COPY_BYTES)
    whose FETCH_SIZE/WRITE_SIZE readings give the counters' scale."""
    lut = hardware.device_palette(device)
    blocks, scales = encoded_weights(torch, [(INTER, HIDDEN)], lut)[(INTER, HIDDEN)]
    handles = [runtime.pack_arrays(blocks, scales, lookahead=args.lookahead or 1)[0] for _ in range(args.layers)]
    x = torch.randn((1, HIDDEN), device=device).to(torch.bfloat16)
    y = torch.empty((1, INTER), device=device, dtype=torch.float32)
    for _ in range(3):
        for handle in handles:
            ext.linear_f32_into(handle, x, y)
    torch.cuda.synchronize()
    src = torch.empty(COPY_BYTES, dtype=torch.uint8, device=device).fill_(1)
    dst = torch.empty_like(src)
    torch.cuda.synchronize()
    dst.copy_(src)
    torch.cuda.synchronize()
    runtime.free(handles)
    print(json.dumps({"kernel_only": True, "launches": 3 * len(handles), "bytes_per_launch": gemv_bytes(INTER, HIDDEN),
                      "copy_bytes": COPY_BYTES}), flush=True)
    return 0


def prefill_only(torch, ext, runtime, hardware, device, args) -> int:
    """Launches for counter runs: the 5120->27648 prefill GEMM at ``--prompt`` tokens (the library's
    default tile for that shape, or candidate ``--tile``) on ``--layers`` distinct copies, twice each."""
    lut = hardware.device_palette(device)
    blocks, scales = encoded_weights(torch, [(INTER, HIDDEN)], lut)[(INTER, HIDDEN)]
    handles = [runtime.pack_arrays(blocks, scales)[0] for _ in range(args.layers)]
    if args.tile:
        for handle in handles:
            ext.set_prefill_backend(handle, args.tile)
    x = torch.randn((args.prompt, HIDDEN), device=device).to(torch.bfloat16)
    for _ in range(2):
        for handle in handles:
            ext.linear(handle, x)
    torch.cuda.synchronize()
    runtime.free(handles)
    print(json.dumps({"prefill_only": True, "launches": 2 * len(handles), "tokens": args.prompt, "tile": args.tile,
                      "flops_per_launch": 2 * args.prompt * INTER * HIDDEN}), flush=True)
    return 0


# The reference's FP4 hybrid shapes (texelator/runtime.py:66-131: its MLP at 512 tokens), as (M, K).
FP4_SHAPES = [(17408, 5120), (5120, 17408)]


def fp4_only(torch, ext, runtime, hardware, device, args) -> int:
    """The FP4 hybrid prefill at ``--prompt`` tokens on the reference's two MLP shapes, each stage
    timed over ``--layers`` distinct weight copies (back-to-back launches, HIP events): activation
    quantization, weight requantization from the BC4 tiles, the block-scaled GEMM, and the bf16
    prefill GEMM of the same matrices for comparison."""
    lut = hardware.device_palette(device)
    weights = encoded_weights(torch, FP4_SHAPES, lut)
    stream = torch.cuda.current_stream()
    tokens = args.prompt
    out = {}
    for m, k in FP4_SHAPES:
        blocks, scales = weights[(m, k)]
        handles = [runtime.pack_arrays(blocks, scales)[0] for _ in range(args.layers)]
        x = torch.randn((tokens, k), device=device).to(torch.bfloat16)
        xp, xs = ext.quantize_activation_fp4(x)
        staged = [ext.decode_weight_fp4(h) for h in handles]
        n = len(handles)
        for h in handles:
            ext.linear(h, x)
        times = {
            "bf16_prefill_us": timed_launches(torch, stream, lambda i: ext.linear(handles[i % n], x), 2 * n),
            "quantize_us": timed_launches(torch, stream, lambda i: ext.quantize_activation_fp4_out(x, xp, xs), 2 * n),
            "requantize_us": timed_launches(torch, stream, lambda i: ext.decode_weight_fp4_out(handles[i % n], *staged[i % n]),
                                            2 * n),
            "gemm_us": timed_launches(torch, stream, lambda i: ext.fp4_gemm(xp, xs, *staged[i % n]), 2 * n),
        }
        row = {key: round(value * 1e6, 2) for key, value in times.items()}
        row["fp4_total_us"] = round(row["quantize_us"] + row["requantize_us"] + row["gemm_us"], 2)
        row["gemm_tflops"] = round(2 * tokens * m * k / (times["gemm_us"] * 1e12), 1)
        out[f"{m}x{k}"] = row
        del staged
        runtime.free(handles)
    print(json.dumps({"fp4_only": True, "tokens": tokens, "copies": args.layers, "shapes": out}), flush=True)
    return 0


def model_section(torch, args, model_name: str | None = None, context: int | None = None) -> dict:
    """Prefill tok/s at ``--prompt`` tokens (reference protocol, texelator/prefill.py:63-131) and
    graph-replayed greedy decode tok/s from the prompt up to ``context``, on a random-init BC4
    decoder of the 27B class (27b) or the 3B class (3b) whose linears are BC4-encoded by this build's
    encoder (``--model-weights uniform``: uniform random block bytes instead). If the prefill path
    fails the protocol's correctness gate, the failure is reported and the prefill is not timed."""
    from texelator_amd import modeling, prefill

    model_name = model_name or args.model
    context = context or args.context
    config = modeling.DecoderConfig.class_27b() if model_name == "27b" else modeling.DecoderConfig.qwen25_3b_style()
    model = modeling.BC4Decoder(config, max_context=context, seed=SEED, weights=args.model_weights)
    gate_failed = None
    try:
        try:
            pre = prefill.benchmark_prefill(model, tokens=args.prompt, warmup=2, runs=5)
        except prefill.GateFailed as error:
            log(str(error))
            pre, gate_failed = None, error.correctness
        dec = prefill.benchmark_decode(model, prompt_tokens=args.prompt, context=context)
    finally:
        model.close()
    bytes_per_token = config.bc4_bytes() + 2 * config.vocab * config.hidden
    weights = ("BC4-encoded (this build's PTQ encoder on the GPU) N(0, 0.02^2) weights, "
               f"{modeling.DISTINCT_LAYERS} distinct layer sets" if args.model_weights == "encoded"
               else "uniform random BC4 block bytes")
    out = {
        "config": model_name, "layers": config.layers, "hidden": config.hidden, "bc4_bytes": config.bc4_bytes(),
        "weights": args.model_weights,
        "prefill_tokens": args.prompt,
        "prefill_tok_s": round(pre["fused_bc4_mfma"]["gpu_tokens_per_second"], 1) if pre else None,
        "prefill_ms": round(pre["fused_bc4_mfma"]["gpu_seconds_median"] * 1e3, 2) if pre else None,
        "prefill_gemv_only_tok_s": round(pre["scalar_gemv"]["gpu_tokens_per_second"], 1) if pre else None,
        "prefill_correctness": pre["correctness"] if pre else gate_failed,
        "prefill_gate_failed": gate_failed is not None,
        "decode_context": [args.prompt, context],
        "decode_tok_s": round(dec["gpu_tokens_per_second"], 2),
        "decode_ms_per_token": round(dec["ms_per_token"], 3),
        "decode_timed_steps": dec["timed_steps"],
        "decode_per_bucket_tok_s": {k: round(v["tokens_per_second"], 2) for k, v in dec["per_bucket"].items()},
        "decode_weight_bytes_per_token": bytes_per_token,
        "data": f"random-init {weights} (GPT-2 depth-scaled init), uniform random prompt",
    }
    return out


def hf_section(torch, args) -> dict:
    """The 3B-class decoder through the reference's calling path: a Hugging Face Qwen2 with
    TexelatorLinear modules (``texelator_amd.hf.build_qwen2``), the reference's prefill protocol on
    it (``model.model(input_ids=...)``) and greedy ``model.generate`` of 256 tokens after a 512-token
    prompt, timed on the host clock (``hf.benchmark_generate``); then the same model decoding 256
    tokens through ``hf.GraphedGreedy`` (static cache, the library's attention, norms, fused gate/up
    SwiGLU GEMV, rotary embedding kernel, joined q|k|v GEMV with its biases in the epilogue, the
    attention's residual add in the post-attention norm, graph replays)."""
    from texelator_amd import hf, modeling, prefill
    from texelator_amd.runtime import free

    config = modeling.DecoderConfig.qwen25_3b_style()
    model, handles = hf.build_qwen2(config, seed=SEED, weights=args.model_weights)
    try:
        try:
            pre = prefill.benchmark_prefill(model, tokens=args.prompt, warmup=1, runs=3)
            gate_failed = None
        except prefill.GateFailed as error:
            log(str(error))
            pre, gate_failed = None, error.correctness
        gen = hf.benchmark_generate(model, prompt_tokens=args.prompt, new_tokens=256, runs=2)
        hf.use_texelator_norms(model)
        hf.use_texelator_residuals(model)
        hf.use_texelator_mlp(model)
        hf.use_texelator_rope(model)
        handles += hf.use_texelator_qkv(model)
        graphed = hf.GraphedGreedy(model, max_cache_len=args.prompt + 264).benchmark(args.prompt, 256)
    finally:
        free(handles)
        del model
        torch.cuda.empty_cache()
    return {
        "config": "3b", "path": "transformers Qwen2ForCausalLM + TexelatorLinear (install_standalone form)",
        "weights": args.model_weights,
        "prefill_tokens": args.prompt,
        "prefill_tok_s": round(pre["fused_bc4_mfma"]["gpu_tokens_per_second"], 1) if pre else None,
        "prefill_gemv_only_tok_s": round(pre["scalar_gemv"]["gpu_tokens_per_second"], 1) if pre else None,
        "prefill_correctness": pre["correctness"] if pre else gate_failed,
        "prefill_gate_failed": gate_failed is not None,
        "generate_new_tokens": gen["new_tokens"],
        "decode_tok_s": round(gen["decode_tok_s"], 2),
        "generate_tok_s": round(gen["generate_tok_s"], 2),
        "generate_seconds": round(gen["generate_seconds"], 3),
        "graphed_decode_tok_s": round(graphed["decode_tok_s"], 2),
        "graphed_path": "hf.GraphedGreedy: static KV cache, the library's attention and RMSNorm kernels "
                        "(hf.use_texelator_norms), the gate/up SwiGLU GEMV (hf.use_texelator_mlp), the rotary "
                        "embedding kernel (hf.use_texelator_rope), one GEMV over the joined q|k|v handle with the "
                        "biases in its epilogue (hf.use_texelator_qkv, tx_concat_rows + tx_linear_add_bias), the "
                        "attention's residual add fused into the post-attention norm and the MLP's into the down GEMV "
                        "(hf.use_texelator_residuals), one token's k/v appended to the static cache in one launch, "
                        "the one-token forward replayed from a HIP graph "
                        "(device clock)",
    }


def main() -> int:
    parser = argparse.ArgumentParser(description=__doc__.splitlines()[0])
    parser.add_argument("--gpus", type=int, default=1)
    parser.add_argument("--steps", type=int, default=200)
    parser.add_argument("--warmup", type=int, default=20)
    parser.add_argument("--layers", type=int, default=8, help="distinct layer copies swept per step")
    parser.add_argument("--lookahead", type=int, default=0, help="GEMV lookahead (0 = library default)")
    parser.add_argument("--cpu-runs", type=int, default=5, help="runs per CPU-baseline median")
    parser.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    parser.add_argument("--no-graph", action="store_true", help="launch eagerly instead of replaying a graph")
    parser.add_argument("--no-prefill", action="store_true", help="skip the prefill GEMM measurements")
    parser.add_argument("--model", choices=("27b", "3b", "none"), default="27b",
                        help="model-level decode/prefill tok/s on a random-init 27B- or 3B-class decoder")
    parser.add_argument("--context", type=int, default=4096, help="decode up to this context")
    parser.add_argument("--no-small-model", action="store_true",
                        help="skip the Qwen2.5-3B-style decoder after the 27B-class one")
    parser.add_argument("--prompt", type=int, default=512, help="prefill tokens")
    parser.add_argument("--model-weights", choices=("encoded", "uniform"), default="encoded",
                        help="BC4 data of the model-level decoders: encoded random-init weights or uniform bytes")
    parser.add_argument("--no-hf", action="store_true",
                        help="skip the Hugging Face (reference calling path) measurement of the 3B-class decoder")
    parser.add_argument("--hf-only", action="store_true",
                        help="run only the 3B model through Hugging Face modules (the model_3b_hf section)")
    parser.add_argument("--model-only", action="store_true",
                        help="profiling mode: only the model-level prefill and decode measurement (its JSON)")
    parser.add_argument("--prefill-only", action="store_true",
                        help="profiling mode: only the gate/up prefill GEMM at --prompt tokens over the layer copies")
    parser.add_argument("--tile", type=int, default=0, choices=range(0, 10),
                        help="with --prefill-only: prefill tile candidate 5..9 (0: the library's default)")
    parser.add_argument("--fp4-only", action="store_true",
                        help="only the FP4 hybrid prefill stages and the bf16 prefill on the reference's MLP "
                             "shapes at --prompt tokens (its JSON)")
    parser.add_argument("--kernel-only", action="store_true",
                        help="profiling mode: only the gate/up GEMV over the layer copies, then a plain copy of "
                             "COPY_BYTES bytes that calibrates the HBM byte counters")
    args = parser.parse_args()

    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) > 1:
        print("bench.py measures one GPU only: the BC4 GEMV path has no multi-GPU mode in this build "
              "(run with --gpus 1)", file=sys.stderr)
        return 2

    import torch

    from texelator_amd import hardware, runtime

    if not torch.cuda.is_available():
        print("bench.py needs a visible GPU", file=sys.stderr)
        return 1
    ext = runtime.extension()
    device = torch.device("cuda", 0)
    torch.cuda.set_device(device)

    if args.kernel_only:
        return kernel_only(torch, ext, runtime, hardware, device, args)
    if args.prefill_only:
        return prefill_only(torch, ext, runtime, hardware, device, args)
    if args.fp4_only:
        return fp4_only(torch, ext, runtime, hardware, device, args)
    if args.hf_only:
        print(json.dumps({"hf_only": True, "model_3b_hf": hf_section(torch, args)}), flush=True)
        return 0
    if args.model_only:
        print(json.dumps({"model_only": True, "model": model_section(torch, args)}), flush=True)
        return 0

    log("probing palette and encoding weights")
    lut = hardware.device_palette(device)
    unique = sorted({(m, k) for _, m, k in LAYER})
    weights = encoded_weights(torch, unique, lut)
    del lut

    log(f"packing {args.layers} layer copies")
    handles = []  # (name, m, k, handle)
    for _ in range(args.layers):
        for name, m, k in LAYER:
            blocks, scales = weights[(m, k)]
            (handle,) = runtime.pack_arrays(blocks, scales, lookahead=args.lookahead or 1)
            if args.lookahead:
                ext.set_lookahead(handle, args.lookahead)
            handles.append((name, m, k, handle))
    lookahead = ext.lookahead(handles[0][3])
    generator = torch.Generator(device="cuda").manual_seed(SEED + 1)
    xs = {k: torch.randn((1, k), device=device, generator=generator).to(torch.bfloat16) for k in (HIDDEN, INTER)}
    ys = [torch.empty((1, m), device=device, dtype=torch.float32) for _, m, _, _ in handles]
    step_bytes = sum(gemv_bytes(m, k) for _, m, k, _ in handles)

    def step():
        for (_, _, k, handle), y in zip(handles, ys):
            ext.linear_f32_into(handle, xs[k], y)

    stream = torch.cuda.Stream(device)
    graph = None
    with torch.cuda.stream(stream):
        step()
        torch.cuda.synchronize()
        if not args.no_graph:
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                step()
            torch.cuda.synchronize()
        run = graph.replay if graph is not None else step

        log(f"warmup {args.warmup} steps")
        for _ in range(args.warmup):
            run()
        torch.cuda.synchronize()

        log(f"timing {args.steps} steps")
        start = time.perf_counter()
        for _ in range(args.steps):
            run()
        torch.cuda.synchronize()
        elapsed = time.perf_counter() - start

        # Dominant kernel: back-to-back gate/up launches between two events on this stream,
        # queued behind a spin kernel so that host launch cost is hidden.
        dominant = [(h, y, k, m) for (name, m, k, h), y in zip(handles, ys) if name in DOMINANT]
        repeats = 8
        torch.cuda.synchronize()
        torch.cuda._sleep(20_000_000)
        begin = torch.cuda.Event(enable_timing=True)
        end = torch.cuda.Event(enable_timing=True)
        begin.record(stream)
        for _ in range(repeats):
            for h, y, k, _ in dominant:
                ext.linear_f32_into(h, xs[k], y)
        end.record(stream)
        torch.cuda.synchronize()
        launches = repeats * len(dominant)
        dominant_s = begin.elapsed_time(end) / 1e3 / launches

        # Per-shape averages, same method (reported for context).
        per_shape = {}
        for name, m, k in LAYER:
            group = [(h, y) for (n, _, _, h), y in zip(handles, ys) if n == name]
            torch.cuda._sleep(20_000_000)
            b = torch.cuda.Event(enable_timing=True)
            e = torch.cuda.Event(enable_timing=True)
            b.record(stream)
            for _ in range(repeats):
                for h, y in group:
                    ext.linear_f32_into(h, xs[k], y)
            e.record(stream)
            torch.cuda.synchronize()
            t = b.elapsed_time(e) / 1e3 / (repeats * len(group))
            per_shape[f"{name}_{k}x{m}"] = {"us": round(t * 1e6, 3), "GB/s": round(gemv_bytes(m, k) / t / 1e9, 1)}

    gate_m, gate_k = INTER, HIDDEN
    achieved = gemv_bytes(gate_m, gate_k) / dominant_s / 1e9
    value = step_bytes * args.steps / elapsed / 1e9
    result = {
        "metric": "BC4 GEMV GB/s (% HBM peak); decode tok/s; prefill tok/s @512 tokens",
        "value": round(value, 2),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(elapsed / args.steps * 1e3, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic: W~N(0,0.02^2)*LogNormal(0,0.3) per input channel, BC4-encoded on device; x~N(0,1) bf16",
        "config": {
            "workload": "decode GEMV sweep, batch 1, 27B-class shapes q,k,v,o 5120->5120/1024, "
                        "gate/up 5120->27648, down 27648->5120, fp32 outputs",
            "layers": args.layers,
            "linears_per_step": len(handles),
            "bytes_per_step": step_bytes,
            "graph": graph is not None,
            "lookahead": lookahead,
            "parallelism": "single GPU",
        },
        "roofline": {
            "bound": "hbm",
            "achieved": round(achieved, 1),
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": round(achieved / HBM_PEAK_GBS, 4),
            "traffic": read_traffic(),
            "kernel": "gemv 5120->27648 (gate/up)",
            "bytes_per_launch": gemv_bytes(gate_m, gate_k),
            "avg_launch_us": round(dominant_s * 1e6, 3),
        },
        "per_shape": per_shape,
    }
    log("streaming-read reference")
    result["hbm_stream_read"] = stream_read(torch, stream, args.layers)
    result["roofline"]["frac_of_stream_read"] = round(achieved / result["hbm_stream_read"]["GB/s"], 4)
    if not args.no_prefill:
        log("prefill GEMM")
        with torch.cuda.stream(stream):
            result["prefill"] = prefill_section(torch, ext, stream, handles)
    del graph
    runtime.free([h for _, _, _, h in handles])
    handles = []
    if args.model != "none":
        log(f"model-level tok/s ({args.model})")
        result["model"] = model_section(torch, args)
    if args.model == "27b" and not args.no_small_model:
        # the 3B-class decoder: 512-token prompt, then 256 greedy decode steps
        log("model-level tok/s (3b)")
        result["model_3b"] = model_section(torch, args, "3b", args.prompt + 256)
    if args.model != "none" and not args.no_hf:
        log("model-level tok/s (3b, Hugging Face calling path)")
        result["model_3b_hf"] = hf_section(torch, args)
    if "model" in result:
        # the metric's second and third figures (27B-class decoder), fully timed; a prefill that
        # fails the reference protocol's correctness gate is reported as failed, not timed
        result["prefill_tok_s_512"] = result["model"]["prefill_tok_s"]
        result["prefill_gate_failed"] = result["model"]["prefill_gate_failed"]
        result["decode_tok_s"] = result["model"]["decode_tok_s"]
    if not args.no_cpu:
        log("cpu baseline")
        result["cpu_baseline"] = cpu_baseline(weights, args.cpu_runs)
    else:
        result["cpu_baseline"] = None

    print(json.dumps(result), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
