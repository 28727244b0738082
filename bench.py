"""Benchmark of the exact-verify MTP hot path on one MI355X.

Default workload (``--workload mtp_round``): the full exact-verify MTP decode round of a random-init 9B-class qwen35
hybrid (32 layers: 24 Gated-DeltaNet + 8 GQA, hidden 4096, FFN 12288, vocab 248320, nextn draft block; every matrix
Q6_K with seeded weights) at context 4096 and 65536.  One step = one verify round (draft + 2-column verify + greedy
acceptance + GDN rollback, one hipGraph launch).  Per context: a non-MTP greedy run (the stream every MTP run must
reproduce bit for bit), then MTP runs with the draft forced to acceptance 0, 0.5 and 1.0.  The context state is
synthesized from a seed (KV cache fp16 N(0,1), GDN state N(0,0.05^2)) instead of prefilled.

``--workload verify_gemv``: the 2-column verify GEMV pair with both fused epilogues (up||gate 24576x4096 ncols=2,
then down 4096x12288 ncols=2 with residual + partials), >= 1 GiB of rotating weight replicas.

``--workload ingest``: the prompt-ingest leg alone (4096 seeded tokens at batch 16, in wide chunks of 1024; also part of
mtp_round's line), the workload of the ingest kernel trace.

Prints ONE JSON line.  For mtp_round, ``value`` is tok/s at context 4096 and acceptance 0.5; ``roofline`` is the
up||gate verify GEMV's algorithmic bytes / its mean launch time from HIP events on its launch stream (measured in the
same run); ``cpu_baseline`` is one verify round on this host's cores: the reference's CPU arithmetic as a SIMD
timing build (oracle/cpu_round.c), every GEMV shape, GDN layer and attention of the round timed as a leg and summed.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

METRIC = "MTP verify-round µs + tok/s (9B Q6_K, ctx 4K/64K); GEMV HBM GB/s % of peak"
HBM_PEAK_GBS = 8000.0

# config 2 shapes and their algorithmic bytes (weights once for both columns + activations + epilogue traffic)
UG_ROWS, UG_IN = 24576, 4096
DN_ROWS, DN_IN = 4096, 12288
Q6 = 210


def q6_bytes(rows, n_in):
    return rows * (n_in // 256) * Q6


UG_BYTES = q6_bytes(UG_ROWS, UG_IN) + 2 * (UG_IN // 32) * 36 + 2 * UG_ROWS * 4            # 82,781,184
DN_BYTES = (q6_bytes(DN_ROWS, DN_IN) + 2 * (DN_IN // 32) * 36 + 2 * DN_ROWS * 4 * 2
            + 2 * (DN_ROWS // 4) * 4)                                                       # 41,389,056
PAIR_BYTES = UG_BYTES + DN_BYTES                                                             # 124,170,240
# the round's up||gate kernel: GEMV + SwiGLU + Q8_1 in one launch (weights, Q8_1 in, Q8_1 out of the 12288 products)
UGS_BYTES = q6_bytes(UG_ROWS, UG_IN) + 2 * (UG_IN // 32) * 36 + 2 * (UG_ROWS // 2 // 32) * 36  # 82,612,224

# HBM traffic of one fused up||gate + SwiGLU ncols=2 launch: L2-to-memory request counts from two rocprofv3 --pmc passes
# over `bench.py --workload traffic_probe` (profiles/gemv_up_gate_swiglu_traffic.md).  On gfx950 a TCC_EA0_RDREQ that is
# not a 32-byte request moves 128 bytes (the same process's copy kernel reads 256 MiB in 2,097,401 requests), and a
# TCC_EA0_WRREQ is 64 bytes (TCC_EA0_WRREQ_64B) or 32.
PMC_UG_RDREQ, PMC_UG_RDREQ_32B = 648172, 0
PMC_UG_WRREQ, PMC_UG_WRREQ_64B = 768, 384


def ea_bytes(rdreq, rdreq_32b, wrreq, wrreq_64b):
    """HBM bytes from the TCC/EA request counters: 128-byte and 32-byte reads, 64-byte and 32-byte writes"""
    return 128 * (rdreq - rdreq_32b) + 32 * rdreq_32b + 64 * wrreq_64b + 32 * (wrreq - wrreq_64b)


UG_TRAFFIC_BYTES = ea_bytes(PMC_UG_RDREQ, PMC_UG_RDREQ_32B, PMC_UG_WRREQ, PMC_UG_WRREQ_64B)   # 83,002,880


def cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


# the 9B verify round's work at two columns: (n_in, n_out, residual, launches per round); the draft block adds one
# attention layer (qkv, out_proj, FFN), eh_proj and a second lm_head pass
ROUND_GEMVS = [(4096, 12352, False, 24), (4096, 10240, False, 9), (4096, 4096, True, 33), (4096, 24576, False, 33),
               (12288, 4096, True, 33), (8192, 4096, False, 1)]
LM_HEAD_ROWS, LM_HEAD_PASSES = 248320, 2
ROUND_GDN, ROUND_ATTN = 24, 9


def cpu_baseline(ctx: int = 4096, leg_s: float = 0.6):
    """The reference's CPU path for one verify round, restated as a SIMD timing build (oracle/cpu_round.c: AVX2 /
    AVX-512 VNNI integer dots, OpenMP), timed leg by leg on this host: each distinct GEMV shape of the round at two
    columns (the lm_head on a 24576-row slice, scaled by rows), the 2-token GDN layer and the 2-query attention at ctx,
    each repeated for ~leg_s; the round is the sum of legs times their launches per round.  Config 1 (Q6_K 12288x4096
    GEMV, one column, residual) is timed on all the threads and on one."""
    import numpy as np

    import oracle
    threads = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else os.cpu_count()
    threads = max(1, min(threads, 16))   # a one-GPU box's CPU share
    simd = oracle.cpr().cpr_simd_level()

    def timed(fn):
        fn()
        n, t0 = 0, time.perf_counter()
        while True:
            fn()
            n += 1
            el = time.perf_counter() - t0
            if el >= leg_s and n >= 2:
                return el / n

    t_start = time.perf_counter()
    legs, round_s = {}, 0.0
    for n_in, n_out, res, count in ROUND_GEMVS:
        w = oracle.gen_q6k(n_out, n_in, seed=n_in + n_out)
        xq = oracle.quantize_q8_1(oracle.normal(2 * n_in, seed=7), n_in, 2)
        r = oracle.normal(2 * n_out, seed=8) if res else None
        t = timed(lambda: oracle.cpr_q6k_gemv(w, xq, n_in, n_out, ncols=2, res=r, partials=res, threads=threads))
        legs[f"gemv {n_out}x{n_in}{' res' if res else ''} x{count}"] = round(t * 1e6, 1)
        round_s += count * t
        if (n_in, n_out) == (4096, 24576):   # the lm_head: the same rows of 4096, scaled to its 248320 rows
            t_head = t * LM_HEAD_ROWS / n_out
            legs[f"lm_head {LM_HEAD_ROWS}x4096 x{LM_HEAD_PASSES} (scaled from 24576 rows)"] = round(t_head * 1e6, 1)
            round_s += LM_HEAD_PASSES * t_head
        del w
    h_k, h_v, S = 16, 32, 128
    ch = (2 * h_k + h_v) * S
    stride = ch + h_v * S
    g = dict(qkvz=oracle.normal(2 * stride, seed=11), ab=oracle.normal(4 * h_v, seed=12),
             conv_w=oracle.normal(4 * ch, seed=13, std=0.5), dt=np.zeros(h_v, np.float32),
             ssm_a=(-np.exp(oracle.normal(h_v, seed=14, std=0.5))).astype(np.float32),
             gamma=(1 + oracle.normal(S, seed=15, std=0.1)).astype(np.float32),
             hist=oracle.normal(3 * ch, seed=16, std=0.5), state=oracle.normal(S * h_v * S, seed=17, std=0.05))
    t = timed(lambda: oracle.cpr_gdn_layer(g["qkvz"], stride, g["ab"], g["conv_w"], g["dt"], g["ssm_a"], g["gamma"],
                                           1e-6, g["hist"], g["state"], h_k, h_v, 2, threads=threads))
    legs[f"gdn layer 2 tokens x{ROUND_GDN}"] = round(t * 1e6, 1)
    round_s += ROUND_GDN * t
    kc = oracle.normal(ctx * 4 * 256, seed=18).astype(np.float16).view(np.uint16)
    vc = oracle.normal(ctx * 4 * 256, seed=19).astype(np.float16).view(np.uint16)
    q = oracle.normal(2 * 16 * 256, seed=20)
    t = timed(lambda: oracle.cpr_gqa_decode(q, kc, vc, 16, 4, 256, ctx - 2, 2, 1 / 16, threads=threads))
    legs[f"attention 2 queries ctx {ctx} x{ROUND_ATTN}"] = round(t * 1e6, 1)
    round_s += ROUND_ATTN * t
    # config 1: one column with the residual, all threads and one
    w = oracle.gen_q6k(12288, 4096, seed=21)
    xq = oracle.quantize_q8_1(oracle.normal(4096, seed=22), 4096, 1)
    r = oracle.normal(12288, seed=23)
    c1 = timed(lambda: oracle.cpr_q6k_gemv(w, xq, 4096, 12288, ncols=1, res=r, partials=True, threads=threads))
    c1_one = timed(lambda: oracle.cpr_q6k_gemv(w, xq, 4096, 12288, ncols=1, res=r, partials=True, threads=1))
    tok_round = tokens_for_rounds(ACCEPT_PATTERNS["0.5"], 20) / 20
    return {"value": round(tok_round / round_s, 4), "unit": "tok/s", "cores": threads, "kind": "port",
            "sample": f"one verify round of the 9B-class model at ctx {ctx}, acceptance 0.5 ({tok_round:.2f} tokens per "
                      "round), summed from legs timed on this host: every distinct GEMV shape at two columns, the GDN "
                      "layer and the attention, each repeated ~%.1f s (%.1f s in all)"
                      % (leg_s, time.perf_counter() - t_start),
            "us_per_round": round(round_s * 1e6, 1),
            "legs_us": legs,
            "cpu_model": cpu_model(),
            "simd": "avx512-vnni" if simd >= 2 else "avx2",
            "config1": {"workload": "Q6_K 12288x4096 GEMV, ncols=1, residual + partials",
                        "us": round(c1 * 1e6, 1), "GB_s": round(q6_bytes(12288, 4096) / c1 / 1e9, 2),
                        "us_1thread": round(c1_one * 1e6, 1),
                        "GB_s_1thread": round(q6_bytes(12288, 4096) / c1_one / 1e9, 2)}}


def run_verify_gemv(args):
    import torch

    import rapier_amd as rmi
    torch.cuda.set_device(0)
    stream = torch.cuda.Stream(device=0)          # explicit, default priority: the entry points reject NULL
    torch.cuda.set_stream(stream)

    # >= 1.2 GB of distinct weights so consecutive steps never re-read a cached replica
    reps = max(2, -(-1_200_000_000 // PAIR_BYTES))
    ug = [torch.empty(q6_bytes(UG_ROWS, UG_IN), dtype=torch.uint8, device="cuda") for _ in range(reps)]
    dn = [torch.empty(q6_bytes(DN_ROWS, DN_IN), dtype=torch.uint8, device="cuda") for _ in range(reps)]
    for i in range(reps):
        rmi.gen_q6_k(ug[i], UG_ROWS * UG_IN // 256, seed=1000 + i)
        rmi.gen_q6_k(dn[i], DN_ROWS * DN_IN // 256, seed=2000 + i)
    x_ug = torch.empty(2 * UG_IN, device="cuda")
    x_dn = torch.empty(2 * DN_IN, device="cuda")
    rmi.gen_normal(x_ug, x_ug.numel(), seed=3)
    rmi.gen_normal(x_dn, x_dn.numel(), seed=4)
    xq_ug = torch.empty(rmi.native_q8_1_bytes(UG_IN, 2), dtype=torch.uint8, device="cuda")
    xq_dn = torch.empty(rmi.native_q8_1_bytes(DN_IN, 2), dtype=torch.uint8, device="cuda")
    rmi.native_quantize_q8_1(x_ug, xq_ug, UG_IN, 2)
    rmi.native_quantize_q8_1(x_dn, xq_dn, DN_IN, 2)
    res = torch.empty(2 * DN_ROWS, device="cuda")
    rmi.gen_normal(res, res.numel(), seed=5)
    y_ug = torch.empty(2 * UG_ROWS, device="cuda")
    y_dn = torch.empty(2 * DN_ROWS, device="cuda")
    part = torch.empty(2 * (DN_ROWS // 4), device="cuda")

    def step(i, ev=None):
        r = i % reps
        if ev is not None:
            ev[0].record(stream)
        rmi.native_q6_k_mmvq(ug[r], xq_ug, y_ug, UG_IN, UG_ROWS, 2, stream)
        if ev is not None:
            ev[1].record(stream)
        rmi.native_q6_k_mmvq_res_n(dn[r], xq_dn, y_dn, res, part, DN_IN, DN_ROWS, 2, stream)

    for i in range(args.warmup):
        step(i)
    torch.cuda.synchronize()
    t_start, t_end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    t_start.record(stream)
    for i in range(args.steps):
        step(args.warmup + i)
    t_end.record(stream)
    torch.cuda.synchronize()
    total_ms = t_start.elapsed_time(t_end)
    ms_per_step = total_ms / args.steps
    value = PAIR_BYTES / (ms_per_step * 1e-3) / 1e9


    # roofline leg: the round's up||gate kernel (GEMV + SwiGLU + Q8_1, one launch) on SwiGLU-packed (wave-tiled)
    # copies of the up||gate replicas, as the engine packs them.  Blocks of back-to-back launches over the rotating
    # replicas, one HIP event pair per block on the launch stream (per-launch event pairs would add the event's own
    # cost to every launch).
    ugp = [torch.empty(rmi.q6_k_packed_bytes(UG_IN, UG_ROWS), dtype=torch.uint8, device="cuda") for _ in range(reps)]
    for i in range(reps):
        rmi.q6_k_pack_swiglu(ug[i], ugp[i], UG_IN, UG_ROWS // 2, stream)
    q_ug = torch.empty(rmi.native_q8_1_bytes(UG_ROWS // 2, 2), dtype=torch.uint8, device="cuda")
    for i in range(reps):
        rmi.native_q6_k_swiglu_packed(ugp[i], xq_ug, q_ug, UG_IN, UG_ROWS // 2, 2, stream)
    blocks, per_block = 5, 2 * reps
    evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(blocks)]
    torch.cuda.synchronize()
    for b in range(blocks):
        evs[b][0].record(stream)
        for i in range(per_block):
            rmi.native_q6_k_swiglu_packed(ugp[i % reps], xq_ug, q_ug, UG_IN, UG_ROWS // 2, 2, stream)
        evs[b][1].record(stream)
    torch.cuda.synchronize()
    ug_us = sorted(a.elapsed_time(b) * 1e3 / per_block for a, b in evs)
    ug_mean_us = sum(ug_us) / len(ug_us)
    achieved = UGS_BYTES / (ug_mean_us * 1e-6) / 1e9
    del ugp
    c1 = run_config1(stream, blocks=5)

    # the same pair through the same entry points once native_q6_k_pack has given every replica a library-owned
    # packed copy (the reference's opt-in registry, mmvq:2930-2960, looked up at mmvq:3629): the packed kernels, the
    # same bits (timed after the other legs, which it leaves as they were)
    for i in range(reps):
        assert rmi.native_q6_k_pack(ug[i], UG_IN, UG_ROWS) and rmi.native_q6_k_pack(dn[i], DN_IN, DN_ROWS)
    for i in range(args.warmup):
        step(i)
    torch.cuda.synchronize()
    t_start.record(stream)
    for i in range(args.steps):
        step(args.warmup + i)
    t_end.record(stream)
    torch.cuda.synchronize()
    reg_ms_per_step = t_start.elapsed_time(t_end) / args.steps
    for i in range(reps):
        rmi.native_q6_k_unpack(ug[i])
        rmi.native_q6_k_unpack(dn[i])
    del ug, dn
    out = {
        "metric": METRIC,
        "value": round(value, 1),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "int8 dot, f32 accumulate",
        "data": "synthetic (seeded Q6_K weights per config: codes U{0..63}, sc U[-32,31], d=|N(0,1e-3)|; N(0,1) "
                "activations and residuals)",
        "config": {
            "workload": "2-column verify GEMV pair: up||gate Q6_K 24576x4096 ncols=2, then down Q6_K 4096x12288 "
                        "ncols=2 with fused residual + sum-of-squares partials",
            "algorithmic_bytes_per_step": PAIR_BYTES,
            "us_per_pair": round(ms_per_step * 1e3, 2),
            "hbm_frac_of_peak": round(value / HBM_PEAK_GBS, 4),
            "registry_packed_us_per_pair": round(reg_ms_per_step * 1e3, 2),
            "registry_packed_hbm_frac_of_peak": round(PAIR_BYTES / (reg_ms_per_step * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
            "weight_replicas": reps,
            "rotated_bytes": reps * (q6_bytes(UG_ROWS, UG_IN) + q6_bytes(DN_ROWS, DN_IN)),
            "config1": c1,
        },
        "roofline": {
            "kernel": "q6k_packed_swiglu<2, 8, 4, 2, false> (up||gate 24576x4096 GEMV + SwiGLU + Q8_1, ncols=2, "
                      "SwiGLU-packed wave-tile layout; 192 workgroups of 8 waves, two 32-output groups each)",
            "bound": "hbm",
            "achieved": round(achieved, 1),
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": round(achieved / HBM_PEAK_GBS, 4),
            "traffic": UG_TRAFFIC_BYTES,
            "traffic_over_algorithmic": round(UG_TRAFFIC_BYTES / UGS_BYTES, 4),
            "algorithmic_bytes_per_launch": UGS_BYTES,
            "mean_launch_us": round(ug_mean_us, 3),
            "launches_timed": blocks * per_block,
        },
    }
    return out


# config 1: Q6_K 12288 x 4096, one column, residual + partials; algorithmic bytes = weights + Q8_1 x + res read +
# y write + partials
C1_ROWS, C1_IN = 12288, 4096
C1_BYTES = q6_bytes(C1_ROWS, C1_IN) + (C1_IN // 32) * 36 + 2 * C1_ROWS * 4 + (C1_ROWS // 4) * 4   # 41,402,880


def run_config1(stream, blocks=5):
    """config 1 on the GPU: the drop-in residual GEMV on GGUF blocks (rmi_native_q6_k_mmvq_res, the reference's call)
    and on the engine's packed copy, over >= 1.2 GB of rotating replicas, one HIP event pair per block of launches"""
    import torch

    import rapier_amd as rmi
    reps = max(2, -(-1_200_000_000 // q6_bytes(C1_ROWS, C1_IN)))
    ws = [torch.empty(q6_bytes(C1_ROWS, C1_IN), dtype=torch.uint8, device="cuda") for _ in range(reps)]
    for i in range(reps):
        rmi.gen_q6_k(ws[i], C1_ROWS * C1_IN // 256, seed=4000 + i)
    x = torch.empty(C1_IN, device="cuda")
    rmi.gen_normal(x, C1_IN, seed=41)
    xq = torch.empty(rmi.native_q8_1_bytes(C1_IN, 1), dtype=torch.uint8, device="cuda")
    rmi.native_quantize_q8_1(x, xq, C1_IN, 1)
    y = torch.empty(C1_ROWS, device="cuda")
    rmi.gen_normal(y, C1_ROWS, seed=42)
    part = torch.empty(C1_ROWS // 4, device="cuda")

    def time_it(fn):
        for i in range(reps):
            fn(i)
        evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(blocks)]
        torch.cuda.synchronize()
        for b in range(blocks):
            evs[b][0].record(stream)
            for i in range(2 * reps):
                fn(i % reps)
            evs[b][1].record(stream)
        torch.cuda.synchronize()
        return sum(a.elapsed_time(b) * 1e3 / (2 * reps) for a, b in evs) / blocks

    gguf_us = time_it(lambda i: rmi.native_q6_k_mmvq_res(ws[i], xq, y, y, part, C1_IN, C1_ROWS, stream))
    wp = [torch.empty(rmi.q6_k_packed_bytes(C1_IN, C1_ROWS), dtype=torch.uint8, device="cuda") for _ in range(reps)]
    for i in range(reps):
        rmi.q6_k_pack(ws[i], wp[i], C1_IN, C1_ROWS, stream)
    packed_us = time_it(lambda i: rmi.native_q6_k_mmvq_packed_res_n(wp[i], xq, y, y, part, C1_IN, C1_ROWS, 1, stream))
    del wp
    for i in range(reps):   # the reference's call again, on library-owned packed copies (native_q6_k_pack)
        assert rmi.native_q6_k_pack(ws[i], C1_IN, C1_ROWS)
    reg_us = time_it(lambda i: rmi.native_q6_k_mmvq_res(ws[i], xq, y, y, part, C1_IN, C1_ROWS, stream))
    for i in range(reps):
        rmi.native_q6_k_unpack(ws[i])
    del ws
    return {"workload": "config 1: Q6_K 12288x4096 GEMV, ncols=1, residual + partials (y aliases res)",
            "algorithmic_bytes": C1_BYTES,
            "gguf_layout_us": round(gguf_us, 2), "gguf_layout_GB_s": round(C1_BYTES / gguf_us / 1e3, 1),
            "registry_packed_us": round(reg_us, 2), "registry_packed_GB_s": round(C1_BYTES / reg_us / 1e3, 1),
            "packed_us": round(packed_us, 2), "packed_GB_s": round(C1_BYTES / packed_us / 1e3, 1)}


def run_traffic_probe():
    """Workload for the rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE passes: one fused up||gate + SwiGLU ncols=2 launch
    (SwiGLU-packed weights) after a 1 GiB
    fill has evicted L2 and the Infinity Cache, then a copy-like kernel of known size (reads 256 MiB, writes
    256 MiB) that calibrates both counters in the same process."""
    import torch

    import rapier_amd as rmi
    torch.cuda.set_device(0)
    stream = torch.cuda.Stream(device=0)
    torch.cuda.set_stream(stream)
    wg = torch.empty(q6_bytes(UG_ROWS, UG_IN), dtype=torch.uint8, device="cuda")
    rmi.gen_q6_k(wg, UG_ROWS * UG_IN // 256, seed=1)
    w = torch.empty(rmi.q6_k_packed_bytes(UG_IN, UG_ROWS), dtype=torch.uint8, device="cuda")
    rmi.q6_k_pack_swiglu(wg, w, UG_IN, UG_ROWS // 2, stream)
    del wg
    x = torch.empty(2 * UG_IN, device="cuda")
    rmi.gen_normal(x, x.numel(), seed=2)
    xq = torch.empty(rmi.native_q8_1_bytes(UG_IN, 2), dtype=torch.uint8, device="cuda")
    rmi.native_quantize_q8_1(x, xq, UG_IN, 2)
    y = torch.empty(rmi.native_q8_1_bytes(UG_ROWS // 2, 2), dtype=torch.uint8, device="cuda")
    a = torch.ones(COPY_KIB_ELEMS, device="cuda")
    b = torch.empty_like(a)
    junk = torch.empty(256 * 1024 * 1024, device="cuda")
    torch.cuda.synchronize()
    junk.fill_(1.0)
    torch.cuda.synchronize()
    rmi.native_q6_k_swiglu_packed(w, xq, y, UG_IN, UG_ROWS // 2, 2, stream)
    torch.cuda.synchronize()
    junk.fill_(2.0)
    torch.cuda.synchronize()
    torch.add(a, 1.0, out=b)
    torch.cuda.synchronize()
    print(json.dumps({"workload": "traffic_probe", "gemv_launches": 1, "copy_read_bytes": a.numel() * 4,
                      "copy_write_bytes": b.numel() * 4}), flush=True)


COPY_KIB_ELEMS = 64 * 1024 * 1024   # floats: the probe's copy kernel reads 256 MiB and writes 256 MiB

# the round's Q6_K GEMVs at two columns, as the engine launches them on its packed copies: (name, n_in, n_out, kind,
# launches per round); kind "res" = residual + partials epilogue, "swiglu" = up||gate + SwiGLU + Q8_1 (n_out = 2 ff)
ROUND_KERNEL_GEMVS = [
    ("gdn in_proj qkv|z|beta|alpha", 4096, 12352, "plain", 24),
    ("attn qkv", 4096, 10240, "plain", 9),
    ("out_proj (ssm_out / wo)", 4096, 4096, "res", 33),
    ("up||gate + SwiGLU", 4096, 24576, "swiglu", 33),
    ("ffn down", 12288, 4096, "res", 33),
    ("draft eh_proj", 8192, 4096, "plain", 1),
    ("lm_head", 4096, 248320, "plain", 2),
]


def gemv_algorithmic_bytes(n_in, n_out, kind, ncols=2):
    """weights once + Q8_1 inputs + outputs (fp32 rows, or the Q8_1 of the ff SwiGLU products) + the residual read
    and 4-row partials of a residual GEMV"""
    b = q6_bytes(n_out, n_in) + ncols * (n_in // 32) * 36
    if kind == "swiglu":
        return b + ncols * (n_out // 2 // 32) * 36
    b += ncols * n_out * 4
    if kind == "res":
        b += ncols * n_out * 4 + ncols * (n_out // 4) * 4
    return b


def time_blocks(stream, launch, nrot, blocks=5, per_block=None):
    """mean launch time (us) from HIP events around blocks of back-to-back launches over nrot rotating buffer sets"""
    import torch
    per_block = per_block or max(2 * nrot, 20)
    for r in range(nrot):
        launch(r)
    evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(blocks)]
    torch.cuda.synchronize()
    for b in range(blocks):
        evs[b][0].record(stream)
        for i in range(per_block):
            launch(i % nrot)
        evs[b][1].record(stream)
    torch.cuda.synchronize()
    return sum(a.elapsed_time(b) * 1e3 / per_block for a, b in evs) / blocks, blocks * per_block


def time_graph(stream, launch, nrot, blocks=5):
    """mean launch time (us) of back-to-back launches over nrot rotating buffer sets, captured once into a HIP graph
    and replayed (the launches of a round are graph nodes too; a host loop of ctypes calls would time the host for
    kernels of a few microseconds)"""
    import torch
    for r in range(nrot):
        launch(r)
    torch.cuda.synchronize()
    per_graph = 2 * nrot
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        for i in range(per_graph):
            launch(i % nrot)
    g.replay()
    torch.cuda.synchronize()
    evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(blocks)]
    for b in range(blocks):
        evs[b][0].record(stream)
        g.replay()
        evs[b][1].record(stream)
    torch.cuda.synchronize()
    return sum(a.elapsed_time(b) * 1e3 / per_graph for a, b in evs) / blocks, blocks * per_graph


def time_read_ref(stream, nbytes):
    """the single-launch streaming-read reference for nbytes (rmi_stream_read, rotating replicas >= 1 GB), best of a
    few grids: what one kernel that only reads those bytes takes here, launch and ramp included"""
    import torch

    import rapier_amd as rmi
    nbytes = nbytes // 16 * 16
    nrot = max(2, -(-1_000_000_000 // nbytes))
    bufs = [torch.full((nbytes,), r, dtype=torch.uint8, device="cuda") for r in range(nrot)]
    out = torch.zeros(1, dtype=torch.int32, device="cuda")
    best = None
    for grid in (512, 1024, 2048, 4096):
        us, _ = time_blocks(stream, lambda r: rmi.stream_read(bufs[r], nbytes, grid, out, stream), nrot, blocks=3)
        if best is None or us < best[0]:
            best = (us, grid)
    del bufs
    return best


def time_gdn_layer(stream):
    """the verify round's GDN layer launch (rmi_gdn_layer_tokens_x, 2 tokens: conv + SiLU + L2, delta-rule step, RMSNorm
    * SiLU gate, Q8_1; after-token-0 state to the rollback buffer) at the 9B shapes, rotating over 80 layers' state
    (320 MB, above the Infinity Cache).  Algorithmic bytes: state read + state written twice + history and conv taps
    + inputs + y and its Q8_1."""
    import torch

    import rapier_amd as rmi
    h_k, h_v, S = 16, 32, 128
    ch = 2 * h_k * S + h_v * S
    stride = ch + h_v * S + 2 * h_v                    # the engine's in_proj rows: q|k|v|z|beta|alpha
    nrot = 80
    st = torch.empty(nrot, 2, S * h_v * S, device="cuda")
    rmi.gen_normal(st, st.numel(), seed=31, std=0.05)
    hist = torch.empty(nrot, 2, h_v * 3 * S * 3, device="cuda")
    rmi.gen_normal(hist, hist.numel(), seed=32, std=0.5)
    proj = torch.empty(2 * stride, device="cuda")
    rmi.gen_normal(proj, proj.numel(), seed=33)
    conv_w = torch.empty(4 * ch, device="cuda")
    rmi.gen_normal(conv_w, conv_w.numel(), seed=34, std=0.5)
    dt = torch.zeros(h_v, device="cuda")
    ssm_a = -torch.ones(h_v, device="cuda")
    gamma = torch.ones(S, device="cuda")
    sel = torch.zeros(1, dtype=torch.int32, device="cuda")
    y = torch.empty(2 * h_v * S, device="cuda")
    q8b = rmi.native_q8_1_bytes(h_v * S, 1)
    q8 = torch.empty(2 * q8b, dtype=torch.uint8, device="cuda")

    xch = torch.zeros(rmi.gdn_exchange_bytes(h_v), dtype=torch.uint8, device="cuda")

    def launch(r):
        rmi.gdn_layer_tokens_x(st[r, 0], st[r, 1], hist[r, 0], hist[r, 1], sel, proj, stride, proj[ch + h_v * S:],
                               stride, conv_w, dt, ssm_a, gamma, 1e-6, y, h_v * S, q8, q8b, h_k, h_v, 2, xch, stream)

    us, n = time_graph(stream, launch, nrot)
    state = S * h_v * S * 4
    nbytes = 3 * state + 2 * 2 * h_v * 3 * S * 3 * 4 + 4 * ch * 4 + 2 * stride * 4 + 2 * (h_v * S * 4 + q8b)
    return {"kernel": "gdn layer, 2 tokens (rmi_gdn_layer_tokens_x: four workgroups per value head)", "per_round": ROUND_GDN, "algorithmic_bytes": nbytes,
            "us": round(us, 3), "GB_s": round(nbytes / us / 1e3, 1), "launches_timed": n}


def time_attention(stream, ctx):
    """the verify round's attention launch pair as the engine runs it (rmi_gqa_flash_decode_prep: the per-head norm,
    RoPE and the new K / V rows in the split-K partial, then the merge with the sigmoid gate and Q8_1) for 2 queries at
    positions ctx - 2, ctx - 1 over a fp16 KV cache of the 9B shapes (4 KV heads x 256), with the engine's chunk size
    (a full cache is one partial workgroup per CU), rotating over enough caches to exceed the Infinity Cache.
    Algorithmic bytes: K + V rows read once."""
    import torch

    import rapier_amd as rmi
    n_head, n_kv, hd = 16, 4, 256
    max_ctx = ctx + 512
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    chunks = max(1, cus // n_kv)
    nsub = max(2, min(64, -(-max_ctx // (64 * chunks))))
    row = n_kv * hd
    nrot = max(2, -(-400_000_000 // (2 * max_ctx * row * 2)))
    kv = torch.empty(nrot, 2, max_ctx * row, dtype=torch.float16, device="cuda")
    rmi.gen_normal_f16(kv, kv.numel(), seed=41)
    q3_stride = 2 * n_head * hd + 2 * row   # per token [n_head x (q | gate) | k | v], the qkv GEMV's output
    q3 = torch.empty(2 * q3_stride, device="cuda")
    rmi.gen_normal(q3, q3.numel(), seed=42)
    qn = torch.ones(hd, device="cuda")
    kn = torch.ones(hd, device="cuda")
    pos = torch.tensor([ctx - 2], dtype=torch.int32, device="cuda")
    yb = torch.empty(2 * n_head * hd, device="cuda")
    q8b = rmi.native_q8_1_bytes(n_head * hd, 1)
    q8 = torch.empty(2 * q8b, dtype=torch.uint8, device="cuda")
    ws = torch.empty(rmi.gqa_workspace_bytes(max_ctx, n_kv, nsub), dtype=torch.uint8, device="cuda")

    def launch(r):
        rmi.gqa_flash_decode_prep(q3, q3_stride, qn, kn, kv[r, 0], kv[r, 1], pos, yb, n_head * hd, q8, q8b, ws,
                                  n_head, n_kv, hd, 64, 1e7, 1.0, 4096.0, 1e-6, 2, max_ctx, nsub, 1.0 / 16,
                                  stream=stream)

    us, n = time_graph(stream, launch, nrot)
    nbytes = 2 * ctx * row * 2
    return {"kernel": f"attention, 2 queries, ctx {ctx} (rmi_gqa_flash_decode_prep: norm + RoPE + partial, then "
                      f"merge; nsub {nsub})",
            "per_round": ROUND_ATTN, "algorithmic_bytes": nbytes, "us": round(us, 3),
            "GB_s": round(nbytes / us / 1e3, 1), "frac": round(nbytes / us / 1e3 / HBM_PEAK_GBS, 4),
            "launches_timed": n}


def run_kernels(args):
    """Each GEMV shape of the verify round at two columns, on the packed layout the engine runs, over >= 1 GB of
    rotating replicas (so no launch finds its weights in the 256 MB Infinity Cache): mean launch time from HIP events
    around blocks of back-to-back launches, algorithmic GB/s and fraction of peak.  Also the workload of the rocprofv3
    counter passes over the same kernels."""
    import torch

    import rapier_amd as rmi
    torch.cuda.set_device(0)
    stream = torch.cuda.Stream(device=0)
    torch.cuda.set_stream(stream)
    only = set(args.shapes.split(",")) if args.shapes else None
    out = []
    for i_shape, (name, n_in, n_out, kind, per_round) in enumerate(ROUND_KERNEL_GEMVS):
        if only is not None and str(i_shape) not in only:
            continue
        wbytes = q6_bytes(n_out, n_in)
        reps = max(2, -(-1_000_000_000 // wbytes))
        src = torch.empty(wbytes, dtype=torch.uint8, device="cuda")
        wp = []
        for r in range(reps):
            rmi.gen_q6_k(src, n_out * n_in // 256, seed=7000 + 31 * i_shape + r)
            w = torch.empty(rmi.q6_k_packed_bytes(n_in, n_out), dtype=torch.uint8, device="cuda")
            if kind == "swiglu":
                rmi.q6_k_pack_swiglu(src, w, n_in, n_out // 2, stream)
            else:
                rmi.q6_k_pack(src, w, n_in, n_out, stream)
            wp.append(w)
        del src
        x = torch.empty(2 * n_in, device="cuda")
        rmi.gen_normal(x, x.numel(), seed=11 + i_shape)
        xq = torch.empty(rmi.native_q8_1_bytes(n_in, 2), dtype=torch.uint8, device="cuda")
        rmi.native_quantize_q8_1(x, xq, n_in, 2, stream)
        y = torch.empty(2 * n_out, device="cuda")
        rmi.gen_normal(y, y.numel(), seed=12 + i_shape)
        part = torch.empty(2 * (n_out // 4), device="cuda")
        yq = torch.empty(rmi.native_q8_1_bytes(max(n_out // 2, 32), 2), dtype=torch.uint8, device="cuda")

        def launch(r):
            if kind == "swiglu":
                rmi.native_q6_k_swiglu_packed(wp[r], xq, yq, n_in, n_out // 2, 2, stream)
            elif kind == "res":
                rmi.native_q6_k_mmvq_packed_res_n(wp[r], xq, y, y, part, n_in, n_out, 2, stream)
            else:
                rmi.native_q6_k_mmvq_packed(wp[r], xq, y, n_in, n_out, 2, stream)

        for r in range(reps):
            launch(r)
        blocks, per_block = 5, max(2 * reps, 20)
        evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(blocks)]
        torch.cuda.synchronize()
        for b in range(blocks):
            evs[b][0].record(stream)
            for i in range(per_block):
                launch(i % reps)
            evs[b][1].record(stream)
        torch.cuda.synchronize()
        us = sum(a.elapsed_time(b) * 1e3 / per_block for a, b in evs) / blocks
        nbytes = gemv_algorithmic_bytes(n_in, n_out, kind)
        del wp
        torch.cuda.synchronize()
        ref_us, ref_grid = time_read_ref(stream, nbytes)
        row = {"gemv": name, "n_in": n_in, "n_out": n_out, "kind": kind, "per_round": per_round,
               "algorithmic_bytes": nbytes, "us": round(us, 3), "GB_s": round(nbytes / us / 1e3, 1),
               "frac": round(nbytes / us / 1e3 / HBM_PEAK_GBS, 4), "launches_timed": blocks * per_block,
               "read_ref_us": round(ref_us, 3), "read_ref_grid": ref_grid, "over_read_ref": round(us / ref_us, 3)}
        out.append(row)
        print(json.dumps(row), file=sys.stderr, flush=True)
    others = []
    n = len(ROUND_KERNEL_GEMVS)
    if only is None or str(n) in only:
        others.append(time_gdn_layer(stream))
    for i, ctx in enumerate((4096, 65536)):
        if only is None or str(n + 1 + i) in only:
            others.append(time_attention(stream, ctx))
    for r in others:
        print(json.dumps(r), file=sys.stderr, flush=True)
    tot_us = sum(r["us"] * r["per_round"] for r in out)
    tot_b = sum(r["algorithmic_bytes"] * r["per_round"] for r in out)
    print(json.dumps({"workload": "kernels", "gemvs": out, "others": others,
                      "round_gemv_us": round(tot_us, 1), "round_gemv_bytes": tot_b,
                      "round_gemv_frac": round(tot_b / tot_us / 1e3 / HBM_PEAK_GBS, 4) if tot_us else None}),
          flush=True)

ACCEPT_PATTERNS = {"0": [0], "0.5": [1, 0], "1.0": [1]}


def gdn_timeouts():
    import rapier_amd as rmi
    return int(rmi.gdn_exchange_timeouts())


def tokens_for_rounds(pattern, rounds):
    """tokens a forced run emits in exactly `rounds` rounds (2 per accepted round, 1 per rejected)."""
    return sum(2 if pattern[r % len(pattern)] else 1 for r in range(rounds))


def run_mtp_rounds(args, contexts=(4096, 65536)):
    import torch

    import rapier_amd.engine as E
    torch.cuda.set_device(0)
    stream = torch.cuda.Stream(device=0)
    torch.cuda.set_stream(stream)
    K, W = args.steps, args.warmup
    table, identical, info = {}, True, None
    for ctx in contexts:
        n_tok = tokens_for_rounds([1], K)          # greedy reference length covers every forced run
        eng = E.Engine(E.qwen35_9b_config(), seed=2024, max_ctx=ctx + 2 * (K + W) + 256, stream=stream)
        info = eng.info()
        first = eng.synth_context(ctx, seed=ctx, last_token=1000)
        pos0, cur0 = eng.state()
        eng.save_state()
        eng.generate(max(W, 1), mode=E.GREEDY)      # warm the single-token graph
        eng.restore_state(pos0, cur0)
        ref, st_g = eng.generate(n_tok, mode=E.GREEDY)
        row = {"greedy": {"tok_s": round(n_tok / (st_g["gpu_ms"] / 1e3), 2),
                          "ms_per_token": round(st_g["gpu_ms"] / n_tok, 4), "tokens": n_tok}}
        for name, pat in ACCEPT_PATTERNS.items():
            eng.restore_state(pos0, cur0)
            if W:
                eng.generate(tokens_for_rounds(pat, W), mode=E.MTP_FORCED, ref_tokens=ref, ref_base=pos0 + 1,
                             pattern=pat)                                  # untimed warmup rounds (graph capture)
                eng.restore_state(pos0, cur0)
            n = tokens_for_rounds(pat, K)
            toks, st = eng.generate(n, mode=E.MTP_FORCED, ref_tokens=ref, ref_base=pos0 + 1, pattern=pat)
            same = toks == ref[:n]
            identical &= same
            row[name] = {"us_per_round": round(st["gpu_ms"] * 1e3 / st["rounds"], 2),
                         "tok_s": round(n / (st["gpu_ms"] / 1e3), 2), "rounds": st["rounds"],
                         "accepted": st["accepted"], "tokens": n, "stream_identical": same}
        table[str(ctx)] = row
        eng.close()
        del eng
        torch.cuda.synchronize()
    return table, identical, info


def run_round(args):
    """Verify rounds only, at the first context of --ctx and forced acceptance 0.5: the workload of the whole-round
    counter passes (HBM bytes per round) and of quick round timings.  The greedy stream is generated first, as every
    forced MTP run needs it, and the MTP stream is checked against it."""
    import torch

    import rapier_amd.engine as E
    torch.cuda.set_device(0)
    stream = torch.cuda.Stream(device=0)
    torch.cuda.set_stream(stream)
    ctx = int(args.ctx.split(",")[0])
    K, W = args.steps, args.warmup
    pat = ACCEPT_PATTERNS["0.5"]
    eng = E.Engine(E.qwen35_9b_config(), seed=2024, max_ctx=ctx + 2 * (K + W) + 256, stream=stream)
    info = eng.info()
    eng.synth_context(ctx, seed=ctx, last_token=1000)
    pos0, cur0 = eng.state()
    eng.save_state()
    ref, _ = eng.generate(tokens_for_rounds([1], K + W), mode=E.GREEDY)
    eng.restore_state(pos0, cur0)
    if W:
        eng.generate(tokens_for_rounds(pat, W), mode=E.MTP_FORCED, ref_tokens=ref, ref_base=pos0 + 1, pattern=pat)
        eng.restore_state(pos0, cur0)
    n = tokens_for_rounds(pat, K)
    toks, st = eng.generate(n, mode=E.MTP_FORCED, ref_tokens=ref, ref_base=pos0 + 1, pattern=pat)
    eng.close()
    torch.cuda.synchronize()
    us = st["gpu_ms"] * 1e3 / st["rounds"]
    print(json.dumps({"workload": "round", "ctx": ctx, "rounds": st["rounds"], "us_per_round": round(us, 2),
                      "tok_s": round(n / (st["gpu_ms"] / 1e3), 2), "stream_identical": toks == ref[:n],
                      "round_weight_bytes": info["round_weight_bytes"], "kv_bytes_per_pos": info["kv_bytes_per_pos"],
                      "gdn_exchange_timeouts": gdn_timeouts()}),
          flush=True)


def run_ingest(n_prompt=4096, batch=16, n_check=93):
    """Prompt ingest on the 9B-class model: n_prompt seeded random tokens from position 0 at the largest batch, which runs
    them in wide chunks of up to 1024 tokens (one weight pass per chunk), timed by the host clock around the call (token
    upload, chunks, the final sync).  The token-by-token path is timed on the first n_check tokens.  The state the two paths
    leave is compared behind two ingests of n_check tokens: one wide chunk, and (n_check // 3 at a time, too short for one)
    16-token chunks on the chunk graph with their tail."""
    import numpy as np
    import torch

    import rapier_amd.engine as E
    stream = torch.cuda.Stream(device=0)
    torch.cuda.set_stream(stream)
    eng = E.Engine(E.qwen35_9b_config(), seed=2024, max_ctx=n_prompt + 256, stream=stream)
    prompt = [int(t) for t in np.random.default_rng(4096).integers(0, 248320, size=n_prompt)]
    eng.prefill(prompt[:2 * n_check], batch=batch)               # the kernels' first launches
    t0 = time.perf_counter()
    eng.prefill(prompt, batch=batch)
    dt = time.perf_counter() - t0
    t1 = time.perf_counter()
    first1 = eng.prefill(prompt[:n_check], batch=1)
    dt1 = time.perf_counter() - t1
    h1 = eng.read(E.BUF_HIDDEN, 0, 4 * 4096)
    same = True
    for step in (n_check, n_check // 3):
        eng.reset()
        for i in range(0, n_check, step):
            first = eng.ingest(prompt[i:min(i + step, n_check)], batch=batch)
        same = same and first == first1 and np.array_equal(h1, eng.read(E.BUF_HIDDEN, 0, 4 * 4096))
    eng.close()
    torch.cuda.synchronize()
    chunks = (n_prompt + 1023) // 1024
    return {"prompt_tokens": n_prompt, "batch": batch, "tok_s": round(n_prompt / dt, 1),
            "chunks": chunks, "ms_per_chunk": round(dt * 1e3 / chunks, 3),
            "per_token_tok_s": round(n_check / dt1, 1),
            "identical_to_per_token": bool(same),
            "note": "host clock around rmi_engine_prefill_batch, chunks of up to 1024 tokens; per-token path timed on the "
                    f"first {n_check} tokens; identical = first token and final hidden bit-equal after {n_check} tokens, "
                    "ingested as one wide chunk and in 16-token chunks"}


def qwen35_9b_tensors(plan="q6_k"):
    """(name, ggml type, dims) of a 9B-class qwen35 GGUF with the reference's tensor names (qw:2003-2127).
    plan "q6_k": every matrix Q6_K.  plan "q5_k_m": a Q5_K_M-like mix (llama.cpp's rule for that file type): Q5_K
    matrices and token table, Q6_K output, attn_v and ffn_down Q6_K in the first and last eighth of the layers and in
    every third layer between, Q5_K elsewhere - so q|k|v groups mix types in those layers."""
    E, F, V, NL, HK, HV, NH, NKV, HD = 4096, 12288, 248320, 32, 16, 32, 16, 4, 256
    ch = (2 * HK + HV) * 128
    mixed = plan == "q5_k_m"
    mat = 13 if mixed else 14

    def more_bits(il):
        return il < NL // 8 or il >= 7 * NL // 8 or (il - NL // 8) % 3 == 2

    t = [("token_embd.weight", mat, (E, V)), ("output.weight", 14, (E, V)), ("output_norm.weight", 0, (E,))]

    def attn(il):
        p = f"blk.{il}."
        vt = 14 if not mixed or more_bits(il) else 13
        return [(p + "attn_norm.weight", 0, (E,)), (p + "post_attention_norm.weight", 0, (E,)),
                (p + "attn_q.weight", mat, (E, 2 * NH * HD)), (p + "attn_k.weight", mat, (E, NKV * HD)),
                (p + "attn_v.weight", vt, (E, NKV * HD)), (p + "attn_output.weight", mat, (NH * HD, E)),
                (p + "attn_q_norm.weight", 0, (HD,)), (p + "attn_k_norm.weight", 0, (HD,))]

    def ffn(il):
        p = f"blk.{il}."
        dt = 14 if not mixed or more_bits(il) else 13
        return [(p + "ffn_up.weight", mat, (E, F)), (p + "ffn_gate.weight", mat, (E, F)),
                (p + "ffn_down.weight", dt, (F, E))]

    for il in range(NL):
        p = f"blk.{il}."
        if (il + 1) % 4 == 0:
            t += attn(il)
        else:
            t += [(p + "attn_norm.weight", 0, (E,)), (p + "post_attention_norm.weight", 0, (E,)),
                  (p + "attn_qkv.weight", mat, (E, ch)), (p + "attn_gate.weight", mat, (E, HV * 128)),
                  (p + "ssm_beta.weight", mat, (E, HV)), (p + "ssm_alpha.weight", mat, (E, HV)),
                  (p + "ssm_out.weight", mat, (HV * 128, E)), (p + "ssm_conv1d.weight", 0, (4, ch)),
                  (p + "ssm_dt.bias", 0, (HV,)), (p + "ssm_a", 0, (HV,)), (p + "ssm_norm.weight", 0, (128,))]
        t += ffn(il)
    t += attn(NL) + ffn(NL) + [(f"blk.{NL}.nextn.eh_proj.weight", mat, (2 * E, E))]
    t += [(f"blk.{NL}.nextn.{w}.weight", 0, (E,)) for w in ("enorm", "hnorm", "shared_head_norm")]
    meta = [("general.architecture", 8, "qwen35"), ("qwen35.block_count", 4, NL + 1),
            ("qwen35.nextn_predict_layers", 4, 1), ("qwen35.attention.layer_norm_rms_epsilon", 6, 1e-6),
            ("qwen35.rope.freq_base", 6, 1e7), ("qwen35.rope.dimension_count", 4, 64)]
    return t, meta


BLOCK = {14: 210, 13: 176, 12: 144}   # bytes per 256 weights of Q6_K, Q5_K, Q4_K


def write_synthetic_gguf(path, tensors, meta, seed=7):
    """Stream a GGUF v3 file (the published layout: header, key/values, tensor infos, data aligned to 32): random
    Q6_K / Q5_K / Q4_K blocks with valid fp16 scales, unit norms, ssm_a = -1, small conv taps.  Returns the file
    size."""
    import struct

    import numpy as np
    rng = np.random.default_rng(seed)
    s = lambda x: struct.pack("<Q", len(x.encode())) + x.encode()   # noqa: E731
    fmt = {4: "<I", 6: "<f"}
    kv = b"".join(s(k) + struct.pack("<I", t) + (s(v) if t == 8 else struct.pack(fmt[t], v)) for k, t, v in meta)
    sizes = [(n, tp, d, (int(np.prod(d)) // 256 * BLOCK[tp]) if tp in BLOCK else int(np.prod(d)) * 4)
             for n, tp, d in tensors]
    infos, off, offs = b"", 0, []
    for n, tp, d, nb in sizes:
        infos += s(n) + struct.pack("<I", len(d)) + b"".join(struct.pack("<Q", x) for x in d) + struct.pack("<IQ", tp, off)
        offs.append(off)
        off = (off + nb + 31) // 32 * 32
    head = b"GGUF" + struct.pack("<IQQ", 3, len(tensors), len(meta)) + kv + infos
    with open(path, "wb") as f:
        f.write(head + b"\0" * ((-len(head)) % 32))
        pos = 0
        for (n, tp, d, nb), o in zip(sizes, offs):
            f.write(b"\0" * (o - pos))
            if tp in BLOCK:
                bb = BLOCK[tp]
                for r0 in range(0, nb, bb << 16):           # 65536 blocks at a time
                    blk = rng.integers(0, 256, min(bb << 16, nb - r0), dtype=np.uint8).reshape(-1, bb)
                    if tp == 14:
                        blk[:, 208:210] = np.frombuffer(np.float16(1e-3).tobytes(), np.uint8)
                    else:                                   # d, dmin at the block head
                        blk[:, 0:2] = np.frombuffer(np.float16(2e-3).tobytes(), np.uint8)
                        blk[:, 2:4] = np.frombuffer(np.float16(1e-3).tobytes(), np.uint8)
                    f.write(blk.tobytes())
            else:
                v = np.ones(nb // 4, np.float32)
                if n.endswith("ssm_a"):
                    v[:] = -1.0
                elif n.endswith("conv1d.weight") or n.endswith("dt.bias"):
                    v = (0.1 * rng.standard_normal(nb // 4)).astype(np.float32)
                f.write(v.tobytes())
            pos = o + nb
    return os.path.getsize(path)


def serve_leg(path, n_gen):
    """The --serve protocol through the engine executable on the same file: JSON lines over pipes, the way the
    reference's server drives its engine.  Times a 4096-token ingest (gen 1), then greedy (top-40 list per token) and
    MTP runs of n_gen tokens from a 64-token prompt, each from the request write to its done line."""
    import subprocess

    import numpy as np
    exe = os.path.join(ROOT, "rapier_amd", "rmi_engine")
    if not os.path.exists(exe):
        return {"skipped": "the engine executable is not built"}
    env = dict(os.environ, QWYTHOS_MAXCTX="8192")
    p = subprocess.Popen([exe, "--model", path, "--serve"], stdin=subprocess.PIPE, stdout=subprocess.PIPE,
                         stderr=subprocess.PIPE, text=True, bufsize=1, env=env)
    try:
        seen = []
        for line in p.stderr:                                # the runtime may print notices first
            seen.append(line.strip())
            if "ready" in line or len(seen) > 50:
                break
        if not seen or "ready" not in seen[-1]:
            return {"error": " | ".join(seen)[-300:]}
        rng = np.random.default_rng(3)

        def run(req):
            t0 = time.perf_counter()
            p.stdin.write(json.dumps(req, separators=(",", ":")) + "\n")
            p.stdin.flush()
            ids, t_first = [], None
            while True:
                o = json.loads(p.stdout.readline())
                if "id" in o:
                    ids.append(o["id"])
                    if t_first is None:
                        t_first = time.perf_counter()
                elif "done" in o or "error" in o or "ok" in o:
                    return ids, t_first - t0 if t_first else None, time.perf_counter() - t0, o

        run({"op": "reset"})
        prompt = rng.integers(0, 248320, 4096).tolist()
        _, t_first, _, _ = run({"op": "run", "tokens": prompt, "gen": 1, "mtp": False})
        out = {"ingest_tokens": 4096, "ingest_tok_s": round(4096 / t_first, 1)}
        short = rng.integers(0, 248320, 64).tolist()
        for mtp in (False, True):
            run({"op": "reset"})
            ids, t_first, t_all, done = run({"op": "run", "tokens": short, "gen": n_gen, "mtp": mtp})
            key = "mtp" if mtp else "greedy"
            out[key + "_tok_s"] = round((len(ids) - 1) / (t_all - t_first), 1)
            out[key + "_ids"] = ids
        out["mtp_identical"] = out.pop("mtp_ids") == out.pop("greedy_ids")
        return out
    finally:
        p.stdin.close()
        p.wait(timeout=120)


def run_gguf_load(args):
    """Load a 9B-class qwen35 GGUF (written to local disk first, so the load reads the page cache) through
    rmi_engine_create_gguf and decode from it; then serve from the same file through the engine executable."""
    import tempfile

    import torch

    import rapier_amd.engine as E
    torch.cuda.set_device(0)
    stream = torch.cuda.Stream(device=0)
    torch.cuda.set_stream(stream)
    import shutil
    tensors, meta = qwen35_9b_tensors(args.plan)
    tmp = os.environ.get("TMPDIR", "/tmp")
    if shutil.disk_usage(tmp).free < 16e9:
        print(json.dumps({"workload": "gguf_load", "skipped": f"less than 16 GB free under {tmp}"}), flush=True)
        return
    with tempfile.TemporaryDirectory(dir=tmp) as d:
        path = os.path.join(d, "qwen35-9b-synthetic.gguf")
        t0 = time.perf_counter()
        size = write_synthetic_gguf(path, tensors, meta)
        t_write = time.perf_counter() - t0
        print(f"gguf written: {size / 1e9:.2f} GB in {t_write:.1f} s", file=sys.stderr, flush=True)
        t0 = time.perf_counter()
        eng = E.Engine.from_gguf(path, max_ctx=4096 + 512, stream=stream)
        t_load = time.perf_counter() - t0
        info = eng.info()
        first = eng.prefill(list(range(1000, 1064)), batch=16)
        pos0, cur0 = eng.state()
        eng.save_state()
        n = args.steps
        ref, st_g = eng.generate(n, mode=E.GREEDY)
        eng.restore_state(pos0, cur0)
        toks, st_m = eng.generate(n, mode=E.MTP)
        eng.close()
        torch.cuda.synchronize()
        print(f"in-process decode done; serving from the file", file=sys.stderr, flush=True)
        serve = serve_leg(path, n)
    print(json.dumps({"workload": "gguf_load", "plan": args.plan, "file_bytes": size, "load_s": round(t_load, 3),
                      "load_GB_s": round(size / t_load / 1e9, 2), "write_s": round(t_write, 2),
                      "round_weight_bytes": info["round_weight_bytes"], "first_token": first,
                      "greedy_tok_s": round(n / (st_g["gpu_ms"] / 1e3), 1),
                      "mtp_tok_s_natural": round(n / (st_m["gpu_ms"] / 1e3), 1), "mtp_identical": toks == ref,
                      "serve": serve,
                      "note": "random K-quant blocks, unit norms: a load and shape check, not a trained model (draft "
                              "acceptance near 0); the file is read from the page cache right after it was written; "
                              "serve rates are wall-clock over pipes, from the first token line to the done line"}),
          flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200, help="timed verify rounds per run (mtp_round) or GEMV pairs")
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--workload", default="mtp_round",
                    choices=["mtp_round", "verify_gemv", "traffic_probe", "gguf_load", "kernels", "round", "ingest"])
    ap.add_argument("--shapes", default="", help="kernels: comma-separated indices of the GEMV shapes to run")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--plan", default="q6_k", choices=["q6_k", "q5_k_m"], help="gguf_load: the file's type plan")
    ap.add_argument("--ctx", default="4096,65536",
                    help="comma-separated context lengths for mtp_round; value is quoted at the first")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print(f"bench.py: this build measures one MI355X; --gpus {args.gpus} is not supported: the path runs on one GPU "
              f"in this build", file=sys.stderr)
        sys.exit(2)
    if args.workload == "traffic_probe":
        run_traffic_probe()
        return
    if args.workload == "gguf_load":
        run_gguf_load(args)
        return
    if args.workload == "kernels":
        run_kernels(args)
        return
    if args.workload == "round":
        run_round(args)
        return
    if args.workload == "ingest":
        print(json.dumps({"workload": "ingest", **run_ingest()}), flush=True)
        return
    gemv_args =argparse.Namespace(steps=50 if args.workload == "mtp_round" else args.steps,
                                   warmup=10 if args.workload == "mtp_round" else args.warmup)
    gemv = run_verify_gemv(gemv_args)
    cpu = None if args.no_cpu else cpu_baseline(int(args.ctx.split(",")[0]))
    if args.workload == "verify_gemv":
        gemv["cpu_baseline"] = cpu
        print(json.dumps(gemv), flush=True)
        return
    ctxs = tuple(int(c) for c in args.ctx.split(","))
    table, identical, info = run_mtp_rounds(args, ctxs)
    ingest = run_ingest()
    head = table[str(ctxs[0])]["0.5"]
    out = {
        "metric": METRIC,
        "value": head["tok_s"],
        "unit": "tok/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(head["us_per_round"] / 1e3, 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "int8 dot, f32 accumulate (Q6_K x Q8_1 GEMVs); f32 GDN/attention over fp16 KV",
        "data": "synthetic: seeded random-init Q6_K weights (codes U{0..63}, sc U[-32,31], d=|N(0,1e-3)|); context "
                "state synthesized from a seed (fp16 KV N(0,1), GDN state N(0,0.05^2)), not prefilled",
        "config": {
            "workload": "exact-verify MTP round, random-init 9B-class qwen35 (32 layers: 24 GDN + 8 GQA, hidden 4096, "
                        f"FFN 12288, vocab 248320, nextn draft), one hipGraph per round; value = ctx {ctxs[0]}, "
                        "forced acceptance 0.5",
            "model": "qwen35-9B-class random-init Q6_K",
            "ctx": list(ctxs),
            "forced_acceptance": [0, 0.5, 1.0],
            "runs": table,
            "mtp_stream_identical_to_greedy": identical,
            "round_weight_bytes": info["round_weight_bytes"],
            "token_weight_bytes": info["token_weight_bytes"],
            "kv_bytes_per_pos": info["kv_bytes_per_pos"],
            "round_hbm_frac_at_first_ctx_accept05": round(
                (info["round_weight_bytes"] + info["kv_bytes_per_pos"] * ctxs[0]) /
                (head["us_per_round"] * 1e-6) / 1e9 / HBM_PEAK_GBS, 4),
            "verify_gemv_pair": {"GB_s": gemv["value"], "us_per_pair": gemv["config"]["us_per_pair"],
                                 "hbm_frac_of_peak": gemv["config"]["hbm_frac_of_peak"],
                                 "registry_packed_us_per_pair": gemv["config"]["registry_packed_us_per_pair"],
                                 "registry_packed_hbm_frac_of_peak":
                                     gemv["config"]["registry_packed_hbm_frac_of_peak"]},
            "config1_gpu": gemv["config"]["config1"],
            "ingest": ingest,
            # bounded waits of the GDN layer kernel that ran out in this process (the engine calls fail if any did)
            "gdn_exchange_timeouts": gdn_timeouts(),
        },
        "roofline": gemv["roofline"],
    }
    out["cpu_baseline"] = cpu
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
