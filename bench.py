#!/usr/bin/env python3
"""Benchmark: BASELINE configs[3] on one MI355X.

Workload (one "step"): the 2B hybrid (24 layers, 3:1 gated-delta-net : attention, int4 group-32
weights, random init, vocab 151936) encodes a 512-token state of uniform-random ids once
(Engine::forward with keep), then answers 3 questions of 40 random tokens each from the state's
snapshot (2, 3 and 5 option rows + the last row), the pointer head scoring each.  That is the
reference's Decider::ask_all (src/lib.rs:183-199) on token ids; the three question forwards run as
independent sequences of one batched forward (the same results as three forwards), and the head
(src/head.rs:55-77, f64) runs on the device after it.

Reported: `value` = prefill tokens/s (512-token state forwards), `ask_all_ms` = the latency of
ask_all as sd_ask_ids serves it (one forward of the state with the questions as branches of it,
then the head), `ms_per_step` = the whole step (the snapshot path below, then that ask_all), plus
the snapshot path's phases (prefill_ms: the state's forward with keep; questions_ms: the batched
question forward from the snapshot with the pointer head on the device; their sum
ask_all_snapshot_path_ms), the roofline of the dominant kernel
class (the prefill int4 GEMM, timed live with HIP events on the stream it runs on) and the CPU
baseline (the C oracle on the host cores, a bounded prefill sample of the same model).
"""
import argparse
import json
import os
import statistics
import sys
import tempfile
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

STATE_LEN, N_QUESTIONS, Q_LEN = 512, 3, 40
OPTIONS = [[3, 17], [5, 12, 30], [2, 9, 18, 27, 36]]
PEAK_MFMA_F16 = 2500.0   # TFLOP/s, MI355X dense fp16
PEAK_HBM = 8000.0        # GB/s


def log(*a):
    print(*a, file=sys.stderr, flush=True)


GEMM_LABELS = ("in_proj", "out_proj", "qkv", "o_proj", "gate_up", "down")
TRAFFIC_SUMMARY = os.path.join(ROOT, "profiles", "gemm_w4_prefill_512_traffic.txt")


def gemm_shapes(cfg):
    """(label, N, K) of every int4 GEMM launch of one forward, in plan order (src/engine.rs:475-518)."""
    import sdamd.synth as synth
    d, inter = cfg["hidden_size"], cfg["intermediate_size"]
    H, dv = cfg["linear_num_key_heads"], cfg["linear_value_head_dim"]
    hq, hd = cfg["num_attention_heads"], cfg["head_dim"]
    out = []
    for kind in cfg["layer_types"]:
        if kind == "linear_attention":
            out += [("in_proj", synth.in_proj_rows(cfg), d), ("out_proj", d, H * dv)]
        else:
            out += [("qkv", synth.qkv_rows(cfg), d), ("o_proj", d, hq * hd)]
        out += [("gate_up", 2 * inter, d), ("down", d, inter)]
    return out


def read_traffic():
    """HBM bytes per GEMM launch from the committed rocprofv3 counter summary, or None."""
    try:
        with open(TRAFFIC_SUMMARY) as f:
            for line in f:
                if line.startswith("traffic_bytes_per_launch:"):
                    return float(line.split(":", 1)[1])
    except OSError:
        pass
    return None


def gemm_roofline(eng, state, cfg, reps=5):
    """The prefill int4 GEMM (k_gemm_w4, M = 512) inside the engine's own 512-token forward: each
    GEMM is one launch whose own start and end HIP records into a pair of events on the engine's
    stream (hipExtLaunchKernel, Engine.profile).  achieved = algorithmic flops per launch / average
    launch duration."""
    shapes = gemm_shapes(cfg)
    M = len(state)
    total_ms = []
    for _ in range(reps):
        prof = dict(eng.profile(state))
        total_ms.append(sum(prof[k] for k in GEMM_LABELS))
    ms = statistics.median(total_ms)
    launches = len(shapes)
    avg_s = ms / 1e3 / launches
    flops = sum(2.0 * M * N * K for _, N, K in shapes) / launches
    achieved = flops / avg_s / 1e12
    return {"bound": "mfma", "achieved": round(achieved, 2), "peak": PEAK_MFMA_F16, "unit": "TFLOP/s",
            "frac": round(achieved / PEAK_MFMA_F16, 4), "traffic": read_traffic(),
            # rocprofv3 counters cannot be read from inside this run: traffic is the committed
            # two-pass FETCH_SIZE / WRITE_SIZE measurement of the same prefill GEMMs
            "traffic_source": "profiles/gemm_w4_prefill_512_traffic.txt (rocprofv3 --pmc FETCH_SIZE, WRITE_SIZE "
                              "of bench.py --pmc-workload segment 1, copy-kernel scaled); not measured in this run",
            "kernel": "k_gemm_w4 (int4 g32 fused-dequant MFMA GEMM, prefill M=512, the 2B's 96 GEMMs)",
            "avg_launch_us": round(avg_s * 1e6, 2), "flops_per_launch": flops,
            "algorithmic_bytes_per_launch": sum(N * K // 2 + N * K // 16 + 2 * M * K + 2 * M * N
                                                for _, N, K in shapes) / launches,
            "launches_timed": launches * reps}


def peak_measure(pkg, full=False):
    """Achievable ceilings on this GPU (libsdpeak.so, include/sdpeak.h): the f16 MFMA instruction of
    the prefill GEMM alone and inside the GEMM's own loop mix (dequant + LDS fragments, no memory
    traffic), for about 50 ms of back-to-back launches (the clock a sustained workload gets; the
    benchmark's steps run back to back), each on patterned operands (few switching bits: the
    instruction rate) and on random ones (the power-limited clock a GEMM on real data runs at), and
    streaming HBM reads.  full: also 20-us and 2-ms bursts after an idle pause, the (4,1) mix, every
    occupancy and the copy rate (bench.py --peak)."""
    res = {}

    def mfma(variant, wg, us_per_launch, total_ms):
        # calibrate the loop trips per launch from a short launch, then time the real ones
        probe = pkg.peak_mfma(variant, wg, 200, 1)
        per_iter_ms = probe["ms"] / 200
        iters = max(10, int(us_per_launch / 1e3 / per_iter_ms))
        launches = max(1, int(total_ms / (iters * per_iter_ms)))
        r = pkg.peak_mfma(variant, wg, iters, launches)
        r.update(iters=iters, launches=launches)
        return r

    best = None
    for wg in ((1, 2, 3) if full else (1, 2)):
        r = mfma(0, wg, 2000, 50)
        res[f"mfma_sustained_wg{wg}"] = r
        if best is None or r["tflops"] > best["tflops"]:
            best = r
    res["mfma_sustained"] = best
    bestmix = None
    for wg in ((1, 2, 3) if full else (2, 3)):
        r = mfma(1, wg, 2000, 50)
        res[f"gemm_mix_2x1_sustained_wg{wg}"] = r
        if bestmix is None or r["tflops"] > bestmix["tflops"]:
            bestmix = r
    res["gemm_mix_2x1_sustained"] = bestmix
    for name, variant, wgs in (("mfma_random", 3, (1, 2)), ("gemm_mix_2x1_random", 4, (2, 3))):
        b = None
        for wg in ((1, 2, 3) if full else wgs):
            r = mfma(variant, wg, 2000, 50)
            res[f"{name}_sustained_wg{wg}"] = r
            if b is None or r["tflops"] > b["tflops"]:
                b = r
        res[f"{name}_sustained"] = b
    res["hbm_read"] = pkg.peak_hbm(0, 2 << 30, 10)
    if full:
        for wg in (1, 2, 3):
            res[f"gemm_mix_4x1_sustained_wg{wg}"] = mfma(2, wg, 2000, 50)
            res[f"gemm_mix_4x1_random_sustained_wg{wg}"] = mfma(5, wg, 2000, 50)
        time.sleep(0.2)
        res["mfma_burst_20us"] = mfma(0, 2, 20, 0.02)
        time.sleep(0.2)
        res["mfma_burst_2ms"] = mfma(0, 2, 2000, 2)
        res["hbm_copy"] = pkg.peak_hbm(1, 2 << 30, 10)
    return res


def _marker():
    """A one-element fill kernel of torch's: separates the segments of a profiled run."""
    import torch
    torch.ones(1, device="cuda")
    torch.cuda.synchronize()


def pmc_workload(eng, head, state, questions, temp, pkg):
    """What the rocprofv3 counter runs profile, in segments separated by marker kernels:
    0. a plain copy kernel of known size (torch.neg over 256 MiB of f32: 256 MiB read + 256 MiB
       written), which calibrates FETCH_SIZE and WRITE_SIZE;
    1. one eager 512-token prefill (the launches the roofline times);
    2. the same prefill from its captured graph, keeping the snapshot;
    3. the batched question forward of ask_all (3 x 40 tokens from the snapshot) and the device head;
    4. configs[1] at M = 8 (the seven GEMV-class GEMMs) and configs[2] (one gated delta net layer)."""
    import numpy as np
    import torch
    import sdamd.synth as synth
    n = 64 << 20
    src = torch.empty(n, dtype=torch.float32, device="cuda")  # contents do not matter to byte counts
    dst = torch.empty_like(src)
    for _ in range(3):
        torch.neg(src, out=dst)
    torch.cuda.synchronize()
    del src, dst
    _marker()
    eng.profile(state)
    _marker()
    snap = eng.forward(state, [], keep=True).snapshot
    _marker()
    eng.ask_batch(head, questions, OPTIONS, [temp] * len(questions), cache=snap)
    snap.free()
    _marker()
    st = torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(0)
    for _, N, K in CFG1_LAYER:
        M = 8
        dA = _dev(rng.standard_normal((M, K)).astype(np.float16))
        dW = _dev(synth.pack_nibbles(rng.integers(0, 16, size=(N, K), dtype=np.uint32)))
        dS = _dev(rng.uniform(0.005, 0.02, size=(N, K // 32)).astype(np.float16))
        dY = torch.empty(M * N * 2, dtype=torch.uint8, device="cuda")
        pkg.op_repack_w4(dW.data_ptr(), dS.data_ptr(), N, K, st)
        pkg.op_matmul(dA.data_ptr(), dW.data_ptr(), dS.data_ptr(), dY.data_ptr(), M, N, K, True, -1, True, st)
    torch.cuda.synchronize()
    g = _gdn_inputs(rng)
    pkg.op_gdn(*g["args"], st)
    torch.cuda.synchronize()
    log(f"pmc workload done: copy kernel of {4 * n} bytes each way, {len(state)}-token prefill (eager, graph), "
        f"{len(questions)} batched questions, configs[1] at M = 8, configs[2]")


# the GEMM set of one decoder layer (name, N, K)
CFG1_LAYER = [("q", 2048, 2048), ("k", 512, 2048), ("v", 512, 2048), ("o", 2048, 2048), ("gate", 6144, 2048),
              ("up", 6144, 2048), ("down", 2048, 6144)]
GDN_T, GDN_H, GDN_DK, GDN_DV = 512, 16, 128, 128


def _gdn_inputs(rng):
    """q, k L2-normalized per head (the kernel normalizes again), v ~ N(0,1); a, b ~
    N(0,1) with negA = -1 and dt_bias = 0 (g = -softplus(a), beta = sigmoid(b)); zero state."""
    import numpy as np
    import torch
    T, H, dk, dv = GDN_T, GDN_H, GDN_DK, GDN_DV
    C = 2 * H * dk + H * dv
    qkv = rng.standard_normal((T, C)).astype(np.float32)
    for j in range(2 * H):
        blk = qkv[:, j * dk:(j + 1) * dk]
        blk /= np.linalg.norm(blk, axis=1, keepdims=True)
    big = np.zeros((T, 2 * H), np.float16)
    big[:, :H] = rng.standard_normal((T, H)).astype(np.float16)
    big[:, H:] = rng.standard_normal((T, H)).astype(np.float16)
    keep = {"qkv": _dev(qkv), "big": _dev(big), "nA": _dev(np.full(H, -1.0, np.float32)),
            "dtb": _dev(np.zeros(H, np.float32)),
            "state": _dev(np.zeros(H * dk * dv, np.float32)),
            "o": torch.empty(T * H * dv, dtype=torch.float32, device="cuda")}
    keep["args"] = (keep["qkv"].data_ptr(), keep["big"].data_ptr(), 2 * H, 0, H, keep["nA"].data_ptr(),
                    keep["dtb"].data_ptr(), T, H, dk, dv, keep["state"].data_ptr(), 0, keep["o"].data_ptr())
    return keep


def _kernel_short(name):
    """k_gemm_w4m<2,1,false,true,1> from the (demangled or mangled) kernel name."""
    import re
    m = re.match(r"_ZN2sd12_GLOBAL__N_1(\d+)", name)
    if m:  # mangled: length-prefixed name, then I<template args>E of integer/bool literals
        n = int(m.group(1))
        base = name[m.end():m.end() + n]
        rest = name[m.end() + n:]
        if rest.startswith("I"):
            args = re.findall(r"L([ib])(\d+)E", rest[:rest.find("EE") + 2])
            base += "<" + ",".join(v if t == "i" else ("true" if v == "1" else "false") for t, v in args) + ">"
        return base
    name = name.replace("void ", "").replace("sd::(anonymous namespace)::", "")
    return name.split("(")[0]


def _is_marker(name):
    """torch's fill kernel (torch.ones(1) in _marker); the workloads launch no other fill."""
    return "FillFunctor" in name


def _segments(rows):
    """rows: [(order, kernel name, payload)] of one profiled run of --pmc-workload, in dispatch
    order -> the dispatches of its segments (split at the marker kernels; the copy kernel is
    segment 0)."""
    segs, cur = [], []
    for r in rows:
        if _is_marker(r[1]):
            segs.append(cur)
            cur = []
        else:
            cur.append(r)
    segs.append(cur)
    return segs


def _algorithmic(cfg, seg, dispatches):
    """Algorithmic bytes (and MFMA flops for the GEMMs) of each dispatch of a --pmc-workload
    segment: [(bytes or None, flops or None)].  The GEMM launches follow the plan order of
    gemm_shapes(); the per-layer kernels of the 2B have fixed shapes (L tokens after P)."""
    d, inter = cfg["hidden_size"], cfg["intermediate_size"]
    H, dk, dv = cfg["linear_num_key_heads"], cfg["linear_key_head_dim"], cfg["linear_value_head_dim"]
    hq, hk, hd = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
    C = 2 * H * dk + H * dv
    if seg in (1, 2):
        L, P, shapes = STATE_LEN, 0, gemm_shapes(cfg)
    elif seg == 3:
        L, P, shapes = N_QUESTIONS * Q_LEN, STATE_LEN, gemm_shapes(cfg)
    else:
        L, P, shapes = 8, 0, [(n, N, K) for n, N, K in CFG1_LAYER]
    gi, out = 0, []
    for name in dispatches:
        k = _kernel_short(name)
        b = f = None
        if k.startswith("k_gemm_w4") or k.startswith("k_gemv"):
            if gi < len(shapes):
                _, N, K = shapes[gi]
                b = N * K // 2 + N * K // 16 + 2 * L * K + 2 * L * N
                f = 2.0 * L * N * K
            gi += 1
        elif seg == 4 and k.startswith("k_gdn_prep"):
            T = GDN_T
            b = 4 * T * GDN_H * (2 * GDN_DK + GDN_DV) + 4 * T * GDN_H
        elif seg == 4 and k.startswith("k_gdn_scan"):
            T = GDN_T
            b = 4 * T * GDN_H * GDN_DV + 4 * GDN_H * GDN_DK * GDN_DV
        elif k.startswith("k_gdn_prep"):  # q, k, v (f32), a, b (f16) in
            b = 4 * L * C + 4 * L * H
        elif k.startswith("k_gdn_scan"):  # o out, the state in (with a prefix) and out
            b = 4 * L * H * dv + 4 * H * dk * dv * (2 if P else 1)
        elif k.startswith("k_gdn_recur"):
            b = 4 * L * C + 4 * L * H + 4 * L * H * dv + 4 * H * dk * dv * (2 if P else 1)
        elif k.startswith("k_conv"):  # f16 channels in, f32 out, 4 taps per channel, the history
            b = 2 * L * C + 4 * L * C + 16 * C + 2 * 3 * C
        elif k.startswith("k_gnorm"):  # o f32 + z f16 in, f16 out
            b = L * H * dv * (4 + 2 + 2) + 4 * dv
        elif k.startswith("k_add_norm"):  # x f32 in and out, y f16 in, h f16 out
            b = L * d * (4 + 4 + 2 + 2) + 4 * d
        elif k.startswith("k_qk_prep"):  # q, gate-free k, v f16 in; Q, K, V f16 out
            b = 2 * L * (hq * hd + 2 * hk * hd) * 2
        elif k.startswith(("k_attn<", "k_attn_rows<")):  # Q, gate in; K, V of P + L keys; out f16
            b = 2 * L * hq * hd * 3 + 2 * (P + L) * hk * hd * 2
        out.append((b, f))
    return out


def counter_summary(trace_dir, pmc_dirs, cfg):
    """Per-kernel counter evidence for one --pmc-workload run: durations from a --kernel-trace run,
    FETCH_SIZE / WRITE_SIZE scaled by the copy kernel's known bytes, and the SQ / GRBM counters
    (MFMA busy cycles and f16 flops, LDS bank conflicts) from the other --pmc runs, per segment
    and kernel."""
    import csv
    import glob
    trace = []
    for path in glob.glob(os.path.join(trace_dir, "**", "*kernel_trace.csv"), recursive=True):
        with open(path) as f:
            for r in csv.DictReader(f):
                trace.append((int(r["Start_Timestamp"]), r["Kernel_Name"], (int(r["End_Timestamp"]) - int(r["Start_Timestamp"])) / 1e3))
    trace.sort()
    tsegs = _segments(trace)
    counters = {}  # counter -> segments of [(order, name, value)]
    for d in pmc_dirs:
        per = {}
        for path in glob.glob(os.path.join(d, "**", "*counter_collection.csv"), recursive=True):
            with open(path) as f:
                for r in csv.DictReader(f):
                    key = int(r.get("Dispatch_Id") or r.get("Correlation_Id"))
                    per.setdefault(r["Counter_Name"], {}).setdefault(key, [r["Kernel_Name"], 0.0])
                    per[r["Counter_Name"]][key][1] += float(r["Counter_Value"])
        for cn, disp in per.items():
            rows = [(k, v[0], v[1]) for k, v in sorted(disp.items())]
            counters[cn] = _segments(rows)
    copy_bytes = 4 * (64 << 20)
    scale = {}
    for cn in ("FETCH_SIZE", "WRITE_SIZE"):
        if cn in counters:
            cp = [v for _, k, v in counters[cn][0] if "neg_kernel" in k]
            scale[cn] = copy_bytes / (statistics.median(cp) * 1024) if cp else None
    names = ["", "eager 512-token prefill", "512-token prefill from its graph (keep)",
             f"batched question forward ({N_QUESTIONS} x {Q_LEN} tokens after {STATE_LEN}) + device head",
             "configs[1] at M = 8 (GEMV) and configs[2] (one gated delta net layer)"]
    print("# per-kernel counters (rocprofv3 --pmc, one pass per counter group) and durations (--kernel-trace)")
    print("# FETCH/WRITE scaled by the copy kernel: " +
          ", ".join(f"{cn} x{v:.4f}" for cn, v in scale.items() if v))
    print("# columns: dispatches, avg us (trace), algorithmic MB / dispatch, counter HBM MB / dispatch (FETCH + WRITE),")
    print("#   algorithmic GB/s and its fraction of 8 TB/s, MFMA busy % (SQ_VALU_MFMA_BUSY_CYCLES / (GRBM_GUI_ACTIVE x 1024")
    print("#   SIMDs)), f16 MFMA TFLOP/s from SQ_INSTS_VALU_MFMA_MOPS_F16 x 512 / trace duration and its fraction of")
    print("#   2.5 PFLOP/s, LDS bank-conflict cycles per LDS-active cycle")
    for si in range(1, len(tsegs)):
        tseg = tsegs[si]
        if not tseg:
            continue
        alg = _algorithmic(cfg, si, [n for _, n, _ in tseg])
        cseg = {cn: (segs[si] if si < len(segs) else []) for cn, segs in counters.items()}
        agg = {}
        for i, (_, name, us) in enumerate(tseg):
            a = agg.setdefault(_kernel_short(name), {"n": 0, "us": 0.0, "alg": 0.0, "alg_n": 0, "fl": 0.0, "idx": []})
            a["n"] += 1
            a["us"] += us
            a["idx"].append(i)
            if alg[i][0] is not None:
                a["alg"] += alg[i][0]
                a["alg_n"] += 1
            if alg[i][1] is not None:
                a["fl"] += alg[i][1]

        def csum(cn, idx):
            rows = cseg.get(cn) or []
            if len(rows) != len(tseg):
                return None  # the counter run does not line up with the trace (missing dispatches)
            return sum(rows[i][2] for i in idx)

        print()
        print(f"## segment {si}: {names[si] if si < len(names) else ''}: {len(tseg)} dispatches, "
              f"{sum(u for _, _, u in tseg):.1f} us of kernels")
        print(f"  {'kernel':36s} {'n':>4s} {'avg us':>8s} {'alg MB':>8s} {'hbm MB':>8s} {'alg GB/s':>9s} "
              f"{'of HBM':>7s} {'mfma %':>7s} {'TFLOP/s':>8s} {'of MFMA':>8s} {'lds cf':>7s}")
        for k, a in sorted(agg.items(), key=lambda kv: -kv[1]["us"]):
            n, us = a["n"], a["us"]
            algmb = a["alg"] / a["alg_n"] / 1e6 if a["alg_n"] else None
            fe, wr = csum("FETCH_SIZE", a["idx"]), csum("WRITE_SIZE", a["idx"])
            hbm = ((fe * scale["FETCH_SIZE"] + wr * scale["WRITE_SIZE"]) * 1024 / n / 1e6
                   if fe is not None and wr is not None and scale.get("FETCH_SIZE") and scale.get("WRITE_SIZE") else None)
            gbs = a["alg"] / (us * 1e-6) / 1e9 if a["alg_n"] == n else None
            busy, gui = csum("SQ_VALU_MFMA_BUSY_CYCLES", a["idx"]), csum("GRBM_GUI_ACTIVE", a["idx"])
            mfma = 100 * busy / (gui / 8 * 1024) if busy is not None and gui else None
            mops = csum("SQ_INSTS_VALU_MFMA_MOPS_F16", a["idx"])
            tf = mops * 512 / (us * 1e-6) / 1e12 if mops else None
            bc, la = csum("SQ_LDS_BANK_CONFLICT", a["idx"]), csum("SQ_LDS_IDX_ACTIVE", a["idx"])
            cf = bc / la if bc is not None and la else None

            def fm(v, w, p):
                return f"{v:{w}.{p}f}" if v is not None else f"{'-':>{w}s}"
            print(f"  {k[:36]:36s} {n:4d} {us / n:8.2f} {fm(algmb, 8, 2)} {fm(hbm, 8, 2)} {fm(gbs, 9, 0)} "
                  f"{fm(gbs / PEAK_HBM if gbs else None, 7, 3)} {fm(mfma, 7, 1)} {fm(tf, 8, 1)} "
                  f"{fm(tf / PEAK_MFMA_F16 if tf else None, 8, 3)} {fm(cf, 7, 3)}")
        fl = sum(a["fl"] for a in agg.values())
        gus = sum(a["us"] for k, a in agg.items() if k.startswith("k_gemm_w4") or k.startswith("k_gemv"))
        if fl and gus:
            print(f"  GEMMs: {fl / 1e9:.1f} GFLOP in {gus:.1f} us = {fl / gus / 1e6:.1f} TFLOP/s "
                  f"({fl / gus / 1e6 / PEAK_MFMA_F16:.3f} of 2.5 PFLOP/s)")


def traffic_summary(fetch_dir, write_dir, cfg, state_len):
    """Reads the per-dispatch FETCH_SIZE and WRITE_SIZE (KiB) of the two counter runs, scales each
    by the ratio of the copy kernel's known bytes to its counter reading, and prints the summary
    that read_traffic() parses."""
    import csv
    import glob

    def per_kernel(d, counter):
        disp = {}
        for path in glob.glob(os.path.join(d, "**", "*counter_collection.csv"), recursive=True):
            with open(path) as f:
                for r in csv.DictReader(f):
                    if r["Counter_Name"] == counter:
                        key = int(r.get("Dispatch_Id") or r.get("Correlation_Id"))
                        disp.setdefault(key, [r["Kernel_Name"], 0.0])[1] += float(r["Counter_Value"])
        if not disp:
            raise SystemExit(f"no {counter} rows under {d}")
        segs = _segments([(k, v[0], v[1]) for k, v in sorted(disp.items())])
        copy = [v for _, k, v in segs[0] if "neg_kernel" in k]
        # segment 1: the eager prefill whose GEMM launches the roofline times
        gemm = [v for _, k, v in (segs[1] if len(segs) > 1 else []) if "k_gemm_w4" in k]
        if not copy or not gemm:
            raise SystemExit(f"{counter}: copy kernel or GEMM dispatches missing under {d}")
        return statistics.median(copy), sum(gemm) / len(gemm), len(gemm)

    copy_bytes = 4 * (64 << 20)
    fc, fg, nf = per_kernel(fetch_dir, "FETCH_SIZE")
    wc, wg, nw = per_kernel(write_dir, "WRITE_SIZE")
    kf, kw = copy_bytes / (fc * 1024), copy_bytes / (wc * 1024)
    traffic = fg * 1024 * kf + wg * 1024 * kw
    shapes = gemm_shapes(cfg)
    alg = sum(N * K // 2 + N * K // 16 + 2 * state_len * K + 2 * state_len * N for _, N, K in shapes) / len(shapes)
    print(f"# HBM traffic of k_gemm_w4 in one eager {state_len}-token prefill of the 2B (rocprofv3 --pmc; segment 1 "
          "of the --pmc-workload run)")
    print("# commands (R = repository root, run from /tmp):")
    print("#   rocprofv3 --pmc FETCH_SIZE --output-format csv -d FETCH_DIR -o run -- python3 $R/bench.py --pmc-workload")
    print("#   rocprofv3 --pmc WRITE_SIZE --output-format csv -d WRITE_DIR -o run -- python3 $R/bench.py --pmc-workload")
    print("#   python3 $R/bench.py --traffic-summary FETCH_DIR WRITE_DIR")
    print(f"# copy kernel (torch.neg, {copy_bytes} B each way): FETCH_SIZE {fc:.1f} KiB -> factor {kf:.4f}; "
          f"WRITE_SIZE {wc:.1f} KiB -> factor {kw:.4f}")
    print(f"# k_gemm_w4: {nf} dispatches, mean FETCH_SIZE {fg:.1f} KiB, mean WRITE_SIZE {wg:.1f} KiB")
    print(f"# algorithmic bytes per launch (weights + scales + A + Y as f16): {alg:.0f}")
    print(f"fetch_bytes_per_launch: {fg * 1024 * kf:.0f}")
    print(f"write_bytes_per_launch: {wg * 1024 * kw:.0f}")
    print(f"traffic_bytes_per_launch: {traffic:.0f}")


def trace_summary(trace_dir):
    """Per-kernel totals of a `rocprofv3 --kernel-trace` run of this script, then the kernels of the
    last state prefill, of the last batched question forward and of the last one-forward ask_all,
    then the GEMM launches of the roofline's eager forwards.  Each forward starts with one k_embed
    launch; a step's forwards are prefill, questions, ask_all; the roofline's forwards follow a
    marker kernel of torch's."""
    import csv
    import glob
    rows = []
    for path in glob.glob(os.path.join(trace_dir, "**", "*kernel_trace.csv"), recursive=True):
        with open(path) as f:
            for r in csv.DictReader(f):
                rows.append((int(r["Start_Timestamp"]), int(r["End_Timestamp"]), r["Kernel_Name"]))
    if not rows:
        raise SystemExit(f"no kernel_trace.csv under {trace_dir}")
    rows.sort()

    short = _kernel_short

    def table(rs, title):
        agg = {}
        for s, e, k in rs:
            a = agg.setdefault(short(k), [0, 0.0])
            a[0] += 1
            a[1] += (e - s) / 1e3
        busy = sum(v[1] for v in agg.values())
        print(title)
        print(f"  {'kernel':44s} {'calls':>6s} {'total us':>10s} {'avg us':>8s} {'%':>6s}")
        for k, (n, us) in sorted(agg.items(), key=lambda kv: -kv[1][1]):
            print(f"  {k:44s} {n:6d} {us:10.1f} {us / n:8.2f} {100 * us / busy:6.2f}")
        return busy

    table(rows, "# per-kernel totals over the whole run")

    is_marker = _is_marker
    mark = next((i for i, r in enumerate(rows) if is_marker(r[2])), len(rows))
    steps_rows, roof_rows = rows[:mark], [r for r in rows[mark:] if not is_marker(r[2])]
    starts = [i for i, r in enumerate(steps_rows) if "k_embed" in r[2]]
    fwd = [steps_rows[a:b] for a, b in zip(starts, starts[1:] + [len(steps_rows)])]
    for kind, idx in (("state prefill", range(0, len(fwd), 3)), ("batched question forward", range(1, len(fwd), 3)),
                      ("ask_all forward (the state with the questions as its branches)", range(2, len(fwd), 3))):
        idx = list(idx)
        if not idx:
            continue
        f = fwd[idx[-1]]
        print()
        span = (f[-1][1] - f[0][0]) / 1e3
        busy = table(f, f"# one {kind} (last of {len(idx)}): {len(f)} kernels, first start to last end "
                        f"{span:.1f} us")
        print(f"  kernel busy {busy:.1f} us, gaps {span - busy:.1f} us")
        g = [(e - s) / 1e3 for s, e, k in f if "k_gemm_w4" in k]
        if g:
            print(f"  k_gemm_w4 launches in this forward: {len(g)}, average duration {sum(g) / len(g):.2f} us")
    g = [(e - s) / 1e3 for s, e, k in roof_rows if "k_gemm_w4" in k]
    if g:
        n_fwd = sum(1 for r in roof_rows if "k_embed" in r[2])
        print()
        print(f"# roofline: the GEMM launches of its {n_fwd} eager {STATE_LEN}-token forwards (Engine.profile)")
        print(f"  k_gemm_w4 launches: {len(g)}, average duration {sum(g) / len(g):.2f} us")


def _dev(a):
    """numpy array -> device bytes (torch is only the allocator)."""
    import numpy as np
    import torch
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.uint8).reshape(-1).copy()).cuda()


def _timed(fn, reps):
    """Average device ms of fn(stream) over reps calls.  The calls are captured into one graph
    (after an eager warm-up that lets the entry points size their workspaces) and the graph is
    replayed between two events: eager launches through ctypes take several microseconds of host
    time each, which would otherwise be what a microsecond kernel is timed at."""
    import torch
    fn(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        st = torch.cuda.current_stream().cuda_stream
        for _ in range(reps):
            fn(st)
    g.replay()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    best = float("inf")
    for _ in range(3):
        e0.record()
        g.replay()
        e1.record()
        e1.synchronize()
        best = min(best, e0.elapsed_time(e1) / reps)
    return best


def kernel_bench(pkg, reps=50):
    """BASELINE configs[0..2] as kernel-level measurements (parity for them is in tests/): the int4
    GEMM on one linear layer, the GEMM set of one decoder layer at M = 512 and M = 8, and one gated
    delta net layer.  Weights are repacked once (sd_op_repack_w4), as the engine does at load."""
    import numpy as np
    import torch
    import sdamd.synth as synth
    rng = np.random.default_rng(0)
    out = {"metric": "kernel-level configs[0..2] (int4 GEMM, layer GEMM set, gated delta net layer), 1 GPU",
           "unit": "us", "data": "synthetic (BASELINE configs distributions, seed 0)"}

    def gemm(M, N, K):
        A = rng.standard_normal((M, K)).astype(np.float16)
        W = synth.pack_nibbles(rng.integers(0, 16, size=(N, K), dtype=np.uint32))
        S = rng.uniform(0.005, 0.02, size=(N, K // 32)).astype(np.float16)
        dA, dW, dS = _dev(A), _dev(W), _dev(S)
        dY = torch.empty(M * N * 2, dtype=torch.uint8, device="cuda")
        pkg.op_repack_w4(dW.data_ptr(), dS.data_ptr(), N, K, torch.cuda.current_stream().cuda_stream)
        exact = M <= 20
        ms = _timed(lambda st: pkg.op_matmul(dA.data_ptr(), dW.data_ptr(), dS.data_ptr(), dY.data_ptr(), M, N, K, exact,
                                             -1, True, st), reps)
        wbytes = N * K // 2 + N * K // 16
        io = 2 * M * K + 2 * M * N
        return {"M": M, "N": N, "K": K, "us": round(ms * 1e3, 2),
                "tflops": round(2.0 * M * N * K / ms / 1e9, 1),
                "mfma_frac": round(2.0 * M * N * K / ms / 1e9 / PEAK_MFMA_F16, 4),
                "gbps": round((wbytes + io) / ms / 1e6, 1),
                "hbm_frac": round((wbytes + io) / ms / 1e6 / PEAK_HBM, 4)}

    out["cfg0_linear"] = gemm(128, 6144, 2048)
    layer = CFG1_LAYER
    fused = [("qkv", 5120, 2048), ("in_proj", 8256, 2048), ("gate_up", 12288, 2048), ("o", 2048, 2048),
             ("down", 2048, 6144)]
    for M in (512, 8):
        rs = {name: gemm(M, N, K) for name, N, K in layer}
        tot_us = sum(r["us"] for r in rs.values())
        flops = sum(2.0 * M * N * K for _, N, K in layer)
        wbytes = sum(N * K // 2 + N * K // 16 for _, N, K in layer)
        out[f"cfg1_layer_M{M}"] = {"shapes": rs, "total_us": round(tot_us, 2),
                                   "tflops": round(flops / tot_us / 1e6, 1),
                                   "mfma_frac": round(flops / tot_us / 1e6 / PEAK_MFMA_F16, 4),
                                   "weight_gbps": round(wbytes / tot_us / 1e3, 1),
                                   "hbm_frac": round(wbytes / tot_us / 1e3 / PEAK_HBM, 4)}
        if M == 8:
            # the same layer as the engine launches it at M <= 20 (the f32-dequant GEMV): q/k/v (or
            # the GDN layer's in_proj) and gate/up as one fused matrix each; gate_up timed with f16
            # output (the engine applies SiLU * mul in the same kernel's epilogue)
            fz = {name: gemm(M, N, K) for name, N, K in fused}
            att = fz["qkv"]["us"] + fz["o"]["us"] + fz["gate_up"]["us"] + fz["down"]["us"]
            gdn = fz["in_proj"]["us"] + fz["o"]["us"] + fz["gate_up"]["us"] + fz["down"]["us"]
            out["cfg1_fused_M8"] = {"shapes": fz, "attention_layer_us": round(att, 2), "gdn_layer_us": round(gdn, 2)}
        if M == 512:
            out["cfg1_fused_M512"] = {name: gemm(M, N, K) for name, N, K in fused}
            # the vendor library's f16 GEMM (torch.matmul -> hipBLASLt) on the same shapes, with f16
            # weights (4x the weight bytes, no dequant): what the hardware gives a plain GEMM here
            for name, N, K in fused:
                a16 = torch.randn(M, K, dtype=torch.float16, device="cuda")
                b16 = torch.randn(N, K, dtype=torch.float16, device="cuda")
                ms = _timed(lambda st: torch.matmul(a16, b16.t()), reps)
                out["cfg1_fused_M512"][name]["hipblaslt_f16_us"] = round(ms * 1e3, 2)
    # one gated delta net layer (prep + scan), T = 512, 16 heads, dk = dv = 128
    T, H, dk, dv = GDN_T, GDN_H, GDN_DK, GDN_DV
    g = _gdn_inputs(rng)
    ms = _timed(lambda st: pkg.op_gdn(*g["args"], st), reps)
    alg = 4 * T * H * (2 * dk + dv) + 8 * T * H + 4 * T * H * dv + 4 * H * dk * dv
    out["cfg2_gdn_layer"] = {"T": T, "H": H, "us": round(ms * 1e3, 2), "algorithmic_bytes": alg,
                             "gbps": round(alg / ms / 1e6, 1), "hbm_frac": round(alg / ms / 1e6 / PEAK_HBM, 4),
                             "recurrent_equiv_tflops": round(7.0 * T * H * dk * dv / ms / 1e9, 2)}
    return out


def sweep_bench(pkg, eng, head, temp, n_states=64, n_q=8, seed=4):
    """64 independent states of U[128, 2048] random tokens, each encoded once
    (forward with keep), then 8 questions of U[24, 64] tokens answered from its snapshot as one
    batched forward with the device head.  Aggregate prefill tokens/s; per-question latency = the
    wall time of the batch that answers it.  Then each state's ask_all as sd_ask_ids serves it (one
    forward of the state with its 8 questions as branches): its latency per state.  A first pass over
    the same inputs builds the per-length plans (captured graphs) and is reported separately as the
    cold pass."""
    import numpy as np
    import sdamd.synth as synth
    rng = np.random.default_rng(seed)
    work = []
    for _ in range(n_states):
        L = int(rng.integers(128, 2049))
        state = rng.integers(0, synth.VOCAB_2B, L).astype(np.uint32)
        qs = [rng.integers(0, synth.VOCAB_2B, int(rng.integers(24, 65))).astype(np.uint32) for _ in range(n_q)]
        opts = [sorted(rng.choice(len(q) - 1, int(rng.integers(2, 6)), replace=False).tolist()) for q in qs]
        work.append((state, qs, opts))

    def run_pass():
        pre_tok, pre_s, q_lat, a_lat = 0, 0.0, [], []
        for state, qs, opts in work:
            t0 = time.perf_counter()
            snap = eng.forward(state, [], keep=True).snapshot
            t1 = time.perf_counter()
            eng.ask_batch(head, qs, opts, [temp] * n_q, cache=snap)
            t2 = time.perf_counter()
            snap.free()
            pkg.ask_ids(eng, head, state, qs, opts, [temp] * n_q)
            t3 = time.perf_counter()
            pre_tok += len(state)
            pre_s += t1 - t0
            q_lat.extend([t2 - t1] * n_q)
            a_lat.append(t3 - t2)
        q_lat.sort()
        a_lat.sort()
        return pre_tok / pre_s, q_lat, a_lat

    t = time.perf_counter()
    cold_rate, _, _ = run_pass()
    log(f"sweep cold pass (plans built) in {time.perf_counter() - t:.1f} s")
    rate, q_lat, a_lat = run_pass()
    return {"metric": "configs[4] sweep: aggregate prefill tokens/s, per-question latency p50/p99 (ms)",
            "prefill_tokens_per_s": round(rate, 1), "cold_pass_prefill_tokens_per_s": round(cold_rate, 1),
            "states": n_states, "questions_per_state": n_q,
            "question_p50_ms": round(1e3 * q_lat[len(q_lat) // 2], 3),
            "question_p99_ms": round(1e3 * q_lat[min(len(q_lat) - 1, int(0.99 * len(q_lat)))], 3),
            "ask_all_p50_ms": round(1e3 * a_lat[len(a_lat) // 2], 3),
            "ask_all_p99_ms": round(1e3 * a_lat[min(len(a_lat) - 1, int(0.99 * len(a_lat)))], 3),
            "data": "synthetic: random-init 2B, uniform-random ids; lengths U[128, 2048], questions U[24, 64], "
                    "2-5 options each"}


def cpu_baseline(model_dir, vocab, temp, n_tokens=STATE_LEN):
    """The C oracle (a CPU port of the reference kernels) on the host cores, one step of the same
    workload: the prefill of n_tokens random ids with a snapshot (`value` is its tokens/s, the bench
    line's metric), then the 3 x 40-token questions, each from the snapshot, and the f64 pointer head
    (about 12 s on 16 cores)."""
    import numpy as np
    from oracle import torso
    om = torso.OracleModel(model_dir)
    rng = np.random.default_rng(7)
    ids = rng.integers(0, vocab, n_tokens)
    questions = [rng.integers(0, vocab, Q_LEN) for _ in range(N_QUESTIONS)]
    t = time.perf_counter()
    _, snap = om.forward(ids, [n_tokens - 1], keep=True)
    dt = time.perf_counter() - t
    for q, o in zip(questions, OPTIONS):
        hid, _ = om.forward(q, list(o) + [len(q) - 1], cache=snap)
        om.probs(hid, temp)
    dq = time.perf_counter() - t - dt
    return {"value": round(n_tokens / dt, 3), "unit": "tokens/s", "cores": torso.lib().or_num_threads(),
            "kind": "port", "ask_all_ms": round(1e3 * (dt + dq), 1), "questions_ms": round(1e3 * dq, 1),
            "sample": f"one ask_all step on the same 2B model: the prefill of {n_tokens} random tokens "
                      f"({dt:.1f} s) and {N_QUESTIONS} x {Q_LEN}-token questions from its snapshot with the head "
                      f"({dq:.1f} s); the reference's wgpu/lavapipe path cannot be built here: no cargo, no "
                      f"Vulkan ICD"}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--model-dir", default=os.path.join(tempfile.gettempdir(), "sd_bench_2b"))
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-roofline", action="store_true")
    ap.add_argument("--profile", action="store_true", help="also print the per-kernel-label breakdown")
    ap.add_argument("--pmc-workload", action="store_true",
                    help="run only the workload of the rocprofv3 counter runs (copy kernel + one prefill)")
    ap.add_argument("--traffic-summary", nargs=2, metavar=("FETCH_DIR", "WRITE_DIR"),
                    help="print the HBM traffic summary from two rocprofv3 --pmc output folders (no GPU)")
    ap.add_argument("--counter-summary", nargs="+", metavar="DIR",
                    help="TRACE_DIR PMC_DIR...: per-kernel counter summary of --pmc-workload runs (no GPU)")
    ap.add_argument("--trace-summary", metavar="TRACE_DIR",
                    help="print the kernel summary of a rocprofv3 --kernel-trace output folder (no GPU)")
    ap.add_argument("--kernels", action="store_true",
                    help="kernel-level BASELINE configs[0..2] instead of the ask_all workload (one JSON line)")
    ap.add_argument("--peak", action="store_true",
                    help="achievable-peak microbenchmarks (MFMA alone, the GEMM's loop mix, HBM) as one JSON line")
    ap.add_argument("--sweep", action="store_true",
                    help="BASELINE configs[4] (64 states, 8 questions each) instead of the ask_all workload")
    args = ap.parse_args()
    if args.trace_summary:
        trace_summary(args.trace_summary)
        return
    if args.counter_summary:
        import __graft_entry__ as entry
        entry._import_pkg()
        import sdamd.synth as synth
        counter_summary(args.counter_summary[0], args.counter_summary[1:], synth.CONFIG_2B)
        return
    if args.traffic_summary:
        import __graft_entry__ as entry
        entry._import_pkg()
        import sdamd.synth as synth
        traffic_summary(*args.traffic_summary, synth.CONFIG_2B, STATE_LEN)
        return
    if args.gpus != 1:
        print(f"bench.py runs on one GPU only (asked for {args.gpus}): every state and question is independent, "
              "so more GPUs would each run their own requests; there is no multi-GPU path to measure.", file=sys.stderr)
        sys.exit(2)

    import numpy as np
    import torch

    import __graft_entry__ as entry
    pkg = entry._import_pkg()
    pkg.lib()
    import sdamd.synth as synth
    if args.kernels:
        print(json.dumps(kernel_bench(pkg)), flush=True)
        return
    if args.peak:
        r = peak_measure(pkg, full=True)
        r["peak_published"] = {"mfma_f16_tflops": PEAK_MFMA_F16, "hbm_gbps": PEAK_HBM}
        print(json.dumps(r), flush=True)
        return

    t = time.perf_counter()
    model_dir = synth.write_model(args.model_dir, synth.CONFIG_2B, vocab=synth.VOCAB_2B, seed=0)
    log(f"model ready in {time.perf_counter() - t:.1f} s: {model_dir}")
    t = time.perf_counter()
    eng, head, dcfg = pkg.load_decider(model_dir)
    log(f"{eng.adapter}: weights loaded in {time.perf_counter() - t:.1f} s")
    d = eng.hidden_size()
    rng = np.random.default_rng(2026)
    state = rng.integers(0, synth.VOCAB_2B, STATE_LEN).astype(np.uint32)
    questions = [rng.integers(0, synth.VOCAB_2B, Q_LEN).astype(np.uint32) for _ in range(N_QUESTIONS)]
    temp = float(dcfg["temperature"])
    if args.pmc_workload:
        pmc_workload(eng, head, state, questions, temp, pkg)
        return
    if args.sweep:
        print(json.dumps(sweep_bench(pkg, eng, head, temp)), flush=True)
        return

    def step():
        t0 = time.perf_counter()
        out = eng.forward(state, [], keep=True, timed=True)
        t1 = time.perf_counter()
        snap = out.snapshot
        # the questions continue from the snapshot as independent sequences of one batched forward,
        # the pointer head runs on the device behind it
        probs, qgpu = eng.ask_batch(head, questions, OPTIONS, [temp] * N_QUESTIONS, cache=snap, timed=True)
        t2 = time.perf_counter()
        snap.free()
        # ask_all as the library serves it (sd_ask_ids): one forward of the state with the three
        # questions as branches of it, then the device head
        tprobs = pkg.ask_ids(eng, head, state, questions, OPTIONS, [temp] * N_QUESTIONS)
        t3 = time.perf_counter()
        return t1 - t0, t2 - t1, t3 - t2, out.gpu_ms, [qgpu], probs, tprobs

    for i in range(args.warmup):
        step()
        log(f"warmup {i + 1}/{args.warmup} done")
    torch.cuda.synchronize()
    pre, qs, ask, pre_gpu, q_gpu = [], [], [], [], []
    t_start = time.perf_counter()
    for i in range(args.steps):
        a, b, c, g, qg, probs, tprobs = step()
        pre.append(a)
        qs.append(b)
        ask.append(c)
        pre_gpu.append(g)
        q_gpu.extend(qg)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t_start
    log(f"timed {args.steps} steps in {wall:.3f} s")
    snap_ask = [a + b for a, b in zip(pre, qs)]
    # the two ask_all paths agree (the questions' matmul sizes and summation orders differ)
    tree_dp = max(float(abs(x - y).max()) for x, y in zip(probs, tprobs))
    value = STATE_LEN * len(pre) / sum(pre)
    res = {
        "metric": "prefill tokens/s + ask_all latency (ms), 2B hybrid, 512-tok state, 1 GPU",
        "value": round(value, 1),
        "unit": "tokens/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(1e3 * wall / args.steps, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f16 x int4 (f32 accumulate; f32 recurrent state)",
        "data": "synthetic: random-init 2B weights (seed 0), uniform-random token ids",
        "config": {"workload": "configs[3]: 2B hybrid, 512-token state prefill + ask_all of 3 x 40-token questions",
                   "layers": 24, "hidden": d, "vocab": synth.VOCAB_2B, "state_tokens": STATE_LEN,
                   "questions": N_QUESTIONS, "question_tokens": Q_LEN, "options": [len(o) for o in OPTIONS]},
        "ask_all_ms": round(1e3 * statistics.mean(ask), 3),
        "ask_all_p50_ms": round(1e3 * statistics.median(ask), 3),
        "ask_all_snapshot_path_ms": round(1e3 * statistics.mean(snap_ask), 3),
        "ask_all_paths_max_dprob": tree_dp,
        "prefill_ms": round(1e3 * statistics.mean(pre), 3),
        "prefill_gpu_ms": round(statistics.mean(pre_gpu), 3),
        "questions_ms": round(1e3 * statistics.mean(qs), 3),
        "questions_gpu_ms": round(statistics.mean(q_gpu), 3),
        "probs_last_step": [[round(float(x), 5) for x in p] for p in probs],
    }
    if args.profile:
        prof = eng.profile(state)
        res["profile_prefill_ms"] = {k: round(v, 4) for k, v in prof}
        prof_q = eng.profile(questions[0])
        res["profile_question_ms"] = {k: round(v, 4) for k, v in prof_q}
    if not args.no_roofline:
        # a marker kernel of torch's separates the timed steps from the roofline's forwards in a
        # kernel trace of this script (see trace_summary)
        torch.ones(1, device="cuda")
        torch.cuda.synchronize()
        rl = gemm_roofline(eng, state, synth.CONFIG_2B)
        # the achievable ceilings, measured in this run after the timed steps (about 0.4 s)
        pk = peak_measure(pkg)
        a0, a1 = pk["mfma_random_sustained"], pk["gemm_mix_2x1_random_sustained"]
        p0, p1 = pk["mfma_sustained"], pk["gemm_mix_2x1_sustained"]
        rl["achievable"] = round(a0["tflops"], 2)
        rl["achievable_frac"] = round(rl["achieved"] / a0["tflops"], 4)
        rl["achievable_source"] = (f"v_mfma_f32_32x32x16_f16 loop from registers on random f16 operands (the GEMM's "
                                   f"data: random signs and mantissas), {a0['cus']} CUs, about 50 ms of back-to-back "
                                   f"launches: {a0['tflops']:.0f} TFLOP/s at a {a0['clock_ghz']:.2f} GHz shader clock "
                                   f"(libsdpeak.so, measured in this run; on patterned operands the same loop runs "
                                   f"{p0['tflops']:.0f} TFLOP/s at {p0['clock_ghz']:.2f} GHz: the clock is power-limited)")
        rl["achievable_gemm_mix"] = round(a1["tflops"], 2)
        rl["achievable_gemm_mix_frac"] = round(rl["achieved"] / a1["tflops"], 4)
        rl["achievable_gemm_mix_source"] = (f"the GEMM's (2,1) inner loop without memory traffic (int4 dequant, 2 LDS "
                                            f"fragments, 2 MFMAs per word) on random data, sustained: "
                                            f"{a1['tflops']:.0f} TFLOP/s at {a1['clock_ghz']:.2f} GHz (patterned "
                                            f"operands: {p1['tflops']:.0f} at {p1['clock_ghz']:.2f} GHz)")
        rl["hbm_read_achievable_gbps"] = round(pk["hbm_read"]["gbps"], 1)
        res["roofline"] = rl
    if not args.no_cpu_baseline:
        eng.free()
        res["cpu_baseline"] = cpu_baseline(model_dir, synth.VOCAB_2B, temp)
    print(json.dumps(res), flush=True)


if __name__ == "__main__":
    main()
