"""Benchmark of the MI355X W8A8 arctic-embed-s forward pass (one GPU).

A step is one device forward pass over one token-packed batch (256 sequences,
lengths U{16..512} with [CLS]/[SEP], ids U[1000,30522), seed 3) on the seeded
synthetic model.  Inputs are resident in HBM
before the timed region; `value` is embeddings/s over exactly --steps passes.

Also reported: per-kernel device time (HIP events on the workspace stream over
the timed region) and the roofline of the dominant kernel, ms/seq at 128 tokens,
the end-to-end roofline (the sum over launches of each kernel's
ideal time against the measured pass), and the CPU baseline: the oracle's
restatement of the reference's best x86 backend (AVX-VNNI, else AVX2) under the
reference's embed_batch policy on the host's cores.
"""
import argparse
import json
import os
import shutil
import sys
import tempfile
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "snowflake-arctic-embed-s-rust_amd"))

METRIC = "embeddings/sec @ ragged 16\u2013512-tok batch; int8 MFMA % of peak; ms/seq @128"
MODEL_SEED = 0xAE85EED
PEAK_INT8_TOPS = 5000.0    # MI355X dense int8 MFMA
PEAK_FP32_TFLOPS = 157.3   # MI355X dense fp32 MFMA
PEAK_HBM_GBS = 8000.0      # MI355X HBM3E


def make_batch(n, lo, hi, seed):
    rng = np.random.default_rng(seed)
    lens = rng.integers(lo, hi + 1, n)
    return [np.concatenate([[101], rng.integers(1000, 30522, int(L) - 2), [102]]).astype(np.uint16) for L in lens]


# (sequences, shortest, longest, seed) of each workload
SHAPES = {"c1": (1, 128, 128, 1), "c3": (256, 16, 512, 3), "c4": (64, 512, 512, 4), "c5": (8192, 8, 64, 5)}
CONFIGS = {
    "c1": (lambda: make_batch(1, 128, 128, 1), "c1_1x128"),
    "c3": (lambda: make_batch(256, 16, 512, 3), "c3_ragged_256x16-512"),
    "c4": (lambda: make_batch(64, 512, 512, 4), "c4_64x512"),
    "c5": (lambda: make_batch(8192, 8, 64, 5), "c5_8192x8-64"),
}


def kernel_work(kind, T, B, lens):
    """Algorithmic work of one launch of `kind` on a packed batch (unit, amount, bound, peak)."""
    sum_l2 = float(sum(int(L) * int(L) for L in lens))
    if kind == "gemm_ffn_up":
        return "TOPS", 2.0 * T * 1536 * 384, "mfma", PEAK_INT8_TOPS
    if kind == "gemm_ffn_down":
        return "TOPS", 2.0 * T * 384 * 1536, "mfma", PEAK_INT8_TOPS
    if kind == "ffn_fused":  # FFN-up + FFN-down in one kernel
        return "TOPS", 4.0 * T * 1536 * 384, "mfma", PEAK_INT8_TOPS
    if kind == "gemm_qkv":
        return "TOPS", 2.0 * T * 1152 * 384, "mfma", PEAK_INT8_TOPS
    if kind == "gemm_attn_out":
        return "TOPS", 2.0 * T * 384 * 384, "mfma", PEAK_INT8_TOPS
    if kind == "attention":  # QK^T + PV, 12 heads, head_dim 32, f32
        return "TFLOP/s", 4.0 * 12 * 32 * sum_l2, "mfma", PEAK_FP32_TFLOPS
    if kind in ("ln1", "ln2"):  # read f32 row, write f32 row + int8 row + scale
        return "GB/s", T * (384 * 4 * 2 + 384 + 4), "hbm", PEAK_HBM_GBS
    if kind == "embed_ln":  # gather 2 int8 rows + 2 scales, write f32 row + int8 row + scale
        return "GB/s", T * (2 * 384 + 8 + 384 * 4 + 384 + 4), "hbm", PEAK_HBM_GBS
    return None


def roofline_step_ms(T, B, lens, ffn_fused=False, attn_ln_fused=False):
    """Ideal time of one forward pass: the sum over launches of max(ops / peak, bytes / HBM) with
    algorithmic ops and bytes (weights read once per launch), per kernel kind (ms per step).
    ffn_fused: the FFN block is one kernel (int8 A, f32 residual and output, no intermediate), and
    LN2 then stores (mean, rstd) per row instead of its f32 output (the next attention-output
    kernel recomputes it from LN2's input rows).
    attn_ln_fused: the attention output GEMM and LN1 are one kernel (f32 ctx and residual in, the
    LayerNorm's f32 row, int8 row and scale out; no intermediate)."""
    sum_l2 = float(sum(int(L) * int(L) for L in lens))
    hbm = PEAK_HBM_GBS * 1e9

    def gemm(M, N, K, a_bytes, res):
        ops = 2.0 * M * N * K
        byts = a_bytes * M * K + 4 * M + N * K + 8 * N + 4 * M * N * (2 if res else 1)
        return max(ops / (PEAK_INT8_TOPS * 1e12), byts / hbm)

    per = {
        "embed_ln": T * (2 + 2 * 384 + 8 + 384 * 4 + 384 + 4) / hbm,
        "gemm_qkv": 11 * gemm(T, 1152, 384, 1, False),
        "attention": 11 * max(4.0 * 12 * 32 * sum_l2 / (PEAK_FP32_TFLOPS * 1e12), T * (1152 + 384) * 4 / hbm),
        "gemm_attn_out": 11 * gemm(T, 384, 384, 4, True),
        "ln1": 11 * T * (384 * 4 * 2 + 384 + 4) / hbm,
        "gemm_ffn_up": 11 * gemm(T, 1536, 384, 1, False),
        "gemm_ffn_down": 11 * gemm(T, 384, 1536, 4, True),
        "ln2": 11 * T * (384 * 4 + (8 if ffn_fused else 384 * 4) + 384 + 4) / hbm,
        "ffn_fused": 11 * max(4.0 * T * 1536 * 384 / (PEAK_INT8_TOPS * 1e12),
                              (T * (384 + 4 + 2 * 384 * 4) + 2 * 1536 * 384 + 1536 * 12 + 384 * 8) / hbm),
        # layer 11: K/V for all tokens, the [CLS] query's attention over them, then the B-row tail
        "layer11_tail": gemm(T, 768, 384, 1, False) + T * 768 * 4 / hbm
        + gemm(B, 384, 384, 1, False) + gemm(B, 384, 384, 4, True) + gemm(B, 1536, 384, 1, False)
        + gemm(B, 384, 1536, 4, True) + 3 * B * 3460 / hbm,
    }
    for k in (("gemm_ffn_up", "gemm_ffn_down") if ffn_fused else ("ffn_fused",)):
        del per[k]
    if attn_ln_fused:
        per["gemm_attn_out"] = 11 * max(2.0 * T * 384 * 384 / (PEAK_INT8_TOPS * 1e12),
                                        (T * (3 * 384 * 4 + 384 + 8) + 384 * 384 + 384 * 16) / hbm)
        del per["ln1"]
    return {k: v * 1e3 for k, v in per.items()}


def host_cpu():
    """The host's CPU: /proc/cpuinfo's model name with its family / model / stepping numbers
    (some hosts report only a generic name), and the ISA extensions the reference's x86 dispatch
    looks at."""
    info, flags = {}, set()
    try:
        for ln in open("/proc/cpuinfo"):
            k, _, v = ln.partition(":")
            k = k.strip()
            if k in ("model name", "vendor_id", "cpu family", "model", "stepping") and k not in info:
                info[k] = v.strip()
            elif k == "flags" and not flags:
                flags = set(v.split())
    except OSError:
        pass
    model = "%s (%s family %s model %s stepping %s)" % (info.get("model name", "unknown"), info.get("vendor_id", "?"),
                                                         info.get("cpu family", "?"), info.get("model", "?"),
                                                         info.get("stepping", "?"))
    return model, [f for f in ("avx2", "fma", "avx_vnni", "avx512f", "avx512_vnni") if f in flags]


def gemm_microbench(ae, torch, iters):
    """The standalone W8A8 GEMM, f32 output + bias, through the C ABI."""
    rng = np.random.default_rng(2)
    rows = []
    for (k, n) in [(384, 1152), (384, 384), (384, 1536), (1536, 384)]:
        w = rng.integers(-127, 128, (n, k), dtype=np.int8)
        ws_ = rng.uniform(0.0002, 0.0006, n).astype(np.float32)
        bias = rng.normal(0, 0.02, n).astype(np.float32)
        lin = ae.Linear(w, ws_, bias, np.ones(k, np.float32))
        for m in (128, 4096, 32768):
            a = torch.from_numpy(rng.integers(-127, 128, (m, k), dtype=np.int8)).cuda()
            sa = torch.from_numpy(rng.uniform(0.01, 0.1, m).astype(np.float32)).cuda()
            out = torch.empty((m, n), dtype=torch.float32, device="cuda")
            for _ in range(3):
                lin.gemm(m, a.data_ptr(), sa.data_ptr(), None, out.data_ptr())
            torch.cuda.synchronize()
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(iters):
                lin.gemm(m, a.data_ptr(), sa.data_ptr(), None, out.data_ptr())
            e1.record()
            torch.cuda.synchronize()
            us = e0.elapsed_time(e1) * 1e3 / iters
            ops = 2.0 * m * n * k
            byts = m * k + n * k + 4 * m + 8 * n + 4 * m * n
            rows.append({"M": m, "K": k, "N": n, "us": round(us, 2), "TOPS": round(ops / us / 1e6, 1),
                         "mfma_frac": round(ops / us / 1e6 / PEAK_INT8_TOPS, 4),
                         "GBs": round(byts / us / 1e3, 1), "hbm_frac": round(byts / us / 1e3 / PEAK_HBM_GBS, 4)})
        lin.close()
    return rows


def measured_traffic(kind, workload):
    """HBM bytes per launch of `kind` on `workload`, from a committed rocprofv3 --pmc summary
    (profiles/<kind>_<workload>_traffic.txt, line `hbm_bytes_per_launch: N`), or None."""
    path = os.path.join(ROOT, "profiles", "%s_%s_traffic.txt" % (kind, workload))
    try:
        for ln in open(path):
            if ln.startswith("hbm_bytes_per_launch:"):
                return int(float(ln.split(":", 1)[1]))
    except OSError:
        return None
    return None


def load_cpu_oracle():
    """The oracle (scalar restatement of the reference), used only by the cpu_baseline leg."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle as orc
    return orc


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--config", default="c3", choices=sorted(CONFIGS))
    ap.add_argument("--cpu-sample", type=int, default=256, help="sequences of the workload timed on the CPU")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-c1", action="store_true", help="skip the 128-token latency measurement")
    ap.add_argument("--no-quantized", action="store_true", help="skip the quantized-attention mode pass")
    ap.add_argument("--no-embed-batch", action="store_true", help="skip the host-to-host embed_batch measurement")
    ap.add_argument("--gemm", action="store_true", help="run only the standalone GEMM microbench")
    ap.add_argument("--calib-copy-mib", type=int, default=0,
                    help="run one plain device copy of this many MiB first (calibrates rocprofv3 byte counters)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py: runs on exactly one GPU (the forward pass is data-parallel over sequences "
              "with no cross-GPU exchange; --gpus %d is not supported)" % args.gpus, file=sys.stderr)
        sys.exit(2)

    import torch
    import arctic_embed_amd as ae

    if args.gemm:
        rows = gemm_microbench(ae, torch, max(args.steps, 10))
        print(json.dumps({"gemm_microbench": rows}), flush=True)
        return

    tmp = tempfile.mkdtemp(prefix="ae_bench_")
    try:
        ae.write_synthetic_ae8(os.path.join(tmp, "model.ae8"), MODEL_SEED)
        shutil.copyfile(os.path.join(ROOT, "tests", "golden", "vocab.txt"), os.path.join(tmp, "vocab.txt"))
        engine = ae.Engine.from_dir(tmp)
    finally:
        shutil.rmtree(tmp, ignore_errors=True)

    make, workload = CONFIGS[args.config]
    seqs = make()
    lens = [len(s) for s in seqs]
    B, T = len(seqs), int(sum(lens))
    ws = engine.workspace(max(T, 512), B)
    ids_d = torch.from_numpy(np.concatenate(seqs).view(np.int16)).cuda()
    cu_d = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).cuda()
    out_d = torch.zeros((B, 384), dtype=torch.float32, device="cuda")
    stream = torch.cuda.ExternalStream(ws.stream)

    def step():
        engine.forward_packed_device(ws, ids_d.data_ptr(), cu_d.data_ptr(), B, T, out_d.data_ptr(), ws.stream,
                                     max_seq_len=max(lens))

    if args.calib_copy_mib > 0:  # one copy kernel of known size: reads N MiB, writes N MiB
        src = torch.ones(args.calib_copy_mib << 18, dtype=torch.float32, device="cuda")
        dst = torch.empty_like(src)
        torch.cuda.synchronize()
        dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst
    for _ in range(max(2, args.warmup)):  # the second pass captures the forward graph
        step()
    torch.cuda.synchronize()
    # timed region: exactly --steps passes (graph replay), HIP events on the workspace stream
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    ev0.record(stream)
    for _ in range(args.steps):
        step()
    ev1.record(stream)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    gpu_ms = ev0.elapsed_time(ev1)
    # per-kernel device times: the same passes again, launched eagerly with events around each kernel kind
    ws.set_timing(True)
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    ktimes = ws.kernel_times()
    # above 1024 tokens the FFN block is one kernel, timed under gemm_ffn_up (gemm_ffn_down: 0 launches)
    ffn_fused = ktimes["gemm_ffn_down"][1] == 0 and ktimes["gemm_ffn_up"][1] > 0
    if ffn_fused:
        ktimes["ffn_fused"] = ktimes.pop("gemm_ffn_up")
        del ktimes["gemm_ffn_down"]
    ws.set_timing(False)
    ms_per_step = gpu_ms / args.steps
    value = B * args.steps / (gpu_ms / 1e3)
    emb = out_d.cpu().numpy()
    norms_ok = bool(np.all(np.isfinite(emb)) and np.abs(np.linalg.norm(emb.astype(np.float64), axis=1) - 1).max() < 1e-4)

    # roofline of the dominant kernel kind
    kernel_ms = {k: v[0] / max(1, args.steps) for k, v in ktimes.items()}
    dom = max((k for k in kernel_ms if kernel_work(k, T, B, lens)), key=lambda k: kernel_ms[k])
    unit, amount, bound, peak = kernel_work(dom, T, B, lens)
    launches = ktimes[dom][1]
    avg_launch_s = ktimes[dom][0] / 1e3 / max(1, launches)
    achieved = amount / avg_launch_s / (1e9 if unit == "GB/s" else 1e12)
    roofline = {"kernel": dom, "bound": bound, "achieved": round(achieved, 3), "peak": peak,
                "unit": unit, "frac": round(achieved / peak, 4), "traffic": measured_traffic(dom, workload),
                "avg_launch_us": round(avg_launch_s * 1e6, 2), "algorithmic_per_launch": amount}
    # end-to-end: the sum of every kernel's roofline time against the measured pass
    attn_ln_fused = ktimes["ln1"][1] == 0 and ktimes["gemm_attn_out"][1] > 0
    roof = roofline_step_ms(T, B, lens, ffn_fused, attn_ln_fused)
    e2e = {"t_roof_ms": round(sum(roof.values()), 4), "t_measured_ms": round(ms_per_step, 4),
           "frac": round(sum(roof.values()) / ms_per_step, 4),
           "per_kernel_frac": {k: round(roof[k] / kernel_ms[k], 4) for k in roof if kernel_ms.get(k)}}
    # the FFN GEMMs' fraction of dense int8 MFMA peak (the metric's second part)
    ffn = {}
    for k in (("ffn_fused",) if ffn_fused else ("gemm_ffn_up", "gemm_ffn_down")):
        u, a, _, p = kernel_work(k, T, B, lens)
        s = ktimes[k][0] / 1e3 / max(1, ktimes[k][1])
        ffn[k] = round(a / s / 1e12 / p, 4)

    # the reference's ArmSme attention (int8 Q/K/V, int16 P; AE_ATTENTION_QUANTIZED) on the same batch:
    # an optional mode, reported beside the exact path's figures, never as `value`
    quant = None
    if not args.no_quantized:
        ws.set_attention_mode(True)
        for _ in range(max(2, args.warmup)):
            step()
        torch.cuda.synchronize()
        q0, q1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        q0.record(stream)
        for _ in range(args.steps):
            step()
        q1.record(stream)
        torch.cuda.synchronize()
        q_ms = q0.elapsed_time(q1)
        emb_q = out_d.cpu().numpy().astype(np.float64)
        ws.set_timing(True)
        for _ in range(args.steps):
            step()
        torch.cuda.synchronize()
        kq = ws.kernel_times()
        ws.set_timing(False)
        ws.set_attention_mode(False)
        e64 = emb.astype(np.float64)
        cos_q = float(((e64 * emb_q).sum(1) / (np.linalg.norm(e64, axis=1) * np.linalg.norm(emb_q, axis=1))).min())
        quant = {"value": round(B * args.steps / (q_ms / 1e3), 2), "unit": "embeddings/s",
                 "ms_per_step": round(q_ms / args.steps, 4),
                 "attention_ms_per_step": round(kq["attention"][0] / max(1, args.steps), 4),
                 "min_cos_vs_exact": round(cos_q, 6)}

    # The drop-in embed_batch, PCIe included: host ids in, host embeddings out, through the C ABI's
    # ae_embed_batch_tokens on the engine's own workspace (ws = NULL, as the Rust binding calls it:
    # grown once to the request, batches queued with one synchronization), a fresh batch of the
    # workload's distribution every step (new lengths, so no captured graph is replayed). Never `value`.
    eb = None
    if not args.no_embed_batch:
        n_s, lo, hi, seed = SHAPES[args.config]
        fresh = [make_batch(n_s, lo, hi, 1000 + seed * 100 + k) for k in range(args.steps + 2)]
        for b in fresh[:2]:  # growth of the engine's workspace, warm-up
            engine.embed_batch_tokens(None, b)
        t0 = time.perf_counter()
        for b in fresh[2:]:
            emb_h = engine.embed_batch_tokens(None, b)
        eb_s = time.perf_counter() - t0
        n_emb = sum(len(b) for b in fresh[2:])
        n_tok = sum(sum(len(x) for x in b) for b in fresh[2:])
        eb = {"value": round(n_emb / eb_s, 2), "unit": "embeddings/s", "ratio_to_value": round(n_emb / eb_s / value, 4),
              "ms_per_step": round(eb_s * 1e3 / args.steps, 4), "tokens_per_s": round(n_tok / eb_s, 1),
              "steps": args.steps, "outputs_unit_norm": bool(np.abs(np.linalg.norm(
                  emb_h.astype(np.float64), axis=1) - 1).max() < 1e-4),
              "path": "host ids -> ae_embed_batch_tokens(engine, NULL workspace) -> host embeddings; "
                      "fresh lengths each step; wall clock"}

    # ms/seq @ 128 tokens (the metric's third part): single-sequence latency, device-resident input
    c1_ms = None
    if not args.no_c1:
        c1 = make_batch(1, 128, 128, 1)[0]
        ws1 = engine.workspace(512, 1)
        ids1 = torch.from_numpy(c1.view(np.int16)).cuda()
        cu1 = torch.tensor([0, 128], dtype=torch.int32, device="cuda")
        out1 = torch.zeros((1, 384), dtype=torch.float32, device="cuda")
        s1 = torch.cuda.ExternalStream(ws1.stream)
        for _ in range(3):
            engine.forward_packed_device(ws1, ids1.data_ptr(), cu1.data_ptr(), 1, 128, out1.data_ptr(), ws1.stream,
                                         128)
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(s1)
        n1 = 50
        for _ in range(n1):
            engine.forward_packed_device(ws1, ids1.data_ptr(), cu1.data_ptr(), 1, 128, out1.data_ptr(), ws1.stream,
                                         128)
        e1.record(s1)
        torch.cuda.synchronize()
        c1_ms = round(e0.elapsed_time(e1) / n1, 4)
        ws1.close()

    cpu = None
    if not args.no_cpu:
        orc = load_cpu_oracle()
        # all the host cores this process may use (the reference's bin uses available_parallelism,
        # src/bin/arctic_embed.rs:324-326), capped at the 16 CPUs a one-GPU job gets on the GPU box
        usable = len(os.sched_getaffinity(0))
        threads = max(1, min(16, usable))
        sample = seqs[: args.cpu_sample]
        m = None
        tmp = tempfile.mkdtemp(prefix="ae_cpu_")
        try:
            ae.write_synthetic_ae8(os.path.join(tmp, "model.ae8"), MODEL_SEED)
            m = orc.OracleModel(os.path.join(tmp, "model.ae8"))
        finally:
            shutil.rmtree(tmp, ignore_errors=True)
        # the reference's best x86 backend (AVX-VNNI, else AVX2; restated in oracle/x86.c) under its
        # embed_batch policy: warm-up on the first 32 items (src/bin/arctic_embed.rs:338), then the
        # median of 5 full runs; the scalar restatement only on a host without AVX2+FMA
        backend = orc.x86_backend()

        def run(s, n_threads):
            return m.x86_embed_batch_tokens(s, n_threads) if backend else m.embed_batch_tokens(s, n_threads)

        def median_s(fn, reps):
            ts = []
            for _ in range(reps):
                t0 = time.perf_counter()
                fn()
                ts.append(time.perf_counter() - t0)
            return sorted(ts)[reps // 2]

        run(sample[:32], threads)
        ref = run(sample, threads)
        cpu_s = median_s(lambda: run(sample, threads), 5)
        # ms/seq at 128 tokens: one thread, and all threads (the reference's
        # embed_batch gives one sequence to one thread, so more threads cannot shorten it); median of 5
        c1seq = make_batch(1, 128, 128, 1)
        run(c1seq, 1)
        cpu_c1_ms = median_s(lambda: run(c1seq, 1), 5) * 1e3
        cpu_c1_all_ms = median_s(lambda: run(c1seq, threads), 5) * 1e3
        m.close()
        g = emb[: len(sample)].astype(np.float64)
        r = np.asarray(ref, np.float64)
        cos = float(((g * r).sum(1) / (np.linalg.norm(g, axis=1) * np.linalg.norm(r, axis=1))).min())
        cpu_model, isa = host_cpu()
        cpu = {"value": round(len(sample) / cpu_s, 3), "unit": "embeddings/s", "cores": threads, "kind": "port",
               "backend": backend or "scalar", "os_cpu_count": os.cpu_count(), "usable_cpus": usable,
               "tokens_per_s": round(sum(len(s) for s in sample) / cpu_s, 1),
               "ms_per_seq_128_1thread": round(cpu_c1_ms, 3), "ms_per_seq_128_all_threads": round(cpu_c1_all_ms, 3),
               "cpu_model": cpu_model, "isa": isa,
               "sample": "first %d sequences (%d tokens) of the %s batch, median of 5 runs on %d threads (all usable "
                         "CPUs, at most the GPU box's 16 per GPU); restatement of the reference's %s backend under "
                         "its embed_batch policy"
                         % (len(sample), sum(len(s) for s in sample), workload, threads,
                            {"avx_vnni": "AVX-VNNI", "avx2": "AVX2"}.get(backend, "scalar")),
               "gpu_vs_cpu_min_cos": round(cos, 9)}

    line = {
        "metric": METRIC, "value": round(value, 2), "unit": "embeddings/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(ms_per_step, 4), "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "int8", "data": "synthetic",
        "config": {"workload": workload, "n_seqs": B, "tokens": T, "model": "arctic-embed-s synthetic seed 0xAE85EED"},
        "tokens_per_s": round(T * args.steps / (gpu_ms / 1e3), 1),
        "wall_s": round(wall, 4), "outputs_unit_norm": norms_ok,
        "ffn_int8_mfma_frac": ffn, "ms_per_seq_128": c1_ms,
        "kernel_ms_per_step": {k: round(v, 4) for k, v in kernel_ms.items()},
        "roofline": roofline, "e2e_roofline": e2e, "cpu_baseline": cpu, "quantized_attention_mode": quant,
        "embed_batch_pcie": eb,
    }
    print(json.dumps(line), flush=True)
    ws.close()
    engine.close()


if __name__ == "__main__":
    main()
